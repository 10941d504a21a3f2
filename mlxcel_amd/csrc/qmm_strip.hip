// qmm_strip.hip — plan and launch of the strip kernel (qmm_strip.hpp), and
// its bfloat16 instantiations for 4/8-bit affine codes and mxfp4.
#include <algorithm>
#include <cmath>

#include "qmm_strip.hpp"

namespace mlxq {

namespace {

size_t strip_lds(int mt, int nwn, int gs, int64_t experts) {
  const int sr = (8 / nwn) * 128 * strip_wps(mt, nwn);
  return (size_t)2 * mt * 16 * sr * 2 + (size_t)2 * (sr / gs) * (16 * nwn + 16) * 4 + 16 +
         (experts > 0 && experts <= kStripRunsMax ? (size_t)(2 * experts + 9) * 4 : 0);
}

constexpr int kTilesM[5] = {1, 2, 3, 4, 8};  // 16-row activation tiles per pass
// Microseconds of a dense launch on MI355X:
//   start + rounds * passes * (pass + window * windows of a wave) + partial sums
// a pass is longer the fuller the round and where rows of the result cannot
// be written 16 bytes at a time; rounds of workgroups past one count `whole`
// of the way to the next integer (14336 x 4096 in 448 workgroups of 32 rows
// 19.5 us, 8192 x 4096 in 256 of them 10.6).  Fitted to 80000 graph-timed
// launches (5-128 rows, and passes of 128 to 1024; N 64-151936, K 256-14336),
// 4-11% rms; [kTilesM index][log2(nwn)], window 0: not built.
struct StripCost {
  float start, pass, pass_fill, narrow, window, whole, sum, sum_each;
};
constexpr StripCost kCost[5][3] = {
    {{3.6f, 0.4f, 0.4f, 0.6f, 0.94f, 0.64f, 2.3f, 13.9f}, {2.3f, 1.8f, 0.7f, 0.6f, 0.73f, 0.97f, 2.4f, 11.0f}, {3.6f, 0.0f, 0.9f, 0.6f, 0.64f, 0.78f, 2.7f, 1.8f}},
    {{1.9f, 2.6f, 0.5f, 0.6f, 1.38f, 0.93f, 2.2f, 9.5f}, {2.1f, 1.8f, 0.6f, 0.6f, 1.02f, 0.83f, 2.4f, 4.8f}, {3.4f, 0.0f, 0.8f, 0.7f, 0.82f, 0.60f, 2.8f, 2.3f}},
    {{}, {1.8f, 2.4f, 0.7f, 0.7f, 1.32f, 0.94f, 2.3f, 4.7f}, {3.7f, 0.0f, 0.8f, 0.9f, 1.05f, 0.67f, 2.5f, 3.7f}},
    {{}, {1.9f, 2.7f, 0.9f, 0.7f, 1.49f, 0.95f, 2.3f, 3.8f}, {1.9f, 1.9f, 1.3f, 1.0f, 1.12f, 0.95f, 2.7f, 2.9f}},
    {{}, {}, {1.5f, 2.9f, 1.5f, 2.3f, 1.84f, 0.96f, 2.8f, 2.3f}}};
// the same by width of the codes
constexpr float kBitsCost[9] = {1.f, 1.f, 0.97f, 0.99f, 0.97f, 1.04f, 1.03f, 1.f, 1.f};


// Microseconds of a sorted gather spread evenly over its experts:
//   start + rounds * (round + passes * (pass + window * windows of a wave))
// window for 4-bit codes, `bits8` more of it for 8-bit ones and `fill` more in
// a full round.  Fitted to 5900 graph-timed calls on MI355X (8-256 experts of
// N 64-5760, K 512-4096; 8-200 entries each), 8-18% rms.
struct GatherCost {
  int mt, nwn, slots;  // slots: workgroups per CU
  float start, round, pass, narrow, window, bits8, fill, whole;
};
constexpr GatherCost kGather[] = {
    {1, 4, 1, 5.3f, 0.0f, 1.4f, 0.2f, 0.24f, 0.85f, 1.28f, 0.68f}, {2, 2, 1, 3.1f, 0.1f, 2.3f, 0.4f, 0.76f, 0.12f, 0.48f, 0.50f},
    {2, 4, 1, 4.4f, 0.0f, 1.3f, 0.3f, 0.72f, 0.25f, 0.03f, 0.59f}, {3, 2, 2, 2.2f, 0.6f, 2.9f, 0.5f, 1.23f, 0.15f, 0.62f, 0.50f},
    {3, 4, 1, 5.4f, 0.5f, 1.2f, 0.6f, 0.88f, 0.52f, 0.00f, 0.65f}, {8, 4, 1, 3.1f, 2.1f, 1.2f, 0.4f, 1.71f, 0.00f, 0.70f, 0.63f}};

float gather_us(int bits, int64_t N, int64_t B, int64_t E, const StripPlan& p, int cus) {
  for (const GatherCost& c : kGather) {
    if (c.mt != p.mt || c.nwn != p.nwn) continue;
    const float x = (float)(E * p.row_blocks) / (float)(c.slots * cus);
    const float rounds = std::max(1.f, c.whole * std::ceil(x) + (1.f - c.whole) * x);
    const float window = c.window * (bits == 8 ? 1.f + c.bits8 : 1.f) * (1.f + c.fill * std::min(x, 1.f));
    return c.start + rounds * (c.round + mean_passes((double)B / E, 16 * p.mt) * (c.pass + (N % 8 != 0 ? c.narrow : 0.f) + window * p.windows));
  }
  return 0.f;
}

}  // namespace

float mean_passes(double avg, int rows) {
  double sum = 1.0;  // P(more than j passes' entries) over j
  for (int j = 1;; j++) {
    const double more = 0.5 * (1.0 - std::erf((j * (double)rows + 0.5 - avg) / std::sqrt(2.0 * avg)));
    sum += more;
    if (more < 1e-3) return (float)sum;
  }
}

StripPlan strip_plan(int fmt, int bits, int gs, int64_t rows, int64_t N, int64_t K, int64_t experts, int cus,
                     int nwn_req, int mt_req, int ks_req) {
  StripPlan p;
  if (rows < 1 || N < 1 || K < 32 || K % 32 != 0 || K % gs != 0 || (fmt == MXFP4 && gs != 32)) return p;
  if (rows * K * 2 >= ((int64_t)1 << 31) || N * (K / 32) * bits * 4 >= ((int64_t)1 << 31) || N * (K / gs) * 2 >= ((int64_t)1 << 31))
    return p;
  const int64_t per = experts > 0 ? (rows + experts - 1) / experts : rows;
  int lm = per <= 16 ? 0 : per <= 32 ? 1 : per <= 48 ? 2 : per <= 64 ? 3 : 4;
  // an expert's rows spread around the average and are taken 16 mt at a
  // time: 48 at a time measured fastest from 25 to ~100 rows per expert (128
  // experts of 768 x 2048, 32 rows each: 57 us, 79 with 32 at a time, 83 with
  // 64; 64 rows each 100, 118, 137), 32 below that (16 rows each 48.6 us vs
  // 52.3), 128 past it (8 experts of 4096 x 2048, 256 rows each: 114 vs 127
  // with 32)
  if (experts > 0) lm = per <= 11 ? 0 : per <= 24 ? 1 : per <= 100 ? 2 : 4;
  for (int i = 0; i < 5; i++)
    if (mt_req == kTilesM[i]) lm = i;
  const int mt = kTilesM[lm];
  const float passes = experts > 0 ? mean_passes((double)rows / experts, 16 * mt) : (float)((rows + 16 * mt - 1) / (16 * mt));
  float best = 0.f;
  for (int ln = 0; ln < 3; ln++) {
    const int nwn = 1 << ln;
    const StripCost& c = kCost[lm][ln];
    if (c.window == 0.f || (nwn_req > 0 && nwn != nwn_req)) continue;
    const int wps = strip_wps(mt, nwn), sr = (8 / nwn) * 128 * wps;
    if (sr < 2 * gs || strip_lds(mt, nwn, gs, experts) > kQmvLdsMax) continue;
    const int64_t blocks = (N + 16 * nwn - 1) / (16 * nwn);
    const int64_t steps = (K + sr - 1) / sr;
    const int64_t ks_max = experts > 0 ? 1 : ks_req > 0 ? ks_req : std::min<int64_t>(16, std::max<int64_t>(1, cus / blocks));
    for (int64_t ks = ks_req > 0 && experts <= 0 ? ks_req : 1; ks <= ks_max; ks++) {
      const int64_t per_split = (steps + ks - 1) / ks;
      const int64_t ksr = (steps + per_split - 1) / per_split;
      const int64_t windows = (per_split + 1) / 2 * 2 * wps;  // steps run in pairs
      const float x = (float)(blocks * ksr * std::max<int64_t>(experts, 1)) / cus;
      const float rounds = std::max(1.f, c.whole * std::ceil(x) + (1.f - c.whole) * x);
      const bool narrow = N % (ksr > 1 ? 4 : 8) != 0;
      const float us = kBitsCost[bits] * (c.start + rounds * passes * (c.pass + c.pass_fill * std::min(x, 1.f) + (narrow ? c.narrow : 0.f) + c.window * windows) +
                                          (ksr > 1 ? c.sum + c.sum_each * (float)ksr * rows * N * 1e-6f : 0.f));
      if (p.ok && us >= best) continue;
      best = us;
      p.ok = true;
      p.mt = mt;
      p.nwn = nwn;
      p.row_blocks = (int)blocks;
      p.ks = (int)ksr;
      p.k_per_split = (int)std::min<int64_t>(per_split * sr, (int64_t)1 << 30);
      p.windows = (int)(experts > 0 ? windows : windows * (int64_t)passes);
      p.us = us;
      p.lds = strip_lds(mt, nwn, gs, experts);
    }
  }
  if (p.ok && experts > 0) p.us = gather_us(bits, N, rows, experts, p, cus);
  if (p.ok && (p.row_blocks * (int64_t)16 * p.nwn >= ((int64_t)1 << 31) || p.ks > 65535 || experts > 65535)) p.ok = false;
  return p;
}

hipError_t strip_launch(int fmt, int bits, const StripArgs& a_in, const StripPlan& p, hipStream_t stream) {
  if (!p.ok) return hipErrorInvalidValue;
  StripArgs a = a_in;
  a.ks = p.ks;
  a.k_per_split = p.k_per_split;
  const dim3 grid((unsigned)p.row_blocks, (unsigned)(a.rhs ? a.E : p.ks));
  if (a.rhs) {  // bfloat16 4- and 8-bit codes only
    if (fmt == MXFP4 || a.xt != 0 || (bits != 4 && bits != 8)) return hipErrorInvalidValue;
    return bits == 4 ? strip_launch_fmt<AFF4, 4, 0, true>(a, p, grid, stream) : strip_launch_fmt<AFF4, 8, 0, true>(a, p, grid, stream);
  }
  if (fmt == MXFP4) return a.xt == 0 ? strip_launch_fmt<MXFP4, 4, 0>(a, p, grid, stream) : hipErrorInvalidValue;
  if (bits == 4 || bits == 8) {
    if (a.xt != 0) return strip_launch_f16(bits, a, p, grid, stream);
    return bits == 4 ? strip_launch_fmt<AFF4, 4, 0>(a, p, grid, stream) : strip_launch_fmt<AFF4, 8, 0>(a, p, grid, stream);
  }
  return a.xt != 0 ? strip_launch_f16_odd(bits, a, p, grid, stream) : strip_launch_odd(bits, a, p, grid, stream);
}

}  // namespace mlxq
