// qmm_strip.hpp — the strip kernel: quantized matmul of a few to ~100
// activation rows for gfx950, weights dequantized in registers, straight into MFMA operands.
//
//   y[m][n] = sum_k x[m][k] * W[n][k],  W = T(s * q + b)  (affine, T the
//   16-bit type of x, the rounding of the prefill and general kernels) or
//   fp4(q) * 2^(e - 127) (mxfp4, exact), fp32 accumulation, one rounding.
//
// A workgroup of 8 waves owns 16 NWN weight rows: NWN waves along the rows
// (16 each) times 8 / NWN along K.  K goes in windows of 128 positions per
// wave: lane i holds 32 consecutive codes (BITS words, one quantization
// group) of weight row i % 16 at 32 (i / 16), dequantizes them eight at a
// time into the B operand of four v_mfma_f32_16x16x32 and multiplies all MT
// 16-row activation tiles with them, so every code is widened once however
// many activation rows there are.  The sum over k does not care which k a
// lane's eight slots hold as long as both operands agree: the activations
// sit in LDS and each lane reads the chunk its codes belong to.
//
// Activations and scales of one step (SR = 128 WPS (8 / NWN) positions) are
// staged in double-buffered LDS with one barrier per step; a step's loads
// are in flight during the step before it.  Rows of activations are XOR
// swizzled in 16-byte chunks so the 16 rows of an operand read fall on
// distinct banks.  Weights never touch LDS: a ring of RD windows per wave is
// in flight in registers.
//
// What bounds it (MI355X, 14336 x 4096, 3-bit g64, 8 rows, 13.8 us, 62.6 on
// the general tile kernel; timing-only copies with 32 weight rows per workgroup,
// 14.6 us, where 64 are taken now): 7.4 us are left with the dequantization, the
// staging and the weight stream all taken out (launch, first loads, sum over the
// K waves), the dequantization (2.6 VALU per code) adds 2.5, staging and barriers
// 2; the 25.7 MB of weights (3.2 us at 8 TB/s) hide under these.  Per
// 128-position window a wave spends 0.64 us at 16 activation rows, 0.82 at 32,
// 1.05 at 48, 1.12 at 64 and 1.84 at 128 (64 weight rows per workgroup; the
// planner's table in qmm_strip.hip has the others).  Two windows per
// step (one past 16 rows) and a ring of two steps measured best of 1, 2 and
// 4 windows and rings of 2 to 8; two workgroups per CU instead of one
// changed nothing.
//
// Gathers sorted by expert (GATHER): workgroup row y takes expert y, whose
// entries are found by binary search in the sorted indices, 16 MT of them at
// a pass.  Routing that sends much of a batch to a few experts would leave
// their passes to a few workgroups: where one run exceeds a.long_run entries,
// the first a.deal workgroup rows find all runs (strip_runs) and deal the
// passes of all experts out in turn (128 experts of 768 x 2048, 1024 tokens
// top 8 all on the same 8 experts: 309 us without, 82 with; spread evenly 107
// either way).

#pragma once

#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"

namespace mlxq {

typedef float sf32x2 __attribute__((ext_vector_type(2)));
constexpr uint32_t kBigScale = (127u + 100u) << 7;  // exponent field of a bfloat16 2^100

template <int XT>
__device__ __forceinline__ uint32_t strip_pack(float lo, float hi) {
  if constexpr (XT == 0) return __builtin_bit_cast(uint32_t, __builtin_convertvector(sf32x2{lo, hi}, bf16x2));
  else {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(sf32x2{lo, hi}, h2));
  }
}

// Sorted gathers whose longest run is far above the average: every expert's
// entries, found by scanning the indices.  Expert e's run from `at[e]` to
// `at[e + 1]` goes in passes of ROWS entries, the first of them number
// `pass0[e]`; returns the number of passes.  (Called by all 512 threads, E <=
// 512; at: E + 1 words, pass0: E + 8.)  Indices that are not sorted give runs
// that overlap or lack entries, within [0, M].
template <int ROWS>
__device__ __forceinline__ int strip_runs(const StripArgs& a, int t, int* at, int* pass0) {
  const int E = a.E, M = a.M, st = a.rhs_stride > 1 ? 2 : 1;
  for (int e = t; e <= E; e += 512) at[e] = M;
  __syncthreads();
  for (int i0 = t; i0 < M; i0 += 512 * 8) {  // 16 loads in flight
    uint32_t cur[8], prev[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int i = i0 + 512 * u;
      cur[u] = a.rhs[(uint32_t)(min(i, M - 1) * st)];
      prev[u] = a.rhs[(uint32_t)(max(min(i, M) - 1, 0) * st)];
    }
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int i = i0 + 512 * u;
      if (i >= M) break;
      const int c = (int)min(cur[u], (uint32_t)(E - 1)), p = i > 0 ? (int)min(prev[u], (uint32_t)(E - 1)) : -1;
      for (int e = p + 1; e <= c; e++) at[e] = i;  // the first entry of every expert up to c
    }
  }
  __syncthreads();
  const int own = t < E ? (max(0, at[t + 1] - at[t]) + ROWS - 1) / ROWS : 0, lane = t & 63;
  int sum = own;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int v = __shfl_up(sum, d);
    if (lane >= d) sum += v;
  }
  if (lane == 63) pass0[E + (t >> 6)] = sum;
  __syncthreads();
  int before = sum - own, all = 0;
#pragma unroll
  for (int w = 0; w < 8; w++) {
    const int v = pass0[E + w];
    all += v;
    if (w < (t >> 6)) before += v;
  }
  if (t < E) pass0[t] = before;
  return all;
}

template <int FMT, int BITS, int XT, int MT, int NWN, bool GATHER>
__global__ __launch_bounds__(512, 2) void qmm_strip_kernel(const StripArgs a) {
  constexpr bool AFF = FMT != MXFP4;
  constexpr int WPS = strip_wps(MT, NWN);    // windows per wave and step
  constexpr int RD = 2 * WPS;                // windows of weights in flight per wave
  constexpr int NWK = 8 / NWN;               // waves along K
  constexpr int RW = 16 * NWN;               // weight rows per workgroup
  constexpr int SRW = 128 * WPS;             // K positions per wave and step
  constexpr int SR = NWK * SRW;              // K positions per step
  constexpr int U = RD / WPS;                // steps of weights in flight
  constexpr int CPR = SR / 8;                // 16-byte chunks per staged row
  constexpr int XL = MT * 16 * CPR / 512;    // activation loads per thread and step
  constexpr int XROWS = 512 / CPR;           // rows per load pass
  constexpr int XB = MT * 16 * SR * 2;       // bytes of one activation buffer
  constexpr int TP = RW + 16;                // words per group of the scale table
  constexpr int SL = AFF ? (WPS + 1) / 2 : WPS;  // scale loads per thread and step (groups of 32)
  static_assert(RD % (2 * WPS) == 0 && XL >= 1 && XL * 512 == MT * 16 * CPR && CPR <= 512, "step shape");

  extern __shared__ __align__(16) unsigned char lds[];
  const int gs_shift = a.gs_shift;
  const int GS = SR >> gs_shift;             // groups per step (>= 2)
  unsigned char* xs = lds;                   // [2][MT * 16][SR] 16-bit
  uint32_t* tbl = reinterpret_cast<uint32_t*>(lds + 2 * XB);  // [2][GS][TP]

  // set where a scale of 2^100 or more has been staged
  volatile uint32_t* big = reinterpret_cast<volatile uint32_t*>(tbl + 2 * GS * TP);

  const int t = threadIdx.x;
  if (t == 0) *big = 0u;
  __syncthreads();
  const int lane = t & 63, wave = t >> 6;
  const int nwave = __builtin_amdgcn_readfirstlane(wave % NWN), kwave = __builtin_amdgcn_readfirstlane(wave / NWN);
  const int r = lane & 15, q = lane >> 4;
  const int N = a.N, K = a.K;
  const int n0 = blockIdx.x * RW;

  // gathers: workgroup y takes expert y's run of entries; where some run is
  // far above the average, passes y, y + deal, ... of all experts' instead
  int first = 0, end = a.M;
  int64_t e = 0;
  bool even = true;
  int passes = 0;
  volatile int* turn = reinterpret_cast<volatile int*>(big + 1);  // expert, first entry and end of a pass
  int* at = reinterpret_cast<int*>(tbl + 2 * GS * TP) + 4;        // E + 1 words
  int* pass0 = at + a.E + 1;                                      // E + 8
  auto take = [&](int pass) {
    __syncthreads();  // pass0 is written, the last turn read
    if (t < a.E) {
      const int i = (pass - pass0[t]) * (16 * MT), from = at[t], to = at[t + 1];
      if (i >= 0 && from + i < to) {  // one thread's
        turn[0] = t;
        turn[1] = from + i;
        turn[2] = min(to, from + i + 16 * MT);
      }
    }
    __syncthreads();
    e = __builtin_amdgcn_readfirstlane(turn[0]);
    first = __builtin_amdgcn_readfirstlane(turn[1]);
    end = __builtin_amdgcn_readfirstlane(turn[2]);
  };
  if constexpr (GATHER) {
    e = blockIdx.y;
    // A run longer than long_run + half covers some pair of entries long_run
    // apart that starts at a multiple of half.  Every wave looks for itself
    // (64 pairs a time, in flight beside the search): no barrier, and the same
    // answer in all.
    const int half = (a.long_run + 1) / 2, st = a.rhs_stride > 1 ? 2 : 1;
    auto pair_at = [&](int i, uint32_t* v) {  // (past the end: one entry twice, masked by equal)
      v[0] = a.rhs[(uint32_t)(min(i, a.M - 1) * st)];
      v[1] = a.rhs[(uint32_t)(min(i + a.long_run, a.M - 1) * st)];
    };
    auto equal = [&](int i, const uint32_t* v) { return a.long_run > 0 && i + a.long_run < a.M && v[0] == v[1]; };
    uint32_t v0[2];
    sorted_run(a.rhs, a.rhs_stride, a.M, a.E, (int)e, lane, first, end, [&] { pair_at(lane * half, v0); });
    even = __ballot(equal(lane * half, v0)) == 0ull;
    for (int i = (64 + lane) * half; even && a.long_run > 0 && (i - lane * half) + a.long_run < a.M; i += 64 * half) {
      uint32_t v[2];
      pair_at(i, v);
      even = __ballot(equal(i, v)) == 0ull;
    }
    if (even) {
      if (first >= end) return;  // the same in every wave
    } else {
      if ((int)blockIdx.y >= a.deal) return;
      passes = __builtin_amdgcn_readfirstlane(strip_runs<16 * MT>(a, t, at, pass0));
      if ((int)blockIdx.y >= passes) return;
      take(blockIdx.y);
    }
  }
  // A dense call's expert and first row stay values in registers: with them
  // folded away the compiler schedules the kernels differently, some worse
  // (float16 2-bit 64 rows 13-17% slower at 64 weight rows a workgroup, bfloat16
  // 3-bit 8-16 rows 4-7%) and some better (bfloat16 2-6-bit 128 rows 18-26%
  // faster, float16 3-5-bit 48 rows 7-10%, float16 6-bit 8-16 rows 24% over
  // 14336 x 4096 and equal over 4096 x 4096 and 4096 x 14336).
  if constexpr (!GATHER) {
    asm volatile("" : "+s"(e));
    asm volatile("" : "+s"(first));
  }
  const int z = GATHER ? 0 : blockIdx.y;
  const int kbeg = z * a.k_per_split, kend = min(K, kbeg + a.k_per_split);
  const int nsteps = (kend - kbeg + SR - 1) / SR;

  const int G = K >> gs_shift;
  const uint32_t RB = (uint32_t)(K / 32 * BITS) * 4u;
  constexpr uint32_t SE = AFF ? 2u : 1u;     // bytes per scale

  // weights of this lane: row n0 + 16 nwave + r, codes 32 q .. + 31 of each
  // window; positions past K read the next row's codes (finite, and their
  // scale and bias are 0 in the table)
  const int wn = n0 + 16 * nwave + r;
  const uint32_t woff = wn < N ? (uint32_t)wn * RB + (uint32_t)(((kbeg + kwave * SRW) >> 5) + q) * (uint32_t)(BITS * 4) : kDeadOfs;
  uint32_t wv[RD][BITS];

  // activations: thread t stages chunk t % CPR of rows t / CPR + XROWS i
  const int xrow = t / CPR, xch = t % CPR;
  const int xcol = (xch & ~15) | ((xch & 3) << 2) | ((xch >> 2) & 3);
  uint32_t xoff[XL];
  u32x4 xreg[2][XL];
  // scales: pairs of groups (affine), single groups (mxfp4); thread t takes
  // entry (t + 512 i) % GPT of row (t + 512 i) / GPT
  const int GPT = AFF ? GS >> 1 : GS;
  const int gp_shift = 31 - __builtin_clz(GPT);
  uint32_t soff[SL], sreg[2][SL][2], breg[2][SL][2];
  const bool g_even = (G & 1) == 0;
#pragma unroll
  for (int i = 0; i < SL; i++) {
    const int row = (t + 512 * i) >> gp_shift, e = (t + 512 * i) & (GPT - 1);
    const int n = n0 + row, g = (kbeg >> gs_shift) + (AFF ? 2 * e : e);
    soff[i] = row < RW && n < N ? ((uint32_t)n * (uint32_t)G + (uint32_t)g) * SE : kDeadOfs;
  }

  const __amdgpu_buffer_rsrc_t xr = buffer_rsrc(a.x, (uint32_t)((int64_t)a.M * K * 2));
  // empty resources for the loads of steps past the end
  const __amdgpu_buffer_rsrc_t x0 = buffer_rsrc(a.x, 0u), w0 = buffer_rsrc(a.w, 0u), s0r = buffer_rsrc(a.scales, 0u);
  for (int c0 = first, pass = blockIdx.y; GATHER || c0 < end;) {
    const int rows = min(16 * MT, end - c0);
    const int64_t sofs = e * a.s_expert_stride * SE;
    const __amdgpu_buffer_rsrc_t wr = buffer_rsrc(a.w + e * a.w_expert_stride, (uint32_t)((int64_t)N * RB));
    const __amdgpu_buffer_rsrc_t sr =
        buffer_rsrc(static_cast<const uint8_t*>(a.scales) + sofs, (uint32_t)((int64_t)N * G * SE));
    const __amdgpu_buffer_rsrc_t br =
        buffer_rsrc(AFF ? (const void*)(static_cast<const uint8_t*>(a.biases) + sofs) : a.scales,
                    AFF ? (uint32_t)((int64_t)N * G * SE) : 0u);
    auto load_window = [&](int slot, int step, int w) {
      const bool live = step < nsteps;
      load_codes<BITS>(live ? wr : w0, woff, live ? (step * (SR / 32) + w * 4) * (BITS * 4) : 0, wv[slot]);
    };
#pragma unroll
    for (int i = 0; i < XL; i++) {
      const int row = xrow + XROWS * i;
      xoff[i] = row < rows ? ((uint32_t)(c0 + row) * (uint32_t)K + (uint32_t)(kbeg + 8 * xch)) * 2u : kDeadOfs;
    }
    auto load_x = [&](int set, int step) {
      const bool live = step < nsteps;
      const __amdgpu_buffer_rsrc_t rs = live ? xr : x0;
      const int so = live ? step * (SR * 2) : 0;
      const bool in = 8 * xch < kend - kbeg - step * SR;  // past K: zeros
#pragma unroll
      for (int i = 0; i < XL; i++)
        xreg[set][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, in ? xoff[i] : kDeadOfs, so, 0));
    };
    auto write_x = [&](int buf) {  // from register set `buf`
#pragma unroll
      for (int i = 0; i < XL; i++) {
        const int row = xrow + XROWS * i;
        *reinterpret_cast<u32x4*>(xs + buf * XB + row * (SR * 2) + ((xcol ^ (row & 15)) << 4)) = xreg[buf][i];
      }
    };
    auto load_s = [&](int set, int step) {
      const bool live = step < nsteps;
      const __amdgpu_buffer_rsrc_t rs = live ? sr : s0r, rb = live ? br : s0r;
      const int so = live ? step * GS * (int)SE : 0;
      const int left = kend - kbeg - step * SR;
#pragma unroll
      for (int i = 0; i < SL; i++) {
        const int e = (t + 512 * i) & (GPT - 1);
        if constexpr (AFF) {
          const bool in0 = ((2 * e) << gs_shift) < left;
          if (g_even) {  // both groups in range together, 4-byte aligned
            const uint32_t o = in0 ? soff[i] : kDeadOfs;
            sreg[set][i][0] = __builtin_amdgcn_raw_buffer_load_b32(rs, o, so, 0);
            breg[set][i][0] = __builtin_amdgcn_raw_buffer_load_b32(rb, o, so, 0);
          } else {
            const bool in1 = ((2 * e + 1) << gs_shift) < left;
            const uint32_t o0 = in0 ? soff[i] : kDeadOfs, o1 = in1 ? soff[i] + 2u : kDeadOfs;
            sreg[set][i][0] = __builtin_amdgcn_raw_buffer_load_b16(rs, o0, so, 0);
            sreg[set][i][1] = __builtin_amdgcn_raw_buffer_load_b16(rs, o1, so, 0);
            breg[set][i][0] = __builtin_amdgcn_raw_buffer_load_b16(rb, o0, so, 0);
            breg[set][i][1] = __builtin_amdgcn_raw_buffer_load_b16(rb, o1, so, 0);
          }
        } else {
          const bool in = (e << gs_shift) < left;
          sreg[set][i][0] = __builtin_amdgcn_raw_buffer_load_b8(rs, in ? soff[i] : kDeadOfs, so, 0);
        }
      }
    };
    auto write_s = [&](int step, int buf) {
      const int left = kend - kbeg - step * SR;
#pragma unroll
      for (int i = 0; i < SL; i++) {
        const int row = (t + 512 * i) >> gp_shift, e = (t + 512 * i) & (GPT - 1);
        if (row >= RW) continue;
        if constexpr (AFF) {
          if (XT == 0) {
            const uint32_t hi = g_even ? sreg[buf][i][0] >> 16 : sreg[buf][i][1];
            if (max(sreg[buf][i][0] & 0x7F80u, hi & 0x7F80u) >= kBigScale) *big = 1u;
          }
          uint32_t* d = tbl + (buf * GS + 2 * e) * TP + row;
          d[0] = __builtin_amdgcn_perm(breg[buf][i][0], sreg[buf][i][0], 0x05040100u);
          d[TP] = g_even ? __builtin_amdgcn_perm(breg[buf][i][0], sreg[buf][i][0], 0x07060302u)
                         : __builtin_amdgcn_perm(breg[buf][i][1], sreg[buf][i][1], 0x05040100u);
        } else {
          // past K the activations are 0: any finite scale does
          tbl[(buf * GS + e) * TP + row] = (e << gs_shift) < left ? sreg[buf][i][0] : 127u;
        }
      }
    };

    f32x4 acc[MT];
    // B operand chunk j of this lane reads activation chunk 4 q + j of the window
    uint32_t xo[4];
#pragma unroll
    for (int j = 0; j < 4; j++) xo[j] = (uint32_t)(r * (SR * 2) + kwave * (SRW * 2) + (((4 * j + q) ^ r) << 4));
    const uint32_t tlane = (uint32_t)((((kwave * SRW + 32 * q) >> gs_shift) * TP + 16 * nwave + r) * 4);

    // the whole K range into acc; BIG: scales past 2^100 among them
    auto run = [&](auto big_tag) __attribute__((always_inline)) {
      constexpr bool BIG = decltype(big_tag)::value;
#pragma unroll
      for (int i = 0; i < MT; i++) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      load_x(0, 0);
      load_s(0, 0);
#pragma unroll
      for (int s = 0; s < RD; s++) load_window(s, s / WPS, s % WPS);
      load_x(1, 1);
      load_s(1, 1);
      write_x(0);
      write_s(0, 0);
      __syncthreads();
      for (int s0 = 0; s0 < nsteps; s0 += U) {
#pragma unroll
        for (int u = 0; u < U; u++) {
          const int step = s0 + u, buf = u & 1;
          load_x(buf, step + 2);
          load_s(buf, step + 2);
          const unsigned char* xb = xs + buf * XB;
          const unsigned char* tb = reinterpret_cast<const unsigned char*>(tbl) + tlane + (uint32_t)(buf * GS * TP * 4);
#pragma unroll
          for (int w = 0; w < WPS; w++) {
            const int slot = u * WPS + w;
            const uint32_t sb = *reinterpret_cast<const uint32_t*>(tb + (uint32_t)(((w * 128) >> gs_shift) * (TP * 4)));
            u32x4 o[4];
            if constexpr (AFF) {
              const float sc = xt_to_f32<XT>(sb & 0xFFFFu), bi = xt_to_f32<XT>(sb >> 16);
              const float s24 = sc * 16777216.f;
#pragma unroll
              for (int j = 0; j < 4; j++)
#pragma unroll
                for (int h = 0; h < 4; h++) {
                  const uint32_t q0 = code_at<BITS>(wv[slot], 8 * j + 2 * h), q1 = code_at<BITS>(wv[slot], 8 * j + 2 * h + 1);
                  if constexpr (BIG) {
                    o[j][h] = strip_pack<XT>(__builtin_fmaf(sc, (float)q0, bi), __builtin_fmaf(sc, (float)q1, bi));
                  } else {
                    // a code as the low half of a register is the float16
                    // subnormal q 2^-24: one mixed-precision FMA with 2^24 s
                    // is fma(s, q, b) exactly
                    o[j][h] = strip_pack<XT>(__builtin_fmaf((float)__builtin_bit_cast(_Float16, (uint16_t)q0), s24, bi),
                                             __builtin_fmaf((float)__builtin_bit_cast(_Float16, (uint16_t)q1), s24, bi));
                  }
                }
            } else {
              // normal scales fold into the fp4 conversion (exact); 2^-127 and
              // NaN (codes 0 and 255) multiply afterwards
              const float sc = e8m0_to_f32(sb);
              const bool special = sb - 1u >= 254u;
              const float cs = special ? 1.0f : sc;
              const bool any = __ballot(special) != 0ull;
#pragma unroll
              for (int j = 0; j < 4; j++) {
                uint32_t v[4];
                unpack_mxfp4_scaled(wv[slot][j], cs, v);
                if (__builtin_expect(any, 0)) {
#pragma unroll
                  for (int h = 0; h < 4; h++) {
                    const uint32_t p = strip_pack<0>(bf16_bits_to_f32(v[h] & 0xFFFFu) * sc, bf16_bits_to_f32(v[h] >> 16) * sc);
                    v[h] = special ? p : v[h];
                  }
                }
                o[j] = u32x4{v[0], v[1], v[2], v[3]};
              }
            }
            load_window(slot, step + U, w);  // the slot's next window
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
              for (int i = 0; i < MT; i++) {
                const u32x4 xv = *reinterpret_cast<const u32x4*>(xb + xo[j] + w * 256 + i * (16 * SR * 2));
                acc[i] = mfma16x16x32_xt<XT>(xv, o[j], acc[i]);
              }
          }
          write_x(buf ^ 1);
          write_s(step + 1, buf ^ 1);
          __syncthreads();
        }
      }
    };
    run(std::false_type{});
    if constexpr (AFF && XT == 0) {
      // a scale of 2^100 or more was staged (2^24 s may have overflowed):
      // once more with the codes converted
      if (__builtin_expect(*big != 0u, 0)) run(std::true_type{});
    }

    // sum over the K waves through LDS, in wave order
    float* red = reinterpret_cast<float*>(lds);  // [NWK][16 MT][RW]
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int e = 0; e < 4; e++) red[(kwave * 16 * MT + 16 * i + 4 * q + e) * RW + 16 * nwave + r] = acc[i][e];
    __syncthreads();
    constexpr int OC = RW / 8;
    const bool vec = (N & 7) == 0 && (reinterpret_cast<uintptr_t>(a.out) & 15) == 0;
    for (int idx = t; idx < 16 * MT * OC; idx += 512) {
      const int m = idx / OC, c = idx % OC;
      const int n = n0 + 8 * c;
      if (m >= rows || n >= N) continue;
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; e++) v[e] = 0.f;
#pragma unroll
      for (int kw = 0; kw < NWK; kw++) {
        const f32x4* p = reinterpret_cast<const f32x4*>(red + (kw * 16 * MT + m) * RW + 8 * c);
        const f32x4 lo = p[0], hi = p[1];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          v[e] += lo[e];
          v[4 + e] += hi[e];
        }
      }
      if (a.ks > 1) {
        float* d = a.ws + ((int64_t)z * a.M + c0 + m) * N + n;
        if (vec) {
          reinterpret_cast<f32x4*>(d)[0] = f32x4{v[0], v[1], v[2], v[3]};
          reinterpret_cast<f32x4*>(d)[1] = f32x4{v[4], v[5], v[6], v[7]};
        } else {
          for (int e = 0; e < 8 && n + e < N; e++) d[e] = v[e];
        }
      } else {
        uint16_t* d = a.out + (int64_t)(c0 + m) * N + n;
        const u32x4 p = {strip_pack<XT>(v[0], v[1]), strip_pack<XT>(v[2], v[3]), strip_pack<XT>(v[4], v[5]),
                         strip_pack<XT>(v[6], v[7])};
        if (vec) {
          *reinterpret_cast<u32x4*>(d) = p;
        } else {
          for (int e = 0; e < 8 && n + e < N; e++) d[e] = (uint16_t)(p[e >> 1] >> (16 * (e & 1)));
        }
      }
    }
    __syncthreads();  // the sums have been read before the next rows are staged
    if constexpr (!GATHER) {
      c0 += 16 * MT;
    } else if (even) {
      c0 += 16 * MT;
      if (c0 >= end) break;
    } else {
      pass += a.deal;
      if (pass >= passes) break;
      take(pass);
      c0 = first;
    }
  }
}

template <int FMT, int BITS, int XT, bool GATHER = false>
hipError_t strip_launch_fmt(const StripArgs& a, const StripPlan& p, dim3 grid, hipStream_t stream) {
#define STRIP_CASE(MT_, NWN_)                                                                                      \
  if (p.mt == MT_ && p.nwn == NWN_) {                                                                              \
    hipLaunchKernelGGL((qmm_strip_kernel<FMT, BITS, XT, MT_, NWN_, GATHER>), grid, dim3(512), p.lds, stream, a);   \
    return hipGetLastError();                                                                                      \
  }
  STRIP_CASE(1, 1)
  STRIP_CASE(1, 2)
  STRIP_CASE(1, 4)
  STRIP_CASE(2, 1)
  STRIP_CASE(2, 2)
  STRIP_CASE(2, 4)
  STRIP_CASE(3, 2)
  STRIP_CASE(3, 4)
  STRIP_CASE(4, 2)
  STRIP_CASE(4, 4)
  STRIP_CASE(8, 4)
#undef STRIP_CASE
  return hipErrorInvalidValue;
}

// one source file each (compile time)
hipError_t strip_launch_odd(int bits, const StripArgs& a, const StripPlan& p, dim3 grid, hipStream_t stream);
hipError_t strip_launch_f16(int bits, const StripArgs& a, const StripPlan& p, dim3 grid, hipStream_t stream);
hipError_t strip_launch_f16_odd(int bits, const StripArgs& a, const StripPlan& p, dim3 grid, hipStream_t stream);

}  // namespace mlxq
