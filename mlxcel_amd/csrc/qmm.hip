// qmm.hip — prefill quantized matmul (many activation rows) for gfx950.
//
// Replaces the reference's prefill route: affine dequantize to a bf16
// temporary and a hipBLASLt GEMM (overlays/rocm/mlx/backend/rocm/quantized/
// affine_quantize.hip:127-167 + qmm.hip:1376-1617, 3689-3892).  Here the
// dequantization happens on the way into LDS, so the bf16 weights never
// touch HBM: y = x @ W^T with W = bf16(s*q + b) (affine; the reference GPU
// dequantizer's rounding, affine_quantize.hip:164) or fp4(q) * 2^(e-127)
// (mxfp4, exact), fp32 accumulation, one bf16 rounding on store.
//
// Two kernels:
//  * qmm_tile_kernel (dense prefill, and grouped gathers at tiles 4-8): tiles
//    of 128 x 128 to 256 x 256 on 4 or 8 waves of v_mfma_f32_32x32x16_bf16
//    (or _f16), K in steps of 64 through double-buffered, XOR-swizzled LDS;
//    described above the kernel;
//  * qmm_kernel (grouped gathers at tiles 0-3): 4 waves (2 x 2) of
//    v_mfma_f32_16x16x32_bf16 over padded LDS rows [BM][64 + 8] and
//    [BN][64 + 8] (the 8-element pad puts the 16 rows a fragment read
//    touches on distinct banks), the next K-step's loads issued before the
//    current step's MFMAs, one barrier per K-step.
// When the grid would leave CUs idle (short M), K is split across
// workgroups and the fp32 partials are summed by a second kernel in a fixed
// order (bitwise reproducible).
#include <algorithm>
#include <cmath>

#include "qmm_tile.hpp"

namespace mlxq {

namespace {
constexpr int LDSK = BK + 8;  // padded row length (bf16)
constexpr int NT = 256;       // threads per workgroup (4 waves, 2 x 2)
}  // namespace

// BM x BN output tile per workgroup; each wave owns (BM/2) x (BN/2).
template <int FMT, int BM, int BN>
__global__ __launch_bounds__(NT) void qmm_kernel(const QmmArgs a) {
  constexpr int TM = BM / 2, TN = BN / 2;  // wave tile
  constexpr int FM = TM / 16, FN = TN / 16;  // 16 x 16 MFMA tiles per wave
  constexpr bool AFF = FMT != MXFP4;
  constexpr int BITS = FMT == AFF8 ? 8 : 4;
  constexpr int WT = BK * BITS / 8 / 16;   // threads per weight row per K-step (16 bytes each)
  constexpr int WROWS = NT / WT;           // weight rows loaded per pass
  constexpr int WPASS = BN / WROWS;        // passes per K-step
  constexpr int VPL = 128 / BITS;          // values per 16-byte load
  constexpr int XPASS = BM * BK * 2 / 16 / NT;  // 16-byte activation loads per thread per K-step

  __shared__ __align__(16) uint16_t xs[2][BM * LDSK];
  __shared__ __align__(16) uint16_t wsm[2][BN * LDSK];

  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = t >> 6;
  const int wm = wave >> 1, wn = wave & 1;  // wave position in the 2 x 2 grid
  static_assert(BN % WROWS == 0, "weight rows per pass must divide BN");
  const int n0 = blockIdx.x * BN;
  const int M = a.M, N = a.N, K = a.K;
  const int nks = a.ksteps_per_split;
  const int ks0 = blockIdx.z * nks;
  const int ks1 = min(ks0 + nks, K / BK);

  // Rows of this tile: rows m0 .. m0+rows-1 of x / y, or (gathers grouped by
  // expert) table entry blockIdx.y: grouped rows r0 .. r0+rows-1 of one
  // expert, read and written through xrows / orows.
  int m0 = blockIdx.y * BM, rows = min(BM, M - m0), r0 = 0;
  int64_t wbase = 0, sbase = 0;
  if (a.seg) {
    if ((int)blockIdx.y >= (int)a.nseg_dev[0]) return;
    const int expert = (int)a.seg[3 * blockIdx.y];
    r0 = (int)a.seg[3 * blockIdx.y + 1];
    rows = (int)a.seg[3 * blockIdx.y + 2];
    m0 = 0;
    wbase = (int64_t)expert * a.w_expert_stride;
    sbase = (int64_t)expert * a.s_expert_stride;
  }

  const __amdgpu_buffer_rsrc_t xr = buffer_rsrc(a.x, (uint32_t)((int64_t)a.x_rows * K * 2));
  const uint32_t RB = (uint32_t)(K * BITS / 8);  // bytes per weight row
  const __amdgpu_buffer_rsrc_t wr = buffer_rsrc(a.w + wbase, (uint32_t)((int64_t)N * RB));
  const int G = K >> a.gs_shift;
  const __amdgpu_buffer_rsrc_t sr =
      buffer_rsrc(reinterpret_cast<const uint8_t*>(a.scales) + sbase * (AFF ? 2 : 1), (uint32_t)((int64_t)N * G * (AFF ? 2 : 1)));
  const __amdgpu_buffer_rsrc_t br =
      buffer_rsrc(AFF ? (const void*)(a.biases + sbase) : a.scales, (uint32_t)(AFF ? (int64_t)N * G * 2 : 0));

  // ---- global -> register staging of one K-step ----------------------------
  // activations: thread t loads row (t / 8) + 32 i, 16-byte chunk t % 8
  const int xrow = t >> 3, xch = t & 7;
  // weights: thread t loads row (t / WT) + WROWS p, 16-byte piece t % WT
  const int wrow = t / WT, wpc = t % WT;
  uint32_t xbase[XPASS];  // byte offset of each staged x row (tile rows past `rows` read 0)
#pragma unroll
  for (int i = 0; i < XPASS; i++) {
    const int tr = xrow + 32 * i;
    const uint32_t xrw = a.seg ? (tr < rows ? a.xrows[r0 + tr] : 0u) : (uint32_t)(m0 + tr);
    xbase[i] = tr < rows ? xrw * (uint32_t)K * 2u + (uint32_t)xch * 16u : kDeadOfs;
  }
  u32x4 xreg[XPASS];
  u32x4 wreg[WPASS];
  uint32_t sreg[WPASS], breg[WPASS];
  auto load_step = [&](int ks) {
    const int k0 = ks * BK;
#pragma unroll
    for (int i = 0; i < XPASS; i++)
      xreg[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xr, xbase[i] + (uint32_t)k0 * 2u, 0, 0));
#pragma unroll
    for (int p = 0; p < WPASS; p++) {
      const int n = n0 + wrow + WROWS * p;
      const bool live = n < N;
      const uint32_t off = live ? (uint32_t)n * RB + (uint32_t)(k0 * BITS / 8 + wpc * 16) : kDeadOfs;
      wreg[p] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wr, off, 0, 2 /* nt */));
      const int g = (k0 + wpc * VPL) >> a.gs_shift;
      const uint32_t so = live ? (uint32_t)(n * G + g) : kDeadOfs;
      if constexpr (AFF) {
        sreg[p] = __builtin_amdgcn_raw_buffer_load_b16(sr, so * 2u, 0, 0);
        breg[p] = __builtin_amdgcn_raw_buffer_load_b16(br, so * 2u, 0, 0);
      } else {
        sreg[p] = __builtin_amdgcn_raw_buffer_load_b8(sr, so, 0, 0);
        breg[p] = 0u;
      }
    }
  };

  // ---- register -> LDS (activations as is, weights dequantized) ------------
  auto store_step = [&](int buf) {
#pragma unroll
    for (int i = 0; i < XPASS; i++)
      *reinterpret_cast<u32x4*>(&xs[buf][(xrow + 32 * i) * LDSK + xch * 8]) = xreg[i];
#pragma unroll
    for (int p = 0; p < WPASS; p++) {
      const u32x4 w = wreg[p];
      uint32_t o[VPL / 2];
      if constexpr (AFF) {
        const float sc = bf16_bits_to_f32(sreg[p]);
        const float bi = bf16_bits_to_f32(breg[p]);
        if constexpr (BITS == 4) {
          // nibbles 2j (low half of byte j) and 2j+1 (high half)
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const uint32_t lo = w[e] & 0x0F0F0F0Fu, hi = (w[e] >> 4) & 0x0F0F0F0Fu;
#pragma unroll
            for (int j = 0; j < 4; j++)
              o[e * 4 + j] = pack_bf16x2(__builtin_fmaf(sc, ubyte(lo, j), bi), __builtin_fmaf(sc, ubyte(hi, j), bi));
          }
        } else {
#pragma unroll
          for (int e = 0; e < 4; e++)
#pragma unroll
            for (int j = 0; j < 4; j += 2)
              o[e * 2 + j / 2] =
                  pack_bf16x2(__builtin_fmaf(sc, ubyte(w[e], j), bi), __builtin_fmaf(sc, ubyte(w[e], j + 1), bi));
        }
      } else {
        // fp4 code points times a power of two are exact in bf16: for normal
        // scales (e8m0 1..254) the gfx950 scaled conversion does it in one
        // instruction per pair; 2^-127 and NaN take the explicit product.
        const float sc = e8m0_to_f32(sreg[p]);
        if (sreg[p] - 1u < 254u) {
#pragma unroll
          for (int e = 0; e < 4; e++) unpack_mxfp4_scaled(w[e], sc, &o[e * 4]);
        } else {
#pragma unroll
          for (int e = 0; e < 4; e++) {
            uint32_t v[4];
            unpack_mxfp4(w[e], v);  // pairs (2h, 2h+1) of the code points
#pragma unroll
            for (int h = 0; h < 4; h++)
              o[e * 4 + h] = pack_bf16x2(bf16_bits_to_f32(v[h] & 0xFFFFu) * sc, bf16_bits_to_f32(v[h] >> 16) * sc);
          }
        }
      }
      uint16_t* dst = &wsm[buf][(wrow + WROWS * p) * LDSK + wpc * VPL];
#pragma unroll
      for (int c = 0; c < VPL / 8; c++)
        *reinterpret_cast<u32x4*>(dst + 8 * c) = u32x4{o[4 * c], o[4 * c + 1], o[4 * c + 2], o[4 * c + 3]};
    }
  };

  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; i++)
#pragma unroll
    for (int j = 0; j < FN; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int fr = lane & 15;         // fragment row (A) / column (B)
  const int fk = (lane >> 4) * 8;   // fragment k offset within 32

  if (ks0 < ks1) {
    load_step(ks0);
    store_step(0);
    __syncthreads();
    for (int ks = ks0; ks < ks1; ks++) {
      const int buf = (ks - ks0) & 1;
      if (ks + 1 < ks1) load_step(ks + 1);
#pragma unroll
      for (int kk = 0; kk < BK; kk += 32) {
        bf16x8 af[FM], bfr[FN];
#pragma unroll
        for (int i = 0; i < FM; i++)
          af[i] = *reinterpret_cast<const bf16x8*>(&xs[buf][(wm * TM + i * 16 + fr) * LDSK + kk + fk]);
#pragma unroll
        for (int j = 0; j < FN; j++)
          bfr[j] = *reinterpret_cast<const bf16x8*>(&wsm[buf][(wn * TN + j * 16 + fr) * LDSK + kk + fk]);
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
          for (int j = 0; j < FN; j++) acc[i][j] = mfma16x16x32(af[i], bfr[j], acc[i][j]);
      }
      if (ks + 1 < ks1) store_step(buf ^ 1);
      __syncthreads();
    }
  }

  // ---- epilogue: lane holds rows 4 (lane / 16) + q of each 16 x 16 tile ------
  const bool split = a.ksplit > 1;
#pragma unroll
  for (int i = 0; i < FM; i++)
#pragma unroll
    for (int j = 0; j < FN; j++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int tr = wm * TM + i * 16 + 4 * (lane >> 4) + q;
        const int c = n0 + wn * TN + j * 16 + fr;
        if (tr < rows && c < N) {
          const int64_t r = a.seg ? (int64_t)a.orows[r0 + tr] : (int64_t)(m0 + tr);
          if (split) a.ws[((int64_t)blockIdx.z * M + r) * N + c] = acc[i][j][q];
          else a.out[r * N + c] = (uint16_t)f32_to_bf16_bits(acc[i][j][q]);
        }
      }
}

// ---- host ------------------------------------------------------------------

namespace {
// Tile codes: 0 = 256 x 128, 1 = 256 x 256, 2 = 128 x 128, 3 = 64 x 128
// (16x16-MFMA kernel, grid (n, m, split)); 4 = 256 x 256 (8 waves), 5 = 256 x 128,
// 6 = 128 x 128, 7 = 256 x 256 (4 waves), 8 = 256 x 128 (8 waves, 4 x 2)
// (32x32-MFMA tile kernel, 1-D XCD-ordered grid).
constexpr int kTiles = 9;
const int kBM[kTiles] = {256, 256, 128, 64, 256, 256, 128, 256, 256};
const int kBN[kTiles] = {128, 256, 128, 128, 256, 128, 128, 256, 128};
bool is_tile_kernel(int tile) { return tile >= 4; }
}  // namespace

int qmm_tile_rows(int tile) { return tile >= 0 && tile < kTiles ? kBM[tile] : 0; }

namespace {
// Microseconds of a launch of tiles 4, 6 and 8 on MI355X:
//   start + rounds * (round + K-steps * (step + step_fill * fill)) + partial sums
// fill: workgroups over what one round of the CUs holds, at most 1; rounds: 1,
// or the exact number of them, `whole` of the way to the next integer (part-full
// rounds of one tile per CU cost more than a full one); a round's own
// time grows with the fill and is longer where rows of the result cannot be
// written 16 bytes at a time.  Fitted to 280000 graph-timed launches (129-2048
// rows; 17-128 rows for `few`; N 64-151936, K 256-14336, half of them with N
// not a multiple of 8), 5-6% rms.
struct TileCost {
  int slots;  // workgroups per CU
  float start, round[2], round_fill[2], step, step_fill, whole, sum, sum_each;  // [0] 16-byte rows of the result, [1] others
};
constexpr TileCost kCost4 = {1, 0.1f, {4.3f, 9.9f}, {7.4f, 13.3f}, 0.86f, 0.65f, 1.71f, 4.8f, 0.95f};
constexpr TileCost kCost6 = {2, 3.3f, {2.1f, 6.1f}, {4.1f, 6.4f}, 0.81f, 0.34f, 0.54f, 3.3f, 1.43f};
constexpr TileCost kCost8 = {1, 3.4f, {1.8f, 5.8f}, {3.9f, 5.8f}, 0.78f, 0.23f, 1.28f, 3.6f, 1.49f};
constexpr TileCost kCost6Few = {2, 0.8f, {4.4f, 6.4f}, {0.9f, 1.5f}, 0.81f, 0.40f, 0.51f, 3.0f, 2.23f};
constexpr TileCost kCost4Odd = {1, 3.7f, {2.6f, 8.8f}, {6.4f, 12.4f}, 1.01f, 0.65f, 1.57f, 4.9f, 0.91f};
constexpr TileCost kCost6Odd = {2, 4.3f, {1.2f, 5.0f}, {4.2f, 6.8f}, 0.86f, 0.38f, 0.54f, 3.2f, 1.38f};

float tile_us(int tile, bool odd, int64_t M, int64_t N, int nks, int ks, int num_cus) {
  const TileCost& c = tile == 4 ? (odd ? kCost4Odd : kCost4) : tile == 8 ? kCost8 : odd ? kCost6Odd : M <= 128 ? kCost6Few : kCost6;
  const int steps = (nks + ks - 1) / ks, ksr = (nks + steps - 1) / steps;
  const int64_t tiles = ((M + kBM[tile] - 1) / kBM[tile]) * ((N + kBN[tile] - 1) / kBN[tile]);
  const float x = (float)(tiles * ksr) / (float)((int64_t)c.slots * num_cus), fill = std::min(x, 1.f);
  const float rounds = std::max(1.f, c.whole * std::ceil(x) + (1.f - c.whole) * x);
  const int narrow = N % (ksr > 1 ? 4 : 8) != 0;
  return c.start + rounds * (c.round[narrow] + c.round_fill[narrow] * fill + steps * (c.step + c.step_fill * fill)) +
         (ksr > 1 ? c.sum + c.sum_each * (float)ksr * M * N * 1e-6f : 0.f);
}

// The cheapest tile and K split by that price, among each tile with no split,
// the split that fills a round and one less, for a grid of up to about one
// round (129-1024 rows; the 2-, 3-, 5- and 6-bit codes, which have tiles 4 and
// 6 only, at any row count).  The plan whose splits are powers of two
// (tile_in, ks_in; 0: none) is kept unless another is 3% cheaper.  Over 10900
// timed calls at 129-1024 rows the choice is 2.5% off the fastest (tile, split)
// measured, that plan 18%; 1% of them are more than 5% slower than on that
// plan (4% with prices without the round's own time and the narrow rows: 4-bit
// 469 rows over 17388 x 1152 64 us vs 50).
int plan_mid(bool odd, int64_t M, int64_t N, int nks, int num_cus, int tile_in, int ks_in, int& ks_out) {
  int best_tile = tile_in;
  float best = ks_in > 0 ? 0.97f * tile_us(tile_in, odd, M, N, nks, ks_in, num_cus) : 0.f;
  ks_out = ks_in;
  for (int tile : {4, 6, 8}) {
    if (odd && tile == 8) continue;
    const int64_t tiles = ((M + kBM[tile] - 1) / kBM[tile]) * ((N + kBN[tile] - 1) / kBN[tile]);
    const int64_t slots = (int64_t)(tile == 6 ? 2 : 1) * num_cus;
    const int mx = (int)std::max<int64_t>(1, std::min<int64_t>(std::min<int64_t>(slots / tiles, nks / 4), 16));
    for (int ks : {1, mx - 1, mx}) {
      if (ks < 1) continue;
      const float us = tile_us(tile, odd, M, N, nks, ks, num_cus);
      if (best > 0.f && us >= best) continue;
      best = us;
      best_tile = tile;
      ks_out = ks;
    }
  }
  return best_tile;
}
}  // namespace

QmmPlan qmm_plan(int fmt, int gs, int64_t M, int64_t N, int64_t K, int num_cus, int tile_req, int ksplit_req,
                 int mix, int streamk, bool fit_round) {
  QmmPlan p;
  if (fmt >= kAffOdd && !fit_round) return p;
  const int bits = fmt_bits(fmt);
  const bool odd = fmt >= kAffOdd;  // tiles 4 and 6 only
  if (odd && tile_req != 4 && tile_req != 6) tile_req = -1;
  if (K % BK != 0 || K % gs != 0 || M <= 0 || N <= 0) return p;
  if (M * K * 2 >= ((int64_t)1 << 31) || N * K * bits / 8 >= ((int64_t)1 << 31)) return p;
  const int nks = (int)(K / BK);
  auto tiles_of = [&](int t) { return ((M + kBM[t] - 1) / kBM[t]) * ((N + kBN[t] - 1) / kBN[t]); };
  int tile, ks_planned = 0;
  // K split by powers of two while the grid covers less than the CUs (up to
  // two workgroups per CU for few rows, where each tile is cheap) and each
  // split keeps >= 8 K-steps (gate/up M=32-128: 448 workgroups 31-38 us, 896
  // 37-50 us)
  auto pow2_split = [&](int t) {
    const int64_t n = tiles_of(t), fit = M <= 128 ? 2 * (int64_t)num_cus : num_cus;
    int ks = 1;
    while (n * ks * 2 <= fit && nks / (ks * 2) >= 8) ks *= 2;
    return ks;
  };
  if (tile_req >= 0 && tile_req < kTiles) {
    tile = tile_req;
  } else if (odd) {
    tile = plan_mid(true, M, N, nks, num_cus, 0, 0, ks_planned);
  } else {
    // 256 x 256 (8 waves) when there are enough tiles or K is long enough
    // for a K split to fill the CUs; else 128 x 128, two workgroups per CU.
    // Up to ~512 rows, 256 x 128 on 8 waves where it measured faster: long K
    // (split, down projections: 88-89 us vs 91-93 at M=512), 8-bit codes
    // with ~one tile per CU (gate/up M=512: 83 us vs 94) and 4-bit codes
    // with 0.75-1 tile per CU (gate/up M=384-512: 83-85 us vs 95, steady
    // state; at M=768, 1.3 tiles per CU, 162 vs 127).  Measured on MI355X at
    // the Llama-3-8B prefill shapes.
    // At 129-256 rows (less than one 256 x 128 tile per CU) the same tile
    // with a K split measured best too (gate/up M=256: 51.8 us vs 62 on 128 x
    // 128).
    const bool mid_rows = M > 128 && M <= 768;
    const int64_t t8 = tiles_of(8);
    const bool one_round8 = (fmt == AFF8 && t8 * 4 >= (int64_t)num_cus * 3) || (fmt != MXFP4 && t8 <= num_cus);
    if (mid_rows && (K >= 8192 || one_round8)) tile = 8;
    else tile = (M > 128 && (tiles_of(4) >= num_cus / 2 || K >= 8192)) ? 4 : 6;
    if (fit_round && ksplit_req <= 0 && M > 128 && M <= 1024 && tiles_of(4) <= num_cus)
      tile = plan_mid(false, M, N, nks, num_cus, tile, pow2_split(tile), ks_planned);
  }
  p.tile = tile;
  p.rows_per_tile = kBM[tile];
  p.tiles_n = (int)((N + kBN[tile] - 1) / kBN[tile]);
  p.tiles_m = (int)((M + kBM[tile] - 1) / kBM[tile]);
  const int64_t tiles = (int64_t)p.tiles_n * p.tiles_m;
  const int ks = ksplit_req > 0 ? ksplit_req : ks_planned > 0 ? ks_planned : pow2_split(tile);
  p.ksteps_per_split = (nks + ks - 1) / ks;
  p.ksplit = (nks + p.ksteps_per_split - 1) / p.ksteps_per_split;
  // consecutive tiles along M share weights, along N share activations: walk
  // along the dimension whose operand is the smaller of the two to re-read
  p.m_fast = M * K * 2 <= N * K * bits / 8 ? 1 : 0;
  p.ok = tiles * p.ksplit < ((int64_t)1 << 31);
  if (tile == 4 || tile == 6 || tile == 8) p.us = tile_us(tile, odd, M, N, nks, ks, num_cus);
  // Part-full last round: more 256 x 256 tiles than CUs, and the columns
  // past the whole rounds fit one round of 256 x 128 tiles.  Whole columns
  // of 256 x 256 tiles fill the full rounds, the rest runs as that one round
  // of the narrower tile, about 0.65 of a 256 x 256 tile's time (MI355X,
  // gate/up K=4096: M=1280-1536 x N=14336 202 us vs 233, M=2048 x N=12288
  // 214 vs 234).  A 256 x 192 tail for M=2048 x N=14336 measured slower
  // than the second 256 x 256 round (246 vs 240), so none is planned there.
  // Stream-K: one workgroup per CU takes an equal run of the 256 x 256
  // tiles' K-steps laid end to end, so a last round holding only a few tiles
  // does not leave the other CUs idle; a tile cut by a run boundary meets
  // through one fp32 partial.  Runs of at least a tile's K plus 8 steps keep
  // a cut tile's tail (the start of the next run) well ahead of its head
  // (the end of this run).  Taken when the last round holds at most 1/8 of
  // the CUs' tiles: the runs start their tiles at different K-steps, so
  // workgroups that share operands no longer read them from L2 at the same
  // time, which costs ~30% per step (MI355X, K=4096, 4-bit: 12288 x 1536
  // rows, 1.125 rounds, 170.5 us vs 196.6 on the two-launch plan; 14336 x
  // 2048 rows, 1.75 rounds, 269 vs 233).  streamk > 1 forces that run length.
  if (streamk && !odd && tile_req < 0 && ksplit_req <= 0 && p.tile == 4 && p.ksplit == 1 && tiles > num_cus &&
      fmt != MXFP4 && (streamk > 1 || (tiles < 2 * (int64_t)num_cus && (tiles - num_cus) * 8 <= num_cus))) {
    const int64_t steps = tiles * nks;
    const int64_t len = streamk > 1 ? streamk : (steps + num_cus - 1) / num_cus;
    if (len >= nks + 8 && len < ((int64_t)1 << 30) && (steps + len - 1) / len <= num_cus) {
      p.sk_len = (int)len;
      p.sk_wgs = (int)((steps + len - 1) / len);
      return p;
    }
  }
  if (mix && !odd && tile_req < 0 && ksplit_req <= 0 && p.tile == 4 && p.ksplit == 1 && tiles > num_cus) {
    const int64_t nb = (tiles / num_cus) * num_cus / p.tiles_m;  // 256-wide column tiles in whole rounds
    const int64_t n1 = nb * kBN[4];
    const int64_t tn2 = (N - n1 + kBN[8] - 1) / kBN[8];
    if (n1 > 0 && n1 < N && tn2 * p.tiles_m <= num_cus) {
      p.tile2 = 8;
      p.n_first = (int)n1;
      p.tiles_n2 = (int)tn2;
      p.tiles_n = (int)nb;
    }
  }
  return p;
}

namespace {
template <int FMT, int XT>
void qmm_tile_launch1(const QmmArgs& a, int tile, int ksplit, hipStream_t stream) {
  const dim3 grid((unsigned)((int64_t)a.tiles_m * a.tiles_n * ksplit));
  switch (tile) {
    case 4: hipLaunchKernelGGL((qmm_tile_kernel<FMT, 256, 256, 2, 4, XT>), grid, dim3(512), 0, stream, a); break;
    case 5: hipLaunchKernelGGL((qmm_tile_kernel<FMT, 256, 128, 2, 2, XT>), grid, dim3(256), 0, stream, a); break;
    case 7: hipLaunchKernelGGL((qmm_tile_kernel<FMT, 256, 256, 2, 2, XT>), grid, dim3(256), 0, stream, a); break;
    case 8: hipLaunchKernelGGL((qmm_tile_kernel<FMT, 256, 128, 4, 2, XT>), grid, dim3(512), 0, stream, a); break;
    default: hipLaunchKernelGGL((qmm_tile_kernel<FMT, 128, 128, 2, 2, XT>), grid, dim3(256), 0, stream, a); break;
  }
}

template <int FMT, int XT>
void qmm_tile_launch(const QmmArgs& a, const QmmPlan& p, hipStream_t stream) {
  if (p.sk_len > 0) {
    QmmArgs ak = a;
    ak.sk_len = p.sk_len;
    if constexpr (FMT != MXFP4)
      hipLaunchKernelGGL((qmm_tile_kernel<FMT, 256, 256, 2, 4, XT, true>), dim3((unsigned)p.sk_wgs), dim3(512), 0,
                         stream, ak);
    return;
  }
  if (p.tile2 < 0) {
    qmm_tile_launch1<FMT, XT>(a, p.tile, p.ksplit, stream);
    return;
  }
  // columns [0, n_first) on p.tile, then [n_first, N) on p.tile2: the second
  // launch sees the weight rows, scale rows and result columns from n_first
  // on, with the result's full row stride
  QmmArgs a1 = a;
  a1.N = p.n_first;
  a1.ldo = a.N;
  qmm_tile_launch1<FMT, XT>(a1, p.tile, 1, stream);
  constexpr int BITS = FMT == AFF8 ? 8 : 4;
  const int64_t n1 = p.n_first;
  const int64_t groups = (int64_t)a.K >> a.gs_shift;
  QmmArgs a2 = a;
  a2.w = a.w + n1 * ((int64_t)a.K * BITS / 32);
  a2.scales = reinterpret_cast<const uint8_t*>(a.scales) + n1 * groups * (FMT != MXFP4 ? 2 : 1);
  a2.biases = a.biases ? a.biases + n1 * groups : a.biases;
  a2.out = a.out + n1;
  a2.N = a.N - p.n_first;
  a2.ldo = a.N;
  a2.tiles_n = p.tiles_n2;
  qmm_tile_launch1<FMT, XT>(a2, p.tile2, 1, stream);
}

template <int FMT>
void qmm_launch_fmt(const QmmArgs& a, const QmmPlan& p, hipStream_t stream) {
  if (is_tile_kernel(p.tile)) {
    if constexpr (FMT != MXFP4) {
      if (a.xt == 1) {
        qmm_tile_launch<FMT, 1>(a, p, stream);
        return;
      }
    }
    qmm_tile_launch<FMT, 0>(a, p, stream);
    return;
  }
  const dim3 grid((unsigned)p.tiles_n, (unsigned)p.tiles_m, (unsigned)p.ksplit);
  switch (p.tile) {
    case 1: hipLaunchKernelGGL((qmm_kernel<FMT, 256, 256>), grid, dim3(NT), 0, stream, a); break;
    case 2: hipLaunchKernelGGL((qmm_kernel<FMT, 128, 128>), grid, dim3(NT), 0, stream, a); break;
    case 3: hipLaunchKernelGGL((qmm_kernel<FMT, 64, 128>), grid, dim3(NT), 0, stream, a); break;
    default: hipLaunchKernelGGL((qmm_kernel<FMT, 256, 128>), grid, dim3(NT), 0, stream, a); break;
  }
}
}  // namespace

// start (the index and grouping launches) + per entry + rounds * (round +
// K-steps * (step + step_fill * fill)), as above; 8-bit codes take `bits8` more
// per step.  Fitted to 3500 graph-timed gathers on MI355X (8-256 experts, 8-200
// entries each, spread evenly), 8% rms.
float grouped_us(int bits, int64_t N, int64_t K, int64_t E, int64_t B, int cus) {
  struct Cost {
    int slots;
    float start, entry, round, step, step_fill, whole, bits8;
  };
  const int tile = grouped_tile(B / E);
  const Cost c = tile == 3   ? Cost{2, 12.1f, 2.7e-3f, 2.7f, 0.91f, 0.64f, 0.58f, 0.35f}
                 : tile == 2 ? Cost{2, 10.9f, 2.0e-3f, 11.2f, 1.08f, 0.88f, 0.47f, 0.30f}
                             : Cost{1, 13.7f, 1.5e-3f, 24.2f, 1.49f, 0.24f, 0.76f, 0.52f};
  const float x = (float)((N + kBN[tile] - 1) / kBN[tile] * E) * mean_passes((double)B / E, kBM[tile]) / (float)(c.slots * cus);
  const float fill = std::min(x, 1.f), rounds = std::max(1.f, c.whole * std::ceil(x) + (1.f - c.whole) * x);
  const float step = (c.step + c.step_fill * fill) * (bits == 8 ? 1.f + c.bits8 : 1.f);
  return c.start + c.entry * B + rounds * (c.round + step * (float)(K / BK));
}

QmmPlan qmm_plan_grouped(int fmt, int gs, int64_t N, int64_t K, int tile) {
  QmmPlan p;
  const int bits = fmt == AFF8 ? 8 : 4;
  if (K % BK != 0 || K % gs != 0 || N <= 0 || tile < 0 || tile >= kTiles) return p;
  if (N * K * bits / 8 >= ((int64_t)1 << 31)) return p;
  p.tile = tile;
  p.rows_per_tile = kBM[tile];
  p.tiles_n = (int)((N + kBN[tile] - 1) / kBN[tile]);
  p.tiles_m = 0;  // the caller sets the segment count
  p.ksplit = 1;
  p.ksteps_per_split = (int)(K / BK);
  p.m_fast = 0;
  p.ok = true;
  return p;
}

hipError_t qmm_launch(int fmt, const QmmArgs& a_in, const QmmPlan& p, hipStream_t stream) {
  if (!p.ok) return hipErrorInvalidValue;
  // float16: affine codes on the 32x32-MFMA tile kernel only
  if (a_in.xt != 0 && (fmt == MXFP4 || !is_tile_kernel(p.tile))) return hipErrorInvalidValue;
  if (p.sk_len > 0 && (p.tile != 4 || !a_in.ws || !a_in.cnt || a_in.seg || fmt == MXFP4)) return hipErrorInvalidValue;
  QmmArgs a = a_in;
  a.tiles_m = p.tiles_m;
  a.tiles_n = p.tiles_n;
  a.m_fast = p.m_fast;
  if (p.sk_len <= 0) a.sk_len = 0;
  if (fmt >= kAffOdd) {
    if ((p.tile != 4 && p.tile != 6) || p.tile2 >= 0 || p.sk_len > 0 || a.seg) return hipErrorInvalidValue;
    qmm_launch_odd(fmt - kAffOdd, a, p.tile, p.ksplit, stream);
  } else switch (fmt) {
    case AFF4: qmm_launch_fmt<AFF4>(a, p, stream); break;
    case AFF8: qmm_launch_fmt<AFF8>(a, p, stream); break;
    default: qmm_launch_fmt<MXFP4>(a, p, stream); break;
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || p.ksplit == 1) return e;
  return launch_splitk_reduce(a.ws, a.out, (int64_t)a.M * a.N, p.ksplit, stream, a.xt);
}

}  // namespace mlxq
