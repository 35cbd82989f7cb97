// q8_gemm.hip -- the Q8_0 quantized linear for gfx950: y = x * W^T (+ bias)
// with W stored as GGML Q8_0 (int8 values, one scale per 32 along K).
//
// Semantics (bf16 x): W is dequantized exactly as the Q8_0 -> bf16 op does
// it (w = RNE_bf16(f32(q) * d), the product q * d being exact in f32), x is
// bf16, products accumulate in f32 on the matrix cores
// (v_mfma_f32_32x32x16_bf16), the bias is added in f32 and the result is
// rounded once to y's dtype. That is candle's dequantize-then-matmul path
// with a bf16 dequant target.
//
// Weights are first repacked once (q8_0_repack_kernel, the load-time step
// the reference takes in QMatMul::from_qtensor) from 34-byte blocks, which
// are only 2-byte aligned, into int8 [N, K] row-major plus f32 scales
// [N, K/32], so the GEMM streams them with 16-byte loads.
//
// Four GEMM kernels (each one rounding of the f32 sum per output):
// - q8_0_few_rows_kernel (K % 64 == 0, up to 16 rows or few tiles): workgroups of
//   16 weight rows whose wavefronts split k.
// - q8_0_gemm_ring_kernel (K % 64 == 0, the common case): a workgroup of NW
//   wavefronts (8, or 4 for small shapes) computes a BM x 32 NW tile (BM 32 to
//   256); x, the
//   int8 weights and the scales stream through a 3-stage LDS ring by direct
//   global->LDS loads; each wavefront dequantises its own 32 weight columns
//   once per k-step.
// - q8_0_gemm_kernel (K % 64 == 32): a 256-thread workgroup computes a
//   128 x 128 tile; x and the dequantised W are staged as bf16 in LDS,
//   double-buffered, through registers.
// - q8_0_gemm_x3_kernel (f32 x, K % 64 == 0): f32 arithmetic on the bf16
//   matrix cores, x split exactly into three bf16 terms, the int8 weights
//   exact in bf16 and each Q8_0 block's scale applied to its block sum.
// Within a k-step the kernels assign k to MFMA sub-steps differently, so
// their outputs can differ in the last bit of the f32 sum; each is
// deterministic.
#include "common.hpp"
#include "kernels.hpp"
#include "q8_tiles.hpp"

namespace lux3d {

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr int kBK = 32;                   // the k granularity (one Q8_0 block)
constexpr int kGemmThreads = 256;

// ---- repack: GGML blocks -> int8 [N, K] + f32 scales [N, K/32] -------------

__global__ __launch_bounds__(256) void q8_0_repack_kernel(const uint8_t *blocks, int64_t nblocks, int8_t *qs,
                                                          float *scales) {
  const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;  // one thread per 8 values
  if (g >= nblocks * 4) return;
  const int64_t blk = g >> 2;
  const int q = (int)(g & 3);
  const uint16_t *w = reinterpret_cast<const uint16_t *>(blocks + blk * 34);
  uint32_t lo = (uint32_t)w[1 + q * 4] | ((uint32_t)w[2 + q * 4] << 16);
  uint32_t hi = (uint32_t)w[3 + q * 4] | ((uint32_t)w[4 + q * 4] << 16);
  // blocks are row-major over (n, k/32): block blk holds row n = blk / (K/32)
  // values k = (blk % (K/32)) * 32 + ...; so the int8 stream is contiguous
  *reinterpret_cast<uint2 *>(qs + g * 8) = make_uint2(lo, hi);
  if (q == 0) scales[blk] = f16_bits_to_f32(w[0]);
}

// ---- GEMM -------------------------------------------------------------------

// Block tile BM x BN, k-step BK (one or two Q8_0 blocks); the four
// wavefronts form a 2 x 2 grid, each owning (BM/2) x (BN/2) = TM x TN MFMA
// tiles of 32 x 32. MINW is the minimum number of wavefronts per SIMD the
// register allocation must allow.
template <typename OUT, int BM, int BN, int BK, int MINW>
__global__ __launch_bounds__(kGemmThreads, MINW) void q8_0_gemm_kernel(Q8GemmParams p) {
  constexpr int TM = BM / 64, TN = BN / 64;
  constexpr int LDS_ROW = BK + 8;                    // bf16 per LDS row (odd multiple of 16 bytes)
  constexpr int A_CPR = BK / 8;                      // 16-byte chunks per x row per k-step
  constexpr int A_CHUNKS = BM * A_CPR / kGemmThreads;
  constexpr int B_CPR = BK / 16;                     // 16-int8 chunks per weight row per k-step
  constexpr int B_CHUNKS = BN * B_CPR / kGemmThreads;
  static_assert(A_CHUNKS >= 1 && B_CHUNKS >= 1, "tile too small for 256 threads");
  static_assert(BK % 32 == 0, "k-steps are whole Q8_0 blocks");
  __shared__ __align__(16) __bf16 As[2][BM * LDS_ROW];
  __shared__ __align__(16) __bf16 Bs[2][BN * LDS_ROW];

  const int t = threadIdx.x;
  const int lane = t & 63, wave = t >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int64_t m0 = (int64_t)blockIdx.y * BM, n0 = (int64_t)blockIdx.x * BN;
  const int64_t nblk = p.K / 32;  // Q8_0 blocks per weight row
  const int64_t nk = p.K / BK;

  // global -> register staging: x row chunks and weight row chunks. Rows past
  // M (N) are clamped to M - 1 (N - 1): loaded, computed, never stored.
  int64_t a_off[A_CHUNKS];
  int a_lds[A_CHUNKS];
#pragma unroll
  for (int i = 0; i < A_CHUNKS; ++i) {
    const int c = t + i * kGemmThreads, r = c / A_CPR, part = c % A_CPR;
    const int64_t gr = m0 + r < p.M ? m0 + r : p.M - 1;
    a_off[i] = (gr * p.ldx + part * 8) * 2;
    a_lds[i] = r * LDS_ROW + part * 8;
  }
  int64_t b_row[B_CHUNKS];
  int b_part[B_CHUNKS], b_lds[B_CHUNKS];
#pragma unroll
  for (int i = 0; i < B_CHUNKS; ++i) {
    const int c = t + i * kGemmThreads, r = c / B_CPR;
    b_part[i] = c % B_CPR;
    b_row[i] = n0 + r < p.N ? n0 + r : p.N - 1;
    b_lds[i] = r * LDS_ROW + b_part[i] * 16;
  }

  const char *xbase = reinterpret_cast<const char *>(p.x);
  uint4 ra[A_CHUNKS], rb[B_CHUNKS];
  float rd[B_CHUNKS];
  auto load_step = [&](int64_t kt) {
    const int64_t k0 = kt * BK;
#pragma unroll
    for (int i = 0; i < A_CHUNKS; ++i) ra[i] = ld16<false>(xbase + a_off[i] + k0 * 2);
#pragma unroll
    for (int i = 0; i < B_CHUNKS; ++i) {
      rb[i] = ld16<false>(p.qs + b_row[i] * p.K + k0 + b_part[i] * 16);
      rd[i] = p.scales[b_row[i] * nblk + k0 / 32 + b_part[i] / 2];
    }
  };
  auto store_step = [&](int buf) {
#pragma unroll
    for (int i = 0; i < A_CHUNKS; ++i) *reinterpret_cast<uint4 *>(&As[buf][a_lds[i]]) = ra[i];
#pragma unroll
    for (int i = 0; i < B_CHUNKS; ++i) {
      // dequant: 16 int8 -> bf16(f32(q) * d), RNE (q * d is exact in f32)
      const uint32_t w4[4] = {rb[i].x, rb[i].y, rb[i].z, rb[i].w};
      uint32_t pk[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t v = w4[j];
        const float f0 = (float)(int8_t)(v & 0xFFu) * rd[i], f1 = (float)(int8_t)((v >> 8) & 0xFFu) * rd[i];
        const float f2 = (float)(int8_t)((v >> 16) & 0xFFu) * rd[i], f3 = (float)(int8_t)(v >> 24) * rd[i];
        pk[2 * j] = pack_bf16x2(f0, f1);
        pk[2 * j + 1] = pack_bf16x2(f2, f3);
      }
      uint4 *dst = reinterpret_cast<uint4 *>(&Bs[buf][b_lds[i]]);
      dst[0] = make_uint4(pk[0], pk[1], pk[2], pk[3]);
      dst[1] = make_uint4(pk[4], pk[5], pk[6], pk[7]);
    }
  };

  f32x16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x16_t{};

  load_step(0);
  store_step(0);
  lds_barrier();

  const int lrow = lane & 31, lk = (lane >> 5) * 8;
  for (int64_t kt = 0; kt < nk; ++kt) {
    const int buf = (int)(kt & 1);
    if (kt + 1 < nk) load_step(kt + 1);
#pragma unroll
    for (int s = 0; s < BK / 16; ++s) {
      bf16x8_t a[TM], b[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i)
        a[i] = *reinterpret_cast<const bf16x8_t *>(&As[buf][(wm * (BM / 2) + i * 32 + lrow) * LDS_ROW + s * 16 + lk]);
#pragma unroll
      for (int j = 0; j < TN; ++j)
        b[j] = *reinterpret_cast<const bf16x8_t *>(&Bs[buf][(wn * (BN / 2) + j * 32 + lrow) * LDS_ROW + s * 16 + lk]);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    if (kt + 1 < nk) store_step(buf ^ 1);
    lds_barrier();
  }

  // epilogue: lane holds C[8*(e/4) + 4*(lane/32) + e%4][lane%32] of each tile
  char *ybase = reinterpret_cast<char *>(p.y);
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int64_t col = n0 + wn * (BN / 2) + j * 32 + (lane & 31);
    if (col >= p.N) continue;
    const float bias = p.bias ? p.bias[col] : 0.f;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int64_t row = m0 + wm * (BM / 2) + i * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
        if (row >= p.M) continue;
        const float v = acc[i][j][e] + bias;
        if constexpr (OUT::code == LUX3D_F32) {
          reinterpret_cast<float *>(ybase)[row * p.ldy + col] = v;
        } else {
          store1<OUT>(ybase, row * p.ldy + col, v);
        }
      }
  }
}

// ---- GEMM through an LDS ring fed by direct loads ---------------------------
//
// A workgroup of NW wavefronts computes a BM x 32 NW tile of y (256 x 256 where
// the problem fills the chip with them, down to 32 x 128). Its wavefronts each
// own 32 columns and all BM rows (BM / 32 MFMA tiles of
// 32 x 32), so every weight element is dequantised by exactly one wavefront
// and amortised over BM rows of x.
//
// Operands reach LDS by direct global->LDS loads (buffer_load ... lds, 16 or
// 4 bytes per lane, written in lane order at the address in M0) through a
// RING_STAGES-deep ring; no global load targets registers inside the k loop,
// so the loads of the next stages stay in flight across k-steps. One stage
// (k-step of 64) holds:
//   x       BM rows x 128 bytes, chunk c of row r in slot c ^ ((r >> 1) & 7)
//           (conflict-free fragment reads without padding);
//   weights per wavefront 2 KB: lane l's 16-byte half q (q = 0, 1) of the
//           32 int8 it needs at q * 1024 + l * 16;
//   scales  per wavefront 256 bytes: lane l's f32 scale at l * 4.
// k order: within a k-step, lane half h (lane / 32) of sub-step s holds
// k = 32 h + 8 s + e (e < 8) for both operands, so each lane's weight bytes
// for the step are 32 contiguous int8 of one Q8_0 block with one scale.
// The loads are inline assembly: the compiler then neither counts them nor
// inserts conservative waits for them, and the waits below are explicit
// (vmcnt counts a wavefront's own loads in issue order).
//
// Sub-steps are software-pipelined: the fragments and dequantised weights of
// sub-step s + 1 are produced while the MFMAs of s run; the barrier sits
// before the last sub-step's MFMAs, which then overlap the first reads of the
// next stage. The epilogue stages each wavefront's block through the ring
// (bias added, rounded once) and writes whole 16-byte row pieces.

constexpr int kRingStages = 3;

// 8 int8 (two dwords) -> bf16(f32(q) * d), RNE; q * d is exact in f32
__device__ __forceinline__ bf16x8_t dequant8(uint32_t lo, uint32_t hi, float d) {
  uint32_t pk[4];
  const uint32_t w2[2] = {lo, hi};
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const uint32_t v = w2[j];
    const float f0 = (float)(int8_t)(v & 0xFFu) * d, f1 = (float)(int8_t)((v >> 8) & 0xFFu) * d;
    const float f2 = (float)(int8_t)((v >> 16) & 0xFFu) * d, f3 = (float)(int8_t)(v >> 24) * d;
    pk[2 * j] = pack_bf16x2(f0, f1);
    pk[2 * j + 1] = pack_bf16x2(f2, f3);
  }
  return __builtin_bit_cast(bf16x8_t, make_uint4(pk[0], pk[1], pk[2], pk[3]));
}

// Needs K % 64 == 0 and every descriptor extent below 2^31 bytes (checked by
// the dispatcher). Tile order: workgroup ids are dealt round-robin to the 8
// XCDs; they are renumbered so that each XCD takes a contiguous range, walked
// in groups of GM row tiles (columns fastest within a group), so the tiles
// running on one XCD share x rows and weight columns in its L2.
template <typename OUT, int GM, int BM, int NW = 8>
__global__ __launch_bounds__(64 * NW, 1) void q8_0_gemm_ring_kernel(Q8GemmParams p, int tiles_m, int tiles_n) {
  // NW wavefronts, each owning 32 columns: BN = 32 NW (256 or 128); BM a multiple of 32 up to 256
  constexpr int BN = 32 * NW, BK = 64, TM = BM / 32, NS = kRingStages;
  constexpr int RW = BN * 64, RS = BN * 8;          // weights and scales per stage
  constexpr int kRingA = BM * 128, kRingStage = kRingA + RW + RS;  // 51,200 / 34,816 / 25,600 bytes
  constexpr int SEGW = BM / (8 * NW);              // x segments (1 KB = 8 rows) per wavefront
  constexpr int kRingOps = SEGW + 2 + 1;           // direct loads per wavefront per stage
  static_assert(BM % 32 == 0 && BM <= 256 && BM % (8 * NW) == 0 && (NW == 4 || NW == 8) && SEGW >= 1,
                "tile shape");
  __shared__ __align__(16) char ring[NS * kRingStage];

  const int G = tiles_m * tiles_n, bid = (int)blockIdx.x;
  const int per = G / 8, rem = G % 8, xcd = bid % 8, pos = bid / 8;
  const int lid = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + pos;
  const int group = lid / (GM * tiles_n), first_m = group * GM;
  const int gsize = tiles_m - first_m < GM ? tiles_m - first_m : GM;
  const int in_group = lid - group * GM * tiles_n;
  const int tm = first_m + in_group % gsize, tn = in_group / gsize;

  const int t = threadIdx.x;
  const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), h = lane >> 5, lrow = lane & 31;
  const int64_t m0 = (int64_t)tm * BM, c0 = (int64_t)tn * BN;
  const int64_t ncol = c0 + wave * 32 + lrow, nc = ncol < p.N ? ncol : p.N - 1;  // past N: clamped, never stored
  const int64_t nblk = p.K / 32;
  const int nk = (int)(p.K / BK);

  // direct-load sources: descriptors on the tile's first row / column, a
  // fixed per-lane offset, the k-step advance in the scalar offset
  uint32_t xoff[SEGW];
#pragma unroll
  for (int i = 0; i < SEGW; ++i) {
    const int g = wave * SEGW + i;  // 1 KB segment = 8 rows
    const int r = 8 * g + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    const int64_t gr = m0 + r < p.M ? m0 + r : p.M - 1;  // rows past M: clamped, never stored
    xoff[i] = (uint32_t)(((gr - m0) * p.ldx + 8 * c) * 2);
  }
  // each descriptor spans just the tile's rows / columns
  const int64_t last_row = p.M - 1 - m0 < BM - 1 ? p.M - 1 - m0 : BM - 1;
  const int64_t ncols = p.N - c0 < BN ? p.N - c0 : BN;
  const i32x4_t xr = buffer_rsrc(reinterpret_cast<const char *>(p.x) + m0 * p.ldx * 2, (last_row * p.ldx + p.K) * 2);
  const i32x4_t wr = buffer_rsrc(p.qs + c0 * p.K, ncols * p.K);
  const i32x4_t sr = buffer_rsrc(p.scales + c0 * nblk, ncols * nblk * 4);
  const uint32_t woff = (uint32_t)((nc - c0) * p.K + 32 * h);
  const uint32_t soff = (uint32_t)(((nc - c0) * nblk + h) * 4);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)ring;
  auto issue = [&](int kt, int buf) {
    const uint32_t st = lds0 + buf * kRingStage;
#pragma unroll
    for (int i = 0; i < SEGW; ++i)
      lds_load16(xr, xoff[i], (uint32_t)kt * BK * 2, __builtin_amdgcn_readfirstlane(st + (wave * SEGW + i) * 1024));
    lds_load16(wr, woff, (uint32_t)kt * BK, __builtin_amdgcn_readfirstlane(st + kRingA + wave * 2048));
    lds_load16(wr, woff, (uint32_t)kt * BK + 16, __builtin_amdgcn_readfirstlane(st + kRingA + wave * 2048 + 1024));
    lds_load4(sr, soff, (uint32_t)kt * 8, __builtin_amdgcn_readfirstlane(st + kRingA + RW + wave * 256));
  };

  // fragment of M-tile i, sub-step s at fbase[s] + i * 4096 (the swizzle only
  // depends on the row within a 32-row tile)
  int fbase[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) fbase[s] = lrow * 128 + (((4 * h + s) ^ ((lrow >> 1) & 7)) << 4);
  uint4 w0, w1;
  float sc;
  auto read_w = [&](const char *st) {
    w0 = *reinterpret_cast<const uint4 *>(st + kRingA + wave * 2048 + lane * 16);
    w1 = *reinterpret_cast<const uint4 *>(st + kRingA + wave * 2048 + 1024 + lane * 16);
    sc = *reinterpret_cast<const float *>(st + kRingA + RW + wave * 256 + lane * 4);
  };
  auto make_b = [&](int s) {
    const uint4 &v = s < 2 ? w0 : w1;
    return (s & 1) ? dequant8(v.z, v.w, sc) : dequant8(v.x, v.y, sc);
  };
  auto read_a = [&](const char *st, int s, bf16x8_t (&a)[TM]) {
#pragma unroll
    for (int i = 0; i < TM; ++i) a[i] = *reinterpret_cast<const bf16x8_t *>(st + fbase[s] + i * 4096);
  };
  f32x16_t acc[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) acc[i] = f32x16_t{};
  auto mfmas = [&](const bf16x8_t (&a)[TM], bf16x8_t b) {
#pragma unroll
    for (int i = 0; i < TM; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b, acc[i], 0, 0, 0);
  };

  // Prologue: stages 0 .. NS-2. The loop body is branch-free: past the last
  // k-step it reloads the last stage (in bounds) into a slot that is not read
  // for data again, so the wait counts are the same every step.
#pragma unroll
  for (int st = 0; st < NS - 1; ++st) issue(st < nk ? st : nk - 1, st);
  __builtin_amdgcn_s_waitcnt(waitcnt_vm((NS - 2) * kRingOps));  // stage 0 landed
  __builtin_amdgcn_s_barrier();

  bf16x8_t a0[TM], a1[TM], b0, b1;
  read_w(ring);
  read_a(ring, 0, a0);
  b0 = make_b(0);
  for (int kt = 0; kt < nk; ++kt) {
    // the slot refilled here was last read in step kt - 1, before its barrier
    issue(kt + NS - 1 < nk ? kt + NS - 1 : nk - 1, (kt + NS - 1) % NS);
    __builtin_amdgcn_sched_barrier(0);
    const char *st = ring + (kt % NS) * kRingStage;
    read_a(st, 1, a1);
    b1 = make_b(1);
    mfmas(a0, b0);
    __builtin_amdgcn_sched_barrier(0);
    read_a(st, 2, a0);
    b0 = make_b(2);
    mfmas(a1, b1);
    __builtin_amdgcn_sched_barrier(0);
    read_a(st, 3, a1);
    b1 = make_b(3);
    mfmas(a0, b0);
    __builtin_amdgcn_sched_barrier(0);
    // stage kt + 1 landed (only the stages issued after it may be in flight)
    // and this wavefront's reads of stage kt are done; then every one's
    __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0((NS - 2) * kRingOps));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    const char *nx = ring + ((kt + 1) % NS) * kRingStage;
    read_w(nx);
    read_a(nx, 0, a0);
    mfmas(a1, b1);
    b0 = make_b(0);
    __builtin_amdgcn_sched_barrier(0);
  }
  __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(0));  // the trailing reloads and reads

  char *ybase = reinterpret_cast<char *>(p.y);
  const float bias = (p.bias && ncol < p.N) ? p.bias[ncol] : 0.f;
  constexpr int EB = OUT::code == LUX3D_F32 ? 4 : 2;
  if (((uintptr_t)p.y % 16 == 0) && ((p.ldy * EB) % 16 == 0)) {
    // stage the wavefront's BM x 32 block through the ring, RP rows per
    // pass (rows padded by 16 bytes), and store whole 16-byte row pieces
    constexpr int ROW_B = 32 * EB, LROW = ROW_B + 16, CPR = ROW_B / 16, EPC = 16 / EB;
    // RP rows per pass: a multiple of 32 that divides BM and fits the ring
    constexpr int CAP = NS * kRingStage;
    constexpr int RP = NW * BM * LROW <= CAP ? BM
                       : (BM % 128 == 0 && NW * 128 * LROW <= CAP) ? 128
                       : (BM % 64 == 0 && NW * 64 * LROW <= CAP) ? 64 : 32;
    constexpr int REGION = RP * LROW;
    static_assert(NW * REGION <= CAP && BM % RP == 0, "epilogue staging fits the ring");
    __builtin_amdgcn_s_barrier();  // every wavefront is done with the ring
    char *reg = ring + wave * REGION;
    const int64_t c0w = c0 + wave * 32;
#pragma unroll
    for (int pass = 0; pass < BM / RP; ++pass) {
#pragma unroll
      for (int ii = 0; ii < RP / 32; ++ii)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int r = ii * 32 + 8 * (e >> 2) + 4 * h + (e & 3);
          const float v = acc[pass * (RP / 32) + ii][e] + bias;
          if constexpr (EB == 4) *reinterpret_cast<float *>(reg + r * LROW + lrow * 4) = v;
          else if constexpr (OUT::code == LUX3D_BF16)
            *reinterpret_cast<uint16_t *>(reg + r * LROW + lrow * 2) = (uint16_t)(pack_bf16x2(v, 0.f) & 0xFFFFu);
          else *reinterpret_cast<uint16_t *>(reg + r * LROW + lrow * 2) = (uint16_t)(pack_f16x2(v, 0.f) & 0xFFFFu);
        }
#pragma unroll
      for (int it = 0; it < RP * CPR / 64; ++it) {
        const int q = it * 64 + lane, r = q / CPR, part = q % CPR;
        const int64_t row = m0 + pass * RP + r, col = c0w + part * EPC;
        if (row >= p.M || col >= p.N) continue;
        const uint4 v = *reinterpret_cast<const uint4 *>(reg + r * LROW + part * 16);
        char *dst = ybase + (row * p.ldy + col) * EB;
        if (col + EPC <= p.N) {
          *reinterpret_cast<uint4 *>(dst) = v;
        } else {
          const uint32_t w4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
          for (int k = 0; k < EPC; ++k)
            if (col + k < p.N) {
              if constexpr (EB == 4) reinterpret_cast<uint32_t *>(dst)[k] = w4[k];
              else reinterpret_cast<uint16_t *>(dst)[k] = (uint16_t)(w4[k >> 1] >> (16 * (k & 1)));
            }
        }
      }
    }
    return;
  }
  // y rows not 16-byte aligned: one element per store
  if (ncol < p.N) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int64_t row = m0 + i * 32 + 8 * (e >> 2) + 4 * h + (e & 3);
        if (row >= p.M) continue;
        store1<OUT>(ybase, row * p.ldy + ncol, acc[i][e] + bias);
      }
  }
}

// ---- f32 activations on the bf16 matrix cores -------------------------------------
//
// y = sum over Q8_0 blocks b of d_b * (sum_{k in b} x_k q_k): each int8 q is
// exact in bf16, each f32 x is split exactly into three bf16 terms (x = x1 +
// x2 + x3, split3_bf16), so x q = x1 q + x2 q + x3 q with every product
// exact in f32. A 32-deep block of a 32 x 32 tile is six bf16 MFMAs (three
// terms x two 16-deep sub-steps) into a zeroed f32 block sum, which one FMA
// per element scales by the column's d and adds to the accumulator. That is
// the reference's f32 dequantize-then-matmul (w = q d exact in f32, f32
// products and sums, nn_blocks.rs:140) up to the order of the sums, at 6/16
// of the matrix-core cycles of v_mfma_f32_32x32x2_f32 per block. It replaced
// a ring kernel on v_mfma_f32_32x32x2_f32 (4096 x 2048 -> 8192: 994 -> 430
// us, same-box A/B).
//
// 128 x 256 tiles, 8 wavefronts as 2 (rows) x 4 (columns), 64 x 64 each; where
// those would leave CUs idle, 64 x 128 or 32 x 128 tiles of 4 wavefronts, whose
// KG groups take every KG th k-step into rings of their own and add their sums
// in LDS at the end (a step's chain of MFMAs, not memory, bounds a lone tile).
// 32-deep k-steps through a 4-stage LDS ring filled by direct global -> LDS
// loads: x (BM rows x 128 bytes, row-major), the int8 weights (32 columns x
// 32 bytes per 1 KB segment; lane l holds column l % 32, bytes 16 (l / 32)
// .. + 15) and the scales (32 columns per wavefront, both lane halves). Each
// step one cooperative pass splits the next stage's x into three bf16 planes
// (double-buffered; 64-byte rows, 16-byte chunk c of row r in slot c ^ ((r
// >> 2) & 3), so fragment reads are conflict-free). k order: in sub-step s,
// lane half h holds k = 16 h + 8 s + e on both operands. One barrier per
// step: wait for stage kt + 1, barrier, issue stage kt + 3, split stage
// kt + 1, compute stage kt.
constexpr int kX3Stages = 4;

// KG groups of WM x WN wavefronts, each wavefront TI x TJ tiles of 32 x 32.
template <int WM, int WN, int TI, int TJ>
struct X3Tile {
  static constexpr int NW = WM * WN, BM = 32 * WM * TI, BN = 32 * WN * TJ;
  static constexpr int SX = BM / 8 / NW, SW = BN / 32 / NW;  // 1 KB segments of x and of the weights a wavefront loads
  static constexpr int XL = BM * 128, WB = BN * 32, SB = BN * 8, STAGE = XL + WB + SB;
  static constexpr int PLANE = BM * 64;                      // one bf16 plane of BM rows x 32 k
  static constexpr int OPS = SX + 2 * SW;                    // direct loads per wavefront per stage
  static constexpr int LDS = kX3Stages * STAGE + 2 * 3 * PLANE;
  static_assert(BM % (8 * NW) == 0 && BN % (32 * NW) == 0, "whole segments per wavefront");
};

template <typename OUT, int GM, int WM, int WN, int TI, int TJ, int KG>
__global__ __launch_bounds__(64 * WM * WN * KG, 1) void q8_0_gemm_x3_kernel(Q8GemmParams p, int tiles_m, int tiles_n) {
  using T = X3Tile<WM, WN, TI, TJ>;
  constexpr int BM = T::BM, BN = T::BN, BK = 32, NS = kX3Stages;
  __shared__ __align__(16) char lds_all[KG * T::LDS];

  const int G = tiles_m * tiles_n, bid = (int)blockIdx.x;
  const int per = G / 8, rem = G % 8, xcd = bid % 8, pos = bid / 8;
  const int lid = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + pos;
  const int group = lid / (GM * tiles_n), first_m = group * GM;
  const int gsize = tiles_m - first_m < GM ? tiles_m - first_m : GM;
  const int in_group = lid - group * GM * tiles_n;
  const int tm = first_m + in_group % gsize, tn = in_group / gsize;

  const int kg = KG > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / (64 * T::NW)) : 0;
  const int t = KG > 1 ? threadIdx.x - kg * 64 * T::NW : threadIdx.x;
  const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), h = lane >> 5, l32 = lane & 31;
  const int wm = wave / WN, wn = wave % WN;
  char *const lds = lds_all + kg * T::LDS, *const planes = lds + NS * T::STAGE;
  const int64_t m0 = (int64_t)tm * BM, c0 = (int64_t)tn * BN;
  const int64_t nblk = p.K / 32;
  const int nk = (int)nblk, nit = (nk + KG - 1) / KG;  // group kg takes steps kg, kg + KG, ...

  // direct-load offsets (rows and columns past the matrix clamp to the last)
  uint32_t xoff[T::SX];
#pragma unroll
  for (int i = 0; i < T::SX; ++i) {
    const int r = 8 * (T::SX * wave + i) + (lane >> 3);
    const int64_t gr = m0 + r < p.M ? m0 + r : p.M - 1;
    xoff[i] = (uint32_t)(((gr - m0) * p.ldx + 4 * (lane & 7)) * 4);
  }
  const int64_t last_row = p.M - 1 - m0 < BM - 1 ? p.M - 1 - m0 : BM - 1;
  const int64_t ncols = p.N - c0 < BN ? p.N - c0 : BN;
  const i32x4_t xr = buffer_rsrc(reinterpret_cast<const char *>(p.x) + m0 * p.ldx * 4, (last_row * p.ldx + p.K) * 4);
  const i32x4_t wr = buffer_rsrc(p.qs + c0 * p.K, ncols * p.K);
  const i32x4_t sr = buffer_rsrc(p.scales + c0 * nblk, ncols * nblk * 4);
  uint32_t woff[T::SW], soff[T::SW];
#pragma unroll
  for (int i = 0; i < T::SW; ++i) {
    const int64_t col = c0 + 32 * (T::SW * wave + i) + l32, wc = col < p.N ? col : p.N - 1;
    woff[i] = (uint32_t)((wc - c0) * p.K + 16 * h);
    soff[i] = (uint32_t)((wc - c0) * nblk * 4);
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)lds;
  auto issue = [&](int it, int slot) {
    const int step = it * KG + kg, kt = step < nk ? step : nk - 1;
    const uint32_t st = lds0 + slot * T::STAGE;
#pragma unroll
    for (int i = 0; i < T::SX; ++i)
      lds_load16(xr, xoff[i], (uint32_t)kt * BK * 4, __builtin_amdgcn_readfirstlane(st + (T::SX * wave + i) * 1024));
#pragma unroll
    for (int i = 0; i < T::SW; ++i) {
      const int seg = T::SW * wave + i;
      lds_load16(wr, woff[i], (uint32_t)kt * BK, __builtin_amdgcn_readfirstlane(st + T::XL + seg * 1024));
      lds_load4(sr, soff[i], (uint32_t)kt * 4, __builtin_amdgcn_readfirstlane(st + T::XL + T::WB + seg * 256));
    }
  };
  // the split pass: thread t of a group takes every 64 NW th 16-byte chunk of
  // the stage's x from t (row q / 8, k 4 (q % 8) .. + 3)
  auto split = [&](int slot, int pb) {
    const char *xs = lds + slot * T::STAGE;
    char *pl = planes + pb * 3 * T::PLANE;
#pragma unroll
    for (int i = 0; i < BM * 8 / (64 * T::NW); ++i) {
      const int q = t + i * 64 * T::NW, r = q >> 3, c = q & 7;
      const float4 v = *reinterpret_cast<const float4 *>(xs + q * 16);
      const Split3 lo = split3_bf16(v.x, v.y), hi = split3_bf16(v.z, v.w);
      const int off = r * 64 + (((c >> 1) ^ ((r >> 2) & 3)) << 4) + (c & 1) * 8;
      *reinterpret_cast<uint2 *>(pl + off) = make_uint2(lo.t1, hi.t1);
      *reinterpret_cast<uint2 *>(pl + T::PLANE + off) = make_uint2(lo.t2, hi.t2);
      *reinterpret_cast<uint2 *>(pl + 2 * T::PLANE + off) = make_uint2(lo.t3, hi.t3);
    }
  };
  // fragment offsets: A rows (wm TI + i) * 32 + l32, chunk 2 h + s
  int aoff[TI][2];
#pragma unroll
  for (int i = 0; i < TI; ++i) {
    const int r = (wm * TI + i) * 32 + l32;
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) aoff[i][s2] = r * 64 + (((2 * h + s2) ^ ((r >> 2) & 3)) << 4);
  }
  f32x16_t acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[i][j] = f32x16_t{};
  auto compute = [&](int slot, int pb) {
    const char *st = lds + slot * T::STAGE;
    const char *pl = planes + pb * 3 * T::PLANE;
    // weights of columns (wn TJ + j) * 32 + l32: 16 int8 -> two bf16x8 (sub-steps)
    bf16x8_t b[TJ][2];
    float d[TJ];
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
      const uint4 w = *reinterpret_cast<const uint4 *>(st + T::XL + (wn * TJ + j) * 1024 + lane * 16);
      d[j] = *reinterpret_cast<const float *>(st + T::XL + T::WB + (wn * TJ + j) * 256 + l32 * 4);
      const uint32_t wv[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        uint32_t pk[4];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const uint32_t v = wv[2 * s2 + u];
          pk[2 * u] = pack_bf16x2((float)(int8_t)(v & 0xFFu), (float)(int8_t)((v >> 8) & 0xFFu));
          pk[2 * u + 1] = pack_bf16x2((float)(int8_t)((v >> 16) & 0xFFu), (float)(int8_t)(v >> 24));
        }
        b[j][s2] = __builtin_bit_cast(bf16x8_t, u32x4_t{pk[0], pk[1], pk[2], pk[3]});
      }
    }
#pragma unroll
    for (int i = 0; i < TI; ++i) {
      bf16x8_t a[3][2];
#pragma unroll
      for (int q = 0; q < 3; ++q)
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) a[q][s2] = *reinterpret_cast<const bf16x8_t *>(pl + q * T::PLANE + aoff[i][s2]);
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
        // block sum, smallest terms first, then scaled by the column's d
        f32x16_t blk = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[2][0], b[j][0], f32x16_t{}, 0, 0, 0);
        blk = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[2][1], b[j][1], blk, 0, 0, 0);
        blk = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1][0], b[j][0], blk, 0, 0, 0);
        blk = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1][1], b[j][1], blk, 0, 0, 0);
        blk = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0][0], b[j][0], blk, 0, 0, 0);
        blk = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0][1], b[j][1], blk, 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = __builtin_fmaf(blk[e], d[j], acc[i][j][e]);
      }
    }
  };

#pragma unroll
  for (int s2 = 0; s2 < NS - 1; ++s2) issue(s2, s2);
  __builtin_amdgcn_s_waitcnt(waitcnt_vm((NS - 2) * T::OPS));
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  split(0, 0);
  for (int it = 0; it < nit; ++it) {
    // stage it + 1 landed (it + 2 may be in flight); every wavefront is done
    // with compute(it - 1) and split(it)
    __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(T::OPS));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    issue(it + NS - 1, (it + NS - 1) % NS);
    __builtin_amdgcn_sched_barrier(0);
    if (it + 1 < nit) split((it + 1) % NS, (it + 1) & 1);
    if (KG == 1 || it * KG + kg < nk) compute(it % NS, it & 1);
  }
  __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(0));
  __builtin_amdgcn_s_barrier();  // every wavefront is done with the ring and the planes

  if constexpr (KG > 1) {
    // the groups' sums in group order, through LDS
    constexpr int PART = TI * TJ * 16 * 64;
    static_assert((KG - 1) * T::NW * PART * 4 <= KG * T::LDS, "partial sums fit");
    float *const part = reinterpret_cast<float *>(lds_all) + wave * PART;
    if (kg > 0) {
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e)
            part[(kg - 1) * T::NW * PART + ((i * TJ + j) * 16 + e) * 64 + lane] = acc[i][j][e];
    }
    __syncthreads();
    if (kg == 0) {
#pragma unroll
      for (int g = 1; g < KG; ++g)
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
          for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e)
              acc[i][j][e] += part[(g - 1) * T::NW * PART + ((i * TJ + j) * 16 + e) * 64 + lane];
    }
    __syncthreads();
    if (kg > 0) return;
  }

  // epilogue: each wavefront's 32 TI x 32 TJ block through LDS, bias added, one
  // rounding, 16-byte row pieces
  char *ybase = reinterpret_cast<char *>(p.y);
  constexpr int EB = OUT::code == LUX3D_F32 ? 4 : 2;
  float bias[TJ];
#pragma unroll
  for (int j = 0; j < TJ; ++j) {
    const int64_t col = c0 + (wn * TJ + j) * 32 + l32;
    bias[j] = (p.bias && col < p.N) ? p.bias[col] : 0.f;
  }
  if (((uintptr_t)p.y % 16 == 0) && ((p.ldy * EB) % 16 == 0)) {
    constexpr int ROW_B = 32 * TJ * EB, LROW = ROW_B + 16, CPR = ROW_B / 16, EPC = 16 / EB;
    constexpr int REGION = 32 * TI * LROW;
    static_assert(T::NW * REGION <= T::LDS, "epilogue staging fits");
    char *reg = lds + wave * REGION;
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int r = i * 32 + 8 * (e >> 2) + 4 * h + (e & 3), cl = j * 32 + l32;
          const float v = acc[i][j][e] + bias[j];
          if constexpr (EB == 4) *reinterpret_cast<float *>(reg + r * LROW + cl * 4) = v;
          else if constexpr (OUT::code == LUX3D_BF16)
            *reinterpret_cast<uint16_t *>(reg + r * LROW + cl * 2) = (uint16_t)(pack_bf16x2(v, 0.f) & 0xFFFFu);
          else *reinterpret_cast<uint16_t *>(reg + r * LROW + cl * 2) = (uint16_t)(pack_f16x2(v, 0.f) & 0xFFFFu);
        }
    const int64_t r0 = m0 + wm * TI * 32, cw = c0 + wn * TJ * 32;
#pragma unroll
    for (int it = 0; it < 32 * TI * CPR / 64; ++it) {
      const int q = it * 64 + lane, r = q / CPR, part = q % CPR;
      const int64_t row = r0 + r, col = cw + part * EPC;
      if (row >= p.M || col >= p.N) continue;
      const uint4 v = *reinterpret_cast<const uint4 *>(reg + r * LROW + part * 16);
      char *dst = ybase + (row * p.ldy + col) * EB;
      if (col + EPC <= p.N) {
        *reinterpret_cast<uint4 *>(dst) = v;
      } else {
        const uint32_t w4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int kk = 0; kk < EPC; ++kk)
          if (col + kk < p.N) {
            if constexpr (EB == 4) reinterpret_cast<uint32_t *>(dst)[kk] = w4[kk];
            else reinterpret_cast<uint16_t *>(dst)[kk] = (uint16_t)(w4[kk >> 1] >> (16 * (kk & 1)));
          }
      }
    }
    return;
  }
  // y rows not 16-byte aligned: one element per store
#pragma unroll
  for (int j = 0; j < TJ; ++j) {
    const int64_t col = c0 + (wn * TJ + j) * 32 + l32;
    if (col >= p.N) continue;
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int64_t row = m0 + (wm * TI + i) * 32 + 8 * (e >> 2) + 4 * h + (e & 3);
        if (row >= p.M) continue;
        store1<OUT>(ybase, row * p.ldy + col, acc[i][j][e] + bias[j]);
      }
  }
}

// ---- few rows --------------------------------------------------------------------
//
// One modulation or conditioning vector per batch element, short sequences: the
// weights' bytes bound them, and tiles of 128 rows leave most CUs idle (72
// workgroups at N 9216) behind a serial k loop. A workgroup owns 16 weight rows
// and 16 MT rows of x; its NW wavefronts take pairs of 64-deep chunks of k in
// turn, and their sums (v_mfma_f32_16x16x32_bf16: x rows x weight rows) are
// added in wavefront order through LDS. A turn of the loop takes U chunks, but
// as compiled a wavefront waits for each chunk's loads and multiplies before it
// issues the next chunk's (the branch after each chunk keeps them apart: 51
// VGPRs): one chunk is in flight per wavefront, and only the other wavefronts
// of the SIMD cover its latency. k order inside a chunk: lane group g = lane / 16 holds weights
// 16 g .. 16 g + 15 of its row as one 16-byte load (one Q8_0 block, one scale),
// bytes 8 s .. + 7 in MFMA s, and x alike. XF32: f32 x in three exact bf16
// terms, the int8 weights exact, one MFMA per term and Q8_0 block (lane group
// g: weights 8 g .. + 7), the block's sum scaled by d, as q8_0_gemm_x3_kernel
// does. Before / after, us: M 2, K 1536 -> N 9216 16.9 / 8.0 in bf16 (16 MB of
// weights: 3.1 us at the copy rate) and 71 / 10.8 in f32; M 64, K 8192 -> N
// 2048 68 / 38 and 363 / 69.
template <typename OUT, bool XF32, int NW, int MT>
__global__ __launch_bounds__(64 * NW) void q8_0_few_rows_kernel(Q8GemmParams p) {
  typedef float f32x4_t __attribute__((ext_vector_type(4)));
  constexpr int U = MT == 1 ? (XF32 ? 4 : 8) : 2;  // chunks per turn
  __shared__ float part[NW][MT * 256];
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), g = lane >> 4;
  const int64_t n0 = (int64_t)blockIdx.x * 16, m0 = (int64_t)blockIdx.y * 16 * MT;
  // rows past N and M are clamped: loaded, computed, never stored
  const int64_t n = n0 + (lane & 15) < p.N ? n0 + (lane & 15) : p.N - 1;
  const int64_t nch = p.K / 64;
  const int8_t *wr = p.qs + n * p.K;
  const float *sr = p.scales + n * (p.K / 32);
  const char *xr[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int64_t m = m0 + 16 * i + (lane & 15);
    xr[i] = reinterpret_cast<const char *>(p.x) + (m < p.M ? m : p.M - 1) * p.ldx * (XF32 ? 4 : 2);
  }
  f32x4_t acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = f32x4_t{};
  // chunks go to the wavefronts in pairs: whole 128-byte lines of the weights
  for (int64_t c0 = 2 * wave; c0 < nch; c0 += U * NW) {
    auto chunk = [&](int u) { return c0 + (int64_t)(u / 2) * 2 * NW + (u & 1); };
    if constexpr (!XF32) {
      uint4 w[U], x[U][MT][2];
      float d[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t c = chunk(u) < nch ? chunk(u) : c0;
        w[u] = ld16<false>(wr + c * 64 + 16 * g);
        d[u] = sr[c * 2 + (g >> 1)];
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          x[u][i][0] = ld16<false>(xr[i] + (c * 64 + 16 * g) * 2);
          x[u][i][1] = ld16<false>(xr[i] + (c * 64 + 16 * g) * 2 + 16);
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (chunk(u) >= nch) break;  // uniform
        const bf16x8_t b0 = dequant8(w[u].x, w[u].y, d[u]), b1 = dequant8(w[u].z, w[u].w, d[u]);
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, x[u][i][0]), b0, acc[i], 0, 0, 0);
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, x[u][i][1]), b1, acc[i], 0, 0, 0);
        }
      }
    } else {
      uint2 w[U][2];
      float d[U][2], x[U][2][MT][8];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t c = chunk(u) < nch ? chunk(u) : c0;
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          w[u][b] = *reinterpret_cast<const uint2 *>(wr + c * 64 + 32 * b + 8 * g);
          d[u][b] = sr[c * 2 + b];
#pragma unroll
          for (int i = 0; i < MT; ++i) Chunk<F32>::load<false>(xr[i] + (c * 64 + 32 * b + 8 * g) * 4, x[u][b][i]);
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (chunk(u) >= nch) break;  // uniform
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const bf16x8_t q = dequant8(w[u][b].x, w[u][b].y, 1.f);
#pragma unroll
          for (int i = 0; i < MT; ++i) {
            uint32_t x1[4], x2[4], x3[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const Split3 r = split3_bf16(x[u][b][i][2 * e], x[u][b][i][2 * e + 1]);
              x1[e] = r.t1;
              x2[e] = r.t2;
              x3[e] = r.t3;
            }
            f32x4_t blk = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(bf16x8_t, u32x4_t{x3[0], x3[1], x3[2], x3[3]}), q, f32x4_t{}, 0, 0, 0);
            blk = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(bf16x8_t, u32x4_t{x2[0], x2[1], x2[2], x2[3]}), q, blk, 0, 0, 0);
            blk = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(bf16x8_t, u32x4_t{x1[0], x1[1], x1[2], x1[3]}), q, blk, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i][e] = __builtin_fmaf(blk[e], d[u][b], acc[i][e]);
          }
        }
      }
    }
  }
  // lane holds rows 4 g + e, column lane % 16 of each 16-row tile
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) part[wave][i * 256 + e * 64 + lane] = acc[i][e];
  __syncthreads();
  for (int o = t; o < MT * 256; o += 64 * NW) {
    const int64_t row = m0 + o / 256 * 16 + 4 * ((o & 63) >> 4) + (o >> 6 & 3), col = n0 + (o & 15);
    if (row >= p.M || col >= p.N) continue;
    float v = part[0][o];
#pragma unroll
    for (int w = 1; w < NW; ++w) v += part[w][o];
    store1<OUT>(p.y, row * p.ldy + col, v + (p.bias ? p.bias[col] : 0.f));
  }
}

template <typename OUT, bool XF32, int MT>
hipError_t launch_few_rows(const Q8GemmParams &p, hipStream_t s) {
  // 2048 wavefronts (two per SIMD), or as many as k has chunk pairs
  const int64_t tn = (p.N + 15) / 16, tm = (p.M + 16 * MT - 1) / (16 * MT);
  if (tn > INT32_MAX || tm > 65535) return hipErrorInvalidValue;
  const dim3 grid((unsigned)tn, (unsigned)tm);
  if (tn * tm * 4 >= 2048 || p.K <= 512)
    hipLaunchKernelGGL((q8_0_few_rows_kernel<OUT, XF32, 4, MT>), grid, dim3(256), 0, s, p);
  else if (tn * tm * 8 >= 2048 || p.K <= 1024)
    hipLaunchKernelGGL((q8_0_few_rows_kernel<OUT, XF32, 8, MT>), grid, dim3(512), 0, s, p);
  else
    hipLaunchKernelGGL((q8_0_few_rows_kernel<OUT, XF32, 16, MT>), grid, dim3(1024), 0, s, p);
  return hipGetLastError();
}

template <typename OUT, int WM, int WN, int TI, int TJ, int KG>
hipError_t launch_x3(const Q8GemmParams &p, hipStream_t s) {
  using T = X3Tile<WM, WN, TI, TJ>;
  const int64_t tiles_m = (p.M + T::BM - 1) / T::BM, tiles_n = (p.N + T::BN - 1) / T::BN;
  if (tiles_m * tiles_n > 0x7FFFFFFF) return hipErrorInvalidValue;
  hipLaunchKernelGGL((q8_0_gemm_x3_kernel<OUT, 8, WM, WN, TI, TJ, KG>), dim3((unsigned)(tiles_m * tiles_n)),
                     dim3(64 * T::NW * KG), 0, s, p, (int)tiles_m, (int)tiles_n);
  return hipGetLastError();
}

template <typename OUT>
hipError_t launch_f32(const Q8GemmParams &p, hipStream_t s) {
  const Q8Tile tile = q8_tile_f32(p.M, p.N, p.K);
  if (tile.few()) return tile.rows == 16 ? launch_few_rows<OUT, true, 1>(p, s) : launch_few_rows<OUT, true, 4>(p, s);
  if (tile.rows == 128) return launch_x3<OUT, 2, 4, 2, 2, 1>(p, s);
  if (tile.rows == 32) return launch_x3<OUT, 1, 4, 1, 1, 3>(p, s);
  return tile.groups == 1 ? launch_x3<OUT, 2, 2, 1, 2, 1>(p, s) : launch_x3<OUT, 2, 2, 1, 2, 2>(p, s);
}

// The ring kernel's buffer descriptors span one tile (at most 256 rows of x,
// 256 weight rows and their scales) and must stay below 2^31 bytes; its
// per-lane offsets are 32-bit.
bool ring_fits(const Q8GemmParams &p) {
  const int64_t lim = 0x7FFFFFFF;
  return p.K % 64 == 0 && (255 * p.ldx + p.K) * 2 <= lim && 256 * p.K <= lim &&
         (p.M + 127) / 128 * ((p.N + 255) / 256) <= INT32_MAX;
}

template <typename OUT, int BM, int NW>
hipError_t launch_ring(const Q8GemmParams &p, hipStream_t s) {
  const int64_t tiles_m = (p.M + BM - 1) / BM, tiles_n = (p.N + 32 * NW - 1) / (32 * NW);
  if (tiles_m * tiles_n > INT32_MAX) return hipErrorInvalidValue;
  hipLaunchKernelGGL((q8_0_gemm_ring_kernel<OUT, 8, BM, NW>), dim3((unsigned)(tiles_m * tiles_n)), dim3(64 * NW), 0, s,
                     p, (int)tiles_m, (int)tiles_n);
  return hipGetLastError();
}

template <typename OUT>
hipError_t launch_bf16(const Q8GemmParams &p, hipStream_t s) {
  const Q8Tile tile = q8_tile_bf16(p.M, p.N, p.K);
  if (tile.few()) return tile.rows == 16 ? launch_few_rows<OUT, false, 1>(p, s) : launch_few_rows<OUT, false, 4>(p, s);
  if (tile.cols == 256) return tile.rows == 256 ? launch_ring<OUT, 256, 8>(p, s) : launch_ring<OUT, 128, 8>(p, s);
  switch (tile.rows) {
    case 32: return launch_ring<OUT, 32, 4>(p, s);
    case 64: return launch_ring<OUT, 64, 4>(p, s);
    case 128: return launch_ring<OUT, 128, 4>(p, s);
  }
  return launch_ring<OUT, 160, 4>(p, s);
}

template <typename OUT>
hipError_t launch_tiles(const Q8GemmParams &p, hipStream_t s) {
  if (p.x_f32) return launch_f32<OUT>(p, s);  // K % 64 == 0, checked by the caller
  if (ring_fits(p)) return launch_bf16<OUT>(p, s);
  // K % 64 == 32, or rows too far apart for the ring's offsets
  const dim3 grid((unsigned)((p.N + 127) / 128), (unsigned)((p.M + 127) / 128));
  hipLaunchKernelGGL((q8_0_gemm_kernel<OUT, 128, 128, 32, 1>), grid, dim3(kGemmThreads), 0, s, p);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_q8_0_repack(const uint8_t *blocks, int64_t nblocks, int8_t *qs, float *scales, hipStream_t s) {
  if (nblocks <= 0) return hipSuccess;
  const int64_t threads = nblocks * 4;
  hipLaunchKernelGGL(q8_0_repack_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, blocks, nblocks,
                     qs, scales);
  return hipGetLastError();
}

// ---- integer-dot Q8_0 linear: candle's CPU QMatMul semantics ----------------
//
// The reference's quantized Linear::forward (runtime/nn_blocks.rs:80-93) on
// the CPU quantizes each x row to Q8_0 blocks and takes integer dot
// products with the weight blocks (candle-core quantized/k_quants.rs,
// BlockQ8_0::from_float and vec_dot). Here:
// - q8_0_quantize_rows_kernel: eight lanes per 32-value block (16 bytes
//   each): amax = max |x| (NaN ignored, at least 0), d = amax / 127, id =
//   d != 0 ? 1 / d : 0 (correctly rounded f32 divisions), q = round half
//   away from zero of x * id, saturated to int8 with NaN -> 0, and d rounded
//   to f16 (RNE) and widened back to f32;
// - q8_0_int8_gemm_kernel: one v_mfma_i32_32x32x32_i8 per 32 x 32 tile and
//   Q8_0 block gives that block's exact int32 dot products; each is then
//   folded into the f32 sum as candle's generic vec_dot does, in block
//   order: acc = acc + ((f32)isum * wd) * xd, every operation rounded
//   (mul_rn / add_rn: no contraction), and y = acc + bias. The result is
//   bit-identical to candle's CPU path. The f32 fold (4 VALU operations per
//   output and block) bounds the kernel, not the int8 matrix rate.

__global__ __launch_bounds__(256) void q8_0_quantize_rows_kernel(Q8IntParams p) {
  const int64_t nb = p.K / 32;
  const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t blk = g >> 3;
  const int part = (int)(g & 7);
  const bool live = blk < p.M * nb;
  const int64_t bc = live ? blk : 0;
  const int64_t m = bc / nb, b = bc - m * nb;
  const float4 v = *reinterpret_cast<const float4 *>(p.x + m * p.ldx + b * 32 + part * 4);
  const float xv[4] = {v.x, v.y, v.z, v.w};
  // f32::max ignores a NaN operand; fmaxf (IEEE maxNum) does the same
  float a = fmaxf(fmaxf(fabsf(xv[0]), fabsf(xv[1])), fmaxf(fabsf(xv[2]), fabsf(xv[3])));
  a = fmaxf(a, dpp<DPP_XOR1>(a));
  a = fmaxf(a, dpp<DPP_XOR2>(a));
  a = fmaxf(a, dpp<DPP_HALF_MIRROR>(a));  // the 8 lanes of the block
  const float amax = fmaxf(a, 0.0f);       // candle starts its maximum at 0
  const float d = amax / 127.0f;
  const float id = d != 0.0f ? 1.0f / d : 0.0f;
  uint32_t packed = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float r = roundf(mul_rn(xv[k], id));
    const int q = r != r ? 0 : (r >= 127.0f ? 127 : (r <= -128.0f ? -128 : (int)r));
    packed |= ((uint32_t)(uint8_t)(int8_t)q) << (8 * k);
  }
  if (!live) return;
  *reinterpret_cast<uint32_t *>(p.xq + m * p.K + b * 32 + part * 4) = packed;
  if (part == 0) p.xd[b * p.ldxd + m] = (float)(_Float16)d;  // block-major
}

// 256 threads (2 x 2 wavefronts of 32 x 32 tiles) per 64 x 64 tile of y; a
// stage is two Q8_0 blocks (k-step 64), double-buffered through LDS: rows of
// 64 int8 at an 80-byte stride (conflict-free 16-byte fragment reads) and
// the stage's block scales of the tile's 64 x rows and 64 weight rows. The
// second block's MFMA is issued before the first block's f32 fold, so the
// matrix core runs beside the fold's VALU work. An odd last block is loaded
// twice and folded once.
constexpr int kI8Tile = 64, kI8Row = 80;
__global__ __launch_bounds__(256) void q8_0_int8_gemm_kernel(Q8IntParams p, int tiles_n) {
  typedef int i32x4_t_ __attribute__((ext_vector_type(4)));
  typedef int i32x16_t_ __attribute__((ext_vector_type(16)));
  __shared__ __align__(16) int8_t As[2][kI8Tile * kI8Row];
  __shared__ __align__(16) int8_t Bs[2][kI8Tile * kI8Row];
  __shared__ __align__(16) float Ad[2][2][kI8Tile];  // [buffer][block of the stage][row]
  __shared__ __align__(16) float Bd[2][2][kI8Tile];
  (void)tiles_n;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), wm = wave >> 1,
            wn = wave & 1;
  const int64_t m0 = (int64_t)blockIdx.y * kI8Tile, n0 = (int64_t)blockIdx.x * kI8Tile;
  const int64_t nb = p.K / 32, nst = (nb + 1) / 2;
  // loaders: thread t moves the 16 bytes (t & 3) of x row t / 4 and of weight
  // row t / 4 per stage (rows past M / N clamped: loaded, computed, never
  // stored); wavefronts 0-1 the x scales (block wave & 1 of the stage, row
  // lane), 2-3 the weight scales
  const int lr = t >> 2, lq = t & 3;
  const int64_t ra = m0 + lr < p.M ? m0 + lr : p.M - 1, rb = n0 + lr < p.N ? n0 + lr : p.N - 1;
  const int8_t *sa = p.xq + ra * p.K + lq * 16, *sb = p.qs + rb * p.K + lq * 16;
  const int so = lr * kI8Row + lq * 16;
  const int sr = lane, sbk = wave & 1;
  const bool sx = wave < 2;
  const int64_t swr = n0 + sr < p.N ? n0 + sr : p.N - 1;
  // the thread's scale column: x scales are block-major (stride ldxd per
  // block), weight scales row-major (stride 1); the stride is wave-uniform
  const float *sp = sx ? p.xd + m0 + sr : p.scales + swr * nb;
  const int64_t sstep = sx ? p.ldxd : 1;
  // an odd last stage holds block nb - 1 in both halves: threads of the
  // second half (lq 2, 3) read 32 bytes back, and both scale rows read it
  const int back = lq >= 2 ? 32 : 0;
  uint4 va, vb;
  float vs;
  auto load = [&](int64_t st) {
    int64_t o = st * 64, kb = 2 * st + sbk;
    if (2 * st + 1 == nb) {
      o -= back;
      kb = 2 * st;
    }
    va = *reinterpret_cast<const uint4 *>(sa + o);
    vb = *reinterpret_cast<const uint4 *>(sb + o);
    vs = sp[kb * sstep];
  };
  auto store = [&](int buf) {
    *reinterpret_cast<uint4 *>(&As[buf][so]) = va;
    *reinterpret_cast<uint4 *>(&Bs[buf][so]) = vb;
    (sx ? Ad[buf][sbk] : Bd[buf][sbk])[sr] = vs;
  };
  load(0);
  store(0);
  lds_barrier();

  float acc[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = 0.f;
  const int fr = lane & 31, fk = (lane >> 5) * 16;
  auto fold = [&](const i32x16_t_ &c, int buf, int blk) {
    const float wd = Bd[buf][blk][wn * 32 + fr];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      // rows 8q + 4 (lane / 32) + 0..3 of the wavefront's 32
      const float4 xd4 = *reinterpret_cast<const float4 *>(&Ad[buf][blk][wm * 32 + 8 * q + 4 * (lane >> 5)]);
      const float xd[4] = {xd4.x, xd4.y, xd4.z, xd4.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int e = 4 * q + i;
        acc[e] = add_rn(acc[e], mul_rn(mul_rn((float)c[e], wd), xd[i]));
      }
    }
  };
  // a wavefront whose 32 rows all lie past M (in the last row of tiles) only
  // loads and synchronises: its products would never be stored
  const bool rows_live = m0 + wm * 32 < p.M;  // wave-uniform
  for (int64_t st = 0; st < nst; ++st) {
    const int buf = (int)(st & 1);
    if (st + 1 < nst) load(st + 1);
    if (rows_live) {
      const int8_t *a = &As[buf][(wm * 32 + fr) * kI8Row + fk], *b = &Bs[buf][(wn * 32 + fr) * kI8Row + fk];
      const i32x16_t_ c0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(*reinterpret_cast<const i32x4_t_ *>(a),
                                                                 *reinterpret_cast<const i32x4_t_ *>(b), i32x16_t_{},
                                                                 0, 0, 0);
      // an odd last stage holds block nb - 1 in both halves: its second
      // product is computed and not folded
      const i32x16_t_ c1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(*reinterpret_cast<const i32x4_t_ *>(a + 32),
                                                                 *reinterpret_cast<const i32x4_t_ *>(b + 32),
                                                                 i32x16_t_{}, 0, 0, 0);
      fold(c0, buf, 0);
      if (2 * st + 1 < nb) fold(c1, buf, 1);
    }
    if (st + 1 < nst) store(buf ^ 1);
    lds_barrier();
  }
  // lane holds y[8 (e / 4) + 4 (lane / 32) + e % 4][lane % 32] of its 32 x 32 tile
  const int64_t col = n0 + wn * 32 + fr;
  if (col >= p.N) return;
  const float bias = p.bias ? p.bias[col] : 0.f;
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const int64_t row = m0 + wm * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
    if (row < p.M) p.y[row * p.ldy + col] = p.bias ? add_rn(acc[e], bias) : acc[e];
  }
}

hipError_t launch_q8_0_gemm(int out_dt, const Q8GemmParams &p, hipStream_t s) {
  if (p.M <= 0 || p.N <= 0) return hipSuccess;
  if (p.K <= 0 || p.K % kBK) return hipErrorInvalidValue;
  if (p.x_f32 && (p.K % 64 || (127 * p.ldx + p.K) * 4 > 0x7FFFFFFF || 256 * p.K > 0x7FFFFFFF))
    return hipErrorInvalidValue;
  if ((p.N + 127) / 128 > INT32_MAX || (p.M + 127) / 128 > 65535) return hipErrorInvalidValue;
  switch (out_dt) {
    case LUX3D_BF16: return launch_tiles<BF16>(p, s);
    case LUX3D_F16: return launch_tiles<F16>(p, s);
    case LUX3D_F32: return launch_tiles<F32>(p, s);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_q8_0_quantize_rows(const Q8IntParams &p, hipStream_t s) {
  if (p.M <= 0) return hipSuccess;
  if (p.K <= 0 || p.K % 32) return hipErrorInvalidValue;
  const int64_t lanes = p.M * (p.K / 32) * 8;
  if ((lanes + 255) / 256 > INT32_MAX) return hipErrorInvalidValue;
  hipLaunchKernelGGL(q8_0_quantize_rows_kernel, dim3((unsigned)((lanes + 255) / 256)), dim3(256), 0, s, p);
  return hipGetLastError();
}

hipError_t launch_q8_0_int8_gemm(const Q8IntParams &p, hipStream_t s) {
  if (p.M <= 0 || p.N <= 0) return hipSuccess;
  if (p.K <= 0 || p.K % 32 || p.ldxd < (p.M + kI8Tile - 1) / kI8Tile * kI8Tile) return hipErrorInvalidValue;
  const int64_t tn = (p.N + kI8Tile - 1) / kI8Tile, tm = (p.M + kI8Tile - 1) / kI8Tile;
  if (tn > INT32_MAX || tm > 65535) return hipErrorInvalidValue;
  hipLaunchKernelGGL(q8_0_int8_gemm_kernel, dim3((unsigned)tn, (unsigned)tm), dim3(256), 0, s, p, (int)tn);
  return hipGetLastError();
}

}  // namespace lux3d
