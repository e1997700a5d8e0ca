// gemm.hip — LoRA-linear GEMMs for gfx950 (CDNA4): C[M,N] = A[M,K]·op(B), B
// [K,N] (frozen W in the forward, tied embedding in the LM-head backward) or
// [N,K] (W in dX = dY·Wᵀ, embedding in the LM-head forward).
//
// gemm(): fp32 operands (or fp16 B of a shape the fp16 kernel does not take)
// on the bf16 matrix cores, every fp32 value as three bf16 terms
// (gemm_x.hip), or, small products of the operators, on the fp32 matrix cores.  gemm_h(): fp16 B on the fp16 matrix cores, the fp32 operand
// as two fp16 terms with a row scale.  Both fuse bias, the rank-r LoRA term
// scale·P[M,r]·Q, a residual add and accumulation into C; split-K partials
// are summed with the epilogue (and a row norm) by a second launch.
#include <cfloat>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <type_traits>

#include <hip/hip_ext.h>

#include "gemm_common.h"

namespace mft {
namespace {

// Sum of the split-K partials in split order plus the epilogue.  Rows are
// blockIdx.y; each thread takes four consecutive columns (128-bit partial
// loads when N is a multiple of 4).
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ partial, int splits,
                                                            int M, int N, float* C, int64_t ldc,
                                                            GemmEpilogue ep) {
  const int n0 = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (n0 >= N) return;
  const int64_t total = (int64_t)M * N;
  for (int m = blockIdx.y; m < M; m += gridDim.y) {
    const float* src = partial + (int64_t)m * N + n0;
    if ((N & 3) == 0) {
      floatx4 s = *reinterpret_cast<const floatx4*>(src);
      for (int z = 1; z < splits; ++z) s += *reinterpret_cast<const floatx4*>(src + (int64_t)z * total);
#pragma unroll
      for (int e = 0; e < 4; ++e) epilogue_store(ep, s[e], m, n0 + e, C, ldc);
    } else {
      for (int e = 0; e < 4 && n0 + e < N; ++e) {
        float s = 0.f;
        for (int z = 0; z < splits; ++z) s += src[(int64_t)z * total + e];
        epilogue_store(ep, s, m, n0 + e, C, ldc);
      }
    }
  }
}

// ---- small fp32 products -------------------------------------------------------
// C = A·op(B) on the fp32 matrix cores for products of few tiles (plan_gemm_x
// chooses; both sides' times stand there).  gemm_x_kernel's panel step is a
// chain of splitting instructions, 0.42 µs however small the tile; here it is
// 16 MFMAs a wave, 0.21 µs of the matrix core, and 0.31 with the barrier and
// the LDS reads that nothing hides at one workgroup a CU.  Half the tile, so
// that small outputs reach more CUs.
// Workgroup tile 32×64, four waves as 2×2, each owning 16×32 outputs as two
// v_mfma_f32_16x16x4_f32 tiles; K in panels of 32.  Lane (i, g) supplies
// A[row i][k g] and B[k g][col i] and holds D[row 4g+v][col i]; over four
// consecutive MFMAs lane group g takes k = 4g..4g+3 of a 16-wide k block, so
// an A or [N,K] B fragment is one 128-bit LDS read; with B as [K,N] the
// wave's two column tiles interleave (tile b holds columns 2i + b) and one
// 64-bit read a k gives a lane its B values of both.
//
// Every k step of two panels has accumulators of its own (sixteen sets of 8
// registers, added pairwise at the end): no MFMA waits for the one before it,
// and a chain holds K/16 products, so that from K = 256 on the sums are as
// close to 64 bits as gemm_x_kernel's.
//
// Panel entry j lives in LDS stage j % 3 and is stored two steps before it is
// multiplied, so that in step j every wave already holds the fragments of the
// first k block of entry j+1; global loads run four entries ahead through two
// register sets.  One barrier a step.  The loop runs two steps per iteration:
// an odd panel count starts with an entry of zeros, and loads past the last
// panel re-read it.  TAIL: K not a multiple of 32, or fp16 B; elements of the
// last panel at k ≥ K are zeroed at the store.
template <bool B_NK, bool B_F16, bool RANK, bool TAIL>
__global__ __launch_bounds__(256) void gemm_s_kernel(GemmParams p) {
  constexpr int BM = 32, BN = 64, BK = 32;
  constexpr int PA = BK + 4;
  // [K,N] B: 4·PB ≡ 32 (mod 64) puts lane groups g and g+1 of a 64-bit
  // fragment read in disjoint LDS bank halves
  constexpr int PB = B_NK ? BK + 4 : BN + 8;
  constexpr int A_STAGE = BM * PA, STAGE = A_STAGE + (B_NK ? BN : BK) * PB;
  constexpr int N_LD = 3;  // 16-byte chunks of a panel per thread: one of A, two of B
  constexpr int BES = B_F16 ? 2 : 4;
  __shared__ __attribute__((aligned(16))) float smem[3 * STAGE];

  int tile, split;
  float* raw_tile;
  if (!tile_slice<BM, BN>(p, tile, split, raw_tile)) return;
  const int m0 = tile % p.tiles_m * BM, n0 = tile / p.tiles_m * BN;
  const int kbeg = split * p.k_chunk;
  const int klen = tile < p.full_tiles ? p.K : min(p.K - kbeg, p.k_chunk);
  const int nk = (klen + BK - 1) / BK, odd = nk & 1;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = (wave & 1) * 16, wn = (wave >> 1) * 32;
  const int li = lane & 15, lg = lane >> 4;

  floatx4 acc[16][2];
#pragma unroll
  for (int t = 0; t < 16; ++t)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[t][b] = floatx4{0.f, 0.f, 0.f, 0.f};

  // buffer resources based at the tile's first row / column of its K-slice
  const __amdgpu_buffer_rsrc_t rsa = buf_rsrc(p.A + (int64_t)m0 * p.lda + kbeg);
  const __amdgpu_buffer_rsrc_t rsb =
      buf_rsrc(static_cast<const char*>(p.B) + (B_NK ? (int64_t)n0 * p.ldb + kbeg : (int64_t)kbeg * p.ldb + n0) * BES);
  const int a_row = tid / 8, kq = tid % 8 * 4;  // of [rows][32] chunks
  const uint32_t a_off = (uint32_t)(((int64_t)(min(m0 + a_row, p.M - 1) - m0) * p.lda + kq) * 4);
  uint32_t b_off[2];
  int b_lds[2];  // LDS offsets (floats) within a stage
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    if constexpr (B_NK) {
      const int row = a_row + 32 * it;
      b_off[it] = (uint32_t)(((int64_t)(min(n0 + row, p.N - 1) - n0) * p.ldb + kq) * BES);
      b_lds[it] = A_STAGE + row * PB + kq;
    } else {
      const int k = tid / 16 + 16 * it, nq = tid % 16 * 4;
      b_off[it] = (uint32_t)(((int64_t)k * p.ldb + (n0 + nq < p.N ? nq : 0)) * BES);
      b_lds[it] = A_STAGE + k * PB + nq;
    }
  }

  floatx4 rs[2][N_LD];  // register staging sets
  // entry j holds panel j − odd, clamped to the slice's
  auto kof = [&](int j) { return min(max(j - odd, 0), nk - 1) * BK; };
  // TAIL: chunks at k ≥ klen re-read the row's first of the panel, rows at
  // k ≥ klen the panel's first row
  auto gload = [&](auto sc, int j) {
    constexpr int S = decltype(sc)::value;
    const int kc = kof(j);
    const uint32_t kback = TAIL && kc + kq >= klen ? (uint32_t)kq : 0u;
    rs[S][0] = buf_load4(rsa, a_off - kback * 4u, (uint32_t)kc * 4u);
    const uint32_t boff = (uint32_t)((B_NK ? (int64_t)kc : (int64_t)kc * p.ldb) * BES);
#pragma unroll
    for (int it = 0; it < 2; ++it) {
      const int k = tid / 16 + 16 * it;
      const uint32_t back = B_NK ? kback * BES : TAIL && kc + k >= klen ? (uint32_t)((int64_t)k * p.ldb) * BES : 0u;
      if constexpr (B_F16) rs[S][1 + it] = stash_f16(buf_load2u(rsb, b_off[it] - back, boff));
      else rs[S][1 + it] = buf_load4(rsb, b_off[it] - back, boff);
    }
  };
  auto lstore = [&](auto sc, int stage, int j) {
    constexpr int S = decltype(sc)::value;
    float* st = smem + stage * STAGE;
#pragma unroll
    for (int it = 0; it < N_LD; ++it) {
      floatx4 v = rs[S][it];
      if (B_F16 && it > 0) v = unstash_f16(v);
      if (TAIL) {  // without a branch, which would end the schedule of the step
        const bool row = !B_NK && it > 0;  // the chunk lies along N
        const int k = kof(j) + (row ? tid / 16 + 16 * (it - 1) : kq);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = k + (row ? 0 : e) < klen ? v[e] : 0.f;
      }
      *reinterpret_cast<floatx4*>(st + (it == 0 ? a_row * PA + kq : b_lds[it - 1])) = v;
    }
  };
  struct Frags {
    floatx4 a, b[2];
  };
  auto read_frags = [&](Frags& f, int stage, int kb) {
    const float* as = smem + stage * STAGE;
    const float* bs = as + A_STAGE;
    f.a = *reinterpret_cast<const floatx4*>(as + (wm + li) * PA + kb + 4 * lg);
    if constexpr (B_NK) {
#pragma unroll
      for (int b = 0; b < 2; ++b) f.b[b] = *reinterpret_cast<const floatx4*>(bs + (wn + 16 * b + li) * PB + kb + 4 * lg);
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const float2 v = *reinterpret_cast<const float2*>(bs + (kb + 4 * lg + t) * PB + wn + 2 * li);
        f.b[0][t] = v.x;
        f.b[1][t] = v.y;
      }
    }
  };
  auto mfmas = [&](const Frags& f, auto sc, auto qc) {
    constexpr int T = 8 * decltype(sc)::value + 4 * decltype(qc)::value;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int b = 0; b < 2; ++b)
        acc[T + t][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.a[t], f.b[b][t], acc[T + t][b], 0, 0, 0);
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;

  constexpr int N_RD = 1 + (B_NK ? 2 : 4);  // LDS read instructions per read_frags
  Frags F[2];
  int s_cur = 0, s_nxt = 1, s_st = 2;  // stages of entries j, j+1, j+2 (wave-uniform)
  auto step = [&](auto sc, int j) {
    read_frags(F[1], s_cur, 16);
    mfmas(F[0], sc, I0{});
    read_frags(F[0], s_nxt, 0);  // entry j+1, visible since the last barrier
    lstore(sc, s_st, j + 2);     // loaded two steps ago
    gload(sc, j + 4);            // into the same register set
    mfmas(F[1], sc, I1{});
    __builtin_amdgcn_sched_group_barrier(0x100, N_RD, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, N_RD, 0);
#pragma unroll
    for (int i = 0; i < N_LD; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
    }
#pragma unroll
    for (int i = 0; i < N_LD; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 8 - 2 * N_LD, 0);
    __syncthreads();
    const int t = s_cur;
    s_cur = s_nxt;
    s_nxt = s_st;
    s_st = t;
  };
  gload(I0{}, 0);
  gload(I1{}, 1);
  if (odd) {  // the entry of zeros
    for (int i = tid; i < STAGE / 4; i += 256) reinterpret_cast<floatx4*>(smem)[i] = floatx4{0.f, 0.f, 0.f, 0.f};
  } else {
    lstore(I0{}, 0, 0);
  }
  lstore(I1{}, 1, 1);
  gload(I0{}, 2);
  gload(I1{}, 3);
  __syncthreads();
  read_frags(F[0], 0, 0);
  for (int j = 0; j < nk + odd; j += 2) {
    step(I0{}, j);
    step(I1{}, j + 1);
  }
#pragma unroll
  for (int o = 8; o >= 1; o /= 2)
#pragma unroll
    for (int t = 0; t < o; ++t)
#pragma unroll
      for (int b = 0; b < 2; ++b) acc[t][b] += acc[t + o][b];

  // Rank-r LoRA term: one more K panel of depth r, staged in the ring's LDS
  // after the last step's barrier; split 0 only.
  if (RANK && split == 0) {
    const int r = p.ep.r, rp = (r + 3) & ~3, pr = rp + 1;
    float* Ps = smem;
    float* Qs = smem + BM * pr;
    for (int i = tid; i < BM * rp; i += 256) {
      const int row = i / rp, j = i % rp, m = m0 + row;
      Ps[row * pr + j] = (m < p.M && j < r) ? p.ep.P[(int64_t)m * r + j] : 0.f;
    }
    for (int i = tid; i < BN * rp; i += 256) {
      const int col = i / rp, j = i % rp, n = n0 + col;
      Qs[col * pr + j] = (n < p.N && j < r) ? p.ep.lscale * p.ep.Q[(int64_t)n * p.ep.qsn + (int64_t)j * p.ep.qsj] : 0.f;
    }
    __syncthreads();
    for (int t = 0; t < rp / 4; ++t) {
      const float fp = Ps[(wm + li) * pr + 4 * t + lg];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const float fq = Qs[(wn + (B_NK ? 16 * b + li : 2 * li + b)) * pr + 4 * t + lg];
        acc[0][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(fp, fq, acc[0][b], 0, 0, 0);
      }
    }
  }
  tile_out<BM, BN, 3 * STAGE * 4>(p, smem, m0, n0, split, [&](auto&& put) {
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int v = 0; v < 4; ++v) put(wm + 4 * lg + v, wn + (B_NK ? 16 * b + li : 2 * li + b), acc[0][b][v]);
  }, raw_tile);
}

// ---- fp16 matrix-core path ---------------------------------------------------
// Frozen W stored as fp16 is exact in fp16, so y = x·W can run on the fp16
// matrix cores (v_mfma_f32_16x16x32_f16: 8× the fp32 MFMA rate) once the fp32
// operand x is carried by two fp16 values.  Row m of x is scaled by
// s_m = 2^(14 − ⌊log2 max|x_m|⌋), so that max|x_m·s_m| ∈ [2^14, 2^15) sits
// inside fp16's range, and split into hi = fp16(x·s) and lo = fp16(x·s − hi),
// both rounded to nearest even (x·s and x·s − hi are exact in fp32).  The
// pair keeps x·s to within 2^-22·|x·s| (or 2^-25 absolute where lo is
// subnormal, far below the row maximum): 22 of fp32's 24 significand bits.
// Products of fp16 values are exact in fp32 and the matrix cores accumulate
// in fp32, so diag(1/s)·(hi·W + lo·W) differs from the fp32 product by a few
// units of 2^-22 relative.  The GEMM splits its A tiles while staging them
// into LDS; the row scales come from a pass that already reads every row
// (the rank-r projections of the LoRA branch, rank_batch) or from
// row_scale_kernel.  inv_s[m] = 1/s_m is a power of two.
// inv_s[m] of rows x[m, 0:K) (K a multiple of 4), one workgroup per row.
// fmaxf drops NaN operands; NaN and ±inf entries pass through the split
// unchanged (their rows' products are NaN / inf as in fp32).
__global__ __launch_bounds__(256) void row_scale_kernel(const float* __restrict__ x, int64_t ldx, int K,
                                                        float* __restrict__ inv_s) {
  __shared__ float red[4];
  const int m = blockIdx.x, tid = threadIdx.x;
  const float* xr = x + (int64_t)m * ldx;
  float mx = 0.f;
  for (int k = 4 * tid; k < K; k += 1024) {
    const floatx4 v = *reinterpret_cast<const floatx4*>(xr + k);
    mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))));
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  if ((tid & 63) == 0) red[tid >> 6] = mx;
  __syncthreads();
  if (tid == 0) inv_s[m] = row_inv_scale(fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])));
}

// hi/lo split of two fp32 values x0, x1 scaled by s, packed two fp16 per
// register: hi = fp16(x·s), lo = fp16(x·s − hi), both rounded to nearest
// even from the exact fp32 value (the fma forms x·s − hi exactly).  Four
// mixed-precision fmas write each half in place (mixlo keeps the high half,
// mixhi the low), instead of converts plus shift-and-or packing.
__device__ __forceinline__ void split2_f16(float x0, float x1, float s, uint32_t& hi, uint32_t& lo) {
  asm("v_fma_mixlo_f16 %0, %2, %4, 0\n\t"
      "v_fma_mixhi_f16 %0, %3, %4, 0\n\t"
      "v_fma_mixlo_f16 %1, %2, %4, -%0 op_sel_hi:[0,0,1]\n\t"
      "v_fma_mixhi_f16 %1, %3, %4, -%0 op_sel:[0,0,1] op_sel_hi:[0,0,1]"
      : "=&v"(hi), "=&v"(lo)
      : "v"(x0), "v"(x1), "v"(s));
}

typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));

// A column segment of a segmented launch: output columns [n0, next n0) of
// the launch take their own B, C and rank-r panel (P, Q) — the q, k and v
// (or gate and up) projections of one shared input in one launch.
struct GemmHSegment {
  int n0;
  const uint16_t* B;
  int64_t ldb;
  float* C;
  int64_t ldc;
  const float* P;
  const float* Q;
};
constexpr int kMaxGemmHSegments = 3;
// A K segment of a K-segmented launch ([N,K] B only): reduction indices
// [k0, next k0) take their own B (fp16 [N][ldb]), the row scales of their A
// columns and their rank-r panel — dX = Σ_g dY_g·W_gᵀ over the q, k and v (or
// gate and up) projections, whose dY are column blocks of one A.
struct GemmHKSegment {
  int k0;
  const uint16_t* B;
  int64_t ldb;
  const float* inv_s;
  const float* P;
  const float* Q;
};

struct GemmHParams {
  const float* A;      // fp32 [M][lda]
  const float* inv_s;  // [M] row scales 1/s_m (powers of two), or null (s = 1)
  const uint16_t* B;   // fp16 [N][ldb] (B_NK) or [K][ldb]
  float* C;
  int64_t lda, ldb, ldc;
  int M, N, K;
  int k_chunk;
  int tiles_m, tiles_n, tiles_per_xcd;
  int splits, spread;
  float* partial;
  int out_vec;  // output rows allow 128-bit stores (tile_out)
  GemmEpilogue ep;
  int nseg;  // > 1: column segments (unsplit K, every segment a whole number of BN-wide tiles)
  GemmHSegment seg[kMaxGemmHSegments];
  int nkseg;  // > 1: K segments (B_NK; every segment a whole number of 32-deep panels)
  GemmHKSegment kseg[kMaxGemmHSegments];
};

// Workgroup → (tile, split) of a 1-D grid.  Workgroup L runs on XCD L % 8
// (round-robin dispatch), each XCD with its own L2.  With s ≤ 8 splits, the
// s K-slices take 8/s XCDs each and their tiles are cut into contiguous
// ranges among those XCDs, M-fastest, so an XCD reads whole column bands of
// B and the A rows of only its own K-slice (a split-K launch that spread
// every slice over every XCD would fetch the whole of A into each of the 8
// L2s).  With `spread` (used for s > 8) every K-slice covers all 8 XCDs.
// Host side: tiles_per_xcd = ceil(tiles / (8/s)), or ceil(tiles/8) spread.
__device__ __forceinline__ bool tile_of(const GemmHParams& p, int& tile, int& split) {
  const int L = blockIdx.x, xcd = L % 8, idx = L / 8;
  const int tiles = p.tiles_m * p.tiles_n;
  if (p.spread) {
    const int per = 8 * p.tiles_per_xcd, r = L % per;
    split = L / per;
    tile = (r % 8) * p.tiles_per_xcd + r / 8;
  } else {  // s ≤ 8
    const int g = 8 / p.splits;  // XCDs per split
    split = xcd / g;
    tile = (xcd % g) * p.tiles_per_xcd + idx;
  }
  return tile < tiles && split < p.splits;
}

// C = diag(inv_s)·(hi + lo)·op(B) (+ a rank-r panel on the fp32 matrix cores,
// and tile_out's epilogue), hi/lo the fp16 split of diag(s)·A made while A's fp32
// panel is staged into LDS.  Workgroup tile BM×BN, four waves as 2×2, each
// owning (BM/2)×(BN/2) outputs as 16×16 tiles; K in panels of 32 (one
// v_mfma_f32_16x16x32_f16 k-block: lane l holds row l%16, k 8(l/16)..+7 of
// each operand).  LDS per stage: the hi and lo A planes [BM][32] and B as
// [BN][32] (B_NK) or [32][BN] (k-major, as W [K,N] is stored): k-major B
// fragments come out of LDS through ds_read_b64_tr_b16, which hands lane
// 4a+e of every 16-lane group element e of the 8-byte rows addressed by
// lanes a, a+4, a+8, a+12 — lanes addressing rows k..k+3 at columns
// n0 + 4·(0..3) give each lane four consecutive k of its own column, so W
// needs no transposed copy.  Pipeline: a three-stage LDS ring stored two
// steps ahead, global loads PIPE + 2 steps ahead in PIPE register sets,
// fragments of the next stage read at the top of each step, one barrier per
// step.  Row pitches: 40 halves (A, [N,K] B: 16-byte
// fragment reads conflict-free over 8 lanes), BN + 16 halves (k-major B:
// the four rows of a 16-lane transposed read fall in disjoint banks).
template <int BM, int BN, bool B_NK, bool RANK, int PIPE>
__global__ __launch_bounds__(256) void gemm_h_kernel(GemmHParams p) {
  constexpr int BK = 32;
  constexpr int TA = BM / 32, TB = BN / 32;  // 16×16 tiles per wave along M and N
  constexpr int PA = BK + 8;
  constexpr int PT = BN + 16;
  constexpr int A_PL = BM * PA;
  constexpr int B_PL = B_NK ? BN * PA : BK * PT;
  constexpr int STAGE = 2 * A_PL + B_PL;  // halves
  constexpr int A_ITEMS = BM * BK / 4 / 256;  // 16-byte fp32 chunks of A per thread
  constexpr int B_ITEMS = BN * BK / 8 / 256;  // 16-byte fp16 chunks of B per thread
  constexpr int N_ST = A_ITEMS + B_ITEMS;     // global loads per panel
  constexpr int N_WR = 2 * A_ITEMS + B_ITEMS; // LDS stores per panel
  static_assert(A_ITEMS >= 1 && B_ITEMS >= 1 && TA >= 1 && TB >= 1, "tile config");
  __shared__ __attribute__((aligned(16))) uint16_t smem[3 * STAGE];

  int tile, split;
  if (!tile_of(p, tile, split)) return;
  const int tm_idx = tile % p.tiles_m;
  const int tn_idx = tile / p.tiles_m;
  const int m0 = tm_idx * BM;
  int n0 = tn_idx * BN;
  static_assert(kMaxGemmHSegments == 3, "segment selects below");
  if (p.nseg > 1) {  // the tile's column segment (uniform): its operands, columns relative to it
    // selects over constant indices only: a computed index into the kernel
    // arguments would copy them to scratch memory
    const int g = p.nseg > 2 && n0 >= p.seg[2].n0 ? 2 : n0 >= p.seg[1].n0 ? 1 : 0;
#define MFT_SEG(f) (g == 0 ? p.seg[0].f : g == 1 ? p.seg[1].f : p.seg[2].f)
    const int nb = MFT_SEG(n0);
    const int ne = g == 0 ? p.seg[1].n0 : g == 1 && p.nseg > 2 ? p.seg[2].n0 : p.N;
    p.B = MFT_SEG(B);
    p.ldb = MFT_SEG(ldb);
    p.C = MFT_SEG(C);
    p.ldc = MFT_SEG(ldc);
    p.ep.P = MFT_SEG(P);
    p.ep.Q = MFT_SEG(Q);
#undef MFT_SEG
    n0 -= nb;
    p.N = ne - nb;
  }
  const int kbeg = split * p.k_chunk;
  const int kend = min(p.K, kbeg + p.k_chunk);
  const int nk = (kend - kbeg) / BK;  // whole panels (checked on the host)
  const int pad = (PIPE - nk % PIPE) % PIPE;  // leading zero entries: the step loop runs PIPE steps per iteration
  const int T = nk + pad;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = (wave & 1) * (BM / 2), wn = (wave >> 1) * (BN / 2);
  const int li = lane & 15, lg = lane >> 4;

  floatx4 acc[TA][TB];
#pragma unroll
  for (int a = 0; a < TA; ++a)
#pragma unroll
    for (int b = 0; b < TB; ++b) acc[a][b] = floatx4{0.f, 0.f, 0.f, 0.f};

  // buffer resources based at the tile's first row / column of its K-slice
  const __amdgpu_buffer_rsrc_t rsa = buf_rsrc(p.A + (int64_t)m0 * p.lda + kbeg);
  const __amdgpu_buffer_rsrc_t rsb =
      buf_rsrc(p.B + (B_NK ? (int64_t)n0 * p.ldb + kbeg : (int64_t)kbeg * p.ldb + n0));
  // K segments: every segment's B based at the tile's first column (its own
  // pitch); a panel takes the segment holding its first k (selects over
  // constant indices keep the kernel arguments in scalar registers)
  static_assert(kMaxGemmHSegments == 3, "K-segment selects below");
  const bool kseg = B_NK && p.nkseg > 1;

  const int64_t kldb1 = p.kseg[1].ldb, kldb2 = p.kseg[2].ldb;
  const int kk1 = p.kseg[1].k0, kk2 = p.kseg[2].k0;
  // 1/s_m of row m: with K segments the largest of the segments' scales
  // (their A blocks share one row scale, so the products sum in one accumulator)
  auto row_isc = [&](int m) {
    if (!kseg) return p.inv_s[m];
    float v = fmaxf(p.kseg[0].inv_s[m], p.kseg[1].inv_s[m]);
    return p.nkseg > 2 ? fmaxf(v, p.kseg[2].inv_s[m]) : v;
  };
  uint32_t a_off[A_ITEMS], b_off[B_ITEMS];
  int b_row[B_ITEMS], b_kq[B_ITEMS];   // [N,K] B chunk: row within the tile, k within the panel
  int a_lds[A_ITEMS], b_lds[B_ITEMS];  // LDS offsets (halves) within a stage
  float a_sc[A_ITEMS];                 // s_m of each A chunk's row
#pragma unroll
  for (int it = 0; it < A_ITEMS; ++it) {
    const int flat = tid + 256 * it;
    const int row = flat / 8, kq = (flat % 8) * 4;
    const int mr = min(m0 + row, p.M - 1);
    a_off[it] = (uint32_t)(((int64_t)(mr - m0) * p.lda + kq) * 4);
    a_lds[it] = row * PA + kq;
    a_sc[it] = p.inv_s ? 1.f / row_isc(mr) : 1.f;  // exact: a power of two
  }
#pragma unroll
  for (int it = 0; it < B_ITEMS; ++it) {
    const int flat = tid + 256 * it;
    if constexpr (B_NK) {
      const int row = flat / 4, kq = (flat % 4) * 8;
      b_row[it] = min(n0 + row, p.N - 1) - n0;
      b_kq[it] = kq;
      b_off[it] = (uint32_t)(((int64_t)b_row[it] * p.ldb + kq) * 2);
      b_lds[it] = 2 * A_PL + row * PA + kq;
    } else {
      const int k = flat / (BN / 8), nq = (flat % (BN / 8)) * 8;
      b_off[it] = (uint32_t)(((int64_t)k * p.ldb + (n0 + nq < p.N ? nq : 0)) * 2);
      b_lds[it] = 2 * A_PL + k * PT + nq;
    }
  }

  floatx4 rs[PIPE][N_ST];  // register staging sets (16-byte chunks as floats); entry e in set e % PIPE
  auto gload = [&](auto sc, int j) {
    constexpr int S = decltype(sc)::value;
    const int kc = min(max(j - pad, 0), nk - 1) * BK;
#pragma unroll
    for (int it = 0; it < A_ITEMS; ++it) rs[S][it] = buf_load4(rsa, a_off[it], (uint32_t)kc * 4u);
    if constexpr (B_NK) {
      // selects only (no branch): the panel's segment — always 0 without K
      // segments, where segment 0's B is the whole of B
      const int kg = kbeg + kc;  // the panel's first k in the whole reduction
      const int g = !kseg ? 0 : p.nkseg > 2 && kg >= kk2 ? 2 : kg >= kk1 ? 1 : 0;
      // the pointer is selected, then made a resource (selecting among three
      // resources, or among pointers computed ahead of the loop, puts them in
      // scratch memory)
      const __amdgpu_buffer_rsrc_t rb = buf_rsrc(
          g == 0 ? (kseg ? p.kseg[0].B + (int64_t)n0 * p.kseg[0].ldb : p.B + (int64_t)n0 * p.ldb)
                 : g == 1 ? p.kseg[1].B + (int64_t)n0 * kldb1 : p.kseg[2].B + (int64_t)n0 * kldb2);
      const int64_t ldb = g == 1 ? kldb1 : kldb2;
      const uint32_t boff = (uint32_t)(kg - (g == 0 ? 0 : g == 1 ? kk1 : kk2)) * 2u;
#pragma unroll
      for (int it = 0; it < B_ITEMS; ++it)
        rs[S][A_ITEMS + it] =
            buf_load4(rb, g == 0 ? b_off[it] : (uint32_t)(((int64_t)b_row[it] * ldb + b_kq[it]) * 2), boff);
    } else {
      const uint32_t boff = (uint32_t)((int64_t)kc * p.ldb * 2);
#pragma unroll
      for (int it = 0; it < B_ITEMS; ++it) rs[S][A_ITEMS + it] = buf_load4(rsb, b_off[it], boff);
    }
  };
  auto lstore = [&](auto sc, int stage) {
    constexpr int S = decltype(sc)::value;
    uint16_t* st = smem + stage * STAGE;
#pragma unroll
    for (int it = 0; it < A_ITEMS; ++it) {
      uint2 h, l;
      split2_f16(rs[S][it][0], rs[S][it][1], a_sc[it], h.x, l.x);
      split2_f16(rs[S][it][2], rs[S][it][3], a_sc[it], h.y, l.y);
      *reinterpret_cast<uint2*>(st + a_lds[it]) = h;
      *reinterpret_cast<uint2*>(st + A_PL + a_lds[it]) = l;
    }
#pragma unroll
    for (int it = 0; it < B_ITEMS; ++it) *reinterpret_cast<floatx4*>(st + b_lds[it]) = rs[S][A_ITEMS + it];
  };
  struct Frags {
    halfx8 h[TA], l[TA], b[TB];
  };
  auto read_frags = [&](Frags& f, int stage) {
    const uint16_t* st = smem + stage * STAGE;
#pragma unroll
    for (int a = 0; a < TA; ++a) {
      const int o = (wm + 16 * a + li) * PA + 8 * lg;
      f.h[a] = *reinterpret_cast<const halfx8*>(st + o);
      f.l[a] = *reinterpret_cast<const halfx8*>(st + A_PL + o);
    }
    const uint16_t* bs = st + 2 * A_PL;
    if constexpr (B_NK) {
#pragma unroll
      for (int b = 0; b < TB; ++b) f.b[b] = *reinterpret_cast<const halfx8*>(bs + (wn + 16 * b + li) * PA + 8 * lg);
    } else {
      const int r = 8 * lg + (li >> 2);
#pragma unroll
      for (int b = 0; b < TB; ++b) {
        const int c = wn + 16 * b + 4 * (li & 3);
        const shortx4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4*)(bs + r * PT + c));
        const shortx4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4*)(bs + (r + 4) * PT + c));
        f.b[b] = __builtin_bit_cast(halfx8, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
      }
    }
  };
  auto mfmas = [&](const Frags& f) {
#pragma unroll
    for (int a = 0; a < TA; ++a)
#pragma unroll
      for (int b = 0; b < TB; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f.h[a], f.b[b], acc[a][b], 0, 0, 0);
#pragma unroll
    for (int a = 0; a < TA; ++a)
#pragma unroll
      for (int b = 0; b < TB; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f.l[a], f.b[b], acc[a][b], 0, 0, 0);
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;

  constexpr int N_RD = 2 * TA + (B_NK ? TB : 2 * TB);  // LDS read instructions per read_frags
  constexpr int N_MF = 2 * TA * TB;                     // MFMAs per step
  Frags F[PIPE];                                        // entry e's fragments in F[e % PIPE]
  int s_nxt = 1, s_st = 2;  // stages of entries j+1, j+2 (wave-uniform); entry j sits in the third
  // Step j (fc = j % PIPE, sc = (j + 2) % PIPE): read entry j+1's fragments,
  // store entry j+2 (loaded PIPE steps ago) and load entry j+2+PIPE into its
  // register set, multiply entry j.
  auto step = [&](auto fc, auto sc, int j) {
    constexpr int FC = decltype(fc)::value;
    read_frags(F[(FC + 1) % PIPE], s_nxt);  // entry j+1, visible since the last barrier
    lstore(sc, s_st);
    gload(sc, j + 2 + PIPE);
    mfmas(F[FC]);
    __builtin_amdgcn_sched_group_barrier(0x100, N_RD, 0);
    if constexpr (N_MF >= N_WR + N_ST) {
#pragma unroll
      for (int i = 0; i < N_WR; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
      }
#pragma unroll
      for (int i = 0; i < N_ST; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, N_MF - N_WR - N_ST, 0);
    } else {
      __builtin_amdgcn_sched_group_barrier(0x200, N_WR, 0);
      __builtin_amdgcn_sched_group_barrier(0x020, N_ST, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, N_MF, 0);
    }
    __syncthreads();
    const int t = s_nxt;  // the stage of entry j (just multiplied) takes entry j+3
    s_nxt = s_st;
    s_st = (t + 2) % 3;
  };
  // Prologue: entries 0 .. PIPE-1 into their sets, entries 0 and 1 stored
  // (zero stages for leading pad entries), then entries PIPE, PIPE+1.
  auto zero_stage = [&](int stage) {
    for (int i = tid; i < STAGE / 8; i += 256)
      reinterpret_cast<floatx4*>(smem + stage * STAGE)[i] = floatx4{0.f, 0.f, 0.f, 0.f};
  };
  gload(I0{}, 0);
  gload(I1{}, 1);
  if constexpr (PIPE == 3) gload(I2{}, 2);
  if (pad > 0) zero_stage(0);
  else lstore(I0{}, 0);
  if (pad > 1) zero_stage(1);
  else lstore(I1{}, 1);
  gload(I0{}, PIPE);
  gload(I1{}, PIPE + 1);
  __syncthreads();
  read_frags(F[0], 0);
  if constexpr (PIPE == 2) {
    for (int j = 0; j < T; j += 2) {
      step(I0{}, I0{}, j);
      step(I1{}, I1{}, j + 1);
    }
  } else {
    for (int j = 0; j < T; j += 3) {
      step(I0{}, I2{}, j);
      step(I1{}, I0{}, j + 1);
      step(I2{}, I1{}, j + 2);
    }
  }

  // undo the row scale
  if (p.inv_s) {
#pragma unroll
    for (int a = 0; a < TA; ++a)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float f = row_isc(min(m0 + wm + 16 * a + 4 * lg + v, p.M - 1));
#pragma unroll
        for (int b = 0; b < TB; ++b) acc[a][b][v] *= f;
      }
  }

  // Rank-r LoRA term in fp32 (v_mfma_f32_16x16x4_f32), split 0 only, staged
  // in the ring's LDS after the last step's barrier.
  if (RANK && split == 0) {
    // with K segments the panels of the segments side by side: rank index
    // j = g·r + jj takes segment g's P[m][jj] and Q(n, jj)
    const int r = p.ep.r, rt = kseg ? p.nkseg * r : r, rp = (rt + 3) & ~3, pr = rp + 1;
    const float *kP0 = p.kseg[0].P, *kP1 = p.kseg[1].P, *kP2 = p.kseg[2].P;
    const float *kQ0 = p.kseg[0].Q, *kQ1 = p.kseg[1].Q, *kQ2 = p.kseg[2].Q;
    float* Ps = reinterpret_cast<float*>(smem);
    float* Qs = Ps + BM * pr;
    for (int i = tid; i < BM * rp; i += 256) {
      const int row = i / rp, j = i % rp, m = m0 + row;
      const int g = j / r, jj = j % r;
      const float* P = !kseg ? p.ep.P : g == 0 ? kP0 : g == 1 ? kP1 : kP2;
      Ps[row * pr + j] = (m < p.M && j < rt) ? P[(int64_t)m * r + jj] : 0.f;
    }
    for (int i = tid; i < BN * rp; i += 256) {
      const int col = i / rp, j = i % rp, n = n0 + col;
      const int g = j / r, jj = j % r;
      const float* Q = !kseg ? p.ep.Q : g == 0 ? kQ0 : g == 1 ? kQ1 : kQ2;
      Qs[col * pr + j] = (n < p.N && j < rt) ? p.ep.lscale * Q[(int64_t)n * p.ep.qsn + (int64_t)jj * p.ep.qsj] : 0.f;
    }
    __syncthreads();
    for (int t = 0; t < rp / 4; ++t) {
      float fp[TA], fq[TB];
#pragma unroll
      for (int a = 0; a < TA; ++a) fp[a] = Ps[(wm + 16 * a + li) * pr + 4 * t + lg];
#pragma unroll
      for (int b = 0; b < TB; ++b) fq[b] = Qs[(wn + 16 * b + li) * pr + 4 * t + lg];
#pragma unroll
      for (int a = 0; a < TA; ++a)
#pragma unroll
        for (int b = 0; b < TB; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(fp[a], fq[b], acc[a][b], 0, 0, 0);
    }
  }

  tile_out<BM, BN, 3 * STAGE * 2>(p, reinterpret_cast<float*>(smem), m0, n0, split, [&](auto&& put) {
#pragma unroll
    for (int a = 0; a < TA; ++a)
#pragma unroll
      for (int b = 0; b < TB; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v) put(wm + 16 * a + 4 * lg + v, wn + 16 * b + li, acc[a][b][v]);
  });
}

}  // namespace
thread_local const KernelEvents* t_gemm_events = nullptr;
thread_local hipEvent_t t_tail_start = nullptr, t_tail_stop = nullptr;
namespace {

// The timing events of the launches in a scope; none are left behind by one that throws.
struct GemmEventScope {
  explicit GemmEventScope(const KernelEvents* ev) { t_gemm_events = ev; }
  ~GemmEventScope() { t_gemm_events = nullptr; }
};

// After the main launch: the split-K reduction with the epilogue (and the
// row norm, fused into it where splitk_norm can), or the row norm alone.
void gemm_finish(hipStream_t s, int splits, bool dispatch_events, const KernelEvents* ev, const float* partial,
                 int M, int N, float* C, int64_t ldc, const GemmEpilogue& ep, const RowNorm* nm) {
  MFT_CHECK_ARG(!nm || ldc == N, "a row norm needs ldc == N");
  if (splits > 1) {
    // The split-K reduction (with the epilogue and, when fused, the row
    // norm) belongs to the GEMM's time: bracket it with the tail events.
    const bool tail = ev && ev->tail_start && ev->tail_stop;
    if (tail) {
      ev->tail_used = true;
      if (dispatch_events) {
        t_tail_start = ev->tail_start;
        t_tail_stop = ev->tail_stop;
      } else {
        MFT_HIP(hipEventRecord(ev->tail_start, s));
      }
    }
    struct TailReset {
      ~TailReset() { t_tail_start = t_tail_stop = nullptr; }
    } tail_reset;
    const bool fused = nm && splitk_norm(s, partial, splits, M, N, C, ldc, ep, *nm);
    if (!fused) {
      MFT_LAUNCH_TAIL(splitk_reduce_kernel, dim3((unsigned)cdiv(N, 1024), (unsigned)std::min(M, 65535)), dim3(256),
                      0, s, partial, splits, M, N, C, ldc, ep);
    }
    t_tail_start = t_tail_stop = nullptr;
    if (tail && !dispatch_events) MFT_HIP(hipEventRecord(ev->tail_stop, s));
    MFT_LAUNCH_CHECK();
    if (!fused && nm) row_norm(s, C, M, N, *nm);
  } else if (nm) {
    row_norm(s, C, M, N, *nm);
  }
}


// ---- small fp32 GEMM launch ----
template <bool B_NK, bool B_F16, bool TAIL>
void launch_s_rank(hipStream_t s, const GemmParams& p, dim3 grid) {
  if (p.ep.P != nullptr) launch_gemm_kernel(gemm_s_kernel<B_NK, B_F16, true, TAIL>, grid, dim3(256), s, p);
  else launch_gemm_kernel(gemm_s_kernel<B_NK, B_F16, false, TAIL>, grid, dim3(256), s, p);
}
}  // namespace
void gemm_s_launch(hipStream_t s, const GemmParams& p, dim3 grid, bool b_nk, bool b_f16) {
  if (b_f16) {
    if (b_nk) launch_s_rank<true, true, true>(s, p, grid);
    else launch_s_rank<false, true, true>(s, p, grid);
  } else if (p.K % 32 == 0) {
    if (b_nk) launch_s_rank<true, false, false>(s, p, grid);
    else launch_s_rank<false, false, false>(s, p, grid);
  } else {
    if (b_nk) launch_s_rank<true, false, true>(s, p, grid);
    else launch_s_rank<false, false, true>(s, p, grid);
  }
  MFT_LAUNCH_CHECK();
}
namespace {

// ---- fp16 matrix-core GEMM launch ----
dim3 xcd_grid(GemmHParams& p, int splits) {
  static const int spread = [] {  // tuning hook: MFT_GEMM_SPREAD=1 spreads every K-slice over all XCDs
    const char* e = getenv("MFT_GEMM_SPREAD");
    return e ? atoi(e) : 0;
  }();
  const int tiles = p.tiles_m * p.tiles_n;
  p.splits = splits;
  // up to eight slices have XCDs of their own (1024×1152×6912 60 µs, spread
  // 65; the other fp16 layer shapes level); beyond there is none left for each
  p.spread = spread || splits > 8;
  if (p.spread) {
    p.tiles_per_xcd = (int)cdiv(tiles, 8);
    return dim3((unsigned)(p.tiles_per_xcd * 8 * splits), 1);
  }
  p.tiles_per_xcd = (int)cdiv(tiles, 8 / splits);
  return dim3((unsigned)(p.tiles_per_xcd * 8), 1);
}
template <int BM, int BN, bool RANK>
void launch_h_rank(hipStream_t s, GemmHParams& p, bool b_nk, int splits) {
  p.tiles_m = (int)cdiv(p.M, BM);
  p.tiles_n = (int)cdiv(p.N, BN);
  const dim3 grid = xcd_grid(p, splits), block(256);
  if (p.nseg <= 1) p.out_vec = out_vec(p);  // gemm_h_segments looks at every segment
  static const int pipe = [] {  // tuning hook: MFT_GEMMH_PIPE = 2 or 3 register staging sets
    const char* e = getenv("MFT_GEMMH_PIPE");
    return e && atoi(e) == 2 ? 2 : 3;
  }();
  if (pipe == 3) {
    if (b_nk) launch_gemm_kernel(gemm_h_kernel<BM, BN, true, RANK, 3>, grid, block, s, p);
    else launch_gemm_kernel(gemm_h_kernel<BM, BN, false, RANK, 3>, grid, block, s, p);
  } else {
    if (b_nk) launch_gemm_kernel(gemm_h_kernel<BM, BN, true, RANK, 2>, grid, block, s, p);
    else launch_gemm_kernel(gemm_h_kernel<BM, BN, false, RANK, 2>, grid, block, s, p);
  }
  MFT_LAUNCH_CHECK();
}
template <int BM, int BN>
void launch_h(hipStream_t s, GemmHParams& p, bool b_nk, int splits) {
  if (p.ep.P != nullptr) launch_h_rank<BM, BN, true>(s, p, b_nk, splits);
  else launch_h_rank<BM, BN, false>(s, p, b_nk, splits);
}

// Tile shape and split-K of the fp16 GEMM.  A panel step's time is the
// larger of a per-shape latency floor and the step's operand bytes (fp32 A,
// fp16 B) times the workgroups resident at once over an effective L2 rate;
// a launch runs ceil(workgroups / capacity) rounds of k_chunk/32 steps
// (capacity = 256 CUs × 1, 2 or 3 workgroups of the 128×128, 64×128 and
// 64×64 tiles, from their LDS rings), plus 5 µs per launch and, split, 2 µs
// plus the partials at 3 MB/µs.  Fitted to MI355X sweeps of the Gemma-3 1B
// linear shapes (M = 1024, 18 plans each), it picks within 6% of the best
// measured plan in total; K-slices deeper than 1024 measured slower than
// the model says (the fp32 A rows of a deep slice fall out of L2), so deep
// reductions split until a slice is at most 1024 deep.
struct PlanH {
  int bm, bn, splits;
};
PlanH plan_gemm_h(int M, int N, int K, size_t ws_bytes, bool stats) {
  struct Shape {
    int bm, bn, occ;
    double lat_us;
  };
  static const Shape shapes[] = {{128, 128, 1, 1.0}, {64, 128, 2, 0.4}, {64, 64, 3, 0.3}};
  PlanH best{64, 64, 1};
  double best_t = 1e30;
  for (const Shape& sh : shapes) {
    if (stats && sh.bn != 128) continue;  // row statistics: 64-column blocks per wave, unsplit K
    const int64_t tiles = cdiv(M, sh.bm) * cdiv(N, sh.bn);
    for (int sp : {1, 2, 3, 4, 6, 8, 16, 32}) {
      const int64_t kc = cdiv(cdiv(K, sp), 32) * 32;
      if (cdiv(K, kc) != sp) continue;
      if (stats && sp > 1) continue;
      if (sp > 1 && (kc < 128 || (size_t)sp * M * N * sizeof(float) > ws_bytes)) continue;
      if (K >= 4096 && kc > 1024 && sp < 8) continue;
      const int64_t wgs = tiles * sp, cap = 256 * sh.occ;
      const double conc = (double)std::min<int64_t>(wgs, cap);
      const double step_bytes = sh.bm * 32.0 * 4 + sh.bn * 32.0 * 2;
      const double tau = std::max(sh.lat_us, conc * step_bytes / 11e6);  // µs per panel step
      double t = 5.0 + (double)cdiv(wgs, cap) * (double)(kc / 32) * tau;
      if (sp > 1) t += 2.0 + sp * (double)M * N * 8 / 3e6;
      if (t < best_t) {
        best_t = t;
        best = {sh.bm, sh.bn, sp};
      }
    }
  }
  return best;
}
}  // namespace

// Tuning hooks MFT_GEMM_PLAN / MFT_GEMMH_PLAN: "bm,bn,splits" forces every
// launch; "M,N,K:bm,bn,splits;..." forces the listed shapes only.  Returns
// false when the variable forces nothing for this shape.
static bool forced_plan(const char* env, int M, int N, int K, int& bm, int& bn, int& sp) {
  if (!env) return false;
  if (!strchr(env, ':')) return sscanf(env, "%d,%d,%d", &bm, &bn, &sp) == 3;
  for (const char* e = env; e && *e; e = strchr(e, ';') ? strchr(e, ';') + 1 : nullptr) {
    int m = 0, n = 0, k = 0;
    if (sscanf(e, "%d,%d,%d:%d,%d,%d", &m, &n, &k, &bm, &bn, &sp) == 6 && m == M && n == N && k == K) return true;
  }
  return false;
}

void gemm(hipStream_t s, const float* A, int64_t lda, const void* B, int64_t ldb, bool b_nk,
          bool b_f16, float* C, int64_t ldc, int M, int N, int K, const GemmEpilogue& ep,
          Scratch ws, const KernelEvents* ev) {
  MFT_CHECK_ARG(M > 0 && N > 0 && K > 0, "empty GEMM");
  MFT_CHECK_ARG(lda % 4 == 0 && lda >= K, "lda must be a multiple of 4 and >= K");
  MFT_CHECK_ARG(!b_nk || ldb >= K, "ldb must be >= K for [N,K] B");
  MFT_CHECK_ARG(b_nk || ldb >= N, "ldb must be >= N for [K,N] B");
  MFT_CHECK_ARG(ldc >= N, "ldc must be >= N");
  MFT_CHECK_ARG(ep.r <= 32, "LoRA rank > 32 unsupported");
  MFT_CHECK_ARG(((uintptr_t)A & 15) == 0, "A must be 16-byte aligned");
  GemmParams p{};
  p.A = A; p.B = B; p.C = C;
  p.lda = lda; p.ldb = ldb; p.ldc = ldc;
  p.M = M; p.N = N; p.K = K;
  p.ep = ep;
  if (ldb % 4 != 0 || ((uintptr_t)B & (b_f16 ? 7 : 15)) != 0) {
    // The kernel reads B as aligned 4-vectors; repack an unaligned or
    // odd-pitch B into the workspace with a padded pitch first.
    const size_t esz = b_f16 ? 2 : 4;
    const int64_t rows = b_nk ? N : K, cols = b_nk ? K : N;
    const int64_t pitch = (cols + 3) / 4 * 4;
    const size_t need = (size_t)rows * pitch * esz;
    MFT_CHECK_ARG(ws.ptr && ws.bytes >= need + 256, "unaligned B needs a workspace for repacking");
    char* dst = reinterpret_cast<char*>(ws.ptr);
    MFT_HIP(hipMemcpy2DAsync(dst, pitch * esz, B, ldb * esz, cols * esz, rows, hipMemcpyDeviceToDevice, s));
    p.B = dst;
    p.ldb = pitch;
    const size_t used = (need + 255) / 256 * 256;
    ws.ptr = reinterpret_cast<float*>(dst + used);
    ws.bytes -= used;
  }
  MFT_CHECK_ARG(!ep.stats || (ep.stats_ld >= cdiv(N, 64) && !ep.bias && !ep.resid && ep.beta == 0.f && !ep.gelu_out &&
                              !ep.gelu_grad_of && !ep.P && !(ep.norm && ep.norm->kind != NORM_NONE)),
                "row statistics describe plain logits (no epilogue terms)");
  // a tile's K-slice is addressed through 32-bit buffer offsets from the
  // tile's first row / column: the deepest slice they reach in both operands
  const int64_t reach = (int64_t(1) << 32) / (b_f16 ? 2 : 4) - 1;
  const int64_t k_max =
      std::min((int64_t(1) << 30) - 1 - 128 * lda, b_nk ? reach - 128 * p.ldb : (reach - 128) / p.ldb);

  const RowNorm* nm = ep.norm && ep.norm->kind != NORM_NONE ? ep.norm : nullptr;
  const size_t skew = ws.ptr ? (16 - ((uintptr_t)ws.ptr & 15)) & 15 : 0;  // partials are moved 16 bytes at a time
  float* wsp = ws.ptr ? reinterpret_cast<float*>(reinterpret_cast<char*>(ws.ptr) + skew) : nullptr;
  const size_t ws_bytes = ws.ptr && ws.bytes > skew ? ws.bytes - skew : 0;
  XPlan pl = plan_gemm_x(M, N, K, k_max, ws_bytes, nm != nullptr && N % 4 == 0 && N <= 4096 && ldc == N,
                         ep.stats != nullptr, ep.small_tiles, b_f16 || K % 32 != 0);
  // Tuning hook: MFT_GEMM_PLAN="bm,bn,splits" (or per shape, "M,N,K:bm,bn,splits;...") forces tiles and a uniform split.
  static const char* forced_env = getenv("MFT_GEMM_PLAN");
  int bm = 0, bn = 0, sp = 0;
  if (!ep.stats && !b_f16 && forced_plan(forced_env, M, N, K, bm, bn, sp) &&
      ((bm == 32 && bn == 64) || (bm == 64 && bn == 64) || (bm == 64 && bn == 128) || (bm == 128 && bn == 128)) &&
      sp >= 1 && (sp == 1 || (size_t)sp * M * N * sizeof(float) <= ws_bytes))
    pl = {bm, bn, sp, (int)(cdiv(M, bm) * cdiv(N, bn)), 0};
  MFT_CHECK_ARG(!ep.stats || (pl.bn == 128 && pl.splits == 1 && pl.tail_splits <= 1),
                "row statistics need whole 128-wide tiles");
  MFT_CHECK_ARG(gemm_x_depth(pl, p) <= k_max, "GEMM operand too large for 32-bit buffer offsets");
  static const bool log_plans = getenv("MFT_GEMM_PLAN_LOG") != nullptr;  // tuning hook: print each launch's plan
  if (log_plans)
    fprintf(stderr, "gemm %d,%d,%d:%d,%d,%d full=%d tail=%d norm=%d\n", M, N, K, pl.bm, pl.bn, pl.splits, pl.full,
            pl.tail_splits, nm ? 1 : 0);

  // Timing: events recorded by the dispatch itself, except under stream
  // capture, where they are separate event records around the launch.
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (ev) MFT_HIP(hipStreamIsCapturing(s, &cap));
  const bool dispatch_events = ev && ev->start && ev->stop && cap == hipStreamCaptureStatusNone;
  if (ev && ev->start && !dispatch_events) MFT_HIP(hipEventRecord(ev->start, s));
  KernelEvents tev;
  if (dispatch_events && pl.tail_splits > 1 && ev->tail_start && ev->tail_stop) {
    ev->tail_used = true;  // the sums of the split tiles
    tev.start = ev->tail_start;
    tev.stop = ev->tail_stop;
  }
  {
    const GemmEventScope scope(dispatch_events ? ev : nullptr);
    gemm_x_launch(s, p, pl, b_nk, b_f16, wsp, tev.start ? &tev : nullptr);
  }
  if (ev && ev->stop && !dispatch_events) MFT_HIP(hipEventRecord(ev->stop, s));

  gemm_finish(s, p.partial ? p.tail_splits : 1, dispatch_events, ev, wsp, M, N, C, ldc, ep, nm);
}

void row_scales(hipStream_t s, const float* x, int64_t ldx, int M, int K, float* inv_s) {
  MFT_CHECK_ARG(M > 0 && K > 0 && K % 4 == 0 && ldx % 4 == 0 && ((uintptr_t)x & 15) == 0, "row_scales shape");
  hipLaunchKernelGGL(row_scale_kernel, dim3((unsigned)M), dim3(256), 0, s, x, ldx, K, inv_s);
  MFT_LAUNCH_CHECK();
}

bool gemm_h_ok(int N, int K, bool b_nk, int r) { return K % 32 == 0 && (b_nk || N % 8 == 0) && r <= 32; }

void gemm_h(hipStream_t s, const float* A, int64_t lda, const float* inv_s, const uint16_t* B, int64_t ldb, bool b_nk,
            float* C, int64_t ldc, int M, int N, int K, const GemmEpilogue& ep, Scratch ws, const KernelEvents* ev) {
  MFT_CHECK_ARG(M > 0 && N > 0 && K > 0, "empty GEMM");
  MFT_CHECK_ARG(gemm_h_ok(N, K, b_nk, ep.r), "fp16 GEMM takes K % 32 == 0, N % 8 == 0 for [K,N] B, r <= 32");
  MFT_CHECK_ARG(A && lda >= K && lda % 4 == 0, "lda must be a multiple of 4 and >= K");
  MFT_CHECK_ARG(b_nk ? ldb >= K : ldb >= N, "ldb too small");
  MFT_CHECK_ARG(ldb % 8 == 0, "ldb must be a multiple of 8");
  MFT_CHECK_ARG(ldc >= N, "ldc must be >= N");
  MFT_CHECK_ARG((((uintptr_t)A | (uintptr_t)B) & 15) == 0, "GEMM operands must be 16-byte aligned");
  MFT_CHECK_ARG(!ep.stats || (ep.stats_ld >= cdiv(N, 64) && !ep.bias && !ep.resid && ep.beta == 0.f && !ep.gelu_out &&
                              !ep.gelu_grad_of && !ep.P && !(ep.norm && ep.norm->kind != NORM_NONE)),
                "row statistics describe plain logits (no epilogue terms)");
  GemmHParams p{};
  p.A = A; p.inv_s = inv_s; p.B = B; p.C = C;
  p.lda = lda; p.ldb = ldb; p.ldc = ldc;
  p.M = M; p.N = N; p.K = K;
  p.ep = ep;
  p.partial = nullptr;
  PlanH pl = plan_gemm_h(M, N, K, ws.ptr ? ws.bytes : 0, ep.stats != nullptr);
  // Tuning hook: MFT_GEMMH_PLAN="bm,bn,splits" (or per shape, "M,N,K:bm,bn,splits;...") forces the launch shape.
  static const char* forced_env = getenv("MFT_GEMMH_PLAN");
  int bm = 0, bn = 0, sp = 0;
  const bool forced = forced_plan(forced_env, M, N, K, bm, bn, sp);
  if (forced && !ep.stats) {
    if (sp >= 1 && sp <= 64 &&
        ((bm == 128 && bn == 128) || (bm == 64 && bn == 128) || (bm == 64 && bn == 64)) &&
        (sp == 1 || (size_t)sp * M * N * sizeof(float) <= ws.bytes))
      pl = {bm, bn, sp};
  }
  const RowNorm* nm = ep.norm && ep.norm->kind != NORM_NONE ? ep.norm : nullptr;
  // as in gemm(): a row norm rides in the split-K reduction for free
  if (nm && !forced && !ep.stats && pl.splits == 1 && K >= 512 && N % 4 == 0 && N <= 4096 && ldc == N &&
      (size_t)2 * M * N * sizeof(float) <= ws.bytes)
    pl.splits = 2;
  int splits = pl.splits;
  p.k_chunk = (int)(cdiv(cdiv(K, splits), 32) * 32);
  splits = (int)cdiv(K, p.k_chunk);
  static const bool log_plans = getenv("MFT_GEMM_PLAN_LOG") != nullptr;
  if (log_plans) fprintf(stderr, "gemm_h %d,%d,%d:%d,%d,%d norm=%d\n", M, N, K, pl.bm, pl.bn, splits, nm ? 1 : 0);
  MFT_CHECK_ARG(((int64_t)pl.bm * p.lda + p.k_chunk) * 4 < (int64_t(1) << 32) &&
                    (b_nk ? (int64_t)pl.bn * p.ldb + p.k_chunk : (int64_t)p.k_chunk * p.ldb + pl.bn) * 2 <
                        (int64_t(1) << 32),
                "GEMM operand too large for 32-bit buffer offsets");
  if (splits > 1) p.partial = ws.ptr;

  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (ev) MFT_HIP(hipStreamIsCapturing(s, &cap));
  const bool dispatch_events = ev && ev->start && ev->stop && cap == hipStreamCaptureStatusNone;
  if (ev && ev->start && !dispatch_events) MFT_HIP(hipEventRecord(ev->start, s));
  {
    const GemmEventScope scope(dispatch_events ? ev : nullptr);
    if (pl.bm == 128) launch_h<128, 128>(s, p, b_nk, splits);
    else if (pl.bn == 128) launch_h<64, 128>(s, p, b_nk, splits);
    else launch_h<64, 64>(s, p, b_nk, splits);
  }
  if (ev && ev->stop && !dispatch_events) MFT_HIP(hipEventRecord(ev->stop, s));
  gemm_finish(s, splits, dispatch_events, ev, ws.ptr, M, N, C, ldc, ep, nm);
}

bool segments_out_vec(const GemmHSegmentArg* seg, int nseg) {
  bool vec = true;
  for (int g = 0; g < nseg; ++g) vec = vec && seg[g].ldc % 4 == 0 && ((uintptr_t)seg[g].C & 15) == 0;
  return vec;
}

bool gemm_h_segments(hipStream_t s, const float* A, int64_t lda, const float* inv_s, bool b_nk,
                     const GemmHSegmentArg* seg, int nseg, int M, int K, const GemmEpilogue& ep,
                     const KernelEvents* ev) {
  MFT_CHECK_ARG(seg && nseg >= 2 && nseg <= kMaxGemmHSegments && M > 0 && K > 0, "segmented GEMM: 2 or 3 segments");
  MFT_CHECK_ARG(A && lda >= K && lda % 4 == 0 && ((uintptr_t)A & 15) == 0, "segmented GEMM: A");
  MFT_CHECK_ARG(!ep.bias && !ep.resid && ep.beta == 0.f && !ep.gelu_out && !ep.gelu_grad_of && !ep.stats &&
                    !(ep.norm && ep.norm->kind != NORM_NONE),
                "segmented GEMM: plain outputs plus the rank-r panel only");
  int N = 0;
  bool all64 = true, all128 = true;
  for (int g = 0; g < nseg; ++g) {
    const GemmHSegmentArg& a = seg[g];
    MFT_CHECK_ARG(a.B && a.C && a.N > 0 && gemm_h_ok(a.N, K, b_nk, ep.r) && a.ldb % 8 == 0 &&
                      (b_nk ? a.ldb >= K : a.ldb >= a.N) && a.ldc >= a.N && ((uintptr_t)a.B & 15) == 0,
                  "segmented GEMM: segment shape");
    MFT_CHECK_ARG((ep.r > 0) == (a.P != nullptr && a.Q != nullptr), "segmented GEMM: rank panel per segment");
    all64 = all64 && a.N % 64 == 0;
    all128 = all128 && a.N % 128 == 0;
    N += a.N;
  }
  PlanH pl = plan_gemm_h(M, N, K, 0, false);  // no workspace: unsplit
  static const char* forced_env = getenv("MFT_GEMMH_PLAN");
  int bm = 0, bn = 0, sp = 0;
  if (forced_plan(forced_env, M, N, K, bm, bn, sp) && sp == 1 &&
      ((bm == 128 && bn == 128) || (bm == 64 && bn == 128) || (bm == 64 && bn == 64)))
    pl = {bm, bn, 1};
  if (pl.bn == 128 && !all128) pl = {64, 64, 1};
  if (!all64) return false;
  GemmHParams p{};
  p.A = A; p.inv_s = inv_s; p.B = seg[0].B; p.C = seg[0].C;
  p.lda = lda; p.ldb = seg[0].ldb; p.ldc = seg[0].ldc;
  p.M = M; p.N = N; p.K = K;
  p.ep = ep;
  p.ep.P = seg[0].P;  // selects the rank-panel kernel; each tile takes its segment's panel
  p.ep.Q = seg[0].Q;
  p.partial = nullptr;
  p.k_chunk = K;
  p.nseg = nseg;
  p.out_vec = segments_out_vec(seg, nseg);
  for (int g = 0, n0 = 0; g < nseg; n0 += seg[g].N, ++g) {
    p.seg[g] = GemmHSegment{n0, seg[g].B, seg[g].ldb, seg[g].C, seg[g].ldc, seg[g].P, seg[g].Q};
    MFT_CHECK_ARG((b_nk ? (int64_t)pl.bn * seg[g].ldb + K : (int64_t)K * seg[g].ldb + pl.bn) * 2 < (int64_t(1) << 32),
                  "GEMM operand too large for 32-bit buffer offsets");
  }
  MFT_CHECK_ARG(((int64_t)pl.bm * lda + K) * 4 < (int64_t(1) << 32), "GEMM operand too large for 32-bit buffer offsets");
  static const bool log_plans = getenv("MFT_GEMM_PLAN_LOG") != nullptr;
  if (log_plans) fprintf(stderr, "gemm_h_seg %d,%d,%d:%d,%d,1 nseg=%d\n", M, N, K, pl.bm, pl.bn, nseg);
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (ev) MFT_HIP(hipStreamIsCapturing(s, &cap));
  const bool dispatch_events = ev && ev->start && ev->stop && cap == hipStreamCaptureStatusNone;
  if (ev && ev->start && !dispatch_events) MFT_HIP(hipEventRecord(ev->start, s));
  {
    const GemmEventScope scope(dispatch_events ? ev : nullptr);
    if (pl.bm == 128) launch_h<128, 128>(s, p, b_nk, 1);
    else if (pl.bn == 128) launch_h<64, 128>(s, p, b_nk, 1);
    else launch_h<64, 64>(s, p, b_nk, 1);
  }
  if (ev && ev->stop && !dispatch_events) MFT_HIP(hipEventRecord(ev->stop, s));
  return true;
}

void gemm_h_ksegments(hipStream_t s, const float* A, int64_t lda, const GemmHKSegmentArg* seg, int nseg, float* C,
                      int64_t ldc, int M, int N, const GemmEpilogue& ep, Scratch ws, const KernelEvents* ev) {
  MFT_CHECK_ARG(seg && nseg >= 2 && nseg <= kMaxGemmHSegments && M > 0 && N > 0, "K-segmented GEMM: 2 or 3 segments");
  MFT_CHECK_ARG(A && lda % 4 == 0 && ((uintptr_t)A & 15) == 0, "K-segmented GEMM: A");
  MFT_CHECK_ARG(ldc >= N && nseg * ep.r <= 32, "K-segmented GEMM: ldc or rank");
  MFT_CHECK_ARG(!ep.stats && !ep.gelu_out && !ep.gelu_grad_of, "K-segmented GEMM: no statistics or GELU terms");
  int K = 0;
  for (int g = 0; g < nseg; ++g) {
    const GemmHKSegmentArg& a = seg[g];
    MFT_CHECK_ARG(a.B && a.inv_s && a.K > 0 && a.K % 32 == 0 && a.ldb >= a.K && a.ldb % 8 == 0 &&
                      ((uintptr_t)a.B & 15) == 0,
                  "K-segmented GEMM: segment shape");
    MFT_CHECK_ARG((ep.r > 0) == (a.P != nullptr && a.Q != nullptr), "K-segmented GEMM: rank panel per segment");
    K += a.K;
  }
  MFT_CHECK_ARG(lda >= K, "K-segmented GEMM: lda < K");
  GemmHParams p{};
  p.A = A; p.inv_s = seg[0].inv_s; p.B = seg[0].B; p.C = C;
  p.lda = lda; p.ldb = seg[0].ldb; p.ldc = ldc;
  p.M = M; p.N = N; p.K = K;
  p.ep = ep;
  p.ep.P = seg[0].P;  // selects the rank-panel kernel; the panel reads every segment's P, Q
  p.ep.Q = seg[0].Q;
  p.partial = nullptr;
  p.nkseg = nseg;
  for (int g = 0, k0 = 0; g < nseg; k0 += seg[g].K, ++g)
    p.kseg[g] = GemmHKSegment{k0, seg[g].B, seg[g].ldb, seg[g].inv_s, seg[g].P, seg[g].Q};
  for (int g = nseg; g < kMaxGemmHSegments; ++g) p.kseg[g] = p.kseg[nseg - 1];  // never selected
  PlanH pl = plan_gemm_h(M, N, K, ws.ptr ? ws.bytes : 0, false);
  static const char* forced_env = getenv("MFT_GEMMH_PLAN");
  int bm = 0, bn = 0, sp = 0;
  const bool forced = forced_plan(forced_env, M, N, K, bm, bn, sp);
  if (forced && sp >= 1 && sp <= 64 && ((bm == 128 && bn == 128) || (bm == 64 && bn == 128) || (bm == 64 && bn == 64)) &&
      (sp == 1 || (size_t)sp * M * N * sizeof(float) <= ws.bytes))
    pl = {bm, bn, sp};
  const RowNorm* nm = ep.norm && ep.norm->kind != NORM_NONE ? ep.norm : nullptr;
  if (nm && !forced && pl.splits == 1 && K >= 512 && N % 4 == 0 && N <= 4096 && ldc == N &&
      (size_t)2 * M * N * sizeof(float) <= ws.bytes)
    pl.splits = 2;  // a row norm rides in the split-K reduction
  p.k_chunk = (int)(cdiv(cdiv(K, pl.splits), 32) * 32);
  const int splits = (int)cdiv(K, p.k_chunk);
  for (int g = 0; g < nseg; ++g)
    MFT_CHECK_ARG(((int64_t)pl.bn * seg[g].ldb + seg[g].K) * 2 < (int64_t(1) << 32),
                  "GEMM operand too large for 32-bit buffer offsets");
  MFT_CHECK_ARG(((int64_t)pl.bm * lda + p.k_chunk) * 4 < (int64_t(1) << 32), "GEMM operand too large for 32-bit buffer offsets");
  if (splits > 1) p.partial = ws.ptr;
  static const bool log_plans = getenv("MFT_GEMM_PLAN_LOG") != nullptr;
  if (log_plans) fprintf(stderr, "gemm_h_kseg %d,%d,%d:%d,%d,%d nseg=%d norm=%d\n", M, N, K, pl.bm, pl.bn, splits, nseg, nm ? 1 : 0);
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (ev) MFT_HIP(hipStreamIsCapturing(s, &cap));
  const bool dispatch_events = ev && ev->start && ev->stop && cap == hipStreamCaptureStatusNone;
  if (ev && ev->start && !dispatch_events) MFT_HIP(hipEventRecord(ev->start, s));
  {
    const GemmEventScope scope(dispatch_events ? ev : nullptr);
    if (pl.bm == 128) launch_h<128, 128>(s, p, true, splits);
    else if (pl.bn == 128) launch_h<64, 128>(s, p, true, splits);
    else launch_h<64, 64>(s, p, true, splits);
  }
  if (ev && ev->stop && !dispatch_events) MFT_HIP(hipEventRecord(ev->stop, s));
  gemm_finish(s, splits, dispatch_events, ev, ws.ptr, M, N, C, ldc, ep, nm);
}

bool gemm_f16w(hipStream_t s, const float* x, int64_t ldx, const void* W, int64_t ldw, bool b_nk, float* C,
               int64_t ldc, int M, int N, int K, const GemmEpilogue& ep, Scratch ws, const KernelEvents* ev) {
  static const int mode = [] {  // tuning hook: MFT_GEMM_F16=0 keeps fp16 W on the fp32 kernels
    const char* e = getenv("MFT_GEMM_F16");
    return e ? atoi(e) : 1;
  }();
  if (!mode || ep.stats || !gemm_h_ok(N, K, b_nk, ep.r) || ldx % 4 != 0 || ldx < K || ((uintptr_t)x & 15) != 0 ||
      ldw % 8 != 0 || ((uintptr_t)W & 15) != 0)
    return false;
  const size_t need = ((size_t)M * sizeof(float) + 255) / 256 * 256;
  const size_t pad = ws.ptr ? (256 - ((uintptr_t)ws.ptr & 255)) & 255 : 0;
  if (!ws.ptr || ws.bytes < need + pad) return false;
  char* base = reinterpret_cast<char*>(ws.ptr) + pad;
  float* inv_s = reinterpret_cast<float*>(base);
  row_scales(s, x, ldx, M, K, inv_s);
  Scratch rest;
  rest.ptr = reinterpret_cast<float*>(base + need);
  rest.bytes = ws.bytes - need - pad;
  gemm_h(s, x, ldx, inv_s, static_cast<const uint16_t*>(W), ldw, b_nk, C, ldc, M, N, K, ep, rest, ev);
  return true;
}

}  // namespace mft
