// gemm_common.h — what the GEMM kernels share: parameters, tile order, epilogue,
// softmax row statistics, launch with timing events.
#ifndef MFT_GEMM_COMMON_H
#define MFT_GEMM_COMMON_H
#include <cfloat>
#include <type_traits>

#include <hip/hip_ext.h>

#include "common.h"

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef short shortx4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) shortx4 lds_shortx4;

namespace mft {

struct GemmParams {
  const float* A;
  const void* B;
  float* C;
  int64_t lda, ldb, ldc;
  int M, N, K;
  int tiles_m, tiles_n;
  // The first full_tiles tiles take the whole K; the others are cut into
  // tail_splits slices of k_chunk, whose raw sums go to partial
  // ([slice][M][N]) or, if that is null, tile by tile to
  // tail_out[tile − full_tiles][slice][BM][BN].
  int full_tiles, tail_splits, k_chunk;
  int full_per_xcd, tail_per_xcd;  // workgroups of either kind per XCD
  float* partial;
  float* tail_out;
  int out_vec;  // output rows allow 128-bit stores (tile_out)
  GemmEpilogue ep;
};

constexpr float kLog2eG = 1.4426950408889634f;

// Softmax statistics of one logits row segment of 64 values held in LDS
// (row-major, 16-byte aligned): (max t, Σ 2^(t − max)) with t = value·log2e.
// Entries past the matrix edge hold −FLT_MAX (their terms flush to 0; the
// first entry is always inside).  The max runs over the raw values (scaling
// by log2e is monotonic) as IEEE maximum, which needs no canonicalised
// operands.
__device__ __forceinline__ float2 row_stats64(const float* row) {
  const float4* r4 = reinterpret_cast<const float4*>(row);
  float v[64];
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const float4 t = r4[q];
    v[4 * q] = t.x;
    v[4 * q + 1] = t.y;
    v[4 * q + 2] = t.z;
    v[4 * q + 3] = t.w;
  }
  float mx = v[0];
#pragma unroll
  for (int c = 1; c + 1 < 64; c += 2) mx = __builtin_elementwise_maximum(mx, __builtin_elementwise_maximum(v[c], v[c + 1]));
  mx = __builtin_elementwise_maximum(mx, v[63]);
  const float ml = mx * kLog2eG;
  float s0 = 0.f, s1 = 0.f;
#pragma unroll
  for (int c = 0; c < 64; c += 2) {
    s0 += __builtin_amdgcn_exp2f(fmaf(v[c], kLog2eG, -ml));
    s1 += __builtin_amdgcn_exp2f(fmaf(v[c + 1], kLog2eG, -ml));
  }
  return make_float2(ml, s0 + s1);
}

// Workgroup → (tile, K-slice) of a GemmParams launch, and where a split
// tile's raw sums go (null: the whole output or [slice][M][N] partials).
// Workgroup L runs on XCD L % 8, each with its own L2: the whole tiles first,
// contiguous runs of them (M-fastest) to an XCD, so that it reads whole column
// bands of B; then the slices of the others, the slices of one K range
// together, so that an XCD reads the A rows of few slices.
template <int BM, int BN>
__device__ __forceinline__ bool tile_slice(const GemmParams& p, int& tile, int& split, float*& raw_tile) {
  const int xcd = blockIdx.x % 8, idx = blockIdx.x / 8, rem = p.tiles_m * p.tiles_n - p.full_tiles;
  raw_tile = nullptr;
  split = 0;
  if (idx < p.full_per_xcd) {
    tile = xcd * p.full_per_xcd + idx;
    return tile < p.full_tiles;
  }
  const int u = xcd * p.tail_per_xcd + idx - p.full_per_xcd;
  if (u >= rem * p.tail_splits) return false;
  split = u / rem;
  tile = p.full_tiles + u % rem;
  if (!p.partial) raw_tile = p.tail_out + ((int64_t)(u % rem) * p.tail_splits + split) * (min(BM, p.M) * BN);
  return true;
}

// Bias, residual and β·C; the rank-r term is accumulated on the matrix
// cores before the epilogue.
__device__ __forceinline__ float epilogue_value(const GemmEpilogue& ep, float acc, int m, int n,
                                                const float* C, int64_t ldc) {
  float v = acc;
  if (ep.bias) v += ep.bias[n];
  if (ep.resid) v += ep.resid[(int64_t)m * ldc + n];
  if (ep.beta != 0.f) v = fmaf(ep.beta, C[(int64_t)m * ldc + n], v);
  return v;
}

// Final value of C[m][n] (epilogue_value, then the fused GELU variants) and
// its store; with gelu_out also stores the activation.
__device__ __forceinline__ void epilogue_store(const GemmEpilogue& ep, float acc, int m, int n, float* C,
                                               int64_t ldc) {
  const int64_t at = (int64_t)m * ldc + n;
  float v = epilogue_value(ep, acc, m, n, C, ldc);
  if (ep.gelu_grad_of) v *= gelu_tanh_grad(ep.gelu_grad_of[at]);
  C[at] = v;
  if (ep.gelu_out) ep.gelu_out[at] = gelu_tanh(v);
}

// Four neighbouring outputs of a row (n a multiple of 4, 16-byte rows).
template <bool GELU>
__device__ __forceinline__ void epilogue_store4(const GemmEpilogue& ep, floatx4 v, floatx4 bias, int64_t at, float* C) {
  v += bias;
  if (ep.resid) v += *reinterpret_cast<const floatx4*>(ep.resid + at);
  if (ep.beta != 0.f) {
    const floatx4 c = *reinterpret_cast<const floatx4*>(C + at);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = fmaf(ep.beta, c[e], v[e]);
  }
  if constexpr (GELU) {
    if (ep.gelu_grad_of) {
      const floatx4 x = *reinterpret_cast<const floatx4*>(ep.gelu_grad_of + at);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] *= gelu_tanh_grad(x[e]);
    }
  }
  *reinterpret_cast<floatx4*>(C + at) = v;
  if constexpr (GELU) {
    if (ep.gelu_out) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = gelu_tanh(v[e]);
      *reinterpret_cast<floatx4*>(ep.gelu_out + at) = v;
    }
  }
}

// Output of a 2×2-wave tile (gemm_s_kernel, gemm_h_kernel, gemm_x_kernel):
// partials of a split K, or the epilogue.  The tile goes
// through the idle LDS ring (row pitch BN + 4 floats), so that a thread
// handles 16-byte runs of whole rows: loads and stores of 256 or 512
// contiguous bytes, and one small loop for the whole tile.  Straight from
// the accumulator layout the epilogue was unrolled once per element, 20 KB
// (64×64) to 80 KB (128×128) of code that every workgroup ran through once:
// a launch two panels deep took 7 and 20 µs, most of it instruction fetch.
// BN = 128 also emits the LM head's softmax row statistics (row_stats64),
// one thread per row and 64-column block; a block wholly past N writes none.
// each(put) calls put(row, col, value) for every accumulator of the thread.
// raw_tile (nullable): the raw tile's rows inside the matrix go there, BN apart.
template <int BM, int BN, int RING_BYTES, class Params, class Each>
__device__ __forceinline__ void tile_out(const Params& p, float* ring, int m0, int n0, int split, Each&& each,
                                         float* raw_tile = nullptr) {
  constexpr int SP = BN + 4;
  static_assert(BM * SP * 4 <= RING_BYTES, "LDS ring too small for the output tile");
  const int tid = threadIdx.x;
  const bool split_out = p.partial != nullptr;
  const bool stats = BN == 128 && p.ep.stats && !split_out;
  __syncthreads();  // every wave is done with the ring
  each([&](int row, int col, float v) {
    // columns past N take no part in the statistics
    ring[row * SP + col] = stats && n0 + col >= p.N ? -FLT_MAX : v;
  });
  __syncthreads();
  if constexpr (BN == 128) {
    if (stats && tid < 2 * BM) {
      const int row = tid % BM, blk = tid / BM, m = m0 + row, nb = n0 + 64 * blk;
      if (m < p.M && nb < p.N) p.ep.stats[(int64_t)m * p.ep.stats_ld + nb / 64] = row_stats64(ring + row * SP + 64 * blk);
    }
  }
  float* dst = split_out ? p.partial + (int64_t)split * p.M * p.N : p.C;
  const int64_t ld = split_out ? p.N : p.ldc;
  constexpr int CH = BN / 4, RP = 256 / CH;  // chunks of a row, rows per pass
  const int c = 4 * (tid % CH), n = n0 + c, r0 = tid / CH;
  const int rows = min(BM, p.M - m0);
  if (raw_tile) {
#pragma unroll 4
    for (int r = r0; r < rows; r += RP)
      *reinterpret_cast<floatx4*>(raw_tile + r * BN + c) = *reinterpret_cast<const floatx4*>(ring + r * SP + c);
  } else if (p.out_vec && n + 3 < p.N) {
    const float* src = ring + r0 * SP + c;
    int64_t at = (int64_t)(m0 + r0) * ld + n;
    if (split_out) {
#pragma unroll 4
      for (int r = r0; r < rows; r += RP, src += RP * SP, at += RP * ld)
        *reinterpret_cast<floatx4*>(dst + at) = *reinterpret_cast<const floatx4*>(src);
    } else {
      const floatx4 bias =
          p.ep.bias ? *reinterpret_cast<const floatx4*>(p.ep.bias + n) : floatx4{0.f, 0.f, 0.f, 0.f};
      if (p.ep.gelu_out || p.ep.gelu_grad_of) {
#pragma unroll 1
        for (int r = r0; r < rows; r += RP, src += RP * SP, at += RP * ld)
          epilogue_store4<true>(p.ep, *reinterpret_cast<const floatx4*>(src), bias, at, dst);
      } else {
#pragma unroll 4
        for (int r = r0; r < rows; r += RP, src += RP * SP, at += RP * ld)
          epilogue_store4<false>(p.ep, *reinterpret_cast<const floatx4*>(src), bias, at, dst);
      }
    }
  } else if (n < p.N) {  // unaligned rows, or the last columns of a ragged width
#pragma unroll 1
    for (int r = r0; r < rows; r += RP)
#pragma unroll 1
      for (int e = 0; e < 4 && n + e < p.N; ++e) {
        const float v = ring[r * SP + c + e];
        if (split_out) dst[(int64_t)(m0 + r) * ld + n + e] = v;
        else epilogue_store(p.ep, v, m0 + r, n + e, dst, ld);
      }
  }
}
// Whether tile_out may use 16-byte rows (host side).
template <class Params>
int out_vec(const Params& p) {
  if (p.partial) return p.N % 4 == 0 && ((uintptr_t)p.partial & 15) == 0;
  return p.ldc % 4 == 0 && (((uintptr_t)p.C | (uintptr_t)p.ep.bias | (uintptr_t)p.ep.resid | (uintptr_t)p.ep.gelu_out |
                             (uintptr_t)p.ep.gelu_grad_of) & 15) == 0;
}

// The same for a column-segmented launch, whose tiles store to their own segment's C.
bool segments_out_vec(const GemmHSegmentArg* seg, int nseg);

// Launch of the GEMM kernel proper.  With timing events set, the dispatch
// itself records them (hipExtLaunchKernel: the timestamps bracket the
// kernel's execution), so timing adds no event packets to the stream and the
// measured span matches a kernel trace's duration.
extern thread_local const KernelEvents* t_gemm_events;

template <typename Kern, class Params>
void launch_gemm_kernel(Kern kernel, dim3 grid, dim3 block, hipStream_t s, const Params& p) {
  if (t_gemm_events)
    hipExtLaunchKernelGGL(kernel, grid, block, 0, s, t_gemm_events->start, t_gemm_events->stop, 0, p);
  else
    hipLaunchKernelGGL(kernel, grid, block, 0, s, p);
}

// gemm_x.hip.  How gemm_x_launch runs C = A·op(B): tiles bm×bn of 32×64
// (gemm_s_kernel), 64×64, 64×128 or 128×128 (gemm_x_kernel); with splits > 1 every tile in that many K-slices to
// [slice][M][N] partials in ws, which the caller reduces; else the first
// `full` tiles whole and the others in tail_splits slices, summed by a second
// launch.
struct XPlan {
  int bm, bn, splits, full, tail_splits;
};
// norm: a row norm of the finished output follows (it rides in the
// reduction of a uniform split); stats: 128-wide tiles, none split.
// small: 32×64 tiles too; k_max: the deepest K-slice a tile may take; tail: K
// not in whole panels, or fp16 B.
XPlan plan_gemm_x(int M, int N, int K, int64_t k_max, size_t ws_bytes, bool norm, bool stats, bool small, bool tail);
int gemm_x_depth(const XPlan& pl, const GemmParams& p);  // the deepest K-slice of a plan
void gemm_x_launch(hipStream_t s, GemmParams& p, const XPlan& pl, bool b_nk, bool b_f16, float* ws,
                   const KernelEvents* tail_ev);
// gemm.hip: gemm_s_kernel on a grid of tile_slice.
void gemm_s_launch(hipStream_t s, const GemmParams& p, dim3 grid, bool b_nk, bool b_f16);

}  // namespace mft
#endif
