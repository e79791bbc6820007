// K split over workgroups for the kernels whose tiles are large for few rows: workgroup (tile, split) multiplies
// split's share of K and writes its fp32 sums to the workspace, [split][M][ksplit_row(N)]; a second launch adds the
// splits in order, the bias, and writes C.
#pragma once
#include "cascmm_tile_kernel.h"

namespace cascmm {

constexpr int kMaxKSplits = 16;

// The workgroups of a launch: (split, tile), the splits' tile rows one below the other, so that an XCD's contiguous range
// lies in one split or two and its L2 holds their share of K only (512 x 5120 x 1280 prepared in four splits: with every
// XCD at work on all splits of its tiles 35 us, so 31).  In: the row of the stack.  Out: the tile row, returns the split.
__device__ __forceinline__ int ksplit_of_row(int& tm, int tiles_m, int k_per, int K) {
  if (k_per >= K) return 0;
  const int split = tm / tiles_m;
  tm -= split * tiles_m;
  return split;
}

// k of a split (all but the last): whole 64-k stages, so that only the last one can end inside a stage
inline int64_t ksplit_k(int64_t K, int splits) { return ((K + splits - 1) / splits + 63) / 64 * 64; }
// a count of splits of which none is empty
inline bool ksplit_valid(int64_t K, int splits) { return splits >= 1 && splits <= kMaxKSplits && (splits - 1) * ksplit_k(K, splits) < K; }
// floats of a row of partial results: whole 16-byte chunks
inline int64_t ksplit_row(int64_t N) { return (N + 3) / 4 * 4; }
inline size_t ksplit_bytes(int64_t M, int64_t N, int splits) { return splits > 1 ? (size_t)splits * (size_t)M * (size_t)ksplit_row(N) * sizeof(float) : 0; }

// A thread adds four consecutive columns of one row; the loads of up to eight splits are in flight.  Bound by its
// latency, not by bytes: 2.5 - 4.2 us (kernel trace, medians) for 0.3 to 10 MB of partial results alike
// (profiles/cascmm_ksplit_kernels.txt).
template <int IODT>
__global__ __launch_bounds__(256) void ksplit_reduce_kernel(const float* __restrict__ parts, int splits, int M, int N, const void* __restrict__ bias,
                                                           void* __restrict__ C, int64_t ldc, int vec_out) {
  typedef IoType<IODT> Io;
  typedef typename Io::T E;
  const int quads = (N + 3) >> 2;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, total = (int64_t)M * quads;
  if (i >= total) return;
  const int m = (int)(i / quads), n = (int)(i - (int64_t)m * quads) * 4;
  const f32x4* src = (const f32x4*)parts + i;
  f32x4 s = src[0];
  for (int k = 1; k < splits; k += 7) {
    f32x4 v[7];
#pragma unroll
    for (int u = 0; u < 7; ++u) v[u] = src[(int64_t)(k + u < splits ? k + u : 0) * total];
#pragma unroll
    for (int u = 0; u < 7; ++u)
      if (k + u < splits) s += v[u];
  }
  E* c = (E*)C + (int64_t)m * ldc + n;
  typedef E e4 __attribute__((ext_vector_type(4)));
  if (bias) {
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] += n + e < N ? Io::load((const E*)bias + n + e) : 0.f;
  }
  if (vec_out) {   // N % 4 == 0, rows of C on whole quads
    *(e4*)c = __builtin_convertvector(s, e4);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < N) Io::store(c + e, s[e]);
  }
}

// Host side of a split launch: the launch functions' own check of what the caller has decided
inline int ksplit_check(const GroupParams& p) {
  if (p.count != 1 || p.glu || !ksplit_valid(p.K, p.k_splits) || p.k_per != ksplit_k(p.K, p.k_splits)) return CASCMM_ERR_BAD_VARIANT;
  if (!p.workspace || p.workspace_bytes < ksplit_bytes(p.M, p.N, p.k_splits)) return CASCMM_ERR_WORKSPACE;
  return (uintptr_t)p.workspace % 16 == 0 ? CASCMM_OK : CASCMM_ERR_ALIGNMENT;
}
template <int IODT> int launch_ksplit_reduce(const GroupParams& p, hipStream_t stream) {
  typedef typename IoType<IODT>::T E;
  const int64_t total = (int64_t)p.M * ((p.N + 3) / 4);
  const int vec_out = p.N % 4 == 0 && p.ldc % 4 == 0 && (uintptr_t)p.C[0] % (4 * sizeof(E)) == 0;
  return launch_kernel(ksplit_reduce_kernel<IODT>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, (const float*)p.workspace, p.k_splits,
                       p.M, p.N, p.bias[0], p.C[0], p.ldc, vec_out) == hipSuccess
             ? CASCMM_OK
             : CASCMM_ERR_LAUNCH;
}

}  // namespace cascmm
