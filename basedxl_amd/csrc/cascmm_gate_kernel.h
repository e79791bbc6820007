// The gate of a gated projection whose product no kernel stores gated (columns off the tiles, a weight that is not kept split and rows off
// them, ...): out = value * gelu(gate) from h = [value | gate], gelu(x) = x (1 + erf(x / sqrt 2)) / 2 in fp32 whatever the elements are.
//
// Bound by memory: h is read once and the result written once, where an elementwise gelu and a product read and write gelu(gate) besides.
// A thread takes runs of VEC elements (16 bytes where the rows allow them) and asks for all of its own before the first is used.
// 16-bit elements take the gated stores' gelu (3.8e-6 relative at most where it matters, an element's half ulp is 4.9e-4): with erff, some 40
// instructions an element beside half the bytes, 4000 x 2560 took 14.5 us.
// Measured (graph replay, us, rows x inner; in brackets gelu and product as two launches): fp32 4000 x 2560 21.0 (47.1, 5.8 TB/s), 700 x 2560
// 6.2 (11.3), 120 x 2560 4.7 (7.0), single elements 4000 x 2559 27.3 (47.0); fp16 4000 x 2560 12.5 (31.5), 120 x 2560 4.3 (8.0), in 4-byte
// runs 4000 x 2558 16.7 (31.4), single elements 4000 x 2559 22.9 (31.3).
#pragma once
#include "cascmm_common.h"

namespace cascmm {

// runs of a row: 32-bit numbers (checked by the host), UNROLL of them a thread, 256 apart
template <int IODT, int VEC, int UNROLL>
__global__ __launch_bounds__(256) void cascmm_gate_kernel(const typename IoType<IODT>::T* __restrict__ h, int64_t ldh,
                                                          typename IoType<IODT>::T* __restrict__ out, int64_t ldo, unsigned per_row, unsigned total,
                                                          int64_t inner) {
  typedef typename IoType<IODT>::T T;
  struct alignas(VEC * sizeof(T)) Run { T v[VEC]; };
  Run value[UNROLL], gate[UNROLL];
  const unsigned first = blockIdx.x * (256u * UNROLL) + threadIdx.x;
#pragma unroll
  for (int u = 0; u < UNROLL; ++u) {
    const unsigned i = first + 256u * u;
    if (i >= total) continue;
    const unsigned row = i / per_row;
    const T* src = h + (int64_t)row * ldh + (int64_t)(i - row * per_row) * VEC;
    value[u] = *(const Run*)src;
    gate[u] = *(const Run*)(src + inner);
  }
#pragma unroll
  for (int u = 0; u < UNROLL; ++u) {
    const unsigned i = first + 256u * u;
    if (i >= total) continue;
    const unsigned row = i / per_row;
    Run r;
    float g[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) g[e] = IoType<IODT>::load(&gate[u].v[e]);
    if constexpr (sizeof(T) == 2) {
      gelu_values(g);
    } else {
#pragma unroll
      for (int e = 0; e < VEC; ++e) g[e] = 0.5f * g[e] * (1.f + erff(g[e] * 0.70710678118654752f));
    }
#pragma unroll
    for (int e = 0; e < VEC; ++e) IoType<IODT>::store(&r.v[e], IoType<IODT>::load(&value[u].v[e]) * g[e]);
    *(Run*)(out + (int64_t)row * ldo + (int64_t)(i - row * per_row) * VEC) = r;
  }
}

template <int IODT, int VEC, int UNROLL>
hipError_t launch_gate_runs(const void* h, int64_t ldh, void* out, int64_t ldo, int64_t rows, int64_t inner, hipStream_t stream) {
  typedef typename IoType<IODT>::T T;
  const int64_t total = rows * (inner / VEC);
  hipError_t err = hipSuccess;
  CASCMM_LAUNCH(err, (cascmm_gate_kernel<IODT, VEC, UNROLL>), dim3((unsigned)((total + 256 * UNROLL - 1) / (256 * UNROLL))), dim3(256), 0, stream,
                (const T*)h, ldh, (T*)out, ldo, (unsigned)(inner / VEC), (unsigned)total, inner);
  return err;
}
// 16-byte runs where rows, gates and results start on 16 bytes, else 4 bytes or single elements
template <int IODT>
hipError_t launch_gate(const void* h, int64_t ldh, void* out, int64_t ldo, int64_t rows, int64_t inner, hipStream_t stream) {
  constexpr int ES = (int)sizeof(typename IoType<IODT>::T), WIDE = 16 / ES;
  const auto fits = [&](int64_t n) {
    return inner % n == 0 && ldh % n == 0 && ldo % n == 0 && ((uintptr_t)h | (uintptr_t)out) % (uint64_t)(n * ES) == 0;
  };
  if (fits(WIDE)) return launch_gate_runs<IODT, WIDE, 1>(h, ldh, out, ldo, rows, inner, stream);
  if constexpr (ES == 2) {
    if (fits(2)) return launch_gate_runs<IODT, 2, 4>(h, ldh, out, ldo, rows, inner, stream);
  }
  return launch_gate_runs<IODT, 1, 4>(h, ldh, out, ldo, rows, inner, stream);
}

}  // namespace cascmm
