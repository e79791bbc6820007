// Instantiations: 16-bit tensors as one term of their own format (the dtype the reference runs its UNet in).
#include "cascmm_variants.h"
#include "cascmm_h16_kernel.h"

namespace cascmm {

template <class T, int FMT, int RAWB, int GLU>
static int launch_h16_kernel(const GroupParams& p, hipStream_t stream) {
  auto kfn = cascmm_h16_kernel<T, FMT, RAWB, GLU>;
  if (T::LDS_BYTES > 64 * 1024) {
    static LdsFlags lds_set;
    if (!ensure_lds((const void*)kfn, T::LDS_BYTES, lds_set)) return CASCMM_ERR_LAUNCH;
  }
  const dim3 grid((unsigned)(p.tiles_m * p.tiles_n * p.k_splits), (unsigned)p.count);
  return launch_kernel(kfn, grid, dim3(T::NT), (size_t)T::LDS_BYTES, stream, p) == hipSuccess ? CASCMM_OK : CASCMM_ERR_LAUNCH;
}

template <class T, int FMT, int RAWB, int GLU>
static int launch_h16(const GroupParams& p, hipStream_t stream) {
  if (p.kernel_out) { *p.kernel_out = (const void*)cascmm_h16_kernel<T, FMT, RAWB, 0>; return CASCMM_OK; }
  if (p.count < 1 || p.lda % 2 != 0 || (p.glu && !GLU)) return CASCMM_ERR_BAD_VARIANT;
  if (RAWB && (p.N % 2 != 0 || p.ldb % 2 != 0)) return CASCMM_ERR_BAD_VARIANT;
  if (p.lda * 2 * 512 >= 0x7FFFFFFF || (RAWB ? ((int64_t)p.K + 64) * p.ldb * 2 : ((int64_t)p.K + 63) / 64 * 128 * p.N) > 0x7FFFFFFF)
    return CASCMM_ERR_TOO_LARGE;
  if constexpr (GLU) {
    if (p.glu) return launch_h16_kernel<T, FMT, 0, 1>(p, stream);
  }
  if (p.k_splits > 1) {
    const int st = ksplit_check(p);
    if (st != CASCMM_OK) return st;
    GroupParams q = p;
    q.bias[0] = nullptr;
    const int sg = launch_h16_kernel<T, FMT, RAWB, 0>(q, stream);
    return sg == CASCMM_OK ? launch_ksplit_reduce<H16Elem<FMT>::DT>(p, stream) : sg;
  }
  return launch_h16_kernel<T, FMT, RAWB, 0>(p, stream);
}

// WM, WN, WK, MT, NTL, BK, NS: see H16.  An even NTL has the gated store.
#define H16_ROW(NAME, RAWB, FMT, DT, ...)                                                                               \
  {NAME, KIND_H16, DT, FMT, 1, false, H16<__VA_ARGS__>::BM, H16<__VA_ARGS__>::BN, H16<__VA_ARGS__>::BK, H16<__VA_ARGS__>::NT, \
   H16<__VA_ARGS__>::LDS_BYTES, true, true, &launch_h16<H16<__VA_ARGS__>, FMT, RAWB, (!RAWB && H16<__VA_ARGS__>::NTL % 2 == 0) ? 1 : 0>, \
   RAWB == 0, RAWB == 0 && H16<__VA_ARGS__>::NTL % 2 == 0}
#define H16_TILE(TILE, ...)                                                                            \
  H16_ROW(TILE "_h16_fp16x1_bpre_ioh", 0, CASCMM_FMT_FP16, CASCMM_DT_F16, __VA_ARGS__),                \
  H16_ROW(TILE "_h16_fp16x1_io16h", 1, CASCMM_FMT_FP16, CASCMM_DT_F16, __VA_ARGS__),                   \
  H16_ROW(TILE "_h16_bf16x1_bpre_iob", 0, CASCMM_FMT_BF16, CASCMM_DT_BF16, __VA_ARGS__),               \
  H16_ROW(TILE "_h16_bf16x1_io16b", 1, CASCMM_FMT_BF16, CASCMM_DT_BF16, __VA_ARGS__)

static const VariantDesc kTable[] = {
    // (stages in LDS: with more than these the first MFMA waits behind the loads of stages that are needed late:
    // 2048 x 2048 x 2048 on 128 x 128: 20.8 us with three, 22.0 with four, 23.5 with five)
    H16_TILE("t256x320x32", 4, 1, 1, 2, 10, 32, 4),
    H16_TILE("t256x256x32", 2, 2, 1, 4, 4, 32, 4),
    H16_TILE("t128x256x64", 2, 2, 1, 2, 4, 64, 3),
    H16_TILE("t128x160x64", 4, 1, 1, 1, 5, 64, 3),
    H16_TILE("t128x128x64", 2, 2, 1, 2, 2, 64, 3),
    H16_TILE("t64x160x64", 2, 1, 2, 1, 5, 64, 3),
    H16_TILE("t64x128x64", 2, 2, 1, 1, 2, 64, 3),   // (this and the next two: two workgroups on a CU)
    H16_TILE("t128x64x64", 2, 2, 1, 2, 1, 64, 3),
    H16_TILE("t64x64x64", 2, 2, 1, 1, 1, 64, 4),
};

const VariantDesc* variants_h16(int* n) {
  *n = (int)(sizeof(kTable) / sizeof(kTable[0]));
  return kTable;
}

}  // namespace cascmm
