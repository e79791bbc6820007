// Instantiations: 16-bit tensors as one term of their own format, small problems with K split over the waves of a workgroup.
#include "cascmm_variants.h"
#include "cascmm_hwk_kernel.h"

namespace cascmm {

template <int MB, int NB, int FMT, int RAWB, int GLU>
static int launch_hwk_kernel(const GroupParams& p, hipStream_t stream) {
  typedef HWK<MB, NB, RAWB> T;
  auto kfn = cascmm_hwk_kernel<MB, NB, FMT, RAWB, GLU>;
  if (T::LDS_BYTES > 64 * 1024) {
    static LdsFlags lds_set;
    if (!ensure_lds((const void*)kfn, T::LDS_BYTES, lds_set)) return CASCMM_ERR_LAUNCH;
  }
  const int64_t grid = (int64_t)p.count * p.tiles_m * p.tiles_n;
  if (grid <= 0 || grid > 0x7FFFFFFF) return CASCMM_ERR_TOO_LARGE;
  return launch_kernel(kfn, dim3((unsigned)grid), dim3(T::NT), (size_t)T::LDS_BYTES, stream, p) == hipSuccess ? CASCMM_OK : CASCMM_ERR_LAUNCH;
}

template <int MB, int NB, int FMT, int RAWB>
static int launch_hwk(const GroupParams& p, hipStream_t stream) {
  constexpr bool kGlu = !RAWB && NB == 4;
  if (p.kernel_out) { *p.kernel_out = (const void*)cascmm_hwk_kernel<MB, NB, FMT, RAWB, 0>; return CASCMM_OK; }
  if (p.count < 1 || p.K <= 0 || p.k_splits > 1 || p.lda % 2 != 0 || (p.glu && (!kGlu || p.glu != 1 || p.N % 64 != 0))) return CASCMM_ERR_BAD_VARIANT;
  if (RAWB && (p.N % 2 != 0 || p.ldb % 2 != 0)) return CASCMM_ERR_BAD_VARIANT;
  if (p.lda * 2 * 512 >= 0x7FFFFFFF || (RAWB ? ((int64_t)p.K + 64) * p.ldb * 2 : ((int64_t)p.K + 63) / 64 * 128 * p.N) > 0x7FFFFFFF)
    return CASCMM_ERR_TOO_LARGE;
  if constexpr (kGlu) {
    if (p.glu) return launch_hwk_kernel<MB, NB, FMT, 0, 1>(p, stream);
  }
  return launch_hwk_kernel<MB, NB, FMT, RAWB, 0>(p, stream);
}

#define HWK_ROW(NAME, MB, NB, RAWB, FMT, DT)                                                                                   \
  {NAME, KIND_HWK, DT, FMT, 1, false, HWK<MB, NB, RAWB>::BM, HWK<MB, NB, RAWB>::BN, HWK<MB, NB, RAWB>::BK, HWK<MB, NB, RAWB>::NT, \
   HWK<MB, NB, RAWB>::LDS_BYTES, true, true, &launch_hwk<MB, NB, FMT, RAWB>, RAWB == 0, RAWB == 0 && NB == 4, true}
#define HWK_BPRE(TILE, MB, NB)                                                                  \
  HWK_ROW(TILE "_hwk_fp16x1_bpre_ioh", MB, NB, 0, CASCMM_FMT_FP16, CASCMM_DT_F16),              \
  HWK_ROW(TILE "_hwk_bf16x1_bpre_iob", MB, NB, 0, CASCMM_FMT_BF16, CASCMM_DT_BF16)
#define HWK_RAW(TILE, MB, NB)                                                                   \
  HWK_ROW(TILE "_hwk_fp16x1_io16h", MB, NB, 1, CASCMM_FMT_FP16, CASCMM_DT_F16),                 \
  HWK_ROW(TILE "_hwk_bf16x1_io16b", MB, NB, 1, CASCMM_FMT_BF16, CASCMM_DT_BF16)

static const VariantDesc kTable[] = {
    HWK_BPRE("t16x16x64", 1, 1), HWK_BPRE("t16x32x64", 1, 2), HWK_BPRE("t16x64x64", 1, 4), HWK_BPRE("t32x32x64", 2, 2), HWK_BPRE("t32x64x64", 2, 4),
    HWK_BPRE("t64x64x64", 4, 4),   // (chosen for the gated store only)
    HWK_RAW("t16x32x64", 1, 2), HWK_RAW("t16x64x64", 1, 4), HWK_RAW("t32x32x64", 2, 2), HWK_RAW("t32x64x64", 2, 4),
};

const VariantDesc* variants_hwk(int* n) {
  *n = (int)(sizeof(kTable) / sizeof(kTable[0]));
  return kTable;
}

}  // namespace cascmm
