// Instantiations: right operand prepared (split once, stored as operand slots), fp32 left operand.
#include "cascmm_variants.h"

namespace cascmm {

#define BF CASCMM_FMT_BF16
#define FP CASCMM_FMT_FP16
#define F8 CASCMM_FMT_FP8

static const VariantDesc kTable[] = {
    // name, BM, BN, BK, WM, WN, WK, DEPTH, producer waves
    CASCMM_TILE_VARIANT_BPRE("t64x160x64_w2x1x2_d2_bf16x2_tri_bpre", 64, 160, 64, 2, 1, 2, 2, 4, BF, 2, false),
    CASCMM_TILE_VARIANT_BPRE("t64x160x64_w2x1x2_d3_bf16x2_tri_bpre", 64, 160, 64, 2, 1, 2, 3, 4, BF, 2, false),
    CASCMM_TILE_VARIANT_BPRE("t128x128x64_w2x2x1_d2_bf16x2_tri_bpre", 128, 128, 64, 2, 2, 1, 2, 4, BF, 2, false),
    CASCMM_TILE_VARIANT_BPRE("t128x160x32_w2x1x2_d3_bf16x2_tri_bpre", 128, 160, 32, 2, 1, 2, 3, 4, BF, 2, false),
    CASCMM_TILE_VARIANT_BPRE("t256x128x32_w4x1x1_d2_bf16x2_tri_bpre", 256, 128, 32, 4, 1, 1, 2, 4, BF, 2, false),
    CASCMM_TILE_VARIANT_BPRE("t64x64x64_w2x2x1_d3_bf16x2_tri_bpre", 64, 64, 64, 2, 2, 1, 3, 4, BF, 2, false),
    CASCMM_TILE_VARIANT_BPRE("t64x256x32_w1x4x1_d3_bf16x2_tri_bpre", 64, 256, 32, 1, 4, 1, 3, 4, BF, 2, false),
    CASCMM_TILE_VARIANT_BPRE("t256x160x32_w4x1x1_d2_bf16x2_tri_bpre", 256, 160, 32, 4, 1, 1, 2, 4, BF, 2, false),
    // the large-tile kernel fed with prepared slots of B (A still raw fp32, split at fragment-read time)
    CASCMM_W512_VARIANT("t256x320x32_w512_bf16x2_tri_bpre", 1),
    CASCMM_W512_EDGE_VARIANT("t256x320x32_w512_edge_bf16x2_tri_bpre", 1, 5),
    CASCMM_W512_EDGE_VARIANT("t256x256x32_w512_edge_bf16x2_tri_bpre", 1, 4),
    CASCMM_W512_EDGE_VARIANT("t256x192x32_w512_narrow_bf16x2_tri_bpre", 1, 3),
    CASCMM_W512_EDGE_VARIANT("t256x128x32_w512_narrow_bf16x2_tri_bpre", 1, 2),
    // K split over the eight waves of a workgroup: small problems
    CASCMM_WAVEK_VARIANT_B("t16x16x32_wavek_bf16x2_tri_bpre", 16, 1, 1, BF, 2, 1),
    CASCMM_WAVEK_VARIANT_B("t16x32x32_wavek_bf16x2_tri_bpre", 16, 1, 2, BF, 2, 1),
    CASCMM_WAVEK_VARIANT_B("t16x64x32_wavek_bf16x2_tri_bpre", 16, 1, 4, BF, 2, 1),
    CASCMM_WAVEK_VARIANT_B("t32x32x32_wavek_bf16x2_tri_bpre", 32, 1, 1, BF, 2, 1),
    CASCMM_WAVEK_VARIANT_B("t32x64x32_wavek_bf16x2_tri_bpre", 16, 2, 4, BF, 2, 1),
    CASCMM_WAVEK_VARIANT_B("t64x64x32_wavek_bf16x2_tri_bpre", 16, 4, 4, BF, 2, 1),
    CASCMM_TILE_VARIANT_BPRE("t128x128x32_w4x2x1_d2_bf16x3_tri_bpre", 128, 128, 32, 4, 2, 1, 2, 4, BF, 3, false),
    CASCMM_TILE_VARIANT_BPRE("t128x128x32_w4x2x1_d2_fp16x3_tri_bpre", 128, 128, 32, 4, 2, 1, 2, 4, FP, 3, false),
    CASCMM_TILE_VARIANT_BPRE("t128x128x32_w4x2x1_d2_fp8x3_tri_bpre", 128, 128, 32, 4, 2, 1, 2, 4, F8, 3, false),
};

const VariantDesc* variants_bpre(int* n) {
  *n = (int)(sizeof(kTable) / sizeof(kTable[0]));
  return kTable;
}

}  // namespace cascmm
