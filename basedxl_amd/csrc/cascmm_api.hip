// extern "C" entry points: argument checks, kernel selection, small utility kernels.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <dlfcn.h>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "cascmm_gate_kernel.h"
#include "cascmm_variants.h"

namespace cascmm {

// ---------------------------------------------------------------------------------------
// variant table (immutable after first use)
// ---------------------------------------------------------------------------------------
static const std::vector<VariantDesc>& table() {
  static const std::vector<VariantDesc> t = [] {
    std::vector<VariantDesc> v;
    int n = 0;
    const VariantDesc* p = variants_bf16(&n);
    v.insert(v.end(), p, p + n);
    p = variants_fp16(&n);
    v.insert(v.end(), p, p + n);
    p = variants_fp8(&n);
    v.insert(v.end(), p, p + n);
    p = variants_io16(&n);
    v.insert(v.end(), p, p + n);
    p = variants_bpre(&n);
    v.insert(v.end(), p, p + n);
    p = variants_chain(&n);
    v.insert(v.end(), p, p + n);
    p = variants_h16(&n);
    v.insert(v.end(), p, p + n);
    p = variants_hwk(&n);
    v.insert(v.end(), p, p + n);
    return v;
  }();
  return t;
}

struct TunedCost;
struct CallCost;
// per variant, resolved once when the table is built: its measured cost constants (or none) and what
// kind of kernel its name says it is
struct VariantInfo {
  const TunedCost* tuned;
  const CallCost *call, *gated, *shape;   // (shape: for the selection functions)
  bool p8, bdirect;
};
static const std::vector<VariantInfo>& variant_info();

static bool aligned_to(const void* p, size_t a) { return ((uintptr_t)p % a) == 0; }
static size_t dtype_size(int dt) { return dt == CASCMM_DT_F32 ? 4 : 2; }

struct Problem {
  int64_t M, N, K, lda, ldb, ldc;
  int dtype, fmt, terms, products;
  bool bpre = false;  // B is a prepared (already split) weight buffer
  bool glu = false;   // gated epilogue: B prepared by cascmm_prepare_weight_glu, C has N / 2 columns
  bool glu_slots = false;   // ... written as the left operand slots of the next GEMM (large-tile kernel only)
  // the rows of A are whole 16-byte chunks with zeros between K and the last chunk's end: fp32 with K % 4 == 0, 16-bit
  // with K % 8 == 0, or rows padded in the workspace (relay)
  bool chunked = false;
  // a call (not the selection functions, which answer for a shape): the small tiles of KIND_WAVEK are open too, and rows that
  // are not chunked, which these kernels read where they lie (what lies past K is masked)
  bool call = false;
  // three fp8 / fp16 terms: only the kernels that split both operands into slots first; K is rounded up to whole
  // stages, of which the operands hold k_valid, and their rows need no alignment
  bool split_first = false;
  int64_t k_valid = 0;
  bool whole_k = false;   // no K split over workgroups (cascmm_ksplit.h)
};

// Three fp8 terms with K a multiple of 64 are prepared for the fp8-rate kernel: [term][K/16][N] slots
// of 16 k each (the gated layout keeps the older form, whose kernels have the gated store)
static bool prepared_as_k16_slots(int64_t K, int fmt, int terms, bool glu) {
  return fmt == CASCMM_FMT_FP8 && terms == 3 && K > 0 && K % F8K64::BK == 0 && !glu;
}

// a x b x c > 2^31 - 1, for any non-negative 64-bit factors (the product itself may not fit 64 bits)
static bool beyond_i32(int64_t a, int64_t b, int64_t c) {
  int64_t ab = 0, abc = 0;
  return __builtin_mul_overflow(a, b, &ab) || __builtin_mul_overflow(ab, c, &abc) || abc > INT32_MAX;
}

// bytes of a prepared weight: planes x prepared_kgroups(K) x N operand slots of 16 bytes
static int64_t prepared_bytes(int64_t K, int64_t N, int fmt, int terms, bool glu = false) {
  if (prepared_as_k16_slots(K, fmt, terms, glu)) return f8k64_slot_bytes(N, K);
  const int planes = fmt == CASCMM_FMT_FP8 ? (terms + 1) / 2 : terms;
  int64_t slots = 0, bytes = 0;   // (saturates instead of overflowing: callers compare the result with limits)
  if (__builtin_mul_overflow((int64_t)planes * prepared_kgroups(K), N, &slots) || __builtin_mul_overflow(slots, (int64_t)16, &bytes))
    return INT64_MAX;
  return bytes;
}

static int check_problem(const Problem& q) {
  if (q.dtype != CASCMM_DT_F32 && q.dtype != CASCMM_DT_F16 && q.dtype != CASCMM_DT_BF16) return CASCMM_ERR_BAD_DTYPE;
  if (q.fmt != CASCMM_FMT_BF16 && q.fmt != CASCMM_FMT_FP16 && q.fmt != CASCMM_FMT_FP8) return CASCMM_ERR_BAD_FORMAT;
  if (q.terms < 1 || q.terms > 3) return CASCMM_ERR_BAD_FORMAT;
  if (q.products != CASCMM_PROD_TRI && q.products != CASCMM_PROD_FULL) return CASCMM_ERR_BAD_FORMAT;
  if (q.M < 0 || q.N < 0 || q.K < 0) return CASCMM_ERR_BAD_SHAPE;
  if (q.M > INT32_MAX || q.N > INT32_MAX || q.K > INT32_MAX) return CASCMM_ERR_TOO_LARGE;
  if (q.lda < (q.split_first ? q.k_valid : q.K) || q.ldb < q.N || q.ldc < (q.glu ? q.N / 2 : q.N)) return CASCMM_ERR_BAD_SHAPE;
  return CASCMM_OK;
}

// 16-bit tensors multiplied as one term of their own format: exact operands, nothing to split
static bool own_format16(const Problem& q) {
  return q.terms == 1 && ((q.dtype == CASCMM_DT_F16 && q.fmt == CASCMM_FMT_FP16) || (q.dtype == CASCMM_DT_BF16 && q.fmt == CASCMM_FMT_BF16));
}

// What the rows of the operands allow.  FIT_DWORD: 32-bit byte offsets inside a tile and down a column block of B
// (buffer offsets are 32-bit): the kernels whose loads are checked against the buffers' ends dword by dword take any
// alignment and any N.  FIT_FAST: 16-byte aligned rows and N % 4 == 0 too, which the other fast kernels need (K % BK is
// checked per kernel).  16-bit tensors have one kind of fast kernel: rows on dwords.
enum RowFit { FIT_NONE = 0, FIT_DWORD = 1, FIT_FAST = 2 };
static RowFit row_fit(const Problem& q, const void* A, const void* B) {
  if (q.dtype != CASCMM_DT_F32) {
    // 16-bit operands: only as one term of their own format
    return own_format16(q) && q.lda % 2 == 0 && (A == nullptr || aligned_to(A, 4)) && q.lda * 2 * 512 < INT32_MAX &&
                   (q.bpre || (q.ldb % 2 == 0 && q.N % 2 == 0 && (B == nullptr || aligned_to(B, 4))))
               ? FIT_FAST
               : FIT_NONE;
  }
  if (q.split_first) return FIT_FAST;
  if (!(q.lda * 4 * 512 < INT32_MAX && (q.bpre || (q.ldb * 4 * 136 < INT32_MAX && q.K * q.ldb * 4 < INT32_MAX)))) return FIT_NONE;
  return q.lda % 4 == 0 && (A == nullptr || aligned_to(A, 16)) &&
                 (q.bpre || (q.ldb % 4 == 0 && q.N % 4 == 0 && (B == nullptr || aligned_to(B, 16))))
             ? FIT_FAST
             : FIT_DWORD;
}

static bool variant_matches(const VariantDesc& v, const Problem& q, RowFit fit) {
  const int full = (q.products == CASCMM_PROD_FULL && q.terms > 1) ? 1 : 0;
  if (v.iodt != q.dtype || v.fmt != q.fmt || v.terms != q.terms || v.full != full || v.bpre != q.bpre) return false;
  if (q.split_first && v.kind != KIND_F8K64 && v.kind != KIND_F16K) return false;
  const bool any_rows = v.kind == KIND_WAVEK || v.kind == KIND_SLOTK;
  if (v.fast && fit < (any_rows ? FIT_DWORD : FIT_FAST)) return false;
  // K in whole 32-k steps, or a tail of whole 16-byte chunks (a weight less than one 64-k stage deep is not worth keeping
  // split: such a prepared operand is refused)
  if ((v.kind == KIND_SLOTK || v.kind == KIND_W512E) && (q.K == 0 || (q.K % 32 != 0 && !(q.chunked && (!q.bpre || q.K >= 64))))) return false;
  if (v.fast && !any_rows && v.kind != KIND_H16 && v.kind != KIND_HWK && (v.kind != KIND_W512E || q.glu) && q.K % v.BK != 0) return false;
  if (v.kind == KIND_SPLITK && (q.M > 5 * v.BM || q.K < 4 * v.BK)) return false;  // skinny: few row tiles, deep K
  if (v.kind == KIND_F8K64 && (q.products != CASCMM_PROD_TRI || q.K % v.BK != 0 || q.K == 0 || q.glu ||
                               f8k64_slot_bytes(q.M, q.K) > INT32_MAX || f8k64_slot_bytes(q.N, q.K) > INT32_MAX))
    return false;
  if (v.kind == KIND_F16K && (q.products != CASCMM_PROD_TRI || q.K % v.BK != 0 || q.K == 0 || q.glu || q.bpre ||
                              (v.BM == F16K::BM && q.K > F16K::MAX_K) || q.K * q.ldb * 4 > INT32_MAX ||
                              f16k_slot_bytes(q.M, q.K) > INT32_MAX || f16k_slot_bytes(q.N, q.K) > INT32_MAX))
    return false;
  if (v.bpre && v.kind != KIND_F8K64 && prepared_as_k16_slots(q.K, q.fmt, q.terms, q.glu)) return false;   // other layout
  if (v.kind == KIND_W512 && (q.M % v.BM != 0 || q.N % v.BN != 0 || q.M * q.lda * 4 > INT32_MAX ||
                              (!q.bpre && q.K * q.ldb * 4 > INT32_MAX) || q.ldc * (int64_t)(v.BM * 4) > INT32_MAX))
    return false;
  if (v.kind == KIND_W512E && (q.M < W512_EDGE_ROWS || q.N < v.BN || (q.glu && v.BN == W512::BN && q.N % v.BN != 0) || q.lda < 32 || q.M * q.lda * 4 > INT32_MAX ||
                               (!q.bpre && beyond_i32(q.K + 32, q.ldb, 4)) || q.ldc * (int64_t)(v.BM * 4) > INT32_MAX))
    return false;
  // (rows that are not chunked: up to four rounds of tiles, larger problems are worth a copy of A)
  if (v.kind == KIND_WAVEK && q.bpre && q.K % 32 != 0 && !(q.chunked && q.K >= 64)) return false;   // (as KIND_SLOTK)
  if (v.kind == KIND_WAVEK && (q.K == 0 || (q.K % 32 != 0 && !q.chunked && (!q.call || ((q.M + v.BM - 1) / v.BM) * ((q.N + v.BN - 1) / v.BN) > 4 * kNumCUs)) || (v.call_only && !q.call) || beyond_i32(q.M, q.lda, 4))) return false;
  if (v.kind == KIND_SLOTK && (q.lda < 32 || q.glu || q.M * q.lda * 4 > INT32_MAX || q.ldc * (int64_t)(v.BM * 4) > INT32_MAX))
    return false;
  // (32-bit byte offsets down B, a raw one's two stages past the end included, and inside a tile of A, see row_fit; K in whole 16-byte chunks)
  if ((v.kind == KIND_HWK || v.kind == KIND_W512E) && v.call_only && !q.call) return false;
  if ((v.kind == KIND_H16 || v.kind == KIND_HWK) && ((q.K % 8 != 0 && !q.chunked) || q.K == 0 || (q.bpre ? beyond_i32((q.K + 63) / 64, q.N, 128) : beyond_i32(q.K + 64, q.ldb, 2))))
    return false;
  if (q.glu && !v.glu) return false;
  if (q.glu_slots && v.kind != KIND_W512) return false;
  return true;
}

// Cost model.  The two-term bf16 and three-term fp8 kernels, which carry the SDXL workload, are costed from
// constants measured on MI355X (sweep over the UNet's Linear shapes, HIP-graph replay): a launch
// takes  rounds x (K/64 x step64 + fixed)  microseconds, where a partly filled last round counts
// as  tail + (1 - tail) x fill  of a full one, with one `tail` for a launch that has no full
// round (its tiles run faster: less contention for the caches) and one for later rounds.  Other kernels use the analytic form the constants were first fitted with: a
// 64-deep K step of a full round costs about (BM*BN + 64*(BM+BN)) / 20000 microseconds (MFMA
// work grows with BM*BN; loading, splitting and staging grow with BM+BN and weigh about as much
// at these tile sizes).
struct TunedCost { const char* name; double step64_us, fixed_us, tail_first, tail_later; };
static const TunedCost kTuned[] = {
    {"t64x160x64_w2x1x2_d2_bf16x2_tri", 1.228, 4.34, 1.00, 0.80},
    {"t256x128x32_w4x1x1_d2_bf16x2_tri", 2.294, 7.99, 0.80, 0.80},
    {"t128x128x32_w4x1x1_d3_bf16x2_tri", 1.464, 5.83, 0.90, 0.80},
    {"t128x128x64_w2x1x2_d2_bf16x2_tri", 1.189, 8.10, 0.90, 0.80},
    {"t64x128x64_w2x1x2_d3_bf16x2_tri", 0.922, 4.17, 1.00, 0.90},
    {"t64x64x64_w2x2x1_d3_bf16x2_tri", 0.671, 2.34, 1.00, 1.00},
    {"t64x160x64_w2x1x2_d2_p8_bf16x2_tri", 1.064, 4.69, 0.90, 0.80},
    {"t128x128x64_w4x1x1_d2_p8_bf16x2_tri", 1.224, 6.84, 0.80, 0.70},
    {"t256x160x32_w4x1x1_d2_bf16x2_tri", 3.200, 6.50, 0.70, 0.50},
    // (the large tiles on raw weights: partly filled rounds are faster than full ones, the board's power goes to fewer CUs: 64 of 256
    // tiles 0.62 of a round, 144 tiles 0.7, 192 tiles 0.88; on prepared ones: kLargeTileCost)
    {"t256x320x32_w512_bf16x2_tri", 5.65, 16.0, 0.50, 0.50},
    {"t256x320x32_w512_edge_bf16x2_tri", 5.65, 17.0, 0.50, 0.50},
    {"t256x256x32_w512_edge_bf16x2_tri", 4.60, 10.5, 0.45, 0.45},
    // three fp16 / bf16 terms
    {"t128x128x32_w4x2x1_d2_fp16x3_tri", 3.107, 7.22, 0.90, 0.80},
    {"t64x64x32_w2x2x1_d3_fp16x3_tri", 1.088, 2.27, 1.00, 1.00},
    {"t128x128x32_w4x2x1_d2_bf16x3_tri", 2.596, 7.02, 0.80, 0.70},
    {"t64x64x32_w2x2x1_d3_bf16x3_tri", 0.910, 2.20, 1.00, 1.00},
    // three fp8 terms (static tensor scales)
    {"t128x128x32_w4x2x1_d2_fp8x3_tri", 2.547, 6.33, 1.00, 0.90},
    {"t64x64x64_w2x2x1_d2_fp8x3_tri", 1.016, 2.50, 1.00, 1.00},
    {"t128x128x32_w2x2x1_d2_fp8x3_tri", 2.211, 6.93, 0.90, 0.80},
    {"t64x128x64_w2x2x2_d2_fp8x3_tri", 1.409, 4.91, 1.00, 0.90},
    // right operand prepared (sweep over M in 1024..8192 of the UNet's (K, N) pairs)
    {"t64x160x64_w2x1x2_d2_bf16x2_tri_bpre", 0.925, 5.57, 0.80, 0.60},
    {"t64x160x64_w2x1x2_d3_bf16x2_tri_bpre", 0.891, 6.26, 0.90, 0.80},
    {"t128x128x64_w2x2x1_d2_bf16x2_tri_bpre", 1.193, 6.27, 0.90, 0.80},
    {"t128x160x32_w2x1x2_d3_bf16x2_tri_bpre", 1.501, 9.45, 0.70, 0.50},
    {"t256x128x32_w4x1x1_d2_bf16x2_tri_bpre", 2.192, 9.64, 0.70, 0.70},
    {"t64x64x64_w2x2x1_d3_bf16x2_tri_bpre", 0.515, 2.08, 1.00, 1.00},
    {"t64x256x32_w1x4x1_d3_bf16x2_tri_bpre", 1.250, 5.89, 0.80, 0.50},
    {"t256x160x32_w4x1x1_d2_bf16x2_tri_bpre", 2.837, 12.00, 0.60, 0.50},
    // K split over the waves: a round of 256 tiles costs 0.011 us per k + 8 us, and rounds do not overlap
    // (2048 x {1280, 5120} x 1280: 21.7 / 64.3 us; 1024 x 1280 x 1280: 17.4 us -- 7 % less than with raw A fetched
    // in half lines, A/B on one card)
    {"k64x160x16_wk4_bf16x2_tri_bpre", 0.71, 8.0, 0.65, 0.95},
    {"k64x80x32_wk4_bf16x2_tri_bpre", 0.445, 5.4, 0.69, 0.95},
    // ... both operands raw (2048 x {1280, 5120} x 1280: 24.0 / 77.2 us; 8192 x 2560 x 640, two rounds: 79.3 us)
    {"k64x160x16_wk4_bf16x2_tri", 0.887, 6.3, 0.65, 0.95},
};

constexpr int kMaxTileSplits = 4;
// kernels that split K over workgroups as cascmm_ksplit.h describes
static bool ksplit_kind(const VariantDesc& v) { return v.kind == KIND_H16 || v.kind == KIND_SLOTK; }
// the fp8-rate kernel with K over the waves: us per 64-k stage of a wave, and per round of tiles
constexpr double kF8WKStageUs = 2.25, kF8WKFixedUs = 6.0;   // (fit: 2048 x {1280, 5120} x 1280, 4096 x {640, 2560} x 640)


// Calls with two bf16 terms, plain products.  A launch of `tiles` tiles on 256 CUs, k in units of the kernel's loop (KIND_WAVEK and
// KIND_HWK: steps per wave; K over four waves: trips of 256 k, in 64s; else 64 k):  c0 + full (c1 + k r1) + |k s0, fill k s1 + MB of B / bw|_x
// (the x-norm), where full rounds of 256 tiles go before one that is `fill` full.  The small tiles have rounds like the others, though several fit
// a CU: the one CU that gets a second tile runs both at once, and each takes longer (200 x 2560 x 640 prepared: 260 tiles of 16 x 32 14.8 us,
// 200 of them for 154 rows 9.8; 70 of 32 x 32 10.9).  deep: what a step past the straight code's adds; for the
// kernels without any, us per 1e9 multiply-adds (tiles filled up) at the board's power, which deep products of many tiles run into.  edge: tiles over
// an edge of C, us per round (their store is the checked one); of the small ones the share that the form for the right edge costs.
// MB: both operands.  Fitted to 1633 prepared and 1526 raw shapes of 2 - 9000 rows, K 256 - 5120, widths 256 - 10240, a fifth of them the sizes that
// models have and squares (graph replay over three sets of operands, every kernel forced in turn), mean error 0.02 - 0.09.  The kernel chosen
// is behind the fastest of all, on average and in one of twenty: 2 - 2048 rows 0.5 and 3.0 % (prepared), 0.5 and 1.8 % (raw); 600 - 9000 rows 1.0 and 5.7 %,
// 1.0 and 6.8 %; products beyond 1.2e10 multiply-adds 0.2 and 1.0 %, 0.1 and 0 %; sizes of models 0.4 and 3.0 %, 0.7 and 4.6 %.  (With constants fitted to one set of
// operands, which the L2s kept, small tiles without rounds and B's bytes alone: 1.5 and 9.9 %, 1.3 and 11 %; 1.7 and 10 %, 2.2 and 16 %; 0.5 and 2.6 %, 0.9 and 8.3 %;
// 1.3 and 9.6 %, 1.5 and 11 %: 7296 x 1198 x 283 54.7 us, 43.9 with these.)  The eight-wave tiles' errors are on the low side behind a full round
// (7 %) and with more than 5 MB of A (10 %; rows off 16 bytes of 20 MB and more 25 %, where a copy of A is the alternative), which their estimates are
// raised by.  Groups: the tiles of all their problems; there the eight-wave tiles are 5 - 8 % faster than that and the prepared 64 x 160 one 8 % slower (305 groups
// of two and three, 0.6 and 0.8 % behind the fastest on average, 2.5 and 3.5 % in one of twenty).
// The large tiles of 192 and 128 columns, and all gated large tiles, are fitted to 230 shapes each (raw, prepared, gated; 300 - 9000 rows).  On 376 raw,
// 380 prepared and 380 gated others they are chosen for 38, 35 and 23, which take 0.92, 0.91 and 0.87 of the time of what was chosen before
// (one of them more than 3 % longer: gated 1289 x 576 x 4608 28.5 us, 26.5); the kernel chosen is 0.3 - 0.6 % behind the fastest of all on average.
// The selection functions, which answer for shapes, keep the constants above but for KIND_WAVEK.
struct CallCost { const char* name; double c0, s0, s1, c1, bw, x, r1, deep, edge; };
static const CallCost kCallCost[] = {
    {"t16x16x32_wavek_bf16x2_tri", 2.45, 0.392, 0.199, 0, 26, 1, 0.477, 0.125, 0.0733},
    {"t16x32x32_wavek_bf16x2_tri", 2.43, 0.679, 0.376, 0, 19.2, 1.44, 0.656, 0.0251, 0.0805},
    {"t16x64x32_wavek_bf16x2_tri", 2.5, 0.887, 0.404, 1.12, 25.1, 1, 1.06, 0, 0.0803},
    {"t32x32x32_wavek_bf16x2_tri", 2.48, 0.877, 0.553, 0.589, 60, 1.29, 1.2, 0, 0.0976},
    {"t32x64x32_wavek_bf16x2_tri", 3.09, 1.09, 0.626, 1.69, 60, 1, 1.44, 0, 0.0651},
    {"t64x64x32_wavek_bf16x2_tri", 5.14, 1.28, 1.23, 2.43, 60, 1.23, 2.22, 0, 0.037},
    {"k64x160x16_wk4_bf16x2_tri", 6.72, 0.598, 0.632, 5.15, 19.2, 2.19, 0.817, 5.44, 0.178},
    {"bd64x128x64_d3_p4_bf16x2_tri", 4.36, 1.08, 0.735, 1.88, 15.8, 2.88, 1.1, 5.63, 0.77},
    {"bd96x128x64_d3_p4_bf16x2_tri", 5.62, 1.23, 0.828, 3.35, 7.45, 2.89, 1.28, 6.21, 1.54},
    {"bd128x128x32_d3_p4_bf16x2_tri", 5.03, 1.49, 1.22, 3.44, 60, 2.71, 1.53, 6.29, 1.88},
    {"bd192x128x64_d2_p4_bf16x2_tri", 7.19, 1.87, 1.37, 4.95, 5, 3.33, 2.03, 5.64, 3.33},
    {"t64x64x64_w2x2x1_d3_bf16x2_tri", 4.77, 0.691, 0.166, 0.732, 60, 1.21, 0.704, 0.0299, 0.612},
    {"t64x160x64_w2x1x2_d2_p8_bf16x2_tri", 6.13, 0.882, 0.448, 2.91, 60, 1.56, 0.914, 7.15, 3.83},
    {"t128x128x64_w4x1x1_d2_p8_bf16x2_tri", 7.79, 0.949, 1.03, 3.05, 14.8, 2.11, 1.24, 5.44, 4.31},
    {"t256x128x32_w4x1x1_d2_bf16x2_tri", 8.14, 1.84, 1.92, 4.28, 5.15, 3.21, 2.37, 4.76, 10.8},
    {"t256x160x32_w4x1x1_d2_bf16x2_tri", 10.6, 2.12, 2.43, 5.46, 7.3, 3.16, 2.67, 4.77, 12.2},
    {"t256x128x32_w512_narrow_bf16x2_tri", 10, 1.97, 1.97, 6.25, 7.12, 3.15, 2.7, 5.3, 0},
    {"t256x192x32_w512_narrow_bf16x2_tri", 11.6, 2.48, 3.1, 8.09, 5, 3.95, 3.66, 4.74, 0.115},
    {"t256x256x32_w512_edge_bf16x2_tri", 10.8, 2.93, 4.76, 9.03, 51.2, 3.72, 4.87, 0, 1.43},
    {"t256x320x32_w512_edge_bf16x2_tri", 12.5, 3.48, 5.85, 13.5, 60, 3.47, 5.71, 0.153, 1.61},
    {"t256x320x32_w512_bf16x2_tri", 12.4, 3.45, 5.79, 13.4, 60, 3.47, 5.65, 0.151, 0},
    // three fp16 terms (448 shapes; the tile chosen is 0.06 % behind the fastest of the three, without rounds 0.4 %, at most 26 %)
    {"t16x16x32_wavek_fp16x3_tri", 2.47, 0.728, 0.176, 0.125, 28.6, 1, 0.664, 0.051, 0},
    {"t16x32x32_wavek_fp16x3_tri", 2.44, 1.13, 0.236, 0.804, 38.3, 1, 1.23, 0, 0},
    {"t32x32x32_wavek_fp16x3_tri", 2.79, 1.5, 0.319, 1.57, 60, 1, 1.62, 0, 0},
    // ... tiles that scale themselves: the same, select_scaled_rows adds what the maxima take
    {"t16x16x32_wavek_fp16x3_tri_scaled", 2.47, 0.728, 0.176, 0.125, 28.6, 1, 0.664, 0.051, 0},
    {"t16x32x32_wavek_fp16x3_tri_scaled", 2.44, 1.13, 0.236, 0.804, 38.3, 1, 1.23, 0, 0},
    {"t32x32x32_wavek_fp16x3_tri_scaled", 2.79, 1.5, 0.319, 1.57, 60, 1, 1.62, 0, 0},
    // three fp8 terms (493 shapes, hardly ever behind the fastest; without rounds 0.6 %, at most 33 %)
    {"t16x16x32_wavek_fp8x3_tri", 2.54, 0.713, 0.229, 0.147, 28.1, 1, 0.655, 0.00446, 0},
    {"t16x32x32_wavek_fp8x3_tri", 2.57, 1.1, 0.207, 1.1, 26.9, 1, 1.24, 0, 0},
    {"t32x32x32_wavek_fp8x3_tri", 2.91, 1.4, 0.425, 2.04, 60, 1, 4.23, 0.0301, 0},
    // prepared weights
    {"t16x16x32_wavek_bf16x2_tri_bpre", 2.63, 0.241, 0.211, 0.112, 20.1, 1.25, 0.347, 0.0308, 0.0554},
    {"t16x32x32_wavek_bf16x2_tri_bpre", 2.6, 0.367, 0.314, 0, 19.2, 1.27, 0.547, 0.0707, 0.036},
    {"t16x64x32_wavek_bf16x2_tri_bpre", 2.69, 0.604, 0.365, 0.906, 26.6, 1, 0.986, 0.155, 0.0211},
    {"t32x32x32_wavek_bf16x2_tri_bpre", 2.67, 0.592, 0.597, 0.772, 29, 1.53, 0.986, 0, 0.0563},
    {"t32x64x32_wavek_bf16x2_tri_bpre", 2.97, 0.872, 0.585, 1.22, 60, 1, 1.32, 0, 0.0249},
    {"t64x64x32_wavek_bf16x2_tri_bpre", 4.59, 1.13, 0.884, 1.99, 60, 1.04, 2.03, 0, 0.0331},
    {"k64x80x32_wk4_bf16x2_tri_bpre", 5.85, 0.322, 0.13, 4.01, 60, 1, 0.433, 5.65, 0},
    {"k64x160x16_wk4_bf16x2_tri_bpre", 7.2, 0.561, 0.597, 5.11, 18.8, 3.01, 0.738, 4.98, 0.181},
    {"t64x64x64_w2x2x1_d3_bf16x2_tri_bpre", 4.84, 0.42, 0.155, 0.696, 60, 1.04, 0.515, 7.64, 0.667},
    {"t64x160x64_w2x1x2_d2_bf16x2_tri_bpre", 7.56, 0.676, 0.654, 2.64, 11.4, 2.59, 0.847, 6.02, 1.9},
    {"t64x256x32_w1x4x1_d3_bf16x2_tri_bpre", 7.06, 0.989, 1.13, 1.76, 60, 2.59, 1.29, 5.41, 2.23},
    {"t128x128x64_w2x2x1_d2_bf16x2_tri_bpre", 8.38, 0.911, 1.17, 1.53, 11.9, 3.15, 1.25, 4.85, 2.13},
    {"t128x160x32_w2x1x2_d3_bf16x2_tri_bpre", 8.7, 1.09, 1.2, 2.33, 6.04, 2.66, 1.48, 4.52, 5.43},
    {"t256x128x32_w4x1x1_d2_bf16x2_tri_bpre", 8.58, 1.54, 1.81, 3.81, 13.7, 2.3, 2.26, 4.32, 3.23},
    {"t256x160x32_w4x1x1_d2_bf16x2_tri_bpre", 9.46, 1.98, 2.55, 1.51, 9.49, 4.62, 2.69, 4.44, 8.45},
    {"t256x128x32_w512_narrow_bf16x2_tri_bpre", 8.82, 1.83, 2.08, 5.36, 5.45, 4.23, 2.57, 4.58, 0.358},
    {"t256x192x32_w512_narrow_bf16x2_tri_bpre", 11.6, 2.25, 2.83, 6.84, 5.08, 4.16, 3.5, 4.59, 0.0827},
    {"t256x256x32_w512_edge_bf16x2_tri_bpre", 11.4, 2.77, 4.31, 9.8, 14.7, 3.83, 4.45, 3.63, 0.921},
    {"t256x320x32_w512_edge_bf16x2_tri_bpre", 12, 3.27, 5.17, 11, 22.9, 2.97, 5.43, 0.301, 2.16},
    {"t256x320x32_w512_bf16x2_tri_bpre", 11.9, 3.24, 5.12, 10.9, 22.9, 2.97, 5.38, 0.298, 0},
};
// Gated calls on prepared weights (N: the projection's width; 1096 shapes, fitted in the same way: 0.2 - 0.7 % behind the fastest on average, 5 % in one of
// twenty; with the eight-wave tiles priced by the plain products' constants and the others by the ones above 1.5 and 9 %: 893 x 320 x 2240 16.6 us,
// 12.3 on 64 x 64 tiles; 4736 x 4256 x 256 84 and 73)
static const CallCost kGatedCost[] = {
    {"t16x64x32_wavek_bf16x2_tri_bpre", 2.56, 0.634, 0.372, 0.75, 19.8, 1, 0.976, 0.0835, 0},
    {"t32x64x32_wavek_bf16x2_tri_bpre", 2.89, 0.876, 0.596, 0.944, 60, 1, 1.38, 0, 0},
    {"t64x64x32_wavek_bf16x2_tri_bpre", 4.74, 0.71, 1.13, 1.92, 60, 1.12, 2.1, 0.426, 0},
    {"t64x256x32_w1x4x1_d3_bf16x2_tri_bpre", 7.36, 0.951, 0.377, 0.872, 60, 1.26, 1.32, 5.89, 2.34},
    {"t128x128x64_w2x2x1_d2_bf16x2_tri_bpre", 8.87, 0.909, 1.03, 0.863, 18.9, 3.8, 1.29, 5.41, 2.07},
    {"t256x128x32_w4x1x1_d2_bf16x2_tri_bpre", 9.06, 1.51, 1.84, 2.77, 60, 2.29, 2.4, 4.47, 4.59},
    {"t256x128x32_w512_narrow_bf16x2_tri_bpre", 9.33, 1.72, 1.89, 6.09, 60, 2.35, 2.47, 4.94, 0},
    {"t256x256x32_w512_edge_bf16x2_tri_bpre", 13.4, 2.63, 3.27, 8.56, 5.22, 2.67, 4.26, 3.78, 0.127},
    {"t256x320x32_w512_edge_bf16x2_tri_bpre", 16.2, 3.08, 4.34, 10, 60, 2.08, 5.34, 3.48, 1.52},
    {"t256x320x32_w512_bf16x2_tri_bpre", 16, 3.05, 4.3, 9.9, 60, 2.08, 5.29, 3.44, 0},
};
// What the selection functions, and with them the limits of cascmm_gemm_noalloc, price the two tiles of KIND_WAVEK by that they know
static const CallCost kShapeCost[] = {
    {"t32x32x32_wavek_bf16x2_tri", 1.98, 1, 1.02, 0.468, 37.6, 2.39, 1.23, 0, 0},
    {"t32x64x32_wavek_bf16x2_tri", 2.68, 1.22, 0.589, 0.662, 40, 1.12, 1.77, 0, 0},
};
static const std::vector<VariantInfo>& variant_info() {
  static const std::vector<VariantInfo> info = [] {
    std::vector<VariantInfo> v;
    for (const VariantDesc& d : table()) {
      VariantInfo i{nullptr, nullptr, nullptr, nullptr, strstr(d.name, "_p8_") != nullptr, d.name[0] == 'b' && d.name[1] == 'd'};
      for (const TunedCost& t : kTuned)
        if (strcmp(t.name, d.name) == 0) i.tuned = &t;
      for (const CallCost& t : kCallCost)
        if (strcmp(t.name, d.name) == 0) i.call = &t;
      for (const CallCost& t : kGatedCost)
        if (strcmp(t.name, d.name) == 0) i.gated = &t;
      for (const CallCost& t : kShapeCost)
        if (strcmp(t.name, d.name) == 0) i.shape = &t;
      v.push_back(i);
    }
    return v;
  }();
  return info;
}
static double call_estimate_us(const CallCost& t, const VariantDesc& v, const Problem& q, int count, double tiles, int64_t k_per) {
  const double k = v.kind == KIND_WAVEK || v.kind == KIND_HWK ? (double)(((k_per + v.BK - 1) / v.BK + 7) / 8) : v.kind == KIND_SLOTK ? (double)((k_per + 255) / 256 * 4) : (double)k_per / 64.0;
  const double per = tiles / kNumCUs, mb = (double)count * (double)q.K * (double)(q.call ? q.M + q.N : q.N) * (double)dtype_size(q.dtype) * 1.0e-6;
  const double few = v.kind == KIND_HWK ? kHwkStraight : wavek_straight(v.BM * v.BN);
  const double full = std::ceil(per) - 1.0, fill = per - full;
  const bool small = v.kind == KIND_WAVEK || v.kind == KIND_HWK;
  const double lone = k * t.s0 + (small && k > few ? t.deep * (k - few) : 0.0), shared = fill * k * t.s1 + mb / t.bw;
  const double us = t.c0 + full * (t.c1 + k * t.r1) + std::pow(std::pow(lone, t.x) + std::pow(shared, t.x), 1.0 / t.x);
  if (small) {
    const double late = v.kind != KIND_WAVEK || !q.call || q.glu ? 1.0
                        : count > 1 ? (v.BM * v.BN == 4096 ? 0.92 : 0.95)
                        : (full > 0 ? 1.07 : 1.0) * ((double)q.M * (double)q.K > 5.0e6 ? 1.25 : (double)q.M * (double)q.K > 1.25e6 ? 1.1 : 1.0);
    return late * (q.N % v.BN != 0 ? us * (1.0 + t.edge) : us);
  }
  // (The gated 256 x 128 tile with producer waves: a wave's rows over the edge are stored one by one, which few of them do quickly: 1289 x 576 x
  // 4608 28.1 us, 29.5 on the large tile of 128 columns; 3087 x 384 x 2304 22.3, 24.2.  The smaller tiles with less of an edge lost 14 - 22 % to
  // the eight-wave ones: 530 x 832 x 3200, 295 x 1088 x 6528)
  const double rows_over = q.glu && v.kind == KIND_TILE && v.BM == 256 && q.N % v.BN == 0 ? std::min(1.0, (double)(q.M % v.BM) / 64.0) : 1.0;
  const double edged = q.N % v.BN != 0 || q.M % v.BM != 0 ? us + t.edge * rows_over * (full + 1.0) : us;
  const double power = t.deep * tiles * v.BM * v.BN * (double)k_per * 1.0e-9;
  // (the large tiles of 192 and 128 columns, prepared: with a margin; without one 3072^3 took 153 us on 192, 138 on 256 x 160)
  const double margin = count > 1 && q.bpre && v.BM == 64 && v.BN == 160 ? 1.08 : q.bpre && v.kind == KIND_W512E && v.call_only ? 1.03 : 1.0;
  return std::pow(std::pow(edged, 8.0) + std::pow(power, 8.0), 0.125) * margin;
}
static bool wavek_eligible(const Problem& q) {
  return q.dtype == CASCMM_DT_F32 && q.fmt == CASCMM_FMT_BF16 && q.terms == 2 && q.products == CASCMM_PROD_TRI && !q.bpre &&
         !q.glu && q.K > 0 && !beyond_i32(q.M, q.lda, 4);
}
// a call whose kernels all have such constants
static bool costed_call(const Problem& q) {
  return q.call && q.dtype == CASCMM_DT_F32 && q.fmt == CASCMM_FMT_BF16 && q.terms == 2 && q.products == CASCMM_PROD_TRI && (!q.glu || q.bpre);
}
static double wavek_estimate_us(const Problem& q, int count) {
  double best = 1e9;
  for (size_t i = 0; i < table().size(); ++i) {
    const VariantDesc& v = table()[i];
    const VariantInfo& info = variant_info()[i];
    if (v.kind != KIND_WAVEK || v.bpre || !(q.call ? info.call : info.shape)) continue;
    best = std::min(best, call_estimate_us(q.call ? *info.call : *info.shape, v, q, count, (double)count * (double)((q.M + v.BM - 1) / v.BM) * (double)((q.N + v.BN - 1) / v.BN), q.K));
  }
  return best;
}
// The skinny split-K path for comparison (its 32-row variant, the one preferred among them): two
// launches, a workgroup's (32 + 128) x K / splits x 4 bytes at 70 bytes per ns, the partial results
// written and read back at about 4 TB/s (fitted on the same shapes).
static double skinny_estimate_us(const Problem& q) {
  const int sp = skinny_splits(q.M, q.N, q.K, 32, 128, 64);
  return 8.5 + 160.0 * (double)(q.K / sp) * 4.0 / 70.0e3 + 2.0 * sp * (double)q.M * (double)q.N * 4.0 / 4.0e6;
}

// The 16-bit kernels (KIND_H16).  A workgroup's k costs s1 with every CU at work (L2 or the board's power is shared)
// and s0 with few; a round of 256 tiles adds `end` for its store, a launch `start`.  raw: the factor on k of a right
// operand that the LDS transposes.  Measured on the Linear shapes of a UNet and on squares (graph replay, every tile
// forced in turn), before the two tiles of 32-k stages loaded pairs of them: those run in 0.83 - 1.00 of what is said here, in pairs of 32 k, and
// are left out now and then.  Looked at again with every kernel forced on 600 shapes: the one chosen is 0.3 - 1.2 % behind the fastest on average (raw,
// few rows 1.8), 2 - 6 % in one of twenty (16); with k rounded to the pairs' 64 here two choices changed, both for the worse.
struct H16Cost { int BM, BN; double s0, s1, start, end, raw; };
static const H16Cost kH16Cost[] = {
    {256, 320, 0.0205, 0.0315, 3.8, 8.0, 1.06}, {256, 256, 0.0175, 0.0255, 4.0, 6.5, 1.03}, {128, 256, 0.0090, 0.0138, 3.5, 3.5, 1.04},
    {128, 160, 0.0058, 0.0092, 3.5, 2.4, 1.17}, {128, 128, 0.0056, 0.0077, 3.3, 1.8, 1.16}, {64, 160, 0.0047, 0.0053, 3.7, 2.7, 1.10},
    {64, 128, 0.0042, 0.0046, 3.3, 1.1, 1.06},  {128, 64, 0.0044, 0.0050, 3.5, 1.1, 1.02},  {64, 64, 0.0026, 0.0033, 3.2, 1.0, 1.20},
};
static double h16_estimate_us(const VariantDesc& v, const Problem& q, double tiles, int64_t k_per) {
  for (const H16Cost& c : kH16Cost)
    if (c.BM == v.BM && c.BN == v.BN) {
      const double full = (double)(int64_t)(tiles / kNumCUs), rem = tiles / kNumCUs - full;
      const double last = rem > 0 ? (c.s1 * rem > c.s0 ? c.s1 * rem : c.s0) : 0.0;
      const double k = (double)((k_per + v.BK - 1) / v.BK * v.BK) * (q.bpre ? 1.0 : c.raw);
      return c.start + (full + (rem > 0 ? 1.0 : 0.0)) * c.end + k * (full * c.s1 + last);
    }
  return 1e9;
}

// The same problems with K over eight waves (KIND_HWK), with a launch's constants of kCallCost (`form`: 0 prepared, 1 raw, 2 gated).
// Fitted as those to 642 prepared and 383 raw shapes of 2 - 2048 rows (fp16), and 262 gated ones.  They win where the tiles about fit the CUs at once
// (2 x 1280 x 1280 prepared 3.2 us, 6.9 on the four-wave kernels; 154 x 2048 x 1280 5.6, 10.3), and lose behind that, where every tile pays its launch and
// its meeting in LDS (2048 x 640 x 640 raw 12.0 us, 7.3).  The estimates decide; raw weights deeper than the straight
// code's four steps a wave stay with the four-wave kernels (10 x 2496 x 760 6.4 us, here 7.4).  The kernel chosen is 0.3 % (prepared) and 0.6 % (raw) behind the
// fastest of all on average, 2.0 and 3.9 % in one of twenty; prepared 1.2 and 9.0 % with the small tiles priced without rounds
// (41 x 4000 x 1624: 104 tiles of 32 x 32 9.2 us, 153 of 16 x 32 8.0; 8.5 on the four-wave kernels).  64 x 64 tiles
// gained only with the gated store (plain, by index only: 976 x 2048 x 640 9.1 us on the four-wave kernels, 10.6 on them).
struct HwkCost { int BM, BN, form; CallCost c; };
static const HwkCost kHwkCost[] = {
    {16, 16, 0, {nullptr, 3.13, 0.0911, 0.117, 0.239, 19.1, 1, 0.286, 0.237, 0}},
    {16, 32, 0, {nullptr, 3.04, 0.221, 0.18, 0.249, 18.8, 1, 0.409, 0.294, 0}},
    {16, 64, 0, {nullptr, 3.07, 0.471, 0.246, 0.59, 19.2, 1, 0.831, 0.444, 0}},
    {32, 32, 0, {nullptr, 3.16, 0.344, 0.328, 1.06, 33.6, 1, 0.75, 0.215, 0}},
    {32, 64, 0, {nullptr, 3.22, 0.608, 0.561, 1.44, 43.3, 1, 1.07, 0.3, 0}},
    {16, 32, 1, {nullptr, 2.99, 0.459, 0.308, 0.135, 17.3, 1.23, 0.679, 0.614, 0}},
    {16, 64, 1, {nullptr, 3.04, 0.843, 0.221, 0.966, 23.6, 1, 1.18, 0.607, 0}},
    {32, 32, 1, {nullptr, 3.1, 0.52, 0.535, 0.895, 30.1, 1.2, 1.03, 0.561, 0}},
    {32, 64, 1, {nullptr, 3.25, 0.935, 0.471, 1.38, 27.2, 1, 1.36, 0.509, 0}},
    {16, 64, 2, {nullptr, 3.32, 0.463, 0.236, 0.562, 16.3, 1, 0.778, 0.427, 0}},
    {32, 64, 2, {nullptr, 3.53, 0.594, 0.474, 1.27, 33.8, 1, 1.23, 0.353, 0}},
    {64, 64, 2, {nullptr, 3.84, 0.862, 0.823, 1.92, 60, 1, 1.61, 0.195, 0}},
};
static double hwk_estimate_us(const VariantDesc& v, const Problem& q, int count, double tiles) {
  if (!q.bpre && q.K > 2048) return 1e9;
  for (const HwkCost& t : kHwkCost)
    if (t.BM == v.BM && t.BN == v.BN && t.form == (q.glu ? 2 : q.bpre ? 0 : 1)) return call_estimate_us(t.c, v, q, count, tiles, q.K);
  return 1e9;
}

// The K-over-waves kernels (KIND_SLOTK): whole trips of four stages per wave, K in steps of 256; tiles over the edge of C
// were 3 - 9 % slower than their whole neighbours (320 x 956 x 1792, 800 x 896 x 2688); over several rounds of
// raw operands that is lost in the rest (2500^3 119 us, 131 on the tile it would leave it to), not with the weight prepared
// (3000 x 2048 x 2048 85 us, 78 there).
static double slotk_estimate_us(const TunedCost& t, const VariantDesc& v, const Problem& q, double tiles, int64_t k_per) {
  const double full = (double)(int64_t)(tiles / kNumCUs), rem = tiles - full * kNumCUs;
  const double tail = full == 0 ? t.tail_first : t.tail_later;
  const double rounds = full + (rem > 0 ? tail + (1.0 - tail) * rem / kNumCUs : 0.0);
  const double edge = (full == 0 || q.bpre) && (q.N % v.BN != 0 || q.M % v.BM != 0) ? 1.05 : 1.0;
  return edge * rounds * ((double)((k_per + 255) / 256 * 256) / 64.0 * t.step64_us + t.fixed_us);
}

// The large tiles on prepared weights.  A round of a few tiles takes a us per 64 k and b; one that fills the chip A and B, for the
// clock that the board's power leaves; in between by the cube of what is filled, and a round behind another starts c earlier.  Fitted
// to 128 shapes each of 64 - 8192 rows, K and widths from 320 (gated: 66 and 44), within 5 %: 256 x 256, us: 4928 x 384 x 1152 29.4, 6976 x
// 320 x 960 26.2, 4096^3 300; gated 1709 x 448 x 3584 33.6, 1500 x 1280 x 10240 99.4.  (With a partly filled round as 0.45 of a full one
// and a share of the rest the small ones were priced at 18 - 26 us and came here from tiles that run them in 20 - 25: 3072 x 576 x
// 1728 36 us, 25 on 256 x 128; 4928 x 384 x 1152 28, 22.  Raw weights keep that rule: the other tiles' entries for them lie as far off.)
struct LargeTileCost { int BN; bool glu; double a, b, A, B, c; };
static const LargeTileCost kLargeTileCost[] = {
    {256, false, 2.845, 10.34, 4.415, 12.13, 3.0}, {320, false, 3.438, 12.08, 5.382, 13.81, 3.7},
    {256, true, 2.830, 12.33, 4.507, 13.15, 6.0},  {320, true, 3.470, 16.43, 5.254, 18.72, 6.6},
};
static double large_tile_us(const VariantDesc& v, const Problem& q, double tiles) {
  for (const LargeTileCost& t : kLargeTileCost)
    if (t.BN == v.BN && t.glu == q.glu) {
      const double k = (double)((q.K + 31) / 32) * 0.5, full = (double)(int64_t)(tiles / kNumCUs), part = tiles / kNumCUs - full;
      const double few = t.a * k + t.b, all = t.A * k + t.B;
      const double us = full * all + (part > 0 ? few - (full > 0 ? t.c : 0.0) + part * part * part * (all - few) : 0.0);
      return v.kind == KIND_W512 ? 0.99 * us : us;   // (whole tiles: no test per load of A)
    }
  return 1e9;
}

// K split over workgroups (cascmm_ksplit.h): where the tiles leave CUs idle, `estimate(tiles, k of a split)` with the
// chip filled against the second launch and the partial results, written and read back.  Measured (graph replay): 7 x 3264 x 880
// fp16 14.8 -> 6.2 us in thirteen splits, 256 x 5120 x 1280 23.0 -> 14.0 in six, 34 x 2008 x 2176 fp32 prepared 15.5 -> 9.5 in
// eight, 154 x 2048 x 2560 raw 18.4 -> 15.6 in four.  Below 11 us the second launch, 3 us of the
// host's time, costs an eager call more than it gives (keys and values 40 x 1664 x 768 fp16 8.4 -> 11.5 us).
template <class F>
static double ksplit_best(const Problem& q, int count, double tiles, size_t ws_bytes, double launch_us, double bytes_per_us, int* splits, F estimate) {
  double best = estimate(tiles, q.K);
  *splits = 1;
  if (count != 1 || q.glu || q.whole_k || best < 11.0) return best;
  for (int sp = 2; sp <= kMaxKSplits && tiles * sp <= kNumCUs; ++sp) {
    if (!ksplit_valid(q.K, sp) || ksplit_bytes(q.M, q.N, sp) > ws_bytes) continue;
    const double c = estimate(tiles * sp, ksplit_k(q.K, sp)) + launch_us + (double)ksplit_bytes(q.M, q.N, sp) / bytes_per_us;
    if (c < best) { best = c; *splits = sp; }
  }
  return best;
}

// ws_bytes: workspace the caller brought; *splits_out: K split the cost was computed for (the
// LDS-tiled two-term bf16 kernels may split K over up to kMaxTileSplits work items per tile when a
// single problem has too few tiles to occupy the chip and the workspace holds the partials)
static double variant_cost(int vi, const Problem& q, int count, size_t ws_bytes = 0, int* splits_out = nullptr) {
  const VariantDesc& v = table()[vi];
  const VariantInfo& info = variant_info()[vi];
  if (splits_out) *splits_out = 1;
  const double tiles = (double)count * (double)((q.M + v.BM - 1) / v.BM) * (double)((q.N + v.BN - 1) / v.BN);
  const double full = (double)(int64_t)(tiles / kNumCUs);
  const double rem = tiles - full * kNumCUs;
  if (v.kind == KIND_HWK) return hwk_estimate_us(v, q, count, tiles);
  if (v.kind == KIND_SPLITK) {
    if (q.call) return 1e9;   // (the small tiles of KIND_WAVEK and the K-over-waves tiles: 3 x 4416 x 2752 18 us here, 12.1 there)
    // Problems with too few tiles to occupy the chip: splitting K wins whenever the plain tile
    // kernels would leave more than half of the CUs idle; among the split-K variants the
    // smaller row tile was faster wherever both were measured.
    if ((double)((q.M + 63) / 64) * (double)((q.N + 127) / 128) >= kNumCUs / 2) return 1e9;
    // ... unless the one-launch kernel that splits K over its waves is expected to be faster
    const double skinny_us = skinny_estimate_us(q);
    if (wavek_eligible(q) && wavek_estimate_us(q, count) < skinny_us) return 1e9;
    // ... or the K-over-waves tiles, K split over workgroups too (64 x 5120 x 1280: 17.1 us here, 15.2 there)
    for (int i = 0; i < (int)table().size(); ++i)
      if (table()[i].kind == KIND_SLOTK && variant_matches(table()[i], q, FIT_DWORD) && variant_cost(i, q, count, ws_bytes) < skinny_us) return 1e9;
    return 1e-6 * (double)(((q.M + v.BM - 1) / v.BM) * v.BM) + 1e-8 * v.BM;
  }
  const bool costed = costed_call(q);
  const CallCost* c = costed && q.glu ? info.gated : !q.call && info.shape ? info.shape : info.call;
  if (costed && !c && v.fast) return 1e9;   // (nowhere the fastest)
  if (c && (costed || v.kind == KIND_WAVEK)) {
    if (v.kind != KIND_SLOTK) return call_estimate_us(*c, v, q, count, tiles, q.K);
    int ks = 1;
    const double us = ksplit_best(q, count, tiles, ws_bytes, 2.85, 9.0e6, &ks, [&](double n, int64_t k) { return call_estimate_us(*c, v, q, count, n, k); });
    if (splits_out) *splits_out = ks;
    return us;
  }
  if ((v.kind == KIND_W512E || v.kind == KIND_W512) && q.bpre) return large_tile_us(v, q, tiles);
  int ks = 1;
  if (v.kind == KIND_H16 || (v.kind == KIND_SLOTK && info.tuned)) {
    const double us = v.kind == KIND_H16
        // (calls on prepared weights, 255 shapes: 2 x 4928 x 2880 in eleven splits 10.2 us, not the 8.0 of the constants before)
        ? ksplit_best(q, count, tiles, ws_bytes, q.call && q.bpre ? 1.65 : 1.6, q.call && q.bpre ? 1.5e6 : 3.8e6, &ks, [&](double t, int64_t k) { return h16_estimate_us(v, q, t, k); })
        : ksplit_best(q, count, tiles, ws_bytes, 2.8, 12.0e6, &ks, [&](double t, int64_t k) { return slotk_estimate_us(*info.tuned, v, q, t, k); });
    if (splits_out) *splits_out = ks;
    return us;
  }
  if (v.kind == KIND_F8K64) {
    // stages of 64 k at ~2.1 us per resident round, the K split the launcher will use, and the passes
    // around the GEMM: the split of A (and of B unless prepared), the reduction of a K split
    const int sp = f8k64_splits(q.M, q.N, q.K, v.BM);
    const double items = tiles * sp;
    const double rounds_ = items <= kNumCUs ? 1.0 : (double)(int64_t)(items / kNumCUs) + ((int64_t)items % kNumCUs ? 0.8 : 0.0);
    // (the 64-row tile splits K over the four waves of its workgroup: a quarter of the stages per wave, in pairs,
    // and rounds of one tile per CU that do not overlap)
    const double gemm_us = v.BM == F8WK::BM ? rounds_ * ((double)((q.K / 64 + 7) / 8 * 2) * kF8WKStageUs + kF8WKFixedUs)
                                            : rounds_ * ((double)(q.K / 64 / sp) * f8k64_stage_us(v.BM) + (v.BM == 256 ? 6.0 : 4.0));
    double us = gemm_us + 6.0 + (double)q.M * q.K * 7.0 / 4.0e6;
    if (!q.bpre) us += 3.0 + (double)q.K * q.N * 7.0 / 4.0e6;
    if (sp > 1) us += 3.0 + (double)(sp + 1) * q.M * q.N * 4.0 / 4.0e6;
    return us;
  }
  if (v.kind == KIND_F16K) {
    // Stages of 32 k (the K-over-waves kernel: a wave's own stages, in pairs) at the measured 3.0 / 2.45 us with 10 / 8 us
    // per round beside them (fit: 2048 x {1280, 5120} x 1280, 2048 x 1280 x {3840, 10240}, 8192 x 640 x 5120), and the
    // two passes around the GEMM: both operands read twice and written once as slots, 14 bytes per element at 5.7 TB/s.
    const double rounds_ = tiles <= kNumCUs ? 1.0 : (double)(int64_t)(tiles / kNumCUs) + ((int64_t)tiles % kNumCUs ? 0.8 : 0.0);
    const double gemm_us = v.BM == F16WK::BM ? rounds_ * ((double)((q.K / 32 + 7) / 8 * 2) * 3.0 + 10.0)
                                             : rounds_ * ((double)(q.K / 32) * 2.45 + 8.0);
    return gemm_us + 4.0 + ((double)q.M * q.K + (double)q.K * q.N) * 14.0 / 5.7e6;
  }
  if (info.tuned) {
    const TunedCost& t = *info.tuned;
    const double tail = full == 0 ? t.tail_first : t.tail_later;
    const double rounds = full + (rem > 0 ? tail + (1.0 - tail) * rem / kNumCUs : 0.0);
    // tiles that hang over the edge of C take the bounds-checked epilogue and load clamped
    // columns: measured about a quarter slower (32768 x 640 x 320 on the 128-wide tile)
    const double edge = v.kind != KIND_W512E && (q.N % v.BN != 0 || q.M % v.BM != 0) ? 1.25 : 1.0;
    double best = edge * rounds * ((double)q.K / 64.0 * t.step64_us + t.fixed_us);
    if (v.kind == KIND_TILE && count == 1 && q.dtype == CASCMM_DT_F32 && q.N % 4 == 0 && full == 0 && !q.glu) {
      const int64_t ksteps = (q.K + v.BK - 1) / v.BK;
      for (int sp = 2; sp <= kMaxTileSplits; ++sp) {
        if (ksteps % sp != 0 || ksteps / sp < 4 || tiles * sp > kNumCUs) continue;
        if (ws_bytes < (size_t)sp * q.M * q.N * sizeof(float)) continue;
        const double r = t.tail_first + (1.0 - t.tail_first) * tiles * sp / kNumCUs;
        // the second pass: a launch plus writing and reading the partial results at about 4 TB/s
        const double reduce_us = 2.0 + (double)(sp + 1) * q.M * q.N * 4.0 / 4.0e6;
        const double c = edge * r * ((double)q.K / sp / 64.0 * t.step64_us + t.fixed_us) + reduce_us;
        if (c < best) {
          best = c;
          if (splits_out) *splits_out = sp;
        }
      }
    }
    return best;
  }
  const double rounds = full + (rem > 0 ? 0.55 + 0.45 * rem / kNumCUs : 0.0);
  double step = ((double)v.BM * v.BN + 64.0 * (v.BM + v.BN)) / 20000.0;
  if (info.p8) step *= 0.94;
  const double ksteps = (double)((q.K + 63) / 64);
  // the plain B-direct kernels were slower than the LDS-tiled ones on every shape measured:
  // they stay selectable by index only
  if (info.bdirect) return 1e6 + rounds * step * ksteps;
  double best = rounds * (step * ksteps + 5.0) + (v.fast ? 0.0 : 1e3);
  // the same K split as above for the kernels without measured constants (three-term and fp8
  // cascades on the shapes that leave CUs idle)
  if (v.fast && count == 1 && q.dtype == CASCMM_DT_F32 && q.N % 4 == 0 && full == 0 && !q.glu && !q.bpre) {
    const int64_t bk_steps = (q.K + v.BK - 1) / v.BK;
    for (int sp = 2; sp <= kMaxTileSplits; ++sp) {
      if (bk_steps % sp != 0 || bk_steps / sp < 4 || tiles * sp > kNumCUs) continue;
      if (ws_bytes < (size_t)sp * q.M * q.N * sizeof(float)) continue;
      const double r = 0.55 + 0.45 * tiles * sp / kNumCUs;
      const double reduce_us = 2.0 + (double)(sp + 1) * q.M * q.N * 4.0 / 4.0e6;
      const double c = r * (step * ksteps / sp + 5.0) + reduce_us;
      if (c < best) {
        best = c;
        if (splits_out) *splits_out = sp;
      }
    }
  }
  return best;
}

// Three terms on K over eight waves, by the tiles of 32 x 32 (graph replay, 150 shapes of 2 - 1500 rows each).
// fp16: only in the place of the tile kernels, which split the operands as they are too (the slot kernels scale both first and so take
// values beyond fp16's range: of their calls the tiles that scale themselves take some, see select_scaled_rows), up to two tiles per CU, of deep K up to one, and up to three where the other kernel is
// the bounds-checked one.  0.47 of the tile kernels' time (2 x 1280 x 1280 12.8 us, here 6.1; 38 x 256 x 448 9.9, 3.3; 222 x 4352 x 704 32.9,
// 28.6; 788 x 659 x 818 bounds-checked 35.0, 23.0), 2 % behind the fastest of all; beyond: 391 x 384 x 1984 13.6, here 16.7; 96 x 2048 x 8192
// 41.0, 45.3 (eager); 1136 x 3200 x 256 42.8, 44.9.
// fp8: in the place of the slot kernels too (all scale by the same exponents), whose passes it does without, up to one tile per CU: 0.56 of the
// time (2 x 1280 x 1280 11.7, here 6.3; 18 x 2688 x 384 20.4, 10.3), for 16 rows up to 400 tiles (2 x 320 x 10240 14.8, 10.9; 16 x 1280 x 12800
// 32.7, 23.6); beyond, the fp8-rate instruction wins: 391 x 384 x 1984 11.8, here 17.3; 222 x 4352 x 704 27.4, 28.1.  Deep K, of few tiles: 4 x
// 4372 x 1728 50.4, 21.6; 8 x 8192 x 2048 48.0, 31.3; 40 x 6144 x 1280 39.7, 27.9; but 154 x 10240 x 640 43.5, here 52.1; 20 x 20480 x 1280 74.6,
// 84.6; 64 x 8192 x 2560 49.6, 56.2.
static bool wavek_three_terms(const VariantDesc& v) { return v.kind == KIND_WAVEK && v.terms == 3; }
static bool few_tiles_three_terms(const Problem& q, int count, bool bounds_checked) {
  const int64_t tiles = (int64_t)count * ((q.M + 31) / 32) * ((q.N + 31) / 32);
  if (q.fmt == CASCMM_FMT_FP8) return q.K > 4096 ? tiles <= 640 * 1024 / q.K : tiles <= (q.M <= 16 ? 400 : kNumCUs);
  return tiles <= (bounds_checked ? 3 : q.K <= 2048 ? 2 : 1) * kNumCUs;
}

// ws_bytes: workspace the caller brought (split-K variants that need more are skipped)
// The selection walks the whole table and costs every candidate; a model calls the same few dozen
// problems over and over (eagerly, ~750 Linear calls per UNet step), so the answers are remembered.
struct SelectKey {
  int64_t M, N, K;
  size_t ws_bytes;
  // flags: bpre << 1 | glu << 2, what variant_matches reads of the leading dimensions (the 32-bit addressing limits of
  // some kernels: M lda, K ldb, 1024 ldc and 256 ldc beyond 2^31 bytes << 3, 4, 5, 15; lda below 32 << 7), glu_slots << 6,
  // chunked << 8, split_first << 9, the fit of the rows << 10, whole_k << 12, K ldb as the kernels state it with
  // stages past K, of four-byte and two-byte elements << 13, 14, call << 16
  int dtype, fmt, terms, products, count, flags;
  bool operator==(const SelectKey& o) const {
    return M == o.M && N == o.N && K == o.K && ws_bytes == o.ws_bytes && dtype == o.dtype && fmt == o.fmt &&
           terms == o.terms && products == o.products && count == o.count && flags == o.flags;
  }
};
struct SelectKeyHash {
  size_t operator()(const SelectKey& k) const {
    uint64_t h = 1469598103934665603ull;
    auto mix = [&](uint64_t v) { h = (h ^ v) * 1099511628211ull; };
    mix((uint64_t)k.M); mix((uint64_t)k.N); mix((uint64_t)k.K); mix((uint64_t)k.ws_bytes);
    mix(((uint64_t)k.dtype << 40) ^ ((uint64_t)k.fmt << 32) ^ ((uint64_t)k.terms << 24) ^ ((uint64_t)k.products << 16) ^
        ((uint64_t)k.count << 8) ^ (uint64_t)k.flags);
    return (size_t)h;
  }
};
struct SelectHit { int variant, splits; };

static int select_variant_uncached(const Problem& q, RowFit fit, int count, size_t ws_bytes, int* splits_out);

static int select_variant(const Problem& q, RowFit fit, int count, size_t ws_bytes = (size_t)-1,
                          int* splits_out = nullptr) {
  static std::mutex mu;
  static std::unordered_map<SelectKey, SelectHit, SelectKeyHash> memo;
  const SelectKey key{q.M, q.N, q.K, ws_bytes, q.dtype, q.fmt, q.terms, q.products, count,
                      (q.lda < 32 ? 128 : 0) | (q.chunked ? 256 : 0) | (q.split_first ? 512 : 0) | ((int)fit << 10) | (q.whole_k ? 4096 : 0) | (q.call ? 65536 : 0) | (q.bpre ? 2 : 0) | (q.glu ? 4 : 0) | (q.glu_slots ? 64 : 0) | (beyond_i32(q.M, q.lda, 4) ? 8 : 0) |
                          (beyond_i32(q.K, q.ldb, 4) ? 16 : 0) | (beyond_i32(q.ldc, 1024, 1) ? 32 : 0) | (beyond_i32(q.ldc, 256, 1) ? 32768 : 0) | (beyond_i32(q.K + 32, q.ldb, 4) ? 8192 : 0) |
                          (beyond_i32(q.K + 64, q.ldb, 2) ? 16384 : 0)};
  {
    std::lock_guard<std::mutex> lock(mu);
    auto it = memo.find(key);
    if (it != memo.end()) {
      if (splits_out) *splits_out = it->second.splits;
      return it->second.variant;
    }
  }
  int splits = 1;
  const int v = select_variant_uncached(q, fit, count, ws_bytes, &splits);
  {
    std::lock_guard<std::mutex> lock(mu);
    if (memo.size() >= 4096) memo.clear();
    memo[key] = SelectHit{v, splits};
  }
  if (splits_out) *splits_out = splits;
  return v;
}

static int select_variant_uncached(const Problem& q, RowFit fit, int count, size_t ws_bytes, int* splits_out) {
  const auto& t = table();
  int best = -1;
  double best_cost = 0;
  if (splits_out) *splits_out = 1;
  for (int i = 0; i < (int)t.size(); ++i) {
    if (wavek_three_terms(t[i]) || !variant_matches(t[i], q, fit)) continue;
    if (count > 1 && !t[i].grouped) continue;
    if (t[i].kind == KIND_SPLITK &&
        skinny_workspace_bytes(q.M, q.N, q.K, t[i].BM, t[i].BN, t[i].BK) > ws_bytes)
      continue;
    if (t[i].kind == KIND_F8K64 && f8k64_workspace_bytes(q.M, q.N, q.K, q.bpre, t[i].BM) > ws_bytes) continue;
    if (t[i].kind == KIND_F16K && f16k_workspace_bytes(q.M, q.N, q.K) > ws_bytes) continue;
    int sp = 1;
    const double c = variant_cost(i, q, count, ws_bytes, &sp);
    if (best < 0 || c < best_cost) {
      best = i;
      best_cost = c;
      if (splits_out) *splits_out = sp;
    }
  }
  if (best >= 0 && (t[best].kind == KIND_TILE || t[best].kind == KIND_F8K64) && few_tiles_three_terms(q, count, !t[best].fast)) {
    best_cost = 1e9;
    for (int i = 0; i < (int)t.size(); ++i) {
      if (!wavek_three_terms(t[i]) || t[i].scaled || !variant_matches(t[i], q, fit) || variant_cost(i, q, count) >= best_cost) continue;
      best = i;
      best_cost = variant_cost(i, q, count);
      if (splits_out) *splits_out = 1;
    }
  }
  // A group in one launch has fewer kernels to choose from than its problems one behind the other (the large tiles on prepared weights with K off 32, K over
  // four waves): 3 x (2592 x 552 x 3840) prepared 238 us in one launch, 126 in three.  From 10 us a problem on: an eager launch is 3 us of the
  // host's time.  (No kernel: the launch then takes the problems one by one.)
  if (best >= 0 && count > 1 && costed_call(q)) {
    const int one = select_variant_uncached(q, fit, 1, ws_bytes, nullptr);
    const double us = one < 0 ? 1e9 : variant_cost(one, q, 1, ws_bytes);
    if (us >= 10.0 && 1.03 * count * us < best_cost) return CASCMM_ERR_BAD_FORMAT;
  }
  return best < 0 ? (int)CASCMM_ERR_BAD_FORMAT : best;
}
// what such a call is expected to take
static double call_cost_us(const Problem& q, RowFit fit, int count) {
  const int v = select_variant(q, fit, count), one = v < 0 && count > 1 ? select_variant(q, fit, 1) : -1;
  return v >= 0 ? variant_cost(v, q, count) : one >= 0 ? count * variant_cost(one, q, 1) : 1e9;
}

// ---------------------------------------------------------------------------------------
// utility kernels
// ---------------------------------------------------------------------------------------
template <int IODT>
__global__ void fill_bias_kernel(void* C, const void* bias, int M, int N, int64_t ldc) {
  typedef typename IoType<IODT>::T T;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)M * N) return;
  const int r = (int)(i / N), c = (int)(i % N);
  IoType<IODT>::store((T*)C + (int64_t)r * ldc + c, bias ? IoType<IODT>::load((const T*)bias + c) : 0.f);
}

// fp8 tensor scale, three stream-ordered steps on the caller's int32: zero it, fold in the bit
// pattern of max|x| (non-negative floats order like their bit patterns), turn it into the
// exponent e with max|x| * 2^e in (224, 448]
__global__ void amax_begin_kernel(int32_t* exp_out) { *exp_out = 0; }

template <int IODT>
__global__ __launch_bounds__(256) void amax_kernel(const void* x, int64_t rows, int64_t cols, int64_t ld, int32_t* exp_out) {
  const unsigned best = amax_scan<IODT>(x, rows, cols, ld);
  if ((threadIdx.x & 63) == 0 && best != 0) atomicMax((unsigned*)exp_out, best);
}

__global__ void amax_end_kernel(int32_t* exp_out) { *exp_out = exp_of_amax((unsigned)*exp_out); }

// The same search in ONE launch.  scratch = {running max, arrival count}, both zero on entry: every
// workgroup folds its maximum in, fences, and takes a ticket; the one that draws the last ticket sees
// every other workgroup's contribution, writes {e_x, *second} and leaves the scratch zeroed for the
// next call.  No workgroup waits for another.
template <int IODT>
__global__ __launch_bounds__(1024) void amax_single_launch_kernel(const void* x, int64_t rows, int64_t cols, int64_t ld,
                                                                  const int32_t* second, int32_t* exps_out, unsigned* scratch) {
  __shared__ unsigned wave_best[16];
  const unsigned best = amax_scan<IODT>(x, rows, cols, ld);
  if ((threadIdx.x & 63) == 0) wave_best[threadIdx.x >> 6] = best;
  __syncthreads();
  if (threadIdx.x != 0) return;
  unsigned b = 0;
  for (unsigned w = 0; w < (blockDim.x >> 6); ++w) b = wave_best[w] > b ? wave_best[w] : b;
  // atomics of all workgroups on one word run one after another: skip the one that cannot raise
  // the maximum (the running value only grows within a call, so a stale read errs on the safe side)
  if (b > __hip_atomic_load(&scratch[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(&scratch[0], b);
  __threadfence();
  const unsigned ticket = atomicAdd(&scratch[1], 1u);
  if (ticket != gridDim.x - 1) return;
  __threadfence();
  const unsigned bits = atomicExch(&scratch[0], 0u);
  atomicExch(&scratch[1], 0u);
  exps_out[0] = exp_of_amax(bits);
  if (second) exps_out[1] = *second;
}

template <int IODT, int FMT, int TERMS>
__global__ void split_terms_kernel(const void* x, float* out, int64_t n, int tensor_exp) {
  typedef typename IoType<IODT>::T T;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float r[8];
  r[0] = IoType<IODT>::load((const T*)x + i) * __builtin_ldexpf(1.0f, tensor_exp);
#pragma unroll
  for (int e = 1; e < 8; ++e) r[e] = 0.f;
  u32x4 t[Lowp<FMT>::planes(TERMS)];
  split8<FMT, TERMS>(r, t);
#pragma unroll
  for (int k = 0; k < TERMS; ++k) {
    out[(int64_t)k * n + i] = Lowp<FMT>::element0(t[Lowp<FMT>::plane(k)], k);
  }
}

template <int IODT, int FMT>
static int launch_split(const void* x, float* out, int64_t n, int terms, int tensor_exp, hipStream_t s) {
  const unsigned grid = (unsigned)((n + 255) / 256);
  hipError_t err = hipSuccess;
  switch (terms) {
    case 1: CASCMM_LAUNCH(err, (split_terms_kernel<IODT, FMT, 1>), dim3(grid), dim3(256), 0, s, x, out, n, tensor_exp); break;
    case 2: CASCMM_LAUNCH(err, (split_terms_kernel<IODT, FMT, 2>), dim3(grid), dim3(256), 0, s, x, out, n, tensor_exp); break;
    case 3: CASCMM_LAUNCH(err, (split_terms_kernel<IODT, FMT, 3>), dim3(grid), dim3(256), 0, s, x, out, n, tensor_exp); break;
    default: return CASCMM_ERR_BAD_FORMAT;
  }
  return err == hipSuccess ? CASCMM_OK : CASCMM_ERR_LAUNCH;
}

// Splits a weight once: thread (kg, n) reads the 8 values B[8 kg .. 8 kg + 7][n] (zero beyond K),
// splits them like the GEMM kernels do and writes one 16-byte operand slot per plane to
// out[(plane * K/8 + kg) * N + n].
template <int IODT, int FMT, int TERMS>
__global__ __launch_bounds__(256) void prepare_weight_kernel(const void* B, int K, int N, int64_t ldb,
                                                            const int32_t* tensor_exp, u32x4* out, int flags) {
  typedef typename IoType<IODT>::T T;
  const int glu = flags & 1, chained = flags & 2;
  const int kgs = chained ? K / 8 : (int)prepared_kgroups(K);
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)kgs * N) return;
  const int kg = (int)(i / N), n = (int)(i - (int64_t)kg * N);
  // gated layout: prepared columns alternate 32 value columns (first half of B) and their 32
  // gate columns (second half)
  const int src = glu ? (n >> 6) * 32 + (n & 31) + ((n >> 5) & 1) * (N >> 1) : n;
  float r[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    // chained: the k order of the left operand's slots as the gated store writes them (see
    // cascmm_prepare_left): positions 0..3 are k = 16 t + 4 g + 0..3 and 4..7 the same + 8, kg = 2 t + g
    const int k = chained ? 16 * (kg >> 1) + 8 * (e >> 2) + 4 * (kg & 1) + (e & 3) : kg * 8 + e;
    r[e] = k < K ? IoType<IODT>::load((const T*)B + (int64_t)k * ldb + src) : 0.f;
  }
  constexpr int PL = Lowp<FMT>::planes(TERMS);
  u32x4 t[PL];
  float scale = 1.f;
  if constexpr (Lowp<FMT>::kTensorScaled) {
    if (tensor_exp) scale = __builtin_ldexpf(1.f, *tensor_exp);
  }
  split8<FMT, TERMS>(r, t, scale);
#pragma unroll
  for (int pl = 0; pl < PL; ++pl) out[((int64_t)pl * kgs + kg) * N + n] = t[pl];
}

template <int IODT, int FMT>
static int launch_prepare(const void* B, int K, int N, int64_t ldb, int terms, const int32_t* e, u32x4* out, hipStream_t s,
                          int glu) {
  const int64_t total = ((glu & 2) ? (int64_t)(K / 8) : prepared_kgroups(K)) * N;
  const unsigned grid = (unsigned)((total + 255) / 256);
  hipError_t err = hipSuccess;
  switch (terms) {
    case 1: CASCMM_LAUNCH(err, (prepare_weight_kernel<IODT, FMT, 1>), dim3(grid), dim3(256), 0, s, B, K, N, ldb, e, out, glu); break;
    case 2: CASCMM_LAUNCH(err, (prepare_weight_kernel<IODT, FMT, 2>), dim3(grid), dim3(256), 0, s, B, K, N, ldb, e, out, glu); break;
    case 3: CASCMM_LAUNCH(err, (prepare_weight_kernel<IODT, FMT, 3>), dim3(grid), dim3(256), 0, s, B, K, N, ldb, e, out, glu); break;
    default: return CASCMM_ERR_BAD_FORMAT;
  }
  return err == hipSuccess ? CASCMM_OK : CASCMM_ERR_LAUNCH;
}

template <int IODT>
static int launch_prepare_fmt(const void* B, int K, int N, int64_t ldb, int fmt, int terms, const int32_t* e, u32x4* out,
                              hipStream_t s, int glu) {
  if (fmt == CASCMM_FMT_BF16) return launch_prepare<IODT, CASCMM_FMT_BF16>(B, K, N, ldb, terms, e, out, s, glu);
  if (fmt == CASCMM_FMT_FP16) return launch_prepare<IODT, CASCMM_FMT_FP16>(B, K, N, ldb, terms, e, out, s, glu);
  if (fmt == CASCMM_FMT_FP8) return launch_prepare<IODT, CASCMM_FMT_FP8>(B, K, N, ldb, terms, e, out, s, glu);
  return CASCMM_ERR_BAD_FORMAT;
}

// ---------------------------------------------------------------------------------------
// operands whose rows no fast kernel reads, copied into the workspace first
// ---------------------------------------------------------------------------------------
// Workgroups 0 .. a_blocks - 1: rows of A [M][K] (row stride lda) as rows of a_chunks 16-byte chunks, zeros past K; a
// thread writes one chunk.  The others (16-bit elements as one term of their own format only): B [K][N] as operand
// slots [4 ceil(K/32)][N], a thread the eight k of a column.  E: an unsigned type of the elements' size; bits are moved.
// (chunks are counted in 32 bits: the copies are below 2 GiB)
// A whole chunk of A is one 16-byte load, which wants its address on a dword; of 16-bit rows that start between two, the five dwords that
// hold it, shifted (each of them holds an element of the chunk, so none lies outside the tensor's memory).
// Bound by memory and the launch.  Whole calls, us, before (an element at a time, 64-bit counts) and now: fp16 4305 x 1201 x 1201 33.5, 31.3;
// 4000 x 639 x 640 16.3, 15.0; 2048 x 1279 x 2560 28.6, 27.3; fp32 4000 x 639 x 640 26.9, 26.1.
template <typename E>
__global__ __launch_bounds__(256) void relay_kernel(const E* __restrict__ A, int M, int K, int64_t lda, int a_chunks, u32x4* __restrict__ a_out,
                                                   int a_blocks, const E* __restrict__ B, int N, int64_t ldb, u32x4* __restrict__ b_out) {
  constexpr int PER = 16 / sizeof(E);
  typedef E chunk_t __attribute__((ext_vector_type(PER)));
  typedef unsigned dwords_t __attribute__((ext_vector_type(4), aligned(4)));
  chunk_t c;
  if ((int)blockIdx.x < a_blocks) {
    const unsigned i = blockIdx.x * 256u + threadIdx.x;
    if (i >= (unsigned)M * (unsigned)a_chunks) return;
    const int row = (int)(i / (unsigned)a_chunks), k0 = (int)(i - (unsigned)row * (unsigned)a_chunks) * PER;
    const E* src = A + (int64_t)row * lda + k0;
    if (k0 + PER <= K) {
      const unsigned off = sizeof(E) == 2 ? (unsigned)((uintptr_t)src & 2u) : 0u;
      const unsigned* from = (const unsigned*)((const char*)src - off);
      u32x4 w = *(const dwords_t*)from;
      if (off != 0) {
        const unsigned last = from[4];
        w = (u32x4){__builtin_amdgcn_alignbit(w[1], w[0], 16), __builtin_amdgcn_alignbit(w[2], w[1], 16), __builtin_amdgcn_alignbit(w[3], w[2], 16),
                    __builtin_amdgcn_alignbit(last, w[3], 16)};
      }
      a_out[i] = w;
      return;
    }
#pragma unroll
    for (int e = 0; e < PER; ++e) c[e] = k0 + e < K ? src[e] : (E)0;
    a_out[i] = __builtin_bit_cast(u32x4, c);
  } else {
    const unsigned i = (blockIdx.x - (unsigned)a_blocks) * 256u + threadIdx.x;
    if (i >= (unsigned)prepared_kgroups(K) * (unsigned)N) return;
    const int kg = (int)(i / (unsigned)N), n = (int)(i - (unsigned)kg * (unsigned)N);
#pragma unroll
    for (int e = 0; e < PER; ++e) c[e] = kg * PER + e < K ? B[(int64_t)(kg * PER + e) * ldb + n] : (E)0;
    b_out[i] = __builtin_bit_cast(u32x4, c);
  }
}

// What a problem needs copied before the fast kernels take it (nothing: neither flag), and the bytes of one such copy,
// rounded up to whole 256.  fp32 (two bf16 terms): rows of A whose length is not a multiple of 4; everything else is read
// where it lies.  16-bit: rows of A that are not whole chunks or do not start on dwords, and a raw B of odd N or ldb.
// The bounds-checked kernels, which read element by element, stay for callers without a workspace: 7488 x 1061 x 3192
// fp32 601 us, copied first 248; 37 x 2139 x 6528 fp16 238 against 15; and where nothing is copied, 333 x 456 x 211 18.6
// against 6.4, 44 x 1124 x 1728 42.5 against 8.7.
struct Relay { bool a = false, b = false; size_t a_bytes = 0, b_bytes = 0; int a_chunks = 0; };
// the problem that is left once its operands are copied
static Problem relayed(const Problem& q0, const Relay& r) {
  Problem q = q0;
  if (r.a) q.lda = r.a_chunks * (16 / (int64_t)dtype_size(q.dtype));
  q.chunked = true;
  q.bpre = r.b;
  if (r.b) q.ldb = q.N;
  return q;
}
// where_it_lies: nothing is copied for the kernels that need no copy where they are expected to be faster
static Relay relay_of(const Problem& q0, int count, const void* const* A, const void* const* B, bool where_it_lies = true) {
  Problem q = q0;
  q.call = true;
  Relay r;
  if (q.bpre || q.split_first || q.K == 0) return r;
  const bool f32 = q.dtype == CASCMM_DT_F32;
  if (f32 ? !(q.fmt == CASCMM_FMT_BF16 && q.terms == 2 && (q.products == CASCMM_PROD_TRI)) : !own_format16(q)) return r;
  const int64_t es = f32 ? 4 : 2, per = 16 / es;
  r.a = q.K % per != 0 || (!f32 && q.lda % 2 != 0);
  r.b = !f32 && (q.N % 2 != 0 || q.ldb % 2 != 0);
  for (int i = 0; i < count; ++i) {
    r.a = r.a || (!f32 && A && !aligned_to(A[i], 4));
    r.b = r.b || (!f32 && B && !aligned_to(B[i], 4));
  }
  const int64_t lines = (q.K * es + 127) / 128;   // (rows of whole cache lines)
  int64_t a_bytes = 0, b_bytes = r.b ? prepared_bytes(q.K, q.N, q.fmt, 1) : 0;
  if (__builtin_mul_overflow(q.M, lines * 128, &a_bytes) || a_bytes > INT32_MAX || b_bytes > INT32_MAX) return Relay();
  r.a_chunks = (int)lines * 8;
  r.a_bytes = r.a ? f8k64_up(a_bytes) : 0;
  r.b_bytes = f8k64_up(b_bytes);
  // (small problems have a kernel that reads rows of any length where they lie; the copy is a launch of 4 us: 122 x 2382 x 1480
  // 17.3 us with it)
  if (f32 && r.a && where_it_lies) {
    RowFit fit = FIT_FAST;
    for (int i = 0; i < count; ++i) fit = std::min(fit, row_fit(q, A ? A[i] : nullptr, B ? B[i] : nullptr));
    const Problem e = relayed(q, r);
    const int direct = select_variant(q, fit, count);
    if (direct >= 0 && table()[direct].kind == KIND_WAVEK &&
        variant_cost(direct, q, count) < call_cost_us(e, row_fit(e, nullptr, nullptr), count) + 3.5 + (double)a_bytes * 2.0 / 4.0e6)
      return Relay();
  }
  // (a copied B is a prepared one, which the bounds-checked kernels do not take: without a kernel for what is left, rows of A
  // too far apart for 32-bit offsets for instance, nothing is copied and the operands are read where they lie)
  if (r.b) {
    const Problem e = relayed(q, r);
    if (select_variant(e, row_fit(e, nullptr, nullptr), count) < 0) return Relay();
  }
  return r;
}
static size_t relay_bytes(const Relay& r, int count) { return (size_t)count * (r.a_bytes + r.b_bytes); }
// what the partial results of the chosen kernel's K split take, at most `room`
static size_t ksplit_need(const Problem& q, RowFit fit, size_t room) {
  int splits = 1;
  const int v = select_variant(q, fit, 1, room, &splits);
  return v >= 0 && ksplit_kind(table()[v]) ? ksplit_bytes(q.M, q.N, splits) : 0;
}

// three fp8 / fp16 terms that the slot kernels take once K is rounded up to their stages: they split both operands in a
// pass of their own, which fills the rest with zeros and reads rows of any alignment
static Problem rounded_up(const Problem& q, RowFit fit) {
  Problem e = q;
  e.k_valid = q.K;
  const int64_t step = q.fmt == CASCMM_FMT_FP8 ? 64 : 32;
  if (q.dtype == CASCMM_DT_F32 && !q.bpre && !q.glu && q.terms == 3 && q.products == CASCMM_PROD_TRI && q.fmt != CASCMM_FMT_BF16 &&
      (fit != FIT_FAST || q.K % step != 0) && q.K > 0 && !beyond_i32(q.K, q.ldb, 4)) {
    e.split_first = true;
    e.K = (q.K + step - 1) / step * step;
  }
  return e;
}

// The slot kernel for such a problem, or a negative status: none, no room, or the bounds-checked kernel, which needs one
// launch where these need three, is expected to be faster (a 32-k step of its 64 x 64 tiles 1.35 us: 100 x 300 x 200
// fp16 x 3 16.5 us against 21; 300 x 500 x 1001 25.9 against 24, fp8 x 3 35 against 26, 3740 x 1090 x 992 fp16 x 3 132 against 81).
// Three fp8 terms need three launches more, of 3 us of the host's time each, behind a scale search that keeps the host
// busy already: eager calls take 36 us in slots however small they are, so what the bounds-checked kernel runs in less stays
// there (8 x 632 x 576: 31 us; graph replay 30 and 23), and the launches count as 5 us.  A step of the bounds-checked fp8
// tiles takes 1.1 us where there are few and 1.9 on 130 CUs (640 x 768 x 814: 49 us).
static int select_rounded_up(const Problem& q, RowFit fit, size_t room, Problem* e) {
  *e = rounded_up(q, fit);
  if (!e->split_first) return CASCMM_ERR_BAD_FORMAT;
  // (up to one tile per CU, of 16 columns for 16 rows and fewer, K over eight waves on the rows as they lie: 6 x 2455 x 1079 12.2 us, 33.3
  // in slots; 153 x 1368 x 728 11.5, 23.5.  Wider results of few rows are left to the comparison below, as before: 5 x 939 x 5189 24.7 in
  // slots, 8.8 here)
  const int64_t wide = q.M <= 16 ? 16 : 32;
  if (q.call && q.fmt == CASCMM_FMT_FP8 && fit != FIT_NONE && ((q.M + wide - 1) / wide) * ((q.N + wide - 1) / wide) <= kNumCUs &&
      few_tiles_three_terms(q, 1, false) && !beyond_i32(q.M, q.lda, 4))
    return CASCMM_ERR_BAD_FORMAT;
  const int v = select_variant(*e, FIT_FAST, 1, room);
  if (v < 0) return v;
  const double tiles = (double)((q.M + 63) / 64) * (double)((q.N + 63) / 64);
  const double rounds = (double)(int64_t)((tiles + kNumCUs - 1) / kNumCUs);
  const bool fp8 = q.fmt == CASCMM_FMT_FP8;
  const double step = fp8 ? std::min(1.2 + 0.006 * tiles, 2.7) : 1.35, slots = variant_cost(v, *e, 1);
  return (fp8 ? std::max(slots + 5.0, 32.0) : slots) < 3.5 + step * rounds * (double)((q.K + 31) / 32) ? v : (int)CASCMM_ERR_BAD_FORMAT;
}

// A call that an fp16 slot kernel would take if it had all the workspace that it wants: K over eight waves on the rows as they lie, which scales
// its tiles itself and needs no workspace, or -1.  (A tile costs 1.15 of the unscaled kernels' time in the median of 119 shapes.)  Up to two tiles
// of 32 x 32 per CU: 330 tiles of 71 x 3801 x 3520 96.4 us in slots, here 54.8 (66.1 where the values are scaled); 286 of 341 x 3577 x 832 75.4,
// 53.0 (66.7); beyond 389 x 1152 x 2175 41.3, 47.7; 421 x 760 x 2496 32.8, 41.3.
static bool few_scaled_tiles(const Problem& q) {
  return q.call && q.dtype == CASCMM_DT_F32 && q.fmt == CASCMM_FMT_FP16 && q.terms == 3 && !q.bpre && !q.glu && !q.split_first &&
         ((q.M + 31) / 32) * ((q.N + 31) / 32) <= 2 * kNumCUs;
}
static int select_scaled_rows(const Problem& q, RowFit fit) {
  const auto& t = table();
  if (!few_scaled_tiles(q)) return -1;
  Problem e;
  int v = select_rounded_up(q, fit, (size_t)-1, &e);
  if (v < 0) {
    e = q;
    v = select_variant(q, fit, 1);
  }
  if (v < 0 || t[v].kind != KIND_F16K) return -1;
  int best = -1;
  double best_cost = variant_cost(v, e, 1);
  for (int i = 0; i < (int)t.size(); ++i) {
    if (!t[i].scaled || !variant_matches(t[i], q, fit)) continue;
    const double cost = 1.15 * variant_cost(i, q, 1);
    if (cost >= best_cost) continue;
    best = i;
    best_cost = cost;
  }
  return best;
}

// The launch itself, on operands as they lie (exps_dyn, b_exp_src: see gemm_impl)
static int gemm_on_rows(int count, const void* const* A, const void* const* B, void* const* C, const void* const* bias, const Problem& q0,
                        const int32_t* tensor_exps, void* workspace, size_t workspace_bytes, hipStream_t stream, int variant,
                        int32_t* exps_dyn = nullptr, const int32_t* b_exp_src = nullptr) {
  Problem q = q0;
  const size_t es = dtype_size(q.dtype);
  RowFit fit = FIT_FAST;
  for (int i = 0; i < count; ++i) {
    if (!A[i] || !B[i]) return CASCMM_ERR_NULL_POINTER;
    if (!aligned_to(A[i], es) || !aligned_to(B[i], q.bpre ? 16 : es)) return CASCMM_ERR_ALIGNMENT;
    fit = std::min(fit, row_fit(q, A[i], q.bpre ? nullptr : B[i]));
  }
  if (q.bpre) {
    // prepared weights only have the fast kernels: K and the rows of A as the kernel needs them (checked per
    // variant), and a buffer the 32-bit offsets can span
    if (fit == FIT_NONE) return CASCMM_ERR_ALIGNMENT;
    if (prepared_bytes(q.K, q.N, q.fmt, q.terms, q.glu) > INT32_MAX) return CASCMM_ERR_TOO_LARGE;
  }
  // (a prepared weight that no kernel takes with these rows: ALIGNMENT where they are off 16-byte boundaries, which all of
  // the kernels take)
  bool off16 = false;
  for (int i = 0; i < count; ++i) off16 = off16 || !aligned_to(A[i], 16) || q.lda * (int64_t)es % 16 != 0;
  const auto none = [&](int status) { return q.bpre && off16 ? (int)CASCMM_ERR_ALIGNMENT : status; };

  const auto& t = table();
  int splits = 1;
  if (variant < 0) {
    // (with room for slots a call of select_scaled_rows is one that a slot kernel would take: the others do not pay for its answer)
    const size_t room = workspace ? workspace_bytes : 0;
    const RowFit rows_fit = fit;
    const bool no_slots = count == 1 && few_scaled_tiles(q) && f16k_workspace_bytes(q.M, q.N, rounded_up(q, fit).K) > room;
    int rows = no_slots ? select_scaled_rows(q, fit) : -1;
    if (count == 1 && !q.split_first && rows < 0) {
      Problem e;
      if (select_rounded_up(q, fit, room, &e) >= 0) {
        q = e;
        fit = FIT_FAST;
      }
    }
    variant = rows >= 0 ? rows : select_variant(q, fit, count, room, &splits);
    if (count == 1 && variant >= 0 && t[variant].kind == KIND_F16K && (rows = select_scaled_rows(q0, rows_fit)) >= 0) {
      variant = rows;
      q = q0;
    }
    if (variant < 0 && count > 1) {
      // no kernel takes these problems in one launch (the fp8-rate kernel runs one at a time): one
      // launch each, in order on the stream, sharing the workspace
      for (int i = 0; i < count; ++i) {
        const void* bi = bias ? bias[i] : nullptr;
        const int st1 = gemm_on_rows(1, A + i, B + i, C + i, bias ? &bi : nullptr, q, tensor_exps ? tensor_exps + 2 * i : nullptr,
                                  workspace, workspace_bytes, stream, -1);
        if (st1 != CASCMM_OK) return st1;
      }
      return CASCMM_OK;
    }
    if (variant < 0) return none(variant);
  } else {
    splits = (variant >> 16) > 0 ? (variant >> 16) : 1;   // forced: kernel index | K splits << 16
    variant &= 0xFFFF;
    if (variant >= (int)t.size()) return CASCMM_ERR_BAD_VARIANT;
    if (splits > (ksplit_kind(t[variant]) ? kMaxKSplits : kMaxTileSplits)) return CASCMM_ERR_BAD_VARIANT;
    if (!variant_matches(t[variant], q, fit)) return none(CASCMM_ERR_BAD_VARIANT);
  }
  const VariantDesc& v = t[variant];
  if (exps_dyn && (v.kind != KIND_F8K64 || count != 1)) return CASCMM_ERR_BAD_VARIANT;
  if (count > 1 && !v.grouped) {
    // a forced kernel that runs one problem per launch: one launch each, in order on the stream
    if (v.kind == KIND_SPLITK) return CASCMM_ERR_BAD_VARIANT;
    for (int i = 0; i < count; ++i) {
      const void* bi = bias ? bias[i] : nullptr;
      const int st1 = gemm_on_rows(1, A + i, B + i, C + i, bias ? &bi : nullptr, q, tensor_exps ? tensor_exps + 2 * i : nullptr,
                                workspace, workspace_bytes, stream, variant | (splits > 1 ? splits << 16 : 0));
      if (st1 != CASCMM_OK) return st1;
    }
    return CASCMM_OK;
  }
  GroupParams p;
  memset(&p, 0, sizeof(p));
  p.M = (int)q.M; p.N = (int)q.N; p.K = (int)q.K;
  p.k_valid = (int)(q.split_first ? q.k_valid : q.K);
  p.lda = q.lda; p.ldb = q.ldb; p.ldc = q.ldc;
  const int64_t tm = (q.M + v.BM - 1) / v.BM, tn = (q.N + v.BN - 1) / v.BN;
  if (tm * tn * count > INT32_MAX) return CASCMM_ERR_TOO_LARGE;
  p.tiles_m = (int)tm; p.tiles_n = (int)tn;
  p.count = count;
  p.workspace = workspace;
  p.workspace_bytes = workspace_bytes;
  p.k_splits = v.kind == KIND_TILE ? splits : 1;
  p.k_per = p.K;
  if (ksplit_kind(v) && splits > 1 && count == 1 && !q.glu) {
    // (a forced count of which some would be empty: the others; without room for the partial results: K whole)
    const int64_t k_per = ksplit_k(q.K, splits);
    splits = (int)((q.K + k_per - 1) / k_per);
    if (workspace && aligned_to(workspace, 16) && ksplit_bytes(q.M, q.N, splits) <= workspace_bytes && splits > 1) {
      p.k_splits = splits;
      p.k_per = (int)k_per;
    }
  }
  p.tensor_exps = q.fmt == CASCMM_FMT_FP8 ? tensor_exps : nullptr;
  p.glu = q.glu_slots ? 2 : (q.glu ? 1 : 0);
  p.exps_dyn = exps_dyn;
  p.b_exp_src = b_exp_src;
  for (int i = 0; i < count; ++i) {
    p.A[i] = A[i]; p.B[i] = B[i]; p.C[i] = C[i]; p.bias[i] = bias ? bias[i] : nullptr;
  }
  return v.launch(p, stream);
}

// whether the rows of A are whole 16-byte chunks by K alone
static bool chunked_by_k(const Problem& q) { return q.K % (q.dtype == CASCMM_DT_F32 ? 4 : 8) == 0; }

// the kernel for a shape whose operands lie well (what the selection functions of the ABI answer: the launch may copy
// rows first and then take another)
static int select_for_shape(Problem q, int count) {
  q.chunked = q.K % 8 == 0;
  return select_variant(q, row_fit(q, nullptr, nullptr), count);
}

// One launch for `count` problems of one shape (count == 1: a plain GEMM), behind a copy of operands whose rows need one.
// exps_dyn (fp8-rate kernel only, count == 1): the launch finds the left operand's scale exponent
// itself and leaves {e_A, *b_exp_src} there; CASCMM_ERR_BAD_VARIANT when another kernel is selected.
static int gemm_impl(int count, const void* const* A, const void* const* B, void* const* C, const void* const* bias,
                     const Problem& q0, const int32_t* tensor_exps, void* workspace, size_t workspace_bytes,
                     hipStream_t stream, int variant, int32_t* exps_dyn = nullptr, const int32_t* b_exp_src = nullptr) {
  Problem q = q0;
  int st = check_problem(q);
  if (st != CASCMM_OK) return st;
  if (count < 1 || count > kMaxGroup) return CASCMM_ERR_BAD_SHAPE;
  if (q.M == 0 || q.N == 0) return CASCMM_OK;
  const size_t es = dtype_size(q.dtype);
  for (int i = 0; i < count; ++i) {
    if (!C[i]) return CASCMM_ERR_NULL_POINTER;
    if (!aligned_to(C[i], es) || (bias && !aligned_to(bias[i], es))) return CASCMM_ERR_ALIGNMENT;
  }
  if (q.glu && (q.N % 64 != 0 || q.K == 0)) return CASCMM_ERR_BAD_SHAPE;
  if (q.K == 0) {
    const int64_t total = q.M * q.N;
    const unsigned grid = (unsigned)((total + 255) / 256);
    hipError_t err = hipSuccess;
    for (int i = 0; i < count; ++i) {
      const void* b = bias ? bias[i] : nullptr;
      if (q.dtype == CASCMM_DT_F32)
        CASCMM_LAUNCH(err, (fill_bias_kernel<CASCMM_DT_F32>), dim3(grid), dim3(256), 0, stream, C[i], b, (int)q.M, (int)q.N, q.ldc);
      else if (q.dtype == CASCMM_DT_F16)
        CASCMM_LAUNCH(err, (fill_bias_kernel<CASCMM_DT_F16>), dim3(grid), dim3(256), 0, stream, C[i], b, (int)q.M, (int)q.N, q.ldc);
      else
        CASCMM_LAUNCH(err, (fill_bias_kernel<CASCMM_DT_BF16>), dim3(grid), dim3(256), 0, stream, C[i], b, (int)q.M, (int)q.N, q.ldc);
    }
    return err == hipSuccess ? CASCMM_OK : CASCMM_ERR_LAUNCH;
  }
  q.chunked = chunked_by_k(q);
  q.call = true;
  // Calls of several launches that meet in the workspace go to the stream as a whole: two threads that share a stream, and
  // with it the workspace, must not put one call's launches between another's.
  static std::mutex workspace_mu;
  std::unique_lock<std::mutex> whole(workspace_mu, std::defer_lock);
  if (workspace) whole.lock();
  if (variant < 0) {
    const Relay r = relay_of(q, count, A, B);
    if ((r.a || r.b) && workspace && aligned_to(workspace, 16) && workspace_bytes >= relay_bytes(r, count)) {
      const void* ap[kMaxGroup];
      const void* bp[kMaxGroup];
      char* ws = (char*)workspace;
      for (int i = 0; i < count; ++i) {
        if (!A[i] || !B[i]) return CASCMM_ERR_NULL_POINTER;
        if (!aligned_to(A[i], es) || !aligned_to(B[i], es)) return CASCMM_ERR_ALIGNMENT;
        // (the same operand twice in one group is copied once)
        bool copy_a = r.a, copy_b = r.b;
        ap[i] = A[i];
        bp[i] = B[i];
        for (int j = 0; j < i; ++j) {
          if (copy_a && A[j] == A[i]) { ap[i] = ap[j]; copy_a = false; }
          if (copy_b && B[j] == B[i]) { bp[i] = bp[j]; copy_b = false; }
        }
        if (copy_a) { ap[i] = ws; ws += r.a_bytes; }
        if (copy_b) { bp[i] = ws; ws += r.b_bytes; }
        const unsigned a_blocks = copy_a ? (unsigned)((q.M * r.a_chunks + 255) / 256) : 0;
        const unsigned b_blocks = copy_b ? (unsigned)((prepared_kgroups(q.K) * q.N + 255) / 256) : 0;
        if (a_blocks + b_blocks == 0) continue;
        hipError_t err = hipSuccess;
        if (q.dtype == CASCMM_DT_F32)
          CASCMM_LAUNCH(err, (relay_kernel<unsigned>), dim3(a_blocks), dim3(256), 0, stream, (const unsigned*)A[i], (int)q.M, (int)q.K, q.lda, r.a_chunks,
                        (u32x4*)ap[i], (int)a_blocks, (const unsigned*)nullptr, 0, (int64_t)0, (u32x4*)nullptr);
        else
          CASCMM_LAUNCH(err, (relay_kernel<unsigned short>), dim3(a_blocks + b_blocks), dim3(256), 0, stream, (const unsigned short*)A[i], (int)q.M,
                        (int)q.K, q.lda, r.a_chunks, (u32x4*)ap[i], (int)a_blocks, (const unsigned short*)B[i], (int)q.N, q.ldb, (u32x4*)bp[i]);
        if (err != hipSuccess) return CASCMM_ERR_LAUNCH;
      }
      const size_t rest = workspace_bytes - relay_bytes(r, count);
      return gemm_on_rows(count, ap, bp, C, bias, relayed(q, r), tensor_exps, rest > 0 ? (char*)workspace + relay_bytes(r, count) : nullptr, rest, stream, -1);
    }
  }
  return gemm_on_rows(count, A, B, C, bias, q, tensor_exps, workspace, workspace_bytes, stream, variant, exps_dyn, b_exp_src);
}

}  // namespace cascmm

using namespace cascmm;

// Built-in scratch of cascmm_gemm_noalloc: the K-split partial results that cascmm_gemm keeps in the
// caller's workspace.  One copy per GPU the library runs on, held until the process ends.  In host
// code the array's name is only a handle for hipGetSymbolAddress; the device address it returns
// (per device) is what kernels and copies are given.
static __device__ __align__(256) unsigned char scratch[CASCMM_NOALLOC_SCRATCH_BYTES];

static int noalloc_scratch(void** out) {
  static std::mutex mu;
  static void* ptr_of_device[kMaxDevices] = {nullptr};
  const int d = device_index();
  if (d < 0) return CASCMM_ERR_LAUNCH;
  std::lock_guard<std::mutex> lock(mu);
  if (!ptr_of_device[d]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return CASCMM_ERR_LAUNCH;
    ptr_of_device[d] = p;
  }
  *out = ptr_of_device[d];
  return CASCMM_OK;
}

extern "C" {

int cascmm_init(void) {
  void* p = nullptr;
  return noalloc_scratch(&p);
}

int cascmm_gemm_noalloc(const void* A, const void* B, void* C, const void* bias, int64_t M, int64_t N, int64_t K,
                        int64_t lda, int64_t ldb, int64_t ldc, int dtype, int fmt, int terms, int products,
                        const int32_t* tensor_exps, void* stream) {
  Problem q{M, N, K, lda, ldb, ldc, dtype, fmt, terms, products};
  const int st = check_problem(q);
  if (st != CASCMM_OK) return st;
  if (M == 0 || N == 0 || K == 0) return cascmm_gemm(A, B, C, bias, M, N, K, lda, ldb, ldc, dtype, fmt, terms, products,
                                                     tensor_exps, nullptr, 0, stream);
  // the scratch that the kernel cascmm_gemm would pick with an unlimited workspace needs for this problem
  size_t need = 0;
  const void* const a1[1] = {A};
  const void* const b1[1] = {B};
  const Relay relay = relay_of(q, 1, a1, b1);
  if (relay.a || relay.b) {
    need = relay_bytes(relay, 1);
    if (need > (size_t)CASCMM_NOALLOC_SCRATCH_BYTES) need = 0;   // (the bounds-checked kernels need no copy)
    else need += ksplit_need(relayed(q, relay), FIT_FAST, (size_t)CASCMM_NOALLOC_SCRATCH_BYTES - need);
  } else if (A && B) {
    const RowFit fit = row_fit(q, A, B);
    // (what the kernels known to the selection functions would need: the call itself may take a small tile that needs none)
    q.chunked = chunked_by_k(q);
    Problem e;
    int splits = 1;
    int v = select_rounded_up(q, fit, (size_t)CASCMM_NOALLOC_SCRATCH_BYTES, &e);
    if (v < 0) {
      e = q;
      v = select_variant(q, fit, 1, (size_t)-1, &splits);
    }
    if (v < 0) return v;
    bool as_chosen = true;
    if (ksplit_kind(table()[v]) && ksplit_bytes(M, N, splits) > (size_t)CASCMM_NOALLOC_SCRATCH_BYTES) {
      // (a K split over workgroups is a choice: without it the call is refused or taken as the other kernels need)
      e.whole_k = true;
      v = select_variant(e, fit, 1, (size_t)-1, &splits);
      if (v < 0) return v;
      as_chosen = table()[v].kind == KIND_TILE && splits > 1;
    }
    // (refused where nothing comes near the tile kernels' own K split: few rows have the one-launch kernel)
    if (table()[v].kind == KIND_TILE && splits > 1 && (size_t)splits * (size_t)M * (size_t)N * sizeof(float) > (size_t)CASCMM_NOALLOC_SCRATCH_BYTES &&
        wavek_eligible(e) && (M <= 160 || wavek_estimate_us(e, 1) < 1.8 * variant_cost(v, e, 1, (size_t)-1)))
      as_chosen = false;
    if (!as_chosen || (table()[v].kind == KIND_F8K64 && f8k64_workspace_bytes(M, N, e.K, false, table()[v].BM) > (size_t)CASCMM_NOALLOC_SCRATCH_BYTES) ||
        (table()[v].kind == KIND_F16K && f16k_workspace_bytes(M, N, e.K) > (size_t)CASCMM_NOALLOC_SCRATCH_BYTES)) {
      // the fp8-rate kernel is a choice, not a need: without room for its operand slots the choice is
      // made among the kernels that split inside the GEMM
      v = select_variant(q, fit, 1, (size_t)CASCMM_NOALLOC_SCRATCH_BYTES, &splits);
      if (v < 0) return v;
    }
    const VariantDesc& d = table()[v];
    if (d.kind == KIND_SPLITK) need = skinny_workspace_bytes(M, N, K, d.BM, d.BN, d.BK);
    else if (d.kind == KIND_F8K64) need = f8k64_workspace_bytes(M, N, e.K, false, d.BM);
    else if (d.kind == KIND_F16K) need = f16k_workspace_bytes(M, N, e.K);
    else if (ksplit_kind(d)) need = ksplit_bytes(M, N, splits);
    else if (splits > 1) need = (size_t)splits * (size_t)M * (size_t)N * sizeof(float);
  }
  if (need > (size_t)CASCMM_NOALLOC_SCRATCH_BYTES) return CASCMM_ERR_SCRATCH_LIMIT;
  void* ws = nullptr;
  if (need > 0) {
    const int ss = noalloc_scratch(&ws);
    if (ss != CASCMM_OK) return ss;
  }
  // (nothing in the scratch has to start at zero: a launch reads back only the partial results it wrote)
  return gemm_impl(1, &A, &B, &C, bias ? &bias : nullptr, q, tensor_exps, ws, need, (hipStream_t)stream, -1);
}

int cascmm_gemm_variant(const void* A, const void* B, void* C, const void* bias, int64_t M, int64_t N, int64_t K,
                        int64_t lda, int64_t ldb, int64_t ldc, int dtype, int fmt, int terms, int products,
                        const int32_t* tensor_exps, void* workspace, size_t workspace_bytes, void* stream,
                        int variant) {
  const Problem q{M, N, K, lda, ldb, ldc, dtype, fmt, terms, products};
  return gemm_impl(1, &A, &B, &C, bias ? &bias : nullptr, q, tensor_exps, workspace, workspace_bytes, (hipStream_t)stream,
                   variant);
}

int cascmm_gemm_grouped(int count, const void* const* A, const void* const* B, void* const* C, const void* const* bias,
                        int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int dtype, int fmt,
                        int terms, int products, const int32_t* tensor_exps, void* workspace, size_t workspace_bytes,
                        void* stream, int variant) {
  if (!A || !B || !C) return CASCMM_ERR_NULL_POINTER;
  const Problem q{M, N, K, lda, ldb, ldc, dtype, fmt, terms, products};
  return gemm_impl(count, A, B, C, bias, q, tensor_exps, workspace, workspace_bytes, (hipStream_t)stream, variant);
}

int cascmm_select_variant_glu(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int dtype, int fmt,
                              int terms, int products) {
  Problem q{M, N, K, lda, ldb, ldc, dtype, fmt, terms, products};
  q.glu = true;
  const int st = check_problem(q);
  if (st != CASCMM_OK) return st;
  if (N % 64 != 0 || K == 0) return CASCMM_ERR_BAD_SHAPE;
  q.chunked = chunked_by_k(q);
  const RowFit fit = row_fit(q, nullptr, nullptr);
  const int v = select_variant(q, fit, 1);
  if (v < 0) return v;
  // worth it?  The alternative is the plain product, as a call takes it, plus cascmm_gate, which reads M x N values and writes half as many
  // (5.8 TB/s, and a launch); the kernel with the gated store may be a poor fit for the shape (too few tiles for the chip).
  // Over 78 shapes of 512 - 8192 rows 0.2 % behind the faster of the two on average, 1.0 % with gelu and product as two launches in mind and the
  // selection functions' kernels: 2048 x 320 x 2560 gated 34.5 us, plain and gate 30.2; 1792 x 640 x 5120 53.8, 50.3; 3072 x 960 x 7680 165, 159.
  Problem plain = q;
  plain.glu = false;
  plain.call = true;
  plain.ldc = N;
  const int vp = select_variant(plain, fit, 1);
  if (vp >= 0) {
    const double gate_us = 2.0 + (double)M * (double)N * 6.0 / 5.8e6;
    if (variant_cost(v, q, 1) > variant_cost(vp, plain, 1) + gate_us) return CASCMM_ERR_BAD_FORMAT;
  }
  return v;
}

int cascmm_gemm_glu(const void* A, const void* B, void* C, const void* bias, int64_t M, int64_t N, int64_t K, int64_t lda,
                    int64_t ldb, int64_t ldc, int dtype, int fmt, int terms, int products, void* stream, int variant) {
  Problem q{M, N, K, lda, ldb, ldc, dtype, fmt, terms, products};
  q.glu = true;
  return gemm_impl(1, &A, &B, &C, bias ? &bias : nullptr, q, nullptr, nullptr, 0, (hipStream_t)stream, variant);
}

int cascmm_gemm(const void* A, const void* B, void* C, const void* bias, int64_t M, int64_t N, int64_t K, int64_t lda,
                int64_t ldb, int64_t ldc, int dtype, int fmt, int terms, int products, const int32_t* tensor_exps,
                void* workspace, size_t workspace_bytes, void* stream) {
  return cascmm_gemm_variant(A, B, C, bias, M, N, K, lda, ldb, ldc, dtype, fmt, terms, products, tensor_exps,
                             workspace, workspace_bytes, stream, -1);
}

size_t cascmm_prepared_bytes(int64_t K, int64_t N, int fmt, int terms) {
  if (K < 0 || N < 0 || terms < 1 || terms > 3) return 0;
  if (fmt != CASCMM_FMT_BF16 && fmt != CASCMM_FMT_FP16 && fmt != CASCMM_FMT_FP8) return 0;
  // (three fp8 terms have two layouts, for the plain and the gated preparation: room for either)
  return (size_t)std::max(prepared_bytes(K, N, fmt, terms, false), prepared_bytes(K, N, fmt, terms, true));
}

static int prepare_weight_impl(const void* B, int64_t K, int64_t N, int64_t ldb, int dtype, int fmt, int terms,
                               const int32_t* tensor_exp, void* out, size_t out_bytes, void* stream, int glu) {
  if (K < 0 || N < 0 || ldb < N || (glu && N % 64 != 0)) return CASCMM_ERR_BAD_SHAPE;
  if (K > INT32_MAX || N > INT32_MAX) return CASCMM_ERR_TOO_LARGE;
  if (terms < 1 || terms > 3) return CASCMM_ERR_BAD_FORMAT;
  if (fmt != CASCMM_FMT_BF16 && fmt != CASCMM_FMT_FP16 && fmt != CASCMM_FMT_FP8) return CASCMM_ERR_BAD_FORMAT;
  if (K == 0 || N == 0) return CASCMM_OK;
  if (!B || !out) return CASCMM_ERR_NULL_POINTER;
  if (!aligned_to(out, 16)) return CASCMM_ERR_ALIGNMENT;
  if (out_bytes < (size_t)prepared_bytes(K, N, fmt, terms, glu != 0)) return CASCMM_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  if (prepared_as_k16_slots(K, fmt, terms, glu != 0)) {
    // the layout of the fp8-rate kernel: [term][K/16][N] slots of 16 k
    if (dtype != CASCMM_DT_F32) return CASCMM_ERR_BAD_DTYPE;
    const int64_t units = (K >> 4) * N;
    return launch_kernel(f8k64_split_cols_kernel<0>, dim3((unsigned)((units + 255) / 256)), dim3(256), 0, s, (const float*)B, (int)K,
                         (int)K, (int)N, ldb, tensor_exp, (u32x4*)out) == hipSuccess ? CASCMM_OK : CASCMM_ERR_LAUNCH;
  }
  if (dtype == CASCMM_DT_F32) return launch_prepare_fmt<CASCMM_DT_F32>(B, (int)K, (int)N, ldb, fmt, terms, tensor_exp, (u32x4*)out, s, glu);
  if (dtype == CASCMM_DT_F16) return launch_prepare_fmt<CASCMM_DT_F16>(B, (int)K, (int)N, ldb, fmt, terms, tensor_exp, (u32x4*)out, s, glu);
  if (dtype == CASCMM_DT_BF16) return launch_prepare_fmt<CASCMM_DT_BF16>(B, (int)K, (int)N, ldb, fmt, terms, tensor_exp, (u32x4*)out, s, glu);
  return CASCMM_ERR_BAD_DTYPE;
}

int cascmm_prepare_weight(const void* B, int64_t K, int64_t N, int64_t ldb, int dtype, int fmt, int terms,
                          const int32_t* tensor_exp, void* out, size_t out_bytes, void* stream) {
  return prepare_weight_impl(B, K, N, ldb, dtype, fmt, terms, tensor_exp, out, out_bytes, stream, 0);
}

int cascmm_prepare_weight_glu(const void* B, int64_t K, int64_t N, int64_t ldb, int dtype, int fmt, int terms,
                              const int32_t* tensor_exp, void* out, size_t out_bytes, void* stream) {
  return prepare_weight_impl(B, K, N, ldb, dtype, fmt, terms, tensor_exp, out, out_bytes, stream, 1);
}

int cascmm_gemm_prepared_glu(int count, const void* const* A, const void* const* Bprep, void* const* C,
                             const void* const* bias, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldc,
                             int dtype, int fmt, int terms, int products, const int32_t* tensor_exps, void* stream,
                             int variant) {
  if (!A || !Bprep || !C) return CASCMM_ERR_NULL_POINTER;
  Problem q{M, N, K, lda, N, ldc, dtype, fmt, terms, products};
  q.bpre = true;
  q.glu = true;
  return gemm_impl(count, A, Bprep, C, bias, q, tensor_exps, nullptr, 0, (hipStream_t)stream, variant);
}

int cascmm_gemm_prepared(int count, const void* const* A, const void* const* Bprep, void* const* C,
                         const void* const* bias, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldc, int dtype,
                         int fmt, int terms, int products, const int32_t* tensor_exps, void* workspace,
                         size_t workspace_bytes, void* stream, int variant) {
  if (!A || !Bprep || !C) return CASCMM_ERR_NULL_POINTER;
  Problem q{M, N, K, lda, N, ldc, dtype, fmt, terms, products};
  q.bpre = true;
  return gemm_impl(count, A, Bprep, C, bias, q, tensor_exps, workspace, workspace_bytes, (hipStream_t)stream, variant);
}

int cascmm_select_variant_prepared(int count, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldc, int dtype, int fmt,
                                   int terms, int products) {
  if (count < 1 || count > kMaxGroup) return CASCMM_ERR_BAD_SHAPE;
  Problem q{M, N, K, lda, N, ldc, dtype, fmt, terms, products};
  q.bpre = true;
  const int st = check_problem(q);
  if (st != CASCMM_OK) return st;
  return select_for_shape(q, count);
}

size_t cascmm_workspace_bytes(int64_t M, int64_t N, int64_t K, int dtype, int fmt, int terms, int products) {
  // upper bound over the skinny variants that could be selected for this problem (the
  // selection also depends on pointer alignment, which is not known here)
  Problem q{M, N, K, K, N, N, dtype, fmt, terms, products};
  if (check_problem(q) != CASCMM_OK) return 0;
  q.chunked = chunked_by_k(q);
  const RowFit fit = row_fit(q, nullptr, nullptr);
  // rows of A (and, 16-bit, all of B) copied first
  const Relay relay = relay_of(q, 1, nullptr, nullptr, false);
  size_t need = relay_bytes(relay, 1);
  // K split over workgroups, behind such a copy or on the operands as they lie, raw or prepared
  size_t parts = 0;
  for (int pre = 0; pre < 2; ++pre) {
    Problem e = relay.a || relay.b ? relayed(q, relay) : q;
    e.bpre = e.bpre || pre != 0;
    for (int vi = 0; vi < (int)table().size(); ++vi) {
      if (!ksplit_kind(table()[vi]) || !variant_matches(table()[vi], e, FIT_FAST)) continue;
      int sp = 1;
      variant_cost(vi, e, 1, (size_t)-1, &sp);
      parts = std::max(parts, ksplit_bytes(M, N, sp));
    }
  }
  need += parts;
  for (const auto& v : table()) {
    if (v.kind != KIND_SPLITK || !variant_matches(v, q, fit)) continue;
    const size_t n = skinny_workspace_bytes(M, N, K, v.BM, v.BN, v.BK);
    need = n > need ? n : need;
  }
  // three fp8 terms on the fp8-rate kernel, three fp16 terms on operand slots: the slots of A and B
  const Problem e = rounded_up(q, fit);
  for (const auto& v : table()) {
    if ((v.kind != KIND_F8K64 && v.kind != KIND_F16K) || v.bpre || !variant_matches(v, e, e.split_first ? FIT_FAST : fit)) continue;
    const size_t n = v.kind == KIND_F8K64 ? f8k64_workspace_bytes(M, N, e.K, false, v.BM) : f16k_workspace_bytes(M, N, e.K);
    need = n > need ? n : need;
  }
  // K split of the LDS-tiled kernels: up to kMaxTileSplits partial results when some kernel
  // would run the problem with at most half the CUs busy
  if (dtype == CASCMM_DT_F32 && N % 4 == 0) {
    for (int vi = 0; vi < (int)table().size(); ++vi) {
      const VariantDesc& v = table()[vi];
      if (v.kind != KIND_TILE || !variant_matches(v, q, fit)) continue;
      int sp = 1;
      variant_cost(vi, q, 1, (size_t)-1, &sp);
      const size_t n = sp > 1 ? (size_t)kMaxTileSplits * M * N * sizeof(float) : 0;
      need = n > need ? n : need;
    }
  }
  return need;
}

int cascmm_select_variant(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int dtype, int fmt,
                          int terms, int products) {
  const Problem q{M, N, K, lda, ldb, ldc, dtype, fmt, terms, products};
  const int st = check_problem(q);
  if (st != CASCMM_OK) return st;
  return select_for_shape(q, 1);
}

int cascmm_call_variant(const void* A, const void* B, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc,
                        int dtype, int fmt, int terms, int products, size_t workspace_bytes) {
  Problem q{M, N, K, lda, ldb, ldc, dtype, fmt, terms, products};
  const int st = check_problem(q);
  if (st != CASCMM_OK) return st;
  q.chunked = chunked_by_k(q);
  q.call = true;
  // (as gemm_impl and gemm_on_rows go about it)
  const Relay r = relay_of(q, 1, &A, &B);
  if ((r.a || r.b) && workspace_bytes >= relay_bytes(r, 1)) {
    const Problem e = relayed(q, r);
    return select_variant(e, row_fit(e, r.a ? nullptr : A, r.b ? nullptr : B), 1, workspace_bytes - relay_bytes(r, 1));
  }
  const RowFit fit = row_fit(q, A, B);
  const int rows = select_scaled_rows(q, fit);
  if (rows >= 0) return rows;
  Problem e;
  const int v = select_rounded_up(q, fit, workspace_bytes, &e);
  return v >= 0 ? v : select_variant(q, fit, 1, workspace_bytes);
}

int cascmm_call_variant_prepared(const void* A, int glu, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldc, int dtype, int fmt,
                                 int terms, int products, size_t workspace_bytes) {
  Problem q{M, N, K, lda, N, ldc, dtype, fmt, terms, products};
  q.bpre = true;
  q.glu = glu != 0;
  const int st = check_problem(q);
  if (st != CASCMM_OK) return st;
  if (q.glu && (N % 64 != 0 || K == 0)) return CASCMM_ERR_BAD_SHAPE;
  if (prepared_bytes(K, N, fmt, terms, q.glu) > INT32_MAX) return CASCMM_ERR_TOO_LARGE;
  q.chunked = chunked_by_k(q);
  q.call = true;
  return select_variant(q, row_fit(q, A, nullptr), 1, q.glu ? 0 : workspace_bytes);
}

int cascmm_select_variant_grouped(int count, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc,
                                  int dtype, int fmt, int terms, int products) {
  if (count < 1 || count > kMaxGroup) return CASCMM_ERR_BAD_SHAPE;
  const Problem q{M, N, K, lda, ldb, ldc, dtype, fmt, terms, products};
  const int st = check_problem(q);
  if (st != CASCMM_OK) return st;
  return select_for_shape(q, count);
}

int cascmm_variant_count(void) { return (int)table().size(); }

const char* cascmm_variant_name(int variant) {
  if (variant < 0 || variant >= (int)table().size()) return nullptr;
  return table()[variant].name;
}

const char* cascmm_variant_kernel(int variant) {
  return cascmm_launched_kernel(variant, 40960, 40960, 40960);   // (a multiple of every tile and stage)
}

const char* cascmm_launched_kernel(int variant, int64_t M, int64_t N, int64_t K) {
  if (variant < 0 || variant >= (int)table().size() || M < 0 || N < 0 || K < 0 || M > INT32_MAX || N > INT32_MAX || K > INT32_MAX) return nullptr;
  const void* handle = nullptr;
  GroupParams p;
  memset(&p, 0, sizeof(p));
  p.M = (int)M; p.N = (int)N; p.K = (int)K;
  p.kernel_out = &handle;
  if (table()[variant].launch(p, nullptr) != CASCMM_OK || !handle) return nullptr;
  // the handle of a kernel is an exported object of this library that carries the kernel's name
  Dl_info info;
  if (!dladdr(handle, &info) || !info.dli_sname || info.dli_saddr != handle) return nullptr;
  return info.dli_sname;
}

int cascmm_tensor_exp(const void* x, int64_t rows, int64_t cols, int64_t ld, int dtype, int32_t* exp_out,
                      void* stream) {
  if (dtype != CASCMM_DT_F32 && dtype != CASCMM_DT_F16 && dtype != CASCMM_DT_BF16) return CASCMM_ERR_BAD_DTYPE;
  if (rows < 0 || cols < 0 || ld < cols) return CASCMM_ERR_BAD_SHAPE;
  if (!exp_out || (rows * cols > 0 && !x)) return CASCMM_ERR_NULL_POINTER;
  if (rows > INT32_MAX || cols > INT32_MAX) return CASCMM_ERR_TOO_LARGE;
  hipStream_t s = (hipStream_t)stream;
  // *exp_out holds the bit pattern of the running max|x| until the last kernel replaces it
  hipError_t err = hipSuccess;
  CASCMM_LAUNCH(err, amax_begin_kernel, dim3(1), dim3(1), 0, s, exp_out);
  const int64_t total = rows * cols;
  if (total > 0) {
    const unsigned grid = (unsigned)std::min<int64_t>((total + 4095) / 4096, 1024);
    if (dtype == CASCMM_DT_F32)
      CASCMM_LAUNCH(err, (amax_kernel<CASCMM_DT_F32>), dim3(grid), dim3(256), 0, s, x, rows, cols, ld, exp_out);
    else if (dtype == CASCMM_DT_F16)
      CASCMM_LAUNCH(err, (amax_kernel<CASCMM_DT_F16>), dim3(grid), dim3(256), 0, s, x, rows, cols, ld, exp_out);
    else
      CASCMM_LAUNCH(err, (amax_kernel<CASCMM_DT_BF16>), dim3(grid), dim3(256), 0, s, x, rows, cols, ld, exp_out);
  }
  CASCMM_LAUNCH(err, amax_end_kernel, dim3(1), dim3(1), 0, s, exp_out);
  return err == hipSuccess ? CASCMM_OK : CASCMM_ERR_LAUNCH;
}

int cascmm_tensor_exps(const void* x, int64_t rows, int64_t cols, int64_t ld, int dtype, const int32_t* second_exp,
                       int32_t* exps_out, int32_t* scratch, void* stream) {
  if (dtype != CASCMM_DT_F32 && dtype != CASCMM_DT_F16 && dtype != CASCMM_DT_BF16) return CASCMM_ERR_BAD_DTYPE;
  if (rows < 0 || cols < 0 || ld < cols) return CASCMM_ERR_BAD_SHAPE;
  if (!exps_out || !scratch || (rows * cols > 0 && !x)) return CASCMM_ERR_NULL_POINTER;
  if (rows > INT32_MAX || cols > INT32_MAX) return CASCMM_ERR_TOO_LARGE;
  hipStream_t s = (hipStream_t)stream;
  const int64_t total = rows * cols;
  // (an empty tensor: one workgroup that scans nothing and writes e = 0)
  hipError_t err = hipSuccess;
  // few, large workgroups: every workgroup ends in a ticket atomic on one word, and those serialise
  const unsigned grid = (unsigned)std::max<int64_t>(1, std::min<int64_t>((total + 16383) / 16384, device_cus() / 2));
  if (dtype == CASCMM_DT_F32)
    CASCMM_LAUNCH(err, (amax_single_launch_kernel<CASCMM_DT_F32>), dim3(grid), dim3(1024), 0, s, x, rows, cols, ld, second_exp,
                       exps_out, (unsigned*)scratch);
  else if (dtype == CASCMM_DT_F16)
    CASCMM_LAUNCH(err, (amax_single_launch_kernel<CASCMM_DT_F16>), dim3(grid), dim3(1024), 0, s, x, rows, cols, ld, second_exp,
                       exps_out, (unsigned*)scratch);
  else
    CASCMM_LAUNCH(err, (amax_single_launch_kernel<CASCMM_DT_BF16>), dim3(grid), dim3(1024), 0, s, x, rows, cols, ld, second_exp,
                       exps_out, (unsigned*)scratch);
  return err == hipSuccess ? CASCMM_OK : CASCMM_ERR_LAUNCH;
}

int cascmm_gate(const void* h, void* out, int64_t rows, int64_t inner, int64_t ldh, int64_t ldo, int dtype, void* stream) {
  if (dtype != CASCMM_DT_F32 && dtype != CASCMM_DT_F16 && dtype != CASCMM_DT_BF16) return CASCMM_ERR_BAD_DTYPE;
  if (rows < 0 || inner < 0 || ldh < 2 * inner || ldo < inner) return CASCMM_ERR_BAD_SHAPE;
  if (rows == 0 || inner == 0) return CASCMM_OK;
  if (!h || !out) return CASCMM_ERR_NULL_POINTER;
  if (!aligned_to(h, dtype_size(dtype)) || !aligned_to(out, dtype_size(dtype))) return CASCMM_ERR_ALIGNMENT;
  // (the kernel counts a row's elements, and all runs, in 32 bits, in steps of 256 past the last)
  if (inner > INT32_MAX || rows > INT32_MAX || rows * inner > (int64_t)UINT32_MAX - 4096) return CASCMM_ERR_TOO_LARGE;
  const hipStream_t s = (hipStream_t)stream;
  const hipError_t err = dtype == CASCMM_DT_F32   ? launch_gate<CASCMM_DT_F32>(h, ldh, out, ldo, rows, inner, s)
                         : dtype == CASCMM_DT_F16 ? launch_gate<CASCMM_DT_F16>(h, ldh, out, ldo, rows, inner, s)
                                                  : launch_gate<CASCMM_DT_BF16>(h, ldh, out, ldo, rows, inner, s);
  return err == hipSuccess ? CASCMM_OK : CASCMM_ERR_LAUNCH;
}

int cascmm_gemm_fp8_autoscale(const void* A, const void* B, int b_prepared, void* C, const void* bias, int64_t M, int64_t N,
                              int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int terms, int products, const int32_t* b_exp,
                              int32_t* exps_out, int32_t* scratch, void* workspace, size_t workspace_bytes, void* stream) {
  if (!exps_out || !scratch) return CASCMM_ERR_NULL_POINTER;
  Problem q{M, N, K, lda, b_prepared ? N : ldb, ldc, CASCMM_DT_F32, CASCMM_FMT_FP8, terms, products};
  q.bpre = b_prepared != 0;
  const int st = check_problem(q);
  if (st != CASCMM_OK) return st;
  q.chunked = chunked_by_k(q);
  q.call = true;
  const void* bias1 = bias;
  if (M > 0 && N > 0 && K > 0 && A && B) {
    // the fp8-rate kernel splits A in a pass of its own anyway: the search rides on it
    const RowFit fit = row_fit(q, A, q.bpre ? nullptr : B);
    if (!q.bpre || fit == FIT_FAST) {
      const size_t room = workspace ? workspace_bytes : 0;
      Problem e;
      int v = q.bpre ? (int)CASCMM_ERR_BAD_FORMAT : select_rounded_up(q, fit, room, &e);
      if (v < 0) {
        e = q;
        v = select_variant(q, fit, 1, room);
      }
      if (v >= 0 && table()[v].kind == KIND_F8K64)
        return gemm_impl(1, &A, &B, &C, bias ? &bias1 : nullptr, e, nullptr, workspace, workspace_bytes, (hipStream_t)stream, v,
                         exps_out, b_exp);
    }
  }
  // any other kernel: the one-launch search, then the GEMM with its result
  const int se = cascmm_tensor_exps(A, M, K, lda, CASCMM_DT_F32, b_exp, exps_out, scratch, stream);
  if (se != CASCMM_OK) return se;
  if (!b_exp) {
    // (exps_out[1] must be defined: a NULL b_exp means e_B = 0)
    hipError_t err = hipSuccess;
    CASCMM_LAUNCH(err, amax_begin_kernel, dim3(1), dim3(1), 0, (hipStream_t)stream, exps_out + 1);
    if (err != hipSuccess) return CASCMM_ERR_LAUNCH;
  }
  return gemm_impl(1, &A, &B, &C, bias ? &bias1 : nullptr, q, exps_out, workspace, workspace_bytes, (hipStream_t)stream, -1);
}

int cascmm_split_terms(const void* x, float* out, int64_t n, int dtype, int fmt, int terms, int tensor_exp,
                       void* stream) {
  if (n < 0) return CASCMM_ERR_BAD_SHAPE;
  if (n == 0) return CASCMM_OK;
  if (!x || !out) return CASCMM_ERR_NULL_POINTER;
  if (dtype != CASCMM_DT_F32) return CASCMM_ERR_BAD_DTYPE;
  hipStream_t s = (hipStream_t)stream;
  if (fmt == CASCMM_FMT_BF16) return launch_split<CASCMM_DT_F32, CASCMM_FMT_BF16>(x, out, n, terms, tensor_exp, s);
  if (fmt == CASCMM_FMT_FP16) return launch_split<CASCMM_DT_F32, CASCMM_FMT_FP16>(x, out, n, terms, tensor_exp, s);
  if (fmt == CASCMM_FMT_FP8) return launch_split<CASCMM_DT_F32, CASCMM_FMT_FP8>(x, out, n, terms, tensor_exp, s);
  return CASCMM_ERR_BAD_FORMAT;
}

const char* cascmm_strerror(int status) {
  switch (status) {
    case CASCMM_OK: return "ok";
    case CASCMM_ERR_NULL_POINTER: return "null pointer argument";
    case CASCMM_ERR_BAD_SHAPE: return "bad shape or leading dimension";
    case CASCMM_ERR_BAD_DTYPE: return "unsupported element type";
    case CASCMM_ERR_BAD_FORMAT: return "unsupported format / terms / products combination";
    case CASCMM_ERR_WORKSPACE: return "workspace missing or too small";
    case CASCMM_ERR_ALIGNMENT: return "pointer not aligned to its element size";
    case CASCMM_ERR_LAUNCH: return "HIP launch failed";
    case CASCMM_ERR_BAD_VARIANT: return "kernel variant unknown or unable to run this problem";
    case CASCMM_ERR_TOO_LARGE: return "dimension too large";
    case CASCMM_ERR_SCRATCH_LIMIT: return "problem needs more scratch than the library's built-in buffer holds (use cascmm_gemm with a workspace)";
    default: return "unknown status";
  }
}

int cascmm_selftest(void) {
  int bad = 0;
  const auto& t = table();
  for (const TunedCost& c : kTuned) {
    int hits = 0;
    for (const VariantDesc& d : t) hits += strcmp(c.name, d.name) == 0 ? 1 : 0;
    bad += hits == 1 ? 0 : 1;
  }
  std::vector<CallCost> calls(std::begin(kCallCost), std::end(kCallCost));
  calls.insert(calls.end(), std::begin(kGatedCost), std::end(kGatedCost));
  for (const CallCost& c : calls) {
    int hits = 0;
    for (const VariantDesc& d : t) hits += strcmp(c.name, d.name) == 0 ? 1 : 0;
    bad += hits == 1 ? 0 : 1;
  }
  for (size_t i = 0; i < t.size(); ++i)
    for (size_t j = i + 1; j < t.size(); ++j) bad += strcmp(t[i].name, t[j].name) == 0 ? 1 : 0;
  return bad;
}

// ---- chained feed-forward: both operands as slots -------------------------------------------------
size_t cascmm_left_slots_bytes(int64_t M, int64_t K) {
  if (M <= 0 || K <= 0 || K % 16 != 0) return 0;
  int64_t mk = 0, bytes = 0;
  if (__builtin_mul_overflow(M, K, &mk) || __builtin_mul_overflow(mk, (int64_t)4, &bytes)) return 0;
  return (size_t)bytes;
}

int cascmm_prepare_left(const void* A, int64_t M, int64_t K, int64_t lda, void* out, size_t out_bytes, void* stream) {
  if (M < 0 || K < 0 || lda < K || K % 16 != 0) return CASCMM_ERR_BAD_SHAPE;
  if (M > INT32_MAX || K > INT32_MAX) return CASCMM_ERR_TOO_LARGE;
  if (M == 0 || K == 0) return CASCMM_OK;
  if (!A || !out) return CASCMM_ERR_NULL_POINTER;
  if (!aligned_to(A, 16) || !aligned_to(out, 16) || lda % 4 != 0) return CASCMM_ERR_ALIGNMENT;
  const size_t need = cascmm_left_slots_bytes(M, K);
  if (need == 0 || need > (size_t)INT32_MAX) return CASCMM_ERR_TOO_LARGE;
  if (out_bytes < need) return CASCMM_ERR_WORKSPACE;
  return launch_prepare_left((const float*)A, (int)M, (int)K, lda, out, (hipStream_t)stream);
}

int cascmm_prepare_weight_chained(const void* B, int64_t K, int64_t N, int64_t ldb, void* out, size_t out_bytes, void* stream) {
  if (K < 0 || N < 0 || ldb < N || K % 16 != 0) return CASCMM_ERR_BAD_SHAPE;
  if (K > INT32_MAX || N > INT32_MAX) return CASCMM_ERR_TOO_LARGE;
  if (K == 0 || N == 0) return CASCMM_OK;
  if (!B || !out) return CASCMM_ERR_NULL_POINTER;
  if (!aligned_to(out, 16)) return CASCMM_ERR_ALIGNMENT;
  if (out_bytes < (size_t)prepared_bytes(K, N, CASCMM_FMT_BF16, 2)) return CASCMM_ERR_WORKSPACE;
  return launch_prepare<CASCMM_DT_F32, CASCMM_FMT_BF16>(B, (int)K, (int)N, ldb, 2, nullptr, (u32x4*)out, (hipStream_t)stream, 2);
}

int cascmm_gemm_glu_chained(const void* A, const void* B, int b_prepared, void* out_slots, size_t out_bytes, const void* bias,
                            int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, void* stream) {
  if (N % 64 != 0) return CASCMM_ERR_BAD_SHAPE;
  Problem q{M, N, K, lda, b_prepared ? N : ldb, N / 2, CASCMM_DT_F32, CASCMM_FMT_BF16, 2, CASCMM_PROD_TRI};
  q.bpre = b_prepared != 0;
  q.glu = true;
  q.glu_slots = true;
  const int st = check_problem(q);
  if (st != CASCMM_OK) return st;
  if (M == 0 || N == 0) return CASCMM_OK;
  if (!out_slots) return CASCMM_ERR_NULL_POINTER;
  if (!aligned_to(out_slots, 16)) return CASCMM_ERR_ALIGNMENT;
  const size_t need = cascmm_left_slots_bytes(M, N / 2);
  if (need == 0 || need > (size_t)INT32_MAX) return CASCMM_ERR_TOO_LARGE;
  if (out_bytes < need) return CASCMM_ERR_WORKSPACE;
  return gemm_impl(1, &A, &B, &out_slots, bias ? &bias : nullptr, q, nullptr, nullptr, 0, (hipStream_t)stream, -1);
}

int cascmm_chained_supported(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K < 16 || K % 16 != 0) return 0;
  if (M > INT32_MAX || N > INT32_MAX || K > INT32_MAX) return 0;
  if (beyond_i32(M, K, 4) || beyond_i32(N, K, 4)) return 0;   // both slot buffers below 2 GiB
  return 1;
}

int cascmm_gemm_chained(const void* Aslots, const void* Bslots, void* C, const void* bias, int64_t M, int64_t N, int64_t K,
                        int64_t ldc, void* stream) {
  if (M < 0 || N < 0 || K < 0 || ldc < N) return CASCMM_ERR_BAD_SHAPE;
  if (M == 0 || N == 0) return CASCMM_OK;
  if (!cascmm_chained_supported(M, N, K)) return CASCMM_ERR_BAD_FORMAT;
  if (!Aslots || !Bslots || !C) return CASCMM_ERR_NULL_POINTER;
  if (!aligned_to(Aslots, 16) || !aligned_to(Bslots, 16) || !aligned_to(C, 4) || !aligned_to(bias, 4)) return CASCMM_ERR_ALIGNMENT;
  if (beyond_i32(ldc, SlotK::BM, 4)) return CASCMM_ERR_TOO_LARGE;
  SlotKParams q;
  memset(&q, 0, sizeof(q));
  q.a = Aslots; q.b_slots = Bslots; q.C = (float*)C; q.bias = (const float*)bias;
  q.M = (int)M; q.N = (int)N; q.K = (int)K; q.ldc = ldc;
  return launch_slotk(q, 0, (hipStream_t)stream);
}

int cascmm_version(void) { return CASCMM_VERSION; }

}  // extern "C"
