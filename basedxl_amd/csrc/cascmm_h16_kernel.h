// Plain 16-bit GEMM (fp16 or bf16 tensors as ONE term of their own format, fp32 accumulation; gfx950).
//
// Eight consecutive elements of a row of A already are one lane's MFMA operand, and so is one 16-byte operand
// slot of a prepared B (cascmm_prepare_weight); a raw B [K][N] is transposed by the LDS itself on the way to the
// registers (ds_read_b64_tr_b16: sixteen lanes read 4 rows x 16 columns and every lane gets one column's four k).
// So nothing passes the VALU: every operand byte goes memory -> LDS by `buffer_load ... lds` and LDS -> MFMA.
//
// Workgroup: four waves, one per SIMD, WM x WN over the tile (WK = 2: two wave groups take alternate 16-k slices
// of every stage and meet in LDS at the end).  NS stages of BK k in LDS, one barrier per stage.  It sits in front of
// a stage's last slice, whose fragments are in registers by then: behind it stage s + 1 has landed, so the last
// slice's MFMAs hide the first fragment reads of the next stage, and the buffer of stage s is free, so the loads of
// stage s + NS start at once: NS - 1 stages are in flight (with the barrier at the top of a stage it was one less).
//
// What bounds it: one product per element leaves three times fewer MFMA cycles per byte than the two-term
// cascade, so a tile is as good as its bytes per multiply-add: (BM + BN) x 2 bytes per k through the CU's share
// of the L2s against BM x BN / 2048 matrix cycles.  Measured (fp16, weight prepared / raw, graph replay, all on one card, others are up to a
// tenth faster; in brackets before rows of A came in whole lines, sums stayed in place and fragments were read earlier): 2048 x 1280 x
// 10240 on 256 x 320 52.3 / 52.8 us (62.4 / 64.4), its loop at the board's power with random operands (zeros: a third faster); 4096^3 on
// 256 x 256 115.3 / 114.4 us (121.4 / 123.2); 8192 x 2560 x 640 33.7 / 34.3 us (33.7 / 35.0); 2048^3 on 128 x 128 22.3 / 22.6 us (22.6 /
// 23.7), its loop at 66 bytes per ns and CU from the L2s; 2048 x 1280 x 1280 13.3 / 14.0 us (13.5 / 15.0); 512 x 1280 x 1280 on 64 x 64 8.2 /
// 9.0 us (8.4 / 9.5); gated 2048 x 1280 x 10240 56.2 (60.2), 8192 x 640 x 5120 66.1 (69.6).  Kernel times and counters of the earlier state:
// profiles/cascmm_h16_kernel_fp16.txt.
//
// The MFMAs take their operands swapped (B first): a lane then holds ONE ROW of C and four consecutive columns
// per register quad, which are packed to 8 bytes, turned row-wise through LDS and stored 16 bytes per lane.
#pragma once
#include <type_traits>

#include "cascmm_ksplit.h"

namespace cascmm {

template <int WM_, int WN_, int WK_, int MT_, int NTL_, int BK_, int NS_>
struct H16 {
  static constexpr int WM = WM_, WN = WN_, WK = WK_, MT = MT_, NTL = NTL_, BK = BK_, NS = NS_, NT = 256;
  static constexpr int WTM = 32 * MT, WTN = 32 * NTL, BM = WM * WTM, BN = WN * WTN;
  // 32-k stages take half a 128-byte line of a row of A: its rows are loaded for two stages at once
  static constexpr bool PAIR = BK == 32;
  static constexpr int AK = PAIR ? 2 * BK : BK;      // k of a row of A that are loaded together
  static constexpr int KG = AK / 8;                  // 16-byte chunks of that
  static constexpr int SLW = BK / 16 / WK;           // 16-k slices of a stage that a wave multiplies
  static constexpr int A_BUF = BM * AK * 2, B_STAGE = BN * BK * 2;
  static constexpr int A_STEP = PAIR ? 0 : A_BUF + B_STAGE, B_STEP = PAIR ? B_STAGE : A_STEP;   // from one stage's LDS to the next one's
  static constexpr int B_AREA = PAIR ? 2 * A_BUF : A_BUF;   // (pairs: two of A, then the stages of B)
  static constexpr int A_LOADS = A_BUF / 4096, B_LOADS = B_STAGE / 4096, LOADS = A_LOADS + B_LOADS;   // per wave: A (pairs: of two stages), B of a stage
  static constexpr int OUT_ROW = WTN * 2 + 16;       // bytes of a row of C in the store's LDS area (padded: banks)
  static constexpr int SUM_WAVE = WK == 2 ? (NTL + 1) / 2 * 4096 : 0;   // the other wave group's sums of this wave's blocks
  static constexpr int OUT_WAVE = 32 * OUT_ROW + WTN * 4 > SUM_WAVE ? 32 * OUT_ROW + WTN * 4 : SUM_WAVE;
  static constexpr int RING_BYTES = PAIR ? B_AREA + NS * B_STAGE : NS * B_STEP;
  static constexpr int LDS_BYTES = RING_BYTES > 4 * OUT_WAVE ? RING_BYTES : 4 * OUT_WAVE;
  // tile rows an XCD walks down before moving one tile to the right: about square in bytes
  static constexpr int GROUP_M = BN >= 2 * BM ? 8 : 4;
  static_assert(WM * WN * WK == 4 && (BK == 32 || BK == 64) && SLW % 2 == 0 && NS >= 3, "layout");
  // (pairs: the prologue issues the first pair of A before all of B and one pair more, so the wait counts at the first stages hold for four
  // stages only: with five, two pairs would be taken to be in flight behind stage 1's B, which is read then)
  static_assert(!PAIR || (WK == 1 && NS == 4 && A_LOADS % 2 == 0), "pairs");
  static_assert(A_BUF % 4096 == 0 && B_STAGE % 4096 == 0, "every wave issues the same number of loads");
  static_assert((NS - 1) * LOADS <= 63, "the wait counter has six bits");
  static_assert(LDS_BYTES <= 160 * 1024, "LDS");
};

typedef __attribute__((address_space(3))) void* h16_lds_ptr;

// (functions of their own: in a call whose arguments depend on a template parameter the host pass of the compiler
// rejects the builtin without a message and then leaves out the kernel's launch stub)
__device__ __forceinline__ void h16_load_lds(__amdgpu_buffer_rsrc_t rsrc, unsigned char* dst, int voffset, int soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (h16_lds_ptr)dst, 16, voffset, soffset, 0, 0);
}
// Transposing read, as assembly: in front of the builtin the compiler waits for every `buffer_load ... lds` in
// flight (it cannot see that they write other buffers), which serialised loads and MFMAs.  The caller waits for the
// result itself.
template <int OFF> __device__ __forceinline__ u32x2 h16_read_tr(unsigned lds_addr) {
  u32x2 v;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(lds_addr), "n"(OFF));
  return v;
}

// MFMA with the accumulator in ordinary vector registers: there are sixteen blocks' worth of accumulation registers,
// which is where the compiler puts every accumulator of an MFMA that it selects itself
template <int FMT> __device__ __forceinline__ void h16_mfma_v(u32x4 a, u32x4 b, f32x16& c) {
  if constexpr (FMT == CASCMM_FMT_BF16) asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
  else asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
}

template <int FMT> struct H16Elem;
template <> struct H16Elem<CASCMM_FMT_BF16> { typedef __bf16 T; static constexpr int DT = CASCMM_DT_BF16; };
template <> struct H16Elem<CASCMM_FMT_FP16> { typedef _Float16 T; static constexpr int DT = CASCMM_DT_F16; };

// Host-checked: the rows of A start on dwords and are whole 16-byte chunks, zeros past K (K % 8 == 0, or padded), 512 of
// them below 2 GiB; RAWB = 0: B prepared (prepared_kgroups(K) x N slots, zeros beyond K), 2 GiB not reached with K rounded up to 64; RAWB = 1: B [K][ldb] with
// N % 2 == 0 and rows on dwords, K * ldb * 2 below 2 GiB.  Any M and N: rows and columns past the edge are loaded as zeros or as
// some other column's values and not stored.  grid.y: the problem of a group.  k_splits > 1: K in splits of k_per (a
// multiple of 64), fp32 sums to the workspace instead of a result, see cascmm_ksplit.h.
// GLU: gated store (see GroupParams; RAWB = 0, NTL even: a wave owns whole value / gate pairs of blocks).
template <class T, int FMT, int RAWB, int GLU>
__global__ __launch_bounds__(T::NT, 1) void cascmm_h16_kernel(const GroupParams p) {
  typedef typename H16Elem<FMT>::T E;
  typedef IoType<H16Elem<FMT>::DT> Io;
  static_assert(!GLU || (!RAWB && T::NTL % 2 == 0), "the gated store pairs a wave's blocks");
  extern __shared__ __attribute__((aligned(1024))) unsigned char h16_smem[];
  unsigned char* smem = h16_smem;
  const int tid = threadIdx.x, lane = tid & 63, l31 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = wave / (T::WM * T::WN), wmn = wave % (T::WM * T::WN);
  const int wm0 = (wmn / T::WN) * T::WTM, wn0 = (wmn % T::WN) * T::WTN;
  const int prob = blockIdx.y;
  // The arguments that A's first loads need, all requested here: left to themselves the reads sink to their uses and wait one
  // behind the other, which with a descriptor per tile was 0.2 us of a call with new operands (2048 x 1280 x 1280, three
  // weights in turn: 12.52 us, so 12.26; 512 x 1280 x 1280 6.7 us, with N among them 7.0).
  int tiles_m = p.tiles_m, tiles_n = p.tiles_n, k_splits = p.k_splits, M = p.M, K_all = p.K, k_per = p.k_per, lda = (int)p.lda;
  const void *A = p.A[prob], *B = p.B[prob];
  asm volatile("" : "+s"(tiles_m), "+s"(tiles_n), "+s"(k_splits), "+s"(M), "+s"(K_all), "+s"(k_per), "+s"(lda), "+s"(A), "+s"(B));
  int tm, tn;
  tile_coords(blockIdx.x, tiles_m * k_splits, tiles_n, tm, tn, T::GROUP_M < tiles_m || k_splits == 1 ? T::GROUP_M : tiles_m);
  const int split = ksplit_of_row(tm, tiles_m, k_per, K_all);
  const int m0 = tm * T::BM, n0 = tn * T::BN;
  const int k0 = split * k_per;
  const int K = K_all - k0 < k_per ? K_all - k0 : k_per;
  const int ksteps = T::PAIR ? (K + 63) / 64 * 2 : (K + T::BK - 1) / T::BK;

  // A's buffer starts with the tile's first row, so A itself may be of any size: the offsets inside a tile stay below
  // 512 rows.  Rows past M read as zero (it ends with row M - 1), and so does everything past B's last row or slot row
  const int kgs = (K + 31) / 32 * 4;   // prepared_kgroups
  const int rows = M - m0 < T::BM ? M - m0 : T::BM;
  const int a_bytes = ((rows - 1) * lda + (K + 7) / 8 * 8) * 2;
  const int64_t b_bytes = RAWB ? ((int64_t)(K - 1) * p.ldb + p.N) * 2 : (int64_t)kgs * p.N * 16;
  const int64_t b_first = RAWB ? (int64_t)k0 * p.ldb * 2 : (int64_t)(k0 / 8) * p.N * 16;
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)((const E*)A + (int64_t)m0 * lda + k0), 0, a_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void*)((const char*)B + b_first), 0, (int)b_bytes, 0x00020000);

  // ---- loads: this wave's kilobytes of a stage ----
  // A: row r of the BM x 64 block at r * 128 bytes; position pos of a row holds chunk (pos - r / 2) mod 8: the sixteen
  // lanes a 16-byte LDS read serves together hit every bank once
  static_assert(T::KG == 8, "rotation");
  constexpr int RSH = 1;
  int a_voff[T::A_LOADS], a_k[T::A_LOADS];   // (a_k: pairs have two values only, even and odd loads)
#pragma unroll
  for (int j = 0; j < T::A_LOADS; ++j) {
    const int row = (wave * T::A_LOADS + j) * (64 / T::KG) + lane / T::KG;
    const int chunk = (lane % T::KG - (row >> RSH)) & (T::KG - 1);   // (rows / 2 mod 8: load j's lanes as load j + 2's)
    a_k[j] = chunk * 8;
    a_voff[j] = row < rows ? (row * lda + chunk * 8) * 2 : 0x7FFFFFFF;
  }
  // B prepared: slot (k group, column) at (kg * BN + column) * 16.  B raw: row k at 2 BN k bytes, its 16-byte chunks
  // (8 columns) permuted by an XOR so that the four rows of a transposing read lie on different banks
  constexpr int CPR = T::BN / 8;   // chunks per row of raw B
  constexpr int XSH = (T::BN * 2) % 256 == 0 ? 0 : (T::BN * 2) % 256 == 128 ? 1 : 2;
  auto xor_of = [](int row) { return XSH == 0 ? 4 * (row & 3) : XSH == 1 ? 4 * ((row >> 1) & 1) : 0; };
  int b_voff[T::B_LOADS];
#pragma unroll
  for (int j = 0; j < T::B_LOADS; ++j) {
    const int s = (wave * T::B_LOADS + j) * 64 + lane;
    if (RAWB) b_voff[j] = (int)(((int64_t)(s / CPR) * p.ldb + n0 + ((s % CPR) ^ xor_of(s / CPR)) * 8) * 2);
    else b_voff[j] = ((s / T::BN) * p.N + n0 + s % T::BN) * 16;
  }
  const int b_step = RAWB ? (int)(T::BK * p.ldb * 2) : T::BK / 8 * p.N * 16;
  // load j of A's rows from stage `step` on (pairs: an even one)
  auto issue_a = [&](int step, int buf, int j) {
    // (past K: beyond the buffer's end, zeros)
    const int v = a_k[T::PAIR ? j & 1 : j] < K - step * T::BK ? a_voff[j] : 0x7FFFFFFF;
    h16_load_lds(ra, smem + (T::PAIR ? (step & 2) * (T::A_BUF / 2) : buf * T::A_STEP) + (wave * T::A_LOADS + j) * 1024, v, step * T::BK * 2);
  };
  auto issue_b = [&](int step, int buf, int j) {
    const int bs = (step < ksteps ? step : ksteps) * b_step;
    h16_load_lds(rb, smem + T::B_AREA + buf * T::B_STEP + (wave * T::B_LOADS + j) * 1024, b_voff[j], bs);
  };
  // load j of the window that stage `s` opens (its buffers are free then): A and B of stage s + NS; pairs: B of that stage,
  // and, odd stages before it, the rows of A of the pair after the next
  auto issue = [&](int s, int buf, auto odd_tag, int j) {
    constexpr bool A = !T::PAIR || decltype(odd_tag)::value != 0;
    if (A && j < T::A_LOADS) issue_a(T::PAIR ? s + 3 : s + T::NS, buf, j);
    else issue_b(s + T::NS, buf, A ? j - T::A_LOADS : j);
  };

  // ---- fragments: slice sl of a stage ----
  const int a_row = wm0 + l31;
  constexpr int SLICES = T::PAIR ? 2 * T::SLW : T::SLW;
  int a_frag[SLICES];
#pragma unroll
  for (int x = 0; x < SLICES; ++x) {
    const int sl = T::WK == 1 ? x : 2 * x + wk;
    a_frag[x] = a_row * T::AK * 2 + ((2 * sl + g + (a_row >> RSH)) & (T::KG - 1)) * 16;
  }
  // raw B: lane i = lane % 16 of a group of sixteen reads row 8 g + i / 4 (+ 4), columns 16 (lane / 16 % 2) + 4 (i % 4)
  int b_frag[RAWB ? T::NTL : 1];
  const int b_slice = RAWB ? 16 * T::BN * 2 : 2 * T::BN * 16;
  if (RAWB) {
    const int i = lane & 15, row = 8 * g + (i >> 2);
#pragma unroll
    for (int ni = 0; ni < T::NTL; ++ni) {
      const int chunk = (wn0 + ni * 32) / 8 + 2 * ((lane >> 4) & 1) + ((i & 3) >> 1);
      b_frag[ni] = T::B_AREA + wk * b_slice + row * T::BN * 2 + (chunk ^ xor_of(row)) * 16 + (i & 1) * 8;
    }
  } else {
    b_frag[0] = T::B_AREA + wk * b_slice + (g * T::BN + wn0 + l31) * 16;
  }
  // How many slices ahead fragments are read: a slice of few MFMAs is over before the next one's are there.  Two on 128 x 128 (loop of 2048^3
  // 23.7 -> 23.0 k cycles); the smaller tiles gained nothing, the larger ones have MFMAs
  // enough, and raw, the reads written as assembly must not be in flight where the loop closes.
  constexpr int PF = !T::PAIR && T::WK == 1 && !RAWB && T::MT * T::NTL == 4 ? 2 : 1;
  u32x4 Af[2 * PF][T::MT], Bf[2 * PF][T::NTL];
  auto read = [&](const unsigned char* sa, int xa, const unsigned char* st, int x, int buf, int r) {   // r: A's blocks, then B's
    if (r < T::MT) Af[buf][r] = *(const u32x4*)(sa + a_frag[xa] + r * 32 * T::AK * 2);
    else if (RAWB) {
      const unsigned src = (unsigned)(uintptr_t)(h16_lds_ptr)(st + b_frag[r - T::MT] + x * T::WK * b_slice);
      const u32x2 lo = h16_read_tr<0>(src), hi = h16_read_tr<8 * T::BN>(src);   // (four rows further down)
      Bf[buf][r - T::MT] = (u32x4){lo[0], lo[1], hi[0], hi[1]};
    } else {
      Bf[buf][r - T::MT] = *(const u32x4*)(st + b_frag[0] + x * T::WK * b_slice + (r - T::MT) * 512);
    }
  };

#define H16_FENCE() __builtin_amdgcn_sched_barrier(0)
  f32x16 acc[T::MT][T::NTL];
  // Loads of a window: the first P with the last PF slices of its stage, the others with the first slices of the next one.
  typedef std::integral_constant<int, 0> Even;
  typedef std::integral_constant<int, 1> Odd;
  constexpr int WIN[2] = {T::PAIR ? T::B_LOADS : T::LOADS, T::LOADS};   // of an even stage, of an odd one
  constexpr int P[2] = {(PF * WIN[0] + T::SLW - 1) / T::SLW, (PF * WIN[1] + T::SLW - 1) / T::SLW};
  constexpr int FIRST = T::SLW - PF;   // the slice that a stage's barrier stands in front of
  static_assert(PF == 1 || (T::SLW == 2 * PF && !T::PAIR), "a slice's fragments have their buffer");
  // (as if stages -NS ... -1 had opened their windows)
  if constexpr (T::PAIR) {
#pragma unroll
    for (int j = 0; j < T::A_LOADS; ++j) issue_a(0, 0, j);
  }
#pragma unroll
  for (int s = 0; s < T::NS - 1; ++s)
#pragma unroll
    for (int j = 0; j < WIN[0]; ++j) issue(s - T::NS, s, Even(), j);
#pragma unroll
  for (int j = 0; j < P[1]; ++j) issue(-1, T::NS - 1, Odd(), j);
  H16_FENCE();
  // (cleared while the first loads are in flight; the empty statements make the zeros real here)
#pragma unroll
  for (int mi = 0; mi < T::MT; ++mi)
#pragma unroll
    for (int ni = 0; ni < T::NTL; ++ni) {
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[mi][ni][e] = 0.f;
      if (mi * T::NTL + ni < 16) asm volatile("" : "+a"(acc[mi][ni]));
      else asm volatile("" : "+v"(acc[mi][ni]));
    }
  H16_FENCE();
  // What may be in flight: while stage 0 is waited for, and at the barrier of an even and of an odd stage for the next one (pairs:
  // an odd one waits for the pair of A too, which only two stages of B are younger than)
  constexpr int W0 = (T::NS - 2) * WIN[0] + P[1];
  constexpr int W1[2] = {(T::NS - 2) * WIN[0] + (T::PAIR ? (T::NS - 1) / 2 * T::A_LOADS : 0), (T::PAIR ? 2 : T::NS - 2) * WIN[0]};
  static_assert(W0 <= 63 && W1[0] <= 63, "the wait counter has six bits");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (W0 & 0xF) | ((W0 >> 4) << 14));   // stage 0 has landed
  __builtin_amdgcn_s_barrier();
  H16_FENCE();
#pragma unroll
  for (int r = 0; r < PF * (T::MT + T::NTL); ++r) read(smem, r / (T::MT + T::NTL), smem, r / (T::MT + T::NTL), r / (T::MT + T::NTL), r % (T::MT + T::NTL));
  if (RAWB) __builtin_amdgcn_s_waitcnt(0xC07F);

  int cur = 0, before = T::NS - 1;   // LDS buffers of this stage and of the one before it
  // one stage; odd_tag: pairs' second
  auto stage = [&](int s, auto odd_tag) {
    constexpr int ODD = decltype(odd_tag)::value;
    typedef std::integral_constant<int, T::PAIR ? 1 - ODD : 0> Before;   // the stage before it
    const int nx = cur == T::NS - 1 ? 0 : cur + 1;
    const unsigned char* st0 = smem + cur * T::B_STEP;
    const unsigned char* st1 = smem + nx * T::B_STEP;
    const unsigned char* sa0 = T::PAIR ? smem + (s & 2) * (T::A_BUF / 2) : st0;
    const unsigned char* sa1 = !T::PAIR ? st1 : ODD ? smem + ((s + 1) & 2) * (T::A_BUF / 2) : sa0;
    constexpr int XA = ODD * T::SLW, XN = T::PAIR && !ODD ? T::SLW : 0;   // A's first slice of this stage, of the next one
#pragma unroll
    for (int x = 0; x < T::SLW; ++x) {
      const int buf = x % (2 * PF), to = (x + PF) % (2 * PF);
      const bool late = x >= FIRST;
      if (x == FIRST) {
        // own loads of stage s + 1 have landed and own reads of stage s are over, then everybody's
        __builtin_amdgcn_s_waitcnt(0x0070 | (W1[ODD] & 0xF) | ((W1[ODD] >> 4) << 14));
        __builtin_amdgcn_s_barrier();
        H16_FENCE();
      }
      // between the MFMAs of a slice: first the fragment reads of the next one, then this slice's share of the loads
      constexpr int READS = T::MT + T::NTL, MF = T::MT * T::NTL, PB = P[Before::value], WB = WIN[Before::value];
      const int l0 = late ? (x - FIRST) * P[ODD] / PF : PB + x * (WB - PB) / FIRST, l1 = late ? (x - FIRST + 1) * P[ODD] / PF : PB + (x + 1) * (WB - PB) / FIRST;
      // gaps that take the reads.  Of four, the first two: spread over all of them the last one is waited for (loop of 2048^3 on 128 x 128
      // raw 32.4 -> 28.2 k cycles, prepared 25.4 -> 23.7; with two reads a gap 64 x 160 raw lost 7 %, 128 x 160 4 %)
      constexpr int RG = MF == 4 ? 2 : MF >= READS ? READS : (MF + 1) / 2;
#pragma unroll
      for (int mf = 0; mf < MF; ++mf) {
        const int ni = mf / T::MT, mi = mf % T::MT;
        auto multiply = [&]() {
          if (mi * T::NTL + ni < 16)
            acc[mi][ni] = Lowp<FMT>::mfma(Lowp<FMT>::operand(Bf[buf][ni], 0), Lowp<FMT>::operand(Af[buf][mi], 0), acc[mi][ni]);
          else
            h16_mfma_v<FMT>(Bf[buf][ni], Af[buf][mi], acc[mi][ni]);
          H16_FENCE();
        };
        // (Of one or two MFMAs a slice's reads go out first: behind them the next slice waited for all of its reads.  512 x 1280 x 1280 on 64 x
        // 64 9.1 -> 8.35 us, raw 9.6 -> 9.0; 1000 x 2560 x 1280 on 128 x 64 17.1 -> 16.9; of four, raw 128 x 128 lost 3 %)
        if (MF > 2) multiply();
#pragma unroll
        for (int r = 0; r < READS; ++r) {
          if (r * RG / READS != mf) continue;
          if (late) read(sa1, XN + x - FIRST, st1, x - FIRST, to, r);
          else read(sa0, XA + x + PF, st0, x + PF, to, r);
        }
#pragma unroll
        for (int j = 0; j < T::LOADS; ++j) {
          if (j < l0 || j >= l1 || (j - l0) * MF / (l1 - l0) != mf) continue;
          if (late) issue(s, cur, odd_tag, j);
          else issue(s - 1, before, Before(), j);
        }
        H16_FENCE();
        if (MF <= 2) multiply();
      }
      if (RAWB) {   // (results of reads written as assembly: the compiler does not wait for them)
        __builtin_amdgcn_s_waitcnt(0xC07F);
        H16_FENCE();
      }
    }
    before = cur;
    cur = nx;
  };
  for (int s = 0; s < ksteps; s += T::PAIR ? 2 : 1) {
    stage(s, Even());
    if constexpr (T::PAIR) stage(s + 1, Odd());
  }
#undef H16_FENCE
  __builtin_amdgcn_s_waitcnt(0x0F70);   // the loads past the last stage have landed before LDS is used again
  // (the MFMAs written as assembly are invisible to the compiler's hazard handling)
  asm volatile("s_nop 7\n s_nop 7\n s_nop 7" ::: "memory");
  __syncthreads();

  // ---- two wave groups: each finishes its share of the blocks, the other one's sums come through LDS ----
  constexpr int OB = GLU ? T::NTL / 2 : T::NTL;              // 32-column blocks of C per row block
  constexpr int HALF = T::WK == 2 ? (OB + 1) / 2 : OB;       // wave group 0: blocks 0 .. HALF - 1, group 1: the others
  unsigned char* area = smem + wave * T::OUT_WAVE;
  // (The store is straight-line code that every wave runs once, so its length is time: instructions come from L2 at
  // some 10 KB per us.  With or without a bias, 16-byte or single stores are therefore separate copies.)
  auto finish = [&](auto first_tag, auto count_tag, auto bias_tag) {
    constexpr int B0 = decltype(first_tag)::value, NB = decltype(count_tag)::value;
    constexpr bool BIAS = decltype(bias_tag)::value != 0;
    if constexpr (!BIAS && !GLU) {
      if (p.k_splits > 1) {   // (a lane's four consecutive columns of its row; the wave's rows of a block, 32 bytes each)
        const int row = (p.N + 3) & ~3, col0 = n0 + wn0 + 32 * B0;
        float* part = (float*)p.workspace + ((int64_t)split * p.M + m0 + wm0) * row + col0;
        const int64_t bytes = ((int64_t)(p.M - 1 - m0 - wm0) * row + (row - col0)) * 4;
        const i32x4 rp = make_rsrc(part, bytes < 0 ? 0 : bytes);
#pragma unroll
        for (int mi = 0; mi < T::MT; ++mi)
#pragma unroll
          for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const f32x16& v = acc[mi][B0 + b];
              const int col = 32 * b + 8 * q + 4 * g;
              llvm_raw_buffer_store_v4f32((f32x4){v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]}, rp,
                                          col0 + col < row ? ((mi * 32 + l31) * row + col) * 4 : 0x7FFFFFFF, 0, 0);
            }
        return;
      }
    }
    // ---- store: of block (mi, ni) a lane holds row 32 mi + l31, columns 32 ni + 8 q + 4 g + e in register 4 q + e ----
    const int no = GLU ? p.N >> 1 : p.N;
    const int oc0 = (GLU ? (n0 + wn0) >> 1 : n0 + wn0) + 32 * B0;
    float* bl = (float*)(area + 32 * T::OUT_ROW);   // the wave's bias values, in the order of its columns
    if constexpr (BIAS) {
      const E* bias = (const E*)p.bias[prob];
      for (int c = lane; c < NB * (GLU ? 64 : 32); c += 64) {
        // (gated: blocks alternate value and gate columns)
        const int col = GLU ? oc0 + (c >> 6) * 32 + (c & 31) : oc0 + c;
        bl[c] = col < no ? Io::load(bias + (GLU && (c & 32) ? no : 0) + col) : 0.f;
      }
    }
    E* C = (E*)p.C[prob] + (int64_t)(m0 + wm0) * p.ldc + oc0;
    // Stores of 16 bytes, of two elements or of one, as width and alignment of the rows allow, with 32-bit offsets over the wave's
    // rows; rows too far apart for those are addressed one by one.
    const bool near_rows = p.ldc * (2 * T::WTM) <= 0x7FFFFFFF;
    const bool vec = near_rows && (p.ldc & 7) == 0 && (no & 7) == 0 && ((uintptr_t)p.C[prob] & 15) == 0;
    const bool pairs = (p.ldc & 1) == 0 && (no & 1) == 0 && ((uintptr_t)p.C[prob] & 3) == 0;
    // rows past M fall beyond the end of the buffer and are dropped, columns past the last one are sent there too
    const int64_t c_bytes = ((int64_t)(p.M - 1 - m0 - wm0) * p.ldc + (no - oc0)) * 2;
    const i32x4 rc = make_rsrc(C, c_bytes < 0 ? 0 : c_bytes);
    const int ldc_bytes = (int)p.ldc * 2;
    constexpr int CHUNKS = 4 * NB, ITS = 2 * NB;   // 16-byte chunks of a row; of 32 rows, per lane
    // 32 rows in W elements a lane, eight reads and then eight stores at a time.  (One element behind the other, each store waiting for
    // its read, a width off 8 took 6016 x 2240 x 754 from the 27.6 us of 752 to 40, 4096 x 640 x 639 from 7.7 to 13.6.)
    auto narrow = [&](int mi, auto width_tag) {
      constexpr int W = decltype(width_tag)::value, PER_ROW = 32 * NB / W;
      typedef typename std::conditional<W == 2, unsigned, unsigned short>::type U;
#pragma unroll 1
      for (int i0 = lane; i0 < 32 * PER_ROW; i0 += 8 * 64) {
        U v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int i = i0 + 64 * u;
          v[u] = *(const U*)(area + (i / PER_ROW) * T::OUT_ROW + (i % PER_ROW) * (2 * W));
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int i = i0 + 64 * u, c = (i % PER_ROW) * W;
          const int voff = oc0 + c < no ? (mi * 32 + i / PER_ROW) * ldc_bytes + c * 2 : 0x7FFFFFFF;
          if constexpr (W == 2) llvm_raw_buffer_store_f32(__builtin_bit_cast(float, v[u]), rc, voff, 0, 0);
          else llvm_raw_buffer_store_i16(__builtin_bit_cast(short, v[u]), rc, voff, 0, 0);
        }
      }
    };
#pragma unroll
    for (int mi = 0; mi < T::MT; ++mi) {
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        // (The large tiles' sums stay in the accumulation registers up to here.  Left alone the compiler moves all of them to ordinary ones
        // behind the loop, through scratch memory what does not fit: 26 k cycles of store in place of 16 k on 256 x 320, 16 k in place of
        // 10 k on 256 x 256; gated, and of smaller tiles, its own order is the better one.)
        if (!GLU && T::MT * T::NTL >= 16 && mi * T::NTL + B0 + b < 16) asm volatile("" : "+a"(acc[mi][B0 + b]));
        // (a block's bias values at once: quad by quad, every quad waits for its own)
        f32x4 bv[4], bg[4];
        if constexpr (BIAS) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            bv[q] = *(const f32x4*)(bl + (GLU ? 64 : 32) * b + 8 * q + 4 * g);
            if constexpr (GLU) bg[q] = *(const f32x4*)(bl + 64 * b + 32 + 8 * q + 4 * g);
          }
        }
        auto sum = [&](int block, const f32x4* bias4, int q, int x) { return BIAS ? acc[mi][block][4 * q + x] + bias4[q][x] : acc[mi][block][4 * q + x]; };
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          typedef E e2 __attribute__((ext_vector_type(2)));
          float y[4];
          if constexpr (GLU) {
#pragma unroll
            for (int x = 0; x < 4; ++x) y[x] = sum(2 * b + 1, bg, q, x);
            gelu_values(y);
#pragma unroll
            for (int x = 0; x < 4; ++x) y[x] *= sum(2 * b, bv, q, x);
          } else {
#pragma unroll
            for (int x = 0; x < 4; ++x) y[x] = sum(B0 + b, bv, q, x);
          }
          const u32x2 out = {__builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){y[0], y[1]}, e2)),
                             __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){y[2], y[3]}, e2))};
          *(u32x2*)(area + l31 * T::OUT_ROW + (32 * b + 8 * q + 4 * g) * 2) = out;
        }
      }
      if (vec) {
        // (a few at a time: the reads' latency overlaps, the registers last)
        constexpr int GRP = ITS <= 8 ? ITS : ITS == 10 ? 5 : 4;
        static_assert(ITS % GRP == 0, "groups");
#pragma unroll
        for (int i0 = 0; i0 < ITS; i0 += GRP) {
          u32x4 v[GRP];
#pragma unroll
          for (int it = 0; it < GRP; ++it) {
            const int i = (i0 + it) * 64 + lane;
            v[it] = *(const u32x4*)(area + (i / CHUNKS) * T::OUT_ROW + (i % CHUNKS) * 16);
          }
#pragma unroll
          for (int it = 0; it < GRP; ++it) {
            const int i = (i0 + it) * 64 + lane, c = i % CHUNKS;
            llvm_raw_buffer_store_v4f32(__builtin_bit_cast(f32x4, v[it]), rc, oc0 + c * 8 < no ? (mi * 32 + i / CHUNKS) * ldc_bytes + c * 16 : 0x7FFFFFFF, 0, 0);
          }
        }
      } else if (near_rows) {
        if (pairs) narrow(mi, std::integral_constant<int, 2>{});
        else narrow(mi, std::integral_constant<int, 1>{});
      } else {
#pragma unroll 1
        for (int i = lane; i < 32 * NB * 32; i += 64) {
          const int row = i / (32 * NB), c = i % (32 * NB);
          const E h = *(const E*)(area + row * T::OUT_ROW + c * 2);
          if (m0 + wm0 + mi * 32 + row < p.M && oc0 + c < no) C[(int64_t)(mi * 32 + row) * p.ldc + c] = h;
        }
      }
    }
  };
  auto with_bias = [&](auto first, auto count) {
    if (p.bias[prob]) finish(first, count, std::integral_constant<int, 1>{});
    else finish(first, count, std::integral_constant<int, 0>{});
  };
  if constexpr (T::WK == 2) {
    static_assert(T::MT == 1 && !GLU, "one row block per wave");
    unsigned char* other = smem + (wave ^ (T::WM * T::WN)) * T::OUT_WAVE;
#pragma unroll
    for (int b = 0; b < T::NTL; ++b)
      if ((b < HALF) == (wk == 1))   // the other group's block
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x16& v = acc[0][b];
          *(f32x4*)(other + ((b % HALF) * 4 + q) * 1024 + lane * 16) = (f32x4){v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
        }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < T::NTL; ++b)
      if ((b < HALF) == (wk == 0))
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x4 o = *(const f32x4*)(area + ((b % HALF) * 4 + q) * 1024 + lane * 16);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[0][b][4 * q + e] += o[e];
        }
    if (wk == 0) with_bias(std::integral_constant<int, 0>{}, std::integral_constant<int, HALF>{});
    else with_bias(std::integral_constant<int, HALF>{}, std::integral_constant<int, OB - HALF>{});
  } else {
    with_bias(std::integral_constant<int, 0>{}, std::integral_constant<int, OB>{});
  }
}

}  // namespace cascmm
