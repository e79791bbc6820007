// Skinny problems (few rows, e.g. the two rows of a time embedding, the 77 or 154 text tokens of a cross-attention K/V
// projection) and small ones in ONE launch and without partial results in memory: K is split over the eight waves of a
// workgroup instead of over workgroups, so the partial sums meet in LDS.
//
// One workgroup computes a (W MB) x (W NB) tile of C over the whole K, in blocks of the 16 x 16 x 32 (W = 16) or
// 32 x 32 x 16 (W = 32) MFMA.  Wave w takes
// the 32-wide K steps w, w + 8, w + 16, ...; it streams its own operands and shares nothing with the other waves
// until the end, so the main loop has no barrier:
//   * A (32 k fp32 of a row are one 128-byte line) goes to the wave's private LDS ring without passing registers
//     (AL `buffer_load ... lds` of 1 KB, eight rows each: eight consecutive lanes fetch the eight 16-byte chunks
//     of one row, rotated inside the row so that the fragment reads spread over all banks);
//   * B needs no transposition: lane (c, g) of an MFMA wants B[k0 + 8 g + e][column c], e = 0..7, which is one
//     4-, 8- or 16-byte load per e straight into registers: the wave's NB column blocks are the columns NB c + nb.
// NS - 1 steps beyond the current one are in flight.  The values are split in registers right before their MFMAs, like
// in the large-tile kernel.  At the end the eight partial tiles are added in wave order through LDS (deterministic)
// and written with the bias.
//
// The shape is bound by what one CU can pull in, W (MB + NB) x K x 4 bytes, at the 64 bytes per clock of its vector
// memory path, by the instructions of the split (three per element with two bf16 terms, about eight with three fp16 or fp8
// terms) and by latencies, not by HBM (the weights are 10 MB) and not by the MFMAs.  A CU keeps about 0.4 requests per ns going,
// whatever it asks for (26 bytes per ns in 64-byte pieces of a row, 42 in 128-byte ones, 71 in 256-byte ones; more steps in
// flight change nothing), so few columns are spread over as many CUs as there are 16-wide tiles, and 64 x 64 tiles serve the
// problems of some 256 of them.  Measured (graph replay, us; in brackets the one 32 x 32 / 32 x 64 kernel before, whose steps stood
// behind branches): 2 x 1280 x 1280 4.2 (7.6), 2 x 320 x 1280 2.6 (4.9), 32 x 1024 x 384 3.6 (7.1), 128 x 1952 x 448 6.5 (10.3),
// 333 x 456 x 211 3.6 (5.7), 640^3 7.4 (10.6), 768^3 10.7 and 1024^3 13.6 (12.5 and 15.9 on the LDS-tiled kernel), 154 x 2048 x 1280
// 11.7 (11.4).  Three fp16 terms: 2 x 1280 x 1280 6.1 (12.8 on the 64 x 64 tile kernel with its K split), 38 x 256 x 448 3.3 (9.9), 154 x
// 2048 x 1280 17.3 (20.8), 333 x 456 x 211 5.1 (23.3 on the bounds-checked kernel); their accumulators fill the registers on tiles beyond
// 32 x 32.  Three fp8 terms, scales given: 2 x 1280 x 1280 6.3 (11.7), 18 x 2688 x 384 10.3 (20.4).  With the weight prepared, two 16-byte loads per step and 16 columns and half the instructions: 2 x 2816 x 1280 5.7 (9.3
// raw), 154 x 2048 x 1280 9.5, x 640 7.6, 77 x 2048 x 2560 9.5, 108 x 592 x 3155 6.3 (10.0 on the 64 x 80 tile, eager).
#pragma once
#include <type_traits>

#include "cascmm_f16k_kernel.h"

namespace cascmm {

// steps of a wave that have straight code, by the tile's size, and in cascmm_hwk_kernel.h
constexpr int wavek_straight(int area) { return area == 256 ? 8 : area == 512 ? 6 : area <= 2048 ? 4 : 2; }
constexpr int kHwkStraight = 4;

// AL: loads of A per step and wave (W MB / 8: all rows of the tile); B_LOADS: those of B
template <int W, int MB, int NB, int AL, int B_LOADS>
struct WaveK {
  static constexpr int BM = W * MB, BN = W * NB, BK = 32, NW = 8, NT = 512;
  static constexpr int KM = 512 / W, HALVES = BK / KM;     // k of an MFMA, MFMAs per step
  static constexpr int REGS = W * W / 64;                  // accumulator registers of a block
  static constexpr int LOADS = AL + B_LOADS;               // per wave and step
  static constexpr int NS = BM == 16 && LOADS <= 15 ? 5 : BM <= 32 ? (LOADS <= 20 ? 4 : 3) : 2;               // steps in LDS and registers
  static constexpr int STRAIGHT = wavek_straight(BM * BN);
  static constexpr int A_STAGE = AL * 1024;
  static constexpr int RING = NS * A_STAGE;                // per wave
  static constexpr int PART = BM * BN * 4;                 // a wave's partial tile
  static constexpr int LDS_BYTES = NW * (RING > PART ? RING : PART);
  static_assert((NS - 1) * LOADS <= 60, "the wait counter has six bits");
};

typedef __attribute__((address_space(3))) void* wavek_lds_ptr;

// 64 lanes x 16 bytes from a buffer straight into LDS at dst + 16 lane.  (Not called from the kernel
// template directly: in a call whose arguments depend on a template parameter the host pass of the
// compiler rejects the builtin without a message and then leaves out the kernel's launch stub.)
__device__ __forceinline__ void wavek_load_lds(__amdgpu_buffer_rsrc_t rsrc, unsigned char* dst, int voffset, int soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (wavek_lds_ptr)dst, 16, voffset, soffset, 0, 0);
}
// The same with the instruction's immediate offset, kb KB (0 .. 3): it is added to the LDS address AND to the memory
// address, so loads into consecutive kilobytes of LDS can share one M0 (one scalar instruction less per load) if the
// lane offset makes up for it on the memory side.
__device__ __forceinline__ void wavek_load_lds_kb(__amdgpu_buffer_rsrc_t rsrc, unsigned char* dst, int voffset, int soffset, int kb) {
  switch (kb) {
    case 0: __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (wavek_lds_ptr)dst, 16, voffset, soffset, 0, 0); break;
    case 1: __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (wavek_lds_ptr)dst, 16, voffset, soffset, 1024, 0); break;
    case 2: __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (wavek_lds_ptr)dst, 16, voffset, soffset, 2048, 0); break;
    default: __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (wavek_lds_ptr)dst, 16, voffset, soffset, 3072, 0); break;
  }
}
// waits until at most N of the wave's loads are outstanding
template <int N>
__device__ __forceinline__ void wavek_wait_loads() {
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 0xF) | ((N >> 4) << 14));
}
// f(0), f(1), ... f(N - 1) with the number as a constant; the second form as long as cond(number) holds, in nested branches
template <int N, int I = 0, class F>
__device__ __forceinline__ void wavek_each(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    wavek_each<N, I + 1>(f);
  }
}
template <int N, int I = 0, class C, class F>
__device__ __forceinline__ void wavek_each_while(C&& cond, F&& f) {
  if constexpr (I < N) {
    if (cond(std::integral_constant<int, I>{})) {
      f(std::integral_constant<int, I>{});
      wavek_each_while<N, I + 1>(cond, f);
    }
  }
}
template <int FMT, int W, class ACC>
__device__ __forceinline__ ACC wavek_mfma(typename Lowp<FMT>::Vec a, typename Lowp<FMT>::Vec b, ACC c) {
  if constexpr (W == 32) return Lowp<FMT>::mfma(a, b, c);
  else if constexpr (FMT == CASCMM_FMT_BF16) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  else if constexpr (FMT == CASCMM_FMT_FP16) return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  else return __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(a, b, c, 0, 0, 0);
}

// Three fp16 terms on values as they are: what the largest element of an operand has to reach.  The terms are whole multiples of 2^-46,
// 2^-38 of that element: what the slots hold (their smallest term is kept at 2^-35 of elements scaled to 14 at most).  The products
// that are left out are 2^-33 of a product, and the roundings of the sums 2^-24.  (At 2^-13 a tile's elements 2^-16 below its largest one
// were off by 2.9e-6 of themselves, in slots by 1.0e-7.)
constexpr float kWaveKLeast = 0x1p-8f;
// A wave whose first step has nothing from kWaveKLeast on, or something beyond kWaveKMost, scales: that step's largest element to 2^-6, so
// that later ones may be 2^22 times as large
constexpr float kWaveKMost = 0x1p15f;
__device__ __forceinline__ int wavek_exp(unsigned bits) {
  const int e = exp_of_amax(bits) - 14;
  return e < -60 ? -60 : e > 60 ? 60 : e;
}
// (in assembly: the compiler quiets values from memory, in an instruction each, before it compares them.  A NaN stays in top.)
__device__ __forceinline__ void wavek_top(float& top, const float (&x)[8]) {
#pragma unroll
  for (int e = 0; e < 8; e += 2) asm("v_maximum3_f32 %0, %0, |%1|, |%2|" : "+v"(top) : "v"(x[e]), "v"(x[e + 1]));
}
__device__ __forceinline__ unsigned wavek_bits(float top) { return __builtin_bit_cast(unsigned, top) & 0x7FFFFFFFu; }

// A's rows in a stage: position pos of row r holds chunk (pos - wavek_rot(r / 2)) mod 8 (16-row blocks: the rotations of
// cascmm_slotn_kernel.h, which explains them)
template <int W>
__host__ __device__ constexpr int wavek_rot(int h) {
  return W == 32 ? (h & 7) : (int)((0x75642031u >> (4 * (h & 7))) & 7u);
}
// Byte, in a block of rows of a stage, of half x (16 bytes) of what a lane hands to MFMA h.  With fewer than W rows in the stage the
// other lanes read rows 0 .. 8 AL - 1 again: what they compute is not stored.
template <int W, int AL>
__host__ __device__ constexpr int wavek_fragment(int lane, int h, int x) {
  const int row = lane & (W - 1) & (8 * AL - 1), kg = lane / W;
  return row * 128 + ((h * (128 / W) + 2 * kg + x + wavek_rot<W>(row >> 1)) & 7) * 16;
}
template <int W, int MB, int AL>
constexpr bool wavek_fragments_inside() {
  for (int lane = 0; lane < 64; ++lane)
    for (int h = 0; h < W / 16; ++h)
      for (int x = 0; x < 2; ++x)
        if (wavek_fragment<W, AL>(lane, h, x) + (MB - 1) * W * 128 + 16 > AL * 1024) return false;
  return true;
}

// The sizes of one kernel: its launch has to bring the LDS that these stages take, and their number depends on the loads
template <int W, int MB, int NB, int AL, int FMT, int TERMS, int BPRE>
using WaveKOf = WaveK<W, MB, NB, AL, BPRE ? Lowp<FMT>::planes(TERMS) * NB * (W / 16) : W / 2>;

// Host-checked: fp32 operands, 'tri' products; M * lda * 4 and K * ldb * 4 below 2 GiB.  Rows need no alignment (a 16-byte
// buffer load wants its address on a dword, and its dwords are checked against the buffer's end one by one).
// TAIL = 0: K % 32 == 0 and N % (W NB) == 0.  TAIL = 1: any N and K: the rows of B past K lie beyond its buffer (zeros),
// chunks of A past K are fetched from beyond the buffer, what a row's last chunk holds past K is masked.
// AL < W MB / 8: only the first 8 AL rows of A are fetched (M <= 8 AL), the lanes of the others read those again.
// BPRE = 1: B is a prepared weight, [plane][4 ceil(K/32)][N] operand slots, a load per plane and column block (block nb: columns
// W nb + c).  GLU = 1 (prepared, 64-wide tiles): the gated store, C has N / 2 columns, B alternates 32 value and 32 gate columns.
// SCALED = 1 (three fp16 terms, raw): for the calls of the slot kernels (cascmm_f16k_kernel.h), which find the maxima of both operands and
// scale them before they split, in launches of their own.  Here a wave looks at its first step: values within fp16's range and not too small are
// computed as they are, others scaled by that step's maxima, undone on the wave's sums.  Where that was not enough, a sum is not
// finite or all of the tile's rows of A or columns of B lie below kWaveKLeast, the workgroup computes the tile again, scaled by its operands'
// maxima, which the first pass has kept (infinities and NaN among them: the largest finite ones, read once more).  Tiles of zeros are not
// computed again.  Three launches and the slots' trip through memory are saved, and the tiles are small (us, graph replay: in slots on 64 x 160
// tiles; here; here with values that are scaled): 5 x 3165 x 3136 79.9, 15.0, 19.5; 33 x 1613 x 1374 46.0, 11.8, 19.4; 223 x 1401 x 1024 43.1,
// 14.9, 21.5; 71 x 3801 x 3520 96.4, 54.8, 66.1.  A second pass is dearer: with one element of A beyond the range 33.3, 29.7, 33.0, 86.6, with A's
// first 512 k 2^30 below the others 37.9, 37.1, 39.2, 128.9.  Errors against 64 bits: 1.1 to 7.2 1e-9 (rms, of the sum of magnitudes), 6.1e-9
// to 1.2e-8 in slots.
template <int W, int MB, int NB, int AL, int TAIL, int FMT, int TERMS, int BPRE = 0, int GLU = 0, int SCALED = 0>
__global__ __launch_bounds__(512) void cascmm_wavek_kernel(const GroupParams p) {
  static_assert(!GLU || (BPRE && W == 16 && NB == 4), "a value block and its gate block in one tile");
  static_assert(!SCALED || (FMT == CASCMM_FMT_FP16 && TERMS == 3 && !BPRE && TAIL), "for the calls of the slot kernels");
  typedef WaveKOf<W, MB, NB, AL, FMT, TERMS, BPRE> T;
  typedef Lowp<FMT> L;
  constexpr int KM = T::KM, HALVES = T::HALVES, REGS = T::REGS;
  typedef float acc_t __attribute__((ext_vector_type(REGS)));
  constexpr int PL = L::planes(TERMS);
  constexpr int CL = AccClasses<FMT, TERMS, false>::kCount;
  constexpr bool kFold = AccClasses<FMT, TERMS, false>::kChunked;   // the class-0 sum in blocks of NS steps
  extern __shared__ __attribute__((aligned(1024))) unsigned char wavek_smem[];
  const int tid = threadIdx.x, lane = tid & 63, lw = lane & (W - 1), kg = lane / W;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned char* ring = wavek_smem + wave * T::RING;

  // work item: consecutive items run down the row tiles of one column band, and an XCD (which
  // gets every eighth workgroup) takes a contiguous range of items, so a band of B is pulled
  // into one L2 only
  const int tiles = p.tiles_m * p.tiles_n;
  const int total = tiles * p.count;
  const int per = total >> 3;
  int id = blockIdx.x;
  if (id < (per << 3)) id = (id & 7) * per + (id >> 3);
  const void *pa = p.A[0], *pb = p.B[0], *pbias = p.bias[0];
  void* pc = p.C[0];
  int prob = 0;
  if (p.count > 1) {
    prob = id / tiles;
    pa = p.A[prob]; pb = p.B[prob]; pbias = p.bias[prob]; pc = p.C[prob];
  }
  const int t = id - prob * tiles;
  const int tn = t / p.tiles_m, tm = t - tn * p.tiles_m;
  const int m0 = tm * T::BM, n0 = tn * T::BN;
  const int steps = (p.K + T::BK - 1) / T::BK;                // all of them
  const int my_steps = (steps - wave + T::NW - 1) / T::NW;    // those of this wave: wave, wave + 8, ...
  const int ldb_bytes = (int)p.ldb * 4;

  // rows past M read as zero: the buffer ends with row M - 1 (B: with row K - 1)
  const int a_end = (int)(((int64_t)(p.M - 1) * p.lda + p.K) * 4), b_plane = BPRE ? (int)prepared_kgroups(p.K) * p.N * 16 : 0,
            b_end = BPRE ? PL * b_plane : (int)(((int64_t)(p.K - 1) * p.ldb + p.N) * 4);
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)pa, 0, a_end, 0x00020000);
  const i32x4 rb = make_rsrc(pb, b_end);
  // load j of a step brings rows 8 j + lane / 8 to LDS bytes 1024 j + 16 lane, their chunks rotated (wavek_rot)
  int a_voff[2], a_k[2];
#pragma unroll
  for (int jp = 0; jp < 2; ++jp) {
    const int chunk = ((lane & 7) - wavek_rot<W>(4 * jp + (lane >> 4))) & 7;
    a_k[jp] = chunk * 4;
    a_voff[jp] = (int)(((int64_t)(m0 + (lane >> 3)) * p.lda + chunk * 4) * 4);
  }
  const int rows8 = (int)p.lda * 32;
  const int b_voff = BPRE ? (kg * p.N + n0 + lw) * 16 : 8 * kg * ldb_bytes + (n0 + NB * lw) * 4;
  // fragment of a block of rows: row lw, the chunks of k group kg of MFMA h at their rotated places
  static_assert(wavek_fragments_inside<W, MB, AL>(), "a fragment is read from the stage that was waited for");
  int a_frag[HALVES][2];
#pragma unroll
  for (int h = 0; h < HALVES; ++h)
#pragma unroll
    for (int x = 0; x < 2; ++x) a_frag[h][x] = wavek_fragment<W, AL>(lane, h, x);

  typedef float bvec __attribute__((ext_vector_type(NB)));
  // B of the steps in flight, raw or as slots
  bvec Bv[BPRE ? 1 : T::NS][HALVES][8];
  u32x4 Bp[BPRE ? T::NS : 1][HALVES][NB][PL];

  // the loads of this wave's i-th step; past its last step they name places beyond the buffers (zeros, nothing is fetched)
  auto issue = [&](int i, int st) {
    const int k0 = (wave + i * T::NW) * T::BK;
    const bool real = i < my_steps;
#pragma unroll
    for (int j = 0; j < AL; ++j)
      wavek_load_lds(ra, ring + st * T::A_STAGE + j * 1024, !TAIL || a_k[j & 1] < p.K - k0 ? a_voff[j & 1] : 0x7FFFFFFF,
                     real ? k0 * 4 + j * rows8 : a_end);
#pragma unroll
    for (int h = 0; h < HALVES; ++h)
#pragma unroll
      for (int e = 0; e < (BPRE ? 0 : 8); ++e) {
        const int soff = real ? (k0 + KM * h + e) * ldb_bytes : b_end;
        if constexpr (NB == 1) Bv[st][h][e] = (bvec){llvm_raw_buffer_load_f32(rb, b_voff, soff, 0)};
        else if constexpr (NB == 2) Bv[st][h][e] = __builtin_bit_cast(bvec, llvm_raw_buffer_load_v2f32(rb, b_voff, soff, 0));
        else Bv[st][h][e] = __builtin_bit_cast(bvec, llvm_raw_buffer_load_v4f32(rb, b_voff, soff, 0));
      }
    if constexpr (BPRE) {
#pragma unroll
      for (int h = 0; h < HALVES; ++h)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int pl = 0; pl < PL; ++pl)
            Bp[st][h][nb][pl] = __builtin_bit_cast(u32x4, llvm_raw_buffer_load_v4f32(rb, b_voff + nb * (W * 16), real ? ((k0 + KM * h) >> 3) * p.N * 16 + pl * b_plane : b_end, 0));
    }
    __builtin_amdgcn_sched_barrier(0);   // (steps in this order: the waits count the loads of younger ones)
  };

  acc_t acc[CL][MB][NB], master[kFold ? MB : 1][kFold ? NB : 1];
  const acc_t zero = {};
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
      for (int c = 0; c < CL; ++c) acc[c][mb][nb] = zero;
      if constexpr (kFold) master[mb][nb] = zero;
    }

  // fp8 terms: the tensors' scales, powers of two
  constexpr bool kScaled8 = FMT == CASCMM_FMT_FP8;
  float scale_a = 1.f, scale_b = 1.f, scale_out = 1.f, scale_wave = 1.f;   // (scale_wave: of this wave's sums, SCALED)
  if constexpr (kScaled8) {
    if (p.tensor_exps) {
      const int ea = p.tensor_exps[2 * prob], eb = p.tensor_exps[2 * prob + 1];
      scale_a = __builtin_ldexpf(1.f, ea);
      scale_b = __builtin_ldexpf(1.f, eb);
      scale_out = __builtin_ldexpf(1.f, -(ea + eb));
    }
  }
  // SCALED: the largest magnitude that a lane has seen of A, and of its columns of B
  float top_a = 0.f, top_b[SCALED ? NB : 1] = {};
  // how a step takes its values
  typedef std::integral_constant<int, 0> AsTheyAre;
  typedef std::integral_constant<int, 1> Scaled;
  typedef std::integral_constant<int, 2> ScaledAgain;   // the maxima are known
  auto step = [&](int i, auto U, auto how) {
    constexpr int u = decltype(U)::value;
    constexpr bool kScale = decltype(how)::value != 0, kTop = SCALED && decltype(how)::value != 2;
    const unsigned char* stp = ring + u * T::A_STAGE;
#pragma unroll
    for (int h = 0; h < HALVES; ++h) {
      const int left = p.K - (wave + i * T::NW) * T::BK - KM * h - 8 * kg;   // elements of this lane's k group that exist
      u32x4 ta[MB][PL];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        const unsigned char* src = stp + mb * (W * 128);
        const f32x4 x0 = *(const f32x4*)(src + a_frag[h][0]), x1 = *(const f32x4*)(src + a_frag[h][1]);
        float xa[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
        if constexpr (TAIL) {
#pragma unroll
          for (int e = 0; e < 8; ++e) xa[e] = e < left ? xa[e] : 0.f;
        }
        if constexpr (kTop) wavek_top(top_a, xa);
        if constexpr (kScale) {
#pragma unroll
          for (int e = 0; e < 8; ++e) xa[e] *= scale_a;
        }
        split8<FMT, TERMS>(xa, ta[mb], scale_a);
      }
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        u32x4 tb[PL];
        if constexpr (BPRE) {
#pragma unroll
          for (int pl = 0; pl < PL; ++pl) tb[pl] = Bp[u][h][nb][pl];
        } else {
          float xb[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) xb[e] = Bv[u][h][e][nb];
          if constexpr (kTop) wavek_top(top_b[nb], xb);
          if constexpr (kScale) {
#pragma unroll
            for (int e = 0; e < 8; ++e) xb[e] *= scale_b;
          }
          split8<FMT, TERMS>(xb, tb, scale_b);
        }
        // smallest products first
#pragma unroll
        for (int s = TERMS - 1; s >= 0; --s)
#pragma unroll
          for (int ia = s; ia >= 0; --ia)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
              acc_t& c = acc[AccClasses<FMT, TERMS, false>::index(s)][mb][nb];
              c = wavek_mfma<FMT, W>(L::operand(ta[mb][L::plane(ia)], ia), L::operand(tb[L::plane(s - ia)], s - ia), c);
            }
      }
    }
  };
  auto fold = [&]() {
    if constexpr (kFold) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          master[mb][nb] += acc[0][mb][nb];
          acc[0][mb][nb] = zero;
        }
    }
  };
  // SCALED: the first step's maxima, once its loads have landed; whether the wave scales, by scale_a and scale_b
  auto scales = [&]() {
    float first_a = 0.f, first_b = 0.f;
    const int left = p.K - wave * T::BK - 8 * kg;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const unsigned char* src = ring + mb * (W * 128);
      const f32x4 x0 = *(const f32x4*)(src + a_frag[0][0]), x1 = *(const f32x4*)(src + a_frag[0][1]);
      float xa[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
#pragma unroll
      for (int e = 0; e < 8; ++e) xa[e] = e < left ? xa[e] : 0.f;
      wavek_top(first_a, xa);
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      float xb[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) xb[e] = n0 + NB * lw + nb < p.N ? Bv[0][0][e][nb] : 0.f;
      wavek_top(first_b, xb);
    }
    const bool take_a = __any(first_a >= kWaveKLeast) && !__any(first_a > kWaveKMost), take_b = __any(first_b >= kWaveKLeast) && !__any(first_b > kWaveKMost);
    if (take_a && take_b) return false;
    unsigned bits_a = wavek_bits(first_a), bits_b = wavek_bits(first_b);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const unsigned a = (unsigned)__shfl_xor((int)bits_a, off, 64), b = (unsigned)__shfl_xor((int)bits_b, off, 64);
      bits_a = a > bits_a ? a : bits_a;
      bits_b = b > bits_b ? b : bits_b;
    }
    // (zeros, infinities and NaN say nothing)
    const int ea = take_a || bits_a == 0 || bits_a >= 0x7F800000u ? 0 : wavek_exp(bits_a), eb = take_b || bits_b == 0 || bits_b >= 0x7F800000u ? 0 : wavek_exp(bits_b);
    scale_a = __builtin_ldexpf(1.f, ea);
    scale_b = __builtin_ldexpf(1.f, eb);
    scale_wave = __builtin_ldexpf(1.f, -(ea + eb));
    return __builtin_amdgcn_readfirstlane(ea | eb) != 0;
  };
  bool scaled = false;
  // Up to T::STRAIGHT steps: straight code for their number, which issues no load that nobody needs (a step's loads past the
  // end of the buffers cost 0.25 us).  More: trips of NS steps without a branch inside, then those that are left, whose loads
  // are under way already.  In both every path into a step has issued the same loads, so the compiler knows how many are
  // younger than the ones it waits for.  (With steps skipped by branches it assumed the fewest, and the waits in front of the
  // splits of B left half the steps in flight.)
  constexpr int NS = T::NS, L1 = T::LOADS;
  wavek_each<T::STRAIGHT>([&](auto Z) {
    constexpr int S = decltype(Z)::value + 1;
    if (my_steps == S) {
      constexpr int AHEAD = S < NS - 1 ? S : NS - 1;
      wavek_each<AHEAD>([&](auto U) { issue(decltype(U)::value, decltype(U)::value); });
      if constexpr (SCALED) {
        wavek_wait_loads<(AHEAD - 1) * L1>();
        scaled = scales();
        if (scaled) return;
      }
      wavek_each<S>([&](auto U) {
        constexpr int u = decltype(U)::value, younger = S - 1 - u < NS - 1 ? S - 1 - u : NS - 1;
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (u + NS - 1 < S) issue(u + NS - 1, (u + NS - 1) % NS);
        wavek_wait_loads<younger * L1>();
        step(u, std::integral_constant<int, u % NS>{}, AsTheyAre{});
      });
    }
  });
  if (my_steps > T::STRAIGHT) {
    wavek_each<NS - 1>([&](auto U) { issue(decltype(U)::value, decltype(U)::value); });
    if constexpr (SCALED) {
      wavek_wait_loads<(NS - 2) * L1>();
      scaled = scales();
    }
    int i = SCALED && scaled ? my_steps : 0;
    for (; i + NS <= my_steps; i += NS) {
      wavek_each<NS>([&](auto U) {
        constexpr int u = decltype(U)::value;
        issue(i + u + NS - 1, (u + NS - 1) % NS);
        wavek_wait_loads<(NS - 1) * L1>();
        step(i + u, U, AsTheyAre{});
      });
      fold();
    }
    wavek_each_while<NS - 1>([&](auto U) { return i + decltype(U)::value < my_steps; },
                             [&](auto U) {
                               constexpr int u = decltype(U)::value;
                               __builtin_amdgcn_sched_barrier(0);
                               wavek_wait_loads<(NS - 2 - u) * L1>();
                               step(i + u, U, AsTheyAre{});
                             });
  }
  fold();
  // all steps, scaled, from the first one on (those past the last one add products of zeros)
  auto scaled_steps = [&](auto how) {
    wavek_wait_loads<0>();
    __builtin_amdgcn_sched_barrier(0);
    wavek_each<NS - 1>([&](auto U) { issue(decltype(U)::value, decltype(U)::value); });
    for (int i = 0; i < my_steps; i += NS) {
      wavek_each<NS>([&](auto U) {
        constexpr int u = decltype(U)::value;
        issue(i + u + NS - 1, (u + NS - 1) % NS);
        wavek_wait_loads<(NS - 1) * L1>();
        step(i + u, U, how);
      });
      fold();
    }
  };
  if constexpr (SCALED) {
    if (scaled) scaled_steps(Scaled{});
  }
  wavek_wait_loads<0>();   // the loads past the last step land before the ring is reused
  __syncthreads();

  // ---- the eight partial tiles meet in LDS: [wave][mb][nb][reg][lane] fp32 -------------------------
  float* part = (float*)wavek_smem;
  auto wave_sum = [&](int mb, int nb, int e) {
    float v = acc[CL - 1][mb][nb][e];
    if constexpr (CL > 1) {
#pragma unroll
      for (int c = CL - 2; c >= 0; --c) v = __builtin_fmaf(v, AccClasses<FMT, TERMS, false>::kFoldScale, acc[c][mb][nb][e]);
    }
    if constexpr (kFold) v += master[mb][nb][e];
    return v;
  };
  // (these loops stand here and not in a lambda that a scaled tile calls twice: with it the compiler ordered the straight code
  // above otherwise, prepared 12 x 4096 x 512 7.86 -> 8.05 us)
  bool finite = true;   // SCALED: the sums of the columns that exist
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int e = 0; e < REGS; ++e) {
        const float v = SCALED ? wave_sum(mb, nb, e) * scale_wave : wave_sum(mb, nb, e);
        if constexpr (SCALED) finite = finite && (__builtin_fabsf(v) < __builtin_inff() || n0 + NB * lw + nb >= p.N);
        part[(((wave * MB + mb) * NB + nb) * REGS + e) * 64 + lane] = v;
      }
  unsigned* word = (unsigned*)(wavek_smem + T::LDS_BYTES);   // (SCALED: eight words behind the tiles)
  float top = 0.f;                                           // (SCALED: of this lane's columns of B that exist)
  if constexpr (SCALED) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      float xb[8] = {n0 + NB * lw + nb < p.N ? top_b[nb] : 0.f};
      wavek_top(top, xb);
    }
    const unsigned mine = (__any(top_a * scale_a >= kWaveKLeast) ? 1u : 0u) | (__any(top * scale_b >= kWaveKLeast) ? 2u : 0u) | (__any(!finite) ? 4u : 0u);
    if (lane == 0) word[wave] = mine;
  }
  __syncthreads();
  bool again = false;
  if constexpr (SCALED) {
    unsigned all = 0;
#pragma unroll
    for (int w = 0; w < T::NW; ++w) all |= word[w];
    all = __builtin_amdgcn_readfirstlane(all);
    if (all != 3) {
      // the largest elements of the tile's rows of A and columns of B
      const auto most = [&](unsigned a, unsigned b) {
        __syncthreads();
        if (tid < 2) word[tid] = 0;
        __syncthreads();
        atomicMax(&word[0], a);
        atomicMax(&word[1], b);
        __syncthreads();
      };
      most(wavek_bits(top_a), wavek_bits(top));
      if (__builtin_amdgcn_readfirstlane(word[0] >= 0x7F800000u || word[1] >= 0x7F800000u)) {
        // infinities or NaN among the values: the largest finite ones (rows past the last one: that one again)
        unsigned best_a = 0, best_b = 0;
        const auto look = [](unsigned& best, float x) {
          const unsigned bits = __builtin_bit_cast(unsigned, x) & 0x7FFFFFFFu;
          best = bits < 0x7F800000u && bits > best ? bits : best;
        };
        for (int k = tid; k < p.K; k += T::NT) {
          float x[T::BM];
#pragma unroll
          for (int r = 0; r < T::BM; ++r) x[r] = ((const float*)pa)[(int64_t)(m0 + r < p.M ? m0 + r : p.M - 1) * p.lda + k];
#pragma unroll
          for (int r = 0; r < T::BM; ++r) look(best_a, x[r]);
        }
        constexpr int ROWS = T::NT / T::BN, U = 16;
        const float* col = (const float*)pb + (n0 + tid % T::BN < p.N ? n0 + tid % T::BN : p.N - 1);
        for (int k = tid / T::BN; k < p.K; k += ROWS * U) {
          float x[U];
#pragma unroll
          for (int u = 0; u < U; ++u) x[u] = col[(int64_t)(k + u * ROWS < p.K ? k + u * ROWS : p.K - 1) * p.ldb];
#pragma unroll
          for (int u = 0; u < U; ++u) look(best_b, x[u]);
        }
        most(best_a, best_b);
      }
      // (finite sums of zeros are what they are)
      again = __builtin_amdgcn_readfirstlane((all & 4) != 0 || (word[0] != 0 && word[1] != 0));
    }
    if (again) {
      const int ea = f16k_exp_of_amax(word[0]), eb = f16k_exp_of_amax(word[1]);
      scale_a = __builtin_ldexpf(1.f, ea);
      scale_b = __builtin_ldexpf(1.f, eb);
      scale_out = __builtin_ldexpf(1.f, -(ea + eb));
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
          for (int c = 0; c < CL; ++c) acc[c][mb][nb] = zero;
          if constexpr (kFold) master[mb][nb] = zero;
        }
      scaled_steps(ScaledAgain{});
      wavek_wait_loads<0>();
      __syncthreads();
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int e = 0; e < REGS; ++e) part[(((wave * MB + mb) * NB + nb) * REGS + e) * 64 + lane] = wave_sum(mb, nb, e);
      __syncthreads();
    }
  }
  // thread -> (mb, nb, reg, lane) positions tid, tid + 512, ...; of a block a lane holds column lw, rows 4 kg + reg (of 32
  // rows: 8 (reg / 4) + 4 kg + reg % 4)
  float* C = (float*)pc;
  const float* bias = (const float*)pbias;
  if constexpr (GLU) {
    // the gate blocks are two further on
    const int half = p.N >> 1;
#pragma unroll
    for (int q = 0; q < T::BM * 32 / T::NT; ++q) {
      const int pos = q * T::NT + tid;
      const int blk = pos / 256, e = (pos / 64) % 4, ln = pos % 64;
      const int row = m0 + 16 * (blk >> 1) + 4 * (ln >> 4) + e, pair = blk & 1;
      const int col = (n0 >> 1) + 16 * pair + (ln & 15);
      const int at = (((blk >> 1) * 4 + pair) * 4 + e) * 64 + ln;
      float v = 0.f, g = 0.f;
#pragma unroll
      for (int w = 0; w < T::NW; ++w) {
        v += part[w * (MB * 4 * 256) + at];
        g += part[w * (MB * 4 * 256) + at + 2 * 256];
      }
      if (row < p.M) C[(int64_t)row * p.ldc + col] = gated_value(v + (bias ? bias[col] : 0.f), g + (bias ? bias[half + col] : 0.f));
    }
    return;
  }
  constexpr int OUT = T::BM * T::BN;
#pragma unroll
  for (int q = 0; q < (OUT + T::NT - 1) / T::NT; ++q) {
    const int pos = q * T::NT + tid;
    if (OUT % T::NT != 0 && pos >= OUT) break;
    const int blk = pos / (W * W), e = (pos / 64) % REGS, ln = pos % 64;
    const int row = m0 + W * (blk / NB) + 8 * (e >> 2) + 4 * (ln / W) + (e & 3);
    const int col = n0 + (BPRE ? W * (blk % NB) + (ln & (W - 1)) : NB * (ln & (W - 1)) + blk % NB);
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < T::NW; ++w) sum += part[((w * MB * NB + blk) * REGS + e) * 64 + ln];
    if constexpr (kScaled8 || SCALED) sum *= scale_out;
    if (row < p.M && (!TAIL || col < p.N)) C[(int64_t)row * p.ldc + col] = sum + (bias ? bias[col] : 0.f);
  }
}

}  // namespace cascmm
