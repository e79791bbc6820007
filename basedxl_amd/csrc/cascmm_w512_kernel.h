// Large-tile kernel of the two-term bf16 cascade (gfx950): four waves with 512 registers each.
//
// One workgroup = four waves (one per SIMD, 2 x 2) computes a 256 x 320 tile of C; a wave owns
// 128 x 160 of it, twenty 32 x 32 accumulator blocks: sixteen in the 256 accumulation registers
// and four in ordinary vector registers.  Against a 64 x 160 wave tile this cuts the LDS bytes read per
// MFMA by a third and the bytes staged per MFMA by 30 %, and those bytes, not issue slots, are what
// the chip's power management charges for: with every CU busy the clock settles where the power
// fits, so fewer bytes moved per MFMA is a higher clock.
//
// There are no producer waves (a kernel has one register allocation, so a wave with 512 registers
// fills its SIMD).  Both operands reach LDS as raw fp32 without passing registers (wave-wide
// `buffer_load ... lds`, 1 KB each), and every wave splits the values of its own fragments in
// registers right after reading them:
//   * A: 256 rows x 32 k, two stages at once; eight consecutive lanes fetch the eight 16-byte chunks of one row's
//     128 bytes (a whole cache line; in halves, a stage at a time, every line was fetched twice: 4096^3 329.8 us, 320.6 since), rotated
//     inside the row so that the fragment reads (lane l: row l%32, two chunks of a stage's four) spread over all banks;
//   * B: 16 k rows x 320 columns per stage, 256 consecutive floats per load; lane l of a fragment reads
//     column l%32 at k = 8 (l/32) .. +7 with eight ds_read_b32 (rows of the odd k-group are rotated by
//     32 columns, which keeps the two half waves on different banks).
// Two waves share every row block and every column block, so each value is split twice per
// workgroup; the split's VALU work issues in the gaps between the wave's own MFMAs, as do the LDS
// reads and the loads of later stages, and it costs no measurable time there.
//
// Stages are 16 k deep (60 MFMAs per wave), two pairs of A and four stages of B in LDS (144 KB).  At the barrier that opens
// stage s, stage s + 1 has landed as well, so the first fragments of the next stage are read before
// its barrier and no LDS latency is exposed after it; later loads are issued during stage s into what it has freed.
// Loads are issued unconditionally (past the last stage the last one is fetched again into
// a dead buffer): a wave that is alone on its SIMD pays tens of cycles for every branch.
//
// The order of everything between two MFMAs is pinned with scheduling fences; the four blocks held
// in vector registers use the MFMA through inline assembly, because the compiler gives every MFMA it
// selects an accumulator in the accumulation registers (of which there are sixteen blocks' worth).
#pragma once
#include "cascmm_tile_kernel.h"

namespace cascmm {

template <int NTL_>
struct W512Tile {
  static constexpr int NTL = NTL_;                  // column blocks of a wave
  static constexpr int BM = 256, BN = 64 * NTL, BK = 16, NT = 256;
  // stages of B and pairs of stages of A in LDS: the narrower tiles' stages are shorter (24 and 36 MFMAs), so more of them are in flight
  static constexpr int NS = NTL == 2 ? 6 : NTL == 3 ? 5 : 4, NPA = NTL <= 3 ? 3 : 2;
  static constexpr int WTM = 128, WTN = 32 * NTL, MT = 4;
  static constexpr int A_PAIR = BM * 2 * BK * 4;    // raw fp32, two stages: 128 bytes per row
  static constexpr int B_STAGE = BK * BN * 4;       // raw fp32
  static constexpr int B_AREA = NPA * A_PAIR;       // the pairs of A, then NS stages of B
  static constexpr int LDS_BYTES = B_AREA + NS * B_STAGE;   // 144 KB (NTL = 4: 128 KB, 3: 156 KB)
  static_assert(LDS_BYTES <= 160 * 1024, "LDS");
  static constexpr int A_LOADS = 8;                 // direct loads per wave: a pair of A; a stage of B has NTL
};
typedef W512Tile<5> W512;
constexpr int W512_EDGE_ROWS = 64;   // EDGE: the fewest rows

typedef __attribute__((address_space(3))) void* w512_lds_ptr;

// one wave-wide direct load, j KB behind the LDS address (and the lane offset)
__device__ __forceinline__ void w512_load0(__amdgpu_buffer_rsrc_t r, w512_lds_ptr dst, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, dst, 16, voff, soff, 0, 0);
}
__device__ __forceinline__ void w512_load1(__amdgpu_buffer_rsrc_t r, w512_lds_ptr dst, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, dst, 16, voff, soff, 1024, 0);
}
__device__ __forceinline__ void w512_load2(__amdgpu_buffer_rsrc_t r, w512_lds_ptr dst, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, dst, 16, voff, soff, 2048, 0);
}
__device__ __forceinline__ void w512_load3(__amdgpu_buffer_rsrc_t r, w512_lds_ptr dst, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, dst, 16, voff, soff, 3072, 0);
}

// MFMA with the accumulator in ordinary vector registers
__device__ __forceinline__ void w512_mfma_v(u32x4 a, u32x4 b, f32x16& c) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
}
__device__ __forceinline__ f32x16 w512_mfma_a(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// an empty statement that uses a block where it is kept
__device__ __forceinline__ void w512_in_acc(f32x16& c) { asm volatile("" : "+a"(c)); }
__device__ __forceinline__ void w512_in_vec(f32x16& c) { asm volatile("" : "+v"(c)); }

// NTL: column blocks of a wave; 5 is the 256 x 320 tile described above, 4 the same on 256 x 256 (sixteen blocks, all in
// the accumulation registers), 3 and 2 on 256 x 192 and 256 x 128, for problems that the wider ones leave CUs idle with: a stage has
// 36 and 24 MFMAs, more stages are in flight, and a block splits up to two row blocks of A.  In brackets the fastest other kernel, us:
// raw 1971 x 440 x 2624 24.8 (33.7), 7986 x 320 x 832 21.3 (26.6), 5494 x 448 x 3648 67.3 (76.8), prepared 63.8 (69.5); gated 2028 x 384 x 2432
// 20.2 (27.0).  The loop keeps the pace of the wider tiles where the chip is full (raw 1976 x 1280 x 3840 67.1, 72.9 on the 256 x 128
// tile of the kernels with producer waves; with the weight prepared that one stays the faster, 61 against 68).
// EDGE = 1: tiles may hang over the edges of C: rows and columns past the end are loaded as copies of the last one, which
// costs the loop nothing, and the stores past it go beyond the descriptor's end; the last stages may hang over K.
// Measured (graph replay, raw / prepared weight, all on one card, others are up to a tenth faster; in brackets before rows of A came in
// whole lines): 1976 x 1280 x 10240 on 256 x 320 142.5 / 140.7 us (143.8 / 138.3: the board's power), its gated form 127.4 (132.9);
// 7800 x 640 x 5120 145.7 / 137.9 (145.1 / 141.1); 1500 x 1280 x 10240 on 256 x 256 109.9 / 103.0 (111.3 / 103.4); 4096^3 323.8 / 303.8
// (326.7 / 311.4) = 1.27 / 1.36 PFLOP/s of MFMA work, as on the wider tile: what is left is the clock the board's power allows.  K off its
// steps 3700^3 281 / 263 us (283 / 264; the K-over-waves kernel, the only other one that takes it, 1.25 times that).  The test per load of A
// costs whole K nothing that can be measured.  Traces and counters: profiles/cascmm_w512_edge_kernels.txt.
// Host-checked: M % 256 == 0, N % BN == 0 (EDGE: M >= 64, N >= BN, raw B: N % 4 == 0; with the gated store N % 320 == 0 on the wider
// tile), K % 32 == 0 (EDGE: rows of A of whole 16-byte chunks, zeros between K and the last one's end), lda % 4 == 0, ldb % 4 == 0, A and B 16-byte
// aligned, M * lda * 4 and K * ldb * 4 below 2 GiB, C rows addressable with 32-bit byte offsets
// inside a tile.
// GLU = 1: the gated store (C has N / 2 columns, see GroupParams); a raw operand's gate columns are
// fetched from N / 2 further right, so that both kinds of operand fill the same accumulator blocks.
// (An instantiation of its own: the plain kernel stays as it is, without the scratch bytes this epilogue's
// register allocation asks for.)
// GLU = 2: the gated store writes its result as the LEFT OPERAND SLOTS of the next GEMM (two bf16 terms,
// [term][(N / 2) / 8][M] x 16 bytes at C) instead of fp32.  The MFMAs then take their operands the other
// way round, which leaves every accumulator block transposed in the registers: a lane holds one row of C
// and four consecutive columns per register quad, i.e. half a slot per quad -- the slot of k group
// 2 t + g holds columns 16 t + 4 g + 0..3 and 16 t + 8 + 4 g + 0..3 -- and 32 consecutive lanes write 32
// consecutive slots, 512 contiguous bytes.  (cascmm_prepare_weight_chained gives the next GEMM's weight
// the same order of k.)
// BPRE = 1: the right operand comes already split (cascmm_prepare_weight: 16-byte slots of 8 k of one
// column of one term, [term][K/8][N], below 2 GiB).  A stage then holds the same 20 KB of B as slots
// [term][k group][320], copied by the same twenty 1 KB loads; a lane reads its two operands with two
// 16-byte reads instead of eight 4-byte ones, and the split of B, 55 % of the kernel's VALU work,
// is gone.  Same terms, same order of products: the results equal the raw kernel's bit for bit.
// (a template, so that only the translation unit that lists the variant compiles it)
template <int BPRE, int GLU = 0, int NTL = 5, int EDGE = 0>
__global__ __launch_bounds__(W512Tile<NTL>::NT) __attribute__((amdgpu_waves_per_eu(1, 1))) void cascmm_w512_kernel(const GroupParams p) {
  typedef W512Tile<NTL> T;
  static_assert(NTL >= 2 && NTL <= 5, "");
  static_assert(!GLU || NTL == 5 || (GLU == 1 && BPRE && EDGE && NTL != 3), "");
  static_assert(GLU != 2 || !EDGE, "");
  extern __shared__ __attribute__((aligned(1024))) unsigned char w512_smem[];
  unsigned char* smem = w512_smem;
  const int tid = threadIdx.x, lane = tid & 63, l31 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm0 = (wave >> 1) * T::WTM, wn0 = (wave & 1) * T::WTN;
  int tm, tn;
  tile_coords(blockIdx.x, p.tiles_m, p.tiles_n, tm, tn);
  const int m0 = tm * T::BM, n0 = tn * T::BN;
  const int ksteps = EDGE ? (p.K + 31) / 32 * 2 : p.K / T::BK;
  const int ldb_bytes = (int)p.ldb * 4;

  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)p.A[0], 0, 0x7FFFFFFF, 0x00020000);
  // (one record fewer than A's: with equal words the compiler keeps one copy of them and rebuilds this descriptor from it
  // in front of every B load)
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void*)p.B[0], 0, EDGE && !BPRE ? (int)((((int64_t)p.K - 1) * p.ldb + p.N) * 4) : 0x7FFFFFFE, 0x00020000);
  // per wave: 8 loads of A for two stages (8 rows x 128 bytes each; LDS position 8 row + pos holds chunk
  // (pos - row / 2) mod 8 of the row) and NTL loads of B for every stage (256 consecutive floats of the stage's
  // [16][BN] area)
  const int a_chunk = ((lane & 7) - (lane >> 4)) & 7;   // of the even loads (their first row is a multiple of 16); the odd ones': ^ 4
  int a_voff[T::A_LOADS], b_voff[T::NTL];
#pragma unroll
  for (int j = 0; j < T::A_LOADS; ++j) {
    const int row = (wave * T::A_LOADS + j) * 8 + (lane >> 3);
    const int arow = EDGE && m0 + row >= p.M ? p.M - 1 : m0 + row;
    a_voff[j] = (int)(((int64_t)arow * p.lda + (a_chunk ^ 4 * (j & 1)) * 4) * 4) - (j & 3) * 1024;
  }
#pragma unroll
  for (int j = 0; j < T::NTL; ++j) {
    const int inst = wave * T::NTL + j;
    if (BPRE) {
      // run inst = (term * 2 + k group) * NTL + run of 64 columns; lane = column inside the run
      const int tk = inst / T::NTL, run = inst % T::NTL;
      int col = n0 + run * 64 + lane;
      if (EDGE && col >= p.N) col = p.N - 1;
      b_voff[j] = (((tk >> 1) * (int)prepared_kgroups(p.K) + (tk & 1)) * p.N + col) * 16;
    } else {
      const int f = inst * 256 + lane * 4;
      const int k = f / T::BN, pos = f % T::BN;
      int n = pos - 32 * ((k >> 3) & 1);
      n = n < 0 ? n + T::BN : n;
      int col = n0 + n;
      // gated store: the tile's ten column blocks are value 0, gate 0, value 1, ... of output columns
      // n0 / 2 + 32 j + l; the raw operand keeps its gate columns N / 2 further right
      if (GLU) col = ((n >> 5) & 1) * (p.N >> 1) + (n0 >> 1) + 32 * (n >> 6) + (n & 31);
      if (EDGE && col >= p.N) col = p.N - 4;   // (four columns at a time, N a multiple of 4)
      b_voff[j] = k * ldb_bytes + col * 4;
    }
  }
  const int b_step = BPRE ? 2 * p.N * 16 : T::BK * ldb_bytes;   // bytes of B per stage
  // The loads of a wave land in consecutive kilobytes of LDS: the LDS address is M0 plus the instruction's immediate
  // offset, so a wave's A loads of a stage share one M0 and differ in the immediate; the immediate moves the memory
  // address too, which the lane offsets make up for (they stay non-negative: load j starts at least j KB into its
  // operand, at an edge as well: 64 rows of 32 k and BN columns are more than 3 KB).  The second four of A and the fifth of B are
  // 4 KB further, beyond the immediate's range, and take an M0 of their own.
#pragma unroll
  for (int j = 1; j < (T::NTL < 4 ? T::NTL : 4); ++j) b_voff[j] -= j * 1024;
  // load j of the pair of stages that starts with stage `first` (even), into buffer `buf`
  auto issue_a = [&](int first, int buf, int j) {
    const int step = first < ksteps - 2 ? first : ksteps - 2;
    const w512_lds_ptr al = (w512_lds_ptr)(smem + buf * T::A_PAIR + wave * (T::A_LOADS * 1024) + (j >> 2) * 4096);
    const int as = step * T::BK * 4;
    // EDGE: chunks past K come from beyond the buffer, as zeros (B's rows past K do by themselves: its buffer ends there, or
    // its slots hold zeros)
    const int av = EDGE && (a_chunk ^ 4 * (j & 1)) * 4 >= p.K - step * T::BK ? 0x7FFFFFFF : a_voff[j];
    switch (j & 3) {
      case 0: w512_load0(ra, al, av, as); break;
      case 1: w512_load1(ra, al, av, as); break;
      case 2: w512_load2(ra, al, av, as); break;
      default: w512_load3(ra, al, av, as); break;
    }
  };
  auto issue_b = [&](int step_, int buf, int j) {
    const int step = step_ < ksteps - 1 ? step_ : ksteps - 1;
    const w512_lds_ptr bl = (w512_lds_ptr)(smem + T::B_AREA + buf * T::B_STAGE + wave * (T::NTL * 1024) + (j >> 2) * 4096);
    const int bs = step * b_step;
    switch (j & 3) {
      case 0: w512_load0(rb, bl, b_voff[j], bs); break;
      case 1: w512_load1(rb, bl, b_voff[j], bs); break;
      case 2: w512_load2(rb, bl, b_voff[j], bs); break;
      default: w512_load3(rb, bl, b_voff[j], bs); break;
    }
  };

  // fragment addresses: of A inside a pair, the second stage's chunks are four further (^ 64 bytes); of B inside a stage
  const int a_row = wm0 + l31;                          // + mi * 32 rows = mi * 4096 bytes (same rotation: 32 / 2 = 2 x 8)
  const int a_frag0 = a_row * 128 + ((2 * g + (a_row >> 1)) & 7) * 16;
  const int a_frag1 = a_row * 128 + ((2 * g + 1 + (a_row >> 1)) & 7) * 16;
  int b_frag[T::NTL];
#pragma unroll
  for (int ni = 0; ni < T::NTL; ++ni) {
    int pos = wn0 + ni * 32 + l31 + 32 * g;
    pos = pos >= T::BN ? pos - T::BN : pos;
    b_frag[ni] = (8 * g * T::BN + pos) * 4;   // + e * BN * 4
    // prepared: slot (term 0, k group g, column) -- term 1 is 2 * BN slots further
    if (BPRE) b_frag[ni] = (g * T::BN + wn0 + ni * 32 + l31) * 16;
  }

  f32x16 acc[T::MT][T::NTL];

  // ---- software pipeline ---------------------------------------------------------------------
  // Blocks are numbered t = stage * NTL + ni.  While the 12 MFMAs of block t issue, the raw B values of
  // block t + 2 are read from LDS and those of block t + 1 (read one block earlier) are split; the A
  // values of the next stage's row blocks are read and split during the blocks that RB_OF gives them to (five and four
  // blocks: row block ni during block ni), and loads of later stages are issued: one per block of an even stage (B), up to SLOTS per block
  // of an odd one (a pair of A, then B).
#define W512_FENCE() __builtin_amdgcn_sched_barrier(0)
  u32x4 Af[2][2][T::MT];   // [buffer][hi / lo][mi]
  float R[2][8];           // raw B values of two blocks in flight
  constexpr int RBS = T::NTL < 4 ? 2 : 1;   // row blocks of A that a block takes care of, at most
  float RA[RBS][8];        // their raw values, of the next stage
  u32x4 H[2], L[2];        // split B of the current / next block
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  typedef float f32x2v __attribute__((ext_vector_type(2)));

  auto read_raw = [&](float (&dst)[8], const unsigned char* stp, int ni, int e0, int e1) {
#pragma unroll
    for (int e = e0; e < e1; ++e) dst[e] = *(const float*)(stp + b_frag[ni] + e * T::BN * 4);
  };
  // prepared B: the two terms of a block (the second term is needed four MFMAs later than the first)
  auto read_slot_hi = [&](int buf, const unsigned char* stp, int ni) { H[buf] = *(const u32x4*)(stp + b_frag[ni]); };
  auto read_slot_lo = [&](int buf, const unsigned char* stp, int ni) { L[buf] = *(const u32x4*)(stp + b_frag[ni] + 2 * T::BN * 16); };
  // the split of one pair of consecutive k in two halves of three VALU instructions each
  auto split_1 = [&](float (&x)[8], u32x4& hi, int e) {
    const f32x2v v = {x[2 * e], x[2 * e + 1]};
    const unsigned hp = __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
    hi[e] = hp;
    x[2 * e] = x[2 * e] - __builtin_bit_cast(float, hp << 16);
  };
  auto split_2 = [&](float (&x)[8], const u32x4& hi, u32x4& lo, int e) {
    const f32x2v r = {x[2 * e], x[2 * e + 1] - __builtin_bit_cast(float, hi[e] & 0xFFFF0000u)};
    lo[e] = __builtin_bit_cast(unsigned, __builtin_convertvector(r, bf16x2));
  };

  // Stage v issues stage v + NS - 1 of B, an odd one before that the pair (v - 1) / 2 + NPA of A, whose buffer the stage before it has
  // read last.  Here: what the stages before the first one would have issued.
#pragma unroll
  for (int v = -2 * T::NPA; v < 0; ++v) {
    const int pair = (v - 1) / 2 + T::NPA, sb = v + T::NS - 1;   // (v odd: v - 1 is even)
    if (v & 1) {
#pragma unroll
      for (int j = 0; j < T::A_LOADS; ++j)
        if (pair >= 0) issue_a(2 * pair, pair, j);
    }
#pragma unroll
    for (int j = 0; j < T::NTL; ++j)
      if (sb >= 0) issue_b(sb, sb, j);
  }
  // the accumulators are cleared while the first loads are in flight: not before them, which would hold
  // the loads back, and not after the barrier, where the first MFMA would wait for it
  W512_FENCE();
#pragma unroll
  for (int mi = 0; mi < T::MT; ++mi)
#pragma unroll
    for (int ni = 0; ni < T::NTL; ++ni)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[mi][ni][e] = 0.f;
  // (an empty statement that "uses" every block makes the zeros real here; left alone the compiler creates them
  // right before the first MFMAs)
#pragma unroll
  for (int mi = 0; mi < T::MT; ++mi)
#pragma unroll
    for (int ni = 0; ni < T::NTL; ++ni) {
      if (ni < 4) w512_in_acc(acc[mi][ni]);
      else w512_in_vec(acc[mi][ni]);
    }
  W512_FENCE();
  // Loads that may be in flight: what the last NS - 3 stages have issued (W0: all but pair 0 and stage 0)
  constexpr int WEVEN = (T::NS - 3) * T::NTL + (T::NS - 2) / 2 * T::A_LOADS, WODD = (T::NS - 3) * T::NTL + (T::NS - 3) / 2 * T::A_LOADS;
  constexpr int W0 = (T::NPA - 1) * T::A_LOADS + (T::NS - 2) * T::NTL;
  static_assert(2 * T::NPA - 2 >= T::NS - 2, "an odd stage finds the pair of A that it waits for among the older loads");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (W0 & 0xF) | ((W0 >> 4) << 14));   // pair 0 and stage 0 have landed
  __builtin_amdgcn_s_barrier();
  {
    const unsigned char* b0 = smem + T::B_AREA;
#pragma unroll
    for (int mi = 0; mi < T::MT; ++mi) {
      const f32x4 x0 = *(const f32x4*)(smem + a_frag0 + mi * 4096), x1 = *(const f32x4*)(smem + a_frag1 + mi * 4096);
      float x[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        split_1(x, Af[0][0][mi], e);
        split_2(x, Af[0][0][mi], Af[0][1][mi], e);
      }
    }
    if (BPRE) {
      read_slot_hi(0, b0, 0);
      read_slot_lo(0, b0, 0);
    } else {
      read_raw(R[0], b0, 0, 0, 8);
      read_raw(R[1], b0, 1, 0, 8);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        split_1(R[0], H[0], e);
        split_2(R[0], H[0], L[0], e);
      }
    }
  }

  int sbuf = 0, pbuf = 0;   // the buffers of stage s of B and of its pair of A
  auto stage_buf = [&](int k) { return T::NS == 4 ? (sbuf + k) & 3 : sbuf + k >= T::NS ? sbuf + k - T::NS : sbuf + k; };   // of stage s + k
  for (int s = 0; s < ksteps; s += 2) {
    const int pnext = T::NPA == 2 ? pbuf ^ 1 : pbuf == T::NPA - 1 ? 0 : pbuf + 1;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      // top of stage s + j: the own loads of stage s + j + 1 have landed, then everybody's
      if (j == 0) __builtin_amdgcn_s_waitcnt(0x0F70 | (WEVEN & 0xF) | ((WEVEN >> 4) << 14));
      else __builtin_amdgcn_s_waitcnt(0x0F70 | (WODD & 0xF) | ((WODD >> 4) << 14));
      __builtin_amdgcn_s_barrier();
      const unsigned char* st0 = smem + T::B_AREA + stage_buf(j) * T::B_STAGE;       // this stage of B
      const unsigned char* st1 = smem + T::B_AREA + stage_buf(j + 1) * T::B_STAGE;   // the next one
      const unsigned char* an = smem + (j == 0 ? pbuf : pnext) * T::A_PAIR;          // the pair of A that the next stage lies in
#pragma unroll
      for (int ni = 0; ni < T::NTL; ++ni) {
        const int t = j * T::NTL + ni;        // block number inside the trip: its parity is static
        const int cur = t & 1, nxt = cur ^ 1;
        const int n2 = (ni + 2) % T::NTL;
        const unsigned char* st2 = (ni + 2 < T::NTL) ? st0 : st1;
        const int n1 = (ni + 1) % T::NTL;                                  // prepared B: the next block's slots are read whole
        const unsigned char* stn = (ni + 1 < T::NTL) ? st0 : st1;
        u32x4(&Ah)[T::MT] = Af[j][0];
        u32x4(&Al)[T::MT] = Af[j][1];
        // products lo.hi, hi.lo, hi.hi of the four row blocks: smallest first, consecutive MFMAs on
        // different accumulators
        auto mm = [&](int idx) {
          const int prod = idx >> 2, mi = idx & 3;
          const u32x4 a = prod == 0 ? Al[mi] : Ah[mi];
          const u32x4 b = prod == 1 ? L[cur] : H[cur];
          if (GLU == 2) {   // operands swapped: the block comes out transposed
            if (ni < 4) acc[mi][ni] = w512_mfma_a(b, a, acc[mi][ni]);
            else w512_mfma_v(b, a, acc[mi][ni]);
          } else {
            if (ni < 4) acc[mi][ni] = w512_mfma_a(a, b, acc[mi][ni]);
            else w512_mfma_v(a, b, acc[mi][ni]);
          }
        };
        // loads of a stage: NTL of B, one behind each block; the odd stages' blocks have more slots, for the pair of A
        constexpr int SLOTS = (T::A_LOADS + 2 * T::NTL - 1) / T::NTL;   // of a block of an odd stage
        auto dl = [&](int k) {
          if (k == 1 && j == 0) issue_b(s + T::NS - 1, stage_buf(T::NS - 1), ni);
          if (j == 0 || k >= SLOTS) return;
          const int slot = ni * SLOTS + k;
          if (slot < T::A_LOADS) issue_a(s + 2 * T::NPA, pbuf, slot);
          else if (slot < T::A_LOADS + T::NTL) issue_b(s + T::NS, stage_buf(0), slot - T::A_LOADS);
        };
        // row blocks of A that the block reads and splits for the next stage
        constexpr int RB_OF[4][6] = {{0, 2, 4}, {0, 2, 3, 4}, {0, 1, 2, 3, 4}, {0, 1, 2, 3, 4, 4}};
        const int rb0 = RB_OF[T::NTL - 2][ni], rbs = RB_OF[T::NTL - 2][ni + 1] - rb0;
        // What goes between MFMA g and MFMA g + 1 of the block.  A wave alone on its SIMD issues one instruction
        // every four cycles or so, whatever its kind, and an MFMA holds the matrix pipe for 32: more than six
        // instructions in a gap leave the pipe waiting.  The sixteen half-splits of the block (three VALU
        // instructions each: B's in gaps 0 .. 7, A's in gaps 4 .. 11) and the LDS reads and loads are spread so
        // that no gap holds more than six (2202 shader-clock cycles per stage against 2228 with the LDS reads in
        // gaps 0 .. 2 and all the splits in gaps 3 .. 10; 1920 are the MFMAs).
        // LDS answers in order: one wait at the top of a block covers everything the block before it read (the
        // compiler would put a wait of its own, an instruction each, in front of the first use of every read),
        // a second one in gap 4 the block's A fragments (younger than them: the raw B reads of gaps 1 and 2)
        auto gap = [&](int gi) {
          if (gi == 0) { __builtin_amdgcn_s_waitcnt(0xC07F); W512_FENCE(); }                          // lgkmcnt(0)
          if (gi == 4 && rbs > 0) { __builtin_amdgcn_s_waitcnt(BPRE ? 0xC07F : 0xC47F); W512_FENCE(); }   // lgkmcnt(0) / lgkmcnt(4)
          if (gi == 0) {   // row blocks of the next stage
            const int half = j == 0 ? 64 : 0;
#pragma unroll
            for (int x = 0; x < RBS; ++x) {
              if (x >= rbs) continue;
              const f32x4 x0 = *(const f32x4*)(an + (a_frag0 ^ half) + (rb0 + x) * 4096), x1 = *(const f32x4*)(an + (a_frag1 ^ half) + (rb0 + x) * 4096);
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                RA[x][e] = x0[e];
                RA[x][4 + e] = x1[e];
              }
            }
          }
          if (!BPRE && gi == 1) read_raw(R[cur], st2, n2, 0, 4);
          if (!BPRE && gi == 2) read_raw(R[cur], st2, n2, 4, 8);
          if (!BPRE) {   // (two row blocks of A: both halves of a pair in each of the gaps in front of theirs)
#pragma unroll
            for (int h = 0; h < 8; ++h) {
              if ((rbs == 2 ? h >> 1 : h) != gi) continue;
              if (h & 1) split_2(R[nxt], H[nxt], L[nxt], h >> 1);
              else split_1(R[nxt], H[nxt], h >> 1);
            }
          }
          if (gi >= 4) {
            const int h = gi - 4;
#pragma unroll
            for (int x = 0; x < RBS; ++x) {
              if (x >= rbs) continue;
              if (h & 1) split_2(RA[x], Af[j ^ 1][0][rb0 + x], Af[j ^ 1][1][rb0 + x], h >> 1);
              else split_1(RA[x], Af[j ^ 1][0][rb0 + x], h >> 1);
            }
          }
          if (BPRE && gi == 4) read_slot_hi(nxt, stn, n1);     // seven MFMAs before the next block's first
          if (BPRE && gi == 8) read_slot_lo(nxt, stn, n1);
          // the stage's loads, apart from each other: an even stage's one in gap 9, an odd stage's two to five in every other gap
          // (several loads in neighbouring gaps of one block cost 30 cycles each: counted)
          if (gi == 3) dl(0);
          if (gi == 9) dl(1);
          if (gi == 11) dl(2);
          if (gi == 7) dl(3);
          if (gi == 5) dl(4);
        };
#pragma unroll
        for (int gi = 0; gi < 12; ++gi) {
          mm(gi); W512_FENCE();
          gap(gi); W512_FENCE();
        }
      }
    }
    sbuf = stage_buf(2);
    pbuf = pnext;
  }
#undef W512_FENCE
  __builtin_amdgcn_s_waitcnt(0x0F70);   // the redundant loads of the last stages land before LDS is given up
  // the MFMAs written as assembly are invisible to the compiler's hazard handling: their passes
  // must have drained before the accumulators are read
  asm volatile("s_nop 7\n s_nop 7\n s_nop 7" ::: "memory");

  // ---- epilogue: of every block a lane holds column l31, rows 8 q + 4 g + e -----------------------
  // (the lane number is taken afresh: a register kept alive through the main loop for it would be spilled)
  const int elane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  const int el31 = elane & 31, eg = elane >> 5;
  const float* bias = (const float*)p.bias[0];
  const int ldc_bytes = (int)p.ldc * 4;
  if constexpr (GLU == 2) {
    // Gated store as operand slots.  Blocks are transposed: of block (mi, ni) a lane holds row 32 mi + l31
    // and columns 8 q + 4 g + e in register 4 q + e.  Pairs of blocks as below (value j, gate j); the gate
    // of pair 2 crosses from the right wave to the left one through LDS, same lanes and registers.
    const int half = p.N >> 1, c0 = n0 >> 1;
    const int kgroups = half >> 3;                                  // k groups of the next GEMM
    float* xbuf = (float*)smem + (wave >> 1) * (T::MT * 16 * 64);
    __builtin_amdgcn_s_barrier();
    auto bias_at = [&](int col) { return bias ? bias[col] : 0.f; };
    if (wave & 1) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float bg = bias_at(half + c0 + 64 + 8 * (r >> 2) + 4 * eg + (r & 3));
        float gate[T::MT];
#pragma unroll
        for (int mi = 0; mi < T::MT; ++mi) gate[mi] = acc[mi][0][r] + bg;
        gelu_values(gate);
#pragma unroll
        for (int mi = 0; mi < T::MT; ++mi) xbuf[(mi * 16 + r) * 64 + elane] = gate[mi];
      }
    }
    __syncthreads();
    // 4 M K2 bytes of slots, below 2 GiB (host-checked)
    const i32x4 rc = make_rsrc(p.C[0], (int64_t)2 * kgroups * p.M * 16);
    const int voff = (eg * p.M + m0 + wm0 + el31) * 16;             // + mi * 512
    const int term1 = kgroups * p.M * 16;
    auto out_pair = [&](int pair, int vb, int gb, bool gate_in_lds) {
      const int col0 = c0 + 32 * pair;                              // first output column of the pair
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {                              // k groups 4 (col0 / 32) + 2 s2 + g
        float bv[8], bgt[8];
#pragma unroll
        for (int x = 0; x < 8; ++x) {
          const int col = col0 + 16 * s2 + 8 * (x >> 2) + 4 * eg + (x & 3);
          bv[x] = bias_at(col);
          bgt[x] = gate_in_lds ? 0.f : bias_at(half + col);
        }
        const int soff = ((col0 >> 3) + 2 * s2) * p.M * 16;
#pragma unroll
        for (int mi = 0; mi < T::MT; ++mi) {
          float r8[8], gl[8];
#pragma unroll
          for (int x = 0; x < 8; ++x) {
            const int r = 8 * s2 + x;                               // register 4 q + e with q = 2 s2 + x / 4
            gl[x] = gate_in_lds ? xbuf[(mi * 16 + r) * 64 + elane] : acc[mi][gb][r] + bgt[x];
          }
          if (!gate_in_lds) gelu_values(gl);
#pragma unroll
          for (int x = 0; x < 8; ++x) {
            r8[x] = (acc[mi][vb][8 * s2 + x] + bv[x]) * gl[x];
            // the slots are the split of this product ROUNDED to fp32, as a separate pass over the fp32
            // result would split it: keep the compiler from folding the multiplication into the split's
            // subtraction (a fused multiply-subtract would take the residual of the unrounded product)
            asm volatile("" : "+v"(r8[x]));
          }
          u32x4 t[2];
          split8<CASCMM_FMT_BF16, 2>(r8, t);
          llvm_raw_buffer_store_v4f32(__builtin_bit_cast(f32x4, t[0]), rc, voff + mi * 512, soff, kLargeTileStoreAux);
          llvm_raw_buffer_store_v4f32(__builtin_bit_cast(f32x4, t[1]), rc, voff + mi * 512, soff + term1, kLargeTileStoreAux);
        }
      }
    };
    if ((wave & 1) == 0) {
      out_pair(0, 0, 1, false);
      out_pair(1, 2, 3, false);
      out_pair(2, 4, 0, true);
    } else {
      out_pair(3, 1, 2, false);
      out_pair(4, 3, 4, false);
    }
    return;
  }
  if constexpr (GLU == 1 && NTL != 5) {
    // Gated store of the 256 and 128 wide tiles: a wave's blocks are value 0, gate 0, value 1, ... of its own columns.
    const int half = p.N >> 1, rows = p.M - (m0 + wm0);
    const i32x4 re = make_rsrc((float*)p.C[0] + (int64_t)(m0 + wm0) * p.ldc, rows > 0 ? (int64_t)(rows < T::WTM ? rows : T::WTM) * ldc_bytes : 0);
#pragma unroll
    for (int pair = 0; pair < NTL / 2; ++pair) {
      const int col = ((n0 + wn0) >> 1) + 32 * pair + el31, read = col < half ? col : half - 1;
      const float bv = bias ? bias[read] : 0.f, bg = bias ? bias[half + read] : 0.f;
      const int voff = col < half ? eg * 4 * ldc_bytes + col * 4 : 0x7FFFFFFF;
#pragma unroll
      for (int mi = 0; mi < T::MT; ++mi)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float gate[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) gate[e] = acc[mi][2 * pair + 1][4 * q + e] + bg;
          gelu_values(gate);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            llvm_raw_buffer_store_f32((acc[mi][2 * pair][4 * q + e] + bv) * gate[e], re,
                                      (int)((unsigned)voff + (unsigned)((mi * 32 + q * 8 + e) * ldc_bytes)), 0, kLargeTileStoreAux);
        }
    }
    return;
  } else if constexpr (GLU == 1) {
    // Gated store: C[m][n0 / 2 + 32 j + l] = (value j + bias) x gelu(gate j + bias), j = 0 .. 4.  The
    // left wave of a row pair holds value 0, gate 0, value 1, gate 1, value 2, the right one gate 2,
    // value 3, gate 3, value 4, gate 4: pair 2 is the only one that spans two waves.  Each evaluates half of its gates: the
    // left wave hands its values of the upper two row blocks over, the right one its gates of the lower two, same lanes and
    // registers, through the LDS the main loop has given up.  (The gates are what this store takes: with all of pair 2's on the
    // right wave, and the left one waiting for them, 192 a lane one behind the other in place of 160.)
    const int half = p.N >> 1, c0 = n0 >> 1;
    float* xbuf = (float*)smem + (wave >> 1) * (4 * 16 * 64);        // 16 KB per row pair of waves: 32 values, 32 gates a lane
    __builtin_amdgcn_s_barrier();                                    // every wave has read its last fragments
    const float b2 = bias ? bias[(wave & 1 ? half : 0) + c0 + 64 + el31] : 0.f;   // of pair 2's columns that this wave holds
    if (wave & 1) {
#pragma unroll
      for (int r = 0; r < 32; ++r) xbuf[(32 + r) * 64 + elane] = acc[2 + r / 16][0][r & 15] + b2;
    } else {
#pragma unroll
      for (int r = 0; r < 32; ++r) xbuf[r * 64 + elane] = acc[r / 16][4][r & 15] + b2;
    }
    __syncthreads();
    float* C = (float*)p.C[0] + (int64_t)(m0 + wm0) * p.ldc + c0;
    // (EDGE: the descriptor ends with the last row of C, the row offsets are part of the checked lane offset)
    const int rows = p.M - (m0 + wm0);
    const i32x4 rc = make_rsrc(C, !EDGE ? 0x7FFFFFFF : rows > 0 ? (int64_t)(rows < T::WTM ? rows : T::WTM) * ldc_bytes - c0 * 4 : 0);
    // row blocks first .. last - 1 of a pair; value and gate: its sums with the bias
    auto out_pair = [&](int pair, int first, int last, auto value, auto gate) {
      const int voff = eg * 4 * ldc_bytes + (pair * 32 + el31) * 4;
#pragma unroll
      for (int mi = first; mi < last; ++mi)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float gl[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) gl[e] = gate(mi, 4 * q + e);
          gelu_values(gl);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int roff = (mi * 32 + q * 8 + e) * ldc_bytes;
            llvm_raw_buffer_store_f32(value(mi, 4 * q + e) * gl[e], rc, EDGE ? voff + roff : voff, EDGE ? 0 : roff, kLargeTileStoreAux);
          }
        }
    };
    auto own_pair = [&](int pair, int vb, int gb) {
      const float bv = bias ? bias[c0 + 32 * pair + el31] : 0.f, bg = bias ? bias[half + c0 + 32 * pair + el31] : 0.f;
      out_pair(pair, 0, T::MT, [&](int mi, int r) { return acc[mi][vb][r] + bv; }, [&](int mi, int r) { return acc[mi][gb][r] + bg; });
    };
    if ((wave & 1) == 0) {
      own_pair(0, 0, 1);
      own_pair(1, 2, 3);
      out_pair(2, 2, 4, [&](int mi, int r) { return acc[mi][4][r] + b2; }, [&](int mi, int r) { return xbuf[(mi * 16 + r) * 64 + elane]; });
    } else {
      out_pair(2, 0, 2, [&](int mi, int r) { return xbuf[(mi * 16 + r) * 64 + elane]; }, [&](int mi, int r) { return acc[mi][0][r] + b2; });
      own_pair(3, 1, 2);
      own_pair(4, 3, 4);
    }
    return;
  }
  float* C = (float*)p.C[0] + (int64_t)(m0 + wm0) * p.ldc + n0 + wn0;
  const i32x4 rc = make_rsrc(C, 0x7FFFFFFF);
  if (EDGE && (m0 + T::BM > p.M || n0 + T::BN > p.N)) {
    // The descriptor ends with the last row of C and a lane past the last column points beyond any descriptor, so the
    // stores need no branches (with a test per store such a tile took 28 us longer, and the launch with it).
    const int rows = p.M - (m0 + wm0);
    const i32x4 re = make_rsrc((float*)p.C[0] + (int64_t)(m0 + wm0) * p.ldc, rows > 0 ? (int64_t)(rows < T::WTM ? rows : T::WTM) * ldc_bytes : 0);
#pragma unroll
    for (int ni = 0; ni < T::NTL; ++ni) {
      const int col = n0 + wn0 + ni * 32 + el31;
      const float bv = bias ? bias[col < p.N ? col : p.N - 1] : 0.f;
      const int voff = col < p.N ? eg * 4 * ldc_bytes + col * 4 : 0x7FFFFFFF;
#pragma unroll
      for (int mi = 0; mi < T::MT; ++mi)
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            llvm_raw_buffer_store_f32(acc[mi][ni][4 * q + e] + bv, re, (int)((unsigned)voff + (unsigned)((mi * 32 + q * 8 + e) * ldc_bytes)), 0,
                                      kLargeTileStoreAux);
    }
    return;
  }
#pragma unroll
  for (int ni = 0; ni < T::NTL; ++ni) {
    const float bv = bias ? bias[n0 + wn0 + ni * 32 + el31] : 0.f;
    const int voff = eg * 4 * ldc_bytes + (ni * 32 + el31) * 4;
#pragma unroll
    for (int mi = 0; mi < T::MT; ++mi)
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          llvm_raw_buffer_store_f32(acc[mi][ni][4 * q + e] + bv, rc, voff, (mi * 32 + q * 8 + e) * ldc_bytes, kLargeTileStoreAux);
  }
}

}  // namespace cascmm
