// Plain 16-bit GEMM (fp16 or bf16 tensors as ONE term of their own format) for skinny and small problems in one launch: K is
// split over the eight waves of a workgroup, the counterpart of cascmm_wavek_kernel.h for the operands of cascmm_h16_kernel.h.
//
// One workgroup computes a (16 MB) x (16 NB) tile of C over the whole K in blocks of the 16 x 16 x 32 MFMA.  Wave w takes the
// 64-wide K steps w, w + 8, ... and shares nothing with the other waves until the end, so the loop has no barrier:
//   * A (64 k of a row are one 128-byte line) goes to the wave's private LDS ring without passing registers, eight rows per
//     `buffer_load ... lds`, the chunks of a row rotated so that the fragment reads spread over all banks;
//   * a prepared B is read as operand slots, 16 bytes per lane and MFMA; of a raw one a lane loads its NB adjacent columns of
//     eight rows (4 or 8 bytes each) and puts the halves together in registers (four permutes per MFMA).
// NS - 1 steps beyond the current one are in flight; the partial tiles are added in wave order through LDS (deterministic).
//
// Bound by the launch, one pass of latencies and what a CU pulls in, 32 (MB + NB) bytes per k, not by the MFMAs.  The four-wave
// kernels walk K stage by stage behind barriers, 2.6 - 3.3 ns per k on their 64 x 64 tile (K = 1280: 3 - 4 of 7 - 8 us); here a
// wave has an eighth of it and all its loads in flight at once.
// Measured (fp16, graph replay over three sets of operands, us; in brackets the four-wave kernels): weight prepared 2 x 1280 x 1280
// 3.2 (6.9), 16 x 320 x 1280 2.9 (3.9), 77 x 2048 x 1280 4.5 (8.5), 154 x 2048 x 1280 5.6 (10.3), x 2560 7.7 (9.5), gated 120 x 384 x
// 3072 4.1 (5.3), 64 x 1280 x 10240 9.1 (10.3); raw 2 x 1280 x 1280 4.0 (7.0), 154 x 2048 x 1280 6.9 (10.5), 256^3 3.2 (4.1), 512^3 3.9
// (5.1).  Behind one tile per CU they lose: 1024 x 640 x 640 6.2 (5.0), 2048 x 640 x 640 raw 12.0 (7.3).
#pragma once
#include "cascmm_h16_kernel.h"
#include "cascmm_wavek_kernel.h"

namespace cascmm {

template <int MB_, int NB_, int RAWB>
struct HWK {
  static constexpr int MB = MB_, NB = NB_, BM = 16 * MB, BN = 16 * NB, BK = 64, NW = 8, NT = 512;
  static constexpr int A_LOADS = 2 * MB, B_LOADS = RAWB ? 16 : 2 * NB, LOADS = A_LOADS + B_LOADS;   // per wave and step
  static constexpr int NS = MB == 1 ? 4 : MB == 2 ? 3 : 2;   // steps in LDS and registers
  static constexpr int STRAIGHT = kHwkStraight;
  static constexpr int A_STAGE = A_LOADS * 1024, RING = NS * A_STAGE, PART = BM * BN * 4;
  static constexpr int LDS_BYTES = NW * (RING > PART ? RING : PART);
  static_assert((NS - 1) * LOADS <= 60, "the wait counter has six bits");
  static_assert(LDS_BYTES <= 160 * 1024, "LDS");
};

// Host-checked, as for cascmm_h16_kernel: the rows of A start on dwords and are whole 16-byte chunks, zeros past K (K % 8 == 0, or
// padded); RAWB = 0: B prepared (prepared_kgroups(K) x N slots, zeros beyond K), 2 GiB not reached with K rounded up to 64; RAWB = 1:
// B [K][ldb] with N % 2 == 0 and rows on dwords, (K + 64) * ldb * 2 below 2 GiB.  Any M and N: rows past M read as zero, columns past the
// edge as some other column's, neither is stored.  GLU (RAWB = 0, NB = 4): the gated store, C has N / 2 columns, B alternates 32
// value and 32 gate columns.
template <int MB, int NB, int FMT, int RAWB, int GLU>
__global__ __launch_bounds__(512) void cascmm_hwk_kernel(const GroupParams p) {
  typedef HWK<MB, NB, RAWB> T;
  typedef Lowp<FMT> L;
  typedef typename H16Elem<FMT>::T E;
  typedef IoType<H16Elem<FMT>::DT> Io;
  static_assert(!GLU || (!RAWB && NB == 4), "a value block and its gate block in one tile");
  static_assert(!RAWB || NB == 2 || NB == 4, "whole dwords of a row of B");
  extern __shared__ __attribute__((aligned(1024))) unsigned char hwk_smem[];
  const int tid = threadIdx.x, lane = tid & 63, lw = lane & 15, kg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned char* ring = hwk_smem + wave * T::RING;

  // consecutive items run down the row tiles of one column band, and an XCD takes a contiguous range of items: a band of B is
  // pulled into one L2 only
  // (the arguments are requested together: left to themselves the reads sink to their uses and wait one behind the other)
  int tiles_m = p.tiles_m, tiles_n = p.tiles_n, count = p.count, M = p.M, N = p.N, K = p.K, lda = (int)p.lda, ldb = (int)p.ldb;
  const void *A = p.A[0], *B = p.B[0];
  asm volatile("" : "+s"(tiles_m), "+s"(tiles_n), "+s"(count), "+s"(M), "+s"(N), "+s"(K), "+s"(lda), "+s"(ldb), "+s"(A), "+s"(B));
  const int tiles = tiles_m * tiles_n, total = tiles * count, per = total >> 3;
  int id = blockIdx.x;
  if (id < (per << 3)) id = (id & 7) * per + (id >> 3);
  int prob = 0;
  if (count > 1) {
    prob = id / tiles;
    A = p.A[prob];
    B = p.B[prob];
  }
  const int t = id - prob * tiles;
  const int tn = t / tiles_m, tm = t - tn * tiles_m;
  const int m0 = tm * T::BM, n0 = tn * T::BN;
  const int steps = (K + T::BK - 1) / T::BK;
  const int my_steps = (steps - wave + T::NW - 1) / T::NW;   // wave, wave + 8, ...

  // A's buffer starts with the tile's first row (A itself may be of any size) and ends with row M - 1; B's ends with its last row or slot row
  const int rows = M - m0 < T::BM ? M - m0 : T::BM;
  const int a_end = ((rows - 1) * lda + (K + 7) / 8 * 8) * 2;
  const int ldb_bytes = ldb * 2;
  const int b_end = RAWB ? (K - 1) * ldb_bytes + N * 2 : (int)prepared_kgroups(K) * N * 16;
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)((const E*)A + (int64_t)m0 * lda), 0, a_end, 0x00020000);
  const i32x4 rb = make_rsrc(B, b_end);
  // load j of a step brings rows 8 j + lane / 8 to LDS bytes 1024 j + 16 lane; position pos of row r holds chunk (pos - r / 2) mod 8
  int a_voff[2], a_k[2];
#pragma unroll
  for (int jp = 0; jp < 2; ++jp) {
    const int chunk = ((lane & 7) - (4 * jp + (lane >> 4))) & 7;
    a_k[jp] = chunk * 8;
    a_voff[jp] = ((lane >> 3) * lda + chunk * 8) * 2;
  }
  const int rows8 = lda * 16;
  const int b_voff = RAWB ? 8 * kg * ldb_bytes + (n0 + NB * lw) * 2 : (kg * N + n0 + lw) * 16;
  int a_frag[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) a_frag[h] = lw * 128 + ((4 * h + kg + (lw >> 1)) & 7) * 16;

  typedef unsigned rvec __attribute__((ext_vector_type(NB >= 2 ? NB / 2 : 1)));   // (a lane's columns of a row of raw B)
  rvec Bv[RAWB ? T::NS : 1][2][8];
  u32x4 Bp[RAWB ? 1 : T::NS][2][NB];
  // the loads of this wave's i-th step; past its last step they name places beyond the buffers (zeros, nothing is fetched)
  auto issue = [&](int i, int st) {
    const int k0 = (wave + i * T::NW) * T::BK;
    const bool real = i < my_steps;
#pragma unroll
    for (int j = 0; j < T::A_LOADS; ++j)
      wavek_load_lds(ra, ring + st * T::A_STAGE + j * 1024, a_k[j & 1] < K - k0 ? a_voff[j & 1] : 0x7FFFFFFF, real ? k0 * 2 + j * rows8 : a_end);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if constexpr (RAWB) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int soff = real ? (k0 + 32 * h + e) * ldb_bytes : b_end;
          if constexpr (NB == 2) Bv[st][h][e] = (rvec){__builtin_bit_cast(unsigned, llvm_raw_buffer_load_f32(rb, b_voff, soff, 0))};
          else Bv[st][h][e] = __builtin_bit_cast(rvec, llvm_raw_buffer_load_v2f32(rb, b_voff, soff, 0));
        }
      } else {
        const int soff = real ? ((k0 >> 3) + 4 * h) * N * 16 : b_end;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) Bp[st][h][nb] = __builtin_bit_cast(u32x4, llvm_raw_buffer_load_v4f32(rb, b_voff + nb * 256, soff, 0));
      }
    }
    __builtin_amdgcn_sched_barrier(0);   // (steps in this order: the waits count the loads of younger ones)
  };

  typedef f32x4 acc_t;
  acc_t acc[MB][NB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = (acc_t){0.f, 0.f, 0.f, 0.f};

  // (operands swapped, B first: a lane then holds one row of C)
  auto step = [&](auto U) {
    constexpr int u = decltype(U)::value;
    const unsigned char* stp = ring + u * T::A_STAGE;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      u32x4 a[MB];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) a[mb] = *(const u32x4*)(stp + mb * 2048 + a_frag[h]);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        u32x4 b;
        if constexpr (RAWB) {
#pragma unroll
          for (int r = 0; r < 4; ++r) b[r] = __builtin_amdgcn_perm(Bv[u][h][2 * r + 1][nb >> 1], Bv[u][h][2 * r][nb >> 1], nb & 1 ? 0x07060302u : 0x05040100u);
        } else {
          b = Bp[u][h][nb];
        }
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[mb][nb] = wavek_mfma<FMT, 16>(L::operand(b, 0), L::operand(a[mb], 0), acc[mb][nb]);
      }
    }
  };
  // Straight code for up to STRAIGHT steps, trips of NS steps and their rest for more: cascmm_wavek_kernel.h says why
  constexpr int NS = T::NS, L1 = T::LOADS;
  wavek_each<T::STRAIGHT>([&](auto Z) {
    constexpr int S = decltype(Z)::value + 1;
    if (my_steps == S) {
      wavek_each<(S < NS - 1 ? S : NS - 1)>([&](auto U) { issue(decltype(U)::value, decltype(U)::value); });
      wavek_each<S>([&](auto U) {
        constexpr int u = decltype(U)::value, younger = S - 1 - u < NS - 1 ? S - 1 - u : NS - 1;
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (u + NS - 1 < S) issue(u + NS - 1, (u + NS - 1) % NS);
        wavek_wait_loads<younger * L1>();
        step(std::integral_constant<int, u % NS>{});
      });
    }
  });
  if (my_steps > T::STRAIGHT) {
    wavek_each<NS - 1>([&](auto U) { issue(decltype(U)::value, decltype(U)::value); });
    int i = 0;
    for (; i + NS <= my_steps; i += NS) {
      wavek_each<NS>([&](auto U) {
        constexpr int u = decltype(U)::value;
        issue(i + u + NS - 1, (u + NS - 1) % NS);
        wavek_wait_loads<(NS - 1) * L1>();
        step(U);
      });
    }
    wavek_each_while<NS - 1>([&](auto U) { return i + decltype(U)::value < my_steps; },
                             [&](auto U) {
                               constexpr int u = decltype(U)::value;
                               __builtin_amdgcn_sched_barrier(0);
                               wavek_wait_loads<(NS - 2 - u) * L1>();
                               step(U);
                             });
  }
  wavek_wait_loads<0>();   // the loads past the last step land before the ring is reused
  __syncthreads();

  // ---- the partial tiles meet in LDS, [wave][mb][quad][lane] x 16 bytes.  A lane holds row lw of block mb; its NB quads of four
  // adjacent columns: prepared, quad nb = columns 16 nb + 4 kg + e; raw, columns 4 NB kg + 4 i + 0..3, which are columns NB c + nb of
  // the blocks' c = 4 kg + e ----
  f32x4* part = (f32x4*)hwk_smem;
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = RAWB ? acc[mb][(4 * i + e) % NB][(4 * i + e) / NB] : acc[mb][i][e];
      part[((wave * MB + mb) * NB + i) * 64 + lane] = v;
    }
  __syncthreads();
  const int no = GLU ? N >> 1 : N;
  E* C = (E*)p.C[prob];
  const E* bias = (const E*)p.bias[prob];
  typedef E e4 __attribute__((ext_vector_type(4)));
  const bool vec = (p.ldc & 3) == 0 && (no & 3) == 0 && ((uintptr_t)C & 7) == 0;
  constexpr int OB = GLU ? NB / 2 : NB, QUADS = MB * OB * 64;
#pragma unroll
  for (int q = 0; q < (QUADS + T::NT - 1) / T::NT; ++q) {
    const int pos = q * T::NT + tid;
    if (QUADS % T::NT != 0 && pos >= QUADS) break;
    const int blk = pos >> 6, ln = pos & 63, mb = blk / OB, i = blk % OB;
    const int row = m0 + 16 * mb + (ln & 15);
    const int col = (GLU ? n0 >> 1 : n0) + (RAWB ? 4 * NB * (ln >> 4) + 4 * i : 16 * i + 4 * (ln >> 4));
    f32x4 s = {0.f, 0.f, 0.f, 0.f}, g = s;
#pragma unroll
    for (int w = 0; w < T::NW; ++w) {
      s += part[((w * MB + mb) * NB + i) * 64 + ln];
      if constexpr (GLU) g += part[((w * MB + mb) * NB + i + 2) * 64 + ln];
    }
    if (row >= M || col >= no) continue;
    if (bias) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (col + e < no) {
          s[e] += Io::load(bias + col + e);
          if constexpr (GLU) g[e] += Io::load(bias + no + col + e);
        }
    }
    if constexpr (GLU) {
      float gate[4] = {g[0], g[1], g[2], g[3]};
      gelu_values(gate);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] *= gate[e];
    }
    E* c = C + (int64_t)row * p.ldc + col;
    if (vec) *(e4*)c = __builtin_convertvector(s, e4);
    else
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (col + e < no) Io::store(c + e, s[e]);
  }
}

}  // namespace cascmm
