// BF16 GEMM for gfx950 with operands moved straight to LDS (lds_dma.h).
//
//   C[b](m,n) = epilogue( sum_k A[b](m,k) B[b](n,k) )   (both operands K-contiguous bf16 rows)
//   SPLIT:   operands a = a_hi + a_lo, products hi*hi + hi*lo + lo*hi (FP32 accumulation)
//
// WR x WC waves, wave tile 16 TM x 16 TN of v_mfma_f32_16x16x32_bf16 tiles, a ring of STAGES LDS
// stages (64 k, or 32 k of both planes), one barrier per stage. Four forms are used:
//   256 x 256, 16 waves of 64 x 64, 2 stages: large products. What bounds the 128 x 128
//     register-staged tiles of gemm_bf16_kernel is LDS traffic (fragment reads plus staged writes
//     come to the 128 bytes a CU moves per cycle at half of the MFMA rate); twice the tile edge halves
//     the writes, which the loads do themselves, and four waves per SIMD cover the barrier. Stage 1
//     of the Hd contraction at 128700 x 3000 x 900, split / plain: 2.64 / 0.98 ms with 128 x 128
//     tiles, 2.00 / 0.83 here (347 / 840 TFLOP/s); eight waves of 128 x 64 2.11 / 0.85, of 64 x 128
//     2.12 / 0.84, 256 x 128 tiles 2.42 / 1.01; the same without the stores 1.65 / 0.60.
//   128 x 128, 8 waves of 32 x 64, 2 stages: split products with fewer columns or a shorter K, plain ones with a
//     short K; two workgroups per CU, one's epilogue under the other's products (three stages leave room for one: 20-30% slower).
//   256 rows x (16 TN) columns, 8 waves of 32 rows, 3 stages: second-stage products that fill their
//     rounds (900 x 100 per vector, K = 29744, 30 vectors: 1193 -> 1054 us split, 440 -> 410 plain).
//   32 rows x (32, 64, 128) columns, 2 x 2 waves, 4 stages: the same with few outputs, where each
//     workgroup walks a long K alone and the ring hides the latency (210 x 30 per vector,
//     K = 30720 in 4 splits, 8 vectors: 197 -> 67 us split, 99 -> 35 plain).
//
// The MFMAs take B as their first operand, so a lane holds four consecutive n of one m (n =
// 4 (lane / 16) + r, m = lane % 16). Every output accumulates its 32-k steps in order, per step
// hi*hi, hi*lo, lo*hi, as in gemm_bf16_kernel: the results are those of the 128 x 128 tiles bit for bit.
#pragma once
#include "lds_dma.h"

namespace xg {

// Epilogues whose rows are BF16 planes (kPlanes): the kernel rounds to hi (and lo, planes() == 2). Row m
// carries factor(m). width(): w = 4, 2 or 1 columns from a multiple of w are adjacent in memory, 2w-byte aligned.
template <class E, class = void>
struct epi_planes { static constexpr bool value = false; };
template <class E>
struct epi_planes<E, decltype((void)E::kPlanes)> { static constexpr bool value = E::kPlanes; };

typedef unsigned short us4v __attribute__((ext_vector_type(4)));
typedef unsigned short us2v __attribute__((ext_vector_type(2)));

template <int TM, int TN, int WR, int WC, int STAGES, bool SPLIT, class Epi>
__global__ __launch_bounds__(64 * WR * WC) void gemm_bf16_ring_kernel(
    GemmDims d, Opnd<unsigned short> A, Opnd<unsigned short> B, Epi epi) {
  constexpr int NW = WR * WC;
  constexpr int KSTEP = SPLIT ? 32 : 64;  // k per stage
  constexpr int NSUB = SPLIT ? 1 : 2;     // 32-k steps per stage
  constexpr int NP = SPLIT ? 2 : 1;       // planes
  constexpr int ROWB = 128;
  constexpr int WM = 16 * TM, WN = 16 * TN;
  constexpr int BM = WR * WM, BN = WC * WN;
  constexpr int STAGE_BYTES = (BM + BN) * ROWB;
  constexpr int G = STAGE_BYTES / 1024;       // 8-row groups, one load instruction each
  constexpr int LPW = (G + NW - 1) / NW;      // load instructions per wave per stage
  constexpr bool PADDED = G % NW != 0;        // some waves issue a load more: the others aim at a spare group
  static_assert(STAGES >= 2 && (STAGES - 2) * LPW <= 63, "vmcnt range");
  // the planes' epilogue turns 32 x WN pieces of both planes per wave in the same memory
  constexpr int EPI_BYTES = epi_planes<Epi>::value && WN == 64 && TM % 2 == 0 ? NW * 2 * 32 * (2 * WN + 16) : 0;
  constexpr int RING_BYTES = STAGES * STAGE_BYTES + (PADDED ? 1024 : 0);
  constexpr int LDS_BYTES = RING_BYTES > EPI_BYTES ? RING_BYTES : EPI_BYTES;
  static_assert(LDS_BYTES <= 160 * 1024, "LDS of a CU");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[LDS_BYTES];

  int tm, tn;
  tile_of_block(d, tm, tn);
  const int b = blockIdx.z, ks = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm0 = (wave / WC) * WM, wn0 = (wave % WC) * WN;
  const int m0 = tm * BM, n0 = tn * BN;
  const int kbeg = ks * d.kchunk;
  const int kend = min(d.K, kbeg + d.kchunk);
  const int nk = kend > kbeg ? (kend - kbeg + KSTEP - 1) / KSTEP : 0;
  // a wave outside the matrix, or above the diagonal of a lower triangle, only loads
  const bool active = m0 + wm0 < d.M && n0 + wn0 < d.N && !(d.lower && m0 + wm0 + WM <= n0 + wn0);

  // this lane's source and first k for each of the wave's loads; rows past M / N read the last row (their
  // results are not stored), k past the chunk reads the zero page
  const unsigned short* zp = reinterpret_cast<const unsigned short*>(g_zero_page);
  const unsigned short* src[LPW];
  int kof[LPW];
#pragma unroll
  for (int j = 0; j < LPW; ++j) {
    const int gi = NW * j + wave;
    const int rr = 8 * gi + (lane >> 3);
    const int c = lds_slot(rr, lane & 7);
    const bool lo = SPLIT && c >= 4;
    kof[j] = kbeg + (SPLIT ? 8 * (c & 3) : 8 * c);
    if (PADDED && gi >= G) kof[j] = d.K;  // always the zero page
    src[j] = (gi < BM / 8 ? (lo ? A.lo : A.p) + (long)b * A.bs + (long)min(m0 + rr, d.M - 1) * A.ld
                          : (lo ? B.lo : B.p) + (long)b * B.bs + (long)min(n0 + rr - BM, d.N - 1) * B.ld) +
             kof[j];
  }
  const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(lds_u4*)lds);
  auto issue = [&](int stage, int dk) {  // the stage that starts dk after kbeg
#pragma unroll
    for (int j = 0; j < LPW; ++j) {
      const unsigned short* g = kof[j] + dk < kend ? src[j] + dk : zp;
      const int gi = NW * j + wave;
      dma16(g, lds0 + (unsigned)(!PADDED || gi < G ? stage * STAGE_BYTES + gi * 1024 : STAGES * STAGE_BYTES));
    }
  };

  f4v acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = (f4v){0.f, 0.f, 0.f, 0.f};

  const int r16 = lane & 15, q = lane >> 4;
  const unsigned char* fa = lds + (wm0 + r16) * ROWB;
  const unsigned char* fb = lds + (BM + wn0 + r16) * ROWB;
  // tile rows are multiples of 16, so a lane's slot depends on r16 and the chunk only
  int slot[2];  // chunk q, chunk q + 4: the planes (SPLIT) or the 32-k halves
#pragma unroll
  for (int h = 0; h < 2; ++h) slot[h] = lds_slot(r16, q + 4 * h) * 16;

  auto compute = [&](int stage) {
    const unsigned char* sa = fa + stage * STAGE_BYTES;
    const unsigned char* sb = fb + stage * STAGE_BYTES;
#pragma unroll
    for (int sub = 0; sub < NSUB; ++sub) {
      bf8v bf[NP][TN], af[2][NP];
      auto read_a = [&](int i) {
#pragma unroll
        for (int p = 0; p < NP; ++p)
          af[i & 1][p] = *reinterpret_cast<const bf8v*>(sa + i * 16 * ROWB + slot[SPLIT ? p : sub]);
      };
      read_a(0);
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int p = 0; p < NP; ++p)
          bf[p][j] = *reinterpret_cast<const bf8v*>(sb + j * 16 * ROWB + slot[SPLIT ? p : sub]);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        if (i + 1 < TM) read_a(i + 1);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[0][j], af[i & 1][0], acc[i][j], 0, 0, 0);
          if constexpr (SPLIT) {
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[1][j], af[i & 1][0], acc[i][j], 0, 0, 0);
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[0][j], af[i & 1][1], acc[i][j], 0, 0, 0);
          }
        }
      }
    }
  };

#pragma unroll
  for (int t = 0; t < STAGES - 1; ++t)
    if (t < nk) issue(t, t * KSTEP);
  int cur = 0, fill = STAGES - 1;  // stage read in this step, stage filled during it
  for (int t = 0; t < nk; ++t) {
    // this wave's loads of step t have landed once at most the later issued steps' remain
    if (STAGES >= 3 && t + STAGES - 2 < nk)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((STAGES - 2) * LPW) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // then every wave's have, and every wave has read the stage that the next issue fills
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (t + STAGES - 1 < nk) issue(fill, (t + STAGES - 1) * KSTEP);
    if (active) compute(cur);
    cur = cur + 1 == STAGES ? 0 : cur + 1;
    fill = fill + 1 == STAGES ? 0 : fill + 1;
  }
  // lane: m = 16 i + lane % 16, n = 16 j + 4 (lane / 16) + r
  if constexpr (epi_planes<Epi>::value && WN == 64 && TM % 2 == 0) {
    // A store of the fragments as they lie touches 16 rows in 32-byte pieces (70 cycles an
    // instruction, a fifth of the whole product at K = 900), so each wave turns 32 rows at a time in
    // LDS and stores 128-byte pieces of four rows. The pieces straddle cache lines (a vector's rows
    // are not multiples of 128 bytes), so the stores stay in the L2 until their lines are whole:
    // non-temporal ones wrote 4.2 GB instead of 3.5 per 3.2 GB and took 4.24 / 1.84 ms instead of
    // 4.04 / 1.64 (split / plain, 257400 x 3000 x 900).
    constexpr int RS = 2 * WN + 16;  // LDS row: 36 dwords, conflict-free in both directions
    constexpr int PLANE = 32 * RS;
    __syncthreads();  // every wave has read the last stage
    unsigned char* mine = lds + wave * (2 * PLANE);
    const bool two = SPLIT && epi.planes() == 2;
    // 16 lanes of four columns to a row, 32 of two or 64 of one, as vectors end (31 columns, 900 x 250 rows, K = 250, split / plain: 173 / 81 us;
    // 8-byte stores at odd 2-byte offsets, with the cut groups one by one: 190 / 88)
    const int width = epi.width();
    const int gn = n0 + wn0 + (width == 4 ? 4 * r16 : width == 2 ? 2 * (lane & 31) : lane);
    const long co = gn < d.N ? epi.col(b, gn) : 0;
#pragma unroll
    for (int h = 0; h < TM / 2; ++h) {
#pragma unroll
      for (int i2 = 0; i2 < 2; ++i2) {
        const int i = 2 * h + i2;
        const float f = epi.factor(min(m0 + wm0 + 16 * i + r16, d.M - 1));
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          us4v vh, vl;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float x = acc[i][j][r] * f;
            vh[r] = bf16_bits_rn(x);
            vl[r] = bf16_bits_rn(x - bf16_bits_to_f(vh[r]));
          }
          unsigned char* at = mine + (16 * i2 + r16) * RS + (16 * j + 4 * q) * 2;
          *reinterpret_cast<us4v*>(at) = vh;
          if (two) *reinterpret_cast<us4v*>(at + PLANE) = vl;
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (width == 4) {
#pragma unroll
        for (int it = 0; it < 8; ++it) {
          const int row = 4 * it + q, gm = m0 + wm0 + 32 * h + row;
          const unsigned char* at = mine + row * RS + r16 * 8;
          const us4v vh = *reinterpret_cast<const us4v*>(at);
          const us4v vl = *reinterpret_cast<const us4v*>(at + PLANE);
          if (gm < d.M && gn < d.N) {
            const long idx = epi.row(b, ks, gm).off + co;
            *reinterpret_cast<us4v*>(epi.Sh + idx) = vh;
            if (two) *reinterpret_cast<us4v*>(epi.Sl + idx) = vl;
          }
        }
      } else {
        const int mh = m0 + wm0 + 32 * h;
        const long ro = epi.row(b, ks, min(mh + (lane & 31), d.M - 1)).off;
        if (width == 2) {
#pragma unroll 8
          for (int it = 0; it < 16; ++it) {
            const int row = 2 * it + (lane >> 5);
            const unsigned char* at = mine + row * RS + (lane & 31) * 4;
            const us2v vh = *reinterpret_cast<const us2v*>(at);
            const us2v vl = *reinterpret_cast<const us2v*>(at + PLANE);
            const long r0 = lane_value(ro, 2 * it), r1 = lane_value(ro, 2 * it + 1);
            const long idx = (lane < 32 ? r0 : r1) + co;
            if (mh + row < d.M && gn < d.N) {
              *reinterpret_cast<us2v*>(epi.Sh + idx) = vh;
              if (two) *reinterpret_cast<us2v*>(epi.Sl + idx) = vl;
            }
          }
        } else
#pragma unroll 8
        for (int row = 0; row < 32; ++row) {
          if (mh + row >= d.M) break;
          const unsigned char* at = mine + row * RS + lane * 2;
          const unsigned short vh = *reinterpret_cast<const unsigned short*>(at);
          const unsigned short vl = *reinterpret_cast<const unsigned short*>(at + PLANE);
          const long idx = lane_value(ro, row) + co;
          if (gn < d.N) {
            epi.Sh[idx] = vh;
            if (two) epi.Sl[idx] = vl;
          }
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    return;
  }
  if (!active) return;
  const int mb = m0 + wm0 + r16, nb = n0 + wn0 + 4 * q;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int gm = mb + 16 * i;
    if (gm >= d.M) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gn = nb + 16 * j + r;
        if (gn < d.N) epi(b, ks, gm, gn, acc[i][j][r]);
      }
  }
}

template <int TM, int TN, int WR, int WC, int STAGES, class Epi>
inline hipError_t launch_bf16_ring(hipStream_t st, const GemmDims& d, Opnd<unsigned short> A, Opnd<unsigned short> B,
                                   bool split, Epi epi) {
  const dim3 grid(gemm_tiles(d), d.ksplit, d.batch), block(64 * WR * WC);
  if (split)
    hipLaunchKernelGGL((gemm_bf16_ring_kernel<TM, TN, WR, WC, STAGES, true, Epi>), grid, block, 0, st, d, A, B, epi);
  else
    hipLaunchKernelGGL((gemm_bf16_ring_kernel<TM, TN, WR, WC, STAGES, false, Epi>), grid, block, 0, st, d, A, B, epi);
  return hipGetLastError();
}

// Tiles of a second-stage product: M rows per batch entry, N <= 128 columns, a long K in ksplit chunks.
enum class Bf16Second { kStaged, kRows256, kRows32 };

// The form that gives the CU with the most workgroups the least to do. `c` workgroups of a form on one of the 256 CUs
// take, per K, c times the weight below: 32-row tiles (2 to 5 of them run at a time) by their width, 256-row tiles (one at a
// time), register-staged 128 x 128 tiles two at a time, or one for somewhat more than half of that (the plain
// one of up to 64 columns for somewhat more). Weights: ns per 10^4 k of the split form, of which the plain
// one takes 0.40 to 0.45. Rows beyond the product load one and the same line, so products of few rows take less of a tile's
// time: of two register-staged ones 0.65 up to 59 rows and all from 91 on; of a 256-row one 0.6 up to 94 and all from 212
// on, with split operands of more than 64 columns 2.2 per row and column, from 300 to 600. `own_cols`: the columns' operand
// is each batch entry's own and is read again by each tile of its rows; that, or few rows, costs the 32-row tiles of
// split operands where several share a CU. Over 1390 products of 7-900 rows and 16-128 columns on all three forms the choice is
// within 5 % of the fastest on 1353, 0.4 % off it on average, and more than 3 % behind the register-staged tiles on 16 (0.65
// of their time on average); over 1258 with `own_cols` more than 3 % behind on 6 (0.56, both stages).
// One threshold on the workgroups had missed the rounds (staged / 256 / 32 rows, split, us): 303 rows, 102 columns, 45
// vectors, K = 105040 in 3: 270 of the 256-row tiles, 2706 / 4706 / 4218; 640, 100, 30, 72800 in 3: 270, 1922 / 2799 / 3599; 256,
// 100, 20, 104000 in 4: 640 of the 32-row ones, 940 / 1457 / 1443; full tiles' weights for all had missed the few rows: 54,
// 77, 45, 45680 in 4: 344 / 314 / 421; 57, 114, 64, 90360 in 4: 782 / 662 / 901; 89, 124, 45, 117632 in 4: 1014 / 1298 / 1457;
// own columns (both stages): 197, 112, 45, 128576: 5601 / 6914 / 6316. Where all had been right: 300, 97, 28, 93600 in 4: 1734 /
// 1377 / 1901; 210, 30, 15, 30720 in 4: 251 / 319 / 143.
inline Bf16Second bf16_second_form(int M, int N, int batch, int ksplit, bool split, bool own_cols) {
  const long n = (long)batch * ksplit;
  auto per_cu = [&](int rows) { return ((M + rows - 1) / rows * n + 255) / 256; };
  const bool narrow = N <= 64;
  const long c = per_cu(128);
  const double pair = std::max(0.65, std::min(1.0, M / 91.0)) * (narrow ? 520 : 720);
  const double staged = c / 2 * pair + c % 2 * (!narrow ? 410 : split ? 310 : 340);
  const double rows256 = per_cu(256) * (split && !narrow ? std::max(300.0, std::min(600.0, 2.2 * (std::min(M, 256) + N)))
                                                         : std::max(0.6, std::min(1.0, 0.28 + M / 294.0)) * (narrow ? 490 : 600));
  const bool reread = split && per_cu(32) > 1 && ((own_cols && N > 96) || M <= 100);
  const double rows32 = per_cu(32) * (N <= 32 ? 95 : narrow ? 108 : reread ? 210 : 187);
  if (staged <= rows256 && staged <= rows32) return Bf16Second::kStaged;
  return rows256 <= rows32 ? Bf16Second::kRows256 : Bf16Second::kRows32;
}

// The 256-row or 32-row tiles. bk: what K chunks are multiples of (64 / 128, as for the 128 x 128 tiles).
template <class Epi>
inline hipError_t launch_bf16_tall(hipStream_t st, Bf16Second form, int M, int N, int K, int batch, int ksplit, int bk,
                                   Opnd<unsigned short> A, Opnd<unsigned short> B, bool split, Epi epi) {
  if (form == Bf16Second::kRows256) {
    const int tn = (N + 15) / 16;
#define XG_TALL(TN) \
  return launch_bf16_ring<2, TN, 8, 1, 3>(st, make_dims<256, 16 * TN>(M, N, K, batch, ksplit, bk, false), A, B, split, epi)
    if (tn <= 2) XG_TALL(2);
    if (tn <= 4) XG_TALL(4);
    if (tn <= 6) XG_TALL(6);
    if (tn == 7) XG_TALL(7);
    XG_TALL(8);
#undef XG_TALL
  }
  if (N <= 32) return launch_bf16_ring<1, 1, 2, 2, 4>(st, make_dims<32, 32>(M, N, K, batch, ksplit, bk, false), A, B, split, epi);
  if (N <= 64) return launch_bf16_ring<1, 2, 2, 2, 4>(st, make_dims<32, 64>(M, N, K, batch, ksplit, bk, false), A, B, split, epi);
  return launch_bf16_ring<1, 4, 2, 2, 4>(st, make_dims<32, 128>(M, N, K, batch, ksplit, bk, false), A, B, split, epi);
}

}  // namespace xg
