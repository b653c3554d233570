// FP64 GEMM for gfx950 with operands moved straight to LDS.
//
//   C[b](m,n) = epilogue( sum_k A[b](m,k) s[b](k) B[b](n,k) )   (both operands K-contiguous rows)
//
// Block tile BM x BN = (16 TM WR) x (16 TN WC), WR x WC waves, wave tile 16 TM x 16 TN of
// v_mfma_f64_16x16x4f64 tiles, K step 16 (one 128-byte line of every operand row). What bounds it
// is the FP64 matrix pipe, which one wave alone keeps half busy: a register-only loop of these MFMAs
// runs at 36 TFLOP/s with one wave per SIMD and at 77 with two or more, so a kernel with two waves
// per SIMD falls to half rate whenever one of them waits at a barrier (82 % busy, 62 TFLOP/s on the
// Hd stage-1 product with 64 x 64 wave tiles). Hence small wave tiles and four waves per SIMD (two
// workgroups of eight waves per CU), global_load_lds_dwordx4 filling the next stage while this one
// is multiplied, one barrier per K step, no staging registers and no transposing LDS stores. A
// 16-byte LDS read hands a lane two consecutive k: the lanes' k of the two MFMAs of a pair are
// {8u + 2q} and {8u + 2q + 1} (q = lane / 16) for A and B alike, a permutation inside the sum. The
// 16-byte chunk c of LDS row r sits at slot c ^ ((r & 7) ^ ((r >> 3) & 1)): a fragment read (16 rows,
// one chunk) touches 16 distinct bank groups. A wave whose tile lies outside the matrix, or above the
// diagonal of a lower-triangle product, takes part in the loads and barriers only, so edges cost
// in steps of a wave tile. HAS_S: the weights of a K step are one more 128-byte LDS row and multiply
// the B fragment after its read (TN multiplies against TM TN MFMAs), so no scaled copy of B is written.
#pragma once
#include "lds_dma.h"

namespace xg {

typedef double d2v __attribute__((ext_vector_type(2)));

// One output tile over k in [kbeg, kend): store(acc, row_of, col_of) receives the wave's result
// fragments (row_of(i, r), col_of(j): global row and column); called by active waves only.
template <int TM, int TN, int WR, int WC, bool HAS_S, class Store>
__device__ __forceinline__ void f64_lds_tile(const GemmDims& d, const Opnd<double>& A, const Opnd<double>& B,
                                             const double* __restrict__ s, long s_bs, int tm, int tn, int b, int kbeg,
                                             int kend, const Store& store) {
  constexpr int NW = WR * WC;
  constexpr int WM = 16 * TM, WN = 16 * TN;
  constexpr int BM = WR * WM, BN = WC * WN, BK = 16, ROWB = 128;
  constexpr int RG = (BM + BN) / 8;          // 8-row groups of operand rows, one load instruction each
  constexpr int G = RG + (HAS_S ? 1 : 0);    // + the weights
  constexpr int LPW = (G + NW - 1) / NW;     // load instructions per wave per stage
  constexpr int STAGE_BYTES = G * 1024;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * STAGE_BYTES];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm0 = (wave / WC) * WM, wn0 = (wave % WC) * WN;
  const int m0 = tm * BM, n0 = tn * BN;
  const int nk = kend > kbeg ? (kend - kbeg + BK - 1) / BK : 0;
  const bool active = m0 + wm0 < d.M && n0 + wn0 < d.N && !(d.lower && m0 + wm0 + WM <= n0 + wn0);

  // this lane's source and first k for each of the wave's load instructions; rows past M / N read the
  // last row (their results are not stored), k past the chunk reads the zero page
  const double* zp = reinterpret_cast<const double*>(g_zero_page);
  const double* src[LPW];
  int kof[LPW];
#pragma unroll
  for (int j = 0; j < LPW; ++j) {
    const int gi = NW * j + wave;
    const int rr = 8 * gi + (lane >> 3);
    int k = 2 * lds_slot(rr, lane & 7);
    const double* p = zp;
    if (gi < BM / 8) {
      p = A.p + (long)b * A.bs + (long)min(m0 + rr, d.M - 1) * A.ld;
    } else if (gi < RG) {
      p = B.p + (long)b * B.bs + (long)min(n0 + rr - BM, d.N - 1) * B.ld;
    } else if (HAS_S && gi == RG && lane < 8) {
      p = s + (long)b * s_bs;
      k = 2 * lane;
    } else {
      k = d.K;  // spare lanes: always the zero page
    }
    kof[j] = kbeg + k;
    src[j] = p + kof[j];
  }
  const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(lds_u4*)lds);

  auto issue = [&](int stage, int dk) {  // the K step that starts dk after kbeg
#pragma unroll
    for (int j = 0; j < LPW; ++j) {
      const int gi = NW * j + wave;
      if (G % NW != 0 && gi >= G) continue;
      const double* g = kof[j] + dk < kend ? src[j] + dk : zp;
      dma16(g, lds0 + (unsigned)(stage * STAGE_BYTES + gi * 1024));
    }
  };

  d4v acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = (d4v){0.0, 0.0, 0.0, 0.0};

  const int r16 = lane & 15, q = lane >> 4;
  auto compute = [&](int stage) {
    const unsigned char* sA = lds + stage * STAGE_BYTES;
    const unsigned char* sB = sA + BM * ROWB;
#pragma unroll
    for (int u = 0; u < 2; ++u) {  // 8 k each
      const int c = 4 * u + q;
      d2v a[TM], bb[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int row = wm0 + 16 * i + r16;
        a[i] = *reinterpret_cast<const d2v*>(sA + row * ROWB + lds_slot(row, c) * 16);
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int row = wn0 + 16 * j + r16;
        bb[j] = *reinterpret_cast<const d2v*>(sB + row * ROWB + lds_slot(row, c) * 16);
      }
      if constexpr (HAS_S) {
        const d2v w = *reinterpret_cast<const d2v*>(sA + RG * 1024 + c * 16);
#pragma unroll
        for (int j = 0; j < TN; ++j) bb[j] *= w;
      }
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i][e], bb[j][e], acc[i][j], 0, 0, 0);
    }
  };

  if (nk > 0) issue(0, 0);
  for (int t = 0; t < nk; ++t) {
    // every wave's loads of step t are in LDS, and every wave has read the stage the next issue fills
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (t + 1 < nk) issue((t + 1) & 1, (t + 1) * BK);
    if (active) compute(t & 1);
  }
  if (active)
    store(acc, [&](int i, int r) { return m0 + wm0 + i * 16 + (lane >> 4) + 4 * r; },
          [&](int j) { return n0 + wn0 + j * 16 + (lane & 15); });
}

template <int TM, int TN, int WR, int WC, class Epi>
__global__ __launch_bounds__(64 * WR * WC) __attribute__((amdgpu_waves_per_eu(4))) void gemm_f64_lds_kernel(
    GemmDims d, Opnd<double> A, Opnd<double> B, Epi epi) {
  int tm, tn;
  tile_of_block(d, tm, tn);
  const int b = blockIdx.z, ks = blockIdx.y;
  f64_lds_tile<TM, TN, WR, WC, false>(
      d, A, B, nullptr, 0, tm, tn, b, ks * d.kchunk, min(d.K, (ks + 1) * d.kchunk),
      [&](const auto& acc, auto row_of, auto col_of) { epilogue_store<TM, TN, 4>(d, epi, b, ks, acc, row_of, col_of); });
}

// Lower-triangle products of `batch` weight vectors over shared operands (eps at several
// frequencies), dealt evenly: the units (tile, `flock` batches), form one line of units * steps
// K steps, and each flock of workgroups, one per batch, takes an equal share of it. (With a workgroup
// per tile the 432 tiles of P = 937 and 12 frequencies leave 80 of 256 CUs with one workgroup and 176
// with two.) The workgroups of a flock walk the same k of the same operand panels on one XCD, so
// one of them misses its L2 and the others hit. A (unit, batch) that one workgroup covers goes to
// the epilogue; parts go to part[(2 wg + slot) BM BN], slot 0 for a unit an earlier workgroup began,
// slot 1 for one begun here and not finished, and even_reduce_kernel adds them in order. A part holds the
// fragments as the lanes do, value by value.
// One accumulator takes at most 4096 k; the sums of longer shares are added up in the slot. The rounding
// of a sum of K products grows with the partial sums it passes through, and with one accumulator over all of K
// the error of eps (2-norm, against 80 bits) was 6.2e-15 at P = 2000, K = 90000, 12 frequencies and 1.3e-15 at 937,
// 6293; it is 3.3e-16 and 7.2e-16. The slot's traffic costs 0.4-2 % (74.5 -> 75.1 and 1.347 -> 1.351 ms; P = 1535,
// K = 27000: 14.1 -> 14.4); 1024 k give 2.4e-16 at P = 937, for 6 % at 1535.
struct EvenShare {
  long units, steps, groups;  // groups: flocks
  int flock, bgroups;         // workgroups of a flock; batch groups (units = tiles * bgroups)
  __host__ __device__ long begin(long g) const {
    const long t = units * steps;
    return t / groups * g + t % groups * g / groups;
  }
  // the flock that holds step x of the line
  __device__ long owner(long x) const {
    long g = (long)((double)x / ((double)units * (double)steps) * (double)groups);
    g = g < 0 ? 0 : (g >= groups ? groups - 1 : g);
    while (g > 0 && begin(g) > x) --g;
    while (g + 1 < groups && begin(g + 1) <= x) ++g;
    return g;
  }
};

__device__ __forceinline__ void lower_tile(int tile, int& tm, int& tn) {
  tm = (int)((sqrt(8.0 * (double)tile + 1.0) - 1.0) * 0.5);
  while ((tm + 1) * (tm + 2) / 2 <= tile) ++tm;
  while (tm * (tm + 1) / 2 > tile) --tm;
  tn = tile - tm * (tm + 1) / 2;
}

template <int TM, int TN, int WR, int WC, class Epi>
__global__ __launch_bounds__(64 * WR * WC) __attribute__((amdgpu_waves_per_eu(4))) void gemm_f64_even_kernel(
    GemmDims d, EvenShare sh, Opnd<double> A, Opnd<double> B, const double* __restrict__ s, long s_bs, Epi epi,
    double* __restrict__ part) {
  constexpr int BM = 16 * TM * WR, BN = 16 * TN * WC, BK = 16, NT = 64 * WR * WC;
  // consecutive workgroups on one XCD (block b runs on XCD b % 8)
  const long nb = sh.groups * sh.flock, q = nb >> 3, rem = nb & 7, x = blockIdx.x & 7;
  const long wg = x * q + (x < rem ? x : rem) + (blockIdx.x >> 3);
  // 64-bit divisions leave their results in vector registers, of which the products need all 128
  const long g = lane_value(wg / sh.flock, 0);
  const int member = (int)(wg - g * sh.flock);
  const long end = lane_value(sh.begin(g + 1), 0);
  constexpr long kChain = 4096 / BK;
  for (long pos = lane_value(sh.begin(g), 0); pos < end;) {
    const long u = lane_value(pos / sh.steps, 0), t0 = pos - u * sh.steps;
    const long t1 = min(sh.steps, t0 + (end - pos));
    pos += t1 - t0;
    const int tile = (int)lane_value(u / sh.bgroups, 0), b = (int)(u - (long)tile * sh.bgroups) * sh.flock + member;
    int tm, tn;
    lower_tile(tile, tm, tn);
    tm = __builtin_amdgcn_readfirstlane(tm);
    tn = __builtin_amdgcn_readfirstlane(tn);
    const bool whole = t0 == 0 && t1 == sh.steps;
    double* out = part + (2 * wg + (t0 == 0 ? 1 : 0)) * BM * BN;
    for (long t = t0; t < t1; t += kChain) {
      const long te = min(t1, t + kChain);
      f64_lds_tile<TM, TN, WR, WC, true>(
          d, A, B, s, s_bs, tm, tn, b, (int)t * BK, min(d.K, (int)te * BK),
          [&](auto& acc, auto row_of, auto col_of) {
            auto each = [&](auto f) {
#pragma unroll
              for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                  unsigned at = threadIdx.x + (i * TN + j) * 4 * NT;
                  asm volatile("" : "+v"(at)::"memory");  // else every address is computed ahead and held
#pragma unroll
                  for (int r = 0; r < 4; ++r) f(acc[i][j], r, out[at + r * NT]);
                }
            };
            if (t > t0) each([](d4v& v, int r, const double& o) { v[r] += o; });
            if (whole && te == t1)
              epilogue_store<TM, TN, 4>(d, epi, b, 0, acc, row_of, col_of);
            else
              each([](const d4v& v, int r, double& o) { o = v[r]; });
          });
      __syncthreads();  // the next piece refills the LDS stages
    }
  }
}

// The units that several workgroups share: their parts added in order, then the epilogue.
template <int TM, int TN, int WR, int WC, class Epi>
__global__ __launch_bounds__(256) void even_reduce_kernel(GemmDims d, EvenShare sh, const double* __restrict__ part,
                                                          Epi epi) {
  constexpr int BM = 16 * TM * WR, BN = 16 * TN * WC, NT = 64 * WR * WC;
  const long u = blockIdx.x;
  const int member = blockIdx.y;
  const long g0 = sh.owner(u * sh.steps), g1 = sh.owner(u * sh.steps + sh.steps - 1);
  const int tile = (int)(u / sh.bgroups), b = (int)(u - (long)tile * sh.bgroups) * sh.flock + member;
  if (g0 == g1) return;
  int tm, tn;
  lower_tile(tile, tm, tn);
  for (int e = threadIdx.x; e < BM * BN; e += 256) {
    const int row = e / BN, col = e % BN, m = tm * BM + row, n = tn * BN + col;
    if (m >= d.M || n >= d.N || m < n) continue;
    const int value = ((row / 16 % TM) * TN + col / 16 % TN) * 4 + (row & 15) / 4;
    const int wave = row / (16 * TM) * WC + col / (16 * TN);
    const double* q = part + value * NT + 64 * wave + 16 * (row & 3) + (col & 15);
    double acc = q[(2 * (g0 * sh.flock + member) + 1) * BM * BN];
    for (long g = g0 + 1; g <= g1; ++g) acc += q[2 * (g * sh.flock + member) * BM * BN];
    epi(b, 0, m, n, acc);
  }
}

// Both operands K-contiguous with 16-byte aligned rows, K even.
inline bool f64_lds_ok(const Opnd<double>& A, const Opnd<double>& B, int K) {
  return A.p && B.p && vec_ok(A, K, 2) && vec_ok(B, K, 2);
}

// Full outputs, 128 x 64 tiles, eight waves of 32 x 32 (at 16384 x 3072, K = 896 / 4096: 67.8 / 69.1
// TFLOP/s; 128 x 128 tiles of eight 64 x 32 waves 65.0 / 70.3, of four 64 x 64 waves 65.2 / 66.7).
template <class Epi>
inline hipError_t launch_f64_big(hipStream_t st, const GemmDims& d, Opnd<double> A, Opnd<double> B, Epi epi) {
  const dim3 grid(gemm_tiles(d), d.ksplit, d.batch);
  hipLaunchKernelGGL((gemm_f64_lds_kernel<2, 2, 4, 2, Epi>), grid, dim3(512), 0, st, d, A, B, epi);
  return hipGetLastError();
}

// 64 x 64 tiles, four waves of 32 x 32.
template <class Epi>
inline hipError_t launch_f64_mid(hipStream_t st, const GemmDims& d, Opnd<double> A, Opnd<double> B, Epi epi) {
  const dim3 grid(gemm_tiles(d), d.ksplit, d.batch);
  hipLaunchKernelGGL((gemm_f64_lds_kernel<2, 2, 2, 2, Epi>), grid, dim3(256), 0, st, d, A, B, epi);
  return hipGetLastError();
}

// Full output of few columns: 128-row tiles as wide as N in steps of 16, eight waves one above the
// other, so a 30- or 100-column product multiplies 32 or 112 columns and not 64 or 128.
template <int TN, class Epi>
inline hipError_t launch_f64_narrow_tn(hipStream_t st, int M, int N, int K, int batch, int ksplit, Opnd<double> A,
                                       Opnd<double> B, Epi epi) {
  const GemmDims d = make_dims<128, 16 * TN>(M, N, K, batch, ksplit, 16, false);
  const dim3 grid(gemm_tiles(d), d.ksplit, d.batch);
  hipLaunchKernelGGL((gemm_f64_lds_kernel<1, TN, 8, 1, Epi>), grid, dim3(512), 0, st, d, A, B, epi);
  return hipGetLastError();
}

// The even deal of `batch` weighted lower-triangle products (weights s + b s_bs) of order d.M over K:
// 128 x 128 tiles (2 workgroups of 8 waves per CU), which do a given area in 0.87 of the time, or 64 x 64 (4 of 4 waves), whose
// edges waste less: the larger ones unless they compute 1.13 times as much, from an order of 1536 (64 / 128, ms, K = 27000:
// 1600, 12 frequencies 16.08 / 15.46) or of 1217 with three weight vectors or more (K = 27000: 1400, 11 and 12 frequencies 12.25 / 10.32
// and 12.20 / 11.11; K = 24000: 1250, 1, 2 and 3 0.87 / 1.07, 1.57 / 1.62, 2.32 / 2.22; 1300, 12, at 1.14 times the area, 9.63 / 9.94);
// below, their few units are cut into many parts (K = 20000: 1100, 4 and 12 1.77 / 1.78 and 5.10 / 4.97; 6293: 937, 12 1.39 / 1.53).
// At least 8 K steps a workgroup, so a small matrix is not cut into more parts than it has work for.
struct EvenPlan {
  int tile;
  EvenShare sh;
  long workgroups() const { return sh.groups * sh.flock; }
  size_t part_bytes() const { return (size_t)workgroups() * 2 * tile * tile * 8; }
};
inline EvenPlan f64_even_plan(long P, long K, long batch, long cus) {
  EvenPlan p;
  auto area = [&](long t) {
    const long n = (P + t - 1) / t;
    return n * (n + 1) / 2 * t * t;
  };
  p.tile = (P >= 1536 || (P > 1216 && batch >= 3)) && area(128) * 100 <= area(64) * 113 ? 128 : 64;
  const long tl = (P + p.tile - 1) / p.tile;
  // the widest flock without idle members (P = 2000, K = 90000: 3 frequencies by 1 / 3 21.1 / 19.5 ms, 9 by 2 (one in ten
  // idle) / 1 / 3 66.4 / 61.2 / 57.5, 11 by 4 / 1 76.8 / 74.0, 12 by 1 / 2 / 3 / 4 80.0 / 78.0 / 77.1 / 76.0)
  for (p.sh.flock = 4; p.sh.flock > 1 && batch % p.sh.flock != 0;) --p.sh.flock;
  p.sh.bgroups = (int)(batch / p.sh.flock);
  p.sh.units = tl * (tl + 1) / 2 * p.sh.bgroups;
  p.sh.steps = (K + 15) / 16;
  const long resident = (p.tile == 128 ? 2 : 4) * cus / p.sh.flock;
  p.sh.groups = std::max<long>(1, std::min<long>(resident, p.sh.units * p.sh.steps / 8));
  return p;
}
template <class Epi>
inline hipError_t launch_f64_even(hipStream_t st, const EvenPlan& p, int P, int K, int batch, Opnd<double> A,
                                  Opnd<double> B, const double* s, long s_bs, double* part, Epi epi) {
  const dim3 grid((unsigned)p.workgroups()), red((unsigned)p.sh.units, (unsigned)p.sh.flock);
  if (p.tile == 128) {
    const GemmDims d = make_dims<128, 128>(P, P, K, batch, 1, 16, true);
    hipLaunchKernelGGL((gemm_f64_even_kernel<4, 2, 2, 4, Epi>), grid, dim3(512), 0, st, d, p.sh, A, B, s, s_bs, epi, part);
    if (p.sh.groups > 1)
      hipLaunchKernelGGL((even_reduce_kernel<4, 2, 2, 4, Epi>), red, dim3(256), 0, st, d, p.sh, part, epi);
  } else {
    const GemmDims d = make_dims<64, 64>(P, P, K, batch, 1, 16, true);
    hipLaunchKernelGGL((gemm_f64_even_kernel<4, 1, 1, 4, Epi>), grid, dim3(256), 0, st, d, p.sh, A, B, s, s_bs, epi, part);
    if (p.sh.groups > 1)
      hipLaunchKernelGGL((even_reduce_kernel<4, 1, 1, 4, Epi>), red, dim3(256), 0, st, d, p.sh, part, epi);
  }
  return hipGetLastError();
}

// 16-column steps of the narrow tile for an N-column product: the fewest columns in all, the widest
// tile among those.
inline int f64_narrow_tn(int N) {
  int best = 8, cols = 1 << 30;
  for (int tn = 8; tn >= 1; --tn) {
    const int c = (N + 16 * tn - 1) / (16 * tn) * 16 * tn;
    if (c < cols) { cols = c; best = tn; }
  }
  return best;
}

template <class Epi>
inline hipError_t launch_f64_narrow(hipStream_t st, int M, int N, int K, int batch, int ksplit, Opnd<double> A,
                                    Opnd<double> B, Epi epi) {
  switch (f64_narrow_tn(N)) {
    case 1: return launch_f64_narrow_tn<1>(st, M, N, K, batch, ksplit, A, B, epi);
    case 2: return launch_f64_narrow_tn<2>(st, M, N, K, batch, ksplit, A, B, epi);
    case 3: return launch_f64_narrow_tn<3>(st, M, N, K, batch, ksplit, A, B, epi);
    case 4: return launch_f64_narrow_tn<4>(st, M, N, K, batch, ksplit, A, B, epi);
    case 5: return launch_f64_narrow_tn<5>(st, M, N, K, batch, ksplit, A, B, epi);
    case 6: return launch_f64_narrow_tn<6>(st, M, N, K, batch, ksplit, A, B, epi);
    case 7: return launch_f64_narrow_tn<7>(st, M, N, K, batch, ksplit, A, B, epi);
    default: return launch_f64_narrow_tn<8>(st, M, N, K, batch, ksplit, A, B, epi);
  }
}

}  // namespace xg
