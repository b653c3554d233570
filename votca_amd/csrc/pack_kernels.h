// Operator set-up on the device: the padded layouts of the operator's blocks of M^P_{mn} and the aux sums of its
// diagonal. All of it is bound by the memory: a layout is written in one pass over its elements (with its
// BF16 planes, where the operator holds them), and no index of it is divided.
#pragma once
#include "kernels_misc.h"

namespace xg {

// dst row a n1 + b (wp doubles, wp a multiple of 8) = [scale[b]] src[a sa + b sb + 0 .. w - 1], then zeros, and the
// row's BF16 planes (split_bf16) where hi is given. L lanes to a row, two elements a lane and step.
// 1280 x 280 x 320 (40 occupied, 280 virtual levels): block and planes in 425 us, 5.1 TB/s; a pass with 64-bit
// divisions per element and one that splits its result took 343 + 250 us.
template <int L>
__global__ __launch_bounds__(256) void pack_rows_kernel(const double* __restrict__ src, long sa, long sb, long n0,
                                                        long n1, int w, int wp, const double* __restrict__ scale,
                                                        double* __restrict__ dst, unsigned short* __restrict__ hi,
                                                        unsigned short* __restrict__ lo) {
  const long b = blockIdx.x * (long)(256 / L) + threadIdx.x / L;
  if (b >= n1) return;
  for (long a = blockIdx.y; a < n0; a += gridDim.y) {
    const double* s = src + a * sa + b * sb;
    const long o = (a * n1 + b) * wp;
    for (int j = 2 * (threadIdx.x % L); j < wp; j += 2 * L) {
      double x[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) x[e] = j + e < w ? (scale ? scale[b] * s[j + e] : s[j + e]) : 0.0;
      *reinterpret_cast<double2*>(dst + o + j) = make_double2(x[0], x[1]);
      if (hi) {
        ushort2 h, l;
        split_bf16(x[0], h.x, l.x);
        split_bf16(x[1], h.y, l.y);
        *reinterpret_cast<ushort2*>(hi + o + j) = h;
        *reinterpret_cast<ushort2*>(lo + o + j) = l;
      }
    }
  }
}

inline void pack_rows(hipStream_t st, const double* src, long sa, long sb, long n0, long n1, int w, int wp,
                      const double* scale, double* dst, unsigned short* hi, unsigned short* lo) {
  if (n0 <= 0 || n1 <= 0) return;
  const unsigned gy = (unsigned)std::min<long>(n0, 65535);
  // the narrowest group of lanes that takes a row in one step
#define XG_PACK(L)                                                                                              \
  hipLaunchKernelGGL((pack_rows_kernel<L>), dim3((unsigned)((n1 + 256 / L - 1) / (256 / L)), gy), dim3(256), 0, \
                     st, src, sa, sb, n0, n1, w, wp, scale, dst, hi, lo)
  if (wp <= 16) XG_PACK(8);
  else if (wp <= 32) XG_PACK(16);
  else if (wp <= 64) XG_PACK(32);
  else XG_PACK(64);
#undef XG_PACK
  XG_HIP(hipGetLastError());
}

// dst[(a n1 + b) ldd + p] = src[p sp + a sa + b] for p < P, zero for P <= p < ldd: 32 x 32 tiles turned in LDS, so
// that both sides move whole 256-byte runs. 40 x 280 x 1280: 48 us (reads of one element per line, 160).
__global__ __launch_bounds__(256) void pack_turned_kernel(const double* __restrict__ src, long sp, long sa, long n0,
                                                          long n1, long P, long ldd, double* __restrict__ dst) {
  __shared__ double t[32][33];
  const int x = threadIdx.x & 31, y = threadIdx.x >> 5;
  const long pt = (ldd + 31) / 32, b0 = (blockIdx.x / pt) * 32, p0 = (blockIdx.x % pt) * 32;
  for (long a = blockIdx.y; a < n0; a += gridDim.y) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const long p = p0 + y + 8 * i, b = b0 + x;
      t[y + 8 * i][x] = p < P && b < n1 ? src[p * sp + a * sa + b] : 0.0;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const long b = b0 + y + 8 * i, p = p0 + x;
      if (b < n1 && p < ldd) dst[(a * n1 + b) * ldd + p] = t[x][y + 8 * i];
    }
    __syncthreads();
  }
}

inline void pack_turned(hipStream_t st, const double* src, long sp, long sa, long n0, long n1, long P, long ldd,
                        double* dst) {
  if (n0 <= 0 || n1 <= 0 || ldd <= 0) return;
  const dim3 grid((unsigned)(((n1 + 31) / 32) * ((ldd + 31) / 32)), (unsigned)std::min<long>(n0, 65535));
  hipLaunchKernelGGL(pack_turned_kernel, grid, dim3(256), 0, st, src, sp, sa, n0, n1, P, ldd, dst);
  XG_HIP(hipGetLastError());
}

// Aux sums of the operator's diagonal, element (p, s, r) of the tensor at D[p ps + s nt + r], v over levels
// v0 .., c over levels c0 ..:
//   part[z][v ct + c] = sum over the z-th share of p of
//     fx (p,v,c)^2 - fd (p,c,c) E_p (p,v,v) - fd2 (p,c,v) E_p (p,v,c)
// A workgroup takes 64 c (lanes) x 8 v and a share of the aux functions, which its four waves split; (p,c,c), one
// line to a lane, is read once for the eight v. The shares make about 1024 workgroups: the sum over
// 1280 aux functions as one serial chain per (v, c) took 975 us at 40 x 280, this and the sum of
// its shares 90.
constexpr int kDiagV = 8;
__global__ __launch_bounds__(256) void diag_sums_kernel(const double* __restrict__ D, long ps, long nt, long v0, long c0,
                                                        long vt, long ct, long P, const double* __restrict__ E,
                                                        double fx, double fd, double fd2, double* __restrict__ part) {
  __shared__ double red[3][kDiagV][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const long c = blockIdx.x * 64l + lane, cc = min(c, ct - 1);
  const long vb = blockIdx.y * (long)kDiagV;
  const long share = (P + gridDim.z - 1) / gridDim.z, p0 = blockIdx.z * share, p1 = min(P, p0 + share);
  double s[kDiagV];
#pragma unroll
  for (int j = 0; j < kDiagV; ++j) s[j] = 0.0;
  for (long p = p0 + w; p < p1; p += 4) {
    const double* M = D + p * ps;
    const double e = E ? E[p] : 0.0;
    const double mc = fd != 0.0 ? M[(c0 + cc) * nt + c0 + cc] * e : 0.0;
#pragma unroll
    for (int j = 0; j < kDiagV; ++j) {
      const long v = v0 + min(vb + j, vt - 1);
      const double m = fx != 0.0 || fd2 != 0.0 ? M[v * nt + c0 + cc] : 0.0;
      if (fx != 0.0) s[j] += fx * (m * m);
      if (fd != 0.0) s[j] -= fd * (mc * M[v * nt + v]);
      if (fd2 != 0.0) s[j] -= fd2 * (M[(c0 + cc) * nt + v] * e * m);
    }
  }
  if (w > 0)
#pragma unroll
    for (int j = 0; j < kDiagV; ++j) red[w - 1][j][lane] = s[j];
  __syncthreads();
  if (w == 0 && c < ct)
#pragma unroll
    for (int j = 0; j < kDiagV; ++j)
      if (vb + j < vt)
        part[blockIdx.z * (vt * ct) + (vb + j) * ct + c] = ((s[j] + red[0][j][lane]) + red[1][j][lane]) + red[2][j][lane];
}

// Number of shares of the aux sum, for about 1024 workgroups of at least 16 aux functions each.
inline long diag_shares(long vt, long ct, long P) {
  const long wg = ((ct + 63) / 64) * ((vt + kDiagV - 1) / kDiagV);
  return std::max<long>(1, std::min((1024 + wg - 1) / wg, (P + 15) / 16));
}

inline void diag_sums(hipStream_t st, const double* D, long ps, long nt, long v0, long c0, long vt, long ct, long P,
                      const double* E, double fx, double fd, double fd2, long shares, double* part) {
  const dim3 grid((unsigned)((ct + 63) / 64), (unsigned)((vt + kDiagV - 1) / kDiagV), (unsigned)shares);
  hipLaunchKernelGGL(diag_sums_kernel, grid, dim3(256), 0, st, D, ps, nt, v0, c0, vt, ct, P, E, fx, fd, fd2, part);
  XG_HIP(hipGetLastError());
}

}  // namespace xg
