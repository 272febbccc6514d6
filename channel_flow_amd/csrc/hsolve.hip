// Per-mode v and omega_y solves (PF:242-394) with the diagonalised operators of
// helmholtz.h, and the mean mode (PF:401-474).
//
// Per parity half system and real column (Re or Im of one mode):
//   omega_y:  x = Q V diag(1 / sigma) L b
//   v:        x = Q V s (L b + a l1 - B q),  a, B from the two wall conditions
// with L, V, the eigenvalues and the wall vectors shared by all modes and by
// both equations.  A block takes one parity and 64 or 32 real columns: the right-hand
// sides are staged in LDS, Y = L B runs on the FP64 matrix cores, Y is scaled
// per (row, mode) and corrected (v) in registers and written back to LDS as the B
// operand of X = V Y; the first coefficient is minus the sum of the others (the
// wall condition x(1) = 0), so it costs adds, not a row block.
//
// Bound: the matrix products, 2 m^2 multiply-adds per real column and parity
// (5 GFLOP per equation at 256x193x256, 35 TFLOP/s for v and 41 for omega_y,
// against the 72 that a large FP64 library product reaches); the rest is the
// blocks' loads, scaling and stores (65 of 138 us, 51 of 119), which overlap the
// products of other blocks in part only.  They replace a
// stream of stored v inverses (1.55 GB, one pair per k^2), which HBM bound:
// v 0.429 -> 0.131 ms and omega_y 0.139 -> 0.110 ms at 256x193x256, v 3.0 ->
// 0.85 ms at 512x257x512.
#include "chf_internal.h"
#include "mfma.h"

namespace chf {

struct HsArgs {
  const double2 *L[2], *V[2];  // per parity: packed A fragments (pack_pairs in api.hip)
  const double* vec[2];        // per parity: lam, w1, w2, l1, q, each [16 MB]
  const double* wall[2];       // per parity: [column][4], (d1, d2) -> (a, B)  (v)
  const double2* rhs[2][2];    // per equation (0 = v) and parity: folded right-hand sides [rows][ncol]
  double* out[2];              // v, omega_y, real view [Ny][2 ncol]
  const double *al, *be;
  int m[2];
  int Mx, Mz;
  long ncol;
  double c;
  // mean mode (the v launch's first block)
  double2 *au0, *w0;
  const double2 *c1n, *c1p, *c3n, *c3p;  // mean Lamb point values, n and n-1
  const double* tmean;                   // [l][p]: T0 + c T2 transposed
  const double* inv0;                    // k^2 = 0 half-system inverses [row j][even | odd]
  int N, Ny, ne, no;
  double dt;
};

// U and W (PF:401-474): right-hand side (T0 + c T2) U - dt/2 (3 L^n - L^(n-1))
// folded by parity, times the stored inverse of the k^2 = 0 operator.  One
// thread per row with lanes along the contiguous index of both matrices.
__device__ void mean_mode_block(const HsArgs& a, double* sm) {
  const int Ny = a.Ny, N = a.N, ne = a.ne, no = a.no;
  double* x = sm;            // [Ny][4]: U.re U.im W.re W.im
  double* b = sm + 4 * Ny;   // [Ny][4]: even rows, then odd rows
  for (int l = threadIdx.x; l < Ny; l += blockDim.x) {
    const double2 U = a.au0[l], W = a.w0[l];
    x[4 * l] = U.x; x[4 * l + 1] = U.y; x[4 * l + 2] = W.x; x[4 * l + 3] = W.y;
  }
  __syncthreads();
  for (int row = threadIdx.x; row < Ny; row += blockDim.x) {
    const bool odd = row >= ne;
    const int p = odd ? row - ne : row, q = N - p;
    double acc[4] = {0, 0, 0, 0};
    if (p >= 1) {
#pragma unroll 8
      for (int l = odd ? 1 : 0; l <= N; l += 2) {
        const double t = a.tmean[(long)l * Ny + p];
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] += t * x[4 * l + i];
      }
      const double hd = -1.0 * a.dt / 2.0, s = odd ? -1.0 : 1.0;
      const double2 hn[2] = {a.c1n[p], a.c3n[p]}, hp[2] = {a.c1p[p], a.c3p[p]};
      const double2 gn[2] = {a.c1n[q], a.c3n[q]}, gp[2] = {a.c1p[q], a.c3p[q]};
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const double fx = hd * (3.0 * hn[i].x - hp[i].x), fy = hd * (3.0 * hn[i].y - hp[i].y);
        const double gx = hd * (3.0 * gn[i].x - gp[i].x), gy = hd * (3.0 * gn[i].y - gp[i].y);
        acc[2 * i] += p == q ? fx : 0.5 * (fx + s * gx);
        acc[2 * i + 1] += p == q ? fy : 0.5 * (fy + s * gy);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) b[4 * row + i] = acc[i];
  }
  __syncthreads();
  const int neP = ne + (ne & 1), noP = no + (no & 1), rowlen = neP + noP;
  for (int row = threadIdx.x; row < Ny; row += blockDim.x) {
    const bool odd = row >= ne;
    const int i = odd ? row - ne : row, n = odd ? no : ne;
    const double* M = a.inv0 + (odd ? neP : 0) + i;
    const double* r = b + (odd ? 4 * ne : 0);
    double acc[4] = {0, 0, 0, 0};
#pragma unroll 8
    for (int j = 0; j < n; ++j) {
      const double t = M[(long)j * rowlen];
#pragma unroll
      for (int k = 0; k < 4; ++k) acc[k] = fma(t, r[4 * j + k], acc[k]);
    }
    const int l = 2 * i + (odd ? 1 : 0);
    a.au0[l] = make_double2(acc[0], acc[1]);
    a.w0[l] = make_double2(acc[2], acc[3]);
  }
}

// IS_V: the v system (right-hand-side rows from p = 2) or omega_y (from p = 1).
// A block takes CT real columns; its WR x WC waves split the 16-row blocks into
// WR groups of up to RB and the columns into WC groups of CB 16-column blocks.
template <bool IS_V, int CT, int WR, int WC, int RB>
__device__ __forceinline__ void hsolve_block(const HsArgs& a, double* sB) {
  using MF = Mf<double>;
  constexpr int CB = CT / 16 / WC, NT = 64 * WR * WC;
  const int par = blockIdx.y;
  const int tile = (int)blockIdx.x - 1;
  if (tile < 0) {
    if (IS_V && par == 0) mean_mode_block(a, sB);
    return;
  }
  const int m = par ? a.m[1] : a.m[0];
  const int MB = (m + 15) / 16, KP = (m + 7) / 8, R = 16 * MB;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wr = wave / WC, wc = wave % WC;
  const int rb0 = wr * RB;  // this wave's row blocks rb0 .. rb0 + RB - 1 (those < MB)
  const int cl = wc * CB * 16 + (lane & 15);  // its first column in the tile
  const long col0 = (long)tile * (CT / 2);    // first complex column
  double* red = sB;  // [WR][CT][2], between the products' uses of sB

  // stage B: matrix row r holds the right-hand side of point p = r + 1; rows
  // without one (v at p = 1, the padding) and columns past the end are zero
  {
    const double2* ro = IS_V ? (par ? a.rhs[0][1] : a.rhs[0][0]) : (par ? a.rhs[1][1] : a.rhs[1][0]);
    constexpr int off = IS_V ? 1 : 0, SL = (16 * WR * RB * CT / 2 + NT - 1) / NT;  // every load in flight at once
    const int nst = R * (CT / 2), last = m - 1 - off;
    for (int i0 = threadIdx.x; i0 < nst; i0 += SL * NT) {
      double2 v[SL];
#pragma unroll
      for (int u = 0; u < SL; ++u) {
        const int idx = i0 + u * NT, r = idx / (CT / 2) - off;
        const long cc = col0 + idx % (CT / 2);
        const bool in = idx < nst && r >= 0 && r <= last && cc < a.ncol;
        v[u] = in ? ro[(long)r * a.ncol + cc] : make_double2(0, 0);
      }
#pragma unroll
      for (int u = 0; u < SL; ++u) {
        const int idx = i0 + u * NT;
        if (idx < nst) *reinterpret_cast<double2*>(sB + 2 * idx) = v[u];
      }
    }
  }
  __syncthreads();

  MF::acc acc[RB][CB];
  // acc = A B over the m rows of B, eight at a time: a lane's A values of two
  // k blocks come as one 16-byte load (from L2), requested one step ahead
  auto product = [&](const double2* A) {
#pragma unroll
    for (int t = 0; t < RB; ++t)
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) acc[t][cb] = MF::acc{0, 0, 0, 0};
    double2 fa[RB], fb[RB];
    auto fetch = [&](double2 (&f)[RB], int kp) {
#pragma unroll
      for (int t = 0; t < RB; ++t) f[t] = A[((long)min(rb0 + t, MB - 1) * KP + min(kp, KP - 1)) * 64 + lane];
    };
    auto use = [&](const double2 (&f)[RB], int kp) {
      double b[2][CB];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) b[h][cb] = sB[(8 * kp + 4 * h + (lane >> 4)) * CT + cl + 16 * cb];
#pragma unroll
      for (int t = 0; t < RB; ++t) {
        if (rb0 + t < MB) {
#pragma unroll
          for (int cb = 0; cb < CB; ++cb) {
            acc[t][cb] = MF::mma(f[t].x, b[0][cb], acc[t][cb]);
            acc[t][cb] = MF::mma(f[t].y, b[1][cb], acc[t][cb]);
          }
        }
      }
    };
    fetch(fa, 0);
    for (int kp = 0; kp < KP; kp += 2) {
      fetch(fb, kp + 1);
      use(fa, kp);
      if (kp + 1 >= KP) break;
      fetch(fa, kp + 2);
      use(fb, kp + 1);
    }
  };
  product(par ? a.L[1] : a.L[0]);
  __syncthreads();

  // scale per (row, mode); v: the two wall conditions
  const double* vec = par ? a.vec[1] : a.vec[0];
  double k2[CB];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    const long cm = min(col0 + ((cl + 16 * cb) >> 1), a.ncol - 1);
    const int kz = (int)((unsigned)cm / (unsigned)a.Mx), kx = (int)(cm - (long)kz * a.Mx);
    const double alx = a.al[kx], bez = a.be[kz];
    k2[cb] = alx * alx + bez * bez;
  }
  if constexpr (!IS_V) {
#pragma unroll
    for (int t = 0; t < RB; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = 16 * (rb0 + t) + MF::row(lane, e);
        if (row >= R) continue;
        const double lam = vec[row];
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) sB[row * CT + cl + 16 * cb] = acc[t][cb][e] / (1.0 + a.c * (k2[cb] - lam));
      }
  } else {
    // s is formed twice: holding it across the wall sums costs a wave per SIMD
    auto scale = [&](double lam, double k) { return 1.0 / ((1.0 + a.c * (k - lam)) * (lam - k)); };
    double d1[CB] = {}, d2[CB] = {};
#pragma unroll
    for (int t = 0; t < RB; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = min(16 * (rb0 + t) + MF::row(lane, e), R - 1);
        const bool in = rb0 + t < MB;
        const double lam = vec[row], w1 = in ? vec[R + row] : 0.0, w2 = in ? vec[2 * R + row] : 0.0;
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
          const double x = acc[t][cb][e] * scale(lam, k2[cb]);
          d1[cb] += w1 * x;
          d2[cb] += w2 * x;
        }
      }
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
#pragma unroll
      for (int o = 16; o < 64; o <<= 1) {
        d1[cb] += __shfl_xor(d1[cb], o);
        d2[cb] += __shfl_xor(d2[cb], o);
      }
      if (WR > 1 && lane < 16) {
        red[(wr * CT + cl + 16 * cb) * 2] = d1[cb];
        red[(wr * CT + cl + 16 * cb) * 2 + 1] = d2[cb];
      }
    }
    if constexpr (WR > 1) __syncthreads();
    const double* wall = par ? a.wall[1] : a.wall[0];
    double wa[CB], wb[CB];
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      double e1 = d1[cb], e2 = d2[cb];
      if constexpr (WR > 1) {
        const double* r0 = red + (cl + 16 * cb) * 2;
        e1 = r0[0];
        e2 = r0[1];
#pragma unroll
        for (int g = 1; g < WR; ++g) {
          e1 += r0[2 * CT * g];
          e2 += r0[2 * CT * g + 1];
        }
      }
      const double* w = wall + 4 * min(col0 + ((cl + 16 * cb) >> 1), a.ncol - 1);
      wa[cb] = w[0] * e1 + w[1] * e2;
      wb[cb] = w[2] * e1 + w[3] * e2;
    }
    if constexpr (WR > 1) __syncthreads();
#pragma unroll
    for (int t = 0; t < RB; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = 16 * (rb0 + t) + MF::row(lane, e);
        if (row >= R) continue;
        const double lam = vec[row], l1 = vec[3 * R + row], q = vec[4 * R + row];
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
          sB[row * CT + cl + 16 * cb] = scale(lam, k2[cb]) * (acc[t][cb][e] + (wa[cb] * l1 - wb[cb] * q));
      }
  }
  __syncthreads();
  product(par ? a.V[1] : a.V[0]);

  if constexpr (WR > 1) __syncthreads();
  // x_0 = -sum of x_1 .. x_m (padding rows are zero)
  double sum[CB] = {};
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
#pragma unroll
    for (int t = 0; t < RB; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[cb] += acc[t][cb][e];
#pragma unroll
    for (int o = 16; o < 64; o <<= 1) sum[cb] += __shfl_xor(sum[cb], o);
    if (WR > 1 && lane < 16) red[wr * CT + cl + 16 * cb] = sum[cb];
  }
  if constexpr (WR > 1) __syncthreads();
  // the mean mode and the span Nyquist column are not solved here (PF:247)
  const long ncold = 2 * a.ncol;
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    const long col = 2 * col0 + cl + 16 * cb, cm = col >> 1;
    if (cm >= a.ncol || cm == 0 || (int)((unsigned)cm / (unsigned)a.Mx) == a.Mz / 2) continue;
    double* o = (IS_V ? a.out[0] : a.out[1]) + (long)par * ncold + col;
    if (wr == 0 && lane < 16) {
#pragma unroll
      for (int g = 1; g < WR; ++g) sum[cb] += red[g * CT + cl + 16 * cb];
      o[0] = -sum[cb];
    }
#pragma unroll
    for (int t = 0; t < RB; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = 16 * (rb0 + t) + MF::row(lane, e);
        if (row < m) o[2L * (row + 1) * ncold] = acc[t][cb][e];
      }
  }
}

// Both equations in one launch (first = 0, two layers), or one of them.
template <int CT, int WR, int WC, int RB, int WPS>
__global__ __launch_bounds__(64 * WR * WC, WPS) void k_hsolve(HsArgs a, int first) {
  extern __shared__ double sB[];  // [16 MB rows][CT]
  if (first + blockIdx.z == 0) hsolve_block<true, CT, WR, WC, RB>(a, sB);
  else hsolve_block<false, CT, WR, WC, RB>(a, sB);
}

// The wall matrices of every column and parity (wall_matrix of helmholtz.h).
__global__ __launch_bounds__(256) void k_wall(HsArgs a, double* out0, double* out1) {
  const int par = blockIdx.y;
  const int R = 16 * (((par ? a.m[1] : a.m[0]) + 15) / 16), m = par ? a.m[1] : a.m[0];
  const double* vec = par ? a.vec[1] : a.vec[0];
  const long cm = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (cm >= a.ncol) return;
  const int kz = (int)((unsigned)cm / (unsigned)a.Mx), kx = (int)(cm - (long)kz * a.Mx);
  const double k2 = a.al[kx] * a.al[kx] + a.be[kz] * a.be[kz];
  double m11 = 0, m12 = 0, m21 = 0, m22 = -1.0 / a.c;
  for (int j = 0; j < m; ++j) {
    const double lam = vec[j], s = 1.0 / ((1.0 + a.c * (k2 - lam)) * (lam - k2));
    const double w1 = vec[R + j] * s, w2 = vec[2 * R + j] * s, l1 = vec[3 * R + j], q = vec[4 * R + j];
    m11 += w1 * l1;
    m12 -= w1 * q;
    m21 += w2 * l1;
    m22 -= w2 * q;
  }
  const double det = m11 * m22 - m12 * m21;
  double* o = (par ? out1 : out0) + 4 * cm;
  o[0] = -m22 / det;
  o[1] = m12 / det;
  o[2] = m21 / det;
  o[3] = -m11 / det;
}

static HsArgs hs_args(const Ctx& c) {
  const Dims& d = c.d;
  HsArgs a{};
  for (int p = 0; p < 2; ++p) {
    a.L[p] = c.hL[p];
    a.V[p] = c.hV[p];
    a.vec[p] = c.hvec[p];
    a.wall[p] = c.hwall[p];
  }
  a.al = c.alpha;
  a.be = c.beta;
  a.m[0] = d.ne - 1;
  a.m[1] = d.no - 1;
  a.Mx = d.Mx;
  a.Mz = d.Mz;
  a.ncol = d.ncol;
  a.c = c.prm.dt * 0.5 / c.prm.re;
  a.N = d.N;
  a.Ny = d.Ny;
  a.ne = d.ne;
  a.no = d.no;
  a.dt = c.prm.dt;
  return a;
}

hipError_t launch_wall_setup(Ctx& c) {
  const HsArgs a = hs_args(c);
  hipLaunchKernelGGL(k_wall, dim3((unsigned)((c.d.ncol + 255) / 256), 2), dim3(256), 0, c.stream, a, c.hwall[0],
                     c.hwall[1]);
  return hipGetLastError();
}

template <int CT, int WR, int WC, int RB, int WPS>
static hipError_t run_hsolve(Ctx& c, const HsArgs& a, int first, int count) {
  const size_t shm = sizeof(double) * (size_t)CT * 16 * ((a.m[0] + 15) / 16);
  const unsigned tiles = (unsigned)((2 * a.ncol + CT - 1) / CT);
  if (sizeof(double) * 8ull * a.Ny > shm) return hipErrorInvalidValue;  // the mean-mode block's arrays
  hipLaunchKernelGGL((k_hsolve<CT, WR, WC, RB, WPS>), dim3(tiles + 1, 2, count), dim3(64 * WR * WC), shm, c.stream, a,
                     first);
  return hipGetLastError();
}

hipError_t launch_hsolve(Ctx& c, int first, int count) {
  HsArgs a = hs_args(c);
  a.rhs[0][0] = c.rvE;
  a.rhs[0][1] = c.rvO;
  a.rhs[1][0] = c.roE;
  a.rhs[1][1] = c.roO;
  a.out[0] = reinterpret_cast<double*>(c.v);
  a.out[1] = reinterpret_cast<double*>(c.oy);
  a.au0 = c.au0;
  a.w0 = c.w0;
  a.c1n = c.cl1[c.hcur];
  a.c1p = c.cl1[1 - c.hcur];
  a.c3n = c.cl3[c.hcur];
  a.c3p = c.cl3[1 - c.hcur];
  a.tmean = c.tmean;
  a.inv0 = c.inv0;
  // CT, WR, WC, RB by the row blocks of the even half system (the odd one has as
  // many or one less).  The resident blocks run in step (they start together and
  // a launch is a few rounds of them), so loads, products and stores overlap the
  // less the longer a block is: with 32 columns and a wave's tile of 2 x 2 (7, 8
  // row blocks) instead of 64 and 4 x 2, 16 waves a CU fit in the place of 8, and
  // the products reach 49 TFLOP/s in the place of 43 (v / omega_y, us: 256x257x256
  // 235 / 202 -> 204 / 176, 256x225x256 200 / 175 -> 175 / 150; 96x97x96 21 / 15.3
  // -> 17.5 / 14.1; 64x65x64 11.4 / 8.9 -> 10.0 / 7.8).  From 4 to 6 row blocks
  // 64 columns stay: 256x193x256 138 / 117, with 32 columns 148 / 123 to 152 / 132
  // (one wave per row block 181 / 148: six waves load the four SIMDs unevenly),
  // 192x161x192 76 / 63 against 76 / 62, 128x129x128 30 / 23 against 34 / 23.
  switch ((a.m[0] + 15) / 16) {
    case 1: return run_hsolve<64, 1, 4, 1, 3>(c, a, first, count);
    case 2: return run_hsolve<32, 2, 2, 1, 4>(c, a, first, count);
    case 3: return run_hsolve<32, 3, 1, 1, 4>(c, a, first, count);
    case 4: return run_hsolve<64, 2, 2, 2, 3>(c, a, first, count);
    case 5: case 6: return run_hsolve<64, 2, 2, 3, 3>(c, a, first, count);
    case 7: case 8: return run_hsolve<32, 4, 1, 2, 4>(c, a, first, count);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace chf
