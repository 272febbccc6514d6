// Passes along the degree of every (kx, kz) column: the kinematics after a solve
// and the h assembly after the products.
//
//   kinematics : u, w, omega_x, omega_z and the next solve's right-hand-side
//                brackets from v, omega_y (getvelocityandvorticity PF:2347-2407)
//   hassemble  : h_v = k^2 L_y + i alpha D L_x + i beta D L_z,
//                h_g = i alpha L_z - i beta L_x (PF:1502-1540, dz PF:570-599)
//
// Both rest on the coefficient derivative b_k = b_(k+2) + 2 (k+1) a_(k+1), a suffix
// sum over the degrees of one parity.  Large grids run it as a serial chain, one
// thread per column, whose loads stream; small grids, where those chains leave
// the chip idle for the latency of every batch of loads, in segments.
#include "chf_internal.h"
#include "fftreg.h"
#include "segments.h"

namespace chf {

// ------------------------------------------------------------- kinematics

// getvelocityandvorticity (PF:2347-2407) for every mode with k^2 != 0:
//   u = (i alpha Dv - i beta omega_y)/k^2,  w = (i beta Dv + i alpha omega_y)/k^2,
//   omega_x = Dw - i beta v,                omega_z = -Du + i alpha v,
// and for the mean mode (PF:435-438, 469-472) u = U, w = W, omega_z = -DU,
// omega_x = DW.  D is the coefficient-space derivative of dz (PF:570-599),
// b_k = b_{k+2} + 2(k+1) a_{k+1}, b_0 halved.
//
// The recurrences split into two independent chains by degree parity: chain q
// reads v at degrees of parity q and omega_y at parity 1-q, and produces
// Dv, u, w at parity 1-q and Du, Dw, omega_x, omega_z at parity q.  One thread
// runs one chain of one mode, backwards over the degree, with its loads issued
// eight degrees ahead.  Its outputs are stored non-temporally: the next
// kernels read them, this one does not (the padded synthesis that reads u, w,
// omega_x, omega_z runs 5% faster, this pass 3% slower).
//
// The same pass forms the explicit-operator brackets of the next solve's
// right-hand sides (get_coef_rhs / get_rhs_omegay, PF:252-257, 335-340):
//   g_v = c D^4 v + (1 - 2 c k^2) D^2 v - k^2 (1 - c k^2) v   (at parity q)
//   g_w = c D^2 omega_y + (1 - c k^2) omega_y                  (at parity 1-q)
// whose chains read the same v and omega_y degrees as chain q.
struct KinArgs {
  const double2 *v, *oy, *au0, *w0;
  double2 *u, *w, *ox, *oz;
  float2 *uf, *wf, *oxf, *ozf;  // F32: u, w, omega_x, omega_z rounded to FP32, written instead
  double2 *gv, *go;  // brackets for the next solve
  const double *al, *be;
  int* nonfinite;    // set to 1 when v, omega_y, U or W hold a NaN or an infinity
  int Mx, Mz, N, Ny;
  long ncol;
  double c;          // dt / (2 re)
};

// u, w, omega_x, omega_z at one offset: FP64, or (F32) rounded to FP32
template <bool F32>
__device__ __forceinline__ void kin_store(const KinArgs& a, int which, long off, double2 v) {
  if constexpr (F32) {
    float2* p = which == 0 ? a.uf : which == 1 ? a.wf : which == 2 ? a.oxf : a.ozf;
    st_nt(p + off, make_float2((float)v.x, (float)v.y));
  } else {
    double2* p = which == 0 ? a.u : which == 1 ? a.w : which == 2 ? a.ox : a.oz;
    st_nt(p + off, v);
  }
}

template <bool F32>
__global__ __launch_bounds__(256) void k_kinematics(KinArgs a) {
  const int q = blockIdx.y;  // chain: parity of the v degrees it reads
  const int N = a.N;
  if (blockIdx.x == gridDim.x - 1) {
    // mean mode, one block: U, W staged in LDS, derivatives by lanes 0..3
    if (q != 0) return;
    extern __shared__ double sm[];
    double* x = sm;              // U.re U.im W.re W.im   [4][Ny]
    double* d = sm + 4 * a.Ny;   // DU.re DU.im DW.re DW.im
    bool finite = true;
    for (int k = threadIdx.x; k < a.Ny; k += blockDim.x) {
      const double2 U = a.au0[k], W = a.w0[k];
      x[0 * a.Ny + k] = U.x; x[1 * a.Ny + k] = U.y; x[2 * a.Ny + k] = W.x; x[3 * a.Ny + k] = W.y;
      finite = finite && isfinite(U.x) && isfinite(U.y) && isfinite(W.x) && isfinite(W.y);
    }
    if (!finite) a.nonfinite[0] = 1;
    __syncthreads();
    if (threadIdx.x < 4) {
      const double* xa = x + threadIdx.x * a.Ny;
      double* b = d + threadIdx.x * a.Ny;
      double b2 = 0.0, b1 = 0.0;
      b[N] = 0.0;
      for (int k = N - 1; k >= 0; --k) {
        const double bk = b2 + 2.0 * (k + 1) * xa[k + 1];
        b2 = b1;
        b1 = bk;
        b[k] = (k == 0) ? 0.5 * bk : bk;
      }
    }
    __syncthreads();
    for (int k = threadIdx.x; k < a.Ny; k += blockDim.x) {
      const long off = (long)k * a.ncol;
      kin_store<F32>(a, 0, off, make_double2(x[0 * a.Ny + k], x[1 * a.Ny + k]));
      kin_store<F32>(a, 1, off, make_double2(x[2 * a.Ny + k], x[3 * a.Ny + k]));
      kin_store<F32>(a, 3, off, make_double2(-1.0 * d[0 * a.Ny + k], -1.0 * d[1 * a.Ny + k]));
      kin_store<F32>(a, 2, off, make_double2(d[2 * a.Ny + k], d[3 * a.Ny + k]));
    }
    return;
  }
  const long cm = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (cm >= a.ncol || cm == 0) return;
  const int kz = (int)((unsigned)cm / (unsigned)a.Mx);
  const int kx = (int)(cm - (long)kz * a.Mx);
  if (kz == a.Mz / 2) return;  // span Nyquist: never solved, stays zero (PF:247)
  const double al = a.al[kx], be = a.be[kz];
  const double k2 = al * al + be * be;
  double2 vp = make_double2(0, 0);                    // v_{k+1}
  double2 dv2 = make_double2(0, 0);                   // Dv_{k+2} (unhalved)
  double2 up = make_double2(0, 0), wp = make_double2(0, 0);    // u_{k+1}, w_{k+1}
  double2 du2 = make_double2(0, 0), dw2 = make_double2(0, 0);  // Du_{k+2}, Dw_{k+2}
  // bracket chains: latest unhalved D^2 v, D^3 v, D^4 v, D omega, D^2 omega and omega_{k+1}
  double2 d2s = make_double2(0, 0), d3s = make_double2(0, 0), d4s = make_double2(0, 0);
  double2 e1s = make_double2(0, 0), e2s = make_double2(0, 0), wn = make_double2(0, 0);
  const double cc = a.c, c2 = 1.0 - 2.0 * cc * k2, c0 = k2 * (1.0 - cc * k2), cw = 1.0 - cc * k2;
  // x * 0 is 0 for every finite x and NaN for a NaN or an infinity: one
  // multiply-add per value, no branch between the batched loads
  double probe = 0.0;
  for (int k0 = N; k0 >= 0; k0 -= 8) {
    double2 in[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int k = k0 - s;
      if (k >= 0) in[s] = (((k & 1) == q) ? a.v : a.oy)[(long)k * a.ncol + cm];
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int k = k0 - s;
      if (k < 0) break;
      const long off = (long)k * a.ncol + cm;
      const double f = 2.0 * (k + 1);
      if ((k & 1) == q) {
        // Du_k, Dw_k from u_{k+1}, w_{k+1}; omega_x, omega_z with v_k
        double2 du = make_double2(du2.x + f * up.x, du2.y + f * up.y);
        double2 dw = make_double2(dw2.x + f * wp.x, dw2.y + f * wp.y);
        du2 = du;
        dw2 = dw;
        if (k == 0) {
          du.x *= 0.5; du.y *= 0.5; dw.x *= 0.5; dw.y *= 0.5;
        }
        const double2 vk = in[s];
        kin_store<F32>(a, 2, off, make_double2(dw.x + be * vk.y, dw.y - be * vk.x));
        kin_store<F32>(a, 3, off, make_double2(-du.x - al * vk.y, -du.y + al * vk.x));
        // brackets: D^2 v, D^4 v at k from D v, D^3 v at k+1; D omega at k from omega_{k+1}
        double2 q2 = make_double2(d2s.x + f * dv2.x, d2s.y + f * dv2.y);
        double2 q4 = make_double2(d4s.x + f * d3s.x, d4s.y + f * d3s.y);
        e1s = make_double2(e1s.x + f * wn.x, e1s.y + f * wn.y);
        d2s = q2;
        d4s = q4;
        if (k == 0) {
          q2.x *= 0.5; q2.y *= 0.5; q4.x *= 0.5; q4.y *= 0.5;
        }
        st_nt(&a.gv[off], make_double2(cc * q4.x + c2 * q2.x - c0 * vk.x, cc * q4.y + c2 * q2.y - c0 * vk.y));
        vp = vk;
      } else {
        // Dv_k from v_{k+1}; u_k, w_k with omega_y_k
        double2 dv = make_double2(dv2.x + f * vp.x, dv2.y + f * vp.y);
        dv2 = dv;
        if (k == 0) {
          dv.x *= 0.5; dv.y *= 0.5;
        }
        const double omr = in[s].x, omi = in[s].y;
        const double2 uk = make_double2(-1.0 * al * dv.y / k2 + be * omi / k2, al * dv.x / k2 - be * omr / k2);
        const double2 wk = make_double2(-1.0 * dv.y * be / k2 - 1.0 * omi * al / k2, be * dv.x / k2 + al * omr / k2);
        kin_store<F32>(a, 0, off, uk);
        kin_store<F32>(a, 1, off, wk);
        up = uk;
        wp = wk;
        // brackets: D^3 v at k from D^2 v at k+1; D^2 omega at k from D omega at k+1
        d3s = make_double2(d3s.x + f * d2s.x, d3s.y + f * d2s.y);
        double2 r2 = make_double2(e2s.x + f * e1s.x, e2s.y + f * e1s.y);
        e2s = r2;
        if (k == 0) {
          r2.x *= 0.5; r2.y *= 0.5;
        }
        st_nt(&a.go[off], make_double2(cc * r2.x + cw * omr, cc * r2.y + cw * omi));
        wn = in[s];
      }
      probe = fma(in[s].x, 0.0, fma(in[s].y, 0.0, probe));
    }
  }
  if (probe != probe) a.nonfinite[0] = 1;
}

// ---------------------------------------------------------------- h assembly

// L^n coefficients in FP64, or (mixed form with FFT transforms) in FP32: the
// FP32 analysis's results, exact in either width
struct LIn {
  const double2* d;
  const float2* f;
  // the stored value (float2 or double2); widened where it is used, so that
  // a batch of loads stays in flight
  template <bool F32>
  __device__ __forceinline__ auto raw(long i) const {
    if constexpr (F32) return f[i];
    else return d[i];
  }
  template <bool F32>
  __device__ __forceinline__ double2 at(long i) const {
    const auto v = raw<F32>(i);
    return make_double2(v.x, v.y);
  }
};

template <class V>
__device__ __forceinline__ double2 widen(V v) {
  return make_double2(v.x, v.y);
}

struct MArgs {
  LIn lx, lz;
  double2 *o1, *o3;
  const double* costab;  // cos(pi n / 2N), n < 4N
  int N, Pn;
  long ncol;
};

// The cosines come from LDS: read as table rows from the L2, whose latency every
// few degrees waited for, they made this block the longest of a small grid's launch
// (us, rows / LDS: 128x97x128 mixed 22.9 / 15.8, 96x101x96 FP64 21.3 / 14.9,
// 128x129x128 33.2 / 27.5, 64x65x64 9.9 / 8.2; eight or sixteen rows in flight 27 to 54).
template <bool F32>
__device__ void mean_points_block(const MArgs& a) {
  __shared__ double2 s1[260], s3[260];
  __shared__ double ct[512];  // cos(pi m / N), m < 2N
  for (int l = threadIdx.x; l <= a.N; l += blockDim.x) {
    s1[l] = a.lx.at<F32>((long)l * a.ncol);
    s3[l] = a.lz.at<F32>((long)l * a.ncol);
  }
  for (int m = threadIdx.x; m < 2 * a.N; m += blockDim.x) ct[m] = a.costab[2 * m];
  __syncthreads();
  for (int jj = threadIdx.x; jj < a.Pn; jj += blockDim.x) {
    double2 e1 = make_double2(0, 0), o1 = make_double2(0, 0);
    double2 e3 = make_double2(0, 0), o3 = make_double2(0, 0);
    int m = 0;  // l jj mod 2N: T_l(y_jj) = cos(pi l jj / N)
#pragma unroll 4
    for (int l = 0; l <= a.N; ++l) {
      const double t = ct[m];
      m += jj;
      if (m >= 2 * a.N) m -= 2 * a.N;
      const double2 x1 = s1[l], x3 = s3[l];
      if (l & 1) {
        o1.x += t * x1.x; o1.y += t * x1.y;
        o3.x += t * x3.x; o3.y += t * x3.y;
      } else {
        e1.x += t * x1.x; e1.y += t * x1.y;
        e3.x += t * x3.x; e3.y += t * x3.y;
      }
    }
    a.o1[jj] = make_double2(e1.x + o1.x, e1.y + o1.y);
    a.o3[jj] = make_double2(e3.x + o3.x, e3.y + o3.y);
    const int q = a.N - jj;
    if (q != jj) {
      a.o1[q] = make_double2(e1.x - o1.x, e1.y - o1.y);
      a.o3[q] = make_double2(e3.x - o3.x, e3.y - o3.y);
    }
  }
}

struct HArgs {
  LIn lx, ly, lz;
  double2 *hv, *hg;
  const double *al, *be;
  int Mx, N;
  long ncol;
};

// One thread per complex column; the derivative runs the backward recurrence
// c_k b_k = b_{k+2} + 2 (k+1) a_{k+1}, which equals the reference's explicit
// sum b_k = (2/c_k) sum_{j>k, j+k odd} j a_j.
// The launch carries one extra block that computes the mean-mode Lamb point
// values (mean_points_block) from the same coefficients.
template <bool F32>
__global__ __launch_bounds__(256) void k_hassemble(HArgs a, MArgs m) {
  if (blockIdx.x == gridDim.x - 1) {
    mean_points_block<F32>(m);
    return;
  }
  const long cm = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (cm >= a.ncol) return;
  const int kz = (int)((unsigned)cm / (unsigned)a.Mx);
  const int kx = (int)(cm - (long)kz * a.Mx);
  const double al = a.al[kx], be = a.be[kz];
  const double k2 = al * al + be * be;
  const int N = a.N;
  double2 bx2 = make_double2(0, 0), bx1 = make_double2(0, 0);
  double2 bz2 = make_double2(0, 0), bz1 = make_double2(0, 0);
  double2 lxn = make_double2(0, 0), lzn = make_double2(0, 0);  // a_{k+1}
  for (int k0 = N; k0 >= 0; k0 -= 4) {
    // loads issued four degrees ahead of the recurrence
    decltype(a.lx.raw<F32>(0)) pl[4][3];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int k = k0 - t;
      if (k >= 0) {
        const long off = (long)k * a.ncol + cm;
        pl[t][0] = a.lx.raw<F32>(off);
        pl[t][1] = a.ly.raw<F32>(off);
        pl[t][2] = a.lz.raw<F32>(off);
      }
    }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int k = k0 - t;
    if (k < 0) break;
    const long off = (long)k * a.ncol + cm;
    const double2 lx = widen(pl[t][0]), ly = widen(pl[t][1]), lz = widen(pl[t][2]);
    double2 dx, dz;
    if (k == N) {
      dx = make_double2(0, 0);
      dz = make_double2(0, 0);
    } else {
      const double f = 2.0 * (k + 1);
      dx = make_double2(bx2.x + f * lxn.x, bx2.y + f * lxn.y);
      dz = make_double2(bz2.x + f * lzn.x, bz2.y + f * lzn.y);
    }
    bx2 = bx1;
    bx1 = dx;
    bz2 = bz1;
    bz1 = dz;
    if (k == 0) {
      dx.x *= 0.5;
      dx.y *= 0.5;
      dz.x *= 0.5;
      dz.y *= 0.5;
    }
    // h_v = (k^2 L_y + i alpha D L_x) + i beta D L_z
    double hvr = k2 * ly.x - al * dx.y;
    double hvi = k2 * ly.y + al * dx.x;
    hvr = hvr - be * dz.y;
    hvi = hvi + be * dz.x;
    // h_g = i alpha L_z - i beta L_x
    const double hgr = -1.0 * al * lz.y + be * lx.y;
    const double hgi = al * lz.x - be * lx.x;
    a.hv[off] = make_double2(hvr, hvi);
    a.hg[off] = make_double2(hgr, hgi);
    lxn = lx;
    lzn = lz;
  }
  }
}

// ------------------------------------------------------------ segmented forms

// A block takes kSegCols columns; thread (s, tx) holds the degrees s SL .. s SL +
// SL - 1 (SL even) of column tx in registers, all loads in flight at once, and a
// derivative is the local suffix sums plus the totals of the segments above,
// exchanged through LDS.  Bound: the latency of one load, one to four exchanges
// and the stores, against that of every batch of the serial chain.
constexpr int kSegCols = 8, kMaxSegs = 28;

// Degrees per segment: the smallest even count that covers N + 1 degrees with
// kMaxSegs segments (2 .. 10).
static int seg_len(int Ny) {
  int sl = 2;
  while ((Ny + sl - 1) / sl > kMaxSegs) sl += 2;
  return sl;
}

struct SegTotals {
  double2 t[kMaxSegs][2][kSegCols];  // per segment: sums over even, odd degrees
};

// In place, one segment of a -> its derivative's (local part), and the segment's
// totals of 2 p a_p per parity.
template <int SL>
__device__ __forceinline__ void seg_derive(double2 (&a)[SL], int k0, int s, int tx, SegTotals& tot) {
  double2 acc[2] = {make_double2(0, 0), make_double2(0, 0)};
#pragma unroll
  for (int i = SL - 1; i >= 0; --i) {
    const double f = 2.0 * (k0 + i);
    const double2 x = a[i];
    a[i] = acc[(i + 1) & 1];
    acc[i & 1] = make_double2(acc[i & 1].x + f * x.x, acc[i & 1].y + f * x.y);
  }
  tot.t[s][0][tx] = acc[0];
  tot.t[s][1][tx] = acc[1];
}

// Adds the totals of the segments above (after a barrier).
template <int SL>
__device__ __forceinline__ void seg_add(double2 (&a)[SL], int k0, int s, int G, int tx, const SegTotals& tot) {
  double2 off[2] = {make_double2(0, 0), make_double2(0, 0)};
  for (int q = G - 1; q > s; --q)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const double2 v = tot.t[q][e][tx];
      off[e] = make_double2(off[e].x + v.x, off[e].y + v.y);
    }
#pragma unroll
  for (int i = 0; i < SL; ++i) a[i] = make_double2(a[i].x + off[(i + 1) & 1].x, a[i].y + off[(i + 1) & 1].y);
  if (k0 == 0) a[0] = make_double2(0.5 * a[0].x, 0.5 * a[0].y);
}

// k_kinematics in segments.  The derivatives of u and w come from those of v and
// omega_y.  One extra block runs the mean mode (U in v's place, W in omega_y's).
template <bool F32, int SL>
__global__ __launch_bounds__(kSegCols* kMaxSegs) void k_kinematics_seg(KinArgs a) {
  __shared__ SegTotals tot[2][2];
  const int s = threadIdx.x / kSegCols, tx = threadIdx.x - s * kSegCols, G = blockDim.x / kSegCols;
  const bool mean = blockIdx.x == gridDim.x - 1;
  const long cm = mean ? 0 : (long)blockIdx.x * kSegCols + tx;
  const int kz = (int)((unsigned)cm / (unsigned)a.Mx), kx = (int)(cm - (long)kz * a.Mx);
  // not solved: the span Nyquist column and, but in the mean block, (0,0) (PF:247)
  const bool valid = mean ? tx == 0 : cm < a.ncol && cm != 0 && kz != a.Mz / 2;
  const int k0 = s * SL;
  double2 v[SL], o[SL], d[SL], e[SL];
  double probe = 0.0;
#pragma unroll
  for (int i = 0; i < SL; ++i) {
    const int k = k0 + i;
    const bool in = valid && k <= a.N;
    const long off = mean ? k : (long)k * a.ncol + cm;
    v[i] = in ? (mean ? a.au0 : a.v)[off] : make_double2(0, 0);
    o[i] = in ? (mean ? a.w0 : a.oy)[off] : make_double2(0, 0);
  }
#pragma unroll
  for (int i = 0; i < SL; ++i) {
    probe = fma(v[i].x, 0.0, fma(v[i].y, 0.0, fma(o[i].x, 0.0, fma(o[i].y, 0.0, probe))));
    d[i] = v[i];
    e[i] = o[i];
  }
  if (probe != probe) a.nonfinite[0] = 1;
  const double al = valid ? a.al[kx] : 0.0, be = valid ? a.be[kz] : 0.0;
  const double k2 = al * al + be * be;
  const double ia = valid && !mean ? al / k2 : 0.0, ib = valid && !mean ? be / k2 : 0.0;
  // D v, D omega_y
  seg_derive<SL>(d, k0, s, tx, tot[0][0]);
  seg_derive<SL>(e, k0, s, tx, tot[0][1]);
  __syncthreads();
  seg_add<SL>(d, k0, s, G, tx, tot[0][0]);
  seg_add<SL>(e, k0, s, G, tx, tot[0][1]);
  if (mean) {  // u = U, w = W, omega_x = DW, omega_z = -DU (PF:435-438, 469-472)
    if (valid)
#pragma unroll
      for (int i = 0; i < SL; ++i) {
        if (k0 + i > a.N) break;
        const long off = (long)(k0 + i) * a.ncol;
        kin_store<F32>(a, 0, off, v[i]);
        kin_store<F32>(a, 1, off, o[i]);
        kin_store<F32>(a, 2, off, e[i]);
        kin_store<F32>(a, 3, off, make_double2(-d[i].x, -d[i].y));
      }
    return;
  }
  if (valid)
#pragma unroll
    for (int i = 0; i < SL; ++i) {
      if (k0 + i > a.N) break;
      const long off = (long)(k0 + i) * a.ncol + cm;
      kin_store<F32>(a, 0, off, make_double2(ib * o[i].y - ia * d[i].y, ia * d[i].x - ib * o[i].x));
      kin_store<F32>(a, 1, off, make_double2(-ib * d[i].y - ia * o[i].y, ib * d[i].x + ia * o[i].x));
    }
  // D^2 v (in d), D^2 omega_y (in e2)
  double2 e2[SL];
#pragma unroll
  for (int i = 0; i < SL; ++i) e2[i] = e[i];
  seg_derive<SL>(d, k0, s, tx, tot[1][0]);
  seg_derive<SL>(e2, k0, s, tx, tot[1][1]);
  __syncthreads();
  seg_add<SL>(d, k0, s, G, tx, tot[1][0]);
  seg_add<SL>(e2, k0, s, G, tx, tot[1][1]);
  const double cc = a.c, c2 = 1.0 - 2.0 * cc * k2, c0 = k2 * (1.0 - cc * k2), cw = 1.0 - cc * k2;
  double2 g[SL];
#pragma unroll
  for (int i = 0; i < SL; ++i) {
    if (valid && k0 + i <= a.N) {
      const long off = (long)(k0 + i) * a.ncol + cm;
      // Dw = i (ib D^2 v + ia D omega_y), Du = i (ia D^2 v - ib D omega_y)
      kin_store<F32>(a, 2, off, make_double2(be * v[i].y - ib * d[i].y - ia * e[i].y,
                                             ib * d[i].x + ia * e[i].x - be * v[i].x));
      kin_store<F32>(a, 3, off, make_double2(ia * d[i].y - ib * e[i].y - al * v[i].y,
                                             ib * e[i].x - ia * d[i].x + al * v[i].x));
      st_nt(&a.go[off], make_double2(cc * e2[i].x + cw * o[i].x, cc * e2[i].y + cw * o[i].y));
    }
    g[i] = make_double2(c2 * d[i].x - c0 * v[i].x, c2 * d[i].y - c0 * v[i].y);
  }
  // D^3 v, D^4 v
  seg_derive<SL>(d, k0, s, tx, tot[0][0]);
  __syncthreads();
  seg_add<SL>(d, k0, s, G, tx, tot[0][0]);
  seg_derive<SL>(d, k0, s, tx, tot[1][0]);
  __syncthreads();
  seg_add<SL>(d, k0, s, G, tx, tot[1][0]);
  if (valid)
#pragma unroll
    for (int i = 0; i < SL; ++i) {
      if (k0 + i > a.N) break;
      st_nt(&a.gv[(long)(k0 + i) * a.ncol + cm], make_double2(cc * d[i].x + g[i].x, cc * d[i].y + g[i].y));
    }
}

// k_hassemble in segments: one derivative, of alpha L_x + beta L_z.
template <bool F32, int SL>
__global__ __launch_bounds__(kSegCols* kMaxSegs) void k_hassemble_seg(HArgs a, MArgs m) {
  if (blockIdx.x == 0) {  // first, so that it overlaps the others
    mean_points_block<F32>(m);
    return;
  }
  __shared__ SegTotals tot;
  const int s = threadIdx.x / kSegCols, tx = threadIdx.x - s * kSegCols, G = blockDim.x / kSegCols;
  const long cm = (long)(blockIdx.x - 1) * kSegCols + tx;
  const bool valid = cm < a.ncol;
  const int kz = valid ? (int)((unsigned)cm / (unsigned)a.Mx) : 0, kx = valid ? (int)(cm - (long)kz * a.Mx) : 0;
  const double al = a.al[kx], be = a.be[kz], k2 = al * al + be * be;
  const int k0 = s * SL;
  decltype(a.lx.raw<F32>(0)) x[SL], y[SL], z[SL];
#pragma unroll
  for (int i = 0; i < SL; ++i) {
    const bool in = valid && k0 + i <= a.N;
    const long off = in ? (long)(k0 + i) * a.ncol + cm : 0;
    x[i] = a.lx.raw<F32>(off);
    y[i] = a.ly.raw<F32>(off);
    z[i] = a.lz.raw<F32>(off);
    if (!in) x[i].x = x[i].y = z[i].x = z[i].y = 0;
  }
  double2 d[SL];
#pragma unroll
  for (int i = 0; i < SL; ++i) {
    const double2 lx = widen(x[i]), lz = widen(z[i]);
    d[i] = make_double2(al * lx.x + be * lz.x, al * lx.y + be * lz.y);
    // h_g = i (alpha L_z - beta L_x)
    if (valid && k0 + i <= a.N)
      a.hg[(long)(k0 + i) * a.ncol + cm] = make_double2(be * lx.y - al * lz.y, al * lz.x - be * lx.x);
  }
  seg_derive<SL>(d, k0, s, tx, tot);
  __syncthreads();
  seg_add<SL>(d, k0, s, G, tx, tot);
  // h_v = k^2 L_y + i D (alpha L_x + beta L_z)
  if (valid)
#pragma unroll
    for (int i = 0; i < SL; ++i) {
      if (k0 + i > a.N) break;
      const double2 ly = widen(y[i]);
      a.hv[(long)(k0 + i) * a.ncol + cm] = make_double2(k2 * ly.x - d[i].y, k2 * ly.y + d[i].x);
    }
}

template <int SL>
static hipError_t run_kin_seg(Ctx& c, const KinArgs& a, bool f32) {
  const dim3 grid((unsigned)((a.ncol + kSegCols - 1) / kSegCols) + 1), block(kSegCols * ((a.Ny + SL - 1) / SL));
  if (f32) hipLaunchKernelGGL((k_kinematics_seg<true, SL>), grid, block, 0, c.stream, a);
  else hipLaunchKernelGGL((k_kinematics_seg<false, SL>), grid, block, 0, c.stream, a);
  return hipGetLastError();
}

template <int SL>
static hipError_t run_hasm_seg(Ctx& c, const HArgs& a, const MArgs& m, bool f32) {
  const dim3 grid((unsigned)((a.ncol + kSegCols - 1) / kSegCols) + 1), block(kSegCols * ((a.N + SL) / SL));
  if (f32) hipLaunchKernelGGL((k_hassemble_seg<true, SL>), grid, block, 0, c.stream, a, m);
  else hipLaunchKernelGGL((k_hassemble_seg<false, SL>), grid, block, 0, c.stream, a, m);
  return hipGetLastError();
}

hipError_t launch_kinematics(Ctx& c, bool f32) {
  if (f32 && !c.uf) return hipErrorInvalidValue;
  const Dims& d = c.d;
  KinArgs a{};
  a.uf = c.uf;
  a.wf = c.wf;
  a.oxf = c.oxf;
  a.ozf = c.ozf;
  a.v = c.v;
  a.oy = c.oy;
  a.au0 = c.au0;
  a.w0 = c.w0;
  a.u = c.u;
  a.w = c.w;
  a.ox = c.ox;
  a.oz = c.oz;
  a.gv = c.gv;
  a.go = c.go;
  a.al = c.alpha;
  a.be = c.beta;
  a.nonfinite = c.nonfinite;
  a.Mx = d.Mx;
  a.Mz = d.Mz;
  a.N = d.N;
  a.Ny = d.Ny;
  a.ncol = d.ncol;
  a.c = c.prm.dt * 0.5 / c.prm.re;
  if (kinematics_in_segments(d.ncol, c.f32_fields)) {
    const int sl = seg_len(d.Ny);
    switch (sl) {
      case 2: return run_kin_seg<2>(c, a, f32);
      case 4: return run_kin_seg<4>(c, a, f32);
      case 6: return run_kin_seg<6>(c, a, f32);
      case 8: return run_kin_seg<8>(c, a, f32);
      case 10: return run_kin_seg<10>(c, a, f32);
      default: return hipErrorInvalidValue;
    }
  }
  const unsigned nb = (unsigned)((d.ncol + kColumnThreads - 1) / kColumnThreads) + 1;  // + the mean-mode block
  const size_t shm = sizeof(double) * 8ull * d.Ny;
  const void* k = f32 ? (const void*)k_kinematics<true> : (const void*)k_kinematics<false>;
  if (shm > 65536) {
    hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
    if (e != hipSuccess) return e;
  }
  if (f32)
    hipLaunchKernelGGL(k_kinematics<true>, dim3(nb, 2), dim3(kColumnThreads), shm, c.stream, a);
  else
    hipLaunchKernelGGL(k_kinematics<false>, dim3(nb, 2), dim3(kColumnThreads), shm, c.stream, a);
  return hipGetLastError();
}

hipError_t launch_hassemble(Ctx& c) {
  HArgs a{};
  const bool f32 = c.f32_fields;  // the analysis wrote L^n in FP32 (Lcf)
  a.lx = LIn{c.Lc[0], f32 ? c.Lcf[0] : nullptr};
  a.ly = LIn{c.Lc[1], f32 ? c.Lcf[1] : nullptr};
  a.lz = LIn{c.Lc[2], f32 ? c.Lcf[2] : nullptr};
  a.hv = c.hvc;
  a.hg = c.hgc;
  a.al = c.alpha;
  a.be = c.beta;
  a.Mx = c.d.Mx;
  a.N = c.d.N;
  a.ncol = c.d.ncol;
  MArgs m{};
  m.lx = a.lx;
  m.lz = a.lz;
  m.o1 = c.cl1[1 - c.hcur];
  m.o3 = c.cl3[1 - c.hcur];
  m.costab = c.costab;
  m.N = c.d.N;
  m.Pn = c.d.Pn;
  m.ncol = c.d.ncol;
  if (hassemble_in_segments(a.ncol, f32)) {
    switch (seg_len(c.d.Ny)) {
      case 2: return run_hasm_seg<2>(c, a, m, f32);
      case 4: return run_hasm_seg<4>(c, a, m, f32);
      case 6: return run_hasm_seg<6>(c, a, m, f32);
      case 8: return run_hasm_seg<8>(c, a, m, f32);
      case 10: return run_hasm_seg<10>(c, a, m, f32);
      default: return hipErrorInvalidValue;
    }
  }
  const dim3 grid((unsigned)((a.ncol + kColumnThreads - 1) / kColumnThreads) + 1);
  if (f32)
    hipLaunchKernelGGL(k_hassemble<true>, grid, dim3(kColumnThreads), 0, c.stream, a, m);
  else
    hipLaunchKernelGGL(k_hassemble<false>, grid, dim3(kColumnThreads), 0, c.stream, a, m);
  return hipGetLastError();
}

}  // namespace chf
