// Per-(kx,|kz|) solves of the v and omega_y equations with stored inverses
// (PF:242-394; the path taken when the diagonalised operators of hsolve.hip do
// not verify), with their mean mode (PF:401-474), and the GPU set-up of the
// operator inverses (PF:181-204).
//
// The collocation operators of get_coef_v (PF:3348-3381) and get_coef_omegay
// (PF:3432-3455) depend on (kx, kz) through k^2 only, so the modes +kz and
// -kz share one matrix, and with the grid symmetric about y = 0 each
// operator decouples into an even-degree and an odd-degree system:
//   v   : rows (r0+r1)/2, (r2-r3)/2 and the symmetric parts at points
//         p = 2..N/2 (even);  (r0-r1)/2, (r2+r3)/2 and the antisymmetric parts
//         at p = 2..(N-1)/2 (odd);
//   w_y : row (r0+-r1)/2 and the (anti)symmetric parts at p = 1..N/2.
// Set-up inverts each half system once (Gauss-Jordan with partial pivoting in
// LDS); a step multiplies the stored inverses, as the reference multiplies the
// zgetri inverses with a_multiply_x (PF:4123-4139).
#include "chf_internal.h"
#include "fftreg.h"

namespace chf {

// ------------------------------------------------------------------ set-up

struct SetupArgs {
  const double *t0, *t2, *t4;
  const double *al, *be;
  double* inv;      // v halves (null: not stored)
  double* inv_w;    // omega halves
  int Mx, N, Ny, ne, no;
  long stride, row, stride_w, row_w;
  const int* crep;  // representative group of each operator class
  double dt, re;
};

__device__ inline double op_v(const SetupArgs& a, double k2, int p, int l) {
  // get_coef_v interior row (PF:3361-3362)
  const int o = p * a.Ny + l;
  return -a.t4[o] * a.dt * 0.5 / a.re + (1 + k2 * a.dt / a.re) * a.t2[o] -
         k2 * (1 + k2 * a.dt * 0.5 / a.re) * a.t0[o];
}

__device__ inline double op_w(const SetupArgs& a, double k2, int p, int l) {
  // get_coef_omegay interior row (PF:3444); at k^2 = 0 this is get_coef_u0 (PF:3502)
  const int o = p * a.Ny + l;
  return -a.t2[o] * a.dt * 0.5 / a.re + (1 + k2 * a.dt * 0.5 / a.re) * a.t0[o];
}

// grid: (operator classes, 4) ; blockIdx.y = eq*2 + parity (eq 0 = v, 1 = omega_y).
// A class is the set of groups whose k^2 is bitwise equal; it is inverted once,
// at its first group's k^2.
__global__ __launch_bounds__(256) void k_setup(SetupArgs a) {
  extern __shared__ double sm[];
  __shared__ int piv[160];
  __shared__ double colk[160];
  const int cls = blockIdx.x;
  const int g = a.crep[cls];
  const int eq = blockIdx.y >> 1, par = blockIdx.y & 1;
  const int kx = g % a.Mx, kz = g / a.Mx;
  const double k2 = a.al[kx] * a.al[kx] + a.be[kz] * a.be[kz];
  const int n = par ? a.no : a.ne;
  const int nP = n + (n & 1);  // even width: 16-byte aligned row pairs
  const int neP = a.ne + (a.ne & 1);
  if (eq == 0 && !a.inv) return;
  const long orow = eq ? a.row_w : a.row;
  double* out = (eq ? a.inv_w + (long)cls * a.stride_w : a.inv + (long)cls * a.stride) + par * neP;
  if (eq == 0 && g == 0) {  // k^2 = 0 has no v system (PF:184, 247)
    for (int idx = threadIdx.x; idx < a.ne * nP; idx += blockDim.x)
      out[(long)(idx / nP) * orow + idx % nP] = 0.0;
    return;
  }
  double* A = sm;  // n x n row-major
  for (int idx = threadIdx.x; idx < n * n; idx += blockDim.x) {
    const int i = idx / n, j = idx - i * n;
    const int l = 2 * j + par;
    double val;
    if (eq == 0) {
      if (i == 0) val = 1.0;
      else if (i == 1) val = (double)l * (double)l;
      else val = op_v(a, k2, i, l);                 // point p = i (rows 2..)
    } else {
      if (i == 0) val = 1.0;
      else val = op_w(a, k2, i, l);                 // point p = i (rows 1..)
    }
    A[idx] = val;
  }
  __syncthreads();
  const int lane = threadIdx.x & 63;
  for (int k = 0; k < n; ++k) {
    if (threadIdx.x < 64) {
      double best = -1.0;
      int bi = n;
      for (int i = k + lane; i < n; i += 64) {
        const double v = fabs(A[i * n + k]);
        if (v > best) { best = v; bi = i; }
      }
      for (int off = 32; off > 0; off >>= 1) {
        const double ob = __shfl_xor(best, off);
        const int oi = __shfl_xor(bi, off);
        if (ob > best || (ob == best && oi < bi)) { best = ob; bi = oi; }
      }
      if (lane == 0) piv[k] = bi;
    }
    __syncthreads();
    const int pr = piv[k];
    if (pr != k) {
      for (int j = threadIdx.x; j < n; j += blockDim.x) {
        const double t = A[k * n + j];
        A[k * n + j] = A[pr * n + j];
        A[pr * n + j] = t;
      }
      __syncthreads();
    }
    const double pinv = 1.0 / A[k * n + k];
    for (int i = threadIdx.x; i < n; i += blockDim.x) colk[i] = A[i * n + k];
    __syncthreads();
    for (int j = threadIdx.x; j < n; j += blockDim.x) A[k * n + j] = (j == k ? 1.0 : A[k * n + j]) * pinv;
    __syncthreads();
    for (int idx = threadIdx.x; idx < n * n; idx += blockDim.x) {
      const int i = idx / n, j = idx - i * n;
      if (i == k) continue;
      const double base = (j == k) ? 0.0 : A[idx];
      A[idx] = base - colk[i] * A[k * n + j];
    }
    __syncthreads();
  }
  // undo the row interchanges as column interchanges, last first
  for (int k = n - 1; k >= 0; --k) {
    const int pr = piv[k];
    if (pr != k) {
      for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const double t = A[i * n + k];
        A[i * n + k] = A[i * n + pr];
        A[i * n + pr] = t;
      }
    }
    __syncthreads();
  }
  // transposed store: row j, entry i = Ainv[i][j]; zero padding for i >= n and j >= n
  for (int idx = threadIdx.x; idx < a.ne * nP; idx += blockDim.x) {
    const int j = idx / nP, i = idx - j * nP;
    out[(long)j * orow + i] = (i < n && j < n) ? A[i * n + j] : 0.0;
  }
}

hipError_t launch_setup_inverses(Ctx& c) {
  const Dims& d = c.d;
  SetupArgs a{};
  a.t0 = c.t0;
  a.t2 = c.t2;
  a.t4 = c.t4;
  a.al = c.alpha;
  a.be = c.beta;
  a.inv = c.inv;
  a.inv_w = const_cast<double*>(c.inv_w);
  a.Mx = d.Mx;
  a.N = d.N;
  a.Ny = d.Ny;
  a.ne = d.ne;
  a.no = d.no;
  a.stride = d.inv_stride;
  a.row = d.inv_row;
  a.stride_w = c.stride_w;
  a.row_w = c.row_w;
  a.crep = c.crep;
  a.dt = c.prm.dt;
  a.re = c.prm.re;
  size_t shm = sizeof(double) * (size_t)d.ne * d.ne;
  if (shm > 65536) {
    hipError_t e = hipFuncSetAttribute((const void*)k_setup, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(k_setup, dim3(d.nclass, 4), dim3(256), shm, c.stream, a);
  return hipGetLastError();
}

// ------------------------------------------------------------------- solve

struct SolveArgs {
  const double2 *rvE, *rvO;        // v right-hand sides, [row][column] per parity
  const double2 *roE, *roO;        // omega_y right-hand sides, [row][column] per parity
  const double* inv;
  const double* inv_w;
  double2 *vst, *oy;  // v by group (record [l][side], see KinArgs), omega_y
  double2 *au0, *w0;
  const double2 *c1n, *c1p, *c3n, *c3p;  // mean Lamb point values, n and n-1
  const double *t0, *t2;
  int Mx, Mz, N, Ny, ne, no;
  long stride, row, stride_w, row_w, ncol;
  const int *bmat, *bg0, *bg1;  // per block: operator class, first and second group (-1: none)
  double dt, re;
};

// Block -> solve block in XCD-contiguous order: every XCD takes a contiguous
// run of blocks, so the neighbouring kx columns whose 16-byte values share a
// cache line are read and written through the same L2.
__device__ __forceinline__ int xcd_group(int b, int nb) { return (int)xcd_order(b, nb); }

// 16-byte load of inverse data that is read once per step: marked non-temporal
// so the 4.9 GB stream does not evict the right-hand sides and fields from L2.
__device__ __forceinline__ double2 stream_load(const double* p) {
  typedef double nt2 __attribute__((ext_vector_type(2)));
  const nt2 t = __builtin_nontemporal_load(reinterpret_cast<const nt2*>(p));
  return make_double2(t.x, t.y);
}

// One block per (operator class, up to two groups).  A group (kx, |kz|) holds
// the modes m0 = (kz, kx) and m1 = (Mz - kz, kx); groups with the same k^2
// share the operator, so the block streams the class's half-system inverses
// once, multiplies each by the 4 real right-hand-side vectors (Re, Im of both
// modes) of each of its groups, and writes v^{n+1} and omega_y^{n+1} (PF:242-394).  The block holding group 0 is
// the mean mode (PF:401-474): U and W with the omega_y-type operator at k^2 = 0.
// Matrix columns per load batch in the streaming loop of k_solve; two batches
// alternate, so the next batch is in flight while the current one is used.
// Measured at 256x193x256: 6 (12 loads in flight per lane, 2 waves per SIMD)
// beats 4 (8 loads, 3 waves), 5 and 8.
constexpr int kSolveSU = 6;

__global__ __launch_bounds__(512) void k_solve(SolveArgs a) {
  extern __shared__ double rb[];  // [slot][Ny][4 vec], slot = group * neq + eq
  constexpr int SU = kSolveSU, neq = 2;
  const int b = xcd_group(blockIdx.x, gridDim.x);
  const int Ny = a.Ny, N = a.N, ne = a.ne, no = a.no;
  const int mat = a.bmat[b];
  const int gs0 = a.bg0[b], gs1 = a.bg1[b];
  const int ngr = gs1 >= 0 ? 2 : 1;
  const bool mean = (gs0 == 0);
  const double c = a.dt * 0.5 / a.re;

  // ---- this thread's task: one row pair (2i, 2i+1) of one half system of one
  // equation (the launch has at least as many threads as tasks).  Its first SU
  // matrix columns are requested before the right-hand-side gather, so the
  // gather's latency overlaps the start of the stream.
  const int neP = ne + (ne & 1), noP = no + (no & 1);
  const int pe = neP / 2, po = noP / 2;  // row pairs per half system
  const int ntask = (mean ? 1 : neq) * (pe + po);
  const int t = threadIdx.x;
  const bool active = t < ntask;
  const int eq = mean ? 1 : t / (pe + po);
  const int rr = mean ? t : t - eq * (pe + po);
  const bool odd = rr >= pe;
  const int i2 = 2 * (odd ? rr - pe : rr);
  const int n = odd ? no : ne;
  const long nP = eq ? a.row_w : a.row;
  const double* M = (eq ? a.inv_w + (long)mat * a.stride_w : a.inv + (long)mat * a.stride) + (odd ? neP : 0) + i2;
  double2 ma[SU], mb[SU];
#pragma unroll
  for (int u = 0; u < SU; ++u) ma[u] = (active && u < n) ? stream_load(M + (long)u * nP) : make_double2(0, 0);

  // ---- right-hand sides, parity-folded (rows of the half systems)
  if (!mean) {
    for (int gi = 0; gi < ngr; ++gi) {
      const int g = gi ? gs1 : gs0;
      const int kx = g % a.Mx, kzab = g / a.Mx;
      const long col0 = (long)kzab * a.Mx + kx, col1 = (long)(kzab ? a.Mz - kzab : 0) * a.Mx + kx;
      for (int idx = threadIdx.x; idx < neq * Ny; idx += blockDim.x) {
        const int eq = idx / Ny, row = idx - eq * Ny;
        // row < ne: even system row; else odd system row (row - ne)
        const bool odd = row >= ne;
        const int i = odd ? row - ne : row;
        const int nbc = eq ? 1 : 2;
        double2 x0 = make_double2(0, 0), x1 = make_double2(0, 0);
        if (i >= nbc) {
          const int r = i - nbc;
          const double2* src = eq ? (odd ? a.roO : a.roE) : (odd ? a.rvO : a.rvE);
          x0 = src[(long)r * a.ncol + col0];
          if (kzab > 0) x1 = src[(long)r * a.ncol + col1];
        }
        double* dst = rb + ((gi * neq + eq) * Ny + row) * 4;
        dst[0] = x0.x;
        dst[1] = x0.y;
        dst[2] = x1.x;
        dst[3] = x1.y;
      }
    }
  } else {
    // mean mode: U (vectors 0,1) and W (vectors 2,3) with the omega_y-type
    // operator at k^2 = 0; forcing -dt/2 (3 L^n - L^{n-1}) (PF:403-404, 441-442)
    for (int row = threadIdx.x; row < Ny; row += blockDim.x) {
      const bool odd = row >= ne;
      const int i = odd ? row - ne : row;
      double acc[4] = {0, 0, 0, 0};
      if (i >= 1) {
        const int p = i, q = N - p;
        for (int l = odd ? 1 : 0; l <= N; l += 2) {
          const double t = a.t0[p * Ny + l] + c * a.t2[p * Ny + l];
          const double2 U = a.au0[l], W = a.w0[l];
          acc[0] += t * U.x; acc[1] += t * U.y; acc[2] += t * W.x; acc[3] += t * W.y;
        }
        const double2 f1p = a.c1n[p], f1q = a.c1n[q], g1p = a.c1p[p], g1q = a.c1p[q];
        const double2 f3p = a.c3n[p], f3q = a.c3n[q], g3p = a.c3p[p], g3q = a.c3p[q];
        const double hd = -1.0 * a.dt / 2.0;
        const double2 Fp = make_double2(hd * (3.0 * f1p.x - g1p.x), hd * (3.0 * f1p.y - g1p.y));
        const double2 Fq = make_double2(hd * (3.0 * f1q.x - g1q.x), hd * (3.0 * f1q.y - g1q.y));
        const double2 Gp = make_double2(hd * (3.0 * f3p.x - g3p.x), hd * (3.0 * f3p.y - g3p.y));
        const double2 Gq = make_double2(hd * (3.0 * f3q.x - g3q.x), hd * (3.0 * f3q.y - g3q.y));
        const double s = odd ? -1.0 : 1.0;
        if (p == q) {
          acc[0] += Fp.x; acc[1] += Fp.y; acc[2] += Gp.x; acc[3] += Gp.y;
        } else {
          acc[0] += 0.5 * (Fp.x + s * Fq.x); acc[1] += 0.5 * (Fp.y + s * Fq.y);
          acc[2] += 0.5 * (Gp.x + s * Gq.x); acc[3] += 0.5 * (Gp.y + s * Gq.y);
        }
      }
      for (int q4 = 0; q4 < 4; ++q4) rb[row * 4 + q4] = acc[q4];  // slot 0
    }
  }
  __syncthreads();
  // ---- dense half-system inverses x = Einv be, Oinv bo: 16-byte matrix loads,
  // accumulating the vectors of every group of the block.
  if (active) {
    const int ns = mean ? 1 : ngr;  // vector sets (slots) for this equation
    const double* rhs0 = rb + ((mean ? 0 : eq) * Ny + (odd ? ne : 0)) * 4;
    const double* rhs1 = rb + ((neq + eq) * Ny + (odd ? ne : 0)) * 4;
    double x[2][8] = {};
    // The right-hand sides are the same for every lane (LDS broadcasts); a
    // scheduling barrier per column keeps their reads next to their use, so
    // they hold registers for one column only and the load depth, not the
    // right-hand sides, fills the registers.
    auto column = [&](const double2 m, int jj) {
      __builtin_amdgcn_sched_barrier(0);
      const double* r0 = rhs0 + jj * 4;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        x[0][q] = fma(m.x, r0[q], x[0][q]);
        x[0][4 + q] = fma(m.y, r0[q], x[0][4 + q]);
      }
      if (ns > 1) {
        const double* r1 = rhs1 + jj * 4;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          x[1][q] = fma(m.x, r1[q], x[1][q]);
          x[1][4 + q] = fma(m.y, r1[q], x[1][4 + q]);
        }
      }
    };
    // batches [j, j + SU) alternate between ma and mb; the first was requested
    // before the gather.  The next batch is always requested (its columns
    // clamped to n - 1), so the number of loads in flight is fixed and the
    // current batch waits for its own loads only.
    int j = 0;
    if (n < SU) {
#pragma unroll
      for (int u = 0; u < SU; ++u)
        if (u < n) column(ma[u], u);
      j = n;
    } else {
      while (true) {
#pragma unroll
        for (int u = 0; u < SU; ++u) mb[u] = stream_load(M + (long)min(j + SU + u, n - 1) * nP);
#pragma unroll
        for (int u = 0; u < SU; ++u) column(ma[u], j + u);
        j += SU;
        if (j + SU > n) break;
#pragma unroll
        for (int u = 0; u < SU; ++u) ma[u] = stream_load(M + (long)min(j + SU + u, n - 1) * nP);
#pragma unroll
        for (int u = 0; u < SU; ++u) column(mb[u], j + u);
        j += SU;
        if (j + SU > n) break;
      }
    }
    for (; j < n; ++j) {
      const double2 m = stream_load(M + (long)j * nP);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const double r = rhs0[j * 4 + q];
        x[0][q] = fma(m.x, r, x[0][q]);
        x[0][4 + q] = fma(m.y, r, x[0][4 + q]);
        if (ns > 1) {
          const double r1 = rhs1[j * 4 + q];
          x[1][q] = fma(m.x, r1, x[1][q]);
          x[1][4 + q] = fma(m.y, r1, x[1][4 + q]);
        }
      }
    }
    for (int gi = 0; gi < ns; ++gi) {
      const int g = gi ? gs1 : gs0;
      const int kx = g % a.Mx, kzab = g / a.Mx;
      const long col0 = (long)kzab * a.Mx + kx, col1 = (long)(kzab ? a.Mz - kzab : 0) * a.Mx + kx;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int i = i2 + h;
        if (i >= n) break;
        const int l = 2 * i + (odd ? 1 : 0);
        const double* xx = x[gi];
        if (mean) {
          a.au0[l] = make_double2(xx[4 * h + 0], xx[4 * h + 1]);
          a.w0[l] = make_double2(xx[4 * h + 2], xx[4 * h + 3]);
        } else if (eq == 0) {
          // v: the group's record is written by this block alone, in full
          // lines (scattered 16-byte column stores cost a third of the solve)
          double2* rec = a.vst + (long)g * Ny * 2;
          rec[2 * l] = make_double2(xx[4 * h + 0], xx[4 * h + 1]);
          if (kzab > 0) rec[2 * l + 1] = make_double2(xx[4 * h + 2], xx[4 * h + 3]);
        } else {
          a.oy[(long)l * a.ncol + col0] = make_double2(xx[4 * h + 0], xx[4 * h + 1]);
          if (kzab > 0) a.oy[(long)l * a.ncol + col1] = make_double2(xx[4 * h + 2], xx[4 * h + 3]);
        }
      }
    }
  }
}

// v from the solve's per-group records (record g = |kz| Mx + kx holds
// [l][side], side 0 for kz = |kz|, 1 for kz = Mz - |kz|) into the field layout
// [l][kz][kx].  Block = one |kz| and VL degrees: it reads the 256-byte record
// segments of its Mx groups whole and writes Mx-long rows of both kz.  The
// mean column and the span Nyquist row are not written.
constexpr int kVL = 8;

__global__ __launch_bounds__(256) void k_vtranspose(const double2* __restrict__ vst, double2* __restrict__ v,
                                                    int Mx, int Mz, int Ny, long ncol) {
  extern __shared__ double2 tile[];  // [VL][2][Mx]
  const int kzab = blockIdx.x, l0 = blockIdx.y * kVL;
  const int nl = min(kVL, Ny - l0);
  const int per = 2 * kVL;  // double2 per record segment
  for (int i = threadIdx.x; i < Mx * per; i += blockDim.x) {
    const int kx = i / per, e = i - kx * per;
    const int l = e >> 1, side = e & 1;
    if (l < nl) tile[(l * 2 + side) * Mx + kx] = vst[((long)(kzab * Mx + kx) * Ny + l0 + l) * 2 + side];
  }
  __syncthreads();
  const int nside = kzab ? 2 : 1;
  for (int i = threadIdx.x; i < nl * nside * Mx; i += blockDim.x) {
    const int kx = i % Mx, ls = i / Mx;
    const int l = ls / nside, side = ls - l * nside;
    const int kz = side ? Mz - kzab : kzab;
    if (kz == 0 && kx == 0) continue;  // the mean column: U, W are solved instead
    v[(long)(l0 + l) * ncol + (long)kz * Mx + kx] = tile[(l * 2 + side) * Mx + kx];
  }
}

static SolveArgs solve_args(const Ctx& c) {
  const Dims& d = c.d;
  SolveArgs a{};
  a.rvE = c.rvE;
  a.rvO = c.rvO;
  a.roE = c.roE;
  a.roO = c.roO;
  a.inv = c.inv;
  a.inv_w = c.inv_w;
  a.vst = c.vst;
  a.oy = c.oy;
  a.au0 = c.au0;
  a.w0 = c.w0;
  a.c1n = c.cl1[c.hcur];
  a.c1p = c.cl1[1 - c.hcur];
  a.c3n = c.cl3[c.hcur];
  a.c3p = c.cl3[1 - c.hcur];
  a.t0 = c.t0;
  a.t2 = c.t2;
  a.Mx = d.Mx;
  a.Mz = d.Mz;
  a.N = d.N;
  a.Ny = d.Ny;
  a.ne = d.ne;
  a.no = d.no;
  a.stride = d.inv_stride;
  a.row = d.inv_row;
  a.stride_w = c.stride_w;
  a.row_w = c.row_w;
  a.bmat = c.bmat;
  a.bg0 = c.bg0;
  a.bg1 = c.bg1;
  a.ncol = d.ncol;
  a.dt = c.prm.dt;
  a.re = c.prm.re;
  return a;
}

// LDS bytes (two groups per block, two equations each) and threads of the
// solve blocks: one thread per task, a row pair of a half system.
static void solve_shape(const Ctx& c, size_t* shm, int* threads) {
  const Dims& d = c.d;
  *shm = sizeof(double) * 4ull * d.Ny * 2 * 2;
  const int pairs = (d.ne + (d.ne & 1)) / 2 + (d.no + (d.no & 1)) / 2;
  *threads = (2 * pairs + 63) / 64 * 64;
}

static hipError_t allow_shm(const void* kernel, size_t shm) {
  if (shm <= 65536) return hipSuccess;
  return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
}

hipError_t launch_vtranspose(Ctx& c) {
  const Dims& d = c.d;
  const size_t tshm = sizeof(double2) * 2ull * kVL * d.Mx;
  if (tshm > 65536) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_vtranspose, dim3(d.Mz / 2, (d.Ny + kVL - 1) / kVL), dim3(256), tshm, c.stream,
                     (const double2*)c.vst, c.v, d.Mx, d.Mz, d.Ny, d.ncol);
  return hipGetLastError();
}

hipError_t launch_solve(Ctx& c) {
  const SolveArgs a = solve_args(c);
  size_t shm;
  int threads;
  solve_shape(c, &shm, &threads);
  if (threads > 512) return hipErrorInvalidValue;
  hipError_t e = allow_shm((const void*)k_solve, shm);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_solve, dim3(c.d.nblocks), dim3(threads), shm, c.stream, a);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  return launch_vtranspose(c);
}

}  // namespace chf
