// Unpadded physical fields and plane statistics, computed where the fields
// live.
//
//   physical: transform(1, .) (PF:948-961 with fourtrx_zcomp(+1), PF:774-860):
//             Chebyshev coefficients -> values at y_k = cos(pi k/N), span
//             modes -> nny points (Nyquist slot zeroed), streamwise modes ->
//             nnx real points (Hermitian fill, Re of the kx = 0 entry), i.e.
//             the reference's real*8 (0:nnx-1, 0:nny-1, 0:N) == [Ny][nny][nnx].
//   plane statistics: the plane means, covariances and extrema of the
//             physical u, v, w that statistics (PF:2816-3020) reduces.
//
// A streamwise line of nnx = 2 M real values comes from one complex transform
// of M points: with X the line's modes (X_M = 0),
//   z_m = (X_m + conj X_(M-m)) + i w (X_m - conj X_(M-m)),  w = e^(2 pi i m / nnx),
// and its transform holds x_(2j) + i x_(2j+1).  Bound: HBM (a line is read and
// written once); the LDS kernel of fft.hip, which transforms all nnx complex
// points, serves the lengths without a split.  256x193x256: three physical
// fields 0.81 -> 0.36 ms (with the span step's register FFT), the statistics
// 1.11 -> 0.36 ms (their planes are no longer stored and read twice); 32x33x32
// 0.077 -> 0.054 and 0.044 ms, launches.
#include <algorithm>

#include "chf_internal.h"
#include "fftreg.h"

namespace chf {

struct LineArgs {
  const double2* in[3];  // [Ny][Mz][Mx], span points
  double* out;           // [Ny][Mz][nnx], or the statistics' partial sums [Ny][splits][12]
  const double2* tw;     // e^(-2 pi i m / nnx)
  int Mz, splits;
  long nlines;
};

// Geometry of a block: NG lines, G = N2 threads each.
template <int N1, int N2>
struct LineGeo {
  static_assert(N1 <= N2, "thread t < N2 of a group holds N1 values");
  static constexpr int M = N1 * N2, G = N2, NG = 256 / G, NT = NG * G, TILE = N1 * (N2 + 1);
  static constexpr size_t shm = sizeof(double2) * (2 * M + (size_t)NG * TILE);
};

// A block's lines are consecutive in memory: its NT threads read them as one
// run, N1 values each (0 past the last line).
template <int N1, int N2>
__device__ __forceinline__ void lines_load(const double2* f, int nvalid, double2 (&r)[N1]) {
  using Ge = LineGeo<N1, N2>;
#pragma unroll
  for (int i = 0; i < N1; ++i) {
    const int idx = i * Ge::NT + threadIdx.x;
    r[i] = (int)threadIdx.x < Ge::NT && idx < nvalid * Ge::M ? f[idx] : make_double2(0, 0);
  }
}

// The values of a line by the G threads of its group g: thread t holds z[k1] =
// (x_2j, x_(2j+1)) at j = k1 N2 + t.  All threads of the block call it together
// with what lines_load gave them (threads past NT idle); `tw` is
// e^(-2 pi i m / nnx), m < nnx, and `tiles` the NG line tiles, in LDS.
template <int N1, int N2>
__device__ __forceinline__ void lines_c2r(const double2 (&r)[N1], const double2* tw, double2* tiles, int g, int t,
                                          double2 (&z)[N1]) {
  using Ge = LineGeo<N1, N2>;
  double2* buf = tiles + min(g, Ge::NG - 1) * Ge::TILE;
  __syncthreads();  // the tiles are free (and the table is written)
#pragma unroll
  for (int i = 0; i < N1; ++i) {
    const int idx = i * Ge::NT + threadIdx.x, ln = idx / Ge::M;
    if ((int)threadIdx.x < Ge::NT) tiles[ln * Ge::TILE + idx - ln * Ge::M] = r[i];
  }
  __syncthreads();
  const bool a_thread = g < Ge::NG && t < N1;
  double2 x[N2];
  if (a_thread) {
#pragma unroll
    for (int n2 = 0; n2 < N2; ++n2) {
      const int m = n2 * N1 + t;
      double2 X = buf[m], Y = buf[m ? Ge::M - m : 0];
      if (m == 0) {
        X.y = 0.0;                  // Re of the kx = 0 entry (PF:1116-1118)
        Y = make_double2(0, 0);     // X_M, the Nyquist mode
      }
      const double2 w = tw[m];
      const double2 e = make_double2(X.x + Y.x, X.y - Y.y), o = make_double2(X.x - Y.x, X.y + Y.y);
      const double2 ow = make_double2(o.x * w.x + o.y * w.y, o.y * w.x - o.x * w.y);  // o conj(w)
      x[n2] = make_double2(e.x - ow.y, e.y + ow.x);
    }
  }
  __syncthreads();
  if (a_thread) {
    Dft<N2, +1, double2>::run(x);
#pragma unroll
    for (int k2 = 0; k2 < N2; ++k2) {
      double2 w = tw[2 * t * k2];
      w.y = -w.y;
      buf[t * (N2 + 1) + k2] = (k2 == 0) ? x[0] : cmulv(x[k2], w);
    }
  }
  __syncthreads();
  if (g < Ge::NG) fft_stepB<N1, N2, +1>(z, buf, t);
}

template <int N1, int N2>
__global__ __launch_bounds__(256) void k_line_c2r(LineArgs a) {  // NT threads
  using Ge = LineGeo<N1, N2>;
  extern __shared__ __align__(16) unsigned char smraw[];
  double2* tw = reinterpret_cast<double2*>(smraw);
  const int g = threadIdx.x / Ge::G, t = threadIdx.x - g * Ge::G;
  const long line0 = (long)blockIdx.x * Ge::NG;
  double2 r[N1], z[N1];
  lines_load<N1, N2>(a.in[0] + line0 * Ge::M, (int)min((long)Ge::NG, a.nlines - line0), r);
  for (int i = threadIdx.x; i < 2 * Ge::M; i += Ge::NT) tw[i] = a.tw[i];
  lines_c2r<N1, N2>(r, tw, tw + 2 * Ge::M, g, t, z);
  if (line0 + g < a.nlines) {
    double2* o = reinterpret_cast<double2*>(a.out) + (line0 + g) * Ge::M;
#pragma unroll
    for (int k1 = 0; k1 < N1; ++k1) o[k1 * N2 + t] = z[k1];
  }
}

// Sum over the block of one value per thread (every thread gets it).
__device__ __forceinline__ double block_sum(double v, double* red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  v = 0.0;
  for (int w = 0; w < (int)(blockDim.x >> 6); ++w) v += red[w];
  return v;
}

constexpr int kStatsThreads = 256;

// Plane statistics without storing the physical fields: a block transforms
// some of a plane's lines of u, v, w, keeps them in registers and sums the
// products about the plane means and the extrema.  The mean of a field over the
// plane is the mean over the span of its lines' (real) kx = 0 modes, and NaN where a
// value of the plane is not finite, as a sum over the values is: the squares' sum is
// NaN where a value is (no term of it is negative), and an infinity is the largest
// value (a test of every value costs 2%).
template <int N1, int N2>
__global__ __launch_bounds__(kStatsThreads, 2) void k_line_stats(LineArgs a) {
  using Ge = LineGeo<N1, N2>;
  extern __shared__ __align__(16) unsigned char smraw[];
  __shared__ double red[8];
  double2* tw = reinterpret_cast<double2*>(smraw);
  const int g = threadIdx.x / Ge::G, t = threadIdx.x - g * Ge::G;
  for (int i = threadIdx.x; i < 2 * Ge::M; i += blockDim.x) tw[i] = a.tw[i];
  const int k = blockIdx.x;
  const long plane = (long)k * a.Mz;
  double mean[3];
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    double v = 0.0;
    for (int l = threadIdx.x; l < a.Mz; l += blockDim.x) v += a.in[q][(plane + l) * Ge::M].x;
    mean[q] = block_sum(v, red) / (double)a.Mz;
  }
  double acc[6] = {}, big[3] = {};
  double2 r[N1];
  for (int l0 = blockIdx.y * Ge::NG; l0 < a.Mz; l0 += a.splits * Ge::NG) {
    const int nvalid = min(Ge::NG, a.Mz - l0);
    const bool valid = g < nvalid;
    double2 z[3][N1];
    lines_load<N1, N2>(a.in[0] + (plane + l0) * Ge::M, nvalid, r);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      lines_c2r<N1, N2>(r, tw, tw + 2 * Ge::M, g, t, z[q]);
      if (q < 2) lines_load<N1, N2>(a.in[q + 1] + (plane + l0) * Ge::M, nvalid, r);
    }
    if (valid) {
#pragma unroll
      for (int k1 = 0; k1 < N1; ++k1)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const double u = h ? z[0][k1].y : z[0][k1].x, v = h ? z[1][k1].y : z[1][k1].x,
                       w = h ? z[2][k1].y : z[2][k1].x;
          const double du = u - mean[0], dv = v - mean[1], dw = w - mean[2];
          acc[0] += du * du;
          acc[1] += dv * dv;
          acc[2] += dw * dw;
          acc[3] += du * dv;
          acc[4] += du * dw;
          acc[5] += dv * dw;
          big[0] = fmax(big[0], fabs(u));
          big[1] = fmax(big[1], fabs(v));
          big[2] = fmax(big[2], fabs(w));
        }
    }
  }
  double* p = a.out + ((long)k * a.splits + blockIdx.y) * 12;
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    const double v = block_sum(acc[i], red);
    if (threadIdx.x == 0) p[3 + i] = v;
    if (i < 3 && v != v) mean[i] = v;
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    double v = big[i];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int w = 1; w < (int)(blockDim.x >> 6); ++w) v = fmax(v, red[w]);
      p[9 + i] = v;
      p[i] = isinf(v) ? v - v : mean[i];
    }
  }
}

// The splits' partial results [Ny][splits][12] to out [12][Ny]; no branch in a loop,
// so that its loads are in flight together.
__global__ __launch_bounds__(256) void k_stats_final(const double* __restrict__ part, int splits, int Ny, double coef,
                                                     double* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 12 * Ny) return;
  const int q = i / Ny, k = i - q * Ny;
  const double* p = part + (long)k * splits * 12 + q;
  double v = p[0];
#pragma unroll 8
  for (int s = 1; s < splits; ++s) {
    const double x = p[12 * s];
    v = q < 3 ? (x == x ? v : x) : q < 9 ? v + x : fmax(v, x);  // the same mean in every split, but for NaN
  }
  out[i] = (q >= 3 && q < 9) ? v * coef : v;
}

// One block per wall-normal point k of three physical fields [Ny][nny][nnx].
// out (12 x Ny, quantity-major): ua va wa uu vv ww uv uw vw max|u| max|v| max|w|
__global__ __launch_bounds__(256) void k_plane_stats(const double* __restrict__ u, const double* __restrict__ v,
                                                     const double* __restrict__ w, long plane, int Ny,
                                                     double* __restrict__ out) {
  __shared__ double red[6][256];
  const int k = blockIdx.x;
  const double* pu = u + (long)k * plane;
  const double* pv = v + (long)k * plane;
  const double* pw = w + (long)k * plane;
  double s[6] = {0, 0, 0, 0, 0, 0};
  for (long i = threadIdx.x; i < plane; i += blockDim.x) {
    const double a = pu[i], b = pv[i], c = pw[i];
    s[0] += a;
    s[1] += b;
    s[2] += c;
    s[3] = fmax(s[3], fabs(a));
    s[4] = fmax(s[4], fabs(b));
    s[5] = fmax(s[5], fabs(c));
  }
  for (int q = 0; q < 6; ++q) red[q][threadIdx.x] = s[q];
  __syncthreads();
  for (int h = blockDim.x / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) {
      for (int q = 0; q < 3; ++q) red[q][threadIdx.x] += red[q][threadIdx.x + h];
      for (int q = 3; q < 6; ++q) red[q][threadIdx.x] = fmax(red[q][threadIdx.x], red[q][threadIdx.x + h]);
    }
    __syncthreads();
  }
  const double coef = 1.0 / (double)plane;
  const double ma = red[0][0] * coef, mb = red[1][0] * coef, mc = red[2][0] * coef;
  const double xa = red[3][0], xb = red[4][0], xc = red[5][0];
  __syncthreads();
  double t[6] = {0, 0, 0, 0, 0, 0};
  for (long i = threadIdx.x; i < plane; i += blockDim.x) {
    const double a = pu[i] - ma, b = pv[i] - mb, c = pw[i] - mc;
    t[0] += a * a;
    t[1] += b * b;
    t[2] += c * c;
    t[3] += a * b;
    t[4] += a * c;
    t[5] += b * c;
  }
  for (int q = 0; q < 6; ++q) red[q][threadIdx.x] = t[q];
  __syncthreads();
  for (int h = blockDim.x / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h)
      for (int q = 0; q < 6; ++q) red[q][threadIdx.x] += red[q][threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[0 * Ny + k] = ma;
    out[1 * Ny + k] = mb;
    out[2 * Ny + k] = mc;
    for (int q = 0; q < 6; ++q) out[(3 + q) * Ny + k] = red[q][0] * coef;
    out[9 * Ny + k] = xa;
    out[10 * Ny + k] = xb;
    out[11 * Ny + k] = xc;
  }
}

// Calls run.operator()<N1, N2>() for the split of a line of M complex points
// (N1 <= N2: a thread keeps N1 values of each field); false without one.
template <class F>
static bool with_line_split(int M, F& run) {
  switch (M) {
    case 8: run.template operator()<2, 4>(); return true;
    case 12: run.template operator()<3, 4>(); return true;
    case 16: run.template operator()<4, 4>(); return true;
    case 18: run.template operator()<3, 6>(); return true;
    case 24: run.template operator()<4, 6>(); return true;
    case 32: run.template operator()<4, 8>(); return true;
    case 36: run.template operator()<6, 6>(); return true;
    case 48: run.template operator()<6, 8>(); return true;
    case 54: run.template operator()<6, 9>(); return true;
    case 64: run.template operator()<8, 8>(); return true;
    case 72: run.template operator()<8, 9>(); return true;
    case 96: run.template operator()<8, 12>(); return true;
    case 108: run.template operator()<9, 12>(); return true;
    case 128: run.template operator()<8, 16>(); return true;
    case 144: run.template operator()<9, 16>(); return true;
    case 192: run.template operator()<8, 24>(); return true;
    case 256: run.template operator()<16, 16>(); return true;
    default: return false;
  }
}

// Lines that a block of a split transforms at a time; 0 without a split.
struct LinesPerBlock {
  int n = 0;
  template <int N1, int N2>
  void operator()() {
    n = LineGeo<N1, N2>::NG;
  }
};

static int lines_per_block(int M) {
  LinesPerBlock lines;
  with_line_split(M, lines);
  return lines.n;
}

struct RunC2r {
  Ctx& c;
  const LineArgs& a;
  hipError_t e = hipSuccess;
  template <int N1, int N2>
  void operator()() {
    using Ge = LineGeo<N1, N2>;
    static_assert(Ge::shm <= 160 * 1024, "line tiles exceed the LDS");
    if (Ge::shm > 65536)
      e = hipFuncSetAttribute((const void*)k_line_c2r<N1, N2>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)Ge::shm);
    if (e != hipSuccess) return;
    hipLaunchKernelGGL((k_line_c2r<N1, N2>), dim3((unsigned)((a.nlines + Ge::NG - 1) / Ge::NG)),
                       dim3(Ge::NG * Ge::G), Ge::shm, c.stream, a);
    e = hipGetLastError();
  }
};

struct RunStats {
  Ctx& c;
  const LineArgs& a;
  hipError_t e = hipSuccess;
  template <int N1, int N2>
  void operator()() {
    using Ge = LineGeo<N1, N2>;
    if (Ge::shm + 64 > 65536)
      e = hipFuncSetAttribute((const void*)k_line_stats<N1, N2>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)Ge::shm);
    if (e != hipSuccess) return;
    hipLaunchKernelGGL((k_line_stats<N1, N2>), dim3(c.d.Ny, a.splits), dim3(kStatsThreads), Ge::shm, c.stream, a);
    e = hipGetLastError();
  }
};

hipError_t launch_stream_c2r_unpadded(Ctx& c, const double2* in, double* out) {
  LineArgs a{};
  a.in[0] = in;
  a.out = out;
  a.tw = c.twxu;
  a.nlines = (long)c.d.Ny * c.d.Mz;
  RunC2r run{c, a};
  if (with_line_split(c.d.Mx, run)) return run.e;
  return launch_stream_c2r_lds(c, in, out);
}

hipError_t launch_physical(Ctx& c, const double2* field, double2* work, double* out) {
  // Chebyshev synthesis at the N+1 points into the complex work plane (every
  // point of every column is written, so the work needs no clearing)
  const double2* in1[1] = {field};
  double2* o1[1] = {work};
  hipError_t e = launch_synth_points(c, in1, o1, 1);
  if (e != hipSuccess) return e;
  e = launch_span_inverse_unpadded(c, o1, 1);
  if (e != hipSuccess) return e;
  return launch_stream_c2r_unpadded(c, work, out);
}

// Blocks per plane of the statistics: enough for six on every CU, each with at
// least 16 lines and one group of lines (more of them would sum the plane means
// for nothing: 16x33x512, 64 lines a group, 76 us with 32 blocks, 63 with 8).
int stats_splits(const Ctx& c) {
  const int ng = lines_per_block(c.d.Mx);
  return ng ? std::max(1, std::min({1536 / c.d.Ny, c.d.Mz / 16, (c.d.Mz + ng - 1) / ng})) : 1;
}

bool stats_in_lines(const Ctx& c) { return lines_per_block(c.d.Mx) > 0; }

hipError_t launch_statistics(Ctx& c, const double2* const* fields, double2* const* work, double* const* phys,
                             double* part, double* out) {
  const Dims& d = c.d;
  hipError_t e = launch_synth_points(c, fields, work, 3);
  if (e != hipSuccess) return e;
  e = launch_span_inverse_unpadded(c, work, 3);
  if (e != hipSuccess) return e;
  if (!stats_in_lines(c)) {
    for (int q = 0; q < 3 && e == hipSuccess; ++q) e = launch_stream_c2r_unpadded(c, work[q], phys[q]);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_plane_stats, dim3(d.Ny), dim3(256), 0, c.stream, phys[0], phys[1], phys[2],
                       (long)d.Mz * 2 * d.Mx, d.Ny, out);
    return hipGetLastError();
  }
  LineArgs a{};
  for (int q = 0; q < 3; ++q) a.in[q] = work[q];
  a.out = part;
  a.tw = c.twxu;
  a.Mz = d.Mz;
  a.splits = stats_splits(c);
  RunStats run{c, a};
  with_line_split(d.Mx, run);
  if (run.e != hipSuccess) return run.e;
  hipLaunchKernelGGL(k_stats_final, dim3((12 * d.Ny + 255) / 256), dim3(256), 0, c.stream, part, a.splits, d.Ny,
                     1.0 / ((double)d.Mz * 2 * d.Mx), out);
  return hipGetLastError();
}

}  // namespace chf
