// loma_yops.hip -- dispatch of the y-direction kernels over the chunk size M
// (rows of a y-column per lane); the kernels are in loma_yops_impl.h and are
// instantiated one M per translation unit (loma_yops_m<M>.hip).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "loma_kernels.h"

namespace loma {

template <int M>
int launch_dy_m(int, const YTab&, const double*, double*, int, hipStream_t);
template <int M>
int launch_lapvdvhom_m(const YTab&, const double*, int, const double*, double*, double*,
                       const double*, int, int, hipStream_t);
template <int M>
int launch_helm_bc_m(const YTab&, const double*, int, double*, double*, int, hipStream_t);
template <int M>
int launch_inty8_m(const YTab&, const double*, double*, hipStream_t);
template <int M>
int launch_visc_m(const YTab&, const double*, const double*, int, double*, double*, double*,
                  double*, double*, double*, const double*, double, double, double, int,
                  hipStream_t);
template <int M>
int launch_phase_m(int, bool, const PhaseArgs&, hipStream_t);
template <int M>
int launch_ic_m(const IcArgs&, hipStream_t);
template <int M>
int launch_thickness_m(bool, const PhaseArgs&, const double*, double, int, hipStream_t);
template <int M>
int launch_stats_m(bool, int, const StatsArgs&, hipStream_t);
template <int M>
int launch_phase_batch_m(int, bool, const PhaseArgs*, const int*, int, int, hipStream_t);

RkCoef rk_coefficients() {
  RkCoef r;
  const double p0 = 5.0 / 66.0, p1 = -1.0;
  const double g[3] = {8.0 / 15.0, 5.0 / 12.0, 3.0 / 4.0};
  const double xi[3] = {0.0, -17.0 / 60.0, -5.0 / 12.0};
  const double b3 = (p1 * (g[0] * g[2] + g[1] * g[2] + xi[1] * g[2] + g[0] * xi[2]) -
                     g[0] * g[1] * g[2] - g[0] * g[1] * xi[2]) /
                    (p1 - g[0] * g[1]);
  for (int q = 0; q < 3; ++q) { r.gama[q] = g[q]; r.xi[q] = xi[q]; }
  r.beta[0] = g[0] - p0; r.beta[1] = p1; r.beta[2] = b3;
  r.alpha[0] = p0; r.alpha[1] = g[1] + xi[1] - p1; r.alpha[2] = g[2] + xi[2] - r.beta[2];
  return r;
}


#define LOMA_DISPATCH_M(M, ...)                 \
  switch (M) {                                  \
    case 3: { constexpr int MM = 3; return __VA_ARGS__; } \
    case 4: { constexpr int MM = 4; return __VA_ARGS__; } \
    case 5: { constexpr int MM = 5; return __VA_ARGS__; } \
    case 6: { constexpr int MM = 6; return __VA_ARGS__; } \
    case 7: { constexpr int MM = 7; return __VA_ARGS__; } \
    case 8: { constexpr int MM = 8; return __VA_ARGS__; } \
    case 9: { constexpr int MM = 9; return __VA_ARGS__; } \
    case 10: { constexpr int MM = 10; return __VA_ARGS__; } \
    case 12: { constexpr int MM = 12; return __VA_ARGS__; } \
    case 14: { constexpr int MM = 14; return __VA_ARGS__; } \
    case 16: { constexpr int MM = 16; return __VA_ARGS__; } \
    default: return (int)hipErrorInvalidValue;  \
  }

int launch_dy(int M, int order, const YTab& T, const double* u, double* du, int ncols,
              hipStream_t st) {
  if (ncols <= 0) return 0;
  LOMA_DISPATCH_M(M, launch_dy_m<MM>(order, T, u, du, ncols, st));
}
int launch_lapvdvhom(int M, const YTab& T, const double* lu, const double* phi, double* v,
                     double* dv, const double* rK, int ncols, int mode, hipStream_t st) {
  if (ncols <= 0) return 0;
  LOMA_DISPATCH_M(M, launch_lapvdvhom_m<MM>(T, lu, 5 * WAVE * MM, phi, v, dv, rK, ncols, mode,
                                            st));
}
int launch_helm_bc(int M, const YTab& T, const double* lu, double* bc, double* h, int nclass,
                   hipStream_t st) {
  if (nclass <= 0) return 0;
  LOMA_DISPATCH_M(M, launch_helm_bc_m<MM>(T, lu, 5 * WAVE * MM, bc, h, nclass, st));
}
int launch_inty8(int M, const YTab& T, const double* du, double* u, hipStream_t st) {
  LOMA_DISPATCH_M(M, launch_inty8_m<MM>(T, du, u, st));
}
int launch_visc(int M, const YTab& T, const double* lu1, const double* lu2, double* vorwk,
                double* vor, double* phi, double* v, double* dvdy,
                double* phiwk, const double* rk2, double dalbe, double dtri, double dtxi,
                int ncols, hipStream_t st) {
  if (ncols <= 0) return 0;
  LOMA_DISPATCH_M(M, launch_visc_m<MM>(T, lu1, lu2, 5 * WAVE * MM, vorwk, vor, phi, v,
                                       dvdy, phiwk, rk2, dalbe, dtri, dtxi, ncols, st));
}
int launch_phaseA(int M, bool fp32, const PhaseArgs& a, hipStream_t st) {
  if (a.nmodes <= 0) return 0;
  LOMA_DISPATCH_M(M, launch_phase_m<MM>(0, fp32, a, st));
}
int launch_phaseC(int M, bool fp32, const PhaseArgs& a, hipStream_t st) {
  if (a.nmodes <= 0) return 0;
  LOMA_DISPATCH_M(M, launch_phase_m<MM>(1, fp32, a, st));
}
int launch_phaseC2(int M, bool fp32, const PhaseArgs& a, hipStream_t st) {
  if (a.nmodes <= 0) return 0;
  LOMA_DISPATCH_M(M, launch_phase_m<MM>(2, fp32, a, st));
}
int launch_phase_batch(int M, bool fp32, int which, const PhaseArgs* args, const int* first,
                       int nrun, int nblocks, hipStream_t st) {
  if (nblocks <= 0 || nrun <= 0) return 0;
  LOMA_DISPATCH_M(M, launch_phase_batch_m<MM>(which, fp32, args, first, nrun, nblocks, st));
}
// the grids of launch_phase_m: 4 wavefronts (modes, or Helmholtz classes
// for phase C2) per 256-thread block
int phase_blocks(int which, const RunConst& rc) {
  const int n = which == 2 ? rc.nplanes * (rc.nz + 1) : rc.nplanes * rc.mz;
  return (n + 3) / 4;
}
int launch_ic(int M, const IcArgs& a, hipStream_t st) {
  LOMA_DISPATCH_M(M, launch_ic_m<MM>(a, st));
}
int launch_thickness(int M, bool fp32, const PhaseArgs& a, const double* hy, double ly,
                     int which, hipStream_t st) {
  LOMA_DISPATCH_M(M, launch_thickness_m<MM>(fp32, a, hy, ly, which, st));
}

// LU of (dt22 - s dt21), s = shifts[.] + shift, with identity end rows
// (Lapvdvhom laps.f:349-366), one thread per system.  Output per system:
// lane-major streams over 64*M rows, first lo1, lo2 (lower multipliers by
// destination row), then inv, up1, up2; zero beyond row my-1.
// The rows are a serial chain, and with a few wavefronts on the card its
// instructions are what it costs: the band rows wait in LDS and are read one
// row ahead, the three rows in flight rotate by name (no moves), the interior
// rows run without edge tests, and stores take a scalar offset.
// 92 -> 36 us for 441 systems of 129 rows and 230 -> 67 us for 7,225 of 257,
// against one that cleared its tables first and walked them with index
// divisions (64 or fewer systems a wavefront make no difference).
__global__ __launch_bounds__(64) void k_helm_factor(const double* __restrict__ dt21,
                                                    const double* __restrict__ dt22, int my,
                                                    int M, const double* __restrict__ shifts,
                                                    double shift, int nsys,
                                                    double* __restrict__ lu) {
  extern __shared__ __align__(16) double g[];  // rows of dt22, then of dt21
  for (int q0 = threadIdx.x; q0 < 5 * my; q0 += 64 * 8) {
    double c2[8], c1[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int q = min(q0 + 64 * i, 5 * my - 1);
      c2[i] = dt22[q];
      c1[i] = dt21[q];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int q = min(q0 + 64 * i, 5 * my - 1);
      g[q] = c2[i];
      g[5 * my + q] = c1[i];
    }
  }
  __syncthreads();
  const int s = blockIdx.x * 64 + threadIdx.x;
  const int stride = 5 * WAVE * M * 8;  // bytes of a system's table
  const auto out = make_rsrc(lu + (size_t)blockIdx.x * 64 * (5 * WAVE * M), 0x7fffffff);
  const int vo = threadIdx.x * stride;
  const int ubase = 2 * WAVE * M * 8;
  // The rows past my-1 are zero.  A batch of a few systems clears them with the
  // lanes along the rows, system by system (0.24 us for 64 rows of one), others
  // with each lane its own system's behind the chain (0.09 us a row, whatever
  // the systems): one visc of 17 rows, 175 of 192 to clear, 58 against 89 us.
  const int pad = WAVE * M - my, nb = min(64, nsys - (int)blockIdx.x * 64);
  const bool together = 4 * nb * ((pad + 63) / 64) < pad;
  if (together)
    for (int q = 0; q < nb; ++q)
      for (int r = my + (int)threadIdx.x; r < WAVE * M; r += 64) {
        typedef unsigned u2v __attribute__((ext_vector_type(2)));
        const int l = r / M, t = r - l * M, sys = q * stride;
#pragma unroll
        for (int e = 0; e < 3; ++e)
          __builtin_amdgcn_raw_buffer_store_b64(
              u2v{0, 0}, out, sys + ubase + stream_index(3 * M, 3 * t + e, l, 2) * 8, 0, 0);
#pragma unroll
        for (int e = 0; e < 2; ++e)
          __builtin_amdgcn_raw_buffer_store_b64(
              u2v{0, 0}, out, sys + stream_index(2 * M, 2 * t + e, l, 2) * 8, 0, 0);
      }
  if (s >= nsys) return;
  const double sh = shifts[s] + shift;
  auto put = [&](int so, double v) {
    typedef unsigned u2v __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2v, v), out, vo, so, 0);
  };
  auto put_lo = [&](int l, int t, double a, double b) {
    typedef unsigned u4v __attribute__((ext_vector_type(4)));
    typedef double d2v __attribute__((ext_vector_type(2)));
    d2v v;
    v[0] = a;
    v[1] = b;
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4v, v), out, vo,
                                           (t * WAVE + l) * 16, 0);
  };
  int l = 0, t = 0, ln = 0, tn = 1;  // lane and slot of rows k and k+1 (M >= 3)
  double l2 = 0.0;                   // row k-1's multiplier into row k+1
  const int utail = ubase + (3 * M - 1) * (WAVE * 8);
  const int tlast = (M & 1) ? M - 1 : -1;  // slot whose up2 lies behind the vectors
  auto store_row = [&](double iv, double u1, double u2, double m1, double m2) {
    // entries 3t .. 3t+2 of lane l's U stream, two to a 16-byte vector
    const int odd = t & 1, ub = ubase + ((3 * t) >> 1) * (WAVE * 16) + l * 16;
    const int in = ub + WAVE * 16 + odd * 8, tail = utail + l * 8;
    put(ub + odd * 8, iv);
    put(ub + 8 + odd * (WAVE * 16 - 8), u1);
    put(t == tlast ? tail : in, u2);
    if (ln < WAVE) put_lo(ln, tn, m1, l2);
    l2 = m2;
    const bool wrap = tn + 1 == M;
    l = ln;
    t = tn;
    tn = wrap ? 0 : tn + 1;
    ln = wrap ? ln + 1 : ln;
  };
  double n2[5], n1[5];               // the row after those in flight
  auto ahead = [&](int j) {
    const double* p = g + 5 * j;
#pragma unroll
    for (int d = 0; d < 5; ++d) {
      n2[d] = p[d];
      n1[d] = p[5 * my + d];
    }
  };
  auto interior = [&](double (&r)[5]) {
#pragma unroll
    for (int d = 0; d < 5; ++d) r[d] = n2[d] - sh * n1[d];
  };
  // eliminates column k (pivot row a) from rows b and c
  auto eliminate = [&](const double (&a)[5], double (&b)[5], double (&c)[5], double& iv,
                       double& m1, double& m2) {
    iv = 1.0 / a[2];
    m1 = b[1] * iv;
    b[2] -= m1 * a[3];
    b[3] -= m1 * a[4];
    m2 = c[0] * iv;
    c[1] -= m2 * a[3];
    c[2] -= m2 * a[4];
  };
  put_lo(0, 0, 0.0, 0.0);
  double w0[5] = {0.0, 0.0, 1.0, 0.0, 0.0}, w1[5], w2[5];
  ahead(1);
  interior(w1);
  ahead(2);
  interior(w2);
  ahead(3);
  // rows k whose incoming row k+3 is an interior one
  auto step = [&](int k, double (&a)[5], double (&b)[5], double (&c)[5]) {
    double iv, m1, m2;
    eliminate(a, b, c, iv, m1, m2);
    store_row(iv, a[3], a[4], m1, m2);
    interior(a);
    ahead(k + 4);
  };
  int k = 0;
  for (; k + 2 <= my - 5; k += 3) {
    step(k, w0, w1, w2);
    step(k + 1, w1, w2, w0);
    step(k + 2, w2, w0, w1);
  }
  // the last rows: the incoming row is an interior one, the identity (row
  // my-1) or none
  for (; k < my; ++k) {
    double iv, m1, m2;
    eliminate(w0, w1, w2, iv, m1, m2);
    store_row(iv, k + 1 < my ? w0[3] : 0.0, k + 2 < my ? w0[4] : 0.0, k + 1 < my ? m1 : 0.0,
              k + 2 < my ? m2 : 0.0);
    const int j = k + 3;
    double w3[5];
    if (j < my - 1) {
      ahead(j);
      interior(w3);
    } else {
#pragma unroll
      for (int d = 0; d < 5; ++d) w3[d] = d == 2 && j == my - 1 ? 1.0 : 0.0;
    }
#pragma unroll
    for (int d = 0; d < 5; ++d) { w0[d] = w1[d]; w1[d] = w2[d]; w2[d] = w3[d]; }
  }
  if (!together)
    for (; k < WAVE * M; ++k) store_row(0.0, 0.0, 0.0, 0.0, 0.0);
}

int launch_helm_factor(const double* dt21, const double* dt22, int my, int M,
                       const double* shifts, double shift, int nsys, double* lu,
                       hipStream_t st) {
  if (nsys <= 0) return 0;
  hipLaunchKernelGGL(k_helm_factor, dim3((nsys + 63) / 64), dim3(64), 10 * (size_t)my * 8, st, dt21, dt22,
                     my, M, shifts, shift, nsys, lu);
  return (int)hipGetLastError();
}

// end of step: time += dt; dt <- CFL estimate (cross.f:1196-1204,
// 1769-1818) from the maxima of the x-line tiles, reduced here by one
// workgroup.  NaN flag from the CFL maxima.
constexpr int FINISH_THREADS = 1024;
__device__ __forceinline__ void finish_body(DevScalars* sc, const RunConst& rc, int icfl,
                                            const double* cflp, int ntile) {
  __shared__ double red[FINISH_THREADS / 64][4];
  double c[4] = {0.0, 0.0, 0.0, 0.0};
  if (icfl) {
    for (int t = threadIdx.x; t < ntile; t += FINISH_THREADS) {
      const double2 p = ((const double2*)cflp)[2 * (size_t)t];
      const double2 q = ((const double2*)cflp)[2 * (size_t)t + 1];
      c[0] = max_nan(c[0], p.x);
      c[1] = max_nan(c[1], p.y);
      c[2] = max_nan(c[2], q.x);
      c[3] = max_nan(c[3], q.y);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
      for (int d = 32; d >= 1; d >>= 1) c[k] = max_nan(c[k], __shfl_xor(c[k], d));
    if ((threadIdx.x & 63) == 0)
      for (int k = 0; k < 4; ++k) red[threadIdx.x >> 6][k] = c[k];
    __syncthreads();
    if (threadIdx.x == 0)
      for (int w = 1; w < FINISH_THREADS / 64; ++w)
        for (int k = 0; k < 4; ++k) c[k] = max_nan(c[k], red[w][k]);
  }
  if (threadIdx.x != 0) return;
  sc->time = sc->time + sc->dt;
  if (icfl) {
    const double cx = c[0], cy = c[1], cz = c[2], cd = c[3];
    const double conv = cx * rc.hxalp * 0.5 + cy + cz * rc.hzbet * 0.5;
    double dtr = rc.cfl / (conv + cd);
    if (rc.dt_fp32) dtr = (double)(float)dtr;
    if (!(dtr > 0.0) || isinf(dtr)) sc->nan = 1;
    sc->dtr = dtr;
    sc->dt = dtr;
  }
}
__global__ __launch_bounds__(FINISH_THREADS) void k_finish_step(DevScalars* sc, RunConst rc,
                                                                 int icfl, const double* cflp,
                                                                 int ntile) {
  finish_body(sc, rc, icfl, cflp, ntile);
}
// one workgroup per run
__global__ __launch_bounds__(FINISH_THREADS) void k_finish_batch(const FinishArgs* args) {
  const FinishArgs& f = args[blockIdx.x];
  finish_body(f.sc, f.rc, f.icfl, f.cflp, f.ntile);
}
int launch_finish_batch(const FinishArgs* args, int nrun, hipStream_t st) {
  if (nrun <= 0) return 0;
  hipLaunchKernelGGL(k_finish_batch, dim3(nrun), dim3(FINISH_THREADS), 0, st, args);
  return (int)hipGetLastError();
}


// The step's per-chunk sums into the accumulated columns: one wavefront per
// (y row, quantity) adds the row's chunk partials (contiguous in memory),
// each lane a fixed strided subset in order and then a fixed shuffle tree,
// so the sum does not depend on scheduling.  Quantities: Tp, then up, vp,
// wp, uvr, uwr, vwr, w1p, w2p, w3p, thep, theup, ep; the last index takes
// the line sums of 1/T over z (rhom).  The plane-summed intensities of this
// step are kept for uner (cross.f:802-816).
__global__ __launch_bounds__(64) void k_stats_reduce(StatsArgs a) {
  const int my = a.rc.my;
  const int j = blockIdx.x, q = blockIdx.y, lane = threadIdx.x;
  constexpr int col[STAT_NPART + 4] = {20, 11, 12, 13, 14, 15, 16, 17, 18,
                                       19, 29, 30, 21, 28, 22, 25, 27};
  double s = 0.0;
  if (q < STAT_NPART) {
    const double* p = a.part + ((size_t)q * my + j) * a.nw;
    for (int w = lane; w < a.nw; w += 64) s += p[w];
  } else {
    const double* p = a.lines + (size_t)(q - STAT_NPART) * a.rc.mgalz * my;
    for (int z = lane; z < a.rc.mgalz; z += 64) s += p[(size_t)z * my + j];
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) s += __shfl_xor(s, d);
  if (lane == 0) {
    a.acc[(size_t)col[q] * my + j] += s;
    if (q >= 1 && q <= 9) a.last[(size_t)(q - 1) * my + j] = s;
  }
}

int launch_stats(int M, bool fp32, int which, const StatsArgs& a, hipStream_t st) {
  if (which == 3) {
    hipLaunchKernelGGL(k_stats_reduce, dim3(a.rc.my, STAT_NPART + 4), dim3(64), 0, st, a);
    return (int)hipGetLastError();
  }
  LOMA_DISPATCH_M(M, launch_stats_m<MM>(fp32, which, a, st));
}

int launch_finish_step(DevScalars* sc, RunConst rc, int icfl, const double* cflp, int ntile,
                       hipStream_t st) {
  if (icfl && (!cflp || ntile <= 0 || ntile > cfl_tiles_max(rc.my, rc.mgalz)))
    return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(k_finish_step, dim3(1), dim3(FINISH_THREADS), 0, st, sc, rc, icfl, cflp,
                     ntile);
  return (int)hipGetLastError();
}

// n doubles (an even number) rounded to floats in host memory: the link bounds
// it, so few workgroups do
__global__ __launch_bounds__(256) void k_narrow(const double2* __restrict__ src,
                                                float* __restrict__ dst, size_t n) {
  const size_t step = (size_t)gridDim.x * 256;
  for (size_t q = blockIdx.x * 256 + threadIdx.x; q < n / 4; q += step) {
    const double2 a = src[2 * q], b = src[2 * q + 1];
    ((float4*)dst)[q] = float4{(float)a.x, (float)a.y, (float)b.x, (float)b.y};
  }
  if (n % 4 && blockIdx.x == 0 && threadIdx.x == 0) {
    const double2 a = src[n / 2 - 1];
    ((float2*)dst)[n / 2 - 1] = float2{(float)a.x, (float)a.y};
  }
}
int launch_narrow(const double* src, float* dst, size_t n, hipStream_t st) {
  if (!n) return 0;
  const unsigned g = (unsigned)std::min<size_t>(128, (n / 4 + 255) / 256 + 1);
  hipLaunchKernelGGL(k_narrow, dim3(g), dim3(256), 0, st, (const double2*)src, dst, n);
  return (int)hipGetLastError();
}

}  // namespace loma
