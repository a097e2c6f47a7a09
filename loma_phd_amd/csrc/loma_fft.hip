// loma_fft.hip -- x/z Fourier transforms between spectral planes and
// physical lines, and the fused physical-space kernel.
//
// Reference: foup2 (trunk/lomacte3/src/cross.f:1282-1430), fourz/fourx
// (fou3D.f:29-95), FFTPACK conventions (cftsingle.f:2-66, rftsingle.f:25-96),
// phys2 (cross.f:1440-1828).
//
// Layouts (complex T2 = float2 or double2):
//   spectral S  : [i][k][j]       (kx plane, kz mode, y)   -- y fastest
//   z-physical W: [i][z][j]       (kx plane, z point, y)   -- y fastest
//   rhst/rhsz   : [z][j][x] FP64  (physical history of RHS(T) / RHS(Z))
// Every FFT is a Stockham autosort transform in LDS with mixed radices
// 8/4/2/3/5 (Govindaraju et al., SC'08 formulation), one workgroup per tile.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "loma_kernels.h"

namespace loma {

FftPlan make_plan(int n) {
  FftPlan p;
  p.n = n;
  p.npass = 0;
  int m = n;
  while (m % 8 == 0 && m > 1) { p.rad[p.npass++] = 8; m /= 8; }
  while (m % 4 == 0 && m > 1) { p.rad[p.npass++] = 4; m /= 4; }
  while (m % 2 == 0 && m > 1) { p.rad[p.npass++] = 2; m /= 2; }
  while (m % 3 == 0 && m > 1) { p.rad[p.npass++] = 3; m /= 3; }
  while (m % 5 == 0 && m > 1) { p.rad[p.npass++] = 5; m /= 5; }
  if (m != 1) p.npass = -1;  // unsupported length
  for (int q = 0, ns = 1; q < p.npass; ns *= p.rad[q], ++q) {
    p.inb[q] = (float)p.rad[q] / (float)n;
    p.ins[q] = 1.0f / (float)ns;
  }
  return p;
}

// x / d for 0 <= x < 2^20 from the rounded reciprocal of d: (x + 1/2) / d is at
// least 1/(2d) from an integer and its rounding error below x / d 2^-22.  The
// run-time plans divide several times per butterfly, and an integer division is
// some 20 instructions: 144x450x120 with Z, FP64 z transforms 0.37 -> 0.26 ms
// and x lines 1.41 -> 1.31 ms a launch, step 7.8 -> 6.9 ms
__device__ __forceinline__ int fast_div(int x, float inv) {
  return (int)(((float)x + 0.5f) * inv);
}

template <typename T2>
__device__ __forceinline__ T2 cmul(T2 a, T2 b) {
  T2 r;
  r.x = a.x * b.x - a.y * b.y;
  r.y = a.x * b.y + a.y * b.x;
  return r;
}
template <typename T2>
__device__ __forceinline__ T2 cadd(T2 a, T2 b) { T2 r; r.x = a.x + b.x; r.y = a.y + b.y; return r; }
template <typename T2>
__device__ __forceinline__ T2 csub(T2 a, T2 b) { T2 r; r.x = a.x - b.x; r.y = a.y - b.y; return r; }
// multiply by s*i (s = +1 or -1)
template <typename T2>
__device__ __forceinline__ T2 cmuli(T2 a, int s) { T2 r; r.x = -s * a.y; r.y = s * a.x; return r; }

// in-register DFT of size R: V_k = sum_r v_r exp(s 2 pi i r k / R)
template <typename T, typename T2>
__device__ __forceinline__ void dft2(T2* v) {
  T2 a = v[0], b = v[1];
  v[0] = cadd(a, b);
  v[1] = csub(a, b);
}
template <typename T, typename T2>
__device__ __forceinline__ void dft4(T2* v, int s) {
  T2 t0 = cadd(v[0], v[2]), t1 = csub(v[0], v[2]);
  T2 t2 = cadd(v[1], v[3]), t3 = cmuli(csub(v[1], v[3]), s);
  v[0] = cadd(t0, t2);
  v[2] = csub(t0, t2);
  v[1] = cadd(t1, t3);
  v[3] = csub(t1, t3);
}
template <typename T, typename T2>
__device__ __forceinline__ void dft8(T2* v, int s) {
  T2 e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
  dft4<T, T2>(e, s);
  dft4<T, T2>(o, s);
  const T h = (T)0.70710678118654752440;
  T2 w1, w3;
  w1.x = h; w1.y = s * h;     // exp(s i pi/4)
  w3.x = -h; w3.y = s * h;    // exp(s 3 i pi/4)
  T2 o1 = cmul(o[1], w1), o2 = cmuli(o[2], s), o3 = cmul(o[3], w3);
  v[0] = cadd(e[0], o[0]);
  v[4] = csub(e[0], o[0]);
  v[1] = cadd(e[1], o1);
  v[5] = csub(e[1], o1);
  v[2] = cadd(e[2], o2);
  v[6] = csub(e[2], o2);
  v[3] = cadd(e[3], o3);
  v[7] = csub(e[3], o3);
}
template <typename T, typename T2>
__device__ __forceinline__ void dft3(T2* v, int s) {
  const T c = (T)-0.5, sn = (T)(0.86602540378443864676) * (T)s;
  T2 a = v[0], b = v[1], d = v[2];
  T2 sum = cadd(b, d), dif = csub(b, d);
  v[0] = cadd(a, sum);
  T2 m;
  m.x = a.x + c * sum.x;
  m.y = a.y + c * sum.y;
  T2 r;
  r.x = -sn * dif.y;
  r.y = sn * dif.x;
  v[1] = cadd(m, r);
  v[2] = csub(m, r);
}
template <typename T, typename T2>
__device__ __forceinline__ void dft6(T2* v, int s) {
  T2 e[3] = {v[0], v[2], v[4]}, o[3] = {v[1], v[3], v[5]};
  dft3<T, T2>(e, s);
  dft3<T, T2>(o, s);
  const T c = (T)0.5, h = (T)(0.86602540378443864676) * (T)s;
  const T2 o1 = cmul(o[1], T2{c, h}), o2 = cmul(o[2], T2{-c, h});  // exp(s i pi k/3)
  v[0] = cadd(e[0], o[0]);
  v[3] = csub(e[0], o[0]);
  v[1] = cadd(e[1], o1);
  v[4] = csub(e[1], o1);
  v[2] = cadd(e[2], o2);
  v[5] = csub(e[2], o2);
}
template <typename T, typename T2>
__device__ __forceinline__ void dft5(T2* v, int s) {
  const T c1 = (T)0.30901699437494742410, c2 = (T)-0.80901699437494742410;
  const T s1 = (T)0.95105651629515357212 * (T)s, s2 = (T)0.58778525229247312917 * (T)s;
  T2 a = v[0];
  T2 b1 = cadd(v[1], v[4]), d1 = csub(v[1], v[4]);
  T2 b2 = cadd(v[2], v[3]), d2 = csub(v[2], v[3]);
  v[0].x = a.x + b1.x + b2.x;
  v[0].y = a.y + b1.y + b2.y;
  T2 m1, m2, r1, r2;
  m1.x = a.x + c1 * b1.x + c2 * b2.x; m1.y = a.y + c1 * b1.y + c2 * b2.y;
  m2.x = a.x + c2 * b1.x + c1 * b2.x; m2.y = a.y + c2 * b1.y + c1 * b2.y;
  // r = i*(s1 d1 + s2 d2), i*(s2 d1 - s1 d2)
  r1.x = -(s1 * d1.y + s2 * d2.y); r1.y = s1 * d1.x + s2 * d2.x;
  r2.x = -(s2 * d1.y - s1 * d2.y); r2.y = s2 * d1.x - s1 * d2.x;
  v[1] = cadd(m1, r1);
  v[4] = csub(m1, r1);
  v[2] = cadd(m2, r2);
  v[3] = csub(m2, r2);
}

// LDS layout of FFT work buffers: one pad entry after every 8, so that the
// stride-R butterfly writes of the first passes spread over the banks.
#ifndef LOMA_LDS_PAD
#define LOMA_LDS_PAD 0
#endif
// waves per SIMD the x-line and z-transform kernels are compiled for
#ifndef LOMA_XL_WPE
#define LOMA_XL_WPE 2
#endif
#ifndef LOMA_ZF_WPE
#define LOMA_ZF_WPE 4
#endif
template <int PAD = LOMA_LDS_PAD>
__device__ __forceinline__ int lds_i(int i) { return PAD ? i + (i >> 3) : i; }
__host__ __device__ inline int lds_entries(int n, int pad = LOMA_LDS_PAD) {
  return pad ? n + (n >> 3) + 1 : n;
}
// Row-major LDS rows of a z-transform tile: entry i of row `row` at
// row * rs + lds_i<PAD>(i).  The in-row pad spreads the stride-R butterfly
// writes over the banks; the row stride is odd (in entries) so that the
// tile's global loads and stores, which walk down a column (consecutive
// rows, same i), hit distinct banks.
__host__ __device__ inline int lds_row_stride(int n, int pad) { return n + (pad ? n / 8 : 0) + 1; }
#ifndef LOMA_ZF_PAD32
#define LOMA_ZF_PAD32 1
#endif
template <typename T>
constexpr int zf_pad() { return sizeof(T) == 8 ? 1 : LOMA_ZF_PAD32; }

// Twiddles of one butterfly: w[r] *= tw[jm * r * tstep] (conjugated for
// s > 0), r = 1..R-1.  With LOMA_TW_REC = 1 (default) only tw[jm * tstep]
// is loaded and its powers are formed by products (at most three
// multiplications deep), which trades six table loads per butterfly for
// complex multiplications: 5.75 against 5.97 ms per FP64 x-line launch and
// 1.64 against 1.74 ms per FP64 forward z launch at 512x513x256.
#ifndef LOMA_TW_REC
#define LOMA_TW_REC 1
#endif
// the powers of a loaded first twiddle p1 (LOMA_TW_REC's products)
template <int R, typename T2>
__device__ __forceinline__ void twiddle_pow(T2* w, T2 p1, int s) {
  T2 p[R];
  p[1] = p1;
  if (s > 0) p[1].y = -p[1].y;
  if constexpr (R >= 3) p[2] = cmul(p[1], p[1]);
  if constexpr (R >= 4) p[3] = cmul(p[2], p[1]);
  if constexpr (R >= 5) p[4] = cmul(p[2], p[2]);
  if constexpr (R >= 6) p[5] = cmul(p[4], p[1]);
  if constexpr (R >= 8) {
    p[6] = cmul(p[3], p[3]);
    p[7] = cmul(p[4], p[3]);
  }
#pragma unroll
  for (int r = 1; r < R; ++r) w[r] = cmul(w[r], p[r]);
}
// The same with the third power p3 from the table too: no power is more than
// two multiplications away from a table entry.  The recursion from p1 alone
// makes most of a transform's error and grows with the radices of the later
// passes (rms of 256 points in eps: passes 8, 8, 4 1.02 FP32 and 1.09 FP64;
// 4, 8, 8 1.40 and 1.30, with p3 0.79 and 0.70).
template <int R, typename T2>
__device__ __forceinline__ void twiddle_pow3(T2* w, T2 p1, T2 p3, int s) {
  if constexpr (R < 4) {
    twiddle_pow<R>(w, p1, s);
  } else {
    T2 p[R];
    p[1] = p1;
    p[3] = p3;
    if (s > 0) {
      p[1].y = -p[1].y;
      p[3].y = -p[3].y;
    }
    p[2] = cmul(p[1], p[1]);
    if constexpr (R >= 5) p[4] = cmul(p[3], p[1]);
    if constexpr (R >= 6) p[5] = cmul(p[3], p[2]);
    if constexpr (R >= 8) {
      p[6] = cmul(p[3], p[3]);
      p[7] = cmul(p[4], p[3]);
    }
#pragma unroll
    for (int r = 1; r < R; ++r) w[r] = cmul(w[r], p[r]);
  }
}
template <int R, typename T2>
__device__ __forceinline__ void twiddle(T2* w, const T2* __restrict__ tw, int jm, int tstep,
                                        int s) {
  if constexpr (LOMA_TW_REC) {
    twiddle_pow<R>(w, tw[jm * tstep], s);
  } else {
#pragma unroll
    for (int r = 1; r < R; ++r) {
      T2 t = tw[jm * r * tstep];
      if (s > 0) t.y = -t.y;
      w[r] = cmul(w[r], t);
    }
  }
}

template <int R, typename T, typename T2, int PAD = LOMA_LDS_PAD>
__device__ __forceinline__ void stockham_item(const T2* __restrict__ src, T2* __restrict__ dst,
                                              int rowbase, int j, int nb, int Ns, float ins,
                                              int tstep, const T2* __restrict__ tw, int s) {
  T2 v[R];
  const int jq = fast_div(j, ins), jm = j - jq * Ns;
#pragma unroll
  for (int r = 0; r < R; ++r) v[r] = src[lds_i<PAD>(rowbase + j + r * nb)];
  if (Ns > 1) twiddle<R>(v, tw, jm, tstep, s);
  if (R == 2) dft2<T, T2>(v);
  if (R == 3) dft3<T, T2>(v, s);
  if (R == 4) dft4<T, T2>(v, s);
  if (R == 5) dft5<T, T2>(v, s);
  if (R == 8) dft8<T, T2>(v, s);
  const int idxD = rowbase + jq * Ns * R + jm;
#pragma unroll
  for (int r = 0; r < R; ++r) dst[lds_i<PAD>(idxD + r * Ns)] = v[r];
}

// nrows independent length-N transforms of rows stored with stride N in a
// (LDS, padded layout lds_i); b is scratch of the same size.  Returns the
// buffer holding the result.  s = -1 forward (e^{-i}), +1 inverse; unscaled.
// Ends with a barrier.
template <typename T, typename T2, int PAD = LOMA_LDS_PAD>
__device__ __forceinline__ T2* fft_rows(T2* a, T2* b, int N, int RS, int nrows, const FftPlan& pl,
                        const T2* __restrict__ tw, int s) {
  int Ns = 1;
  for (int p = 0; p < pl.npass; ++p) {
    const int R = pl.rad[p];
    const int nb = N / R;
    const int tstep = N / (Ns * R);
    const int total = nrows * nb;
    const float inb = pl.inb[p], ins = pl.ins[p];
    for (int it = threadIdx.x; it < total; it += blockDim.x) {
      const int row = fast_div(it, inb), j = it - row * nb;
      const int rb = row * RS;
      switch (R) {
        case 2: stockham_item<2, T, T2, PAD>(a, b, rb, j, nb, Ns, ins, tstep, tw, s); break;
        case 3: stockham_item<3, T, T2, PAD>(a, b, rb, j, nb, Ns, ins, tstep, tw, s); break;
        case 4: stockham_item<4, T, T2, PAD>(a, b, rb, j, nb, Ns, ins, tstep, tw, s); break;
        case 5: stockham_item<5, T, T2, PAD>(a, b, rb, j, nb, Ns, ins, tstep, tw, s); break;
        default: stockham_item<8, T, T2, PAD>(a, b, rb, j, nb, Ns, ins, tstep, tw, s); break;
      }
    }
    __syncthreads();
    T2* t = a;
    a = b;
    b = t;
    Ns *= R;
  }
  return a;
}

// In-place variant for one LDS buffer: each pass loads its items into
// registers, synchronises, writes the butterflies back, synchronises.
// nrows * N <= blockDim.x * E (E = complex entries per thread).
template <int R, typename T, typename T2, int PAD>
__device__ __forceinline__ void radix_pass_ip(T2* a, int N, int RS, int nrows, int Ns, int tstep,
                                              float inb, float ins, const T2* __restrict__ tw,
                                              int s, T2* v, int nitems) {
  const int nb = N / R;
  const int total = nrows * nb;
#pragma unroll
  for (int k = 0; k < nitems; ++k) {
    const int it = threadIdx.x + k * blockDim.x;
    if (it < total) {
      const int row = fast_div(it, inb), j = it - row * nb;
#pragma unroll
      for (int r = 0; r < R; ++r) v[k * R + r] = a[row * RS + lds_i<PAD>(j + r * nb)];
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < nitems; ++k) {
    const int it = threadIdx.x + k * blockDim.x;
    if (it < total) {
      const int row = fast_div(it, inb), j = it - row * nb;
      const int jq = fast_div(j, ins), jm = j - jq * Ns;
      T2* w = v + k * R;
      if (Ns > 1) twiddle<R>(w, tw, jm, tstep, s);
      if (R == 2) dft2<T, T2>(w);
      if (R == 3) dft3<T, T2>(w, s);
      if (R == 4) dft4<T, T2>(w, s);
      if (R == 5) dft5<T, T2>(w, s);
      if (R == 8) dft8<T, T2>(w, s);
      const int idxD = jq * Ns * R + jm;
#pragma unroll
      for (int r = 0; r < R; ++r) a[row * RS + lds_i<PAD>(idxD + r * Ns)] = w[r];
    }
  }
  __syncthreads();
}

template <typename T, typename T2, int E, int PAD>
__device__ void fft_rows_ip(T2* a, int N, int nrows, const FftPlan& pl,
                            const T2* __restrict__ tw, int s) {
  T2 v[E + 8];
  const int RS = lds_row_stride(N, PAD);
  int Ns = 1;
  for (int p = 0; p < pl.npass; ++p) {
    const int R = pl.rad[p];
    const int tstep = N / (Ns * R);
    const float inb = pl.inb[p], ins = pl.ins[p];
    switch (R) {
      case 2: radix_pass_ip<2, T, T2, PAD>(a, N, RS, nrows, Ns, tstep, inb, ins, tw, s, v, (E + 1) / 2); break;
      case 3: radix_pass_ip<3, T, T2, PAD>(a, N, RS, nrows, Ns, tstep, inb, ins, tw, s, v, (E + 2) / 3); break;
      case 4: radix_pass_ip<4, T, T2, PAD>(a, N, RS, nrows, Ns, tstep, inb, ins, tw, s, v, (E + 3) / 4); break;
      case 5: radix_pass_ip<5, T, T2, PAD>(a, N, RS, nrows, Ns, tstep, inb, ins, tw, s, v, (E + 4) / 5); break;
      default: radix_pass_ip<8, T, T2, PAD>(a, N, RS, nrows, Ns, tstep, inb, ins, tw, s, v, (E + 7) / 8); break;
    }
    Ns *= R;
  }
}

// Compile-time plans for the production lengths: the same radix sequence as
// make_plan (8s, then 4, 2, 3, 5), with every stride, index split and
// twiddle step a constant, so the index arithmetic folds into shifts and
// multiplies.  Results are identical to the run-time plan.
constexpr int ct_radix(int m) {
  return m % 8 == 0 ? 8 : (m % 4 == 0 ? 4 : (m % 2 == 0 ? 2 : (m % 3 == 0 ? 3 : 5)));
}

template <typename T, typename T2, int E, int N, int Ns, int NT, int PAD, int NSTOP = N>
__device__ __forceinline__ void fft_rows_ip_ct(T2* a, int nrows, const T2* __restrict__ tw,
                                               int s, T2* v) {
  if constexpr (Ns < NSTOP) {
    constexpr int R = ct_radix(N / Ns);
    constexpr int nb = N / R;
    constexpr int tstep = N / (Ns * R);
    constexpr int nitems = (E + R - 1) / R;
    constexpr int RS = N + (PAD ? N / 8 : 0) + 1;
    const int total = nrows * nb;
    int t0 = threadIdx.x;
    asm volatile("" : "+v"(t0));
#pragma unroll
    for (int k = 0; k < nitems; ++k) {
      const int it = t0 + k * NT;
      if (it < total) {
        const int row = it / nb, j = it - row * nb;
#pragma unroll
        for (int r = 0; r < R; ++r) v[k * R + r] = a[row * RS + lds_i<PAD>(j + r * nb)];
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < nitems; ++k) {
      const int it = t0 + k * NT;
      if (it < total) {
        const int row = it / nb, j = it - row * nb;
        const int jm = j % Ns;
        T2* w = v + k * R;
        if (Ns > 1) twiddle<R>(w, tw, jm, tstep, s);
        if (R == 2) dft2<T, T2>(w);
        if (R == 3) dft3<T, T2>(w, s);
        if (R == 4) dft4<T, T2>(w, s);
        if (R == 5) dft5<T, T2>(w, s);
        if (R == 8) dft8<T, T2>(w, s);
        const int idxD = (j / Ns) * Ns * R + jm;
#pragma unroll
        for (int r = 0; r < R; ++r) a[row * RS + lds_i<PAD>(idxD + r * Ns)] = w[r];
      }
    }
    __syncthreads();
    fft_rows_ip_ct<T, T2, E, N, Ns * R, NT, PAD, NSTOP>(a, nrows, tw, s, v);
  }
}

// Ns of the last pass of the compile-time plan of length N
constexpr int ct_last_ns(int N) {
  int Ns = 1;
  while (Ns * ct_radix(N / Ns) < N) Ns *= ct_radix(N / Ns);
  return Ns;
}
template <int R, typename T, typename T2>
__device__ __forceinline__ void dft_r(T2* w, int s) {
  if constexpr (R == 2) dft2<T, T2>(w);
  if constexpr (R == 3) dft3<T, T2>(w, s);
  if constexpr (R == 4) dft4<T, T2>(w, s);
  if constexpr (R == 5) dft5<T, T2>(w, s);
  if constexpr (R == 6) dft6<T, T2>(w, s);
  if constexpr (R == 8) dft8<T, T2>(w, s);
}

// NN > 0: compile-time length NN; NN = 0: the run-time plan
template <typename T, typename T2, int E, int NN, int NT, int PAD>
__device__ __forceinline__ void fft_any_ip(T2* a, int N, int nrows, const FftPlan& pl,
                                           const T2* __restrict__ tw, int s) {
  if constexpr (NN > 0) {
    T2 v[E + 8];
    fft_rows_ip_ct<T, T2, E, NN, 1, NT, PAD>(a, nrows, tw, s, v);
  } else {
    fft_rows_ip<T, T2, E, PAD>(a, N, nrows, pl, tw, s);
  }
}

// ------------------------------------------------------------------------
// z transforms: spectral [i][k][j] <-> z-physical [i][z][j]
// (localyz2zy + fourz(+1), fou3D.f:103-146 / fourz(-1) + localzy2yz)
// ------------------------------------------------------------------------
// z transform of a J-row tile with register-resident ends (compile-time
// length N).  The first radix pass takes its items row-fastest (lanes
// 0..J-1 are the J y rows at one z), so its R inputs per item come straight
// from HBM in runs of J entries; it has no twiddles and writes LDS.  The
// middle passes run in LDS; the last pass, again row-fastest, writes its
// outputs z = j + r*Ns straight to HBM.  This saves the staging of the tile
// through LDS on the way in and on the way out (two LDS passes, two
// barriers).  INV: spectral [i][k][j] -> z-physical [i][z][j] (the dealiased
// band reads as zero); else the reverse, scaled by 1/N, dealiased modes
// dropped.
#ifndef LOMA_ZF_REG
#define LOMA_ZF_REG 1
#endif
template <typename T, typename T2, int E, int N, int PAD, bool INV>
__device__ __forceinline__ void zfft_reg(const T2* __restrict__ src, T2* __restrict__ dst,
                                         T2* A, int i, int j0, int J, int my, int myp, int mz,
                                         int nz, const T2* __restrict__ tw) {
  constexpr int RS = N + (PAD ? N / 8 : 0) + 1;
  constexpr int R1 = ct_radix(N), nb1 = N / R1;
  constexpr int NSL = ct_last_ns(N), RL = N / NSL, nbL = N / RL;
  static_assert(NSL > 1, "at least two passes");
  const int sgn = INV ? +1 : -1;
  T2 v[E + 8];
  // first pass
  {
    constexpr int nit = (E + R1 - 1) / R1;
    const int total = J * nb1;
#pragma unroll
    for (int q = 0; q < nit; ++q) {
      const int it = threadIdx.x + q * 256;
      if (it < total) {
        const int jj = it % J, j = it / J, jy = j0 + jj;
        T2* w = v + q * R1;
#pragma unroll
        for (int r = 0; r < R1; ++r) {
          const int z = j + r * nb1;
          T2 x = T2{0, 0};
          if (jy < my) {
            if constexpr (INV) {
              const int k = z <= nz ? z : (z >= N - nz ? z - N + mz : -1);
              if (k >= 0) x = src[((size_t)i * mz + k) * myp + jy];
            } else {
              x = src[((size_t)i * N + z) * myp + jy];
            }
          }
          w[r] = x;
        }
      }
    }
#pragma unroll
    for (int q = 0; q < nit; ++q) {
      const int it = threadIdx.x + q * 256;
      if (it < total) {
        const int jj = it % J, j = it / J;
        T2* w = v + q * R1;
        dft_r<R1, T, T2>(w, sgn);
#pragma unroll
        for (int r = 0; r < R1; ++r) A[jj * RS + lds_i<PAD>(j * R1 + r)] = w[r];
      }
    }
  }
  __syncthreads();
  // middle passes (Ns = R1 .. NSL)
  fft_rows_ip_ct<T, T2, E, N, R1, 256, PAD, NSL>(A, J, tw, sgn, v);
  // last pass.  FP64: every item's first twiddle is loaded before the first
  // store (a load after a store waits for it: vmcnt counts both, in order)
  // and pinned there so that the compiler does not sink the loads below the
  // earlier items' stores: 0.949 -> 0.920 ms (inverse) and 1.224 -> 1.214 ms
  // (forward) per launch at 512x513x256.  FP32 lost with it (inverse 0.458
  // -> 0.478 ms) and loads each item's twiddle in the item.
  {
    constexpr int nit = (E + RL - 1) / RL;
    const int total = J * nbL;
    const T sc = INV ? (T)1 : (T)(1.0 / (double)N);
    constexpr bool TWA = sizeof(T) == 8 && LOMA_TW_REC;
    T2 tw1[nit];
    if constexpr (TWA) {
#pragma unroll
      for (int q = 0; q < nit; ++q) {
        const int it = threadIdx.x + q * 256;
        tw1[q] = it < total ? tw[it / J] : T2{1, 0};
      }
#pragma unroll
      for (int q = 0; q < nit; ++q) asm volatile("" : "+v"(tw1[q].x), "+v"(tw1[q].y));
    }
#pragma unroll
    for (int q = 0; q < nit; ++q) {
      const int it = threadIdx.x + q * 256;
      if (it < total) {
        const int jj = it % J, j = it / J, jy = j0 + jj;
        T2* w = v + q * RL;
#pragma unroll
        for (int r = 0; r < RL; ++r) w[r] = A[jj * RS + lds_i<PAD>(j + r * nbL)];
        if constexpr (TWA) twiddle_pow<RL>(w, tw1[q], sgn);
        else twiddle<RL>(w, tw, j, 1, sgn);
        dft_r<RL, T, T2>(w, sgn);
        if (jy < my) {
#pragma unroll
          for (int r = 0; r < RL; ++r) {
            const int z = j + r * NSL;
            if constexpr (INV) {
              dst[((size_t)i * N + z) * myp + jy] = w[r];
            } else {
              const int k = z <= nz ? z : (z >= N - nz ? z - N + mz : -1);
              if (k >= 0) {
                T2 y = w[r];
                y.x *= sc;
                y.y *= sc;
                dst[((size_t)i * mz + k) * myp + jy] = y;
              }
            }
          }
        }
      }
    }
  }
}

// One workgroup: J consecutive y entries of one kx plane of one field, all
// z; one LDS buffer, in-place FFT (J * mgalz <= 256 * E).
template <typename T, int E, int NN>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(LOMA_ZF_WPE))) void k_zfft_inv(FftArgs a) {
  const int bx = blockIdx.x, by = blockIdx.y;
#include "loma_zfft_inv_body.inc"
}
template <typename T, int E, int NN>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(LOMA_ZF_WPE))) void k_zfft_inv_batch(
    const FftArgs* __restrict__ args, const int* __restrict__ first, int nrun) {
  const int r = batch_run(first, nrun, blockIdx.x);
  const FftArgs& a = args[r];
  const int bx = blockIdx.x - first[r], by = blockIdx.y;
#include "loma_zfft_inv_body.inc"
}

template <typename T, int E, int NN>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(LOMA_ZF_WPE))) void k_zfft_fwd(FftArgs a) {
  const int bx = blockIdx.x, by = blockIdx.y;
#include "loma_zfft_fwd_body.inc"
}
template <typename T, int E, int NN>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(LOMA_ZF_WPE))) void k_zfft_fwd_batch(
    const FftArgs* __restrict__ args, const int* __restrict__ first, int nrun) {
  const int r = batch_run(first, nrun, blockIdx.x);
  const FftArgs& a = args[r];
  const int bx = blockIdx.x - first[r], by = blockIdx.y;
#include "loma_zfft_fwd_body.inc"
}

// ------------------------------------------------------------------------
// x lines at the lengths of the run-time plan: inverse x transform of the 7 (11
// with Z) transform inputs, phys2 algebra, forward x transform of the 10 (11)
// outputs (foup2: 8 and 11), for 2*pairs lines
// (fixed z, consecutive y) per 256-thread workgroup.  Two real lines share
// one complex FFT.  The algebra runs in two passes so that only rho*u_i, T
// and one accumulator per point stay in registers:
//   pass 1: T, rho u, rho v, rho w -> u_i = rho u_i T and the six rho u_i u_j
//   pass 2: lap T, T_x, T_y, T_z (and Z's) accumulated into
//           r = T (lap T / Pe - rho u . grad T), then DT, drho (and DZ).
// Every global access of a field is a run of 2*PAIRS consecutive y entries.
// ------------------------------------------------------------------------
// 256 threads per x-line workgroup (512 measured slower on MI355X: more
// spills at the 128-VGPR budget that 8 waves per SIMD pair impose)
#ifndef LOMA_XL_THREADS
#define LOMA_XL_THREADS 256
#endif
constexpr int XL_THREADS = LOMA_XL_THREADS;

// Workgroups are dealt to the 8 XCDs round-robin; this maps the launch so
// that tiles t, t+1, ... (neighbouring y runs that share cache lines) run on
// one XCD and share its L2.  Launch 8*ceil(n/8) groups; tiles >= n idle.
__device__ __forceinline__ int xcd_tile(int b, int n) {
  const int per = (n + 7) / 8;
  return (b & 7) * per + (b >> 3);
}
__host__ inline int xcd_groups(int n) { return 8 * ((n + 7) / 8); }

// Per-thread share of one input field's lines: XR (kx, line pair) items of
// two complex coefficients, all loaded before the first is packed.
template <typename T2, int XR>
struct XlIn {
  T2 a[XR], b[XR];
};

template <typename T2, int XR>
__device__ __forceinline__ void xl_fetch(const FftArgs& a, const T2* __restrict__ src, int z,
                                         int j0, int pairs, XlIn<T2, XR>& v) {
  const int np = a.rc.nplanes, my = a.rc.my, mgz = a.rc.mgalz;
  const int lp = __builtin_ctz(pairs);  // pairs is a power of two
#pragma unroll
  for (int r = 0; r < XR; ++r) {
    const int it = threadIdx.x + r * XL_THREADS;
    T2 ca = T2{0, 0}, cb = T2{0, 0};
    if (it < np * pairs) {
      const int ii = it >> lp, p = it & (pairs - 1);
      const int ja = j0 + 2 * p, jb = ja + 1;
      const size_t base = ((size_t)ii * mgz + z) * a.rc.myp;
      if (ja < my) ca = src[base + ja];
      if (jb < my) cb = src[base + jb];
    }
    v.a[r] = ca;
    v.b[r] = cb;
  }
}

// Fields per x transform.  The rows of field f are f*pairs ..
// f*pairs+pairs-1, so one transform of 2*pairs rows keeps every thread of
// a radix pass busy where pairs alone is too few rows: FP64 at 480 points
// has 2 pairs, 120 radix-8 butterflies for 256 threads (two fields per
// transform 2.65 against 3.39 ms an x-line launch at 480x257x240, 0.143
// against 0.176 at 100x129x90).  FP32, with 4 pairs, carries one (2.11 ms;
// two would take 1.90, and 0.092 instead of 0.109 at 100x129x90).
#ifndef LOMA_XL_DUAL64
#define LOMA_XL_DUAL64 1
#endif
#ifndef LOMA_XL_DUAL32
#define LOMA_XL_DUAL32 0
#endif
template <typename T>
constexpr int xl_nf() {
  return (sizeof(T) == 8 ? LOMA_XL_DUAL64 : LOMA_XL_DUAL32) ? 2 : 1;
}
// x-line LDS rows: one pad entry after every eight (lds_i<1>) spreads the
// strided butterfly writes of the first radix-8 passes over the banks.  FP64
// (16-byte entries): 2.65 against 2.69 ms a launch at 480x257x240, but 0.143
// against 0.132 at 100x129x90; FP32 is slower padded (2.19 against 2.11 and
// 0.121 against 0.109 ms) and stays unpadded.
#ifndef LOMA_XL_PAD64
#define LOMA_XL_PAD64 1
#endif
#ifndef LOMA_XL_PAD32
#define LOMA_XL_PAD32 0
#endif
template <typename T>
constexpr int xl_pad() {
  return sizeof(T) == 8 ? LOMA_XL_PAD64 : LOMA_XL_PAD32;
}

// fetched lines of NF fields (xl_fetch) -> Hermitian-packed complex rows in
// A (row f*pairs + p = lines j0+2p, j0+2p+1 of field f); no barrier.
template <typename T, typename T2, int XR, int NF>
__device__ __forceinline__ void xl_pack_from(const FftArgs& a, const XlIn<T2, XR>* v, T2* A,
                                             int pairs, int dx) {
  constexpr int XP = xl_pad<T>();
  const int N = a.rc.mgalx, np = a.rc.nplanes;
  const int lp = __builtin_ctz(pairs);
  const int RS = N;
  // the dealiased band np..N-np is zero
  const int nzero = N - 2 * np + 1;
  const float iz = 1.0f / (float)nzero;
  for (int it = threadIdx.x; it < NF * pairs * nzero; it += XL_THREADS) {
    const int p = fast_div(it, iz), q = it - p * nzero;
    A[lds_i<XP>(p * RS + np + q)] = T2{0, 0};
  }
#pragma unroll
  for (int f = 0; f < NF; ++f) {
#pragma unroll
    for (int r = 0; r < XR; ++r) {
      const int it = threadIdx.x + r * XL_THREADS;
      if (it < np * pairs) {
        const int ii = it >> lp, p = it & (pairs - 1);
        const T2 ca = v[f].a[r], cb = v[f].b[r];
        const int rb = (f * pairs + p) * RS;
        if (f == dx) {                // ikx times this field, rounded once (XRow::pack_dx)
          const double kx = a.rc.alp * ii;
          const double ax = -kx * ca.y, ay = kx * ca.x, bx = -kx * cb.y, by = kx * cb.x;
          if (ii == 0) {
            A[lds_i<XP>(rb)] = T2{(T)ax, (T)bx};
          } else {
            A[lds_i<XP>(rb + ii)] = T2{(T)(ax - by), (T)(ay + bx)};
            A[lds_i<XP>(rb + N - ii)] = T2{(T)(ax + by), (T)(-ay + bx)};
          }
          continue;
        }
        if (ii == 0) {
          // the imaginary part of the kx=0 coefficient is ignored (rft, rftsingle.f:87-91)
          A[lds_i<XP>(rb)] = T2{ca.x, cb.x};
        } else {
          A[lds_i<XP>(rb + ii)] = T2{ca.x - cb.y, ca.y + cb.x};           // X_a + i X_b
          A[lds_i<XP>(rb + N - ii)] = T2{ca.x + cb.y, -ca.y + cb.x};      // conj(X_a) + i conj(X_b)
        }
      }
    }
  }
}
// lines of NF fields (W layout [i][z][j]; src1 unused for NF = 1) -> the
// packed rows in A; no barrier.
template <typename T, typename T2, int XR, int NF>
__device__ __forceinline__ void xl_pack(const FftArgs& a, const T2* __restrict__ src0,
                                        const T2* __restrict__ src1, T2* A, int z, int j0,
                                        int pairs, int dx) {
  XlIn<T2, XR> v[NF];
  xl_fetch<T2, XR>(a, src0, z, j0, pairs, v[0]);
  if constexpr (NF > 1) xl_fetch<T2, XR>(a, src1, z, j0, pairs, v[1]);
  xl_pack_from<T, T2, XR, NF>(a, v, A, pairs, dx);
}

// Hermitian unpacking of the transformed pairs in R into fields dst0 (rows
// 0..pairs-1) and dst1 (rows pairs..2*pairs-1), scaled by 1/N; no barrier.
template <typename T, typename T2, int NF>
__device__ __forceinline__ void xl_unpack(const FftArgs& a, const T2* R, T2* __restrict__ dst0,
                                          T2* __restrict__ dst1, int z, int j0, int pairs) {
  constexpr int XP = xl_pad<T>();
  const int N = a.rc.mgalx, np = a.rc.nplanes, my = a.rc.my, mgz = a.rc.mgalz;
  const int lp = __builtin_ctz(pairs);
  const int RS = N;
  const T hs = (T)(0.5 / (double)N);
  const int per = np * pairs;
  for (int it = threadIdx.x; it < NF * per; it += XL_THREADS) {
    const int f = NF > 1 && it >= per ? 1 : 0, jt = it - f * per;
    const int ii = jt >> lp, p = jt & (pairs - 1);
    const int ja = j0 + 2 * p, jb = ja + 1;
    const int rb = (f * pairs + p) * RS;
    const T2 zk = R[lds_i<XP>(rb + ii)];
    T2 zc = R[lds_i<XP>(rb + (ii ? N - ii : 0))];
    zc.y = -zc.y;
    T2 ya{(zk.x + zc.x) * hs, (zk.y + zc.y) * hs};
    T2 yb{(zk.y - zc.y) * hs, -(zk.x - zc.x) * hs};  // (zk - zc) / (2i)
    if (ii == 0) { ya.y = 0; yb.y = 0; }
    T2* dst = f ? dst1 : dst0;
    const size_t base = ((size_t)ii * mgz + z) * a.rc.myp;
    if (ja < my) dst[base + ja] = ya;
    if (jb < my) dst[base + jb] = yb;
  }
}

// pack, then the inverse FFT; the derivative d/dx of field dx (-1: of none).
// Returns the buffer holding the physical pairs.
template <typename T, typename T2, int XR, int NF>
__device__ __forceinline__ T2* xl_inverse(const FftArgs& a, const T2* __restrict__ src0,
                          const T2* __restrict__ src1, T2* A, T2* B, int z, int j0, int pairs,
                          int dx = -1) {
  xl_pack<T, T2, XR, NF>(a, src0, src1, A, z, j0, pairs, dx);
  __syncthreads();
  const int N = a.rc.mgalx;
  return fft_rows<T, T2, xl_pad<T>()>(A, B, N, N, NF * pairs, a.plx, (const T2*)a.twx, +1);
}

// forward FFT of A (rows of NF outputs, filled by the caller, then
// synchronised here) and the unpacking
template <typename T, typename T2, int NF>
__device__ __forceinline__ void xl_forward(const FftArgs& a, T2* __restrict__ dst0, T2* __restrict__ dst1,
                           T2* A, T2* B, int z, int j0, int pairs) {
  const int N = a.rc.mgalx;
  __syncthreads();
  const T2* R = fft_rows<T, T2, xl_pad<T>()>(A, B, N, N, NF * pairs, a.plx, (const T2*)a.twx, -1);
  xl_unpack<T, T2, NF>(a, R, dst0, dst1, z, j0, pairs);
  __syncthreads();
}

// Mean split: the transform inputs carry no 00 mode; its y-profile comes in
// FP64 (mean_in) and is added back here, per line.  Each output has an FP64
// per-y estimate g (the same algebra on the profiles) subtracted before the
// forward transform and stored in mean_out for phase C to add back, so the
// transforms (FP32 in mixed mode) only carry perturbation-sized values.
constexpr int XL_MAXL = 32;  // lines per workgroup (2 * pairs, pairs <= 16)

// Makes register arrays opaque to the optimiser at a loop head, so that
// per-output expressions are not hoisted out of the output loop and kept
// live for all outputs at once.
template <typename T, int E>
__device__ __forceinline__ void opaque_regs(T (&v)[E][2]) {
#pragma unroll
  for (int m = 0; m < E; ++m)
#pragma unroll
    for (int h = 0; h < 2; ++h) asm volatile("" : "+v"(v[m][h]));
}

// RK3 coefficients of a substep times dt; dtalpha = ab * dtbeta, so that
// the constraint source drho = d/(T T+ dtbeta) - ab r/T^2 takes one division:
// (d T - dtalpha r T+) / (T^2 T+ dtbeta)
struct XlRk {
  double dtxi, dtgamma, dtbeta, ab, dtalpha;
};
__device__ __forceinline__ XlRk xl_rk(double dt, int rkstep) {
  const double gam[3] = {8.0 / 15.0, 5.0 / 12.0, 3.0 / 4.0};
  const double xis[3] = {0.0, -17.0 / 60.0, -5.0 / 12.0};
  const double p0 = 5.0 / 66.0, p1 = -1.0;
  const double b3 = (p1 * (gam[0] * gam[2] + gam[1] * gam[2] + xis[1] * gam[2] + gam[0] * xis[2]) -
                     gam[0] * gam[1] * gam[2] - gam[0] * gam[1] * xis[2]) /
                    (p1 - gam[0] * gam[1]);
  const double betas[3] = {gam[0] - p0, p1, b3};
  const double alphas[3] = {p0, gam[1] + xis[1] - p1, gam[2] + xis[2] - b3};
  const int rk = rkstep - 1;
  return XlRk{dt * xis[rk], dt * gam[rk], dt * betas[rk], alphas[rk] / betas[rk],
              dt * alphas[rk]};
}

// Compiled for two waves per SIMD (LOMA_XL_WPE; FP64 always): at three,
// FP64 spilled heavily (and its Z-transport build gave wrong results), and
// FP32 spilled enough to measure slower (3.33 vs 3.22 ms at 512x513x256, when
// this kernel served 512 points).
template <typename T, bool WZ, int EPT>
__global__ __launch_bounds__(XL_THREADS)
__attribute__((amdgpu_waves_per_eu(XL_THREADS == 512 ? 4 : (sizeof(T) == 8 ? 2 : LOMA_XL_WPE)))) void k_xline(FftArgs a) {
  const int bx = blockIdx.x;
#include "loma_xline_body.inc"
}
template <typename T, bool WZ, int EPT>
__global__ __launch_bounds__(XL_THREADS)
__attribute__((amdgpu_waves_per_eu(XL_THREADS == 512 ? 4 : (sizeof(T) == 8 ? 2 : LOMA_XL_WPE)))) void k_xline_batch(
    const FftArgs* __restrict__ args, const int* __restrict__ first, int nrun) {
  const int r = batch_run(first, nrun, blockIdx.x);
  const FftArgs& a = args[r];
  const int bx = blockIdx.x - first[r];
#include "loma_xline_body.inc"
}

// ------------------------------------------------------------------------
// x lines, a wavefront (or an aligned part of one) per transform row, for
// rows of N = 64, 128, 256, 512 (E = 8) and 96, 192, 384 (E = 6) points.
// RL = N / E lanes own a row, E entries each, jl + RL r: what the last inverse
// pass (radix E) leaves in a lane's registers, what the physics takes there
// and what the first forward pass (radix E) starts from.  The passes stay
// inside the row's lanes and run in place in LDS between wavefront barriers;
// workgroup barriers remain around the pack and the unpack, whose lanes walk
// the y runs.  Rows carry one pad entry per eight and four more: pack, passes
// and unpack of the powers of two are free of bank conflicts.  FP64 transforms
// two fields at once (a thread holds 4 entries of each field, not 8: at 8 its
// registers allow one wavefront per SIMD) and its waves exchange entries
// through the rows.
// Radices: E = 8: R0 = N / 64, 8, 8 (inverse), 8, 8, R0 (forward); E = 6:
// 8, RB = N / 48, 6 and 6, 8, RB.
// ------------------------------------------------------------------------
__device__ __forceinline__ double uniform(double v) {
  const long long b = __builtin_bit_cast(long long, v);
  const unsigned lo = __builtin_amdgcn_readfirstlane((int)b);
  const unsigned hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
  return __builtin_bit_cast(double, (long long)(((unsigned long long)hi << 32) | lo));
}
template <typename T, int N_>
struct XRow {
  using T2 = typename std::conditional<sizeof(T) == 4, float2, double2>::type;
  static constexpr int N = N_, NP = N / 3, E = N % 3 ? 8 : 6, RL = N / E;
  static constexpr int R0 = N / 64, RB = N / 48;
  static constexpr int NF = sizeof(T) == 8 ? 2 : 1;   // fields per transform
  static constexpr int EF = E / NF;                   // entries of a thread per field
  static constexpr int pairs_of(int cap) {            // line pairs: a power of two, at most 16
    int p = 16;
    while (p * N > cap) p /= 2;
    return p;
  }
  static constexpr int P = pairs_of(sizeof(T) == 8 ? 1024 : 2048);
  static constexpr int GT = P * RL, NT = NF * GT, ROWS = NF * P;
  static constexpr int RS = N + N / 8 + 4;
  static constexpr int NBUF = sizeof(T) == 8 ? 1 : 2;   // row buffers
  static constexpr int XR = (NP * P + GT - 1) / GT;
  static constexpr int NL = E == 8 ? (R0 > 1 ? 8 / R0 : 1) : (48 + RL - 1) / RL;
  __device__ static __forceinline__ constexpr int li(int i) { return i + (i >> 3); }
  // position of entry jl + RL r (RL is a multiple of 8)
  __device__ static __forceinline__ int at(int jl, int r) { return li(jl) + RL / 8 * 9 * r; }
  // Twiddles of lane jl, passes 0: first inverse, 1: second inverse, 2: first
  // forward, 3 + q: second forward (items q).  The first powers are kept in
  // registers; the third powers come from `t3` (pass -> value).
  static constexpr int NTW = 3 + NL;
  __device__ static __forceinline__ int tw_index(int k, int jl) {
    if (k == 0) return E == 8 ? jl % R0 * (N / (8 * R0)) : jl % 8 * 6;
    if (k == 1) return jl;
    if (k == 2) return jl % E * (N / (8 * E));
    const int j = jl + RL * (k - 3);
    return E == 8 || j < 48 ? j : 0;
  }
  struct Tw {
    T2 p[NTW];
  };
  // the first (pw = 1) or third (pw = 3) powers
  __device__ static __forceinline__ Tw twiddles(const T2* __restrict__ tw, int jl, int pw) {
    Tw t;
#pragma unroll
    for (int k = 0; k < NTW; ++k) t.p[k] = tw[pw * tw_index(k, jl) % N];
    return t;
  }
  // This thread's (kx, line pair) items of a field: byte offset in the field
  // and the row entries X_k and X_{N-k} go to.  Items past the last read item
  // 0 and write the pad entries behind the row, as X_N of kx = 0 does.  Offsets
  // have 64 bits (fields of 4 GiB and more; with 32 a launch at 512x513x256 takes
  // the same 2.39 ms FP64 and 1.20 ms mixed).
  struct Items {
    size_t off[XR];
    int lo[XR], hi[XR];
  };
  __device__ static __forceinline__ Items items(int tg, int mgz, int z, int myp, int j0, int my) {
    Items t;
#pragma unroll
    for (int r = 0; r < XR; ++r) {
      const int it = tg + r * GT;
      const bool ok = it < NP * P;
      const int ii = ok ? it / P : 0, q = it % P;
      // tiles of up to 16 lines end inside the row's padding to a multiple of 16
      const int j = 2 * P <= 16 || j0 + 2 * q < my ? j0 + 2 * q : j0;
      t.off[r] = (((size_t)ii * mgz + z) * myp + j) * sizeof(T2);
      t.lo[r] = q * RS + (ok ? li(ii) : li(N) + 1);
      t.hi[r] = q * RS + li(N - ii);
    }
    return t;
  }
  __device__ static __forceinline__ void fetch(const T2* __restrict__ src, const Items& t,
                                               XlIn<T2, XR>& v) {
    typedef T vec __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int r = 0; r < XR; ++r) {
      const vec q = *(const vec*)((const char*)src + t.off[r]);
      v.a[r] = T2{q[0], q[1]};
      v.b[r] = T2{q[2], q[3]};
    }
  }
  // the coefficients times ikx (FP64; FP32 rows take pack_dx)
  __device__ static __forceinline__ void ikx(XlIn<T2, XR>& v, int tg, double alp) {
    static_assert(sizeof(T) == 8, "kx and the products are FP64");
#pragma unroll
    for (int r = 0; r < XR; ++r) {
      const T kx = (T)(alp * ((tg + r * GT) / P));
      v.a[r] = T2{-v.a[r].y * kx, v.a[r].x * kx};
      v.b[r] = T2{-v.b[r].y * kx, v.b[r].x * kx};
    }
  }
  // left: lines of the tile inside the grid (the others read as zero); the
  // imaginary part of the kx = 0 coefficient is ignored (rft, rftsingle.f:87-91)
  __device__ static __forceinline__ void mask(XlIn<T2, XR>& v, int tg, int left) {
    if (left < 2 * P) {
#pragma unroll
      for (int r = 0; r < XR; ++r) {
        const int l = 2 * ((tg + r * GT) % P);
        v.a[r].x = l < left ? v.a[r].x : (T)0;
        v.a[r].y = l < left ? v.a[r].y : (T)0;
        v.b[r].x = l + 1 < left ? v.b[r].x : (T)0;
        v.b[r].y = l + 1 < left ? v.b[r].y : (T)0;
      }
    }
    v.a[0].y = tg < P ? (T)0 : v.a[0].y;
    v.b[0].y = tg < P ? (T)0 : v.b[0].y;
  }
  // two real lines to one complex row
  __device__ static __forceinline__ void pack(XlIn<T2, XR> v, T2* A, int tg, const Items& t,
                                              int left) {
    mask(v, tg, left);
#pragma unroll
    for (int r = 0; r < XR; ++r) {
      const T2 ca = v.a[r], cb = v.b[r];
      A[t.lo[r]] = T2{ca.x - cb.y, ca.y + cb.x};      // X_a + i X_b
      A[t.hi[r]] = T2{ca.x + cb.y, -ca.y + cb.x};     // conj(X_a) + i conj(X_b)
    }
  }
  // the rows of d/dx: X = ikx times the coefficients, formed and summed in FP64
  // and rounded once (kx and the products rounded to FP32 on their own put two
  // more roundings on dT/dx)
  __device__ static __forceinline__ void pack_dx(XlIn<T2, XR> v, T2* A, int tg, const Items& t,
                                                 int left, double alp) {
    mask(v, tg, left);
#pragma unroll
    for (int r = 0; r < XR; ++r) {
      const double kx = alp * ((tg + r * GT) / P);
      const double ax = -kx * v.a[r].y, ay = kx * v.a[r].x;
      const double bx = -kx * v.b[r].y, by = kx * v.b[r].x;
      A[t.lo[r]] = T2{(T)(ax - by), (T)(ay + bx)};
      A[t.hi[r]] = T2{(T)(ax + by), (T)(-ay + bx)};
    }
  }
  // entry jl + c of a packed row (c a multiple of 8); NP .. N-NP are zero
  // (dealiased) and not stored
  __device__ static __forceinline__ T2 packed(const T2* A, int jl, int c) {
    if (c >= NP && c + RL - 1 <= N - NP) return T2{0, 0};
    const int i = jl + c;
    if (c + RL <= NP || c > N - NP) return A[li(jl) + c / 8 * 9];
    return i < NP || i > N - NP ? A[li(jl) + c / 8 * 9] : T2{0, 0};
  }
  template <typename T3>
  __device__ static __forceinline__ void inverse(T2* A, int jl, const Tw& tw, const T3& t3,
                                                 T2 (&w)[E]) {
    if constexpr (E == 8) {
      if constexpr (R0 > 1) {
#pragma unroll
        for (int q = 0; q < 8 / R0; ++q)
#pragma unroll
          for (int r = 0; r < R0; ++r) w[q * R0 + r] = packed(A, jl, RL * q + 64 * r);
        wave_sync();
#pragma unroll
        for (int q = 0; q < 8 / R0; ++q) {
          dft_r<R0, T, T2>(w + q * R0, +1);
          const int o = li((jl + RL * q) * R0);
#pragma unroll
          for (int r = 0; r < R0; ++r) A[o + r] = w[q * R0 + r];
        }
        wave_sync();
      }
#pragma unroll
      for (int r = 0; r < 8; ++r) w[r] = R0 > 1 ? A[at(jl, r)] : packed(A, jl, RL * r);
      if constexpr (R0 > 1) twiddle_pow3<8>(w, tw.p[0], t3(0), +1);
      dft8<T, T2>(w, +1);
      wave_sync();
      const int o = li(jl / R0 * (R0 * 8) + jl % R0);
#pragma unroll
      for (int r = 0; r < 8; ++r) A[o + r * R0 + (r * R0 >> 3)] = w[r];
    } else {
      const bool on = jl < N / 8;
      T2 u[8];
      if (on) {
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          const int i = jl + r * (N / 8);
          u[r] = i < NP || i > N - NP ? A[li(i)] : T2{0, 0};
        }
      }
      wave_sync();
      if (on) {
        dft8<T, T2>(u, +1);
#pragma unroll
        for (int r = 0; r < 8; ++r) A[9 * jl + r] = u[r];
      }
      wave_sync();
      T2 v[NL * RB];
#pragma unroll
      for (int q = 0; q < NL; ++q)
        if (48 % RL == 0 || jl + RL * q < 48)
#pragma unroll
          for (int r = 0; r < RB; ++r) v[q * RB + r] = A[li(jl) + RL / 8 * 9 * q + 54 * r];
      wave_sync();
#pragma unroll
      for (int q = 0; q < NL; ++q)
        if (48 % RL == 0 || jl + RL * q < 48) {
          twiddle_pow3<RB>(v + q * RB, tw.p[0], t3(0), +1);
          dft_r<RB, T, T2>(v + q * RB, +1);
          const int j = jl + RL * q, o = j / 8 * (9 * RB) + j % 8;
#pragma unroll
          for (int r = 0; r < RB; ++r) A[o + 9 * r] = v[q * RB + r];
        }
    }
    wave_sync();
#pragma unroll
    for (int r = 0; r < E; ++r) w[r] = A[at(jl, r)];
    twiddle_pow3<E>(w, tw.p[1], t3(1), +1);
    dft_r<E, T, T2>(w, +1);
  }
  // Transform of sign s (first twiddles of sign -1) of the row whose entries
  // jl + RL r are in w; the results stay in registers, v[q][r] = entry
  // jl + RL q + NLAST r of the row (lanes of q with jl + RL q < NLAST).
  static constexpr int RLAST = E == 8 ? (R0 > 1 ? R0 : 8) : RB;  // radix of the last pass
  static constexpr int NLAST = N / RLAST;
  __device__ static __forceinline__ bool last_on(int jl, int q) {
    return NLAST % RL == 0 || jl + RL * q < NLAST;
  }
  // position of entry jl + RL q + NLAST r (NLAST is a multiple of 8)
  __device__ static __forceinline__ int last_at(int jl, int q, int r) {
    return li(jl) + RL / 8 * 9 * q + NLAST / 8 * 9 * r;
  }
  template <typename T3>
  __device__ static __forceinline__ void row_fft(T2* A, int jl, const Tw& tw, const T3& t3, int s,
                                                 T2 (&w)[E], T2 (&v)[NL][RLAST]) {
    dft_r<E, T, T2>(w, s);
#pragma unroll
    for (int r = 0; r < E; ++r) A[E == 8 ? 9 * jl + r : li(6 * jl + r)] = w[r];
    wave_sync();
    const bool on = E == 8 || jl < N / 8;
    T2 u[8];
    if (on) {
#pragma unroll
      for (int r = 0; r < 8; ++r) u[r] = A[E == 8 ? at(jl, r) : li(jl + r * (N / 8))];
    }
    if constexpr (E == 8 && R0 == 1) {
      twiddle_pow3<8>(u, tw.p[3], t3(3), s);
      dft8<T, T2>(u, s);
#pragma unroll
      for (int r = 0; r < 8; ++r) v[0][r] = u[r];
    } else {
      wave_sync();
      if (on) {
        twiddle_pow3<8>(u, tw.p[2], t3(2), s);
        dft8<T, T2>(u, s);
        const int o = jl / E * (8 * E) + jl % E;
#pragma unroll
        for (int r = 0; r < 8; ++r) A[E == 8 ? li(o) + 9 * r : li(o + 6 * r)] = u[r];
      }
      wave_sync();
#pragma unroll
      for (int q = 0; q < NL; ++q)
        if (last_on(jl, q)) {
#pragma unroll
          for (int r = 0; r < RLAST; ++r) v[q][r] = A[last_at(jl, q, r)];
          twiddle_pow3<RLAST>(v[q], tw.p[3 + q], t3(3 + q), s);
          dft_r<RLAST, T, T2>(v[q], s);
        }
    }
  }
  template <typename T3>
  __device__ static __forceinline__ void forward(T2* A, int jl, const Tw& tw, const T3& t3,
                                                 T2 (&w)[E]) {
    T2 v[NL][RLAST];
    row_fft(A, jl, tw, t3, -1, w, v);
    wave_sync();
#pragma unroll
    for (int q = 0; q < NL; ++q)
      if (last_on(jl, q)) {
#pragma unroll
        for (int r = 0; r < RLAST; ++r) A[last_at(jl, q, r)] = v[q][r];
      }
  }
  // Hermitian unpacking into a field, scaled by 1/N (lines past my go to the
  // row's padding, which is never read, or are dropped)
  __device__ static __forceinline__ void unpack(const T2* A, T2* __restrict__ dst, int tg,
                                                const Items& t, int left) {
    typedef T vec __attribute__((ext_vector_type(4)));
    const T hs = (T)(0.5 / (double)N);
#pragma unroll
    for (int r = 0; r < XR; ++r) {
      const int it = tg + r * GT, q = it % P;
      const T2 zk = A[t.lo[r]];
      T2 zc = A[r == 0 && tg < P ? q * RS : t.hi[r]];
      zc.y = -zc.y;
      vec y;
      y[0] = (zk.x + zc.x) * hs;
      y[1] = (zk.y + zc.y) * hs;
      y[2] = (zk.y - zc.y) * hs;  // (zk - zc) / (2i)
      y[3] = -(zk.x - zc.x) * hs;
      if (r == 0) {
        y[1] = tg < P ? (T)0 : y[1];
        y[3] = tg < P ? (T)0 : y[3];
      }
      if ((r < XR - 1 || it < NP * P) && (2 * P <= 16 || 2 * q < left))
        *(vec*)((char*)dst + t.off[r]) = y;
    }
  }
};

template <typename T, bool WZ, int N>
__global__ __launch_bounds__((XRow<T, N>::NT))
__attribute__((amdgpu_waves_per_eu(2))) void k_xrow(FftArgs a) {
  const int bx = blockIdx.x;
#include "loma_xrow_body.inc"
}
template <typename T, bool WZ, int N>
__global__ __launch_bounds__((XRow<T, N>::NT))
__attribute__((amdgpu_waves_per_eu(2))) void k_xrow_batch(
    const FftArgs* __restrict__ args, const int* __restrict__ first, int nrun) {
  const int r = batch_run(first, nrun, blockIdx.x);
  const FftArgs& a = args[r];
  const int bx = blockIdx.x - first[r];
#include "loma_xrow_body.inc"
}

// fourz on standalone rows (FFTPACK convention), for the per-operator API.
// Lengths of XRow: RL lanes of a wavefront per row, from and to HBM in
// registers (runs of RL entries), two exchanges through the row's LDS and no
// workgroup barrier: 87,210 rows of 256 take 144 us, 5.0 TB/s where a large copy
// reaches 5.6; one workgroup a row took 321
template <int N>
__global__ __launch_bounds__(256) void k_fourz_row(const double2* __restrict__ tw, double2* c,
                                                   int nrows, int iopt) {
  using C = XRow<double, N>;
  constexpr int RL = C::RL, ROWS = 256 / RL;
  __shared__ double2 buf[ROWS * C::RS];
  const int lr = threadIdx.x / RL, jl = threadIdx.x - lr * RL;
  const long long row = (long long)blockIdx.x * ROWS + lr;
  if (row >= nrows) return;
  const typename C::Tw twd = C::twiddles(tw, jl, 1), tw3 = C::twiddles(tw, jl, 3);
  double2* p = c + row * N + jl;
  double2 w[C::E], v[C::NL][C::RLAST];
#pragma unroll
  for (int r = 0; r < C::E; ++r) w[r] = p[RL * r];
  C::row_fft(buf + lr * C::RS, jl, twd, [&](int k) { return tw3.p[k]; }, iopt < 0 ? -1 : 1, w, v);
  const double sc = iopt < 0 ? 1.0 / N : 1.0;
#pragma unroll
  for (int q = 0; q < C::NL; ++q)
    if (C::last_on(jl, q)) {
#pragma unroll
      for (int r = 0; r < C::RLAST; ++r) {
        double2 y = v[q][r];
        y.x *= sc;
        y.y *= sc;
        p[RL * q + C::NLAST * r] = y;
      }
    }
}
// other lengths: as many rows a workgroup as fill its threads, run-time plan
__global__ __launch_bounds__(256) void k_fourz(FftPlan pl, const double2* tw, double2* c,
                                               int nrows, int iopt, int per) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int N = pl.n;
  double2* A = (double2*)smem;
  double2* B = A + lds_entries(N * per);
  const long long row0 = (long long)blockIdx.x * per;
  const int nr = (int)min((long long)per, nrows - row0);
  double2* p = c + row0 * N;
  for (int it = threadIdx.x; it < nr * N; it += blockDim.x) A[lds_i(it)] = p[it];
  __syncthreads();
  double2* R = fft_rows<double, double2>(A, B, N, N, nr, pl, tw, iopt < 0 ? -1 : 1);
  const double sc = iopt < 0 ? 1.0 / N : 1.0;
  for (int it = threadIdx.x; it < nr * N; it += blockDim.x) {
    double2 v = R[lds_i(it)];
    v.x *= sc;
    v.y *= sc;
    p[it] = v;
  }
}

// ------------------------------------------------------------------------
// launchers
// ------------------------------------------------------------------------
static size_t zfft_lds(bool fp32, const FftArgs& a) {
  return (size_t)a.J * lds_row_stride(a.rc.mgalz, fp32 ? LOMA_ZF_PAD32 : 1) * (fp32 ? 8 : 16);
}
static size_t xline_lds(bool fp32, const FftArgs& a) {
  const int nf = fp32 ? xl_nf<float>() : xl_nf<double>();
  const int pad = fp32 ? xl_pad<float>() : xl_pad<double>();
  return (size_t)2 * lds_entries(nf * (a.L / 2) * a.rc.mgalx, pad) *
         (fp32 ? 8 : 16);
}

// kernel instance for a transform length: compile-time plans for the
// production lengths, the run-time plan otherwise
#define LOMA_BY_LENGTH(n, LAUNCH)              \
  switch (n) {                                 \
    case 64: { constexpr int NN = 64; LAUNCH; break; }   \
    case 96: { constexpr int NN = 96; LAUNCH; break; }   \
    case 128: { constexpr int NN = 128; LAUNCH; break; } \
    case 192: { constexpr int NN = 192; LAUNCH; break; } \
    case 256: { constexpr int NN = 256; LAUNCH; break; } \
    case 384: { constexpr int NN = 384; LAUNCH; break; } \
    case 512: { constexpr int NN = 512; LAUNCH; break; } \
    default: { constexpr int NN = 0; LAUNCH; break; }    \
  }

int launch_zfft_inv(bool fp32, const FftArgs& a, hipStream_t st) {
  const int nyb = (a.rc.my + a.J - 1) / a.J;
  dim3 g(a.rc.nplanes * nyb, a.nfields), b(256);
  const size_t lds = zfft_lds(fp32, a);
  // J * mgalz <= 256 * E (checked at init)
  if (fp32) {
    LOMA_BY_LENGTH(a.rc.mgalz, hipLaunchKernelGGL((k_zfft_inv<float, LOMA_ZF_E32, NN>), g, b, lds, st, a));
  } else {
    LOMA_BY_LENGTH(a.rc.mgalz, hipLaunchKernelGGL((k_zfft_inv<double, LOMA_ZF_E64, NN>), g, b, lds, st, a));
  }
  return (int)hipGetLastError();
}

int launch_zfft_fwd(bool fp32, const FftArgs& a, hipStream_t st) {
  const int nyb = (a.rc.my + a.J - 1) / a.J;
  dim3 g(a.rc.nplanes * nyb, a.nfields), b(256);
  const size_t lds = zfft_lds(fp32, a);
  if (fp32) {
    LOMA_BY_LENGTH(a.rc.mgalz, hipLaunchKernelGGL((k_zfft_fwd<float, LOMA_ZF_E32, NN>), g, b, lds, st, a));
  } else {
    LOMA_BY_LENGTH(a.rc.mgalz, hipLaunchKernelGGL((k_zfft_fwd<double, LOMA_ZF_E64, NN>), g, b, lds, st, a));
  }
  return (int)hipGetLastError();
}

// k_xrow serves the production lengths at the tile the plan gives them
// (L = 2 P lines); other lengths take k_xline with its run-time plan.
template <typename T>
static bool xrow_tile(const FftArgs& a) {
  switch (a.rc.mgalx) {
    case 64: return a.L == 2 * XRow<T, 64>::P;
    case 96: return a.L == 2 * XRow<T, 96>::P;
    case 128: return a.L == 2 * XRow<T, 128>::P;
    case 192: return a.L == 2 * XRow<T, 192>::P;
    case 256: return a.L == 2 * XRow<T, 256>::P;
    case 384: return a.L == 2 * XRow<T, 384>::P;
    case 512: return a.L == 2 * XRow<T, 512>::P;
    default: return false;
  }
}
bool xrow_serves(bool fp32, const FftArgs& a) {
  return fp32 ? xrow_tile<float>(a) : xrow_tile<double>(a);
}

// x-line kernel of a run's length
#define LOMA_XROW_BY_LENGTH(n, LAUNCH)                   \
  switch (n) {                                           \
    case 64: { constexpr int NN = 64; LAUNCH; break; }   \
    case 96: { constexpr int NN = 96; LAUNCH; break; }   \
    case 128: { constexpr int NN = 128; LAUNCH; break; } \
    case 192: { constexpr int NN = 192; LAUNCH; break; } \
    case 256: { constexpr int NN = 256; LAUNCH; break; } \
    case 384: { constexpr int NN = 384; LAUNCH; break; } \
    case 512: { constexpr int NN = 512; LAUNCH; break; } \
  }

template <typename T, bool WZ>
static void launch_xline_t(const FftArgs& a, dim3 g, size_t lds, hipStream_t st) {
  // entries per thread of k_xline: pairs * mgalx <= XL_THREADS * EPT, i.e. at
  // most 1024 (FP64) / 2048 (FP32) entries per workgroup (checked at init)
  constexpr int EPT = (sizeof(T) == 8 ? 1024 : 2048) / XL_THREADS;
  if (a.xrow) {
    LOMA_XROW_BY_LENGTH(a.rc.mgalx, hipLaunchKernelGGL((k_xrow<T, WZ, NN>), g, dim3(XRow<T, NN>::NT), 0, st, a));
  } else {
    hipLaunchKernelGGL((k_xline<T, WZ, EPT>), g, dim3(XL_THREADS), lds, st, a);
  }
}

int launch_xline(bool fp32, const FftArgs& a, hipStream_t st) {
  const int nyb = (a.rc.my + a.L - 1) / a.L;
  dim3 g(xcd_groups(a.rc.mgalz * nyb));
  const size_t lds = xline_lds(fp32, a);
  if (fp32) {
    if (a.with_z) launch_xline_t<float, true>(a, g, lds, st);
    else launch_xline_t<float, false>(a, g, lds, st);
  } else {
    if (a.with_z) launch_xline_t<double, true>(a, g, lds, st);
    else launch_xline_t<double, false>(a, g, lds, st);
  }
  return (int)hipGetLastError();
}

// ---- batched launches (one class of runs: same length, tiles, fields) ----
int zfft_blocks(const FftArgs& a) { return a.rc.nplanes * ((a.rc.my + a.J - 1) / a.J); }
int xline_blocks(const FftArgs& a) {
  return xcd_groups(a.rc.mgalz * ((a.rc.my + a.L - 1) / a.L));
}

int launch_zfft_batch(bool fp32, bool inv, const FftArgs& proto, const FftArgs* args,
                      const int* first, int nrun, int nblocks, hipStream_t st) {
  if (nblocks <= 0 || nrun <= 0) return 0;
  dim3 g(nblocks, proto.nfields), b(256);
  const size_t lds = zfft_lds(fp32, proto);
  if (fp32) {
    if (inv) {
      LOMA_BY_LENGTH(proto.rc.mgalz, hipLaunchKernelGGL((k_zfft_inv_batch<float, LOMA_ZF_E32, NN>), g, b, lds, st, args, first, nrun));
    } else {
      LOMA_BY_LENGTH(proto.rc.mgalz, hipLaunchKernelGGL((k_zfft_fwd_batch<float, LOMA_ZF_E32, NN>), g, b, lds, st, args, first, nrun));
    }
  } else {
    if (inv) {
      LOMA_BY_LENGTH(proto.rc.mgalz, hipLaunchKernelGGL((k_zfft_inv_batch<double, LOMA_ZF_E64, NN>), g, b, lds, st, args, first, nrun));
    } else {
      LOMA_BY_LENGTH(proto.rc.mgalz, hipLaunchKernelGGL((k_zfft_fwd_batch<double, LOMA_ZF_E64, NN>), g, b, lds, st, args, first, nrun));
    }
  }
  return (int)hipGetLastError();
}

template <typename T, bool WZ>
static void launch_xline_batch_t(const FftArgs& proto, dim3 g, size_t lds, hipStream_t st,
                                 const FftArgs* args, const int* first, int nrun) {
  constexpr int EPT = (sizeof(T) == 8 ? 1024 : 2048) / XL_THREADS;
  if (proto.xrow) {
    LOMA_XROW_BY_LENGTH(proto.rc.mgalx, hipLaunchKernelGGL((k_xrow_batch<T, WZ, NN>), g, dim3(XRow<T, NN>::NT), 0, st, args, first, nrun));
  } else {
    hipLaunchKernelGGL((k_xline_batch<T, WZ, EPT>), g, dim3(XL_THREADS), lds, st, args, first, nrun);
  }
}

int launch_xline_batch(bool fp32, const FftArgs& proto, const FftArgs* args, const int* first,
                       int nrun, int nblocks, hipStream_t st) {
  if (nblocks <= 0 || nrun <= 0) return 0;
  dim3 g(nblocks);
  const size_t lds = xline_lds(fp32, proto);
  if (fp32) {
    if (proto.with_z) launch_xline_batch_t<float, true>(proto, g, lds, st, args, first, nrun);
    else launch_xline_batch_t<float, false>(proto, g, lds, st, args, first, nrun);
  } else {
    if (proto.with_z) launch_xline_batch_t<double, true>(proto, g, lds, st, args, first, nrun);
    else launch_xline_batch_t<double, false>(proto, g, lds, st, args, first, nrun);
  }
  return (int)hipGetLastError();
}

int launch_fourz(const FftPlan& pl, const double2* tw, double2* c, int nrows, int iopt,
                 hipStream_t st) {
  if (nrows <= 0) return 0;
  switch (pl.n) {
#define LOMA_FOURZ_ROW(n)                                                                       \
    case n: {                                                                                   \
      constexpr int rows = 256 / XRow<double, n>::RL;                                           \
      hipLaunchKernelGGL((k_fourz_row<n>), dim3((nrows + rows - 1) / rows), dim3(256), 0, st, tw, \
                         c, nrows, iopt);                                                       \
      break;                                                                                    \
    }
    LOMA_FOURZ_ROW(64) LOMA_FOURZ_ROW(96) LOMA_FOURZ_ROW(128) LOMA_FOURZ_ROW(192)
    LOMA_FOURZ_ROW(256) LOMA_FOURZ_ROW(384) LOMA_FOURZ_ROW(512)
#undef LOMA_FOURZ_ROW
    default: {
      // 1024 entries a workgroup (both buffers 32 KiB: five workgroups a CU hide
      // each other's barriers); longer rows go one to a workgroup.  2048 entries
      // leave two a CU: 50,001 rows of 480 take 341 us so, 224 with 1024 and 299
      // with one row a workgroup; 5,003 rows of 1000 take 66, 51 and 53.  Few rows
      // are spread over the chip first, four workgroups to a CU: 734 rows of 216
      // take 20 us nine to a workgroup and 17 us one to a workgroup
      const int per = std::max(1, std::min(1024 / pl.n, nrows / 1024));
      hipLaunchKernelGGL(k_fourz, dim3((nrows + per - 1) / per), dim3(256),
                         (size_t)2 * lds_entries(pl.n * per) * 16, st, pl, tw, c, nrows, iopt, per);
    }
  }
  return (int)hipGetLastError();
}

}  // namespace loma
