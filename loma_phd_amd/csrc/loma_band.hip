// loma_band.hip -- batched pentadiagonal solves in isolation: LU without
// pivoting (bandec, trunk/lomacte3/src/cfdiff.f:977-1022) and the two
// triangular sweeps (banbks, cfdiff.f:954-974) for many independent systems
// with complex right-hand sides, FP64 arithmetic.
//
// A lane carries one system through both sweeps (W systems a wavefront): row
// j is reduced by the two rows before it and scaled by its pivot at once, so
// that {U1, U2, Y} / pivot, 32 bytes, is all that the backward sweep needs
// (errors against extended precision 1.33e-16, 1.66e-16 and 5.4e-16 for bands
// dominant by 2.5 and 1.01 times and close to a Helmholtz operator's; dividing
// by the pivot last gave 1.34e-16, 1.67e-16 and 5.5e-16).
// Every lane reads its own rows from HBM to registers, 16 bytes a load (the
// 128-byte lines that the 64 lanes walk stay in L1), with two chunks of CH rows
// in flight; the loops hold whole chunks and read on to a clamped row at their
// ends, because a chunk fetched under a condition is copied where the paths
// meet, behind a wait for every load.  The scratch rows have the group's
// systems fastest.
//
// The chain from row to row, a division and two multiply-adds, bounds small
// batches (about 270 cycles a row): 2653 systems of 422 rows 339 -> 83 us,
// 16 of 257 172 -> 49 us.  Traffic bounds large ones (72 bytes a row in and
// out, 64 of scratch): 16,384 systems of 513 rows 482 -> 257 us, of 257 rows
// with an FP32 right-hand side 334 -> 122 us, 4.5 TB/s.  Before, two waves
// per 64 systems staged system-major tiles through LDS, 152 bytes a row.
#include <hip/hip_runtime.h>

#include <mutex>
#include <type_traits>
#include <vector>

#include "loma_internal.h"
#include "loma_kernels.h"

namespace loma {

constexpr int CH = 8;  // rows per chunk of loads, two chunks in flight

// 16 bytes at the alignment the arrays have
typedef double v2d __attribute__((ext_vector_type(2), aligned(8)));
typedef float v4f __attribute__((ext_vector_type(4), aligned(4)));

// F32: the right-hand side is complex FP32 (else FP64).  rhs and x may be
// the same buffer (an FP64 solve in place), so neither is restrict.
template <bool F32, int W>
__global__ __launch_bounds__(64) void k_band5(const double* __restrict__ band, const void* rhs,
                                              double* x, double* __restrict__ scr, int n,
                                              int nsys) {
  using Y = typename std::conditional<F32, float, double>::type;
  const int lane = threadIdx.x, s0 = blockIdx.x * W, gs = min(W, nsys - s0);
  if (lane >= gs) return;
  const size_t s = (size_t)s0 + lane;
  const double* b = band + s * n * 5;
  const Y* rh = (const Y*)rhs + s * n * 2;
  // scratch of the group: row k's {U1, U2} and {Re Y, Im Y}, systems fastest
  char* const sg = (char*)(scr + (size_t)s0 * n * 4);
  const unsigned row16 = gs * 16, lane16 = lane * 16;
  double a[2][CH * 5];
  Y y[2][CH * 2];
  auto fetch = [&](int q, int r0) __attribute__((always_inline)) {  // rows r0 .. r0 + CH - 1
    const v2d* p = (const v2d*)(b + (size_t)r0 * 5);
#pragma unroll
    for (int e = 0; e < CH * 5 / 2; ++e) {
      const v2d t = p[e];
      a[q][2 * e] = t.x;
      a[q][2 * e + 1] = t.y;
    }
    if constexpr (F32) {
      const v4f* r = (const v4f*)(rh + (size_t)r0 * 2);
#pragma unroll
      for (int e = 0; e < CH / 2; ++e) {
        const v4f t = r[e];
        y[q][4 * e] = t.x;
        y[q][4 * e + 1] = t.y;
        y[q][4 * e + 2] = t.z;
        y[q][4 * e + 3] = t.w;
      }
    } else {
      const v2d* r = (const v2d*)(rh + (size_t)r0 * 2);
#pragma unroll
      for (int e = 0; e < CH; ++e) {
        const v2d t = r[e];
        y[q][2 * e] = t.x;
        y[q][2 * e + 1] = t.y;
      }
    }
  };
  // the entries left of the matrix, of rows 0 and 1
  auto left = [&]() __attribute__((always_inline)) { a[0][0] = a[0][1] = a[0][5] = 0.0; };
  // scaled rows j - 1 and j - 2 of the factor and the right-hand side
  double U1[2] = {0.0, 0.0}, U2[2] = {0.0, 0.0}, Yr[2] = {0.0, 0.0}, Yi[2] = {0.0, 0.0};
  auto row = [&](const double* w, Y br, Y bi, int j) __attribute__((always_inline)) {
    const double a0 = w[0];
    const double a1 = w[1] - a0 * U1[1];
    const double d = w[2] - a0 * U2[1] - a1 * U1[0];
    const double u1 = w[3] - a1 * U2[0], u2 = w[4];
    const double yr = br - a0 * Yr[1] - a1 * Yr[0];
    const double yi = bi - a0 * Yi[1] - a1 * Yi[0];
    const double iv = 1.0 / d;
    U1[1] = U1[0];
    U2[1] = U2[0];
    Yr[1] = Yr[0];
    Yi[1] = Yi[0];
    U1[0] = u1 * iv;
    U2[0] = u2 * iv;
    Yr[0] = yr * iv;
    Yi[0] = yi * iv;
    char* o = sg + (size_t)j * 2 * row16;
    *(double2*)(o + lane16) = double2{U1[0], U2[0]};
    *(double2*)(o + row16 + lane16) = double2{Yr[0], Yi[0]};
  };
  // rows 0 .. h - 1 come first, so that pairs of whole chunks are left
  const int h = n % (2 * CH);
  if (n < 2 * CH) {
    for (int j = 0; j < n; ++j) {
      const double* p = b + j * 5;
      const double w[5] = {j < 2 ? 0.0 : p[0], j < 1 ? 0.0 : p[1], p[2], p[3], p[4]};
      row(w, rh[2 * j], rh[2 * j + 1], j);
    }
  } else if (h) {
    fetch(0, 0);
    fetch(1, CH);
    left();
#pragma unroll
    for (int t = 0; t < 2 * CH - 1; ++t)
      if (t < h) row(a[t / CH] + t % CH * 5, y[t / CH][t % CH * 2], y[t / CH][t % CH * 2 + 1], t);
  }
  if (n >= 2 * CH) {
    fetch(0, h);
    fetch(1, h + CH);
    if (h == 0) left();
    if (h == 1) a[0][0] = 0.0;
#pragma unroll 1
    for (int r0 = h; r0 < n; r0 += 2 * CH)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
#pragma unroll
        for (int t = 0; t < CH; ++t)
          row(a[q] + t * 5, y[q][t * 2], y[q][t * 2 + 1], r0 + q * CH + t);
        fetch(q, min(r0 + (q + 2) * CH, n - CH));  // past the end: read and not used
      }
  }
  // columns n and n + 1 are not in the matrix
  *(double2*)(sg + (size_t)(n - 2) * 2 * row16 + lane16) = double2{U1[1], 0.0};
  *(double2*)(sg + (size_t)(n - 1) * 2 * row16 + lane16) = double2{0.0, 0.0};
  // backward sweep x_k = Y_k - U1 x_{k+1} - U2 x_{k+2}
  double2 u[2][CH], v[2][CH];
  auto sload = [&](int q, int r0) __attribute__((always_inline)) {  // rows r0 .. r0 + CH - 1
    const char* o = sg + (size_t)r0 * 2 * row16;
#pragma unroll
    for (int t = 0; t < CH; ++t) {
      u[q][t] = *(const double2*)(o + lane16);
      v[q][t] = *(const double2*)(o + row16 + lane16);
      o += 2 * row16;
    }
  };
  double xr[2] = {0.0, 0.0}, xi[2] = {0.0, 0.0};
  v2d* xo = (v2d*)(x + s * n * 2);
  auto back = [&](double2 u, double2 v, int k) __attribute__((always_inline)) {
    const double zr = v.x - u.y * xr[1] - u.x * xr[0];
    const double zi = v.y - u.y * xi[1] - u.x * xi[0];
    xr[1] = xr[0];
    xi[1] = xi[0];
    xr[0] = zr;
    xi[0] = zi;
    xo[k] = v2d{zr, zi};
  };
  if (n >= 2 * CH) {
    sload(0, n - CH);
    sload(1, n - 2 * CH);
#pragma unroll 1
    for (int r0 = n - CH; r0 > h; r0 -= 2 * CH)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
#pragma unroll
        for (int t = CH - 1; t >= 0; --t) back(u[q][t], v[q][t], r0 - q * CH + t);
        sload(q, max(r0 - (q + 2) * CH, 0));
      }
    if (h) {
      sload(0, 0);
      sload(1, CH);
#pragma unroll
      for (int t = 2 * CH - 2; t >= 0; --t)
        if (t < h) back(u[t / CH][t % CH], v[t / CH][t % CH], t);
    }
  } else {
    for (int k = n - 1; k >= 0; --k) {
      const char* o = sg + (size_t)k * 2 * row16;
      back(*(const double2*)(o + lane16), *(const double2*)(o + row16 + lane16), k);
    }
  }
}

// Systems a wavefront: 64 use the cache lines and the scratch rows best, but a
// batch has to reach every compute unit first, and a load that touches 64 lines
// takes four times the cycles of one that touches 16.  2653 systems of 422 rows:
// 83 us with 16, 88 with 32, 98 with 64; 16,384 of 513: 290, 272 and 257.  8 were
// no faster than 16 at 1024 systems (97 and 98 us for 513 rows).
int launch_band5(const double* band, const void* rhs, double* x, double* scratch, int n,
                 int nsys, int rhs_fp32, hipStream_t st) {
  if (nsys <= 0 || n <= 0) return 0;
  const dim3 b(64);
#define LOMA_BAND5(W)                                                                          \
  do {                                                                                         \
    const dim3 g((nsys + W - 1) / W);                                                          \
    if (rhs_fp32)                                                                              \
      hipLaunchKernelGGL((k_band5<true, W>), g, b, 0, st, band, rhs, x, scratch, n, nsys);     \
    else                                                                                       \
      hipLaunchKernelGGL((k_band5<false, W>), g, b, 0, st, band, rhs, x, scratch, n, nsys);    \
  } while (0)
  if (nsys <= 16 * 256) LOMA_BAND5(16);
  else if (nsys <= 32 * 256) LOMA_BAND5(32);
  else LOMA_BAND5(64);
#undef LOMA_BAND5
  return (int)hipGetLastError();
}

// ---- the allocation-free variant -------------------------------------------
// Scratch of loma_band5_solve_dev_noalloc: a fixed device array that every
// GPU the library runs on holds until the process ends.  Host code never
// passes the array's name to a kernel (on the host it is only a stand-in
// symbol); it uses the device address that hipGetSymbolAddress returns for
// the current device, kept per device in g_scr_dev.  A row takes four doubles;
// the limit of five, n*5*nsys, is the entry's own and stays.
constexpr size_t BAND5_SCRATCH_DOUBLES = (size_t)1 << 22;  // 4194304 doubles, 32 MiB
static __device__ __align__(256) double scratch[BAND5_SCRATCH_DOUBLES];

static std::mutex g_scr_mu;
static std::vector<double*> g_scr_dev;  // device address of scratch, per device

static int scratch_address(int dev, double** out) {
  std::lock_guard<std::mutex> lk(g_scr_mu);
  if ((int)g_scr_dev.size() <= dev) g_scr_dev.resize(dev + 1, nullptr);
  if (!g_scr_dev[dev]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) {
      set_error("loma_band5_solve_dev_noalloc: no device address for the scratch array");
      return LOMA_ERR_DEVICE;
    }
    g_scr_dev[dev] = (double*)p;
  }
  *out = g_scr_dev[dev];
  return LOMA_OK;
}

}  // namespace loma

extern "C" int loma_band5_solve_dev_noalloc(const double* band, void* rhs, double* x, int n,
                                            int nsys, int rhs_fp32, void* stream) {
  using namespace loma;
  if (!band || !rhs || n < 3 || nsys < 0 || (rhs_fp32 && !x)) {
    set_error("loma_band5_solve_dev_noalloc: bad arguments (n >= 3; x required for float rhs)");
    return LOMA_ERR_ARG;
  }
  if ((size_t)n * 5 * (size_t)nsys > BAND5_SCRATCH_DOUBLES) {
    set_error("loma_band5_solve_dev_noalloc: n*5*nsys exceeds the fixed scratch of "
              "4194304 doubles (32 MiB); split the batch");
    return LOMA_ERR_ARG;
  }
  if (nsys == 0) return LOMA_OK;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) {
    set_error("loma_band5_solve_dev_noalloc: hipGetDevice failed");
    return LOMA_ERR_DEVICE;
  }
  double* scr = nullptr;
  int e = scratch_address(dev, &scr);
  if (e) return e;
  hipStream_t st = (hipStream_t)stream;
  // every scratch entry the kernel reads it wrote first in the same launch,
  // so nothing is cleared
  e = launch_band5(band, rhs, x ? x : (double*)rhs, scr, n, nsys, rhs_fp32, st);
  if (e) {
    set_error("loma_band5_solve_dev_noalloc: launch failed");
    return LOMA_ERR_DEVICE;
  }
  if (hipStreamSynchronize(st) != hipSuccess) {
    set_error("loma_band5_solve_dev_noalloc: solve failed");
    return LOMA_ERR_DEVICE;
  }
  return LOMA_OK;
}

