// gp_dns.hip -- the spectral DNS field supplier on the GPU: the reference's
// pseudo-spectral Navier-Stokes step (ADV_FLUID, adv_fluid.f90:78-234) with
// its rotational-form nonlinear term (NONLINEAR_TERMS, nonlinear_terms.f90:
// 96-206), divergence projection (PROJ_DIVFREE, proj_divfree.f90:46-60),
// smooth dealiasing filter (MESHING, meshing.f90:151-180), STEADY forcing
// (ADV_FORCING / ADD_FORCING3) and CHECK_CFL, in double precision.
//
// Layout: physical arrays [3][n][n][n] (x fastest, index (k n + j) n + i);
// spectral arrays [3][n][n][pitch] (the halved x axis fastest, as the
// reference's FSTART(1):FEND(1)), complex interleaved, n/2 + 1 of pitch
// columns used.  Transforms are unnormalised both ways as P3DFFT's; the
// forward result is multiplied by FACTOR = 1/n^3 inside the kernel that
// consumes it.
//
// A transform is three passes (x, y, z lines), each of them bound by memory,
// so the step's own work rides in the passes that hold the values anyway
// (gp_fft.h: a pass starts and ends with them in registers).  One ADV_FLUID,
// F being three fields read or written once:
//   k_fx_r2c     u -> A                                            2 F
//   k_fy         A, forward                                        2 F
//   k_fz ENTRY   forward z, U = A FACTOR, A = i k x U, backward z  3 F
//   k_fy         A, backward                                       2 F
//   k_fx_cross   backward x of A (vorticity), u x z, forward x     3 F
//   k_fy         A, forward                                        2 F
//   k_fz STAGE1  forward z; RHS = F + P(A FACTOR); Un = (U + dt/2 RHS) E,
//                V = (U + dt RHS) E; B = V, A = i k x V, backward z
//                of both                                           5 F
//   k_fy         A and B, backward                                 4 F
//   k_fx_cross   backward x of both, their product, forward x      3 F
//   k_fy         A, forward                                        2 F
//   k_fz STAGE2  forward z; RHS; U = Un + dt/2 RHS, projection, FILTER;
//                B = U, backward z                                 4 F
//   k_fy         B, backward                                       2 F
//   k_fx_c2r     B -> u                                            2 F
// 36 F in all, against 63 F for seven library transforms and separate
// element-wise kernels.  Measured, us a step, library transforms -> these
// passes: 32^3 121 -> 63, 48^3 187 -> 125, 64^3 184 -> 111, 80^3 239 -> 195, 96^3
// 378 -> 231, 100^3 415 -> 263, 128^3 691 -> 375, 144^3 1048 -> 714, 160^3 1291
// -> 1010, 192^3 2435 -> 1712, 256^3 6500 -> 3355 (36 F = 15.4 GB with the
// padding, 4.6 TB/s), 320^3 12524 -> 8717, 384^3 24650 -> 14490, 512^3 53460 ->
// 31100.  Error of the velocity against 80-bit arithmetic, rms: 64^3 after 40
// steps 8.4e-15 -> 6.8e-15, 128^3 after 16 6.5e-15 -> 2.4e-15, 256^3 after 3
// 1.4e-15 -> 7.9e-16.  (E = exp(-VISC |k|^2 DTIME), P the projection of
// NONLINEAR_TERMS's RHS assembly.)
//
// Lengths without a plan in gp_fft.h take rocFFT's batched transforms and
// one kernel for each element-wise step (pitch n/2 + 1):
//   u -> z (copy), R2C z -> U                       (entry transform)
//   k_scale_curl: U *= FACTOR, A = i k x U
//   C2R A -> z (vorticity), k_cross: z = u x z, EPS_FLU partials
//   R2C z -> A, k_stage1
//   C2R B -> u (stage velocity), C2R A -> z, k_cross, R2C z -> A
//   k_stage2, C2R B -> u
#include <hip/hip_runtime.h>
#include <rocfft/rocfft.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/gazpart_gpu.h"
#include "gp_fft.h"
#include "gp_xfer.h"

namespace gpdns {

constexpr int BLOCK = 256;
constexpr double ZERO_R = 1.0e-33;      // mod_dns_dim.f90:136
constexpr double INF_R = 1.0e33;        // mod_dns_dim.f90:137 INFINITY
constexpr double RTRUNC = 8.0 / 9.0;    // meshing.f90:38
constexpr int RED_BLOCKS = 1024;

struct Grid {
  int n, nh;            // n, n/2 + 1
  int pitch;            // columns of a spectral row in memory (nh or more)
  long long plane;      // values from one z plane to the next (n pitch or more)
  long long nr, nc;     // n^3, n plane
  double kf;            // KFIRST = 2 pi / L (init_run.f90:128)
  double klast;         // KLAST = pi / (L / n) (init_run.f90:129)
  double ikl2;          // 1 / KLAST^2
};

// wavenumbers of spectral element (i, j, k) (meshing.f90:96-121)
__device__ __forceinline__ void wavenum_at(const Grid& g, int i, int j, int k, double& kx,
                                           double& ky, double& kz) {
  kx = (double)i * g.kf;
  ky = (double)(j <= g.n / 2 ? j : j - g.n) * g.kf;
  kz = (double)(k <= g.n / 2 ? k : k - g.n) * g.kf;
}
// of element e of an array of pitch nh
__device__ __forceinline__ void wavenum(const Grid& g, long long e, double& kx, double& ky,
                                        double& kz) {
  const int i = (int)(e % g.nh);
  const long long r = e / g.nh;
  wavenum_at(g, i, (int)(r % g.n), (int)(r / g.n), kx, ky, kz);
}

// i k x U as nonlinear_terms.f90:104-112 forms it, term by term
__device__ __forceinline__ void curl(double kx, double ky, double kz, double2 u, double2 v,
                                     double2 w, double2& ox, double2& oy, double2& oz) {
  // (i a) k = (-a.y k, a.x k)
  ox.x = (-w.y * ky) - (-v.y * kz); ox.y = (w.x * ky) - (v.x * kz);
  oy.x = (-u.y * kz) - (-w.y * kx); oy.y = (u.x * kz) - (w.x * kx);
  oz.x = (-v.y * kx) - (-u.y * ky); oz.y = (v.x * kx) - (u.x * ky);
}

// RHS = F + P(T) (nonlinear_terms.f90:187-200): P = 1 - k k / |k|^2, and 0
// for the mean (the reference divides by INFINITY there).  One division a
// mode instead of nine quotients.
__device__ __forceinline__ void project_rhs(double kx, double ky, double kz, double2 t0,
                                            double2 t1, double2 t2, double2 f0, double2 f1,
                                            double2 f2, double2& r0, double2& r1, double2& r2) {
  const double k2 = kx * kx + ky * ky + kz * kz;
  const bool mean = k2 <= ZERO_R;
  const double q = mean ? 0.0 : 1.0 / k2, one = mean ? 0.0 : 1.0;
  const double dx = q * (kx * t0.x + ky * t1.x + kz * t2.x),
               dy = q * (kx * t0.y + ky * t1.y + kz * t2.y);
  r0.x = f0.x + (one * t0.x - kx * dx); r0.y = f0.y + (one * t0.y - kx * dy);
  r1.x = f1.x + (one * t1.x - ky * dx); r1.y = f1.y + (one * t1.y - ky * dy);
  r2.x = f2.x + (one * t2.x - kz * dx); r2.y = f2.y + (one * t2.y - kz * dy);
}

__device__ __forceinline__ double2 cmul(double2 a, double s) { return make_double2(a.x * s, a.y * s); }
__device__ __forceinline__ double2 cadd(double2 a, double2 b) {
  return make_double2(a.x + b.x, a.y + b.y);
}

// the forcing of mode e (fmap: -1 or its index among nf modes)
__device__ __forceinline__ void forcing_at(const int* fmap, const double2* fc, int nf, long long e,
                                           double2& f0, double2& f1, double2& f2) {
  f0 = f1 = f2 = make_double2(0.0, 0.0);
  if (!fmap) return;
  const int m = fmap[e];
  if (m < 0) return;
  f0 = fc[m]; f1 = fc[nf + m]; f2 = fc[2 * nf + m];
}

__global__ __launch_bounds__(BLOCK) void k_scale_curl(Grid g, double2* __restrict__ U,
                                                      double2* __restrict__ A, double factor) {
  for (long long e = (long long)blockIdx.x * BLOCK + threadIdx.x; e < g.nc;
       e += (long long)gridDim.x * BLOCK) {
    double kx, ky, kz;
    wavenum(g, e, kx, ky, kz);
    const double2 u = cmul(U[e], factor), v = cmul(U[g.nc + e], factor),
                  w = cmul(U[2 * g.nc + e], factor);
    U[e] = u; U[g.nc + e] = v; U[2 * g.nc + e] = w;
    double2 ox, oy, oz;
    curl(kx, ky, kz, u, v, w, ox, oy, oz);
    A[e] = ox; A[g.nc + e] = oy; A[2 * g.nc + e] = oz;
  }
}

// z = u x z (nonlinear_terms.f90:131-136); with part != nullptr also the
// sum of z^2 per workgroup (EPS_FLU, :124-128)
__global__ __launch_bounds__(BLOCK) void k_cross(Grid g, const double* __restrict__ u,
                                                 double* __restrict__ z, double* part) {
  __shared__ double s[BLOCK];
  double acc = 0.0;
  for (long long p = (long long)blockIdx.x * BLOCK + threadIdx.x; p < g.nr;
       p += (long long)gridDim.x * BLOCK) {
    const double ux = u[p], uy = u[g.nr + p], uz = u[2 * g.nr + p];
    const double zx = z[p], zy = z[g.nr + p], zz = z[2 * g.nr + p];
    if (part) acc += zx * zx + zy * zy + zz * zz;
    z[p] = uy * zz - uz * zy;
    z[g.nr + p] = uz * zx - ux * zz;
    z[2 * g.nr + p] = ux * zy - uy * zx;
  }
  if (!part) return;
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int w = BLOCK / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = s[0];
}

// first stage (adv_fluid.f90:113-131) and the curl of its result for the
// second stage's nonlinear term
__global__ __launch_bounds__(BLOCK) void k_stage1(Grid g, double2* __restrict__ A,
                                                  double2* __restrict__ U, double2* __restrict__ Un,
                                                  double2* __restrict__ B, double factor,
                                                  double visc, double dt, const int* fmap,
                                                  const double2* fc, int nf) {
  for (long long e = (long long)blockIdx.x * BLOCK + threadIdx.x; e < g.nc;
       e += (long long)gridDim.x * BLOCK) {
    double kx, ky, kz;
    wavenum(g, e, kx, ky, kz);
    double2 f0, f1, f2, r0, r1, r2;
    forcing_at(fmap, fc, nf, e, f0, f1, f2);
    project_rhs(kx, ky, kz, cmul(A[e], factor), cmul(A[g.nc + e], factor),
                cmul(A[2 * g.nc + e], factor), f0, f1, f2, r0, r1, r2);
    const double ef = exp(-visc * (kx * kx + ky * ky + kz * kz) * dt);
    const double h = dt / 2;
    const double2 rr[3] = {r0, r1, r2};
    double2 un[3];
    for (int c = 0; c < 3; ++c) {
      const double2 u0 = U[c * g.nc + e];
      Un[c * g.nc + e] = cmul(cadd(u0, cmul(rr[c], h)), ef);
      un[c] = cmul(cadd(u0, cmul(rr[c], dt)), ef);
      U[c * g.nc + e] = un[c];
      B[c * g.nc + e] = un[c];
    }
    double2 ox, oy, oz;
    curl(kx, ky, kz, un[0], un[1], un[2], ox, oy, oz);
    A[e] = ox; A[g.nc + e] = oy; A[2 * g.nc + e] = oz;
  }
}

// second stage's update of one mode (adv_fluid.f90:166-190): U = Un + dt/2
// RHS, PROJ_DIVFREE, FILTER
__device__ __forceinline__ void stage2_mode(const Grid& g, double kx, double ky, double kz,
                                            double dt, double2 r0, double2 r1, double2 r2,
                                            double2 n0, double2 n1, double2 n2, double2& u,
                                            double2& v, double2& w) {
  const double h = dt / 2;
  u = cadd(n0, cmul(r0, h));
  v = cadd(n1, cmul(r1, h));
  w = cadd(n2, cmul(r2, h));
  // PROJ_DIVFREE
  const double k2 = kx * kx + ky * ky + kz * kz;
  const double q = k2 <= ZERO_R ? 0.0 : 1.0 / k2;
  const double dx = q * (kx * u.x + ky * v.x + kz * w.x),
               dy = q * (kx * u.y + ky * v.y + kz * w.y);
  u.x -= kx * dx; u.y -= kx * dy;
  v.x -= ky * dx; v.y -= ky * dy;
  w.x -= kz * dx; w.y -= kz * dy;
  // FILTER, ALIASCONTROL = 2
  const double k2s = k2 * g.ikl2;
  double fl = 1.0;
  if (k2s > RTRUNC * RTRUNC && k2s <= 1.0) {
    const double c = cos((M_PI / 2.0) * (sqrt(k2s) - RTRUNC) / (1.0 - RTRUNC));
    fl = (c * c) * (c * c);
  } else if (k2s > 1.0) {
    fl = 0.0;
  }
  u = cmul(u, fl); v = cmul(v, fl); w = cmul(w, fl);
}

// second stage over all modes; B = U for the backward transform
__global__ __launch_bounds__(BLOCK) void k_stage2(Grid g, const double2* __restrict__ A,
                                                  double2* __restrict__ U,
                                                  const double2* __restrict__ Un,
                                                  double2* __restrict__ B, double factor,
                                                  double dt, const int* fmap, const double2* fc,
                                                  int nf) {
  for (long long e = (long long)blockIdx.x * BLOCK + threadIdx.x; e < g.nc;
       e += (long long)gridDim.x * BLOCK) {
    double kx, ky, kz;
    wavenum(g, e, kx, ky, kz);
    double2 f0, f1, f2, r0, r1, r2, u, v, w;
    forcing_at(fmap, fc, nf, e, f0, f1, f2);
    project_rhs(kx, ky, kz, cmul(A[e], factor), cmul(A[g.nc + e], factor),
                cmul(A[2 * g.nc + e], factor), f0, f1, f2, r0, r1, r2);
    stage2_mode(g, kx, ky, kz, dt, r0, r1, r2, Un[e], Un[g.nc + e], Un[2 * g.nc + e], u, v, w);
    U[e] = u; U[g.nc + e] = v; U[2 * g.nc + e] = w;
    B[e] = u; B[g.nc + e] = v; B[2 * g.nc + e] = w;
  }
}

__global__ __launch_bounds__(BLOCK) void k_curl(Grid g, const double2* __restrict__ U,
                                                double2* __restrict__ A) {
  for (long long e = (long long)blockIdx.x * BLOCK + threadIdx.x; e < g.nc;
       e += (long long)gridDim.x * BLOCK) {
    double kx, ky, kz;
    wavenum(g, e, kx, ky, kz);
    double2 ox, oy, oz;
    curl(kx, ky, kz, U[e], U[g.nc + e], U[2 * g.nc + e], ox, oy, oz);
    A[e] = ox; A[g.nc + e] = oy; A[2 * g.nc + e] = oz;
  }
}

// ---------------------------------------------------------------------------
// the fused passes (gp_fft.h).  What bounds them is memory: at 256^3 a pass
// over three fields moves 0.83 to 2.1 GB.  y and z lines are read in tiles of
// W neighbouring columns, so that every access is whole cache lines (rows are
// padded to a multiple of 8 columns, 128 bytes); x lines lie in rows and two
// real lines share one complex transform.
// ---------------------------------------------------------------------------
template <int N, int K> constexpr int tile_w() { return gpfft::Plan<N, K>::T >= 8 ? 8 : 16; }
template <int N, int K> constexpr int col_threads() { return gpfft::Plan<N, K>::T * tile_w<N, K>(); }

// exchange of a tile of columns through LDS, column fastest (eight lanes
// cover the 128 bytes that LDS moves a clock); two buffers in turn where
// they fit, so that one barrier an exchange is enough
template <int N, int K> struct ColX {
  static constexpr int W = tile_w<N, K>();
  static constexpr bool two = 2 * N * W * (int)sizeof(double2) <= 65536;
  static constexpr int elems = (two ? 2 : 1) * N * W;
  double2* s;
  int w;
  int turn = 0;
  __device__ __forceinline__ void again(int) {
    if (two) turn ^= 1;
    else __syncthreads();
  }
  __device__ __forceinline__ void ready(int) { __syncthreads(); }
  __device__ __forceinline__ void put(int, int i, double2 v) { s[(turn * N + i) * W + w] = v; }
  __device__ __forceinline__ double2 get(int, int i) { return s[(turn * N + i) * W + w]; }
};

// exchange of one row among its T threads, padded against bank conflicts;
// LDS serves a wavefront in order, so a row inside one wavefront needs no
// barrier
template <int N, int K> struct RowX {
  static constexpr int T = gpfft::Plan<N, K>::T;
  static constexpr bool wave = T <= 64 && 64 % T == 0;
  // rows of a workgroup: one wavefront where the grid has few rows
  static constexpr int G = N <= 128 && T <= 64 ? 64 / T : 256 / T;
  static constexpr int threads = G * T;
  static constexpr int elems = N + N / 8;
  double2* s;
  static __device__ __forceinline__ int at(int i) { return i + (i >> 3); }
  __device__ __forceinline__ void sync() {
    if (wave) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
      __syncthreads();
    }
  }
  __device__ __forceinline__ void again(int) { sync(); }
  __device__ __forceinline__ void ready(int) { sync(); }
  __device__ __forceinline__ void put(int, int i, double2 v) { s[at(i)] = v; }
  __device__ __forceinline__ double2 get(int, int i) { return s[at(i)]; }
};

// the value `off` bytes (the lane's part) from a pointer that is the same for
// the whole wavefront: one 32-bit register a lane for all the values of a
// thread, where 64-bit addresses took dozens (a field is below 4 GB)
template <typename T> __device__ __forceinline__ T& at_byte(T* base, unsigned off) {
  return *reinterpret_cast<T*>(
      reinterpret_cast<std::conditional_t<std::is_const_v<T>, const char*, char*>>(base) + off);
}

// the twiddle table in LDS, for kernels whose many transforms read it again
// and again
template <int N> __device__ __forceinline__ void stage_twiddles(double2* s, const double2* tw) {
  for (int k = threadIdx.x; k < N; k += blockDim.x) s[k] = tw[k];
  __syncthreads();
}

// y lines of gridDim.z fields, in place
template <int N, int DIR>
__global__ __launch_bounds__((col_threads<N, 0>())) void k_fy(double2* __restrict__ a, Grid g,
                                                         const double2* __restrict__ tw) {
  using PL = gpfft::Plan<N, 0>;
  constexpr int W = tile_w<N, 0>(), E = PL::E, T = PL::T;
  __shared__ double2 lds[ColX<N, 0>::elems];
  const int w = threadIdx.x % W, t = threadIdx.x / W;
  const int i = blockIdx.x * W + w;
  const bool on = i < g.nh;
  double2* p = a + blockIdx.z * g.nc + blockIdx.y * g.plane;
  const unsigned off = (unsigned)(t * g.pitch + i) * 16u;
  double2 v[1][E];
#pragma unroll
  for (int m = 0; m < E; ++m)
    v[0][m] = on ? at_byte(p + T * m * g.pitch, off) : double2{0.0, 0.0};
  ColX<N, 0> x{lds, w};
  gpfft::fft<N, 0, DIR, 1>(v, x, tw, t);
  if (on)
#pragma unroll
    for (int m = 0; m < E; ++m) at_byte(p + T * m * g.pitch, off) = v[0][m];
}

// z lines with the element-wise work on the modes between the forward and
// the backward transform.  ENTRY: A -> U, curl -> A; SPECTRAL: A -> U;
// CURL: U -> curl -> A; STAGE1: A, U -> Un, B, curl -> A; STAGE2: A, Un -> U,
// B.
enum { FZ_ENTRY, FZ_SPECTRAL, FZ_CURL, FZ_STAGE1, FZ_STAGE2 };

struct ZArgs {
  double2 *A, *B, *U, *Un;
  double factor, visc, dt;
  const int* fmap;
  const double2* fc;
  int nf;
};

// component c of i k x U as curl() forms it
__device__ __forceinline__ double2 curl_c(int c, double kx, double ky, double kz, double2 u,
                                          double2 v, double2 w) {
  double2 o[3];
  curl(kx, ky, kz, u, v, w, o[0], o[1], o[2]);
  return o[c];
}

template <int N, int MODE>
__global__ __launch_bounds__((col_threads<N, 1>())) void k_fz(ZArgs za, Grid g,
                                                         const double2* __restrict__ gtw) {
  using PL = gpfft::Plan<N, 1>;
  constexpr int W = tile_w<N, 1>(), E = PL::E, T = PL::T;
  __shared__ double2 lds[ColX<N, 1>::elems];
  __shared__ double2 tw[N];
  stage_twiddles<N>(tw, gtw);
  const int w = threadIdx.x % W, t = threadIdx.x / W;
  const int e = blockIdx.x * W + w;               // j pitch + i
  const int j = e / g.pitch, i = e - j * g.pitch;
  const bool on = i < g.nh;
  const unsigned off = ((unsigned)t * (unsigned)g.plane + (unsigned)e) * 16u;
  auto at = [&](auto* f, int c, int m) -> auto& {
    return at_byte(f + (c * g.nc + T * m * g.plane), off);
  };
  ColX<N, 1> x{lds, w};
  double2 v[3][E];
  const double2* in = MODE == FZ_CURL ? za.U : za.A;
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int m = 0; m < E; ++m) v[c][m] = on ? at(in, c, m) : double2{0.0, 0.0};
  if (MODE != FZ_CURL) gpfft::fft<N, 1, -1, 3>(v, x, tw, t);
#pragma unroll
  for (int m = 0; m < E; ++m) {
    const int k = t + T * m;
    double kx, ky, kz;
    wavenum_at(g, i, j, k, kx, ky, kz);
    if (MODE == FZ_ENTRY || MODE == FZ_SPECTRAL) {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        v[c][m] = cmul(v[c][m], za.factor);
        if (on) at(za.U, c, m) = v[c][m];
      }
    }
    if (MODE == FZ_STAGE1 || MODE == FZ_STAGE2) {
      double2 f0, f1, f2, r[3];
      f0 = f1 = f2 = make_double2(0.0, 0.0);
      if (on) forcing_at(za.fmap, za.fc, za.nf, ((long long)k * N + j) * g.nh + i, f0, f1, f2);
      project_rhs(kx, ky, kz, cmul(v[0][m], za.factor), cmul(v[1][m], za.factor),
                  cmul(v[2][m], za.factor), f0, f1, f2, r[0], r[1], r[2]);
      if (MODE == FZ_STAGE1) {
        // adv_fluid.f90:113-131
        const double ef = exp(-za.visc * (kx * kx + ky * ky + kz * kz) * za.dt);
        const double h = za.dt / 2;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const double2 u0 = on ? at(za.U, c, m) : double2{0.0, 0.0};
          if (on) at(za.Un, c, m) = cmul(cadd(u0, cmul(r[c], h)), ef);
          v[c][m] = cmul(cadd(u0, cmul(r[c], za.dt)), ef);
        }
      } else {
        double2 n[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) n[c] = on ? at(za.Un, c, m) : double2{0.0, 0.0};
        stage2_mode(g, kx, ky, kz, za.dt, r[0], r[1], r[2], n[0], n[1], n[2], v[0][m], v[1][m],
                    v[2][m]);
        if (on)
#pragma unroll
          for (int c = 0; c < 3; ++c) at(za.U, c, m) = v[c][m];
      }
    }
    // one value's loads and divisions at a time: spread over all of them
    // they take the registers of a second wavefront
    __builtin_amdgcn_sched_barrier(0);
  }
  if (MODE == FZ_SPECTRAL) return;
  if (MODE == FZ_STAGE1 || MODE == FZ_STAGE2) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      double2 b[1][E];
#pragma unroll
      for (int m = 0; m < E; ++m) b[0][m] = v[c][m];
      gpfft::fft<N, 1, 1, 1>(b, x, tw, t);
      if (on)
#pragma unroll
        for (int m = 0; m < E; ++m) at(za.B, c, m) = b[0][m];
    }
  }
  if (MODE != FZ_STAGE2) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      double2 b[1][E];
#pragma unroll
      for (int m = 0; m < E; ++m) {
        double kx, ky, kz;
        wavenum_at(g, i, j, t + T * m, kx, ky, kz);
        b[0][m] = curl_c(c, kx, ky, kz, v[0][m], v[1][m], v[2][m]);
      }
      gpfft::fft<N, 1, 1, 1>(b, x, tw, t);
      if (on)
#pragma unroll
        for (int m = 0; m < E; ++m) at(za.A, c, m) = b[0][m];
    }
  }
}

// the complex line whose backward transform has the real lines of the half
// spectra a and b as its parts (as a complex-to-real transform does, the
// imaginary parts of the first and the last column count for nothing); row:
// the byte offset of the thread's row in both
template <int N, int K>
__device__ __forceinline__ void load_pair(const double2* __restrict__ a,
                                          const double2* __restrict__ b, unsigned row, bool on,
                                          int t, double2* v) {
  using PL = gpfft::Plan<N, K>;
#pragma unroll
  for (int m = 0; m < PL::E; ++m) {
    const int e = t + PL::T * m;
    const unsigned q = row + 16u * (unsigned)(e <= N / 2 ? e : N - e);
    const double2 p = on ? at_byte(a, q) : double2{0.0, 0.0},
                  r = on ? at_byte(b, q) : double2{0.0, 0.0};
    if (e == 0 || e == N / 2) v[m] = {p.x, r.x};
    else if (e < N / 2) v[m] = {p.x - r.y, p.y + r.x};
    else v[m] = {p.x + r.y, r.x - p.y};
  }
}

// the half spectra of the two real lines whose pair was transformed
template <int N, int K>
__device__ __forceinline__ void store_pair(RowX<N, K>& x, const double2* v, bool on, int t,
                                           double2* __restrict__ a, double2* __restrict__ b,
                                           unsigned row) {
  using PL = gpfft::Plan<N, K>;
  x.again(0);
#pragma unroll
  for (int m = 0; m < PL::E; ++m) x.put(0, t + PL::T * m, v[m]);
  x.ready(0);
  if (!on) return;
#pragma unroll
  for (int m = 0; m < PL::E / 2; ++m) {
    const int e = t + PL::T * m;
    const double2 z = x.get(0, e), y = x.get(0, e ? N - e : 0);
    at_byte(a, row + 16u * e) = {0.5 * (z.x + y.x), 0.5 * (z.y - y.y)};
    at_byte(b, row + 16u * e) = {0.5 * (z.y + y.y), 0.5 * (y.x - z.x)};
  }
  if (t == 0) {
    const double2 z = x.get(0, N / 2);
    at_byte(a, row + 8u * N) = {z.x, 0.0};
    at_byte(b, row + 8u * N) = {z.y, 0.0};
  }
}

// the row pair of a thread: rows 2 pr and 2 pr + 1 of the n^2 rows of a field
// (n is even: both in one plane)
template <int N, int K> struct RowOf {
  int t, gr;
  long long pr;
  bool on;
  __device__ __forceinline__ RowOf()
      : t(threadIdx.x % RowX<N, K>::T), gr(threadIdx.x / RowX<N, K>::T),
        pr((long long)blockIdx.x * RowX<N, K>::G + threadIdx.x / RowX<N, K>::T),
        on(pr < (long long)N * N / 2) {}
  // the first row's place in a spectral field, in bytes
  __device__ __forceinline__ unsigned at(const Grid& g) const {
    const unsigned k = (unsigned)(pr / (N / 2)), j = 2u * (unsigned)(pr % (N / 2));
    return (k * (unsigned)g.plane + j * (unsigned)g.pitch) * 16u;
  }
  // and value e of it in a physical one
  __device__ __forceinline__ unsigned real(int e) const { return ((unsigned)pr * 2u * N + e) * 8u; }
};

template <int N>
__global__ __launch_bounds__((RowX<N, 0>::threads)) void k_fx_r2c(const double* __restrict__ u,
                                                             double2* __restrict__ A, Grid g,
                                                             const double2* __restrict__ tw) {
  using PL = gpfft::Plan<N, 0>;
  __shared__ double2 lds[RowX<N, 0>::G * RowX<N, 0>::elems];
  const RowOf<N, 0> ro;
  RowX<N, 0> x{lds + ro.gr * RowX<N, 0>::elems};
#pragma unroll 1
  for (int c = 0; c < 3; ++c) {
    const double* p = u + c * g.nr;
    double2 v[1][PL::E];
#pragma unroll
    for (int m = 0; m < PL::E; ++m) {
      const unsigned q = ro.real(ro.t + PL::T * m);
      v[0][m] = ro.on ? double2{at_byte(p, q), at_byte(p + N, q)} : double2{0.0, 0.0};
    }
    gpfft::fft<N, 0, -1, 1>(v, x, tw, ro.t);
    double2* r = A + c * g.nc;
    store_pair<N, 0>(x, v[0], ro.on, ro.t, r, r + g.pitch, ro.at(g));
  }
}

template <int N>
__global__ __launch_bounds__((RowX<N, 0>::threads)) void k_fx_c2r(const double2* __restrict__ B,
                                                             double* __restrict__ u, Grid g,
                                                             const double2* __restrict__ tw) {
  using PL = gpfft::Plan<N, 0>;
  __shared__ double2 lds[RowX<N, 0>::G * RowX<N, 0>::elems];
  const RowOf<N, 0> ro;
  RowX<N, 0> x{lds + ro.gr * RowX<N, 0>::elems};
#pragma unroll 1
  for (int c = 0; c < 3; ++c) {
    const double2* r = B + c * g.nc;
    double2 v[1][PL::E];
    load_pair<N, 0>(r, r + g.pitch, ro.at(g), ro.on, ro.t, v[0]);
    gpfft::fft<N, 0, 1, 1>(v, x, tw, ro.t);
    double* p = u + c * g.nr;
    if (ro.on)
#pragma unroll
      for (int m = 0; m < PL::E; ++m) {
        const unsigned q = ro.real(ro.t + PL::T * m);
        at_byte(p, q) = v[0][m].x;
        at_byte(p + N, q) = v[0][m].y;
      }
  }
}

// u x vorticity of a row pair (nonlinear_terms.f90:131-136) between the
// backward and the forward x transforms.  FIRST: the velocity is u, and the
// squares of the vorticity are summed per workgroup (EPS_FLU, :124-128);
// else the velocity is B's.
template <int N, bool FIRST>
__global__ __launch_bounds__((RowX<N, 1>::threads)) void k_fx_cross(const double* __restrict__ u,
                                                               const double2* __restrict__ B,
                                                               double2* __restrict__ A, Grid g,
                                                               const double2* __restrict__ gtw,
                                                               double* __restrict__ part) {
  using PL = gpfft::Plan<N, 1>;
  constexpr int E = PL::E;
  __shared__ double2 tw[N];
  stage_twiddles<N>(tw, gtw);
  __shared__ double2 lds[RowX<N, 1>::G * RowX<N, 1>::elems];
  __shared__ double red[FIRST ? RowX<N, 1>::threads : 1];
  const RowOf<N, 1> ro;
  RowX<N, 1> x{lds + ro.gr * RowX<N, 1>::elems};
  const unsigned r0 = ro.at(g);
  double2 v[3][E];
  if (FIRST) {
#pragma unroll
    for (int c = 0; c < 3; ++c)
      load_pair<N, 1>(A + c * g.nc, A + c * g.nc + g.pitch, r0, ro.on, ro.t, v[c]);
#pragma unroll
    for (int c = 0; c < 3; ++c)
      gpfft::fft<N, 1, 1, 1>(&v[c], x, tw, ro.t);
    double acc = 0.0;
#pragma unroll
    for (int m = 0; m < E; ++m) {
      const unsigned q = ro.real(ro.t + PL::T * m);
      double a[3], b[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        a[c] = ro.on ? at_byte(u + c * g.nr, q) : 0.0;
        b[c] = ro.on ? at_byte(u + c * g.nr + N, q) : 0.0;
      }
      const double2 zx = v[0][m], zy = v[1][m], zz = v[2][m];
      acc += zx.x * zx.x + zy.x * zy.x + zz.x * zz.x;
      acc += zx.y * zx.y + zy.y * zy.y + zz.y * zz.y;
      v[0][m] = {a[1] * zz.x - a[2] * zy.x, b[1] * zz.y - b[2] * zy.y};
      v[1][m] = {a[2] * zx.x - a[0] * zz.x, b[2] * zx.y - b[0] * zz.y};
      v[2][m] = {a[0] * zy.x - a[1] * zx.x, b[0] * zy.y - b[1] * zx.y};
    }
    red[threadIdx.x] = acc;   // rows out of range hold zeros
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {   // at most 256 threads
      if ((int)threadIdx.x < h && (int)threadIdx.x + h < RowX<N, 1>::threads)
        red[threadIdx.x] += red[threadIdx.x + h];
      __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
  } else {
    // A pair of lines is always two rows of one quantity: the rounding of a
    // transform goes by the larger of its two parts, and velocity and
    // vorticity differ by the wavenumber, that is, by the unit of length
    double2 p[3][E];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      load_pair<N, 1>(B + c * g.nc, B + c * g.nc + g.pitch, r0, ro.on, ro.t, p[c]);
      gpfft::fft<N, 1, 1, 1>(&p[c], x, tw, ro.t);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      load_pair<N, 1>(A + c * g.nc, A + c * g.nc + g.pitch, r0, ro.on, ro.t, v[c]);
      gpfft::fft<N, 1, 1, 1>(&v[c], x, tw, ro.t);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int m = 0; m < E; ++m) {
      const double2 zx = v[0][m], zy = v[1][m], zz = v[2][m];
      v[0][m] = {p[1][m].x * zz.x - p[2][m].x * zy.x, p[1][m].y * zz.y - p[2][m].y * zy.y};
      v[1][m] = {p[2][m].x * zx.x - p[0][m].x * zz.x, p[2][m].y * zx.y - p[0][m].y * zz.y};
      v[2][m] = {p[0][m].x * zy.x - p[1][m].x * zx.x, p[0][m].y * zy.y - p[1][m].y * zx.y};
    }
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    gpfft::fft<N, 1, -1, 1>(&v[c], x, tw, ro.t);
    store_pair<N, 1>(x, v[c], ro.on, ro.t, A + c * g.nc, A + c * g.nc + g.pitch, r0);
  }
}

// the sum of n partials in a fixed order, one workgroup
__global__ __launch_bounds__(BLOCK) void k_sum(const double* __restrict__ part, int n,
                                               double* __restrict__ out) {
  __shared__ double s[BLOCK];
  double acc = 0.0;
  for (int p = threadIdx.x; p < n; p += BLOCK) acc += part[p];
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int h = BLOCK / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) s[threadIdx.x] += s[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = s[0];
}

// per-workgroup max |a| of the three components
__global__ __launch_bounds__(BLOCK) void k_absmax3(Grid g, const double* __restrict__ u,
                                                   double* part) {
  __shared__ double s[3][BLOCK];
  double m[3] = {0.0, 0.0, 0.0};
  for (long long p = (long long)blockIdx.x * BLOCK + threadIdx.x; p < g.nr;
       p += (long long)gridDim.x * BLOCK)
    for (int c = 0; c < 3; ++c) m[c] = fmax(m[c], fabs(u[c * g.nr + p]));
  for (int c = 0; c < 3; ++c) s[c][threadIdx.x] = m[c];
  __syncthreads();
  for (int w = BLOCK / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w)
      for (int c = 0; c < 3; ++c) s[c][threadIdx.x] = fmax(s[c][threadIdx.x], s[c][threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0)
    for (int c = 0; c < 3; ++c) part[3 * blockIdx.x + c] = s[c][0];
}

// ---------------------------------------------------------------------------
// the reference's RAN1 (Park-Miller minimal standard, Schrage's method,
// Bays-Durham shuffle of 32) and GAUSS (polar Box-Muller, one value kept),
// adv_forcing.f90:130-215, as a host-side generator
// ---------------------------------------------------------------------------
struct Ran1 {
  static constexpr int IA = 16807, IM = 2147483647, IQ = 127773, IR = 2836, NTAB = 32;
  int iv[NTAB] = {};
  int iy = 0;
  int iset = 0;
  double gset = 0.0;
  int idum = 0;
  static int lcg(int x) {
    const int k = x / IQ;
    x = IA * (x - k * IQ) - IR * k;
    return x < 0 ? x + IM : x;
  }
  double ran1() {
    const int ndiv = 1 + (IM - 1) / NTAB;
    const double am = 1.0 / IM, rnmx = 1.0 - 1.2e-7;
    if (idum <= 0 || iy == 0) {
      idum = std::max(-idum, 1);
      for (int j = NTAB + 8; j >= 1; --j) {
        idum = lcg(idum);
        if (j <= NTAB) iv[j - 1] = idum;
      }
      iy = iv[0];
    }
    idum = lcg(idum);
    const int j = iy / ndiv;
    iy = iv[j];
    iv[j] = idum;
    return std::min(am * iy, rnmx);
  }
  double gauss() {
    if (iset != 0) {
      iset = 0;
      return gset;
    }
    double v1, v2, rsq;
    do {
      v1 = 2.0 * ran1() - 1.0;
      v2 = 2.0 * ran1() - 1.0;
      rsq = v1 * v1 + v2 * v2;
    } while (!(rsq < 1.0 && rsq != 0.0));
    const double fac = std::sqrt(-2.0 * std::log(rsq) / rsq);
    gset = v1 * fac;
    iset = 1;
    return v2 * fac;
  }
};

}  // namespace gpdns

using namespace gpdns;

// the forcing of several steps goes to the device at once: at most FORCE_STEPS,
// and FORCE_BYTES of amplitudes unless one step has more (a band of all modes:
// 3 GB at 512^3)
constexpr int FORCE_STEPS = 16;
constexpr size_t FORCE_BYTES = (size_t)4 << 20;

struct gp_dns {
  gp_dns_params prm{};
  Grid g{};
  hipStream_t st = nullptr;
  double* u = nullptr;     // [3][nr] velocity
  double* z = nullptr;     // [3][nr] vorticity / u x omega / copies
  double2* U = nullptr;    // [3][nc]
  double2* Un = nullptr;   // [3][nc] first-stage U_NP1
  double2* A = nullptr;    // [3][nc] curl / transformed products
  double2* B = nullptr;    // [3][nc] backward-transform inputs
  double* part = nullptr;  // reduction partials (and, last, their sum)
  int npart = 0;
  double2* tw = nullptr;   // exp(-2 pi i k / n), lengths with a plan; else null
  rocfft_plan fwd = nullptr, bwd = nullptr;
  rocfft_execution_info info = nullptr;
  void* work = nullptr;
  gpx::Xfer xf;            // transfers with the caller's memory
  bool have_u = false;
  double eps = 0.0;
  // forcing: modes in the reference's loop order, amplitudes (host), the
  // dense mode map and the amplitudes on the device
  std::vector<long long> fmode;
  std::vector<double> fkf;
  std::vector<double> famp;    // [3][nf][2]
  int* fmap = nullptr;
  int fsteps = FORCE_STEPS;    // steps whose forcing goes to the device at once
  double2* fdev = nullptr;     // their amplitudes
  double* fpin = nullptr;      // and their page-locked staging
  Ran1 rng;
  std::string err;
};

namespace {

#define DCHK(call)                                                        \
  do {                                                                    \
    hipError_t e_ = (call);                                               \
    if (e_ != hipSuccess) {                                               \
      d->err = std::string(#call " failed: ") + hipGetErrorString(e_);    \
      return GP_ERR_HIP;                                                  \
    }                                                                     \
  } while (0)

#define FCHK(call)                                                        \
  do {                                                                    \
    rocfft_status s_ = (call);                                            \
    if (s_ != rocfft_status_success) {                                    \
      d->err = std::string(#call " failed with rocfft status ") +        \
               std::to_string((int)s_);                                   \
      return GP_ERR_HIP;                                                  \
    }                                                                     \
  } while (0)

unsigned grid_of(long long n) {
  const long long b = (n + BLOCK - 1) / BLOCK;
  return (unsigned)std::min<long long>(b, 65536);
}

int r2c(gp_dns* d, double* in, double2* out) {
  void* ib[1] = {in};
  void* ob[1] = {out};
  FCHK(rocfft_execute(d->fwd, ib, ob, d->info));
  return GP_OK;
}

int c2r(gp_dns* d, double2* in, double* out) {
  void* ib[1] = {in};
  void* ob[1] = {out};
  FCHK(rocfft_execute(d->bwd, ib, ob, d->info));
  return GP_OK;
}

// ADV_FORCING (adv_forcing.f90:33-125) on the host for the next ns steps (it
// depends on nothing but its own sequence): one copy to the device for all
// of them.  The stream is idle here (gp_dns_step).

int advance_forcing(gp_dns* d, int ns) {
  const int nf = (int)d->fmode.size();
  if (!d->prm.forcing || nf == 0) return GP_OK;
  const double dt = d->prm.dtime;
  const double alpha = dt / d->prm.time_force;
  const double beta = std::pow(2.0 * d->prm.sigma_force * d->prm.sigma_force * dt /
                                   d->prm.time_force, 0.5);
  const double kmax = d->prm.kforce_max;
  for (int s = 0; s < ns; ++s) {
    for (int m = 0; m < nf; ++m) {
      const double xampf = (kmax - d->fkf[m]) / 0.20 / kmax;
      const double xampl = (std::exp(2.0 * xampf) - 1.0) / (std::exp(2.0 * xampf) + 1.0);
      for (int c = 0; c < 3; ++c) {
        double* a = d->famp.data() + ((size_t)c * nf + m) * 2;
        double xe = d->rng.gauss() * xampl;
        const double re = a[0] * (1.0 - alpha) + xe * beta;
        xe = d->rng.gauss() * xampl;
        const double im = a[1] * (1.0 - alpha) + xe * beta;
        a[0] = re;
        a[1] = im;
      }
    }
    std::copy(d->famp.begin(), d->famp.end(), d->fpin + (size_t)s * d->famp.size());
  }
  DCHK(hipMemcpyAsync(d->fdev, d->fpin, (size_t)ns * d->famp.size() * sizeof(double),
                      hipMemcpyHostToDevice, d->st));
  return GP_OK;
}

// the passes of one length
template <int N> struct Passes {
  template <int DIR> static void y(gp_dns* d, double2* a, int fields) {
    hipLaunchKernelGGL((k_fy<N, DIR>), dim3((d->g.nh + tile_w<N, 0>() - 1) / tile_w<N, 0>(), N, fields),
                       dim3(col_threads<N, 0>()), 0, d->st, a, d->g, (const double2*)d->tw);
  }
  template <int MODE> static void z(gp_dns* d, const int* fmap, const double2* fc) {
    ZArgs za{d->A, d->B, d->U, d->Un, 1.0 / (double)d->g.nr, d->prm.visc, d->prm.dtime,
             fmap, fc, (int)d->fmode.size()};
    hipLaunchKernelGGL((k_fz<N, MODE>), dim3((unsigned)(N * d->g.pitch / tile_w<N, 1>())),
                       dim3(col_threads<N, 1>()), 0, d->st, za, d->g, (const double2*)d->tw);
  }
  template <int K> static unsigned rows() {
    return (unsigned)((N * N / 2 + RowX<N, K>::G - 1) / RowX<N, K>::G);
  }
  static void r2c(gp_dns* d, const double* u) {
    hipLaunchKernelGGL((k_fx_r2c<N>), dim3(rows<0>()), dim3(RowX<N, 0>::threads), 0, d->st, u, d->A,
                       d->g, (const double2*)d->tw);
  }
  static void c2r(gp_dns* d, const double2* a, double* u) {
    hipLaunchKernelGGL((k_fx_c2r<N>), dim3(rows<0>()), dim3(RowX<N, 0>::threads), 0, d->st, a, u, d->g,
                       (const double2*)d->tw);
  }
  template <bool FIRST> static void cross(gp_dns* d) {
    hipLaunchKernelGGL((k_fx_cross<N, FIRST>), dim3(rows<1>()), dim3(RowX<N, 1>::threads), 0, d->st,
                       (const double*)d->u, (const double2*)d->B, d->A, d->g,
                       (const double2*)d->tw, d->part);
  }
  static void step(gp_dns* d, const int* fmap, const double2* fc) {
    if (d->prm.reuse_spectral) {
      z<FZ_CURL>(d, nullptr, nullptr);
    } else {
      r2c(d, d->u);
      y<-1>(d, d->A, 3);
      z<FZ_ENTRY>(d, nullptr, nullptr);
    }
    y<1>(d, d->A, 3);
    cross<true>(d);
    y<-1>(d, d->A, 3);
    z<FZ_STAGE1>(d, fmap, fc);
    y<1>(d, d->A, 6);   // A and B, which follows it
    cross<false>(d);
    y<-1>(d, d->A, 3);
    z<FZ_STAGE2>(d, fmap, fc);
    y<1>(d, d->B, 3);
    c2r(d, d->B, d->u);
  }
  // U from u
  static void spectral(gp_dns* d) {
    r2c(d, d->u);
    y<-1>(d, d->A, 3);
    z<FZ_SPECTRAL>(d, nullptr, nullptr);
  }
  // z = curl of U, in physical space
  static void vorticity(gp_dns* d) {
    z<FZ_CURL>(d, nullptr, nullptr);
    y<1>(d, d->A, 3);
    c2r(d, d->A, d->z);
  }
};

// f(Passes<n>) for the lengths that have a plan; false for the others
template <typename F> bool with_passes(int n, F&& f) {
  switch (n) {
#define GP_LEN(N_) case N_: f(Passes<N_>{}); return true;
    GP_LEN(32) GP_LEN(48) GP_LEN(64) GP_LEN(80) GP_LEN(96) GP_LEN(100) GP_LEN(128) GP_LEN(144)
    GP_LEN(160) GP_LEN(192) GP_LEN(256) GP_LEN(320) GP_LEN(384) GP_LEN(512)
#undef GP_LEN
  }
  return false;
}

// one ADV_FLUID (asynchronous); fc: its forcing amplitudes
int one_step(gp_dns* d, const double2* fc) {
  const Grid& g = d->g;
  const double factor = 1.0 / (double)g.nr;
  const int nf = (int)d->fmode.size();
  const int* fmap = (d->prm.forcing && nf) ? d->fmap : nullptr;
  if (d->tw) {
    with_passes(g.n, [&](auto ps) { ps.step(d, fmap, fc); });
    DCHK(hipGetLastError());
    return GP_OK;
  }
  const unsigned gc = grid_of(g.nc), gr = grid_of(g.nr);
  int rc;
  if (d->prm.reuse_spectral) {
    // U is the spectral state u came from (set_velocity or the last step)
    hipLaunchKernelGGL(k_curl, dim3(gc), dim3(BLOCK), 0, d->st, g, (const double2*)d->U, d->A);
  } else {
    // entry transform of the velocity (adv_fluid.f90:86-94); u is kept
    DCHK(hipMemcpyAsync(d->z, d->u, 3 * g.nr * sizeof(double), hipMemcpyDeviceToDevice, d->st));
    if ((rc = r2c(d, d->z, d->U))) return rc;
    hipLaunchKernelGGL(k_scale_curl, dim3(gc), dim3(BLOCK), 0, d->st, g, d->U, d->A, factor);
  }
  // stage 1
  if ((rc = c2r(d, d->A, d->z))) return rc;
  hipLaunchKernelGGL(k_cross, dim3(RED_BLOCKS), dim3(BLOCK), 0, d->st, g, (const double*)d->u,
                     d->z, d->part);
  if ((rc = r2c(d, d->z, d->A))) return rc;
  hipLaunchKernelGGL(k_stage1, dim3(gc), dim3(BLOCK), 0, d->st, g, d->A, d->U, d->Un, d->B,
                     factor, d->prm.visc, d->prm.dtime, fmap, fc, nf);
  // stage 2
  if ((rc = c2r(d, d->B, d->u))) return rc;
  if ((rc = c2r(d, d->A, d->z))) return rc;
  hipLaunchKernelGGL(k_cross, dim3(gr), dim3(BLOCK), 0, d->st, g, (const double*)d->u, d->z,
                     (double*)nullptr);
  if ((rc = r2c(d, d->z, d->A))) return rc;
  hipLaunchKernelGGL(k_stage2, dim3(gc), dim3(BLOCK), 0, d->st, g, (const double2*)d->A, d->U,
                     (const double2*)d->Un, d->B, factor, d->prm.dtime, fmap, fc, nf);
  if ((rc = c2r(d, d->B, d->u))) return rc;
  DCHK(hipGetLastError());
  return GP_OK;
}

// EPS_FLU = VISC * sum(zeta^2) of the last step's first stage (waits for it)
int read_eps(gp_dns* d) {
  double s = 0.0;
  double* out = d->part + d->npart;
  hipLaunchKernelGGL(k_sum, dim3(1), dim3(BLOCK), 0, d->st, (const double*)d->part, d->npart, out);
  DCHK(hipGetLastError());
  DCHK(hipMemcpyAsync(&s, out, sizeof(double), hipMemcpyDeviceToHost, d->st));
  DCHK(hipStreamSynchronize(d->st));
  d->eps = d->prm.visc * s;
  return GP_OK;
}

}  // namespace

extern "C" {

int gp_dns_create(const gp_dns_params* p, gp_dns** out) {
  if (!p || !out) return GP_ERR_ARG;
  *out = nullptr;
  if (p->n < 4 || p->n % 2 || p->n > 2048 || !(p->L > 0) || !(p->visc >= 0) ||
      !(p->dtime > 0))
    return GP_ERR_ARG;
  if (p->forcing && !(p->time_force > 0 && p->kforce_max > 0)) return GP_ERR_ARG;
  gp_dns* d = new gp_dns();
  d->prm = *p;
  Grid& g = d->g;
  g.n = p->n;
  g.nh = p->n / 2 + 1;
  g.nr = (long long)p->n * p->n * p->n;
  const bool own = with_passes(p->n, [](auto) {});
  g.pitch = own ? (g.nh + 7) / 8 * 8 : g.nh;
  // planes 256 bytes apart from a power of two times the row: the z lines of
  // a tile then spread over the memory channels (256^3: STAGE1 608 -> 589 us)
  g.plane = (long long)p->n * g.pitch + (own ? 16 : 0);
  g.nc = p->n * g.plane;
  g.kf = 2.0 * M_PI / p->L;
  g.klast = M_PI / (p->L / p->n);
  g.ikl2 = 1.0 / (g.klast * g.klast);
  auto fail = [&](int rc) {
    gp_dns_destroy(d);
    return rc;
  };
  if (hipStreamCreate(&d->st) != hipSuccess) return fail(GP_ERR_HIP);
  const size_t rb = 3 * (size_t)g.nr * sizeof(double), cb = 3 * (size_t)g.nc * sizeof(double2);
  // partials of the vorticity's squares: one a workgroup of the first product
  d->npart = RED_BLOCKS;
  with_passes(g.n, [&](auto ps) { d->npart = (int)ps.template rows<1>(); });
  const size_t np = std::max<size_t>((size_t)d->npart + 1, 3 * RED_BLOCKS);
  if (hipMalloc((void**)&d->u, rb) != hipSuccess || hipMalloc((void**)&d->z, rb) != hipSuccess ||
      hipMalloc((void**)&d->U, cb) != hipSuccess || hipMalloc((void**)&d->Un, cb) != hipSuccess ||
      hipMalloc((void**)&d->A, 2 * cb) != hipSuccess ||
      hipMalloc((void**)&d->part, np * sizeof(double)) != hipSuccess)
    return fail(GP_ERR_NOMEM);
  d->B = d->A + 3 * g.nc;   // one array of six fields: k_fy takes both at once
  if (own) {
    std::vector<double2> tw((size_t)g.n);
    for (int k = 0; k < g.n; ++k) {
      const long double a = 2.0L * acosl(-1.0L) * (long double)k / (long double)g.n;
      tw[(size_t)k] = make_double2((double)cosl(a), (double)-sinl(a));
    }
    if (hipMalloc((void**)&d->tw, tw.size() * sizeof(double2)) != hipSuccess)
      return fail(GP_ERR_NOMEM);
    if (hipMemcpy(d->tw, tw.data(), tw.size() * sizeof(double2), hipMemcpyHostToDevice) !=
        hipSuccess)
      return fail(GP_ERR_HIP);
  } else {
    if (rocfft_setup() != rocfft_status_success) return fail(GP_ERR_HIP);
    const size_t len[3] = {(size_t)g.n, (size_t)g.n, (size_t)g.n};
    if (rocfft_plan_create(&d->fwd, rocfft_placement_notinplace, rocfft_transform_type_real_forward,
                           rocfft_precision_double, 3, len, 3, nullptr) != rocfft_status_success ||
        rocfft_plan_create(&d->bwd, rocfft_placement_notinplace, rocfft_transform_type_real_inverse,
                           rocfft_precision_double, 3, len, 3, nullptr) != rocfft_status_success)
      return fail(GP_ERR_HIP);
    size_t w1 = 0, w2 = 0;
    rocfft_plan_get_work_buffer_size(d->fwd, &w1);
    rocfft_plan_get_work_buffer_size(d->bwd, &w2);
    const size_t wb = std::max(w1, w2);
    if (rocfft_execution_info_create(&d->info) != rocfft_status_success) return fail(GP_ERR_HIP);
    if (wb) {
      if (hipMalloc(&d->work, wb) != hipSuccess) return fail(GP_ERR_NOMEM);
      if (rocfft_execution_info_set_work_buffer(d->info, d->work, wb) != rocfft_status_success)
        return fail(GP_ERR_HIP);
    }
    if (rocfft_execution_info_set_stream(d->info, d->st) != rocfft_status_success)
      return fail(GP_ERR_HIP);
  }
  // forcing modes in the order of adv_forcing.f90:45-62 (K, J, I)
  if (p->forcing) {
    const size_t nm = (size_t)g.n * g.n * g.nh;
    std::vector<int> map(nm, -1);
    for (int k = 0; k < g.n; ++k)
      for (int j = 0; j < g.n; ++j)
        for (int i = 0; i < g.nh; ++i) {
          const double kx = i * g.kf, ky = (j <= g.n / 2 ? j : j - g.n) * g.kf,
                       kz = (k <= g.n / 2 ? k : k - g.n) * g.kf;
          const double kfm = std::pow(kx * kx + ky * ky + kz * kz, 0.5);
          if (kfm >= p->kforce_min && kfm <= p->kforce_max) {
            const long long e = ((long long)k * g.n + j) * g.nh + i;
            map[(size_t)e] = (int)d->fmode.size();
            d->fmode.push_back(e);
            d->fkf.push_back(kfm);
          }
        }
    const size_t nf = d->fmode.size();
    d->famp.assign(3 * nf * 2, 0.0);   // INITIATION_FORCING_NEW: F = 0
    d->rng.idum = p->seed;
    const size_t one = std::max<size_t>(3 * nf, 1) * sizeof(double2);
    d->fsteps = (int)std::min<size_t>(FORCE_STEPS, std::max<size_t>(FORCE_BYTES / one, 1));
    const size_t fb = one * (size_t)d->fsteps;
    if (hipMalloc((void**)&d->fmap, nm * sizeof(int)) != hipSuccess ||
        hipMalloc((void**)&d->fdev, fb) != hipSuccess ||
        hipHostMalloc((void**)&d->fpin, fb) != hipSuccess)
      return fail(GP_ERR_NOMEM);
    if (hipMemcpy(d->fmap, map.data(), map.size() * sizeof(int), hipMemcpyHostToDevice) !=
            hipSuccess ||
        hipMemset(d->fdev, 0, fb) != hipSuccess)
      return fail(GP_ERR_HIP);
  }
  *out = d;
  return GP_OK;
}

int gp_dns_destroy(gp_dns* d) {
  if (!d) return GP_ERR_ARG;
  if (d->st) hipStreamSynchronize(d->st);
  if (d->fwd) rocfft_plan_destroy(d->fwd);
  if (d->bwd) rocfft_plan_destroy(d->bwd);
  if (d->info) rocfft_execution_info_destroy(d->info);
  void* bufs[] = {d->u, d->z, d->U, d->Un, d->A, d->part, d->tw, d->work, d->fmap, d->fdev};
  for (void* b : bufs)
    if (b) hipFree(b);
  if (d->fpin) hipHostFree(d->fpin);
  d->xf.release();
  if (d->st) hipStreamDestroy(d->st);
  delete d;
  return GP_OK;
}

const char* gp_dns_error_string(const gp_dns* d) { return d ? d->err.c_str() : "null handle"; }

int gp_dns_set_velocity(gp_dns* d, const double* uvw) {
  if (!d || !uvw) return GP_ERR_ARG;
  DCHK(d->xf.h2d(d->u, uvw, 3 * (size_t)d->g.nr * sizeof(double), d->st));
  // the spectral state of this velocity (for gp_dns_get_vorticity / bind)
  if (d->tw) {
    with_passes(d->g.n, [&](auto ps) { ps.spectral(d); });
  } else {
    DCHK(hipMemcpyAsync(d->z, d->u, 3 * d->g.nr * sizeof(double), hipMemcpyDeviceToDevice, d->st));
    int rc;
    if ((rc = r2c(d, d->z, d->U))) return rc;
    hipLaunchKernelGGL(k_scale_curl, dim3(grid_of(d->g.nc)), dim3(BLOCK), 0, d->st, d->g, d->U,
                       d->A, 1.0 / (double)d->g.nr);
  }
  DCHK(hipGetLastError());
  DCHK(hipStreamSynchronize(d->st));
  d->have_u = true;
  return GP_OK;
}

int gp_dns_get_velocity(gp_dns* d, double* uvw) {
  if (!d || !uvw) return GP_ERR_ARG;
  if (!d->have_u) {
    d->err = "no velocity (gp_dns_set_velocity)";
    return GP_ERR_STATE;
  }
  DCHK(d->xf.d2h(uvw, d->u, 3 * (size_t)d->g.nr * sizeof(double), d->st));
  return GP_OK;
}

static int vorticity_dev(gp_dns* d) {
  // i k x U -> z (z is free between steps)
  if (d->tw) {
    with_passes(d->g.n, [&](auto ps) { ps.vorticity(d); });
    DCHK(hipGetLastError());
    return GP_OK;
  }
  hipLaunchKernelGGL(k_curl, dim3(grid_of(d->g.nc)), dim3(BLOCK), 0, d->st, d->g,
                     (const double2*)d->U, d->A);
  DCHK(hipGetLastError());
  return c2r(d, d->A, d->z);
}

int gp_dns_get_vorticity(gp_dns* d, double* w) {
  if (!d || !w) return GP_ERR_ARG;
  if (!d->have_u) {
    d->err = "no velocity (gp_dns_set_velocity)";
    return GP_ERR_STATE;
  }
  int rc;
  if ((rc = vorticity_dev(d))) return rc;
  DCHK(d->xf.d2h(w, d->z, 3 * (size_t)d->g.nr * sizeof(double), d->st));
  return GP_OK;
}

int gp_dns_step(gp_dns* d, int nsteps) {
  if (!d || nsteps < 0) return GP_ERR_ARG;
  if (!d->have_u) {
    d->err = "no velocity (gp_dns_set_velocity)";
    return GP_ERR_STATE;
  }
  // in turns of fsteps steps
  for (int s0 = 0; s0 < nsteps; s0 += d->fsteps) {
    const int ns = std::min(d->fsteps, nsteps - s0);
    int rc = advance_forcing(d, ns);
    for (int s = 0; s < ns && !rc; ++s)
      rc = one_step(d, d->fdev ? d->fdev + 3 * (size_t)s * d->fmode.size() : nullptr);
    if (!rc && s0 + ns >= nsteps) rc = read_eps(d);
    if (rc) return rc;
    // the staging of the next turn's forcing
    if (d->prm.forcing) DCHK(hipStreamSynchronize(d->st));
  }
  return GP_OK;
}

static int absmax(gp_dns* d, double m[3]) {
  hipLaunchKernelGGL(k_absmax3, dim3(RED_BLOCKS), dim3(BLOCK), 0, d->st, d->g,
                     (const double*)d->u, d->part);
  DCHK(hipGetLastError());
  std::vector<double> h(3 * RED_BLOCKS);
  DCHK(hipMemcpyAsync(h.data(), d->part, h.size() * sizeof(double), hipMemcpyDeviceToHost,
                      d->st));
  DCHK(hipStreamSynchronize(d->st));
  m[0] = m[1] = m[2] = 0.0;
  for (int b = 0; b < RED_BLOCKS; ++b)
    for (int c = 0; c < 3; ++c) m[c] = std::max(m[c], h[3 * b + c]);
  return GP_OK;
}

int gp_dns_cfl(gp_dns* d, double dtime_user, double* dtime) {
  if (!d) return GP_ERR_ARG;
  if (!d->have_u) {
    d->err = "no velocity (gp_dns_set_velocity)";
    return GP_ERR_STATE;
  }
  double m[3];
  int rc;
  if ((rc = absmax(d, m))) return rc;
  // check_cfl.f90:61-92 with DX = DY = DZ = L / (n - 1) (meshing.f90:45-47)
  const double dx = d->prm.L / (double)(d->g.n - 1);
  double dtc = INF_R;
  for (int c = 0; c < 3; ++c) dtc = std::min(dtc, m[c] > ZERO_R ? 0.05 * dx / m[c] : INF_R);
  const double dtf = std::min(INF_R, 1.0 * dx * dx / d->prm.visc);
  d->prm.dtime = std::min(std::min(dtc, dtf), dtime_user);
  if (dtime) *dtime = d->prm.dtime;
  return GP_OK;
}

int gp_dns_info(gp_dns* d, double* eps, double* umax3, int* nforce) {
  if (!d) return GP_ERR_ARG;
  if (eps) *eps = d->eps;
  if (nforce) *nforce = (int)d->fmode.size();
  if (umax3) {
    if (!d->have_u) {
      d->err = "no velocity (gp_dns_set_velocity)";
      return GP_ERR_STATE;
    }
    return absmax(d, umax3);
  }
  return GP_OK;
}

int gp_dns_bind(gp_dns* d, gp_ctx* ctx, int mesh_vorticity) {
  if (!d || !ctx) return GP_ERR_ARG;
  if (!d->have_u) {
    d->err = "no velocity (gp_dns_set_velocity)";
    return GP_ERR_STATE;
  }
  int rc;
  if ((rc = vorticity_dev(d))) return rc;
  const double vs = mesh_vorticity ? (double)(d->g.n - 1) / (double)d->g.n : 1.0;
  DCHK(hipStreamSynchronize(d->st));
  const int rc2 = gp_bind_field_planar(ctx, d->g.n, d->u, d->z, vs);
  if (rc2) d->err = gp_last_error_string(ctx);
  return rc2;
}

}  // extern "C"
