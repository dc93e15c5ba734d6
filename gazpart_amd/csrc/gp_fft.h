// gp_fft.h -- FP64 complex transforms of one length in registers, for the
// DNS supplier's fused passes (gp_dns.hip).
//
// A line of N values belongs to T = N / E threads; thread t holds the E
// values t + T m (m = 0..E-1), before and after a transform, so a pass that
// works on transformed values (a projection, a curl, a product) runs on
// the registers of the transform and the next one starts from them.  A
// transform is the Stockham autosort form: passes of radix R | E, each on
// values that are N/R apart (always a thread's own), with an exchange
// through LDS between two passes and none after the last one.
#pragma once

#include <hip/hip_runtime.h>

namespace gpfft {

// E and the radices of the lengths that have a plan.  K = 0: kernels that
// hold one line, few passes (each exchange is a trip through LDS).  K = 1:
// kernels that hold three lines and their own work beside, fewer values a
// thread where the length allows, so that several wavefronts fit on a SIMD
// (256: 8 values leave room for one or two).
template <int N, int K> struct Plan { static constexpr bool ok = false; };
#define GP_FFT_PLAN(N_, K_, E_, ...)                                         \
  template <> struct Plan<N_, K_> {                                          \
    static constexpr bool ok = true;                                         \
    static constexpr int N = N_, E = E_, T = N_ / E_;                        \
    static constexpr int rad[7] = {__VA_ARGS__};                             \
  }
#define GP_FFT_BOTH(N_, E_, ...)                                             \
  GP_FFT_PLAN(N_, 0, E_, __VA_ARGS__);                                       \
  GP_FFT_PLAN(N_, 1, E_, __VA_ARGS__)
GP_FFT_PLAN(32, 0, 8, 8, 4);
GP_FFT_PLAN(32, 1, 4, 4, 4, 2);
GP_FFT_BOTH(48, 12, 12, 4);
GP_FFT_PLAN(64, 0, 8, 8, 8);
GP_FFT_PLAN(64, 1, 4, 4, 4, 4);
GP_FFT_BOTH(80, 10, 10, 2, 2, 2);
GP_FFT_BOTH(96, 12, 12, 4, 2);
GP_FFT_BOTH(100, 10, 10, 10);
GP_FFT_PLAN(128, 0, 8, 8, 4, 4);
GP_FFT_PLAN(128, 1, 4, 4, 4, 4, 2);
GP_FFT_BOTH(144, 12, 12, 12);
GP_FFT_BOTH(160, 10, 10, 2, 2, 2, 2);
GP_FFT_BOTH(192, 12, 12, 4, 4);
GP_FFT_PLAN(256, 0, 8, 8, 8, 4);
GP_FFT_PLAN(256, 1, 4, 4, 4, 4, 4);
GP_FFT_BOTH(320, 10, 10, 2, 2, 2, 2, 2);
GP_FFT_BOTH(384, 12, 12, 4, 4, 2);
GP_FFT_PLAN(512, 0, 8, 8, 8, 8);
GP_FFT_PLAN(512, 1, 4, 4, 4, 4, 4, 2);
#undef GP_FFT_BOTH
#undef GP_FFT_PLAN

__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return {a.x + b.x, a.y + b.y}; }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return {a.x - b.x, a.y - b.y}; }
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
// DIR i a
template <int DIR> __device__ __forceinline__ double2 rot(double2 a) {
  return DIR > 0 ? double2{-a.y, a.x} : double2{a.y, -a.x};
}

// cos of an angle in degrees, of the angles that radices 3, 5, 8, 10 and 12
// have, to the last bit (a constant that is one bit off is off in every
// transform of a run: 1e-14 after 40 steps)
constexpr double cos_deg(int d) {
  d = d % 360;
  if (d < 0) d += 360;
  if (d > 180) d = 360 - d;
  if (d > 90) return -cos_deg(180 - d);
  return d == 0    ? 1.0
         : d == 18 ? 0.95105651629515357212
         : d == 30 ? 0.86602540378443864676
         : d == 36 ? 0.80901699437494742410
         : d == 45 ? 0.70710678118654752440
         : d == 54 ? 0.58778525229247312917
         : d == 60 ? 0.5
         : d == 72 ? 0.30901699437494742410
                   : 0.0;   // 90
}
// cos and sin of 2 pi k / r, 360 k divisible by r
constexpr double cosk(int k, int r) { return cos_deg(360 * k / r); }
constexpr double sink(int k, int r) { return cos_deg(360 * k / r - 90); }

// R-point transforms of registers, in place, natural order
template <int R, int DIR> struct Dft;
template <int DIR> struct Dft<1, DIR> {
  static __device__ __forceinline__ void run(double2*) {}
};
template <int DIR> struct Dft<2, DIR> {
  static __device__ __forceinline__ void run(double2* a) {
    const double2 t = a[1];
    a[1] = csub(a[0], t);
    a[0] = cadd(a[0], t);
  }
};
template <int DIR> struct Dft<3, DIR> {
  static __device__ __forceinline__ void run(double2* a) {
    constexpr double s = sink(1, 3);
    const double2 p = cadd(a[1], a[2]), m = csub(a[1], a[2]);
    const double2 c = {a[0].x - 0.5 * p.x, a[0].y - 0.5 * p.y};
    const double2 d = rot<DIR>(double2{s * m.x, s * m.y});
    a[0] = cadd(a[0], p);
    a[1] = cadd(c, d);
    a[2] = csub(c, d);
  }
};
template <int DIR> struct Dft<4, DIR> {
  static __device__ __forceinline__ void run(double2* a) {
    const double2 s0 = cadd(a[0], a[2]), d0 = csub(a[0], a[2]);
    const double2 s1 = cadd(a[1], a[3]), d1 = rot<DIR>(csub(a[1], a[3]));
    a[0] = cadd(s0, s1);
    a[1] = cadd(d0, d1);
    a[2] = csub(s0, s1);
    a[3] = csub(d0, d1);
  }
};
template <int DIR> struct Dft<5, DIR> {
  static __device__ __forceinline__ void run(double2* a) {
    constexpr double c1 = cosk(1, 5), c2 = cosk(2, 5), s1 = sink(1, 5), s2 = sink(2, 5);
    const double2 p1 = cadd(a[1], a[4]), m1 = csub(a[1], a[4]);
    const double2 p2 = cadd(a[2], a[3]), m2 = csub(a[2], a[3]);
    const double2 u = {a[0].x + c1 * p1.x + c2 * p2.x, a[0].y + c1 * p1.y + c2 * p2.y};
    const double2 v = {a[0].x + c2 * p1.x + c1 * p2.x, a[0].y + c2 * p1.y + c1 * p2.y};
    const double2 e = rot<DIR>(double2{s1 * m1.x + s2 * m2.x, s1 * m1.y + s2 * m2.y});
    const double2 f = rot<DIR>(double2{s2 * m1.x - s1 * m2.x, s2 * m1.y - s1 * m2.y});
    a[0] = cadd(a[0], cadd(p1, p2));
    a[1] = cadd(u, e);
    a[4] = csub(u, e);
    a[2] = cadd(v, f);
    a[3] = csub(v, f);
  }
};
// A x B: A-point transforms of the values B apart, twiddles, B-point ones
template <int A, int B, int DIR> struct DftAB {
  template <int K1, int N2> static __device__ __forceinline__ double2 tw(double2 v) {
    constexpr int k = K1 * N2;
    if constexpr (k == 0) {
      return v;
    } else {
      constexpr double c = cosk(k, A * B), s = DIR * sink(k, A * B);
      return cmul(v, double2{c, s});
    }
  }
  template <int K1, int N2> static __device__ __forceinline__ void row(double2* x, const double2 (*y)[B]) {
    if constexpr (N2 < B) {
      x[N2] = tw<K1, N2>(y[K1][N2]);
      row<K1, N2 + 1>(x, y);
    }
  }
  template <int K1> static __device__ __forceinline__ void out(double2* a, const double2 (*y)[B]) {
    if constexpr (K1 < A) {
      double2 x[B];
      row<K1, 0>(x, y);
      Dft<B, DIR>::run(x);
#pragma unroll
      for (int k2 = 0; k2 < B; ++k2) a[K1 + A * k2] = x[k2];
      out<K1 + 1>(a, y);
    }
  }
  static __device__ __forceinline__ void run(double2* a) {
    double2 y[A][B];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
      double2 x[A];
#pragma unroll
      for (int n1 = 0; n1 < A; ++n1) x[n1] = a[n1 * B + n2];
      Dft<A, DIR>::run(x);
#pragma unroll
      for (int k1 = 0; k1 < A; ++k1) y[k1][n2] = x[k1];
    }
    out<0>(a, y);
  }
};
template <int DIR> struct Dft<8, DIR> : DftAB<2, 4, DIR> {};
template <int DIR> struct Dft<10, DIR> : DftAB<2, 5, DIR> {};
template <int DIR> struct Dft<12, DIR> : DftAB<3, 4, DIR> {};

// lines in the registers of a thread
template <int N, int K> using Lines = double2 (*)[Plan<N, K>::E];

// NC lines of length N in the registers of thread t of their T threads;
// tw[k] = exp(-2 pi i k / N).  DIR -1 forward, +1 backward, unnormalised.
// X exchanges: X::put(c, index, value), X::get(c, index), X::ready(c)
// between the puts and the gets of line c, X::again(c) before the puts of
// line c (after the gets of earlier ones).
template <int N, int K, int DIR, int NC, int P, int NS, typename X>
__device__ __forceinline__ void fft_pass(Lines<N, K> v, X& x, const double2* tw, int t) {
  using PL = Plan<N, K>;
  constexpr int E = PL::E, T = PL::T, R = PL::rad[P], B = E / R;
  static_assert(B * R == E, "radix divides the values of a thread");
#pragma unroll
  for (int b = 0; b < B; ++b) {
    double2 w[R];
    if constexpr (NS > 1) {
      // every factor from the table: powers formed by multiplication cost a
      // decimal digit over a run's transforms
      const int q = (t + T * b) % NS;
#pragma unroll
      for (int r = 1; r < R; ++r) {
        w[r] = tw[q * r * (N / (NS * R))];
        if (DIR > 0) w[r].y = -w[r].y;
      }
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      double2 a[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        a[r] = v[c][b + B * r];
        if constexpr (NS > 1) {
          if (r > 0) a[r] = cmul(a[r], w[r]);
        }
      }
      Dft<R, DIR>::run(a);
#pragma unroll
      for (int r = 0; r < R; ++r) v[c][b + B * r] = a[r];
    }
  }
  if constexpr (NS * R < N) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      x.again(c);
#pragma unroll
      for (int b = 0; b < B; ++b) {
        const int j = t + T * b, q = j % NS;
#pragma unroll
        for (int r = 0; r < R; ++r) x.put(c, (j / NS) * (NS * R) + q + r * NS, v[c][b + B * r]);
      }
      x.ready(c);
#pragma unroll
      for (int m = 0; m < E; ++m) v[c][m] = x.get(c, t + T * m);
    }
    fft_pass<N, K, DIR, NC, P + 1, NS * R>(v, x, tw, t);
  }
}
template <int N, int K, int DIR, int NC, typename X>
__device__ __forceinline__ void fft(Lines<N, K> v, X& x, const double2* tw, int t) {
  fft_pass<N, K, DIR, NC, 0, 1>(v, x, tw, t);
}

}  // namespace gpfft
