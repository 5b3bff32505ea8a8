// Complex numbers in registers, compile-time loops and compile-time roots of unity for 64-wide CDNA wavefronts.
#pragma once
#include <hip/hip_runtime.h>
#include <utility>

namespace m2 {

struct cf {            // complex float; kept as two scalars so that nothing is forced into pairs
  float re, im;
};

// a b with its roundings said: of the two products of each sum the one with a.re goes into the sum unrounded.  Left to the compiler, which of
// them that was depended on where b came from (memory, or the thread's own transform), and with it the last bit of the result.
__device__ __forceinline__ cf cmul(cf a, cf b) {
  return {fmaf(a.re, b.re, -(a.im * b.im)), fmaf(a.re, b.im, a.im * b.re)};
}
__device__ __forceinline__ cf csquare(cf a) { return {fmaf(a.re, a.re, -(a.im * a.im)), (a.re + a.re) * a.im}; }

template <int I> using ic = std::integral_constant<int, I>;

template <int B, int E, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(ic<B>{});
    static_for<B + 1, E>(f);
  }
}

constexpr int bitrev(int v, int bits) {
  int r = 0;
  for (int i = 0; i < bits; ++i) r |= ((v >> i) & 1) << (bits - 1 - i);
  return r;
}
constexpr int ilog2(int v) { return v <= 1 ? 0 : 1 + ilog2(v >> 1); }

// cos and sin of 2 pi k / n in compile-time double precision: reduction to a quadrant in whole numbers, then the Taylor
// series (|x| <= pi / 2, terms to x^26: below 1e-19)
constexpr double cos_quadrant(double x) {
  double term = 1.0, sum = 1.0;
  for (int i = 1; i <= 13; ++i) {
    term *= -x * x / ((2 * i - 1) * (2 * i));
    sum += term;
  }
  return sum;
}
constexpr double root_cos64(long k, long n) {
  k = ((k % n) + n) % n;
  const long quadrant = 4 * k / n, rest = 4 * k - quadrant * n;      // angle = pi / 2 (quadrant + rest / n)
  const double half_pi = 1.57079632679489661923;
  // an angle and its distance to the next quadrant: the cosine of the one is the sine of the other
  const double c = rest == 0 ? 1.0 : cos_quadrant(half_pi * (double)rest / (double)n);
  const double s = rest == 0 ? 0.0 : cos_quadrant(half_pi * (double)(n - rest) / (double)n);
  return quadrant == 0 ? c : quadrant == 1 ? -s : quadrant == 2 ? -c : s;
}
constexpr double root_sin64(long k, long n) { return root_cos64(4 * k - n, 4 * n); }
constexpr float root_cos(long k, long n) { return (float)root_cos64(k, n); }
constexpr float root_sin(long k, long n) { return root_cos(4 * k - n, 4 * n); }

// v exp(-2 pi i K / N), or with CONJ v exp(+2 pi i K / N)
template <int K, int N, bool CONJ = false>
__device__ __forceinline__ cf mul_root(cf v) {
  constexpr int k = ((K % N) + N) % N;
  if constexpr (k == 0) {
    return v;
  } else {
    constexpr float c = root_cos(k, N), s = CONJ ? root_sin(k, N) : -root_sin(k, N);
    if constexpr (c == 0.f) return {-s * v.im, s * v.re};
    else if constexpr (s == 0.f) return {c * v.re, c * v.im};
    else return {c * v.re - s * v.im, c * v.im + s * v.re};
  }
}

// v exp(-2 pi i K / N), 0 <= K < N / 4, with its roundings said: of the two products of each sum the one with the smaller of cosine and sine
// (LARGE: with the larger one; where they are equal, with v.im) goes into the sum unrounded.
template <int K, int N, bool LARGE>
__device__ __forceinline__ cf mul_root_rounded(cf v) {
  static_assert(K >= 0 && 4 * K < N, "an angle of the first quadrant");
  if constexpr (K == 0) {
    return v;
  } else {
    constexpr float c = root_cos(K, N), s = root_sin(K, N);
    if constexpr (8 * K == N) return {fmaf(s, v.im, c * v.re), fmaf(c, v.im, -(s * v.re))};
    else if constexpr ((8 * K < N) == LARGE) return {fmaf(c, v.re, s * v.im), fmaf(c, v.im, -(s * v.re))};
    else return {fmaf(s, v.im, c * v.re), fmaf(-s, v.re, c * v.im)};
  }
}

}  // namespace m2
