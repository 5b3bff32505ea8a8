// The transform engine of the long convolutions.
//
// A causal-plus-anticausal convolution of a real signal s (L samples) with a 2L-tap window k is a product of polynomials
// modulo z^2L - 1 of which the first L coefficients are wanted.  Write k = lo + z^L hi.  Modulo z^L + i, where z^L = -i,
//
//     s (lo + i hi)  =  (low half of s lo + high half of s hi)  +  i (...)
//
// and the real part is the answer: ONE complex transform of L points per signal, evaluated at the roots of z^L = -i, that is
// at exp(-2 pi i (k + 1/4) / L), a pointwise product with the transform of lo + i hi, and the real part of the inverse.
// Against the transform of 2L points of two signals packed as a + i u (which this took over from) the product needs no pairs of
// mirrored frequencies, the first pass starts from real numbers, the last one ends in them, and a signal that waits takes 32
// registers instead of 64.  At L = 32768 the ring splits once more, z^L + i = (z^H - r)(z^H + r) with H = L / 2, r^2 = -i: two
// transforms of H points at exp(-2 pi i (k + s) / H), s = 1/8 and 5/8.
//
// Butterflies.  A transform at shift s splits like the ring itself: z^2h - w^2 = (z^h - w)(z^h + w), so that every butterfly is
// (a, b) -> (a + w b, a - w b) with a factor w that belongs to the block and not to the position in it: four fused multiply-adds
// for the sum and two for the difference (2 a - sum), and no multiplication by twiddles between the passes.  A radix-R pass needs
// R / 2 different factors, all of them powers of one root times constants.  The inverse runs the transform without shift back
// (factors belong to the position) with the same butterfly and removes the shift at the end, where only the real part is formed.
// A row is three passes, R1 at stride H / R1, R2 at stride R3 and R3 on contiguous groups, or two (R2 = 1); forward leaves
// bit-reversed registers in natural slots, so the spectra lie in whatever order the last pass leaves them in.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fft_regs.h"
#include "m2_internal.h"

namespace m2 {

template <int LOGH_, int R1_, int R2_, int R3_, int E_>
struct TwistPlan {
  static constexpr int LOGH = LOGH_, H = 1 << LOGH_, R1 = R1_, R2 = R2_, R3 = R3_;
  static constexpr int E = E_;                     // points per thread
  static constexpr int T = H / E;                  // threads per transform
  static constexpr int S1 = H / R1;                // stride of the first pass; of the second: R3
  static constexpr int NB1 = E / R1, NB2 = E / R2, NG = E / R3;
  static constexpr bool THREE = R2 > 1;
  // LDS padding in complex slots.  Two passes: one slot after every group, so that the groups of consecutive lanes start in
  // consecutive banks; a row ends where the next one's lanes use the banks it leaves free (T lanes of 8 bytes).  Three passes: one
  // slot after every 16 and one more after every 256, the least conflicts by counter among the paddings that keep offsets linear.
  __host__ __device__ static constexpr int phys(int p) { return THREE ? p + (p >> 4) + (p >> 8) : p + p / R3; }
  static constexpr int kRaw = THREE ? H + (H >> 4) + (H >> 8) : H + H / R3;
  static constexpr int ROW = THREE || T >= 32 ? kRaw : kRaw + ((T - kRaw) % 32 + 32) % 32;
  // Tables of factors in LDS, two slots of padding behind each row.  Three passes: of the second, R2 / 2 factors per block (forward)
  // and per position (inverse).  Two passes: of the last forward one, R3 / 2 per group, and of the last inverse one, R1 / 2 per position.
  static constexpr int FR = THREE ? R2 : R3, IR = THREE ? R2 : R1;      // radices
  static constexpr int FS = FR / 2 + 2, IS = IR / 2 + 2;                // slots per row
  static constexpr int TAB = R1 * FS + R3 * IS;
  static_assert(R1 * R2 * R3 == H && E % R1 == 0 && E % R2 == 0 && E % R3 == 0, "radices");
  static_assert(!THREE || R3 == 16, "padding");
};

// phys(base + o) == phys(base) + phys(o) for every (base, offset) pair of the three passes, and every slot inside the row
template <class P>
constexpr bool twist_offsets_ok() {
  for (int q = 0; q < P::S1; ++q)
    for (int j = 0; j < P::R1; ++j)
      if (P::phys(q + j * P::S1) != P::phys(q) + P::phys(j * P::S1)) return false;
  if (P::THREE)
    for (int b = 0; b < P::R1; ++b)
      for (int m = 0; m < P::R3; ++m)
        for (int j = 0; j < P::R2; ++j)
          if (P::phys(b * P::S1 + m + j * P::R3) != P::phys(b * P::S1 + m) + P::phys(j * P::R3)) return false;
  for (int g = 0; g < P::H / P::R3; ++g)
    for (int j = 0; j < P::R3; ++j)
      if (P::phys(P::R3 * g + j) != P::phys(P::R3 * g) + j) return false;
  return P::phys(P::H - 1) < P::ROW;
}

__device__ __forceinline__ cf lds_get(const float2* p, int off) {
  const float2 v = p[off];
  return {v.x, v.y};
}
__device__ __forceinline__ void lds_put(float2* p, int off, cf v) { p[off] = make_float2(v.re, v.im); }

// exp(-2 pi i m / n), n a power of two
__device__ __forceinline__ cf unit_root(int m, int n) {
  float s, c;
  sincospif(2.0f * (float)m / (float)n, &s, &c);
  return {c, -s};
}

// Synchronisation of N consecutive threads (aligned runs, N a power of two).  Up to 64 lie inside one wavefront: its LDS
// instructions execute in program order, so a later read by any lane sees an earlier write by any other lane and only the
// compiler has to be kept from reordering them.  More need the workgroup barrier, across which the scheduler is not to move code
// either: the phases on its two sides each fit the register budget, a merged schedule of both does not.
template <int N>
__device__ __forceinline__ void sync_threads() {
  if constexpr (N <= 64) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  } else {
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
  }
}

// The thread's number, to the compiler another value each time: what is formed from it is formed anew and not kept in registers across
// the passes, which would spill it.
__device__ __forceinline__ int anew(int t) {
  asm volatile("" : "+v"(t));
  return t;
}

// ------------------------------------------------------------------------------------------
// radix-R transforms in registers.  The factor of stage S (blocks of R / 2^S), number e < max(1, 2^(S-1)), at shift sigma is
// exp(-i pi (sigma + e) / 2^S); the other half of a stage's factors are these times -i.
// ------------------------------------------------------------------------------------------
// (a, b) <- (a + w b, a - w b), w or conj(w), times -i (conj: i) with ROT
template <bool CONJ, bool ROT>
__device__ __forceinline__ void butterfly(cf& a, cf& b, cf w) {
  const float wr = ROT ? w.im : w.re, wi = (ROT ? -w.re : w.im) * (CONJ ? -1.f : 1.f);
  const cf s = {fmaf(-wi, b.im, fmaf(wr, b.re, a.re)), fmaf(wi, b.re, fmaf(wr, b.im, a.im))};
  b = {fmaf(2.f, a.re, -s.re), fmaf(2.f, a.im, -s.im)};
  a = s;
}
// the same with w = exp(-2 pi i K / N), or its conjugate
template <bool CONJ, int K, int N>
__device__ __forceinline__ void butterfly_const(cf& a, cf& b) {
  constexpr int k = ((K % N) + N) % N;
  if constexpr (k == 0 || 4 * k == N) {
    const cf v = k == 0 ? b : CONJ ? cf{-b.im, b.re} : cf{b.im, -b.re};
    b = {a.re - v.re, a.im - v.im};
    a = {a.re + v.re, a.im + v.im};
  } else {
    butterfly<CONJ, false>(a, b, cf{root_cos(k, N), -root_sin(k, N)});
  }
}

// Registers of a finished butterfly are handed on at once (`out(register)`, in BASE .. BASE + R - 1), so that their LDS stores leave
// while the rest of the last stage is computed: the scheduler would collect them behind it.  The barriers keep it from that.
struct KeepAll {
  template <class R>
  __device__ __forceinline__ void operator()(R) const {}
};
template <bool LAST, int A, int B, bool HOLD, class OUT>
__device__ __forceinline__ void hand_on(OUT&& out) {
  if constexpr (LAST && !std::is_same<std::decay_t<OUT>, KeepAll>::value) {
    out(ic<A>{});
    out(ic<B>{});
    if constexpr (HOLD) __builtin_amdgcn_sched_barrier(0);
  }
}

// forward, shift S8 / 8 known at compile time: natural order in, bit-reversed out.  REAL: the imaginary parts of the input are zero
// and not read.
template <int R, int BASE, int S8, bool REAL, int NREG, class OUT>
__device__ __forceinline__ void fwd_const(cf (&x)[NREG], OUT&& out) {
  static_for<0, ilog2(R)>([&](auto ss) {
    constexpr int S = decltype(ss)::value, h = R >> (S + 1);
    static_for<0, (1 << S)>([&](auto bb) {
      constexpr int b = decltype(bb)::value, k = S8 + 8 * bitrev(b, S), n = 16 << S, at = BASE + 2 * h * b;
      static_for<0, h>([&](auto jj) {
        constexpr int j = decltype(jj)::value;
        if constexpr (REAL && S == 0) {
          const float p = x[at + j].re, q = x[at + h + j].re, im = -root_sin(k, n) * q;
          x[at + j] = {fmaf(root_cos(k, n), q, p), im};
          x[at + h + j] = {fmaf(-root_cos(k, n), q, p), -im};
        } else {
          butterfly_const<false, k, n>(x[at + j], x[at + h + j]);
        }
        hand_on<S + 1 == ilog2(R), at + j, at + h + j, (b & 1) == 1>(out);
      });
    });
  });
}
// forward with factors w(stage, number)
template <int R, int BASE, int NREG, class W, class OUT>
__device__ __forceinline__ void fwd_factors(cf (&x)[NREG], W&& w, OUT&& out) {
  static_for<0, ilog2(R)>([&](auto ss) {
    constexpr int S = decltype(ss)::value, h = R >> (S + 1);
    static_for<0, (S > 0 ? 1 << (S - 1) : 1)>([&](auto bb) {
      constexpr int b = decltype(bb)::value;
      const cf f = w(ss, ic<bitrev(b, S > 0 ? S - 1 : 0)>{});
      static_for<0, h>([&](auto jj) {
        constexpr int at = BASE + 4 * h * b + decltype(jj)::value;
        butterfly<false, false>(x[at], x[at + h], f);
        if constexpr (S > 0) butterfly<false, true>(x[at + 2 * h], x[at + 3 * h], f);
        hand_on<S + 1 == ilog2(R), at, at + h, false>(out);
        if constexpr (S > 0) hand_on<S + 1 == ilog2(R), at + 2 * h, at + 3 * h, true>(out);
      });
    });
  });
}
// inverse without shift: bit-reversed in, natural out, unscaled
template <int R, int BASE, int NREG, class OUT>
__device__ __forceinline__ void inv_plain(cf (&x)[NREG], OUT&& out) {
  static_for<0, ilog2(R)>([&](auto ss) {
    constexpr int S = decltype(ss)::value, h = 1 << S;
    static_for<0, R / (2 * h)>([&](auto bb) {
      static_for<0, h>([&](auto jj) {
        constexpr int j = decltype(jj)::value, at = BASE + 2 * h * decltype(bb)::value + j;
        butterfly_const<true, j, 2 * h>(x[at], x[at + h]);
        hand_on<2 * h == R, at, at + h, (j & 1) == 1>(out);
      });
    });
  });
}
// inverse of inputs that are to be multiplied by powers of exp(2 pi i sigma / R): conjugates of the factors at shift sigma
template <int R, int BASE, int NREG, class W, class OUT>
__device__ __forceinline__ void inv_factors(cf (&x)[NREG], W&& w, OUT&& out) {
  static_for<0, ilog2(R)>([&](auto ss) {
    constexpr int S = decltype(ss)::value, h = 1 << S;
    static_for<0, (S > 0 ? h / 2 : 1)>([&](auto jj) {
      constexpr int j = decltype(jj)::value;
      const cf f = w(ss, jj);
      static_for<0, R / (2 * h)>([&](auto bb) {
        constexpr int at = BASE + 2 * h * decltype(bb)::value + j;
        butterfly<true, false>(x[at], x[at + h], f);
        if constexpr (S > 0) butterfly<true, true>(x[at + h / 2], x[at + h + h / 2], f);
        hand_on<2 * h == R, at, at + h, false>(out);
        if constexpr (S > 0) hand_on<2 * h == R, at + h / 2, at + h + h / 2, true>(out);
      });
    });
  });
}

// All factors of a radix-R pass from two of them held in registers, those with e = 0 of the last stage and of the last but two:
// the others are squares of these (one or two steps) and constant multiples.  Their roundings are said, and with them the last bit of what is
// transformed: filters' spectra (LARGE, mul_root_rounded) come out the same from the kernel that stores them and in a core that makes its own.
template <int R>
struct Factors {
  cf fine, mid;
  // sigma = num / den, powers of two
  __device__ __forceinline__ void init(int num, int den) {
    fine = unit_root(num, den * R);
    mid = unit_root(num, den * (R / 4));
  }
  template <bool LARGE, class F>
  __device__ __forceinline__ void use(F&& body) const {
    constexpr int last = ilog2(R) - 1;
    cf f = fine, m = mid;
    asm volatile("" : "+v"(f.re), "+v"(f.im), "+v"(m.re), "+v"(m.im));     // rebuilt where used: no long-lived registers
    cf t[last + 1];
    t[last] = f;
    t[last - 1] = csquare(f);
    t[last - 2] = m;
    if constexpr (last > 2) t[last - 3] = csquare(m);
    if constexpr (last > 3) t[last - 4] = csquare(t[last - 3]);
    body([&](auto ss, auto ee) __attribute__((always_inline)) {
      return mul_root_rounded<decltype(ee)::value, (2 << decltype(ss)::value), LARGE>(t[decltype(ss)::value]);
    });
  }
};

// What a thread keeps for its transforms at shift S8 / 8 (nothing with two passes, which have tables)
template <class P, int S8>
struct TwistForward {            // of the last forward pass: group k1 R2 + k2 holds the frequencies k1 + R1 k2 (mod R1 R2)
  Factors<P::R3> last[P::NG];
  __device__ __forceinline__ void init(int t) {
    if constexpr (P::THREE)
      static_for<0, P::NG>([&](auto ii) {
        const int g = t + P::T * decltype(ii)::value;
        last[decltype(ii)::value].init(8 * (g / P::R2 + P::R1 * (g % P::R2)) + S8, 8 * P::R1 * P::R2);
      });
  }
  template <int I>
  __device__ __forceinline__ const Factors<P::R3>& group() const { return last[I]; }
};
template <class P>
struct TwistInverse {            // of the last inverse pass
  Factors<P::R1> first[P::NB1];
  __device__ __forceinline__ void init(int t) {
    if constexpr (P::THREE)
      static_for<0, P::NB1>([&](auto ii) { first[decltype(ii)::value].init(t + P::T * decltype(ii)::value, P::S1); });
  }
};
template <class P, int S8>
struct TwistEnd {                // exp(2 pi i q S8 / 8H): with constants, the removal of the shift
  cf f[P::NB1];
  __device__ __forceinline__ void init(int t) {
    static_for<0, P::NB1>([&](auto ii) {
      const cf w = unit_root((t + P::T * decltype(ii)::value) * S8, 8 * P::H);
      f[decltype(ii)::value] = {w.re, -w.im};
    });
  }
};

// the tables, by all threads of the workgroup; a barrier has to follow
template <class P, int S8>
__device__ __forceinline__ void tables_init(float2* tab) {
  constexpr int fwd = P::FR / 2, inv = P::IR / 2;
  for (int i = threadIdx.x; i < P::R1 * fwd + P::R3 * inv; i += blockDim.x) {
    const bool f = i < P::R1 * fwd;
    const int r = f ? i / fwd : (i - P::R1 * fwd) / inv, n = f ? i % fwd : (i - P::R1 * fwd) % inv;
    const int S = n == 0 ? 0 : 32 - __builtin_clz(n), e = n == 0 ? 0 : n - (1 << (S - 1));       // factor n: stage and number
    // forward row r: sigma = (r + S8 / 8) / R1; inverse row r: sigma = r / R3
    const cf w = f ? unit_root(8 * r + S8 + e * 8 * P::R1, 16 * P::R1 << S) : unit_root(r + e * P::R3, 2 * P::R3 << S);
    tab[f ? r * P::FS + n : P::R1 * P::FS + r * P::IS + n] = make_float2(w.re, w.im);
  }
}
// the factors of one row of the tables, read ahead of their use: all of them, or with R = 32 (no registers for sixteen beside the
// points) the last stage's eight behind the first three stages
template <int R>
struct TableRow {
  static constexpr int kFirst = R / 2 < 8 ? R / 2 : 8;
  cf f[R / 2];
  const float2* tab;
  __device__ __forceinline__ void load(const float2* p) {
    tab = p;
    static_for<0, kFirst>([&](auto nn) { f[decltype(nn)::value] = lds_get(tab, decltype(nn)::value); });
  }
  template <class S, class E>
  __device__ __forceinline__ cf operator()(S, E) {
    if constexpr (R == 32 && S::value == 3 && E::value == 0) {
      __builtin_amdgcn_sched_barrier(0);
      static_for<kFirst, R / 2>([&](auto nn) { f[decltype(nn)::value] = lds_get(tab, decltype(nn)::value); });
    }
    return f[S::value == 0 ? 0 : (1 << (S::value - 1)) + E::value];
  }
};

// ------------------------------------------------------------------------------------------
// passes over a row in LDS; thread t of T.  First-pass layout: register i R1 + j <-> position t + T i + S1 j
// ------------------------------------------------------------------------------------------
template <class P, int S8, bool REAL>
__device__ __forceinline__ void fwd_first(cf (&x)[P::E], int t, float2* row) {
  static_for<0, P::NB1>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    float2* pb = row + P::phys(t + P::T * i);
    fwd_const<P::R1, i * P::R1, S8, REAL>(x, [&](auto rr) __attribute__((always_inline)) {
      constexpr int r = decltype(rr)::value;
      lds_put(pb, P::phys(bitrev(r % P::R1, ilog2(P::R1)) * P::S1), x[r]);
    });
  });
}
// second pass: all of a thread's inputs are requested before the first of its butterflies
template <class P, bool INV>
__device__ __forceinline__ void second(cf (&x)[P::E], int t, float2* row, const float2* tab) {
  constexpr int R = P::R2, bits = ilog2(R);
  auto base = [&](int i) __attribute__((always_inline)) {
    const int q = t + P::T * i;
    return row + P::phys(q / P::R3 * P::S1 + q % P::R3);
  };
  static_for<0, P::NB2>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    const float2* pb = base(i);
    static_for<0, R>([&](auto rr) {
      constexpr int r = decltype(rr)::value;      // forward: natural, inverse: bit-reversed registers
      x[i * R + r] = lds_get(pb, P::phys((INV ? bitrev(r, bits) : r) * P::R3));
    });
  });
  static_for<0, P::NB2>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    const int q = t + P::T * i;
    float2* pb = base(i);
    TableRow<R> w;
    w.load(tab + (INV ? P::R1 * P::FS + q % P::R3 * P::IS : q / P::R3 * P::FS));
    auto put = [&](auto rr) __attribute__((always_inline)) {
      constexpr int r = decltype(rr)::value, at = r % R;
      lds_put(pb, P::phys((INV ? at : bitrev(at, bits)) * P::R3), x[r]);
    };
    if constexpr (INV) inv_factors<R, i * R>(x, w, put);
    else fwd_factors<R, i * R>(x, w, put);
  });
}
// last pass: group I of the thread
template <class P, int I>
__device__ __forceinline__ void load_group(cf (&x)[P::E], int t, const float2* row) {
  const float2* pg = row + P::phys(P::R3 * (t + P::T * I));
  static_for<0, P::R3>([&](auto jj) { x[I * P::R3 + decltype(jj)::value] = lds_get(pg, decltype(jj)::value); });
}
template <class P, int I, bool LARGE, class TF>
__device__ __forceinline__ void fwd_group(cf (&x)[P::E], int t, const float2* tab, const TF& tf) {
  if constexpr (P::THREE) {
    tf.template group<I>().template use<LARGE>([&](auto&& w) __attribute__((always_inline)) { fwd_factors<P::R3, I * P::R3>(x, w, KeepAll{}); });
  } else {
    TableRow<P::R3> w;
    w.load(tab + (t + P::T * I) * P::FS);
    fwd_factors<P::R3, I * P::R3>(x, w, KeepAll{});
  }
}
template <class P, int I>
__device__ __forceinline__ void inv_group(cf (&x)[P::E], int t, float2* row) {
  float2* pg = row + P::phys(P::R3 * (t + P::T * I));
  inv_plain<P::R3, I * P::R3>(x, [&](auto rr) __attribute__((always_inline)) {
    constexpr int r = decltype(rr)::value;
    lds_put(pg, r % P::R3, x[r]);
  });
}
template <class P>
__device__ __forceinline__ void inv_first(cf (&x)[P::E], int t, const float2* row, const float2* tab, const TwistInverse<P>& ti) {
  static_for<0, P::NB1>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    const float2* pb = row + P::phys(t + P::T * i);
    static_for<0, P::R1>([&](auto rr) {
      constexpr int r = decltype(rr)::value;
      x[i * P::R1 + r] = lds_get(pb, P::phys(bitrev(r, ilog2(P::R1)) * P::S1));
    });
    if constexpr (P::THREE) {
      ti.first[i].template use<false>([&](auto&& w) __attribute__((always_inline)) { inv_factors<P::R1, i * P::R1>(x, w, KeepAll{}); });
    } else {
      TableRow<P::R1> w;
      w.load(tab + P::R1 * P::FS + (t + P::T * i) * P::IS);
      inv_factors<P::R1, i * P::R1>(x, w, KeepAll{});
    }
  });
}
// real part of register I R1 + J without the shift
template <class P, int S8, int REG>
__device__ __forceinline__ float end_real(const cf (&x)[P::E], const TwistEnd<P, S8>& te) {
  constexpr int i = REG / P::R1, j = REG % P::R1;
  const cf v = mul_root<j * S8, 8 * P::R1, true>(x[REG]);
  return te.f[i].re * v.re - te.f[i].im * v.im;
}

// x <- x K, K as the spectrum kernels leave it: float4 = registers 2 p and 2 p + 1 of group I, T apart.  (The thread is added last:
// where the row is the same for all lanes its addresses stay in scalar registers.)
template <class P, int I>
__device__ __forceinline__ void load_spectrum(float4 (&K)[P::R3 / 2], const float4* __restrict__ sp, int t) {
  static_for<0, P::R3 / 2>([&](auto pp) { K[decltype(pp)::value] = (sp + (I * (P::R3 / 2) + decltype(pp)::value) * P::T)[(unsigned)t]; });
}
template <class P, int I>
__device__ __forceinline__ void multiply(cf (&x)[P::E], const float4 (&K)[P::R3 / 2]) {
  static_for<0, P::R3 / 2>([&](auto pp) {
    constexpr int p = decltype(pp)::value, r = I * P::R3 + 2 * p;
    x[r] = cmul(x[r], cf{K[p].x, K[p].y});
    x[r + 1] = cmul(x[r + 1], cf{K[p].z, K[p].w});
  });
}
template <class P>
__device__ __forceinline__ void store_spectrum(const cf (&x)[P::E], float scale, float4* __restrict__ sp) {
  static_for<0, P::E / 2>([&](auto pp) {
    constexpr int p = decltype(pp)::value;
    sp[p * P::T] = make_float4(scale * x[2 * p].re, scale * x[2 * p].im, scale * x[2 * p + 1].re, scale * x[2 * p + 1].im);
  });
}

// taps (2 L of one filter and channel) in first-pass layout: lo + i hi, the two halves of the window
template <class P>
__device__ __forceinline__ void load_taps(cf (&x)[P::E], const float* __restrict__ p, int t) {
  static_for<0, P::E>([&](auto rr) {
    constexpr int r = decltype(rr)::value, n = P::T * (r / P::R1) + P::S1 * (r % P::R1);
    x[r] = {(p + n)[(unsigned)t], (p + n + P::H)[(unsigned)t]};
  });
}

// Where a mixer core finds its filters: spectra from memory (m2_filter_spectrum_fwd), or taps that it transforms itself, filter f of
// channel c at taps + (f d + c) 2 L, with skip[f][c] on tap 0.
struct FilterTaps {
  const float* taps;
  const float* const* skip;      // one pointer per filter (entries, or the table, may be null)
  int nfilters;                  // 1: the second filter is zero
};

struct Nothing {
  __device__ __forceinline__ void operator()() const {}
};
// One signal: registers in first-pass layout -> spectrum product -> registers in first-pass layout, still shifted.  Enters and
// leaves by LDS slots of the thread's own, so one may follow another without a barrier.  The groups of the last pass are a thread's
// own too: transformed, multiplied and transformed back one after the other.  `before_last` is called ahead of the last pass, where
// the spectrum's registers are free again: loads that it issues travel under that pass.
template <class P, int S8, bool REAL, class TF, class F = Nothing>
__device__ __forceinline__ void convolve(cf (&x)[P::E], int t, float2* row, const float2* tab, const TF& tf,
                                         const TwistInverse<P>& ti, const float4* __restrict__ sp, F&& before_last = Nothing{}) {
  float4 K[P::R3 / 2];
  if constexpr (!P::THREE) load_spectrum<P, 0>(K, sp, t);      // requested a pass ahead of its use
  fwd_first<P, S8, REAL>(x, t, row);
  sync_threads<P::T>();
  if constexpr (P::THREE) {
    load_spectrum<P, 0>(K, sp, t);
    second<P, false>(x, t, row, tab);
    sync_threads<P::T>();
  }
  static_for<0, P::NG>([&](auto gg) { load_group<P, decltype(gg)::value>(x, t, row); });
  static_for<0, P::NG>([&](auto gg) {
    constexpr int g = decltype(gg)::value;
    fwd_group<P, g, false>(x, t, tab, tf);
    multiply<P, g>(x, K);
    if constexpr (g + 1 < P::NG) load_spectrum<P, g + 1>(K, sp, t);
    inv_group<P, g>(x, t, row);
  });
  sync_threads<P::T>();
  if constexpr (P::THREE) {
    second<P, true>(x, t, row, tab);
    sync_threads<P::T>();
  }
  before_last();
  inv_first<P>(x, t, row, tab, ti);
}
// The same with the spectrum in registers, as `held_spectrum` leaves it.  `behind_product` is called where those registers are free again.
template <class P, int S8, bool REAL, class F>
__device__ __forceinline__ void convolve_held(cf (&x)[P::E], int t, float2* row, const float2* tab, const TwistForward<P, S8>& tf,
                                              const TwistInverse<P>& ti, const cf (&K)[P::E], F&& behind_product) {
  fwd_first<P, S8, REAL>(x, t, row);
  sync_threads<P::T>();
  if constexpr (P::THREE) {
    second<P, false>(x, t, row, tab);
    sync_threads<P::T>();
  }
  static_for<0, P::NG>([&](auto gg) { load_group<P, decltype(gg)::value>(x, t, row); });
  static_for<0, P::NG>([&](auto gg) {
    constexpr int g = decltype(gg)::value;
    fwd_group<P, g, false>(x, t, tab, tf);
    static_for<g * P::R3, (g + 1) * P::R3>([&](auto rr) { x[decltype(rr)::value] = cmul(x[decltype(rr)::value], K[decltype(rr)::value]); });
    inv_group<P, g>(x, t, row);
  });
  behind_product();
  sync_threads<P::T>();
  if constexpr (P::THREE) {
    second<P, true>(x, t, row, tab);
    sync_threads<P::T>();
  }
  inv_first<P>(x, t, row, tab, ti);
}
// the forward half: the spectrum of registers in first-pass layout
template <class P, int S8, bool LARGE>
__device__ __forceinline__ void transform(cf (&x)[P::E], int t, float2* row, const float2* tab, const TwistForward<P, S8>& tf) {
  fwd_first<P, S8, false>(x, t, row);
  sync_threads<P::T>();
  if constexpr (P::THREE) {
    second<P, false>(x, t, row, tab);
    sync_threads<P::T>();
  }
  static_for<0, P::NG>([&](auto gg) { load_group<P, decltype(gg)::value>(x, t, row); });
  static_for<0, P::NG>([&](auto gg) { fwd_group<P, decltype(gg)::value, LARGE>(x, t, tab, tf); });
}
// The spectrum of taps in first-pass layout, kept in registers: what the spectrum kernels leave in memory, value by value.
template <class P, int S8>
__device__ __forceinline__ void held_spectrum(cf (&x)[P::E], int t, float2* row, const float2* tab, const TwistForward<P, S8>& tf) {
  transform<P, S8, true>(x, t, row, tab, tf);
  constexpr float scale = 1.f / (float)P::H;
  static_for<0, P::E>([&](auto rr) { x[decltype(rr)::value] = {scale * x[decltype(rr)::value].re, scale * x[decltype(rr)::value].im}; });
}

// The forward half with fp64 butterflies, for the spectra of the shortest rows: values are rounded to fp32 between the passes and at
// the end.  A signal meets its transform's rounding once, a filter's errors every signal alike: with these spectra the
// core at L = 128 is 1.9e-7 from fp64, with fp32 butterflies 2.2e-7 where the transform of 2 L points of both signals packed, which
// this took over from, had 1.9e-7; from L = 256 on fp32 butterflies come out no further off than that one.  (us for the filters
// of 1 / 12 mixers of 768 channels: 27 / 54, with fp32 butterflies 28 / 51.5, with the packed transform 27 / 53.4.)
template <class P>
constexpr bool fine_spectrum() { return P::H == 128; }
struct cd {
  double re, im;
};
// factors of the last pass as in tables_init: row r, stage and number
template <class P, int S8>
struct FineTable {
  double v[P::R1][P::R3 / 2][2];
  constexpr FineTable() : v{} {
    for (int r = 0; r < P::R1; ++r)
      for (int n = 0; n < P::R3 / 2; ++n) {
        const int S = ilog2(2 * n + 1), e = n == 0 ? 0 : n - (1 << (S - 1));
        v[r][n][0] = root_cos64(8 * r + S8 + e * 8 * P::R1, 16 * P::R1 << S);
        v[r][n][1] = -root_sin64(8 * r + S8 + e * 8 * P::R1, 16 * P::R1 << S);
      }
  }
};
template <class P, int S8>
__device__ constexpr FineTable<P, S8> kFineTable{};
// the factors of the thread's group
template <class P, int S8>
struct FineForward {
  cd f[P::R3 / 2];
  __device__ __forceinline__ void load(int t) {
    static_for<0, P::R3 / 2>([&](auto nn) {
      constexpr int n = decltype(nn)::value;
      f[n] = {kFineTable<P, S8>.v[t][n][0], kFineTable<P, S8>.v[t][n][1]};
    });
  }
};
__device__ __forceinline__ void butterfly(cd& a, cd& b, double wr, double wi) {
  const cd s = {fma(-wi, b.im, fma(wr, b.re, a.re)), fma(wi, b.re, fma(wr, b.im, a.im))};
  b = {fma(2.0, a.re, -s.re), fma(2.0, a.im, -s.im)};
  a = s;
}
template <class P, int S8>
__device__ __forceinline__ void transform_fine(cf (&x)[P::E], int t, float2* row, const FineForward<P, S8>& ff) {
  static_for<0, P::NB1>([&](auto ii) {
    constexpr int i = decltype(ii)::value, R = P::R1;
    cd z[R];
    static_for<0, R>([&](auto rr) { z[decltype(rr)::value] = {x[i * R + decltype(rr)::value].re, x[i * R + decltype(rr)::value].im}; });
    static_for<0, ilog2(R)>([&](auto ss) {
      constexpr int S = decltype(ss)::value, h = R >> (S + 1);
      static_for<0, (1 << S)>([&](auto bb) {
        constexpr int b = decltype(bb)::value, k = S8 + 8 * bitrev(b, S), n = 16 << S, at = 2 * h * b;
        constexpr double wr = root_cos64(k, n), wi = -root_sin64(k, n);
        static_for<0, h>([&](auto jj) { butterfly(z[at + decltype(jj)::value], z[at + h + decltype(jj)::value], wr, wi); });
      });
    });
    float2* pb = row + P::phys(t + P::T * i);
    static_for<0, R>([&](auto rr) {
      constexpr int r = decltype(rr)::value;
      lds_put(pb, P::phys(bitrev(r, ilog2(R)) * P::S1), cf{(float)z[r].re, (float)z[r].im});
    });
  });
  sync_threads<P::T>();
  constexpr int R = P::R3;
  static_assert(P::NG == 1, "one group per thread");
  cd z[R];
  const float2* pg = row + P::phys(R * t);
  static_for<0, R>([&](auto jj) {
    const cf v = lds_get(pg, decltype(jj)::value);
    z[decltype(jj)::value] = {v.re, v.im};
  });
  static_for<0, ilog2(R)>([&](auto ss) {
    constexpr int S = decltype(ss)::value, h = R >> (S + 1);
    static_for<0, (1 << S)>([&](auto bb) {
      constexpr int b = decltype(bb)::value, e = bitrev(b, S), half = S > 0 ? (1 << S) / 2 : 1, at = 2 * h * b;
      const cd w = ff.f[S == 0 ? 0 : half + e % half];
      constexpr bool rot = S > 0 && e >= half;      // the other half of a stage's factors: times -i
      static_for<0, h>([&](auto jj) {
        butterfly(z[at + decltype(jj)::value], z[at + h + decltype(jj)::value], rot ? w.im : w.re, rot ? -w.re : w.im);
      });
    });
  });
  static_for<0, R>([&](auto rr) { x[decltype(rr)::value] = {(float)z[decltype(rr)::value].re, (float)z[decltype(rr)::value].im}; });
}
// the forward transform of a spectrum kernel: what it keeps, and the passes
template <class P, int S8>
struct SpectrumForward {
  typename std::conditional<fine_spectrum<P>(), FineForward<P, S8>, TwistForward<P, S8>>::type tf;
  // (by all threads of the workgroup; a barrier has to follow)
  __device__ __forceinline__ void init(int t, float2* tab) {
    if constexpr (fine_spectrum<P>()) {
      tf.load(t);
    } else {
      tables_init<P, S8>(tab);
      tf.init(t);
    }
  }
  __device__ __forceinline__ void operator()(cf (&x)[P::E], int t, float2* row, const float2* tab) const {
    if constexpr (fine_spectrum<P>()) transform_fine<P, S8>(x, t, row, tf);
    else transform<P, S8, true>(x, t, row, tab, tf);
  }
};

// Workgroups per XCD for `pieces` equal pieces of work that slot s takes at s, s + slots, ... : `cus` compute units, `most` workgroups
// on them at a time.  The unit with the most pieces ends last, and a piece goes faster with its unit to itself, so what counts is how
// many pieces the fullest unit has; among equals the fewest workgroups.  (Only the second rule, "no more workgroups than the rounds need",
// put four rows on half of the units and two on the others where three each were possible.  us of the core, d = 768, bf16, by that
// rule / by this one: L = 512, B = 11 30.1 / 27.7, 1024, 3 21.8 / 19.0, 2048, 3 37.1 / 32.6, 4096, 1 28.4 / 24.9, 4096, 3 63.3 / 56.6.)
inline int slots_for(int pieces, int most, int cus) {
  if (pieces <= most) return pieces;
  const int rounds = (pieces + most - 1) / most, few = (pieces + rounds - 1) / rounds;
  auto fullest = [&](int slots) {
    int worst = 0;
    for (int u = 0; u < cus && u < slots; ++u) {
      int n = 0;
      for (int s = u; s < slots; s += cus) n += (pieces - s + slots - 1) / slots;
      worst = n > worst ? n : worst;
    }
    return worst;
  };
  return fullest(most) < fullest(few) ? most : few;
}

// half transforms and rows by sequence length; the shift of one signal's ring (z^L = -i) in eighths
constexpr int kQuarter = 2;
typedef TwistPlan<7, 8, 1, 16, 16> Twist128;
typedef TwistPlan<8, 16, 1, 16, 16> Twist256;
typedef TwistPlan<9, 32, 1, 16, 32> Twist512;
typedef TwistPlan<10, 32, 1, 32, 32> Twist1024;
typedef TwistPlan<11, 16, 8, 16, 32> Twist2048;
typedef TwistPlan<12, 16, 16, 16, 32> Twist4096;
typedef TwistPlan<13, 32, 16, 16, 32> Twist8192;
typedef TwistPlan<14, 32, 32, 16, 32> Twist16384;

}  // namespace m2
