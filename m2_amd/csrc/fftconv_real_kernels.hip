// L = 32768: the fused mixer core and the filter-spectrum kernel.  One transform of L points does not fit the 160 KB of LDS;
// the ring of fft_twist.h splits once more,
//
//   z^L + i = (z^H - r)(z^H + r),  H = L / 2 = 16384,  r = exp(-i pi / 4)
//
// and every real signal s = s0 + z^H s1 goes through two transforms of H points, of s0 + r s1 at shift 1/8 and of s0 - r s1 at
// shift 5/8.  With P and Q the two products the result is y0 = Re(P + Q), y1 = Re((P - Q) / r) (the factor 1/2 is in the spectra).
//
//   spec[channel][signal][half][register pair 0 .. 15][T]  float4, as in fftconv_kernels.hip
//
// One workgroup of 512 threads fills a compute unit.  A thread holds 32 samples of either half of the row in the layout of the first
// pass (positions t + 512 j and H + t + 512 j), which u and the input of a plain convolution are read in directly, consecutive lanes
// consecutive samples.  The product of the short convolutions, the gate and the results of the mixer are staged through the transform's
// buffer (32768 floats are the 16384 complex slots), 64 consecutive time steps per thread on the global side.
//
// What bounds it: 124 us of vector instructions and 700 MB of memory traffic (B = 1, d = 768, bf16), which with one workgroup per unit
// overlap only where loads are requested ahead of a pass, and registers: a row's state takes 128 - 192 of 256, and what the compiler
// keeps beside it is spilled, each reload a wait for every load and store before it.  So what only depends on the thread is formed
// anew where it is used (`anew`, fft_twist.h) or kept in LDS: 232 bytes of scratch per lane became 12.
// us at d = 768, with addresses and factors kept / now, and of the polyphase form that this took over from, whose product paired
// mirrored frequencies at nine times the multiplications: B = 1 bf16 268 / 232 / 338, fp32 316 / 271 / 397; without u 145 / 122 / 140, fp32
// 191 / 165 / 170; plain convolution, which was staged too, 149 / 86 / 102, fp32 173 / 105 / 125.
// Requesting the next row's inputs or u ahead with both signals needs more registers than there are: with 100 of them spilled the kernel
// took 305 us.
//
// Stands in for the same reference code as fftconv_kernels.hip (bert/src/mm/hyena_utils.py:16-42,
// 231-236; bert/src/mm/monarch_mixer_sequence_mixer.py:112-147).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fft_twist.h"
#include "hyena_filter.h"
#include "row_io.h"

namespace m2 {

typedef Twist16384 RealPlan;      // half transforms
static_assert(twist_offsets_ok<RealPlan>(), "LDS offsets of the plan");
constexpr float kRho = 0.70710678118654752440f;      // r = kRho (1 - i)

// floats of the spectrum buffer per (channel, signal, half)
template <class P>
constexpr long real_spec_block() { return 2L * P::H; }

// Staging of 2 H floats through the transform's buffer: thread t owns the time steps 64 t .. 64 t + 63.  The rows of 64 floats are
// padded by 4 so that the 16-byte accesses of consecutive threads spread over the banks.
constexpr int stage_phys(int n) { return n + 4 * (n >> 6); }

// Causal 3-tap convolution of 8 time steps in registers, w folded as in fftconv_kernels.hip
__device__ __forceinline__ void short_conv8(const float (&in)[10], const float (&w)[3], float f, float (&out)[8]) {
  static_for<0, 8>([&](auto ee) {
    constexpr int e = decltype(ee)::value;
    out[e] = f + w[0] * in[e] + w[1] * in[e + 1] + w[2] * in[e + 2];
  });
}

// The factors of the last forward pass at shift S8 / 8 from those at shift 1/8 by one constant, where they are used: four numbers in
// registers and not eight.
template <class P, int S8>
struct HalfForward {
  const TwistForward<P, 1>& at1;
  template <int I>
  __device__ __forceinline__ Factors<P::R3> group() const {
    cf f = at1.last[I].fine, m = at1.last[I].mid;
    asm volatile("" : "+v"(f.re), "+v"(f.im), "+v"(m.re), "+v"(m.im));
    return {mul_root<S8 - 1, 8 * P::H>(f), mul_root<S8 - 1, 8 * P::H / 4>(m)};
  }
};

// Buffer and tables in LDS; behind them a thread's two factors that remove the shifts, which are read where they are used.
template <class P>
constexpr size_t real_lds_bytes() { return (size_t)(P::ROW + 2 * P::TAB + 2 * P::T) * sizeof(float2); }
template <class P>
__device__ __forceinline__ float4* ends_init(float2* lds, int t) {
  static_assert((P::ROW + 2 * P::TAB) % 2 == 0 && P::NB1 == 1, "16-byte slots, one factor each");
  float4* ends = reinterpret_cast<float4*>(lds + P::ROW + 2 * P::TAB);
  TwistEnd<P, 1> te1;
  TwistEnd<P, 5> te5;
  te1.init(t);
  te5.init(t);
  ends[t] = make_float4(te1.f[0].re, te1.f[0].im, te5.f[0].re, te5.f[0].im);
  return ends;
}

// acc += the convolution of the signal whose samples in first-pass layout are lo(r) and hi(r); sp: the signal's two blocks.  The
// second half asks for them again: at(kUnder1st) is called under the last pass of the first half, at(kBetween) behind it, at(kUnder2nd)
// under the last pass of the second half.
enum { kUnder1st, kBetween, kUnder2nd };
template <class P, class LO, class HI, class F>
__device__ __forceinline__ void convolve_halves(LO&& lo, HI&& hi, F&& at, cf (&acc)[32], int t, float2* row,
                                                const float2* tab1, const float2* tab5, const TwistForward<P, 1>& tf1,
                                                const TwistInverse<P>& ti, const float4* ends, const float4* __restrict__ sp) {
  cf x[32];
  static_for<0, 32>([&](auto rr) {
    const float v = kRho * hi(rr);
    x[decltype(rr)::value] = {lo(rr) + v, -v};
  });
  convolve<P, 1, false>(x, anew(t), row, tab1, HalfForward<P, 1>{tf1}, ti, sp, [&]() __attribute__((always_inline)) { at(ic<kUnder1st>{}); });
  // acc.re: first half of the row, acc.im: second.  P without its shift is f v; P / r = f v exp(i pi / 4)
  const float2 end1 = *reinterpret_cast<const float2*>(ends + anew(t));
  static_for<0, 32>([&](auto rr) {
    constexpr int r = decltype(rr)::value;
    const cf v = mul_root<r, 8 * P::R1, true>(x[r]);
    const float re = end1.x * v.re - end1.y * v.im, im = end1.x * v.im + end1.y * v.re;
    acc[r].re += re;
    acc[r].im = fmaf(kRho, re - im, acc[r].im);
  });
  __builtin_amdgcn_sched_barrier(0);
  at(ic<kBetween>{});
  static_for<0, 32>([&](auto rr) {
    const float v = kRho * hi(rr);
    x[decltype(rr)::value] = {lo(rr) - v, v};
  });
  convolve<P, 5, false>(x, anew(t), row, tab5, HalfForward<P, 5>{tf1}, ti, sp + real_spec_block<P>() / 4,
                        [&]() __attribute__((always_inline)) { at(ic<kUnder2nd>{}); });
  const float2 end5 = reinterpret_cast<const float2*>(ends + anew(t))[1];
  static_for<0, 32>([&](auto rr) {
    constexpr int r = decltype(rr)::value;
    const cf v = mul_root<5 * r, 8 * P::R1, true>(x[r]);
    const float re = end5.x * v.re - end5.y * v.im, im = end5.x * v.im + end5.y * v.re;
    acc[r].re += re;
    acc[r].im = fmaf(-kRho, re - im, acc[r].im);
  });
}

// ------------------------------------------------------------------------------------------
// the fused mixer core, sequence length 2 P::H
// ------------------------------------------------------------------------------------------
// HAS_U: the residual long convolution of the layer input u (uin non-null).  Without it there are registers for the gate's inputs to
// be requested under the last pass and the next row's under the epilogue.
template <class P, typename ACT, bool HAS_U>
__global__ __launch_bounds__(P::T) __attribute__((amdgpu_waves_per_eu(2, 2))) void mixer_real_kernel(
    const ACT* __restrict__ xproj,      // (3d, B, LS): x1 | x2 | v, channel-major
    long ldx,                           // elements between two channels of xproj, B L or more
    const float* __restrict__ uin,      // (d, B, LS)  layer input, channel-major (may be null)
    const float* __restrict__ sw,       // (3d, 3)     short-conv taps
    const float* __restrict__ sb,       // (3d)        short-conv bias
    const float* __restrict__ pbias,    // (3d)        bias of the in-projection, added to xproj on load (may be null)
    const float* __restrict__ spec,     // (d, 2, 2) blocks of real_spec_block<P>() floats
    ACT* __restrict__ y,                // (d, B, LS)
    int B, int d) {
  constexpr int T = P::T, H = P::H;
  constexpr long LS = 2L * H, BLK = real_spec_block<P>();
  static_assert(T == 512 && P::E == 32 && P::NB1 == 1 && stage_phys(2 * H) <= 2 * P::ROW, "512 threads, 64 time steps each");
  extern __shared__ float2 lds[];
  float2* row = lds;
  float* stage = reinterpret_cast<float*>(lds);
  const float2 *tab1 = lds + P::ROW, *tab5 = tab1 + P::TAB;
  const int t = threadIdx.x;

  tables_init<P, 1>(lds + P::ROW);
  tables_init<P, 5>(lds + P::ROW + P::TAB);
  TwistForward<P, 1> tf1;
  TwistInverse<P> ti;
  tf1.init(t);
  ti.init(t);
  float4* ends = ends_init<P>(lds, t);
  sync_threads<T>();

  // workgroup -> (channel, batch row) as in mixer_pair_kernel: XCD e takes the channels c = e (mod 8)
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, slots = gridDim.x >> 3;
  const int rows_per_xcd = (d >> 3) * B;
  RawRow<ACT, 8> r1, rv, r2;
  auto fetch = [&](RawRow<ACT, 8>& r, int third, int j) __attribute__((always_inline)) {
    const int c = __builtin_amdgcn_readfirstlane((j / B) * 8 + xcd), bb = __builtin_amdgcn_readfirstlane(j % B);
    const ACT* p = xproj + ((long)third * d + c) * ldx + (long)bb * LS;
    const int n0 = 64 * anew(t);
    static_for<0, 8>([&](auto qq) { r.template fetch<decltype(qq)::value>(p, n0 + 8 * decltype(qq)::value); });
  };
  if constexpr (!HAS_U) {
    if (slot < rows_per_xcd) {
      fetch(r1, 0, slot);
      fetch(rv, 2, slot);
    }
  }
  for (int j = slot; j < rows_per_xcd; j += slots) {
    // the same for every lane: say so, so that row base addresses live in scalar registers
    const int c = __builtin_amdgcn_readfirstlane((j / B) * 8 + xcd), bb = __builtin_amdgcn_readfirstlane(j % B);
    const float4* sp = reinterpret_cast<const float4*>(spec + (long)c * 4 * BLK);
    float lo[32], hi[32];
    auto get_lo = [&](auto rr) __attribute__((always_inline)) { return lo[decltype(rr)::value]; };
    auto get_hi = [&](auto rr) __attribute__((always_inline)) { return hi[decltype(rr)::value]; };
    cf acc[32];
    static_for<0, 32>([&](auto rr) { acc[decltype(rr)::value] = {0.f, 0.f}; });

    // ---- first signal: a = sc(x1) sc(v), convolved with filter 1
    {
      if constexpr (HAS_U) {
        fetch(r1, 0, j);
        fetch(rv, 2, j);
      }
      float w1[3], wv[3], p1 = 0.f, pbv = 0.f;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        w1[k] = sw[(long)c * 3 + k];
        wv[k] = sw[((long)2 * d + c) * 3 + k];
      }
      if (pbias) { p1 = pbias[c]; pbv = pbias[2 * d + c]; }
      const float f1 = sb[c] + p1 * (w1[0] + w1[1] + w1[2]), fv = sb[2 * d + c] + pbv * (wv[0] + wv[1] + wv[2]);
      const int n0 = 64 * anew(t);
      __builtin_amdgcn_sched_barrier(0);
      static_for<0, 8>([&](auto qq) {
        constexpr int q = decltype(qq)::value;
        const int n = n0 + 8 * q;
        float in[10], a[8], v[8];
        r1.template expand<q>(n, in);
        short_conv8(in, w1, f1, a);
        rv.template expand<q>(n, in);
        short_conv8(in, wv, fv, v);
        if constexpr (q == 0) {
          if (t == 0) {      // time steps 0 and 1: taps that fall on the zero padding, outside the biased signal
            a[0] -= p1 * (w1[0] + w1[1]); a[1] -= p1 * w1[0];
            v[0] -= pbv * (wv[0] + wv[1]); v[1] -= pbv * wv[0];
          }
        }
        static_for<0, 8>([&](auto ee) { a[decltype(ee)::value] *= v[decltype(ee)::value]; });
        float4* dst = reinterpret_cast<float4*>(stage + stage_phys(n0) + 8 * q);
        dst[0] = make_float4(a[0], a[1], a[2], a[3]);
        dst[1] = make_float4(a[4], a[5], a[6], a[7]);
        __builtin_amdgcn_sched_barrier(0);
      });
    }
    sync_threads<T>();
    auto from_stage = [&](auto&& put) __attribute__((always_inline)) {
      const float* pl = stage + stage_phys(anew(t));
      static_for<0, 32>([&](auto rr) {
        constexpr int r = decltype(rr)::value;
        put(rr, pl[stage_phys(512 * r)], pl[stage_phys(H + 512 * r)]);
      });
    };
    from_stage([&](auto rr, float l, float h) __attribute__((always_inline)) {
      lo[decltype(rr)::value] = l;
      hi[decltype(rr)::value] = h;
    });
    sync_threads<T>();                     // the transform's slots overlap the staged row
    convolve_halves<P>(get_lo, get_hi, [&](auto when) __attribute__((always_inline)) {
      if constexpr (!HAS_U && decltype(when)::value == kUnder2nd) fetch(r2, 1, j);
    }, acc, t, row, tab1, tab5, tf1, ti, ends, sp);

    // ---- gate: acc = y1 * sc(x2), by way of the stage
    {
      if constexpr (HAS_U) fetch(r2, 1, j);
      float w2[3], pb2 = 0.f;
#pragma unroll
      for (int k = 0; k < 3; ++k) w2[k] = sw[((long)d + c) * 3 + k];
      if (pbias) pb2 = pbias[d + c];
      const float f2 = sb[d + c] + pb2 * (w2[0] + w2[1] + w2[2]);
      sync_threads<T>();                   // everybody has read the last pass's slots
      float* ps = stage + stage_phys(anew(t));
      static_for<0, 32>([&](auto rr) {
        constexpr int r = decltype(rr)::value;
        ps[stage_phys(512 * r)] = acc[r].re;
        ps[stage_phys(H + 512 * r)] = acc[r].im;
      });
      if constexpr (!HAS_U) {
        __builtin_amdgcn_sched_barrier(0);
        if (j + slots < rows_per_xcd) {
          fetch(r1, 0, j + slots);
          fetch(rv, 2, j + slots);
        } else {      // (values of their own here too: otherwise this row's inputs would stay in registers up to this point)
          static_for<0, 8>([&](auto qq) { r1.clear(qq); rv.clear(qq); });
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      sync_threads<T>();
      const int n0 = 64 * anew(t);
      static_for<0, 8>([&](auto qq) {
        constexpr int q = decltype(qq)::value;
        float in[10], g[8];
        r2.template expand<q>(n0 + 8 * q, in);
        short_conv8(in, w2, f2, g);
        if constexpr (q == 0) {
          if (t == 0) { g[0] -= pb2 * (w2[0] + w2[1]); g[1] -= pb2 * w2[0]; }
        }
        float4* at = reinterpret_cast<float4*>(stage + stage_phys(n0) + 8 * q);
        const float4 v0 = at[0], v1 = at[1];
        const float o[8] = {v0.x * g[0], v0.y * g[1], v0.z * g[2], v0.w * g[3], v1.x * g[4], v1.y * g[5], v1.z * g[6], v1.w * g[7]};
        if constexpr (HAS_U) {
          at[0] = make_float4(o[0], o[1], o[2], o[3]);
          at[1] = make_float4(o[4], o[5], o[6], o[7]);
        } else {
          store8(y + ((long)c * B + bb) * LS, n0 + 8 * q, o);
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      sync_threads<T>();                   // the next row's prologue overwrites what has just been read
      if constexpr (HAS_U) {
        from_stage([&](auto rr, float l, float h) __attribute__((always_inline)) { acc[decltype(rr)::value] = {l, h}; });
        sync_threads<T>();
      }
    }

    // ---- second signal: the layer input u, convolved with filter 2 on top of it; read twice rather than kept across the first half
    if constexpr (HAS_U) {
      const float* pu = uin + ((long)c * B + bb) * LS;
      auto load_u = [&]() __attribute__((always_inline)) {
        int again = 0;
        asm volatile("" : "+s"(again));      // a second load, not the first one's registers kept across the half transform
        const float* p = pu + again;
        static_for<0, 32>([&](auto rr) {
          constexpr int r = decltype(rr)::value;
          lo[r] = (p + 512 * r)[(unsigned)t];
          hi[r] = (p + H + 512 * r)[(unsigned)t];
        });
      };
      load_u();
      convolve_halves<P>(get_lo, get_hi, [&](auto when) __attribute__((always_inline)) {
        if constexpr (decltype(when)::value == kBetween) load_u();
      }, acc, t, row, tab1, tab5, tf1, ti, ends, sp + BLK / 2);
      // results to 64 consecutive time steps per thread
      sync_threads<T>();
      float* ps = stage + stage_phys(anew(t));
      static_for<0, 32>([&](auto rr) {
        constexpr int r = decltype(rr)::value;
        ps[stage_phys(512 * r)] = acc[r].re;
        ps[stage_phys(H + 512 * r)] = acc[r].im;
      });
      sync_threads<T>();
      const int n0 = 64 * anew(t);
      static_for<0, 8>([&](auto qq) {
        constexpr int q = decltype(qq)::value;
        const float4* at = reinterpret_cast<const float4*>(stage + stage_phys(n0) + 8 * q);
        const float4 v0 = at[0], v1 = at[1];
        const float o[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
        store8(y + ((long)c * B + bb) * LS, n0 + 8 * q, o);
      });
      sync_threads<T>();                   // the next row's prologue overwrites what has just been read
    }
  }
}

// A plain long convolution of one input, without short convolutions and gates: samples go straight from memory to the layout of the
// first pass and back, consecutive lanes consecutive samples, so that nothing is staged and no barrier stands between rows; the
// samples are read twice, the second time and the next row's first under a last pass.
template <class P, typename ACT>
__global__ __launch_bounds__(P::T) __attribute__((amdgpu_waves_per_eu(2, 2))) void conv_real_kernel(
    const ACT* __restrict__ x, const float* __restrict__ spec, ACT* __restrict__ y, int B, int d) {
  constexpr int T = P::T, H = P::H;
  constexpr long LS = 2L * H, BLK = real_spec_block<P>();
  static_assert(T == 512 && P::E == 32 && P::NB1 == 1 && P::S1 == 512, "first-pass layout");
  extern __shared__ float2 lds[];
  float2* row = lds;
  const float2 *tab1 = lds + P::ROW, *tab5 = tab1 + P::TAB;
  const int t = threadIdx.x;

  tables_init<P, 1>(lds + P::ROW);
  tables_init<P, 5>(lds + P::ROW + P::TAB);
  TwistForward<P, 1> tf1;
  TwistInverse<P> ti;
  tf1.init(t);
  ti.init(t);
  float4* ends = ends_init<P>(lds, t);
  sync_threads<T>();

  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, slots = gridDim.x >> 3;
  const int rows_per_xcd = (d >> 3) * B;
  ACT lo[32], hi[32];
  auto value = [](ACT v) __attribute__((always_inline)) -> float {
    if constexpr (sizeof(ACT) == 2) return bf16_to_f32(v); else return v;
  };
  auto get_lo = [&](auto rr) __attribute__((always_inline)) { return value(lo[decltype(rr)::value]); };
  auto get_hi = [&](auto rr) __attribute__((always_inline)) { return value(hi[decltype(rr)::value]); };
  auto load = [&](int j) __attribute__((always_inline)) {
    const int c = __builtin_amdgcn_readfirstlane((j / B) * 8 + xcd), bb = __builtin_amdgcn_readfirstlane(j % B);
    int again = 0;
    asm volatile("" : "+s"(again));      // a load of its own, not an earlier one's registers kept
    const ACT* p = x + ((long)c * B + bb) * LS + again;
    static_for<0, 32>([&](auto rr) {
      constexpr int r = decltype(rr)::value;
      lo[r] = (p + 512 * r)[(unsigned)t];
      hi[r] = (p + H + 512 * r)[(unsigned)t];
    });
  };
  if (slot < rows_per_xcd) load(slot);
  for (int j = slot; j < rows_per_xcd; j += slots) {
    const int c = __builtin_amdgcn_readfirstlane((j / B) * 8 + xcd), bb = __builtin_amdgcn_readfirstlane(j % B);
    cf acc[32];
    static_for<0, 32>([&](auto rr) { acc[decltype(rr)::value] = {0.f, 0.f}; });
    convolve_halves<P>(get_lo, get_hi, [&](auto when) __attribute__((always_inline)) {
      if constexpr (decltype(when)::value == kUnder1st) load(j);
      if constexpr (decltype(when)::value == kUnder2nd) load(j + slots < rows_per_xcd ? j + slots : j);
    }, acc, t, row, tab1, tab5, tf1, ti, ends, reinterpret_cast<const float4*>(spec + (long)c * 4 * BLK));
    ACT* py = y + ((long)c * B + bb) * LS;
    static_for<0, 32>([&](auto rr) {
      constexpr int r = decltype(rr)::value;
      if constexpr (sizeof(ACT) == 2) {
        (py + 512 * r)[(unsigned)t] = f32_to_bf16(acc[r].re);
        (py + H + 512 * r)[(unsigned)t] = f32_to_bf16(acc[r].im);
      } else {
        (py + 512 * r)[(unsigned)t] = acc[r].re;
        (py + H + 512 * r)[(unsigned)t] = acc[r].im;
      }
    });
  }
}

// ------------------------------------------------------------------------------------------
// filter taps -> spectra; work item = (channel, filter), both half transforms
// ------------------------------------------------------------------------------------------
template <class P>
__global__ __launch_bounds__(P::T) __attribute__((amdgpu_waves_per_eu(2, 2))) void filter_spectrum_real_kernel(
    const float* taps1,    // (d, 2 LS) bidirectional taps of filter_fn
    const float* taps2,    // (d, 2 LS) bidirectional taps of filter_fn2 (null: its blocks are zeroed)
    const float* D1,       // (d) skip weight of filter_fn, added to tap 0 (may be null)
    const float* D2,       // (d) skip weight of filter_fn2 (may be null)
    float* __restrict__ spec, int d, SpectrumBatch sb) {
  constexpr int H = P::H, T = P::T;
  constexpr long LS = 2L * H, BLK = real_spec_block<P>();
  {
    float* sp = spec;
    select_mixer(sb, d, 2 * LS, taps1, taps2, D1, D2, sp);
    spec = sp;
  }
  extern __shared__ float2 lds[];
  float2* row = lds;
  const float2 *tab1 = lds + P::ROW, *tab5 = tab1 + P::TAB;
  const int t = threadIdx.x;

  tables_init<P, 1>(lds + P::ROW);
  tables_init<P, 5>(lds + P::ROW + P::TAB);
  TwistForward<P, 1> tf1;
  TwistForward<P, 5> tf5;
  tf1.init(t);
  tf5.init(t);
  sync_threads<T>();
  const float scale = 1.f / (float)LS;      // 1/H of the inverse, 1/2 of the two halves

  // the taps row is read once: both halves' inputs are formed, the second waits in registers
  for (int item = blockIdx.x; item < 2 * d; item += gridDim.x) {
    const int c = item >> 1;
    const float* taps = item & 1 ? taps2 : taps1;
    gfloat* D = in_global(item & 1 ? D2 : D1);
    float4* blk = reinterpret_cast<float4*>(spec + (long)item * 2 * BLK) + t;
    if (!taps) {
      static_for<0, 2>([&](auto hh) {
        static_for<0, 16>([&](auto ss) { blk[decltype(hh)::value * (BLK / 4) + decltype(ss)::value * T] = make_float4(0.f, 0.f, 0.f, 0.f); });
      });
      continue;
    }
    // k = lo + i hi over the two halves of the window, k = k0 + z^H k1: k0 +- r k1
    cf x[32], q[32];
    {
      const float* p = taps + (long)c * 2 * LS;
      const float dd = (D && t == 0) ? D[c] : 0.f;      // the skip weight is one more tap at lag 0
      static_for<0, 32>([&](auto rr) {
        constexpr int r = decltype(rr)::value;
        x[r] = {(p + 512 * r)[(unsigned)t], (p + LS + 512 * r)[(unsigned)t]};
        q[r] = {(p + H + 512 * r)[(unsigned)t], (p + LS + H + 512 * r)[(unsigned)t]};
      });
      x[0].re += dd;
      static_for<0, 32>([&](auto rr) {
        constexpr int r = decltype(rr)::value;
        const cf v = {kRho * (q[r].re + q[r].im), kRho * (q[r].im - q[r].re)};
        q[r] = {x[r].re - v.re, x[r].im - v.im};
        x[r] = {x[r].re + v.re, x[r].im + v.im};
      });
    }
    sync_threads<T>();                      // the item before has been read
    transform<P, 1, false>(x, t, row, tab1, tf1);
    store_spectrum<P>(x, scale, blk);
    sync_threads<T>();
    static_for<0, 32>([&](auto rr) { x[decltype(rr)::value] = q[decltype(rr)::value]; });
    transform<P, 5, false>(x, t, row, tab5, tf5);
    store_spectrum<P>(x, scale, blk + BLK / 4);
  }
}

// ------------------------------------------------------------------------------------------
// host-side launchers
// ------------------------------------------------------------------------------------------
template <typename ACT>
static int launch_mixer_real(const void* xproj, long ldx, const float* u, const float* sw, const float* sb, const float* pbias,
                             const float* spec, void* y, int B, int d, hipStream_t stream) {
  typedef RealPlan P;
  const size_t lds_bytes = real_lds_bytes<P>();
  const void* kern = !sw ? (const void*)conv_real_kernel<P, ACT>
                         : u ? (const void*)mixer_real_kernel<P, ACT, true> : (const void*)mixer_real_kernel<P, ACT, false>;
  if (!sw && u) return set_error(M2_ERR_ARG, "mixer_real: a plain convolution takes no second input");
  hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
  if (e != hipSuccess) return set_error(M2_ERR_LAUNCH, "hipFuncSetAttribute(mixer_real): %s", hipGetErrorString(e));
  const int rows_per_xcd = (d / 8) * B;
  int slots = num_cus() / 8;          // one workgroup per compute unit (158 KB of LDS)
  if (slots > rows_per_xcd) slots = rows_per_xcd;
  const int rounds = (rows_per_xcd + slots - 1) / slots;      // every workgroup the same number of rows
  slots = (rows_per_xcd + rounds - 1) / rounds;
  if (!sw)
    hipLaunchKernelGGL((conv_real_kernel<P, ACT>), dim3(8 * slots), dim3(P::T), lds_bytes, stream, (const ACT*)xproj, spec, (ACT*)y, B, d);
  else
    hipLaunchKernelGGL((u ? mixer_real_kernel<P, ACT, true> : mixer_real_kernel<P, ACT, false>), dim3(8 * slots), dim3(P::T), lds_bytes,
                       stream, (const ACT*)xproj, ldx, u, sw, sb, pbias, spec, (ACT*)y, B, d);
  return check_launch("mixer_real");
}

int launch_mixer_real_dispatch(const void* xproj, long ldx, const float* u, const float* sw, const float* sb, const float* pbias,
                               const float* spec, void* y, int B, int d, int act_dtype, hipStream_t stream) {
  return act_dtype == M2_DTYPE_F32 ? launch_mixer_real<float>(xproj, ldx, u, sw, sb, pbias, spec, y, B, d, stream)
                                   : launch_mixer_real<uint16_t>(xproj, ldx, u, sw, sb, pbias, spec, y, B, d, stream);
}

int launch_filter_spectrum_real(const float* taps1, const float* taps2, const float* D1, const float* D2, float* spec,
                                int d, const SpectrumBatch& sb, int nmixers, hipStream_t stream) {
  typedef RealPlan P;
  const size_t lds_bytes = (size_t)(P::ROW + 2 * P::TAB) * sizeof(float2);
  auto kern = filter_spectrum_real_kernel<P>;
  hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
  if (e != hipSuccess) return set_error(M2_ERR_LAUNCH, "hipFuncSetAttribute(filter_spectrum_real): %s", hipGetErrorString(e));
  int grid = num_cus();
  if (grid > 2 * d) grid = 2 * d;
  hipLaunchKernelGGL(kern, dim3(grid, nmixers), dim3(P::T), lds_bytes, stream, taps1, taps2, D1, D2, spec, d, sb);
  return check_launch("filter_spectrum_real");
}

}  // namespace m2
