// The fused mixer core at L = 8192 and 16384, where the row buffers of both signals do not leave room for two workgroups on a
// compute unit (or for one): the signals are convolved one after the other through one buffer of L points, so that at L = 8192 two
// workgroups share a unit and overlap each other's barriers and memory stalls.  See fft_twist.h for the transforms.
//
// A row is staged once, a and u side by side as the real and imaginary part of a slot; in the layout of the first pass a thread
// then holds 32 samples of each.  Every signal enters and leaves its passes by slots of the thread's own, and the results go back to
// them side by side again.
//
// us (bf16, d = 768), against two half transforms of both signals packed: L = 8192, B = 4 171 / 184 (15 % fewer vector instructions;
// the ALU is 72 % busy by counter, and LDS and memory overlap with it only across the workgroups of a unit), L = 16384, B = 2 189 / 218.
// Requesting the next row's inputs under the epilogue gained nothing measurable at B = 4 and 3 % with fp32 inputs.  Addresses are formed
// anew where they are used: kept, they had up to 108 bytes per lane spilled (fp32, L = 16384, B = 1 / 2: 145 / 263, now 130 / 248).
//
// Stands in for the same reference code as fftconv_kernels.hip (bert/src/mm/hyena_utils.py:16-42,
// 231-236; bert/src/mm/monarch_mixer_sequence_mixer.py:112-147).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fft_twist.h"
#include "row_io.h"

namespace m2 {

static_assert(twist_offsets_ok<Twist8192>() && twist_offsets_ok<Twist16384>(), "LDS offsets of the plan");

// FULL: short convolutions and gates (sw, sb non-null); otherwise a plain long convolution of one input.
// HAS_U: the residual long convolution of the layer input u (uin non-null).
// TAPS: the filters come as taps, and every row transforms its channel's own (see mixer_taps_kernels.hip).
template <class P, typename ACT, bool FULL, bool HAS_U, bool TAPS>
__global__ __launch_bounds__(P::T) __attribute__((amdgpu_waves_per_eu(2, 2))) void mixer_long_kernel(
    const ACT* __restrict__ xproj,      // (3d, B, L): x1 | x2 | v, channel-major
    long ldx,                           // elements between two channels of xproj, B L or more
    const float* __restrict__ uin,      // (d, B, L)   layer input, channel-major (may be null)
    const float* __restrict__ sw,       // (3d, 3)     short-conv taps; null = plain convolution of a (d, B, L) input
    const float* __restrict__ sb,       // (3d)        short-conv bias
    const float* __restrict__ pbias,    // (3d)        bias of the in-projection, added to xproj on load (may be null)
    const float4* __restrict__ spec,    // (d, 2, E/2, T)
    ACT* __restrict__ y,                // (d, B, L)
    int B, int d, FilterTaps filters) {
  static_assert(!TAPS || (FULL && sizeof(ACT) == 2), "plain convolutions and fp32 rows read spectra");
  constexpr int L = P::H, T = P::T, E = P::E;
  static_assert(E == 32, "four runs of 8 time steps per thread");
  extern __shared__ float2 lds[];
  float2* row = lds;
  const float2* tab = lds + P::ROW;
  const int t = threadIdx.x;

  tables_init<P, kQuarter>(lds + P::ROW);
  TwistForward<P, kQuarter> tf;
  TwistInverse<P> ti;
  TwistEnd<P, kQuarter> te;
  tf.init(t);
  ti.init(t);
  te.init(t);
  sync_threads<T>();

  // Workgroup ids are dealt round-robin to the 8 XCDs (one L2 each).  XCD e takes the channels
  // c = e (mod 8) and runs the B rows of a channel on neighbouring workgroups at the same time, so a
  // channel's spectrum is fetched into that L2 once and shared.  (d % 8 == 0 is checked by the host.)
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, slots = gridDim.x >> 3;
  const int rows_per_xcd = (d >> 3) * B;

  RawRow<ACT, 4> r1, r2, rv;      // the four accesses of a thread are consecutive
  f32x4_t ru[8];
  auto fetch_row = [&](int j) __attribute__((always_inline)) {
    const int c = (j / B) * 8 + xcd, bb = j % B, n0 = 32 * anew(t);
    static_for<0, 4>([&](auto qq) {
      constexpr int q = decltype(qq)::value;
      const int n = n0 + 8 * q;
      if constexpr (FULL) {
        r1.template fetch<q>(xproj + (long)(0 * d + c) * ldx + (long)bb * L, n);
        rv.template fetch<q>(xproj + (long)(2 * d + c) * ldx + (long)bb * L, n);
        r2.template fetch<q>(xproj + (long)(1 * d + c) * ldx + (long)bb * L, n);
      } else {
        r1.template fetch<q>(xproj + (long)c * ldx + (long)bb * L, n);
      }
      if constexpr (HAS_U) {
        const float* pu = uin + ((long)c * B + bb) * L + n;
        ru[2 * q] = *reinterpret_cast<const f32x4_t*>(pu);
        ru[2 * q + 1] = *reinterpret_cast<const f32x4_t*>(pu + 4);
      }
    });
  };
  if (slot < rows_per_xcd) fetch_row(slot);
  cf K[E];      // TAPS: of the signal's filter, taps and then their transform
  auto fetch_taps = [&](int j, int f) __attribute__((always_inline)) {
    const int c = __builtin_amdgcn_readfirstlane((j / B) * 8 + xcd);
    load_taps<P>(K, filters.taps + ((long)f * d + c) * (2L * L), anew(t));
  };
  auto transform_taps = [&](int c, int f) __attribute__((always_inline)) {
    gfloat* D = filters.skip ? in_global(filters.skip[f]) : nullptr;
    if (D && t == 0) K[0].re += D[c];      // the skip weight is one more tap at lag 0
    held_spectrum<P, kQuarter>(K, anew(t), row, tab, tf);
  };
  if constexpr (TAPS) {
    if (slot < rows_per_xcd) fetch_taps(slot, 0);
  }

  for (int j = slot; j < rows_per_xcd; j += slots) {
    // the same for every lane: say so, so that row base addresses live in scalar registers
    const int c = __builtin_amdgcn_readfirstlane((j / B) * 8 + xcd), bb = __builtin_amdgcn_readfirstlane(j % B);

    if constexpr (TAPS) {
      transform_taps(c, 0);
      sync_threads<T>();
    }

    // ---- prologue: 32 consecutive time steps per thread in chunks of 8 (a mapping with consecutive lanes on
    // consecutive 16-byte pieces was measured 7 % slower): short conv, gate, (a, u) -> LDS
    GateRow<ACT, 4> gate;
    {
      float w1[3], w2[3], wv[3], b1 = 0.f, b2 = 0.f, bv = 0.f, p1 = 0.f, p2 = 0.f, pv = 0.f;
      if constexpr (FULL) {
        const float* w = sw + (long)c * 3;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          w1[k] = w[k];
          w2[k] = w[3 * (long)d + k];
          wv[k] = w[6 * (long)d + k];
        }
        b1 = sb[c]; b2 = sb[d + c]; bv = sb[2 * d + c];
        if (pbias) { p1 = pbias[c]; p2 = pbias[d + c]; pv = pbias[2 * d + c]; }
      }
      // The bias p of the in-projection is not added to the inputs: a 3-tap convolution of (x + p) is the convolution
      // of x plus p (w0 + w1 + w2), which goes into the convolution's own bias -- except for the first two outputs
      // of a row, where one or two taps fall on the zero padding (outside the biased signal): those are corrected.
      const float f1 = b1 + p1 * (w1[0] + w1[1] + w1[2]), f2 = b2 + p2 * (w2[0] + w2[1] + w2[2]),
                  fv = bv + pv * (wv[0] + wv[1] + wv[2]);
      const int n0 = 32 * anew(t);
      __builtin_amdgcn_sched_barrier(0);
      static_for<0, 4>([&](auto qq) {
        constexpr int q = decltype(qq)::value;
        const int n = n0 + 8 * q;
        float in[10], a[8], gt[8];
        r1.template expand<q>(n, in);
        if constexpr (FULL) {
          float cv[8];
          static_for<0, 8>([&](auto ee) {
            constexpr int e = decltype(ee)::value;
            a[e] = f1 + w1[0] * in[e] + w1[1] * in[e + 1] + w1[2] * in[e + 2];
          });
          rv.template expand<q>(n, in);
          static_for<0, 8>([&](auto ee) {
            constexpr int e = decltype(ee)::value;
            cv[e] = fv + wv[0] * in[e] + wv[1] * in[e + 1] + wv[2] * in[e + 2];
          });
          r2.template expand<q>(n, in);
          static_for<0, 8>([&](auto ee) {
            constexpr int e = decltype(ee)::value;
            gt[e] = f2 + w2[0] * in[e] + w2[1] * in[e + 1] + w2[2] * in[e + 2];
          });
          if constexpr (q == 0) {
            if (t == 0) {      // time steps 0 and 1 of the row
              a[0] -= p1 * (w1[0] + w1[1]); a[1] -= p1 * w1[0];
              cv[0] -= pv * (wv[0] + wv[1]); cv[1] -= pv * wv[0];
              gt[0] -= p2 * (w2[0] + w2[1]); gt[1] -= p2 * w2[0];
            }
          }
          static_for<0, 8>([&](auto ee) { a[decltype(ee)::value] *= cv[decltype(ee)::value]; });
        } else {
          // plain long convolution: xproj is a single (d, B, L) signal, no short conv, no gates
          static_for<0, 8>([&](auto ee) {
            constexpr int e = decltype(ee)::value;
            a[e] = in[e + 2];
            gt[e] = 1.f;
          });
        }
        gate.template set<q>(gt);
        f32x4_t u0 = {0.f, 0.f, 0.f, 0.f}, u1 = u0;
        if constexpr (HAS_U) { u0 = ru[2 * q]; u1 = ru[2 * q + 1]; }
        float2* dst = row + P::phys(n);       // 8 consecutive slots never straddle a pad
        dst[0] = make_float2(a[0], u0.x); dst[1] = make_float2(a[1], u0.y);
        dst[2] = make_float2(a[2], u0.z); dst[3] = make_float2(a[3], u0.w);
        dst[4] = make_float2(a[4], u1.x); dst[5] = make_float2(a[5], u1.y);
        dst[6] = make_float2(a[6], u1.z); dst[7] = make_float2(a[7], u1.w);
        __builtin_amdgcn_sched_barrier(0);
      });
    }
    sync_threads<T>();

    const float4* sp = spec + (long)c * 2 * (E / 2) * T;
    cf x[E];
    float u[E], ya[E];
    const int t0 = anew(t);
    static_for<0, P::NB1>([&](auto ii) {
      constexpr int i = decltype(ii)::value;
      const float2* pb = row + P::phys(t0 + T * i);
      static_for<0, P::R1>([&](auto jj) {
        constexpr int r = i * P::R1 + decltype(jj)::value;
        const cf v = lds_get(pb, P::phys(decltype(jj)::value * P::S1));
        x[r] = {v.re, 0.f};
        u[r] = v.im;
      });
    });
    if constexpr (TAPS)
      convolve_held<P, kQuarter, true>(x, anew(t), row, tab, tf, ti, K, [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (HAS_U) fetch_taps(j, 1);
        __builtin_amdgcn_sched_barrier(0);
      });
    else
      convolve<P, kQuarter, true>(x, anew(t), row, tab, tf, ti, sp);
    static_for<0, E>([&](auto rr) {
      constexpr int r = decltype(rr)::value;
      ya[r] = end_real<P, kQuarter, r>(x, te);
      x[r] = {u[r], 0.f};
    });
    if constexpr (HAS_U && TAPS) {
      // (the last pass has read slots of the thread's own, which the first one of the transform writes)
      transform_taps(c, 1);
      sync_threads<T>();                   // its last reads are of a group's slots
      convolve_held<P, kQuarter, true>(x, anew(t), row, tab, tf, ti, K, Nothing{});
    } else if constexpr (HAS_U) {
      convolve<P, kQuarter, true>(x, anew(t), row, tab, tf, ti, sp + (E / 2) * T);
    }
    const int t1 = anew(t);
    static_for<0, P::NB1>([&](auto ii) {
      constexpr int i = decltype(ii)::value;
      float2* pb = row + P::phys(t1 + T * i);
      static_for<0, P::R1>([&](auto jj) {
        constexpr int r = i * P::R1 + decltype(jj)::value;
        lds_put(pb, P::phys(decltype(jj)::value * P::S1), cf{ya[r], HAS_U ? end_real<P, kQuarter, r>(x, te) : 0.f});
      });
    });
    // the next row's inputs, while the results go back through LDS
    __builtin_amdgcn_sched_barrier(0);
    if (j + slots < rows_per_xcd) {
      fetch_row(j + slots);
      if constexpr (TAPS) fetch_taps(j + slots, 0);
    } else {      // (a value of its own here too: otherwise this row's inputs would stay in registers up to this point)
      static_for<0, 4>([&](auto qq) {
        constexpr int q = decltype(qq)::value;
        r1.clear(ic<q>{}); r2.clear(ic<q>{}); rv.clear(ic<q>{});
        ru[2 * q] = ru[2 * q + 1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      });
      if constexpr (TAPS) static_for<0, E>([&](auto rr) { K[decltype(rr)::value] = {0.f, 0.f}; });
    }
    __builtin_amdgcn_sched_barrier(0);
    sync_threads<T>();

    // ---- epilogue: 32 consecutive outputs per thread
    const int n0 = 32 * anew(t);
    static_for<0, 4>([&](auto qq) {
      constexpr int q = decltype(qq)::value;
      const int n = n0 + 8 * q;
      const float2* src = row + P::phys(n);
      float out[8];
      static_for<0, 8>([&](auto ee) {
        constexpr int e = decltype(ee)::value;
        const float2 v = src[e];
        out[e] = v.x * gate.template get<8 * q + e>() + v.y;
      });
      store8(y + ((long)c * B + bb) * L, n, out);
    });
    sync_threads<T>();      // the next row's prologue overwrites what the epilogue has just read
  }
}

template <class P, typename ACT, bool TAPS>
static int launch_mixer_long(const void* xproj, long ldx, const float* u, const float* sw, const float* sb, const float* pbias,
                             const float* spec, const FilterTaps& filters, void* y, int B, int d, hipStream_t stream) {
  const size_t lds_bytes = (size_t)(P::ROW + P::TAB) * sizeof(float2);
  auto kern = u ? mixer_long_kernel<P, ACT, true, true, TAPS> : mixer_long_kernel<P, ACT, true, false, TAPS>;
  if constexpr (!TAPS) {
    if (!sw) kern = mixer_long_kernel<P, ACT, false, false, false>;
  }
  if (!sw && u) return set_error(M2_ERR_ARG, "mixer_long: a plain convolution takes no second input");
  hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
  if (e != hipSuccess) return set_error(M2_ERR_LAUNCH, "hipFuncSetAttribute(mixer_long): %s", hipGetErrorString(e));
  const int rows_per_xcd = (d / 8) * B;
  int per_cu = (int)((160 * 1024) / lds_bytes);
  if (per_cu < 1) per_cu = 1;
  if (per_cu > 512 / P::T) per_cu = 512 / P::T;  // two waves per SIMD at 256 registers
  const int cus = num_cus() / 8, slots = slots_for(rows_per_xcd, cus * per_cu, cus);          // workgroups per XCD
  hipLaunchKernelGGL(kern, dim3(8 * slots), dim3(P::T), lds_bytes, stream, (const ACT*)xproj, ldx, u, sw, sb, pbias,
                     (const float4*)spec, (ACT*)y, B, d, filters);
  return check_launch("mixer_long");
}

}  // namespace m2
