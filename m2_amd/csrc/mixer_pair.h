// The fused mixer core with both signals of a row at the same time (L = 128 .. 8192), and its launcher: a template of the translation
// units that build it, fftconv_kernels.hip on filter spectra and mixer_taps_kernels.hip on filter taps.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fft_twist.h"
#include "row_io.h"

namespace m2 {

// ------------------------------------------------------------------------------------------
// the fused mixer core, both signals of a row at the same time
// ------------------------------------------------------------------------------------------
// Per-row constants of the short convolutions, staged through LDS: the threads of a row share one channel, so
// thread k < 15 of the row fetches constant k and all of them read the set back (one register per thread in
// flight instead of fifteen).  Order: (w0, w1, w2, conv bias, projection bias) of x1, then of v, then of x2.
constexpr int kRowConsts = 16;

template <class P>
struct PairLayout {
  static constexpr int RT = 2 * P::T;                          // threads per row: the first half convolves a, the second u
  static constexpr int WG = RT < 256 ? 256 : RT, RPW = WG / RT;
  static constexpr int Q = P::H / RT / 8;                      // runs of 8 time steps per thread
  // A staged row of floats is padded by four after each thread's run, so that 16-byte accesses of consecutive lanes spread over the banks.
  __host__ __device__ static constexpr int stage(int n) { return n + 4 * (n / (8 * Q)); }
  static_assert(P::T % (8 * Q) == 0 && P::S1 % (8 * Q) == 0 && stage(P::H) <= 2 * P::ROW, "the staged row lies in the transform's buffer");
  static constexpr size_t lds_bytes = (size_t)(RPW * 2 * P::ROW + P::TAB) * sizeof(float2) + (size_t)RPW * kRowConsts * sizeof(float);
};

// A row is staged in LDS between 8 consecutive time steps per thread (16-byte global accesses, short convolutions in registers) and
// the layout of the first pass, as plain rows of floats in the buffers of the two transforms.
//
// What bounds it is the vector ALU: at L = 128, d = 1536, B = 64 about 1300 vector instructions per wave and batch of four rows are
// 52 us at full issue, the kernel takes 49; by counter the ALU is 80 % busy there and 81 % at L = 1024, B = 31.  So the split follows the instruction
// count: 16 or 32 points per thread, so that a row up to L = 1024 is two passes inside one wavefront without a barrier, and both
// signals at once, so that a signal that waits costs no registers and the next rows' inputs can travel in them.  us, against the
// transform of 2 L points per row of both signals packed (three passes): L = 128, d = 768, B = 32 15.5 / 21.3; d = 1536, B = 64
// 49 / 68; L = 512, B = 32 56 / 78; L = 1024, B = 31 117 / 166; L = 2048, d = 960, B = 16 184 / 221; L = 4096, B = 1 28 / 32, B = 8
// 159 / 171.  Relative error of the fp32 core against fp64, now / then (N(0, 1) signals and taps): 1.9e-7 / 1.9e-7 at L = 128, 2.4e-7 /
// 2.4e-7 at 256, 2.5e-7 / 4.0e-7 at 512, 3.0e-7 / 6.8e-7 at 2048, 3.4e-7 / 1.2e-6 at 8192.
// FULL: short convolutions and gates (sw, sb non-null); otherwise a plain long convolution of one input.
// TAPS: the filters come as taps, and every row transforms its channel's own (see mixer_taps_kernels.hip).
template <class P, typename ACT, bool FULL, bool TAPS>
__global__ __launch_bounds__(PairLayout<P>::WG) __attribute__((amdgpu_waves_per_eu(P::E == 16 ? 3 : 2, P::E == 16 ? 3 : 2))) void mixer_pair_kernel(
    const ACT* __restrict__ xproj,      // (3d, B, L): x1 | x2 | v, channel-major
    long ldx,                           // elements between two channels of xproj, B L or more
    const float* __restrict__ uin,      // (d, B, L)   layer input, channel-major (may be null)
    const float* __restrict__ sw,       // (3d, 3)     short-conv taps
    const float* __restrict__ sb,       // (3d)        short-conv bias
    const float* __restrict__ pbias,    // (3d)        bias of the in-projection, added to xproj on load (may be null)
    const float4* __restrict__ spec,    // (d, 2, E/2, T)
    ACT* __restrict__ y,                // (d, B, L)
    int B, int d, FilterTaps filters) {
  static_assert(!TAPS || (FULL && sizeof(ACT) == 2), "plain convolutions and fp32 rows read spectra");
  constexpr int L = P::H, T = P::T, E = P::E, RT = PairLayout<P>::RT, RPW = PairLayout<P>::RPW, Q = PairLayout<P>::Q;
  extern __shared__ float2 lds[];
  const int tid = threadIdx.x;
  const int rloc = tid / RT, tr = tid % RT, sig = tr / T, t = tr % T;
  float2* both = lds + rloc * 2 * P::ROW;
  float2* row = both + sig * P::ROW;                          // of this thread's transform
  float* stage = reinterpret_cast<float*>(row);
  float* stage_a = reinterpret_cast<float*>(both);
  float* stage_u = reinterpret_cast<float*>(both + P::ROW);
  const float2* tab = lds + RPW * 2 * P::ROW;
  float* crow = reinterpret_cast<float*>(lds + RPW * 2 * P::ROW + P::TAB) + rloc * kRowConsts;
  const int n0 = 8 * Q * tr;

  tables_init<P, kQuarter>(lds + RPW * 2 * P::ROW);
  TwistForward<P, kQuarter> tf;
  TwistInverse<P> ti;
  TwistEnd<P, kQuarter> te;
  tf.init(t);
  ti.init(t);
  te.init(t);
  __syncthreads();

  // Workgroup ids are dealt round-robin to the 8 XCDs (one L2 each).  XCD e takes the channels
  // c = e (mod 8) and runs the B rows of a channel on neighbouring workgroups at the same time, so a
  // channel's spectrum is fetched into that L2 once and shared.  (d % 8 == 0 is checked by the host.)
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, slots = gridDim.x >> 3;
  const int rows_per_xcd = (d >> 3) * B;

  // The inputs of a row batch are requested one batch ahead: the loads of batch i + 1 are issued as soon as the
  // registers of batch i have been consumed by its prologue, and travel while batch i is transformed.  Without
  // this the workgroups of a compute unit, which start together, stay in step: all load, then all compute, and
  // memory time adds to arithmetic time instead of hiding behind it.
  RawRow<ACT, Q> r1, r2, rv;
  RawRow<float, Q> ru;
  static_for<0, Q>([&](auto q) { ru.a[decltype(q)::value] = ru.b[decltype(q)::value] = f32x4_t{0.f, 0.f, 0.f, 0.f}; });
  float cst = 0.f;
  auto fetch_batch = [&](int j0) __attribute__((always_inline)) {
    const int j = j0 + rloc;
    const int jj = j < rows_per_xcd ? j : rows_per_xcd - 1;
    const int c = (jj / B) * 8 + xcd, b = jj % B;
    static_for<0, Q>([&](auto qq) {
      constexpr int q = decltype(qq)::value;
      const int n = n0 + 8 * q;
      if constexpr (FULL) {
        r1.template fetch<q>(xproj + (long)(0 * d + c) * ldx + (long)b * L, n);
        rv.template fetch<q>(xproj + (long)(2 * d + c) * ldx + (long)b * L, n);
        r2.template fetch<q>(xproj + (long)(1 * d + c) * ldx + (long)b * L, n);
      } else {
        r1.template fetch<q>(xproj + (long)c * ldx + (long)b * L, n);
      }
      if (uin) {
        const float* pu = uin + ((long)c * B + b) * L + n;
        ru.a[q] = *reinterpret_cast<const f32x4_t*>(pu);
        ru.b[q] = *reinterpret_cast<const f32x4_t*>(pu + 4);
      }
    });
    if (FULL && tr < 15) {
      const int grp = tr / 5, k = tr % 5;
      const long ch = (long)(grp == 0 ? 0 : grp == 1 ? 2 : 1) * d + c;
      cst = k < 3 ? sw[ch * 3 + k] : k == 3 ? sb[ch] : (pbias ? pbias[ch] : 0.f);
    }
  };
  if constexpr (!TAPS) {
    if (slot * RPW < rows_per_xcd) fetch_batch(slot * RPW);
  }
  cf K[E];      // TAPS: of the thread's filter, taps and then their transform
  auto fetch_taps = [&](int j0) __attribute__((always_inline)) {
    const int j = j0 + rloc, c = ((j < rows_per_xcd ? j : rows_per_xcd - 1) / B) * 8 + xcd;
    load_taps<P>(K, filters.taps + ((long)(filters.nfilters == 2 ? sig : 0) * d + c) * (2L * L), anew(t));
  };
  if constexpr (TAPS) {
    if (slot * RPW < rows_per_xcd) fetch_taps(slot * RPW);
  }

  for (int j0 = slot * RPW; j0 < rows_per_xcd; j0 += slots * RPW) {
    const int j = j0 + rloc;
    const bool valid = j < rows_per_xcd;
    const int jj = valid ? j : rows_per_xcd - 1;
    const int c = (jj / B) * 8 + xcd, b = jj % B;

    if constexpr (TAPS) {
      fetch_batch(j0);                     // (travels while the taps are transformed)
      __builtin_amdgcn_sched_barrier(0);
      if (sig < filters.nfilters) {
        gfloat* D = filters.skip ? in_global(filters.skip[sig]) : nullptr;
        if (D && t == 0) K[0].re += D[c];      // the skip weight is one more tap at lag 0
      } else {
        static_for<0, E>([&](auto rr) { K[decltype(rr)::value] = {0.f, 0.f}; });
      }
      held_spectrum<P, kQuarter>(K, anew(t), row, tab, tf);      // (the prologue's first barrier stands between its reads and the stage)
    }

    // ---- prologue: 8 Q consecutive time steps per thread: short conv, gate, stage a and u in LDS ----
    GateRow<ACT, Q> gate;
    {
      float w1[3] = {0.f, 0.f, 0.f}, wv[3] = {0.f, 0.f, 0.f}, w2[3] = {0.f, 0.f, 0.f};
      float f1 = 0.f, fv = 0.f, f2 = 0.f, p1 = 0.f, pv = 0.f, p2 = 0.f;
      if constexpr (FULL) {
        if (tr < 15) crow[tr] = cst;
        sync_threads<RT>();
        const float4 c0 = *reinterpret_cast<const float4*>(crow), c1 = *reinterpret_cast<const float4*>(crow + 4),
                     c2 = *reinterpret_cast<const float4*>(crow + 8), c3 = *reinterpret_cast<const float4*>(crow + 12);
        w1[0] = c0.x; w1[1] = c0.y; w1[2] = c0.z; p1 = c1.x;
        wv[0] = c1.y; wv[1] = c1.z; wv[2] = c1.w; pv = c2.y;
        w2[0] = c2.z; w2[1] = c2.w; w2[2] = c3.x; p2 = c3.z;
        // The bias p of the in-projection is not added to the inputs: a 3-tap convolution of (x + p) is the
        // convolution of x plus p (w0 + w1 + w2), which goes into the convolution's own bias -- except for the first
        // two outputs of a row, where one or two taps fall on the zero padding: those are corrected.
        f1 = c0.w + p1 * (w1[0] + w1[1] + w1[2]);
        fv = c2.x + pv * (wv[0] + wv[1] + wv[2]);
        f2 = c3.y + p2 * (w2[0] + w2[1] + w2[2]);
      }
      static_for<0, Q>([&](auto qq) {
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
            if (n0 == 0) {      // time steps 0 and 1 of the row
              a[0] -= p1 * (w1[0] + w1[1]); a[1] -= p1 * w1[0];
              cv[0] -= pv * (wv[0] + wv[1]); cv[1] -= pv * wv[0];
              gt[0] -= p2 * (w2[0] + w2[1]); gt[1] -= p2 * w2[0];
            }
          }
          static_for<0, 8>([&](auto ee) { a[decltype(ee)::value] *= cv[decltype(ee)::value]; });
        } else {
          // plain long convolution: xproj is a single (d, B, L) signal, no short conv, no gates
          static_for<0, 8>([&](auto ee) {
            a[decltype(ee)::value] = in[decltype(ee)::value + 2];
            gt[decltype(ee)::value] = 1.f;
          });
        }
        gate.template set<q>(gt);
        float4* da = reinterpret_cast<float4*>(stage_a + PairLayout<P>::stage(n0) + 8 * q);
        da[0] = make_float4(a[0], a[1], a[2], a[3]);
        da[1] = make_float4(a[4], a[5], a[6], a[7]);
        f32x4_t* du = reinterpret_cast<f32x4_t*>(stage_u + PairLayout<P>::stage(n0) + 8 * q);
        du[0] = ru.a[q];
        du[1] = ru.b[q];
      });
    }
    // the next batch's loads, behind everything that read this batch's registers; where fp32 inputs and 32 points per thread do not
    // fit the registers together, behind the transforms instead
    constexpr bool kEarly = sizeof(ACT) == 2 || E == 16;
    if constexpr (kEarly && !TAPS) {
      __builtin_amdgcn_sched_barrier(0);
      if (j0 + slots * RPW < rows_per_xcd) fetch_batch(j0 + slots * RPW);
      __builtin_amdgcn_sched_barrier(0);
    }
    sync_threads<RT>();

    cf x[E];
    float* own = stage + PairLayout<P>::stage(t);
    static_for<0, E>([&](auto rr) {
      constexpr int r = decltype(rr)::value;
      x[r] = {own[PairLayout<P>::stage(T * (r / P::R1) + P::S1 * (r % P::R1))], 0.f};
    });
    sync_threads<T>();                    // the transform's slots overlap the staged row
    if constexpr (TAPS) {
      convolve_held<P, kQuarter, true>(x, anew(t), row, tab, tf, ti, K, [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        if (j0 + slots * RPW < rows_per_xcd) fetch_taps(j0 + slots * RPW);
        else static_for<0, E>([&](auto rr) { K[decltype(rr)::value] = {0.f, 0.f}; });
        __builtin_amdgcn_sched_barrier(0);
      });
    } else {
      convolve<P, kQuarter, true>(x, t, row, tab, tf, ti, spec + ((long)c * 2 + sig) * (E / 2) * T);
    }
    if constexpr (!kEarly && !TAPS) {
      __builtin_amdgcn_sched_barrier(0);
      if (j0 + slots * RPW < rows_per_xcd) {
        fetch_batch(j0 + slots * RPW);
      } else {      // (values of their own here too: otherwise this batch's inputs would stay in registers up to this point)
        static_for<0, Q>([&](auto qq) { r1.clear(qq); r2.clear(qq); rv.clear(qq); ru.clear(qq); });
        cst = 0.f;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    sync_threads<T>();
    static_for<0, E>([&](auto rr) {
      constexpr int r = decltype(rr)::value;
      own[PairLayout<P>::stage(T * (r / P::R1) + P::S1 * (r % P::R1))] = end_real<P, kQuarter, r>(x, te);
    });
    sync_threads<RT>();

    // ---- epilogue: 8 Q consecutive outputs per thread ----
    static_for<0, Q>([&](auto qq) {
      constexpr int q = decltype(qq)::value;
      const int n = n0 + 8 * q;
      const float4* pa = reinterpret_cast<const float4*>(stage_a + PairLayout<P>::stage(n0) + 8 * q);
      const float4* pu = reinterpret_cast<const float4*>(stage_u + PairLayout<P>::stage(n0) + 8 * q);
      const float4 a0 = pa[0], a1 = pa[1], u0 = pu[0], u1 = pu[1];
      float out[8];
      out[0] = a0.x * gate.template get<8 * q>() + u0.x; out[1] = a0.y * gate.template get<8 * q + 1>() + u0.y;
      out[2] = a0.z * gate.template get<8 * q + 2>() + u0.z; out[3] = a0.w * gate.template get<8 * q + 3>() + u0.w;
      out[4] = a1.x * gate.template get<8 * q + 4>() + u1.x; out[5] = a1.y * gate.template get<8 * q + 5>() + u1.y;
      out[6] = a1.z * gate.template get<8 * q + 6>() + u1.z; out[7] = a1.w * gate.template get<8 * q + 7>() + u1.w;
      if (valid) store8(y + ((long)c * B + b) * L, n, out);
    });
    sync_threads<RT>();      // the next row's prologue overwrites what the epilogue has just read
  }
}

template <class P, typename ACT, bool TAPS>
static int launch_mixer_pair(const void* xproj, long ldx, const float* u, const float* sw, const float* sb, const float* pbias,
                             const float* spec, const FilterTaps& filters, void* y, int B, int d, hipStream_t stream) {
  typedef PairLayout<P> Lay;
  auto kern = mixer_pair_kernel<P, ACT, true, TAPS>;
  if constexpr (!TAPS) {
    if (!sw) kern = mixer_pair_kernel<P, ACT, false, false>;
  }
  if (Lay::lds_bytes > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)Lay::lds_bytes);
    if (e != hipSuccess) return set_error(M2_ERR_LAUNCH, "hipFuncSetAttribute(mixer_pair): %s", hipGetErrorString(e));
  }
  const int rows_per_xcd = (d / 8) * B;
  const int slots_needed = (rows_per_xcd + Lay::RPW - 1) / Lay::RPW;
  // workgroups that are resident on a compute unit at once (registers or LDS, whichever binds): asked once per
  // kernel, the LDS bound is the fallback
  static int resident_of[2] = {0, 0};
  int& resident = resident_of[sw != nullptr];
  if (resident == 0) {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, (const void*)kern, Lay::WG, Lay::lds_bytes) != hipSuccess || n < 1)
      n = (int)((160 * 1024) / Lay::lds_bytes) < 1 ? 1 : (int)((160 * 1024) / Lay::lds_bytes);
    resident = n;
  }
  const int per_cu = resident;
  const int cus = num_cus() / 8, slots = slots_for(slots_needed, cus * (per_cu > 8 ? 8 : per_cu), cus);          // per XCD
  hipLaunchKernelGGL(kern, dim3(8 * slots), dim3(Lay::WG), Lay::lds_bytes, stream, (const ACT*)xproj, ldx, u, sw, sb, pbias,
                     (const float4*)spec, (ACT*)y, B, d, filters);
  return check_launch("mixer_pair");
}

}  // namespace m2
