// Fused Monarch-Mixer sequence-mixer core for gfx950 (L = 128 .. 8192), the filter-spectrum kernel that feeds it (L up to 16384)
// and the C entry points of all lengths.
//
// One (channel, batch) row of length L: two real signals, a = shortconv(v) * shortconv(x1) and u = the layer input, are convolved
// with a 2L-tap bidirectional filter each (fft_twist.h: one complex transform of L points per signal, real in, real out), and
//
//   y[n] = (a (*) k1)[n] * shortconv(x2)[n] + (u (*) k2)[n]
//
// The skip terms "+ D1 a" and "+ D2 u" of the reference are folded into tap 0 of the filters when
// their spectra are built (k[0] += D), which is the same convolution.
//
// Replaces, for the reference's torch path, bert/src/mm/monarch_mixer_sequence_mixer.py:112-147
// together with bert/src/mm/hyena_utils.py:16-42,231-236 (two fftconv_ref calls, the gating and the
// residual add); the launch granularity corresponds to the reference's optional CUDA kernel
// csrc/flashmm/mm_block_fwd_cuda.cu:173-647 but none of that code is used here.
//
// Spectra: spec[channel][signal][register pair 0 .. E/2-1][thread 0 .. T-1] as float4, two complex numbers in exactly the order
// the multiply consumes them, 16 d L bytes; the spectrum kernel produces that order with the same passes, so the layout is
// private to these files.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fft_twist.h"
#include "hyena_filter.h"
#include "row_io.h"

namespace m2 {

#define M2_FOR_EACH_PAIR_LENGTH(X) X(128) X(256) X(512) X(1024) X(2048) X(4096) X(8192)

#define X(L) static_assert(Twist##L::H == L && twist_offsets_ok<Twist##L>(), "LDS offsets of the plan");
M2_FOR_EACH_PAIR_LENGTH(X)
#undef X

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
template <class P, typename ACT, bool FULL>
__global__ __launch_bounds__(PairLayout<P>::WG) __attribute__((amdgpu_waves_per_eu(P::E == 16 ? 3 : 2, P::E == 16 ? 3 : 2))) void mixer_pair_kernel(
    const ACT* __restrict__ xproj,      // (3d, B, L): x1 | x2 | v, channel-major
    long ldx,                           // elements between two channels of xproj, B L or more
    const float* __restrict__ uin,      // (d, B, L)   layer input, channel-major (may be null)
    const float* __restrict__ sw,       // (3d, 3)     short-conv taps
    const float* __restrict__ sb,       // (3d)        short-conv bias
    const float* __restrict__ pbias,    // (3d)        bias of the in-projection, added to xproj on load (may be null)
    const float4* __restrict__ spec,    // (d, 2, E/2, T)
    ACT* __restrict__ y,                // (d, B, L)
    int B, int d) {
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
  if (slot * RPW < rows_per_xcd) fetch_batch(slot * RPW);

  for (int j0 = slot * RPW; j0 < rows_per_xcd; j0 += slots * RPW) {
    const int j = j0 + rloc;
    const bool valid = j < rows_per_xcd;
    const int jj = valid ? j : rows_per_xcd - 1;
    const int c = (jj / B) * 8 + xcd, b = jj % B;

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
    if constexpr (kEarly) {
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
    convolve<P, kQuarter, true>(x, t, row, tab, tf, ti, spec + ((long)c * 2 + sig) * (E / 2) * T);
    if constexpr (!kEarly) {
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

// ------------------------------------------------------------------------------------------
// filter taps -> spectra; work item = (channel, filter): lo + i hi, the two halves of the 2L-tap window
// ------------------------------------------------------------------------------------------
template <class P>
struct SpectrumLayout {
  static constexpr int WG = P::T < 256 ? 256 : P::T, RPW = WG / P::T;
  static constexpr size_t lds_bytes = (size_t)(RPW * P::ROW + P::TAB) * sizeof(float2);
};

template <class P>
__global__ __launch_bounds__(SpectrumLayout<P>::WG) __attribute__((amdgpu_waves_per_eu(2, 2))) void filter_spectrum_kernel(
    const float* taps1,    // (d, 2L) bidirectional taps of filter_fn
    const float* taps2,    // (d, 2L) bidirectional taps of filter_fn2 (may be null: its spectra are zero)
    const float* D1,       // (d) skip weight of filter_fn, added to tap 0 (may be null)
    const float* D2,       // (d) skip weight of filter_fn2 (may be null)
    float4* __restrict__ spec,          // (d, 2, E/2, T)
    int d, SpectrumBatch sb) {
  constexpr int L = P::H, T = P::T, E = P::E, RPW = SpectrumLayout<P>::RPW;
  extern __shared__ float2 lds[];
  const int rloc = threadIdx.x / T, t = threadIdx.x % T;
  float2* row = lds + rloc * P::ROW;
  const float2* tab = lds + RPW * P::ROW;
  {
    float* sp = reinterpret_cast<float*>(spec);
    select_mixer(sb, d, 2 * L, taps1, taps2, D1, D2, sp);
    spec = reinterpret_cast<float4*>(sp);
  }
  SpectrumForward<P, kQuarter> forward;
  forward.init(t, lds + RPW * P::ROW);
  __syncthreads();

  for (int i0 = blockIdx.x * RPW; i0 < 2 * d; i0 += gridDim.x * RPW) {
    const int item = i0 + rloc < 2 * d ? i0 + rloc : 2 * d - 1, c = item >> 1;
    const float* taps = item & 1 ? taps2 : taps1;
    const float* D = item & 1 ? D2 : D1;
    cf x[E];
    if (taps) {
      const float* p = taps + (long)c * 2 * L + t;
      static_for<0, E>([&](auto rr) {
        constexpr int r = decltype(rr)::value, n = T * (r / P::R1) + P::S1 * (r % P::R1);
        x[r] = {p[n], p[n + L]};
      });
      if (D && t == 0) x[0].re += D[c];      // the skip weight is one more tap at lag 0
    } else {
      static_for<0, E>([&](auto rr) { x[decltype(rr)::value] = {0.f, 0.f}; });
    }
    sync_threads<T>();                       // the item before has been read
    forward(x, t, row, tab);
    if (i0 + rloc < 2 * d) store_spectrum<P>(x, 1.f / (float)L, spec + (long)item * (E / 2) * T + t);
  }
}

// ------------------------------------------------------------------------------------------
// host-side dispatch
// ------------------------------------------------------------------------------------------
template <class P, typename ACT>
static int launch_mixer_pair(const void* xproj, long ldx, const float* u, const float* sw, const float* sb, const float* pbias,
                             const float* spec, void* y, int B, int d, hipStream_t stream) {
  typedef PairLayout<P> Lay;
  auto kern = sw ? mixer_pair_kernel<P, ACT, true> : mixer_pair_kernel<P, ACT, false>;
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
                     (const float4*)spec, (ACT*)y, B, d);
  return check_launch("mixer_pair");
}

template <class P>
static int launch_filter_spectrum(const float* taps1, const float* taps2, const float* D1, const float* D2,
                                  float* spec, int d, const SpectrumBatch& sb, int nmixers, hipStream_t stream) {
  typedef SpectrumLayout<P> Lay;
  auto kern = filter_spectrum_kernel<P>;
  if (Lay::lds_bytes > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)Lay::lds_bytes);
    if (e != hipSuccess) return set_error(M2_ERR_LAUNCH, "hipFuncSetAttribute(filter_spectrum): %s", hipGetErrorString(e));
  }
  const int wgs_needed = (2 * d + Lay::RPW - 1) / Lay::RPW;
  int grid = num_cus() * 2;
  if (grid > wgs_needed) grid = wgs_needed;
  hipLaunchKernelGGL(kern, dim3(grid, nmixers), dim3(Lay::WG), Lay::lds_bytes, stream, taps1, taps2, D1, D2, (float4*)spec, d, sb);
  return check_launch("filter_spectrum");
}

// L = 32768 (two half transforms of 16384 points per signal), defined in fftconv_real_kernels.hip
int launch_mixer_real_dispatch(const void* xproj, long ldx, const float* u, const float* sw, const float* sb, const float* pbias,
                               const float* spec, void* y, int B, int d, int act_dtype, hipStream_t stream);
int launch_filter_spectrum_real(const float* taps1, const float* taps2, const float* D1, const float* D2, float* spec,
                                int d, const SpectrumBatch& sb, int nmixers, hipStream_t stream);

// L = 8192 and 16384, one signal after the other: defined in fftconv_long_kernels.hip
int launch_mixer_long_dispatch(const void* xproj, long ldx, const float* u, const float* sw, const float* sb, const float* pbias,
                               const float* spec, void* y, int B, int L, int d, int act_dtype, hipStream_t stream);

// One mixer given by pointers (sb.taps null, nmixers 1) or a batch of mixers described by `sb`.
int launch_filter_spectrum_any(const float* taps1, const float* taps2, const float* D1, const float* D2, float* spec,
                               int d, int L, const SpectrumBatch& sb, int nmixers, hipStream_t stream) {
  switch (L) {
    case 32768: return launch_filter_spectrum_real(taps1, taps2, D1, D2, spec, d, sb, nmixers, stream);
#define X(LEN)   case LEN: return launch_filter_spectrum<Twist##LEN>(taps1, taps2, D1, D2, spec, d, sb, nmixers, stream);
    M2_FOR_EACH_PAIR_LENGTH(X) X(16384)
#undef X
  }
  return set_error(M2_ERR_UNSUPPORTED, "filter spectrum: no plan for L=%d", L);
}

// sw null: plain convolution of a (d, B, L) input
static int launch_mixer_any(const void* xproj, long ldx, const float* u, const float* sw, const float* sb, const float* pbias,
                            const float* spec, void* y, int B, int L, int d, int act_dtype, hipStream_t s) {
  // L = 8192: with both signals at once a compute unit holds one row, one after the other it holds two and each row takes 1.87 times as
  // long, their barriers hidden behind each other (B = 4: 172 us against 184).  Which of the two leaves fewer units idle in its
  // last round decides where that is more than they differ by (B = 1, d = 768, three rows per unit: 47 us against 56).
  const long rows = (long)d * B, cus = num_cus();
  const bool one_by_one = L == 8192 && (rows + cus - 1) / cus * 100 * cus > 93 * ((rows + 2 * cus - 1) / (2 * cus) * 2 * cus);
  if (L == 16384 || one_by_one) return launch_mixer_long_dispatch(xproj, ldx, u, sw, sb, pbias, spec, y, B, L, d, act_dtype, s);
  switch (L) {
    case 32768: return launch_mixer_real_dispatch(xproj, ldx, u, sw, sb, pbias, spec, y, B, d, act_dtype, s);
#define X(LEN)                                                                                                     case LEN:                                                                                                          return act_dtype == M2_DTYPE_F32 ? launch_mixer_pair<Twist##LEN, float>(xproj, ldx, u, sw, sb, pbias, spec, y, B, d, s)                                      : launch_mixer_pair<Twist##LEN, uint16_t>(xproj, ldx, u, sw, sb, pbias, spec, y, B, d, s);
    M2_FOR_EACH_PAIR_LENGTH(X)
#undef X
  }
  return set_error(M2_ERR_UNSUPPORTED, "mixer core: no plan for L=%d", L);
}

}  // namespace m2

using namespace m2;

extern "C" int m2_fftconv_supported_seqlen(int L) {
  return (L >= 128 && L <= 32768 && (L & (L - 1)) == 0) ? 1 : 0;
}

extern "C" size_t m2_filter_spectrum_bytes(int d, int L) {
  return (size_t)d * (size_t)L * 16;        // d channels x 2 signals x L complex numbers
}

extern "C" int m2_filter_spectrum_fwd(const float* taps1, const float* taps2, const float* D1, const float* D2,
                                      float* spec, int d, int L, void* stream) {
  if (!taps1 || !spec) return set_error(M2_ERR_ARG, "m2_filter_spectrum_fwd: null pointer");
  if (d <= 0) return set_error(M2_ERR_ARG, "m2_filter_spectrum_fwd: d must be positive, got %d", d);
  if (!m2_fftconv_supported_seqlen(L))
    return set_error(M2_ERR_UNSUPPORTED, "m2_filter_spectrum_fwd: L=%d unsupported (need L a power of two in [128, 32768])", L);
  const SpectrumBatch none{nullptr, nullptr, 0, 0};
  return launch_filter_spectrum_any(taps1, taps2, D1, D2, spec, d, L, none, 1, (hipStream_t)stream);
}

static int mixer_core(const char* who, const void* xproj, long ldx, const float* proj_bias, const float* u, const float* short_w,
                                 const float* short_b, const float* spec, void* y, int B, int L, int d, int act_dtype,
                                 void* stream) {
  if (!xproj || !short_w || !short_b || !spec || !y) return set_error(M2_ERR_ARG, "%s: null pointer", who);
  if (B <= 0 || d <= 0 || d % 8 != 0) return set_error(M2_ERR_ARG, "%s: need B > 0 and d a positive multiple of 8 (B=%d d=%d)", who, B, d);
  if ((long)B * 3 * d > 0x7fffffffL) return set_error(M2_ERR_UNSUPPORTED, "%s: B * 3 d = %ld rows do not fit an int", who, (long)B * 3 * d);
  if (act_dtype != M2_DTYPE_F32 && act_dtype != M2_DTYPE_BF16)
    return set_error(M2_ERR_ARG, "%s: act_dtype %d is neither M2_DTYPE_F32 nor M2_DTYPE_BF16", who, act_dtype);
  if (!m2_fftconv_supported_seqlen(L))
    return set_error(M2_ERR_UNSUPPORTED, "%s: L=%d unsupported (need L a power of two in [128, 32768])", who, L);
  if (ldx < (long)B * L || ldx % 8) return set_error(M2_ERR_ARG, "%s: rows of xproj %ld apart, need a multiple of 8 from B * L = %ld on", who, ldx, (long)B * L);
  return launch_mixer_any(xproj, ldx, u, short_w, short_b, proj_bias, spec, y, B, L, d, act_dtype, (hipStream_t)stream);
}

extern "C" int m2_mixer_core_fwd(const void* xproj, const float* proj_bias, const float* u, const float* short_w,
                                 const float* short_b, const float* spec, void* y, int B, int L, int d, int act_dtype,
                                 void* stream) {
  return mixer_core("m2_mixer_core_fwd", xproj, (long)B * L, proj_bias, u, short_w, short_b, spec, y, B, L, d, act_dtype, stream);
}

extern "C" int m2_mixer_core_rows_fwd(const void* xproj, long xproj_row, const float* proj_bias, const float* u, const float* short_w,
                                      const float* short_b, const float* spec, void* y, int B, int L, int d, int act_dtype,
                                      void* stream) {
  return mixer_core("m2_mixer_core_rows_fwd", xproj, xproj_row, proj_bias, u, short_w, short_b, spec, y, B, L, d, act_dtype, stream);
}

extern "C" int m2_fftconv_fwd(const void* x, const float* spec, void* y, int B, int L, int d, int act_dtype,
                              void* stream) {
  if (!x || !spec || !y) return set_error(M2_ERR_ARG, "m2_fftconv_fwd: null pointer");
  if (B <= 0 || d <= 0 || d % 8 != 0) return set_error(M2_ERR_ARG, "m2_fftconv_fwd: need B > 0 and d a positive multiple of 8 (B=%d d=%d)", B, d);
  if ((long)B * d > 0x7fffffffL) return set_error(M2_ERR_UNSUPPORTED, "m2_fftconv_fwd: B * d = %ld rows do not fit an int", (long)B * d);
  if (act_dtype != M2_DTYPE_F32 && act_dtype != M2_DTYPE_BF16)
    return set_error(M2_ERR_ARG, "m2_fftconv_fwd: act_dtype %d is neither M2_DTYPE_F32 nor M2_DTYPE_BF16", act_dtype);
  if (!m2_fftconv_supported_seqlen(L))
    return set_error(M2_ERR_UNSUPPORTED, "m2_fftconv_fwd: L=%d unsupported (need L a power of two in [128, 32768])", L);
  return launch_mixer_any(x, (long)B * L, nullptr, nullptr, nullptr, nullptr, spec, y, B, L, d, act_dtype, (hipStream_t)stream);
}
