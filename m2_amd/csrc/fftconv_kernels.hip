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
#include "mixer_pair.h"

namespace m2 {

#define M2_FOR_EACH_PAIR_LENGTH(X) X(128) X(256) X(512) X(1024) X(2048) X(4096) X(8192)

#define X(L) static_assert(Twist##L::H == L && twist_offsets_ok<Twist##L>(), "LDS offsets of the plan");
M2_FOR_EACH_PAIR_LENGTH(X)
#undef X

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
    gfloat* D = in_global(item & 1 ? D2 : D1);
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
#define X(LEN)                                                                                                     case LEN:                                                                                                          return act_dtype == M2_DTYPE_F32 ? launch_mixer_pair<Twist##LEN, float, false>(xproj, ldx, u, sw, sb, pbias, spec, FilterTaps{}, y, B, d, s)                                      : launch_mixer_pair<Twist##LEN, uint16_t, false>(xproj, ldx, u, sw, sb, pbias, spec, FilterTaps{}, y, B, d, s);
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
