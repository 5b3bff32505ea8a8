// Types shared by the filter-generation translation units (hyena_filter_kernels.hip, filter_fused_kernels.hip):
// the pointer table of a batch of implicit filters and the helpers that turn fp32 values into fp16 parts for
// the matrix cores.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fft_regs.h"
#include "m2_internal.h"

namespace m2 {

constexpr int kOrder = 128;
constexpr int kMaxEmb = 8;

struct MlpPtrs {
  const float *w0, *b0, *w1, *b1, *w2, *b2, *w3;
};
struct FilterPtrs {
  const float *z, *t, *freq, *deltas;
  MlpPtrs mlp[2];                 // [0] forward, [1] reverse (all null when the filter is not bidirectional)
};
// the public struct is the same eighteen pointers in the same order, so a device array of it is a table of these
static_assert(sizeof(FilterPtrs) == sizeof(m2_hyena_filter_params), "pointer table layout");

// A batch of filters reaches the kernels either inside the kernel arguments (up to kMaxFilters: the entry point
// that takes a host array) or as a table in device memory (any number: the entry point for all mixers of a model).
constexpr int kMaxFilters = 4;
struct FilterBatch {
  FilterPtrs f[kMaxFilters];
};
struct TabByValue {
  FilterBatch fb;
  __device__ __forceinline__ const FilterPtrs& at(int i) const { return fb.f[i]; }
};
struct TabByPointer {
  const FilterPtrs* p;
  __device__ __forceinline__ const FilterPtrs& at(int i) const { return p[i]; }
};

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// The matrix products of the filter MLPs: either operand as two fp16 parts, x 2^e = hi + lo, three products (hi lo, lo hi, hi hi),
// fp32 accumulation.  Two parts hold 23 - 24 bits and the product left out is below 2^-24 of the whole one, so a product is good to
// what fp32 arithmetic gives.  fp16 has five bits of exponent: e scales activations (|h| <= 1) by 2^13 and every row of a weight
// so that its largest entry lies in [2^12, 2^13), which keeps entries down to 2^-16 of the largest exact to 2^-24 of themselves and
// all others to 2^-38 of the largest.  (Three bf16 parts and six products, which this took over from, are exact and cost twice the
// matrix instructions, half as many conversions again and half as many registers for stationary weights again.)
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
constexpr float kActScale = 8192.f;      // 2^13

// two values -> their high and low parts, packed
__device__ __forceinline__ void split2(float a, float b, uint32_t& hi, uint32_t& lo) {
  const f16x2 h = __builtin_convertvector(f32x2{a, b}, f16x2);
  const f32x2 back = __builtin_convertvector(h, f32x2);
  hi = __builtin_bit_cast(uint32_t, h);
  lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a - back.x, b - back.y}, f16x2));
}
// Scale of a row whose largest magnitude is m: 2^e.  (A row below 2^-47 is scaled by 2^60, no more: its reciprocal multiplies biases.)
__device__ __forceinline__ float row_scale(float m) {
  int e = 12 - (int)((__float_as_uint(m) >> 23) & 0xff) + 127;      // -116 (infinity) ...
  e = e > 60 ? 60 : e;
  return __uint_as_float((uint32_t)(127 + e) << 23);
}

// Spectrum kernels of a batch of mixers: blockIdx.y selects the mixer.  taps: filter f of mixer m at
// taps + (m fpm + f) d 2L; skip: device array of fpm pointers per mixer (skip weights, entries may be null);
// spectra of mixer m at spec + m spec_stride floats.  taps == nullptr: a single mixer given by the kernel's own
// taps1 / taps2 / D1 / D2 arguments.
struct SpectrumBatch {
  const float* taps;
  const float* const* skip;
  int fpm;
  long spec_stride;
};
__device__ __forceinline__ void select_mixer(const SpectrumBatch& sb, int d, int N, const float*& taps1,
                                             const float*& taps2, const float*& D1, const float*& D2, float*& spec) {
  if (sb.taps == nullptr) return;
  const int m = blockIdx.y;
  taps1 = sb.taps + (long)(m * sb.fpm) * d * N;
  taps2 = sb.fpm == 2 ? taps1 + (long)d * N : nullptr;
  D1 = sb.skip ? sb.skip[m * sb.fpm] : nullptr;
  D2 = (sb.skip && sb.fpm == 2) ? sb.skip[m * sb.fpm + 1] : nullptr;
  spec += (long)m * sb.spec_stride;
}

// launchers defined beside their kernels
int launch_filter_spectrum_any(const float* taps1, const float* taps2, const float* D1, const float* D2, float* spec,
                               int d, int L, const SpectrumBatch& sb, int nmixers, hipStream_t stream);
bool project_spectrum_supported(int L);
int launch_project_spectrum(const FilterPtrs* tab, const float* const* skip, int nmixers, int fpm, int L, int d,
                            float shift, const uint16_t* h_hi, const uint16_t* h_lo, float* spec, long spec_stride,
                            hipStream_t stream);

}  // namespace m2
