// Types shared by the filter-generation translation units (hyena_filter_kernels.hip, filter_fused_kernels.hip):
// the pointer table of a batch of implicit filters and the helpers that turn fp32 values into bf16 or fp16 parts for
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

// The tables hold plain pointers, of which a kernel cannot know that they point to device memory.  Loads through them were flat ones,
// whose results come back out of order with LDS reads: every wait for an LDS read was a wait for them too; and where a kernel stores,
// the pointer itself was loaded again for each use, in a wait for all that was in flight.  So kernels take a filter's pointers
// out of the table once, at their start, through in_global.  us for the filters of a mixer of 768 channels, with the 64-bit vector address
// that each store of a tap had, before / now: 12 mixers at once L = 1024 13.4 / 12.9, 4096 45.2 / 43.4, 8192 82.2 / 80.1, three at 32768
// 336 / 326; one mixer 512 55.0 / 52.9, 1024 45.7 / 43.8, 4096 61.7 / 59.6, 8192 96.8 / 92.5.
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(1))) floatx4 gfloatx4;
typedef floatx4 floatx4_any __attribute__((aligned(4)));      // at any address of a float
typedef const __attribute__((address_space(1))) floatx4_any gfloatx4_any;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// The matrix products of the filter MLPs, fp32 accumulation.
//
// The two 128 x 128 layers: either operand as three bf16 parts, x = hi + mid + lo, which hold all 24 bits of an fp32 value of any size,
// and the six products down to 2^-24 of the whole one (mid lo, lo mid and lo lo, below 2^-24, are left out).  What such a layer loses,
// sin(freq x) of the next one amplifies by its argument.  So the five small products of a sum are added apart from the leading ones: in
// one sum of all six each is a rounding of the whole, which leaves an argument off by 0.9e-7 of itself where it is 0.2e-7 now, and a
// whole fp32 mixer 3.8e-7 from fp64 where it is 2.9e-7 now (L = 128; 4.3e-7 and 3.7e-7 at 8192).  (Two fp16 parts and three products, as
// below, save half of the matrix instructions, 5 to 10 % of filter generation, and with operands whose mantissas lie between two numbers
// of 11 bits they put every argument off by 2.6e-7 of itself.)
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ void split3(float x, float& hi, float& mid, float& lo) {
  hi = bf16_to_f32(f32_to_bf16(x));
  const float r = x - hi;
  mid = bf16_to_f32(f32_to_bf16(r));
  lo = r - mid;                      // the conversion of lo to bf16 happens where it is packed
}

// The output projection, whose result nothing amplifies: two fp16 parts, x 2^e = hi + lo, three products (hi lo, lo hi, hi hi).  The
// parts hold a value to 2^-23 of itself and the product left out is at most 2^-22 of the whole one (the error of a product is 2^-21
// at most and 2^-23.7 in the root mean square).  fp16 has five bits of exponent: every row of the weight is scaled so that its largest
// entry lies in [2^12, 2^13), activations, of which 1 is the largest possible, by 2^13.  What is below 2^-13 of the largest has its low
// part among fp16's subnormal numbers and is held to 2^-38 of the largest: of activations 2^-38, whatever their size (two bf16 parts
// held 2^-17 of any value, which is more for activations that are all below 2^-21).  Two bf16 parts (16 bits, the same matrix instructions) left the taps at 4e-6 from fp64, these
// leave them where fp32 arithmetic does, at 2e-7; a third part would double the instructions.
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
// Scale of a row whose largest magnitude is m: 2^e.  (A row below 2^-47 is scaled by 2^60, no more.)
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
