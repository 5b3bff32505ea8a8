// Helpers shared by the translation units of libm2_amd.so (not part of the public C ABI).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/m2_amd.h"

namespace m2 {

// Records a printf-style message retrievable through m2_last_error() and returns `code`.
int set_error(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
// hipGetLastError() after a launch -> 0 or M2_ERR_LAUNCH (message recorded).
int check_launch(const char* what);
// The direct global -> LDS loads take whole 16-byte pieces at 16-byte addresses.
inline bool aligned16(const void* a, const void* b = nullptr, const void* c = nullptr, const void* d = nullptr) {
  return (((uintptr_t)a | (uintptr_t)b | (uintptr_t)c | (uintptr_t)d) & 15) == 0;
}

// Compute units of the current device (cached per device).
int num_cus();

// Block-diagonal products on the dense kernels (dense_kernels.hip): x (M, nb p) bf16, w (nb, q, p) bf16.
bool glu_few_rows_pays(int M, int nb, int p);
int glu_few_rows(const void* x, const void* w, void* out, int M, int nb, int p, int q, hipStream_t stream);
int blockdiag_linear_engine(const void* x, const void* w, const float* bias, const void* resid, void* out, int M, int nb, int p,
                            int q, hipStream_t stream);

// OUT (N, M) = W (N, K) X (M, K)^T with the weights in registers (dense_ws_kernels.hip), rows of OUT ldo elements apart.
bool dense_ws_serves(int M, int N, int K);
int dense_ws_launch(const void* x, const void* w, void* out, int M, int N, long ldo, hipStream_t stream);

// A pointer that was read from memory, said to point to device memory: loads through it are global ones and not flat ones.
typedef const __attribute__((address_space(1))) float gfloat;
__device__ __forceinline__ gfloat* in_global(const float* p) { return (gfloat*)p; }

// LayerNorm of a row of D values with its roundings said, for the kernels that have to give the same bits.  `sum` and `sq` are the sums over the row of the
// values and of their squared distances to the mean, of which a lane's N values give ln_squares.
template <int D>
__device__ __forceinline__ float ln_centred(float v, float sum) { return fmaf(-sum, 1.0f / (float)D, v); }      // value - mean, one rounding
template <int D, int N>
__device__ __forceinline__ float ln_squares(const float (&v)[N], float sum) {
  const float c0 = ln_centred<D>(v[0], sum);
  float sq = c0 * c0;
#pragma unroll
  for (int i = 1; i < N; ++i) {
    const float c = ln_centred<D>(v[i], sum);
    sq = i == 1 ? fmaf(c0, c0, c * c) : fmaf(c, c, sq);
  }
  return sq;
}
template <int D>
__device__ __forceinline__ float ln_rstd(float sq, float eps) { return rsqrtf(fmaf(sq, 1.0f / (float)D, eps)); }
template <int D>
__device__ __forceinline__ float ln_value(float v, float sum, float rstd, float gamma, float beta) {
  return fmaf(ln_centred<D>(v, sum) * rstd, gamma, beta);
}

// round-to-nearest-even float -> bfloat16 bits (NaN stays NaN)
// float -> bf16 bits, round to nearest even (host restatement of what v_cvt_pk_bf16_f32 does)
__host__ __device__ __forceinline__ uint16_t f32_to_bf16_bits(float f) {
  union { float f; uint32_t u; } v;
  v.f = f;
  if ((v.u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((v.u >> 16) | 0x40u);
  v.u += 0x7fffu + ((v.u >> 16) & 1u);
  return (uint16_t)(v.u >> 16);
}
__host__ __device__ __forceinline__ float bf16_to_f32(uint16_t h) {
  union { float f; uint32_t u; } v;
  v.u = ((uint32_t)h) << 16;
  return v.f;
}

// two floats -> packed bf16 pair (lo in bits 0..15), round to nearest even; one v_cvt_pk_bf16_f32 on the device
__host__ __device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  f32x2 v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
#else
  return (uint32_t)f32_to_bf16_bits(lo) | ((uint32_t)f32_to_bf16_bits(hi) << 16);
#endif
}
__host__ __device__ __forceinline__ uint16_t f32_to_bf16(float f) {
#if defined(__HIP_DEVICE_COMPILE__)
  return (uint16_t)pack_bf16x2(f, 0.f);            // the hardware conversion: no branches
#else
  return f32_to_bf16_bits(f);
#endif
}

}  // namespace m2
