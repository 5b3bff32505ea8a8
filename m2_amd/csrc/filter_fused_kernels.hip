// Implicit-filter generation for short sequences (L <= 512): the 128 -> d output projection of the filter MLPs, the
// exponential decay, the placement of forward and reverse taps in the 2L window, the skip weight and the transform
// to the spectra the mixer core consumes -- as ONE kernel, so the taps never exist in memory
// (bert/src/mm/hyena_utils.py:175,201-217 last Linear + modulation, :231-236 bidirectional window,
// :24-33 rfft(k) / 2L; launch granularity of the reference's native filter kernel,
// csrc/flashmm/flash_mm.cpp:301-362).
//
// A workgroup owns 16 channels of one mixer: 32 rows of L complex points in LDS (one per channel and filter; re = the first half
// of the 2L window, im = the second: fft_twist.h), exactly one batch of rows for its 32 T threads.  Phase 1: wave w projects the positions of
// MLP w mod nmlp (forward / reverse MLP of either filter) for the 16 channels on v_mfma_f32_16x16x32_f16
// (W3 rows as the A operand, split into fp16 hi / lo parts in registers; the last hidden layer's activations,
// which the hidden kernel left in the same form, as the B operand; three products, hyena_filter.h),
// multiplies by exp(-t |delta|) + shift and drops each value at its place in the window.  Phase 2: every row is
// transformed by its T threads (same passes as the stand-alone spectrum kernel) and stored in the mixer core's
// order.  All mixers of a model go in one launch (blockIdx.y).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fft_twist.h"
#include "hyena_filter.h"

namespace m2 {

constexpr int kFusedRows = 16;      // channels per workgroup

template <class P>
__global__ __launch_bounds__(2 * kFusedRows * P::T) void project_spectrum_kernel(
    const FilterPtrs* __restrict__ tab,         // fpm entries per mixer
    const float* const* __restrict__ skip,      // fpm skip-weight pointers per mixer (entries, or the table, may be null)
    int fpm, int d, float shift,
    const uint16_t* __restrict__ h_hi,          // (2 nfilters, L, 128) fp16: high parts of the last hidden layer
    const uint16_t* __restrict__ h_lo,          // low parts
    float4* __restrict__ spec, long spec_stride4) {
  constexpr int L = P::H, T = P::T, NT = 2 * kFusedRows * T, NW = NT / 64;
  extern __shared__ float2 lds[];
  float2* factors = lds + 2 * kFusedRows * P::ROW;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, i16 = lane & 15, q4 = lane >> 4;
  SpectrumForward<P, kQuarter> forward;
  forward.init(tid % T, factors);
  const int mixer = blockIdx.y, c0 = blockIdx.x * kFusedRows;
  const int nmlp = 2 * fpm;

  // parts of the window nobody writes: the second filter's rows without a second filter, the reverse half
  // without reverse MLPs
  const bool bidir = tab[mixer * fpm].mlp[1].w3 != nullptr;
  if (fpm == 1 || !bidir) {
    for (int i = tid; i < 2 * kFusedRows * P::ROW; i += NT) lds[i] = make_float2(0.f, 0.f);
    __syncthreads();
  }

  // ---- phase 1: projection + decay into the window ----
  {
    const int m = __builtin_amdgcn_readfirstlane(wave) % nmlp, which = m >> 1, dir = m & 1;
    const int f = mixer * fpm + which;
    gfloat *const W3 = in_global(tab[f].mlp[dir].w3), *const tt = in_global(tab[f].t), *const deltas = in_global(tab[f].deltas);
    if (W3 != nullptr) {
      f16x8 ahi[kOrder / 32], alo[kOrder / 32];
      float rs[4];                     // reciprocal scales of the lane's four channels
      {
        gfloat* wrow = W3 + (long)(c0 + i16) * kOrder + 8 * q4;
        float v[kOrder / 4], top = 0.f;
#pragma unroll
        for (int ks = 0; ks < kOrder / 32; ++ks) {
          const floatx4 v0 = *(gfloatx4*)(wrow + 32 * ks);
          const floatx4 v1 = *(gfloatx4*)(wrow + 32 * ks + 4);
          v[8 * ks] = v0.x; v[8 * ks + 1] = v0.y; v[8 * ks + 2] = v0.z; v[8 * ks + 3] = v0.w;
          v[8 * ks + 4] = v1.x; v[8 * ks + 5] = v1.y; v[8 * ks + 6] = v1.z; v[8 * ks + 7] = v1.w;
        }
#pragma unroll
        for (int j = 0; j < kOrder / 4; ++j) top = fmaxf(top, fabsf(v[j]));
        top = fmaxf(top, __shfl_xor(top, 16));
        top = fmaxf(top, __shfl_xor(top, 32));
        const float scale = row_scale(top), back = 1.f / (scale * kActScale);
#pragma unroll
        for (int ks = 0; ks < kOrder / 32; ++ks) {
          u32x4 vh, vl;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            uint32_t h, l;
            split2(v[8 * ks + 2 * j] * scale, v[8 * ks + 2 * j + 1] * scale, h, l);
            vh[j] = h;
            vl[j] = l;
          }
          ahi[ks] = __builtin_bit_cast(f16x8, vh);
          alo[ks] = __builtin_bit_cast(f16x8, vl);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) rs[j] = __shfl(back, 4 * q4 + j);
      }
      float adelta[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) adelta[j] = -fabsf(deltas[c0 + 4 * q4 + j]) * 1.44269504088896341f;
      const uint16_t* gh = h_hi + ((long)(2 * f + dir) * L + i16) * kOrder + 8 * q4;
      const uint16_t* gl = h_lo + ((long)(2 * f + dir) * L + i16) * kOrder + 8 * q4;
      // the waves that share an MLP take its 16-position tiles in turn
      for (int pt = wave / nmlp; pt < L / 16; pt += NW / nmlp) {
        u32x4 bh[kOrder / 32], bl[kOrder / 32];
#pragma unroll
        for (int ks = 0; ks < kOrder / 32; ++ks) {
          bh[ks] = *reinterpret_cast<const u32x4*>(gh + (long)pt * 16 * kOrder + 32 * ks);
          bl[ks] = *reinterpret_cast<const u32x4*>(gl + (long)pt * 16 * kOrder + 32 * ks);
        }
        const int p = 16 * pt + i16;
        const float tl = tt[p];
        floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < kOrder / 32; ++ks) {      // smallest terms first
          acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(alo[ks], __builtin_bit_cast(f16x8, bh[ks]), acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi[ks], __builtin_bit_cast(f16x8, bl[ks]), acc, 0, 0, 0);
        }
#pragma unroll
        for (int ks = 0; ks < kOrder / 32; ++ks)
          acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi[ks], __builtin_bit_cast(f16x8, bh[ks]), acc, 0, 0, 0);
        // accumulator element j of lane (i16, q4): channel c0 + 4 q4 + j, position p
        // forward taps fill the first half of the window, reverse taps the second from its end
        float* dst = reinterpret_cast<float*>(lds + (8 * q4 + which) * P::ROW + P::phys(dir == 0 ? p : L - 1 - p)) + dir;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          // (exp(-t |delta|) + shift) r; the bare hardware exp2 flushes results below 2^-126 to zero, which is the value to
          // 1e-38 absolute
          const float decay = fmaf(__builtin_amdgcn_exp2f(tl * adelta[j]), rs[j], shift * rs[j]);
          dst[(long)j * P::ROW * 4] = acc[j] * decay;
        }
      }
    }
  }

  // ---- phase 2: one row per T threads ----
  const int rloc = threadIdx.x / T, t = threadIdx.x % T, which = rloc & 1, c = c0 + (rloc >> 1);
  float2* row = lds + rloc * P::ROW;
  __syncthreads();
  cf x[P::E];
  static_for<0, P::E>([&](auto rr) {
    constexpr int r = decltype(rr)::value;
    x[r] = lds_get(row + P::phys(t + T * (r / P::R1)), P::phys(P::S1 * (r % P::R1)));
  });
  if (t == 0 && skip != nullptr && which < fpm) {      // the skip weight D is one more tap at lag 0
    gfloat* D = in_global(skip[mixer * fpm + which]);
    if (D) x[0].re += D[c];
  }
  forward(x, t, row, factors);
  store_spectrum<P>(x, 1.f / (float)L, spec + (long)mixer * spec_stride4 + ((long)c * 2 + which) * (P::E / 2) * T + t);
}

bool project_spectrum_supported(int L) { return L == 128 || L == 256 || L == 512; }

template <class P>
static int launch_project_spectrum_t(const FilterPtrs* tab, const float* const* skip, int nmixers, int fpm, int d,
                                     float shift, const uint16_t* h_hi, const uint16_t* h_lo, float* spec,
                                     long spec_stride, hipStream_t stream) {
  const size_t lds_bytes = (size_t)(2 * kFusedRows * P::ROW + P::TAB) * sizeof(float2);
  auto kern = project_spectrum_kernel<P>;
  if (lds_bytes > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
    if (e != hipSuccess) return set_error(M2_ERR_LAUNCH, "hipFuncSetAttribute(project_spectrum): %s", hipGetErrorString(e));
  }
  hipLaunchKernelGGL(kern, dim3(d / kFusedRows, nmixers), dim3(2 * kFusedRows * P::T), lds_bytes, stream, tab, skip, fpm, d,
                     shift, h_hi, h_lo, (float4*)spec, spec_stride / 4);
  return check_launch("project_spectrum");
}

int launch_project_spectrum(const FilterPtrs* tab, const float* const* skip, int nmixers, int fpm, int L, int d,
                            float shift, const uint16_t* h_hi, const uint16_t* h_lo, float* spec, long spec_stride,
                            hipStream_t stream) {
  if (d % kFusedRows != 0) return set_error(M2_ERR_UNSUPPORTED, "project_spectrum: d=%d must be a multiple of %d", d, kFusedRows);
  switch (L) {
#define X(LEN) \
  case LEN: return launch_project_spectrum_t<Twist##LEN>(tab, skip, nmixers, fpm, d, shift, h_hi, h_lo, spec, spec_stride, stream);
    X(128) X(256) X(512)
#undef X
  }
  return set_error(M2_ERR_UNSUPPORTED, "project_spectrum: no plan for L=%d", L);
}

}  // namespace m2
