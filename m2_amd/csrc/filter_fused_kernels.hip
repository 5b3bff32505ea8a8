// Implicit-filter generation for short sequences (L <= 512): the 128 -> d output projection of the filter MLPs, the
// exponential decay, the placement of forward and reverse taps in the 2L window, the skip weight and the transform
// to the spectra the mixer core consumes -- as ONE kernel, so the taps never exist in memory
// (bert/src/mm/hyena_utils.py:175,201-217 last Linear + modulation, :231-236 bidirectional window,
// :24-33 rfft(k) / 2L; launch granularity of the reference's native filter kernel,
// csrc/flashmm/flash_mm.cpp:301-362).
//
// A workgroup owns 16 or 32 channels of one filter: as many rows of L complex points in LDS (re = the first half of the 2L window, im = the second:
// fft_twist.h), exactly one batch of rows for its T threads per channel.  Phase 1: wave w projects the positions of the filter's forward (w
// even) or reverse MLP for the channels on v_mfma_f32_16x16x32_f16
// (W3 rows as the A operand, split into fp16 hi / lo parts in registers; the last hidden layer's activations,
// which the hidden kernel left in the same form, as the B operand; three products, hyena_filter.h),
// multiplies by exp(-t |delta|) + shift and drops each value at its place in the window.  Phase 2: every row is
// transformed by its T threads (same passes as the stand-alone spectrum kernel) and stored in the mixer core's
// order.  All mixers of a model go in one launch (blockIdx.y; blockIdx.z = the filter).
//
// What bounds it: a wave's positions are a chain of loads, so four tiles of 16 are requested at once; and every workgroup reads all of
// its filter's h3 out of L2 (512 bytes a position), which many mixers are bound by and 32 channels halve, while a single mixer
// leaves most compute units without a workgroup, of which 16 channels and one filter make the most.
// us for the filters of a mixer of 768 channels (all launches), both filters of 16 channels on one workgroup and one tile at a time / 16
// channels / 32 channels: one mixer L = 128 28.2 / 24.3 / 25.7, 256 37.5 / 30.1 / 32.2, 512 55.3 / 40.7 / 43.2; twelve at once 128
// 4.65 / 4.3 / 4.1, 256 7.25 / 6.6 / 6.5, 512 13.0 / 12.7 / 10.0; twelve of 1792 channels at 512 22.8 / 21.5 / 16.9, 24 of 1536 at 128
// 5.2 / 5.2 / 4.5.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fft_twist.h"
#include "hyena_filter.h"

namespace m2 {

constexpr int kFusedRows = 16;      // channels of a tile

// CT tiles of 16 channels per workgroup.
template <class P, int CT>
__global__ __launch_bounds__(CT * kFusedRows * P::T) void project_spectrum_kernel(
    const FilterPtrs* __restrict__ tab,         // fpm entries per mixer
    const float* const* __restrict__ skip,      // fpm skip-weight pointers per mixer (entries, or the table, may be null)
    int fpm, int d, float shift,
    const uint16_t* __restrict__ h_hi,          // (2 nfilters, L, 128) fp16: high parts of the last hidden layer
    const uint16_t* __restrict__ h_lo,          // low parts
    float4* __restrict__ spec, long spec_stride4) {
  constexpr int L = P::H, T = P::T, ROWS = CT * kFusedRows, NW = ROWS * T / 64;
  constexpr int kTiles = L / 16 / (NW / 2), kAhead = kTiles < 4 ? kTiles : 4;      // tiles of 16 positions of a wave, requested at once
  static_assert(NW % 2 == 0 && kTiles % kAhead == 0, "whole groups of tiles");
  extern __shared__ float2 lds[];
  float2* factors = lds + ROWS * P::ROW;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, i16 = lane & 15, q4 = lane >> 4;
  const int rloc = tid / T, t = tid % T;
  const int mixer = blockIdx.y, c0 = blockIdx.x * ROWS, which = blockIdx.z, c = c0 + rloc;
  spec += (long)mixer * spec_stride4 + ((long)c * 2 + which) * (P::E / 2) * T + t;
  if (which >= fpm) {      // no second filter
    static_for<0, P::E / 2>([&](auto pp) { spec[decltype(pp)::value * T] = make_float4(0.f, 0.f, 0.f, 0.f); });
    return;
  }
  SpectrumForward<P, kQuarter> forward;
  forward.init(t, factors);
  const int f = mixer * fpm + which;

  // ---- phase 1: projection + decay into the window ----
  {
    const int dir = wave & 1;
    gfloat *const W3 = in_global(tab[f].mlp[dir].w3), *const tt = in_global(tab[f].t), *const deltas = in_global(tab[f].deltas);
    // forward taps fill the first half of the window, reverse taps the second from its end
    auto put = [&](int ct, int p, const floatx4& v) __attribute__((always_inline)) {
      float* dst = reinterpret_cast<float*>(lds + (16 * ct + 4 * q4) * P::ROW + P::phys(dir == 0 ? p : L - 1 - p)) + dir;
#pragma unroll
      for (int j = 0; j < 4; ++j) dst[(long)j * P::ROW * 2] = v[j];
    };
    if (W3 == nullptr) {      // not bidirectional: the reverse half is zero
      for (int pt = wave >> 1; pt < L / 16; pt += NW / 2)
        for (int ct = 0; ct < CT; ++ct) put(ct, 16 * pt + i16, floatx4{0.f, 0.f, 0.f, 0.f});
    } else {
      const uint16_t* gh = h_hi + ((long)(2 * f + dir) * L + i16) * kOrder + 8 * q4;
      const uint16_t* gl = h_lo + ((long)(2 * f + dir) * L + i16) * kOrder + 8 * q4;
      u32x4 bh[kAhead][kOrder / 32], bl[kAhead][kOrder / 32];
      float tl[kAhead];
      auto request = [&](int k) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
          const int pt = (wave >> 1) + (k + u) * (NW / 2);
#pragma unroll
          for (int ks = 0; ks < kOrder / 32; ++ks) {
            bh[u][ks] = *reinterpret_cast<const u32x4*>(gh + (long)pt * 16 * kOrder + 32 * ks);
            bl[u][ks] = *reinterpret_cast<const u32x4*>(gl + (long)pt * 16 * kOrder + 32 * ks);
          }
          tl[u] = tt[16 * pt + i16];
        }
      };
      f16x8 ahi[CT][kOrder / 32], alo[CT][kOrder / 32];
      float rs[CT][4], adelta[CT][4];                     // reciprocal scales and decay rates of the lane's four channels of a tile
      float v[CT][kOrder / 4];
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        gfloat* wrow = W3 + (long)(c0 + 16 * ct + i16) * kOrder + 8 * q4;
#pragma unroll
        for (int ks = 0; ks < kOrder / 32; ++ks) {
          const floatx4 v0 = *(gfloatx4*)(wrow + 32 * ks);
          const floatx4 v1 = *(gfloatx4*)(wrow + 32 * ks + 4);
          v[ct][8 * ks] = v0.x; v[ct][8 * ks + 1] = v0.y; v[ct][8 * ks + 2] = v0.z; v[ct][8 * ks + 3] = v0.w;
          v[ct][8 * ks + 4] = v1.x; v[ct][8 * ks + 5] = v1.y; v[ct][8 * ks + 6] = v1.z; v[ct][8 * ks + 7] = v1.w;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) adelta[ct][j] = -fabsf(deltas[c0 + 16 * ct + 4 * q4 + j]) * 1.44269504088896341f;
      }
      request(0);
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        float top = 0.f;
#pragma unroll
        for (int j = 0; j < kOrder / 4; ++j) top = fmaxf(top, fabsf(v[ct][j]));
        top = fmaxf(top, __shfl_xor(top, 16));
        top = fmaxf(top, __shfl_xor(top, 32));
        const float scale = row_scale(top), back = 1.f / (scale * kActScale);
#pragma unroll
        for (int ks = 0; ks < kOrder / 32; ++ks) {
          u32x4 vh, vl;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            uint32_t h, l;
            split2(v[ct][8 * ks + 2 * j] * scale, v[ct][8 * ks + 2 * j + 1] * scale, h, l);
            vh[j] = h;
            vl[j] = l;
          }
          ahi[ct][ks] = __builtin_bit_cast(f16x8, vh);
          alo[ct][ks] = __builtin_bit_cast(f16x8, vl);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) rs[ct][j] = __shfl(back, 4 * q4 + j);
      }
      // the waves that share an MLP take its 16-position tiles in turn
      for (int k = 0;;) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) {
            floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < kOrder / 32; ++ks) {      // smallest terms first
              acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(alo[ct][ks], __builtin_bit_cast(f16x8, bh[u][ks]), acc, 0, 0, 0);
              acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi[ct][ks], __builtin_bit_cast(f16x8, bl[u][ks]), acc, 0, 0, 0);
            }
#pragma unroll
            for (int ks = 0; ks < kOrder / 32; ++ks)
              acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi[ct][ks], __builtin_bit_cast(f16x8, bh[u][ks]), acc, 0, 0, 0);
            // accumulator element j of lane (i16, q4): channel c0 + 16 ct + 4 q4 + j, position i16 of the tile.  (exp(-t |delta|) + shift) r;
            // the bare hardware exp2 flushes results below 2^-126 to zero, which is the value to 1e-38 absolute
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[j] *= fmaf(__builtin_amdgcn_exp2f(tl[u] * adelta[ct][j]), rs[ct][j], shift * rs[ct][j]);
            put(ct, 16 * ((wave >> 1) + (k + u) * (NW / 2)) + i16, acc);
          }
        }
        k += kAhead;
        if (k == kTiles) break;
        request(k);
      }
    }
  }

  // ---- phase 2: one row per T threads ----
  float2* row = lds + rloc * P::ROW;
  __syncthreads();
  cf x[P::E];
  static_for<0, P::E>([&](auto rr) {
    constexpr int r = decltype(rr)::value;
    x[r] = lds_get(row + P::phys(t + T * (r / P::R1)), P::phys(P::S1 * (r % P::R1)));
  });
  if (t == 0 && skip != nullptr) {      // the skip weight D is one more tap at lag 0
    gfloat* D = in_global(skip[f]);
    if (D) x[0].re += D[c];
  }
  forward(x, t, row, factors);
  store_spectrum<P>(x, 1.f / (float)L, spec);
}

bool project_spectrum_supported(int L) { return L == 128 || L == 256 || L == 512; }

template <class P, int CT>
static int launch_project_spectrum_t(const FilterPtrs* tab, const float* const* skip, int nmixers, int fpm, int d,
                                     float shift, const uint16_t* h_hi, const uint16_t* h_lo, float* spec,
                                     long spec_stride, hipStream_t stream) {
  constexpr int rows = CT * kFusedRows;
  const size_t lds_bytes = (size_t)(rows * P::ROW + P::TAB) * sizeof(float2);
  auto kern = project_spectrum_kernel<P, CT>;
  if (lds_bytes > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
    if (e != hipSuccess) return set_error(M2_ERR_LAUNCH, "hipFuncSetAttribute(project_spectrum): %s", hipGetErrorString(e));
  }
  hipLaunchKernelGGL(kern, dim3(d / rows, nmixers, 2), dim3(rows * P::T), lds_bytes, stream, tab, skip, fpm, d,
                     shift, h_hi, h_lo, (float4*)spec, spec_stride / 4);
  return check_launch("project_spectrum");
}

int launch_project_spectrum(const FilterPtrs* tab, const float* const* skip, int nmixers, int fpm, int L, int d,
                            float shift, const uint16_t* h_hi, const uint16_t* h_lo, float* spec, long spec_stride,
                            hipStream_t stream) {
  if (d % kFusedRows != 0) return set_error(M2_ERR_UNSUPPORTED, "project_spectrum: d=%d must be a multiple of %d", d, kFusedRows);
  // 32 channels per workgroup where 16 make more than two workgroups for every compute unit
  const bool two = d % (2 * kFusedRows) == 0 && 2l * (d / kFusedRows) * nmixers > 2l * num_cus();
  switch (L) {
#define X(LEN) \
  case LEN: return two ? launch_project_spectrum_t<Twist##LEN, 2>(tab, skip, nmixers, fpm, d, shift, h_hi, h_lo, spec, spec_stride, stream) \
                       : launch_project_spectrum_t<Twist##LEN, 1>(tab, skip, nmixers, fpm, d, shift, h_hi, h_lo, spec, spec_stride, stream);
    X(128) X(256) X(512)
#undef X
  }
  return set_error(M2_ERR_UNSUPPORTED, "project_spectrum: no plan for L=%d", L);
}

}  // namespace m2
