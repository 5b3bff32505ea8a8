// The pooler behind a forward: out (B, d) = tanh(h W^T + bias) in fp32, h the first token's row of each sequence (rows h_row apart),
// W (d, d) (bert/src/bert_layers.py:816-859).
//
// A few rows of a 768 x 768 product: what it takes is a launch and one trip to memory, which the library's product and the tanh behind it made
// twice (9.4 and 4.9 us in a trace).  us per forward, L = 128, B = 1, before / now: 12 x 768 501 / 492, 24 x 1536 1724 / 1709.  A wave has two columns
// and up to eight rows, its lanes share K, and the sums meet in the lanes.  Every eight rows read the whole weight again: d = 768 B = 8 7.7 us,
// 64 10.8, 256 22, where the library's product with its tanh stays at 7.0, 7.2, 9.3; encoder.py sends it eight sequences at most.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fft_regs.h"
#include "m2_internal.h"

namespace m2 {

typedef float floatx4 __attribute__((ext_vector_type(4)));
constexpr int kPoolCols = 2;      // of a wave; four waves per workgroup

template <int ROWS>
__global__ __launch_bounds__(256) void pooler_kernel(const float* __restrict__ h, long h_row, const float* __restrict__ w,
                                                     const float* __restrict__ bias, float* __restrict__ out, int B, int d) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c0 = (int)(blockIdx.x * 4 + wave) * kPoolCols, b0 = (int)blockIdx.y * ROWS;      // (d is a multiple of 8)
  float acc[ROWS][kPoolCols];
  static_for<0, ROWS>([&](auto r) { static_for<0, kPoolCols>([&](auto c) { acc[decltype(r)::value][decltype(c)::value] = 0.f; }); });
#pragma unroll 4
  for (int k = 4 * lane; k < d; k += 256) {
    floatx4 wv[kPoolCols], hv[ROWS];
    static_for<0, kPoolCols>([&](auto c) { wv[decltype(c)::value] = *reinterpret_cast<const floatx4*>(w + (long)(c0 + decltype(c)::value) * d + k); });
    static_for<0, ROWS>([&](auto r) {
      const int b = b0 + decltype(r)::value < B ? b0 + decltype(r)::value : B - 1;
      hv[decltype(r)::value] = *reinterpret_cast<const floatx4*>(h + b * h_row + k);
    });
    static_for<0, ROWS>([&](auto r) {
      static_for<0, kPoolCols>([&](auto c) {
        const floatx4 a = hv[decltype(r)::value], v = wv[decltype(c)::value];
        float& s = acc[decltype(r)::value][decltype(c)::value];
        s = fmaf(a.x, v.x, s);
        s = fmaf(a.y, v.y, s);
        s = fmaf(a.z, v.z, s);
        s = fmaf(a.w, v.w, s);
      });
    });
  }
  for (int o = 32; o > 0; o >>= 1)
    static_for<0, ROWS>([&](auto r) {
      static_for<0, kPoolCols>([&](auto c) { acc[decltype(r)::value][decltype(c)::value] += __shfl_xor(acc[decltype(r)::value][decltype(c)::value], o); });
    });
  static_for<0, ROWS>([&](auto r) {
    static_for<0, kPoolCols>([&](auto c) {
      constexpr int rr = decltype(r)::value, cc = decltype(c)::value;
      if (lane == rr * kPoolCols + cc && b0 + rr < B) out[(long)(b0 + rr) * d + c0 + cc] = tanhf(acc[rr][cc] + (bias ? bias[c0 + cc] : 0.f));
    });
  });
}

}  // namespace m2

using namespace m2;

extern "C" int m2_pooler_fwd(const float* h, long h_row, const float* w, const float* bias, float* out, int B, int d, void* stream) {
  const char* who = "m2_pooler_fwd";
  if (!h || !w || !out) return set_error(M2_ERR_ARG, "%s: null pointer", who);
  if (B <= 0 || d <= 0 || d % 8 || h_row < d || h_row % 4)
    return set_error(M2_ERR_UNSUPPORTED, "%s: need B > 0, d a multiple of 8 and rows a multiple of 4 apart, d at least (B=%d d=%d h_row=%ld)", who, B, d, h_row);
  if (!aligned16(h, w)) return set_error(M2_ERR_UNSUPPORTED, "%s: operands must be 16-byte aligned", who);
  hipStream_t st = (hipStream_t)stream;
  const unsigned cols = (unsigned)(d / (4 * kPoolCols));
  if (B == 1) hipLaunchKernelGGL(pooler_kernel<1>, dim3(cols, 1), dim3(256), 0, st, h, h_row, w, bias, out, B, d);
  else hipLaunchKernelGGL(pooler_kernel<8>, dim3(cols, (B + 7) / 8), dim3(256), 0, st, h, h_row, w, bias, out, B, d);
  return check_launch("pooler");
}
