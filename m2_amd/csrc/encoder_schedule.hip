// The fused schedule of a stack of encoder layers, enqueued by one call: per layer
//
//   xproj (3d, M) = W_in h16^T                     dense_kernels.hip
//   y     (d, M)  = mixer core(xproj, hT, spec)    fftconv*_kernels.hip
//   a     (M, d)  = y^T W_out^T + b                dense_kernels.hip
//   s     (M, d)  = wo(glu(a)) + b + a, bf16       mlp_fused / glu_stream / dense / blockdiag kernels
//   h16 | hT | out32 = LayerNorm(s)                layernorm_kernels.hip
//
// Host code only: what it saves is the host's time per launch.  Issued module by module from Python a layer takes about
// 170 us of host time whatever its size; here five or six launches of about 3 us each.
#include "m2_internal.h"

using namespace m2;

namespace {
struct Layout {
  long xrow;      // elements between two channels of xproj
  size_t xproj, y, a, g, s, h16, hT, total;
};
Layout layout(long M, long d, long I) {
  auto up = [](size_t v) { return (v + 255) & ~(size_t)255; };
  Layout l;
  l.xrow = m2_dense_channels_row((int)M, (int)(3 * d), (int)d);
  l.xproj = 0;
  l.y = up(l.xproj + (size_t)(3 * d * l.xrow) * 2);
  l.a = up(l.y + (size_t)(d * M) * 2);
  l.g = up(l.a + (size_t)(d * M) * 2);
  l.s = up(l.g + (size_t)(I * M) * 2);
  l.h16 = up(l.s + (size_t)(d * M) * 2);
  l.hT = up(l.h16 + (size_t)(d * M) * 2);
  l.total = up(l.hT + (size_t)(d * M) * 4);
  return l;
}
}  // namespace

extern "C" size_t m2_encoder_layers_workspace_bytes(int M, int d, int intermediate) {
  if (M <= 0 || d <= 0 || intermediate <= 0) return 0;
  return layout(M, d, intermediate).total;
}

// filters: spectra, or with fpm > 0 the taps of fpm filters per layer
static int encoder_layers(const char* who, const m2_layer_params* layers, int nlayers, const float* filters, int fpm, const float* const* skip,
                          const void* h16, const float* h_channel_major, float* const* out_f32, void* workspace, int B, int L, int d,
                          int intermediate, int nblocks, float eps, void* stream) {
  if (!layers || !filters || !h16 || !h_channel_major || !out_f32 || !workspace) return set_error(M2_ERR_ARG, "%s: null pointer", who);
  if (nlayers < 1 || B < 1 || L < 1 || d < 1 || intermediate < 1)
    return set_error(M2_ERR_ARG, "%s: sizes must be positive (layers=%d B=%d L=%d d=%d I=%d)", who, nlayers, B, L, d, intermediate);
  if ((long)B * L > 0x7fffffffL) return set_error(M2_ERR_UNSUPPORTED, "%s: B * L = %ld does not fit an int", who, (long)B * L);
  const int M = B * L;
  if (!aligned16(workspace)) return set_error(M2_ERR_UNSUPPORTED, "%s: the workspace must be 16-byte aligned", who);
  for (int i = 0; i < nlayers; ++i) {
    const m2_layer_params& p = layers[i];
    if (!p.in_w || !p.short_w || !p.short_b || !p.out_w || !p.w_gated || !p.w_out || !p.ln_gamma || !p.ln_beta)
      return set_error(M2_ERR_ARG, "%s: layer %d has a null weight", who, i);
  }
  const Layout l = layout(M, d, intermediate);
  unsigned char* ws = (unsigned char*)workspace;
  void *xproj = ws + l.xproj, *y = ws + l.y, *a = ws + l.a, *g = ws + l.g, *s = ws + l.s, *nh = ws + l.h16;
  float* nt = (float*)(ws + l.hT);
  // a layer's LayerNorm and the next one's in_linear as one kernel, where nobody else reads the normalised rows
  const bool joined = m2_layernorm_to_channels_supported(M, 3 * d, d);
  const m2_layer_params* norm = nullptr;      // of the layer whose sum is still to be normalised
  const size_t stride = fpm ? (size_t)fpm * d * 2 * L : m2_filter_spectrum_bytes(d, L) / sizeof(float);
  for (int i = 0; i < nlayers; ++i) {
    const m2_layer_params& p = layers[i];
    int rc = norm ? m2_layernorm_to_channels_fwd(s, norm->ln_gamma, norm->ln_beta, eps, p.in_w, xproj, l.xrow, nt, M, 3 * d, d, stream)
                  : m2_dense_to_channels_rows_fwd(h16, p.in_w, xproj, l.xrow, M, 3 * d, d, stream);
    if (rc) return rc;
    const float* u = p.residual ? h_channel_major : nullptr;
    rc = fpm ? m2_mixer_core_taps_fwd(xproj, l.xrow, p.in_b, u, p.short_w, p.short_b, filters + i * stride, skip ? skip + i * fpm : nullptr, fpm, y,
                                      B, L, d, stream)
             : m2_mixer_core_rows_fwd(xproj, l.xrow, p.in_b, u, p.short_w, p.short_b, filters + i * stride, y, B, L, d, M2_DTYPE_BF16, stream);
    if (rc) return rc;
    rc = m2_dense_from_channels_fwd(y, p.out_w, p.out_b, a, M, d, d, stream);
    if (rc) return rc;
    if (p.mlp_packed) {
      rc = m2_mlp_fused_fwd(a, p.mlp_packed, p.wo_b, a, s, M, d, intermediate, nblocks, M2_DTYPE_BF16, stream);
    } else {
      rc = p.glu_packed ? m2_glu_stream_fwd(a, p.glu_packed, g, M, d, intermediate, nblocks, stream)
                        : m2_blockdiag_glu_fwd(a, p.w_gated, g, M, d, intermediate, nblocks, stream);
      if (rc) return rc;
      rc = m2_blockdiag_linear_fwd(g, p.w_out, p.wo_b, a, s, M, intermediate, d, nblocks, M2_DTYPE_BF16, stream);
    }
    if (rc) return rc;
    const bool last = i == nlayers - 1;
    h_channel_major = nt;
    norm = joined && !last && !out_f32[i] && aligned16(p.ln_gamma, p.ln_beta) ? &p : nullptr;
    if (norm) continue;
    rc = m2_layernorm_bf16_fwd(s, p.ln_gamma, p.ln_beta, eps, out_f32[i], last ? nullptr : nh, last ? nullptr : nt, M, d, stream);
    if (rc) return rc;
    h16 = nh;
  }
  return M2_OK;
}

extern "C" int m2_encoder_layers_fwd(const m2_layer_params* layers, int nlayers, const float* spectra, const void* h16,
                                     const float* h_channel_major, float* const* out_f32, void* workspace, int B, int L,
                                     int d, int intermediate, int nblocks, float eps, void* stream) {
  return encoder_layers("m2_encoder_layers_fwd", layers, nlayers, spectra, 0, nullptr, h16, h_channel_major, out_f32, workspace, B, L, d,
                        intermediate, nblocks, eps, stream);
}

extern "C" int m2_encoder_layers_taps_fwd(const m2_layer_params* layers, int nlayers, const float* taps, const float* const* skip_dev,
                                          int filters_per_mixer, const void* h16, const float* h_channel_major, float* const* out_f32,
                                          void* workspace, int B, int L, int d, int intermediate, int nblocks, float eps, void* stream) {
  const char* who = "m2_encoder_layers_taps_fwd";
  if (filters_per_mixer < 1 || filters_per_mixer > 2)
    return set_error(M2_ERR_ARG, "%s: filters_per_mixer=%d must be 1 or 2", who, filters_per_mixer);
  return encoder_layers(who, layers, nlayers, taps, filters_per_mixer, skip_dev, h16, h_channel_major, out_f32, workspace, B, L, d, intermediate,
                        nblocks, eps, stream);
}
