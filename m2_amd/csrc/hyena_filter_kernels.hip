// Implicit long-filter generation for the Monarch-Mixer sequence mixer on gfx950.
//
//   h0 = z_l (emb)  ->  h1 = sin(f.(W0 h0 + b0))  ->  h2 = sin(f.(W1 h1 + b1))  ->  h3 = sin(f.(W2 h2 + b2))
//   k[c][l] = (W3 h3)[c] * (exp(-t_l |delta_c|) + shift)
//
// (bert/src/mm/hyena_utils.py:168-175 the MLP, :50-63 Sin, :110-112 modulation, :201-217 filter /
// filter_rev, :231-236 placement of the forward and the flipped reverse taps in a 2L window.)
//
// Three kernels.  `split_weights_kernel` re-splits the weights into parts in MFMA operand layout (hyena_filter.h; a few
// microseconds, once per call) where the next kernel has many workgroups to read them.  `hidden_kernel` evaluates the three sin layers for 32 or 64 positions per workgroup: the first
// (emb -> 128) on the vector ALU, the two 128 x 128 layers as six-product split-bf16 MFMA GEMMs (v_mfma_f32_32x32x16_bf16 on the
// three parts of weights and activations: fp32 products, which matters because sin(freq * x) amplifies any rounding of
// x) with the activations resident in LDS; it writes h3 in two fp16 parts.  `project_kernel` is the 128 -> d projection, three
// products of two fp16 parts, whose epilogue applies the decay and stores the taps channel-major, forward taps at [0, L) and reverse taps
// mirrored into [L, 2L).  For L >= 1024 the last two are one launch (`hidden_kernel<2, ., PROJECT = true>`: the
// workgroup that evaluated the hidden layers of 64 positions goes on to project them, h3 never leaves LDS); for
// L <= 512 the batched entry point hands h3 to the projection + spectrum kernel of filter_fused_kernels.hip instead.
#include <hip/hip_runtime.h>

#include <mutex>

#include "hyena_filter.h"

namespace m2 {

constexpr int kPosTile = 32;      // positions per workgroup in hidden_kernel

// sin(x) by two-constant Cody-Waite reduction to [-pi/2, pi/2] (fused multiply-adds keep the reduction
// exact to ~1e-15 n) and the odd Taylor polynomial to x^11 (truncation 5.6e-8 at pi/2).  Absolute error
// ~1e-7 for |x| up to ~1e4, i.e. fp32 sinf quality over the whole range freq * x can take here, at a
// third of the instructions of the libm routine (which carries a slow path for huge arguments).
__device__ __forceinline__ float sin_reduced(float x) {
  const float n = rintf(x * 0.318309886183790672f);
  float r = fmaf(-n, 3.14159274101257324f, x);
  r = fmaf(-n, -8.74227765734758577e-8f, r);
  const float r2 = r * r;
  float p = -2.50521083854417188e-8f;          // -1/11!
  p = fmaf(p, r2, 2.75573192239858907e-6f);    //  1/9!
  p = fmaf(p, r2, -1.98412698412698413e-4f);   // -1/7!
  p = fmaf(p, r2, 8.33333333333333322e-3f);    //  1/5!
  p = fmaf(p, r2, -1.66666666666666657e-1f);   // -1/3!
  const float s = fmaf(p * r2, r, r);
  return __uint_as_float(__float_as_uint(s) ^ ((uint32_t)static_cast<int>(n) << 31));      // odd n: the other sign
}

// The last hidden layer's, whose fp16 parts end at 8: beyond |x| = 3e7 the reduction leaves arguments of any size, and what the polynomial
// makes of them is no sine, but it has to stay a number.  NaN stays NaN.
__device__ __forceinline__ float sin_bounded(float x) {
  const float s = sin_reduced(x);
  return fabsf(s) > 2.f ? copysignf(1.f, s) : s;
}

// The 128 x 128 weights of the two inner layers, split into three bf16 parts and laid out as MFMA A operands, so
// that hidden_kernel fetches them with coalesced 16-byte loads and no arithmetic:
// wsplit[mlp][layer][part][wave w][K step ks][lane (i, h)] = 8 bf16 of row 32 w + i, K = 16 ks + 8 h .. + 7.
// The d x 128 output projection likewise in two fp16 parts, for the hidden kernel that goes on to project, and with it
// w3scale[mlp][row], the reciprocal 2^-(e + 13) of the row's scale and the activations':
// w3split[mlp][part][32-channel tile][K step ks][lane (i, h)] = 8 fp16 of row 32 tile + i, K = 16 ks + 8 h .. + 7.
// A workgroup of 512 threads takes the 32 rows of one (mlp, layer, wave) or one (mlp, tile).
constexpr int kSplitPerLayer = 3 * kOrder * kOrder;      // bf16 elements per (mlp, layer)
template <class TAB>
__global__ __launch_bounds__(512) void split_weights_kernel(TAB tab, int nmlp, int d, uint16_t* __restrict__ wsplit,
                                                            uint16_t* __restrict__ w3split, float* __restrict__ w3scale) {
  const int inner = nmlp * 2 * 4;
  const int lane = threadIdx.x & 63, i32 = lane & 31, ks = threadIdx.x >> 6;
  if ((int)blockIdx.x < inner) {
    const int w = blockIdx.x & 3, layer = (blockIdx.x >> 2) & 1, m = blockIdx.x >> 3;
    const MlpPtrs W = tab.at(m >> 1).mlp[m & 1];
    if (W.w0 == nullptr) return;
    gfloat* src = in_global(layer == 0 ? W.w1 : W.w2) + (long)(32 * w + i32) * kOrder + 16 * ks + 8 * (lane >> 5);
    u32x4 vh, vm, vl;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float h[2], md[2], l[2];
      split3(src[2 * j], h[0], md[0], l[0]);
      split3(src[2 * j + 1], h[1], md[1], l[1]);
      vh[j] = pack_bf16x2(h[0], h[1]);
      vm[j] = pack_bf16x2(md[0], md[1]);
      vl[j] = pack_bf16x2(l[0], l[1]);
    }
    u32x4* dst = reinterpret_cast<u32x4*>(wsplit + ((long)(m * 2 + layer)) * kSplitPerLayer) + (w * 8 + ks) * 64 + lane;
    dst[0] = vh;
    dst[kOrder * kOrder / 8] = vm;
    dst[2 * kOrder * kOrder / 8] = vl;
    return;
  }
  __shared__ float most[8][32];
  const int ct = ((int)blockIdx.x - inner) % (d / 32), m = ((int)blockIdx.x - inner) / (d / 32);
  const MlpPtrs W = tab.at(m >> 1).mlp[m & 1];
  if (W.w3 == nullptr) return;
  gfloat* src = in_global(W.w3) + (long)(32 * ct + i32) * kOrder + 16 * ks + 8 * (lane >> 5);
  float v[8], top = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    v[j] = src[j];
    top = fmaxf(top, fabsf(v[j]));
  }
  top = fmaxf(top, __shfl_xor(top, 32));
  if (lane < 32) most[ks][lane] = top;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 8; ++j) top = fmaxf(top, most[j][i32]);
  const float scale = row_scale(top);
  u32x4 hi, lo;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    uint32_t h, l;
    split2(v[2 * j] * scale, v[2 * j + 1] * scale, h, l);
    hi[j] = h;
    lo[j] = l;
  }
  u32x4* dst = reinterpret_cast<u32x4*>(w3split + (long)m * 2 * d * kOrder) + (ct * 8 + ks) * 64 + lane;
  dst[0] = hi;
  dst[d * kOrder / 8] = lo;
  if (threadIdx.x < 32) w3scale[(long)m * d + 32 * ct + threadIdx.x] = 1.f / (scale * kActScale);
}

constexpr int kActRowB = 2 * kOrder + 16;     // bytes per padded 16-bit row of an activation part (conflict-free 16-byte reads)

// grid (L / (32 TILES), 2 * nfilters), block 256 = 4 waves.  Wave w owns the output neurons [32 w, 32 w + 32) of all
// TILES tiles of 32 positions of the workgroup.  The activations live in LDS as three bf16 parts (hi, mid, lo:
// together the fp32 value) and every layer overwrites them in place; the two 128 x 128 layers are six-product
// split-bf16 MFMA GEMMs, their weights pre-split by split_weights_kernel and held in registers for all tiles (fetching them is what a short run
// of positions per workgroup pays most for: 96 KB per workgroup and layer from L2).  Within a layer the products of
// tile i + 1 are issued together with the sin epilogue of tile i, so that matrix pipe and vector ALU overlap.
//
// PROJECT = true: the same workgroup goes on to the 128 -> d output projection of its positions (the last hidden
// layer's activations stay in LDS as fp16 hi / lo parts instead of travelling through memory): wave w takes the
// 32-channel tiles w, w + 4, ..., fetches the tile's pre-split weight rows (hi / lo parts in operand layout, from L2:
// every workgroup reads all of them once), multiplies (three products: W_hi h_hi + W_hi h_lo + W_lo h_hi), applies
// exp(-t |delta|) + shift and stores the taps channel-major with streaming stores, forward taps at [0, L), reverse taps
// mirrored into [L, 2L) (bert/src/mm/hyena_utils.py:175,213-217,233-234).
template <int TILES, class TAB, bool PROJECT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void hidden_kernel(TAB tab, int L, int emb, float w_mod,
                                                     const uint16_t* __restrict__ wsplit,
                                                     uint16_t* __restrict__ h_hi /* (2 nf, L, 128) fp16 */,
                                                     uint16_t* __restrict__ h_lo /* (2 nf, L, 128) fp16 */,
                                                     int d, float shift, const uint16_t* __restrict__ w3split, const float* __restrict__ w3scale,
                                                     float* __restrict__ taps /* (nf, d, 2L) */) {
  constexpr int P = 32 * TILES;
  __shared__ __attribute__((aligned(16))) unsigned char act[3][P * kActRowB];
  __shared__ float zt[P * kMaxEmb];
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, i32 = lane & 31, half = lane >> 5;
  const int fi = blockIdx.y >> 1, dir = blockIdx.y & 1;
  const FilterPtrs& F = tab.at(fi);
  const MlpPtrs W = F.mlp[dir];
  gfloat *const z = in_global(F.z), *const tt = in_global(F.t), *const freq = in_global(F.freq), *const deltas = in_global(F.deltas);
  gfloat *const w0 = in_global(W.w0), *const b0 = in_global(W.b0), *const b1 = in_global(W.b1), *const b2 = in_global(W.b2);
  const int l0 = blockIdx.x * P;
  if (W.w0 == nullptr) {                        // not bidirectional: nothing to compute for dir == 1 ...
    if constexpr (PROJECT) {                    // ... and the reverse half of the window is zero
      float* out = taps + (long)fi * d * 2 * L + (2L * L - l0 - P);
      for (int i = tid; i < d * P; i += 256) out[(long)(i / P) * 2 * L + i % P] = 0.f;
    }
    return;
  }

  auto put3 = [&](int pos, int o, const float (&s)[4]) __attribute__((always_inline)) {
    float h[4], m[4], l[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) split3(s[j], h[j], m[j], l[j]);
    const int off = pos * kActRowB + 2 * o;
    *reinterpret_cast<uint2*>(&act[0][off]) = make_uint2(pack_bf16x2(h[0], h[1]), pack_bf16x2(h[2], h[3]));
    *reinterpret_cast<uint2*>(&act[1][off]) = make_uint2(pack_bf16x2(m[0], m[1]), pack_bf16x2(m[2], m[3]));
    *reinterpret_cast<uint2*>(&act[2][off]) = make_uint2(pack_bf16x2(l[0], l[1]), pack_bf16x2(l[2], l[3]));
  };
  auto put2 = [&](int pos, int o, const float (&s)[4]) __attribute__((always_inline)) {
    uint32_t h0, h1, l0, l1;
    split2(s[0] * kActScale, s[1] * kActScale, h0, l0);
    split2(s[2] * kActScale, s[3] * kActScale, h1, l1);
    const int off = pos * kActRowB + 2 * o;
    *reinterpret_cast<uint2*>(&act[0][off]) = make_uint2(h0, h1);
    *reinterpret_cast<uint2*>(&act[1][off]) = make_uint2(l0, l1);
  };

  // Weights of an inner layer -> registers.  Requested one phase early (layer 1's before the vector-ALU layer, layer
  // 2's before the last epilogue of layer 1), so that the 24 KB per wave arrive behind other work.
  // PROJECT: from the split copy.  Otherwise a workgroup splits its own rows, 64 values a lane and layer (about 2 us of vector
  // instructions in all, where a launch ahead of this one took 3 to 7): it has one tile, and few of them share a compute unit.
  bf16x8 ah[8], am[8], al[8];
  floatx4 raw[PROJECT ? 1 : 16];
  gfloat *const w1 = in_global(W.w1), *const w2 = in_global(W.w2);
  auto load_weights = [&](int layer) __attribute__((always_inline)) {
    if constexpr (PROJECT) {
      const u32x4* wp = reinterpret_cast<const u32x4*>(wsplit + ((long)(blockIdx.y * 2 + layer)) * kSplitPerLayer) + w * 8 * 64;
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) {
        ah[ks] = __builtin_bit_cast(bf16x8, (wp + ks * 64)[(unsigned)lane]);
        am[ks] = __builtin_bit_cast(bf16x8, (wp + ks * 64 + kOrder * kOrder / 8)[(unsigned)lane]);
        al[ks] = __builtin_bit_cast(bf16x8, (wp + ks * 64 + 2 * kOrder * kOrder / 8)[(unsigned)lane]);
      }
    } else {
      gfloat* row = (layer == 0 ? w1 : w2) + (32 * w + i32) * kOrder + 8 * half;
#pragma unroll
      for (int i = 0; i < 16; ++i) raw[i] = *(gfloatx4_any*)(row + 16 * (i >> 1) + 4 * (i & 1));
    }
  };
  auto split_weights = [&]() __attribute__((always_inline)) {
    if constexpr (!PROJECT) {
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) {
        u32x4 vh, vm, vl;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float h[2], md[2], l[2];
#pragma unroll
          for (int e = 0; e < 2; ++e) split3(raw[2 * ks + j / 2][2 * (j & 1) + e], h[e], md[e], l[e]);
          vh[j] = pack_bf16x2(h[0], h[1]);
          vm[j] = pack_bf16x2(md[0], md[1]);
          vl[j] = pack_bf16x2(l[0], l[1]);
        }
        ah[ks] = __builtin_bit_cast(bf16x8, vh);
        am[ks] = __builtin_bit_cast(bf16x8, vm);
        al[ks] = __builtin_bit_cast(bf16x8, vl);
      }
    }
  };
  load_weights(0);

  // layer 0 (emb -> 128) on the vector ALU: thread = (4 neurons, P / 8 positions).  The embeddings of the tile
  // (P x emb consecutive floats) go through LDS; weights beyond emb are zero so the dot product has a fixed length.
  {
    for (int i = tid; i < P * kMaxEmb; i += 256) zt[i] = i < P * emb ? z[(long)l0 * emb + i] : 0.f;
    const int o = 4 * (tid & 31), p0 = tid >> 5;          // positions p0, p0 + 8, ...
    float wt[4][kMaxEmb], bb[4], fo[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int e = 0; e < kMaxEmb; ++e) wt[j][e] = e < emb ? w0[(o + j) * emb + e] : 0.f;
      bb[j] = b0[o + j];
      fo[j] = w_mod * freq[o + j];
    }
    __syncthreads();
#pragma unroll 4
    for (int pp = 0; pp < P / 8; ++pp) {
      const int pos = p0 + 8 * pp;
      float s[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float acc = bb[j];
#pragma unroll
        for (int e = 0; e < kMaxEmb; ++e) acc += wt[j][e] * zt[pos * emb + e];      // pos emb + e < P emb + 8 <= P kMaxEmb
        s[j] = sin_reduced(fo[j] * acc);
      }
      put3(pos, o, s);
    }
  }
  // layers 1, 2: D[o'][pos] = sum_o W[o'][o] act[pos][o].  A = weight rows 32 w + i32 (registers), B = positions of the
  // tile (LDS); lane (i32, half) holds K = 16 ks + 8 half .. + 7 of both.
  auto products = [&](int tile, floatx16& acc) __attribute__((always_inline)) {
    floatx16 small;      // the products below the leading one, added at the end: the sum is rounded at its full size once a K step
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = small[v] = 0.f;
    const int boff = (32 * tile + i32) * kActRowB + 16 * half;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      const bf16x8 bh = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(&act[0][boff + 32 * ks]));
      const bf16x8 bm = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(&act[1][boff + 32 * ks]));
      const bf16x8 bl = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(&act[2][boff + 32 * ks]));
      // smallest terms first
      small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[ks], bh, small, 0, 0, 0);
      small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[ks], bl, small, 0, 0, 0);
      small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(am[ks], bm, small, 0, 0, 0);
      small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(am[ks], bh, small, 0, 0, 0);
      small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[ks], bm, small, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[ks], bh, acc, 0, 0, 0);
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] += small[v];
  };
  // accumulator element v: neuron 32 w + 8 (v / 4) + 4 half + v % 4, position i32 of the tile
  float fr[16], bs[16];
  auto load_scales = [&](int layer) __attribute__((always_inline)) {
    gfloat* bias = layer == 0 ? b1 : b2;
#pragma unroll
    for (int vq = 0; vq < 4; ++vq) {
      const int o = 32 * w + 8 * vq + 4 * half;
      const floatx4 fq = *(gfloatx4*)(freq + o);
      const floatx4 bq = *(gfloatx4*)(bias + o);
      fr[4 * vq] = w_mod * fq.x; fr[4 * vq + 1] = w_mod * fq.y; fr[4 * vq + 2] = w_mod * fq.z; fr[4 * vq + 3] = w_mod * fq.w;
      bs[4 * vq] = bq.x; bs[4 * vq + 1] = bq.y; bs[4 * vq + 2] = bq.z; bs[4 * vq + 3] = bq.w;
    }
  };
  auto epilogue = [&](auto ll, int tile, const floatx16& acc) __attribute__((always_inline)) {
    constexpr int layer = decltype(ll)::value;
    const int pos = 32 * tile + i32;
#pragma unroll
    for (int vq = 0; vq < 4; ++vq) {
      const int o = 32 * w + 8 * vq + 4 * half;
      float s[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float arg = fr[4 * vq + j] * (acc[4 * vq + j] + bs[4 * vq + j]);
        s[j] = layer == 0 ? sin_reduced(arg) : sin_bounded(arg);
      }
      if constexpr (layer == 0) {
        put3(pos, o, s);
      } else if constexpr (PROJECT) {           // h3 stays in LDS (parts 0 and 1) for the projection
        put2(pos, o, s);
      } else {
        const long hrow = ((long)blockIdx.y * L + l0 + pos) * kOrder;
        uint32_t h0, h1, lo0, lo1;
        split2(s[0] * kActScale, s[1] * kActScale, h0, lo0);
        split2(s[2] * kActScale, s[3] * kActScale, h1, lo1);
        *reinterpret_cast<uint2*>(h_hi + hrow + o) = make_uint2(h0, h1);
        *reinterpret_cast<uint2*>(h_lo + hrow + o) = make_uint2(lo0, lo1);
      }
    }
  };
  // One layer: products(0); then for every tile "barrier; products(next tile) with epilogue(this tile)".  The barrier
  // before an epilogue says that all four waves have read that tile's operands, so it may be overwritten in place;
  // the barrier that ends the layer says that all of the layer's activations are written.
  auto layer_pass = [&](auto ll) __attribute__((always_inline)) {
    constexpr int layer = decltype(ll)::value;
    floatx16 acc[2];
    products(0, acc[0]);
    static_for<0, TILES>([&](auto tt) {
      constexpr int t = decltype(tt)::value;
      __syncthreads();
      if constexpr (t + 1 < TILES) products(t + 1, acc[(t + 1) & 1]);
      else if constexpr (layer == 0) load_weights(1);      // the products of layer 1 are done: its registers are free
      epilogue(ll, t, acc[t & 1]);
    });
    __syncthreads();
  };
  load_scales(0);
  split_weights();
  __syncthreads();                     // layer 0's activations are complete
  layer_pass(ic<0>{});
  load_scales(1);
  split_weights();
  layer_pass(ic<1>{});

  if constexpr (PROJECT) {
    // the barrier that ended the last layer says h3 (hi in act[0], lo in act[1]) is complete for all P positions
    float* out = taps + (long)fi * d * 2 * L;
    const u32x4* w3 = reinterpret_cast<const u32x4*>(w3split + (long)blockIdx.y * 2 * d * kOrder);
    const float* back = w3scale + (long)blockIdx.y * d;
    float tl[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t) tl[t] = tt[l0 + 32 * t + i32];
    // A operand of a channel tile: weight rows 32 ct + i32, K = 16 ks + 8 half + {0..7}, hi / lo parts as
    // split_weights_kernel left them, and the decay rates and scales of the lane's 16 channels
    struct TileOps {
      f16x8 ahi[kOrder / 16], alo[kOrder / 16];
      floatx4 dq[4], rq[4];
    };
    auto fetch_tile = [&](int ct, TileOps& o) __attribute__((always_inline)) {
#pragma unroll
      for (int ks = 0; ks < kOrder / 16; ++ks) {
        o.ahi[ks] = __builtin_bit_cast(f16x8, (w3 + (ct * 8 + ks) * 64)[(unsigned)lane]);
        o.alo[ks] = __builtin_bit_cast(f16x8, (w3 + (ct * 8 + ks) * 64 + d * kOrder / 8)[(unsigned)lane]);
      }
#pragma unroll
      for (int vq = 0; vq < 4; ++vq) {
        o.dq[vq] = ((gfloatx4*)(deltas + 32 * ct + 8 * vq))[(unsigned)half];
        o.rq[vq] = reinterpret_cast<const floatx4*>(back + 32 * ct + 8 * vq)[(unsigned)half];
      }
    };
    auto project_tile = [&](int ct, const TileOps& o) __attribute__((always_inline)) {
      float adelta[16], rs[16];
#pragma unroll
      for (int vq = 0; vq < 4; ++vq) {
        rs[4 * vq] = o.rq[vq].x; rs[4 * vq + 1] = o.rq[vq].y; rs[4 * vq + 2] = o.rq[vq].z; rs[4 * vq + 3] = o.rq[vq].w;
        adelta[4 * vq] = -fabsf(o.dq[vq].x) * 1.44269504088896341f; adelta[4 * vq + 1] = -fabsf(o.dq[vq].y) * 1.44269504088896341f;
        adelta[4 * vq + 2] = -fabsf(o.dq[vq].z) * 1.44269504088896341f; adelta[4 * vq + 3] = -fabsf(o.dq[vq].w) * 1.44269504088896341f;
      }
#pragma unroll
      for (int t = 0; t < TILES; ++t) {
        const unsigned char* bh = &act[0][(32 * t + i32) * kActRowB + 16 * half];
        const unsigned char* bl = &act[1][(32 * t + i32) * kActRowB + 16 * half];
        floatx16 acc;
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[v] = 0.f;
#pragma unroll
        for (int ks = 0; ks < kOrder / 16; ++ks) {
          const f16x8 bhi = __builtin_bit_cast(f16x8, *reinterpret_cast<const u32x4*>(bh + 32 * ks));
          const f16x8 blo = __builtin_bit_cast(f16x8, *reinterpret_cast<const u32x4*>(bl + 32 * ks));
          acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(o.alo[ks], bhi, acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(o.ahi[ks], blo, acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(o.ahi[ks], bhi, acc, 0, 0, 0);
        }
        // accumulator element v of lane: channel 32 ct + 8 (v / 4) + 4 half + v % 4, position l0 + 32 t + i32
        const int l = l0 + 32 * t + i32;
        // A row is the same for all lanes: its address walks along in scalar registers (kept by the asm, which the compiler would turn into
        // sixteen vector addresses), the lane's place in it is a 32-bit offset.
        typedef __attribute__((address_space(1))) char gbyte;
        gbyte* po = (gbyte*)out + (long)(32 * ct) * 8 * L;
        unsigned at = 4u * (4u * half * 2 * L + (dir == 0 ? l : 2 * L - 1 - l));
        asm volatile("" : "+v"(at));
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          asm volatile("" : "+s"(po));
          // (exp(-t |delta|) + shift) r, r the reciprocal scale of the channel; the bare hardware exp2 flushes results below 2^-126 to zero, which is the value to
          // 1e-38 absolute.  Streaming store: the taps are read once, by a later kernel
          const float decay = fmaf(__builtin_amdgcn_exp2f(tl[t] * adelta[v]), rs[v], shift * rs[v]);
          __builtin_nontemporal_store(acc[v] * decay, (__attribute__((address_space(1))) float*)(po + at));
          po += (v & 3) == 3 ? 40l * L : 8l * L;      // channels 8 (v / 4) + v % 4 of the tile
        }
      }
    };
    // two register sets: the next tile's operands are requested before the products of this one
    TileOps o[2];
    const int last = d / 32 - 1;
    auto fetch = [&](int ct, TileOps& into) __attribute__((always_inline)) { fetch_tile(ct < last ? ct : last, into); };      // (never beyond the weights)
    fetch(w, o[0]);
    for (int ct = w; ct <= last; ct += 8) {
      fetch(ct + 4, o[1]);
      __builtin_amdgcn_sched_barrier(0);
      project_tile(ct, o[0]);
      if (ct + 4 > last) break;
      fetch(ct + 8, o[0]);
      __builtin_amdgcn_sched_barrier(0);
      project_tile(ct + 4, o[1]);
    }
  }
}

// Workgroup = 4 waves = 128 channels; wave w owns channels [c0 + 32 w, + 32) and splits its weight rows itself into fp16 hi / lo
// parts, which stay in registers.  The channels' decay rates and scales do not (with both in registers 34 of them went to scratch and
// back for every tile): they are read from LDS where they are used.  The workgroup walks kPosPerWg positions in tiles of 32:
// the h3 tile (hi and lo parts, 16 KB) is fetched with coalesced 16-byte loads one tile ahead, staged in
// LDS (double buffered, rows padded to 272 bytes so that the 16-byte operand reads of 32 rows spread over
// all banks) and shared by the four waves.
// grid (L / kPosPerWg rounded up, d / 128 rounded up, 2 * nfilters).
constexpr int kPosPerWg = 512;      // at most; 32-position tiles past L are skipped
constexpr int kHRow = 2 * kOrder + 16;   // bytes per padded LDS row of one h3 part
template <class TAB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 4))) void project_kernel(TAB tab, int L, int d, float shift,
                                                      const uint16_t* __restrict__ h_hi, const uint16_t* __restrict__ h_lo,
                                                      float* __restrict__ taps /* (nf, d, 2L) */) {
  __shared__ __attribute__((aligned(16))) unsigned char hbuf[2][2][32 * kHRow];     // [buffer][hi, lo][row]
  __shared__ float4 rate[4][8], back[4][8];        // of a wave's 32 channels: -|delta| log2(e), reciprocal scale
  const int fi = blockIdx.z >> 1, dir = blockIdx.z & 1;
  const FilterPtrs& F = tab.at(fi);
  gfloat *const w3 = in_global(F.mlp[dir].w3), *const tt = in_global(F.t), *const deltas = in_global(F.deltas);
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, i32 = lane & 31, half = lane >> 5;
  const int c0 = blockIdx.y * 128 + wave * 32;
  const bool active = c0 < d;                      // d is a multiple of 64: a wave is all in or all out
  const int lbase = blockIdx.x * kPosPerWg;
  float* out = taps + (long)fi * d * 2 * L;
  if (w3 == nullptr) {
    // not bidirectional: the reverse half of the window is zero
    if (active)
      for (int r = 0; r < 32; ++r)
        for (int p = lane; p < kPosPerWg && lbase + p < L; p += 64) out[(long)(c0 + r) * 2 * L + L + lbase + p] = 0.f;
    return;
  }
  int ntiles = (L - lbase) / 32;
  if (ntiles > kPosPerWg / 32) ntiles = kPosPerWg / 32;

  // staging: thread -> two 16-byte pieces of each part of the (contiguous, 8 KB) tile
  const long tile_elems = 32L * kOrder;
  const uint16_t* gh = h_hi + ((long)blockIdx.z * L + lbase) * kOrder + 8 * tid;
  const uint16_t* gl = h_lo + ((long)blockIdx.z * L + lbase) * kOrder + 8 * tid;
  const int srow0 = tid >> 4, scol = (tid & 15) * 16;              // piece q covers row srow0 + 16 q
  // two register sets: the tile after next is in flight while the next one waits to be staged (a tile's product
  // takes well under a memory latency, so one tile of look-ahead left every iteration waiting for its fetch)
  u32x4 st[2][4];
  auto fetch = [&](int pt, auto ss) __attribute__((always_inline)) {
    constexpr int s = decltype(ss)::value;
    st[s][0] = *reinterpret_cast<const u32x4*>(gh + pt * tile_elems);
    st[s][1] = *reinterpret_cast<const u32x4*>(gh + pt * tile_elems + 16 * kOrder);
    st[s][2] = *reinterpret_cast<const u32x4*>(gl + pt * tile_elems);
    st[s][3] = *reinterpret_cast<const u32x4*>(gl + pt * tile_elems + 16 * kOrder);
  };
  auto stage = [&](int buf, auto ss) __attribute__((always_inline)) {
    constexpr int s = decltype(ss)::value;
    *reinterpret_cast<u32x4*>(&hbuf[buf][0][srow0 * kHRow + scol]) = st[s][0];
    *reinterpret_cast<u32x4*>(&hbuf[buf][0][(srow0 + 16) * kHRow + scol]) = st[s][1];
    *reinterpret_cast<u32x4*>(&hbuf[buf][1][srow0 * kHRow + scol]) = st[s][2];
    *reinterpret_cast<u32x4*>(&hbuf[buf][1][(srow0 + 16) * kHRow + scol]) = st[s][3];
  };
  fetch(0, ic<0>{});
  if (ntiles > 1) fetch(1, ic<1>{});

  // A operand: rows c0 + i32, K = 16 ks + 8 half + {0..7}.  All of a row is requested before the first value is looked at: in four
  // parts, read a second time for the splitting, it took 1.4 us more (taps of one filter, d = 768: L = 128 21.7 us, 512 36.2, 8224 54)
  f16x8 ahi[kOrder / 16], alo[kOrder / 16];
  if (active) {
    gfloat* row = w3 + (long)(c0 + i32) * kOrder + 8 * half;
    float top = 0.f;
#pragma unroll
    for (int ks = 0; ks < kOrder / 16; ++ks)
#pragma unroll
      for (int j = 0; j < 8; ++j) top = fmaxf(top, fabsf(row[16 * ks + j]));
    top = fmaxf(top, __shfl_xor(top, 32));
    const float scale = row_scale(top);
#pragma unroll
    for (int ks = 0; ks < kOrder / 16; ++ks) {
      u32x4 vh, vl;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t h, l;
        split2(row[16 * ks + 2 * j] * scale, row[16 * ks + 2 * j + 1] * scale, h, l);
        vh[j] = h;
        vl[j] = l;
      }
      ahi[ks] = __builtin_bit_cast(f16x8, vh);
      alo[ks] = __builtin_bit_cast(f16x8, vl);
    }
    if (half == 0) {
      reinterpret_cast<float*>(rate[wave])[i32] = -fabsf(deltas[c0 + i32]) * 1.44269504088896341f;
      reinterpret_cast<float*>(back[wave])[i32] = 1.f / (scale * kActScale);
    }
  }
  stage(0, ic<0>{});
  __syncthreads();

  // iteration pt: tile pt is in hbuf[pt & 1], tile pt + 1 in register set (pt + 1) & 1; tile pt + 2 is requested into
  // the set tile pt was staged from
  auto iteration = [&](int pt, auto par) __attribute__((always_inline)) {
    constexpr int P = decltype(par)::value;      // pt & 1
    if (pt + 2 < ntiles) fetch(pt + 2, ic<P>{});
    if (active) {
      const unsigned char* bh = &hbuf[P][0][i32 * kHRow + 16 * half];
      const unsigned char* bl = &hbuf[P][1][i32 * kHRow + 16 * half];
      floatx16 acc;
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[v] = 0.f;
#pragma unroll
      for (int ks = 0; ks < kOrder / 16; ++ks) {
        const f16x8 bhi = __builtin_bit_cast(f16x8, *reinterpret_cast<const u32x4*>(bh + 32 * ks));
        const f16x8 blo = __builtin_bit_cast(f16x8, *reinterpret_cast<const u32x4*>(bl + 32 * ks));
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(alo[ks], bhi, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ahi[ks], blo, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ahi[ks], bhi, acc, 0, 0, 0);
      }
      // accumulator element v of lane: channel c0 + 8 (v / 4) + 4 half + v % 4, position i32
      const int l = lbase + pt * 32 + i32;
      const float tl = tt[l];
      float* po = out + (long)(c0 + 4 * half) * 2 * L + (dir == 0 ? l : (2L * L - 1 - l));
#pragma unroll
      for (int vq = 0; vq < 4; ++vq) {
        const float4 dq = rate[wave][2 * vq + half], rq = back[wave][2 * vq + half];
        const float adelta[4] = {dq.x, dq.y, dq.z, dq.w}, rs[4] = {rq.x, rq.y, rq.z, rq.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          // (exp(-t |delta|) + shift) r, r the reciprocal scale of the channel; the bare hardware exp2 flushes results below 2^-126
          // to zero, which is the value to 1e-38 absolute
          const float decay = fmaf(__builtin_amdgcn_exp2f(tl * adelta[j]), rs[j], shift * rs[j]);
          // streaming store: the taps (100 MB per mixer at L = 8192) are read once, by a later kernel (-5 % for the call)
          __builtin_nontemporal_store(acc[4 * vq + j] * decay, po + (long)(8 * vq + j) * 2 * L);
        }
      }
    }
    if (pt + 1 < ntiles) stage(P ^ 1, ic<P ^ 1>{});
    __syncthreads();
  };
  for (int pt = 0; pt < ntiles; pt += 2) {
    iteration(pt, ic<0>{});
    if (pt + 1 < ntiles) iteration(pt + 1, ic<1>{});
  }
}

}  // namespace m2

using namespace m2;

extern "C" size_t m2_hyena_filter_workspace_bytes(int nfilters, int L, int d, int order) {
  if (nfilters <= 0 || L <= 0 || d <= 0 || order <= 0) return 0;
  // h3 in two fp16 parts; the inner-layer weights of the 2 nfilters MLPs as three bf16 parts each; their output
  // projections as two fp16 parts
  return (size_t)2 * nfilters * L * order * sizeof(float) + (size_t)2 * nfilters * 2 * 3 * order * order * sizeof(uint16_t) +
         (size_t)2 * nfilters * 2 * d * order * sizeof(uint16_t);
}

// Hidden layers and projection as one kernel, whose h3 never leaves the chip.  (No more channels than the room of h3, which is free
// then, has for their scales where a caller's workspace of the documented size is all there is.)
static bool project_with_hidden(int L, int d) { return L >= 1024 && L % 64 == 0 && d <= kOrder * L; }

// The launches of a batch of filters (weight re-split and hidden layers with projection + decay, or hidden layers and projection), the table
// coming either by value or from device memory.  `taps` null: the projection is left to the caller (the fused
// projection + spectrum kernel of short sequences).  Only the first form reads split copies (`wsplit`, `w3split`, `w3scale`); other kernels split
// the weights they keep in registers themselves.
template <class TAB>
static int filter_launches(TAB tab, int nfilters, int L, int d, int emb_dim, float w_mod, float shift, uint16_t* h_hi,
                           uint16_t* h_lo, uint16_t* wsplit, uint16_t* w3split, float* w3scale, float* taps, hipStream_t s) {
  const bool one_kernel = taps && project_with_hidden(L, d);
  if (one_kernel) {
    hipLaunchKernelGGL(split_weights_kernel<TAB>, dim3(2 * nfilters * 2 * 4 + 2 * nfilters * (d / 32)), dim3(512), 0, s, tab, 2 * nfilters, d,
                       wsplit, w3split, w3scale);
    const int rc = check_launch("hyena split_weights_kernel");
    if (rc) return rc;
  }
  // Positions per workgroup: longer runs amortise the weight fetch (96 KB per workgroup and layer, 520 bytes per channel for the
  // projection), short sequences need the workgroups spread over the chip.  128 positions would leave one workgroup on a compute unit
  // (104 KB of activations) and half of them idle for a single mixer.  us for the spectra of 1 / 12 mixers, d = 768: L = 1024 44 / 159,
  // 4096 60 / 508, 8192 93 / 979; with inner layers in two fp16 parts and 128 positions 56 / 151, 71 / 457, 93 / 869.
  if (one_kernel) {
    hipLaunchKernelGGL((hidden_kernel<2, TAB, true>), dim3(L / 64, 2 * nfilters), dim3(256), 0, s, tab, L, emb_dim, w_mod, wsplit,
                       h_hi, h_lo, d, shift, w3split, w3scale, taps);
    return check_launch("hyena hidden + project kernel");
  }
  hipLaunchKernelGGL((hidden_kernel<1, TAB, false>), dim3(L / 32, 2 * nfilters), dim3(256), 0, s, tab, L, emb_dim, w_mod, nullptr,
                     h_hi, h_lo, 0, 0.f, nullptr, nullptr, nullptr);
  const int rc = check_launch("hyena hidden_kernel");
  if (rc || !taps) return rc;
  hipLaunchKernelGGL(project_kernel<TAB>, dim3((L + kPosPerWg - 1) / kPosPerWg, (d + 127) / 128, 2 * nfilters), dim3(256), 0, s, tab, L, d, shift,
                     h_hi, h_lo, taps);
  return check_launch("hyena project_kernel");
}

static int check_filter_sizes(const char* who, int L, int d, int order, int emb_dim) {
  if (order != kOrder) return set_error(M2_ERR_UNSUPPORTED, "%s: order=%d, only 128 is built", who, order);
  if (emb_dim < 3 || emb_dim > kMaxEmb)
    return set_error(M2_ERR_UNSUPPORTED, "%s: emb_dim=%d not in [3, %d]", who, emb_dim, kMaxEmb);
  if (L <= 0 || L % kPosTile != 0)
    return set_error(M2_ERR_UNSUPPORTED, "%s: L=%d must be a positive multiple of %d", who, L, kPosTile);
  if (d <= 0 || d % 64 != 0) return set_error(M2_ERR_UNSUPPORTED, "%s: d=%d must be a positive multiple of 64", who, d);
  return M2_OK;
}

// Shared by the two entry points that take a host array of filters: validation and the launches, `workspace`
// holding the h3 hi / lo parts and the re-split weights.
static int hyena_filter_launch(const char* who, const m2_hyena_filter_params* params, int nfilters, int L, int d,
                               int order, int emb_dim, float w_mod, float shift, void* workspace, float* taps,
                               void* stream) {
  if (nfilters < 1 || nfilters > kMaxFilters)
    return set_error(M2_ERR_UNSUPPORTED, "%s: nfilters=%d not in [1, %d]", who, nfilters, kMaxFilters);
  int rc = check_filter_sizes(who, L, d, order, emb_dim);
  if (rc) return rc;
  TabByValue tab;
  FilterBatch& fb = tab.fb;
  for (int f = 0; f < kMaxFilters; ++f) {
    const m2_hyena_filter_params& p = params[f < nfilters ? f : 0];
    if (!p.z || !p.t || !p.freq || !p.deltas || !p.w0 || !p.b0 || !p.w1 || !p.b1 || !p.w2 || !p.b2 || !p.w3)
      return set_error(M2_ERR_ARG, "%s: filter %d has a null forward-MLP pointer", who, f);
    const bool rev = p.rw0 != nullptr;
    if (rev && (!p.rb0 || !p.rw1 || !p.rb1 || !p.rw2 || !p.rb2 || !p.rw3))
      return set_error(M2_ERR_ARG, "%s: filter %d has a partly null reverse MLP", who, f);
    fb.f[f].z = p.z; fb.f[f].t = p.t; fb.f[f].freq = p.freq; fb.f[f].deltas = p.deltas;
    fb.f[f].mlp[0] = MlpPtrs{p.w0, p.b0, p.w1, p.b1, p.w2, p.b2, p.w3};
    fb.f[f].mlp[1] = rev ? MlpPtrs{p.rw0, p.rb0, p.rw1, p.rb1, p.rw2, p.rb2, p.rw3}
                         : MlpPtrs{nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
  }
  uint16_t* h_hi = reinterpret_cast<uint16_t*>(workspace);
  uint16_t* h_lo = h_hi + (size_t)2 * nfilters * L * order;
  uint16_t* wsplit = h_lo + (size_t)2 * nfilters * L * order;
  uint16_t* w3split = wsplit + (size_t)2 * nfilters * 2 * kSplitPerLayer;
  float* w3scale = reinterpret_cast<float*>(workspace);      // (h3 and these are never in memory in the same call)
  return filter_launches(tab, nfilters, L, d, emb_dim, w_mod, shift, h_hi, h_lo, wsplit, w3split, w3scale, taps, (hipStream_t)stream);
}

extern "C" int m2_hyena_filter_fwd(const m2_hyena_filter_params* params, int nfilters, int L, int d, int order,
                                   int emb_dim, float w_mod, float shift, float* workspace, float* taps,
                                   void* stream) {
  if (!params || !workspace || !taps) return set_error(M2_ERR_ARG, "m2_hyena_filter_fwd: null pointer");
  return hyena_filter_launch("m2_hyena_filter_fwd", params, nfilters, L, d, order, emb_dim, w_mod, shift, workspace,
                             taps, stream);
}

// ---------------------------------------------------------------------------------------------
// The same computation for callers that cannot allocate a workspace: the h3 hi / lo parts go through a
// device array that is part of the library's code object.  Every GPU the library runs on holds its own copy
// of the array at its own address until the process ends; in host code the array's NAME is only a stand-in
// for the symbol, so its device address is looked up once per device (hipGetSymbolAddress) and only that
// address is ever handed to a kernel.
// ---------------------------------------------------------------------------------------------
static __device__ __align__(256) unsigned char scratch[M2_HYENA_FILTER_STATIC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {nullptr};      // device address of `scratch` on device i, once looked up

// Device address of the static scratch array on the current device (looked up on the first call per device).
int static_scratch_for_current_device(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return set_error(M2_ERR_LAUNCH, "m2_hyena_filter_fwd_static: hipGetDevice: %s", hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices)
    return set_error(M2_ERR_UNSUPPORTED, "m2_hyena_filter_fwd_static: device index %d beyond %d", dev, kMaxDevices - 1);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_ptr[dev] == nullptr) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || ptr == nullptr)
      return set_error(M2_ERR_LAUNCH, "m2_hyena_filter_fwd_static: hipGetSymbolAddress(scratch) on device %d: %s", dev,
                       hipGetErrorString(e));
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return M2_OK;
}
}  // namespace

extern "C" int m2_hyena_filter_fwd_static(const m2_hyena_filter_params* params, int nfilters, int L, int d, int order,
                                          int emb_dim, float w_mod, float shift, float* taps, void* stream) {
  if (!params || !taps) return set_error(M2_ERR_ARG, "m2_hyena_filter_fwd_static: null pointer");
  if (nfilters < 1 || L <= 0 || order <= 0)
    return set_error(M2_ERR_ARG, "m2_hyena_filter_fwd_static: sizes must be positive (nfilters=%d L=%d order=%d)", nfilters, L, order);
  const size_t need = m2_hyena_filter_workspace_bytes(nfilters, L, d, order);
  if (need > (size_t)M2_HYENA_FILTER_STATIC_SCRATCH_BYTES)
    return set_error(M2_ERR_UNSUPPORTED,
                     "m2_hyena_filter_fwd_static: nfilters=%d, L=%d needs %zu bytes of scratch, the static array holds %zu "
                     "(m2_hyena_filter_workspace_bytes); use m2_hyena_filter_fwd with a caller workspace",
                     nfilters, L, need, (size_t)M2_HYENA_FILTER_STATIC_SCRATCH_BYTES);
  void* ptr = nullptr;
  int rc = static_scratch_for_current_device(&ptr);
  if (rc) return rc;
  // every element that a kernel reads was written by an earlier kernel of the same call (h3 by hidden_kernel, or the split weights by
  // split_weights_kernel where h3 does not leave the chip), so nothing left by an earlier (possibly longer) call is ever read and nothing
  // needs clearing
  return hyena_filter_launch("m2_hyena_filter_fwd_static", params, nfilters, L, d, order, emb_dim, w_mod, shift, ptr,
                             taps, stream);
}

// ---------------------------------------------------------------------------------------------
// All filters of a batch of mixers -> their spectra, the pointer table in device memory.
// ---------------------------------------------------------------------------------------------
namespace {
struct BatchLayout {
  size_t h_lo, wsplit, w3split, w3scale, taps, total;      // byte offsets into the workspace (h_hi at 0)
  bool fused;                                     // projection + spectrum as one kernel, taps never in memory
};
BatchLayout batch_layout(int nmixers, int fpm, int L, int d) {
  const size_t nf = (size_t)nmixers * fpm;
  auto up = [](size_t v) { return (v + 255) & ~(size_t)255; };
  BatchLayout b;
  b.fused = project_spectrum_supported(L);
  b.h_lo = up(2 * nf * L * kOrder * sizeof(uint16_t));
  b.wsplit = b.h_lo + up(2 * nf * L * kOrder * sizeof(uint16_t));
  // (fused: hidden_kernel and project_spectrum_kernel split their weights themselves)
  b.w3split = b.wsplit + (b.fused ? 0 : up(2 * nf * 2 * (size_t)kSplitPerLayer * sizeof(uint16_t)));
  b.w3scale = b.w3split + (b.fused ? 0 : up(2 * nf * 2 * (size_t)d * kOrder * sizeof(uint16_t)));
  b.taps = b.w3scale + (b.fused ? 0 : up(2 * nf * (size_t)d * sizeof(float)));
  b.total = b.taps + (b.fused ? 0 : up(nf * (size_t)d * 2 * L * sizeof(float)));
  return b;
}
}  // namespace

extern "C" size_t m2_mixer_filters_workspace_bytes(int nmixers, int filters_per_mixer, int L, int d, int order) {
  if (nmixers <= 0 || filters_per_mixer < 1 || filters_per_mixer > 2 || L <= 0 || d <= 0 || order != kOrder) return 0;
  return batch_layout(nmixers, filters_per_mixer, L, d).total;
}

// validation of a batch of mixers, for the entry points whose table lives in device memory
static int check_mixers(const char* who, int nmixers, int filters_per_mixer, int L, int d, int order, int emb_dim) {
  if (filters_per_mixer < 1 || filters_per_mixer > 2)
    return set_error(M2_ERR_ARG, "%s: filters_per_mixer=%d must be 1 or 2", who, filters_per_mixer);
  // the MLPs of the batch (two per filter) are one grid dimension of the hidden-layer launch
  if (nmixers < 1 || (long)nmixers * filters_per_mixer * 2 > 65535)
    return set_error(M2_ERR_ARG, "%s: nmixers=%d with %d filters each: at most 65535 MLPs (two per filter) per call", who, nmixers,
                     filters_per_mixer);
  return check_filter_sizes(who, L, d, order, emb_dim);
}

extern "C" int m2_mixer_filters_fwd(const m2_hyena_filter_params* params_dev, const float* const* skip_dev, int nmixers,
                                    int filters_per_mixer, int L, int d, int order, int emb_dim, float w_mod,
                                    float shift, void* workspace, float* spec, void* stream) {
  const char* who = "m2_mixer_filters_fwd";
  if (!params_dev || !workspace || !spec) return set_error(M2_ERR_ARG, "%s: null pointer", who);
  int rc = check_mixers(who, nmixers, filters_per_mixer, L, d, order, emb_dim);
  if (rc) return rc;
  if (!m2_fftconv_supported_seqlen(L))
    return set_error(M2_ERR_UNSUPPORTED, "%s: L=%d unsupported (need L a power of two in [128, 32768])", who, L);
  const int nf = nmixers * filters_per_mixer;
  const BatchLayout lay = batch_layout(nmixers, filters_per_mixer, L, d);
  unsigned char* ws = reinterpret_cast<unsigned char*>(workspace);
  uint16_t* h_hi = reinterpret_cast<uint16_t*>(ws);
  uint16_t* h_lo = reinterpret_cast<uint16_t*>(ws + lay.h_lo);
  uint16_t* wsplit = lay.fused ? nullptr : reinterpret_cast<uint16_t*>(ws + lay.wsplit);
  uint16_t* w3split = lay.fused ? nullptr : reinterpret_cast<uint16_t*>(ws + lay.w3split);
  float* w3scale = lay.fused ? nullptr : reinterpret_cast<float*>(ws + lay.w3scale);
  float* taps = lay.fused ? nullptr : reinterpret_cast<float*>(ws + lay.taps);
  TabByPointer tab{reinterpret_cast<const FilterPtrs*>(params_dev)};
  hipStream_t s = (hipStream_t)stream;
  rc = filter_launches(tab, nf, L, d, emb_dim, w_mod, shift, h_hi, h_lo, wsplit, w3split, w3scale, taps, s);
  if (rc) return rc;
  const long spec_stride = (long)(m2_filter_spectrum_bytes(d, L) / sizeof(float));
  if (lay.fused)
    return launch_project_spectrum(tab.p, skip_dev, nmixers, filters_per_mixer, L, d, shift, h_hi, h_lo, spec, spec_stride, s);
  SpectrumBatch sb{taps, skip_dev, filters_per_mixer, spec_stride};
  return launch_filter_spectrum_any(nullptr, nullptr, nullptr, nullptr, spec, d, L, sb, nmixers, s);
}

// The taps alone, for a mixer core that transforms them itself: the same two launches, no room for taps in the workspace.
extern "C" size_t m2_mixer_taps_workspace_bytes(int nmixers, int filters_per_mixer, int L, int d, int order) {
  if (nmixers <= 0 || filters_per_mixer < 1 || filters_per_mixer > 2 || d <= 0 || order != kOrder || !project_with_hidden(L, d)) return 0;
  const BatchLayout lay = batch_layout(nmixers, filters_per_mixer, L, d);
  return lay.taps - lay.wsplit;      // (h3 does not leave the chip)
}

extern "C" int m2_mixer_taps_fwd(const m2_hyena_filter_params* params_dev, int nmixers, int filters_per_mixer, int L, int d, int order,
                                 int emb_dim, float w_mod, float shift, void* workspace, float* taps, void* stream) {
  const char* who = "m2_mixer_taps_fwd";
  if (!params_dev || !workspace || !taps) return set_error(M2_ERR_ARG, "%s: null pointer", who);
  int rc = check_mixers(who, nmixers, filters_per_mixer, L, d, order, emb_dim);
  if (rc) return rc;
  if (!project_with_hidden(L, d)) return set_error(M2_ERR_UNSUPPORTED, "%s: L=%d unsupported (need a multiple of 64 from 1024 on)", who, L);
  const BatchLayout lay = batch_layout(nmixers, filters_per_mixer, L, d);
  unsigned char* ws = reinterpret_cast<unsigned char*>(workspace);
  TabByPointer tab{reinterpret_cast<const FilterPtrs*>(params_dev)};
  return filter_launches(tab, nmixers * filters_per_mixer, L, d, emb_dim, w_mod, shift, nullptr, nullptr, reinterpret_cast<uint16_t*>(ws),
                         reinterpret_cast<uint16_t*>(ws + lay.w3split - lay.wsplit), reinterpret_cast<float*>(ws + lay.w3scale - lay.wsplit),
                         taps, (hipStream_t)stream);
}
