// LayerNorm, and embeddings + LayerNorm: rows are normalised and written in the three forms the next layer reads.
// `input_forms_kernel` writes two of them from rows as they are.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fft_regs.h"
#include "m2_internal.h"

namespace m2 {

// LayerNorm over the last dimension of x (M, d) fp32, eps inside the square root.
// Workgroup = 8 waves handles R = 8 RW rows; each wave normalises RW rows at once (all loads in flight
// together) and writes the row-major outputs from registers.  For the channel-major output the
// normalised rows also go through an LDS tile, 384 columns at a time (row pitch 384 + 64 / R floats, so that R
// consecutive tokens of 64 / R neighbouring channels fall in 64 different banks; 25 KB at R = 16), and are written back
// with lanes along the token axis: every store instruction covers R consecutive tokens of 64 / R channels.
// The input is read once.  PER = d / 64 values per lane.
//
// Many rows are bound by memory: bf16 in, bf16 + channel-major fp32 out is 8 bytes per value, 6.3 TB/s at M = 32768,
// d = 768.  Few rows are bound by one wave's serial chain and by how many compute units have a workgroup at all, so the fewer
// rows per workgroup the better down to where the channel-major stores (4 R bytes of a channel) become too short.
// us per call, RW = 1 / 2 / 4 (4: 8 RW = 32 rows, no longer built; at d > 1024 its registers do not fit):
//   d = 768:   M = 128 3.9 / 5.1 / 8.0   2048 6.0 / 6.3 / 9.2    2560 7.1 / 6.5 / 9.5    4096 9.2 / 7.6 / 10.2
//              8192 15.1 / 10.5 / 12.6   16384 27.8 / 16.9 / 17.9   32768 55 / 31.9 / 32.8
//   d = 960:   M = 128 4.3 / 5.9 / 9.4   2048 7.2 / 7.3 / 10.9   2560 8.2 / 7.4 / 11.2   32768 66 / 41.0 / 40.2
//   d = 1536:  M = 128 5.9 / 8.3         2048 9.9 / 10.1         2560 12.3 / 10.6        8192 27.6 / 18.3
//   d = 1792:  M = 128 6.4 / 9.7         2048 11.0 / 11.6        2560 13.2 / 12.0        10240 38.9 / 28.9
template <int PER, int RW>
struct LnShape {
  static constexpr int R = 8 * RW;                  // rows per workgroup
  static constexpr int PC = PER < 6 ? PER : 6;      // 64-column groups per tile pass
  static constexpr int NPASS = (PER + PC - 1) / PC;
  static constexpr int PITCH = 64 * PC + 64 / R;
  static constexpr size_t LDS_BYTES = (size_t)R * PITCH * sizeof(float);
};
// Where the rows come from when the kernel normalises embeddings instead of a matrix:
// row m = word[ids[m]] + type[tt[m] or 0] (+ pos[pos_ids[m] or m % L]).
// Every index is clamped into its table before it is used, so a bad id reads a valid row instead of
// foreign memory; when that happens and `bad_index` is not null the kernel stores 1 there (plain vector
// store; the caller cleared it before the launch and reads it afterwards to report the error).
struct EmbedSource {
  const long long* ids;     // (M)
  const long long* tt;      // (M) or null: type 0
  const long long* pos_ids; // (M) or null: m % L
  const float* word;        // (vocab, d)
  const float* type;        // (type_vocab, d)
  const float* pos;         // (max_positions, d) or null: no position embeddings
  int L;
  int vocab, type_vocab, max_positions;      // rows of the three tables
  int* bad_index;           // or null
};
__device__ __forceinline__ long long clamp_index(long long i, int rows, bool& bad) {
  if (i < 0 || i >= rows) {
    bad = true;
    return i < 0 ? 0 : rows - 1;
  }
  return i;
}
// IN: float, or uint16_t for rows stored as bf16 (the sum the reference's autocast path feeds its LayerNorm).
template <int PER, int RW, bool EMBED, typename IN = float>
__global__ __launch_bounds__(512) void layernorm_kernel(const IN* __restrict__ x, EmbedSource src,
                                                        const float* __restrict__ gamma,
                                                        const float* __restrict__ beta, float eps,
                                                        float* __restrict__ out_f32,       // (M, d) or null
                                                        uint16_t* __restrict__ out_bf16,   // (M, d) or null
                                                        float* __restrict__ out_t,         // (d, M) or null
                                                        int M) {
  using S = LnShape<PER, RW>;
  constexpr int d = 64 * PER, R = S::R, PITCH = S::PITCH;
  constexpr int PC = S::PC, NPASS = S::NPASS;
  extern __shared__ float tile[];                       // [R][PITCH], used only with out_t
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int m0 = blockIdx.x * R;
  float g[PER], bt[PER];
  static_for<0, PER>([&](auto ii) {
    g[decltype(ii)::value] = gamma[lane + 64 * decltype(ii)::value];
    bt[decltype(ii)::value] = beta[lane + 64 * decltype(ii)::value];
  });
  float v[RW][PER];
  float sum[RW], sq[RW];
  static_for<0, RW>([&](auto rr_) {
    constexpr int rr = decltype(rr_)::value;
    int m = m0 + wave * RW + rr;
    m = m < M ? m : M - 1;
    if constexpr (!EMBED) {
      const IN* xr = x + (long)m * d;
      static_for<0, PER>([&](auto ii) {
        if constexpr (sizeof(IN) == 2) v[rr][decltype(ii)::value] = bf16_to_f32(xr[lane + 64 * decltype(ii)::value]);
        else v[rr][decltype(ii)::value] = xr[lane + 64 * decltype(ii)::value];
      });
    } else {
      bool bad = false;
      const float* wr = src.word + clamp_index(src.ids[m], src.vocab, bad) * d;
      const float* tr = src.type + (src.tt ? clamp_index(src.tt[m], src.type_vocab, bad) : 0) * d;
      static_for<0, PER>([&](auto ii) {
        constexpr int i = decltype(ii)::value;
        v[rr][i] = wr[lane + 64 * i] + tr[lane + 64 * i];
      });
      if (src.pos) {
        const float* pr = src.pos + (src.pos_ids ? clamp_index(src.pos_ids[m], src.max_positions, bad)
                                                 : (long long)(m % src.L)) * d;
        static_for<0, PER>([&](auto ii) {
          constexpr int i = decltype(ii)::value;
          v[rr][i] += pr[lane + 64 * i];
        });
      }
      if (bad && src.bad_index && lane == 0) *src.bad_index = 1;
    }
  });
  static_for<0, RW>([&](auto rr_) {
    constexpr int rr = decltype(rr_)::value;
    float s = 0.f;
    static_for<0, PER>([&](auto ii) { s += v[rr][decltype(ii)::value]; });
    sum[rr] = s;
  });
  for (int o = 32; o > 0; o >>= 1)
    static_for<0, RW>([&](auto rr_) { sum[decltype(rr_)::value] += __shfl_xor(sum[decltype(rr_)::value], o); });
  static_for<0, RW>([&](auto rr_) {
    constexpr int rr = decltype(rr_)::value;
    sq[rr] = ln_squares<d>(v[rr], sum[rr]);
  });
  for (int o = 32; o > 0; o >>= 1)
    static_for<0, RW>([&](auto rr_) { sq[decltype(rr_)::value] += __shfl_xor(sq[decltype(rr_)::value], o); });
  static_for<0, RW>([&](auto rr_) {
    constexpr int rr = decltype(rr_)::value;
    const int m = m0 + wave * RW + rr;
    const float rstd = ln_rstd<d>(sq[rr], eps);
    static_for<0, PER>([&](auto ii) {
      constexpr int i = decltype(ii)::value;
      v[rr][i] = ln_value<d>(v[rr][i], sum[rr], rstd, g[i], bt[i]);
      if (m < M) {
        if (out_f32) out_f32[(long)m * d + lane + 64 * i] = v[rr][i];
        if (out_bf16) out_bf16[(long)m * d + lane + 64 * i] = f32_to_bf16(v[rr][i]);
      }
    });
  });
  if (!out_t) return;
  // lane = (token tk, channel offset h): R tokens x (64 / R) channels per store instruction
  constexpr int CH = 64 / R;
  const int tk = lane % R, h = lane / R;
  const int mt = m0 + tk;
  static_for<0, NPASS>([&](auto pp) {
    constexpr int ps = decltype(pp)::value;
    constexpr int i0 = ps * PC, i1 = (i0 + PC < PER) ? i0 + PC : PER;      // 64-column groups of this pass
    if (ps > 0) __syncthreads();                                            // the previous pass has been read
    static_for<0, RW>([&](auto rr_) {
      constexpr int rr = decltype(rr_)::value;
      static_for<i0, i1>([&](auto ii) {
        constexpr int i = decltype(ii)::value;
        tile[(wave * RW + rr) * PITCH + lane + 64 * (i - i0)] = v[rr][i];
      });
    });
    __syncthreads();
    if (mt < M) {
      const float* src = tile + tk * PITCH + h;
      float* dst = out_t + (long)(64 * i0 + h) * M + mt;
#pragma unroll 4
      for (int c0 = wave * CH; c0 < 64 * (i1 - i0); c0 += 8 * CH) dst[(long)c0 * M] = src[c0];
    }
  });
}

// ---------------------------------------------------------------------------------------------
// The two forms the first layer reads, from rows in fp32: bf16 rows and a channel-major fp32 copy, one pass.
// A workgroup takes 64 rows x 64 columns: whole 256-byte pieces in, 128-byte and (through LDS, pitch 65: no bank
// conflicts) 256-byte pieces out.
// Memory-bound: 10 bytes per value, 6.6 TB/s.  us, this against a conversion and a transposing copy: d = 768, M = 128
// 3.5 / 4.2, 4096 7.0 / 19.7, 31744 36.8 / 133; d = 1792, M = 10240 27.9 / 92.7.
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void input_forms_kernel(const float* __restrict__ x, uint16_t* __restrict__ out_bf16,
                                                          float* __restrict__ out_t, int M, int d) {
  __shared__ float tile[64 * 65];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, cols = d >> 6;
  const int c0 = (int)(blockIdx.x % cols) * 64;
  const long m0 = (long)(blockIdx.x / cols) * 64;
  float v[16];
  static_for<0, 16>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    const long m = m0 + 16 * wave + i;
    v[i] = x[(m < M ? m : M - 1) * d + c0 + lane];
  });
  static_for<0, 16>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    const long m = m0 + 16 * wave + i;
    if (m < M) out_bf16[m * d + c0 + lane] = f32_to_bf16(v[i]);
    tile[lane * 65 + 16 * wave + i] = v[i];
  });
  __syncthreads();
  if (m0 + lane >= M) return;
  static_for<0, 16>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    out_t[(long)(c0 + 16 * wave + i) * M + m0 + lane] = tile[(16 * wave + i) * 65 + lane];
  });
}

template <int PER, int RW, bool EMBED, typename IN>
static int launch_layernorm_rw(const IN* x, const EmbedSource& src, const float* gamma, const float* beta, float eps,
                               float* out_f32, uint16_t* out_bf16, float* out_channel_major, int M, hipStream_t st) {
  using S = LnShape<PER, RW>;
  const size_t lds = out_channel_major ? S::LDS_BYTES : 0;
  hipLaunchKernelGGL((layernorm_kernel<PER, RW, EMBED, IN>), dim3((M + S::R - 1) / S::R), dim3(512), lds, st, x, src, gamma,
                     beta, eps, out_f32, out_bf16, out_channel_major, M);
  return check_launch("layernorm");
}

// One row per wave while that gives every compute unit at most one workgroup, two beyond (figures above: the lines cross between
// M = 2048 and 2560 at every width).
static bool ln_one_row_per_wave(int M) { return (M + 7l) / 8 <= num_cus(); }

template <bool EMBED, typename IN = float>
static int launch_layernorm(const IN* x, const EmbedSource& src, const float* gamma, const float* beta, float eps,
                            float* out_f32, void* out_bf16, float* out_channel_major, int M, int d, void* stream) {
  hipStream_t st = (hipStream_t)stream;
  uint16_t* o16 = (uint16_t*)out_bf16;
  const bool one = ln_one_row_per_wave(M);
  switch (d / 64) {
#define LN_CASE(P)                                                                                                            \
  case P:                                                                                                                     \
    return one ? launch_layernorm_rw<P, 1, EMBED, IN>(x, src, gamma, beta, eps, out_f32, o16, out_channel_major, M, st)       \
               : launch_layernorm_rw<P, 2, EMBED, IN>(x, src, gamma, beta, eps, out_f32, o16, out_channel_major, M, st);
    LN_CASE(1) LN_CASE(2) LN_CASE(3) LN_CASE(4) LN_CASE(5) LN_CASE(6) LN_CASE(7) LN_CASE(8) LN_CASE(9) LN_CASE(10) LN_CASE(11)
    LN_CASE(12) LN_CASE(13) LN_CASE(14) LN_CASE(15) LN_CASE(16) LN_CASE(17) LN_CASE(18) LN_CASE(19) LN_CASE(20) LN_CASE(21)
    LN_CASE(22) LN_CASE(23) LN_CASE(24) LN_CASE(25) LN_CASE(26) LN_CASE(27) LN_CASE(28) LN_CASE(29) LN_CASE(30) LN_CASE(31)
    LN_CASE(32)
#undef LN_CASE
  }
  return set_error(M2_ERR_UNSUPPORTED, "layernorm: d=%d", d);
}

}  // namespace m2

using namespace m2;

extern "C" int m2_layernorm_fwd(const float* x, const float* gamma, const float* beta, float eps, float* out_f32,
                                void* out_bf16, float* out_channel_major, int M, int d, void* stream) {
  if (!x || !gamma || !beta) return set_error(M2_ERR_ARG, "m2_layernorm_fwd: null pointer");
  if (M <= 0 || d <= 0 || d % 64 != 0 || d > 2048)
    return set_error(M2_ERR_UNSUPPORTED, "m2_layernorm_fwd: need M > 0 and d a multiple of 64 up to 2048 (M=%d d=%d)", M, d);
  return launch_layernorm<false>(x, EmbedSource{}, gamma, beta, eps, out_f32, out_bf16, out_channel_major, M, d, stream);
}

extern "C" int m2_layernorm_bf16_fwd(const void* x, const float* gamma, const float* beta, float eps, float* out_f32,
                                     void* out_bf16, float* out_channel_major, int M, int d, void* stream) {
  if (!x || !gamma || !beta) return set_error(M2_ERR_ARG, "m2_layernorm_bf16_fwd: null pointer");
  if (M <= 0 || d <= 0 || d % 64 != 0 || d > 2048)
    return set_error(M2_ERR_UNSUPPORTED, "m2_layernorm_bf16_fwd: need M > 0 and d a multiple of 64 up to 2048 (M=%d d=%d)", M, d);
  return launch_layernorm<false, uint16_t>((const uint16_t*)x, EmbedSource{}, gamma, beta, eps, out_f32, out_bf16,
                                           out_channel_major, M, d, stream);
}

extern "C" int m2_embed_layernorm_fwd(const long long* input_ids, const long long* token_type_ids,
                                      const long long* position_ids, const float* word_emb, const float* type_emb,
                                      const float* pos_emb, int vocab_size, int type_vocab_size, int max_positions,
                                      const float* gamma, const float* beta, float eps, float* out_f32, void* out_bf16,
                                      float* out_channel_major, int* bad_index, int B, int L, int d, void* stream) {
  if (!input_ids || !word_emb || !type_emb || !gamma || !beta)
    return set_error(M2_ERR_ARG, "m2_embed_layernorm_fwd: null pointer");
  if (B <= 0 || L <= 0 || d <= 0 || d % 64 != 0 || d > 2048)
    return set_error(M2_ERR_UNSUPPORTED, "m2_embed_layernorm_fwd: need B, L > 0 and d a multiple of 64 up to 2048 (B=%d L=%d d=%d)", B, L, d);
  if ((long)B * L > 0x7fffffffL) return set_error(M2_ERR_UNSUPPORTED, "m2_embed_layernorm_fwd: B * L = %ld does not fit an int", (long)B * L);
  if (position_ids && !pos_emb) return set_error(M2_ERR_ARG, "m2_embed_layernorm_fwd: position_ids without a position table");
  if (vocab_size <= 0 || type_vocab_size <= 0 || (pos_emb && max_positions <= 0))
    return set_error(M2_ERR_ARG, "m2_embed_layernorm_fwd: table sizes must be positive (vocab=%d type_vocab=%d max_positions=%d)",
                     vocab_size, type_vocab_size, max_positions);
  if (pos_emb && !position_ids && L > max_positions)
    return set_error(M2_ERR_ARG, "m2_embed_layernorm_fwd: sequence length %d exceeds the position table (%d rows)", L, max_positions);
  const EmbedSource src{input_ids, token_type_ids, position_ids, word_emb, type_emb, pos_emb, L,
                        vocab_size, type_vocab_size, max_positions, bad_index};
  return launch_layernorm<true>((const float*)nullptr, src, gamma, beta, eps, out_f32, out_bf16, out_channel_major, B * L, d, stream);
}

extern "C" int m2_input_forms_fwd(const float* x, void* out_bf16, float* out_channel_major, int M, int d, void* stream) {
  if (!x || !out_bf16 || !out_channel_major) return set_error(M2_ERR_ARG, "m2_input_forms_fwd: null pointer");
  if (M <= 0 || d <= 0 || d % 64 != 0)
    return set_error(M2_ERR_UNSUPPORTED, "m2_input_forms_fwd: need M > 0 and d a multiple of 64 (M=%d d=%d)", M, d);
  const long groups = ((long)M + 63) / 64 * (d / 64);
  if (groups > 0x7fffffffL) return set_error(M2_ERR_UNSUPPORTED, "m2_input_forms_fwd: too many tiles (M=%d d=%d)", M, d);
  hipLaunchKernelGGL(input_forms_kernel, dim3((unsigned)groups), dim3(256), 0, (hipStream_t)stream, x, (uint16_t*)out_bf16,
                     out_channel_major, M, d);
  return check_launch("input_forms");
}
