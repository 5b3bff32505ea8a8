// Dense and block-diagonal bf16 matrix products on the tile engine (gemm_engine.h) and, for few rows, on a kernel that
// splits K over the waves of a workgroup.
#include "gemm_engine.h"

namespace m2 {

// ---------------------------------------------------------------------------------------------
// Few rows: a 32 x 32 tile of OUT[j][i] per workgroup, K split over its NW waves, every wave's operands requested at
// once straight into registers (no LDS stage, no loop: one memory latency), partial sums added through LDS.  GLU: two
// products (gate block and value block of a gated block-diagonal layer) and gelu(gate) * value on the sums.
// ---------------------------------------------------------------------------------------------
constexpr int kRedRow = 36;      // floats between two j of a partial tile

// JT: 16-wide tiles along j of a workgroup.
template <int NW, int KSMAX, bool QKM, bool GLU, int JT>
struct SmallShape {
  static constexpr int kProd = GLU ? 2 : 1;
  static constexpr int kRed = NW * kProd * 16 * JT * kRedRow * 4;
  static constexpr int kStage = QKM ? NW * KSMAX * 2048 : 0;
  static constexpr int kLds = kRed > kStage ? kRed : kStage;
};

template <int NW, int KSMAX, bool QKM, bool GLU, int JT>
__global__ __launch_bounds__(64 * NW) void small_gemm_kernel(GemmArgs g) {
  using S = SmallShape<NW, KSMAX, QKM, GLU, JT>;
  static_assert(JT == 2 || !QKM, "64-byte rows of a channel-major operand");
  static_assert(!(QKM && GLU), "the gated product reads row-major activations");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, i16 = lane & 15, q4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ntiles = g.ti * g.tj;
  const int xcd = blockIdx.x & 7;
  const int tile = (int)((long)xcd * ntiles / 8) + (int)(blockIdx.x >> 3);
  if (tile >= (int)((long)(xcd + 1) * ntiles / 8)) return;
  int i0, j0, blk;
  tile_origin<32, 16 * JT>(g, tile, i0, j0, blk);
  const int nks = (g.nk + 31) / 32;
  const int s0 = wave * nks / NW, ns = (wave + 1) * nks / NW - s0;
  const u32x4 zero = {0u, 0u, 0u, 0u};

  u32x4 pf[S::kProd][KSMAX][2], qf[S::kProd][KSMAX][JT];
  static_for<0, S::kProd>([&](auto dd) {
    constexpr int D = decltype(dd)::value;
    // GLU: gated columns of weight block blk (gate, read against the same block of Q) and of block blk + nblk (value)
    const int wb = blk + D * g.nblk, qb = GLU ? wb : blk;
    const uint16_t* pb = g.p + wb * g.pblk + 32 * s0 + 8 * q4;
    const uint16_t* qbase = g.q + (long)qb * g.nk + 32 * s0 + 8 * q4;
    static_for<0, 2>([&](auto tt) {
      constexpr int t = decltype(tt)::value;
      int i = i0 + 8 * (i16 >> 2) + 4 * t + (i16 & 3);
      i = i < g.ni ? i : g.ni - 1;
      int j = j0 + 16 * t + i16;
      j = j < g.nj ? j : g.nj - 1;
      static_for<0, KSMAX>([&](auto ss) {
        constexpr int s = decltype(ss)::value;
        pf[D][s][t] = zero;
        if constexpr (!QKM && t < JT) qf[D][s][t] = zero;
        if (s < ns && 32 * (s0 + s) + 8 * q4 < g.nk) {
          pf[D][s][t] = *reinterpret_cast<const u32x4*>(pb + (long)i * g.ldp + 32 * s);
          if constexpr (!QKM && t < JT) qf[D][s][t] = *reinterpret_cast<const u32x4*>(qbase + (long)j * g.ldq + 32 * s);
        }
      });
    });
  });
  if constexpr (QKM) {
    // the wave's k rows (64 bytes = 32 j each) through its own LDS rows, read back transposed
    const unsigned lds0 = (unsigned)(uintptr_t)smem + wave * (KSMAX * 2048);
    int j = j0 + 8 * (lane & 3);
    j = j <= g.nj - 8 ? j : g.nj - 8;
    const unsigned voff = (unsigned)(((long)(lane >> 2) * g.ldq + j) * 2);
    for (int s = 0; s < 2 * ns; ++s)
      load_to_lds(lds0 + s * 1024, voff, (const unsigned char*)g.q + (32l * s0 + 16 * s) * g.ldq * 2);
    __builtin_amdgcn_s_waitcnt(kWaitVm0);
    asm volatile("" ::: "memory");
    typedef __attribute__((address_space(3))) s16x4 lds4;
    const unsigned a0 = lds0 + (8 * q4 + (i16 >> 2)) * 64 + 8 * (i16 & 3);
    static_for<0, KSMAX>([&](auto ss) {
      constexpr int s = decltype(ss)::value;
      static_for<0, 2>([&](auto tt) {
        constexpr int t = decltype(tt)::value;
        qf[0][s][t] = zero;
        if (s < ns) {
          const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)(uintptr_t)(a0 + s * 2048 + 32 * t));
          const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)(uintptr_t)(a0 + s * 2048 + 32 * t + 256));
          qf[0][s][t] = __builtin_bit_cast(u32x4, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
      });
    });
  }
  floatx4 acc[S::kProd][2][JT];
  static_for<0, S::kProd>([&](auto dd) {
    constexpr int D = decltype(dd)::value;
    static_for<0, 2 * JT>([&](auto tt) {
      constexpr int t = decltype(tt)::value / JT, u = decltype(tt)::value % JT;
      floatx4 a = {0.f, 0.f, 0.f, 0.f};
      static_for<0, KSMAX>([&](auto ss) {
        constexpr int s = decltype(ss)::value;
        a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, pf[D][s][t]), __builtin_bit_cast(bf16x8, qf[D][s][u]), a, 0, 0, 0);
      });
      acc[D][t][u] = a;
    });
  });
  float* red = reinterpret_cast<float*>(smem);
  if constexpr (QKM) __syncthreads();      // every wave has read its stage: the partial sums take its place
  static_for<0, S::kProd>([&](auto dd) {
    constexpr int D = decltype(dd)::value;
    static_for<0, 2 * JT>([&](auto tt) {
      constexpr int t = decltype(tt)::value / JT, u = decltype(tt)::value % JT;
      *reinterpret_cast<floatx4*>(red + ((wave * S::kProd + D) * 16 * JT + 16 * u + i16) * kRedRow + 8 * q4 + 4 * t) = acc[D][t][u];
    });
  });
  __syncthreads();
  if (tid >= 128 * JT) return;
  const int j = tid >> 3, i4 = 4 * (tid & 7);
  floatx4 sum[S::kProd];
  static_for<0, S::kProd>([&](auto dd) {
    constexpr int D = decltype(dd)::value;
    floatx4 v = {0.f, 0.f, 0.f, 0.f};
    static_for<0, NW>([&](auto ww) {
      v += *reinterpret_cast<const floatx4*>(red + ((decltype(ww)::value * S::kProd + D) * 16 * JT + j) * kRedRow + i4);
    });
    sum[D] = v;
  });
  const int i = i0 + i4;
  if (i >= g.ni || j0 + j >= g.nj) return;
  const long o = (long)(j0 + j) * g.ldo + blk * g.ni + i;
  float r[4];
  if constexpr (GLU) {
    static_for<0, 4>([&](auto e) { r[decltype(e)::value] = gelu_erf_poly(sum[0][decltype(e)::value]) * sum[1][decltype(e)::value]; });
  } else {
    static_for<0, 4>([&](auto e) { r[decltype(e)::value] = sum[0][decltype(e)::value]; });
    if (g.bias) static_for<0, 4>([&](auto e) { r[decltype(e)::value] += g.bias[blk * g.ni + i + decltype(e)::value]; });
    if (g.resid) {
      const u32x2 rr = *reinterpret_cast<const u32x2*>(g.resid + o);
      r[0] += __uint_as_float(rr.x << 16); r[1] += __uint_as_float(rr.x & 0xffff0000u);
      r[2] += __uint_as_float(rr.y << 16); r[3] += __uint_as_float(rr.y & 0xffff0000u);
    }
  }
  u32x2 pk = {pack_bf16x2(r[0], r[1]), pack_bf16x2(r[2], r[3])};
  *reinterpret_cast<u32x2*>(g.out + o) = pk;
}

template <int NW, int KSMAX, bool QKM, bool GLU, int JT>
static int launch_small_j(GemmArgs g, hipStream_t st) {
  using S = SmallShape<NW, KSMAX, QKM, GLU, JT>;
  auto kern = small_gemm_kernel<NW, KSMAX, QKM, GLU, JT>;
  g.ti = g.nblk * ((g.ni + 31) / 32);
  g.tj = (g.nj + 16 * JT - 1) / (16 * JT);
  if (S::kLds > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, S::kLds);
    if (e != hipSuccess) return set_error(M2_ERR_LAUNCH, "hipFuncSetAttribute(small_gemm): %s", hipGetErrorString(e));
  }
  const int nt = g.ti * g.tj;
  hipLaunchKernelGGL(kern, dim3(8 * ((nt + 7) / 8)), dim3(64 * NW), S::kLds, st, g);
  return check_launch("small_gemm");
}
// 32 x 16 tiles where 32 x 32 ones leave half of the compute units without one: a workgroup fetches 48 operand rows instead of 64.
// us per forward, L = 128, B = 1 (`wo`, 96 tiles of 32 x 32), before / now: 12 x 768 494 / 485, 12 x 960 532 / 520.
template <int NW, int KSMAX, bool QKM, bool GLU>
static int launch_small(const GemmArgs& g, hipStream_t st) {
  if constexpr (!QKM && !GLU) {
    if (2l * g.nblk * ((g.ni + 31) / 32) * ((g.nj + 31) / 32) <= num_cus()) return launch_small_j<NW, KSMAX, QKM, GLU, 1>(g, st);
  }
  return launch_small_j<NW, KSMAX, QKM, GLU, 2>(g, st);
}

// ---------------------------------------------------------------------------------------------
// LayerNorm and in_linear of few rows as one kernel: rows of s (M, d) bf16 are normalised on their way into the product
//   out (N, M) = w (N, d) LayerNorm(s)^T
// A workgroup has 32 rows and 16 JT output channels.  The rows come whole into LDS (48 KB at d = 768), where every wave takes the
// statistics of four as layernorm_kernel does, column by column and lane by lane and by the same functions (ln_squares, ...), so that the
// rows have its bits;
// then every wave normalises its eighth of K in operand layout, and products and sums are small_gemm_kernel's.  The channel-major fp32
// form that the mixer core reads is written by the workgroups of the first d channels' worth of tiles, 32 of its channels each.
//
// What it takes away is a launch in a chain of dependent ones, and a kernel that is a load, a reduction and a store long with 16
// workgroups.  us per forward, two kernels / one, batches of L = 128: 12 x 768 B = 1 551 / 508, 2 617 / 583, 12 x 960 B = 1 605 / 549,
// 24 x 1536 B = 1 1757 / 1724, 2 2018 / 1980, 12 x 1792 B = 1 1098 / 1055, 2 1243 / 1225 (6 to 10 us of the first three are the filters').
// ---------------------------------------------------------------------------------------------
template <int PER, int JT>
struct LnGemmShape {
  static constexpr int d = 64 * PER, KS = (d / 32 + 7) / 8, PITCH = d + 8;      // bf16 per row in LDS: 16-byte accesses of 16 rows spread over the banks
  static constexpr int kRows = 32 * PITCH * 2, kRed = 8 * 16 * JT * kRedRow * 4;
  static constexpr int kLds = (kRows > kRed ? kRows : kRed) + 32 * 8;
};
template <int PER, int JT>
__global__ __launch_bounds__(512) void ln_gemm_kernel(const uint16_t* __restrict__ s, const float* __restrict__ gamma, const float* __restrict__ beta,
                                                      float eps, const uint16_t* __restrict__ w, uint16_t* __restrict__ out, long ldo,
                                                      float* __restrict__ out_t /* (d, M) or null */, int M, int N, int ti, int tj) {
  using S = LnGemmShape<PER, JT>;
  constexpr int d = S::d, KS = S::KS, PITCH = S::PITCH, NKS = d / 32;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  uint16_t* rows = reinterpret_cast<uint16_t*>(smem);
  float2* stats = reinterpret_cast<float2*>(smem + (S::kLds - 32 * 8));      // sum, 1 / deviation
  const int tid = threadIdx.x, lane = tid & 63, i16 = lane & 15, q4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // the tiles of an XCD keep the weights' rows together: they are read by one L2 only
  const int ntiles = ti * tj, xcd = blockIdx.x & 7;
  const int tile = (int)((long)xcd * ntiles / 8) + (int)(blockIdx.x >> 3);
  if (tile >= (int)((long)(xcd + 1) * ntiles / 8)) return;
  const int jt = __builtin_amdgcn_readfirstlane(tile / ti), i0 = 32 * (tile - jt * ti), j0 = 16 * JT * jt;
  const int s0 = wave * NKS / 8, ns = (wave + 1) * NKS / 8 - s0;
  const u32x4 zero = {0u, 0u, 0u, 0u};

  // everything that is read is requested here: rows, weights, the scales of this wave's columns
  constexpr int kPieces = 32 * d / 8, kLoads = (kPieces + 511) / 512;
  u32x4 raw[kLoads];
  static_for<0, kLoads>([&](auto ll) {
    constexpr int l = decltype(ll)::value;
    const int p = tid + 512 * l, r = p / (d / 8), c = p % (d / 8);
    int m = i0 + r;
    m = m < M ? m : M - 1;
    if (512 * (l + 1) <= kPieces || p < kPieces) raw[l] = *reinterpret_cast<const u32x4*>(s + (long)m * d + 8 * c);
  });
  u32x4 qf[JT][KS];
  static_for<0, JT>([&](auto jj) {
    int j = j0 + 16 * decltype(jj)::value + i16;
    j = j < N ? j : N - 1;
    static_for<0, KS>([&](auto ss) {
      constexpr int k = decltype(ss)::value;
      qf[decltype(jj)::value][k] = zero;
      if (k < ns) qf[decltype(jj)::value][k] = *reinterpret_cast<const u32x4*>(w + (long)j * d + 32 * (s0 + k) + 8 * q4);
    });
  });
  float g[KS][8], b[KS][8];
  static_for<0, KS>([&](auto ss) {
    constexpr int k = decltype(ss)::value;
    const int at = k < ns ? 32 * (s0 + k) + 8 * q4 : 0;
    static_for<0, 2>([&](auto hh) {
      constexpr int h = decltype(hh)::value;
      const floatx4 gv = *reinterpret_cast<const floatx4*>(gamma + at + 4 * h), bv = *reinterpret_cast<const floatx4*>(beta + at + 4 * h);
      static_for<0, 4>([&](auto e) {
        g[k][4 * h + decltype(e)::value] = gv[decltype(e)::value];
        b[k][4 * h + decltype(e)::value] = bv[decltype(e)::value];
      });
    });
  });
  static_for<0, kLoads>([&](auto ll) {
    constexpr int l = decltype(ll)::value;
    const int p = tid + 512 * l, r = p / (d / 8), c = p % (d / 8);
    if (512 * (l + 1) <= kPieces || p < kPieces) *reinterpret_cast<u32x4*>(rows + r * PITCH + 8 * c) = raw[l];
  });
  __syncthreads();

  // ---- statistics of the wave's four rows, as in layernorm_kernel
  {
    float v[4][PER], sum[4], sq[4];
    static_for<0, 4>([&](auto rr) {
      constexpr int r = decltype(rr)::value;
      static_for<0, PER>([&](auto ii) { v[r][decltype(ii)::value] = bf16_to_f32(rows[(4 * wave + r) * PITCH + lane + 64 * decltype(ii)::value]); });
      float t = 0.f;
      static_for<0, PER>([&](auto ii) { t += v[r][decltype(ii)::value]; });
      sum[r] = t;
    });
    for (int o = 32; o > 0; o >>= 1) static_for<0, 4>([&](auto rr) { sum[decltype(rr)::value] += __shfl_xor(sum[decltype(rr)::value], o); });
    static_for<0, 4>([&](auto rr) {
      constexpr int r = decltype(rr)::value;
      sq[r] = ln_squares<d>(v[r], sum[r]);
    });
    for (int o = 32; o > 0; o >>= 1) static_for<0, 4>([&](auto rr) { sq[decltype(rr)::value] += __shfl_xor(sq[decltype(rr)::value], o); });
    static_for<0, 4>([&](auto rr) {
      constexpr int r = decltype(rr)::value;
      if (lane == r) stats[4 * wave + r] = make_float2(sum[r], ln_rstd<d>(sq[r], eps));
    });
  }
  __syncthreads();

  // ---- the wave's operands: row 8 (i16 / 4) + 4 t + i16 % 4 of the tile, K = 32 (s0 + k) + 8 q4 .. + 7
  u32x4 pf[2][KS];
  static_for<0, 2>([&](auto tt) {
    constexpr int t = decltype(tt)::value;
    const int r = 8 * (i16 >> 2) + 4 * t + (i16 & 3);
    const float2 st = stats[r];
    static_for<0, KS>([&](auto ss) {
      constexpr int k = decltype(ss)::value;
      const u32x4 x = *reinterpret_cast<const u32x4*>(rows + r * PITCH + (k < ns ? 32 * (s0 + k) + 8 * q4 : 0));
      static_for<0, 4>([&](auto e) {
        constexpr int i = decltype(e)::value;
        const float lo = ln_value<d>(__uint_as_float(x[i] << 16), st.x, st.y, g[k][2 * i], b[k][2 * i]);
        const float hi = ln_value<d>(__uint_as_float(x[i] & 0xffff0000u), st.x, st.y, g[k][2 * i + 1], b[k][2 * i + 1]);
        pf[t][k][i] = k < ns ? pack_bf16x2(lo, hi) : 0u;
      });
    });
  });
  floatx4 acc[2][JT];
  static_for<0, 2>([&](auto tt) {
    constexpr int t = decltype(tt)::value;
    static_for<0, JT>([&](auto jj) {
      constexpr int u = decltype(jj)::value;
      floatx4 a = {0.f, 0.f, 0.f, 0.f};
      static_for<0, KS>([&](auto ss) {
        constexpr int k = decltype(ss)::value;
        a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, pf[t][k]), __builtin_bit_cast(bf16x8, qf[u][k]), a, 0, 0, 0);
      });
      acc[t][u] = a;
    });
  });
  if (out_t && jt < d / 32) {
    const int c = 32 * jt + (tid >> 4), r = 2 * (tid & 15);
    if (i0 + r < M) {      // (M is even)
      const float gc = gamma[c], bc = beta[c];
      const float2 sa = stats[r], sb = stats[r + 1];
      const float va = ln_value<d>(bf16_to_f32(rows[r * PITCH + c]), sa.x, sa.y, gc, bc),
                  vb = ln_value<d>(bf16_to_f32(rows[(r + 1) * PITCH + c]), sb.x, sb.y, gc, bc);
      *reinterpret_cast<float2*>(out_t + (long)c * M + i0 + r) = make_float2(va, vb);
    }
  }
  __syncthreads();      // the partial sums take the rows' place
  float* red = reinterpret_cast<float*>(smem);
  static_for<0, 2>([&](auto tt) {
    constexpr int t = decltype(tt)::value;
    static_for<0, JT>([&](auto jj) {
      constexpr int u = decltype(jj)::value;
      *reinterpret_cast<floatx4*>(red + (wave * 16 * JT + 16 * u + i16) * kRedRow + 8 * q4 + 4 * t) = acc[t][u];
    });
  });
  __syncthreads();
  const int j = tid >> 3, i4 = 4 * (tid & 7);
  if (j >= 16 * JT || j0 + j >= N || i0 + i4 >= M) return;
  floatx4 v = {0.f, 0.f, 0.f, 0.f};
  static_for<0, 8>([&](auto ww) { v += *reinterpret_cast<const floatx4*>(red + (decltype(ww)::value * 16 * JT + j) * kRedRow + i4); });
  u32x2 pk = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
  *reinterpret_cast<u32x2*>(out + (long)(j0 + j) * ldo + i0 + i4) = pk;
}

template <int PER, int JT>
static int launch_ln_gemm(const void* s, const float* gamma, const float* beta, float eps, const void* w, void* out, long ldo, float* out_t,
                          int M, int N, hipStream_t st) {
  using S = LnGemmShape<PER, JT>;
  auto kern = ln_gemm_kernel<PER, JT>;
  if (S::kLds > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, S::kLds);
    if (e != hipSuccess) return set_error(M2_ERR_LAUNCH, "hipFuncSetAttribute(ln_gemm): %s", hipGetErrorString(e));
  }
  const int ti = (M + 31) / 32, tj = (N + 16 * JT - 1) / (16 * JT), nt = ti * tj;
  hipLaunchKernelGGL(kern, dim3(8 * ((nt + 7) / 8)), dim3(512), S::kLds, st, (const uint16_t*)s, gamma, beta, eps, (const uint16_t*)w,
                     (uint16_t*)out, ldo, out_t, M, N, ti, tj);
  return check_launch("ln_gemm");
}

template <int BI, int BJ, int WI, int WJ, int STAGES, bool QKM, int OCC>
static int launch_engine(GemmArgs g, hipStream_t st) {
  using S = GemmShape<BI, BJ, WI, WJ, STAGES, QKM>;
  auto kern = gemm_kernel<BI, BJ, WI, WJ, STAGES, QKM, OCC>;
  hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, S::kLds);
  if (e != hipSuccess) return set_error(M2_ERR_LAUNCH, "hipFuncSetAttribute(gemm): %s", hipGetErrorString(e));
  g.ti = g.nblk * ((g.ni + BI - 1) / BI);
  g.tj = (g.nj + BJ - 1) / BJ;
  const int nt = g.ti * g.tj;
  const int per_xcd = num_cus() / 8 * (160 * 1024 / S::kLds > 2 ? 2 : 160 * 1024 / S::kLds);
  const int need = (nt + 7) / 8;
  hipLaunchKernelGGL(kern, dim3(8 * (need < per_xcd ? need : per_xcd)), dim3(S::kThreads), S::kLds, st, g);
  return check_launch("gemm");
}

// ---------------------------------------------------------------------------------------------
// Which kernel for which size.  A tile step (64 of K) of a workgroup takes a time that depends on its tile and on whether
// the compute unit holds a second workgroup; a launch takes about 2.5 us.  Measured on MI355X (us per step, one / two
// workgroups per compute unit; K = 768 and 1536, M = 128 .. 32768): the table below.  What bounds a step: the small
// tiles their loads (a compute unit gets 50 - 65 GB/s out of L2) and the latency of a step, the two large ones the power
// budget (the clock falls to 1.6 - 1.8 GHz under them).  At 4 widths x 9 row counts the model picks the measured best or
// one within about 10 % of it.
// ---------------------------------------------------------------------------------------------
enum DenseVariant { kVarSmall, kVar64, kVar128, kVarMid, kVarWide, kVar256, kVariants };
struct VariantShape {
  int bi, bj, per_cu;       // tile (QKM: i and j exchanged where they differ), workgroups of a compute unit
  float t1, t2;             // us per step with one and with per_cu workgroups on it
};
static const VariantShape kVariantShapes[kVariants] = {
    {32, 32, 4, 0.f, 0.f},       {64, 128, 2, 0.52f, 0.86f},  {128, 128, 2, 0.80f, 1.14f},
    {128, 192, 2, 1.08f, 1.70f}, {256, 192, 1, 1.65f, 1.65f}, {256, 256, 1, 2.00f, 2.00f}};

static float variant_cost(int v, const GemmArgs& g, bool swap) {
  const VariantShape& s = kVariantShapes[v];
  const int bi = swap ? s.bj : s.bi, bj = swap ? s.bi : s.bj;
  const long tiles = (long)g.nblk * ((g.ni + bi - 1) / bi) * ((g.nj + bj - 1) / bj);
  // few rows: the launch, one memory latency, and 64 operand rows per tile at about 13 TB/s
  if (v == kVarSmall) return g.nk > 2048 ? 1e30f : 4.0f + 128e-6f * (float)tiles * (float)g.nk / 13.f;
  const long cus = num_cus(), slots = cus * s.per_cu;
  const long full = tiles / slots, rest = tiles - full * slots;
  return 2.5f + (float)(g.nk / kGK) * ((float)full * s.t2 + (rest == 0 ? 0.f : rest <= cus ? s.t1 : s.t2));
}
// swap: the long side of the tiles along i instead of j
static int pick_variant(const GemmArgs& g, bool swap) {
  int best = kVarSmall;
  float cost = 1e30f;
  for (int v = 0; v < kVariants; ++v) {
    if (v != kVarSmall && g.nk % kGK != 0) continue;
    const float c = variant_cost(v, g, swap);
    if (c < cost) { cost = c; best = v; }
  }
  return best;
}

template <bool QKM>
static int dense_launch(int variant, GemmArgs g, hipStream_t st) {
  switch (variant) {
    case kVarSmall: {
      // the tiles of an XCD keep the larger operand's rows together: weights are read by one L2 only
      g.jfast = QKM;
      const int ks = ((g.nk + 31) / 32 + 7) / 8;
      if (ks <= 3) return launch_small<8, 3, QKM, false>(g, st);
      if (ks <= 4) return launch_small<8, 4, QKM, false>(g, st);
      if (ks <= 6) return launch_small<8, 6, QKM, false>(g, st);
      return launch_small<8, 8, QKM, false>(g, st);
    }
    case kVar64: return QKM ? launch_engine<128, 64, 2, 2, 3, QKM, 2>(g, st) : launch_engine<64, 128, 2, 2, 3, QKM, 2>(g, st);
    case kVar128: return launch_engine<128, 128, 2, 2, 2, QKM, 2>(g, st);
    case kVarMid: return QKM ? launch_engine<192, 128, 2, 2, 2, QKM, 2>(g, st) : launch_engine<128, 192, 2, 2, 2, QKM, 2>(g, st);
    case kVarWide: return QKM ? launch_engine<192, 256, 2, 4, 2, QKM, 2>(g, st) : launch_engine<256, 192, 4, 2, 2, QKM, 2>(g, st);
    default: return launch_engine<256, 256, 2, 4, 2, QKM, 2>(g, st);
  }
}

// ---- block-diagonal products (declared in m2_internal.h) ----
// weights along i (P), rows of x along j (Q)
static GemmArgs blockdiag_args(const void* x, const void* w, const float* bias, const void* resid, void* out, int M, int nb,
                               int p, int q) {
  return GemmArgs{(const uint16_t*)w, (const uint16_t*)x, (uint16_t*)out, bias, (const uint16_t*)resid, p, (long)nb * p,
                  (long)nb * q, q, M, p, nb, (long)q * p, 0, 0, 0};
}
template <int NW>
static int launch_small_glu(const GemmArgs& g, hipStream_t st) {
  const int ks = ((g.nk + 31) / 32 + NW - 1) / NW;
  if (ks <= 2) return launch_small<NW, 2, false, true>(g, st);
  if (ks <= 3) return launch_small<NW, 3, false, true>(g, st);
  return launch_small<NW, 4, false, true>(g, st);
}
// The gated product + GLU for few rows.  us per call at M = 128 / 256, this against the next best: d = 768 5.5 / 7.0 (the
// weight-stationary kernel 10.1 / 10.4), d = 960 5.2 / 7.7 (the streaming kernel 8.2 / 8.4), d = 1536 10.5 / 19.6
// (12.7 / 13.3): every 32 x 32 tile reads its operands again, so it ends where M times the width passes about 250 thousand.
bool glu_few_rows_pays(int M, int nb, int p) { return (long)M * nb * p <= 245760 && p <= 512; }
int glu_few_rows(const void* x, const void* w, void* out, int M, int nb, int p, int q, hipStream_t st) {
  GemmArgs g = blockdiag_args(x, w, nullptr, nullptr, out, M, nb, p, q);
  g.nblk = nb / 2;
  g.ldo = (long)nb / 2 * q;
  g.jfast = 1;
  return launch_small_glu<4>(g, st);
}
// wo + bias + residual in bf16, p % 64 == 0 and q % 8 == 0.  us per call, this against the LDS-tiled kernels it took over
// from: d = 768 M = 128 5.3 / 13.2, 1024 8.8 / 15.5; d = 1536 M = 512 14 / 22, 1024 15 / 23, 2048 20 / 24, 4096 29 / 33,
// 8192 44 / 48; d = 1792 M = 128 9 / 26, 1024 18 / 31, 4096 36 / 42, 8192 60 / 81; d = 960 (240-wide blocks) M = 128
// 6 / 17, 1024 10 / 17, 8192 23 / 27, 32768 107 / 117.
int blockdiag_linear_engine(const void* x, const void* w, const float* bias, const void* resid, void* out, int M, int nb, int p,
                            int q, hipStream_t st) {
  GemmArgs g = blockdiag_args(x, w, bias, resid, out, M, nb, p, q);
  switch (pick_variant(g, true)) {
    case kVarSmall: {
      g.jfast = 1;
      const int ks = ((p + 31) / 32 + 7) / 8;
      if (ks <= 3) return launch_small<8, 3, false, false>(g, st);
      if (ks <= 4) return launch_small<8, 4, false, false>(g, st);
      if (ks <= 6) return launch_small<8, 6, false, false>(g, st);
      return launch_small<8, 8, false, false>(g, st);
    }
    case kVar64: return launch_engine<128, 64, 2, 2, 3, false, 2>(g, st);
    case kVar128: return launch_engine<128, 128, 2, 2, 2, false, 2>(g, st);
    case kVarMid: return launch_engine<192, 128, 2, 2, 2, false, 2>(g, st);
    case kVarWide: return launch_engine<192, 256, 2, 4, 2, false, 2>(g, st);
    default: return launch_engine<256, 256, 2, 4, 2, false, 2>(g, st);
  }
}

static int check_dense(const char* who, const void* x, const void* w, const void* out, int M, int N, int K) {
  if (!x || !w || !out) return set_error(M2_ERR_ARG, "%s: null pointer", who);
  if (M <= 0 || N <= 0 || K <= 0) return set_error(M2_ERR_ARG, "%s: sizes must be positive (M=%d N=%d K=%d)", who, M, N, K);
  if (!m2_dense_supported(M, N, K))
    return set_error(M2_ERR_UNSUPPORTED, "%s: needs M and N multiples of 8, K a multiple of 64 and operands below 4 GB (M=%d N=%d K=%d)", who, M, N, K);
  if (!aligned16(x, w, out)) return set_error(M2_ERR_UNSUPPORTED, "%s: operands must be 16-byte aligned", who);
  return M2_OK;
}

}  // namespace m2

using namespace m2;

extern "C" int m2_blockdiag_glu_few_rows(int M, int in_features, int nblocks) {
  if (M <= 0 || nblocks <= 0 || in_features <= 0 || in_features % nblocks) return 0;
  return glu_few_rows_pays(M, nblocks, in_features / nblocks) ? 1 : 0;
}

extern "C" int m2_dense_supported(int M, int N, int K) {
  if (M < 8 || N < 8 || K < 64 || M % 8 || N % 8 || K % 64) return 0;
  // the direct loads of the tile engine take 32-bit byte offsets
  return ((long)M * K * 2 < (1l << 32) && (long)N * K * 2 < (1l << 32)) ? 1 : 0;
}

static int dense_to_channels(const char* who, const void* x, const void* w, void* out, int M, int N, int K, long ldo, void* stream) {
  const int rc = check_dense(who, x, w, out, M, N, K);
  if (rc) return rc;
  if (ldo < M || ldo % 8) return set_error(M2_ERR_ARG, "%s: rows of the output %ld apart, need a multiple of 8 from M = %d on", who, ldo, M);
  if (dense_ws_serves(M, N, K)) return dense_ws_launch(x, w, out, M, N, ldo, (hipStream_t)stream);
  GemmArgs g{(const uint16_t*)x, (const uint16_t*)w, (uint16_t*)out, nullptr, nullptr, K, K, ldo, M, N, K, 1, 0, 0, 0, 1};
  return dense_launch<false>(pick_variant(g, false), g, (hipStream_t)stream);
}

extern "C" int m2_dense_to_channels_fwd(const void* x, const void* w, void* out, int M, int N, int K, void* stream) {
  return dense_to_channels("m2_dense_to_channels_fwd", x, w, out, M, N, K, M, stream);
}

extern "C" int m2_dense_to_channels_rows_fwd(const void* x, const void* w, void* out, long out_row, int M, int N, int K, void* stream) {
  return dense_to_channels("m2_dense_to_channels_rows_fwd", x, w, out, M, N, K, out_row, stream);
}

// Rows a multiple of 16 KB apart put everything that the weight-stationary kernel stores at a time into one or few of an XCD's 16 L2
// channels; a line more between them spreads it.  us without / with: M = 32768 130 / 96, 24576 90 / 78, 16384 50.1 / 48.8, 8192 30.4 / 29.8;
// other strides gain nothing (31744 93 / 95, 28672 87 / 87, 20480 60 / 59).
extern "C" long m2_dense_channels_row(int M, int N, int K) {
  return dense_ws_serves(M, N, K) && M % 8192 == 0 ? M + 64l : (long)M;
}

extern "C" int m2_dense_from_channels_fwd(const void* x, const void* w, const float* bias, void* out, int M, int N, int K,
                                          void* stream) {
  const int rc = check_dense("m2_dense_from_channels_fwd", x, w, out, M, N, K);
  if (rc) return rc;
  GemmArgs g{(const uint16_t*)w, (const uint16_t*)x, (uint16_t*)out, bias, nullptr, K, M, N, N, M, K, 1, 0, 0, 0, 0};
  return dense_launch<true>(pick_variant(g, true), g, (hipStream_t)stream);
}

// LayerNorm and in_linear as one kernel where in_linear alone would be the kernel of few rows: every tile normalises its rows again, which
// hides behind the launch it saves only there (up to 256 or 384 rows; figures above).
extern "C" int m2_layernorm_to_channels_supported(int M, int N, int K) {
  if (!m2_dense_supported(M, N, K) || N != 3 * K || (K != 768 && K != 960 && K != 1536 && K != 1792) || dense_ws_serves(M, N, K)) return 0;
  const GemmArgs g{nullptr, nullptr, nullptr, nullptr, nullptr, K, K, M, M, N, K, 1, 0, 0, 0, 1};
  return pick_variant(g, false) == kVarSmall ? 1 : 0;
}

extern "C" int m2_layernorm_to_channels_fwd(const void* s, const float* gamma, const float* beta, float eps, const void* w, void* out, long out_row,
                                            float* out_channel_major, int M, int N, int K, void* stream) {
  const char* who = "m2_layernorm_to_channels_fwd";
  if (!gamma || !beta) return set_error(M2_ERR_ARG, "%s: null pointer", who);
  const int rc = check_dense(who, s, w, out, M, N, K);
  if (rc) return rc;
  if (out_row < M || out_row % 8) return set_error(M2_ERR_ARG, "%s: rows of the output %ld apart, need a multiple of 8 from M = %d on", who, out_row, M);
  if (N != 3 * K) return set_error(M2_ERR_UNSUPPORTED, "%s: N=%d must be 3 K=%d", who, N, 3 * K);
  if (!aligned16(gamma, beta, out_channel_major)) return set_error(M2_ERR_UNSUPPORTED, "%s: operands must be 16-byte aligned", who);
  // 16 JT output channels: the fullest compute unit has the fewest operand rows to fetch
  const long ti = (M + 31) / 32, cus = num_cus();
  auto fetched = [&](long jt) { return (ti * ((N + 16 * jt - 1) / (16 * jt)) + cus - 1) / cus * (32 + 16 * jt); };
  const bool three = fetched(3) < fetched(2);
  hipStream_t st = (hipStream_t)stream;
  switch (K) {
#define X(PER)                                                                                                                          \
  case 64 * PER: return three ? launch_ln_gemm<PER, 3>(s, gamma, beta, eps, w, out, out_row, out_channel_major, M, N, st)               \
                              : launch_ln_gemm<PER, 2>(s, gamma, beta, eps, w, out, out_row, out_channel_major, M, N, st);
    X(12) X(15) X(24) X(28)
#undef X
  }
  return set_error(M2_ERR_UNSUPPORTED, "%s: K=%d, built for 768, 960, 1536 and 1792", who, K);
}
