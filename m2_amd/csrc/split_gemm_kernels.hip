// fp32 matrix products on the bf16 matrix cores: every fp32 operand as three bf16 parts (x = hi + mid + lo, 8 + 8 + 8 mantissa
// bits: exact down to |x| = 2^-110; bf16 ends at 2^-133, so smaller values lose low bits) and the six products down to 2^-24 relative (hi hi, hi mid, mid hi, mid mid, hi lo, lo hi), fp32
// accumulation.  The dense projections and the block-diagonal MLP of fp32 callers outside autocast.
//
// What bounds an fp32 product here is the matrix pipe: 157 TFLOP/s for fp32 operands, 2.5 PFLOP/s for bf16 ones, i.e. 415
// for six bf16 products, and the rounding errors are smaller (a chain of K / 32 additions instead of K / 4).
//
// Layout of split operands: per row and chunk of 32 k the three parts side by side, [row][chunk][part][32] bf16: a step of
// a tile reads 192 contiguous bytes of a row.  A block-diagonal operand has its blocks padded to whole chunks with zeros.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fft_regs.h"
#include "m2_internal.h"
#include "mfma_stream.h"

namespace m2 {

// x = h + m + l.  The rest after an infinite h is 0, and a finite x whose rounded h is infinite is truncated instead: finite
// inputs have finite parts, and the sum of the parts is the input wherever bf16 reaches 24 bits below it (|x| >= 2^-110).
__device__ __forceinline__ void split_parts(float x, float& h, float& m, float& l) {
  h = __uint_as_float(pack_bf16x2(x, 0.f) << 16);
  if (fabsf(h) == INFINITY) h = __uint_as_float(__float_as_uint(x) & 0xffff0000u);
  const float r = fabsf(h) == INFINITY ? 0.f : x - h;
  m = __uint_as_float(pack_bf16x2(r, 0.f) << 16);
  l = r - m;
}
// four consecutive k of a row -> their places in the three parts (dst: the first of them in part 0)
__device__ __forceinline__ void store_parts(uint16_t* dst, const float* v) {
  float h[4], m[4], l[4];
  static_for<0, 4>([&](auto e) { split_parts(v[decltype(e)::value], h[decltype(e)::value], m[decltype(e)::value], l[decltype(e)::value]); });
  *reinterpret_cast<u32x2*>(dst) = u32x2{pack_bf16x2(h[0], h[1]), pack_bf16x2(h[2], h[3])};
  *reinterpret_cast<u32x2*>(dst + 32) = u32x2{pack_bf16x2(m[0], m[1]), pack_bf16x2(m[2], m[3])};
  *reinterpret_cast<u32x2*>(dst + 64) = u32x2{pack_bf16x2(l[0], l[1]), pack_bf16x2(l[2], l[3])};
}

// ---- splitting passes: a workgroup takes 32 rows x 64 k of one block (memory-bound: 4 bytes read, 6 written per value).
// CM: the input is channel-major (K, M), nb = 1; else row-major (M, nb p), with a channel-major fp32 copy on request (nb = 1).
template <bool CM>
__device__ __forceinline__ void split_tile(const float* __restrict__ x, uint16_t* __restrict__ out, float* __restrict__ xt,
                                           int M, int nb, int p, int kx, int m0) {
  __shared__ float tile[64][33];
  const int t = threadIdx.x, pc = (p + 31) / 32, pairs = (pc + 1) / 2;
  const int blk = kx / pairs, k0 = (kx % pairs) * 64;
  const int r = t >> 3, kl = 4 * (t & 7), row = m0 + r;
  const int ck = t >> 2, cm = 8 * (t & 3);           // channel-major side: one k, eight rows
  if constexpr (CM) {
    static_for<0, 2>([&](auto hh) {
      constexpr int h = decltype(hh)::value;
      float4 v = {0.f, 0.f, 0.f, 0.f};
      if (k0 + ck < p && m0 + cm + 4 * h < M) v = *reinterpret_cast<const float4*>(x + (long)(k0 + ck) * M + m0 + cm + 4 * h);
      tile[ck][cm + 4 * h] = v.x; tile[ck][cm + 4 * h + 1] = v.y; tile[ck][cm + 4 * h + 2] = v.z; tile[ck][cm + 4 * h + 3] = v.w;
    });
    __syncthreads();
  }
  static_for<0, 2>([&](auto cc) {
    constexpr int c = decltype(cc)::value;
    const int k = k0 + 32 * c + kl;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    if constexpr (CM) {
      static_for<0, 4>([&](auto e) { v[decltype(e)::value] = tile[32 * c + kl + decltype(e)::value][r]; });
    } else if (row < M && k < p) {
      const float4 f = *reinterpret_cast<const float4*>(x + ((long)row * nb + blk) * p + k);
      v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
    }
    if (!CM && xt) static_for<0, 4>([&](auto e) { tile[32 * c + kl + decltype(e)::value][r] = v[decltype(e)::value]; });
    if (row < M && k0 + 32 * c < 32 * pc)
      store_parts(out + (((long)row * nb + blk) * pc + k0 / 32 + c) * 96 + kl, v);
  });
  if (!CM && xt) {
    __syncthreads();
    static_for<0, 2>([&](auto hh) {
      constexpr int h = decltype(hh)::value;
      const int m = cm + 4 * h;
      if (k0 + ck < p && m0 + m < M)
        *reinterpret_cast<float4*>(xt + (long)(k0 + ck) * M + m0 + m) = float4{tile[ck][m], tile[ck][m + 1], tile[ck][m + 2], tile[ck][m + 3]};
    });
  }
}

__global__ __launch_bounds__(256) void split_channels_kernel(const float* __restrict__ x, uint16_t* __restrict__ out, int M, int K) {
  split_tile<true>(x, out, nullptr, M, 1, K, blockIdx.x, blockIdx.y * 32);
}

// Up to four row-major operands in one launch: an activation and the weights it meets, which are split in every call (nothing
// derived from a weight outlives the call, so a weight may be changed in any way between two calls).  us with the 2.4 M values of one
// mixer's two projections at d = 768: 8.8 behind 128 rows, 10.1 behind 2048; a launch of their own would cost as much again in gaps.
struct SplitJob {
  const float* x;
  uint16_t* out;
  float* xt;
  int M, nb, p, gx;         // gx: pairs of chunks of a row
  unsigned first;           // of its workgroups
};
struct SplitJobs {
  SplitJob job[4];
};
__global__ __launch_bounds__(256) void split_rows_kernel(SplitJobs jobs, int n) {
  int j = 0;
  for (int i = 1; i < n; ++i)
    if (blockIdx.x >= jobs.job[i].first) j = i;
  const SplitJob& s = jobs.job[j];
  const unsigned b = blockIdx.x - s.first;
  split_tile<false>(s.x, s.out, s.xt, s.M, s.nb, s.p, (int)(b % (unsigned)s.gx), (int)(b / (unsigned)s.gx) * 32);
}

// a pointer that is the same in all lanes, kept in scalar registers
__device__ __forceinline__ const unsigned char* scalar_ptr(const unsigned char* p) {
  const uint64_t a = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)a), hi = __builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32));
  return (const unsigned char*)(((uint64_t)hi << 32) | lo);
}

// ---- the products:  OUT[j][i] = sum_k P[i][k] Q[j][k], i contiguous in OUT
struct SplitArgs {
  const uint16_t *p, *q;
  float* out;               // or null (gated product)
  uint16_t* parts;          // gated product: its result split
  const float *bias, *resid;
  long ldp, ldq, ldo;       // elements between rows of P, Q and OUT
  int ni, nj, nc;           // sizes of the product of one block; chunks of 32 k
  int nblk;                 // blocks; block b's P rows start at b ni, its chunks of Q at b nc, its columns of OUT at b ni
  int ti, tj, jfast;
};

constexpr int kRowBytes = 192;      // of an operand row in LDS: one chunk, three parts

// A workgroup computes one BI x BJ tile in steps of 32 k: operands straight from memory into one of two LDS stages, one barrier
// per step, placed where a third of the step's MFMAs is left to cover it and the first operand reads of the next step.  16-byte
// piece c of part s of row r lies in slot 4 s + (c ^ (r / 4 % 4)): sixteen rows 192 bytes apart would meet in a quarter of the
// banks otherwise.  GLU: gate block b and value block b + nblk one after the other, then gelu(gate) * value.
//
// us, against the fp32 GEMM library and the fp32-MFMA kernel this took over from (d = 768, M = 2048 / 16384): in-projection 42 / 278
// against 79 / 416, out-projection 23 / 94 against 30 / 142, gated product with GELU 45 / 351 against 112 / 837, wo 23 / 125
// against 54 / 303; 1.5 PFLOP/s of bf16 products at the largest.  Reading the first operands behind the barrier instead of ahead
// of the last products cost 6 %; a third stage gained nothing; 128 x 128 tiles take 1.3 us per step for 0.64 us of MFMAs (LDS
// reads: 18 per 48 MFMAs of a wave).  Relative error against fp64 (2-norm): 1.6e-7 (library 5.0e-7) at K = 768, 2.5e-7 (7.6e-7) at
// 1792; with one accumulator for all six products 4.3e-7, and at K = 192 more than the fp32-MFMA kernel's.
template <int BI, int BJ, int WI, int WJ, bool GLU>
__global__ __launch_bounds__(64 * WI * WJ, WI * WJ == 12 ? 3 : 2) void split_gemm_kernel(SplitArgs g) {
  constexpr int STAGES = 2, W = WI * WJ, TI = BI / WI / 16, TJ = BJ / WJ / 16, D = GLU ? 2 : 1;
  constexpr int LP = BI * 12 / 64 / W, LQ = BJ * 12 / 64 / W, kStage = (BI + BJ) * kRowBytes;
  static_assert(LP * 64 * W == BI * 12 && LQ * 64 * W == BJ * 12, "whole loads per wave");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, i16 = lane & 15, q4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wi = wave / WJ, wj = wave % WJ;
  const int ntiles = g.ti * g.tj, xcd = blockIdx.x & 7;
  const int tile = (int)((long)xcd * ntiles / 8) + (int)(blockIdx.x >> 3);
  if (tile >= (int)((long)(xcd + 1) * ntiles / 8)) return;
  const int it = g.jfast ? tile / g.tj : tile % g.ti, tib = g.ti / g.nblk, blk = it / tib;
  const int i0 = (it - blk * tib) * BI, j0 = (g.jfast ? tile % g.tj : tile / g.ti) * BJ;

  // ---- direct loads: byte offsets of this lane's pieces inside the block's operands
  unsigned vp[LP], vq[LQ];
  static_for<0, LP>([&](auto jj) {
    const int idx = (wave + W * decltype(jj)::value) * 64 + lane, r = idx / 12, s = idx % 12;
    const int row = i0 + r < g.ni ? i0 + r : g.ni - 1;
    vp[decltype(jj)::value] = (unsigned)((long)row * g.ldp * 2) + 16 * ((s & 12) + ((s ^ (r >> 2)) & 3));
  });
  static_for<0, LQ>([&](auto jj) {
    const int idx = (wave + W * decltype(jj)::value) * 64 + lane, r = idx / 12, s = idx % 12;
    const int row = j0 + r < g.nj ? j0 + r : g.nj - 1;
    vq[decltype(jj)::value] = (unsigned)((long)row * g.ldq * 2) + 16 * ((s & 12) + ((s ^ (r >> 2)) & 3));
  });
  const unsigned lds0 = (unsigned)(uintptr_t)smem;
  const int total = D * g.nc;
  auto load_step = [&](int n) __attribute__((always_inline)) {
    const int second = GLU && n >= g.nc, b = blk + second * g.nblk, c = n - second * g.nc;
    const unsigned st = lds0 + (n % STAGES) * kStage;
    const unsigned char* bp = scalar_ptr((const unsigned char*)(g.p + (long)b * g.ni * g.ldp) + c * kRowBytes);
    const unsigned char* bq = scalar_ptr((const unsigned char*)g.q + ((long)b * g.nc + c) * kRowBytes);
    static_for<0, LP>([&](auto jj) { load_to_lds(st + (wave + W * decltype(jj)::value) * 1024, vp[decltype(jj)::value], bp); });
    static_for<0, LQ>([&](auto jj) { load_to_lds(st + BI * kRowBytes + (wave + W * decltype(jj)::value) * 1024, vq[decltype(jj)::value], bq); });
  };

  // the five small products have accumulators of their own: one rounding of the large sum per 32 k instead of six
  floatx4 acc[D][TI][TJ], rest[TI][TJ];
  static_for<0, D * TI * TJ>([&](auto a) {
    constexpr int d = decltype(a)::value / (TI * TJ), t = decltype(a)::value / TJ % TI, u = decltype(a)::value % TJ;
    acc[d][t][u] = floatx4{0.f, 0.f, 0.f, 0.f};
    if constexpr (d == 0) rest[t][u] = floatx4{0.f, 0.f, 0.f, 0.f};
  });
  auto add_rest = [&](auto dd) __attribute__((always_inline)) {
    static_for<0, TI * TJ>([&](auto a) {
      constexpr int t = decltype(a)::value / TJ, u = decltype(a)::value % TJ;
      acc[decltype(dd)::value][t][u] += rest[t][u];
      rest[t][u] = floatx4{0.f, 0.f, 0.f, 0.f};
    });
  };
  const unsigned pa = (wi * (BI / WI) + i16) * kRowBytes + 16 * (q4 ^ (i16 >> 2));
  const unsigned qa = (BI + wj * (BJ / WJ) + i16) * kRowBytes + 16 * (q4 ^ (i16 >> 2));
  auto frag = [&](unsigned a) __attribute__((always_inline)) { return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(smem + a)); };
  bf16x8 pf[3][TI], qf[3][TJ];
  auto read_p = [&](unsigned st, auto ss) __attribute__((always_inline)) {
    constexpr int s = decltype(ss)::value;
    static_for<0, TI>([&](auto t) { pf[s][decltype(t)::value] = frag(st + pa + 64 * s + decltype(t)::value * 16 * kRowBytes); });
  };
  auto read_q = [&](unsigned st, auto ss) __attribute__((always_inline)) {
    constexpr int s = decltype(ss)::value;
    static_for<0, TJ>([&](auto t) { qf[s][decltype(t)::value] = frag(st + qa + 64 * s + decltype(t)::value * 16 * kRowBytes); });
  };
  auto step = [&](int n, auto dd) __attribute__((always_inline)) {
    auto product = [&](auto sp, auto sq) __attribute__((always_inline)) {
      constexpr int d = decltype(dd)::value;
      __builtin_amdgcn_sched_barrier(0);
      static_for<0, TI>([&](auto tt) {
        static_for<0, TJ>([&](auto uu) {
          constexpr int t = decltype(tt)::value, u = decltype(uu)::value;
          floatx4& a = decltype(sp)::value + decltype(sq)::value == 0 ? acc[d][t][u] : rest[t][u];
          a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf[decltype(sp)::value][t], qf[decltype(sq)::value][u], a, 0, 0, 0);
        });
      });
      __builtin_amdgcn_sched_barrier(0);
    };
    const unsigned st = (n % STAGES) * kStage, stn = ((n + 1) % STAGES) * kStage;
    const bool more = n + 1 < total;
    read_q(st, ic<1>{});
    read_p(st, ic<1>{});
    product(ic<0>{}, ic<0>{});
    read_q(st, ic<2>{});
    product(ic<0>{}, ic<1>{});
    read_p(st, ic<2>{});
    product(ic<0>{}, ic<2>{});
    product(ic<1>{}, ic<0>{});
    // All operands of this step are in registers and this wave's loads of the next step are back.  Behind the barrier that
    // holds for everybody: the stage is free for new loads, the next one complete.
    __builtin_amdgcn_s_waitcnt(0x0070);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (n + STAGES < total) load_step(n + STAGES);
    if (more) read_p(stn, ic<0>{});
    product(ic<2>{}, ic<0>{});
    if (more) read_q(stn, ic<0>{});
    product(ic<1>{}, ic<1>{});
  };
  for (int s = 0; s < STAGES; ++s)
    if (s < total) load_step(s);
  __builtin_amdgcn_s_waitcnt(kWaitVm0);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  read_p(0, ic<0>{});
  read_q(0, ic<0>{});
  for (int n = 0; n < g.nc; ++n) step(n, ic<0>{});
  add_rest(ic<0>{});
  if constexpr (GLU) {
    for (int n = g.nc; n < total; ++n) step(n, ic<1>{});
    add_rest(ic<1>{});
  }

  auto emit = [&](int i, int j, const float (&v)[D][4]) __attribute__((always_inline)) {
    const int col = blk * g.ni + i;
    if constexpr (GLU) {
      float r[4];
      static_for<0, 4>([&](auto e) {
        const float x = v[0][decltype(e)::value];
        r[decltype(e)::value] = x * 0.5f * (1.f + erff(x * 0.70710678118654752440f)) * v[1][decltype(e)::value];
      });
      store_parts(g.parts + (long)j * g.ldo + (col >> 5) * 96 + (col & 31), r);
    } else {
      const long o = (long)j * g.ldo + col;
      float4 r = {v[0][0], v[0][1], v[0][2], v[0][3]};
      if (g.bias) { r.x += g.bias[col]; r.y += g.bias[col + 1]; r.z += g.bias[col + 2]; r.w += g.bias[col + 3]; }
      if (g.resid) {
        const float4 a = *reinterpret_cast<const float4*>(g.resid + o);
        r.x += a.x; r.y += a.y; r.z += a.z; r.w += a.w;
      }
      *reinterpret_cast<float4*>(g.out + o) = r;
    }
  };
  const int il = i0 + wi * (BI / WI) + 4 * q4, jl = j0 + wj * (BJ / WJ) + i16;
  unsigned again = 0;                        // pieces of four results with one that is not finite
  static_for<0, TI>([&](auto tt) {
    static_for<0, TJ>([&](auto uu) {
      constexpr int t = decltype(tt)::value, u = decltype(uu)::value;
      if (il + 16 * t >= g.ni || jl + 16 * u >= g.nj) return;
      float v[D][4];
      bool finite = true;
      static_for<0, 4 * D>([&](auto e) {
        constexpr int d = decltype(e)::value / 4, k = decltype(e)::value % 4;
        v[d][k] = acc[d][t][u][k];
        finite = finite && fabsf(v[d][k]) < INFINITY;
      });
      if (!finite) again |= 1u << (t * TJ + u);
      emit(il + 16 * t, jl + 16 * u, v);
    });
  });
  // A sum that is not finite is formed again from whole values, in order: infinity times a part that happens to be zero, or
  // infinities of both signs among the parts, are none of the caller's.
  for (; again; again &= again - 1) {
    const int tu = __builtin_ctz(again), i = il + 16 * (tu / TJ), j = jl + 16 * (tu % TJ);
    float v[D][4];
    static_for<0, 4 * D>([&](auto e) {
      constexpr int d = decltype(e)::value / 4, k4 = decltype(e)::value % 4;
      const int b = blk + d * g.nblk;
      const uint16_t* pr = g.p + ((long)b * g.ni + i + k4) * g.ldp;
      const uint16_t* qr = g.q + (long)j * g.ldq + (long)b * g.nc * 96;
      float s = 0.f;
      for (int c = 0; c < g.nc && s == s; ++c)
        for (int k = 96 * c; k < 96 * c + 32; ++k)
          s = fmaf(bf16_to_f32(pr[k]) + bf16_to_f32(pr[k + 32]) + bf16_to_f32(pr[k + 64]),
                   bf16_to_f32(qr[k]) + bf16_to_f32(qr[k + 32]) + bf16_to_f32(qr[k + 64]), s);
      v[d][k4] = s;
    });
    emit(i, j, v);
  }
}

template <int BI, int BJ, int WI, int WJ, bool GLU>
static int launch_split(SplitArgs g, hipStream_t st) {
  auto kern = split_gemm_kernel<BI, BJ, WI, WJ, GLU>;
  constexpr int lds = 2 * (BI + BJ) * kRowBytes;
  hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return set_error(M2_ERR_LAUNCH, "hipFuncSetAttribute(split_gemm): %s", hipGetErrorString(e));
  g.ti = g.nblk * ((g.ni + BI - 1) / BI);
  g.tj = (g.nj + BJ - 1) / BJ;
  const long nt = (long)g.ti * g.tj;
  if (nt > (1l << 28)) return set_error(M2_ERR_UNSUPPORTED, "split_gemm: %ld tiles", nt);
  hipLaunchKernelGGL(kern, dim3((unsigned)(8 * ((nt + 7) / 8))), dim3(64 * WI * WJ), lds, st, g);
  return check_launch("split_gemm");
}

// Which tile.  A compute unit works through its tiles at a rate that hardly depends on how many share it, so a product takes
// ceil(tiles / units) x (us per step x steps), and the launch; us per step (32 k) by tile, measured (d = 768 ... 1792, M = 128 ...
// 16384): 64 x 64 0.43, 128 x 64 0.69 (1.0 in a first round, when workgroups share units although others are idle), 128 x 128
// 1.29, 192 x 128 either way round 1.65.  The large tiles have 1.6 times the rate per result (operand reads from LDS and L2), the
// small ones fill the last round.  The gated product's epilogue takes 0.42 us per 1024 results.
template <bool GLU>
static int split_launch(const SplitArgs& g, hipStream_t st) {
  if (!aligned16(g.p, g.q, g.parts)) return set_error(M2_ERR_UNSUPPORTED, "split_gemm: split operands must be 16-byte aligned");
  static const struct { int bi, bj; float first, step; } kTiles[5] = {
      {64, 64, 0.43f, 0.43f}, {128, 64, 1.0f, 0.69f}, {128, 128, 1.29f, 1.29f}, {192, 128, 1.65f, 1.65f}, {128, 192, 1.65f, 1.65f}};
  int best = 0;
  float cost = 1e30f;
  for (int v = 0; v < (GLU ? 3 : 5); ++v) {      // (twelve waves have no registers for two sums)
    const long tiles = (long)g.nblk * ((g.ni + kTiles[v].bi - 1) / kTiles[v].bi) * ((g.nj + kTiles[v].bj - 1) / kTiles[v].bj);
    const long rounds = (tiles + num_cus() - 1) / num_cus();
    const float c = (float)rounds * ((GLU ? 2 : 1) * g.nc * (rounds == 1 ? kTiles[v].first : kTiles[v].step) +
                                     (GLU ? 0.42f / 1024 * kTiles[v].bi * kTiles[v].bj : 0.f));
    if (c < cost) { cost = c; best = v; }
  }
  switch (best) {
    case 0: return launch_split<64, 64, 2, 2, GLU>(g, st);
    case 1: return launch_split<128, 64, 2, 2, GLU>(g, st);
    case 2: return launch_split<128, 128, 4, 2, GLU>(g, st);
    default: break;
  }
  if constexpr (!GLU) {
    if (best == 3) return launch_split<192, 128, 3, 4, false>(g, st);
    return launch_split<128, 192, 4, 3, false>(g, st);
  }
  return set_error(M2_ERR_UNSUPPORTED, "split_gemm: no tile");
}

static bool split_ok(long rows, int nb, int p) {
  const long row = (long)nb * ((p + 31) / 32) * kRowBytes;
  return rows > 0 && nb > 0 && p > 0 && p % 4 == 0 && row < (1l << 31) && rows * row < (1l << 32);
}

}  // namespace m2

using namespace m2;

extern "C" size_t m2_split_bytes(int rows, int nblocks, int p) {
  return split_ok(rows, nblocks, p) ? (size_t)rows * nblocks * ((p + 31) / 32) * kRowBytes : 0;
}

extern "C" int m2_split_jobs_fwd(const m2_split_job* jobs, int njobs, void* stream) {
  const char* who = "m2_split_jobs_fwd";
  if (!jobs) return set_error(M2_ERR_ARG, "%s: null pointer", who);
  if (njobs < 1 || njobs > 4) return set_error(M2_ERR_ARG, "%s: takes one to four operands, got %d", who, njobs);
  SplitJobs sj;
  long groups = 0;
  for (int i = 0; i < njobs; ++i) {
    const m2_split_job& j = jobs[i];
    if (!j.x || !j.out) return set_error(M2_ERR_ARG, "%s: null pointer", who);
    if (!aligned16(j.out)) return set_error(M2_ERR_UNSUPPORTED, "%s: split operands must be 16-byte aligned", who);
    if (!split_ok(j.rows, j.nblocks, j.p)) return set_error(M2_ERR_UNSUPPORTED, "%s: needs p a multiple of 4 and operands below 4 GB (M=%d nb=%d p=%d)", who, j.rows, j.nblocks, j.p);
    if (j.channel_major && (j.nblocks != 1 || j.rows % 4)) return set_error(M2_ERR_UNSUPPORTED, "%s: a channel-major copy needs one block and M a multiple of 4 (M=%d nb=%d)", who, j.rows, j.nblocks);
    const int gx = j.nblocks * (((j.p + 31) / 32 + 1) / 2);
    sj.job[i] = SplitJob{j.x, (uint16_t*)j.out, j.channel_major, j.rows, j.nblocks, j.p, gx, (unsigned)groups};
    groups += (long)gx * ((j.rows + 31l) / 32);
  }
  for (int i = njobs; i < 4; ++i) sj.job[i] = sj.job[0];
  // (operands below 4 GB have fewer than 2^25 rows of 192 bytes, hence fewer than 2^21 groups each)
  hipLaunchKernelGGL(split_rows_kernel, dim3((unsigned)groups), dim3(256), 0, (hipStream_t)stream, sj, njobs);
  return check_launch("split_rows");
}

extern "C" int m2_split_rows_fwd(const float* x, void* out, float* channel_major, int M, int nblocks, int p, void* stream) {
  const m2_split_job job{x, out, channel_major, M, nblocks, p};
  return m2_split_jobs_fwd(&job, 1, stream);
}

extern "C" int m2_split_channels_fwd(const float* x, void* out, int M, int K, void* stream) {
  const char* who = "m2_split_channels_fwd";
  if (!x || !out) return set_error(M2_ERR_ARG, "%s: null pointer", who);
  if (!split_ok(M, 1, K) || M % 4 || M > 65535 * 32)
    return set_error(M2_ERR_UNSUPPORTED, "%s: needs M up to 2097120 and K multiples of 4 and operands below 4 GB (M=%d K=%d)", who, M, K);
  if (!aligned16(out)) return set_error(M2_ERR_UNSUPPORTED, "%s: split operands must be 16-byte aligned", who);
  const int pc = (K + 31) / 32;
  hipLaunchKernelGGL(split_channels_kernel, dim3((pc + 1) / 2, (M + 31) / 32), dim3(256), 0, (hipStream_t)stream, x, (uint16_t*)out, M, K);
  return check_launch("split_channels");
}

extern "C" int m2_split_to_channels_fwd(const void* xs, const void* ws, float* out, int M, int N, int K, void* stream) {
  const char* who = "m2_split_to_channels_fwd";
  if (!xs || !ws || !out) return set_error(M2_ERR_ARG, "%s: null pointer", who);
  if (M % 4 || !split_ok(M, 1, K) || !split_ok(N, 1, K))
    return set_error(M2_ERR_UNSUPPORTED, "%s: needs M and K multiples of 4 and operands below 4 GB (M=%d N=%d K=%d)", who, M, N, K);
  const int nc = (K + 31) / 32;
  SplitArgs g{(const uint16_t*)xs, (const uint16_t*)ws, out, nullptr, nullptr, nullptr, nc * 96l, nc * 96l, M, M, N, nc, 1, 0, 0, 1};
  return split_launch<false>(g, (hipStream_t)stream);
}

extern "C" int m2_split_linear_fwd(const void* xs, const void* ws, const float* bias, const float* residual, float* out, int M,
                                   int nblocks, int p, int q, void* stream) {
  const char* who = "m2_split_linear_fwd";
  if (!xs || !ws || !out) return set_error(M2_ERR_ARG, "%s: null pointer", who);
  if (q <= 0 || q % 4 || !split_ok(M, nblocks, p) || !split_ok((long)nblocks * q, 1, p))
    return set_error(M2_ERR_UNSUPPORTED, "%s: needs p and q multiples of 4 and operands below 4 GB (M=%d nb=%d p=%d q=%d)", who, M, nblocks, p, q);
  const int nc = (p + 31) / 32;
  SplitArgs g{(const uint16_t*)ws, (const uint16_t*)xs, out, nullptr, bias, residual, nc * 96l, (long)nblocks * nc * 96, (long)nblocks * q, q, M, nc, nblocks, 0, 0, 1};
  return split_launch<false>(g, (hipStream_t)stream);
}

extern "C" int m2_split_glu_fwd(const void* xs, const void* ws, void* out, int M, int nblocks, int p, int q, void* stream) {
  const char* who = "m2_split_glu_fwd";
  if (!xs || !ws || !out) return set_error(M2_ERR_ARG, "%s: null pointer", who);
  if (nblocks % 2 || q <= 0 || q % 64 || !split_ok(M, nblocks, p) || !split_ok((long)nblocks * q, 1, p) || !split_ok(M, 1, nblocks / 2 * q))
    return set_error(M2_ERR_UNSUPPORTED, "%s: needs an even number of blocks, p a multiple of 4, q of 64 and operands below 4 GB (M=%d nb=%d p=%d q=%d)", who, M, nblocks, p, q);
  const int nc = (p + 31) / 32;
  SplitArgs g{(const uint16_t*)ws, (const uint16_t*)xs, nullptr, (uint16_t*)out, nullptr, nullptr, nc * 96l, (long)nblocks * nc * 96, nblocks / 2 * (long)q * 3, q, M, nc, nblocks / 2, 0, 0, 1};
  return split_launch<true>(g, (hipStream_t)stream);
}
