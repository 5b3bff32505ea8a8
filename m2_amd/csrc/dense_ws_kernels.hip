// Dense bf16 product with its weights held in registers:  OUT[n][m] = sum_k W[n][k] X[m][k], fp32 accumulation
// (in_linear of the 768-wide models, channel-major output).
//
// A workgroup of four waves, one per SIMD with the whole register file, owns 64 TJ output channels: a wave keeps 16 TJ rows of W, all
// K of them, in registers (384 at K = 768, TJ = 4), and the rows of X stream past, 32 at a time (a slab), through a ring of three LDS
// stages filled by direct loads two slabs ahead, one barrier per slab.  Against tiles that fetch both operands for every product this
// halves what comes out of L2 per operation (48 KB for 12.6 MFLOP where a 256 x 256 tile step takes 64 KB for 8.4) and what the waves
// read from LDS, which is what the power budget goes to: with stores left out the loop runs at 1.5 PFLOP/s, the rate this chip holds for
// matrix instructions alone at these sizes.  The results of a slab leave during the first products of the next one.
//
// us, this / tile engine / library, d = 768 (N = 2304): M = 512 8.6 / 9.4 / 9.1, 2048 14.9 / 15.5 / 16.0, 4096 20 / 24 / 27,
// 8192 30 / 37 / 47, 16384 50 / 64 / 62, 31744 93 / 139 / 124; 32768 130 / 163 / 130 where the rows of OUT are 64 KB apart (all rows of
// a slab's results then sit in one L2 channel) and 96 with 128 bytes between them.  Of the 93 us, 7 are the weights' way into the
// registers and the launch and 15 the stores (80 without them).  Measured and not kept: two slabs' results leaving together as whole
// 128-byte lines, kept in LDS until then (101 us), the workgroups of a row range starting at different slabs (98 to 108; at M = 32768
// 115 without the gap between rows), weights fetched straight into operand layout (64-byte pieces: 14.8 us instead of 7.4 before the
// first product).
#include "gemm_engine.h"

namespace m2 {

struct WsArgs {
  const uint16_t* x;     // (M, K)
  const uint16_t* w;     // (N, K)
  uint16_t* out;         // (N, M), rows ldo apart
  long ldo;              // elements between two rows of out
  int M, groups, ranges; // groups of channels, ranges of rows: a workgroup takes one of each
};

template <bool ACC>
__device__ __forceinline__ void pin(u32x4& v) {
  if constexpr (ACC) asm volatile("" : "+a"(v)); else asm volatile("" : "+v"(v));
}
// One product of 16 x 16 x 32 with everything where it is held: the weight operand in the accumulation half (ACC) or the other half of
// the register file, the sums in the other half, in place.  Inline assembly because the compiler gives the sums of every product new
// registers in the accumulation half, which leaves too few for the weights.  It does not see these as matrix instructions, so the
// distances the hardware asks for are kept by the kernel: sums are read eight or more products after the last that wrote them, and no
// vector instruction writes an operand.
template <bool ACC, bool FIRST>
__device__ __forceinline__ void product(floatx4& c, const bf16x8& x, const u32x4& w) {
  if constexpr (FIRST) {
    if constexpr (ACC) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&v"(c) : "v"(x), "a"(w));
    else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&v"(c) : "v"(x), "v"(w));
  } else {
    if constexpr (ACC) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(x), "a"(w));
    else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(x), "v"(w));
  }
}
// nothing reads these sums ahead of this place
__device__ __forceinline__ void settle(floatx4& a, floatx4& b) { asm volatile("" : "+v"(a), "+v"(b)); }
// s_waitcnt immediate: vector-memory and LDS counters
constexpr int ws_vm(int n, int lgkm) { return 0x70 | (n & 15) | (n >> 4 << 14) | lgkm << 8; }

constexpr int kWsGrid = 256;      // 8 XCDs x 32 compute units, one workgroup each

template <int KS, int TJ, int STAGES>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void dense_ws_kernel(WsArgs g) {
  constexpr int K = 32 * KS, KG = (KS + 3) / 4, kSlab = KG * 8192, LD = 2 * KG, D = 3;
  static_assert(KS % D == 0 && KS % 4 == 0, "the operand ring closes over a slab; whole 256-byte pieces of a row");
  constexpr int kBar = KS - D + 1, kAcc = 64 / TJ;      // k steps whose weights sit in the accumulation registers
  static_assert(3 * TJ >= 8, "the products between the last of a sum (k step KS - 1) and its reading (behind those of tile 0 of k step 1)");
  static_assert(TJ + 1 < kBar, "results leave in k steps 1 .. TJ, the loads behind them and ahead of the barrier");
  static_assert((STAGES - 2) * LD + TJ < 64 && 2 * TJ < 64, "what the waits count");
  static_assert(8 * 16 * TJ * 128 <= kSlab + 16384, "the weights' way through LDS: the last stage and the room behind it");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, i16 = lane & 15, q4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // the workgroups that read the same rows of X sit on one XCD as far as they fit
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int per = kWsGrid / 8 / g.groups;        // whole row ranges of an XCD
  int range, grp;
  if (slot < per * g.groups) {
    range = xcd * per + slot / g.groups;
    grp = slot % g.groups;
  } else {
    const int l = (slot - per * g.groups) * 8 + xcd;
    range = 8 * per + l / g.groups;
    grp = l % g.groups;
  }
  if (range >= g.ranges) return;
  const int slabs = (g.M + 31) / 32;
  const int s0 = (int)((long)range * slabs / g.ranges), s1 = (int)((long)(range + 1) * slabs / g.ranges);
  if (s0 >= s1) return;
  const int n = s1 - s0;

  // ---- staging.  A stage is KG pieces of 128 K, each 32 rows of 256 bytes; the 16-byte piece c of row r sits in slot
  // c ^ (r % 4 + 4 (r / 8 % 4)), so that the sixteen rows an operand read takes lie in sixteen different bank groups.
  const unsigned lds0 = (unsigned)(uintptr_t)smem;
  const unsigned lpiece = 16 * ((lane & 15) ^ ((lane >> 4) | (wave << 2)));
  unsigned v0, v1;
  auto load_rows = [&](int slab) __attribute__((always_inline)) {
    int r = slab * 32 + 8 * wave + (lane >> 4);
    int r0 = r < g.M ? r : g.M - 1, r1 = r + 4 < g.M ? r + 4 : g.M - 1;
    v0 = (unsigned)r0 * (K * 2u) + lpiece;
    v1 = (unsigned)r1 * (K * 2u) + lpiece;
  };
  auto load_one = [&](unsigned stage, auto jj) __attribute__((always_inline)) {
    constexpr int j = decltype(jj)::value;
    load_to_lds(lds0 + stage + (j >> 1) * 8192 + (2 * wave + (j & 1)) * 1024, (j & 1) ? v1 : v0, (const unsigned char*)g.x + (j >> 1) * 256);
  };
  static_for<0, STAGES - 1>([&](auto ss) {
    constexpr int s = decltype(ss)::value;
    if (s < n) {
      load_rows(s0 + s);
      static_for<0, LD>([&](auto jj) { load_one(s * kSlab, jj); });
    }
  });

  // ---- weights: 64 K of the wave's rows at a time through its own part of LDS (the last stage and the hold buffer), two such
  // pieces in flight, so that global memory is read in whole lines
  const int n0 = (grp * 4 + wave) * (16 * TJ);
  u32x4 w[KS][TJ];
  {
    constexpr int kPiece = 16 * TJ * 128, WL = kPiece / 1024;
    const unsigned wbase = (STAGES - 1) * kSlab + wave * (2 * kPiece);
    const unsigned voff = (unsigned)(lane >> 3) * (K * 2u) + 16 * ((lane & 7) ^ (lane >> 3));
    const unsigned char* wp = (const unsigned char*)g.w + (long)n0 * K * 2;
    auto load_piece = [&](int piece, unsigned buf) __attribute__((always_inline)) {
      static_for<0, WL>([&](auto uu) {
        load_to_lds(lds0 + wbase + buf + decltype(uu)::value * 1024, voff, wp + decltype(uu)::value * 8 * K * 2 + piece * 128);
      });
    };
    load_piece(0, 0);
    load_piece(1, kPiece);
    const unsigned wa = wbase + i16 * 128;
    static_for<0, KS / 2>([&](auto pp) {
      constexpr int p = decltype(pp)::value;
      if constexpr (p + 1 < KS / 2) __builtin_amdgcn_s_waitcnt(ws_vm(WL, 15)); else __builtin_amdgcn_s_waitcnt(ws_vm(0, 15));
      asm volatile("" ::: "memory");
      static_for<0, 2 * TJ>([&](auto ii) {
        constexpr int h = decltype(ii)::value / TJ, j = decltype(ii)::value % TJ;
        w[2 * p + h][j] = *reinterpret_cast<const u32x4*>(smem + wa + (p & 1) * kPiece + j * 2048 + 16 * ((4 * h + q4) ^ (i16 & 7)));
      });
      static_for<0, 2 * TJ>([&](auto ii) {
        constexpr int h = decltype(ii)::value / TJ, j = decltype(ii)::value % TJ;
        pin<(2 * p + h < kAcc)>(w[2 * p + h][j]);
      });
      if constexpr (p + 2 < KS / 2) {
        __builtin_amdgcn_s_waitcnt(ws_vm(63, 0));
        asm volatile("" ::: "memory");
        load_piece(p + 2, (p & 1) * kPiece);
      }
    });
  }

  // ---- operand reads: matrix row i16 of tile t is row 8 (i16 / 4) + 4 t + i16 % 4 of the slab, so that a lane ends up with eight
  // consecutive rows of a channel
  const unsigned rrow = (8 * (i16 >> 2) + (i16 & 3)) * 256;
  unsigned ra[4];
  static_for<0, 4>([&](auto cc) { ra[decltype(cc)::value] = rrow + 16 * ((4 * decltype(cc)::value + q4) ^ i16); });
  auto read_x = [&](unsigned stage, auto kk, auto tt) __attribute__((always_inline)) -> bf16x8 {
    constexpr int ks = decltype(kk)::value, t = decltype(tt)::value;
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(smem + stage + ra[ks & 3] + (ks >> 2) * 8192 + t * 1024));
  };

  bf16x8 ring[D][2];
  floatx4 acc[2][2][TJ];
  __builtin_amdgcn_s_waitcnt(kWaitVm0);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  static_for<0, D>([&](auto dd) {
    static_for<0, 2>([&](auto tt) { ring[decltype(dd)::value][decltype(tt)::value] = read_x(0, dd, tt); });
  });

  uint16_t* op = g.out + (long)(n0 + i16) * g.ldo + 8 * q4;
  // the results of slab s leave: one 16-byte store per lane and channel tile, four lanes writing 64 bytes of a row
  auto leave = [&](auto par, auto jj, int s) __attribute__((always_inline)) {
    constexpr int p = decltype(par)::value, j = decltype(jj)::value;
    settle(acc[p][0][j], acc[p][1][j]);
    const floatx4 a = acc[p][0][j], b = acc[p][1][j];
    const u32x4 pk = {pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3]), pack_bf16x2(b[0], b[1]), pack_bf16x2(b[2], b[3])};
    const int m = (s0 + s) * 32;
    if (m + 8 * q4 < g.M) *reinterpret_cast<u32x4*>(op + 16 * j * g.ldo + m) = pk;
  };
  unsigned st = 0;
  int s = 0;
  auto body = [&](auto par) __attribute__((always_inline)) {
    constexpr int P = decltype(par)::value;
    unsigned stn = st == (STAGES - 1) * kSlab ? 0 : st + kSlab;
    unsigned stl = st == 0 ? (STAGES - 1) * kSlab : st - kSlab;      // the stage freed by the last barrier
    asm volatile("" : "+s"(st), "+s"(stn), "+s"(stl));
    const bool more = s + STAGES - 1 < n;
    if (more) load_rows(s0 + s + STAGES - 1);
    static_for<0, KS>([&](auto kk) {
      constexpr int ks = decltype(kk)::value;
      if constexpr (ks == kBar) {
        asm volatile("" ::: "memory");
        // every read of this stage is back and this wave's loads of the next slab have landed (behind them: the stores of the
        // previous slab, which is whole, and the loads of the slab after): the barrier frees this stage and completes the next
        if (more && s > 0) __builtin_amdgcn_s_waitcnt(ws_vm((STAGES - 2) * LD + TJ, 0));
        else if (more) __builtin_amdgcn_s_waitcnt(ws_vm((STAGES - 2) * LD, 0));
        else __builtin_amdgcn_s_waitcnt(ws_vm(0, 0));
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        static_for<0, 2>([&](auto tt) { ring[(ks - 1) % D][decltype(tt)::value] = read_x(stn, ic<0>{}, tt); });
      }
      static_for<0, 2>([&](auto tt) {
        constexpr int t = decltype(tt)::value;
        static_for<0, TJ>([&](auto jj) {
          constexpr int j = decltype(jj)::value;
          product<(ks < kAcc), ks == 0>(acc[P][t][j], ring[ks % D][t], w[ks][j]);
        });
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (ks + D < KS) ring[ks % D][t] = read_x(st, ic<ks + D>{}, tt);
        else if constexpr (ks >= kBar) ring[ks % D][t] = read_x(stn, ic<ks + D - KS>{}, tt);
        if constexpr (t == 0 && ks >= 1 && ks <= TJ) {
          if (s > 0) leave(ic<1 - P>{}, ic<(ks + TJ - 1) % TJ>{}, s - 1);
        }
        // direct loads of the slab STAGES - 1 ahead: behind those stores, all of them before the barrier
        constexpr int idx = 2 * (ks - TJ) - 1 + t, cnt = 2 * (kBar - TJ) - 2;
        constexpr int l0 = idx < 0 ? 0 : idx < cnt ? idx * LD / cnt : LD, l1 = idx + 1 < 0 ? 0 : idx + 1 < cnt ? (idx + 1) * LD / cnt : LD;
        if constexpr (l1 > l0) {
          if (more) static_for<l0, l1>([&](auto ll) { load_one(stl, ll); });
        }
        __builtin_amdgcn_sched_barrier(0);
      });
    });
    st = stn;
  };
  for (;;) {
    body(ic<0>{});
    if (++s == n) {
      asm volatile("s_nop 15\n\ts_nop 15");
      __builtin_amdgcn_sched_barrier(0);
      static_for<0, TJ>([&](auto jj) { leave(ic<0>{}, jj, n - 1); });
      break;
    }
    body(ic<1>{});
    if (++s == n) {
      asm volatile("s_nop 15\n\ts_nop 15");
      __builtin_amdgcn_sched_barrier(0);
      static_for<0, TJ>([&](auto jj) { leave(ic<1>{}, jj, n - 1); });
      break;
    }
  }
  __builtin_amdgcn_s_waitcnt(kWaitVm0);
}

// Fewer rows leave most row ranges empty: M = 128 takes 8.0 us here and 7.6 with K split over the waves (dense_kernels.hip).
bool dense_ws_serves(int M, int N, int K) { return K == 768 && N % 256 == 0 && N <= 256 * 256 && M >= 512 && M % 8 == 0; }

// sizes as above, operands 16-byte aligned and below 4 GB, ldo a multiple of 8 and at least M
int dense_ws_launch(const void* x, const void* w, void* out, int M, int N, long ldo, hipStream_t st) {
  constexpr int kStages = 3, kLds = kStages * 6 * 8192 + 16384;      // the ring, and room for the weights' way through LDS
  auto kern = dense_ws_kernel<24, 4, kStages>;
  hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
  if (e != hipSuccess) return set_error(M2_ERR_LAUNCH, "hipFuncSetAttribute(dense_ws): %s", hipGetErrorString(e));
  const int groups = N / 256;
  WsArgs g{(const uint16_t*)x, (const uint16_t*)w, (uint16_t*)out, ldo, M, groups, kWsGrid / groups};
  hipLaunchKernelGGL(kern, dim3(kWsGrid), dim3(256), kLds, st, g);
  return check_launch("dense_ws");
}

}  // namespace m2
