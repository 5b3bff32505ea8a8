// The tile engine of the dense and block-diagonal bf16 matrix products (dense_kernels.hip):
//
//   OUT[j][i] = sum_k P[i][k] Q[j][k]      i contiguous in OUT, fp32 accumulation
//
// P is stored with k contiguous (row stride ldp), Q either with k contiguous (row stride ldq) or, QKM = true,
// with j contiguous and k as the row index (a channel-major activation: row stride ldq between successive k); those
// operands are read from LDS with the transposing ds_read_b64_tr_b16.
//
// A persistent workgroup walks over its tiles in one flat stream of steps of 64 K: operand tiles go from global memory
// straight into LDS (no registers, XOR-swizzled by permuting which lane fetches which 16-byte piece of a 128-byte line),
// STAGES steps ahead and across tile boundaries; ONE barrier per step, placed where the last operand read of the step
// has had a block of MFMAs to come back: it frees the step's stage and completes the next one.  Operands run ahead of the
// MFMAs through registers and do not drain at the barrier.  The rows of P are permuted so that a lane ends up with eight
// consecutive i of an output row: results leave as 16-byte stores, four lanes of a row writing 64 contiguous bytes, without
// another pass through LDS, and the stores of a tile are not waited for until the step after next.
//
// What bounds it, found with parts removed (256 x 192 tiles, M = 8192, N = 4608, K = 1536: 118 us): without the direct loads
// 94 us, without the LDS reads 116, without barriers 121, without stores 118, MFMAs alone 75 us = 1.55 PFLOP/s -- and the
// clock the chip holds is 1.6 - 1.8 GHz throughout: at these sizes the power budget is spent, so what counts is energy,
// i.e. fewer bytes moved, not better overlap (dropping the waits for the loads changes nothing).  Small tiles are bound by
// the 50 - 65 GB/s a compute unit gets out of L2 and by the latency of a step, not by its depth (4 and 6 stages: no gain).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fft_regs.h"
#include "m2_internal.h"
#include "mfma_stream.h"

namespace m2 {

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));

struct GemmArgs {
  const uint16_t* p;
  const uint16_t* q;
  uint16_t* out;
  const float* bias;        // along i, or null
  const uint16_t* resid;    // as out, or null
  long ldp, ldq, ldo;       // elements
  int ni, nj, nk;           // sizes of the product of one block
  int nblk;                 // blocks of a block-diagonal product (1: dense)
  long pblk;                // elements from one block of P to the next; block b's columns of Q start at b nk, of OUT at b ni
  int ti, tj;               // tiles along i (all blocks) and j
  int jfast;                // order of the tiles of an XCD: neighbours differ in j (1) or in i (0)
};

// tile -> first i of the tile inside its block, first j, block
template <int BI, int BJ>
__device__ __forceinline__ void tile_origin(const GemmArgs& g, int tile, int& i0, int& j0, int& blk) {
  const int it = g.jfast ? tile / g.tj : tile % g.ti;
  j0 = (g.jfast ? tile % g.tj : tile / g.ti) * BJ;
  const int tib = g.ti / g.nblk;
  blk = it / tib;
  i0 = (it - blk * tib) * BI;
}

constexpr int kGK = 64;     // K of one step: one 128-byte line of a k-contiguous row

template <int BI, int BJ, int WI, int WJ, int STAGES, bool QKM>
struct GemmShape {
  static constexpr int kWaves = WI * WJ, kThreads = 64 * kWaves;
  static constexpr int TI = BI / WI / 16, TJ = BJ / WJ / 16;     // 16 x 16 tiles of a wave
  static constexpr int kPB = BI * kGK * 2, kQB = BJ * kGK * 2, kStage = kPB + kQB;
  static constexpr int kLds = STAGES * kStage;
  static constexpr int LP = kPB / 1024 / kWaves, LQ = kQB / 1024 / kWaves;     // direct loads of a wave and step
  static_assert(TI % 2 == 0, "a lane's results are pieces of eight i");
  static_assert(kPB % (1024 * kWaves) == 0 && kQB % (1024 * kWaves) == 0, "whole loads per wave");
};

// Swizzle of a k-contiguous tile: the 16-byte piece c (0 .. 7) of row r sits in slot c ^ key(r).  The key takes bit 3 of
// the row instead of bit 2 because the rows that eight neighbouring lanes of a P operand read are 0 - 3 and 8 - 11.
__device__ __forceinline__ int row_key_p(int r) { return (r & 3) | ((r >> 1) & 4); }
__device__ __forceinline__ int row_key_q(int r) { return r & 7; }

template <int BI, int BJ, int WI, int WJ, int STAGES, bool QKM, int OCC>
__global__ __launch_bounds__(64 * WI * WJ) __attribute__((amdgpu_waves_per_eu(OCC, OCC))) void gemm_kernel(GemmArgs g) {
  using S = GemmShape<BI, BJ, WI, WJ, STAGES, QKM>;
  constexpr int TI = S::TI, TJ = S::TJ, LP = S::LP, LQ = S::LQ, W = S::kWaves;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, i16 = lane & 15, q4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wi = wave / WJ, wj = wave % WJ;

  // tiles of this workgroup: XCD e (workgroup ids are dealt round-robin to the 8 XCDs) owns a contiguous run of tiles
  const int ntiles = g.ti * g.tj;
  const int xcd = blockIdx.x & 7;
  const int t_end = (int)((long)(xcd + 1) * ntiles / 8), t_step = gridDim.x >> 3;
  int tile = (int)((long)xcd * ntiles / 8) + (blockIdx.x >> 3);
  if (tile >= t_end) return;
  const int nsteps = g.nk / kGK;
  const int mytiles = (t_end - tile + t_step - 1) / t_step;
  const int total = mytiles * nsteps;

  // ---- staging
  const unsigned lds0 = (unsigned)(uintptr_t)smem;
  int ltile = tile, lstep = 0;                 // tile and step the next loads belong to
  unsigned vp[LP], vq[LQ];
  const unsigned char *bp, *bq;
  auto load_bases = [&]() __attribute__((always_inline)) {
    int i0, j0, blk;
    tile_origin<BI, BJ>(g, ltile, i0, j0, blk);
    bp = (const unsigned char*)(g.p + blk * g.pblk);
    bq = (const unsigned char*)(g.q + (QKM ? 0l : (long)blk * g.nk));
    static_for<0, LP>([&](auto jj) {
      constexpr int j = decltype(jj)::value;
      const int r = (wave + W * j) * 8 + (lane >> 3);
      int row = i0 + r;
      row = row < g.ni ? row : g.ni - 1;
      vp[j] = (unsigned)((long)row * g.ldp * 2) + 16 * ((lane & 7) ^ row_key_p(r));
    });
    static_for<0, LQ>([&](auto jj) {
      constexpr int j = decltype(jj)::value;
      if constexpr (!QKM) {
        const int r = (wave + W * j) * 8 + (lane >> 3);
        int row = j0 + r;
        row = row < g.nj ? row : g.nj - 1;
        vq[j] = (unsigned)((long)row * g.ldq * 2) + 16 * ((lane & 7) ^ row_key_q(r));
      } else {
        constexpr int SL = BJ / 8;             // 16-byte slots of a k row
        const int idx = (wave + W * j) * 64 + lane;
        const int k = idx / SL, s = (idx % SL) ^ (2 * (k & 3));
        int col = j0 + 8 * s;
        col = col <= g.nj - 8 ? col : g.nj - 8;
        vq[j] = (unsigned)((long)k * g.ldq * 2 + col * 2);
      }
    });
  };
  load_bases();
  auto load_one = [&](int stage, auto jj) __attribute__((always_inline)) {
    constexpr int j = decltype(jj)::value;
    if constexpr (j < LP) {
      load_to_lds(lds0 + stage * S::kStage + (wave + W * j) * 1024, vp[j], bp + lstep * 128);
    } else {
      const long adv = QKM ? (long)lstep * kGK * g.ldq * 2 : (long)lstep * 128;
      load_to_lds(lds0 + stage * S::kStage + S::kPB + (wave + W * (j - LP)) * 1024, vq[j - LP], bq + adv);
    }
  };
  auto advance = [&]() __attribute__((always_inline)) {
    if (++lstep == nsteps) {
      lstep = 0;
      ltile += t_step;
      if (ltile < t_end) load_bases();
    }
  };

  // ---- operand reads
  // P rows: MFMA row i16 of tile t is row 32 (t / 2) + 8 (i16 / 4) + 4 (t % 2) + i16 % 4 of the wave's range, so that
  // a lane's accumulators of two neighbouring tiles are eight consecutive i.
  const unsigned prow = wi * (BI / WI) + 8 * (i16 >> 2) + (i16 & 3);
  const unsigned pkey = (i16 & 3) | (((i16 >> 2) & 1) << 2);
  const unsigned pa0 = prow * 128 + 16 * (q4 ^ pkey);
  const unsigned pa1 = prow * 128 + 16 * ((4 + q4) ^ pkey);
  const unsigned qrow = wj * (BJ / WJ) + i16;
  const unsigned qa0 = S::kPB + qrow * 128 + 16 * (q4 ^ (i16 & 7));
  const unsigned qa1 = S::kPB + qrow * 128 + 16 * ((4 + q4) ^ (i16 & 7));
  // QKM: lane (group q4, i16) reads 8 bytes of k row 8 q4 + i16 / 4 (+ 4), columns 4 (i16 % 4) of a 16-column tile
  const unsigned qk_row = (8 * q4 + (i16 >> 2)) * (BJ * 2) + 8 * (i16 & 3);
  auto read_p = [&](unsigned st, auto kss, auto tt) __attribute__((always_inline)) -> bf16x8 {
    constexpr int ks = decltype(kss)::value, t = decltype(tt)::value;
    constexpr int off = (32 * (t >> 1) + 4 * (t & 1)) * 128;
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(smem + st + (ks ? pa1 : pa0) + off));
  };
  auto read_q = [&](unsigned st, auto kss, auto tt) __attribute__((always_inline)) -> bf16x8 {
    constexpr int ks = decltype(kss)::value, t = decltype(tt)::value;
    if constexpr (!QKM) {
      return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(smem + st + (ks ? qa1 : qa0) + t * 16 * 128));
    } else {
      // 32-byte granule of the tile's 16 columns, swizzled by k % 4 = i16 / 4 (both halves: k + 4 has the same key)
      const unsigned gran = (unsigned)((wj * (BJ / WJ) / 16 + t) ^ (i16 >> 2)) * 32;
      const unsigned a = st + S::kPB + ks * 32 * BJ * 2 + qk_row + gran;
      typedef __attribute__((address_space(3))) s16x4 lds4;
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)(uintptr_t)(lds0 + a));
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)(uintptr_t)(lds0 + a + 4 * BJ * 2));
      const s16x8 r = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      return __builtin_bit_cast(bf16x8, r);
    }
  };

  // H: the operand held over an inner row of MFMAs (the one with fewer tiles), S: the one streamed through a ring
  constexpr bool HQ = TJ <= TI;
  constexpr int NH = HQ ? TJ : TI, NS = HQ ? TI : TJ, DS = NS < 4 ? 2 : (2 * NS) % 4 == 0 ? 4 : 3;
  static_assert((2 * NS) % DS == 0, "the ring closes over a step");
  constexpr int NB = 2 * NS;                  // blocks of NH MFMAs per step
  // The barrier sits before this block.  The last operand read of the step goes out one block earlier, so that four or
  // more MFMAs run while it travels.
  constexpr int kBar = NB - DS + 1;
  bf16x8 hold[2][NH], ring[DS];
  auto read_h = [&](unsigned st, auto kss, auto tt) __attribute__((always_inline)) {
    if constexpr (HQ) return read_q(st, kss, tt); else return read_p(st, kss, tt);
  };
  auto read_s = [&](unsigned st, auto ff) __attribute__((always_inline)) {      // flat index 0 .. NB - 1
    constexpr int f = decltype(ff)::value;
    if constexpr (HQ) return read_p(st, ic<f / NS>{}, ic<f % NS>{}); else return read_q(st, ic<f / NS>{}, ic<f % NS>{});
  };
  floatx4 acc[TI][TJ];
  auto clear = [&]() __attribute__((always_inline)) {
    static_for<0, TI>([&](auto a) { static_for<0, TJ>([&](auto b) { acc[decltype(a)::value][decltype(b)::value] = floatx4{0.f, 0.f, 0.f, 0.f}; }); });
  };
  clear();

  // ---- prologue
  int issued = 0;
  for (int s = 0; s < STAGES; ++s)
    if (issued < total) {
      static_for<0, LP + LQ>([&](auto jj) { load_one(s, jj); });
      advance();
      ++issued;
    }
  __builtin_amdgcn_s_waitcnt(kWaitVm0);      // (once per workgroup)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  static_for<0, NH>([&](auto h) { hold[0][decltype(h)::value] = read_h(0, ic<0>{}, h); });
  static_for<0, DS>([&](auto f) { ring[decltype(f)::value] = read_s(0, f); });

  int stage = 0, step = 0, pend = 0;
  for (int n = 0; n < total; ++n) {
    unsigned st = stage * S::kStage;
    const int nstage = stage == STAGES - 1 ? 0 : stage + 1;
    unsigned stn = nstage * S::kStage;
    asm volatile("" : "+s"(st), "+s"(stn));
    const bool more_loads = issued < total;
    static_for<0, NB>([&](auto bb) {
      constexpr int b = decltype(bb)::value;
      constexpr int ks = b / NS, s = b % NS;
      if constexpr (b == kBar) {
        // every operand read of this step has been issued; once they are back and this wave's loads of the next step
        // have landed, the barrier frees this stage and completes the next one
        asm volatile("" ::: "memory");
        if (pend) { __builtin_amdgcn_s_waitcnt(0x0070 | (0xf & (TI / 2 * TJ)) | ((TI / 2 * TJ) >> 4 << 14)); pend = 0; }
        else if (STAGES > 2 && n + STAGES <= issued) __builtin_amdgcn_s_waitcnt(0x0070 | ((STAGES - 2) * (LP + LQ) & 0xf) | (((STAGES - 2) * (LP + LQ)) >> 4 << 14));
        else __builtin_amdgcn_s_waitcnt(0x0070);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        ring[(b - 1) % DS] = read_s(stn, ic<0>{});
      }
      static_for<0, NH>([&](auto hh) {
        constexpr int h = decltype(hh)::value;
        if constexpr (HQ) acc[s][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ring[b % DS], hold[ks][h], acc[s][h], 0, 0, 0);
        else acc[h][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hold[ks][h], ring[b % DS], acc[h][s], 0, 0, 0);
        // reads of the second K half's held operands, during the first blocks
        if constexpr (b < 2 && h < NH) {
          constexpr int idx = b * NH + h;
          if constexpr (idx % 2 == 0 && idx / 2 < NH) hold[1][idx / 2] = read_h(st, ic<1>{}, ic<idx / 2>{});
        }
        if constexpr (b >= kBar) {
          constexpr int idx = (b - kBar) * NH + h, cnt = (DS - 1) * NH;
          // held operands of the next step, one per two MFMAs, and the direct loads of step n + STAGES
          if constexpr (idx % 2 == 0 && idx / 2 < NH) hold[0][idx / 2] = read_h(stn, ic<0>{}, ic<idx / 2>{});
          constexpr int l0 = idx * (LP + LQ) / cnt, l1 = (idx + 1) * (LP + LQ) / cnt;
          if constexpr (l1 > l0) {
            if (more_loads) static_for<l0, l1>([&](auto jj) { load_one(stage, jj); });
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      if constexpr (b + DS < NB) ring[b % DS] = read_s(st, ic<b + DS>{});
      else if constexpr (b >= kBar) ring[b % DS] = read_s(stn, ic<b + DS - NB>{});
      __builtin_amdgcn_sched_barrier(0);
    });
    if (more_loads) { advance(); ++issued; }
    stage = nstage;
    if (++step == nsteps) {
      step = 0;
      // ---- the tile's results leave
      int i0, j0, blk;
      tile_origin<BI, BJ>(g, tile, i0, j0, blk);
      const bool full = i0 + BI <= g.ni && j0 + BJ <= g.nj;
      i0 += wi * (BI / WI) + 8 * q4;
      j0 += wj * (BJ / WJ) + i16;
      const long o0 = (long)j0 * g.ldo + blk * g.ni + i0;
      static_for<0, TI / 2>([&](auto pp) {
        constexpr int p = decltype(pp)::value;
        const bool iok = full || i0 + 32 * p < g.ni;
        float bv[8];
        static_for<0, 8>([&](auto e) { bv[decltype(e)::value] = 0.f; });
        if (g.bias && iok) static_for<0, 8>([&](auto e) { bv[decltype(e)::value] = g.bias[blk * g.ni + i0 + 32 * p + decltype(e)::value]; });
        u32x4 rr[TJ];
        if (g.resid)
          static_for<0, TJ>([&](auto tt) {
            constexpr int t = decltype(tt)::value;
            if (full || (iok && j0 + 16 * t < g.nj)) rr[t] = *reinterpret_cast<const u32x4*>(g.resid + o0 + (long)(16 * t) * g.ldo + 32 * p);
          });
        static_for<0, TJ>([&](auto tt) {
          constexpr int t = decltype(tt)::value;
          const floatx4 a = acc[2 * p][t], c = acc[2 * p + 1][t];
          float v[8];
          static_for<0, 4>([&](auto e) {
            v[decltype(e)::value] = a[decltype(e)::value] + bv[decltype(e)::value];
            v[decltype(e)::value + 4] = c[decltype(e)::value] + bv[decltype(e)::value + 4];
          });
          if (g.resid) {
            v[0] += __uint_as_float(rr[t].x << 16); v[1] += __uint_as_float(rr[t].x & 0xffff0000u);
            v[2] += __uint_as_float(rr[t].y << 16); v[3] += __uint_as_float(rr[t].y & 0xffff0000u);
            v[4] += __uint_as_float(rr[t].z << 16); v[5] += __uint_as_float(rr[t].z & 0xffff0000u);
            v[6] += __uint_as_float(rr[t].w << 16); v[7] += __uint_as_float(rr[t].w & 0xffff0000u);
          }
          u32x4 pk = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
          u32x4* dst = reinterpret_cast<u32x4*>(g.out + o0 + (long)(16 * t) * g.ldo + 32 * p);
          if (full) *dst = pk;
          else if (iok && j0 + 16 * t < g.nj) *dst = pk;
        });
      });
      pend = full ? 1 : 0;
      clear();
      tile += t_step;
    }
  }
  __builtin_amdgcn_s_waitcnt(kWaitVm0);      // no load may be in flight when the workgroup's LDS goes to the next one
}

}  // namespace m2
