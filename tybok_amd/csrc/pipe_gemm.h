// The many-row GEMMs' common part: y[M, N] tiles of x[M, K] . W[N, K]^T on gfx950, four waves that multiply and four that
// only load.
//
// A block owns BM*32 rows x BN*32 columns and a range of k tiles (of 32).  Both operands go from memory to LDS without
// passing through registers (global_load_lds), a round (128 bytes of every row) at a time, into a ring of NS buffers,
// one barrier a round.  Loading waves of their own, because a wave that both loads and multiplies stands still at every
// load while the compute unit's memory pipe is busy, with its matrix instructions behind it: 16-bit operands, 128 x 128
// blocks, 455 ns a round in one wave, 390 in two, and the loads alone take 350 (32 KiB; 64 KiB of cached data reach a
// compute unit's LDS in 485 ns, reading them back takes 219 and does not slow that down, their 16 matrix instructions a
// SIMD 221).
//   * x rows land as whole 128-byte lines; the 16-byte chunks of a line are permuted by row on the way in (the lane
//     picks its global chunk, the LDS slot is fixed by the instruction), so that operand reads of 32 rows touch all banks;
//   * operands are read one step ahead of their use; the barrier stands in the middle of a round's last step;
//   * each XCD takes an eighth of the tiles in a row.
// The k tiles of an output are added in ascending order whatever the block's shape: the shape does not change the bits.
#pragma once
#include "tk_common.h"
#include "tk_kernels.h"

namespace pipe {

typedef int i32x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// 16 bytes per lane from memory (base + voff) to LDS: lane l's land at lds + 16 * l.  Written as assembly so that the
// compiler does not wait for every such load in front of the next LDS read; load_wait below waits for exactly those that
// are needed.  Always a scalar base and a 32-bit lane offset: with 64-bit lane addresses these loads and the matrix
// instructions of the same SIMD hold each other up (64 KiB a compute unit beside 16 matrix instructions a SIMD, which
// take 220 ns: 690 ns with 64-bit lane addresses, 480 with a scalar base, 485 without any matrix instructions).
__device__ __forceinline__ void dma16(unsigned voff, const void* base, unsigned lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(base), "s"(lds) : "memory", "m0");
}
// the same from an address per lane, for rows of x too far apart for a 32-bit offset
__device__ __forceinline__ void dma16_far(const void* p, unsigned lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(p), "s"(lds) : "memory", "m0");
}
// at most `rounds` (<= MAXR) rounds of I loads each are still on their way
template <int I, int MAXR>
__device__ __forceinline__ void load_wait(int rounds) {
  if constexpr (MAXR == 0) {
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
  } else {
    if (rounds >= MAXR) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(MAXR * I) : "memory");
    else load_wait<I, MAXR - 1>(rounds);
  }
}

// operand types: x and W bf16; both fp16; x bf16 and W e4m3 (decoded exactly to bf16 in registers); both e4m3
enum { BF16, F16, BF16_FP8, FP8 };

__device__ __forceinline__ int swz(int row) { return ((row >> 1) & 3) | (((row & 1) ^ ((row >> 3) & 1)) << 2); }

// The tile of a block: blocks are dealt to the 8 XCDs round-robin; each XCD takes an eighth of the tiles in a row, so that
// no XCD has more to do than another (18 column groups dealt out whole: three on two of the XCDs, two on the others, 15.4
// us against 9.7).  The larger operand is the outer index: weights (a group: n tiles and k range) that several blocks
// share come from memory once and from one XCD's L2 afterwards, or (by_rows) activations do.  Splits of K are the outermost
// part of a group: an XCD then reads one or two splits' columns of the activations, not all of them.
struct Tile {
  int mblock, nblk, split;
  int kt_lo, kt_hi;
};
__device__ __forceinline__ bool tile_of(Tile& t, const GemmArgs& a, int nblk_m, int ngroups, int by_rows) {
  const unsigned x8 = blockIdx.x & 7, total = (unsigned)nblk_m * (unsigned)ngroups, each = total >> 3, more = total & 7;
  if ((blockIdx.x >> 3) >= each + (x8 < more)) return false;
  const unsigned lin = x8 * each + (x8 < more ? x8 : more) + (blockIdx.x >> 3);
  t.mblock = (int)(by_rows ? lin / (unsigned)ngroups : lin % (unsigned)nblk_m);
  const int group = (int)(by_rows ? lin % (unsigned)ngroups : lin / (unsigned)nblk_m);
  const int nblk_n = ngroups / a.ksplit;
  t.split = group / nblk_n;
  t.nblk = group % nblk_n;
  t.kt_lo = t.split * a.kt_q + (t.split < a.kt_r ? t.split : a.kt_r);
  t.kt_hi = t.kt_lo + a.kt_q + (t.split < a.kt_r ? 1 : 0);
  return true;
}
inline unsigned blocks_of(int nblk_m, int ngroups) { return ((unsigned)nblk_m * (unsigned)ngroups + 7) / 8 * 8; }

template <int BM_, int BN_, int WGM_, int WGN_, int NS_, int MODE_>
struct Pipe {
  static constexpr int BM = BM_, BN = BN_, WGM = WGM_, WGN = WGN_, NS = NS_, MODE = MODE_;
  static constexpr int NW = WGM * WGN;                 // multiplying waves; as many more only load
  static constexpr int THREADS = 2 * NW * 64;
  static constexpr int TM = BM / WGM, TN = BN / WGN;   // tiles of a wave
  static constexpr int TILES = TM * TN;
  static constexpr int XE = MODE == FP8 ? 1 : 2;       // bytes of an x element
  static constexpr int RK = MODE == FP8 ? 4 : 2;       // k tiles of a round
  static constexpr int CPC = 16 / XE;                  // columns of a 16-byte chunk of x
  static constexpr int WT = MODE == BF16 || MODE == F16 ? 2048 : 1024;  // bytes of a packed weight tile
  static constexpr int WROUND = RK * WT;               // a round of one n tile: consecutive in memory
  static constexpr int AI = BM * 4 / NW, WI = BN * (WROUND / 1024) / NW;  // loads of a loading wave per round
  static constexpr int W_OFF = BM * 4096, STAGE = W_OFF + BN * WROUND;
  static constexpr int RING = NS * STAGE;
  static constexpr int STEPS = MODE == FP8 ? 2 : 4;    // of a round: one matrix instruction per tile each
  static constexpr int SP = BN * 128 + 16;             // row pitch of the block's fp32 sums in LDS (16 rows' same column: all banks)
  static constexpr int LDS = RING > BM * 32 * SP ? RING : BM * 32 * SP;
  static_assert(NW == 4 && BM % WGM == 0 && BN % WGN == 0 && BN * (WROUND / 1024) % NW == 0, "whole tiles and loads per wave");
  static_assert(LDS <= 160 * 1024 && NS >= 2 && (AI + WI) * (NS - 1) < 64, "LDS of a CU, the load counter's range");

  static __device__ __forceinline__ int next(int buf) { return buf + STAGE == RING ? 0 : buf + STAGE; }
  static __device__ __forceinline__ int rounds(const Tile& t) { return (t.kt_hi - t.kt_lo + RK - 1) / RK; }

  // ---- a loading wave (lw of NW), from its first load to the last barrier of the rounds ----
  static __device__ __forceinline__ void load(const GemmArgs& a, const Tile& t, unsigned char* lds, int lw, int lane) {
    const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)lds;
    const int nrounds = rounds(t);
    const int k_end = t.kt_hi * 32 < a.K ? t.kt_hi * 32 : a.K;
    const int k_last = (t.kt_lo + (nrounds - 1) * RK) * 32;
    // x: instruction i brings rows 8q .. 8q + 7 of the block, q = lw * AI + i; lane l the 16-byte slot l % 8 of row
    // 8q + l / 8, which holds the line's chunk (l % 8) ^ swz(row)
    const char* xp[AI];  // the eight rows' first column of this block's k range, then on
    unsigned xv[AI];     // the lane's chunk from there
    const bool far = (unsigned long long)a.ldx * (7 * XE) + 128 > 0xffffffffull;  // xv: within the row, xd: rows down
    int xd[AI];
    unsigned xfix[2];    // last round: lanes whose chunk is past the k range take the round's first one (zeroed in LDS)
#pragma unroll
    for (int i = 0; i < AI; ++i) {
      const int r0 = t.mblock * (BM * 32) + 8 * (lw * AI + i), rl = lane >> 3, ch = (lane & 7) ^ swz(8 * (lw * AI + i) + rl);
      const int b0 = r0 < a.M ? r0 : a.M - 1;  // rows past M: valid data, never stored
      const int m = r0 + rl < a.M ? r0 + rl : a.M - 1;
      xp[i] = (const char*)a.x + ((size_t)b0 * a.ldx + t.kt_lo * 32) * XE;
      xd[i] = m - b0;
      xv[i] = (far ? 0u : (unsigned)xd[i] * (unsigned)a.ldx * XE) + ch * 16;
      if (i < 2) xfix[i] = k_last + ch * CPC < k_end ? 0 : ch * 16;
    }
    // W: instruction i brings KiB q % PW of the round of n tile q / PW, q = i * NW + lw
    constexpr int PW = WROUND / 1024;
    const char* wp[WI];
#pragma unroll
    for (int i = 0; i < WI; ++i) {
      int ntg = t.nblk * BN + (i * NW + lw) / PW;
      if (ntg > a.ntiles - 1) ntg = a.ntiles - 1;  // overhanging tiles are computed on valid data, never stored
      wp[i] = (const char*)a.w + ((size_t)ntg * a.KT + t.kt_lo) * WT + lw % PW * 1024;
    }
    // last round's k tiles past the matrix: its last one again (their x is zero)
    const int past = t.kt_lo + (nrounds - 1) * RK + lw % PW * 1024 / WT - (a.KT - 1);
    const int w_back = past > 0 ? past * WT : 0;
    const unsigned lane16 = lane * 16;
    int ibuf = 0;  // LDS offset of the buffer that the next round is loaded into
    auto issue = [&](int r) {
      const bool last = r == nrounds - 1;
#pragma unroll
      for (int i = 0; i < AI; ++i) {
        const unsigned v = last ? xv[i] - xfix[i & 1] : xv[i], to = lds0 + (unsigned)(ibuf + (lw * AI + i) * 1024);
        if (far) dma16_far(xp[i] + (size_t)xd[i] * a.ldx * XE + v, to);
        else dma16(v, xp[i], to);
        xp[i] += 128;
      }
#pragma unroll
      for (int i = 0; i < WI; ++i) {
        dma16(lane16, wp[i] - (last ? w_back : 0), lds0 + (unsigned)(ibuf + W_OFF + (i * NW + lw) * 1024));
        wp[i] += WROUND;
      }
      ibuf = next(ibuf);
    };
    // NS rounds asked for; then, round after round: its own loads are there, so are the other waves' (and every multiplying
    // wave has left the round before, whose buffer takes round r - 1 + NS)
#pragma unroll
    for (int r = 0; r < NS; ++r)
      if (r < nrounds) issue(r);
    int buf = 0;
    for (int r = 0; r < nrounds; ++r) {
      const int ahead = nrounds - 1 - r;  // rounds asked for behind this one: at most NS - 2 of them, NS - 1 in the first round
      if (r == 0) load_wait<AI + WI, NS - 1>(ahead);
      else load_wait<AI + WI, NS - 2>(ahead);
      if (r == nrounds - 1 && k_last + RK * 32 > k_end) {  // columns past the k range
#pragma unroll
        for (int i = 0; i < AI; ++i)
          if (xfix[i & 1]) *(i32x4*)(lds + buf + (lw * AI + i) * 1024 + lane * 16) = i32x4{0, 0, 0, 0};
      }
      lds_barrier();
      if (r > 0 && r - 1 + NS < nrounds) issue(r - 1 + NS);
      buf = next(buf);
    }
  }

  // ---- a multiplying wave ----
  static __device__ __forceinline__ void multiply(f32x16 (&acc)[TM][TN], const Tile& t, const unsigned char* lds, int wave, int lane) {
    const int wm = wave / WGN, wn = wave % WGN, half = lane >> 5, l32 = lane & 31;
    const int nrounds = rounds(t);
    // an x operand is 1 (16-bit) or 2 (fp8) chunks of the line: step s, half h of the lanes
    constexpr int XH = MODE == FP8 ? 2 : 1;
    constexpr int WPS = MODE == BF16_FP8 ? 2 : 1;  // steps that one read of the weights serves
    i32x4 xa[2][TM][XH], wb[2][TN][XH];
    int xoff[STEPS][XH];
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
#pragma unroll
      for (int h = 0; h < XH; ++h) {
        const int chunk = MODE == FP8 ? 4 * s + 2 * h + half : (s >> 1) * 4 + 2 * half + (s & 1);
        xoff[s][h] = (wm * TM * 32 + l32) * 128 + ((chunk ^ swz(l32)) << 4);
      }
    const int woff = W_OFF + wn * TN * WROUND + lane * 16;
    // reads of step s, u in [0, RD): a matrix instruction's operands are complete one step before it
    constexpr int RD = (TM + TN) * XH;
    auto read1 = [&](int s, int buf, int u) {
      if (u < TM * XH) {
        xa[s & 1][u / XH][u % XH] = *(const i32x4*)(lds + buf + xoff[s][u % XH] + u / XH * 4096);
      } else if (s % WPS == 0) {
        const int v = u - TM * XH;
        wb[(s / WPS) & 1][v / XH][v % XH] = *(const i32x4*)(lds + buf + woff + v / XH * WROUND + (s / WPS * XH + v % XH) * 1024);
      }
    };
    auto mma1 = [&](int s, int i) {
      const int mt = i % TM, nt = i / TM;
      const i32x4(&w)[XH] = wb[(s / WPS) & 1][nt];
      const i32x4(&x)[XH] = xa[s & 1][mt];
      if constexpr (MODE == BF16)
        acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(w[0]), as_bf16x8(x[0]), acc[mt][nt], 0, 0, 0);
      else if constexpr (MODE == F16)
        acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(as_f16x8(w[0]), as_f16x8(x[0]), acc[mt][nt], 0, 0, 0);
      else if constexpr (MODE == BF16_FP8)
        acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fp8x8_to_bf16x8(w[0][2 * (s & 1)], w[0][2 * (s & 1) + 1]), as_bf16x8(x[0]), acc[mt][nt], 0, 0, 0);
      else
        acc[mt][nt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(i32x8{w[0][0], w[0][1], w[0][2], w[0][3], w[1][0], w[1][1], w[1][2], w[1][3]},
                                                                       i32x8{x[0][0], x[0][1], x[0][2], x[0][3], x[1][0], x[1][1], x[1][2], x[1][3]},
                                                                       acc[mt][nt], 0, 0, 0, 0, 0, 0);
    };
    lds_barrier();
    int buf = 0;
#pragma unroll
    for (int u = 0; u < RD; ++u) read1(0, 0, u);
    for (int r = 0; r < nrounds; ++r) {
#pragma unroll
      for (int s = 0; s < STEPS - 1; ++s)
#pragma unroll
        for (int i = 0; i < TILES; ++i) {
          mma1(s, i);
#pragma unroll
          for (int u = 0; u < RD; ++u)
            if (u * TILES / RD == i) read1(s + 1, buf, u);
          __builtin_amdgcn_sched_barrier(0);
        }
      buf = next(buf);
#pragma unroll
      for (int i = 0; i < (TILES + 1) / 2; ++i) mma1(STEPS - 1, i);
      __builtin_amdgcn_sched_barrier(0);
      if (r + 1 < nrounds) {
        lds_barrier();
#pragma unroll
        for (int u = 0; u < RD; ++u) read1(0, buf, u);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = (TILES + 1) / 2; i < TILES; ++i) mma1(STEPS - 1, i);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  static __device__ __forceinline__ void clear(f32x16 (&acc)[TM][TN]) {
#pragma unroll
    for (int mt = 0; mt < TM; ++mt)
#pragma unroll
      for (int nt = 0; nt < TN; ++nt)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[mt][nt][i] = 0.f;
  }
};

}  // namespace pipe
