// The many-row GEMMs over fp8 weights: kernel, K-split reduction and block shapes shared by the weight-only form (bf16
// activations, pipe::BF16_FP8) and the W8A8 form (per-token quantised activations, pipe::FP8).  Products: pipe_gemm.h.
#pragma once
#include "pipe_gemm.h"

namespace pipe {

// Rounding points of the epilogues.  Weight-only: bf16(acc * sw[n]); W8A8: bf16((acc * sa[m]) * sw[n]), products rounded
// separately (the reference's `acc * a_scale[:, None] * w_scale[None, :]`).
template <int MODE>
__device__ __forceinline__ f32x4 scaled(f32x4 v, float sa, f32x4 sw) {
  if constexpr (MODE == FP8) {
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = mul_rn(mul_rn(v[j], sa), sw[j]);
    return v;
  } else {
    return v * sw;
  }
}

template <int MODE>
__device__ __forceinline__ float gated_act(int act, float g) {
  return act == 0 ? silu_f(g) : MODE == FP8 ? gelu_tanh_rcp_f(g) : gelu_tanh_f(g);
}

// What an epilogue piece (eight output columns of a row) reads from memory besides its sums.
template <int EPI>
struct PieceIn {
  f32x4 s0[2], s1[EPI == 1 ? 2 : 1];  // scales (gated: gate and up)
  f32x4 rf[EPI == 0 ? 2 : 1];         // fp32 residual
  i32x2 rh[EPI == 0 ? 2 : 1];         // bf16 residual
  i32x2 gt[EPI == 0 ? 2 : 1];
  float sa;
};
// m, n: row and first column (n a multiple of 8).  What lies outside the matrix is loaded from inside and not stored.
template <int MODE, int EPI>
__device__ __forceinline__ void ask_scales(PieceIn<EPI>& p, const GemmArgs& a, int n) {
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int nq = n + 4 * q < a.N ? n + 4 * q : a.N - 4;
    p.s0[q] = *(const f32x4*)(a.s0 + nq);
    if constexpr (EPI == 1) p.s1[q] = *(const f32x4*)(a.s1 + nq);
    if constexpr (EPI == 0) {
      if (MODE != FP8 && a.gate) p.gt[q] = *(const i32x2*)(a.gate + nq);
    }
  }
}
template <int MODE, int EPI>
__device__ __forceinline__ void ask_row(PieceIn<EPI>& p, const GemmArgs& a, int m, int n) {
  const int mc = m < a.M ? m : a.M - 1;
  if constexpr (MODE == FP8) p.sa = a.row_scale[mc];
  if constexpr (EPI == 0) {
    if (a.resid) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int nq = n + 4 * q < a.N ? n + 4 * q : a.N - 4;
        if (a.resid_f32) p.rf[q] = *(const f32x4*)((const float*)a.resid + (size_t)mc * a.ldr + nq);
        else p.rh[q] = *(const i32x2*)((const u16*)a.resid + (size_t)mc * a.ldr + nq);
      }
    }
  }
}
// v: the piece's sums (gated: the gate's; u the up projection's)
template <int MODE, int EPI>
__device__ __forceinline__ void finish(const GemmArgs& a, const PieceIn<EPI>& p, const f32x4 (&v)[2], const f32x4 (&u)[2], int m, int n) {
  i32x2 o[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    if constexpr (EPI == 0) {
      o[q] = pack_bf16x4(scaled<MODE>(v[q], p.sa, p.s0[q]));
      if (MODE != FP8 && a.gate) o[q] = pack_bf16x4(unpack_bf16x4(o[q]) * unpack_bf16x4(p.gt[q]));
      if (a.resid) o[q] = pack_bf16x4(unpack_bf16x4(o[q]) + (a.resid_f32 ? p.rf[q] : unpack_bf16x4(p.rh[q])));
    } else {
      const f32x4 gg = unpack_bf16x4(pack_bf16x4(scaled<MODE>(v[q], p.sa, p.s0[q])));
      const f32x4 up = unpack_bf16x4(pack_bf16x4(scaled<MODE>(u[q], p.sa, p.s1[q])));
      f32x4 act;
#pragma unroll
      for (int j = 0; j < 4; ++j) act[j] = gated_act<MODE>(a.act, gg[j]);
      o[q] = pack_bf16x4(unpack_bf16x4(pack_bf16x4(act)) * up);
    }
  }
  if (m >= a.M || n >= a.N) return;
  u16* dst = a.y + (size_t)m * a.ldy + n;
  if (a.vec16 && n + 8 <= a.N) {
    *(i32x4*)dst = i32x4{o[0][0], o[0][1], o[1][0], o[1][1]};
  } else {  // 8-byte aligned rows, or the row's last four columns
    *(i32x2*)dst = o[0];
    if (n + 8 <= a.N) *(i32x2*)(dst + 4) = o[1];
  }
}

// EPI: 0 plain (scale, optional per-column gate, optional residual), 1 gated (gate / up tile pairs).  A K split leaves fp32
// partials [split][M][packed columns] for the reduction launch.
template <int MODE, int EPI, int BM, int BN, int WGM, int WGN, int NS, int OCC>
__global__ __launch_bounds__(2 * WGM * WGN * 64, 2 * OCC) void fp8_pipe_kernel(GemmArgs a, int nblk_m, int ngroups, int by_rows) {
  using P = Pipe<BM, BN, WGM, WGN, NS, MODE>;
  static_assert(P::LDS * OCC <= 160 * 1024, "LDS of a CU");
  __shared__ __align__(1024) unsigned char lds[P::LDS];
  Tile t;
  if (!tile_of(t, a, nblk_m, ngroups, by_rows)) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool loader = wave >= P::NW;

  f32x16 acc[P::TM][P::TN];
  P::clear(acc);
  if (loader) P::load(a, t, lds, wave - P::NW, lane);
  else P::multiply(acc, t, lds, wave, lane);

  // ---- the block's sums go to LDS in fp32; loops over 16-byte pieces of output rows, on all eight waves, finish them ----
  const int m_blk = t.mblock * BM * 32;
  constexpr int CPR = (EPI == 0 ? BN : BN / 2) * 4;  // pieces per row
  constexpr int ITEMS = (BM * 32 * CPR + P::THREADS - 1) / P::THREADS;
  static_assert(P::THREADS % CPR == 0, "a thread keeps its columns");
  const int ch = tid % CPR, row0 = tid / CPR;
  const int n = t.nblk * (EPI == 0 ? BN : BN / 2) * 32 + ch * 8;
  PieceIn<EPI> in;
  if (a.ksplit == 1) ask_scales<MODE, EPI>(in, a, n);
  lds_barrier();  // every wave has left the ring behind
  if (!loader) {
    const int wm = wave / WGN, wn = wave % WGN, half = lane >> 5, l32 = lane & 31;
#pragma unroll
    for (int mt = 0; mt < P::TM; ++mt)
#pragma unroll
      for (int nt = 0; nt < P::TN; ++nt)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x16& c = acc[mt][nt];
          *(f32x4*)(lds + ((wm * P::TM + mt) * 32 + l32) * P::SP + ((wn * P::TN + nt) * 32 + 8 * g + 4 * half) * 4) = f32x4{c[4 * g], c[4 * g + 1], c[4 * g + 2], c[4 * g + 3]};
        }
  }
  if (a.ksplit > 1) {
    lds_barrier();
    const int ldp = a.ntiles * 32, np0 = t.nblk * BN * 32;
    float* dst = a.partial + (size_t)t.split * a.M * ldp;
#pragma unroll 2
    for (int it = tid; it < BM * 32 * BN * 8; it += P::THREADS) {  // pieces of four packed columns
      const int row = it / (BN * 8), np = np0 + it % (BN * 8) * 4;
      if (m_blk + row < a.M && np < ldp) *(f32x4*)(dst + (size_t)(m_blk + row) * ldp + np) = *(const f32x4*)(lds + row * P::SP + it % (BN * 8) * 16);
    }
    return;
  }
  constexpr int PRE = EPI == 0 ? (ITEMS < 4 ? ITEMS : 4) : 1;  // pieces whose row operands are asked for in front of the barrier
  PieceIn<EPI> rows[PRE];
  if (EPI == 0) {
#pragma unroll
    for (int i = 0; i < PRE; ++i) ask_row<MODE, EPI>(rows[i], a, m_blk + row0 + i * (P::THREADS / CPR), n);
  }
  lds_barrier();
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const int row = row0 + i * (P::THREADS / CPR), m = m_blk + row;
    if (BM * 32 * CPR % P::THREADS != 0 && row >= BM * 32) break;
    if (EPI == 0 && i < PRE) {
#pragma unroll
      for (int q = 0; q < (EPI == 0 ? 2 : 1); ++q) {
        in.rf[q] = rows[i < PRE ? i : 0].rf[q];
        in.rh[q] = rows[i < PRE ? i : 0].rh[q];
      }
      in.sa = rows[i < PRE ? i : 0].sa;
    } else {
      ask_row<MODE, EPI>(in, a, m, n);
    }
    // gated: the piece's gate and up sums stand in adjacent packed tiles
    const unsigned char* src = lds + row * P::SP + (EPI == 0 ? ch * 32 : ((ch >> 2) * 64 + (ch & 3) * 8) * 4);
    const f32x4 v[2] = {*(const f32x4*)src, *(const f32x4*)(src + 16)};
    f32x4 u[2] = {v[0], v[1]};
    if (EPI == 1) {
      u[0] = *(const f32x4*)(src + 128);
      u[1] = *(const f32x4*)(src + 144);
    }
    finish<MODE, EPI>(a, in, v, u, m, n);
  }
}

// Second launch of a K split: a thread sums one piece (eight output columns) over the splits in split order and finishes it.
template <int MODE, int EPI>
__global__ __launch_bounds__(256) void fp8_split_reduce_kernel(GemmArgs a) {
  const int cpr = (a.N + 7) / 8;
  const int it = blockIdx.x * 256 + threadIdx.x;
  if (it >= a.M * cpr) return;
  const int m = it / cpr, n = it % cpr * 8, ldp = a.ntiles * 32;
  const int np = EPI == 0 ? n : (n >> 5) * 64 + (n & 31);  // packed column
  PieceIn<EPI> in;
  ask_scales<MODE, EPI>(in, a, n);
  ask_row<MODE, EPI>(in, a, m, n);
  f32x4 v[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}}, u[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  const float* src = a.partial + (size_t)m * ldp + np;
#pragma unroll 4
  for (int s = 0; s < a.ksplit; ++s) {
    const float* p = src + (size_t)s * a.M * ldp;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      v[q] += *(const f32x4*)(p + 4 * q);
      if (EPI == 1) u[q] += *(const f32x4*)(p + 32 + 4 * q);
    }
  }
  finish<MODE, EPI>(a, in, v, u, m, n);
}

template <int MODE, int BM, int BN, int WGM, int WGN, int NS, int OCC>
int launch_fp8_pipe(const GemmArgs& a, hipStream_t st) {
  const int nblk_m = (a.M + BM * 32 - 1) / (BM * 32), ngroups = (a.ntiles + BN - 1) / BN * a.ksplit;
  const int by_rows = (long long)a.M * (MODE == FP8 ? 1 : 2) > (long long)a.ntiles * 32;  // bytes of a k column of x and of W
  const dim3 grid(blocks_of(nblk_m, ngroups)), block(2 * WGM * WGN * 64);
  if (a.s1) hipLaunchKernelGGL((fp8_pipe_kernel<MODE, 1, BM, BN, WGM, WGN, NS, OCC>), grid, block, 0, st, a, nblk_m, ngroups, by_rows);
  else hipLaunchKernelGGL((fp8_pipe_kernel<MODE, 0, BM, BN, WGM, WGN, NS, OCC>), grid, block, 0, st, a, nblk_m, ngroups, by_rows);
  if (a.ksplit > 1) {
    const long long items = (long long)a.M * ((a.N + 7) / 8);
    const dim3 rg((unsigned)((items + 255) / 256));
    if (a.s1) hipLaunchKernelGGL((fp8_split_reduce_kernel<MODE, 1>), rg, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((fp8_split_reduce_kernel<MODE, 0>), rg, dim3(256), 0, st, a);
  }
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

// ---- epilogue of the kernels whose weights go through registers: a wave holds tile pairs of its own ----
constexpr int WIDE_NT = 2;  // n tiles per wave

// LDS row pitch (bytes) of a wave's private 32-row output tile in wide_epilogue
__host__ __device__ constexpr int wide_ep_pitch(int epi) { return (epi == 0 ? WIDE_NT * 32 : 32) * 2 + 16; }

// Epilogue of a wave that holds MT x NT accumulator tiles: rows row0 .. row0 + MT*32 - 1, packed n tiles strip*NT ..
// (EPI 1: the (gate, up) pair of output columns strip*32 ..).  wl: the wave's private LDS tile of 32 rows x
// wide_ep_pitch(EPI) bytes (used when the output is 16-byte aligned); the caller has made sure that no wave still
// reads what that space held before.
template <int MODE, int EPI, int MT>
__device__ __forceinline__ void wide_epilogue(const GemmArgs& a, const f32x16 (&acc)[MT][WIDE_NT], unsigned char* wl, int row0, int strip, int lane) {
  constexpr int NT = WIDE_NT;
  const int half = lane >> 5;
  const int l32 = lane & 31;
  float sa[MT];  // W8A8: the scales of this lane's rows
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = row0 + mt * 32 + l32;
    sa[mt] = MODE == FP8 ? a.row_scale[m < a.M ? m : a.M - 1] : 1.f;
  }
  // ---- epilogue: lane l of a tile owns row m = l % 32 and, per register group g, four
  // consecutive columns 8g + 4*(l/32) .. +3 (the accumulators hold C^T) ----
  if (a.vec16) {
    // Coalesced stores: a lane holds, per tile, row l % 32 and four 4-column pieces 16 bytes apart -- stored as
    // they are, one instruction would touch 32 rows with 16 bytes each.  Each wave therefore passes its 32 rows of
    // an m tile through a private LDS tile (a wave's LDS instructions execute in order, so it needs no barrier
    // of its own) and stores them as 16-byte chunks of consecutive columns: whole 64- or 128-byte row segments
    // per 4 or 8 lanes.
    constexpr int COLS = EPI == 0 ? NT * 32 : 32;  // output columns of a wave per row
    constexpr int EP = COLS * 2 + 16;              // LDS row pitch (bytes)
    constexpr int LPR = COLS / 8;                  // lanes (16-byte chunks) per row
    constexpr int RPI = 64 / LPR;                  // rows per store instruction
    static_assert(EP == wide_ep_pitch(EPI), "the callers size the LDS tiles by wide_ep_pitch");
    const int ncol0 = EPI == 0 ? strip * NT * 32 : strip * 32;  // first output column of this wave
    f32x4 sc0[EPI == 0 ? NT : 1][4], sc1[4], gt[EPI == 0 ? NT : 1][4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      if (EPI == 0) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          int n0 = (strip * NT + nt) * 32 + 8 * g + 4 * half;
          if (n0 > a.N - 4) n0 = a.N - 4;  // columns past N are never stored
          sc0[EPI == 0 ? nt : 0][g] = *(const f32x4*)(a.s0 + n0);
          if (MODE != FP8 && a.gate) gt[EPI == 0 ? nt : 0][g] = unpack_bf16x4(*(const i32x2*)(a.gate + n0));
        }
      } else {
        int col = strip * 32 + 8 * g + 4 * half;
        if (col > a.N - 4) col = a.N - 4;
        sc0[0][g] = *(const f32x4*)(a.s0 + col);
        sc1[g] = *(const f32x4*)(a.s1 + col);
      }
    }
    const int lrow = lane / LPR, lchunk = lane % LPR;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        if (EPI == 0) {
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) {
            const f32x16& c = acc[mt][nt];
            const f32x4 v = {c[4 * g], c[4 * g + 1], c[4 * g + 2], c[4 * g + 3]};
            i32x2 r = pack_bf16x4(scaled<MODE>(v, sa[mt], sc0[EPI == 0 ? nt : 0][g]));
            if (MODE != FP8 && a.gate) r = pack_bf16x4(unpack_bf16x4(r) * gt[EPI == 0 ? nt : 0][g]);
            *(i32x2*)(wl + l32 * EP + (nt * 32 + 8 * g + 4 * half) * 2) = r;
          }
        } else {
          const f32x16& cg = acc[mt][0];
          const f32x16& cu = acc[mt][1];
          const f32x4 vg = {cg[4 * g], cg[4 * g + 1], cg[4 * g + 2], cg[4 * g + 3]};
          const f32x4 vu = {cu[4 * g], cu[4 * g + 1], cu[4 * g + 2], cu[4 * g + 3]};
          const f32x4 gg = unpack_bf16x4(pack_bf16x4(scaled<MODE>(vg, sa[mt], sc0[0][g])));
          const f32x4 up = unpack_bf16x4(pack_bf16x4(scaled<MODE>(vu, sa[mt], sc1[g])));
          f32x4 act;
#pragma unroll
          for (int j = 0; j < 4; ++j) act[j] = gated_act<MODE>(a.act, gg[j]);
          act = unpack_bf16x4(pack_bf16x4(act));
          *(i32x2*)(wl + l32 * EP + (8 * g + 4 * half) * 2) = pack_bf16x4(act * up);
        }
      }
#pragma unroll
      for (int j = 0; j < 32 / RPI; ++j) {
        const int row = j * RPI + lrow;
        const int m = row0 + mt * 32 + row;
        const int n = ncol0 + lchunk * 8;
        i32x4 t = *(const i32x4*)(wl + row * EP + lchunk * 16);
        if (m >= a.M || n >= a.N) continue;
        if (EPI == 0 && a.resid) {
          // bf16(y + resid) on the bf16-rounded product, as the scattered path computes it
          f32x4 r0, r1 = {0.f, 0.f, 0.f, 0.f};
          if (a.resid_f32) {
            const f32x4* rp = (const f32x4*)((const float*)a.resid + (size_t)m * a.ldr + n);
            r0 = rp[0];
            if (n + 8 <= a.N) r1 = rp[1];
          } else if (n + 8 <= a.N) {
            const i32x4 rr = *(const i32x4*)((const u16*)a.resid + (size_t)m * a.ldr + n);
            r0 = unpack_bf16x4(i32x2{rr[0], rr[1]});
            r1 = unpack_bf16x4(i32x2{rr[2], rr[3]});
          } else {
            r0 = unpack_bf16x4(*(const i32x2*)((const u16*)a.resid + (size_t)m * a.ldr + n));
          }
          const i32x2 lo = pack_bf16x4(unpack_bf16x4(i32x2{t[0], t[1]}) + r0), hi = pack_bf16x4(unpack_bf16x4(i32x2{t[2], t[3]}) + r1);
          t = i32x4{lo[0], lo[1], hi[0], hi[1]};
        }
        u16* dst = a.y + (size_t)m * a.ldy + n;
        if (n + 8 <= a.N) *(i32x4*)dst = t;
        else *(i32x2*)dst = i32x2{t[0], t[1]};  // N % 8 == 4: the row's last four columns
      }
    }
    return;
  }
  if (EPI == 0) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int n0 = (strip * NT + nt) * 32 + 8 * g + 4 * half;
        if (n0 >= a.N) continue;
        const f32x4 sc = *(const f32x4*)(a.s0 + n0);
        f32x4 gt = {0.f, 0.f, 0.f, 0.f};
        if (MODE != FP8 && a.gate) gt = unpack_bf16x4(*(const i32x2*)(a.gate + n0));
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const int m = row0 + mt * 32 + l32;
          if (m >= a.M) continue;
          const f32x16& c = acc[mt][nt];
          f32x4 v = {c[4 * g], c[4 * g + 1], c[4 * g + 2], c[4 * g + 3]};
          i32x2 r = pack_bf16x4(scaled<MODE>(v, sa[mt], sc));
          if (MODE != FP8 && a.gate) r = pack_bf16x4(unpack_bf16x4(r) * gt);
          if (a.resid) {
            const f32x4 rv = a.resid_f32 ? *(const f32x4*)((const float*)a.resid + (size_t)m * a.ldr + n0)
                                         : unpack_bf16x4(*(const i32x2*)((const u16*)a.resid + (size_t)m * a.ldr + n0));
            r = pack_bf16x4(unpack_bf16x4(r) + rv);
          }
          *(i32x2*)(a.y + (size_t)m * a.ldy + n0) = r;
        }
      }
  } else {
    // tile pair (gate, up) of logical columns strip*32 ..; I % 32 == 0
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int col = strip * 32 + 8 * g + 4 * half;
      if (col >= a.N) continue;
      const f32x4 scg = *(const f32x4*)(a.s0 + col), scu = *(const f32x4*)(a.s1 + col);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const int m = row0 + mt * 32 + l32;
        if (m >= a.M) continue;
        const f32x16& cg = acc[mt][0];
        const f32x16& cu = acc[mt][1];
        const f32x4 vg = {cg[4 * g], cg[4 * g + 1], cg[4 * g + 2], cg[4 * g + 3]};
        const f32x4 vu = {cu[4 * g], cu[4 * g + 1], cu[4 * g + 2], cu[4 * g + 3]};
        const f32x4 gg = unpack_bf16x4(pack_bf16x4(scaled<MODE>(vg, sa[mt], scg)));
        const f32x4 up = unpack_bf16x4(pack_bf16x4(scaled<MODE>(vu, sa[mt], scu)));
        f32x4 act;
#pragma unroll
        for (int j = 0; j < 4; ++j) act[j] = gated_act<MODE>(a.act, gg[j]);
        act = unpack_bf16x4(pack_bf16x4(act));
        *(i32x2*)(a.y + (size_t)m * a.ldy + col) = pack_bf16x4(act * up);
      }
    }
  }
}


}  // namespace pipe
