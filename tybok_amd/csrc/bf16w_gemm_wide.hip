// 16-bit-weight GEMM for many rows with bias / GELU / residual epilogues on gfx950: the linears of the vision
// towers (q|k|v, out_proj, fc1, fc2 over 256 .. 1024 patches per camera) and the bf16 projections of the VLM
// prefill.
//
//   y[M, N] = bf16( resid + act( bf16( x[M, K] . W[N, K]^T + bias[N] ) ) )
//
// Operands: x bf16 row-major; W in the 2 KiB tile order of tk_pack_bf16_weight (tile (nt, kt): two 1 KiB chunks,
// chunk c of lane l = 8 bf16 of column nt*32 + l%32 at k = 32*kt + 16*(l/32) + 8*c), so a weight operand of
// v_mfma_f32_32x32x16_bf16 is one coalesced 16-byte load per lane.
// The products are those of pipe_gemm.h: loads straight to LDS on waves of their own.
//   * K splits hand fp32 partials through the workspace; the last-arriving block sums them in split order:
//     bit-deterministic;
//   * the epilogue passes the block's fp32 sums through LDS and stores 16-byte row segments on all eight waves; what it
//     reads from memory (bias, residual, rotary positions and table rows) is asked for before the products: 1 - 2 us a
//     launch against asking behind them (the weights and vectors of a layer are cold in every request).
// Measured (cold weights, graph replay, us; before: weights straight into the registers of the four waves that multiply):
// SmolVLA's tower at 3 x 1024 rows q|k|v 21.4 -> 17.8, out_proj 14.4 -> 10.2, fc1 25.8 -> 22.1, fc2 29.0 -> 21.7; pi0.5's
// at 2 x 256 rows 13.0 -> 12.4, 10.7 -> 9.4, 14.4 -> 12.7, 22.9 -> 20.8; pi0.5's prefill at 712 rows q|k|v with the
// rotary epilogue 24.4 -> 14.8, o_proj 15.1 -> 13.3.  Slower than before: K below 600 with the weights already in the L2s (48 x
// 256 -> 112 3.5 -> 4.2), and grids just over a generation of 128 x 128 blocks (1100 rows and 8192 columns, K 256 .. 1536: 8 - 18 %,
// where the former kernel held three 96 x 128 blocks a CU).  A launch of this kind that does nothing takes 1.9 us; what bounds
// them is a compute unit's 133 bytes/ns of loads (0.35 - 0.6 us a round), then the epilogue (0.2 us per 32 x 32 tile).
#include "pipe_gemm.h"

namespace {
using namespace pipe;

// FP16: the operands are fp16 (v_mfma_f32_32x32x16_f16) instead of bf16; same tile order, same epilogues
// ROPE (TN == 2, bf16): the weights are packed in rotary pair order -- the two tiles of a wave hold columns
// (c, c + rope_half) of one head -- and the epilogue is the skinny kernel's rotary one: columns < rope_cols rotated
// by the table row of pos[m] (fp32 products rounded separately, or every product and sum rounded to bf16), columns
// >= vt_col0 also written transposed for the attention kernel.  No bias, activation or residual in this form.
template <int BM, int BN, int WGM, int WGN, int NS, int OCC, bool FP16, bool ROPE = false>
__global__ __launch_bounds__(2 * WGM * WGN * 64, 2 * OCC) void bf16w_wide_kernel(GemmArgs a, int nblk_m, int ngroups, int by_rows) {
  using P = Pipe<BM, BN, WGM, WGN, NS, FP16 ? F16 : BF16>;
  constexpr int NW = P::NW, TM = P::TM, TN = P::TN, TILES = P::TILES, SP = P::SP;
  static_assert(!ROPE || (TN == 2 && !FP16), "the rotary epilogue needs both halves of a pair in one wave");
  static_assert(P::LDS * OCC <= 160 * 1024, "LDS of a CU");
  __shared__ __align__(1024) unsigned char lds[P::LDS];
  Tile tile;
  if (!tile_of(tile, a, nblk_m, ngroups, by_rows)) return;
  const int mblock = tile.mblock, nblk = tile.nblk, split = tile.split;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool loader = wave >= NW;
  const int wm = wave / WGN, wn = wave % WGN;  // a multiplying wave's place
  const int half = lane >> 5;
  const int l32 = lane & 31;

  constexpr int THREADS = P::THREADS, CPR = BN * 4, ITEMS = BM * 32 * CPR / THREADS;  // 16-byte pieces of outputs: per row, per thread
  constexpr int PRE_MAX = OCC == 1 ? 4 : TILES < 4 ? 2 : 1, PRE = ITEMS < PRE_MAX ? ITEMS : PRE_MAX;  // pieces whose residual is asked for here (128 registers at two blocks a compute unit)
  static_assert(BM * 32 * CPR % THREADS == 0, "whole pieces");
  const int m_blk = mblock * BM * 32, n_blk = nblk * BN * 32;
  constexpr int PPR = ROPE ? BN / 2 * 4 : 1, RITEMS = ROPE ? BM * 32 * PPR / THREADS : 1;  // rotary form: pairs of pieces, per row and per thread
  static_assert(!ROPE || BM * 32 * PPR % THREADS == 0, "whole pieces");
  int rope_pos[RITEMS];
  if (ROPE) {
#pragma unroll
    for (int i = 0; i < RITEMS; ++i) {
      const int m = m_blk + (i * THREADS + tid) / PPR;
      rope_pos[i] = a.rope_pos[m < a.M ? m : a.M - 1];
    }
  }

  f32x16 acc[TM][TN];
  P::clear(acc);
  if (loader) P::load(a, tile, lds, wave - NW, lane);

  // Bias and (16-bit) residual are asked for before the products: behind them they would be a round trip of their own,
  // to memory that nothing has touched yet
  i32x2 bias[TN][4];
  if (!ROPE && a.bias && !loader) {
#pragma unroll
    for (int nt = 0; nt < TN; ++nt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int n = n_blk + (wn * TN + nt) * 32 + 8 * g + 4 * half;
        bias[nt][g] = *(const i32x2*)(a.bias + (n < a.N ? n : a.N - 4));  // columns past N are never stored
      }
  }
  i32x2 pre[PRE][2];
  const bool res16 = !ROPE && a.resid && !a.resid_f32;
  auto ask_res = [&](i32x2 (&r)[2], int item) {
    const int idx = item * THREADS + tid, m = m_blk + idx / CPR, n = n_blk + idx % CPR * 8;
    const u16* p = (const u16*)a.resid + (size_t)(m < a.M ? m : a.M - 1) * a.ldr;  // what lies outside is loaded from inside and not stored
    r[0] = *(const i32x2*)(p + (n < a.N ? n : a.N - 4));
    r[1] = *(const i32x2*)(p + (n + 4 < a.N ? n + 4 : a.N - 4));
  };
  if (res16 && !loader) {
#pragma unroll
    for (int i = 0; i < PRE; ++i) ask_res(pre[i], i);
  }

  // rotary form: the first pair of pieces' row of the tables as well (the loading waves ask when they have nothing left to load)
  const int po = ROPE ? a.rope_half >> 5 : 1;
  auto first_col = [&](int pair) { return ((pair / po) * 2 * po + pair % po) * 32; };  // of a pair of physical tiles (pair, 0 / 1)
  struct RopeRow {
    f32x4 cos[2], sin[2];
  } early;
  auto ask_rope = [&](RopeRow& t, int i) {
    const int pc = (i * THREADS + tid) % PPR, ca = first_col(nblk * (BN / 2) + (pc >> 2)) + (pc & 3) * 8;
    int pos = rope_pos[i];
    pos = pos < 0 ? 0 : (pos > a.rope_positions - 1 ? a.rope_positions - 1 : pos);
    const size_t at = (size_t)pos * a.rope_half + ca % (2 * a.rope_half);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      t.cos[q] = *(const f32x4*)(a.rope_cos + at + 4 * q);
      t.sin[q] = *(const f32x4*)(a.rope_sin + at + 4 * q);
    }
  };
  if (ROPE) ask_rope(early, 0);

  if (!loader) P::multiply(acc, tile, lds, wave, lane);

  // ---- K-split hand-off: fp32 partials [(block, split)][wave][tile][group][lane][4] ----
  const int blk_lin = nblk * nblk_m + mblock;
  if (a.ksplit > 1) {
    unsigned long long* pbase = (unsigned long long*)a.partial + ((size_t)wave * TILES * 4 * 64 + lane) * 2;
    unsigned long long* mine = pbase + ((size_t)blk_lin * a.ksplit + split) * (NW * TILES * 4 * 64 * 2);
    if (!loader) {
#pragma unroll
      for (int t = 0; t < TILES; ++t)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x16& c = acc[t / TN][t % TN];
          unsigned long long* dst = mine + (size_t)(t * 4 + g) * 128;
          st_agent64(dst, c[4 * g], c[4 * g + 1]);
          st_agent64(dst + 1, c[4 * g + 2], c[4 * g + 3]);
        }
    }
    int* s_last = (int*)lds;  // (the ring is idle behind the barrier)
    handoff_publish();
    __syncthreads();
    if (threadIdx.x == 0) {
      int old = __hip_atomic_fetch_add(a.counters + blk_lin, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *s_last = (old == a.ksplit - 1);
    }
    __syncthreads();
    if (!*s_last) return;
    handoff_acquire();
    if (threadIdx.x == 0) __hip_atomic_store(a.counters + blk_lin, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int mt = 0; mt < TM; ++mt)
#pragma unroll
      for (int nt = 0; nt < TN; ++nt)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[mt][nt][i] = 0.f;
    for (int s = 0; s < (loader ? 0 : a.ksplit); ++s) {  // split order, whoever arrived last
      const unsigned long long* src = pbase + ((size_t)blk_lin * a.ksplit + s) * (NW * TILES * 4 * 64 * 2);
#pragma unroll
      for (int t = 0; t < TILES; ++t) {
        unsigned long long raw[4][2];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          raw[g][0] = ld_agent64(src + (size_t)(t * 4 + g) * 128);
          raw[g][1] = ld_agent64(src + (size_t)(t * 4 + g) * 128 + 1);
        }
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          f32x16& c = acc[t / TN][t % TN];
          c[4 * g] += __uint_as_float((unsigned)raw[g][0]);
          c[4 * g + 1] += __uint_as_float((unsigned)(raw[g][0] >> 32));
          c[4 * g + 2] += __uint_as_float((unsigned)raw[g][1]);
          c[4 * g + 3] += __uint_as_float((unsigned)(raw[g][1] >> 32));
        }
      }
    }
  }

  // ---- epilogue: lane l of a tile holds row m = l % 32 and, per register group g, four consecutive columns
  // 8g + 4*(l/32) .. +3 (the accumulators are C^T).  All of it goes to LDS as fp32 with the bias added; loops over
  // 16-byte pieces of output rows, on all eight waves, then finish them. ----
  if (res16 && loader) {
#pragma unroll
    for (int i = 0; i < PRE; ++i) ask_res(pre[i], i);
  }
  lds_barrier();  // every wave has left the ring (or the partials) behind
  if (!loader) {
#pragma unroll
    for (int mt = 0; mt < TM; ++mt)
#pragma unroll
      for (int nt = 0; nt < TN; ++nt)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x16& c = acc[mt][nt];
          f32x4 v = {c[4 * g], c[4 * g + 1], c[4 * g + 2], c[4 * g + 3]};
          if (!ROPE && a.bias) v = v + unpack_16x4<FP16>(bias[nt][g]);
          *(f32x4*)(lds + ((wm * TM + mt) * 32 + l32) * SP + ((wn * TN + nt) * 32 + 8 * g + 4 * half) * 4) = v;
        }
  }
  lds_barrier();
  if constexpr (ROPE) {
#pragma unroll
    for (int i = 0; i < RITEMS; ++i) {
      const int it = i * THREADS + tid, row = it / PPR, pc = it % PPR, c8 = (pc & 3) * 8;
      const int m = m_blk + row, ca = first_col(nblk * (BN / 2) + (pc >> 2)) + c8, cb = ca + a.rope_half;
      RopeRow late;
      if (i > 0) ask_rope(late, i);
      const RopeRow& t = i > 0 ? late : early;
      const unsigned char* src = lds + row * SP + ((pc >> 2) * 64 + c8) * 4;
      i32x2 oa[2], ob[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        f32x4 va = unpack_bf16x4(pack_bf16x4(*(const f32x4*)(src + 16 * q)));
        f32x4 vb = unpack_bf16x4(pack_bf16x4(*(const f32x4*)(src + 128 + 16 * q)));
        if (ca < a.rope_cols) {
          const f32x4 cs = t.cos[q], sn = t.sin[q];
          f32x4 ra, rb;
          if (a.rope_bf16) {
            const f32x4 ac = unpack_bf16x4(pack_bf16x4(va * cs)), bs = unpack_bf16x4(pack_bf16x4(vb * sn));
            const f32x4 bc = unpack_bf16x4(pack_bf16x4(vb * cs)), as = unpack_bf16x4(pack_bf16x4(va * sn));
            ra = ac - bs;
            rb = bc + as;
          } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              ra[j] = sub_rn(mul_rn(va[j], cs[j]), mul_rn(vb[j], sn[j]));
              rb[j] = add_rn(mul_rn(vb[j], cs[j]), mul_rn(va[j], sn[j]));
            }
          }
          va = ra;
          vb = rb;
        }
        oa[q] = pack_bf16x4(va);
        ob[q] = pack_bf16x4(vb);
      }
      if (m >= a.M) continue;
      u16* dst = a.y + (size_t)m * a.ldy;  // N is a whole number of heads in this form
      if (ca < a.N) *(i32x4*)(dst + ca) = i32x4{oa[0][0], oa[0][1], oa[1][0], oa[1][1]};
      if (cb < a.N) *(i32x4*)(dst + cb) = i32x4{ob[0][0], ob[0][1], ob[1][0], ob[1][1]};
    }
    if (a.vt) {
      // value columns, transposed for the attention kernel: eight consecutive rows per 16-byte store, four stores in a
      // row; rows past M stay zero (the attention kernel relies on zeros behind the last key)
#pragma unroll 1
      for (int it = tid; it < BM * 4 * BN * 32; it += THREADS) {
        const int col = (it >> 2) % (BN * 32), rg = (it / (BN * 128)) * 4 + (it & 3);
        const int n = first_col(nblk * (BN / 2) + (col >> 6)) + (col & 31) + ((col >> 5) & 1) * a.rope_half;
        const int m0 = m_blk + 8 * rg;
        if (n < a.vt_col0 || n >= a.N || m0 >= a.M) continue;
        i32x4 e;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float lo = *(const float*)(lds + (8 * rg + 2 * r) * SP + col * 4), hi = *(const float*)(lds + (8 * rg + 2 * r + 1) * SP + col * 4);
          e[r] = (int)pack_bf16x2(m0 + 2 * r < a.M ? lo : 0.f, m0 + 2 * r + 1 < a.M ? hi : 0.f);
        }
        *(i32x4*)(a.vt + (size_t)(n - a.vt_col0) * a.vt_ld + m0) = e;
      }
    }
    return;
  }
#pragma unroll
  for (int it = 0; it < ITEMS; ++it) {
    const int idx = it * THREADS + tid, row = idx / CPR, ch = idx % CPR, m = m_blk + row, n = n_blk + ch * 8;
    const unsigned char* src = lds + row * SP + ch * 32;
    i32x2 r16[2];
    i32x4 r32[2];
    if (it >= PRE && res16) ask_res(r16, it);
    if (a.resid && a.resid_f32) {
      const float* p = (const float*)a.resid + (size_t)(m < a.M ? m : a.M - 1) * a.ldr;
      r32[0] = *(const i32x4*)(p + (n < a.N ? n : a.N - 4));
      r32[1] = *(const i32x4*)(p + (n + 4 < a.N ? n + 4 : a.N - 4));
    }
    i32x2 o[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      f32x4 v = *(const f32x4*)(src + 16 * q);
      if (a.act == 1) v = unpack_16x4<FP16>(pack_16x4<FP16>(v));  // the linear's 16-bit output, then the activation on it
      if (a.act) {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = gelu_tanh_rcp_f(v[j]);
      }
      o[q] = pack_16x4<FP16>(v);
      if (a.resid) {
        const f32x4 r = a.resid_f32 ? f32x4{__int_as_float(r32[q][0]), __int_as_float(r32[q][1]), __int_as_float(r32[q][2]), __int_as_float(r32[q][3])}
                                    : unpack_16x4<FP16>(it < PRE ? pre[it < PRE ? it : 0][q] : r16[q]);
        o[q] = pack_16x4<FP16>(unpack_16x4<FP16>(o[q]) + r);
      }
    }
    if (m >= a.M || n >= a.N) continue;
    u16* dst = a.y + (size_t)m * a.ldy + n;
    if (n + 8 <= a.N) *(i32x4*)dst = i32x4{o[0][0], o[0][1], o[1][0], o[1][1]};
    else *(i32x2*)dst = o[0];  // N % 8 == 4: the row's last four columns
  }
  if (a.vt && n_blk + BN * 32 > a.vt_col0) {
    // value columns of a packed q|k|v projection, also written transposed for the attention kernel (no activation or
    // residual in this form): eight consecutive rows of a column per 16-byte store, four stores in a row.  The rows of
    // an m tile belong to one problem (vt_rows is a multiple of 32); rows past M are written as zeros.
#pragma unroll 2
    for (int it = tid; it < BM * 4 * BN * 32; it += THREADS) {
      const int col = (it >> 2) % (BN * 32), rg = (it / (BN * 128)) * 4 + (it & 3);
      const int n = n_blk + col, m0 = m_blk + 8 * rg;
      if (n < a.vt_col0 || n >= a.N || m0 >= a.M) continue;
      i32x4 e;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float lo = *(const float*)(lds + (8 * rg + 2 * r) * SP + col * 4), hi = *(const float*)(lds + (8 * rg + 2 * r + 1) * SP + col * 4);
        const float l = m0 + 2 * r < a.M ? lo : 0.f, h = m0 + 2 * r + 1 < a.M ? hi : 0.f;
        e[r] = (int)(FP16 ? pack_f16x2(l, h) : pack_bf16x2(l, h));
      }
      const int prob = a.vt_rows ? m0 / a.vt_rows : 0, key0 = a.vt_rows ? m0 % a.vt_rows : m0;
      *(i32x4*)(a.vt + (size_t)prob * a.vt_bs + (size_t)(n - a.vt_col0) * a.vt_ld + key0) = e;
    }
  }
}

template <int BM, int BN, int WGM, int WGN, int NS, int OCC, bool ROPE>
int launch(const GemmArgs& a, hipStream_t st) {
  constexpr int NW = WGM * WGN;
  const int nblk_m = (a.M + BM * 32 - 1) / (BM * 32);
  const int nblk_n = (a.ntiles + BN - 1) / BN;
  const int ngroups = nblk_n * a.ksplit;
  const int by_rows = a.M > a.N;
  const unsigned blocks = blocks_of(nblk_m, ngroups);
  if (a.rope_pos) {
    if constexpr (ROPE) {
      if (a.f16) return -1;
      hipLaunchKernelGGL((bf16w_wide_kernel<BM, BN, WGM, WGN, NS, OCC, false, true>), dim3(blocks), dim3(2 * NW * 64), 0, st, a, nblk_m, ngroups, by_rows);
      return hipGetLastError() == hipSuccess ? 0 : -3;
    } else {
      return -1;
    }
  }
  if (a.f16)
    hipLaunchKernelGGL((bf16w_wide_kernel<BM, BN, WGM, WGN, NS, OCC, true>), dim3(blocks), dim3(2 * NW * 64), 0, st, a, nblk_m, ngroups, by_rows);
  else
    hipLaunchKernelGGL((bf16w_wide_kernel<BM, BN, WGM, WGN, NS, OCC, false>), dim3(blocks), dim3(2 * NW * 64), 0, st, a, nblk_m, ngroups, by_rows);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // namespace

int tk_launch_bf16w_wide(const GemmArgs& a, int tile, hipStream_t st) {
  switch (tile) {
    case 42: return launch<4, 8, 1, 4, 3, 1, true>(a, st);
    case 41: return launch<4, 4, 2, 2, 2, 2, false>(a, st);
    case 32: return launch<3, 8, 1, 4, 3, 1, true>(a, st);
    case 31: return launch<3, 4, 1, 4, 5, 1, false>(a, st);
    case 22: return launch<2, 8, 1, 4, 4, 1, true>(a, st);
    case 21: return launch<2, 4, 2, 2, 3, 2, false>(a, st);
    case 12: return launch<1, 8, 1, 4, 4, 1, true>(a, st);
    case 11: return launch<1, 4, 1, 4, 4, 2, false>(a, st);
    case 606: return launch<6, 6, 2, 2, 3, 1, false>(a, st);
    case 404: return launch<4, 4, 2, 2, 4, 1, true>(a, st);
    case 406: return launch<4, 6, 2, 2, 3, 1, false>(a, st);
    case 204: return launch<2, 4, 2, 2, 6, 1, true>(a, st);
    case 202: return launch<2, 2, 2, 2, 5, 2, false>(a, st);
    case 403: return launch<4, 3, 4, 1, 5, 1, false>(a, st);
  }
  return -1;
}
