// fp8-weight GEMM for many rows (the VLM prefill) on gfx950: the weight-only form of pipe_fp8.h, a kernel of its own for the
// largest grids, and the row norm in front of them.
// Measured (us, cold weights, graph replay; before: weights straight into the registers of four multiplying waves): the
// gated block 2048 -> 16384 -> 2048 at 288 / 320 / 555 / 712 / 968 rows 94 -> 78, 100 -> 87, 132 -> 129, 153 -> 149, 189 ->
// 187; 960 -> 2560 -> 960 at 305 / 600 rows 41 -> 24, 42 -> 29.
#include <atomic>

#include "pipe_fp8.h"

namespace {
using pipe::lds_barrier;
using pipe::wide_ep_pitch;
using pipe::wide_epilogue;

constexpr int NT = pipe::WIDE_NT;  // n tiles per wave
constexpr int NW = 4;              // waves per block
constexpr int RK = 2;              // k tiles per round

// Grids that cover the device twice over (from 385 rows of the gated 2048 -> 2 x 16384 launch): there the power of the
// operands' way decides the matrix pipes' clock, and the two kernels below, whose weights go through registers, are about level
// with pipe_fp8.h's.  This one where 64-row blocks waste the least: 555 / 640 / 800 rows 79 / 83 / 110 us against 77 / 79 / 106
// of its 128 x 128 blocks, all shapes timed in turn on one card; on another 555 rows 81 against 83 - 88.
// A block of four waves owns 64 rows x 256 packed columns, two blocks a CU (they cover each other's first loads and
// epilogue); wave w owns n tiles 2w, 2w + 1 for all rows, its weights straight from memory into its registers; a round's
// activations are staged once per block through LDS.  EPI: 0 plain, 1 gated.  PF: rounds in flight (even: round r uses LDS
// buffer r % 2).
template <int EPI, int MT, int PF, int OCC>
__global__ __launch_bounds__(NW * 64, OCC) void fp8w_wide_kernel(GemmArgs a, int nblk_m, int ngroups) {
  constexpr int ROWS = MT * 32;
  constexpr int ROWB = RK * 64;            // bytes of one staged activation row per round
  constexpr int PITCH = ROWB + 16;         // conflict-free 16-byte operand reads, 16-byte aligned
  constexpr int XBUF = ROWS * PITCH;
  constexpr int PPR = ROWB / 16;           // 16-byte pieces per staged row
  constexpr int XPT = ROWS * PPR / (NW * 64);
  constexpr int EPB = NW * 32 * ((EPI == 0 ? NT * 32 : 32) * 2 + 16);  // the epilogue's per-wave tiles
  __shared__ __align__(16) unsigned char lds[2 * XBUF > EPB ? 2 * XBUF : EPB];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5;
  const int l32 = lane & 31;

  // slot s of XCD x (blocks are dealt to the 8 XCDs round-robin) -> group (s / nblk_m) * 8 + x, m block
  // s % nblk_m: the nblk_m blocks of a group (same weights) run back to back on one XCD
  const unsigned id = blockIdx.x;
  const unsigned slot = id >> 3;
  const int mblock = (int)(slot % (unsigned)nblk_m);
  const int group = (int)((slot / (unsigned)nblk_m) * 8 + (id & 7));
  if (group >= ngroups) return;
  const int nblk = group;
  const int nrounds = (a.KT + RK - 1) / RK;

  const int strip = nblk * NW + wave;  // this wave's pair of packed n tiles
  const uint8_t* wbase[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    int ntg = strip * NT + nt;
    if (ntg > a.ntiles - 1) ntg = a.ntiles - 1;  // overhanging tiles are computed on valid data, never stored
    wbase[nt] = a.w + ((size_t)ntg * a.KT) * 1024 + lane * 16;
  }

  const char* xsrc[XPT];
  int xcol[XPT], xdst[XPT];
#pragma unroll
  for (int i = 0; i < XPT; ++i) {
    const int p = tid + i * NW * 64;
    const int r = p / PPR, c = p % PPR;
    int m = mblock * ROWS + r;
    if (m > a.M - 1) m = a.M - 1;  // rows past M: valid data, never stored
    xsrc[i] = (const char*)a.x + (size_t)m * a.ldx * 2;
    xcol[i] = c * 8;
    xdst[i] = r * PITCH + c * 16;
  }

  f32x16 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[mt][nt][i] = 0.f;

  struct WFrag {
    i32x4 w[RK][NT];
  };
  struct XFrag {
    i32x4 v[XPT];
  };
  // One piece of each kind of work, so that a round can deal them out between its matrix instructions: a wave
  // cannot issue anything while it waits for the matrix pipe to take its next instruction, so whatever stands
  // between two groups of matrix instructions in program order runs with the pipe empty.
  auto wload1 = [&](WFrag& f, int r, int j, int nt) {  // k tile j of round r, n tile nt: one 1 KiB tile
    int kt = r * RK + j;
    if (kt > a.KT - 1) kt = a.KT - 1;  // its activation columns are zeroed
    f.w[j][nt] = *(const i32x4*)(wbase[nt] + (size_t)kt * 1024);
  };
  auto xload1 = [&](XFrag& f, int r, int i) {
    int k = r * RK * 32 + xcol[i];
    if (k > a.K - 8) k = a.K - 8;
    f.v[i] = *(const i32x4*)(xsrc[i] + (size_t)k * 2);
  };
  auto xstore1 = [&](const XFrag& f, int r, int b, int i) {
    const i32x4 z = {0, 0, 0, 0};
    *(i32x4*)(lds + b * XBUF + xdst[i]) = r * RK * 32 + xcol[i] < a.K ? f.v[i] : z;
  };
  // operand fragments and converted weights of two k tiles: while the MFMAs of one k tile run, the LDS reads and
  // the e4m3 -> bf16 conversions of the next one are issued between them
  i32x4 xa[2][MT][2];
  bf16x8 wb[2][NT][2];
  auto xread1 = [&](int set, int b, int j, int u) {  // u in [0, 2*MT): k step u%2 of m tile u/2, k tile j
    xa[set][u / 2][u % 2] = *(const i32x4*)(lds + b * XBUF + ((u / 2) * 32 + l32) * PITCH + (j * 32 + 16 * half) * 2 + 16 * (u % 2));
  };
  auto wcvt1 = [&](int set, const WFrag& f, int j, int q) {  // q in [0, 2*NT): k step q%2 of n tile q/2
    wb[set][q / 2][q % 2] = fp8x8_to_bf16x8(f.w[j][q / 2][2 * (q % 2)], f.w[j][q / 2][2 * (q % 2) + 1]);
  };
  auto mma1 = [&](int set, int t) {  // t in [0, 2*MT*NT): k step, m tile, n tile
    const int h2 = t / (MT * NT), mt = (t / NT) % MT, nt = t % NT;
    acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wb[set][nt][h2], as_bf16x8(xa[set][mt][h2]), acc[mt][nt], 0, 0, 0);
  };
  static_assert(RK == 2 && PF % 2 == 0, "a round is two phases; buffer parity follows the pipeline slot");

  // PF rounds in flight; every load is unconditional (clamped addresses; columns past the block's k range are
  // zeroed when staged), so the loop bodies have no branch and the compiler keeps precise wait counts.  Round r,
  // phase A: multiplies k tile 0 while k tile 1's operands are fetched from LDS and its weights converted (their
  // registers are refilled for round r+PF right after), and round r+1 is staged into the other LDS buffer; then
  // the round's only barrier (a wave can write buffer b for round r+2 only after every wave has passed the barrier
  // of round r+1, i.e. has its round-r operands in registers); phase B: fetches round r+1's first operands,
  // converts its first weights (and refills their registers) and multiplies k tile 1.  Each of a phase's
  // 2*MT*NT matrix instructions is followed by its share of the other work, fenced so that the order stands:
  // reads and conversions in the first half of the slots, the loads that refill converted registers in the second.
  constexpr int SLOTS = 2 * MT * NT;
  constexpr int HS = SLOTS / 2;
  static_assert(2 * MT <= SLOTS && 2 * NT <= HS && NT <= HS && XPT <= HS, "the pieces fit the slots");
  WFrag wbuf[PF];
  XFrag xbuf[PF];
#pragma unroll
  for (int p = 0; p < PF; ++p) {
#pragma unroll
    for (int i = 0; i < XPT; ++i) xload1(xbuf[p], p, i);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      wload1(wbuf[p], p, 0, nt);
      wload1(wbuf[p], p, 1, nt);
    }
  }
#pragma unroll
  for (int i = 0; i < XPT; ++i) xstore1(xbuf[0], 0, 0, i);
#pragma unroll
  for (int i = 0; i < XPT; ++i) xload1(xbuf[0], PF, i);
  lds_barrier();
#pragma unroll
  for (int u = 0; u < 2 * MT; ++u) xread1(0, 0, 0, u);
#pragma unroll
  for (int q = 0; q < 2 * NT; ++q) wcvt1(0, wbuf[0], 0, q);
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) wload1(wbuf[0], PF, 0, nt);
  auto round = [&](int p, int r) {
    const int b = p & 1;  // == r & 1: rounds advance PF at a time
    const int pn = (p + 1) % PF;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
      mma1(0, i);
#pragma unroll
      for (int u = 0; u < 2 * MT; ++u)
        if (u * SLOTS / (2 * MT) == i) xread1(1, b, 1, u);
#pragma unroll
      for (int q = 0; q < 2 * NT; ++q)
        if (q * HS / (2 * NT) == i) wcvt1(1, wbuf[p], 1, q);
#pragma unroll
      for (int x = 0; x < XPT; ++x) {
        if (x * HS / XPT == i) xstore1(xbuf[pn], r + 1, b ^ 1, x);
        if (HS + x * HS / XPT == i) xload1(xbuf[pn], r + 1 + PF, x);
      }
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        if (HS + nt * HS / NT == i) wload1(wbuf[p], r + PF, 1, nt);  // converted above
      __builtin_amdgcn_sched_barrier(0);
    }
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
      mma1(1, i);
#pragma unroll
      for (int u = 0; u < 2 * MT; ++u)
        if (u * SLOTS / (2 * MT) == i) xread1(0, b ^ 1, 0, u);
#pragma unroll
      for (int q = 0; q < 2 * NT; ++q)
        if (q * HS / (2 * NT) == i) wcvt1(0, wbuf[pn], 0, q);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        if (HS + nt * HS / NT == i) wload1(wbuf[pn], r + 1 + PF, 0, nt);  // converted above
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  {
    int it = 0;
    for (; it + PF <= nrounds; it += PF) {
#pragma unroll
      for (int p = 0; p < PF; ++p) round(p, it + p);
    }
    const int rem = nrounds - it;  // in [0, PF)
#pragma unroll
    for (int q = 0; q < PF - 1; ++q)
      if (q < rem) round(q, it + q);  // block-uniform
  }

  // ---- epilogue ----
  constexpr int EP = wide_ep_pitch(EPI);
  static_assert(NW * 32 * EP == EPB, "the epilogue tiles fit the LDS array");
  if (a.vec16) lds_barrier();  // every wave has left the staged activations behind
  wide_epilogue<pipe::BF16_FP8, EPI, MT>(a, acc, lds + wave * 32 * EP, mblock * ROWS, strip, lane);
}

// The same where taller blocks waste no more rows: eight waves own 2*WM*32 rows x 256 packed columns, with both operands of a
// round staged through registers and LDS: wave (wm, wn) = (wave / 4, wave % 4) owns rows wm*WM*32 .. of the block and the n
// tile pair wn; a weight tile is fetched and converted to bf16 once per block (512 / 712 / 968 rows 61 / 93 / 118 us against 64 /
// 93 / 122 of the best shape of pipe_fp8.h's kernel).  A round is four k steps of
// 16; operand registers of step s + 1 are read while step s multiplies; one barrier per round, before its last step:
// by then every wave has read the round's operands out of buffer b and written its share of round r + 1 into b ^ 1.
//   staging per thread and round: WM 16-byte pieces of x, 2 pieces of 16 fp8 weights (wave (wm, wn): k tile wm of
//   the round for its own n tile pair); each piece is requested again for round r + 1 + PF right after it is stored.
// LDS: 2 x (2*WM*32 rows x 144 B + 32 KiB of bf16 weight tiles) = 136 KB (WM = 4) / 118 KB (WM = 3), dynamic.
template <int EPI, int WM, int PF>
__global__ __launch_bounds__(512, 1) void fp8w_tile_kernel(GemmArgs a, int nblk_m, int ngroups) {
  constexpr int NWV = 8;
  constexpr int ROWS = 2 * WM * 32;
  constexpr int ROWB = RK * 64;
  constexpr int PITCH = ROWB + 16;
  constexpr int XBUF = ROWS * PITCH;
  constexpr int WBUF = NW * NT * RK * 2048;  // bf16 tiles of the round: [n tile][k tile][k step][lane][16 B]
  constexpr int STAGE = XBUF + WBUF;
  constexpr int XPT = ROWS * (ROWB / 16) / (NWV * 64);
  constexpr int SL = WM * NT;  // matrix instructions per k step
  static_assert(XPT == WM && NWV * 32 * wide_ep_pitch(EPI) <= 2 * STAGE, "staging and epilogue tiles fit");
  extern __shared__ __align__(16) unsigned char lds[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  const int half = lane >> 5;
  const int l32 = lane & 31;

  const unsigned id = blockIdx.x;
  const unsigned slot = id >> 3;
  const int mblock = (int)(slot % (unsigned)nblk_m);
  const int group = (int)((slot / (unsigned)nblk_m) * 8 + (id & 7));
  if (group >= ngroups) return;
  const int nblk = group;
  const int nrounds = (a.KT + RK - 1) / RK;

  const int strip = nblk * NW + wn;
  const uint8_t* wbase[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    int ntg = strip * NT + nt;
    if (ntg > a.ntiles - 1) ntg = a.ntiles - 1;
    wbase[nt] = a.w + ((size_t)ntg * a.KT) * 1024 + lane * 16;
  }
  const char* xsrc[XPT];
  const int xcol = (tid & 7) * 8;
  const int xdst = (tid >> 3) * PITCH + (tid & 7) * 16;  // piece i: + i * 64 rows
#pragma unroll
  for (int i = 0; i < XPT; ++i) {
    int m = mblock * ROWS + i * 64 + (tid >> 3);
    if (m > a.M - 1) m = a.M - 1;
    xsrc[i] = (const char*)a.x + (size_t)m * a.ldx * 2;
  }

  f32x16 acc[WM][NT];
#pragma unroll
  for (int mt = 0; mt < WM; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[mt][nt][i] = 0.f;

  struct Stg {
    i32x4 x[XPT];
    i32x4 w[NT];
  };
  auto xload1 = [&](Stg& f, int r, int i) {
    int k = r * RK * 32 + xcol;
    if (k > a.K - 8) k = a.K - 8;
    f.x[i] = *(const i32x4*)(xsrc[i] + (size_t)k * 2);
  };
  auto wload1 = [&](Stg& f, int r, int nt) {
    int kt = r * RK + wm;
    if (kt > a.KT - 1) kt = a.KT - 1;  // its activation columns are zeroed
    f.w[nt] = *(const i32x4*)(wbase[nt] + (size_t)kt * 1024);
  };
  auto xstore1 = [&](const Stg& f, int r, int b, int i) {
    const i32x4 z = {0, 0, 0, 0};
    *(i32x4*)(lds + b * STAGE + xdst + i * 64 * PITCH) = r * RK * 32 + xcol < a.K ? f.x[i] : z;
  };
  auto wstore1 = [&](const Stg& f, int b, int q) {  // q in [0, 2*NT): k step q%2 of n tile q/2
    *(bf16x8*)(lds + b * STAGE + XBUF + ((((wn * NT + q / 2) * RK + wm) * 2 + q % 2) * 64 + lane) * 16) =
        fp8x8_to_bf16x8(f.w[q / 2][2 * (q % 2)], f.w[q / 2][2 * (q % 2) + 1]);
  };
  i32x4 fa[2][WM];
  bf16x8 fb[2][NT];
  auto fread1 = [&](int b, int s, int u) {  // operand u of k step s: u < WM the m tiles, then the n tiles
    const int set = s & 1, j = s >> 1, h2 = s & 1;
    if (u < WM)
      fa[set][u] = *(const i32x4*)(lds + b * STAGE + ((wm * WM + u) * 32 + l32) * PITCH + (j * 32 + 16 * half) * 2 + 16 * h2);
    else
      fb[set][u - WM] = *(const bf16x8*)(lds + b * STAGE + XBUF + ((((wn * NT + u - WM) * RK + j) * 2 + h2) * 64 + lane) * 16);
  };
  auto mma1 = [&](int set, int t) {
    const int mt = t / NT, nt = t % NT;
    acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[set][nt], as_bf16x8(fa[set][mt]), acc[mt][nt], 0, 0, 0);
  };

  Stg stg[PF];
#pragma unroll
  for (int q = 0; q < PF; ++q) {
#pragma unroll
    for (int i = 0; i < XPT; ++i) xload1(stg[q], q, i);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) wload1(stg[q], q, nt);
  }
#pragma unroll
  for (int i = 0; i < XPT; ++i) {
    xstore1(stg[0], 0, 0, i);
    xload1(stg[0], PF, i);
  }
#pragma unroll
  for (int q = 0; q < 2 * NT; ++q) wstore1(stg[0], 0, q);
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) wload1(stg[0], PF, nt);
  lds_barrier();
#pragma unroll
  for (int u = 0; u < WM + NT; ++u) fread1(0, 0, u);

  auto round = [&](int p, int r) {  // p = r % 2 (the LDS buffer); round r + 1 waits in stg[(p + 1) % PF]
    const int b = p & 1;
    Stg& nx = stg[(p + 1) % PF];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      if (s == 3) lds_barrier();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < SL; ++i) {
        mma1(s & 1, i);
        if (i < WM + NT) fread1(s == 3 ? b ^ 1 : b, (s + 1) & 3, i);
        if (s == 0) {
#pragma unroll
          for (int x = 0; x < XPT; ++x)
            if (x * SL / XPT + 1 == i) {
              xstore1(nx, r + 1, b ^ 1, x);
              xload1(nx, r + 1 + PF, x);
            }
        }
        if (s == 1) {
#pragma unroll
          for (int q = 0; q < 2 * NT; ++q)
            if (q * SL / (2 * NT) + 1 == i) {
              wstore1(nx, b ^ 1, q);
              if (q % 2 == 1) wload1(nx, r + 1 + PF, q / 2);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  {
    int it = 0;
    for (; it + 2 <= nrounds; it += 2) {
      round(0, it);
      round(1, it + 1);
    }
    if (it < nrounds) round(0, it);
  }

  constexpr int EP = wide_ep_pitch(EPI);
  if (a.vec16) lds_barrier();
  wide_epilogue<pipe::BF16_FP8, EPI, WM>(a, acc, lds + wave * 32 * EP, mblock * ROWS + wm * WM * 32, strip, lane);
}

// One block per row: out = bf16 norm of the bf16 row, with the rounding points of the skinny
// kernel's prologues: RMSNorm bf16(w * bf16(x * rstd)); adaptive bf16((x * rstd) * (1 + scale) + shift).
// A thread's first piece of the row and the norm's operands for it are requested together up front and stay in
// registers (rows up to 2048 columns need nothing else): one memory round trip before the store, not three.
__global__ __launch_bounds__(256) void norm_rows_kernel(NormRowsArgs a) {
  __shared__ float part[4];
  const int tid = threadIdx.x;
  const char* row = (const char*)a.x + (size_t)blockIdx.x * a.ldx * 2;
  const int pieces = a.K / 8;
  const int p0 = tid < pieces ? tid : pieces - 1;  // past the row: a valid piece, not used
  union { i32x4 v; bf16x2 h[4]; unsigned u[4]; } x0;
  x0.v = *(const i32x4*)(row + (size_t)p0 * 16);
  union { i32x4 v[2]; float f[8]; } sc0, sh0;
  union { i32x4 v; unsigned u[4]; } nw0;
  if (a.ada_scale) {
    sc0.v[0] = *(const i32x4*)(a.ada_scale + p0 * 8);
    sc0.v[1] = *(const i32x4*)(a.ada_scale + p0 * 8 + 4);
    sh0.v[0] = *(const i32x4*)(a.ada_shift + p0 * 8);
    sh0.v[1] = *(const i32x4*)(a.ada_shift + p0 * 8 + 4);
  } else {
    nw0.v = *(const i32x4*)(a.norm_w + p0 * 8);
  }
  float ss0 = 0.f, ss1 = 0.f;
  auto square = [&](const bf16x2* h) {
    ss0 = __builtin_amdgcn_fdot2_f32_bf16(h[0], h[0], ss0, false);
    ss1 = __builtin_amdgcn_fdot2_f32_bf16(h[1], h[1], ss1, false);
    ss0 = __builtin_amdgcn_fdot2_f32_bf16(h[2], h[2], ss0, false);
    ss1 = __builtin_amdgcn_fdot2_f32_bf16(h[3], h[3], ss1, false);
  };
  if (tid < pieces) square(x0.h);
  for (int p = tid + 256; p < pieces; p += 256) {
    union { i32x4 v; bf16x2 h[4]; } xu;
    xu.v = *(const i32x4*)(row + (size_t)p * 16);
    square(xu.h);
  }
  float ss = ss0 + ss1;
  ss = wave_sum(ss);
  if ((tid & 63) == 0) part[tid >> 6] = ss;
  __syncthreads();
  ss = (part[0] + part[1]) + (part[2] + part[3]);
  const float rstd = rsqrtf(ss / (float)a.K + a.eps);
  char* dst = (char*)a.out + (size_t)blockIdx.x * a.ldo * 2;
  auto norm_piece = [&](const unsigned* xu, const float* sc, const float* sh, const unsigned* nw) {
    union { i32x4 v; unsigned u[4]; } o;
    if (a.ada_scale) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x0f = __uint_as_float(xu[e] << 16), x1f = __uint_as_float(xu[e] & 0xffff0000u);
        const float y0 = add_rn(mul_rn(mul_rn(x0f, rstd), add_rn(1.0f, sc[2 * e])), sh[2 * e]);
        const float y1 = add_rn(mul_rn(mul_rn(x1f, rstd), add_rn(1.0f, sc[2 * e + 1])), sh[2 * e + 1]);
        o.u[e] = pack_bf16x2(y0, y1);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const unsigned u = pack_bf16x2(__uint_as_float(xu[e] << 16) * rstd, __uint_as_float(xu[e] & 0xffff0000u) * rstd);
        o.u[e] = pack_bf16x2(__uint_as_float(nw[e] << 16) * __uint_as_float(u << 16),
                             __uint_as_float(nw[e] & 0xffff0000u) * __uint_as_float(u & 0xffff0000u));
      }
    }
    return o.v;
  };
  if (tid < pieces) *(i32x4*)(dst + (size_t)tid * 16) = norm_piece(x0.u, sc0.f, sh0.f, nw0.u);
  for (int p = tid + 256; p < pieces; p += 256) {
    union { i32x4 v; unsigned u[4]; } xu, nw;
    union { i32x4 v[2]; float f[8]; } sc, sh;
    xu.v = *(const i32x4*)(row + (size_t)p * 16);
    if (a.ada_scale) {
      sc.v[0] = *(const i32x4*)(a.ada_scale + p * 8);
      sc.v[1] = *(const i32x4*)(a.ada_scale + p * 8 + 4);
      sh.v[0] = *(const i32x4*)(a.ada_shift + p * 8);
      sh.v[1] = *(const i32x4*)(a.ada_shift + p * 8 + 4);
    } else {
      nw.v = *(const i32x4*)(a.norm_w + p * 8);
    }
    *(i32x4*)(dst + (size_t)p * 16) = norm_piece(xu.u, sc.f, sh.f, nw.u);
  }
}

template <int EPI>
int launch_wide(const GemmArgs& a, hipStream_t st) {
  const int nblk_m = (a.M + 63) / 64, nblk_n = (a.ntiles + NW * NT - 1) / (NW * NT);
  hipLaunchKernelGGL((fp8w_wide_kernel<EPI, 2, 4, 2>), dim3((unsigned)((nblk_n + 7) / 8) * 8u * (unsigned)nblk_m), dim3(NW * 64), 0, st, a, nblk_m, nblk_n);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

template <int EPI, int WM>
int launch_tile(const GemmArgs& a, hipStream_t st) {
  constexpr int LDS = 2 * (2 * WM * 32 * (RK * 64 + 16) + NW * NT * RK * 2048);
  static std::atomic<int> raised{0};  // more LDS than a launch gets by default: raise the kernel's limit once per process
  if (!raised.load(std::memory_order_acquire)) {
    if (hipFuncSetAttribute((const void*)fp8w_tile_kernel<EPI, WM, 1>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) != hipSuccess) return -3;
    raised.store(1, std::memory_order_release);
  }
  const int nblk_m = (a.M + 2 * WM * 32 - 1) / (2 * WM * 32), nblk_n = (a.ntiles + NW * NT - 1) / (NW * NT);
  hipLaunchKernelGGL((fp8w_tile_kernel<EPI, WM, 1>), dim3((unsigned)((nblk_n + 7) / 8) * 8u * (unsigned)nblk_m), dim3(512), LDS, st, a, nblk_m, nblk_n);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // namespace

// tile: an id of kWideTiles (tk_api.hip); 28, 68, 88: the kernels of this file, 64, 192 or 256 rows (no K split)
int tk_launch_gemm_wide(const GemmArgs& a, int tile, hipStream_t st) {
  using namespace pipe;
  switch (tile) {
    case 28: return a.s1 ? launch_wide<1>(a, st) : launch_wide<0>(a, st);
    case 68: return a.s1 ? launch_tile<1, 3>(a, st) : launch_tile<0, 3>(a, st);
    case 88: return a.s1 ? launch_tile<1, 4>(a, st) : launch_tile<0, 4>(a, st);
    case 404: return launch_fp8_pipe<BF16_FP8, 4, 4, 2, 2, 3, 2>(a, st);
    case 304: return launch_fp8_pipe<BF16_FP8, 3, 4, 1, 4, 3, 2>(a, st);
    case 408: return launch_fp8_pipe<BF16_FP8, 4, 8, 2, 2, 4, 1>(a, st);
    case 208: return launch_fp8_pipe<BF16_FP8, 2, 8, 1, 4, 3, 2>(a, st);
    case 204: return launch_fp8_pipe<BF16_FP8, 2, 4, 2, 2, 4, 2>(a, st);
  }
  return -1;
}

int tk_launch_norm_rows(NormRowsArgs a, hipStream_t st) {
  hipLaunchKernelGGL(norm_rows_kernel, dim3(a.M), dim3(256), 0, st, a);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}
