// W8A8 tier of the VLM prefill MLP on gfx950: per-token activation quantisation and the fp8 x fp8 GEMM.
//
//   quant_act_rows_kernel   x[M,K] bf16 -> a8[M,K] e4m3fn, sa[M] fp32 with sa = amax_k|x| / 448 and
//                           a8 = RNE(x / sa) in fp32 (one rounding); a row whose scale is 0 (all zeros; bf16 mode:
//                           |x| up to 448 * 2^-134 as well, whose scale rounds to 0) gives zero codes.
//   fp8_pipe_kernel<FP8>    (pipe_fp8.h) y[M,N] = bf16((a8 . W8^T) * sa[m] * sw[n]) on v_mfma_f32_32x32x64_f8f6f4 (e4m3 x
//                           e4m3, fp32 accumulate, 64 k per instruction).  The order of k inside an instruction is the
//                           same permutation for both operands (bytes 0-15 of a lane: k tile 2s, bytes 16-31: k tile
//                           2s+1), which a dot product does not see.  Measured (us, before: weights straight into the
//                           registers of four multiplying waves): the whole block 2048 -> 16384 -> 2048, quantisations
//                           included, at 256 / 288 / 555 / 712 / 968 rows 63 -> 60, 82 -> 71, 105 -> 96, 124 -> 110, 151 -> 135.
#include "pipe_fp8.h"

namespace {

// One block per row.  MODE 0: sa = amax / 448 (fp32), a8 = RNE(x / sa) from fp32 -- one rounding.
// MODE 1: the arithmetic of a torch expression on bf16 tensors, `s = x.abs().max() / 448` (a bf16 value) and
// `(x / s).to(float8_e4m3fn)` (quotient rounded to bf16, then to fp8): sa = float(bf16(amax / 448)).
// Bound: memory (a 555 x 16384 row block is 18 MB in, 9 MB out) once the loads of a row are all on their way together (NP of
// them a thread, none under a branch: at the join behind one each would be waited for) and a quotient costs four
// instructions (bf16 mode, one division a value before): 555 rows of 2048 / 16384 columns 4.4 -> 3.3 / 10.3 -> 7.1 us, 968 of 16384
// 14.6 -> 10.4.
constexpr int kQuantMaxPieces = 8;  // 16-byte pieces of a row per thread: K <= 8 * 256 * 8 = 16384
template <int NP, bool BF16_MODE>
__global__ __launch_bounds__(256) void quant_act_rows_kernel(QuantActArgs a) {
  __shared__ float part[4];
  const int tid = threadIdx.x;
  const char* row = (const char*)a.x + (size_t)blockIdx.x * a.ldx * 2;
  const int pieces = a.K / 8;
  i32x4 v[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int p = tid + i * 256 < pieces ? tid + i * 256 : pieces - 1;  // past the row: a piece of it again
    v[i] = *(const i32x4*)(row + (size_t)p * 16);
  }
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < NP; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const unsigned u = (unsigned)v[i][e];
      amax = fmaxf(amax, fmaxf(fabsf(__uint_as_float(u << 16)), fabsf(__uint_as_float(u & 0xffff0000u))));
    }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o));
  if ((tid & 63) == 0) part[tid >> 6] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
  float sa = amax / 448.0f;
  if (BF16_MODE) sa = round_bf16(sa);
  if (tid == 0) a.sa[blockIdx.x] = sa;
  // The IEEE quotient, as the elementwise reference computes it, from the correctly rounded reciprocal: one product and one
  // correction by the exact remainder are again correctly rounded (Markstein).  The sign is the numerator's (the remainder
  // of -0 is +0).  Scales whose reciprocal or remainders would leave the range of normal numbers take the division.
  const float inv = 1.0f / sa;
  unsigned char* dst = (unsigned char*)a.a8 + (size_t)blockIdx.x * a.lda;
  auto codes = [&](auto quotient) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int p = tid + i * 256;
      if (p >= pieces) continue;
      float q[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const unsigned u = (unsigned)v[i][e >> 1];
        q[e] = quotient(__uint_as_float((e & 1) ? (u & 0xffff0000u) : (u << 16)));
        if (BF16_MODE) q[e] = round_bf16(q[e]);
      }
      // four fp32 -> four e4m3fn (RNE, saturating at +-448) per conversion pair
      int lo = 0, hi = 0;
      lo = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], lo, false);
      lo = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], lo, true);
      hi = __builtin_amdgcn_cvt_pk_fp8_f32(q[4], q[5], hi, false);
      hi = __builtin_amdgcn_cvt_pk_fp8_f32(q[6], q[7], hi, true);
      *(i32x2*)(dst + (size_t)p * 8) = i32x2{lo, hi};
    }
  };
  // the row's choice in front of the loop: inside, every element carries both branches (1 x 15776, bf16 mode, 6.2 us instead of 3.8)
  if (sa >= 0x1p-80f && sa <= 0x1p+80f)
    codes([&](float x) {
      const float y = x * inv;
      return __builtin_copysignf(fmaf(fmaf(-sa, y, x), inv, y), x);
    });
  else
    codes([&](float x) { return sa == 0.f ? 0.f : x / sa; });
}

// Rows whose share of a compute unit comes out smallest in 64-row blocks, two a CU (577 .. 640, 769 .. 896 rows of the gated
// 2048 -> 2 x 16384 launch): 608 / 800 / 896 rows 58.1 / 74.6 / 77.3 us against 61.9 / 79.2 / 81.4 of fp8_pipe_kernel's
// blocks of 128 x 256, whose last generation is half empty there (graph replay, cold weights).  A block that also loads on waves of its own does not
// fit a CU twice: registers.
// A block of four waves owns 64 rows x 256 packed columns; wave w owns n tiles 2w, 2w + 1 for all rows, its weights straight from
// memory into its registers; a round's activations (128 columns) are staged once per block through LDS.  No K split.
template <int EPI>
__global__ __launch_bounds__(256, 2) void w8a8_wide_kernel(GemmArgs a, int nblk_m, int ngroups) {
  using namespace pipe;
  constexpr int MT = 2, NT = WIDE_NT, NW = 4;  // 32-row tiles of a block, n tiles of a wave, waves
  constexpr int RK = 4, PF = 3;                // k tiles of a round (two 64-wide product steps), rounds in flight
  constexpr int PITCH = RK * 32 + 16, XBUF = MT * 32 * PITCH;  // of the staged rows
  constexpr int PPR = RK * 2, XPT = MT * 32 * PPR / (NW * 64);  // 16-byte pieces per staged row, per thread
  constexpr int EPB = NW * 32 * wide_ep_pitch(EPI);
  __shared__ __align__(16) unsigned char lds[2 * XBUF > EPB ? 2 * XBUF : EPB];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5;
  const int l32 = lane & 31;

  // slot s of XCD x (blocks are dealt to the 8 XCDs round-robin) -> group (s / nblk_m) * 8 + x, m block s % nblk_m: the
  // nblk_m blocks of a group (same weights) run back to back on one XCD
  const unsigned slot = blockIdx.x >> 3;
  const int mblock = (int)(slot % (unsigned)nblk_m);
  const int nblk = (int)((slot / (unsigned)nblk_m) * 8 + (blockIdx.x & 7));
  if (nblk >= ngroups) return;
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
    const int p = tid + i * NW * 64, r = p / PPR, c = p % PPR;
    int m = mblock * MT * 32 + r;
    if (m > a.M - 1) m = a.M - 1;  // rows past M: valid data, never stored
    xsrc[i] = (const char*)a.x + (size_t)m * a.ldx;
    xcol[i] = c * 16;
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
  // One piece of each kind of work, so that a round can deal them out between its matrix instructions: a wave cannot issue
  // anything while it waits for the matrix pipe to take its next instruction.
  auto wload1 = [&](WFrag& f, int r, int st, int q) {  // q in [0, 2*NT): k tile 2*st + q/NT of round r, n tile q%NT
    const int j = 2 * st + q / NT, nt = q % NT;
    int kt = r * RK + j;
    if (kt > a.KT - 1) kt = a.KT - 1;  // its activation columns are zeroed
    f.w[j][nt] = *(const i32x4*)(wbase[nt] + (size_t)kt * 1024);
  };
  auto xload1 = [&](XFrag& f, int r, int i) {
    int k = r * RK * 32 + xcol[i];
    if (k > a.K - 16) k = a.K - 16;
    f.v[i] = *(const i32x4*)(xsrc[i] + k);
  };
  auto xstore1 = [&](const XFrag& f, int r, int b, int i) {
    const i32x4 z = {0, 0, 0, 0};
    *(i32x4*)(lds + b * XBUF + xdst[i]) = r * RK * 32 + xcol[i] < a.K ? f.v[i] : z;
  };
  i32x4 xa[2][MT][2];  // operands of the round's two steps, as the 16-byte halves they are read in
  auto xread1 = [&](int st, int b, int u) {  // u in [0, 2*MT): half u%2 of m tile u/2
    xa[st][u / 2][u % 2] = *(const i32x4*)(lds + b * XBUF + ((u / 2) * 32 + l32) * PITCH + st * 64 + 16 * half + 32 * (u % 2));
  };
  auto mma1 = [&](const WFrag& f, int st, int t) {  // t in [0, MT*NT): m tile t/NT, n tile t%NT
    const int mt = t / NT, nt = t % NT;
    const i32x4 wl = f.w[2 * st][nt], wh = f.w[2 * st + 1][nt], xl = xa[st][mt][0], xh = xa[st][mt][1];
    acc[mt][nt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(i32x8{wl[0], wl[1], wl[2], wl[3], wh[0], wh[1], wh[2], wh[3]},
                                                                  i32x8{xl[0], xl[1], xl[2], xl[3], xh[0], xh[1], xh[2], xh[3]},
                                                                  acc[mt][nt], 0, 0, 0, 0, 0, 0);
  };
  // PF rounds in flight, every load unconditional (clamped addresses; columns past K are zeroed when staged).  Round r,
  // phase A: multiplies step 0 while step 1's operands are fetched from LDS, round r+1 is staged into the other LDS buffer
  // and the weight registers that round r-1's step 1 has left are refilled; then the round's only barrier (a wave writes
  // buffer b for round r+2 only after every wave has passed the barrier of round r+1, with its round-r operands in
  // registers); phase B: fetches round r+1's first operands, multiplies step 1 and refills step 0's weight registers.  A
  // phase never reloads registers its own matrix instructions read.
  constexpr int SLOTS = MT * NT;
  static_assert(SLOTS == 2 * MT && SLOTS >= 2 * NT && 2 * XPT <= SLOTS, "one operand read per slot; the other pieces fit");
  WFrag wbuf[PF];
  XFrag xbuf[PF];
#pragma unroll
  for (int p = 0; p < PF; ++p) {
#pragma unroll
    for (int i = 0; i < XPT; ++i) xload1(xbuf[p], p, i);
#pragma unroll
    for (int q = 0; q < 2 * NT; ++q) {
      wload1(wbuf[p], p, 0, q);
      wload1(wbuf[p], p, 1, q);
    }
  }
#pragma unroll
  for (int i = 0; i < XPT; ++i) xstore1(xbuf[0], 0, 0, i);
#pragma unroll
  for (int i = 0; i < XPT; ++i) xload1(xbuf[0], PF, i);
  lds_barrier();
#pragma unroll
  for (int u = 0; u < 2 * MT; ++u) xread1(0, 0, u);
  auto round = [&](int p, int r) {
    const int b = r & 1;
    const int pn = (p + 1) % PF, pp = (p + PF - 1) % PF;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
      mma1(wbuf[p], 0, i);
      xread1(1, b, i);
      if (i < XPT) xstore1(xbuf[pn], r + 1, b ^ 1, i);
      if (i >= SLOTS - XPT) xload1(xbuf[pn], r + 1 + PF, i - (SLOTS - XPT));
      if (i < 2 * NT) wload1(wbuf[pp], r - 1 + PF, 1, i);  // the registers round r-1 finished with in its phase B
      __builtin_amdgcn_sched_barrier(0);
    }
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
      mma1(wbuf[p], 1, i);
      xread1(0, b ^ 1, i);
      if (i < 2 * NT) wload1(wbuf[p], r + PF, 0, i);  // step 0's registers: free since phase A
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int it = 0;
  for (; it + PF <= nrounds; it += PF) {
#pragma unroll
    for (int p = 0; p < PF; ++p) round(p, it + p);
  }
#pragma unroll
  for (int q = 0; q < PF - 1; ++q)
    if (q < nrounds - it) round(q, it + q);  // block-uniform

  if (a.vec16) lds_barrier();  // every wave has left the staged activations behind
  wide_epilogue<FP8, EPI, MT>(a, acc, lds + wave * 32 * wide_ep_pitch(EPI), mblock * MT * 32, strip, lane);
}

}  // namespace

int tk_quant_act_max_k() { return kQuantMaxPieces * 256 * 8; }

// tile: an id of kW8a8Tiles (tk_api.hip), or 28: w8a8_wide_kernel (no K split)
int tk_launch_w8a8_gemm(const GemmArgs& a, int tile, hipStream_t st) {
  using namespace pipe;
  switch (tile) {
    case 28: {
      const int nblk_m = (a.M + 63) / 64, nblk_n = (a.ntiles + 7) / 8;
      const dim3 grid((unsigned)((nblk_n + 7) / 8) * 8u * (unsigned)nblk_m), block(256);
      if (a.s1) hipLaunchKernelGGL(w8a8_wide_kernel<1>, grid, block, 0, st, a, nblk_m, nblk_n);
      else hipLaunchKernelGGL(w8a8_wide_kernel<0>, grid, block, 0, st, a, nblk_m, nblk_n);
      return hipGetLastError() == hipSuccess ? 0 : -3;
    }
    case 604: return launch_fp8_pipe<FP8, 6, 4, 2, 2, 4, 1>(a, st);
    case 414: return launch_fp8_pipe<FP8, 4, 4, 2, 2, 4, 1>(a, st);
    case 408: return launch_fp8_pipe<FP8, 4, 8, 2, 2, 3, 1>(a, st);
    case 204: return launch_fp8_pipe<FP8, 2, 4, 2, 2, 3, 2>(a, st);
  }
  return -1;
}

template <bool BF16_MODE>
static void launch_quant(int np, dim3 grid, dim3 block, const QuantActArgs& a, hipStream_t st) {
  if (np <= 1) hipLaunchKernelGGL((quant_act_rows_kernel<1, BF16_MODE>), grid, block, 0, st, a);
  else if (np <= 2) hipLaunchKernelGGL((quant_act_rows_kernel<2, BF16_MODE>), grid, block, 0, st, a);
  else if (np <= 4) hipLaunchKernelGGL((quant_act_rows_kernel<4, BF16_MODE>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((quant_act_rows_kernel<kQuantMaxPieces, BF16_MODE>), grid, block, 0, st, a);
}

int tk_launch_quant_act_rows(QuantActArgs a, hipStream_t st) {
  const int np = (a.K / 8 + 255) / 256;
  const dim3 grid(a.M), block(256);
  if (a.mode == 1) launch_quant<true>(np, grid, block, a, st);
  else launch_quant<false>(np, grid, block, a, st);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}
