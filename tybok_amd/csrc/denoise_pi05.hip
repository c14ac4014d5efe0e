// The pi0.5 flow-matching loop as ONE persistent launch: action embedding, every expert layer, final norm, action
// projection and Euler update of all steps.  Hand-offs, operand order and the bounded waits are those of persist.h.
//
// Bound: latency, then the bytes a compute unit takes in.  A step reads 397 MB of weights (80 us at 5 TB/s) and its
// eighteen layers are 108 dependent phases of 0.3 - 1.5 us of work each; as five launches a layer they took 47 us a layer.
// Here 256 resident blocks run the phases back to back: block (rt, c) works on 16 of the chunk's rows with column share c
// of 64.  Measured (50 action tokens, two cameras and 200 language tokens, 10 steps): the loop 8.5 -> 3.44 ms (19 us a layer;
// stamps of every block, mean: 0.6 - 1.5 us from a phase's result to the next one's first input, 0.6 - 1.5 us until all of a
// block's input is there, from there to the result 0.7 - 1.4 us); 0.8 MB through each compute unit.
//
//   step    E0  v = final_norm(x) . Wa^T + b, x_t += dt v         32 blocks per row group, one action column each
//           E1  hidden = x_t . Wi^T + b                           64 blocks, 16 columns each
//   layer   P1  q | k | v = ada(hidden) . W^T, rotary             one rotary pair of q tiles per block; blocks 0..7 also
//                                                                 one of k, 8..15 two tiles of v
//           P2  one head over an eighth of the keys               block 8 h + split: running maximum, sum, fp32 output
//           PC  the eight splits of a head into 32 columns        (a merge in P3 itself would read 8 x 64 KiB a block)
//           P3  hidden += gate * att . Wo^T                       16 columns
//           P4  h = gelu(g) * u of ada(hidden) . Wgu^T            four gate / up pairs of 16 columns
//           P5  hidden += gate * h . Wd^T                         16 columns
//
// Rows: 16 per block (a chunk of 50 is four groups).  32 rows would halve the weights a compute unit reads (336 KiB a
// layer) but double its activations (320 KiB, of which P5 alone 128), and those are in the chain.
// Place: blocks land round-robin on the eight XCDs, so block i = 64 rt + c puts the row groups' blocks of one column share
// on one XCD: the weights, which are too many for any cache above the XCD's, come there once for four blocks, and a
// key split for 32.  A row group on two XCDs of its own (hand-offs 0.3 us shorter) took 2 us a layer more.
// Weights and keys ahead: loads that the memory pipe still works on stand before the next hand-off's data, so each set is
// asked for where the fewest of them are on that path (the loop, us; first figure: as below).
//   * The keys at P1's end; the values behind the query's arrival in P2 3463 (behind P1's products 3489, at P1's end 3584; the
//     keys in front of P1's barrier 3707, at its input 3787).
//   * P3's weights at PC's input 3538 (in P2 3600).  P4's: half at PC's end, half at P3's input 3493 (all at PC's end 3558, at
//     P3's input 3668; the first half at PC's input 3659).
//   * P5's between P4's products and the barrier of its reduction 3558 (behind it 3714, at P4's input 3596).
//   * P1's at P4's end 3805 (in P5 4017).
// P4's and P5's weights are asked for as data that is read once: a step's weights are more than the memory-side cache holds,
// and the others' then stay there (3550 -> 3517; P1's and P3's instead 3832, all 4073, against 3805).
// With all weights in the XCD's L2 already it would be 0.4 less, but touching them there ahead of time (a load per line, by
// waves that wait at a gate) costs 0 - 0.25, through the scalar cache 0.4 - 0.6.  128 registers a wave is what holds them: loads under a branch, or carried
// into the next layer under one, were spilled as they arrived (31 us a layer).
// Keys: one block per head would read 780 KiB; eight splits of at most five tiles of 32 keys keep that at 96 KiB (two
// cameras).
//
// The adaptive norm x rstd (1 + s) + t: producers exchange bf16(x (1 + s)) with the sums of squares of x beside; rstd is a
// factor of the row and multiplies the accumulator; t . W^T is a constant of the step and comes with the modulations.
// fp32 wherever that costs nothing: the residual stream in its owner's registers, logits, the rotation up to its one
// rounding.  (The launches per layer round these to bf16 where the reference arithmetic does.  Rounding the residual here
// as well was measured: mean distance of a chunk from an fp32-activation run 1.9e-3 instead of 0.8e-3.)
#include <math.h>

#include <atomic>

#include "persist.h"
#include "tk_kernels.h"

namespace {
using namespace persist;

constexpr int E = 1024, H = 8, D = 256, F = 4096, A = 32, SPLITS = 8, TILES = 5;
constexpr int KE = E / 32, KO = H * D / 32, KF = F / 32;
constexpr float kOpenpiMask = -2.3819763e38f;  // additive mask of the pi0.5 path

// the weight blob, bytes per layer (operand order, see persist.h): q|k|v [share 80][tile 2][k tile], o [tile][k tile],
// [gate / up pair][k tile] (a lane's 8 gate codes, then its 8 up codes), down [tile][k tile pair]; then the row scales
constexpr int W_QKV = 0, W_O = W_QKV + 160 * KE * 1024, W_GU = W_O + E / 16 * KO * 1024, W_D = W_GU + F / 16 * KE * 1024,
              W_SG = W_D + E / 16 * (KF / 2) * 1024, W_SU = W_SG + F * 4, W_SD = W_SU + F * 4, W_LAYER = W_SD + E * 4;
// modulations, bytes per (step, layer), layer `layers` being the final norm's
constexpr int M_SIN = 0, M_GIN = E * 4, M_SPOST = 2 * E * 4, M_GPOST = 3 * E * 4, M_BQ = 4 * E * 4, M_BG = M_BQ + 2560 * 4, M_BU = M_BG + F * 4,
              M_LAYER = M_BU + F * 4;

// exchange layout (bytes): progress words; two sets of x_t and embedded rows (alternate steps); a ring of kRing layers
constexpr int SS_B = 16 * 64 * 4, X_B = KE * 1024 + SS_B, XT_B = A * 16 * 4;
constexpr int PW_B = 4 * kProgressBytes;
constexpr int OFF_XT = 0, OFF_HID = 4 * XT_B, HEAD_B = OFF_HID + 4 * X_B;
constexpr int Q_B = H * 8192, K_B = 8192, V_B = 16384, PO_B = H * SPLITS * 16384, ST_B = H * 1024, ATT_B = KO * 1024, HF_B = KF * 1024;
constexpr int OFF_Q = 0, OFF_K = OFF_Q + 4 * Q_B, OFF_V = OFF_K + 4 * K_B, OFF_PO = OFF_V + 2 * V_B, OFF_ST = OFF_PO + 4 * PO_B,
              OFF_ATT = OFF_ST + 4 * ST_B, OFF_X1 = OFF_ATT + 4 * ATT_B, OFF_HF = OFF_X1 + 4 * X_B, OFF_X2 = OFF_HF + 4 * HF_B,
              LAYER_B = OFF_X2 + 4 * X_B;
constexpr int kRing = 4;
constexpr size_t XCHG_B = PW_B + 2 * (size_t)HEAD_B + kRing * (size_t)LAYER_B;

constexpr int PART_B = 64 * 1024;
constexpr int L_RS = 2 * PART_B;                  // sums of squares of the 16 rows, four parts, two buffers
constexpr int L_M = L_RS + 2 * 64 * 4;            // tile maxima [wave][16], sums
constexpr int L_L = L_M + kWaves * 16 * 4;
constexpr int L_XT = L_L + kWaves * 16 * 4;       // x_t [32][16]
constexpr int L_WI = L_XT + A * 16 * 4;           // this block's rows of the action embedding [16][32]
constexpr int L_Q = L_WI + 16 * A * 4;            // the query tile, B operand order
constexpr int L_P = L_Q + D / 32 * 1024;          // probabilities of the block's key tiles, B operand order
constexpr int L_ROPE = L_P + TILES * 1024;        // (cos, sin) pairs of 128 column pairs
constexpr int L_KV = L_ROPE + 128 * 16;           // prefix caches of every layer
constexpr int LDS_B = L_KV + kPiMaxLayers * (int)sizeof(PiCache);
static_assert(LDS_B <= 160 * 1024, "one block's LDS");

__global__ __launch_bounds__(kThreads) void pi_denoise_kernel(PiDenoiseArgs a) {
  extern __shared__ __align__(16) unsigned char lds[];
  Ctx cx;
  cx.tid = threadIdx.x;
  cx.lane = cx.tid & 63;
  cx.wave = __builtin_amdgcn_readfirstlane(cx.tid >> 6);
  cx.g = cx.lane >> 4;
  cx.r = cx.lane & 15;
  cx.spin = a.spin;
  cx.dead = 0;
  // blocks land round-robin on the XCDs: the row groups' blocks of one column share are on one
  int rt = blockIdx.x >> 6, c = blockIdx.x & 63;
  if (rt * 16 >= a.M) return;
  cx.rs = make_rsrc(a.xchg, (unsigned)XCHG_B);
  const rsrc_t wr = make_rsrc(a.blob, (unsigned)a.layers * W_LAYER);
  const rsrc_t mr = make_rsrc(a.mods, (unsigned)(a.steps * (a.layers + 1)) * M_LAYER);
  int &tid = cx.tid, &lane = cx.lane, &wave = cx.wave, &g = cx.g, &r = cx.r;
  const int nsuf = (a.M + 31) >> 5, tp = (a.P + 31) >> 5, ntile = tp + nsuf;
  // this block's key tiles: [t0, t1) of the prefix's, then the action tokens'
  const int t0 = (c & 7) * ntile / SPLITS, t1 = ((c & 7) + 1) * ntile / SPLITS, cnt = t1 - t0;

  float* const ldsf = (float*)lds;
  float* const sM = ldsf + L_M / 4;
  float* const sL = ldsf + L_L / 4;
  float* const sX = ldsf + L_XT / 4;
  float* const sW = ldsf + L_WI / 4;
  int buf = 0;  // partial buffer of the current phase (phases alternate: one barrier each is enough)
  auto part = [&]() { return lds + buf * PART_B; };
  auto sq_s = [&]() { return ldsf + L_RS / 4 + buf * 64; };

  enum { PH_E0, PH_E1, PH_P1, PH_P2, PH_PC, PH_P3, PH_P4, PH_P5 };
  auto id_of = [&](int step, int l, int ph) { return (step * (a.layers + 1) + l + 1) * 8 + ph; };  // E phases: l = -1
  // (everything asked for has arrived by then: told so, the compiler does not wait for the store's acknowledgement where it
  // next uses a loaded register)
  auto arrived = [&]() { __builtin_amdgcn_s_waitcnt(0x0f70); };  // vmcnt(0)
  auto announce = [&](int id) {
    if (tid == 0) st_x(cx.rs, (unsigned)id, 0, rt * kProgressBytes + c * 128);
  };
  auto gate = [&](unsigned long long who, int id) {
    const unsigned mine = wave < 4 ? (unsigned)(who >> (16 * wave)) & 0xffff : 0;
    if (mine) watch<16>(cx, (const char*)a.xchg + rt * kProgressBytes + wave * 2048, mine, id);
    block_barrier();
  };
  constexpr unsigned long long kAll = ~0ull, kAct = (1ull << A) - 1;

  // every phase forms its addresses from values the compiler cannot see through (it would form all of them ahead of the
  // loops and spill them)
  auto fresh = [&]() {
    c = __builtin_amdgcn_readfirstlane(c);
    rt = __builtin_amdgcn_readfirstlane(rt);
    wave = __builtin_amdgcn_readfirstlane(wave);
    asm volatile("" : "+s"(c), "+s"(rt), "+s"(wave));
    asm volatile("" : "+v"(tid));
    lane = tid & 63;
    g = lane >> 4;
    r = lane & 15;
  };

  // ---- constants of the whole run ----
  if (tid < 128) {  // row tid / 8, columns n = 2 (tid & 7) and the next
    const int mg = rt * 16 + (tid >> 3), n = 2 * (tid & 7);
    int p = a.pos[mg < a.M ? mg : a.M - 1];
    p = p < 0 ? 0 : (p > a.positions - 1 ? a.positions - 1 : p);
    f32x2* const o = (f32x2*)(lds + L_ROPE + tid * 16);
    o[0] = *(const f32x2*)(a.rope_cos + (size_t)p * (D / 2) + 16 * (c & 7) + n);
    o[1] = *(const f32x2*)(a.rope_sin + (size_t)p * (D / 2) + 16 * (c & 7) + n);
  }
  if (tid < a.layers * (int)(sizeof(PiCache) / 4)) ((int*)(lds + L_KV))[tid] = ((const int*)a.cache)[tid];
  if (tid < A * 16) {
    const int j = tid >> 4, m = rt * 16 + (tid & 15);
    sX[tid] = m < a.M ? a.x0[m * A + j] : 0.f;
    sW[tid] = a.emb_w[(16 * c + (tid >> 5)) * A + (tid & 31)];
  }
  float xcol = 0.f;  // E0: x_t of row tid (< 16), column c
  if (tid < 16 && c < A && rt * 16 + tid < a.M) xcol = a.x0[(rt * 16 + tid) * A + c];
  // this wave's 16 keys (half a tile) in P2: keys 4 g .. 4 g + 3 of them in this lane; bits 8..11: keys that exist
  const int kt = t0 + (wave >> 1);  // their tile
  unsigned vis;
  {
    const bool suf = kt >= tp;
    const int k0 = 32 * (suf ? kt - tp : kt) + 16 * (wave & 1) + 4 * g, len = suf ? a.M : a.P;
    vis = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = k0 + i;
      if (kt < t1 && key < len) vis |= (0x100u | ((suf || a.pad == nullptr || a.pad[key] != 0) ? 1u : 0u)) << i;
    }
  }

  // where this thread's words go, within a layer of the ring.  P1, q and k: the two words of a rotary pair; v: of two tiles
  auto q_s = [&]() { return OFF_Q + rt * Q_B + (c >> 3) * 8192 + ((c & 7) >> 1) * 1024 + (c & 1) * 512; };
  auto kv_off = [&](const Own& ow, int& off, int& step) {  // blocks 0..15, threads 256..511
    if (c < 8) {
      off = OFF_K + rt * K_B + (c >> 1) * 1024 + (c & 1) * 512 + ow.word;
      step = 4096;
    } else {  // keys n, n + 1 of column m
      off = OFF_V + (rt >> 1) * V_B + 2 * (c - 8) * 1024 + (rt & 1) * 512 + ow.word;
      step = 1024;
    }
  };
  auto po_s = [&](int split) { return OFF_PO + rt * PO_B + ((c & 56) + split) * 16384; };
  auto st_s = [&]() { return OFF_ST + rt * ST_B + (c >> 3) * 1024; };  // [pair of splits][row] of two (maximum, sum)
  auto st_w = [&]() { return ((c & 7) >> 1) * 256 + (c & 1) * 8 + lane * 16; };  // lanes < 16
  auto att_s = [&]() { return OFF_ATT + rt * ATT_B + c * 1024; };
  auto x_s = [&]() { return rt * X_B + (c >> 1) * 1024 + (c & 1) * 512; };
  auto ss_s = [&]() { return rt * X_B + KE * 1024 + c * 64; };
  auto h_s = [&]() { return OFF_HF + rt * HF_B + 2 * c * 1024; };
  auto xt_s = [&]() { return OFF_XT + rt * XT_B + c * 64; };

  float res0 = 0.f, res1 = 0.f;  // the residual stream: row m, columns 16 c + n, n + 1 (threads < 256)
  auto put_hidden = [&](const Own& ow, f32x2 s, int base) {
    if (ow.put) st_x(cx.rs, pack_bf16x2(res0 * (1.0f + s[0]), res1 * (1.0f + s[1])), ow.word, base + x_s());
    const float ss = own_row_sum(fmaf(res0, res0, res1 * res1));
    if (ow.put && ow.n == 0) st_x(cx.rs, __float_as_uint(ss), ow.m * 4, base + ss_s());
  };
  auto add_gated = [&](f32x2 y, f32x2 gate) {
    res0 = fmaf(y[0], gate[0], res0);
    res1 = fmaf(y[1], gate[1], res1);
  };
  auto poison_hidden = [&](const Own& ow, int base) {
    if (ow.put) st_x(cx.rs, 0xffffffffu, ow.word, base + x_s());
    if (ow.put && ow.n == 0) st_x(cx.rs, 0xffffffffu, ow.m * 4, base + ss_s());
  };
  // the sums of squares of the 16 rows: an extra piece of the last four waves, 16 of the 64 column shares each
  auto ask_stats = [&](i32x4& st, int base) {
    const int k = wave - (kWaves - 4);
    st = ld_x(cx.rs, lane_at(k >= 0, lane * 16), base_at(k >= 0, base + rt * X_B + KE * 1024 + k * 1024));
  };
  auto take_stats = [&](i32x4& st, int base) {
    const int k = wave - (kWaves - 4);
    if (k >= 0) {
      for (int n = 0;; ++n) {
        if (__builtin_amdgcn_ballot_w64(unset(st)) == 0 || cx.dead) break;
        if (n >= cx.spin) {
          cx.dead = 1;
          break;
        }
        pin();
        ask_stats(st, base);
      }
      const float ss = share_sum(st);
      if ((lane & 12) == 0) sq_s()[k * 16 + share_row(lane)] = ss;
    }
  };
  auto rstd_of = [&](int m) { return rsqrtf((sq_s()[m] + sq_s()[16 + m] + sq_s()[32 + m] + sq_s()[48 + m]) * (1.0f / E) + a.eps); };

  // four pieces s0, s0 + sd, .. of a buffer in operand order (all of them asked for again until all are there: no copies)
  auto wait_pieces = [&](i32x4 (&v)[4], int base, int s0, int sd) {
    int voff[4], soff[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      voff[i] = lane * 16;
      soff[i] = base + (s0 + sd * i) * 1024;
    }
    wait_all<4>(v, cx, voff, soff);
  };
  // a rotary pair of two columns -> two words
  auto rotate = [&](f32x2 va, f32x2 vb, int slot, unsigned& wa, unsigned& wb) {
    const f32x2 cs = ((const f32x2*)(lds + L_ROPE + slot * 16))[0], sn = ((const f32x2*)(lds + L_ROPE + slot * 16))[1];
    float ra[2], rb[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      ra[j] = va[j] * cs[j] - vb[j] * sn[j];
      rb[j] = vb[j] * cs[j] + va[j] * sn[j];
    }
    wa = pack_bf16x2(ra[0], ra[1]);
    wb = pack_bf16x2(rb[0], rb[1]);
  };

  i32x4 wA[4][2], wB[4], wC[2][4], wD[4], vf[TILES];
  f32x2 bq0, bq1, gin, spost, scg, scu, bg, bu, scd, gpost, snext;
  auto load_A = [&](int step, int l) {
    const int ml = (step * (a.layers + 1) + l) * M_LAYER;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int t = 0; t < 2; ++t) wA[t][i] = ld_w(wr, lane * 16, l * W_LAYER + W_QKV + ((2 * c + t) * KE + wave + 16 * i) * 1024);
    const bool second = wave >= 4;
    const Own ow = own_of(tid);
    const int n4 = second && c >= 8 ? ow.m * 4 : ow.n * 4;
    const int share = second ? 64 + c : c;
    bq0 = ld_f2_if(share < 80, mr, n4, ml + M_BQ + share * 128);
    bq1 = ld_f2_if(share < 80, mr, n4, ml + M_BQ + share * 128 + 64);
  };
  auto load_A2 = [&](int l) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int t = 0; t < 2; ++t) wA[2 + t][i] = ld_w_if(c < 16, wr, lane * 16, l * W_LAYER + W_QKV + ((2 * (64 + c) + t) * KE + wave + 16 * i) * 1024);
  };
  auto load_B = [&](int step, int l) {
    const int ml = (step * (a.layers + 1) + l) * M_LAYER, n4 = own_of(tid).n * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) wB[i] = ld_w(wr, lane * 16, l * W_LAYER + W_O + (c * KO + wave + 16 * i) * 1024);
    gin = ld_f2(mr, n4, ml + M_GIN + 64 * c);
    spost = ld_f2(mr, n4, ml + M_SPOST + 64 * c);
  };
  auto load_C = [&](int l, int q) {
    const int p = 4 * c + 2 * (wave >> 3) + q;
#pragma unroll
    for (int i = 0; i < 4; ++i) wC[q][i] = ld_once(wr, lane * 16, l * W_LAYER + W_GU + (p * KE + (wave & 7) + 8 * i) * 1024);
  };
  auto load_CS = [&](int step, int l) {
    const int ml = (step * (a.layers + 1) + l) * M_LAYER, f = 64 * (wave >> 2) + own_of(tid).n * 4;
    scg = ld_f2(wr, f, l * W_LAYER + W_SG + 256 * c);
    scu = ld_f2(wr, f, l * W_LAYER + W_SU + 256 * c);
    bg = ld_f2(mr, f, ml + M_BG + 256 * c);
    bu = ld_f2(mr, f, ml + M_BU + 256 * c);
  };
  auto load_D = [&](int step, int l) {
    const int ml = (step * (a.layers + 1) + l) * M_LAYER, n4 = own_of(tid).n * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) wD[i] = ld_once(wr, lane * 16, l * W_LAYER + W_D + (c * (KF / 2) + wave + 16 * i) * 1024);
    scd = ld_f2(wr, n4, l * W_LAYER + W_SD + 64 * c);
    gpost = ld_f2(mr, n4, ml + M_GPOST + 64 * c);
    snext = ld_f2(mr, n4, ml + M_LAYER + M_SIN + 64 * c);  // the norm that reads P5's rows
  };
  auto load_K = [&](i32x4 (&kf)[8], int l) {
    const PiCache& L = ((const PiCache*)(lds + L_KV))[l];
    const int sl = __builtin_amdgcn_readfirstlane(L.k_sl);
    const rsrc_t rk = make_rsrc(uniform_ptr(L.k), 2u * ((a.P - 1) * sl + D));
    const int t = t0 + (wave >> 1);
    int key = 32 * t + 16 * (wave & 1) + r;
    if (key > a.P - 1) key = a.P - 1;  // masked below
#pragma unroll
    for (int s = 0; s < 8; ++s) kf[s] = ld_w_if(t < t1 && t < tp, rk, 2 * (key * sl + 8 * g), 64 * s);
  };
  auto load_V = [&](int l) {
    const PiCache& L = ((const PiCache*)(lds + L_KV))[l];
    const int sd = __builtin_amdgcn_readfirstlane(L.vt_sd);
    const rsrc_t rv = make_rsrc(uniform_ptr(L.vt), 2u * ((D - 1) * sd + 32 * tp));
#pragma unroll
    for (int i = 0; i < TILES; ++i) vf[i] = ld_w_if(t0 + i < t1 && t0 + i < tp, rv, 2 * ((16 * wave + r) * sd + 8 * g), 64 * (t0 + i));
  };

  block_barrier();
  load_A(0, 0);
  load_A2(0);

  for (int step = 0; step <= a.steps; ++step) {
    const int cur = PW_B + (step & 1) * HEAD_B, oth = PW_B + ((step + 1) & 1) * HEAD_B;
    auto slot = [&](int l) { return PW_B + 2 * HEAD_B + ((step * a.layers + l) & (kRing - 1)) * LAYER_B; };
    // ---------------- E0: the previous step's velocity and Euler update ----------------
    fresh();
    if (step > 0) {
      if (c < A) {
        const int in_base = slot(-1) + OFF_X2;
        i32x4 v[2];
        f32x4 wa[2][2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const float* w = a.act_w + c * E + 32 * (wave + 16 * i) + 8 * g;
          wa[i][0] = *(const f32x4*)w;
          wa[i][1] = *(const f32x4*)(w + 4);
        }
        const float bias = a.mods[(size_t)((step - 1) * (a.layers + 1) + a.layers) * (M_LAYER / 4) + M_BQ / 4 + c];
        pin();
        gate(kAll, id_of(step - 1, a.layers - 1, PH_P5));
        i32x4 st;
        wait_tiles<2, KE>(v, cx, in_base + rt * X_B, wave, 16, [&] { ask_stats(st, in_base); });
        announce(id_of(step, -1, PH_E0));
        float acc = 0.f;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const unsigned xv = (unsigned)v[i][e >> 1];
            acc = fmaf(__uint_as_float((e & 1) ? (xv & 0xffff0000u) : (xv << 16)), wa[i][e >> 2][e & 3], acc);
          }
        acc = row_sum(acc);
        if (lane < 16) sM[wave * 16 + r] = acc;
        take_stats(st, in_base);
        block_barrier();
        if (tid < 16) {
          float v0 = 0.f;
#pragma unroll
          for (int w = 0; w < kWaves; ++w) v0 += sM[w * 16 + tid];
          xcol = add_rn(xcol, mul_rn(a.dt, v0 * rstd_of(tid) + bias));
          const int m = rt * 16 + tid;
          if (step == a.steps) {
            if (m < a.M) a.out[m * A + c] = xcol;
          } else {
            st_x(cx.rs, __float_as_uint(xcol), tid * 4, cur + xt_s());
          }
        }
        buf ^= 1;
      }
      if (step == a.steps) return;
      gate(kAct, id_of(step, -1, PH_E0));
      if (wave < 2) {
        i32x4 v[1];
        const int voff[1] = {lane * 16}, soff[1] = {cur + OFF_XT + rt * XT_B + wave * 1024};
        wait_x<1>(v, cx, voff, soff, [] {});
        *(i32x4*)(lds + L_XT + wave * 1024 + lane * 16) = v[0];
      }
      block_barrier();
    }
    // ---------------- E1: action embedding ----------------
    fresh();
    announce(id_of(step, -1, PH_E1));
    if (tid < 256) {
      const Own ow = own_of(tid);
      const f32x2 s = ld_f2(mr, ow.n * 4, step * (a.layers + 1) * M_LAYER + M_SIN + 64 * c);
      const f32x2 b = *(const f32x2*)(a.emb_b + 16 * c + ow.n);
      res0 = 0.f;
      res1 = 0.f;
#pragma unroll 8
      for (int j = 0; j < A; ++j) {
        const float x = sX[j * 16 + ow.m];
        res0 = fmaf(x, sW[ow.n * A + j], res0);
        res1 = fmaf(x, sW[(ow.n + 1) * A + j], res1);
      }
      res0 += b[0];
      res1 += b[1];
      put_hidden(ow, s, cur + OFF_HID);
    }

    for (int l = 0; l < a.layers; ++l) {
      const int base = slot(l);
      // the layer whose first weights are asked for in this one (behind the last one: dropped.  Asked for under a condition,
      // their registers would be live through the whole layer)
      const int nl = l + 1 < a.layers ? l + 1 : 0, nstep = nl || step + 1 == a.steps ? step : step + 1;
      const int in_base = l == 0 ? cur + OFF_HID : slot(l - 1) + OFF_X2;  // the layer's input rows
      i32x4 kf[8];  // this wave's 16 keys
      // ---------------- P1: q | k | v ----------------
      fresh();
      {
        i32x4 x[2], st;
        gate(kAll, l == 0 ? id_of(step, -1, PH_E1) : id_of(step, l - 1, PH_P5));
        wait_tiles<2, KE>(x, cx, in_base + rt * X_B, wave, 16, [&] { ask_stats(st, in_base); });
        arrived();
        announce(id_of(step, l, PH_P1));
        f32x4 acc[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const f32x4 z = {0.f, 0.f, 0.f, 0.f};
          // (V^T: the operands swapped, a lane then owns a column and four consecutive keys)
          acc[t] = t >= 2 && c >= 8 ? mfma(x[1], wA[t][1], mfma(x[0], wA[t][0], z)) : mfma(wA[t][1], x[1], mfma(wA[t][0], x[0], z));
        }
#pragma unroll
        for (int t = 0; t < 4; ++t)
          if (t < 2 || c < 16) *(f32x4*)(part() + (wave * 4 + t) * 1024 + part_slot(cx)) = acc[t];
        take_stats(st, in_base);
        block_barrier();
        if (wave < 4 || (wave < 8 && c < 16)) {
          const Own ow = own_of(tid);
          const int t = wave < 4 ? 0 : 2;
          const f32x2 va = sum_part<16, 4>(part(), 0, t, ow), vb = sum_part<16, 4>(part(), 0, t + 1, ow);
          unsigned wa, wb;
          if (t == 0 || c < 8) {
            const float rstd = rstd_of(ow.m);
            rotate(va * rstd + bq0, vb * rstd + bq1, ow.m * 8 + (ow.n >> 1), wa, wb);
          } else {
            const float r0 = rstd_of(ow.n), r1 = rstd_of(ow.n + 1);
            wa = pack_bf16x2(va[0] * r0 + bq0[0], va[1] * r1 + bq0[0]);
            wb = pack_bf16x2(vb[0] * r0 + bq1[0], vb[1] * r1 + bq1[0]);
          }
          int off = ow.word + q_s(), d = 4096;
          if (t) kv_off(ow, off, d);
          if (ow.put) {
            st_x(cx.rs, wa, off, base);
            st_x(cx.rs, wb, off + d, base);
          }
        }
        buf ^= 1;
        pin();
        load_K(kf, l);
      }
      // ---------------- P2: attention of one head over this block's keys ----------------
      fresh();
      {
        const bool has_suf = t1 > tp;
        gate((0xffull << (c & 56)) | (has_suf ? 0xffffull : 0ull), id_of(step, l, PH_P1));
        if (wave < 8) {
          i32x4 q[1];
          const int voff[1] = {lane * 16}, soff[1] = {base + OFF_Q + rt * Q_B + (c >> 3) * 8192 + wave * 1024};
          wait_x<1>(q, cx, voff, soff, [] {});
          *(i32x4*)(lds + L_Q + wave * 1024 + lane * 16) = q[0];
        }
        pin();
        load_V(l);
        pin();
        const int t = t0 + (wave >> 1);
        // the action tokens' own keys and values: 16 keys are the rows of one row group (one that does not exist: repeat)
        i32x4 vs[2];
        auto ask_vs = [&]() {
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const bool own = tp + j >= t0 && tp + j < t1;
            vs[j] = ld_x(cx.rs, lane_at(own, ((16 * (2 * j + 1) >= a.M ? (g & 1) : g) * 16 + r) * 16), base_at(own, base + OFF_V + j * V_B + wave * 1024));
          }
        };
        if (has_suf) {
          if (t < t1 && t >= tp) {
            int grp = 2 * (t - tp) + (wave & 1);
            if (16 * grp >= a.M) grp = 2 * (t - tp);
            int voff[8], soff[8];
#pragma unroll
            for (int s = 0; s < 8; ++s) {
              voff[s] = lane * 16;
              soff[s] = base + OFF_K + grp * K_B + s * 1024;
            }
            wait_all<8>(kf, cx, voff, soff);
          }
          for (int n = 0;; ++n) {
            pin();
            ask_vs();
            if (__builtin_amdgcn_ballot_w64(unset(vs[0]) || unset(vs[1])) == 0 || cx.dead) break;
            if (n >= cx.spin) {
              cx.dead = 1;
              break;
            }
          }
        }
        block_barrier();
        const bool has = t < t1;
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
        if (has) {
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            if (k == 4) pin();  // (four operands of the query on the way, not eight)
            s = mfma(kf[k], *(const i32x4*)(lds + L_Q + k * 1024 + lane * 16), s);
          }
        }
        float p[4], tmax = -INFINITY, ls = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float sv = s[e] * 0.0625f;
          p[e] = (vis >> (8 + e)) & 1u ? ((vis >> e) & 1u ? sv : sv + kOpenpiMask) : -INFINITY;
          tmax = fmaxf(tmax, p[e]);
        }
        tmax = max16(tmax);
        tmax = max32(tmax);
        if (lane < 16) sM[wave * 16 + r] = tmax;
        block_barrier();
        announce(id_of(step, l, PH_P2));
        static_assert(2 * TILES <= 12, "three tiles per lane (without keys: -inf)");
        const float bm = max16(max32(fmaxf(fmaxf(sM[g * 16 + r], sM[(g + 4) * 16 + r]), sM[(g + 8) * 16 + r])));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          p[e] = (vis >> (8 + e)) & 1u ? __expf(p[e] - bm) : 0.f;  // (a block without keys: bm is -inf)
          ls += p[e];
        }
        ls = row_sum(ls);
        // keys 16 (wave & 1) + 4 g .. of the tile, row r, into the B operand
        if (has)
          *(i32x2*)(lds + L_P + (wave >> 1) * 1024 + ((2 * (wave & 1) + (g >> 1)) * 16 + r) * 16 + (g & 1) * 8) =
              i32x2{(int)pack_bf16x2(p[0], p[1]), (int)pack_bf16x2(p[2], p[3])};
        if (lane < 16) sL[wave * 16 + r] = ls;
        block_barrier();
        f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < TILES; ++i)
          if (i < cnt && t0 + i < tp) o = mfma(vf[i], *(const i32x4*)(lds + L_P + i * 1024 + lane * 16), o);
        if (has_suf) {
#pragma unroll
          for (int j = 0; j < 2; ++j)
            if (tp + j >= t0 && tp + j < t1) o = mfma(vs[j], *(const i32x4*)(lds + L_P + (tp + j - t0) * 1024 + lane * 16), o);
        }
        st_x4(cx.rs, __builtin_bit_cast(i32x4, o), lane * 16, base + po_s(c & 7) + wave * 1024);
        if (wave == 0) {
          const float sum = row_sum(sL[g * 16 + r] + sL[(g + 4) * 16 + r] + sL[(g + 8) * 16 + r]);
          if (lane < 16) st_x2(cx.rs, __float_as_uint(bm), __float_as_uint(sum), st_w(), base + st_s());
        }
        pin();
      }
      // ---------------- PC: the splits' outputs into 32 columns of the head ----------------
      fresh();
      {
        gate(0xffull << (c & 56), id_of(step, l, PH_P2));
        i32x4 v[2];
        const int voff[2] = {lane * 16, lane * 16};
        const int soff[2] = {base + po_s(wave >> 1) + (2 * (c & 7) + (wave & 1)) * 1024, base + st_s()};
        wait_x<2>(v, cx, voff, soff, [] {});
        arrived();
        announce(id_of(step, l, PH_PC));
        pin();
        load_B(step, l);
        pin();
        // this lane: splits 2 g, 2 g + 1 of row r
        const float m0 = __int_as_float(v[1][0]), l0 = __int_as_float(v[1][1]), m1 = __int_as_float(v[1][2]), l1 = __int_as_float(v[1][3]);
        float mx = fmaxf(m0, m1);
        mx = max16(mx);
        mx = max32(mx);
        const float e0 = __expf(m0 - mx), e1 = __expf(m1 - mx);
        const float sum = row_sum(e0 * l0 + e1 * l1);
        const float w = __shfl((wave >> 1) & 1 ? e1 : e0, (wave >> 2) * 16 + r) / sum;
        *(f32x4*)(part() + wave * 1024 + part_slot(cx)) = __builtin_bit_cast(f32x4, v[0]) * w;
        block_barrier();
        if (tid < 512) {
          const Own ow = own_of(tid);
          const f32x2 o = sum_part<8, 2>(part(), 0, wave >> 2, ow);
          if (ow.put) st_x(cx.rs, pack_bf16x2(o[0], o[1]), (wave >> 2) * 512 + ow.word, base + att_s());
        }
        buf ^= 1;
        pin();
        load_C(l, 0);
        load_CS(step, l);
      }
      // ---------------- P3: output projection, gated residual ----------------
      fresh();
      {
        i32x4 v[4];
        gate(kAll, id_of(step, l, PH_PC));
        wait_pieces(v, base + OFF_ATT + rt * ATT_B, wave, 16);
        arrived();
        announce(id_of(step, l, PH_P3));
        pin();
        load_C(l, 1);
        pin();
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i) acc = mfma(wB[i], v[i], acc);
        *(f32x4*)(part() + wave * 1024 + part_slot(cx)) = acc;
        block_barrier();
        if (tid < 256) {
          const Own ow = own_of(tid);
          add_gated(sum_part<16, 1>(part(), 0, 0, ow), gin);
          put_hidden(ow, spost, base + OFF_X1);
        }
        buf ^= 1;
        pin();
      }
      // ---------------- P4: gate / up ----------------
      fresh();
      {
        i32x4 v[4], st;
        gate(kAll, id_of(step, l, PH_P3));
        ask_stats(st, base + OFF_X1);
        wait_pieces(v, base + OFF_X1 + rt * X_B, wave & 7, 8);
        arrived();
        announce(id_of(step, l, PH_P4));
        f32x4 acc[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            acc[2 * q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fp8x8_to_bf16x8(wC[q][i][0], wC[q][i][1]), as_bf16x8(v[i]), acc[2 * q], 0, 0, 0);
            acc[2 * q + 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fp8x8_to_bf16x8(wC[q][i][2], wC[q][i][3]), as_bf16x8(v[i]), acc[2 * q + 1], 0, 0, 0);
          }
#pragma unroll
        for (int t = 0; t < 4; ++t) *(f32x4*)(part() + (wave * 4 + t) * 1024 + part_slot(cx)) = acc[t];
        take_stats(st, base + OFF_X1);
        load_D(step, l);
        block_barrier();
        {
          const Own ow = own_of(tid);
          const int w0 = (wave >> 3) * 8, t = 2 * ((wave >> 2) & 1);
          const float rstd = rstd_of(ow.m);
          const f32x2 gt = sum_part<8, 4>(part(), w0, t, ow) * rstd * scg + bg, up = sum_part<8, 4>(part(), w0, t + 1, ow) * rstd * scu + bu;
          const unsigned h = pack_bf16x2(gelu_tanh_f(gt[0]) * up[0], gelu_tanh_f(gt[1]) * up[1]);
          if (ow.put) st_x(cx.rs, h, (wave >> 2) * 512 + ow.word, base + h_s());
        }
        buf ^= 1;
        pin();
        load_A(nstep, nl);
        load_A2(nl);
      }
      // ---------------- P5: down projection, gated residual ----------------
      fresh();
      {
        i32x4 v[8];
        gate(kAll, id_of(step, l, PH_P4));
        int voff[8], soff[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          voff[i] = lane * 16;
          soff[i] = base + OFF_HF + rt * HF_B + (2 * (wave + 16 * (i >> 1)) + (i & 1)) * 1024;
        }
        wait_all<8>(v, cx, voff, soff);
        arrived();
        announce(id_of(step, l, PH_P5));
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 8; ++i)
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fp8x8_to_bf16x8(wD[i >> 1][2 * (i & 1)], wD[i >> 1][2 * (i & 1) + 1]), as_bf16x8(v[i]), acc, 0, 0, 0);
        *(f32x4*)(part() + wave * 1024 + part_slot(cx)) = acc;
        block_barrier();
        if (tid < 256) {
          const Own ow = own_of(tid);
          add_gated(sum_part<16, 1>(part(), 0, 0, ow) * scd, gpost);
          put_hidden(ow, snext, base + OFF_X2);
        }
        buf ^= 1;
        pin();
      }
      // ---- back to all ones: the words of the layer before (this layer's P5 input is made of what every block of the
      // group, and through the keys and values every group, produced after reading them); they are written again three
      // layers on.  x_t and the embedded rows: a step later, likewise ----
      const unsigned ones = 0xffffffffu;
      const i32x4 ones4 = {-1, -1, -1, -1};
      fresh();
      if (step > 0 || l > 0) {
        const int ob = slot(l - 1);
        const Own ow = own_of(tid);
        if (tid < 256) {
          if (ow.put) {
            st_x(cx.rs, ones, ow.word + q_s(), ob);
            st_x(cx.rs, ones, ow.word + q_s() + 4096, ob);
          }
          poison_hidden(ow, ob + OFF_X1);
          poison_hidden(ow, ob + OFF_X2);
        } else if (tid < 512 && c < 16) {
          int off, d;
          kv_off(ow, off, d);
          if (ow.put) {
            st_x(cx.rs, ones, off, ob);
            st_x(cx.rs, ones, off + d, ob);
          }
        }
        st_x4(cx.rs, ones4, lane * 16, ob + po_s(c & 7) + wave * 1024);
        if (tid < 16) st_x2(cx.rs, ones, ones, st_w(), ob + st_s());
        if (tid < 256) st_x(cx.rs, ones, tid * 4, ob + att_s());
        if (tid < 512) st_x(cx.rs, ones, tid * 4, ob + h_s());
        if (l == 0) {
          if (tid < 256) poison_hidden(ow, oth + OFF_HID);
          if (c < A && tid < 16) st_x(cx.rs, ones, tid * 4, oth + xt_s());
        }
      }
    }
  }
}

}  // namespace

size_t tk_pi_denoise_exchange_bytes() { return XCHG_B; }
size_t tk_pi_denoise_blob_bytes() { return W_LAYER; }
size_t tk_pi_denoise_mod_bytes() { return M_LAYER; }
int tk_pi_denoise_max_key_tiles() { return SPLITS * TILES; }

int tk_launch_pi_denoise(const PiDenoiseArgs& a, hipStream_t st) {
  static std::atomic<int> raised{0};  // more LDS than a launch gets by default: raise the kernel's limit once per process
  if (!raised.load(std::memory_order_acquire)) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(&pi_denoise_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, LDS_B) != hipSuccess) return -3;
    raised.store(1, std::memory_order_release);
  }
  if (tk_launch_fill_ones(a.xchg, XCHG_B, st)) return -3;
  hipLaunchKernelGGL(pi_denoise_kernel, dim3(256), dim3(kThreads), LDS_B, st, a);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}
