// The SmolVLA flow-matching loop as ONE persistent launch: suffix embedding, every expert layer (self and cross), final
// norm, action projection and Euler update of all steps.
//
// Bound: latency.  A step's sixteen layers are some 75 dependent phases of 0.1 - 0.5 us of work each; as a launch per
// phase they cost 4 - 11 us apiece (launch gap, cold first loads, statistics, drain).  Here 256 resident blocks run the
// phases back to back: block (rt, c) works on 16 of the chunk's rows with column share c of 64, its weights are on their
// way before its input is, and activations pass through the self-signalling exchange buffers of persist.h.
//
//   step    E0  v = final_norm(x) . Wa^T + b, x_t += dt v         32 blocks per row group, one action column each
//           E1  h = silu(x_t . Ws^T + c_step)                     45 blocks, 16 columns each
//           E2  hidden = h . Wt^T + b  (fp32 products)            45 blocks
//   layer   P1  q | k | v = norm(hidden) . W^T, rotary            50 blocks (self layers), 32 columns each
//           P2  attention of one head over [prefix; action tokens] (self), or norm + q projection + rotary + attention
//               over the prefix's fp32 K / V as bf16 hi + lo planes (cross)                  15 blocks
//           P3  hidden += att . Wo^T                              45 blocks
//           P4  h = silu(g) * u of norm(hidden) . Wgu^T           64 blocks, two gate / up pairs of 16 columns each
//           P5  hidden += h . Wd^T                                45 blocks
//
// Rows: 16 per block (four row groups), so a block's share of a phase's input is 23 - 64 KiB.  The four blocks of one
// column share are on one XCD, whose L2 then fetches their weights once: the loop 2.74 -> 2.55 ms against a row group on
// two XCDs of its own, although a hand-off inside two XCDs is 0.3 us shorter.  Inside a block the 16 waves split K; the partial
// tiles meet in LDS once per phase.  With four waves on every SIMD an instruction costs 16 cycles of the phase, so what
// 64 blocks would repeat is done once by the producer: hidden rows are exchanged as bf16(x * w) with the NEXT norm's
// weight, beside the row's partial sums of squares; 1 / rms is a factor of the whole row and multiplies the accumulator.
// The residual stream never leaves its owner's registers and stays fp32 there.
//
// Measured (50 action tokens, 241 prefix tokens, 16 layers, 10 steps): 1.98 ms, against 4.7 ms of the launches per layer: 12.3 us
// a layer and step, a step's ends included.  With stamps in every block, which the kernel pays for, a self layer takes 13.5 us
// (mean) and a cross layer 12.4: five or four hand-offs of 0.6 - 1 us from a
// phase's result to the next one's first input, 0.3 - 0.7 us until all of a block's input is there (64 bytes a cycle), and
// from there to the result 0.6 us in P3 and P5, 1.0 in P1 and P4, 1.7 in the attention, 3.6 us in a cross layer's.
// Where loads are asked for (the loop, us; first figure: as below):
//   * P1's weights: at P4's end 2185; at the end of P3 2309, at P4's input 2218, in P5 2197.
//   * The cross layers' values: between the query's reduction and its barrier 2240; in front of the reduction 2309, behind
//     the barrier 2300.  Their query weights and K in front of the gate (K behind it 2366).
//   * Everything else of a layer behind P1, in the attention's blocks behind the attention (P5's at P4 2108, P4's at P3 2109,
//     against 2070).
// When a block raises its progress word: in the attention behind its last barrier 1979 (in front of it 2068), in P3 with its
// partial tiles written 1973 (at its input 1985), else when the input is there (P1 behind its barrier 1996).
#include <math.h>

#include <atomic>
#include <type_traits>

#include "persist.h"
#include "tk_kernels.h"

namespace {
using namespace persist;

constexpr int E = 720, H = 15, G = 5, D = 64, F = 2048, A = 32;
constexpr int KE = 23, KO = 30, KF = 64;  // k tiles of 32: hidden (the last one half), attention output, feed-forward
constexpr int NE = E / 16;                // 16-column shares of the hidden size
constexpr int NQ = 50;                    // 32-column shares of q | k | v
// blocks 0 .. 44 of a row group own the hidden columns; the attention runs on 45 .. 59, which sit out P3 and P5 and have
// the next layer's keys and values on the way meanwhile; q | k | v shares: 0 .. 44, 60 .. 63 and (the odd one) 45
constexpr int AT = NE;
constexpr float kF32Min = -3.4028234663852886e38f;

// the weight blob, bytes per layer: [16-column tile][k tile] of 1 KiB in A operand order for the bf16 products;
// [gate / up pair][k tile] of 1 KiB (a lane's 8 gate codes, then its 8 up codes); [tile][k tile pair] of 1 KiB (a lane's
// 8 codes of both k tiles); scales and norm weights
constexpr int W_QKV = 0, W_O = W_QKV + 2 * NQ * KE * 1024, W_GU = W_O + NE * KO * 1024, W_D = W_GU + F / 16 * KE * 1024,
              W_SG = W_D + NE * (KF / 2) * 1024, W_SU = W_SG + F * 4, W_SD = W_SU + F * 4, W_NIN = W_SD + E * 4, W_NPOST = W_NIN + E * 4,
              W_LAYER = (W_NPOST + E * 4 + 1023) / 1024 * 1024;

// exchange layout (bytes): kSets sets, used by the steps in turn; per set a head (per row group: x, h, hidden and its sums of squares), then per layer Q, K, V,
// attention output, hidden after attention, feed-forward intermediate, hidden (hidden rows with sums of squares)
constexpr int SS_B = 48 * 16 * 4;  // partial sums of squares: [column share][row]
constexpr int XT_B = 2048, HE_B = NE * 1024, X_B = KE * 1024 + SS_B;
// A step rewrites the words of the step before with ones, and the keys and values of other row groups are the only words whose
// writers a reader does not follow closely: it waits for all groups once a step (P2), so what it knows of one is that the step
// before the last wait has ended there.  With three sets that is enough: a step reads words that were rewritten two steps ago.
// With two a group that ran a whole step ahead could have read another's words of two steps ago.
constexpr int kSets = 3;
constexpr int OFF_PW = 0, PW_B = 4 * kProgressBytes;  // progress words (one set only)
constexpr int OFF_XT = 0, OFF_HE = OFF_XT + 4 * XT_B, OFF_HID = OFF_HE + 4 * HE_B, HEAD_B = OFF_HID + 4 * X_B;
constexpr int Q_B = H * 2048, KV_B = G * 2 * 4096, ATT_B = KO * 1024, HF_B = KF * 1024;
constexpr int OFF_Q = 0, OFF_K = OFF_Q + 4 * Q_B, OFF_V = OFF_K + KV_B, OFF_ATT = OFF_V + KV_B, OFF_X1 = OFF_ATT + 4 * ATT_B,
              OFF_HF = OFF_X1 + 4 * X_B, OFF_X2 = OFF_HF + 4 * HF_B, LAYER_B = OFF_X2 + 4 * X_B;

// LDS: two partial buffers (phases alternate, so one barrier per phase is enough), then small tables
constexpr int PART_B = 64 * 1024;
constexpr int L_RS = 2 * PART_B;                     // sums of squares of the 16 rows, three parts, two buffers
constexpr int L_M = L_RS + 2 * 48 * 4;               // attention: tile maxima [wave][16], sums
constexpr int L_L = L_M + kWaves * 16 * 4;
constexpr int L_XT = L_L + kWaves * 16 * 4;          // x_t [32][16]
constexpr int L_WS = L_XT + A * 16 * 4;              // this block's rows of the suffix embedding [16][32]
constexpr int L_Q = L_WS + 16 * A * 4;               // cross layers: the query tile in operand order
constexpr int L_ROPE = L_Q + 2048;                   // (cos, sin) pairs of P1's (128) and of the cross q's (256) column pairs
constexpr int L_KV = L_ROPE + 384 * 16;              // prefix caches of every layer
constexpr int LDS_B = L_KV + kSvMaxLayers * (int)sizeof(SvCache);

__global__ __launch_bounds__(kThreads) void sv_denoise_kernel(SvDenoiseArgs a) {
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
  const int set_b = HEAD_B + a.layers * LAYER_B;
  cx.rs = make_rsrc(a.xchg, PW_B + (unsigned)kSets * (unsigned)set_b);
  const rsrc_t wr = make_rsrc(a.blob, (unsigned)a.layers * W_LAYER + E * 4);
  int &tid = cx.tid, &lane = cx.lane, &wave = cx.wave, &g = cx.g, &r = cx.r;
  const int nsuf = (a.M + 31) >> 5, tp = (a.P + 31) >> 5;

  float* const ldsf = (float*)lds;
  float* const sM = ldsf + L_M / 4;
  float* const sL = ldsf + L_L / 4;
  float* const sX = ldsf + L_XT / 4;
  float* const sW = ldsf + L_WS / 4;
  int buf = 0;  // partial buffer of the current phase
  auto part = [&]() { return lds + buf * PART_B; };
  auto sq_s = [&]() { return ldsf + L_RS / 4 + buf * 48; };

  // progress: phase ids grow along the run; `announce` some time before this block's output of a phase leaves, `gate` before asking
  // for data that the blocks `from` .. (and the extra ones) produce in phase `id`
  enum { PH_E0, PH_E1, PH_E2, PH_P1, PH_P2, PH_P3, PH_P4, PH_P5 };
  auto id_of = [&](int step, int l, int ph) { return (step * (a.layers + 1) + l + 1) * 8 + ph; };  // E phases: l = -1
  // (everything asked for has arrived by then: told so, the compiler does not wait for the progress store's acknowledgement
  // where it next uses a loaded register)
  auto arrived = [&]() { __builtin_amdgcn_s_waitcnt(0x0f70); };  // vmcnt(0)
  auto announce = [&](int id) {
    if (tid == 0) st_x(cx.rs, (unsigned)id, 0, OFF_PW + rt * kProgressBytes + c * 128);
  };
  auto gate = [&](unsigned long long who, int id) {
    const unsigned mine = wave < 8 ? (unsigned)(who >> (8 * wave)) & 0xff : 0;
    if (mine) watch<8>(cx, (const char*)a.xchg + OFF_PW + rt * kProgressBytes + wave * 1024, mine, id);
    block_barrier();
  };
  constexpr unsigned long long kHid = (1ull << NE) - 1, kAtt = ((1ull << H) - 1) << AT, kAll = ~0ull, kQkv = kHid | (1ull << AT) | (15ull << 60),
                               kAct = (1ull << A) - 1;

  // Addresses are a few instructions to form, and there are hundreds of them: without this the compiler forms them all
  // once, ahead of the loops, and spills them.  Every phase starts from values it cannot see through.
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
  if (tid < 384) {
    // rotary factors of row t / 8, columns n = 2 (t & 7) and the next: 0..127 P1 (columns 16 (c & 1) + n of a head half),
    // 128..383 the cross q (16 u + n)
    const int t = tid < 128 ? tid : tid - 128;
    const int mg = rt * 16 + ((t >> 3) & 15), mc = mg < a.M ? mg : a.M - 1;
    int p = tid < 128 ? a.pos[mc] : a.pos0[mc];
    p = p < 0 ? 0 : (p > a.positions - 1 ? a.positions - 1 : p);
    const int f = 16 * (tid < 128 ? ((c < 60 ? (c == AT ? NQ - 1 : c) : c - 15) & 1) : t >> 7) + 2 * (t & 7);
    f32x2* const o = (f32x2*)(lds + L_ROPE + tid * 16);
    o[0] = *(const f32x2*)(a.rope_cos + (size_t)p * (D / 2) + f);
    o[1] = *(const f32x2*)(a.rope_sin + (size_t)p * (D / 2) + f);
  }
  if (tid < a.layers * (int)(sizeof(SvCache) / 4)) ((int*)(lds + L_KV))[tid] = ((const int*)a.cache)[tid];
  // step 0's x_t, the suffix embedding's weight rows of this block
  if (tid < A * 16) {
    const int j = tid >> 4, m = rt * 16 + (tid & 15);
    sX[tid] = m < a.M ? a.x0[m * A + j] : 0.f;
    if (c < NE) sW[tid] = a.emb_w[(16 * c + (tid >> 5)) * A + (tid & 31)];
  }
  float xcol = 0.f;  // E0: x_t of row tid (< 16), column c
  if (tid < 16 && c < A && rt * 16 + tid < a.M) xcol = a.x0[(rt * 16 + tid) * A + c];
  // the half k tile behind the last hidden column, and the three unused sums of squares of a row, are zeros for good
  if (c == NE - 1) {
    const i32x4 z = {0, 0, 0, 0};
    for (int i = wave; i < 1 + 2 * a.layers; i += kWaves)
      for (int set = 0; set < kSets; ++set) {
        const int b = PW_B + set * set_b + (i == 0 ? OFF_HID : HEAD_B + ((i - 1) >> 1) * LAYER_B + ((i & 1) ? OFF_X1 : OFF_X2)) + rt * X_B;
        if (lane < 32) st_x4(cx.rs, z, lane * 16, b + (KE - 1) * 1024 + 512);
        if (lane < 48) st_x(cx.rs, 0, lane * 4, b + KE * 1024 + NE * 64);
      }
  }
  // visibility of this wave's prefix key tile: keys 8 g .. 8 g + 7 of it in this lane; bits 8..15: keys that exist
  unsigned vis_in;
  {
    const int key = 32 * wave + (lane & 31);
    const bool ok = key < a.P && (a.pad == nullptr || a.pad[key < a.P ? key : 0] != 0);
    const unsigned bits = (unsigned)__builtin_amdgcn_ballot_w64(ok);
    const int left = a.P - (32 * wave + 8 * g);
    vis_in = ((bits >> (8 * g)) & 0xffu) | ((left >= 8 ? 0xffu : (left > 0 ? (1u << left) - 1u : 0u)) << 8);
  }

  auto q_share = [&]() { return c < NE ? c : (c >= 60 ? c - 15 : (c == AT ? NQ - 1 : -1)); };
  // where this thread's words of P1 go (relative to the layer's buffers): the two words of a rotary pair, or of two V^T tiles
  auto p1_off = [&](const Own& ow, int& off0, int& step) {
    const int u = q_share(), hh = u >> 1, uu = u & 1;
    if (hh < H) {
      off0 = OFF_Q + rt * Q_B + hh * 2048 + uu * 512 + ow.word;
      step = 1024;
    } else if (hh < H + G) {
      const int kk = (rt & 1) * 16 + ow.m, row = 4 * (kk >> 3) + (kk & 3), sub = (kk >> 2) & 1;
      off0 = OFF_K + (((hh - H) * 2 + (rt >> 1)) * 2 + sub) * 2048 + (2 * uu + (ow.n >> 3)) * 256 + row * 16 + (ow.n & 7) * 2;
      step = 1024;
    } else {  // V^T: keys n, n + 1 of column m
      off0 = OFF_V + ((hh - H - G) * 2 + (rt >> 1)) * 4096 + uu * 1024 + (rt & 1) * 512 + ow.word;
      step = 2048;
    }
  };
  // ... and of the other phases: scalar parts of the addresses
  auto att_s = [&]() { return OFF_ATT + rt * ATT_B + 2 * (c - AT) * 1024; };       // P2
  auto x_s = [&]() { return rt * X_B + (c >> 1) * 1024 + (c & 1) * 512; };  // E2 / P3 / P5: threads < 256
  auto ss_s = [&]() { return rt * X_B + KE * 1024 + c * 64; };
  auto h_s = [&]() { return OFF_HF + rt * HF_B + c * 1024; };               // P4: threads < 512
  auto he_s = [&]() { return OFF_HE + rt * HE_B + c * 1024; };              // E1: threads < 256
  auto xt_s = [&]() { return OFF_XT + rt * XT_B + c * 64; };                // E0: threads < 16

  float res0 = 0.f, res1 = 0.f;  // the residual stream: row m, columns 16 c + n, n + 1 (threads < 256 of blocks < 45)
  // hidden values of threads < 256 into an exchange buffer: times the next norm's weight, squares beside
  auto put_hidden = [&](const Own& ow, f32x2 nw, int base) {
    if (ow.put) st_x(cx.rs, pack_bf16x2(res0 * nw[0], res1 * nw[1]), ow.word, base + x_s());
    const float ss = own_row_sum(fmaf(res0, res0, res1 * res1));
    if (ow.put && ow.n == 0) st_x(cx.rs, __float_as_uint(ss), ow.m * 4, base + ss_s());
  };
  auto poison_hidden = [&](const Own& ow, int base) {
    if (ow.put) st_x(cx.rs, 0xffffffffu, ow.word, base + x_s());
    if (ow.put && ow.n == 0) st_x(cx.rs, 0xffffffffu, ow.m * 4, base + ss_s());
  };
  // the sums of squares of the 16 rows of a hidden buffer into LDS: an extra piece of the last three waves, 16 of the 48
  // column shares each, asked for with the wave's share of the rows and looked at after it
  auto ask_stats = [&](i32x4& st, int base) {
    const int k = wave - (kWaves - 3);
    st = ld_x(cx.rs, lane_at(k >= 0, lane * 16), base_at(k >= 0, base + rt * X_B + KE * 1024 + k * 1024));
  };
  auto take_stats = [&](i32x4& st, int base) {
    const int k = wave - (kWaves - 3);
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
  auto rstd_of = [&](int m) { return rsqrtf((sq_s()[m] + sq_s()[16 + m] + sq_s()[32 + m]) * (1.0f / E) + a.eps); };

  // a rotary pair of two columns -> two words
  auto rotate = [&](f32x2 va, f32x2 vb, int slot, unsigned& wa, unsigned& wb) {
    const f32x2 cs = ((const f32x2*)(lds + L_ROPE + slot * 16))[0], sn = ((const f32x2*)(lds + L_ROPE + slot * 16))[1];
    float ra[2], rb[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float x = round_bf16(va[j]), y = round_bf16(vb[j]);
      ra[j] = sub_rn(mul_rn(x, cs[j]), mul_rn(y, sn[j]));
      rb[j] = add_rn(mul_rn(y, cs[j]), mul_rn(x, sn[j]));
    }
    wa = pack_bf16x2(ra[0], ra[1]);
    wb = pack_bf16x2(rb[0], rb[1]);
  };

  // this wave's 32 prefix keys: K rows as the A operand (row 4 q + i of tile `sub` is key 8 q + 4 sub + i, so that a
  // lane's scores are eight consecutive keys: the B operand of the second product), V^T rows as its A operand
  auto load_K = [&](i32x4 (&kf)[2][2], int l, bool lo) {
    const SvCache& L = ((const SvCache*)(lds + L_KV))[l];
    const int sl = __builtin_amdgcn_readfirstlane(L.k_sl), sh = __builtin_amdgcn_readfirstlane(L.k_sh), kvh = (c - AT) / (H / G);
    const rsrc_t rk = make_rsrc(uniform_ptr(lo ? L.k_lo : L.k), 2u * ((a.P - 1) * sl + (G - 1) * sh + D));
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      int key = 32 * wave + 8 * (r >> 2) + 4 * sub + (r & 3);
      if (key > a.P - 1) key = a.P - 1;  // masked below
      const int voff = 2 * (key * sl + 8 * g);
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) kf[sub][ks] = ld_w_if(wave < tp, rk, voff, 2 * kvh * sh + 64 * ks);
    }
  };
  auto load_V = [&](i32x4 (&vf)[4], int l, bool lo) {
    const SvCache& L = ((const SvCache*)(lds + L_KV))[l];
    const int sd = __builtin_amdgcn_readfirstlane(L.vt_sd), sh = __builtin_amdgcn_readfirstlane(L.vt_sh), kvh = (c - AT) / (H / G);
    const rsrc_t rv = make_rsrc(uniform_ptr(lo ? L.vt_lo : L.vt), 2u * ((G - 1) * sh + (D - 1) * sd + 32 * tp));
    const int voff = 2 * (r * sd + 8 * g + 32 * wave);
#pragma unroll
    for (int t = 0; t < 4; ++t) vf[t] = ld_w_if(wave < tp, rv, voff, 2 * (kvh * sh + 16 * t * sd));
  };

  // attention of this block's head: qb = the 16 queries as B operands, this wave's key tile in kf / vf (and kl / vl)
  auto attend = [&](const i32x4 (&qb)[2], const i32x4 (&kf)[2][2], const i32x4 (&kl)[2][2], const i32x4 (&vf)[4], const i32x4 (&vl)[4], int base,
                    int id, auto cross_c, int nw) {
    constexpr bool cross = decltype(cross_c)::value;
    const bool has = wave < nw;
    float p[8];
    float tmax = -INFINITY;
    if (has) {
      f32x4 s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int sub = 0; sub < 2; ++sub)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          s[sub] = mfma(kf[sub][ks], qb[ks], s[sub]);
          if (cross) s[sub] = mfma(kl[sub][ks], qb[ks], s[sub]);
        }
      unsigned vis = vis_in, in = vis_in >> 8;
      if (wave >= tp) {  // action tokens: causal
        const int k0 = 32 * (wave - tp) + 8 * g, left = a.M - k0, see = rt * 16 + r - k0 + 1;
        in = left >= 8 ? 0xffu : (left > 0 ? (1u << left) - 1u : 0u);
        vis = see >= 8 ? 0xffu : (see > 0 ? (1u << see) - 1u : 0u);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float sv = s[e >> 2][e & 3] * 0.125f;
        sv = (vis >> e) & 1u ? sv : kF32Min;
        sv = (in >> e) & 1u ? sv : -INFINITY;
        p[e] = sv;
        tmax = fmaxf(tmax, sv);
      }
      tmax = max16(tmax);
      tmax = max32(tmax);
    }
    if (lane < 16) sM[wave * 16 + r] = tmax;
    block_barrier();
    {
      f32x4 o[4];
      float ls = 0.f;
#pragma unroll
      for (int t = 0; t < 4; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (has) {
        const float bm = max16(max32(fmaxf(fmaxf(sM[g * 16 + r], sM[(g + 4) * 16 + r]), fmaxf(sM[(g + 8) * 16 + r], sM[(g + 12) * 16 + r]))));
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          p[e] = __expf(p[e] - bm);
          ls += p[e];
        }
        ls = row_sum(ls);
        const i32x4 ph = {(int)pack_bf16x2(p[0], p[1]), (int)pack_bf16x2(p[2], p[3]), (int)pack_bf16x2(p[4], p[5]), (int)pack_bf16x2(p[6], p[7])};
        i32x4 pl = ph;
        if (cross) {
          float lo[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) lo[e] = p[e] - round_bf16(p[e]);
          pl = i32x4{(int)pack_bf16x2(lo[0], lo[1]), (int)pack_bf16x2(lo[2], lo[3]), (int)pack_bf16x2(lo[4], lo[5]), (int)pack_bf16x2(lo[6], lo[7])};
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          o[t] = mfma(vf[t], ph, o[t]);
          if (cross) {
            o[t] = mfma(vl[t], ph, o[t]);
            o[t] = mfma(vf[t], pl, o[t]);
          }
        }
      }
      if (lane < 16) sL[wave * 16 + r] = ls;
#pragma unroll
      for (int t = 0; t < 4; ++t) *(f32x4*)(part() + (wave * 4 + t) * 1024 + part_slot(cx)) = o[t];
    }
    block_barrier();
    announce(id);
    {
      const Own ow = own_of(tid);
      const f32x2 o = sum_part<kWaves, 4>(part(), 0, wave >> 2, ow);
      const float* const l0 = sL + ow.from * 16 + ow.m;
      const float inv = 1.0f / sum16(sum32((l0[0] + l0[8 * 16]) + (l0[4 * 16] + l0[12 * 16])));
      if (ow.put) st_x(cx.rs, pack_bf16x2(o[0] * inv, o[1] * inv), (wave >> 2) * 512 + ow.word, base + att_s());
    }
    buf ^= 1;
  };

  // ---------------- P1: q | k | v ----------------
  // Weights.  Loads return in order, so a weight asked for shortly before a phase's input delays that input; and a layer's
  // weights asked for phase by phase come in bursts the fabric needs longer for than the phases last.  So P1's are asked
  // for in P4 of the layer before, and the rest of a layer's behind P1 (behind the attention in its blocks): they arrive
  // while the attention runs.
  i32x4 wA[2][2], wB[2], wC[3], wD[2];
  f32x2 nwp, scg, scu, scd, nwd;  // the next norm's weight (P3, P5), column scales
  auto load_A = [&](int l, bool any) {
    const int u = q_share(), wb = l * W_LAYER + W_QKV + 2 * u * KE * 1024;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int s = wave + 16 * i;
#pragma unroll
      for (int t = 0; t < 2; ++t) wA[t][i] = ld_w_if(any && u >= 0 && s < KE, wr, lane * 16, wb + (t * KE + s) * 1024);
    }
  };
  auto load_rest = [&](int l) {
    const int wl = l * W_LAYER, n4 = own_of(tid).n * 4;
    const bool hid = c < NE;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int s = wave + 16 * i;
      wB[i] = ld_w_if(hid && s < KO, wr, lane * 16, wl + W_O + (c * KO + s) * 1024);
    }
    nwp = ld_f2_if(hid, wr, n4, wl + W_NPOST + 64 * c);
    const int p = 2 * c + (wave >> 3), f = 64 * ((wave >> 2) & 1) + n4;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int s = (wave & 7) + 8 * i;
      wC[i] = ld_w_if(s < KE, wr, lane * 16, wl + W_GU + (p * KE + s) * 1024);
    }
    scg = ld_f2(wr, f, wl + W_SG + 128 * c);
    scu = ld_f2(wr, f, wl + W_SU + 128 * c);
#pragma unroll
    for (int i = 0; i < 2; ++i) wD[i] = ld_w_if(hid, wr, lane * 16, wl + W_D + (c * (KF / 2) + wave + 16 * i) * 1024);
    scd = ld_f2_if(hid, wr, n4, wl + W_SD + 64 * c);
    // the norm that reads P5's rows: the next layer's, behind the last one the closing one
    nwd = ld_f2_if(hid, wr, n4, l + 1 < a.layers ? wl + W_LAYER + W_NIN + 64 * c : a.layers * W_LAYER + 64 * c);
  };
  auto phase1 = [&](int l, int in_base, int base, int in_id, int id, bool rest) {
    i32x4 x[2];
    const int u = q_share();
    gate(kHid, in_id);
    i32x4 st;
    wait_tiles<2, KE>(x, cx, in_base + rt * X_B, wave, 16, [&] { ask_stats(st, in_base); });
    arrived();
    announce(id);
    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    const bool vt = (u >> 1) >= H + G;  // V^T: the operands swapped, a lane then owns a column and four consecutive keys
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int t = 0; t < 2; ++t) acc[t] = vt ? mfma(x[i], wA[t][i], acc[t]) : mfma(wA[t][i], x[i], acc[t]);
#pragma unroll
    for (int t = 0; t < 2; ++t) *(f32x4*)(part() + (wave * 2 + t) * 1024 + part_slot(cx)) = acc[t];
    take_stats(st, in_base);
    block_barrier();
    if (tid < 256) {
      const Own ow = own_of(tid);
      f32x2 va = sum_part<16, 2>(part(), 0, 0, ow), vb = sum_part<16, 2>(part(), 0, 1, ow);
      unsigned wa, wb2;
      if (!vt) {
        const float rstd = rstd_of(ow.m);
        rotate(va * rstd, vb * rstd, ow.m * 8 + (ow.n >> 1), wa, wb2);
      } else {
        const float r0 = rstd_of(ow.n), r1 = rstd_of(ow.n + 1);
        wa = pack_bf16x2(va[0] * r0, va[1] * r1);
        wb2 = pack_bf16x2(vb[0] * r0, vb[1] * r1);
      }
      int off0, step;
      p1_off(ow, off0, step);
      if (ow.put) {
        st_x(cx.rs, wa, off0, base);
        st_x(cx.rs, wb2, off0 + step, base);
      }
    }
    if (rest) load_rest(l);
    buf ^= 1;
  };

  block_barrier();

  int cur = PW_B, oth = PW_B + (kSets - 1) * set_b;  // this step's set and the one of the step before
  for (int step = 0; step <= a.steps; ++step, oth = cur, cur = cur == PW_B + (kSets - 1) * set_b ? PW_B : cur + set_b) {
    // ---------------- E0: the previous step's velocity and Euler update ----------------
    fresh();
    if (step > 0) {
      if (c < A) {
        const int in_base = oth + HEAD_B + (a.layers - 1) * LAYER_B + OFF_X2;
        i32x4 v[2];
        f32x4 wa[2][2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int s = wave + 16 * i < KE ? wave + 16 * i : KE - 1;
          const int k = 32 * s + 8 * g < E ? 32 * s + 8 * g : E - 8;  // (behind the last column the input is zero)
          wa[i][0] = *(const f32x4*)(a.act_w + c * E + k);
          wa[i][1] = *(const f32x4*)(a.act_w + c * E + k + 4);
        }
        const float bias = a.act_b ? a.act_b[c] : 0.f;
        pin();
        gate(kHid, id_of(step - 1, a.layers - 1, PH_P5));
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
          const float vel = v0 * rstd_of(tid) + bias;
          xcol = add_rn(xcol, mul_rn(a.dt, vel));
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
      if (c < NE) {
        gate(kAct, id_of(step, -1, PH_E0));
        if (wave < 2) {
          i32x4 v[1];
          const int voff[1] = {lane * 16}, soff[1] = {cur + OFF_XT + rt * XT_B + wave * 1024};
          wait_x<1>(v, cx, voff, soff, [] {});
          *(i32x4*)(lds + L_XT + wave * 1024 + lane * 16) = v[0];
        }
        block_barrier();
      }
    }
    // ---------------- E1, E2: suffix embedding ----------------
    fresh();
    if (c < NE) {
      const Own ow = own_of(tid);
      i32x4 wt[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const int j = wave + 16 * i < NE ? wave + 16 * i : NE - 1;
        wt[i] = *(const i32x4*)(a.time_w + (size_t)(16 * c + r) * E + 16 * j + 4 * g);
      }
      const f32x2 tb = *(const f32x2*)(a.time_b + 16 * c + ow.n), nw = ld_f2(wr, ow.n * 4, W_NIN + 64 * c);
      announce(id_of(step, -1, PH_E1));
      if (tid < 256) {
        const int n = ((tid >> 6) << 2) | (tid & 3), m = (tid >> 2) & 15;
        float e0 = 0.f, e1 = 0.f;
#pragma unroll
        for (int j = 0; j < A; j += 2) {
          e0 = fmaf(sX[j * 16 + m], sW[n * A + j], e0);
          e1 = fmaf(sX[(j + 1) * 16 + m], sW[n * A + j + 1], e1);
        }
        float e = e0 + e1 + a.emb_b[step * E + 16 * c + n];
        e = e / (1.0f + expf(-e));
        st_x(cx.rs, __float_as_uint(e), tid * 4, cur + he_s());
      }
      i32x4 v[3];
      gate(kHid, id_of(step, -1, PH_E1));
      wait_tiles<3, NE>(v, cx, cur + OFF_HE + rt * HE_B, wave, 16, [] {});
      arrived();
      announce(id_of(step, -1, PH_E2));
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__int_as_float(wt[i][e]), __int_as_float(v[i][e]), acc, 0, 0, 0);
      *(f32x4*)(part() + wave * 1024 + part_slot(cx)) = acc;
      block_barrier();
      if (tid < 256) {
        const f32x2 s = sum_part<16, 1>(part(), 0, 0, ow);
        res0 = s[0] + tb[0];
        res1 = s[1] + tb[1];
        put_hidden(ow, nw, cur + OFF_HID);
      }
      buf ^= 1;
    }
    load_A(0, true);

    for (int l = 0; l < a.layers; ++l) {
      const int base = cur + HEAD_B + l * LAYER_B, obase = oth + HEAD_B + l * LAYER_B;
      const int in_base = l == 0 ? cur + OFF_HID : base - LAYER_B + OFF_X2;  // the layer's input rows
      const bool cross = (a.cross_mask >> l) & 1;
      const int in_id = l == 0 ? id_of(step, -1, PH_E2) : id_of(step, l - 1, PH_P5);
      fresh();
      if (c >= AT && c < AT + H && !cross) {
        // ---------------- P2: self attention (and the odd share of P1) ----------------
        // Keys of later rows are masked.  Only the step's first self layer waits for those of all row groups (kSets), the others
        // for the rows up to their own (the loop 1984 -> 1969 us)
        const bool sync = (~a.cross_mask & ((1u << l) - 1)) == 0;
        const int last = sync ? 3 : rt, nw = tp + (sync ? nsuf : (rt >> 1) + 1), h = c - AT;
        i32x4 kf[2][2], vf[4], v[10];
        load_K(kf, l, false);
        load_V(vf, l, false);
        pin();
        if (c == AT) phase1(l, in_base, base, in_id, id_of(step, l, PH_P1), false);
        gate(kQkv, id_of(step, l, PH_P1));
        {
          // the query tile; for the waves behind the prefix also the action tokens' own keys: 32 of them are the rows of
          // two row groups (a group that does not exist: repeat)
          const int j = wave - tp, kvh = h / (H / G);
          const bool own = wave >= tp && wave < nw, one = 16 * (2 * j + 1) >= a.M || 2 * j + 1 > last;
          const int rr = one ? (r & 7) : r, gg = one ? (g & 1) : g;
          int voff[10], soff[10];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            voff[2 + i] = lane_at(own, (g * 16 + rr) * 16);
            soff[2 + i] = base_at(own, base + OFF_K + (kvh * 2 + j) * 4096 + i * 1024);  // [sub][k step]
            voff[6 + i] = lane_at(own, (gg * 16 + r) * 16);
            soff[6 + i] = base_at(own, base + OFF_V + (kvh * 2 + j) * 4096 + i * 1024);
          }
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            voff[i] = lane_at(wave < nw, lane * 16);
            soff[i] = base_at(wave < nw, base + OFF_Q + rt * Q_B + h * 2048 + i * 1024);
          }
          wait_all<10>(v, cx, voff, soff);
          if (own) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              kf[i >> 1][i & 1] = v[2 + i];
              vf[i] = v[6 + i];
            }
          }
        }
        const i32x4 qb[2] = {v[0], v[1]};
        attend(qb, kf, kf, vf, vf, base, id_of(step, l, PH_P2), std::false_type{}, nw);
        load_rest(l);
      } else if (q_share() >= 0 && !cross) {
        // ---------------- P1 ----------------
        phase1(l, in_base, base, in_id, id_of(step, l, PH_P1), true);
      } else if (c >= AT && c < AT + H) {
        // ---------------- P2: cross attention with its query projection ----------------
        i32x4 x[2], w[4][2], kf[2][2], kl[2][2], vf[4], vl[4];
        const int wb = l * W_LAYER + W_QKV + 4 * (c - AT) * KE * 1024;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int s = wave + 16 * i;
#pragma unroll
          for (int t = 0; t < 4; ++t) w[t][i] = ld_w_if(s < KE, wr, lane * 16, wb + (t * KE + s) * 1024);
        }
        load_K(kf, l, false);
        load_K(kl, l, true);
        pin();
        gate(kHid, in_id);
        i32x4 st;
        wait_tiles<2, KE>(x, cx, in_base + rt * X_B, wave, 16, [&] { ask_stats(st, in_base); });
        f32x4 acc[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = mfma(w[t][1], x[1], mfma(w[t][0], x[0], f32x4{0.f, 0.f, 0.f, 0.f}));
#pragma unroll
        for (int t = 0; t < 4; ++t) *(f32x4*)(part() + (wave * 4 + t) * 1024 + part_slot(cx)) = acc[t];
        take_stats(st, in_base);
        block_barrier();
        if (tid < 512) {
          const Own ow = own_of(tid);
          const float rstd = rstd_of(ow.m);
          const int u = wave >> 2;
          const f32x2 va = sum_part<16, 4>(part(), 0, u, ow) * rstd, vb = sum_part<16, 4>(part(), 0, 2 + u, ow) * rstd;
          unsigned wa, wb2;
          rotate(va, vb, 128 + u * 128 + ow.m * 8 + (ow.n >> 1), wa, wb2);
          if (ow.put) {
            *(unsigned*)(lds + L_Q + u * 512 + ow.word) = wa;
            *(unsigned*)(lds + L_Q + 1024 + u * 512 + ow.word) = wb2;
          }
        }
        buf ^= 1;
        load_V(vf, l, false);
        load_V(vl, l, true);
        pin();
        block_barrier();
        const i32x4 qb[2] = {*(const i32x4*)(lds + L_Q + lane * 16), *(const i32x4*)(lds + L_Q + 1024 + lane * 16)};
        attend(qb, kf, kl, vf, vl, base, id_of(step, l, PH_P2), std::true_type{}, tp);
        load_rest(l);
      } else {
        load_rest(l);
      }
      // ---------------- P3: output projection, residual ----------------
      const bool next_self = l + 1 < a.layers && !((a.cross_mask >> (l + 1)) & 1);
      fresh();
      if (c < NE) {
        const Own ow = own_of(tid);
        i32x4 v[2];
        gate(kAtt, id_of(step, l, PH_P2));
        wait_tiles<2, KO>(v, cx, base + OFF_ATT + rt * ATT_B, wave, 16, [] {});
        arrived();
        const f32x4 acc = mfma(wB[1], v[1], mfma(wB[0], v[0], f32x4{0.f, 0.f, 0.f, 0.f}));
        *(f32x4*)(part() + wave * 1024 + part_slot(cx)) = acc;
        announce(id_of(step, l, PH_P3));
        block_barrier();
        if (tid < 256) {
          const f32x2 s = sum_part<16, 1>(part(), 0, 0, ow);
          res0 = s[0] + res0;
          res1 = s[1] + res1;
          put_hidden(ow, nwp, base + OFF_X1);
        }
        buf ^= 1;
      }
      // ---------------- P4: gate / up ----------------
      fresh();
      {
        i32x4 v[3];
        bf16x8 wg[3], wu[3];
        gate(kHid, id_of(step, l, PH_P3));
        i32x4 st;
        wait_tiles<3, KE>(v, cx, base + OFF_X1 + rt * X_B, wave & 7, 8, [&] {
          ask_stats(st, base + OFF_X1);
          // the weights were asked for long before: decoded while the input is on its way
#pragma unroll
          for (int i = 0; i < 3; ++i) {
            wg[i] = fp8x8_to_bf16x8(wC[i][0], wC[i][1]);
            wu[i] = fp8x8_to_bf16x8(wC[i][2], wC[i][3]);
          }
        });
        arrived();
        announce(id_of(step, l, PH_P4));
        f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wg[i], as_bf16x8(v[i]), acc[0], 0, 0, 0);
          acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wu[i], as_bf16x8(v[i]), acc[1], 0, 0, 0);
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) *(f32x4*)(part() + (wave * 2 + t) * 1024 + part_slot(cx)) = acc[t];
        take_stats(st, base + OFF_X1);
        block_barrier();
        if (tid < 512) {
          const Own ow = own_of(tid);
          const int pair = wave >> 2;
          const float rstd = rstd_of(ow.m);
          const f32x2 gt = sum_part<8, 2>(part(), 8 * pair, 0, ow) * rstd * scg, up = sum_part<8, 2>(part(), 8 * pair, 1, ow) * rstd * scu;
          float h[2];
#pragma unroll
          for (int j = 0; j < 2; ++j) h[j] = silu_f(gt[j]) * up[j];
          if (ow.put) st_x(cx.rs, pack_bf16x2(h[0], h[1]), pair * 512 + ow.word, base + h_s());
        }
        pin();
        load_A(l + 1, next_self);
        pin();
        buf ^= 1;
      }
      // ---------------- P5: down projection, residual ----------------
      fresh();
      if (c < NE) {
        const Own ow = own_of(tid);
        i32x4 v[4];
        bf16x8 wd[4];
        gate(kAll, id_of(step, l, PH_P4));
        int voff[4], soff[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          voff[i] = lane * 16;
          soff[i] = base + OFF_HF + rt * HF_B + (2 * (wave + 16 * (i >> 1)) + (i & 1)) * 1024;
        }
        wait_x<4>(v, cx, voff, soff, [&] {
#pragma unroll
          for (int i = 0; i < 4; ++i) wd[i] = fp8x8_to_bf16x8(wD[i >> 1][2 * (i & 1)], wD[i >> 1][2 * (i & 1) + 1]);
        });
        arrived();
        announce(id_of(step, l, PH_P5));
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wd[i], as_bf16x8(v[i]), acc, 0, 0, 0);
        *(f32x4*)(part() + wave * 1024 + part_slot(cx)) = acc;
        block_barrier();
        if (tid < 256) {
          const f32x2 s = sum_part<16, 1>(part(), 0, 0, ow) * scd;
          res0 = s[0] + res0;
          res1 = s[1] + res1;
          put_hidden(ow, nwd, base + OFF_X2);
        }
        buf ^= 1;
      }
      // ---------------- the set of the step before: this layer's words were read, back to all ones ----------------
      const unsigned ones = 0xffffffffu;
      fresh();
      if (tid < 256) {
        const Own ow = own_of(tid);
        if (!cross && q_share() >= 0) {
          int off0, pstep;
          p1_off(ow, off0, pstep);
          if (ow.put) {
            st_x(cx.rs, ones, off0, obase);
            st_x(cx.rs, ones, off0 + pstep, obase);
          }
        }
        if (c < NE) {
          poison_hidden(ow, obase + OFF_X1);
          // (the closing layer's hidden rows of that set are read by this step's E0: they have been by now)
          poison_hidden(ow, obase + OFF_X2);
          if (l == 0) poison_hidden(ow, oth + OFF_HID);
        }
      }
      if (c >= AT && c < AT + H && tid < 512) st_x(cx.rs, ones, tid * 4, obase + att_s());
      if (tid < 256) st_x(cx.rs, ones, tid * 4, obase + h_s());
      if (l == 0) {
        if (c < NE && tid < 256) st_x(cx.rs, ones, tid * 4, oth + he_s());
        if (c < A && tid < 16) st_x(cx.rs, ones, tid * 4, oth + xt_s());
      }
    }
  }
}

// one layer's weights out of the packed 32 x 32 tiles into the blob, 16 bytes per thread
__global__ void sv_pack_kernel(SvPackArgs a) {
  constexpr int C_QKV = (W_O - W_QKV) / 16, C_O = C_QKV + (W_GU - W_O) / 16, C_GU = C_O + (W_D - W_GU) / 16, C_D = C_GU + (W_SG - W_D) / 16,
                C_ALL = C_D + (2 * F + 3 * E) / 4;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < C_ALL; i += gridDim.x * blockDim.x) {
    const int lane = i & 63, g = lane >> 4, r = lane & 15;
    auto t16 = [&](const uint8_t* w, int KT, int nt, int nh, int s) {
      return *(const i32x4*)(w + ((size_t)(nt * KT + s)) * 2048 + (g & 1) * 1024 + ((g >> 1) * 32 + nh * 16 + r) * 16);
    };
    auto t8 = [&](const uint8_t* w, int KT, int nt, int nh, int s) {
      return *(const i32x2*)(w + ((size_t)(nt * KT + s)) * 1024 + ((g >> 1) * 32 + nh * 16 + r) * 16 + (g & 1) * 8);
    };
    i32x4 v = {0, 0, 0, 0};
    int dst;
    if (i < C_QKV) {
      const int piece = i >> 6, s = piece % KE, t = piece / KE;
      if (a.cross) {
        if (t < H * 4) v = t16(a.wqkv, KE, t >> 1, t & 1, s);
      } else {
        v = t16(a.wqkv, KE, 2 * (t >> 2) + (t & 1), (t >> 1) & 1, s);  // share c = t / 2: head half c & 1 of both rotary halves
      }
      dst = W_QKV + i * 16;
    } else if (i < C_O) {
      const int k = i - C_QKV, piece = k >> 6, t = piece / KO;
      v = t16(a.wo, KO, t >> 1, t & 1, piece % KO);
      dst = W_O + k * 16;
    } else if (i < C_GU) {
      const int k = i - C_O, piece = k >> 6, s = piece % KE, p = piece / KE;
      const i32x2 x = t8(a.wgu, KE, 2 * (p >> 1), p & 1, s), y = t8(a.wgu, KE, 2 * (p >> 1) + 1, p & 1, s);
      v = i32x4{x[0], x[1], y[0], y[1]};
      dst = W_GU + k * 16;
    } else if (i < C_D) {
      const int k = i - C_GU, piece = k >> 6, s = 2 * (piece % (KF / 2)), t = piece / (KF / 2);
      const i32x2 x = t8(a.wd, KF, t >> 1, t & 1, s), y = t8(a.wd, KF, t >> 1, t & 1, s + 1);
      v = i32x4{x[0], x[1], y[0], y[1]};
      dst = W_D + k * 16;
    } else {
      const int k = (i - C_D) * 4;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int q = k + e;
        float f;
        if (q < F) f = a.sg[q];
        else if (q < 2 * F) f = a.su[q - F];
        else if (q < 2 * F + E) f = a.sd[q - 2 * F];
        else if (q < 2 * F + 2 * E) f = bf16_bits_to_f32(a.norm_in[q - 2 * F - E]);
        else f = bf16_bits_to_f32(a.norm_post[q - 2 * F - 2 * E]);
        v[e] = __float_as_int(f);
      }
      dst = W_SG + k * 4;
    }
    *(i32x4*)(a.blob + dst) = v;
  }
}

__global__ void fill_ones_kernel(i32x4* p, size_t n) {
  const i32x4 ones = {-1, -1, -1, -1};
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = ones;
}

}  // namespace

size_t tk_sv_denoise_exchange_bytes(int layers) { return PW_B + kSets * ((size_t)HEAD_B + (size_t)layers * LAYER_B); }
size_t tk_sv_denoise_blob_bytes() { return W_LAYER; }
int tk_sv_denoise_max_key_tiles() { return kWaves; }

int tk_launch_sv_pack(const SvPackArgs& a, hipStream_t st) {
  hipLaunchKernelGGL(sv_pack_kernel, dim3(1024), dim3(256), 0, st, a);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int tk_launch_fill_ones(void* p, size_t bytes, hipStream_t st) {
  hipLaunchKernelGGL(fill_ones_kernel, dim3(1024), dim3(256), 0, st, (i32x4*)p, bytes / 16);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int tk_launch_sv_denoise(const SvDenoiseArgs& a, hipStream_t st) {
  static std::atomic<int> raised{0};  // more LDS than a launch gets by default: raise the kernel's limit once per process
  if (!raised.load(std::memory_order_acquire)) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(&sv_denoise_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, LDS_B) != hipSuccess) return -3;
    raised.store(1, std::memory_order_release);
  }
  if (tk_launch_fill_ones(a.xchg, tk_sv_denoise_exchange_bytes(a.layers), st)) return -3;
  hipLaunchKernelGGL(sv_denoise_kernel, dim3(256), dim3(kThreads), LDS_B, st, a);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}
