// Building blocks of the persistent denoising kernels: one launch whose blocks stay resident for the whole
// flow-matching loop and hand activations to each other through memory, phase after phase.
//
// HAND-OFF.  Every word of an exchange buffer is all-ones (a NaN in bf16 and in fp32) until its producer writes it;
// consumers load the data itself with device-coherent loads and look at it: a lane that still sees an all-ones word
// asks again.  No flag, no counter, no cache flush and no wait for store acknowledgements: a hand-off costs one
// store-to-load trip through the fabric.  Measured with rounds of this kind alone (256 blocks of 16 waves, four groups of
// 64 that exchange 32 KiB among themselves, LDS reduction and barrier included): 1.37 us a round with a gate as below and the
// reduction further down (1.6 as that was at first, and then 2.4 without the gate, 2.35 with acknowledged stores and a flag per
// block instead).  Buffers come in sets, used by the denoising steps in turn; a block rewrites its words of the step
// before with ones (every path from "written" to "rewritten" runs through data that all readers produced after their
// reads), and a word is used again only where every path to its next reader runs through data that its writer produced
// after the rewriting, so that nobody finds an old one.  (The pi0.5 loop keeps a ring
// of four layers instead: a layer's words are rewritten at the end of the next one and used again two layers later.)
//
// GATE.  Loads that come back empty cost the compute unit's memory pipe as much as real ones, so nobody asks before
// there is something to expect: every block keeps a progress word (a line of its own, ever growing) and raises it 0.4 - 1 us
// before a phase's output leaves; a few waves of a consumer block watch its producers' words, the others wait at the block's
// barrier, and the first look at the data usually succeeds.  The watch goes through the scalar cache, which it empties before
// each look: vector loads return in order, and behind the 64 - 128 KiB of weights that a block has on the way at any time a
// look at a word took as long as those.  (SmolVLA's loop 2364 -> 2275 us, pi0.5's 3805 -> 3519; rounds alone with 128 KiB of
// weights from memory 3.56 -> 3.29 us, without any 1.41 -> 1.52.)  A scalar load goes through the XCD's own L2, which the store of a
// block on another XCD passes by; that looks see its word in time is measured, and what public descriptions of these parts lead to
// expect (the memory-side cache keeps track of the lines in the XCDs' L2s), but nothing rests on it: a progress word is a hint,
// and whoever has looked kLooks times goes on and asks for the data, with loads at device scope.
//
// EVERY WAIT ENDS: a wave asks at most `spin` times, then marks itself dead, goes on with what it has (ones = NaN)
// and never waits again, so the grid drains and the result holds NaNs, which the caller can see.  All blocks must be
// resident at the same time for the exchange to make progress: at most one block per compute unit is launched.
//
// OPERANDS.  The products run on v_mfma_f32_16x16x32_bf16 with the weights as the A operand (16 output columns) and 16
// activation rows as the B operand; an accumulator lane then owns one row and four consecutive output columns.
// Activations are exchanged in B operand order: 1 KiB per (16 rows, 32 columns), lane l = 16 g + m holding the 8
// columns 8 g .. of row m, so a wave's load is one contiguous KiB and needs no staging.
#pragma once
#include "tk_common.h"

namespace persist {

typedef __amdgpu_buffer_rsrc_t rsrc_t;
constexpr int kWaves = 16;
constexpr int kThreads = kWaves * 64;
constexpr int kCoherent = 16;  // sc1: device scope

struct Ctx {
  rsrc_t rs;  // the exchange buffers (all sets)
  int tid, lane, wave, g, r;
  int spin;
  int dead;  // this wave gave up a wait
};

__device__ __forceinline__ rsrc_t make_rsrc(const void* p, unsigned bytes) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000); }
__device__ __forceinline__ i32x4 ld_x(rsrc_t rs, int voff, int soff) {
  return __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, voff, soff, kCoherent));
}
__device__ __forceinline__ void st_x(rsrc_t rs, unsigned v, int voff, int soff) { __builtin_amdgcn_raw_buffer_store_b32(v, rs, voff, soff, kCoherent); }
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void st_x2(rsrc_t rs, unsigned v0, unsigned v1, int voff, int soff) {
  __builtin_amdgcn_raw_buffer_store_b64(u32x2{v0, v1}, rs, voff, soff, kCoherent);
}
__device__ __forceinline__ void st_x4(rsrc_t rs, i32x4 v, int voff, int soff) {
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rs, voff, soff, kCoherent);
}
__device__ __forceinline__ bool unset(i32x4 v) {
  const unsigned a = (unsigned)v[0] > (unsigned)v[1] ? v[0] : v[1], b = (unsigned)v[2] > (unsigned)v[3] ? v[2] : v[3];
  return (a > b ? a : b) == 0xffffffffu;
}
// a pointer every lane holds, in scalar registers
template <typename V>
__device__ __forceinline__ V* uniform_ptr(V* p) {
  const unsigned long long u = (unsigned long long)p;
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)u), hi = __builtin_amdgcn_readfirstlane((unsigned)(u >> 32));
  return (V*)(((unsigned long long)hi << 32) | lo);
}
__device__ __forceinline__ void pin() { asm volatile("" ::: "memory"); }

// progress words of a row group: [64 blocks] at 128 bytes
constexpr int kGroup = 64, kProgressBytes = kGroup * 128;
constexpr int kLooks = 400;  // at most so many at the progress words: they only say when to ask for the data
// Until the progress words of the N producers from `at` on have reached `id` (bit i of who: the i-th is one).
// N, us of a loop: SmolVLA 2275 with eight words in each of the first eight waves, 2309 with sixteen in four; pi0.5 3454 and
// 3442, 3550 with four words in all sixteen waves.  The first waves: the last ones instead, 2100 (SmolVLA) and 3505.
template <int N>
__device__ __forceinline__ void watch(const Ctx& cx, const char* at, unsigned who, int id) {
  static_assert(N == 8 || N == 16, "words of one look");
  at = uniform_ptr(at);
  for (int n = 0; n < kLooks && n <= cx.spin && !cx.dead; ++n) {
    int w[N];
    if constexpr (N == 8) {
      asm volatile(
          "s_dcache_inv\n\t"
          "s_load_dword %0, %8, 0x0\n\ts_load_dword %1, %8, 0x80\n\ts_load_dword %2, %8, 0x100\n\ts_load_dword %3, %8, 0x180\n\t"
          "s_load_dword %4, %8, 0x200\n\ts_load_dword %5, %8, 0x280\n\ts_load_dword %6, %8, 0x300\n\ts_load_dword %7, %8, 0x380\n\t"
          "s_waitcnt lgkmcnt(0)"
          : "=&s"(w[0]), "=&s"(w[1]), "=&s"(w[2]), "=&s"(w[3]), "=&s"(w[4]), "=&s"(w[5]), "=&s"(w[6]), "=&s"(w[7])
          : "s"(at)
          : "memory");
    } else {
      asm volatile(
          "s_dcache_inv\n\t"
          "s_load_dword %0, %16, 0x0\n\ts_load_dword %1, %16, 0x80\n\ts_load_dword %2, %16, 0x100\n\ts_load_dword %3, %16, 0x180\n\t"
          "s_load_dword %4, %16, 0x200\n\ts_load_dword %5, %16, 0x280\n\ts_load_dword %6, %16, 0x300\n\ts_load_dword %7, %16, 0x380\n\t"
          "s_load_dword %8, %16, 0x400\n\ts_load_dword %9, %16, 0x480\n\ts_load_dword %10, %16, 0x500\n\ts_load_dword %11, %16, 0x580\n\t"
          "s_load_dword %12, %16, 0x600\n\ts_load_dword %13, %16, 0x680\n\ts_load_dword %14, %16, 0x700\n\ts_load_dword %15, %16, 0x780\n\t"
          "s_waitcnt lgkmcnt(0)"
          : "=&s"(w[0]), "=&s"(w[1]), "=&s"(w[2]), "=&s"(w[3]), "=&s"(w[4]), "=&s"(w[5]), "=&s"(w[6]), "=&s"(w[7]),
            "=&s"(w[8]), "=&s"(w[9]), "=&s"(w[10]), "=&s"(w[11]), "=&s"(w[12]), "=&s"(w[13]), "=&s"(w[14]), "=&s"(w[15])
          : "s"(at)
          : "memory");
    }
    bool all = true;
#pragma unroll
    for (int i = 0; i < N; ++i) all = all && (!((who >> i) & 1) || w[i] >= id);
    if (all) break;
  }
}

// A lane offset behind every buffer: the range check answers such a load with zeros and asks the memory for nothing.
// Used instead of a branch around a load -- at the join behind a branch the compiler waits for the load.  The check
// compares the lane offset with (buffer size - scalar offset), so the scalar offset has to be 0 beside it: one beyond
// the buffer's end would wrap the difference around and let the load through.
constexpr int kNowhere = 0x40000000;
__device__ __forceinline__ int lane_at(bool here, int voff) { return here ? voff : kNowhere; }
__device__ __forceinline__ int base_at(bool here, int soff) { return here ? soff : 0; }

// Wait for T pieces of 1 KiB: piece i at byte offset soff[i] (wave-uniform) + voff[i] (per lane; kNowhere and 0: zeros).
// `meanwhile` runs between the first request and the first look.
template <int T, typename Fn>
__device__ __forceinline__ void wait_x(i32x4 (&v)[T], Ctx& cx, const int (&voff)[T], const int (&soff)[T], Fn meanwhile) {
#pragma unroll
  for (int i = 0; i < T; ++i) v[i] = ld_x(cx.rs, voff[i], soff[i]);
  meanwhile();
  for (int n = 0;; ++n) {
    unsigned bad = 0;
#pragma unroll
    for (int i = 0; i < T; ++i)
      if (__builtin_amdgcn_ballot_w64(unset(v[i])) != 0) bad |= 1u << i;
    if (bad == 0 || cx.dead) break;
    if (n >= cx.spin) {
      cx.dead = 1;
      break;
    }
    pin();
#pragma unroll
    for (int i = 0; i < T; ++i)
      if ((bad >> i) & 1u) v[i] = ld_x(cx.rs, voff[i], soff[i]);
  }
  pin();
}

// The same, asking for every piece again until all are there: no copies of what has arrived (many pieces, few registers).
template <int T>
__device__ __forceinline__ void wait_all(i32x4 (&v)[T], Ctx& cx, const int (&voff)[T], const int (&soff)[T]) {
  for (int n = 0;; ++n) {
    pin();
#pragma unroll
    for (int i = 0; i < T; ++i) v[i] = ld_x(cx.rs, voff[i], soff[i]);
    bool bad = false;
#pragma unroll
    for (int i = 0; i < T; ++i) bad = bad || unset(v[i]);
    if (__builtin_amdgcn_ballot_w64(bad) == 0 || cx.dead) break;
    if (n >= cx.spin) {
      cx.dead = 1;
      break;
    }
  }
  pin();
}

// the pieces s0, s0 + sd, ... (T of them; zeros from KS on) of a buffer in operand order
template <int T, int KS, typename Fn>
__device__ __forceinline__ void wait_tiles(i32x4 (&v)[T], Ctx& cx, int base, int s0, int sd, Fn meanwhile) {
  int voff[T], soff[T];
#pragma unroll
  for (int i = 0; i < T; ++i) {
    const int s = s0 + sd * i;
    voff[i] = lane_at(s < KS, cx.lane * 16);
    soff[i] = base_at(s < KS, base + s * 1024);
  }
  wait_x<T>(v, cx, voff, soff, meanwhile);
}

__device__ __forceinline__ f32x4 mfma(i32x4 a, i32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a), as_bf16x8(b), c, 0, 0, 0);
}

// ---- weights: one blob per model in the order the kernel reads it, so that a load is one lane offset and scalars ----
__device__ __forceinline__ i32x4 ld_w(rsrc_t rs, int voff, int soff) {
  return __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, voff, soff, 0));
}
// the same for bytes that are not to push others out of the caches behind
__device__ __forceinline__ i32x4 ld_once(rsrc_t rs, int voff, int soff) {
  return __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, voff, soff, 2));
}
__device__ __forceinline__ f32x2 ld_f2(rsrc_t rs, int voff, int soff) {
  return __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, voff, soff, 0));
}
__device__ __forceinline__ i32x4 ld_w_if(bool here, rsrc_t rs, int voff, int soff) { return ld_w(rs, lane_at(here, voff), base_at(here, soff)); }
__device__ __forceinline__ f32x2 ld_f2_if(bool here, rsrc_t rs, int voff, int soff) { return ld_f2(rs, lane_at(here, voff), base_at(here, soff)); }

// sum over the four lanes that hold the same row of an operand
__device__ __forceinline__ float row_sum(float v) {
  return sum32(sum16(v));
}
// ---- reduction of the waves' partial tiles through LDS ----
// Partials lie as [wave][tile] of 1 KiB, accumulator lane (g, r) -- row r, columns 4 g .. 4 g + 3 -- at part_slot.  Four waves
// reduce a tile, four rows each: lane = 32 h + 16 d + 4 i + j adds up row 4 (wave & 3) + i, columns 4 j .. 4 j + 3 of every
// fourth partial (of 2 h + d on) and ends with columns 4 j + 2 h and the next; the two lanes d = 0, 1 end with the same, d = 0 stores.
// Bound: the chain of LDS reads behind the barrier, and what the stores look like to the memory.  Measured in rounds of the
// hand-off alone (MI355X, 32 KiB a group): two waves adding up sixteen partials of two columns 1.62 us, this split 1.37 (the
// reads are 128 bits without bank conflicts and a quarter as many in a row); eight waves, whose stores cover 32 bytes of a line
// each, 1.92.
__device__ __forceinline__ int part_slot(const Ctx& cx) { return (cx.g * 16 + (cx.r ^ (4 * cx.g))) * 16; }
struct Own {
  int m, n;   // row and first of two columns within the tile
  int src;    // byte offset of the row's four columns within a partial tile
  int word;   // byte offset of the two bf16 results within the tile's half of an exchange piece
  int from;   // the first partial this lane adds up
  bool put;   // of the two lanes with the same result the one that stores
};
__device__ __forceinline__ Own own_of(int t) {
  const int j = t & 3, h = (t >> 5) & 1;
  Own o;
  o.m = ((t >> 6) & 3) * 4 + ((t >> 2) & 3);
  o.n = 4 * j + 2 * h;
  o.src = (j * 16 + (o.m ^ (4 * j))) * 16;
  o.word = (j >> 1) * 256 + o.m * 16 + (j & 1) * 8 + h * 4;
  o.from = (t >> 4) & 3;
  o.put = (t & 16) == 0;
  return o;
}
// a's sum over the lanes l, l ^ 32 in the lower half of the wave, b's in the upper; the same for l, l ^ 16 and its even and odd rows
__device__ __forceinline__ float fold32(float a, float b) {
  const u32x2 s = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}
__device__ __forceinline__ float fold16(float a, float b) {
  const u32x2 s = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}
// waves w0 .. w0 + KG - 1, tile `tile` of NT per wave
template <int KG, int NT>
__device__ __forceinline__ f32x2 sum_part(const unsigned char* p, int w0, int tile, const Own& o) {
  constexpr int N = KG / 4;
  f32x4 v[N];
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = *(const f32x4*)(p + ((w0 + o.from + 4 * i) * NT + tile) * 1024 + o.src);
#pragma unroll
  for (int d = N / 2; d > 0; d >>= 1)
#pragma unroll
    for (int i = 0; i < d; ++i) v[i] += v[i + d];
  return f32x2{sum16(fold32(v[0][0], v[0][2])), sum16(fold32(v[0][1], v[0][3]))};
}
// the sum over a row's sixteen columns of what its lanes hold, in all of them
__device__ __forceinline__ float own_row_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xb1, 0xf, 0xf, true));  // lane ^ 1
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4e, 0xf, 0xf, true));  // lane ^ 2
  return sum32(v);
}

// ---- sums of squares of the rows: exchanged as [column share][16 rows] floats.  A share's 64 bytes come from one block; as
// [row][column share] every block wrote four bytes of every row's lines, and a hand-off with the sums beside its rows took
// 2.19 us alone, against 1.62 without them and 1.36 in this order.  Sixteen shares are a wave's KiB; st: its 16 bytes of lane l,
// share l / 4, rows 4 (l & 3) .. + 3.  The row whose sum the lane ends with (the same in four lanes): share_row ----
__device__ __forceinline__ float share_sum(i32x4 st) {
  float v = fold16(fold32(__int_as_float(st[0]), __int_as_float(st[2])), fold32(__int_as_float(st[1]), __int_as_float(st[3])));
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x128, 0xf, 0xf, true));         // lane ^ 8
  return v + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x124, 0xf, 0xf, true));  // lane + 4
}
__device__ __forceinline__ int share_row(int lane) { return 4 * (lane & 3) + 2 * (lane >> 5) + ((lane >> 4) & 1); }

__device__ __forceinline__ void block_barrier() {
  // LDS traffic only: global loads stay in flight
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

}  // namespace persist
