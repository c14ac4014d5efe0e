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
//                           included, at 256 / 288 / 555 / 712 / 968 rows 67 -> 62, 84 -> 77, 109 -> 103, 126 -> 117, 152 -> 144.
#include "pipe_fp8.h"

namespace {

// One block per row.  MODE 0: sa = amax / 448 (fp32), a8 = RNE(x / sa) from fp32 -- one rounding.
// MODE 1: the arithmetic of a torch expression on bf16 tensors, `s = x.abs().max() / 448` (a bf16 value) and
// `(x / s).to(float8_e4m3fn)` (quotient rounded to bf16, then to fp8): sa = float(bf16(amax / 448)).
// Bound: memory (a 555 x 16384 row block is 18 MB in, 9 MB out) once the loads of a row are all on their way together (NP of
// them a thread, none under a branch: at the join behind one each would be waited for) and a quotient costs four
// instructions: 555 rows of 2048 / 16384 columns 3.8 -> 2.8 / 9.4 -> 8.3 us, 811 of 16384 12.7 -> 10.5.
constexpr int kQuantMaxPieces = 8;  // 16-byte pieces of a row per thread: K <= 8 * 256 * 8 = 16384
template <int NP>
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
  if (a.mode == 1) sa = round_bf16(sa);
  if (tid == 0) a.sa[blockIdx.x] = sa;
  // The IEEE quotient, as the elementwise reference computes it, from the correctly rounded reciprocal: one product and one
  // correction by the exact remainder are again correctly rounded (Markstein).  The sign is the numerator's (the remainder
  // of -0 is +0).  Scales whose reciprocal or remainders would leave the range of normal numbers take the division.
  const float inv = 1.0f / sa;
  const bool plain = sa >= 0x1p-80f && sa <= 0x1p+80f;
  auto quotient = [&](float x) {
    if (sa == 0.f) return 0.f;
    if (!plain) return x / sa;
    const float y = x * inv;
    return __builtin_copysignf(fmaf(fmaf(-sa, y, x), inv, y), x);
  };
  unsigned char* dst = (unsigned char*)a.a8 + (size_t)blockIdx.x * a.lda;
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int p = tid + i * 256;
    if (p >= pieces) continue;
    float q[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const unsigned u = (unsigned)v[i][e >> 1];
      q[e] = quotient(__uint_as_float((e & 1) ? (u & 0xffff0000u) : (u << 16)));
      if (a.mode == 1) q[e] = round_bf16(q[e]);
    }
    // four fp32 -> four e4m3fn (RNE, saturating at +-448) per conversion pair
    int lo = 0, hi = 0;
    lo = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], lo, false);
    lo = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], lo, true);
    hi = __builtin_amdgcn_cvt_pk_fp8_f32(q[4], q[5], hi, false);
    hi = __builtin_amdgcn_cvt_pk_fp8_f32(q[6], q[7], hi, true);
    *(i32x2*)(dst + (size_t)p * 8) = i32x2{lo, hi};
  }
}

}  // namespace

int tk_quant_act_max_k() { return kQuantMaxPieces * 256 * 8; }

// tile: an id of kW8a8Tiles (tk_api.hip)
int tk_launch_w8a8_gemm(const GemmArgs& a, int tile, hipStream_t st) {
  using namespace pipe;
  switch (tile) {
    case 604: return launch_fp8_pipe<FP8, 6, 4, 2, 2, 4, 1>(a, st);
    case 414: return launch_fp8_pipe<FP8, 4, 4, 2, 2, 4, 1>(a, st);
    case 408: return launch_fp8_pipe<FP8, 4, 8, 2, 2, 3, 1>(a, st);
    case 204: return launch_fp8_pipe<FP8, 2, 4, 2, 2, 3, 2>(a, st);
  }
  return -1;
}

int tk_launch_quant_act_rows(QuantActArgs a, hipStream_t st) {
  const int np = (a.K / 8 + 255) / 256;
  const dim3 grid(a.M), block(256);
  if (np <= 1) hipLaunchKernelGGL(quant_act_rows_kernel<1>, grid, block, 0, st, a);
  else if (np <= 2) hipLaunchKernelGGL(quant_act_rows_kernel<2>, grid, block, 0, st, a);
  else if (np <= 4) hipLaunchKernelGGL(quant_act_rows_kernel<4>, grid, block, 0, st, a);
  else hipLaunchKernelGGL(quant_act_rows_kernel<kQuantMaxPieces>, grid, block, 0, st, a);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}
