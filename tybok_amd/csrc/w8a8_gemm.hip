// W8A8 tier of the VLM prefill MLP on gfx950: per-token activation quantisation and the fp8 x fp8 GEMM.
//
//   quant_act_rows_kernel   x[M,K] bf16 -> a8[M,K] e4m3fn, sa[M] fp32 with sa = amax_k|x| / 448 and
//                           a8 = RNE(x / sa) in fp32 (one rounding); an all-zero row gives sa = 0 and zero codes.
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
constexpr int kQuantMaxPieces = 8;  // 16-byte pieces of a row per thread: K <= 8 * 256 * 8 = 16384
__global__ __launch_bounds__(256) void quant_act_rows_kernel(QuantActArgs a) {
  __shared__ float part[4];
  const int tid = threadIdx.x;
  const char* row = (const char*)a.x + (size_t)blockIdx.x * a.ldx * 2;
  const int pieces = a.K / 8;
  i32x4 v[kQuantMaxPieces];
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < kQuantMaxPieces; ++i) {
    const int p = tid + i * 256;
    v[i] = i32x4{0, 0, 0, 0};
    if (p < pieces) v[i] = *(const i32x4*)(row + (size_t)p * 16);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const unsigned u = (unsigned)v[i][e];
      amax = fmaxf(amax, fmaxf(fabsf(__uint_as_float(u << 16)), fabsf(__uint_as_float(u & 0xffff0000u))));
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o));
  if ((tid & 63) == 0) part[tid >> 6] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
  float sa = amax / 448.0f;
  if (a.mode == 1) sa = round_bf16(sa);
  if (tid == 0) a.sa[blockIdx.x] = sa;
  unsigned char* dst = (unsigned char*)a.a8 + (size_t)blockIdx.x * a.lda;
#pragma unroll
  for (int i = 0; i < kQuantMaxPieces; ++i) {
    const int p = tid + i * 256;
    if (p >= pieces) continue;
    float q[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const unsigned u = (unsigned)v[i][e];
      q[2 * e] = __uint_as_float(u << 16);
      q[2 * e + 1] = __uint_as_float(u & 0xffff0000u);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float y = amax == 0.f ? 0.f : q[e] / sa;  // IEEE division, as the elementwise reference computes it
      if (a.mode == 1) y = round_bf16(y);
      q[e] = y;
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
  hipLaunchKernelGGL(quant_act_rows_kernel, dim3(a.M), dim3(256), 0, st, a);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}
