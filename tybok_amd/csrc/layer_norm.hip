// LayerNorm of the vision towers' token rows with the cast to the GEMM input type folded in:
//   y[m, :] = bf16((x[m, :] - mean) * rstd * w + b),   mean / biased variance / rstd in fp32
// for fp32 rows with fp32 parameters (SigLIP tower of pi0.5: F.layer_norm(x) followed by .to(bf16),
// tybok/policies/pi05/models/vision.py:115-170) or bf16 rows with bf16 parameters (SmolVLA's tower,
// which torch normalises in fp32 and rounds once: tybok/policies/smolvla/models/vision.py:197-257).
// One wave per row, the row stays in registers between the mean, variance and output passes; sums
// across the wave in a fixed order.
// Bound: one trip to memory and the launch itself (rows that another launch has just written: 1 us).  So every load of a
// row is on its way before the first is waited for, none under a branch (at the join behind one the load is waited for: a
// row of 1152 columns took three trips), the sums stay out of the LDS pipe, and a row is a block of its own: 256 rows on
// 256 compute units, not on 64.  With the residual add, us: 256 / 768 rows of 1152 fp32 columns 3.9 -> 2.8 / 4.5 -> 3.8,
// 1024 / 3072 rows of 768 bf16 columns 3.5 -> 2.9 / 5.3 -> 4.5.
#include "tk_common.h"
#include "tk_kernels.h"

namespace {

constexpr int PMAX = 4;  // 8-element pieces per lane: rows up to 64 * 8 * PMAX = 2048 columns
constexpr int ROWS = 1;  // rows (waves) of a block

// ADD: the rows are x + r first (r bf16: the output of the linear that closes a residual branch), the
// sum is written back in x's type (fp32: x + float(r); bf16: rounded once, as torch's bf16 add) and
// normalised -- the residual add and the next LayerNorm of a tower layer in one launch.
template <bool XF32, bool WF32, bool ADD, int NP>
__global__ __launch_bounds__(64 * ROWS) void layer_norm_kernel(LayerNormArgs a) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * ROWS + (threadIdx.x >> 6);
  if (row >= a.M) return;
  const int pieces = a.K / 8;
  int yrow = a.y_rows ? a.y_rows[row] : row;  // (requested with everything else)
  yrow = yrow < 0 ? 0 : (yrow > a.M - 1 ? a.M - 1 : yrow);
  // the parameters of this lane's pieces are requested with the row (they depend on nothing computed here): asked
  // for after the two reductions they would cost the launch one more memory round trip
  i32x4 xq[NP][XF32 ? 2 : 1], rq[NP], wq[NP][WF32 ? 2 : 1], bq[NP][WF32 ? 2 : 1];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int p = lane + 64 * i < pieces ? lane + 64 * i : pieces - 1;  // past the row: a valid piece, not used
    const i32x4* xp = (const i32x4*)((const char*)a.x + ((size_t)row * a.ldx + 8 * p) * (XF32 ? 4 : 2));
    xq[i][0] = xp[0];
    if (XF32) xq[i][XF32 ? 1 : 0] = xp[1];
    if (ADD) rq[i] = *(const i32x4*)(a.r + (size_t)row * a.ldr + 8 * p);
  }
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int p = lane + 64 * i < pieces ? lane + 64 * i : pieces - 1;
    const i32x4* wp = (const i32x4*)((const char*)a.w + 8 * p * (WF32 ? 4 : 2));
    const i32x4* bp = (const i32x4*)((const char*)a.b + 8 * p * (WF32 ? 4 : 2));
    wq[i][0] = wp[0];
    bq[i][0] = bp[0];
    if (WF32) {
      wq[i][WF32 ? 1 : 0] = wp[1];
      bq[i][WF32 ? 1 : 0] = bp[1];
    }
  }
  float v[NP][8];
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int p = lane + 64 * i;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const unsigned xu = (unsigned)xq[i][0][e >> 1];
      v[i][e] = XF32 ? __int_as_float(xq[i][XF32 ? e >> 2 : 0][e & 3]) : __uint_as_float((e & 1) ? (xu & 0xffff0000u) : (xu << 16));
      if (ADD) {
        const unsigned ru = (unsigned)rq[i][e >> 1];
        v[i][e] += __uint_as_float((e & 1) ? (ru & 0xffff0000u) : (ru << 16));
      }
    }
    if (ADD && !XF32) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const unsigned su = pack_bf16x2(v[i][2 * e], v[i][2 * e + 1]);
        rq[i][e] = (int)su;
        v[i][2 * e] = __uint_as_float(su << 16);
        v[i][2 * e + 1] = __uint_as_float(su & 0xffff0000u);
      }
    }
    if (p < pieces) {
      if (ADD && XF32) {
        f32x4* dst = (f32x4*)((float*)a.xsum + (size_t)row * a.ldxs + 8 * p);
        dst[0] = f32x4{v[i][0], v[i][1], v[i][2], v[i][3]};
        dst[1] = f32x4{v[i][4], v[i][5], v[i][6], v[i][7]};
      } else if (ADD) {
        *(i32x4*)((u16*)a.xsum + (size_t)row * a.ldxs + 8 * p) = rq[i];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) sum += v[i][e];
    }
  }
  sum = wave_sum(sum);
  const float mean = sum / (float)a.K;
  float sq = 0.f;
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (lane + 64 * i < pieces) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float d = v[i][e] - mean;
        sq = fmaf(d, d, sq);
      }
    }
  sq = wave_sum(sq);
  const float rstd = rsqrtf(sq / (float)a.K + a.eps);
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int p = lane + 64 * i;
    if (p < pieces) {
      float w[8], b[8];
      if (WF32) {
        union { i32x4 q[2]; float f[8]; } wu, bu;
        wu.q[0] = wq[i][0];
        wu.q[1] = wq[i][WF32 ? 1 : 0];
        bu.q[0] = bq[i][0];
        bu.q[1] = bq[i][WF32 ? 1 : 0];
#pragma unroll
        for (int e = 0; e < 8; ++e) { w[e] = wu.f[e]; b[e] = bu.f[e]; }
      } else {
        union { i32x4 q; unsigned u[4]; } wu, bu;
        wu.q = wq[i][0];
        bu.q = bq[i][0];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          w[2 * e] = __uint_as_float(wu.u[e] << 16);
          w[2 * e + 1] = __uint_as_float(wu.u[e] & 0xffff0000u);
          b[2 * e] = __uint_as_float(bu.u[e] << 16);
          b[2 * e + 1] = __uint_as_float(bu.u[e] & 0xffff0000u);
        }
      }
      union { i32x4 q; unsigned u[4]; } o4;
#pragma unroll
      for (int e = 0; e < 4; ++e)
      {
        const float y0 = (v[i][2 * e] - mean) * rstd * w[2 * e] + b[2 * e], y1 = (v[i][2 * e + 1] - mean) * rstd * w[2 * e + 1] + b[2 * e + 1];
        o4.u[e] = a.y_f16 ? pack_f16x2(y0, y1) : pack_bf16x2(y0, y1);
      }
      *(i32x4*)(a.y + (size_t)yrow * a.ldy + 8 * p) = o4.q;
    }
  }
}

}  // namespace

int tk_layer_norm_max_k() { return 64 * 8 * PMAX; }

template <int NP>
static int launch_np(const LayerNormArgs& a, hipStream_t st) {
  const dim3 grid((a.M + ROWS - 1) / ROWS), block(64 * ROWS);
  const bool add = a.r != nullptr;
  if (a.x_f32 && a.wb_f32) {
    if (add)
      hipLaunchKernelGGL((layer_norm_kernel<true, true, true, NP>), grid, block, 0, st, a);
    else
      hipLaunchKernelGGL((layer_norm_kernel<true, true, false, NP>), grid, block, 0, st, a);
  } else if (!a.x_f32 && !a.wb_f32) {
    if (add)
      hipLaunchKernelGGL((layer_norm_kernel<false, false, true, NP>), grid, block, 0, st, a);
    else
      hipLaunchKernelGGL((layer_norm_kernel<false, false, false, NP>), grid, block, 0, st, a);
  } else {
    return -1;
  }
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int tk_launch_layer_norm(LayerNormArgs a, hipStream_t st) {
  switch ((a.K / 8 + 63) / 64) {  // pieces of a lane: as many loads as the row has
    case 1: return launch_np<1>(a, st);
    case 2: return launch_np<2>(a, st);
    case 3: return launch_np<3>(a, st);
    case 4: return launch_np<4>(a, st);
  }
  return -1;
}
