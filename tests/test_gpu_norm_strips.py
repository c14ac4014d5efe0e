"""Gate/up of a few hundred rows with the RMSNorm prologue (blocks that walk several strips) against the same rows in calls of 32,
which run on the kernel with a block per strip: the same order of all sums, so the same bits.  And the other linears of that prefill whose
blocks changed with it: those that walk a long K whole, the projection of fp32 rows."""

import pytest
import torch

from tybok_amd import ops as tk
from tybok_amd.quant import quantize_weight_rows

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _columns(k, i, first):
    """A down projection that hands on columns of the intermediate as they are: one code per row, the sums exact in any order."""
    w = torch.zeros(k, i)
    w[torch.arange(k), (first + torch.arange(k)) % i] = 1.0
    return tk.pack_fp8_weight(*quantize_weight_rows(w.cuda()))


# rows: the first past 64, edges of 32-row blocks, the most below the many-row kernels; K: whole and partial last tiles, both
# round counts, the smallest and the largest; I: strips that divide evenly among the blocks and that do not
@pytest.mark.parametrize("m,k,i", [(65, 784, 4096), (96, 960, 4096), (97, 960, 2560), (129, 528, 2592), (177, 720, 2048), (241, 960, 2560), (255, 1024, 2560)])
@pytest.mark.parametrize("act", ["silu", "gelu_tanh"])
def test_rows_equal_calls_of_32_rows(m, k, i, act):
    g = torch.Generator().manual_seed(m + k)
    x = torch.randn(m, k, generator=g).to(BF16).cuda()
    (w0, s0), (w1, s1) = (quantize_weight_rows((torch.randn(i, k, generator=g) * 0.05).cuda()) for _ in range(2))
    wgu = tk.pack_fp8_gate_up(w0, s0, w1, s1)
    norm = dict(norm_w=(1.0 + 0.1 * torch.randn(k, generator=g)).to(BF16).cuda(), eps=1e-5)
    for first in range(0, i, k):
        wd = _columns(k, i, first)
        got = tk.fp8w_gated_ffn(x, wgu, wd, act, **norm)
        want = torch.cat([tk.fp8w_gated_ffn(x[r : r + 32], wgu, wd, act, **norm) for r in range(0, m, 32)])
        assert torch.equal(got, want)
        assert got.float().abs().max() > 0


# plain linears whose blocks walk the whole K in 9 .. 12 rounds of eight k tiles (split_k = 1: wherever the rule would split it), and
# as the rule takes them: a round of one tile, partial last tiles, whole ones; one row to several row blocks; one column group, a
# partial tile, and a grid beyond the device
@pytest.mark.parametrize("k", [2064, 2304, 2320, 2560, 2576, 2816, 2832, 3072])
@pytest.mark.parametrize("m,n", [(1, 1600), (50, 960), (97, 250), (255, 960), (241, 4096)])
def test_whole_k_linears(m, k, n):
    g = torch.Generator().manual_seed(m + k)
    x = torch.randn(m, k, generator=g).to(BF16).cuda()
    w8, s = quantize_weight_rows((torch.randn(n, k, generator=g) * 0.05).cuda())
    packed = tk.pack_fp8_weight(w8, s)
    w = w8.double() * s.double()[:, None]
    want = x.double() @ w.t()
    # one rounding to bf16 (8 significant bits: half a step is 2^-8 of the value), one of the scaled sum, K fp32 additions of
    # products of this size
    bound = (2.0**-8 + 2.0**-23) * want.abs() + k * 2.0**-24 * (x.double().abs() @ w.abs().t())
    for split_k in (1, 0):
        assert bool(((tk.fp8w_gemm(x, packed, split_k=split_k).double() - want).abs() <= bound).all())


@pytest.mark.parametrize("m", [65, 177, 256])
def test_norm_of_fp32_rows_equals_calls_of_64_rows(m):
    k, heads, kv = 960, 15, 5
    n = (heads + 2 * kv) * 64
    g = torch.Generator().manual_seed(m)
    x = torch.randn(m, k, generator=g).cuda()
    w = tk.pack_bf16_weight((torch.randn(n, k, generator=g) * 0.05).to(BF16).cuda(), rope_half=32)
    rope = tk.RopeTables(torch.randn(512, 32, generator=g).cuda(), torch.randn(512, 32, generator=g).cuda())
    pos = torch.arange(m, dtype=torch.int32, device="cuda")
    norm = (1.0 + 0.1 * torch.randn(k, generator=g)).to(BF16).cuda()

    def rows(lo, hi):
        return tk.bf16w_linear(x[lo:hi], w, norm_w=norm, eps=1e-5, rope=rope, rope_pos=pos[lo:hi].contiguous(), rope_cols=(heads + kv) * 64)

    assert torch.equal(rows(0, m), torch.cat([rows(r, min(r + 64, m)) for r in range(0, m, 64)]))
