"""Gate/up of a few hundred rows with the RMSNorm prologue (blocks that walk several strips) against the same rows in calls of 32,
which run on the kernel with a block per strip: the same order of all sums, so the same bits."""

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
