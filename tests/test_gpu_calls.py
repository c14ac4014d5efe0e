"""The native side of the single calls (csrc/tk_calls.cpp): what they refuse, in which words, and what they return."""

import threading

import pytest
import torch

from tybok_amd import native
from tybok_amd import ops as tk
from tybok_amd.quant import quantize_weight_rows

BF16 = torch.bfloat16


def test_conversions_refuse_with_python_errors():
    # no GPU needed: every call below ends before its launch
    calls = native.calls()
    x = torch.zeros(3, 64, dtype=BF16)
    w = tk.PackedWeight(x, x, 32, 64)
    with pytest.raises(TypeError, match="activations must be bf16 CUDA tensors"):
        tk.fp8w_gemm(x, w)
    with pytest.raises(TypeError, match="must be a tensor, got list"):
        tk.fp8w_gemm([1.0], w)
    with pytest.raises(TypeError, match="takes 10 arguments, got 1"):
        calls.tk_rope_rows(x)
    with pytest.raises(OverflowError, match="does not fit"):
        calls.tk_rope_rows(x, 1 << 40, None, None, None, 1, 1, 1, 1, 1)
    with pytest.raises(TypeError):
        calls.tk_rope_rows(x, "8", None, None, None, 1, 1, 1, 1, 1)
    with pytest.raises(KeyError):
        tk.fp8w_gated_ffn(x, tk.PackedGateUp(x, x, x, 32, 64), tk.PackedWeight(x, x, 64, 32), "relu")
    with pytest.raises(TypeError, match="q must be bf16"):
        tk.expert_attn(x, None, None, None, tk.MASK_NONE)


def _weights(k=64, i=96):
    g = torch.Generator().manual_seed(0)
    q = [quantize_weight_rows(torch.randn(*s, generator=g) * 0.1) for s in ((i, k), (i, k), (k, i))]
    (wg, sg), (wu, su), (wd, sd) = [(a.cuda(), b.cuda()) for a, b in q]
    return tk.pack_fp8_gate_up(wg, sg, wu, su), tk.pack_fp8_weight(wd, sd), tk.pack_fp8_weight(wg, sg)


@pytest.mark.gpu
def test_single_calls_refuse_what_they_cannot_take():
    wgu, wd, w = _weights()
    x = torch.randn(5, 64, device="cuda").to(BF16)
    vec = torch.ones(64, device="cuda")
    for bad, error, text in [
        (dict(x=x.float()), TypeError, "bf16 CUDA"),
        (dict(x=x[:, :32]), ValueError, r"activations must be \[M, 64\] with unit inner stride, got \(5, 32\)"),
        (dict(x=torch.empty(64, 5, dtype=BF16, device="cuda").t()), ValueError, "unit inner stride"),
        (dict(x=x[0]), ValueError, r"got \(64,\)"),
        (dict(resid=x[:, :32]), ValueError, "residual must be"),
        (dict(resid=x.half()), TypeError, "residual must be bf16 or fp32"),
        (dict(gate=vec), ValueError, "gate must be a contiguous bf16 tensor of 64 elements"),
        (dict(norm_w=vec), ValueError, "norm weight must be a contiguous bf16 tensor of 64 elements"),
        (dict(ada=(vec.to(BF16), vec)), ValueError, "must be fp32 vectors of 64"),
        (dict(ada=(vec, None)), TypeError, "scale / shift must be a tensor"),
        (dict(ada=(vec,)), ValueError, r"ada must be \(scale, shift\)"),
        (dict(wd=w), ValueError, r"down weight must be \[K, I\]"),
        (dict(x=x[:0]), RuntimeError, "tk_fp8w_gated_ffn failed"),
    ]:
        kw = dict(x=x, wgu=wgu, wd=wd) | bad
        with pytest.raises(error, match=text):
            tk.fp8w_gated_ffn(kw.pop("x"), kw.pop("wgu"), kw.pop("wd"), **kw)
    k, vt = torch.zeros(40, 2, 64, dtype=BF16, device="cuda"), torch.zeros(2, 64, 64, dtype=BF16, device="cuda")
    q, pad = torch.zeros(5, 4, 64, dtype=BF16, device="cuda"), torch.ones(40, dtype=torch.bool, device="cuda")
    for bad, error, text in [
        (dict(q=q.half()), TypeError, "q must be bf16"),
        (dict(prefix=tk.PrefixKV(k, vt[:, :, :32])), ValueError, "prefix must hold"),
        (dict(prefix=tk.PrefixKV(k, vt, k_lo=k)), ValueError, "low planes"),
        (dict(suffix=tk.SuffixKV(k[:8, :1], vt[:1])), ValueError, "same number of kv heads"),
        (dict(suffix=tk.SuffixKV(k[:8], vt.float())), ValueError, "suffix must hold"),
        (dict(prefix_pad=pad[:39]), ValueError, "prefix_pad"),
        (dict(prefix_pad=pad.float()), ValueError, "prefix_pad"),
        (dict(mask2d=torch.ones(5, 40, dtype=torch.bool, device="cuda")), ValueError, "mask2d"),
    ]:
        kw = dict(q=q, prefix=tk.PrefixKV(k, vt), suffix=None, prefix_pad=pad, mask_mode=tk.MASK_NONE) | bad
        with pytest.raises(error, match=text):
            tk.expert_attn(**kw)


@pytest.mark.gpu
def test_single_calls_return_the_given_output_and_find_a_workspace():
    _, _, w = _weights()
    x = torch.randn(5, 64, device="cuda").to(BF16)
    want = tk.fp8w_gemm(x, w, ws=tk.Workspace())
    tk._default_ws.clear()
    out = torch.empty_like(want)
    assert tk.fp8w_gemm(x, w, out=out) is out and torch.equal(out, want)
    assert list(tk._default_ws) == [torch.cuda.current_device()]
    # another thread on a stream of its own: its launches go there, and the interpreter is free meanwhile
    got, stream = [], torch.cuda.Stream()

    def work():
        with torch.cuda.stream(stream):
            ws = tk.Workspace()
            got.extend(tk.fp8w_gemm(x, w, ws=ws) for _ in range(50))

    torch.cuda.synchronize()
    t = threading.Thread(target=work)
    t.start()
    here = [tk.fp8w_gemm(x, w) for _ in range(50)]
    t.join()
    torch.cuda.synchronize()
    assert all(torch.equal(y, want) for y in here + got) and len(got) == 50
