"""The work this framework is used for, as cases that can be timed and compared.

Two levels of entry points are covered, because programs use both:

* requests -- ``engine.predict_action_chunk(frame, noise)`` of the two policies, what a robot's control loop
  calls: vision tower, prefix prefill, ten denoising steps, actions back on the host;
* single calls of ``tybok_amd.ops`` -- the fp8-weight GEMM, the gated feed-forward block and the attention over
  a cached prefix, what a program with a model of its own calls.

A case is a dict of plain values; ``kind`` names the entry point, the rest are sizes and options.
"""

from __future__ import annotations

import functools
import os
import random
import tempfile

import torch

from tybok_amd import ops as tk
from tybok_amd.policies.synthetic import write_pi05_checkpoint, write_smolvla_checkpoint
from tybok_amd.quant import quantize_weight_rows
from tybok_amd.registry import create_engine

BF16 = torch.bfloat16

# (hidden, intermediate, activation, norm) of the four feed-forward blocks of the two policies
FFN_BLOCKS = {
    "smolvla_expert": (720, 2048, "silu", "rms"),
    "smolvla_vlm": (960, 2560, "silu", "rms"),
    "pi05_expert": (1024, 4096, "gelu_tanh", "ada"),
    "pi05_vlm": (2048, 16384, "gelu_tanh", "ada"),
}

# (query heads, K/V heads, head size, mask over the action tokens, bf16-rounded logits)
ATTN_HEADS = {
    "smolvla": (15, 5, 64, tk.MASK_CAUSAL, False),
    "pi05": (8, 1, 256, tk.MASK_BIDIR, True),
}

CHUNK, ACTION_WIDTH, STEPS = 50, 32, 10


def listed() -> list[dict]:
    return [
        # the smallest call there is: one row through one small projection (a single-token step of somebody's own loop)
        dict(name="gemm_1_row", kind="gemm", m=1, k=720, n=2048),
        # a whole action chunk through the largest weight matrix: bound by reading the weights
        dict(name="gemm_50_rows_33MB", kind="gemm", m=50, k=2048, n=16384),
        # the action expert's feed-forward block with its norm and residual, 160 times in every request
        dict(name="ffn_expert_50_rows", kind="ffn", block="smolvla_expert", m=50, w8a8=False),
        # a prefix of an odd length through the largest block, activations quantised too: bound by the matrix cores
        dict(name="ffn_prefill_555_rows_w8a8", kind="ffn", block="pi05_vlm", m=555, w8a8=True),
        # action tokens attending to a three-camera prefix and to each other
        dict(name="attn_expert_241_keys", kind="attn", heads="smolvla", m=50, prefix=241),
        # the smallest request: one camera whose frames the engine has to resize, still on the host, a short task
        dict(name="smolvla_1_camera_host", kind="request", model="smolvla", cameras=1, tokens=7, height=480, width=640, host=True, graph=True, w8a8=False),
        # an engine as its constructor makes it by default (no recorded graph): launches and host work count
        dict(name="smolvla_2_cameras_eager", kind="request", model="smolvla", cameras=2, tokens=21, height=512, width=512, host=False, graph=False, w8a8=False),
        # the usual three-camera robot, observation already in device memory
        dict(name="smolvla_3_cameras", kind="request", model="smolvla", cameras=3, tokens=48, height=512, width=512, host=False, graph=True, w8a8=False),
        # one camera and a short prompt in the larger policy: a short, ragged prefix
        dict(name="pi05_1_camera_short", kind="request", model="pi05", cameras=1, tokens=19, height=224, width=224, host=False, graph=True, w8a8=False),
        # the usual two-camera request with the whole language block
        dict(name="pi05_2_cameras", kind="request", model="pi05", cameras=2, tokens=200, height=224, width=224, host=False, graph=True, w8a8=False),
        # frames of another size from the host, the prefix's feed-forward in fp8 x fp8
        dict(name="pi05_2_cameras_host_w8a8", kind="request", model="pi05", cameras=2, tokens=90, height=360, width=640, host=True, graph=True, w8a8=True),
        # the largest request: every camera slot filled
        dict(name="pi05_3_cameras", kind="request", model="pi05", cameras=3, tokens=200, height=224, width=224, host=False, graph=True, w8a8=False),
    ]  # fmt: skip


def _log_int(rng: random.Random, lo: int, hi: int, multiple: int = 1) -> int:
    """An integer spread over the logarithm of ``lo .. hi``, a multiple of ``multiple``."""
    value = lo * (hi / lo) ** rng.random()
    return min(max(round(value / multiple), -(-lo // multiple)), hi // multiple) * multiple


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["gemm", "ffn", "attn", "request", "request", "request", "request"])
    if kind == "gemm":
        # any number of action tokens up to 64, any matrix from 128 KB to 33.5 MB (input sizes are multiples of 16)
        while True:
            k, n = _log_int(rng, 256, 16384, 16), _log_int(rng, 250, 16400)
            if k * n <= 2048 * 16400:
                return dict(kind="gemm", m=_log_int(rng, 1, 64), k=k, n=n)
    if kind == "ffn":
        # the experts run on action chunks, the two prefix stacks on whole prefixes
        block = rng.choice(list(FFN_BLOCKS))
        m = _log_int(rng, 1, 64) if "expert" in block else _log_int(rng, 50, 968)
        return dict(kind="ffn", block=block, m=m, w8a8=block == "pi05_vlm" and m >= 128 and rng.random() < 0.5)
    if kind == "attn":
        heads = rng.choice(list(ATTN_HEADS))
        return dict(kind="attn", heads=heads, m=rng.randint(20, 64), prefix=rng.randint(60, 320) if heads == "smolvla" else rng.randint(240, 968))
    model = rng.choice(["smolvla", "pi05"])
    host = rng.random() < 0.5
    if model == "smolvla":
        size = rng.choice([(512, 512), (480, 640), (rng.randint(240, 720), rng.randint(320, 1280))])
        return dict(kind="request", model=model, cameras=rng.randint(1, 4), tokens=rng.randint(3, 48), height=size[0], width=size[1], host=host,
                    graph=rng.random() < 0.75, w8a8=False)  # fmt: skip
    size = rng.choice([(224, 224), (480, 640), (rng.randint(200, 720), rng.randint(200, 1280))])
    return dict(kind="request", model=model, cameras=rng.randint(1, 3), tokens=_log_int(rng, 5, 200), height=size[0], width=size[1], host=host,
                graph=True, w8a8=rng.random() < 0.5)  # fmt: skip


# ---------------------------------------------------------------------- preparation
@functools.lru_cache(maxsize=None)
def _engine(model: str, graph: bool, w8a8: bool):
    """The policy engine a serving process keeps for its lifetime, every fused / fp8 tier on, random-init weights."""
    path = os.path.join(tempfile.mkdtemp(prefix="tybok_cases_"), model)
    if model == "smolvla":
        return create_engine(
            write_smolvla_checkpoint(path, cameras=4, num_steps=STEPS), device="cuda", graph=graph, graph_cameras=(3,), warmup=True,
            tl_fused_expert=True, tl_fp8_expert_mlp=True, tl_fp8_llm_mlp=True, tl_llm_fused_attn=True, tl_vit_oproj=True,
        )  # fmt: skip
    return create_engine(
        write_pi05_checkpoint(path, cameras=3, num_steps=STEPS), device="cuda", graph=graph, graph_cameras=(2,), warmup=True, pad_free=True,
        tl_fused_expert=True, tl_fp8_expert_mlp=True, tl_fp8_llm_mlp="w8a8" if w8a8 else True, tl_llm_flash_attn=True, tl_fused_vit=True,
    )  # fmt: skip


def _fp8_weight(n: int, k: int, g: torch.Generator):
    return quantize_weight_rows(torch.randn(n, k, generator=g, device="cuda") * 0.02)


def prepare(case: dict, seed: int) -> dict:
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "gemm":
        m, k, n = case["m"], case["k"], case["n"]
        return dict(kind=kind, x=torch.randn(m, k, generator=g, device="cuda").to(BF16), w=tk.pack_fp8_weight(*_fp8_weight(n, k, g)))
    if kind == "ffn":
        k, i, act, norm = FFN_BLOCKS[case["block"]]
        x = torch.randn(case["m"], k, generator=g, device="cuda").to(BF16)
        (wg, sg), (wu, su), (wd, sd) = _fp8_weight(i, k, g), _fp8_weight(i, k, g), _fp8_weight(k, i, g)
        state = dict(kind=kind, x=x, wgu=tk.pack_fp8_gate_up(wg, sg, wu, su), wd=tk.pack_fp8_weight(wd, sd), act=act, w8a8=case["w8a8"])
        if norm == "rms":
            state["norm"] = dict(norm_w=(1.0 + 0.1 * torch.randn(k, generator=g, device="cuda")).to(BF16), eps=1e-5)
        else:
            state["norm"] = dict(ada=(0.1 * torch.randn(k, generator=g, device="cuda"), 0.1 * torch.randn(k, generator=g, device="cuda")), eps=1e-6)
        return state
    if kind == "attn":
        h, kv, d, mask, logits_bf16 = ATTN_HEADS[case["heads"]]
        m, p = case["m"], case["prefix"]
        q, kp, vp, ks, vs = (torch.randn(*s, generator=g, device="cuda").to(BF16) for s in ((m, h, d), (p, kv, d), (p, kv, d), (m, kv, d), (m, kv, d)))
        vt = torch.zeros(kv, d, (m + 31) // 32 * 32, dtype=BF16, device="cuda")
        vt[:, :, :m] = vs.permute(1, 2, 0)
        # a few prefix tokens are padding (the language block is rarely full)
        pad = torch.arange(p, device="cuda") < p - 5
        return dict(kind=kind, q=q, prefix=tk.prepare_prefix_kv(kp, vp), suffix=tk.SuffixKV(ks, vt), pad=pad, mask=mask, logits_bf16=logits_bf16)
    engine = _engine(case["model"], case["graph"], case["w8a8"])
    spec = engine.describe()
    images = {c: torch.randint(0, 256, (3, case["height"], case["width"]), generator=g, device="cuda", dtype=torch.uint8).float() / 255.0
              for c in spec["cameras"][: case["cameras"]]}  # fmt: skip
    frame = engine.make_frame(images, torch.randn(6 if case["model"] == "smolvla" else 8, generator=g, device="cuda"), "pick up the cube")
    # token ids of a prompt with the given number of live tokens, as a tokenizer pads it
    width = engine.config.tokenizer_max_length
    frame["observation.language.tokens"] = torch.randint(0, 32000, (width,), generator=g, device="cuda")
    frame["observation.language.attention_mask"] = torch.arange(width, device="cuda") < case["tokens"]
    noise = torch.randn(1, CHUNK, ACTION_WIDTH, generator=g, device="cuda")
    if case["host"]:
        frame = {k: (v.cpu() if isinstance(v, torch.Tensor) else v) for k, v in frame.items()}
        noise = noise.cpu()
    if case["graph"]:  # a server records a shape once, at its first request
        _recorded(case["model"], case["w8a8"], case["cameras"], case["tokens"] if case["model"] == "pi05" else 0, engine, frame, noise)
    return dict(kind=kind, engine=engine, frame=frame, noise=noise)


_seen_shapes: set = set()


def _recorded(model, w8a8, cameras, tokens, engine, frame, noise) -> None:
    if (model, w8a8, cameras, tokens) not in _seen_shapes:
        engine.predict_action_chunk(frame, noise=noise)
        _seen_shapes.add((model, w8a8, cameras, tokens))


# ---------------------------------------------------------------------- one pass
def run(state: dict):
    kind = state["kind"]
    if kind == "gemm":
        return tk.fp8w_gemm(state["x"], state["w"])
    if kind == "ffn":
        x = state["x"]
        if state["w8a8"]:
            # the W8A8 tier normalises in a launch of its own, as the policy does
            return tk.w8a8_gated_ffn(tk.rms_norm_rows(x, **state["norm"]), state["wgu"], state["wd"], state["act"], resid=x, mode="bf16")
        return tk.fp8w_gated_ffn(x, state["wgu"], state["wd"], state["act"], resid=x, **state["norm"])
    if kind == "attn":
        return tk.expert_attn(state["q"], state["prefix"], state["suffix"], state["pad"], state["mask"], logits_bf16=state["logits_bf16"])
    return state["engine"].predict_action_chunk(state["frame"], noise=state["noise"])


# ---------------------------------------------------------------------- what a pass cannot do without
def _request_work(case: dict) -> tuple[float, float]:
    cams, s = case["cameras"], CHUNK
    if case["model"] == "smolvla":
        hid, kv, exp, layers, steps = 960, 320, 720, 16, STEPS
        rows, p = cams * 1024, cams * 64 + 49  # patches, prefix tokens
        vis = 12 * (4 * 768 * 768 + 2 * 768 * 3072)
        flops = 2.0 * rows * (vis + 768 * 768) + 12 * 4.0 * cams * 1024 * 1024 * 768 + 2.0 * cams * 64 * 12288 * hid
        mlp, att = 3 * hid * 2560, hid * (hid + 2 * kv) + hid * hid
        flops += layers * (2.0 * p * (mlp + att) + 4.0 * p * p * hid)
        e_mlp, e_self, e_cross = 3 * exp * 2048, exp * (hid + 2 * kv) + hid * exp, exp * hid + hid * exp
        flops += 8 * 2.0 * p * 2 * kv * kv
        flops += steps * (layers * 2.0 * s * e_mlp + 8 * (2.0 * s * (e_self + e_cross) + 4.0 * s * (p + s) * hid + 4.0 * s * p * hid))
        # 16-bit projections, fp8 feed-forward weights, fp32 K/V projections of the cross layers; image pixels in fp32
        nbytes = 2.0 * (vis + 768 * 768 + 12288 * hid) + layers * (mlp + 2.0 * att + e_mlp) + 8 * 2.0 * (e_self + e_cross) + 8 * 2 * 4.0 * kv * kv
    else:
        hid, exp, heads, layers, steps = 2048, 1024, 2048, 18, STEPS
        rows = cams * 256
        p = rows + min(200, (case["tokens"] + 15) // 16 * 16)
        vis = 27 * (4 * 1152 * 1152 + 2 * 1152 * 4304)
        flops = 2.0 * rows * (vis + 588 * 1152 + 1152 * hid) + 27 * 4.0 * cams * 256 * 256 * 1152
        mlp, att = 3 * hid * 16384, hid * (heads + 512) + heads * hid
        flops += layers * (2.0 * p * (mlp + att) + 4.0 * p * p * heads)
        e_mlp, e_att = 3 * exp * 4096, exp * (heads + 512) + heads * exp
        flops += steps * layers * (2.0 * s * (e_mlp + e_att) + 4.0 * s * (p + s) * heads)
        nbytes = 2.0 * vis + 4.0 * (588 * 1152 + 1152 * hid) + layers * (mlp + 2.0 * att + e_mlp + 2.0 * e_att)
    nbytes += cams * 3 * case["height"] * case["width"] * 4 + s * ACTION_WIDTH * 8
    return nbytes, flops


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "gemm":
        m, k, n = case["m"], case["k"], case["n"]
        return dict(bytes=float(k * n + 4 * n + 2 * m * k + 2 * m * n), flops=2.0 * m * k * n)
    if kind == "ffn":
        k, i, _, _ = FFN_BLOCKS[case["block"]]
        m = case["m"]
        return dict(bytes=float(3 * k * i + 4 * (2 * i + k) + 2 * m * k * 2 + 8 * k), flops=6.0 * m * k * i)
    if kind == "attn":
        h, kv, d, _, _ = ATTN_HEADS[case["heads"]]
        m, p = case["m"], case["prefix"]
        return dict(bytes=float(2 * (2 * m * h * d + 2 * (p + m) * kv * d) + p), flops=4.0 * m * (p + m) * h * d)
    nbytes, flops = _request_work(case)
    return dict(bytes=nbytes, flops=flops)


def tolerance(case: dict):
    kind = case["kind"]
    if kind == "gemm":
        # one rounding to bf16 of fp32 sums: neighbours of one bf16 step
        return dict(rel=3e-3, max=1e-2)
    if kind == "ffn":
        # bf16 intermediate; with W8A8 an intermediate at a tie takes the neighbouring fp8 code
        return dict(rel=1e-2, max=5e-2) if case["w8a8"] else dict(rel=5e-3, max=3e-2)
    if kind == "attn":
        return dict(rel=5e-3, max=3e-2)
    # bf16 activations through a tower, a prefill and ten steps of sixteen or eighteen layers: two bf16 executions of
    # one request (library products against fused kernels) sit 1.7e-3 .. 2.6e-3 apart, single values up to 1e-2
    return dict(rel=5e-3, max=2.5e-2)
