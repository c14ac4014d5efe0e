"""The pi0.5 flow-matching loop as one persistent launch against the launches per layer it replaces, at the edges of its
row groups, key tiles and key splits; what a launch that cannot get its waits answered leaves behind; argument checks."""

import os
import sys

import pytest
import torch

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "golden"))

import cases  # noqa: E402

import tybok_amd.ops as tk  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def model():
    from tybok_amd.policies.pi05.model import PI05Model

    cfg, sd, _ = cases.pi05_build(cases.PI05_CASES["small"])
    m = PI05Model(cfg, sd, "cuda", fused_expert=True, fp8_expert_mlp=True, fp8_llm_mlp=True, fused_prefill=True)
    assert m.denoise_plan is not None and m.persistent_loop
    return m


def _case(model, m, p, with_kv=False):
    g = torch.Generator().manual_seed(1000 * m + p)
    depth = model.ed["depth"]
    kv = [tuple(torch.randn(1, 1, p, 256, generator=g).to(torch.bfloat16).cuda() for _ in range(2)) for _ in range(depth)]
    pad = torch.rand(1, p, generator=g).cuda() > 0.2
    pos = (int(pad.sum()) + torch.arange(m)).to(torch.int32).cuda()
    x, caches = torch.randn(m, 32, generator=g).cuda(), model.attention_caches(kv)
    return (x, kv, caches, pad, pos) if with_kv else (x, caches, pad, pos)


def _run(model, x, caches, pad, pos):
    return model.denoise_plan.run(x, -1.0 / model.num_steps, caches, pad[0], pos)


def _layer_by_layer_loop(model, x, caches, pad, pos):
    model.vt_suf = torch.zeros(1, 256, (x.shape[0] + 31) // 32 * 32, dtype=torch.bfloat16, device="cuda")
    for step in range(model.num_steps):
        hidden = model.lin("action_in_proj", x).to(torch.bfloat16)
        hidden = model._denoise_layers_fused(pad, caches, hidden, pos, step)
        _, x = tk.expert_tail(
            hidden, model.p["action_out_proj.weight"], model.p["action_out_proj.bias"], ada=model.final_split[step], eps=1e-6, x_t=x, dt=-1.0 / model.num_steps
        )
    return x


# rows: one row group, a full one, one more row, two and a bit, all four; keys: a single one and fewer tiles than splits
# (empty splits), tile edges, the most tiles
@pytest.mark.parametrize("m,p", [(1, 1), (16, 32), (17, 33), (50, 275), (50, 712), (33, 223), (50, 968), (64, 1216)])
@torch.inference_mode()
def test_one_launch_matches_the_launches_per_layer(model, m, p):
    x, caches, pad, pos = _case(model, m, p)
    want = _layer_by_layer_loop(model, x, caches, pad, pos)
    got = _run(model, x, caches, pad, pos)
    assert torch.isfinite(got).all()
    rel = float((got - want).norm() / (want - x).norm())
    print(f"M={m} P={p}: relative difference of the flow {rel:.3g}")
    assert rel < 2e-2  # bf16 rounding: residual rows, logits and rotary products round to bf16 there, fp32 here (3.1e-3 - 3.5e-3)
    assert torch.equal(got, _run(model, x, caches, pad, pos))  # the exchange buffers start clean again


@pytest.mark.parametrize("m,p", [(17, 33), (50, 275), (50, 712)])
@torch.inference_mode()
def test_one_launch_is_no_less_precise_than_the_launches_per_layer(model, m, p):
    # both against the same loop with every activation in fp32 (weights as they are, on the CPU)
    from oracle import pi05 as O
    from oracle.smolvla import Weights

    cfg, sd, _ = cases.pi05_build(cases.PI05_CASES["small"])
    shape = O.PI05Shape(depth=model.ed["depth"], num_steps=model.num_steps, chunk=m)
    w = Weights(sd, O.fp8_linear_names(shape, True, True), act_dtype=torch.float32)
    x, kv, caches, pad, pos = _case(model, m, p, with_kv=True)
    kv = [tuple(t.float().cpu() for t in layer) for layer in kv]
    ref, dt = x.cpu()[None], -1.0 / model.num_steps
    for step in range(model.num_steps):
        ref = ref + dt * O.denoise_step(w, shape, pad.cpu(), kv, ref, 1.0 + step * dt)
    flow = (ref[0] - x.cpu()).norm()
    runs = _run(model, x, caches, pad, pos), _layer_by_layer_loop(model, x, caches, pad, pos)
    loop, layers = (float((t.cpu() - ref[0]).norm() / flow) for t in runs)
    print(f"M={m} P={p}: distance of the flow from the fp32 run: one launch {loop:.3g}, launches per layer {layers:.3g}")
    # fp32 residual rows, logits and rotation, each bf16 in the launches per layer: measured 0.37 - 0.40 of their distance
    # (one draw of the same roundings from another moves it by a tenth); with rounded rows alone it would be theirs
    assert loop <= 0.55 * layers


@torch.inference_mode()
def test_a_run_whose_waits_give_up_ends_with_nans_and_leaves_nothing_behind(model):
    # forced from the host: without a single poll no wave waits; every block still runs to its end
    case = _case(model, 50, 65)
    want = _run(model, *case)
    model.denoise_plan.polls = -1
    try:
        lost = _run(model, *case)
        torch.cuda.synchronize()
    finally:
        model.denoise_plan.polls = 0
    assert torch.isnan(lost).any()
    assert torch.equal(_run(model, *case), want)


@torch.inference_mode()
def test_the_single_launch_ffns_bound_is_not_the_loops(model):
    # the process-wide bound of the single-launch feed-forward says nothing about this launch
    case = _case(model, 50, 65)
    want = _run(model, *case)
    prev = tk.set_handoff_spin(0)
    try:
        got = _run(model, *case)
        torch.cuda.synchronize()
    finally:
        tk.set_handoff_spin(prev)
    assert torch.equal(got, want)


def _request():
    _, _, inp = cases.pi05_build(cases.PI05_CASES["small"])
    return [[t.cuda() for t in inp["images"]], [t.cuda() for t in inp["img_masks"]], inp["lang_tokens"].cuda(), inp["lang_masks"].cuda(), *[inp["noise"].cuda()]]


def _layer_by_layer(model, args):
    model.persistent_loop = False
    try:
        return model.sample_actions(*args)
    finally:
        model.persistent_loop = True


@torch.inference_mode()
def test_a_starved_loop_of_the_model_runs_again_layer_by_layer(model, monkeypatch):
    args = _request()
    want = _layer_by_layer(model, args)
    asked = []
    monkeypatch.setattr(model.denoise_plan, "run", lambda x0, *a: asked.append(1) or torch.full_like(x0, float("nan")))
    assert torch.equal(model.sample_actions(*args), want) and asked == [1]


@torch.inference_mode()
def test_a_graph_of_somebody_else_holds_the_launches_per_layer(model, monkeypatch):
    # (its replays would not take turns with other loops, and nobody would look for NaNs)
    from tybok_amd.graph import CaptureSession

    args = _request()
    want = _layer_by_layer(model, args)
    session, out = CaptureSession("cuda"), []
    session.prime(lambda: model.sample_actions(*args))
    monkeypatch.setattr(model.denoise_plan, "run", lambda *a: pytest.fail("the graph holds the persistent loop"))
    graph = session.capture(lambda: out.append(model.sample_actions(*args)))
    for _ in range(3):
        out[0].zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out[0], want)


def test_bad_arguments_are_refused(model):
    x, caches, pad, pos = _case(model, 50, 65)
    with pytest.raises(ValueError):
        _run(model, torch.zeros(65, 32, device="cuda"), caches, pad, pos)
    with pytest.raises(ValueError):
        _run(model, x, caches, pad, pos.long())
    assert not tk.PiDenoisePlan.covers(50, 1217) and tk.PiDenoisePlan.covers(64, 1216)


@torch.inference_mode()
def test_more_steps_than_one_launch_takes_run_layer_by_layer(model):
    cfg, _, inp = cases.pi05_build(cases.PI05_CASES["small"])
    steps = model.num_steps
    model.set_num_steps(1001)
    try:
        args = ([t.cuda() for t in inp["images"]], [t.cuda() for t in inp["img_masks"]], inp["lang_tokens"].cuda(), inp["lang_masks"].cuda(), inp["noise"].cuda())
        assert torch.isfinite(model.sample_actions(*args)).all()
    finally:
        model.set_num_steps(steps)
    assert not tk.PiDenoisePlan.covers(50, 275, 1001) and tk.PiDenoisePlan.covers(50, 275, 1000)
    assert not tk.SvDenoisePlan.covers(50, 241, 1001) and tk.SvDenoisePlan.covers(50, 241, 1000)
