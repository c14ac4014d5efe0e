"""Several engines in one process: what they share, and replays from two streams."""

import os
import sys
import threading

import numpy as np
import pytest
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden"))

import cases  # noqa: E402

import tybok_amd.ops as tk  # noqa: E402

pytestmark = pytest.mark.gpu


def _model(name, **tiers):
    if name == "smolvla":
        from tybok_amd.policies.smolvla.model import SmolVLAModel

        cfg, sd, inp = cases.smolvla_build(cases.SMOLVLA_CASES["small"])
        return SmolVLAModel(cfg, sd, "cuda", **tiers), inp
    from tybok_amd.policies.pi05.model import PI05Model

    cfg, sd, inp = cases.pi05_build(cases.PI05_CASES["small"])
    return PI05Model(cfg, sd, "cuda", **tiers), inp


ALL = dict(fused_expert=True, fp8_expert_mlp=True, fp8_llm_mlp=True, fused_prefill=True)


@pytest.mark.parametrize("name,tiers", [
    ("smolvla", dict(ALL, fused_vit=True)), ("smolvla", dict(fp8_expert_mlp=True, fp8_llm_mlp=True)), ("smolvla", dict(fused_expert=True)),
    ("pi05", dict(ALL, vit_mlp_dtype=torch.bfloat16, vit_lowp_attn=True)), ("pi05", dict(fp8_expert_mlp=True, fp8_llm_mlp=True, fp8_llm_act=True)),
    ("pi05", dict(fused_expert=True)),
])  # fmt: skip
@torch.inference_mode()
def test_a_models_launches_use_its_own_workspace(name, tiers, monkeypatch):
    # (requests of two models may run at the same time: a workspace both write gives either the other's intermediate)
    model, inp = _model(name, **tiers)
    other, _ = _model(name, **tiers)
    assert model.ws.ptr != other.ws.ptr

    def refuse(device=None):
        raise AssertionError("a launch of the model would use the workspace all models share")

    monkeypatch.setattr(tk, "default_workspace", refuse)
    args = [[t.cuda() for t in inp["images"]], [t.cuda() for t in inp["img_masks"]], inp["lang_tokens"].cuda(), inp["lang_masks"].cuda()]
    if name == "smolvla":
        args.append(inp["state"].cuda())
    assert torch.isfinite(model.sample_actions(*args, inp["noise"].cuda())).all()


ENGINE = dict(tl_fused_expert=True, tl_fp8_llm_mlp=True, tl_llm_fused_attn=True)


def _engine(tmp_path, **flags):
    from tybok_amd.policies.synthetic import write_smolvla_checkpoint
    from tybok_amd.registry import create_engine

    ckpt = write_smolvla_checkpoint(str(tmp_path), cameras=1, seed=5, num_vlm_layers=2, vision_layers=1, num_steps=2)
    return create_engine(ckpt, device="cuda", graph=True, warmup=True, **ENGINE, **flags)


def _sleep_on(stream) -> torch.cuda.Event:
    with torch.cuda.stream(stream):
        torch.cuda._sleep(100_000_000)  # (tens of milliseconds at any clock it may count)
        return stream.record_event()


def _side_by_side(a):
    """A stream whose work does not queue up behind ``a``'s (streams share a few hardware queues)."""
    word = torch.zeros(1, device="cuda")
    for _ in range(8):
        b = torch.cuda.Stream()
        torch.cuda.synchronize()
        end = _sleep_on(a)
        with torch.cuda.stream(b):
            word.add_(1)
        b.synchronize()
        if not end.query():
            return b
    pytest.skip("no two streams run side by side here")


def test_a_replay_without_a_loop_does_not_wait_for_another_streams_work(tmp_path):
    engine = _engine(tmp_path, tl_fp8_expert_mlp=False)  # this tier's loop is one launch per phase
    (call,) = (engine._graph_runner.entry(k) for k in engine._graph_runner.keys())
    a = torch.cuda.Stream()
    b = _side_by_side(a)
    torch.cuda.synchronize()
    with torch.cuda.stream(a):
        call.replay()
    a.synchronize()  # (two replays of one graph must not meet)
    end = _sleep_on(a)
    with torch.cuda.stream(b):
        call.replay(copy=False)
    b.synchronize()
    assert not end.query(), "the replay on stream b waited for what stream a had queued"
    torch.cuda.synchronize()


# with the fp8 feed-forward the expert's loop is one launch, and whole replays take turns; without it they run side by side
@pytest.mark.parametrize("fp8_expert", [True, False])
def test_replays_of_two_engines_from_two_streams(tmp_path, fp8_expert):
    engines = [_engine(tmp_path / str(i), tl_fp8_expert_mlp=fp8_expert) for i in range(2)]
    frame = engines[0]._profile_frame()
    noise = torch.zeros(1, 50, 6)
    want = [e.predict_action_chunk(frame, noise=noise) for e in engines]
    assert all(call.takes_turn == fp8_expert for e in engines for call in (e._graph_runner.entry(k) for k in e._graph_runner.keys()))
    torch.cuda.synchronize()
    wrong: list = []

    def serve(engine, expected):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(20):
                if not np.array_equal(engine.predict_action_chunk(frame, noise=noise), expected):
                    wrong.append(engine)

    threads = [threading.Thread(target=serve, args=pair) for pair in zip(engines, want)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong and all(e.model.persistent_loop == fp8_expert for e in engines)
