"""Several engines in one process: what they share, and replays from two streams."""

import os
import sys

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
