"""Requests whose persistent denoising loop cannot get its waits answered (forced from the host: the launch may not poll),
eager and recorded, of both engines: repeated layer by layer, nothing recorded meanwhile, the loop tried again later."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

ALL = dict(tl_fused_expert=True, tl_fp8_expert_mlp=True, tl_fp8_llm_mlp=True)


def _engine(name, tmp_path, graph, **kw):
    from tybok_amd.policies.synthetic import write_pi05_checkpoint, write_smolvla_checkpoint
    from tybok_amd.registry import create_engine

    if name == "smolvla":
        ckpt = write_smolvla_checkpoint(str(tmp_path), cameras=1, seed=5, num_vlm_layers=2, vision_layers=1, num_steps=2)
        return create_engine(ckpt, device="cuda", graph=graph, warmup=False, seed=3, tl_llm_fused_attn=True, **ALL, **kw)
    ckpt = write_pi05_checkpoint(str(tmp_path), cameras=1, seed=5, depth=2, vision_layers=1, num_steps=2)
    return create_engine(ckpt, device="cuda", graph=graph, warmup=False, seed=3, tl_llm_flash_attn=True, pad_free=True, **ALL, **kw)


@pytest.fixture(params=[(n, g) for n in ("smolvla", "pi05") for g in (False, True)], ids=lambda p: f"{p[0]}-{'graph' if p[1] else 'eager'}", scope="module")
def served(request, tmp_path_factory):
    """An engine, a frame, noise, and the chunks it answers with the loop and layer by layer."""
    name, graph = request.param
    engine = _engine(name, tmp_path_factory.mktemp(name), graph)
    frame, noise = engine._profile_frame(), torch.randn(1, 50, 6, generator=torch.Generator().manual_seed(1))
    loop, layers = engine.predict_action_chunk(frame, noise=noise), _layer_by_layer(engine, frame, noise)
    assert engine.graph_enabled == graph and engine.model.persistent_loop
    assert np.isfinite(loop).all() and not np.array_equal(loop, layers)
    return engine, frame, noise, loop, layers


def _layer_by_layer(engine, frame, noise):
    recorded, looped = engine.graph_enabled, engine.model.persistent_loop
    engine.graph_enabled = engine.model.persistent_loop = False
    try:
        return engine.predict_action_chunk(frame, noise=noise)
    finally:
        engine.graph_enabled, engine.model.persistent_loop = recorded, looped


@pytest.fixture
def starved(served):
    """The same with a loop that may not poll: in a recorded shape, the launch keeps the bound it was recorded with."""
    engine = served[0]
    keys = list(engine._graph_runner.keys())

    def bound(polls):
        engine.model.persistent_loop, engine._loop_rest, engine._loop_pause = True, 0, 2
        engine.model.denoise_plan.polls = polls
        if engine.graph_enabled:
            engine._graph_runner.forget()
            assert engine._graph_runner.precapture(keys)

    bound(-1)
    yield served
    bound(0)


def test_a_starved_request_is_repeated_and_the_loop_tried_again(starved, monkeypatch):
    engine, frame, noise, loop, layers = starved
    recorded, kept = engine.graph_enabled, dict(engine._graph_runner._shapes)
    monkeypatch.setattr(engine, "_capture_graph", lambda *a: pytest.fail("a shape was recorded inside a request"))

    def ask():
        return engine.predict_action_chunk(frame, noise=noise)

    assert np.array_equal(ask(), layers) and engine._loop_rest == 2  # starved, repeated
    assert np.array_equal(ask(), layers) and engine._loop_rest == 1  # the loop rests
    assert np.array_equal(ask(), layers) and engine._loop_rest == 4  # tried again, still starved: rests twice as long
    assert engine.graph_enabled == recorded and dict(engine._graph_runner._shapes) == kept
    # the engine's own noise, drawn once
    engine._loop_rest, engine.model.persistent_loop = 0, True
    drawn = engine.predict_action_chunk(frame)
    assert engine._loop_rest and np.array_equal(drawn, _layer_by_layer(engine, frame, engine._drawn_noise.clone()))


def test_the_loop_comes_back_when_it_answers(served):
    engine, frame, noise, loop, layers = served
    engine.model.persistent_loop, engine._loop_rest, engine._loop_pause = False, 2, 8  # as a starved request leaves it
    assert np.array_equal(engine.predict_action_chunk(frame, noise=noise), layers) and engine._loop_pause == 8
    assert np.array_equal(engine.predict_action_chunk(frame, noise=noise), loop)
    assert engine.model.persistent_loop and engine._loop_rest == 0 and engine._loop_pause == engine._LOOP_PAUSE


def test_a_request_that_is_itself_nan_says_nothing_about_the_loop(served):
    engine, frame, noise, _, _ = served
    assert np.isnan(engine.predict_action_chunk(frame, noise=noise * float("nan"))).any()
    assert engine.model.persistent_loop and engine._loop_rest == 0


def test_validate_repeats_a_starved_chunk(starved, tmp_path):
    engine, frame, _, _, _ = starved
    zeros = torch.zeros(1, 50, engine.config.max_action_dim)
    chunk = torch.from_numpy(_layer_by_layer(engine, frame, zeros))[None]
    torch.save(frame, tmp_path / "frame.pt")
    torch.save({"chunk_post": chunk}, tmp_path / "chunk.pt")
    assert engine.validate(str(tmp_path))["chunk_post.max"] == 0.0


def test_the_loop_can_be_switched_off(served, tmp_path):
    # for a GPU that other processes work on as well: recorded shapes follow, outside a request
    engine, frame, noise, loop, layers = served
    turns = lambda: {call.takes_turn for call in engine._graph_runner._shapes.values()}  # noqa: E731
    recorded = set() if not engine.graph_enabled else {False}
    for on, want, takes in ((False, layers, recorded), (True, loop, {not r for r in recorded})):
        engine.set_persistent_loop(on)
        assert turns() == takes
        for _ in range(3):
            assert np.array_equal(engine.predict_action_chunk(frame, noise=noise), want)
    name = "smolvla" if "smolvla" in type(engine).__module__ else "pi05"
    without = _engine(name, tmp_path, engine.graph_requested, persistent_loop=False)
    assert without.model.denoise_plan is None and np.array_equal(without.predict_action_chunk(frame, noise=noise), layers)
    with pytest.raises(ValueError):
        without.set_persistent_loop(True)
