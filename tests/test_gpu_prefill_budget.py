"""Batched prompts under a VRAM budget: the workspace follows the prompt's
length and leaves a streaming model the room for its layers."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_model import ALL_Q8, STREAM_CFG, _layer_bytes, _load_gpu, _tiny_tensors

pytestmark = pytest.mark.gpu
CFG = dict(STREAM_CFG, context_length=1024, embedding_length=512, feed_forward_length=1024)
CAP = 640
CHARGE = "tmp:prefill"


def _rf():
    import ramforge_amd as rf
    return rf


def _stream(c, T, cache):
    m = _rf().GpuLlamaModel(c, CFG, CAP)
    m.enable_streaming(cache)
    for name, (t, ne0, ne1, arr) in T.items():
        m.set_tensor(name, t, ne0, ne1, arr)
    return m


@pytest.fixture(scope="module")
def model():
    """Tensors, a 600-token prompt, the resident model's hidden state after
    300 and 600 of its tokens, the workspace charges of a 40-token and a
    300-token prompt, and what a streaming model holds without any layer."""
    rf = _rf()
    T = _tiny_tensors(np.random.default_rng(71), CFG, ALL_Q8)
    prompt = [int(v) for v in np.random.default_rng(72).integers(0, CFG["vocab_size"], 600)]
    with rf.Context(0) as c:  # with room to spare the first workspace is the longest
        m = _load_gpu(c, CFG, T, CAP)
        used = c.vram_used
        m.prefill(prompt[:40])
        longest = c.charge(CHARGE)
        m.close()
    with rf.Context(0, used + 2 * longest) as c:
        m = _load_gpu(c, CFG, T, CAP)
        m.prefill(prompt[:40])
        ws = [c.charge(CHARGE)]
        m.reset()
        h = [m.prefill(prompt[:300], want_hidden=True)]
        ws.append(c.charge(CHARGE))
        assert ws[1] == longest
        m.reset()
        m.prefill(prompt[:20])  # a shorter prompt keeps the workspace
        assert c.charge(CHARGE) == ws[1]
        m.reset()
        h.append(m.prefill(prompt, want_hidden=True))
        m.close()
    with rf.Context(0) as c:
        m = _stream(c, T, 0)
        used = c.vram_used
        m.close()
    layer = _layer_bytes(T, 0)
    return dict(T=T, prompt=prompt, h=h, short=ws[0], long=ws[1], used=used, layer=layer)


def _close(got, ref):
    assert np.max(np.abs(got - ref)) <= 2e-4 * max(1.0, np.abs(ref).max())


def test_workspace_follows_the_prompt(model):
    """Up to 64 tokens charge 64 tokens' workspace, whatever the cache holds,
    in a budget that the longest would fill by more than a quarter."""
    assert model["long"] > model["short"] + 2 * model["layer"] > 2 * model["layer"]


@pytest.mark.parametrize("extra", [0.5, 1.5, 2.5])
def test_streaming_prompt_beside_its_layers(model, extra):
    """Budgets between a 64-token workspace with a layer and a long one
    without any: the prompt runs in the chunks that leave a layer room, and
    the model goes on from there."""
    rf = _rf()
    layer = model["layer"]
    budget = model["used"] + model["short"] + int((1 + extra) * layer)
    assert budget < model["used"] + model["long"] + layer
    with rf.Context(0, budget) as c:
        m = _stream(c, model["T"], 0)
        _close(m.prefill(model["prompt"][:300], want_hidden=True), model["h"][0])
        assert c.vram_used == model["used"] and c.vram_peak <= budget
        assert c.charge(CHARGE) is None
        m.forward(model["prompt"][300], 300)
        m.close()


def test_resident_prompt_in_short_chunks(model):
    """A resident model whose budget holds a 64-token workspace and no longer
    one: the same hidden state from 64-token chunks, and a second prompt
    keeps the workspace."""
    rf = _rf()
    with rf.Context(0) as c:
        m = _load_gpu(c, CFG, model["T"], CAP)
        used = c.vram_used
        m.close()
    with rf.Context(0, used + model["short"] + 65536) as c:
        m = _load_gpu(c, CFG, model["T"], CAP)
        for _ in range(2):
            _close(m.prefill(model["prompt"][:300], want_hidden=True), model["h"][0])
            assert c.charge(CHARGE) == model["short"] and m.paths()["batched_prefill"]
            m.reset()
        m.close()


@pytest.mark.parametrize("cache", [0, 1 << 30])
def test_streaming_prompt_over_several_chunks(model, cache):
    """600 tokens: a long chunk and the rest, each layer loaded once per chunk
    where none is cached; the hidden state is the resident model's."""
    rf = _rf()
    with rf.Context(0) as c:
        m = _stream(c, model["T"], cache)
        _close(m.prefill(model["prompt"], want_hidden=True), model["h"][1])
        misses = m.residency_stats()["misses"]
        assert misses == CFG["block_count"] * (1 if cache else 2)
        m.close()


def test_short_prompt_keeps_the_cached_layers(model):
    """A 20-token prompt beside every cached layer needs a 64-token workspace
    only, which fits: no layer is evicted."""
    rf = _rf()
    budget = model["used"] + model["short"] + CFG["block_count"] * model["layer"]
    with rf.Context(0, budget) as c:
        m = _stream(c, model["T"], 1 << 30)
        m.forward(1, 0)
        m.reset()
        m.prefill(model["prompt"][:20])
        assert m.residency_stats()["evictions"] == 0
        m.close()


def test_failed_streaming_prompt_gives_its_workspace_back(model):
    """A budget for the workspace but not for a layer beside it: the prompt is
    refused and the workspace's charge is gone, so single forwards, which
    need a layer only, still run."""
    rf = _rf()
    budget = model["used"] + model["short"] + model["layer"] // 2
    assert model["short"] > model["layer"] // 2
    with rf.Context(0, budget) as c:
        m = _stream(c, model["T"], 0)
        with pytest.raises(rf.RamforgeError, match="insufficient memory"):
            m.prefill(model["prompt"][:40])
        assert c.charge(CHARGE) is None and c.vram_used == model["used"]
        m.reset()
        m.forward(1, 0)
        m.close()


def test_growing_cache_takes_the_workspace_back(model):
    """A resident model whose budget holds the K/V growth or a long prompt's
    workspace, not both: the growth of a later step takes the workspace's
    room, and the next prompt runs in what is left, to the hidden state of a
    model with room to spare."""
    rf = _rf()

    def run(budget):
        with rf.Context(0, budget) as c:
            m = rf.GpuLlamaModel(c, CFG, CAP, kv_initial=256)
            for name, (t, ne0, ne1, arr) in model["T"].items():
                m.set_tensor(name, t, ne0, ne1, arr)
            m.prefill(model["prompt"][:250])
            held, ws = c.vram_used, c.charge(CHARGE)
            for p in range(250, 260):  # the 257th position grows the caches
                h = m.forward(model["prompt"][p], p, want_hidden=True)
            grown = c.charge("kv_cache:k") + c.charge("kv_cache:v")
            h2 = m.prefill(model["prompt"][260:400], want_hidden=True)
            m.close()
            return held, ws, grown, h, h2

    held, ws, _, _, _ = run(0)
    held, ws, grown, h, h2 = run(held + ws)  # not the longest workspace
    assert ws > grown  # so the growth fits where the workspace was
    got = run(held + grown // 2)
    assert got[0] == held
    _close(got[3], h)
    _close(got[4], h2)


@pytest.mark.parametrize("heads,kv,hd,runs", [(4, 2, 64, False), (6, 2, 64, True), (2, 1, 96, True)])
def test_prompt_without_room_for_any_workspace(heads, kv, hd, runs):
    """No room for 64 tokens' workspace: the call fails and nothing is
    forwarded, except for head groups and widths that single forwards serve;
    those give exactly the forwards' hidden state, and paths() says so until a
    prompt is batched again."""
    rf = _rf()
    cfg = dict(STREAM_CFG, context_length=256, head_count=heads, head_count_kv=kv, head_dim=hd)
    T = _tiny_tensors(np.random.default_rng(73), cfg, ALL_Q8)
    prompt = [int(v) for v in np.random.default_rng(74).integers(0, cfg["vocab_size"], 30)]
    with rf.Context(0) as c:
        m = _load_gpu(c, cfg, T, 128)
        used = c.vram_used
        ref = [m.forward(t, p, want_hidden=True) for p, t in enumerate(prompt)][-1]
        m.reset()
        m.prefill(prompt)
        longest = c.charge(CHARGE)
        m.close()
    with rf.Context(0, used + 2 * longest) as c:
        m = _load_gpu(c, cfg, T, 128)
        m.prefill(prompt)
        ws = c.charge(CHARGE)
        m.close()
    with rf.Context(0, used + ws // 2) as c:
        m = _load_gpu(c, cfg, T, 128)
        assert m.paths()["batched_prefill"]
        if runs:
            h = m.prefill(prompt, want_hidden=True)
            assert (h.view(np.uint32) == ref.view(np.uint32)).all()
            assert not m.paths()["batched_prefill"]
        else:
            with pytest.raises(rf.RamforgeError, match="insufficient memory"):
                m.prefill(prompt)
            assert m.seq_len == 0 and c.charge(CHARGE) is None
        m.close()
