"""Attention shapes beyond the powers of two: three, five, six, seven and more
than eight query heads per KV head, head_dim 96 and 256, through decode
attention, a model's decode steps and its batched prefill."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_kernels import _attention_case
from test_gpu_model import ALL_Q4, ALL_Q8, TINY, _load_gpu, _tiny_tensors

pytestmark = pytest.mark.gpu


def _rf():
    import ramforge_amd as rf
    return rf


# 16 heads per KV head and hd 256 with 6: per query head in every regime
@pytest.mark.parametrize("qh,kvh,hd", [(3, 1, 64), (12, 2, 128), (15, 3, 96), (7, 1, 128), (14, 2, 64), (5, 5, 96),
                                       (16, 1, 64), (12, 2, 256), (8, 1, 256)])
@pytest.mark.parametrize("hist", [0, 63, 129, 700, 2600])
def test_attention_groups(ctx, orc, hist, qh, kvh, hd):
    """Both sides of the launch regimes' borders, ragged chunk ends and a
    single position, against the oracle's scalar attention."""
    _attention_case(ctx, orc, hist, qh, kvh, hd, 2600 + hist + qh + hd, rope_pos=hist)


@pytest.mark.parametrize("qh,kvh,hd", [(12, 2, 128), (6, 2, 96), (20, 4, 64)])
def test_attention_groups_equal_the_any_shape_kernel(ctx, qh, kvh, hd):
    """A q that is not 16-byte aligned takes the any-shape kernel: the same
    call on both kernels differs by f32 rounding only (sums of a few hundred
    terms in another order: 1e-5 of the largest output)."""
    rf = _rf()
    hist = 300
    rng = np.random.default_rng(qh + hd)
    q = rng.normal(0, 1, qh * hd + 1).astype(np.float32)
    dev = [ctx.array(rng.normal(0, 1, n * kvh * hd).astype(np.float32)) for n in (hist, hist, 1, 1)]
    dq = [ctx.array(q[1:]), ctx.array(q)]
    out = [ctx.empty((qh * hd,)) for _ in range(2)]
    rf.attention_checked(ctx, dq[0], *dev, hist, qh, kvh, hd, out=out[0])
    rf.attention_checked(ctx, dq[1].ptr + 4, *dev, hist, qh, kvh, hd, out=out[1])
    a, b = out[0].numpy(), out[1].numpy()
    assert np.max(np.abs(a - b)) <= 1e-5 * np.abs(b).max()
    for x in dev + dq + out:
        x.free()


@pytest.mark.parametrize("qh,kvh,hd,runs", [(40, 8, 128, True), (32, 8, 128, False)])
def test_attention_groups_without_room_for_the_records(qh, kvh, hd, runs):
    """A workspace that holds the score rows of 101 positions and not the chunk
    records, and that a capture cannot grow: five heads per KV head run the
    any-shape kernel (f32 sums in another order: 1e-5 of the largest output),
    four heads are refused."""
    rf = _rf()
    hist = 100
    rng = np.random.default_rng(qh)
    with rf.Context(0) as c:
        dev = [c.array(rng.normal(0, 1, n).astype(np.float32))
               for n in (qh * hd, hist * kvh * hd, hist * kvh * hd, kvh * hd, kvh * hd)]
        out = c.empty((qh * hd,))
        rf.attention_checked(c, *dev, 10, qh, kvh, hd, out=out)  # one chunk: no records
        if not runs:
            with pytest.raises(rf.RamforgeError, match="during graph capture"):
                with c.capture():
                    rf.attention_checked(c, *dev, hist, qh, kvh, hd, out=out)
            return
        with c.capture() as cap:
            rf.attention_checked(c, *dev, hist, qh, kvh, hd, out=out)
        cap.graph.replay(2)
        got = out.numpy()
        cap.graph.close()
        rf.attention_checked(c, *dev, hist, qh, kvh, hd, out=out)
        ref = out.numpy()
    assert np.max(np.abs(got - ref)) <= 1e-5 * np.abs(ref).max() and not np.array_equal(got, ref)


@pytest.mark.parametrize("qh,kvh,hd,kind", [(12, 2, 128, "q4"), (6, 2, 64, "q8"), (5, 1, 96, "q8"),
                                            (32, 2, 64, "q8"), (6, 1, 256, "q8"), (7, 1, 64, "q8"),
                                            (14, 2, 128, "q4")])
def test_model_groups(ctx, orc, qh, kvh, hd, kind):
    """A prompt of 150 tokens (batched, on the matrix-core attention where it
    takes the shape and on the split kernel) and 40 teacher-forced steps past
    it, through the o-projections that merge the attention's records: hidden
    states against the oracle's token-by-token forward, within 2e-4 of their
    maximum as in the other model tests."""
    rf = _rf()
    cfg = dict(TINY, head_count=qh, head_count_kv=kvh, head_dim=hd, embedding_length=256, context_length=256)
    rng = np.random.default_rng(qh * 10 + hd)
    T = _tiny_tensors(rng, cfg, ALL_Q4 if kind == "q4" else ALL_Q8)
    tokens = [int(v) for v in rng.integers(0, cfg["vocab_size"], 190)]
    om = orc.Model(cfg, T, kv_capacity=200, threads=8)
    ref = [om.forward(t, p) for p, t in enumerate(tokens)]
    om.close()
    gm = _load_gpu(ctx, cfg, T, 200)
    try:
        assert gm.paths()["split_attention"] and gm.paths()["batched_prefill"]
        for mode in (2, 0):
            rf.tune_prefill_attention(mode)
            gm.reset()
            h = gm.prefill(tokens[:150], want_hidden=True)
            got = [(149, h)] + [(p, gm.forward(tokens[p], p, want_hidden=True)) for p in range(150, 190)]
            for p, h in got:
                assert np.max(np.abs(h - ref[p])) <= 2e-4 * max(1.0, np.abs(ref[p]).max()), (mode, p)
    finally:
        rf.tune_prefill_attention(1)
        gm.close()


@pytest.mark.parametrize("qh,kvh,hd", [(6, 1, 256), (16, 1, 64), (7, 1, 64)])
def test_prompt_groups_past_1024_positions(ctx, orc, qh, kvh, hd):
    """A prompt of 1300 tokens in 512-token chunks, the last over more than one
    1024-position chunk: per query head with the merge where no workgroup
    takes the group (six heads of 256, sixteen), on the matrix cores for seven
    heads; the last hidden state against the oracle's, as above."""
    rf = _rf()
    cfg = dict(TINY, head_count=qh, head_count_kv=kvh, head_dim=hd, embedding_length=128, block_count=1,
               context_length=1400)
    rng = np.random.default_rng(qh + hd)
    T = _tiny_tensors(rng, cfg, ALL_Q8)
    tokens = [int(v) for v in rng.integers(0, cfg["vocab_size"], 1300)]
    om = orc.Model(cfg, T, kv_capacity=1400, threads=8)
    for p, t in enumerate(tokens):
        ref = om.forward(t, p)
    om.close()
    gm = _load_gpu(ctx, cfg, T, 1400)
    try:
        assert gm.paths()["batched_prefill"]
        h = gm.prefill(tokens, want_hidden=True)
        assert np.max(np.abs(h - ref)) <= 2e-4 * max(1.0, np.abs(ref).max())
    finally:
        gm.close()
