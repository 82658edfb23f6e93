"""rf_matmul_packed where a launch of the longest chunk would pass a 32-bit
limit: such calls run in 64-token launches, with the same results."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import Q8_0, random_matrix


def _rf():
    import ramforge_amd as rf
    return rf


def _packed_q8_0(raw, rows, in_dim):
    """The packed regions (codes, scales) of a Q8_0 payload."""
    blocks = raw.reshape(rows * in_dim // 32, 34)
    return np.concatenate([blocks[:, 2:].reshape(-1), blocks[:, :2].reshape(-1)])


def _weights(raw, rows, in_dim):
    blocks = raw.reshape(rows * in_dim // 32, 34)
    d = blocks[:, :2].copy().view(np.float16).astype(np.float64)
    d = np.where(np.abs(d) < 2.0 ** -14, 0.5 * d, d)  # the format's decoder: a subnormal half counts half
    return (d * blocks[:, 2:].view(np.int8)).reshape(rows, in_dim)


def test_tall_matrices_take_short_launches_workspace():
    """2^25 rows: the partials of 32 tokens pass 2^32 bytes, so every launch
    is a 64-token one, whose workspace the query reports (host arithmetic)."""
    from ramforge_amd import _lib

    ws = _lib.load().rf_matmul_workspace_bytes
    for rows in (1 << 25, (1 << 32) // 512):
        assert ws(rows, 32, 512) == ws(rows, 32, 64)
    assert ws((1 << 32) // 512 - 1, 32, 512) > ws((1 << 32) // 512 - 1, 32, 64)


def test_wide_matrices_take_short_launches_workspace():
    """2^20 inputs: 512 tokens of x are 2^31 bytes, the most a launch takes
    being less (host arithmetic)."""
    from ramforge_amd import _lib

    ws = _lib.load().rf_matmul_workspace_bytes
    assert ws(8, 1 << 20, 512) == ws(8, 1 << 20, 64)
    assert ws(8, (1 << 20) - 256, 512) > ws(8, (1 << 20) - 256, 64)


@pytest.mark.gpu
def test_matmul_wide(ctx):
    """2^20 inputs and 512 tokens, each token's x the first one's times a power
    of two: so are its results, bit for bit, and the first token's equal
    float64's within sums of 2^20 terms in f32 (errors of 2^-24 per partial
    sum, the partial sums growing as the square root of their length: far
    below 2^-14 of the sum of magnitudes)."""
    rf = _rf()
    out_dim, in_dim, n = 8, 1 << 20, 512
    rng = np.random.default_rng(62)
    raw = random_matrix(Q8_0, out_dim, in_dim, rng)
    x0 = rng.normal(0, 1, in_dim).astype(np.float32)
    p = (np.arange(n) * 5) % 13 - 6
    with rf.Context(0) as c:
        dx = c.array(np.multiply.outer(np.ldexp(np.float32(1), p), x0))
        w, y = c.array(_packed_q8_0(raw, out_dim, in_dim)), c.empty((n, out_dim))
        rf.matmul_packed(c, Q8_0, w, (out_dim, in_dim), dx, n, y)
        got = y.numpy()
    wd = _weights(raw, out_dim, in_dim)
    base = np.ldexp(got, -p[:, None])
    assert np.array_equal(base.view(np.uint32), np.broadcast_to(base[:1], base.shape).view(np.uint32))
    assert np.all(np.abs(base[0] - wd @ x0.astype(np.float64)) <= np.abs(wd) @ np.abs(x0) * 2.0 ** -14)


@pytest.mark.gpu
def test_matmul_tall(ctx):
    """2^25 + 250 rows of one 32-element block, 65 tokens, against float64:
    the rows repeat with a period that no power of two is a multiple of, so a
    partial that lands elsewhere shows.  Sums of 32 terms in f32: 2^-19 of
    the sum of magnitudes."""
    rf = _rf()
    period, n, in_dim = 1000, 65, 32
    rows = (1 << 25) // period * period + 2 * period
    assert rows > 1 << 25
    rng = np.random.default_rng(61)
    raw = random_matrix(Q8_0, period, in_dim, rng)
    codes, scales = np.split(_packed_q8_0(raw, period, in_dim), [period * in_dim])
    x = rng.normal(0, 1, (n, in_dim)).astype(np.float32)
    with rf.Context(0) as c:
        w = c.array(np.concatenate([np.tile(codes, rows // period), np.tile(scales, rows // period)]))
        dx, y = c.array(x), c.empty((n, rows))
        rf.matmul_packed(c, Q8_0, w, (rows, in_dim), dx, n, y)
        c.synchronize()
        wd = _weights(raw, period, in_dim)
        for t in (0, 31, 32, 63, 64):
            got = rf.DeviceArray(c, y.ptr + 4 * t * rows, 4 * rows, (rows // period, period), np.float32, "").numpy()
            ref, scale = wd @ x[t].astype(np.float64), np.abs(wd) @ np.abs(x[t]).astype(np.float64)
            assert np.all(np.abs(got[0] - ref) <= scale * 2.0 ** -19), t
            assert np.array_equal(got.view(np.uint32), np.broadcast_to(got[:1], got.shape).view(np.uint32)), t
