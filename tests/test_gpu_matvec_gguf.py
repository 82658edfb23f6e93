"""The register matvec on GGUF bytes: odd and even block counts (rows that do
and do not start on a dword), partial 1 KiB chunks, one and several steps per
row, odd weight addresses, and non-finite x against the LDS-tiled kernels."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import GEOM, Q4_0, Q4_K, Q5_0, Q5_K, Q6_K, Q8_0, random_matrix
from test_gpu_kernels import _check_matvec

pytestmark = pytest.mark.gpu
TYPES = [Q8_0, Q4_0, Q5_0, Q4_K, Q5_K, Q6_K]


def _rf():
    import ramforge_amd as rf
    return rf


# in_dim in multiples of 256 (tails of one to eight 32-element blocks follow
# for the 32-block types); 2049+ rows of the second shape: several tasks per wavefront
@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("rows,in_dim,w_off", [(1, 256, 0), (3, 768, 2), (9, 2304, 4), (2100, 4096, 0), (520, 4352, 0),
                                               (40, 14592, 0), (7, 2048, 1), (33, 36864, 0)])
def test_matvec_gguf_rows(ctx, orc, t, rows, in_dim, w_off):
    _check_matvec(ctx, orc, t, rows, in_dim, 5000 + t + rows, w_off=w_off)
    if GEOM[t][0] == 32 and in_dim < 36864:
        for extra in (32, 64):
            _check_matvec(ctx, orc, t, rows, in_dim + extra, 5100 + t + rows, w_off=w_off)


def test_matvec_gguf_tall_q8_0(ctx, orc):
    """Rows enough for the wavefront-staged kernel, at both ends of its widths
    (2112 and 4096 inputs) and one block past its even counts."""
    for in_dim in (2112, 4096, 2144):
        _check_matvec(ctx, orc, Q8_0, 28700, in_dim, 5200 + in_dim)


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("case", ["inf", "both", "nan"])
def test_matvec_gguf_nonfinite_x_as_the_tiled_kernel(ctx, t, case):
    """Each row's kind (NaN or the sign of its infinity) equals the tiled
    kernels', whose kinds other tests hold against the oracle's."""
    rf = _rf()
    rng = np.random.default_rng(t)
    rows, in_dim = 70, 1536
    x = rng.normal(0, 1, in_dim).astype(np.float32)
    x[5] = np.nan if case == "nan" else np.inf
    if case == "both":
        x[700] = -np.inf
    w, dx, y = ctx.array(random_matrix(t, rows, in_dim, rng)), ctx.array(x), ctx.empty((rows,))
    out = []
    try:
        for mode in (2, 1):
            rf.tune_matvec_kernel(mode)
            rf.matvec(ctx, t, w, (rows, in_dim), dx, y)
            out.append(y.numpy())
    finally:
        rf.tune_matvec_kernel(2)
    assert np.array_equal(np.isnan(out[0]), np.isnan(out[1]))
    assert np.array_equal(out[0][~np.isnan(out[0])], out[1][~np.isnan(out[1])])
    for a in (w, dx, y):
        a.free()


_FIRST_USE_SCRIPT = r"""
import sys
import numpy as np
sys.path[:0] = [sys.argv[1], sys.argv[1] + "/tests"]
import ramforge_amd as rf
from helpers import GEOM, NAMES, Q4_0, Q4_K, Q5_0, Q5_K, Q6_K, Q8_0, random_matrix

rng = np.random.default_rng(41)
with rf.Context(0) as c:
    for t in (Q8_0, Q4_0, Q5_0, Q4_K, Q5_K, Q6_K):
        rows, in_dim = 96, 33 * 32 if GEOM[t][0] == 32 else 3 * 256
        w = c.array(np.concatenate([np.zeros(2, np.uint8), random_matrix(t, rows, in_dim, rng)]))
        x, y = c.array(rng.normal(0, 1, in_dim).astype(np.float32)), c.empty((rows,))
        call = lambda: rf.matvec(c, t, w.ptr + 2, (rows, in_dim), x, y, w_bytes=w.nbytes - 2)
        print(NAMES[t], flush=True)
        with c.capture() as cap:  # the kernels' first launch in this process
            call()
        cap.graph.replay(2)
        first = y.numpy()
        cap.graph.close()
        call()
        c.synchronize()
        eager = y.numpy()
        assert np.max(np.abs(first - eager)) <= 1e-5 * np.abs(eager).max() and np.abs(eager).max() > 0
        with c.capture() as cap:
            call()
        for _ in range(2):
            y.upload(np.zeros(rows, np.float32))
            cap.graph.replay(1)
            assert np.array_equal(y.numpy().view(np.uint32), eager.view(np.uint32))
        cap.graph.close()
print("ok")
"""


def test_matvec_gguf_first_launch_inside_a_capture():
    """Rows that are not 16-byte aligned: captured before the register kernel's
    setup the call runs the one-shot tiles (f32 sums of a thousand terms in
    another order: 1e-5 of the largest output), afterwards the register
    kernel, with the eager call's bits."""
    import os
    import subprocess
    import sys

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", _FIRST_USE_SCRIPT, root], capture_output=True, text=True, timeout=240)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr


def _f32(v):
    return v.astype(np.float32).astype(np.float64)


def _chains_of_eight(t, raw, rows, x):
    """y = W x summed in f32 as chains of eight products per lane, scaled, over
    a lane's steps, then over the 64 lanes in pairs: (codes [rows, blocks, lanes
    of a block, 8], x likewise, scale [rows, blocks, lanes])."""
    qk, size = GEOM[t]
    b = raw.reshape(rows, -1, size)
    nb = b.shape[1]

    def half(v):  # the format's decoder: a subnormal half counts half
        h = v.copy().view(np.float16).astype(np.float64)[..., 0]
        return np.where(h < 2.0 ** -14, 0.5 * h, h)

    if t == Q8_0:
        q = b[..., 2:].view(np.int8).reshape(rows, nb, 4, 8).astype(np.float64)
        xs, d = x.reshape(nb, 4, 8), np.repeat(half(b[..., :2])[..., None], 4, 2)
    elif t == Q4_0:
        n = b[..., 2:].reshape(rows, nb, 4, 4)
        q = np.concatenate([n & 15, n >> 4], 3).astype(np.float64) - 8
        xb = x.reshape(nb, 2, 4, 4)
        xs, d = np.concatenate([xb[:, 0], xb[:, 1]], 2), np.repeat(half(b[..., :2])[..., None], 4, 2)
    else:
        ql, qh = b[..., :128].reshape(rows, nb, 2, 2, 32), b[..., 128:192].reshape(rows, nb, 2, 1, 32)
        low = np.concatenate([ql & 15, ql >> 4], 3)
        two = (qh >> np.array([0, 2, 4, 6], np.uint8)[:, None]) & 3
        q = (low | two << 4).astype(np.float64).reshape(rows, nb, 32, 8) - 32
        sc = np.repeat(b[..., 192:208].view(np.int8).astype(np.float64), 2, 2)
        xs, d = x.reshape(nb, 32, 8), half(b[..., 208:210])[..., None]
    s = np.zeros(q.shape[:3])
    for i in range(8):
        s = _f32(s + q[..., i] * xs[..., i])  # a fused multiply-add (53 bits hold it but for rare ties)
    s = _f32(d * _f32(sc * s)) if t == Q6_K else _f32(d * s)
    per = 64 // s.shape[2]  # blocks per step of 64 lanes
    s = np.pad(s, ((0, 0), (0, -nb % per), (0, 0))).reshape(rows, -1, 64)
    acc = np.zeros((rows, 64))
    for k in range(s.shape[1]):
        acc = _f32(acc + s[:, k])
    while acc.shape[1] > 1:
        acc = _f32(acc[:, ::2] + acc[:, 1::2])
    return acc[:, 0]


@pytest.mark.parametrize("t", [Q8_0, Q4_0, Q6_K])
def test_matvec_gguf_sums_round_no_worse_than_chains_of_eight(ctx, orc, t):
    """The rms error against float64 over 16384 rows of 1536 inputs is no larger
    than the same products' summed in chains of eight: 4% for the sample (one
    chain of sixteen per lane is 7 to 11% larger)."""
    rf = _rf()
    rng = np.random.default_rng(600 + t)
    rows, in_dim = 16384, 1536
    raw = random_matrix(t, rows, in_dim, rng)
    x = rng.normal(0, 1, in_dim).astype(np.float32)
    w, dx, y = ctx.array(raw), ctx.array(x), ctx.empty((rows,))
    rf.matvec(ctx, t, w, (rows, in_dim), dx, y)
    ref = orc.dequantize_rows(t, raw, in_dim, rows).astype(np.float64).reshape(rows, in_dim) @ x.astype(np.float64)
    got, eight = (np.sqrt(np.mean((v - ref) ** 2)) for v in (y.numpy().astype(np.float64),
                                                             _chains_of_eight(t, raw, rows, x.astype(np.float64))))
    print(f"  {t}: rms error {got:.4e}, chains of eight {eight:.4e}, ratio {got / eight:.3f}", flush=True)
    for a in (w, dx, y):
        a.free()
    assert got <= 1.04 * eight
