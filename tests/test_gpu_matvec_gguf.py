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
