"""The tiled prefill GEMM (launches of more than 64 tokens): edges of its
32-token tiles, 256-row groups, 64-element stages and split-K chains."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import GEOM, NAMES, Q4_0, Q4_K, Q6_K, Q8_0, pack_host, random_matrix
from test_gpu_prefill import _check_matmul

pytestmark = pytest.mark.gpu
PACKED = [Q8_0, Q4_0, Q4_K, Q6_K]


def _rf():
    import ramforge_amd as rf
    return rf


# token tiles of 3 (padded to 4), 2 x 2, 4 and 5; a full chunk and one token
# more; one row; a half stage (odd multiples of 32); chains of one and several
# flushes (8192 inputs and 16 groups: few splits)
@pytest.mark.parametrize("t", PACKED)
@pytest.mark.parametrize("out_dim,in_dim,n", [(1, 256, 65), (255, 32, 96), (257, 96, 97), (300, 2048, 129),
                                              (520, 1024, 160), (64, 3328, 513), (1000, 5120, 200),
                                              (4096, 8192, 256), (14336, 4096, 128)])
def test_matmul_tile_edges(ctx, orc, t, out_dim, in_dim, n):
    if in_dim % GEOM[t][0]:
        pytest.skip(f"{NAMES[t]} rows are whole {GEOM[t][0]}-element blocks")
    _check_matmul(ctx, orc, t, out_dim, in_dim, n, 4100 + t + out_dim % 997 + n)


@pytest.mark.parametrize("t", [Q8_0, Q4_K])
def test_matmul_tile_unaligned_x_and_short_workspace(ctx, t):
    """x four bytes past alignment gives the same bits as an aligned one (no
    staging copy), also with a workspace fixed at 64 tokens' size, where the
    call runs in 64-token launches instead (other sums: 1e-5 of the largest
    output)."""
    rf = _rf()
    rng = np.random.default_rng(t)
    out_dim, in_dim, n = 700, 1024, 130
    w = pack_host(t, random_matrix(t, out_dim, in_dim, rng), out_dim, in_dim)
    x = rng.normal(0, 1, n * in_dim + 1).astype(np.float32)
    out = []
    for fixed in (False, True):
        with rf.Context(0) as c:
            dw, dx, dx1, y = c.array(w), c.array(x[1:]), c.array(x), c.empty((n * out_dim,))
            if fixed:
                c.reserve(matmul_bytes=c.matmul_workspace_bytes(out_dim, in_dim, 64), staging_bytes=64 * 4 * in_dim,
                          fixed=True)
            used = c.vram_used
            for xd in (dx.ptr, dx1.ptr + 4):
                rf.matmul_packed(c, t, dw, (out_dim, in_dim), xd, n, y)
                out.append(y.numpy().copy())
            assert not fixed or c.vram_used == used
    assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))
    assert np.array_equal(out[2].view(np.uint32), out[3].view(np.uint32))
    assert np.max(np.abs(out[0] - out[2])) <= 1e-5 * np.abs(out[0]).max()


@pytest.mark.parametrize("t", [Q8_0, Q4_0, Q4_K])
def test_matmul_tile_errors_do_not_lean(ctx, orc, t):
    """The matrix cores' chained sums lean towards minus infinity; the signs
    of odd blocks take that off: the mean error over 64 x 128 outputs stays
    below a tenth of the rms error (0.7 of it without the signs; independent
    errors would give about 0.01)."""
    rf = _rf()
    rng = np.random.default_rng(7)
    out_dim, in_dim, n = 64, 14336, 128
    raw = random_matrix(t, out_dim, in_dim, rng)
    x = rng.normal(0, 1, (n, in_dim)).astype(np.float32)
    dev = [ctx.array(pack_host(t, raw, out_dim, in_dim)), ctx.array(x.reshape(-1)), ctx.empty((n * out_dim,))]
    rf.matmul_packed(ctx, t, dev[0], (out_dim, in_dim), dev[1], n, dev[2])
    err = dev[2].numpy().reshape(n, out_dim) - x.astype(np.float64) @ orc.dequantize_rows(
        t, raw, in_dim, out_dim).astype(np.float64).T
    assert abs(err.mean()) <= 0.1 * np.sqrt(np.mean(err ** 2))
    for a in dev:
        a.free()
