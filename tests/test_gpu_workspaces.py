"""Context workspaces: rf_ctx_reserve sizes them up front; with a fixed
reservation no call allocates (a call that needs more is refused), growth is
refused during graph capture, and a graph captured before a workspace was
replaced is refused at replay instead of reading the freed buffer."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _attention_inputs(c, rng, hist, qh=32, kvh=8, hd=128):
    arrs = [rng.normal(0, 1, n).astype(np.float32)
            for n in (qh * hd, max(hist, 1) * kvh * hd, max(hist, 1) * kvh * hd, kvh * hd, kvh * hd)]
    return [c.array(a) for a in arrs]


def test_fixed_reservation_allocates_nothing():
    import ramforge_amd as rf

    rng = np.random.default_rng(31)
    with rf.Context(0) as c:
        # up to 64 positions: 8 chunks per query head at most (the split
        # records of 32 heads, hd + 4 floats each), more than the any-shape
        # kernel's score rows
        need = c.attention_workspace_bytes(64, 32, 8, 128)
        assert need == 8 * 32 * 132 * 4
        dev = _attention_inputs(c, rng, 8191)
        out = c.empty((32 * 128,))
        c.reserve(attention_bytes=need, fixed=True)
        used = c.vram_used
        for hist in (63, 40, 0):
            print(f"  reserved attention hist={hist}", flush=True)
            rf.attention_checked(c, *dev, hist, 32, 8, 128, out=out)
            c.synchronize()
            assert c.vram_used == used, hist
        # 2048 positions take 32 chunks per KV head: more than reserved
        with pytest.raises(rf.RamforgeError, match="fixed"):
            rf.attention_checked(c, *dev, 2047, 32, 8, 128, out=out)
        assert c.vram_used == used
        # a larger reservation lifts the limit again
        c.reserve(attention_bytes=c.attention_workspace_bytes(8192, 32, 8, 128), fixed=True)
        rf.attention_checked(c, *dev, 8191, 32, 8, 128, out=out)
        c.synchronize()


def test_matmul_reservation_covers_the_call():
    import ramforge_amd as rf
    from helpers import Q8_0, pack_host, random_matrix

    rng = np.random.default_rng(32)
    rows, k, n = 512, 1024, 80
    raw = random_matrix(Q8_0, rows, k, rng)
    with rf.Context(0) as c:
        w = c.array(pack_host(Q8_0, raw, rows, k))
        x = c.array(rng.normal(0, 1, (n, k)).astype(np.float32))
        y = c.empty((n, rows))
        c.reserve(matmul_bytes=c.matmul_workspace_bytes(rows, k, n), fixed=True)
        used = c.vram_used
        rf.matmul_packed(c, Q8_0, w, (rows, k), x, n, y)
        c.synchronize()
        assert c.vram_used == used


def test_matmul_reservation_covers_shorter_calls():
    """A workspace fixed for 160 tokens serves 128, whose launch takes more
    splits, with the bits of an unfixed context (the same launch, not two
    64-token ones); without a reservation the shorter call does not replace
    the longer one's workspace."""
    import ramforge_amd as rf
    from helpers import Q8_0, pack_host, random_matrix

    rng = np.random.default_rng(37)
    rows, k = 14336, 4096
    w = pack_host(Q8_0, random_matrix(Q8_0, rows, k, rng), rows, k)
    x = rng.normal(0, 1, (160, k)).astype(np.float32)
    out = []
    for first, fixed in ((128, False), (160, False), (160, True)):
        with rf.Context(0) as c:
            dw, dx, y = c.array(w), c.array(x), c.empty((160, rows))
            if fixed:
                c.reserve(matmul_bytes=c.matmul_workspace_bytes(rows, k, first), fixed=True)
            else:
                rf.matmul_packed(c, Q8_0, dw, (rows, k), dx, first, y)
            used = c.vram_used
            rf.matmul_packed(c, Q8_0, dw, (rows, k), dx, 128, y)
            out.append(y.numpy()[:128])
            assert c.vram_used == used
    for got in out[1:]:
        assert np.array_equal(got.view(np.uint32), out[0].view(np.uint32))


def test_growth_refused_during_capture():
    import ramforge_amd as rf

    rng = np.random.default_rng(33)
    with rf.Context(0) as c:
        dev = _attention_inputs(c, rng, 4095)
        out = c.empty((32 * 128,))
        with pytest.raises(rf.RamforgeError, match="during graph capture"):
            with c.capture():
                rf.attention_checked(c, *dev, 4095, 32, 8, 128, out=out)
        # outside a capture the same call grows the workspace and runs
        rf.attention_checked(c, *dev, 4095, 32, 8, 128, out=out)
        c.synchronize()


def test_stale_graph_refused_after_workspace_growth():
    import ramforge_amd as rf

    rng = np.random.default_rng(34)
    with rf.Context(0) as c:
        dev = _attention_inputs(c, rng, 8191)
        out = c.empty((32 * 128,))
        rf.attention_checked(c, *dev, 100, 32, 8, 128, out=out)  # sizes the workspace
        c.synchronize()
        with c.capture() as cap:
            rf.attention_checked(c, *dev, 100, 32, 8, 128, out=out)
        g = cap.graph
        g.replay(2)
        want = out.numpy()
        rf.attention_checked(c, *dev, 8191, 32, 8, 128, out=out)  # replaces the workspace
        c.synchronize()
        with pytest.raises(rf.RamforgeError, match="captured before"):
            g.replay(1)
        g.close()
        with c.capture() as cap2:  # a new capture uses the new buffer
            rf.attention_checked(c, *dev, 100, 32, 8, 128, out=out)
        cap2.graph.replay(2)
        assert np.array_equal(out.numpy().view(np.uint32), want.view(np.uint32))
        cap2.graph.close()


_SETUP_SCRIPT = r"""
import sys
import numpy as np
sys.path.insert(0, sys.argv[1])
import ramforge_amd as rf
from ramforge_amd import GGML

rng = np.random.default_rng(35)
rows, k = 96, 4096
raw = rng.integers(0, 256, size=(rows, k // 32, 34), dtype=np.uint8)
raw[:, :, 0:2] = np.frombuffer(np.full(rows * k // 32, 0x2000, np.uint16).tobytes(), np.uint8).reshape(rows, -1, 2)
with rf.Context(0) as c:
    w = c.array(raw.reshape(-1))
    p = c.empty((raw.size,), "uint8")
    rf.pack_weights(c, GGML.Q8_0, w, rows, k, p)
    x = c.array(rng.normal(0, 1, k).astype(np.float32))
    y = c.empty((rows,))
    # the first launch of this kernel shape in the process: its setup
    # (dynamic LDS attribute, occupancy) is refused inside a capture
    try:
        with c.capture():
            rf.matvec_packed(c, GGML.Q8_0, p, (rows, k), x, y)
        print("captured without refusal")
        sys.exit(1)
    except rf.RamforgeError as e:
        assert "inside a stream capture" in str(e), str(e)
    # once launched outside a capture, the same shape captures and replays
    rf.matvec_packed(c, GGML.Q8_0, p, (rows, k), x, y)
    c.synchronize()
    want = y.numpy()
    y.upload(np.zeros(rows, np.float32))
    with c.capture() as cap:
        rf.matvec_packed(c, GGML.Q8_0, p, (rows, k), x, y)
    cap.graph.replay(2)
    assert np.array_equal(y.numpy().view(np.uint32), want.view(np.uint32))
    cap.graph.close()
print("ok")
"""


def test_first_launch_setup_refused_inside_capture():
    """A launcher's one-time kernel setup (dynamic LDS attribute, occupancy
    query) is never made inside a stream capture: the first launch of a
    kernel shape inside a capture is refused with a clear error, and the
    same shape captures and replays once it has run outside.  Run in a fresh
    process, where no shape has been set up yet."""
    import os
    import subprocess
    import sys

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", _SETUP_SCRIPT, root], capture_output=True, text=True, timeout=240)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr


def test_calls_after_a_failed_device_allocation():
    """A charge the budget allows and the device cannot hold fails without a
    trace: the ledger is rolled back and the next calls, whose launches check
    the runtime's last error, run."""
    import ramforge_amd as rf
    from helpers import Q8_0, pack_host, random_matrix

    rng = np.random.default_rng(39)
    rows, k, n = 300, 1024, 100
    w = pack_host(Q8_0, random_matrix(Q8_0, rows, k, rng), rows, k)
    x = rng.normal(0, 1, (n, k)).astype(np.float32)
    out = []
    with rf.Context(0, 1 << 50) as c:
        dw, dx, y = c.array(w), c.array(x), c.empty((n, rows))
        for fail in (False, True):
            if fail:
                used = c.vram_used
                with pytest.raises(rf.RamforgeError, match="hipMalloc"):
                    c.alloc(1 << 46)
                assert c.vram_used == used
            rf.matmul_packed(c, Q8_0, dw, (rows, k), dx, n, y)
            out.append(y.numpy())
    assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))


_LONG_THEN_CAPTURE = r"""
import sys
import numpy as np
sys.path[:0] = [sys.argv[1], sys.argv[1] + "/tests"]
import ramforge_amd as rf
from helpers import Q4_0, Q4_K, Q6_K, Q8_0, pack_host, random_matrix

rng = np.random.default_rng(38)
rows, k = 512, 1024
with rf.Context(0) as c:
    for t in (Q8_0, Q4_0, Q4_K, Q6_K):
        w = c.array(pack_host(t, random_matrix(t, rows, k, rng), rows, k))
        x, y = c.array(rng.normal(0, 1, 200 * k + 1).astype(np.float32)), c.empty((200, rows))
        for xp in (x.ptr, x.ptr + 4):
            rf.matmul_packed(c, t, w, (rows, k), xp, 200, y)
            for n in (64, 45, 30, 5):
                print(t, xp & 15, n, flush=True)
                with c.capture() as cap:  # the first launches of this many tokens
                    rf.matmul_packed(c, t, w, (rows, k), xp, n, y)
                y.upload(np.zeros((200, rows), np.float32))
                cap.graph.replay(2)
                got = y.numpy()
                cap.graph.close()
                y.upload(np.zeros((200, rows), np.float32))
                rf.matmul_packed(c, t, w, (rows, k), xp, n, y)
                assert np.array_equal(got.view(np.uint32), y.numpy().view(np.uint32)) and np.any(got[n - 1])
print("ok")
"""


def test_long_call_prepares_captures_of_shorter_ones():
    """After a call of 200 tokens a capture takes any shorter call, aligned x
    or not, though other kernels (whose setup a capture refuses) and the
    scratch copy serve up to 64 tokens.  In a fresh process, where no shape
    has been set up yet."""
    import os
    import subprocess
    import sys

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", _LONG_THEN_CAPTURE, root], capture_output=True, text=True, timeout=240)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr


def test_refused_growth_keeps_the_workspace():
    """A budget for the 64-token launches' workspace and not for the longer
    ones': calls of more tokens run in short launches, each with the same
    buffer, so that a graph captured over it stays valid; the results are the
    long launches' up to the sums' order (1e-5 of the largest output)."""
    import ramforge_amd as rf
    from helpers import Q8_0, pack_host, random_matrix

    rng = np.random.default_rng(36)
    rows, k, n = 700, 1024, 130
    w = pack_host(Q8_0, random_matrix(Q8_0, rows, k, rng), rows, k)
    x = rng.normal(0, 1, (n, k)).astype(np.float32)

    def arrays(c):
        return c.array(w), c.array(x), c.empty((n, rows))

    with rf.Context(0) as c:
        dw, dx, y = arrays(c)
        held, short = c.vram_used, max(c.matmul_workspace_bytes(rows, k, i) for i in range(1, 65))
        assert c.matmul_workspace_bytes(rows, k, n) > short + 65536
        rf.matmul_packed(c, Q8_0, dw, (rows, k), dx, n, y)
        ref = y.numpy()
    with rf.Context(0, held + short + 65536) as c:
        dw, dx, y = arrays(c)
        rf.matmul_packed(c, Q8_0, dw, (rows, k), dx, n, y)
        want, used = y.numpy(), c.vram_used
        assert np.max(np.abs(want - ref)) <= 1e-5 * np.abs(ref).max()
        with c.capture() as cap:
            rf.matmul_packed(c, Q8_0, dw, (rows, k), dx, n, y)
        for _ in range(2):
            y.upload(np.zeros((n, rows), np.float32))
            rf.matmul_packed(c, Q8_0, dw, (rows, k), dx, n, y)
            assert c.vram_used == used
            assert np.array_equal(y.numpy().view(np.uint32), want.view(np.uint32))
            y.upload(np.zeros((n, rows), np.float32))
            cap.graph.replay(1)
            c.synchronize()
            assert np.array_equal(y.numpy().view(np.uint32), want.view(np.uint32))
        cap.graph.close()
