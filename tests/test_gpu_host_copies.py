"""Copies between the host and the activation buffer. Up to 1 MiB they go through pinned staging memory: a write has taken
its bytes over when it returns, is not waited for and reaches the device in the order of the calls; past that they are the
runtime's own, behind a wait."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STAGE = 1 << 18  # floats of a staging area


@pytest.fixture()
def ctx(gq):
    c = gq.Context(act_floats=1 << 22, weight_bytes=1 << 27)
    yield c
    c.close()


def _busy(gq, ctx):
    """A captured list of milliseconds, which later calls queue behind (its output in the first 40000 floats)."""
    rows, cols = 8192, 16384
    off = ctx.upload(gq.Q4_0, rows, cols, np.resize(gq.matrix(gq.Q4_0, 256, cols, seed=0, stream=7), rows * gq.row_bytes(gq.Q4_0, cols)))
    return ctx.graph(gq.gemv(gq.Q4_0, rows, cols, off, 0, cols) * 200)


def _write(ctx, off, a):
    """gemvq_act_write from a's own memory."""
    assert ctx.lib.gemvq_act_write(ctx.h, off, a.ctypes.data_as(C.c_void_p), a.size) == 0, ctx.error()


def test_source_may_change_after_a_write(gq, ctx):
    g = _busy(gq, ctx)
    a = gq.normal(1, 1, 3000)
    want = a.copy()
    ctx.replay(g, 2)
    _write(ctx, 50000, a)  # returns while the replays run
    a[:] = -1.0
    _write(ctx, 60000, a)
    a[:] = np.nan
    assert np.array_equal(ctx.read(50000, 3000), want)
    assert np.array_equal(ctx.read(60000, 3000), np.full(3000, -1.0, np.float32))


def test_writes_past_the_staging_area(gq, ctx):
    """Queued behind running work: writes that fill the area several times over, of odd sizes, and one as large as it."""
    g = _busy(gq, ctx)
    ctx.replay(g, 2)
    sizes = [70001, 1, 100003, 16, 90000, 7, STAGE, 33, STAGE - 16, 16, 17, 120000, 150000, 130001]
    want, off = [], 50000
    for i, n in enumerate(sizes):
        a = gq.normal(2, i, n)
        want.append((off, a.copy()))
        _write(ctx, off, a)
        a[:] = np.nan
        off += n + 3 + i  # offsets of any alignment
    assert off < 1 << 22
    for o, w in want:
        assert np.array_equal(ctx.read(o, w.size), w), (o, w.size)


@pytest.mark.parametrize("n", [0, 1, 63, STAGE - 1, STAGE, STAGE + 1, 3 * STAGE + 5])
def test_both_sides_of_the_staging_size(gq, ctx, n):
    a, b = gq.normal(3, 1, n + 2), gq.normal(3, 2, max(n, 1))
    _write(ctx, 1001, a)
    ctx.write(1002, b[:n])
    got = ctx.read(1001, n + 2)
    assert got[0] == a[0] and got[-1] == a[-1] and np.array_equal(got[1:-1], b[:n])
    assert ctx.read(1002, n).size == n


def test_writes_between_replays(gq, ctx):
    """Writes, replays and a list run now, none waited for in between, take effect in the order of the calls."""
    n, X, Y = 4096, 50000, 60000
    g = [ctx.graph(gq.unary(n, X, 4, Y + 4096 * i)) for i in range(3)]
    v = [gq.normal(4, i, n) for i in range(4)]
    for i in range(3):
        ctx.write(X, v[i])
        ctx.replay(g[i])
    ctx.write(X, v[3])
    assert ctx.run(gq.unary(n, X, 4, Y + 4096 * 3)) == 0, ctx.error()
    for i in range(4):
        assert np.array_equal(ctx.read(Y + 4096 * i, n), v[i]), i
    big = gq.normal(4, 9, STAGE + 100)  # a staged write, then one that is not, on the same memory
    ctx.write(X, v[0])
    ctx.write(X, big)
    ctx.write(X + 5, v[1])
    got = ctx.read(X, big.size)
    assert np.array_equal(got[:5], big[:5]) and np.array_equal(got[5:5 + n], v[1]) and np.array_equal(got[5 + n:], big[5 + n:])
