"""The tile height of the adjoint's products is their own: SGNX_VJP_ROWS sets it,
and no height gives other bits, alone and in a batch (strips of one to five
columns, chunks of one row, of an odd number, with a remainder and of the whole
grid; every side kind). SGNX_SWEEP_ROWS, the forward sweep's height, leaves it: a
height that is poor for a small grid's products (32 rows of 64x32 take them four
times as long) must not lengthen a product; 1.5 tells that from the runs' spread."""
import time

import numpy as np
import pytest

from test_gpu_rhs import assert_bitwise
from test_gpu_vjp_edges import SIDES, _case

pytestmark = pytest.mark.gpu


def _products(c, theta, W, ub):
    """a product and a reverse sweep with recomputed and with kept stages"""
    import sgnx
    s = sgnx.SGN2D(**c.solver_kwargs())
    s.setDepth(theta)
    out = list(s.rhs_vjp(c.U0, W, 0.37))
    for keep in (False, True):
        s.upload(c.U0)
        s.tapeKeepStages(keep)
        s.tapeBegin(1 << 20)
        s.integrateAdaptive(0.1, 1e9, s.cflTimeStep(None, 0.3),
                            sgnx.RkOpts(atol=1e-2, rtol=1e-2, max_accepted=2))
        s.tapeEnd()
        out += s.adjoint(ub, None)
    return s, out


@pytest.mark.parametrize("Nx,Ny,sides", [(2, 2, 0), (4, 7, 1), (5, 2, 3), (6, 5, 2), (13, 4, 0),
                                         (15, 34, 4), (24, 33, 2)])
def test_heights_give_the_same_bits(Nx, Ny, sides, monkeypatch):
    import sgnx
    c = _case(Nx, Ny, SIDES[sides], 3 * Nx + Ny)
    rng = np.random.default_rng(Nx)
    W, ub = rng.normal(size=c.U0.size), rng.normal(size=c.U0.size)
    theta = c.depth["Hnod"]
    first, want = _products(c, theta, W, ub)
    for rows in ("1", "2", "3", "16", "33"):
        monkeypatch.setenv("SGNX_VJP_ROWS", rows)
        s, got = _products(c, theta, W, ub)
        b = sgnx.Batch([first, s, _products(c, theta, W, ub)[0]])
        got += [x for pair in b.adjoint([ub] * 3, None) for x in pair]
        b.close()
        s.close()
        for k, (a, w) in enumerate(zip(got, want + want[-2:] * 3)):
            assert_bitwise(a, w, f"rows {rows}, result {k}")
    first.close()


def test_the_sweeps_height_leaves_the_products(monkeypatch):
    import sgnx
    from sgnx import cases, hip
    c = cases.gate(Nx=64, Ny=32)
    U, W = hip.DeviceArray.from_host(c.U0), hip.DeviceArray.from_host(c.U0)
    out, th = hip.DeviceArray(c.U0.size), hip.DeviceArray(c.nd)
    ss = []
    for rows in (None, "32"):
        if rows:
            monkeypatch.setenv("SGNX_SWEEP_ROWS", rows)
        ss.append(sgnx.SGN2D(**c.solver_kwargs()))
    best = [1e9, 1e9]
    for _ in range(20):
        for k, s in enumerate(ss):
            t = time.perf_counter()
            for _ in range(10):
                s.rhs_vjp_device(U.address, W.address, out.address, th.address, 0.3)
            best[k] = min(best[k], time.perf_counter() - t)
    for s in ss:
        s.close()
    for d in (U, W, out, th):
        d.free()
    assert best[1] < 1.5 * best[0], best
