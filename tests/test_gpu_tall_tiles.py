"""Launches that take a grid in tall tiles first and low ones last: grids just
large enough for each pair of heights, with a partial strip and rows that divide
by neither height. The same grid in one height (the low one, which the error
norm's partial sums follow): right-hand side, state, step log and statistics of
an adaptive run, and a run that records a tape with its gradient, bit for bit;
the right-hand side against the element-row tiles too."""
import numpy as np
import pytest

from test_gpu_rhs import assert_bitwise

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nx,Ny,rows", [(303, 161, 2), (301, 247, 3), (403, 251, 4), (611, 301, 4)])
def test_tall_and_low_tiles_equal_one_height(Nx, Ny, rows, monkeypatch):
    import sgnx
    from sgnx import cases
    c = cases.shoal(seed=5, Nx=Nx, Ny=Ny)
    rng = np.random.default_rng(Nx)
    ub = rng.normal(size=c.U0.size)
    got = []
    for one in (False, True):
        if one:
            monkeypatch.setenv("SGNX_SWEEP_ROWS", str(rows))
        s = sgnx.SGN2D(**c.solver_kwargs())
        assert s.rhs_kernel()[1] == rows
        s.setDepth(c.depth["Hnod"])
        r = s.rhs(c.U0, 0.3)
        s.upload(c.U0)
        s.tapeBegin(1 << 20)
        s.tapeKeepStages(True)
        st, log = s.integrateAdaptive(0.0, 1e9, s.cflTimeStep(None, 0.5),
                                      sgnx.RkOpts(atol=1e-8, rtol=1e-6, max_accepted=2),
                                      step_log_cap=2)
        s.tapeEnd()
        g, th = s.adjoint(ub, None)
        got.append((r, s.download(), np.asarray(log).ravel(), g, th, st.as_dict()))
        if one:
            s.set_rhs_kernel(0, rows)
            assert_bitwise(s.rhs(c.U0, 0.3), r, "element-row tiles")
        s.close()
    for a, b, what in zip(got[0], got[1], ("rhs", "state", "log", "U0bar", "thetaBar")):
        assert_bitwise(a, b, what)
    assert got[0][5] == got[1][5]
