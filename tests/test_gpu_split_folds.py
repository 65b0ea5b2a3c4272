"""Folds of the error norm that the other tests of the tile heights do not reach.
The split of the largest grids, tall tiles of 16 rows over low ones of 4, four
partial triples to a tall tile: a grid just large enough for it, with a partial
strip and rows that divide by neither height, against the same grid in one height
of 4 rows, bit for bit. And a norm folded from a single triple, against the same
run with three and with the element-row tiles' norm of its own: compensated sums
in other orders differ by a few rounding units and step sizes follow from the
norm by a power below one, so a relative 1e-12 over three steps; a triple left
out or taken twice shifts the norm by a third."""
import numpy as np
import pytest

from test_gpu_rhs import assert_bitwise

pytestmark = pytest.mark.gpu


def test_sixteen_and_four_rows_equal_four(monkeypatch):
    import sgnx
    from sgnx import cases
    Nx, Ny, cus = 2003, 487, 256
    strips = -(-Nx // 5)
    assert strips * -(-Ny // 16) >= 12 * 4 * cus     # (the rule of the largest grids)
    c = cases.gate(Nx=Nx, Ny=Ny)
    got = []
    for one in (False, True):
        if one:
            monkeypatch.setenv("SGNX_SWEEP_ROWS", "4")
        s = sgnx.SGN2D(**c.solver_kwargs())
        assert s.rhs_kernel()[1] == 4
        s.upload(c.U0)
        st, log = s.integrateAdaptive(0.0, 1e9, s.cflTimeStep(None, 0.5),
                                      sgnx.RkOpts(atol=1e-8, rtol=1e-6, max_accepted=2),
                                      step_log_cap=4)
        got.append((s.download(), np.asarray(log).ravel(), st.as_dict()))
        s.close()
    for a, b, what in zip(got[0], got[1], ("state", "log")):
        assert_bitwise(a, b, what)
    assert got[0][2] == got[1][2]


@pytest.mark.parametrize("variant,rows", [(1, 1), (0, 3)])
def test_norm_of_a_single_partial(variant, rows):
    import sgnx
    from sgnx import cases
    c = cases.gate(Nx=5, Ny=3)
    logs = []
    for v, r in ((1, 3), (variant, rows)):
        s = sgnx.SGN2D(**c.solver_kwargs())
        s.set_rhs_kernel(v, r)
        s.upload(c.U0)
        st, log = s.integrateAdaptive(0.0, 1e9, s.cflTimeStep(None, 0.5),
                                      sgnx.RkOpts(atol=1e-8, rtol=1e-6, max_accepted=3),
                                      step_log_cap=3)
        logs.append((np.asarray(log), st.tReached, st.maxNormLast))
        s.close()
    (a, ta, ma), (b, tb, mb) = logs
    assert np.allclose(a, b, rtol=1e-12, atol=0.0), (a, b)
    assert abs(ta - tb) <= 1e-12 * tb and abs(ma - mb) <= 1e-12 * mb
