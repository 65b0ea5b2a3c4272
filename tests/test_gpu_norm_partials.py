"""The fold of the error norm's partial sums at their numbers' edges: one
partial, fewer and more than the block's threads, more than a round of them,
with remainders. The same run with a partial per strip and chunk of rows and
with the fewest partials: step sizes follow from the norm by a power below one,
and compensated sums in two orders differ by a few rounding units, so a relative
1e-12 over two steps; a triple left out or taken twice shifts the norm by about
one over their number."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nx,Ny,rows", [(5, 3, 3), (5, 1030, 1), (130, 70, 1), (341, 121, 1),
                                        (203, 211, 1)])
def test_norm_does_not_depend_on_the_number_of_partials(Nx, Ny, rows):
    import sgnx
    from sgnx import cases
    c = cases.gate(Nx=Nx, Ny=Ny)
    logs = []
    for r in (rows, Ny):
        s = sgnx.SGN2D(**c.solver_kwargs())
        s.set_rhs_kernel(1, r)
        s.upload(c.U0)
        st, log = s.integrateAdaptive(0.0, 1e9, s.cflTimeStep(None, 0.5),
                                      sgnx.RkOpts(atol=1e-8, rtol=1e-6, max_accepted=3),
                                      step_log_cap=3)
        logs.append((np.asarray(log), st.tReached, st.maxNormLast))
        s.close()
    (a, ta, ma), (b, tb, mb) = logs
    assert np.allclose(a, b, rtol=1e-12, atol=0.0), (a, b)
    assert abs(ta - tb) <= 1e-12 * tb and abs(ma - mb) <= 1e-12 * mb
