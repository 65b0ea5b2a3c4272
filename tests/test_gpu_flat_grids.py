"""Flat grids: a strip is cut into tall tiles and low ones below them only where
it has a tall tile at all, and, where the strips alone make two sets of workgroups, four
of them; else the rows left beside the tall tiles make more low ones, each with a
border and a line of its own, than their even end is worth. Such grids take the
one height of the rule for it. The right-hand side equals the element-row
tiles' bit for bit on both sides of that line."""
import pytest

from test_gpu_rhs import assert_bitwise

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nx,Ny,rows", [(8201, 2, 2), (8201, 5, 5), (8201, 7, 7), (8201, 16, 4),
                                        (10241, 13, 7), (10241, 51, 13), (10241, 52, 4),
                                        (1300, 37, 2)])
def test_flat_grids_are_cut_only_below_tall_tiles(Nx, Ny, rows):
    import sgnx
    from sgnx import cases
    c = cases.gate(Nx=Nx, Ny=Ny)
    s = sgnx.SGN2D(**c.solver_kwargs())
    try:
        assert s.rhs_kernel()[1] == rows
        r = s.rhs(c.U0, 0.3)
        s.set_rhs_kernel(0, rows)
        assert_bitwise(s.rhs(c.U0, 0.3), r, "element-row tiles")
    finally:
        s.close()
