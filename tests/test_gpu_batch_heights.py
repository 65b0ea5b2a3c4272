"""Batches whose members take tile heights other than their own: with the
default heights, members packed with others are given multiples of what they
run with alone (ragged last chunks, grids of two rows, members that stop early
so that the heights change during the run). The error norm is folded over the
same partial sums either way, so states and step statistics equal the solo
run's bit for bit, as do the batched right-hand side and reverse sweep."""
import numpy as np
import pytest

from test_gpu_rhs import assert_bitwise

pytestmark = pytest.mark.gpu


def _members():
    from sgnx import cases
    sizes = [(20 + 4 * k, 17 + 2 * k) for k in range(18)] + [(2, 2), (3, 41), (61, 2)]
    out = []
    for k, (nx, ny) in enumerate(sizes):
        if k % 2:
            out.append(cases.shoal(seed=k, Nx=nx, Ny=ny))
        else:
            out.append(cases.gate(Nx=nx, Ny=ny))
    return out


@pytest.mark.parametrize("graph", [True, False])
def test_packed_heights_bitwise_vs_solo(graph):
    import sgnx
    from sgnx import hip
    cs = _members()
    ss = [sgnx.SGN2D(**c.solver_kwargs()) for c in cs]
    opts = [sgnx.RkOpts(atol=1e-8, rtol=1e-6, max_accepted=2 + k % 5) for k in range(len(cs))]
    dt0, solo, rhs = [], [], []
    for c, s, o in zip(cs, ss, opts):
        s.upload(c.U0)
        rhs.append(s.rhs(c.U0, 0.3))
        dt0.append(s.cflTimeStep(None, 0.5))
        st = s.integrateAdaptive(0.0, 1e9, dt0[-1], o)
        solo.append((s.download(), st.as_dict()))
        s.upload(c.U0)
    b = sgnx.Batch(ss)
    Us = [hip.DeviceArray.from_host(c.U0) for c in cs]
    dUs = [hip.DeviceArray(c.U0.size) for c in cs]
    b.rhs_device([u.address for u in Us], [d.address for d in dUs], [0.3] * len(cs))
    for i, d in enumerate(dUs):
        assert_bitwise(d.download(), rhs[i], f"member {i} rhs")
    sts = b.integrateAdaptive(0.0, 1e9, dt0, opts, graph=graph)
    for i, (s, st) in enumerate(zip(ss, sts)):
        U, sd = solo[i]
        assert st.as_dict() == sd, (i, st.as_dict(), sd)
        assert_bitwise(s.download(), U, f"member {i}")
    b.close()
    for s in ss:
        s.close()


def test_packed_heights_adjoint_bitwise_vs_solo():
    import sgnx
    cs = _members()[:12]
    rng = np.random.default_rng(5)
    ss, ub, solo = [], [], []
    for k, c in enumerate(cs):
        s = sgnx.SGN2D(**c.solver_kwargs())
        s.setDepth(c.depth["Hnod"])
        s.upload(c.U0)
        s.tapeBegin(1 << 20)
        s.integrateAdaptive(0.0, 1e9, s.cflTimeStep(None, 0.5),
                            sgnx.RkOpts(atol=1e-8, rtol=1e-6, max_accepted=2 + k % 3))
        s.tapeEnd()
        ub.append(rng.normal(size=c.U0.size))
        solo.append(s.adjoint(ub[-1], None))
        ss.append(s)
    b = sgnx.Batch(ss)
    for i, ((U0b, thb), (sU, sT)) in enumerate(zip(b.adjoint(ub, None), solo)):
        assert_bitwise(U0b, sU, f"member {i} U0bar")
        assert_bitwise(thb, sT, f"member {i} thetaBar")
    b.close()
    for s in ss:
        s.close()
