"""The batch autotuner and its members' own launches: members with their default
tile height keep it, and with it the speed of their solo runs; one whose height
was set takes the height that the tuner returns, where that is not the untuned
batch's. Solo and batched runs after it agree bit for bit, with and without the
captured step, and so do their right-hand sides."""
import pytest

from test_gpu_rhs import assert_bitwise

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("preset", [(), (1,), (0, 1, 2, 3)])
def test_members_keep_their_default_heights(preset, graph):
    import sgnx
    from sgnx import cases
    cs = [cases.shoal(seed=2, Nx=64, Ny=33), cases.gate(Nx=100, Ny=50),
          cases.gate(Nx=11, Ny=7), cases.shoal(seed=3, Nx=200, Ny=101)]
    ss = [sgnx.SGN2D(**c.solver_kwargs()) for c in cs]
    for i in preset:
        ss[i].set_rhs_kernel(1, 16)
    for c, s in zip(cs, ss):
        s.upload(c.U0)
    before = [s.rhs_kernel()[1] for s in ss]
    b = sgnx.Batch(ss)
    rows, waves = b.autotune(2)
    assert rows >= 1 and 0 <= waves <= 0xf
    for i, s in enumerate(ss):
        assert_bitwise(s.download(), cs[i].U0, f"member {i} after tuning")
        r = s.rhs_kernel()[1]
        if i not in preset:
            assert r == before[i], (i, r, before)
        elif len(preset) == len(ss):
            assert r == rows and rows in (2, 4, 8, 12, 16, 24, 32)
        else:
            assert r in (16, rows)
    opts = [sgnx.RkOpts(atol=1e-8, rtol=1e-6, max_accepted=2 + k) for k in range(4)]
    dt0 = [s.cflTimeStep(None, 0.5) for s in ss]
    solo = []
    for c, s, o, d in zip(cs, ss, opts, dt0):
        st = s.integrateAdaptive(0.0, 1e9, d, o)
        solo.append((s.download(), st.as_dict()))
        s.upload(c.U0)
    for _ in range(2):
        sts = b.integrateAdaptive(0.0, 1e9, dt0, opts, graph=graph)
        for i, (s, st) in enumerate(zip(ss, sts)):
            assert st.as_dict() == solo[i][1]
            assert_bitwise(s.download(), solo[i][0], f"member {i}")
            s.upload(cs[i].U0)
    b.close()
    for s in ss:
        s.close()


def test_a_height_set_after_tuning_is_taken():
    import sgnx
    from sgnx import cases, hip
    c = cases.gate(Nx=40, Ny=21)
    ss = [sgnx.SGN2D(**c.solver_kwargs()) for _ in range(2)]
    for s in ss:
        s.upload(c.U0)
    b = sgnx.Batch(ss)
    b.autotune(1)
    ss[0].set_rhs_kernel(1, 5)
    assert ss[0].rhs_kernel()[1] == 5
    u = hip.DeviceArray.from_host(c.U0)
    d = [hip.DeviceArray(c.U0.size) for _ in ss]
    b.rhs_device([u.address] * 2, [x.address for x in d], 0.2)
    want = ss[0].rhs(c.U0, 0.2)
    for x in d:
        assert_bitwise(x.download(), want, "rhs")
    b.close()
    for s in ss:
        s.close()
    for x in d + [u]:
        x.free()


def test_the_default_height_can_be_set_again():
    """A member that went to the element-row tiles, or to another height, and back
    to its default height is a default member again: the batch autotuner, which
    gives members with a height of their own the one it picks, leaves it."""
    import sgnx
    from sgnx import cases
    cs = [cases.gate(Nx=8, Ny=6), cases.gate(Nx=24, Ny=17), cases.gate(Nx=200, Ny=101)]
    ss = [sgnx.SGN2D(**c.solver_kwargs()) for c in cs]
    default = [s.rhs_kernel()[1] for s in ss]
    assert 1 in default                       # (no height that a tuner tries)
    for s, c, r in zip(ss, cs, default):
        s.upload(c.U0)
        s.set_rhs_kernel(0, r)
        s.set_rhs_kernel(1, 16)
        s.set_rhs_kernel(1, r)
    b = sgnx.Batch(ss)
    b.autotune(1)
    assert [s.rhs_kernel()[1] for s in ss] == default
    b.close()
    for s in ss:
        s.close()


def test_the_default_height_is_a_candidate():
    """A grid of a few workgroups is fastest at one row, its default, which is none
    of the heights that the tuner tries anyway: tuning keeps it."""
    import sgnx
    from sgnx import cases
    c = cases.gate(Nx=8, Ny=6)
    s = sgnx.SGN2D(**c.solver_kwargs())
    s.upload(c.U0)
    assert s.rhs_kernel()[1] == 1
    assert s.autotune(20)[0] == 1
    s.close()
