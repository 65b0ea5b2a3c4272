"""Which way a batch's reverse sweeps go. Twelve grids of 128x64 leave most of the
GPU idle one after another: their sweeps in lockstep have to end well before the
members' own calls do together (0.6 of their time by the launches' shapes; one
after another it is 1, so 0.85 tells the two apart, the best of five rounds each).
Whatever the way, on device memory and at one, two and three members: the bits of
the members' own sweeps, and the same statistics."""
import ctypes as C
import time

import numpy as np
import pytest

from test_gpu_rhs import assert_bitwise

pytestmark = pytest.mark.gpu


def _taped(c, steps):
    import sgnx
    s = sgnx.SGN2D(**c.solver_kwargs())
    s.setDepth(c.depth["Hnod"])
    s.upload(c.U0)
    s.tapeKeepStages(True)
    s.tapeBegin(1 << 20)
    s.integrateAdaptive(0.1, 1e9, s.cflTimeStep(None, 0.5),
                        sgnx.RkOpts(atol=1e-8, rtol=1e-6, max_accepted=steps))
    s.tapeEnd()
    return s


class _Sweeps:
    """n taped members, their cotangents and results on the device"""

    def __init__(self, cases, steps):
        import sgnx
        from sgnx import hip
        self.s = [_taped(c, steps) for c in cases]
        self.b = sgnx.Batch(self.s)
        rng = np.random.default_rng(3)
        self.w = [hip.DeviceArray.from_host(rng.normal(size=s.nTotal())) for s in self.s]
        self.u = [hip.DeviceArray(s.nTotal()) for s in self.s]
        self.th = [hip.DeviceArray(s.nDof()) for s in self.s]
        self.ptrs = [(C.c_void_p * len(self.s))(*[d.address for d in a])
                     for a in (self.w, self.u, self.th)]

    def alone(self):
        for s, w, u, th in zip(self.s, self.w, self.u, self.th):
            s.adjoint_device(w.address, 0, u.address, th.address)

    def batched(self):
        from sgnx import _lib as L
        w, u, th = self.ptrs
        assert self.b.lib.sgnx_batch_adjoint(self.b.h, w, None, u, th, L.MEM_DEVICE) == L.SGNX_OK

    def results(self):
        return [d.download() for d in self.u + self.th]

    def close(self):
        self.b.close()
        for x in self.s:
            x.close()
        for d in self.w + self.u + self.th:
            d.free()


def test_small_members_are_swept_together():
    from sgnx import cases
    q = _Sweeps([cases.shoal(seed=k, Nx=128, Ny=64) for k in range(12)], 5)
    best = {}
    for _ in range(6):                     # (the first warms up)
        for f in (q.alone, q.batched):
            t = time.perf_counter()
            f()
            best.setdefault(f.__name__, []).append(time.perf_counter() - t)
    q.close()
    alone, batched = (min(best[k][1:]) for k in ("alone", "batched"))
    assert batched < 0.85 * alone, (batched, alone)


@pytest.mark.parametrize("sizes", [[(128, 64)], [(64, 33)], [(128, 64)] * 2, [(200, 100)] * 2,
                                   [(31, 17), (256, 128)], [(256, 128), (96, 50), (203, 101)]])
def test_every_way_gives_the_bits_of_the_members_own_sweeps(sizes):
    from sgnx import cases
    q = _Sweeps([cases.shoal(seed=7 + k, Nx=a, Ny=b) for k, (a, b) in enumerate(sizes)], 3)
    q.alone()
    want, stats = q.results(), [s.adjointStats() for s in q.s]
    q.batched()
    for i, (g, w) in enumerate(zip(q.results(), want)):
        assert_bitwise(g, w, f"result {i}")
    assert [s.adjointStats() for s in q.s] == stats == [(0, 0)] * len(sizes)
    q.close()
