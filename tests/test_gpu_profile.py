"""Profiled evaluations that run as jobs take their HIP events from the chain's pool again: after the
first ones the process creates none.

An event is an object of the runtime on this thread's heap, about 1.1 KB (mallinfo2 counts it), and
a timed launch records two. The runtime's heap grows by itself from launch to launch, so profiled
evaluations are compared with as many plain ones: they may grow it by 1 KB more per record,
half of what creating the events anew takes.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class MallInfo2(ctypes.Structure):
    _fields_ = [(f, ctypes.c_size_t) for f in ("arena", "ordblks", "smblks", "hblks", "hblkhd", "usmblks", "fsmblks",
                                               "uordblks", "fordblks", "keepcost")]


@pytest.mark.parametrize("what", ["grad", "measure_tdgfs", "measure_greens"])
def test_events_are_reused(what):
    import dqmc_amd
    from dqmc_amd import _capi
    dqmc_amd.load()
    libc = ctypes.CDLL(None)
    libc.mallinfo2.restype = MallInfo2
    print("profiled %s" % what, flush=True)
    p = dqmc_amd.Params(L=4, slices=40, safe_mult=5, hoppings=(1.0, 0.5, 0.5, 1.0), lam=1.0, r=1.0)
    c = dqmc_amd.DQMC(p, uniforms=dqmc_amd.UniformStream(1))
    c.init(np.random.default_rng(1).uniform(-1, 1, (3, p.N, p.slices)))
    c.allocate_tdgfs()
    ms, cnt = np.zeros(_capi.K_NCLASS), np.zeros(_capi.K_NCLASS, dtype=np.int64)

    def growth(mask):
        c.lib.dqmc_profile(c.h, mask)
        for k in range(60):
            if k == 10:
                before = libc.mallinfo2().uordblks
            getattr(c, what)()
            _capi.check(c.lib.dqmc_profile_read(c.h, _capi.dptr(ms), cnt.ctypes.data_as(_capi._LL), _capi.K_NCLASS))
        return libc.mallinfo2().uordblks - before

    plain = growth(0)
    assert cnt.sum() == 0
    profiled = growth((1 << _capi.K_NCLASS) - 1)
    assert cnt.sum() > 20 and ms.sum() > 0
    assert profiled - plain < 50 * 1024 * int(cnt.sum())
    c.close()
