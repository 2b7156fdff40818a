"""Windowed local updates (variant 4) against the general path (variant 1: G in global memory, one
rank-4 update per acceptance) on the same field, G and uniforms.

Sizes and workgroup counts where its pieces change: columns resident in LDS or not, one and two
rows per thread at the window's end (n <= 512, above), one column per workgroup up to all of them
(W behind X in one or several chunks, a last tile or a last item of one column), windows of a size
that is no multiple of four sites, odd L (n no multiple of 16, generic checkerboard), the smallest
and the largest n.

Tolerance: the two differ in the order of sums only. An update perturbs G by a few eps times its
entries (|G| of order 1) times the condition of M (below 100 for accepted proposals), N of them in
a slice add up to at most N * 100 * 2.2e-16 < 1e-11 at N = 256.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd():
    import dqmc_amd
    dqmc_amd.load()
    return dqmc_amd


def slices(amd, variant, L, wg, count, **kw):
    p = amd.Params(L=L, slices=20, hoppings=(1.0, 0.5, 0.5, 1.0), lam=1.5, r=0.3, **kw)
    c = amd.DQMC(p, uniforms=amd.UniformStream(5))
    c.set_local_variant(variant)
    c.init(np.random.default_rng(L).uniform(-1, 1, (3, p.N, p.slices)))
    if wg:
        c.set_groups(wg_local=wg)
    c.set_proposal_log(4 * p.N * count)
    for k in range(count):
        if k:
            c.propagate()
        c.local_updates()
    out = c.hsfield, c.greens, c.proposal_log(), c.boson_action, c.stats().accepted
    c.close()
    return out


@pytest.mark.parametrize("L,wgs", [(2, (0, 1)), (3, (0, 1, 2)), (4, (0, 1, 3)), (5, (0, 7)), (6, (0, 2)), (7, (0, 1, 5)),
                                   (9, (0, 1, 2, 24)), (10, (0, 3)), (12, (0, 4)), (13, (0, 2)), (16, (0, 1, 8))])
def test_window_equals_general_path(amd, L, wgs):
    kw = {"bfield": True} if L in (6, 12) else {}
    want = slices(amd, 1, L, 8, 2, **kw)
    for wg in wgs:
        print("windowed updates L=%d workgroups %d" % (L, wg), flush=True)
        got = slices(amd, 4, L, wg, 2, **kw)
        assert np.array_equal(got[0], want[0])
        assert got[4] == want[4]
        assert np.abs(got[1] - want[1]).max() < 1e-11
        assert got[2].shape == want[2].shape and np.abs(got[2] - want[2]).max() < 1e-9 * np.abs(want[2]).max()
        assert abs(got[3] - want[3]) <= 1e-12 * abs(want[3])


@pytest.mark.parametrize("count", [0, 3, 4, 57])
def test_uniforms_run_out(amd, count):
    """The proposals that the stream still covers are made, then the error; as variant 1 does."""
    logs = []
    for variant, wg in ((1, 4), (4, 0), (4, 2)):
        p = amd.Params(L=6, slices=20, hoppings=(1.0, 0.5, 0.5, 1.0), lam=1.0, r=1.0)
        c = amd.DQMC(p)
        c.set_local_variant(variant)
        c.init(np.random.default_rng(1).uniform(-1, 1, (3, p.N, p.slices)))
        if wg:
            c.set_groups(wg_local=wg)
        c.set_proposal_log(4 * p.N)
        u = np.random.default_rng(2).random(max(count, 1))
        ptr = u.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
        assert c.lib.dqmc_set_uniforms(c.h, ptr, count) == 0
        acc = ctypes.c_double()
        assert c.lib.dqmc_local_updates(c.h, p.box, ctypes.byref(acc)) != 0
        n = ctypes.c_longlong()
        log = np.zeros((4 * p.N, 4))
        c.lib.dqmc_get_proposal_log(c.h, log.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), ctypes.byref(n))
        logs.append((n.value, log))
        c.close()
    for n, log in logs[1:]:
        assert n == logs[0][0] and np.abs(log - logs[0][1]).max() < 1e-9 * max(1.0, np.abs(logs[0][1]).max())
