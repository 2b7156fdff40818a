"""Time-displaced Green's functions and the measurement's equal-time one as jobs side by side,
against the sequential pass (which the verbatim UDT route keeps), over the checkerboards, interval
lengths and numbers of intervals where the job lists change: one slice per interval (no fill), more
inversions than one round holds (R = 40: 80 jobs, rounds of 32), an odd number of intervals (the
sequential pass for both, the two halves of unequal length for the equal-time function).

Tolerance: both solve with brackets of condition up to 2e3 for the entries of order 1 of G:
n eps 2e3 < 2e-10 at n = 400.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd():
    import dqmc_amd
    dqmc_amd.load()
    return dqmc_amd


@pytest.mark.parametrize("L,M,s,bfield", [(3, 12, 2, False), (4, 20, 10, False), (4, 6, 1, False), (4, 8, 8, False),
                                          (5, 30, 5, False), (4, 30, 10, True), (6, 80, 2, True), (10, 20, 5, False)])
def test_jobs_equal_the_sequential_pass(amd, L, M, s, bfield):
    print("measurement jobs L=%d M=%d safe_mult=%d" % (L, M, s), flush=True)
    got = []
    for route in (0, 1):
        p = amd.Params(L=L, slices=M, safe_mult=s, hoppings=(1.0, 0.5, 0.5, 1.0), lam=1.0, r=0.5, bfield=bfield)
        c = amd.DQMC(p, uniforms=amd.UniformStream(1))
        c.init(np.random.default_rng(3).uniform(-1, 1, (3, p.N, M)))
        amd._capi.check(c.lib.dqmc_set_udt_route(c.h, route))
        before = c.greens, c.log_det
        out = [c.measure_greens()]
        if M % 2 == 0:
            c.allocate_tdgfs()
            for _ in range(2):  # a second pass on the same storage
                c.measure_tdgfs()
            out += [g for tau in range(1, M + 1) for g in c.tdgf(tau)]
        assert np.array_equal(c.greens, before[0]) and c.log_det == before[1]
        got.append(out)
        c.close()
    for a, b in zip(*got):
        assert np.abs(a - b).max() <= 2e-10 * max(1.0, np.abs(b).max())
