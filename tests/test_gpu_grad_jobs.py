"""dS/dphi with its intervals in parallel against the pass it replaces: build_stack, then one
propagate per slice (down). Compared: the gradient is checked against the oracle elsewhere
(test_gpu_parity.py); here the state the chain is left in -- every stack element, G at slice 1,
log|det G|, the drift statistics, slice and direction -- and a sweep from there.

Shapes: one interval (R = 1), two, several, one slice per interval, odd L with the generic
checkerboard, a magnetic field, eight and more intervals (the matrix-core solve).

Tolerance: both passes form the same products and factorisations; the solve may run on another
kernel (8 jobs and more), so G agrees to rounding times its condition: 1e-12 as for merged sweeps.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd():
    import dqmc_amd
    dqmc_amd.load()
    return dqmc_amd


@pytest.mark.parametrize("L,M,s,bfield,checks", [
    (4, 10, 10, False, True), (4, 20, 10, False, True), (4, 6, 1, False, True), (3, 12, 2, False, True),
    (6, 50, 10, True, False), (10, 90, 10, False, True)])
def test_gradient_jobs_leave_the_sequential_state(amd, L, M, s, bfield, checks):
    print("gradient jobs L=%d M=%d safe_mult=%d" % (L, M, s), flush=True)
    p = amd.Params(L=L, slices=M, safe_mult=s, hoppings=(1.0, 0.5, 0.5, 1.0), lam=1.0, r=1.0, bfield=bfield,
                   all_checks=checks)
    phi = np.random.default_rng(100 * L + M).uniform(-1.0, 1.0, (3, p.N, M))
    a = amd.DQMC(p, uniforms=amd.UniformStream(5))
    b = amd.DQMC(p, uniforms=amd.UniformStream(5))
    for c in (a, b):
        c.init(phi)
        c.reset_stats()
    for _ in range(2):  # the second pass runs on warm job storage
        g, S = a.grad()
    b.build_stack()
    for _ in range(M):
        b.propagate()
    for k in range(M // s + 1):
        for x, y in zip(a.stack_element(k), b.stack_element(k)):
            assert np.abs(x - y).max() <= 1e-12 * max(1.0, np.abs(y).max()), k
    assert np.abs(a.greens - b.greens).max() < 1e-12
    assert abs(a.log_det - b.log_det) < 1e-12 * max(1.0, abs(b.log_det)) * p.N
    sa, sb = a.stats(), b.stats()
    assert abs(sa.drift_max - sb.drift_max) < 1e-12 and abs(sa.drift_last - sb.drift_last) < 1e-12
    assert (a.current_slice, a.direction) == (b.current_slice, b.direction) == (1, -1)
    assert g.shape == (3, p.N, M) and np.isfinite(S)
    for c in (a, b):
        c.sweep(2)
    assert np.array_equal(a.hsfield, b.hsfield)
    assert np.abs(a.greens - b.greens).max() < 1e-11
    a.close()
    b.close()
