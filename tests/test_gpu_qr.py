"""Blocked QR (k_qr_pipe): factors at the sizes and workgroup counts where its tiles, rows per
thread and block ownership change.

n = 4 L^2 covers one to four rows per thread (up to n = 256, 512, 768, 1024), last panels of four
columns (n = 36, 100, 196, 324, 676) and tiles that straddle row 0 (n not a multiple of 16).
Workgroup counts: one (no flags), two (every trailing block on one workgroup), three and five
(blocks dealt round robin; the 16-column trailing update where a workgroup holds 128 columns and
more), and the default.

Tolerances: Householder QR is column-wise backward stable, |A - QR|_j <= c n eps |A_j| with a
small c, and |Q^H Q - I| <= c n eps; c = 8, eps = 2.2e-16.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd():
    import dqmc_amd
    dqmc_amd.load()
    return dqmc_amd


EPS = 2.220446049250313e-16


@pytest.mark.parametrize("L", [3, 4, 5, 7, 8, 9, 10, 12, 13, 14, 16])
def test_blocked_qr_sizes_and_workgroups(amd, L):
    n = 4 * L * L
    rng = np.random.default_rng(L)
    A = (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) * np.exp(rng.uniform(-20, 20, n))
    c = amd.DQMC(amd.Params(L=L, slices=20, hoppings=(1.0, 0.5, 0.5, 1.0), lam=1.0, r=1.0))
    for wg in (0, 1, 2, 3, 5):
        print("blocked QR n=%d workgroups %d" % (n, wg), flush=True)
        if wg:
            c.set_groups(wg_qr=wg)
        U, D, T = c.decompose_udt_prepivoted(A)
        assert np.abs(U.conj().T @ U - np.eye(n)).max() <= 8 * n * EPS
        assert (np.abs((U * D) @ T - A) / np.linalg.norm(A, axis=0)).max() <= 8 * n * EPS
        assert np.all(D > 0)
    c.close()


@pytest.mark.parametrize("L,wgs", [(2, (1, 3)), (4, (1, 3, 4, 8)), (5, (1, 2, 4, 9)), (8, (1, 4, 7, 32)),
                                   (10, (1, 5, 6, 25, 50)), (12, (6, 25, 72)), (13, (10, 84)), (16, (11, 128))])
def test_factors_do_not_depend_on_blocks_per_workgroup(amd, L, wgs):
    """A block's update is the same arithmetic whichever workgroup makes it and whatever that
    workgroup holds besides (fewer than 128 columns each, or a lone workgroup up to n = 512: beyond
    that the 16-column form takes over), so U, D and T are equal bit for bit. Where a workgroup holds several blocks, the waves'
    partial sums of consecutive blocks follow one another through LDS."""
    n = 4 * L * L
    rng = np.random.default_rng(50 + L)
    A = (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) * np.exp(rng.uniform(-20, 20, n))
    c = amd.DQMC(amd.Params(L=L, slices=20, hoppings=(1.0, 0.5, 0.5, 1.0), lam=1.0, r=1.0))
    want = None
    for wg in wgs[::-1]:
        assert n <= 512 if wg == 1 else n < 128 * (wg - 1)
        print("blocked QR n=%d workgroups %d" % (n, wg), flush=True)
        c.set_groups(wg_qr=wg)
        got = c.decompose_udt_prepivoted(A)
        want = want or got
        for x, y in zip(got, want):
            assert np.array_equal(x, y)
    c.close()


@pytest.mark.parametrize("L,wg", [(2, 0), (4, 0), (4, 1), (4, 3), (8, 0), (8, 128)])
def test_pivoted_qr_of_nan_columns(amd, L, wg):
    """Columns without a norm come last, so the pivots before them are those of the same matrix with
    zeros there, and D is NaN from the first of them on (one NaN reflector reaches every column);
    nothing is left of the factorisation before, and the next one is unaffected."""
    n = 4 * L * L
    print("pivoted QR with NaN, n=%d workgroups %d" % (n, wg), flush=True)
    rng = np.random.default_rng(70 + L)
    A = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    c = amd.DQMC(amd.Params(L=L, slices=20, hoppings=(1.0, 0.5, 0.5, 1.0), lam=1.0, r=1.0))
    if wg:
        c.set_groups(wg_qr=wg)
    first = c.decompose_udt(A)
    for bad in ([0], [n - 1], [1, n // 2, n - 2], list(range(n))):
        Z, B = A.copy(), A.copy()
        Z[:, bad] = 0
        B[n // 3, bad] = np.nan
        U, D, T = c.decompose_udt(B)
        good = n - len(bad)
        if good:
            assert np.array_equal(D[:good], c.decompose_udt(Z)[1][:good])
        assert np.isnan(D[good:]).all() and np.isnan(U).any() and np.isnan(T).any()
    for x, y in zip(c.decompose_udt(A), first):
        assert np.array_equal(x, y)
    c.close()


@pytest.mark.parametrize("L,wg,nb", [(2, 0, 8), (4, 0, 8), (4, 1, 8), (4, 3, 16), (8, 0, 8), (10, 0, 16), (16, 0, 8)])
def test_blocked_qr_of_nan_columns(amd, L, wg, nb):
    """As for the pivoted QR: the order puts columns without a norm last, by index, so that R of the
    panels before them is that of the same matrix with zeros there."""
    n = 4 * L * L
    print("blocked QR with NaN, n=%d workgroups %d panels of %d" % (n, wg, nb), flush=True)
    rng = np.random.default_rng(90 + L)
    A = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    c = amd.DQMC(amd.Params(L=L, slices=20, hoppings=(1.0, 0.5, 0.5, 1.0), lam=1.0, r=1.0))
    c.set_qr_panel(nb)
    if wg:
        c.set_groups(wg_qr=wg)
    first = c.decompose_udt_prepivoted(A)
    for bad in ([0], [n - 1], [1, n // 2, n - 2], list(range(n))):
        Z, B = A.copy(), A.copy()
        Z[:, bad] = 0
        B[n // 3, bad] = np.nan
        U, D, T = c.decompose_udt_prepivoted(B)
        whole = (n - len(bad)) // nb * nb  # columns of the panels without a NaN
        assert np.array_equal(D[:whole], c.decompose_udt_prepivoted(Z)[1][:whole])
        assert np.isnan(D[n - len(bad):]).all() and np.isnan(U).any() and np.isnan(T).any()
    for x, y in zip(c.decompose_udt_prepivoted(A), first):
        assert np.array_equal(x, y)
    c.close()


@pytest.mark.parametrize("L,wg", [(12, 1), (12, 4), (13, 1), (16, 1), (16, 3)])
def test_few_workgroups_per_chain_in_a_batch(amd, L, wg):
    """n > 512 on few workgroups (every trailing update in the 16-column form) against the default
    counts: the same factorisations up to the order of sums, G through brackets of condition up to
    2e3, so n eps 2e3 < 5e-10, and the same decisions."""
    print("batch of 2, n=%d, %d workgroups per blocked QR" % (4 * L * L, wg), flush=True)
    p = amd.Params(L=L, slices=10, safe_mult=5, hoppings=(1.0, 0.5, 0.5, 1.0), lam=1.0, r=1.0)
    confs = [np.random.default_rng(k).uniform(-1, 1, (3, p.N, p.slices)) for k in range(2)]
    got = []
    for w in (0, wg):
        b = amd.Batch([p, p], streams=[amd.UniformStream(k) for k in range(2)])
        if w:
            b.set_groups(wg_qr=w)
        b.init(confs)
        b.sweep(1)
        got.append([(b.greens(k), b.get_field(k)) for k in range(2)])
        b.close()
    for (g0, f0), (g1, f1) in zip(*got):
        assert np.array_equal(f0, f1) and np.abs(g0 - g1).max() < 5e-10
