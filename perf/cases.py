"""What the framework is used for, as timed cases: sweeps of one Markov chain and of batches of
chains, single update steps driven from the host, the gradient dS/dphi and HMC, and the fermionic
measurements, over the lattice sizes the library takes (L = 4 .. 16, n = 4 L^2 = 64 .. 1024) and
every hopping option (Assaad checkerboard, with a magnetic field, generic bond checkerboard at odd
L, dense). All in float64 / complex128, the library's only data type. Fields are uniform in
[-1, 1]^3, uniforms are the host MT19937 stream, both from the seed.
"""
import math

import numpy as np
import torch

from dqmc_amd import Batch, DQMC, Params, UniformStream
from dqmc_amd import _capi

HOPPINGS = (1.0, 0.5, 0.5, 1.0)
MU = -0.5
DTAU, SAFE = 0.1, 10
C_BOSON, U_BOSON = 3.0, 1.0
BOX = 0.5


def listed():
    one = {"lam": 1.0, "r": 1.0}
    return [
        # one stabilisation interval of update steps driven one by one, as the reference's update(mc, i)
        # does: the smallest calls, bound by launches and host round trips
        dict(one, name="steps_L4", kind="steps", L=4, M=50, hop="chkr"),
        # the smallest whole sweep, without the checkerboard (matrix products in place of plaquettes)
        dict(one, name="sweep_L4_dense", kind="sweep", L=4, M=50, hop="dense"),
        # a lattice of ordinary size with a magnetic field (complex plaquettes, one block each)
        dict(one, name="sweep_L8_bfield", kind="sweep", L=8, M=100, hop="bfield"),
        # odd L: the generic bond checkerboard, n = 324, nothing a multiple of a tile
        dict(one, name="sweep_L9_generic", kind="sweep", L=9, M=50, hop="chkr"),
        # the headline workload: one chain at L = 10, beta = 20
        dict(one, name="sweep_L10", kind="sweep", L=10, M=200, hop="chkr"),
        # the largest lattice: n = 1024
        dict(one, name="sweep_L16", kind="sweep", L=16, M=100, hop="chkr"),
        # 64 independent chains of the headline workload on one GPU
        dict(one, name="batch64_L10", kind="batch", L=10, M=200, hop="chkr", chains=64),
        # a parameter scan: 64 chains of L in {6, 8, 10, 12}, beta in {5, 10, 20}, per-chain r and lambda
        dict(name="batch64_mixed", kind="scan", chains=64, Ms=200),
        # the force of an HMC or gradient-flow run
        dict(one, name="grad_L12", kind="grad", L=12, M=100, hop="chkr"),
        # one HMC trajectory of a small lattice
        dict(one, name="hmc_L6", kind="hmc", L=6, M=50, hop="chkr", steps=3),
        # a measurement: equal-time and time-displaced Green's functions and their observables
        dict(one, name="measure_L8", kind="measure", L=8, M=100, hop="chkr"),
    ]


def draw(rng):
    kind = rng.choice(("steps", "sweep", "sweep", "batch", "scan", "grad", "hmc", "measure"))
    lam, r = round(rng.uniform(0.5, 2.0), 4), round(rng.uniform(-1.0, 1.0), 4)
    case = {"kind": kind, "lam": lam, "r": r}
    if kind == "scan":
        return {"kind": kind, "chains": rng.randint(8, 48), "Ms": 10 * rng.randint(4, 16)}
    # the lattice over the logarithm of n, the number of slices over its own
    top = {"steps": 16, "sweep": 16, "batch": 11, "grad": 13, "hmc": 9, "measure": 9}[kind]
    L = min(top, max(4, int(round(math.exp(rng.uniform(math.log(4), math.log(top)))))))
    # a sweep costs about M (4 + (L / 6)^3): drawn ones stay below the largest listed
    most = {"steps": 200, "sweep": 200, "batch": 120, "grad": 100, "hmc": 50, "measure": 60}[kind]
    if L > 12:
        most = min(most, 80)
    case.update(L=L, M=10 * int(round(math.exp(rng.uniform(math.log(2), math.log(most / 10))))))
    case["hop"] = rng.choice(("chkr", "chkr", "bfield") + (("dense",) if L <= 8 else ()))
    if kind == "batch":
        case["chains"] = int(round(math.exp(rng.uniform(math.log(2), math.log(64)))))
        if L > 9:
            case["chains"] = min(case["chains"], 40)
    if kind == "hmc":
        case["steps"] = rng.randint(1, 4)
    if kind == "measure":
        case["M"] += 10 * (case["M"] // 10 % 2)  # the two halves of imaginary time are filled apart: M / safe_mult even
    return case


def params(case, L, M, seed, lam, r):
    hop = case.get("hop", "chkr")
    return Params(L=L, slices=M, delta_tau=DTAU, safe_mult=SAFE, hoppings=HOPPINGS, mu1=MU, mu2=MU, lam=lam, r=r,
                  c=C_BOSON, u=U_BOSON, checkerboard=hop != "dense", bfield=hop == "bfield", box=BOX, seed=seed)


def field(L, M, seed):
    return np.random.default_rng(seed).uniform(-1.0, 1.0, (3, L * L, M))


def chain_list(case, seed):
    """(L, M, lam, r, seed) of a batch's chains."""
    if case["kind"] == "batch":
        return [(case["L"], case["M"], case["lam"], case["r"], 1000 * seed + c) for c in range(case["chains"])]
    rng = np.random.default_rng(seed)
    return [((6, 8, 10, 12)[c % 4], (case["Ms"] // 4, case["Ms"] // 2, case["Ms"])[c // 4 % 3] // 10 * 10,
             0.5 + 1.5 * float(rng.uniform()), (-1.0, 0.0, 1.0)[c // 12 % 3], 1000 * seed + c)
            for c in range(case["chains"])]


class State:
    pass


def prepare(case, seed):
    s = State()
    s.case = case
    if case["kind"] in ("batch", "scan"):
        chains = chain_list(case, seed)
        ps = [params(case, L, M, sd, lam, r) for L, M, lam, r, sd in chains]
        s.b = Batch(ps, streams=[UniformStream(sd + 7) for _, _, _, _, sd in chains])
        s.b.init([field(L, M, sd) for L, M, _, _, sd in chains])
        # the arrays a program reads every chain's configuration and Green's function into
        s.sizes = [(3 * L * L * M, 16 * L ** 4) for L, M, _, _, _ in chains]
        s.fields = np.zeros(sum(a for a, _ in s.sizes))
        s.greens = np.zeros(sum(b for _, b in s.sizes), dtype=np.complex128)
        return s
    L, M = case["L"], case["M"]
    s.p = params(case, L, M, seed, case["lam"], case["r"])
    s.c = DQMC(s.p, uniforms=UniformStream(seed + 7))
    s.c.init(field(L, M, seed))
    if case["kind"] == "hmc":
        rng = np.random.default_rng(seed + 3)
        s.momenta, s.u = rng.standard_normal((3, L * L, M)), float(rng.uniform())
    if case["kind"] == "measure":
        s.c.allocate_tdgfs()
    return s


def run(s):
    kind = s.case["kind"]
    if kind in ("batch", "scan"):
        s.b.sweep(1)
        f = g = 0
        for c, (nf, ng) in enumerate(s.sizes):
            _capi.check(s.b.lib.dqmc_batch_get_field(s.b.h, c, _capi.dptr(s.fields[f:f + nf])))
            _capi.check(s.b.lib.dqmc_batch_get_greens(s.b.h, c, _capi.dptr(s.greens[g:g + ng].view(np.float64))))
            f, g = f + nf, g + ng
        return {"field": s.fields, "greens": s.greens}
    c = s.c
    if kind in ("sweep", "steps"):
        if kind == "sweep":
            c.sweep(1)
        else:
            for _ in range(SAFE):
                c.update()
        return {"field": c.hsfield, "greens": c.greens, "boson_action": c.boson_action}
    if kind == "grad":
        g, action = c.grad()
        return {"grad": g, "action": action}
    if kind == "hmc":
        accepted, dh = c.hmc_trajectory(s.momenta, s.case["steps"], 0.02, s.u)
        return {"accepted": accepted, "dh": dh, "field": c.hsfield, "greens": c.greens}
    g = c.measure_greens()
    c.measure_tdgfs()
    pc, cdc = c.measure_etpc(), c.measure_etcdc()
    zpc, zcdc = c.measure_zfpc(), c.measure_zfcdc()
    xx, yy, rho = c.measure_zfccc()
    return {"greens": g, "etpc": list(pc), "etcdc": list(cdc), "zfpc": list(zpc), "zfcdc": list(zcdc),
            "zfccc": [xx, yy], "sfdensity": rho}


# ---------------------------------------------------------------------------------------------
# The work of one pass: the algorithm's own counts, each matrix read and written once per
# operation that needs it whole.
# ---------------------------------------------------------------------------------------------

def sweep_work(L, M):
    n = 4.0 * L * L
    acc = 0.68 * L * L * M                       # accepted proposals of a sweep
    refresh = M / SAFE                           # stack factorisations and Green's functions
    flops = (acc * 34.0 + 3.0 * M * 74.0) * n * n   # rank-4 updates; wraps and stack products
    # per refresh: UDT (QR and Q), its T product; three products, a QR and a solve for G
    flops += refresh * (16 / 3 + 16 / 3 + 8 + 3 * 8 + 16 / 3 + 8) * n ** 3
    # G read and written by each slice's updates and each wrap, the stack by its products
    return (M * (32.0 + 64.0 + 32.0) + refresh * 16.0 * 20) * n * n, flops


def work(case):
    kind = case["kind"]
    if kind in ("batch", "scan"):
        each = [sweep_work(L, M) for L, M, _, _, _ in chain_list(case, 1)]
        return {"bytes": sum(b for b, _ in each), "flops": sum(f for _, f in each)}
    L, M = case["L"], case["M"]
    n = 4.0 * L * L
    b, f = sweep_work(L, M)
    if kind == "steps":
        b, f = b * SAFE / M, f * SAFE / M
    if kind in ("grad", "hmc"):  # no updates of G; the stack is built and then rebuilt on the way down
        f = (4.0 * M * 74.0) * n * n + M / SAFE * (2 * (16 / 3 + 16 / 3 + 8) + 3 * 8 + 16 / 3 + 8) * n ** 3
        b = (M * (64.0 + 64.0) + M / SAFE * 16.0 * 30) * n * n
        if kind == "hmc":
            b, f = b * (case["steps"] + 1), f * (case["steps"] + 1)
    if kind == "measure":
        # four chains of UDTs, two stabilised inversions (3 inverses, 2 UDTs, 6 products) per
        # interval, two propagated matrices per slice
        f = (6.0 * M * 74.0) * n * n + M / SAFE * (4 * (32 / 3 + 8) + 2 * (16 + 64 / 3 + 48)) * n ** 3
        b = (M * (6 * 32.0 + 32.0) + M / SAFE * 16.0 * 80) * n * n
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------------------------------------
# The same results by plain dense linear algebra in 64 bits.
# ---------------------------------------------------------------------------------------------

class Model:
    """B_l = K exp(V(phi_l)): the hopping factor K as four N x N flavour blocks, the
    interaction as a 4 x 4 flavour block per site."""

    def __init__(self, case, phi):
        self.L, self.M = case["L"], case["M"]
        self.N = N = self.L ** 2
        self.n, self.phi, self.lam, self.r = 4 * N, phi, case["lam"], case["r"]
        hop, L = case["hop"], self.L
        site = np.arange(N).reshape(L, L).T  # site y + x L at [y, x]
        self.nb = np.stack([np.roll(site, s, a).T.ravel() for s, a in ((-1, 0), (-1, 1), (1, 0), (1, 1))])
        bonds = [(int(s), int(self.nb[k][s]), k) for s in range(N) for k in (0, 1)]  # up, then right

        def bond_matrix(bs, flux, t):
            T = torch.zeros(N, N, dtype=torch.complex128)
            for a, b, k in bs:
                y, x = a % L, a // L
                ph = (flux * L * x if y == L - 1 else 0.0) if k == 0 else -flux * y
                w = -t[1 - k] * complex(math.cos(ph), math.sin(ph))  # the entry (a, b)
                T[a, b] += w
                T[b, a] += w.conjugate()
            return T

        if hop == "dense":
            groups = [bonds]
        elif L % 2:  # greedy colouring in bond order
            groups, left = [], bonds
            while left:
                free, take, rest = set(range(N)), [], []
                for q in left:
                    if q[0] in free and q[1] in free:
                        free -= {q[0], q[1]}
                        take.append(q)
                    else:
                        rest.append(q)
                groups.append(take)
                left = rest
        else:  # plaquettes with their corner at even (x, y), then those at odd (x, y)
            where = lambda s, g: ((s % L - g) % L // 2, (s // L - g) % L // 2)  # noqa: E731
            groups = [[q for q in bonds if where(q[0], g) == where(q[1], g)] for g in (0, 1)]
        fx, fy = (HOPPINGS[0], HOPPINGS[1]), (HOPPINGS[2], HOPPINGS[3])  # (horizontal, vertical) of the two flavours
        phi0 = 2 * math.pi / N if hop == "bfield" else 0.0
        K, half_inv = [], []
        for t, flux in ((fx, phi0), (fy, phi0), (fx, -phi0), (fy, -phi0)):
            e = [[torch.linalg.matrix_exp(-f * DTAU * bond_matrix(g, flux, t)) for f in (1.0, 0.5, -0.5)] for g in groups]
            P = e[0][0]
            for g in e[1:]:
                P = g[1] @ P @ g[1]
            K.append(P * math.exp(DTAU * MU))
            H = torch.eye(N, dtype=torch.complex128)
            for g in e:
                H = H @ g[2]
            half_inv.append(H)
        self.K = torch.stack(K)
        self.Ki = torch.linalg.inv(self.K)
        self.half_inv = torch.stack(half_inv)  # exp(+dtau T / 2) of the groups, the first one leftmost
        self.half = torch.linalg.inv(self.half_inv)

    def blocks(self, K, X):
        return (K @ X.reshape(4, self.N, -1)).reshape(self.n, -1)

    def ev(self, l, power, phi=None):
        """exp(power V) of a slice (or of the given vectors) as (sites, 4, 4)."""
        f = torch.as_tensor(self.phi[:, :, l] if phi is None else phi)
        nrm = f.square().sum(0).sqrt()
        x = self.lam * DTAU * nrm
        sh = power * torch.sinh(x) / nrm
        S, R, C = torch.complex(-f[0] * sh, f[1] * sh), -f[2] * sh, torch.cosh(x)
        E = torch.zeros(f.shape[1], 4, 4, dtype=torch.complex128)
        for a in range(4):
            E[:, a, a] = C.to(E.dtype)
        E[:, 0, 1] = E[:, 3, 2] = S
        E[:, 1, 0] = E[:, 2, 3] = S.conj()
        E[:, 0, 3] = E[:, 3, 0] = R.to(E.dtype)
        E[:, 1, 2] = E[:, 2, 1] = -R.to(E.dtype)
        return E

    def mix(self, E, X):
        return torch.einsum("iab,bij->aij", E, X.reshape(4, self.N, -1)).reshape(self.n, -1)

    def left(self, l, X):
        return self.blocks(self.K, self.mix(self.ev(l, 1), X))

    def dag(self, l, X):  # B_l^H X; exp(V) is hermitian
        return self.mix(self.ev(l, 1), self.blocks(self.K.mH, X))

    def down(self, l, G):  # B_l^-1 G B_l
        G = self.mix(self.ev(l, -1), self.blocks(self.Ki, G))
        return self.dag(l, G.mH).mH

    def udt(self, X, D, T):
        """U D' T' = X D T."""
        X = X * D
        order = torch.argsort(X.abs().square().sum(0), descending=True)
        Q, R = torch.linalg.qr(X[:, order])
        d = R.diagonal().abs()
        back = torch.empty_like(order)
        back[order] = torch.arange(len(order))
        return Q, d, (R / d[:, None])[:, back] @ T

    def one(self):
        eye = torch.eye(self.n, dtype=torch.complex128)
        return eye, torch.ones(self.n, dtype=torch.float64), eye.clone()

    def lefts(self):
        """UDT of B_(k SAFE) .. B_1 for k = 0 .. M / SAFE."""
        got = [self.one()]
        for k in range(self.M // SAFE):
            U, D, T = got[-1]
            for l in range(k * SAFE, (k + 1) * SAFE):
                U = self.left(l, U)
            got.append(self.udt(U, D, T))
        return got

    def more_right(self, k, right):
        """UDT of (B_M .. B_(k SAFE + 1))^H from that of the interval above."""
        U, D, T = right
        for l in range((k + 1) * SAFE - 1, k * SAFE - 1, -1):
            U = self.dag(l, U)
        return self.udt(U, D, T)

    def greens(self, left, right):
        """[1 + left right^H]^-1 and log |det| of it."""
        (Ul, Dl, Tl), (Ur, Dr, Tr) = left, right
        lb, ls, rb, rs = Dl.clamp(min=1), Dl.clamp(max=1), Dr.clamp(min=1), Dr.clamp(max=1)
        A = (Ul.mH @ Ur) / lb[:, None] / rb + ls[:, None] * (Tl @ Tr.mH) * rs
        G = (Ur / rb) @ torch.linalg.solve(A, Ul.mH / lb[:, None])
        return G, float(-torch.linalg.slogdet(A)[1] - lb.log().sum() - rb.log().sum())

    def downward(self):
        """(l, G(l)) for l = M - 1 .. 0 (0-based slices), where the caller may change G and the
        slice's field before the next."""
        lefts, right, M = self.lefts(), self.one(), self.M
        G, self.log_det = self.greens(lefts[-1], right)
        for l in range(M - 1, -1, -1):
            G = self.down(l, G)
            box = [G]
            yield l, box
            G = box[0]
            if l % SAFE == 0 and l > 0:
                right = self.more_right(l // SAFE, right)
                G = self.greens(lefts[l // SAFE], right)[0]

    def action(self):
        h = self.phi.reshape(3, self.L, self.L, self.M)
        t = [h - np.roll(h, -1, a) for a in (3, 1, 2)]
        sq = (self.phi ** 2).sum(0)
        return (0.5 / DTAU / C_BOSON ** 2 * (t[0] ** 2).sum() + 0.5 * DTAU * ((t[1] ** 2).sum() + (t[2] ** 2).sum()) +
                DTAU * (self.r / 2 * sq + U_BOSON / 4 * sq ** 2).sum())

    def site_updates(self, l, box, uniforms):
        """Metropolis proposals of every site of slice l; returns the change of the action."""
        phi, N, total = self.phi, self.N, 0.0
        G, eye = box[0].resolve_conj().numpy().copy(), np.eye(4)
        old_inv = self.ev(l, -1).numpy()
        time = phi[:, :, (l + 1) % self.M] + phi[:, :, l - 1]
        for i in range(N):
            old = phi[:, i, l].copy()
            new = old + (-BOX + 2 * BOX * np.array([next(uniforms) for _ in range(3)]))
            d, q0, q1 = new - old, old @ old, new @ new
            dS = ((q1 - q0) - time[:, i] @ d) / (DTAU * C_BOSON ** 2)
            dS += 0.5 * DTAU * (4 * (q1 - q0) - 2 * (phi[:, self.nb[:, i], l].sum(1) @ d))
            dS += DTAU * (0.5 * self.r * (q1 - q0) + 0.25 * U_BOSON * (q1 * q1 - q0 * q0))
            delta = old_inv[i] @ self.ev(l, 1, new[:, None]).numpy()[0] - eye
            Mx = eye + delta @ (eye - G[i::N, i::N])
            p = math.exp(-dS) * np.linalg.det(Mx).real
            if p > 1 or next(uniforms) < p:
                phi[:, i, l] = new
                total += dS
                A = G[:, i::N].copy()
                A[i::N] -= eye
                G += (A @ np.linalg.inv(Mx)) @ (delta @ G[i::N])
        box[0] = torch.from_numpy(G)
        return total

    def gradient(self):
        """dS/dphi and S."""
        h = self.phi.reshape(3, self.L, self.L, self.M)
        near = lambda a: 2 * h - np.roll(h, -1, a) - np.roll(h, 1, a)  # noqa: E731
        g = near(3) / (DTAU * C_BOSON ** 2) + DTAU * (near(1) + near(2))
        g += DTAU * (self.r * h + U_BOSON * (h ** 2).sum(0) * h)
        g = g.reshape(3, self.N, self.M)
        for l, box in self.downward():
            f = torch.as_tensor(self.phi[:, :, l].copy()).requires_grad_()
            OG = torch.eye(4, dtype=torch.complex128) - box[0].reshape(4, self.N, 4, self.N).diagonal(dim1=1, dim2=3).permute(2, 0, 1)
            torch.einsum("iab,ibc,ica->", OG, self.ev(l, -1), self.ev(l, 1, f)).real.backward()
            g[:, :, l] -= f.grad.numpy()
        return g, float(self.action()) + self.log_det


def exact(case, seed):
    kind = case["kind"]
    if kind in ("batch", "scan"):
        return None  # the chains are those of "sweep", one by one
    n, M = 4 * case["L"] ** 2, case["M"]
    updates, passes = kind in ("sweep", "steps"), case.get("steps", 0) + 1
    if (updates and n ** 3 * M > 2e9) or n ** 3 * M * passes > 2e10:
        return None  # over 20 seconds
    m = Model(case, field(case["L"], M, seed))
    if kind == "grad":
        g, action = m.gradient()
        return {"grad": g, "action": action}
    if updates:
        rng = np.random.Generator(np.random.MT19937(seed + 7))
        uniforms = (float(u) for _ in iter(int, 1) for u in rng.random(1 << 12))
        todo, action = M if kind == "sweep" else SAFE, float(m.action())
        first = True
        for l, box in m.downward():
            if not first:  # init leaves the chain at the last slice; the first step moves on from it
                action += m.site_updates(l, box, uniforms)
                todo -= 1
                if l == 0 and todo:  # the turning point visits the first slice again
                    action += m.site_updates(l, box, uniforms)
                    todo -= 1
            first, last = False, box[0]
            if not todo:
                break
        return {"field": m.phi, "greens": last.resolve_conj().numpy(), "boson_action": action}
    if kind == "hmc":
        rng = np.random.default_rng(seed + 3)
        p, u, eps = rng.standard_normal(m.phi.shape), float(rng.uniform()), 0.02
        before, start = m.phi.copy(), (p ** 2).sum() / 2
        g, action = m.gradient()
        start += action
        for k in range(case["steps"]):
            p -= (0.5 if k == 0 else 1.0) * eps * g
            m.phi = m.phi + eps * p
            g, action = m.gradient()
        p -= 0.5 * eps * g
        dh = action + (p ** 2).sum() / 2 - start
        accepted = bool(dh <= 0 or u < math.exp(-dh))
        if not accepted:
            m.phi = before
        _, box = next(m.downward())
        return {"accepted": accepted, "dh": dh, "field": m.phi, "greens": box[0].resolve_conj().numpy()}
    # the equal-time Green's function at the first slice, hopping half steps moved to both sides
    G, _ = m.greens(m.lefts()[-1], m.one())
    G = m.blocks(m.half_inv, G)
    G = m.blocks(m.half.mH, G.mH).mH
    none = [None, None]
    return {"greens": G.resolve_conj().numpy(), "etpc": none, "etcdc": none, "zfpc": none, "zfcdc": none, "zfccc": none,
            "sfdensity": None}
