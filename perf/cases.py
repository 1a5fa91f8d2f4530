"""Performance cases of the VMC particle-move engine: what its users run, over the real range.

A case is one call sequence of a QMC program through the public host layer (miniqmc_amd.qmcx) on one
of the prepared systems (NiO-8 cubic, 96 electrons, to NiO-64, 768 electrons).  Its kinds:

  sweep   a block of VMC sweeps of a walker batch (qmcx_run_sweeps), read back as a program does at a
          block's end: log|Psi| after every sweep, accept counts, walker positions
  log     new walkers: positions in, evaluateLog from scratch, G, L and log|Psi| out
  nlpp    one NonLocalPP evaluation: the twelve ratios of every electron-ion pair inside rmax
  flex    the batched stage calls of a host-driven move loop: ratio_grad and accept_restore per
          electron, then completeUpdates and evaluateGL
  ratios  virtual-move ratios of one electron (evaluateRatios)

``listed`` holds the fixed cases, ``draw`` more of the same ranges.  Metropolis acceptance is used in
double precision only: in single precision chains of different rounding part at near ties, after
which they are different (equally valid) walks.

Single-precision batches compute in float32 and hand every result out as double; a program that
keeps log|Psi|, ratios, G and L of such a batch stores them as float32, as ``run`` does.

``exact`` evaluates the same quantities from their definitions in float64 torch (direct inverses,
brute-force Jastrow sums, the walks replayed from the random streams).
"""
from __future__ import annotations

import math

import numpy as np
import torch

from miniqmc_amd import nlpp as nl
from miniqmc_amd import qmcx, systems

TAU = 0.3          # the driver's and the benchmark's time step
SIZES = {"nio8-cubic": (96, 48, 24), "nio16": (192, 96, 32), "nio32": (384, 192, 48), "nio64": (768, 384, 64)}
NPAD = {"nio8-cubic": 48, "nio16": 96, "nio32": 208, "nio64": 384}


# ---------------------------------------------------------------------------------------- the cases
def _sweep(name, system, precision, walkers, delay, rule, sweeps, recompute, jastrow="random", j3=False):
    c = {"kind": "sweep", "system": system, "precision": precision, "walkers": walkers, "delay": delay, "rule": rule,
         "sweeps": sweeps, "recompute": recompute, "jastrow": jastrow, "j3": j3}
    return {"name": name, **c} if name else c


def _other(name, kind, system, precision, walkers, delay, **more):
    c = {"kind": kind, "system": system, "precision": precision, "walkers": walkers, "delay": delay,
         "jastrow": more.pop("jastrow", "random"), "j3": more.pop("j3", False), **more}
    return {"name": name, **c} if name else c


def listed():
    return [
        # the production run: the benchmark's NiO-64 batch, FP32 form with the per-sweep FP64 refresh
        _sweep("sweep-nio64-fp32", "nio64", "fp32", 128, 32, "reference", 3, 1),
        # the medium system with more walkers than CUs
        _sweep("sweep-nio32-fp32", "nio32", "fp32", 256, 32, "reference", 3, 1),
        # an uneven batch at a delay rank that does not divide the orbitals, the reference's own functors
        _sweep("sweep-nio16-fp32-odd", "nio16", "fp32", 37, 20, "reference", 2, 1, "nio"),
        # validation runs: double precision, Sherman-Morrison updates, Metropolis walk
        _sweep("sweep-nio64-fp64-sm", "nio64", "fp64", 48, 1, "metropolis", 1, 0),
        # double precision with delayed updates
        _sweep("sweep-nio32-fp64-delayed", "nio32", "fp64", 64, 16, "reference", 1, 1),
        # the smallest program: one walker of the small cell in double precision, all latency
        _sweep("sweep-nio8-fp64-one", "nio8-cubic", "fp64", 1, 1, "metropolis", 2, 0),
        # the three-body Jastrow (the reference's -j)
        _sweep("sweep-nio32-fp32-j3", "nio32", "fp32", 96, 16, "reference", 1, 1, "nio", True),
        # start of a run, or walkers received from elsewhere
        _other("log-nio64-fp32", "log", "nio64", "fp32", 128, 32),
        # pseudopotential of the benchmark's batch
        _other("nlpp-nio64-fp32", "nlpp", "nio64", "fp32", 128, 32, rmax=1.7, max_pairs=4),
        # and in double precision on an uneven batch
        _other("nlpp-nio32-fp64", "nlpp", "nio32", "fp64", 51, 1, rmax=1.7, max_pairs=4),
        # a host program that keeps its own move loop (flex_* stage calls), 16 electrons of each spin
        _other("flex-nio32-fp32", "flex", "nio32", "fp32", 64, 16, electrons=16),
        # one electron's quadrature points of one walker: the smallest call
        _other("ratios-nio8-fp64-one", "ratios", "nio8-cubic", "fp64", 1, 1, points=12),
    ]


def draw(rng):
    def span(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    kind = rng.choice(["sweep", "sweep", "sweep", "log", "nlpp", "flex", "ratios"])
    system = rng.choice(list(SIZES))
    precision = rng.choice(["fp32", "fp32", "fp64"])
    jastrow = rng.choice(["random", "nio"])
    big = system == "nio64"
    j3 = not big and rng.random() < 0.15
    delay = rng.choice([1, 4, 8, 12, 16, 20, 24, 32])
    if kind == "sweep":
        walkers = span(1, 36 if big and precision == "fp64" else 150 if big else 220)
        rule = "reference" if precision == "fp32" else rng.choice(["reference", "metropolis"])
        if j3 and precision == "fp64" and delay > 8:
            delay = 8
        if precision == "fp32":   # the per-sweep refresh is how the FP32 form is run
            return _sweep(None, system, precision, walkers, delay, rule, rng.randint(1, 3), 1, jastrow, j3)
        return _sweep(None, system, precision, walkers, delay, rule, 1, 1 if rule == "reference" else 0, jastrow, j3)
    if kind == "log":
        return _other(None, kind, system, precision, span(1, 160 if big else 240), delay if not j3 else 8,
                      jastrow=jastrow, j3=j3)
    if kind == "nlpp":
        return _other(None, kind, system, precision, span(1, 128 if big else 200), 8 if j3 else delay,
                      jastrow=jastrow, rmax=round(rng.uniform(1.2, 1.9), 2), max_pairs=rng.randint(4, 8))
    if kind == "flex":
        return _other(None, kind, system, precision, span(1, 128), min(delay, 16), jastrow=jastrow,
                      electrons=rng.randint(4, 20))
    return _other(None, kind, system, precision, span(1, 128), min(delay, 16), jastrow=jastrow, points=12 * rng.randint(1, 4))


# ------------------------------------------------------------------------------- what a program holds
_descs, _devices = {}, {}


def _desc(case):
    """The system's description (lattice, ions, functors, orbital table): one fixed workload per name."""
    key = (case["system"], case["jastrow"], case["j3"])
    if key not in _descs:
        _descs[key] = systems.make_system(case["system"], j_mode=case["jastrow"], j3=case["j3"])
    return _descs[key]


def _precision(case):
    return qmcx.FP32 if case["precision"] == "fp32" else qmcx.FP64


def _device(case):
    """The device-resident system (orbital table uploaded once, as a program does)."""
    key = (case["system"], case["jastrow"], case["j3"], case["precision"])
    if key not in _devices:
        _devices[key] = qmcx.System(_desc(case), precisions=(_precision(case),))
    return _devices[key]


def _inputs(case, seed):
    """The numbers a pass works on, all from the seed."""
    d = _desc(case)
    rng = np.random.default_rng([seed, 77])
    n, N, W = d.nup, d.nel, case["walkers"]
    x = {"R": rng.random((W, N, 3)) @ d.lattice, "seed": seed & 0x7FFFFFFF}
    if case["kind"] == "nlpp":
        x["spheres"] = np.stack([nl.quadrature_knots() @ nl.random_rotation(u).T for u in rng.random((W, 3))])
    if case["kind"] == "flex":
        m = min(case["electrons"], n)
        x["iel"] = [int(i) for i in list(range(m)) + list(range(n, n + m))]
        x["displ"] = math.sqrt(TAU) * rng.standard_normal((2 * m, W, 3))
        x["accept"] = (rng.random((2 * m, W)) < 0.5).astype(np.int32)
    if case["kind"] == "ratios":
        x["iel"] = int(rng.integers(0, N))
        v = rng.standard_normal((W, case["points"], 3))
        v *= rng.uniform(0.3, 1.7, (W, case["points"], 1)) / np.linalg.norm(v, axis=2, keepdims=True)
        x["vpos"] = x["R"][:, x["iel"], None, :] + v
    return x


def prepare(case, seed):
    state = {"case": case, **_inputs(case, seed)}
    wb = qmcx.WalkerBatch(_device(case), case["walkers"], delay_rank=case["delay"], precision=_precision(case))
    wb.set_positions(state["R"])
    if case["kind"] != "log":
        wb.evaluate_log()
    if case["kind"] == "nlpp":   # the program's list of pair ratios: spheres of these radii do not overlap
        state["pair_list"] = np.zeros((case["walkers"] * wb.N, 12), np.float32 if case["precision"] == "fp32" else np.float64)
    state["wb"] = wb
    return state


def run(state):
    case, wb = state["case"], state["wb"]
    kept = (lambda a: a.astype(np.float32)) if case["precision"] == "fp32" else (lambda a: a)
    kind = case["kind"]
    if kind == "sweep":
        mode = qmcx.ACCEPT_REFERENCE if case["rule"] == "reference" else qmcx.ACCEPT_METROPOLIS
        hist = wb.run(case["sweeps"], state["seed"], TAU, mode, recompute_every=case["recompute"])
        return {"log": kept(hist), "accepts": wb.accepts(), "positions": wb.positions()}
    if kind == "log":
        wb.set_positions(state["R"])
        log = wb.evaluate_log()
        G, L, _ = wb.gl()
        return {"log": kept(log), "G": kept(G), "L": kept(L)}
    if kind == "nlpp":
        ratios, pairs = wb.nlpp_evaluate(case["rmax"], state["spheres"], max_pairs=case["max_pairs"])
        used = ratios[np.arange(case["max_pairs"]) < pairs[..., None]]   # [listed pairs][12]
        out = state["pair_list"]
        out[:len(used)] = used
        out[len(used):] = 0
        return {"pairs": pairs, "ratios": out}
    if kind == "flex":
        out = []
        for q, iel in enumerate(state["iel"]):
            out.append(wb.flex_ratio_grad(iel, state["displ"][q]))
            wb.flex_accept_restore(iel, state["accept"][q])
        wb.flex_complete_updates()
        log = wb.flex_evaluate_gl()
        return {"ratio": kept(np.stack([o[0] for o in out])), "grad_now": kept(np.stack([o[1] for o in out])),
                "grad_new": kept(np.stack([o[2] for o in out])), "log": kept(log)}
    return {"ratios": kept(wb.flex_evaluate_ratios(state["iel"], state["vpos"]))}


# ------------------------------------------------------------------------------------ work of a pass
def work(case):
    """Bytes: the orbital table's rows that are needed (each once), the walker state in and out once, the
    results.  Flops: spline sums, dot products, radial functors, rank-1 inverse updates, inversions."""
    N, n, g = SIZES[case["system"]]
    W, npad = case["walkers"], NPAD[case["system"]]
    es = 4 if case["precision"] == "fp32" else 8
    table = (g + 3) ** 3 * npad * es

    def spline(points):
        return min(table, points * 64 * npad * es)

    kind = case["kind"]
    mats = W * 2 * n * n
    inversion = 2.0 * n ** 3 * W * 2
    if kind == "sweep":
        moves = W * N * case["sweeps"]
        flops = moves * (64 * 2 * 3 * n + 16.0 * n + 60.0 * N) + 0.5 * moves * 4.0 * n * n
        if case["recompute"]:
            flops += inversion * case["sweeps"]
        return {"bytes": spline(moves) + 2 * mats * es + W * N * 24 * 2, "flops": flops}
    if kind == "log":
        return {"bytes": spline(W * N) + 6 * mats * es + W * N * (24 + 32),
                "flops": W * N * (64 * 2 * 3 * n + 8.0 * n + 60.0 * N) + inversion}
    if kind == "nlpp":
        d = _desc(case)
        sphere = 4.0 / 3.0 * math.pi * case["rmax"] ** 3
        pairs = W * N * d.nions * sphere / abs(float(np.linalg.det(d.lattice)))
        points = 12.0 * pairs
        return {"bytes": spline(points) + mats * es + points * 8, "flops": points * (64 * 2 * n + 2 * n + 20.0 * N)}
    if kind == "flex":
        moves = W * 2 * min(case["electrons"], n)
        return {"bytes": spline(moves) + (mats * 5 + moves * 8 * n) * es,
                "flops": moves * (64 * 2 * 3 * n + 16.0 * n + 60.0 * N + 2.0 * n * n) + W * N * 8.0 * n}
    points = W * case["points"]
    return {"bytes": spline(points) + W * n * es + points * 32, "flops": points * (64 * 2 * n + 2 * n + 20.0 * N)}


# ---------------------------------------------------------------------------- the same in 64 bits
def _philox(counter, k0, k1):
    """Philox4x64-10 (Salmon et al., SC'11) of the four uint64 arrays `counter`."""
    m = [np.uint64(0xD2E7470EE14C6C93), np.uint64(0xCA5A826395121157)]
    bump = [np.uint64(0x9E3779B97F4A7C15), np.uint64(0xBB67AE8584CAA73B)]
    low, half = np.uint64(0xFFFFFFFF), np.uint64(32)

    def wide(a, b):
        al, ah, bl, bh = a & low, a >> half, b & low, b >> half
        t = ah * bl + ((al * bl) >> half)
        return ah * bh + (t >> half) + (((t & low) + al * bh) >> half), a * b

    c = list(counter)
    k = [np.uint64(k0), np.uint64(k1)]
    with np.errstate(over="ignore"):
        for r in range(10):
            if r:
                k = [k[0] + bump[0], k[1] + bump[1]]
            (h0, l0), (h1, l1) = wide(c[0], m[0]), wide(c[2], m[1])
            c = [h1 ^ c[1] ^ k[0], l1, h0 ^ c[3] ^ k[1], l0]
    return c


def _randoms(seed, sweep, W, N):
    """Displacements [W][N][3] and acceptance uniforms [W][N] of one sweep's random streams."""
    w, e = np.meshgrid(np.arange(W, dtype=np.uint64), np.arange(N, dtype=np.uint64), indexing="ij")
    s = np.full_like(w, sweep)

    def unit(x):
        return (x >> np.uint64(11)).astype(np.float64) / 9007199254740992.0

    a = [unit(x) for x in _philox([e, s, w, np.zeros_like(w)], seed, 0x51A7)]
    u = unit(_philox([e, s, w, np.ones_like(w)], seed, 0x51A7)[0])
    r0, r1 = np.sqrt(-2 * np.log(1 - a[0])), np.sqrt(-2 * np.log(1 - a[2]))
    z = np.stack([r0 * np.cos(2 * np.pi * a[1]), r0 * np.sin(2 * np.pi * a[1]), r1 * np.cos(2 * np.pi * a[3])], axis=-1)
    return math.sqrt(TAU) * z, u


class _Exact:
    """The wave function in float64 torch, from the system's description."""

    def __init__(self, d):
        self.dev = dev = "cuda" if torch.cuda.is_available() else "cpu"
        f = lambda a: torch.as_tensor(np.asarray(a, dtype=np.float64), device=dev)  # noqa: E731
        self.d, self.n, self.N = d, d.nup, d.nel
        self.lat, self.inv = f(d.lattice), f(np.linalg.inv(d.lattice))
        self.spo_inv = f(np.linalg.inv(d.spo_lattice))
        self.ions = f(d.ion_pos)
        self.species = torch.as_tensor(np.asarray(d.ion_species), device=dev).long()
        self.rows = torch.as_tensor(d.coefs, device=dev).reshape(-1, d.npad)
        self.f = f

    # cubic B-spline basis and derivatives at the fraction t: [..., 4]
    @staticmethod
    def basis(t):
        w = torch.stack([(1 - t) ** 3, 3 * t ** 3 - 6 * t ** 2 + 4, -3 * t ** 3 + 3 * t ** 2 + 3 * t + 1, t ** 3], -1) / 6
        dw = torch.stack([-(1 - t) ** 2 / 2, 1.5 * t ** 2 - 2 * t, -1.5 * t ** 2 + t + 0.5, t ** 2 / 2], -1)
        return w, dw, torch.stack([1 - t, 3 * t - 2, 1 - 3 * t, t], -1)

    def spo(self, r, derivs=False):
        """Orbital values [P][n], or with derivs [P][5][n]: value, unit-cell gradient, h_xx."""
        ng = self.d.ng
        u = r @ self.spo_inv
        u = (u - torch.floor(u)) * self.f(ng)
        i = torch.minimum(torch.floor(u), self.f(ng) - 1)
        t, i = u - i, i.long()
        a, da, d2a = self.basis(t)
        o = torch.arange(4, device=self.dev)
        idx = ((i[:, 0, None, None, None] + o[:, None, None]) * (ng[1] + 3) + i[:, 1, None, None, None] + o[:, None]) * (ng[2] + 3) \
            + i[:, 2, None, None, None] + o
        sets = [(a, a, a)]
        scale = [1.0]
        if derivs:
            sets += [(da, a, a), (a, da, a), (a, a, da), (d2a, a, a)]
            scale += [ng[0], ng[1], ng[2], ng[0] * ng[0]]
        out = torch.empty((len(r), len(sets), self.n), dtype=torch.float64, device=self.dev)
        step = max(1, (1 << 25) // (64 * self.n))
        for p in range(0, len(r), step):
            q = slice(p, p + step)
            c = self.rows[idx[q].reshape(-1)][:, :self.n].double().reshape(-1, 64, self.n)
            w = torch.stack([s * torch.einsum("pi,pj,pk->pijk", x[0][q, 0], x[1][q, 1], x[2][q, 2]).reshape(-1, 64)
                             for x, s in zip(sets, scale)], 1)
            out[q] = torch.bmm(w.contiguous(), c.contiguous())
        return out if derivs else out[:, 0]

    def image(self, d):
        """Minimum image of displacements d[..., 3]: the cells are orthogonal, so rounding finds it."""
        return d - torch.round(d @ self.inv) @ self.lat

    def functor(self, F, r):
        """u, u', u'' of a radial functor (zero from its cutoff on)."""
        dr = F.rcut / (F.nparams + 1)
        p = np.asarray(F.params, dtype=np.float64)
        c = np.zeros(F.nparams + 5)
        c[0], c[1:F.nparams + 1] = p[1] - 2 * dr * F.cusp, p
        c = self.f(c)
        x = torch.clamp(r / dr, max=F.nparams + 0.999999)
        i = torch.floor(x).long()
        w = self.basis(x - i)
        cs = c[i[..., None] + torch.arange(4, device=self.dev)]
        inside = r < F.rcut
        return [torch.where(inside, (b * cs).sum(-1) / dr ** k, torch.zeros_like(r)) for k, b in enumerate(w)]

    def j1(self, r):
        """sum u, sum u'/r (R_I - r), -(sum u'' + 2 u'/r) over the ions at points r[..., 3]."""
        out = None
        for s, F in enumerate(self.d.j1):
            out = self._radial(F, self.image(self.ions[self.species == s] - r[..., None, :]), None, out)
        return out

    def j2(self, r, iel, R):
        """The same over the other electrons R[..., N, 3] for electrons iel[...] (index tensor) at r."""
        out = None
        other = torch.arange(self.N, device=self.dev)
        disp = self.image(R - r[..., None, :])
        same = (other < self.n) == (iel[..., None] < self.n)
        for F, mask in ((self.d.j2[0], same), (self.d.j2[1], ~same)):
            out = self._radial(F, disp, mask & (other != iel[..., None]), out)
        return out

    def _radial(self, F, disp, mask, out):
        r = torch.sqrt((disp ** 2).sum(-1))
        u, du, d2u = self.functor(F, r)
        g = torch.where(r > 0, du / r, torch.zeros_like(r))
        if mask is not None:
            u, g, d2u = [torch.where(mask, x, torch.zeros_like(x)) for x in (u, g, d2u)]
        new = [u.sum(-1), (g[..., None] * disp).sum(-2), -(d2u + 2 * g).sum(-1)]
        return new if out is None else [a + b for a, b in zip(out, new)]

    def jastrow(self, R):
        """J1 and J2 of every electron of R[W][N][3]: U [W][N] each, gradient and Laplacian sums."""
        o1 = self.j1(R)
        iel = torch.arange(self.N, device=self.dev)
        o2 = [self.j2(R[w], iel, R[w][None]) for w in range(len(R))]
        o2 = [torch.stack(x) for x in zip(*o2)]
        return o1, o2

    def state(self, R, gl=False):
        """log|Psi| [W] of positions R[W][N][3] (and G [W][N][3], L [W][N])."""
        W, n = len(R), self.n
        o1, o2 = self.jastrow(R)
        log = torch.empty(W, dtype=torch.float64, device=self.dev)
        G, L = torch.empty_like(R), torch.empty_like(R[..., 0])
        for w in range(W):
            p = self.spo(R[w], gl)
            for det in range(2):
                rows = slice(det * n, det * n + n)
                A = p[rows, 0] if gl else p[rows]
                ld = torch.linalg.slogdet(A)[1]
                log[w] = ld if det == 0 else log[w] + ld
                if gl:
                    inv = torch.linalg.inv(A).T
                    g = [(p[rows, k] * inv).sum(1) for k in (1, 2, 3)]
                    G[w, rows] = torch.stack(g, -1)
                    L[w, rows] = (p[rows, 4] * inv).sum(1) - sum(x * x for x in g)
        log += -o1[0].sum(1) - 0.5 * o2[0].sum(1)
        return (log, G + o1[1] + o2[1], L + o1[2] + o2[2]) if gl else log

    def inverses(self, R):
        """(A^-1)^T of both determinants, [W][2][n][n]."""
        M = torch.empty((len(R), 2, self.n, self.n), dtype=torch.float64, device=self.dev)
        for w in range(len(R)):
            p = self.spo(R[w])
            for det in range(2):
                M[w, det] = torch.linalg.inv(p[det * self.n:(det + 1) * self.n]).T
        return M

    def move(self, R, M, iel, new, derivs=False):
        """Ratio of moving electron iel of every walker to new[W][3] (and the orbitals there)."""
        det, row = divmod(iel, self.n)
        e = torch.full((len(R),), iel, device=self.dev)
        p = self.spo(new, True) if derivs else self.spo(new)[:, None]
        rdet = (p[:, 0] * M[:, det, row]).sum(1)
        old1, old2 = self.j1(R[:, iel]), self.j2(R[:, iel], e, R)
        new1, new2 = self.j1(new), self.j2(new, e, R)
        ratio = rdet * torch.exp(old1[0] - new1[0] + old2[0] - new2[0])
        return p, rdet, ratio, (old1[1] + old2[1], new1[1] + new2[1])

    def accept(self, R, M, iel, new, p, rdet, yes):
        det, row = divmod(iel, self.n)
        t = torch.bmm(M[:, det], p[:, 0, :, None].contiguous())[..., 0]
        t[:, row] -= 1
        t = torch.where(yes, 1 / rdet, torch.zeros_like(rdet))[:, None] * t
        M[:, det] -= t[:, :, None] * M[:, det, row].clone()[:, None, :]
        R[:, iel] = torch.where(yes[:, None], new, R[:, iel])


def exact(case, seed):
    if case["j3"] and case["kind"] != "sweep":
        return None
    x, E = _inputs(case, seed), _Exact(_desc(case))
    R = E.f(x["R"])
    W, N, n = case["walkers"], E.N, E.n
    as_np = lambda t: t.cpu().numpy()  # noqa: E731
    kind = case["kind"]
    if kind == "sweep":
        hist, count = [], np.zeros(W, dtype=np.int64)
        M = E.inverses(R) if case["rule"] == "metropolis" and not case["j3"] else None
        if case["rule"] == "metropolis" and M is None:
            return None
        for s in range(case["sweeps"]):
            step, u = _randoms(x["seed"], s, W, N)
            if M is None:   # acceptance does not depend on the wave function
                yes = u < 0.5
                R = R + E.f(step * yes[..., None])
                count += yes.sum(1)
            else:
                step, u = E.f(step), E.f(u)
                for iel in range(N):
                    new = R[:, iel] + step[:, iel]
                    p, rdet, ratio, _ = E.move(R, M, iel, new)
                    yes = u[:, iel] < ratio * ratio
                    E.accept(R, M, iel, new, p, rdet, yes)
                    count += as_np(yes)
            if not case["j3"]:
                hist.append(as_np(E.state(R)))
        return {"log": np.stack(hist) if hist else None, "accepts": count, "positions": as_np(R)}
    if kind == "log":
        log, G, L = E.state(R, gl=True)
        return {"log": as_np(log), "G": as_np(G), "L": as_np(L)}
    M = E.inverses(R)
    if kind == "nlpp":
        sph = E.f(x["spheres"])
        counts, out, at = np.zeros((W, N), dtype=np.int32), np.zeros((W * N, 12)), 0
        iel = torch.arange(N, device=E.dev)
        for w in range(W):
            disp = E.image(E.ions - R[w][:, None, :])
            dist = torch.sqrt((disp ** 2).sum(-1))
            near = dist < case["rmax"]
            counts[w] = as_np(near.sum(1))
            e, ion = torch.nonzero(near, as_tuple=True)
            pts = dist[e, ion][:, None, None] * sph[w] + disp[e, ion][:, None, :] + R[w][e][:, None, :]
            if not len(e):
                continue
            ek = e.repeat_interleave(12)
            pts = pts.reshape(-1, 3)
            det = (E.spo(pts) * M[w].reshape(N, n)[ek]).sum(1)
            old = E.j1(R[w])[0] + E.j2(R[w], iel, R[w][None])[0]
            new = E.j1(pts)[0] + E.j2(pts, ek, R[w][None])[0]
            out[at:at + len(e)] = as_np((det * torch.exp(old[ek] - new)).reshape(-1, 12))
            at += len(e)
        return {"pairs": counts, "ratios": out}
    if kind == "flex":
        got = [[], [], []]
        for q, iel in enumerate(x["iel"]):
            det, row = divmod(iel, n)
            here = (E.spo(R[:, iel], True)[:, 1:4] * M[:, det, row, None]).sum(2)
            new = R[:, iel] + E.f(x["displ"][q])
            p, rdet, ratio, (j_old, j_new) = E.move(R, M, iel, new, True)
            got[0].append(as_np(ratio))
            got[1].append(as_np(here + j_old))
            got[2].append(as_np((p[:, 1:4] * M[:, det, row, None]).sum(2) / rdet[:, None] + j_new))
            E.accept(R, M, iel, new, p, rdet, torch.as_tensor(x["accept"][q] != 0, device=E.dev))
        return {"ratio": np.stack(got[0]), "grad_now": np.stack(got[1]), "grad_new": np.stack(got[2]), "log": as_np(E.state(R))}
    det, row = divmod(x["iel"], n)
    pts = E.f(x["vpos"])
    out = torch.empty(pts.shape[:2], dtype=torch.float64, device=E.dev)
    e = torch.full((1,), x["iel"], device=E.dev)
    for w in range(W):
        d = (E.spo(pts[w]) * M[w, det, row]).sum(1)
        old = E.j1(R[w, x["iel"]][None])[0] + E.j2(R[w, x["iel"]][None], e, R[w][None])[0]
        new = E.j1(pts[w])[0] + E.j2(pts[w], e.expand(len(pts[w])), R[w][None])[0]
        out[w] = d * torch.exp(old - new)
    return {"ratios": as_np(out)}
