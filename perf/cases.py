"""The work that a user of this framework has it do, as cases that can be timed.

Chebyshev moments of tight-binding Hamiltonians and what is read off them: the
density of states (`spectral_moments`, by the direct and by the doubling
recursion, and many jobs at once through `Batch`), conductivities
(`kubo_fft`, `correlation_expansion_moments`), time-dependent correlations,
the non-orthogonal basis, and the energy-grid tools that turn moments into
curves.  Every call goes through the package's public functions with the
states resident on the GPU, as `DeviceStates` keeps them; moments and curves
come back as host arrays, as the functions return them.

Lattices are the repository's own kinds (square and cubic Anderson models,
Haldane and Kane-Mele honeycombs) with periodic boundaries and open choices of
every side, generated here from a seed: on-site disorder always, and with
``bonds`` disorder on every hopping too, which leaves the operator with as
many values as entries.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import linqt_amd as lq
from linqt_amd._lib import LQ_LIN_BASTIN
from linqt_amd.io import CSR

# ---- the cases -----------------------------------------------------------------
# kind: which public call is made.  lattice, lx, ly, lz: the system.  M: moments,
# R: random-phase states.


def listed():
    return [
        # The smallest solve: one state on a system of a thousand sites, as a
        # script does while it is written or for one point of a disorder sweep.
        dict(name="dos_small", kind="dos", lattice="square", lx=33, ly=31, lz=1, bonds=False, M=128, R=1, algo="direct"),
        # The density of states that the benchmark quotes: 256 x 256, M = 1024, R = 8.
        dict(name="dos_square", kind="dos", lattice="square", lx=256, ly=256, lz=1, bonds=False, M=1024, R=8,
             algo="direct"),
        # A large three-dimensional system with random hoppings, odd sides and an
        # odd number of states: memory-bound, the operator's values in full.
        dict(name="dos_bonds", kind="dos", lattice="cubic", lx=81, ly=79, lz=77, bonds=True, M=256, R=5, algo="direct"),
        # Twice the moments for each step by the doubling recursion, on a spinful system.
        dict(name="dos_doubling", kind="dos", lattice="kane_mele", lx=127, ly=129, lz=1, bonds=False, M=1024, R=4,
             algo="doubling"),
        # The headline: both components of the Kubo-Bastin conductivity at 512 x 512 cells.
        dict(name="kubo_bastin", kind="kubo", lx=512, ly=512, M=512, nump=2048, R=4, formula="bastin", comps=2,
             precision="fp64"),
        # An ordinary Kubo-Greenwood solve of ragged sizes: a parameter sweep's step.
        dict(name="kubo_greenwood", kind="kubo", lx=95, ly=95, M=300, nump=640, R=3, formula="greenwood", comps=1,
             precision="fp64"),
        # A small table of two-operator moments, kept in a file for the tools.
        dict(name="corr_small", kind="corr", lx=64, ly=64, M0=100, M1=100, R=1, comps=1, precision="fp64"),
        # The split-precision form of the table, two operators.
        dict(name="corr_int8", kind="corr", lx=181, ly=181, M0=256, M1=256, R=2, comps=2, precision="int8x7"),
        # Time-dependent correlations: states evolved and expanded at each time step.
        dict(name="time_corr", kind="time", lattice="honeycomb", lx=128, ly=130, M=128, nT=8, R=2, dt=2.0),
        # A non-orthogonal basis: an overlap solve for each moment.
        dict(name="nonorth", kind="nonorth", lx=90, ly=91, M=48, R=1),
        # A moment table read, damped and turned into curves by the tools, and a
        # finished Kubo solve into a conductivity.
        dict(name="tools", kind="tools", M=512, nump=2048, broad=20.0),
        # Jobs of uneven size advanced together, as the serving loop does.
        dict(name="batch", kind="batch", jobs=12, nmax=180000, M=512, mix=3),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dos", "dos", "dos", "kubo", "kubo", "corr", "time", "nonorth", "tools", "batch"])
    if kind == "dos":
        lattice = rng.choice(["square", "cubic", "kane_mele", "honeycomb"])
        n = _log(rng, 600, 600000)
        lx, ly, lz = _sides(rng, lattice, n)
        n = _size(lattice, lx, ly, lz)
        R = rng.choice([1, 1, 2, 3, 4, 5, 8, 12, 16])
        M = max(32, min(_log(rng, 64, 2048), int(2.5e9 / (n * R))))
        return dict(kind="dos", lattice=lattice, lx=lx, ly=ly, lz=lz, bonds=rng.random() < 0.3, M=M, R=R,
                    algo=rng.choice(["direct", "direct", "doubling"]))
    if kind in ("kubo", "corr"):
        n = _log(rng, 2000, 400000)
        lx, ly, _ = _sides(rng, "honeycomb", n)
        n = _size("honeycomb", lx, ly, 1)
        R = rng.choice([1, 1, 2, 3, 4])
        comps = rng.choice([1, 2])
        precision = rng.choice(["fp64", "fp64", "fp64", "int8x7"])
        most = 4.0e11 if precision == "fp64" else 1.5e11
        M = max(32, min(_log(rng, 48, 1024), int(math.sqrt(most / (n * R * comps)))))
        if kind == "corr":
            return dict(kind="corr", lx=lx, ly=ly, M0=M, M1=max(24, M - rng.choice([0, 0, 1, 20])), R=R, comps=comps,
                        precision=precision)
        return dict(kind="kubo", lx=lx, ly=ly, M=M, nump=M * rng.choice([1, 2, 4]) + rng.choice([0, 0, 2, 10]), R=R,
                    formula=rng.choice(["bastin", "bastin", "greenwood"]), comps=comps, precision=precision)
    if kind == "time":
        n = _log(rng, 2000, 200000)
        lx, ly, _ = _sides(rng, "honeycomb", n)
        n = _size("honeycomb", lx, ly, 1)
        R = rng.choice([1, 2, 3, 4])
        nT = rng.choice([4, 5, 8, 16])
        M = max(32, min(_log(rng, 32, 512), int(6e8 / (n * R * nT))))
        return dict(kind="time", lattice="honeycomb", lx=lx, ly=ly, M=M, nT=nT, R=R, dt=rng.choice([0.5, 1.0, 2.0, 5.0]))
    if kind == "nonorth":
        n = _log(rng, 1000, 200000)
        lx, ly, _ = _sides(rng, "honeycomb", n)
        return dict(kind="nonorth", lx=lx, ly=ly, M=_log(rng, 16, 80), R=rng.choice([1, 1, 2]))
    if kind == "tools":
        return dict(kind="tools", M=_log(rng, 64, 768), nump=_log(rng, 500, 4000), broad=rng.choice([5.0, 10.0, 20.0]))
    return dict(kind="batch", jobs=rng.randint(3, 16), nmax=_log(rng, 20000, 250000), M=_log(rng, 128, 512),
                mix=rng.randint(4, 1 << 20))


# ---- lattices ------------------------------------------------------------------
_ORBITALS = {"square": 1, "cubic": 1, "honeycomb": 2, "kane_mele": 4}


def _size(lattice, lx, ly, lz=1):
    return _ORBITALS[lattice] * lx * ly * lz


def _sides(rng, lattice, n):
    cells = max(27, n // _ORBITALS[lattice])
    if lattice == "cubic":
        s = max(3, round(cells ** (1 / 3)))
        return s + rng.choice([0, 1]), s, s + rng.choice([0, 0, 1])
    s = max(4, round(cells ** 0.5))
    return s + rng.choice([0, 1, 3]), s, 1


def _bonds(lattice, lx, ly, lz):
    """The forward bonds: (row, column, value, displacement) arrays; each bond's
    reverse is its conjugate.  Site index: orbitals fastest, then x, y, z."""
    cells = np.arange(lx * ly * lz)
    x, y, z = cells % lx, cells // lx % ly, cells // (lx * ly)
    norb = _ORBITALS[lattice]

    def at(dx, dy, dz, o):
        return norb * ((x + dx) % lx + lx * ((y + dy) % ly + ly * ((z + dz) % lz))) + o

    a1, a2 = np.array([1.0, 0.0]), np.array([0.5, math.sqrt(3.0) / 2.0])
    dab = (a1 + a2) / 3.0
    out = []
    if lattice in ("square", "cubic"):
        for d in ((1, 0, 0), (0, 1, 0), (0, 0, 1))[: 2 if lattice == "square" else 3]:
            out.append((at(0, 0, 0, 0), at(*d, 0), -1.0, (float(d[0]), float(d[1]))))
        return out
    first = [((0, 0), dab), ((-1, 0), dab - a1), ((0, -1), dab - a2)]
    second = [((1, 0), a1), ((-1, 1), a2 - a1), ((0, -1), -a2)]
    if lattice == "honeycomb":  # Haldane: second neighbours t2 e^{+-i pi/2}
        for (dx, dy), d in first:
            out.append((at(0, 0, 0, 0), at(dx, dy, 0, 1), -1.0, tuple(d)))
        for (dx, dy), d in second:
            for s, sign in ((0, 1.0), (1, -1.0)):
                out.append((at(0, 0, 0, s), at(dx, dy, 0, s), 0.1j * sign, tuple(d)))
        return out
    for (dx, dy), d in first:  # Kane-Mele: two sites x two spins, Rashba and intrinsic coupling
        ux, uy = d / np.linalg.norm(d)
        rashba = 0.05j * np.array([[0.0, uy + 1j * ux], [uy - 1j * ux, 0.0]])
        for sa in (0, 1):
            for sb in (0, 1):
                v = (-1.0 if sa == sb else 0.0) + rashba[sa, sb]
                out.append((at(0, 0, 0, sa), at(dx, dy, 0, 2 + sb), v, tuple(d)))
    for (dx, dy), d in second:
        for s, nu in ((0, 1.0), (1, -1.0)):
            for sg, sz in ((0, 1.0), (1, -1.0)):
                o = 2 * s + sg
                out.append((at(0, 0, 0, o), at(dx, dy, 0, o), 0.06j * nu * sz, tuple(d)))
    return out


class _Ell:
    """A Hermitian operator as equally long rows: columns and values [n][w], the
    diagonal (if any) among them."""

    def __init__(self, n, cols, vals):
        order = np.argsort(cols, axis=1, kind="stable")
        self.n = n
        self.cols = np.take_along_axis(cols, order, 1)
        self.vals = np.take_along_axis(vals, order, 1)

    def csr(self, upper=True):
        keep = self.cols >= np.arange(self.n)[:, None] if upper else np.ones(self.cols.shape, bool)
        rowptr = np.concatenate([[0], np.cumsum(keep.sum(1))])
        return CSR(self.n, rowptr.astype(np.int32), self.cols[keep].astype(np.int32), self.vals[keep])

    def on(self, device):
        """Columns and values [w][n] as torch tensors."""
        return (torch.as_tensor(np.ascontiguousarray(self.cols.T), device=device),
                torch.as_tensor(np.ascontiguousarray(self.vals.T), device=device).to(torch.complex128))


def _apply(a, x):
    cols, vals = a
    y = vals[0][:, None] * x[cols[0]]
    for j in range(1, cols.shape[0]):
        y.addcmul_(vals[j][:, None].expand_as(x), x[cols[j]])
    return y


def _half_width(lattice, disorder):
    return {"square": 4.0, "cubic": 6.0, "honeycomb": 3.7, "kane_mele": 3.6}[lattice] + disorder / 2 + 0.1


def _system(lattice, lx, ly, lz, bonds, rng, want=()):
    """(Hamiltonian, half width, {"x": V_x, "y": V_y}) with on-site disorder U[-1/2, 1/2]."""
    n = _size(lattice, lx, ly, lz)
    fwd = _bonds(lattice, lx, ly, lz)
    rows, cols, vals, disp = [], [], [], []
    for i, j, v, d in fwd:
        v = np.full(i.shape, v, dtype=np.complex128)
        if bonds:
            v = v * (1.0 + 0.3 * (rng.random(i.shape[0]) - 0.5))
        rows += [i, j]
        cols += [j, i]
        vals += [v, v.conj()]
        disp += [np.broadcast_to(d, (i.shape[0], 2)), np.broadcast_to((-d[0], -d[1]), (i.shape[0], 2))]
    rows, cols, vals, disp = np.concatenate(rows), np.concatenate(cols), np.concatenate(vals), np.concatenate(disp)
    order = np.argsort(rows, kind="stable")
    w = rows.shape[0] // n
    assert w * n == rows.shape[0], "rows of one length"
    cols, vals, disp = cols[order].reshape(n, w), vals[order].reshape(n, w), disp[order].reshape(n, w, 2)
    eps = (rng.random(n) - 0.5).astype(np.complex128)
    H = _Ell(n, np.concatenate([np.arange(n)[:, None], cols], 1), np.concatenate([eps[:, None], vals], 1))
    V = {c: _Ell(n, cols, 1j * disp[:, :, k] * vals) for k, c in ((0, "x"), (1, "y")) if c in want}
    return H, _half_width(lattice, 1.0) * (1.3 if bonds else 1.0), V


def _states(n, R, rng):
    return np.exp(2j * np.pi * rng.random((R, n))) / np.sqrt(n)


def _rng(seed):
    return np.random.Generator(np.random.PCG64(int(seed) & 0x7FFFFFFF))


_PRECISION = {"fp64": lq.LQ_PREC_FP64, "int8x7": lq.LQ_PREC_INT8X7}
_CTX = None


def _ctx():
    # one context for the process, as a program has: its scratch serves every solve
    global _CTX
    if _CTX is None:
        _CTX = lq.Context(0)
    return _CTX


# ---- inputs --------------------------------------------------------------------
def _inputs(case, seed):
    """The case's host inputs: operators as rows, states, tables."""
    rng = _rng(seed)
    kind = case["kind"]
    if kind == "dos":
        H, hw, _ = _system(case["lattice"], case["lx"], case["ly"], case["lz"], case["bonds"], rng)
        return dict(H=H, hw=hw, phi=_states(H.n, case["R"], rng))
    if kind in ("kubo", "corr"):
        H, hw, V = _system("honeycomb", case["lx"], case["ly"], 1, False, rng, "xy" if case["comps"] == 2 else "x")
        return dict(H=H, hw=hw, V=V, phi=_states(H.n, case["R"], rng))
    if kind == "time":
        H, hw, V = _system(case["lattice"], case["lx"], case["ly"], 1, False, rng, "x")
        return dict(H=H, hw=hw, V=V, phi=_states(H.n, case["R"], rng))
    if kind == "nonorth":
        H, hw, _ = _system("honeycomb", case["lx"], case["ly"], 1, False, rng)
        # overlap 1 on site, about 0.08 between first neighbours
        near = np.abs(H.vals) > 0.5
        near &= H.cols != np.arange(H.n)[:, None]
        lo = np.minimum(H.cols, np.arange(H.n)[:, None])
        s = 0.08 + 0.02 * np.cos(0.37 * lo + 0.11 * np.maximum(H.cols, np.arange(H.n)[:, None]))
        own = H.cols == np.arange(H.n)[:, None]
        S = _Ell(H.n, H.cols, np.where(own, 1.0, np.where(near, s, 0.0)).astype(np.complex128))
        return dict(H=H, hw=1.4 * hw, S=S, phi=_states(H.n, case["R"], rng))
    if kind == "tools":
        M, nump = case["M"], case["nump"]
        # a table as a solve leaves it: sum over levels of T_m(x) T_n(y) w, Hermitian, 1/2 on the first row and column
        J = 96
        tx, ty = np.arccos(rng.uniform(-0.93, 0.93, J)), np.arccos(rng.uniform(-0.93, 0.93, J))
        w = (rng.standard_normal(J) + 1j * rng.standard_normal(J)) / J
        m = np.arange(M)[:, None]
        t = (np.cos(m * tx) * w) @ np.cos(m * ty).T
        mu = 2.0 * (t + t.conj().T)
        mu[0] *= 0.5
        mu[:, 0] *= 0.5
        one = np.cos(np.arange(M)[:, None] * tx) @ np.abs(w)
        one[1:] *= 2.0
        k = np.arange(nump)
        th = np.pi * (2 * k + 0.5) / nump
        p = (np.sin(th) ** 4 * np.cos(3 * th + rng.uniform(0, 1))).astype(np.complex128)
        q = 1j * np.sin(th) ** 3 * np.cos(2 * th + rng.uniform(0, 1))
        return dict(mu=mu, one=one.astype(np.complex128), fd=np.concatenate([p, q]), n=524288, W=9.2, Ec=0.0)
    jobs = []
    mix = _rng(case["mix"])  # the sizes are the case's, the disorder and states the seed's
    for j in range(case["jobs"]):
        lattice = ["cubic", "kane_mele"][int(mix.integers(2))]
        n = int(math.exp(mix.uniform(math.log(4096), math.log(case["nmax"]))))
        cells = n // _ORBITALS[lattice]
        if lattice == "cubic":
            s = max(4, round(cells ** (1 / 3)))
            lx, ly, lz = s, s, s + int(mix.integers(2))
        else:
            s = max(4, round(cells ** 0.5))
            lx, ly, lz = s, s + int(mix.integers(2)), 1
        M = max(64, int(case["M"] * mix.uniform(0.5, 1.0)))
        R = [1, 2, 4, 8][int(mix.integers(4))]
        jobs.append((lattice, lx, ly, lz, M, R))
    got = []
    for lattice, lx, ly, lz, M, R in jobs:
        H, hw, _ = _system(lattice, lx, ly, lz, False, rng)
        got.append(dict(H=H, hw=hw, phi=_states(H.n, R, rng), M=M))
    return dict(jobs=got)


def prepare(case, seed):
    d = _inputs(case, seed)
    ctx = _ctx()
    s = dict(case=case, ctx=ctx)
    if case["kind"] == "tools":
        return dict(s, **d)

    def hamiltonian(h, hw):
        return lq.SparseMatrix.from_csr(ctx, h.csr()).Rescale(1.0 / hw, 0.0)

    if case["kind"] == "batch":
        s["batch"] = lq.Batch(ctx)
        s["jobs"] = [(hamiltonian(j["H"], j["hw"]), lq.DeviceStates(ctx, j["phi"]), j["M"]) for j in d["jobs"]]
        return s
    s["H"] = hamiltonian(d["H"], d["hw"])
    s["hw"] = d["hw"]
    s["phi"] = lq.DeviceStates(ctx, d["phi"])
    if "V" in d:
        s["V"] = [lq.SparseMatrix.from_csr(ctx, d["V"][c].csr()) for c in sorted(d["V"])]
    if "S" in d:
        s["S"] = lq.SparseMatrix.from_csr(ctx, d["S"].csr(upper=False), fill=lq.LQ_FILL_GENERAL)
    return s


# ---- one pass ------------------------------------------------------------------
def run(state):
    case, ctx = state["case"], state["ctx"]
    kind = case["kind"]
    if kind == "dos":
        algo = lq.LQ_ALGO_DOUBLING if case["algo"] == "doubling" else lq.LQ_ALGO_DIRECT
        return lq.spectral_moments(state["H"], None, state["phi"], case["M"], algo)
    if kind == "kubo":
        formula = lq.LQ_KUBO_BASTIN if case["formula"] == "bastin" else lq.LQ_KUBO_GREENWOOD
        return lq.kubo_fft(state["H"], state["V"][0], state["V"], state["phi"], case["M"], case["nump"], formula,
                           precision=_PRECISION[case["precision"]])
    if kind == "corr":
        return lq.correlation_expansion_moments(state["H"], state["V"][0], state["V"], state["phi"], case["M0"],
                                                case["M1"], precision=_PRECISION[case["precision"]])
    if kind == "time":
        return lq.time_correlations(state["H"], state["V"][0], state["V"][0], state["phi"], case["M"], case["nT"],
                                    case["dt"], 2.0 * state["hw"], 0.0)
    if kind == "nonorth":
        return lq.spectral_moments_nonorth(state["H"], None, state["S"], state["phi"], case["M"])
    if kind == "batch":
        b = state["batch"]
        ids = [b.submit(H, phi, M) for H, phi, M in state["jobs"]]
        b.run()
        return [b.result(j) for j in ids]
    mu, n, W, Ec = state["mu"], state["n"], state["W"], state["Ec"]
    broad = case["broad"]
    one = lq.jackson_1d(ctx, state["one"], W, broad)
    two = lq.jackson_2d(ctx, mu, W, broad, broad)
    top = max(two.shape)
    E, rho = lq.dos_fftgrid(ctx, one, n, W, Ec, 2 * top)
    Eg, sg = lq.greenwood_fftgrid(ctx, two, n, W, Ec, top)
    Eb, sb = lq.bastin_fftgrid(ctx, two, n, W, Ec, top)
    El, sl = lq.linear_grid(ctx, LQ_LIN_BASTIN, two, n, W, Ec)  # 30 energies for each moment
    Ek, sk, gk = lq.kubo_post(ctx, lq.LQ_KUBO_BASTIN, state["fd"], n, W, Ec)
    return dict(one=one, two=two, E=E, rho=rho, Eg=Eg, sg=sg, Eb=Eb, sb=sb, El=El, sl=sl, Ek=Ek, sk=sk, gk=gk)


# ---- what a pass cannot do without -----------------------------------------------
_ROW = {"square": 5, "cubic": 7, "honeycomb": 10, "kane_mele": 13}


def _op_bytes(n, row):
    return 20.0 * n * (row + 1) / 2 + 4.0 * (n + 1)


def _dos_work(lattice, lx, ly, lz, M, R, doubling):
    n, row = _size(lattice, lx, ly, lz), _ROW[lattice]
    steps, dots = (M // 2, 2) if doubling else (M - 1, 1)
    return (_op_bytes(n, row) + 16.0 * n * R + 16.0 * M, steps * n * R * (8.0 * row + 4.0 + 8.0 * dots))


def work(case):
    kind = case["kind"]
    if kind == "dos":
        b, f = _dos_work(case["lattice"], case["lx"], case["ly"], case["lz"], case["M"], case["R"],
                         case["algo"] == "doubling")
        return {"bytes": b, "flops": f}
    if kind in ("kubo", "corr"):
        n, R, comps = _size("honeycomb", case["lx"], case["ly"]), case["R"], case["comps"]
        M0, M1 = (case["M"], case["M"]) if kind == "kubo" else (case["M0"], case["M1"])
        steps = (M0 + M1) * n * R * (80.0 + 4.0) + (M1 * comps + 1) * n * R * 72.0
        ops = _op_bytes(n, 10) + comps * _op_bytes(n, 9) + 16.0 * n * R
        if kind == "corr":  # the whole table: three real products for a complex one
            return {"bytes": ops + 16.0 * comps * M0 * M1, "flops": steps + 6.0 * M0 * M1 * n * R * comps}
        # the energy sums from transforms over the orders of every site, twice as long as the orders
        f = 2.0 * M0
        sums = n * R * ((2 + comps) * 5.0 * f * math.log2(f) + 3 * comps * 8.0 * f)
        return {"bytes": ops + 32.0 * comps * case["nump"], "flops": steps + sums}
    if kind == "time":
        n, R = _size(case["lattice"], case["lx"], case["ly"]), case["R"]
        x = case["dt"] * _half_width(case["lattice"], 1.0) / 0.6582119624
        terms = x + 12.0
        step = n * R * ((case["M"] - 1) * (80.0 + 12.0) + 2 * terms * (80.0 + 12.0) + 72.0)
        return {"bytes": _op_bytes(n, 10) + _op_bytes(n, 9) + 16.0 * n * R + 16.0 * case["M"] * case["nT"],
                "flops": case["nT"] * step}
    if kind == "nonorth":
        n, R = _size("honeycomb", case["lx"], case["ly"]), case["R"]
        # about four iterations for each solve, two overlap products and six vector updates each
        return {"bytes": _op_bytes(n, 10) + 20.0 * n * 10 + 16.0 * n * R + 16.0 * case["M"],
                "flops": R * case["M"] * n * (80.0 + 4 * (2 * 80.0 + 6 * 8.0))}
    if kind == "tools":
        M = case["M"]
        energies = 32.0 * M
        return {"bytes": 16.0 * M * M * 2 + 16.0 * energies, "flops": energies * (4.0 * M * M + 8.0 * M)}
    d = [_batch_job(j) for j in _batch_sizes(case)]
    return {"bytes": sum(b for b, _ in d), "flops": sum(f for _, f in d)}


def _batch_sizes(case):
    mix = _rng(case["mix"])
    for _ in range(case["jobs"]):
        lattice = ["cubic", "kane_mele"][int(mix.integers(2))]
        n = int(math.exp(mix.uniform(math.log(4096), math.log(case["nmax"]))))
        mix.integers(2)
        M = max(64, int(case["M"] * mix.uniform(0.5, 1.0)))
        yield lattice, n, M, [1, 2, 4, 8][int(mix.integers(4))]


def _batch_job(j):
    lattice, n, M, R = j
    row = _ROW[lattice]
    return _op_bytes(n, row) + 16.0 * n * R + 16.0 * M, (M - 1) * n * R * (8.0 * row + 12.0)


# ---- the same in plain 64-bit torch ------------------------------------------------
def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _scaled(H, hw):
    cols, vals = H.on(_dev())
    return cols, vals / hw


def _moments(H, phi, M, T0=None):
    """sum_r <phi_r|T_m T0_r>, m < M, for phi [n][R]."""
    a = phi if T0 is None else T0
    mu = torch.zeros(M, dtype=torch.complex128, device=phi.device)
    mu[0] = (phi.conj() * a).sum()
    b = _apply(H, a)
    for m in range(1, M):
        mu[m] = (phi.conj() * b).sum()
        if m + 1 < M:
            a, b = b, _apply(H, b).mul_(2.0).sub_(a)
    return mu


def _exact_dos(d, M):
    dev = _dev()
    phi = torch.as_tensor(d["phi"].T.copy(), device=dev)
    mu = _moments(_scaled(d["H"], d["hw"]), phi, M) * (2.0 / phi.shape[1])
    mu[0] *= 0.5
    return mu.cpu().numpy()


def _tables(d, ML, MR):
    """sum_r <phi_r|V_x T_m V_o T_n|phi_r> for every operator o."""
    dev = _dev()
    H = _scaled(d["H"], d["hw"])
    V = [d["V"][c].on(dev) for c in sorted(d["V"])]
    phi = torch.as_tensor(d["phi"].T.copy(), device=dev)
    n, R = phi.shape
    top = max(ML, MR)
    L = torch.empty((ML, n * R), dtype=torch.complex128, device=dev)
    Rs = [torch.empty((MR, n * R), dtype=torch.complex128, device=dev) for _ in V]
    a = torch.cat([_apply(V[0], phi), phi], 1)
    b = None
    for m in range(top):
        if m < ML:
            L[m] = a[:, :R].reshape(-1)
        if m < MR:
            for v, t in zip(V, Rs):
                t[m] = _apply(v, a[:, R:].contiguous()).reshape(-1)
        if m + 1 < top:
            if b is None:
                a, b = _apply(H, a), a
            else:
                a, b = _apply(H, a).mul_(2.0).sub_(b), a
    L.conj_physical_()
    return [L @ t.T for t in Rs], R


def _exact_kubo(case, d):
    M, nump = case["M"], case["nump"]
    tabs, R = _tables(d, M, M)
    m = np.arange(M)
    g = ((M - m + 1.0) * np.cos(np.pi * m / (M + 1.0)) + np.sin(np.pi * m / (M + 1.0)) / np.tan(np.pi / (M + 1.0))) / (
        M + 1.0)
    c = (2.0 - (m == 0)) * g
    k = np.arange(nump)
    th = np.pi * (2 * k + 0.5) / nump
    s = np.where(k < nump // 2, 1.0, -1.0)
    t = c * np.cos(th[:, None] * m)
    e = t + 1j * s[:, None] * c * np.sin(th[:, None] * m)
    out = []
    for tab in tabs:
        mu = tab.cpu().numpy() / R
        tm = t @ mu
        if case["formula"] == "greenwood":
            out.append(np.concatenate([(tm * t).sum(1).real + 0j, np.zeros(nump)]))
            continue
        p = (tm * e).sum(1) + ((e.conj() @ mu) * t).sum(1)
        w = (((m * e).conj() @ mu) * t).sum(1) - (tm * (m * e)).sum(1)
        out.append(np.concatenate([p, w]))
    return np.stack(out)


def _exact_corr(case, d):
    M0, M1 = case["M0"], case["M1"]
    top = max(M0, M1)
    tabs, R = _tables(d, top, top)
    out = []
    for tab in tabs:
        t = tab * (4.0 / R)
        t[0] *= 0.5
        t[:, 0] *= 0.5
        out.append(((t + t.conj().T) / 2)[:M0, :M1].cpu().numpy())
    return np.stack(out)


def _bessel(x, tol=1e-10):
    """J_0(x), J_1(x), ... while |J_k| > tol for k >= 1, by downward recurrence."""
    top = int(x + 60 + 10 * x ** (1 / 3)) // 2 * 2 + 40
    j = np.zeros(top + 2)
    j[top] = 1e-280
    for k in range(top, 0, -1):
        j[k - 1] = 2 * k / x * j[k] - j[k + 1]
        if abs(j[k - 1]) > 1e200:
            j[k - 1:] *= 1e-200
    j /= j[0] + 2 * j[2:top + 1:2].sum()
    n = 1
    while n < top and abs(j[n]) > tol:
        n += 1
    return j[:n]


def _exact_time(case, d):
    dev = _dev()
    H, V = _scaled(d["H"], d["hw"]), d["V"]["x"].on(dev)
    phi = torch.as_tensor(d["phi"].T.copy(), device=dev)
    R = phi.shape[1]
    j = _bessel(case["dt"] * d["hw"] / 0.6582119624)
    coef = [(1.0 if k == 0 else 2.0) * (-1j) ** k * j[k] for k in range(len(j))]
    both = torch.cat([_apply(V, phi), phi], 1)
    out = np.zeros((case["M"], case["nT"]), dtype=np.complex128)
    for t in range(case["nT"]):
        left, right = both[:, :R].contiguous(), both[:, R:].contiguous()
        mu = _moments(H, left, case["M"], _apply(V, right)) * (2.0 / R)
        mu[0] *= 0.5
        out[:, t] = mu.cpu().numpy()
        a, b = both, _apply(H, both)
        acc = coef[0] * a
        for ck in coef[1:]:
            acc += ck * b
            a, b = b, _apply(H, b).mul_(2.0).sub_(a)
        both = acc
    return out


def _solve(S, b, tol=1e-14):
    """S^-1 b by conjugate gradients (S is Hermitian and positive)."""
    x = torch.zeros_like(b)
    r = b.clone()
    p = r.clone()
    rr = (r.conj() * r).sum().real
    stop = tol * tol * rr
    for _ in range(200):
        q = _apply(S, p)
        al = rr / (p.conj() * q).sum().real
        x += al * p
        r -= al * q
        new = (r.conj() * r).sum().real
        if new <= stop:
            break
        p = r + (new / rr) * p
        rr = new
    return x


def _exact_nonorth(case, d):
    dev = _dev()
    H, S = _scaled(d["H"], d["hw"]), d["S"].on(dev)
    out = torch.zeros(case["M"], dtype=torch.complex128, device=dev)
    for r in range(case["R"]):
        phi = torch.as_tensor(d["phi"][r].copy(), device=dev)[:, None]
        a = _solve(S, phi)
        b = _solve(S, _apply(H, a))
        for m in range(case["M"]):
            out[m] += (1.0 if m == 0 else 2.0) / case["R"] * (phi.conj() * a).sum()
            a, b = b, 2.0 * _solve(S, _apply(H, b)) - a
    return out.cpu().numpy()


def _crescent(n):
    j = np.arange(n)
    i = np.where((j < n // 2) | (j >= n - n // 2), n - 1 - j, j)
    return np.where(i < 2 * (n // 2), np.where(i % 2 == 0, i // 2, n - 1 - i // 2), i)


def _exact_tools(case, d):
    M, n, W, Ec, nump = case["M"], d["n"], d["W"], d["Ec"], case["nump"]
    a = W / 2.0
    top = min(M, int(math.ceil(np.pi / (2.0 * case["broad"] / 1000 / W))))
    m = np.arange(top)
    phi = np.pi / (top + 1.0)
    g = ((top - m + 1) * np.cos(phi * m) + np.sin(phi * m) * np.cos(phi) / np.sin(phi)) * phi / np.pi
    one, two = d["one"][:top] * g, d["mu"][:top, :top] * np.outer(g, g)

    def delta(x):
        return np.cos(np.arccos(x)[:, None] * m) / np.sqrt(1 - x * x)[:, None] / np.pi

    def green(x):  # -i z^m / f, z = x - i f = e^{-i arccos x}
        f = np.sqrt(1 - x * x)[:, None]
        return -1j * np.exp(-1j * np.arccos(x)[:, None] * m) / f

    def dgreen(x):
        f = np.sqrt(1 - x * x)[:, None]
        return -1j * np.exp(-1j * np.arccos(x)[:, None] * m) * (x[:, None] + 1j * m * f) / f ** 3

    def kernel(x, right):
        dev = _dev()
        z = torch.as_tensor(delta(x), device=dev).to(torch.complex128) @ torch.as_tensor(two, device=dev)
        return (z.cpu().numpy() * right(x)).sum(1).imag

    nd = 2 * top
    x = np.cos(np.pi * (np.arange(nd) + 0.5) / nd)
    E, rho = x * a + Ec, np.abs(delta(x) @ one.real * (n / a))
    x = np.cos(np.pi * (2 * np.arange(top) + 0.5) / top)
    Eg, sg = (x * a + Ec)[:-1], -(kernel(x, green) * (n / a / a))[:-1]
    x = np.cos(np.pi * (2 * _crescent(top) + 0.5) / top)
    k = kernel(x, dgreen) * (-2.0 * n / a / a)
    Eb, sb = (x * a + Ec)[:-1], np.cumsum((k[:-1] * np.diff(x)))
    nl = 30 * top
    x = -0.99 + np.arange(nl) * 1.98 / (nl - 1)
    k = kernel(x, dgreen) * (-2.0 * n / a / a)
    El, sl = (x * a + Ec)[:-1], np.cumsum(k[:-1] * np.diff(x))
    src = _crescent(nump)
    e = np.cos(np.pi * (2 * src + 0.5) / nump)
    fd = d["fd"]
    gk = (e * fd[src].real - np.sqrt(1 - e * e) * fd[src + nump].imag) / (1 - e * e) ** 2 * (n / (a * a) / np.pi)
    sk = np.concatenate([np.cumsum(gk[:-1] * np.diff(e)), [0.0]])
    return dict(one=one, two=two, E=E, rho=rho, Eg=Eg, sg=sg, Eb=Eb, sb=sb, El=El, sl=sl, Ek=a * e - Ec, sk=sk, gk=gk)


def exact(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    if kind == "dos":
        return _exact_dos(d, case["M"])
    if kind == "kubo":
        return _exact_kubo(case, d)
    if kind == "corr":
        return _exact_corr(case, d)
    if kind == "time":
        return _exact_time(case, d)
    if kind == "nonorth":
        return _exact_nonorth(case, d)
    if kind == "tools":
        return _exact_tools(case, d)
    return [_exact_dos(j, j["M"]) for j in d["jobs"]]
