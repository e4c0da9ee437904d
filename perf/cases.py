"""Performance cases of the engine: the calls a user's program makes, through
the Python mirror of the C ABI, over the lattices the engine is used on.

Kinds of case (what each listed one stands for is said at `listed`):

  energy    ccgpu_energy_noalloc on device buffers of the caller
  iterate   the step API of the Fortran host on its own orbital table: start,
            then `its` times residual, update and energy
  solve     one CCD solve on a lattice that is set up: start, ccd_iter
  lattice   a new interaction on a lattice: V, Fock, start, first iteration
  densities one batch over several densities of one lattice
  twists    one batch over seeded twists of one lattice (shared pp ladder)
  point     a whole deck: V (with the three-nucleon force), CCD, (T)
  triples   (T) on the amplitudes of a solve, its element tables in place
  ccdt1     one triples step of a CCDT-1 iteration
  network   the learned start: training steps, then the start of a lattice

The seed of `prepare` moves the density by up to 2% (and draws the amplitudes,
the network's parameters and the training samples), so the channels of a case
are the same for every seed and its numbers are not.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch   # first: the engine then shares its HIP runtime

HBARC, PMASS, PI = 197.326968, float(np.float32(939.565)), 3.14159265358979


def _package():
    if "ccnm" not in sys.modules:
        path = os.path.join(os.getcwd(), "coupled-cluster-nuclearmatter_amd", "ccnm.py")
        spec = importlib.util.spec_from_file_location("ccnm", path)
        mod = importlib.util.module_from_spec(spec)
        sys.modules["ccnm"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["ccnm"]


def listed():
    return [
        # the energy sum a serving loop enqueues on its own buffers, at the
        # amplitude count of PNM A=66 |n_i|<=4
        {"name": "energy_pnm66_n4", "kind": "energy", "n": 1991568},
        # smallest lattice of the decks: launches and latency are everything
        {"name": "iterate_pnm14_n1", "kind": "iterate", "A": 14, "matter": 0, "rho": 0.16, "nmax": 1, "its": 4},
        # the sample deck's size (SNM A=28 |n_i|<=2), NN only, default options
        {"name": "solve_snm28_n2", "kind": "solve", "A": 28, "matter": 1, "rho": 0.16, "nmax": 2, "twist": 0,
         "precision": 0, "accel": 0, "graph": 0},
        # mixed precision (split bfloat16, FP64 to the end) with the Anderson
        # update on a twisted lattice: the production setting of one twist
        {"name": "solve_pnm66_n3_mixed", "kind": "solve", "A": 66, "matter": 0, "rho": 0.12, "nmax": 3, "twist": 1,
         "precision": 3, "accel": 1, "graph": 1},
        # the plain FP64 solver on the largest lattice, replayed from a graph
        {"name": "solve_pnm66_n4", "kind": "solve", "A": 66, "matter": 0, "rho": 0.16, "nmax": 4, "twist": 0,
         "precision": 0, "accel": 0, "graph": 1},
        # a scan over densities or constants refills V every time; the first
        # iteration reads every block of it
        {"name": "lattice_pnm66_n4", "kind": "lattice", "A": 66, "matter": 0, "rho": 0.16, "nmax": 4, "twist": 0,
         "interaction": 1},
        # the equation of state: four densities in one batch, low precision
        # first, to 1e-5 MeV per nucleon
        {"name": "densities4_pnm66_n4", "kind": "densities", "A": 66, "matter": 0, "nmax": 4, "count": 4,
         "rho": 0.08, "step": 0.04},
        # twist averaging: eight twists in one batch with one V_pppp
        {"name": "twists8_pnm66_n3", "kind": "twists", "A": 66, "matter": 0, "nmax": 3, "rho": 0.16, "count": 8,
         "tseed": 17},
        # the sample deck as a whole: NN and normal-ordered 3NF, CCD, (T)
        {"name": "point_snm28_n2_3nf", "kind": "point", "A": 28, "matter": 1, "rho": 0.16, "nmax": 2, "twist": 0,
         "tnf": 2},
        # (T) of a converged solve, the largest sum listed here
        {"name": "triples_pnm66_n3", "kind": "triples", "A": 66, "matter": 0, "rho": 0.16, "nmax": 3, "twist": 0},
        # CCDT-1 repeats this triples step in every iteration
        {"name": "ccdt1_pnm66_n2", "kind": "ccdt1", "A": 66, "matter": 0, "rho": 0.16, "nmax": 2, "twist": 0},
        # the learned start: Adam steps on minibatches, then its inference
        {"name": "network_pnm66_n2", "kind": "network", "A": 66, "matter": 0, "rho": 0.16, "nmax": 2, "steps": 40,
         "batch": 16384},
    ]


# closed shells of the lattice (particles per nucleon species and spin: 1, 7,
# 19, 27, 33 momenta)
_PNM = {1: (14,), 2: (14, 38, 54, 66), 3: (14, 38, 54, 66), 4: (14, 38, 54, 66)}
_SNM = {1: (4, 28), 2: (4, 28, 76, 108), 3: (4, 28)}


def draw(rng):
    def lattice(nmin, nmax, snm=0.4):
        m = 1 if rng.random() < snm else 0
        n = rng.randint(nmin, min(nmax, 3) if m else nmax)
        return {"A": rng.choice((_SNM if m else _PNM)[n]), "matter": m, "nmax": n,
                "rho": round(math.exp(rng.uniform(math.log(0.06), math.log(0.24))), 4)}

    kind = rng.choice(("energy", "iterate", "solve", "solve", "lattice", "densities", "twists", "point", "triples",
                       "ccdt1", "network"))
    if kind == "energy":
        return {"kind": kind, "n": int(math.exp(rng.uniform(math.log(500), math.log(4e6))))}
    if kind == "iterate":
        return {"kind": kind, **lattice(1, 3), "its": rng.randint(1, 5)}
    if kind == "solve":
        p = rng.choice((0, 0, 1, 2, 3))
        return {"kind": kind, **lattice(1, 4), "twist": rng.choice((0, 1)), "precision": p,
                "accel": 1 if p else rng.choice((0, 1)), "graph": rng.choice((0, 1))}
    if kind == "lattice":
        return {"kind": kind, **lattice(1, 4), "twist": rng.choice((0, 1)), "interaction": rng.choice((0, 1, 1))}
    if kind == "densities":
        return {"kind": kind, **lattice(2, 3, 0.0), "count": rng.randint(2, 5), "step": round(rng.uniform(0.01, 0.04), 3)}
    if kind == "twists":
        return {"kind": kind, **lattice(2, 3, 0.0), "count": rng.randint(2, 12), "tseed": rng.randrange(1000)}
    if kind == "point":
        c = lattice(1, 2)
        c["A"] = min(c["A"], 66)
        return {"kind": kind, **c, "twist": rng.choice((0, 1)), "tnf": rng.choice((-1, 0, 1, 2))}
    if kind == "triples":
        c = lattice(1, 3, 0.3)
        c["A"] = min(c["A"], 66 if c["matter"] == 0 else 28)
        return {"kind": kind, **c, "twist": rng.choice((0, 1))}
    if kind == "ccdt1":
        c = lattice(1, 2, 0.3)
        c["A"] = min(c["A"], 66 if c["matter"] == 0 else 28)
        return {"kind": kind, **c, "twist": rng.choice((0, 1))}
    return {"kind": kind, **lattice(1, 3, 0.0), "steps": rng.randint(5, 60),
            "batch": 64 * int(math.exp(rng.uniform(math.log(1), math.log(1024))))}


def _twist(case):
    return (0.5, 1.0, 1.5) if case.get("twist") else (0.0, 0.0, 0.0)


def _density(case, rng):
    return case["rho"] * (1.0 + 0.04 * (rng.random() - 0.5))


def _solver(ccnm, case, rho, twist=None, tnf=-1, kind=1):
    s = ccnm.Solver(A=case["A"], matter=case["matter"], rho=rho, nmax=case["nmax"],
                    twist=_twist(case) if twist is None else twist)
    if kind == 1:
        s.set_chiral(ccnm.NNLO, 450.0)
        if tnf >= 0:
            s.set_3nf(tnf, 0.017, 0.79, 450.0, 3)
    s.generate_interaction(kind)
    return s


def _twists(case):
    return np.random.default_rng(case["tseed"]).uniform(0.0, PI, (case["count"], 3))


def _orbitals(case, rho):
    """The orbital table of a host program: momenta (2 pi n + theta)/L sorted by
    k^2, spin and isospin within a momentum, the first A states are holes."""
    box = (case["A"] / rho) ** (1.0 / 3.0)
    r = range(-case["nmax"], case["nmax"] + 1)
    n = np.array([(x, y, z) for x in r for y in r for z in r])
    k = (2.0 * PI * n + np.array(_twist(case))) / box
    o = np.argsort(np.round(np.sum(k * k, 1), 10), kind="stable")
    st = [(sz, tz) for sz in (-1, 1) for tz in ((1,) if case["matter"] == 0 else (-1, 1))]
    n, k = np.repeat(n[o], len(st), 0), np.repeat(k[o], len(st), 0)
    st = np.tile(np.array(st), (len(o), 1))
    return {"nx": n[:, 0], "ny": n[:, 1], "nz": n[:, 2], "sz": st[:, 0], "tz": st[:, 1], "kx": k[:, 0], "ky": k[:, 1],
            "kz": k[:, 2], "e": HBARC ** 2 * np.sum(k * k, 1) / (2.0 * PMASS), "A": case["A"], "box": box,
            "volume": box ** 3}


def _labels(o):
    """a < b, i < j of every amplitude that conserves momentum and isospin."""
    A, n = o["A"], np.stack([o["nx"], o["ny"], o["nz"], o["tz"]], 1)

    def pairs(lo, hi):
        x, y = np.triu_indices(hi - lo, 1)
        key = (n[x + lo] + n[y + lo]) @ np.array([1, 64, 4096, 262144])
        return x + lo, y + lo, key

    i, j, kh = pairs(0, A)
    a, b, kp = pairs(A, len(n))
    out = []
    for key in np.unique(kh):
        h, p = np.flatnonzero(kh == key), np.flatnonzero(kp == key)
        ph, pp = np.meshgrid(h, p)
        out.append(np.stack([a[pp].ravel(), b[pp].ravel(), i[ph].ravel(), j[ph].ravel()]))
    return [np.ascontiguousarray(x, np.int32) for x in np.concatenate(out, 1)]


def _energy_inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    mk = lambda s: torch.view_as_complex(  # noqa: E731
        s * torch.randn(case["n"], 2, generator=g, device="cuda", dtype=torch.float64))
    return mk(0.01), mk(0.5)


def prepare(case, seed):
    ccnm = _package()
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    st = {"kind": kind, "case": case, "ccnm": ccnm}
    if kind == "energy":
        st["t"], st["r0"] = _energy_inputs(case, seed)
        st["out"] = torch.zeros(1, dtype=torch.complex128, device="cuda")
        return st
    rho = _density(case, rng)
    if kind == "iterate":
        o = _orbitals(case, rho)
        st["s"] = ccnm.Solver(orbitals=o)
        st["s"].generate_interaction(ccnm.INT_MINNESOTA)
        st["labels"] = _labels(o)
    elif kind == "solve":
        st["s"] = _solver(ccnm, case, rho)
    elif kind == "lattice":
        st["s"] = ccnm.Solver(A=case["A"], matter=case["matter"], rho=rho, nmax=case["nmax"], twist=_twist(case))
    elif kind == "densities":
        st["s"] = [_solver(ccnm, case, rho + case["step"] * k) for k in range(case["count"])]
    elif kind == "twists":
        st["s"] = [_solver(ccnm, case, rho, twist=tuple(t)) for t in _twists(case)]
    elif kind == "point":
        st["s"] = ccnm.Solver(A=case["A"], matter=case["matter"], rho=rho, nmax=case["nmax"], twist=_twist(case))
    elif kind in ("triples", "ccdt1"):
        s = st["s"] = _solver(ccnm, case, rho, tnf=2 if kind == "ccdt1" else -1)
        s.setup_t_amplitudes()
        s.ccd_iter()
        if kind == "ccdt1":
            s.setup_t3()
    else:
        s = _solver(ccnm, case, rho)
        s.setup_t_amplitudes()
        s.ccd_iter()
        st["net"] = ccnm.WarmStart(seed=1)
        st["net"].add_solve(s)
        s.close()
        st["s"] = _solver(ccnm, case, 1.1 * rho)
        # He-normal hidden layers, small output layer, zero biases
        th = np.zeros(ccnm.MLP_NPARAM, np.float32)
        for off, fan, count, gain in ((0, 16, 1024, 2.0), (1088, 64, 4096, 2.0), (5248, 64, 4096, 2.0),
                                      (9408, 64, 64, 0.01)):
            th[off:off + count] = rng.standard_normal(count) * math.sqrt(gain / fan)
        st["theta"], st["seed"] = th, int(seed) % 100000
    return st


def _solve_options(case):
    kw = {"use_graph": case["graph"], "precision": case["precision"], "accel": case["accel"]}
    if case["accel"]:
        kw.update(subspace=8, tol=1e-8)
    if case["precision"]:
        kw.update(fp32_switch=3e-2)
    return kw


def _results(rs):
    return {"iterations": [r["iterations"] for r in rs], "e0": np.array([r["e0"] for r in rs]),
            "embpt2": np.array([r["embpt2"] for r in rs]), "eccd": np.array([r["eccd"] for r in rs])}


def run(st):
    kind, case, ccnm = st["kind"], st["case"], st["ccnm"]
    s = st.get("s")
    if kind == "energy":
        ccnm.energy_noalloc(case["n"], st["t"].data_ptr(), st["r0"].data_ptr(), st["out"].data_ptr(),
                            torch.cuda.current_stream().cuda_stream)
        return st["out"]
    if kind == "iterate":
        e = [s.setup_t_amplitudes()]
        count = nstep = 0
        for _ in range(case["its"]):
            s.t2_intermediate(ccnm.PREC_FP64)
            count, nstep = s.diis_t1t2(count + 1, nstep + 1)
            e.append(s.ccd_energy_save())
        return {"e0": np.array(s.e0()), "energies": np.array(e), "t2": s.get_t2(*st["labels"])}
    if kind == "solve":
        s.setup_t_amplitudes()
        r = s.ccd_iter(**_solve_options(case))
        return {**_results([r]), "t2": s.t2_unique()}
    if kind == "lattice":
        s.generate_interaction(case["interaction"])
        e = [s.e0(), s.setup_t_amplitudes()]
        s.t2_intermediate(ccnm.PREC_FP64)
        s.diis_t1t2(1, 1)
        e.append(s.ccd_energy_save())
        return {"energies": np.array(e), "fock": s.fock_diag(), "t2": s.t2_unique()}
    if kind == "densities":
        for x in s:
            x.setup_t_amplitudes()
        return _results(ccnm.batch_solve(s, subspace=8, tol=1e-5 * case["A"], precision=ccnm.PREC_BF16X3,
                                         tail=ccnm.PREC_V32, fp32_switch=3e-2, use_graph=1, accel=1, confirm=1))
    if kind == "twists":
        for x in s:
            x.setup_t_amplitudes()
        rs = ccnm.batch_solve(s, subspace=8, tol=1e-8, precision=ccnm.PREC_BF16X3, fp32_switch=3e-2, use_graph=1,
                              accel=1)
        return {**_results(rs), "t2": [x.t2_unique() for x in s]}
    if kind == "point":
        s.set_chiral(ccnm.NNLO, 450.0)
        s.set_3nf(case["tnf"], 0.017, 0.79, 450.0, 3)
        s.generate_interaction(ccnm.INT_CHIRAL)
        s.setup_t_amplitudes()
        r = s.ccd_iter()
        et = s.pert_triples2()
        return {**_results([r]), "et": np.array(et), "fock": s.fock_diag(), "t2": s.t2_unique()}
    if kind == "triples":
        return np.array(s.pert_triples2())
    if kind == "ccdt1":
        s.t3_intermediate()
        return np.array(s.t3_energy())
    net = st["net"]
    net.params = st["theta"]
    loss = net.train(case["steps"], batch=case["batch"], lr=1e-3, seed=st["seed"])
    e = net.warm_start(s)
    return {"loss": np.array(loss), "params": net.params, "energy": np.array(e), "t2": s.t2_unique()}


def _triples_count(case):
    """(abc, ijk) elements of equal total momentum and isospin: ordered triples
    of distinct states by inclusion and exclusion on momentum histograms."""
    o = _orbitals(case, case["rho"])
    n = np.stack([o["nx"], o["ny"], o["nz"]], 1)
    A, m = case["A"], 8 * case["nmax"] + 2
    total = 0.0

    def hist(idx, mult):
        h = np.zeros((8, m, m, m))
        np.add.at(h, (mult * (o["tz"][idx] + 1) // 2 % 8, *((mult * n[idx].T) % m)), 1.0)
        return np.fft.fftn(h)

    h, p = np.arange(A), np.arange(A, len(n))
    three = []
    for idx in (h, p):
        f1, f2, f3 = (hist(idx, k) for k in (1, 2, 3))
        three.append(np.fft.ifftn((f1 ** 3 - 3 * f1 * f2 + 2 * f3) / 6).real)
    total = float(np.sum(three[0] * three[1]))
    return max(total, 1.0)


def work(case):
    kind = case["kind"]
    if kind == "energy":
        return {"bytes": 32.0 * case["n"] + 16, "flops": 8.0 * case["n"]}
    twists = [_twist(case)] if kind != "twists" else [tuple(t) for t in _twists(case)]
    d = [_package().plan(case["A"], case["matter"], case["rho"], case["nmax"], t) for t in twists]
    d, n = d[0], len(d)
    nT, nV, ring = 16.0 * d["t2_unique"], 16.0 * d["vpppp_unique"], 16.0 * d["ring_elems"]
    flops = d["pp_ladder_flops"] + d["hh_ladder_flops"] + d["ring_flops"]
    # of an iteration: V_pppp, V_hhpp (also as the ring's block) and T read, T
    # and its history written
    its = nV + 5 * nT + ring
    A, p = case["A"], d["nparticles"]
    if kind == "iterate":
        return {"bytes": case["its"] * its, "flops": case["its"] * flops}
    if kind == "solve":
        # about 13 iterations; the low-precision ones read half of V
        return {"bytes": 13 * (0.6 if case["precision"] else 1.0) * its, "flops": 13 * flops}
    if kind == "lattice":
        return {"bytes": nV + its + 3 * nT, "flops": flops + 250.0 * d["vpppp_unique"]}
    if kind == "densities":
        return {"bytes": 7 * case["count"] * 0.6 * its, "flops": 7 * case["count"] * flops}
    if kind == "twists":
        return {"bytes": 13 * (0.6 * nV + n * (5 * nT + ring)), "flops": 13 * n * flops}
    table = 32.0 * (p * p * A + A * A * p)
    if kind == "point":
        three = 3000.0 * A * (d["vpppp_unique"] / 2 + d["t2_unique"] + p * p * A / 2) if case["tnf"] >= 2 else 0.0
        return {"bytes": 13 * its + nV + 2 * table, "flops": 13 * flops + three + 300.0 * _triples_count(case)}
    if kind == "triples":
        return {"bytes": table + nT, "flops": 300.0 * _triples_count(case)}
    if kind == "ccdt1":
        return {"bytes": table + nT, "flops": 3300.0 * _triples_count(case)}
    # per sample and step: forward, and twice as much backward
    return {"bytes": case["steps"] * (case["batch"] * 36.0 + 9473 * 16.0) + 4 * nT,
            "flops": case["steps"] * case["batch"] * 6.0 * 9280 + 2.0 * 9280 * d["t2_unique"]}


def _minnesota(o, dev):
    """Dense antisymmetrized Minnesota elements <pq||rs> in MeV."""
    n = torch.tensor(np.stack([o["nx"], o["ny"], o["nz"]], 1), device=dev)
    sz, tz = (torch.tensor(o[k], device=dev) for k in ("sz", "tz"))
    f32 = lambda x: float(np.float32(x))  # noqa: E731
    N, unit = len(n), PI / o["box"]

    def ss(a, p):
        """spin (isospin) identity and sigma.sigma between (p q) and (r s)"""
        q, r, s = a[:, None, None], a[None, :, None], a[None, None, :]
        same = ((a[p] == r) & (q == s)).double()
        exch = ((a[p] == s) & (q == r) & (a[p] != q)).double()
        return same, same * (a[p] * q) + 2.0 * exch

    V = torch.zeros(N, N, N, N, dtype=torch.float64, device=dev)
    for p in range(N):
        q, r, s = n[:, None, None], n[None, :, None], n[None, None, :]
        q2 = unit * unit * (n[p] - q - r + s).square().sum(-1).double()
        ds, sg = ss(sz, p)
        dt, ta = ss(tz, p)
        g = [v0 * PI ** 1.5 * torch.exp(-q2 / (4.0 * k)) / k ** 1.5
             for v0, k in ((200.0, f32(1.487)), (-178.0, f32(0.639)), (-f32(91.85), f32(0.465)))]
        v = (g[0] * (3 * ds * dt - ta * ds - sg * dt - ta * sg) / 8
             + g[1] * (3 * ds * dt - 3 * ta * ds + sg * dt - ta * sg) / 16
             + g[2] * (3 * ds * dt + ta * ds - 3 * sg * dt - ta * sg) / 16) / o["volume"]
        ok = (n[p] + q == r + s).all(-1) & (tz[p] + tz[:, None, None] == tz[None, :, None] + tz[None, None, :])
        V[p] = torch.where(ok, v, torch.zeros_like(v))
    return V - V.transpose(2, 3)


def _exact_iterate(case, seed):
    """The CCD equations with every index dense, in 64 bits."""
    o = _orbitals(case, _density(case, np.random.default_rng(seed)))
    A, N = o["A"], len(o["nx"])
    if N > 108 or (N - A) ** 4 * A * A > 4e10:
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    V = _minnesota(o, dev)
    e = torch.tensor(o["e"], device=dev)
    h, p = slice(0, A), slice(A, None)
    f = torch.diag(e) + torch.einsum("piqi->pq", V[:, h, :, h])
    e0 = e[h].sum() + 0.5 * torch.einsum("ijij->", V[h, h, h, h])
    fd = torch.diagonal(f)
    Vhhpp = V[h, h, p, p].contiguous()
    Vpphh = V[p, p, h, h].contiguous()
    fpp, fhh = f[p, p], f[h, h]

    def den(x, y):
        return (x[None, None, :, None] + x[None, None, None, :] - y[:, None, None, None] - y[None, :, None, None])

    def energy(t):
        return 0.25 * torch.sum(Vhhpp.permute(2, 3, 0, 1) * t)

    pab = lambda x: x - x.transpose(0, 1)  # noqa: E731
    pij = lambda x: x - x.transpose(2, 3)  # noqa: E731
    zero = torch.zeros((), dtype=torch.float64, device=dev)
    d0 = den(fd[h], fd[p])
    t = torch.where(Vpphh != 0, Vpphh / d0, zero)
    es = [energy(t)]
    for _ in range(case["its"]):
        x = 0.5 * torch.einsum("klcd,cdil->ki", Vhhpp, t)
        y = 0.5 * torch.einsum("kldc,dakl->ac", Vhhpp, t)
        i9 = V[h, h, h, h] + 0.5 * torch.einsum("klcd,cdij->klij", Vhhpp, t)
        w = V[h, p, p, h] + 0.5 * torch.einsum("klcd,dblj->kbcj", Vhhpp, t)
        r = Vpphh + pab(torch.einsum("bc,acij->abij", fpp - y, t)) - pij(torch.einsum("kj,abik->abij", fhh + x, t))
        r = r + 0.5 * torch.einsum("abcd,cdij->abij", V[p, p, p, p], t) + 0.5 * torch.einsum("klij,abkl->abij", i9, t)
        r = r + pab(pij(torch.einsum("kbcj,acik->abij", w, t)))
        d = den(fd[h] + torch.diagonal(x), fd[p] - torch.diagonal(y))
        t = t + 0.25 * torch.where(Vpphh.abs() + t.abs() + r.abs() > 0, r / d, zero)
        es.append(energy(t))
    lab = [torch.tensor(z, device=dev, dtype=torch.long) for z in _labels(o)]
    t2 = t[lab[0] - A, lab[1] - A, lab[2], lab[3]].cpu().numpy().astype(np.complex128)
    return {"e0": np.array(complex(e0.item())), "energies": np.array([complex(z.item()) for z in es]), "t2": t2}


def exact(case, seed):
    if case["kind"] == "energy":
        t, r0 = _energy_inputs(case, seed)
        return torch.sum(t * r0.conj()).reshape(1)
    if case["kind"] == "iterate":
        return _exact_iterate(case, seed)
    return None
