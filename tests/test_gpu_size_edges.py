"""Kernels at the sizes where their loops and dispatch rules change over:
remainders of unrolled loads, edges of tiles, the smallest and largest of a
rule's range, against the oracle or a plain sum."""
import ctypes as C

import numpy as np
import pytest

import mlp_oracle as mo

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip(ccnm):
    ccnm.lib()   # the library loads the image's HIP runtime; the test uses the same one
    rt = C.CDLL("libamdhip64.so.7")
    rt.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    rt.hipFree.argtypes = [C.c_void_p]
    rt.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    rt.hipDeviceSynchronize.argtypes = []
    return rt


@pytest.mark.parametrize("n", [0, 1, 255, 2047, 2048, 2049, 4096 * 2048, 4096 * 2048 + 1, 4097 * 2048 + 300])
def test_energy_noalloc_sum_at_span_edges(ccnm, hip, n):
    """Spans of 2048 amplitudes up to 4096 partials, then longer ones.  A
    thread adds at most 16 products in a row here (longer spans: 2 x 8), the
    trees above it 6 + 4 + 4 + 6 + 16 more, each rounding by at most 2^-53 of
    the sum of moduli, and a product by 2^-52: 64 * 2^-53 covers them."""
    rng = np.random.default_rng(n)
    t, r0 = (rng.standard_normal(2 * n).view(np.complex128) for _ in range(2))
    dev = []
    try:
        for a in (t, r0, np.full(1, 7.0 + 7.0j)):
            p = C.c_void_p()
            assert hip.hipMalloc(C.byref(p), max(a.nbytes, 16)) == 0
            dev.append(p)
            if a.nbytes:
                assert hip.hipMemcpy(p, a.ctypes.data, a.nbytes, 1) == 0
        out = np.zeros(1, np.complex128)
        for _ in range(2):
            ccnm.energy_noalloc(n, dev[0].value, dev[1].value, dev[2].value, None)
            assert hip.hipDeviceSynchronize() == 0
            assert hip.hipMemcpy(out.ctypes.data, dev[2], 16, 2) == 0
    finally:
        for p in dev:
            hip.hipFree(p)
    prod = t * np.conj(r0)
    want = complex(np.sum(prod.real.astype(np.longdouble)), np.sum(prod.imag.astype(np.longdouble)))
    assert abs(out[0] - want) <= 64 * 2.0 ** -53 * np.sum(np.abs(t) * np.abs(r0))


@pytest.mark.parametrize("n", [1, 15, 64, 65, 255, 257, 513, 576, 131136])
def test_mlp_gradient_at_chunk_edges(ccnm, n):
    """Minibatches whose last chunk leaves remainders of the unrolled loads
    (chunks of 512; 131136 samples make chunks of 528), against the oracle with
    the same BF16 rounding points, at the tolerance of
    test_mlp_gradient_matches_oracle: a dropped MFMA step of 16 samples would
    be 3% of its chunk and show in the small cases as a whole."""
    from test_mlp import random_problem
    theta, x, t = random_problem(n, n)
    net = ccnm.WarmStart(seed=1)
    net.params = theta.astype(np.float32)
    loss, g = net.loss_grad(x, t)
    lo, go = mo.loss_grad(theta, x.astype(np.float64), t.astype(np.float64), bf=True)
    assert abs(loss - lo) < 1e-4 * lo
    o = 0
    for name, shp in mo.SHAPES:
        m = int(np.prod(shp))
        a, b = g[o:o + m], go[o:o + m]
        assert np.linalg.norm(a - b) < 1e-2 * np.linalg.norm(b) + 1e-7, (name, np.linalg.norm(a - b))
        o += m


@pytest.mark.parametrize("batch", [64, 192, 576])
def test_mlp_training_step_takes_the_gradient_of_its_minibatch(ccnm, batch):
    """The first Adam step of train() restated on loss_grad of the same
    minibatch (the splitmix64 draw over the training set) at the same
    parameters.  (From the second step on the parameters differ in their last
    bits and single BF16 weights may round the other way.)"""
    s = ccnm.Solver(A=14, matter=ccnm.PNM, rho=0.16, nmax=1)
    s.generate_interaction()
    s.setup_t_amplitudes()
    s.ccd_iter()
    net, ref = ccnm.WarmStart(seed=5), ccnm.WarmStart(seed=5)
    n = net.add_solve(s)
    f, tgt = net.features(s)
    lr, seed, M64 = 1e-3, 77, (1 << 64) - 1
    loss = net.train(1, batch=batch, lr=lr, seed=seed)
    idx = []
    for pos in range(batch):
        z = (seed + 0x51ED27 + 0x9E3779B97F4A7C15 * (pos + 1)) & M64
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & M64
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & M64
        idx.append((z ^ (z >> 31)) % n)
    th = ref.params
    want, g = ref.loss_grad(f[idx], tgt[idx])
    g = g.astype(np.float64)
    step = lr * g / (np.abs(g) + 1e-8)   # m / (1 - b1) over the root of v / (1 - b2)
    assert abs(loss - want) <= 1e-6 * want
    # float32 powers of beta (1 - beta2 keeps 2^-24 / 1e-3 = 6e-5 relative,
    # half of it after the root) and the roundings of m, v and the step
    assert np.max(np.abs(net.params - (th - step))) <= 1e-4 * lr + 2.0 ** -23 * np.max(np.abs(th))


@pytest.mark.parametrize("A,matter,nmax,twist", [
    (14, "pnm", 1, (0.0, 0.0, 0.0)), (2, "pnm", 1, (0.0, 0.0, 0.0)), (15, "pnm", 1, (0.3, 0.7, 1.1)),
    (13, "pnm", 1, (0.0, 0.0, 0.0)), (4, "snm", 1, (0.0, 0.0, 0.0)), (9, "snm", 1, (0.4, 0.2, 0.9)),
    (28, "snm", 1, (0.0, 0.0, 0.0)), (38, "pnm", 2, (0.5, 1.0, 1.5))])
def test_triples_group_kernel_equals_element_kernels(ccnm, monkeypatch, A, matter, nmax, twist):
    """(T) over spin groups against the kernel that gathers every element and
    the one that evaluates them in place, on closed and open shells (groups
    with one spin state, a group split between holes and particles, fewer than
    three holes).  The same terms in another order: each of the 36 products of
    W and the sum over the elements round by 2^-53 of their moduli; the sum has
    one sign per element (every D is negative here), so 1e-12 leaves room for
    cancellation inside W."""
    s = ccnm.Solver(A=A, matter=ccnm.PNM if matter == "pnm" else ccnm.SNM, rho=0.16, nmax=nmax, twist=twist)
    s.set_chiral(ccnm.NNLO, 450.0)
    s.generate_interaction(ccnm.INT_CHIRAL)
    s.setup_t_amplitudes()
    for _ in range(2):
        s.t2_intermediate()
        s.diis_t1t2(1, 1)
    out = {}
    for variant in (None, "3", "0"):
        if variant is None:
            monkeypatch.delenv("CCGPU_T3_KERNEL", raising=False)
        else:
            monkeypatch.setenv("CCGPU_T3_KERNEL", variant)
        out[variant] = (s.pert_triples2(), s.triples_stats()[0])
    s.close()
    (e, n), (e3, n3), (e0, n0) = out[None], out["3"], out["0"]
    assert n == n3 == n0
    assert abs(e - e3) <= 1e-12 * abs(e3), out
    assert abs(e - e0) <= 1e-12 * abs(e0), out


def test_triples_after_a_new_interaction_and_fock(ccnm):
    """The tables of a handle follow its interaction: (T) after a second
    generation equals that of a fresh handle."""
    def fresh(order):
        s = ccnm.Solver(A=14, matter=ccnm.PNM, rho=0.16, nmax=1)
        s.set_chiral(order, 450.0)
        s.generate_interaction(ccnm.INT_CHIRAL)
        s.setup_t_amplitudes()
        return s
    a = fresh(ccnm.NNLO)
    first = a.pert_triples2()
    a.set_chiral(ccnm.LO, 450.0)
    a.generate_interaction(ccnm.INT_CHIRAL)
    a.setup_t_amplitudes()
    b = fresh(ccnm.LO)
    assert a.pert_triples2() == b.pert_triples2()
    assert abs(first - b.pert_triples2()) > 1e-6


@pytest.mark.parametrize("A,matter,nmax,twist", [
    (2, "pnm", 2, (0.0, 0.0, 0.0)), (14, "pnm", 1, (0.0, 0.0, 0.0)), (15, "pnm", 1, (0.3, 0.6, 0.9)),
    (38, "pnm", 2, (0.5, 1.0, 1.5)), (54, "pnm", 2, (0.0, 0.0, 0.0)), (66, "pnm", 4, (0.0, 0.0, 0.0)),
    (162, "pnm", 3, (0.0, 0.0, 0.0)), (246, "pnm", 3, (0.2, 0.4, 0.6)), (28, "snm", 2, (0.0, 0.0, 0.0)),
    (228, "snm", 3, (0.0, 0.0, 0.0))])
def test_fp64_contraction_tiles_equal_list_kernels(ccnm, monkeypatch, A, matter, nmax, twist):
    """X, I9, the hh ladder and the fused ring against the grouped list kernels
    over the classes of their tiles: ring sides 4, 16, 18, 60 (sides that
    differ by up to 16), 76, 128, 172, 212 (differing by up to 40) and 296, past
    the fused kernel; 1 to 245 hole pairs.  Both sum the same products, k in
    another order: each contraction rounds by at most 2^-53 (K + 8) times four
    (three-product complex terms) of its sum of moduli, K at most 1144, so
    6e-13 of it; the amplitudes after two steps without extrapolation are such
    sums over denominators above 1, and a lost k would be 1e-3 of one."""
    out = []
    for lists in (False, True):
        if lists:
            monkeypatch.setenv("CCGPU_SPLIT_K", "256")   # the lists' own default; they run as soon as one is asked for
        s = ccnm.Solver(A=A, matter=ccnm.PNM if matter == "pnm" else ccnm.SNM, rho=0.16, nmax=nmax, twist=twist)
        s.generate_interaction(ccnm.INT_MINNESOTA)
        s.setup_t_amplitudes()
        for _ in range(2):
            s.t2_intermediate()
            s.diis_t1t2(1, 1)
        out.append(s.t2_unique())
        s.close()
    t, ref = out
    assert np.all(np.isfinite(ref)) and np.abs(ref).max() > 0
    assert np.abs(t - ref).max() <= 1e-12 * np.abs(ref).max()


@pytest.mark.parametrize("A,nmax,precision,graph", [
    (2, 2, 0, 0), (14, 1, 0, 1), (14, 1, 3, 0), (66, 2, 3, 1), (66, 3, 0, 0), (66, 3, 3, 0)])
def test_solve_loop_forms_the_iterates_of_the_step_interface(ccnm, A, nmax, precision, graph):
    """The solve loop leaves each iterate to the next residual's opening pass and
    updates inside the closing one; the step interface runs residual and update
    apart, on T in place.  248 to 720540 amplitudes: fewer than a block, less
    and more than one trip of the grids (524288).  Both add the same terms in
    the same order; 1e-13 of the largest amplitude leaves three iterations of
    contracted or separate roundings (2^-53 each) a factor of hundreds."""
    out = []
    for steps in (False, True):
        s = ccnm.Solver(A=A, matter=ccnm.PNM, rho=0.16, nmax=nmax)
        s.generate_interaction(ccnm.INT_MINNESOTA)
        s.setup_t_amplitudes()
        if steps:
            count = nstep = 0
            for _ in range(3):
                s.t2_intermediate(precision)
                count, nstep = s.diis_t1t2(count + 1, nstep + 1, 6, 6)
            e = s.ccd_energy_save()
        else:
            r = s.ccd_iter(subspace=6, diis_step=6, tol=0.0, maxit=3, precision=precision, fp32_switch=0.0,
                           use_graph=graph)
            assert r["iterations"] == 3
            e = r["ecorr"]
        out.append((s.t2_unique(), e))
        s.close()
    (t, e), (t0, e0) = out
    assert np.all(np.isfinite(t0)) and np.abs(t0).max() > 0
    assert np.abs(t - t0).max() <= 1e-13 * np.abs(t0).max()
    assert abs(e - e0) <= 1e-12 * abs(e0)


@pytest.mark.parametrize("A,matter,nmax,twist", [
    (3, "pnm", 1, (0.0, 0.0, 0.0)), (15, "pnm", 1, (0.5, 1.0, 1.5)), (6, "snm", 1, (0.0, 0.0, 0.0)),
    (14, "pnm", 1, (0.5, 1.0, 1.5)), (38, "pnm", 2, (0.0, 0.0, 0.0))])
@pytest.mark.parametrize("lists", [False, True])
def test_ring_of_channel_pairs_equals_oracle(ccnm, monkeypatch, A, matter, nmax, twist, lists):
    """The ring is contracted in one of the channels K', -K' of each pair.  A = 3, 6
    and 15 leave a momentum half filled, so K' = 0 is its own pair.  The oracle
    contracts every channel in 64 bits; 1e-12 of the largest element as in
    test_residual_terms_elementwise_nmax2.  T~, W0 and R~ of all channels come back
    through the debug arrays: R~ as T~ (W0 + 1/2 V~ T~) channel by channel."""
    import ccd_oracle as co
    import chiral_oracle as ch
    lat = co.Lattice.build(A, matter, 0.16, nmax, twist)
    cc = co.CCD(lat, ch.ChiralInteraction(lat, ch.NNLO, 450.0))
    s = ccnm.Solver(A=A, matter=ccnm.PNM if matter == "pnm" else ccnm.SNM, rho=0.16, nmax=nmax, twist=twist)
    s.set_chiral(ccnm.NNLO, 450.0)
    s.generate_interaction(ccnm.INT_CHIRAL)
    s.setup_t_amplitudes()
    s.t2_intermediate()
    s.diis_t1t2(1, 1)
    t, lab = s.t2_unique(), s.t2_labels()
    a, b, i, j = lab.T
    x = np.zeros(cc.ch.size, np.complex128)
    for (p, q, r_, u), sg in (((a, b, i, j), 1.0), ((b, a, i, j), -1.0), ((a, b, j, i), -1.0), ((b, a, j, i), 1.0)):
        x[cc.ch.flat_index(p, q, r_, u)] = sg * t
    R = cc.flat(cc.residual(cc.unflat(x), 8)[0])[cc.ch.flat_index(a, b, i, j)]
    monkeypatch.setenv("CCGPU_TERMS", "8")
    if lists:
        monkeypatch.setenv("CCGPU_SPLIT_K", "256")
    s.t2_intermediate()
    got = s.debug_fetch("R", len(t))
    assert np.abs(got - R).max() <= 1e-12 * np.abs(R).max()
    n = s.dims["ring_elems"]
    tt, rt = s.debug_fetch("Tt", n), s.debug_fetch("Rt", n)
    r0 = s.debug_fetch("R0", len(t))
    # every amplitude stands in four places of T~
    assert abs(np.sum(np.abs(tt) ** 2) - 4 * np.sum(np.abs(t) ** 2)) <= 1e-12 * np.sum(np.abs(tt) ** 2)
    # sum over the ordered amplitudes of conj(t) (R - conj V) = sum of conj(T~) R~
    want = 4 * np.sum(np.conj(t) * (R - r0))
    assert abs(4 * np.sum(np.conj(tt) * rt) - want) <= 1e-11 * np.sum(np.abs(tt) * np.abs(rt))
    s.close()


@pytest.mark.parametrize("A,matter,nmax,twist", [
    (3, "pnm", 1, (0.0, 0.0, 0.0)), (15, "pnm", 1, (0.3, 0.6, 0.9)), (28, "snm", 2, (0.0, 0.0, 0.0)),
    (66, "pnm", 3, (0.9, 1.35, 1.8)), (108, "snm", 2, (0.0, 0.0, 0.0)), (246, "pnm", 3, (0.2, 0.4, 0.6))])
def test_bf16x3_fused_ring_equals_list_kernels(ccnm, monkeypatch, A, matter, nmax, twist):
    """The BF16x3 ring in one launch against the list kernels: channels of 1 to
    above 256 rows, at most 4 hp pairs, odd counts, one that is its own pair.  Both sum
    the same split products in FP32, k at most some 500 a contraction and two of
    them nested: 2 (2 K + 4) 2^-24 = 1.2e-4 of the sum of moduli, which the largest
    element of the ring bounds within a factor of ten on these amplitudes, and
    rounding errors of that many terms add up to a thirtieth of their bound: 4e-5 of
    the largest element.  A lost k would be 1/256 and more of an element."""
    monkeypatch.setenv("CCGPU_TERMS", "8")
    out = []
    for lists in (False, True):
        if lists:
            monkeypatch.setenv("CCGPU_SPLIT_K", "256")
        s = ccnm.Solver(A=A, matter=ccnm.PNM if matter == "pnm" else ccnm.SNM, rho=0.16, nmax=nmax, twist=twist)
        s.set_chiral(ccnm.NNLO, 450.0)
        s.generate_interaction(ccnm.INT_CHIRAL)
        s.setup_t_amplitudes()
        s.t2_intermediate(ccnm.PREC_BF16X3)
        n = s.dims["t2_unique"]
        out.append(s.debug_fetch("R", n) - s.debug_fetch("R0", n))
        s.close()
    r, ref = out
    assert np.all(np.isfinite(ref)) and np.abs(ref).max() > 0
    assert np.abs(r - ref).max() <= 4e-5 * np.abs(ref).max()


@pytest.mark.parametrize("A,matter,nmax,twist,order", [
    (3, "pnm", 1, (0.0, 0.0, 0.0), "NNLO"), (15, "pnm", 1, (0.3, 0.6, 0.9), "NNLO"), (14, "pnm", 1, (0.0, 0.0, 0.0), "LO"),
    (6, "snm", 1, (0.0, 0.0, 0.0), "NNLO"), (28, "snm", 1, (0.2, 0.4, 0.6), "LO"), (4, "snm", 1, (0.5, 1.0, 1.5), "NNLO")])
def test_chiral_blocks_over_pair_groups_equal_elements(ccnm, monkeypatch, A, matter, nmax, twist, order):
    """The V fill takes the sixteen spin combinations of two pair groups at once; single
    elements come from the general evaluation.  Groups of one to four pairs, with and
    without isospin exchange.  Both round the same few dozen operations: 64 * 2^-53 of
    the largest element, 1e-14."""
    s = ccnm.Solver(A=A, matter=ccnm.PNM if matter == "pnm" else ccnm.SNM, rho=0.16, nmax=nmax, twist=twist)
    s.set_chiral(getattr(ccnm, order), 450.0)
    s.generate_interaction(ccnm.INT_CHIRAL)
    o, nt = s.orbitals(), s.dims["t2_unique"]
    a, b, i, j = s.t2_labels().T
    want = np.conj(s.vnn_elements(i, j, a, b))
    got = s.debug_fetch("R0", nt)
    scale = np.abs(want).max()
    assert np.abs(got - want).max() <= 1e-14 * scale
    # W0((i,a),(j,b)) = -<ib||ja>, channels by (tz, n) of j - b, hp pairs by j and then b
    key = {}
    for h in range(A):
        for p in range(A, s.dims["nsp"]):
            key.setdefault((o["tz"][h] - o["tz"][p], *(o[x][h] - o[x][p] for x in ("nx", "ny", "nz"))), []).append((h, p))
    want = []
    for k in sorted(key):
        if tuple(-x for x in k) not in key:
            continue
        hp = np.array(key[k], np.int32)
        r, c = np.meshgrid(np.arange(len(hp)), np.arange(len(hp)), indexing="ij")
        r, c = r.ravel(), c.ravel()
        want.append(-s.vnn_elements(hp[r, 0], hp[c, 1], hp[c, 0], hp[r, 1]))
    want = np.concatenate(want)
    got = s.debug_fetch("W0", len(want))
    assert np.abs(got - want).max() <= 1e-14 * np.abs(want).max()
    # V_pppp through the pp ladder of random amplitudes
    rng = np.random.default_rng(A)
    t = rng.standard_normal(nt) + 1j * rng.standard_normal(nt)
    s.set_t2_unique(t)
    monkeypatch.setenv("CCGPU_TERMS", "2")
    s.t2_intermediate()
    R = s.debug_fetch("R", nt) - s.debug_fetch("R0", nt)
    at = {}
    for u in range(nt):
        at.setdefault((i[u], j[u]), []).append(u)
    err = top = 0.0
    for us in at.values():
        us = np.array(us)
        r, c = np.meshgrid(us, us, indexing="ij")
        v = s.vnn_elements(a[r].ravel(), b[r].ravel(), a[c].ravel(), b[c].ravel()).reshape(r.shape)
        err, top = max(err, np.abs(R[us] - v @ t[us]).max()), max(top, (np.abs(v) @ np.abs(t[us])).max())
    assert err <= 1e-14 * top
    s.close()


@pytest.mark.parametrize("A,matter,nmax", [(2, "pnm", 1), (14, "pnm", 1), (28, "snm", 2), (38, "pnm", 3), (66, "pnm", 3)])
def test_amplitudes_come_back_whole(ccnm, A, matter, nmax):
    """The copy to host memory goes through pinned halves of 4 MB in pieces of 256 KB: less
    than a piece, some pieces, two and three halves with a ragged end."""
    s = ccnm.Solver(A=A, matter=ccnm.PNM if matter == "pnm" else ccnm.SNM, rho=0.16, nmax=nmax)
    n = s.dims["t2_unique"]
    rng = np.random.default_rng(n)
    for _ in range(3):
        t = rng.standard_normal(2 * n).view(np.complex128)
        s.set_t2_unique(t)
        assert np.array_equal(s.t2_unique(), t)
        assert np.array_equal(s.t2_unique(), s.debug_fetch("T", n))
    s.close()
