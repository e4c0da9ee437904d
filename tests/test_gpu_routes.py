"""Calls that can take one of several kernels, tables or copies: each route
gives what the others give, and what a route needs is made when it is taken."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_ccdt1 import native_3nf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("A,matter,nmax,twist", [(4, "snm", 1, (0.0, 0.0, 0.0)), (14, "pnm", 1, (0.4, 0.9, 1.3))])
def test_in_place_triples_switch_keeps_the_three_body_force(ccnm, monkeypatch, A, matter, nmax, twist):
    """CCGPU_T3_KERNEL=0 asks for the kernel without tables, which evaluates
    |W|^2 with the two-nucleon elements alone: (T) with the normal-ordered
    three-nucleon force, (T) with W3 and the CCDT-1 energy are the same with
    the switch and without it (the same terms, 1e-12 for their order)."""
    for approx in (2, 3):
        s = native_3nf(ccnm, A, matter, 0.16, nmax, twist, approx)
        s.setup_t_amplitudes()
        got = []
        for kernel in (None, "0"):
            if kernel is None:
                monkeypatch.delenv("CCGPU_T3_KERNEL", raising=False)
            else:
                monkeypatch.setenv("CCGPU_T3_KERNEL", kernel)
            v = [s.pert_triples2(), *s.triples_parts(), s.setup_t3()]
            s.t3_intermediate()
            got.append(np.array(v + [s.t3_energy()]))
        assert np.all(got[0][[0, 1, 3, 4]] != 0)
        assert np.max(np.abs(got[1] - got[0])) <= 1e-12 * np.max(np.abs(got[0])), got


def test_refused_allocation_leaves_the_next_call_alone(ccnm):
    """An allocation that the card refuses is an error of that call only: the
    runtime's record of it is not taken for one of a later launch."""
    s = ccnm.Solver(A=14, matter=ccnm.PNM, rho=0.16, nmax=1)
    with pytest.raises(RuntimeError, match="hipMalloc"):
        ccnm.hbm_read_probe(1 << 48, 1)
    s.generate_interaction()
    assert s.setup_t_amplitudes() != 0


@pytest.mark.parametrize("kernel", [None, "1"])
def test_triples_after_a_refused_table_allocation(ccnm, monkeypatch, kernel):
    """A card without room for the tables of (T): the call fails, and the next
    one, with room again, makes all of them and gives the same sum.  PNM A=38
    |n_i|<=1 has more hole than particle groups, so the second group table
    (390 kB) is the larger one."""
    def solver():
        s = native_3nf(ccnm, 38, "pnm", 0.16, 1, (0.0, 0.0, 0.0), 2)
        s.setup_t_amplitudes()
        return s
    if kernel:
        monkeypatch.setenv("CCGPU_T3_KERNEL", kernel)
    want = solver().pert_triples2()
    s = solver()
    monkeypatch.setenv("CCGPU_FORCE_NOMEM", "300000")
    for _ in range(2):
        with pytest.raises(RuntimeError, match="hipMalloc of .* bytes failed"):
            s.pert_triples2()
    monkeypatch.delenv("CCGPU_FORCE_NOMEM")
    assert want != 0 and s.pert_triples2() == want


def device_memory_free():
    rt = C.CDLL("libamdhip64.so.7")
    free, total = C.c_size_t(), C.c_size_t()
    assert rt.hipDeviceSynchronize() == 0
    assert rt.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def polarised(ccnm, A, nmax, both=0):
    """Neutrons of spin up in a box at 0.16 fm^-3, the lowest `both` states with
    their spin-down partners: a table handed over orbital by orbital."""
    n = range(-nmax, nmax + 1)
    up = sorted((x * x + y * y + z * z, x, y, z, 1) for x in n for y in n for z in n)
    st = sorted(up + [(*q[:4], -1) for q in up[:both]])
    box = (A / 0.16) ** (1 / 3)
    f = 2 * np.pi / box
    q = np.array(st)
    o = dict(A=A, nx=q[:, 1], ny=q[:, 2], nz=q[:, 3], sz=q[:, 4], tz=np.ones(len(st)), kx=f * q[:, 1], ky=f * q[:, 2],
             kz=f * q[:, 3], e=197.326968 ** 2 / (2 * 939.565) * f * f * q[:, 0], box=box, volume=box ** 3)
    s = ccnm.Solver(orbitals=o)
    s.set_chiral(ccnm.NNLO, 450.0)
    s.set_3nf(3)
    s.generate_interaction(ccnm.INT_CHIRAL)
    s.setup_t_amplitudes()
    return s


@pytest.mark.parametrize("A,nmax,both", [(19, 1, 0), (27, 2, 0), (38, 2, 19), (7, 1, 0)])
def test_triples_of_spin_polarised_tables_by_every_kernel(ccnm, monkeypatch, A, nmax, both):
    """One spin state per momentum (few and many hole triples per channel) and
    both for the holes alone: the sums over groups, element by element and by
    the rule's own choice are sums of the same terms (1e-12 for their order;
    the sums have one sign per element, W some cancellation inside)."""
    s = polarised(ccnm, A, nmax, both)
    got = {}
    for kernel in (None, "2", "1", "3"):
        if kernel is None:
            monkeypatch.delenv("CCGPU_T3_KERNEL", raising=False)
        else:
            monkeypatch.setenv("CCGPU_T3_KERNEL", kernel)
        et = s.pert_triples2()
        n = s.triples_stats()[0]
        v = [et, *s.triples_parts(), s.setup_t3()]
        s.t3_intermediate()
        got[kernel] = np.array(v + [s.t3_energy(), n])
    assert np.all(got["2"] != 0)
    for kernel in (None, "1", "3"):
        assert got[kernel][-1] == got["2"][-1]
        assert np.all(np.abs(got[kernel] - got["2"]) <= 1e-12 * np.abs(got["2"])), got


def test_triples_tables_of_spin_polarised_matter_stay_within_their_budget(ccnm, monkeypatch):
    """A=33 |n_i|<=3, one spin state per momentum: dense tables of 113 MB, group
    tables of four times that.  (T) makes the dense ones, by its own choice and
    where groups are asked for in a budget that has no room for theirs."""
    s = polarised(ccnm, 33, 3)
    np_ = s.dims["nparticles"]
    dense = 32 * (np_ * np_ * 33 + 2 * 33 * 33 * np_)
    s.set_3nf(2)   # (T) without W3
    monkeypatch.setenv("CCGPU_T3_TABLE_GB", str(1.5 * dense / 1e9))
    monkeypatch.setenv("CCGPU_T3_KERNEL", "2")
    before = device_memory_free()
    first = s.pert_triples2()
    assert before - device_memory_free() < 1.5 * dense
    monkeypatch.delenv("CCGPU_T3_KERNEL")
    monkeypatch.delenv("CCGPU_T3_TABLE_GB")
    assert s.pert_triples2() == first
    assert before - device_memory_free() < 1.5 * dense


def ring_channel(o, x, y):
    """Pandya channel of n_x - n_y, its sign dropped: the channel pair's key."""
    k = tuple(int(o[q][x] - o[q][y]) for q in ("tz", "nx", "ny", "nz"))
    return max(k, tuple(-v for v in k))


@pytest.mark.parametrize("lists", [False, True])
@pytest.mark.parametrize("prec", ["PREC_BF16X3", "PREC_FP32"])
def test_thin_ring_channels_stay_in_fp64_arithmetic(ccnm, monkeypatch, prec, lists):
    """Channel pairs with at most four pairs on either side are contracted in
    FP64 arithmetic under the low precisions (BF16x3: on FP32 blocks).  With one
    amplitude the ring of its channel pair is single products V t away from
    the amplitude itself, so the residual equals the FP64 one to the roundings
    of V, t and the product to FP32 (3 x 2^-24, and 2^-24 for their products), or
    to those of FP64 where the blocks are FP64; split products are off by
    2^-18 to 2^-16."""
    monkeypatch.setenv("CCGPU_TERMS", "8")
    if lists:   # the list kernels in place of the fused ring, at the default split
        monkeypatch.setenv("CCGPU_SPLIT_TILES", "128")
    s = ccnm.Solver(A=14, matter=ccnm.PNM, rho=0.16, nmax=1, twist=(0.5, 1.2, 2.2))
    s.set_chiral(ccnm.NNLO, 450.0)
    s.generate_interaction(ccnm.INT_CHIRAL)
    s.setup_t_amplitudes()
    o, A = s.orbitals(), s.dims["nholes"]
    lab = s.t2_labels()
    size = {}   # (particle, hole) pairs of n_a - n_i = k and of -k
    for a in range(A, s.dims["nsp"]):
        for i in range(A):
            k = tuple(int(o[q][a] - o[q][i]) for q in ("tz", "nx", "ny", "nz"))
            key = max(k, tuple(-v for v in k))
            size.setdefault(key, [0, 0])[0 if k == key else 1] += 1
    thin = {k for k, v in size.items() if min(v) <= 4 < max(v)}
    plus = [ring_channel(o, a, i) for a, b, i, j in lab]
    minus = [ring_channel(o, b, i) for a, b, i, j in lab]
    bound = 4 * 2.0 ** -24 if prec == "PREC_BF16X3" else 8 * 2.0 ** -53
    checked = set()
    for k in sorted(thin):
        u = plus.index(k) if k in plus else None
        if u is None:
            continue
        t = np.zeros(len(lab), np.complex128)
        t[u] = 0.7390851332151607 + 0.5671432904097838j
        r = []
        for p in (ccnm.PREC_FP64, getattr(ccnm, prec)):
            s.set_t2_unique(t)
            s.t2_intermediate(p)
            r.append(s.debug_fetch("R", len(lab)) - s.debug_fetch("R0", len(lab)))
        own = (k, minus[u])
        for v in range(len(lab)):
            if v != u and plus[v] == k and minus[v] not in own and abs(r[0][v]) > 1e-8:
                assert abs(r[1][v] - r[0][v]) <= bound * abs(r[0][v]) + 2.0 ** -50 * abs(t[u]), (k, v, r[0][v], r[1][v])
                checked.add(k)
    assert len(checked) >= 3, checked   # the channel pairs of this lattice with such elements


def test_low_precision_after_a_refused_allocation(ccnm, monkeypatch):
    """A card with room for the FP32 copy of V_pppp and not for what comes with
    it: the residual fails, and the next one, with room again, equals that of a
    handle that was never refused (no copy is taken for filled).  PNM A=38
    |n_i|<=1 has fewer particle than hole pairs, so its split T is the larger."""
    def solver():
        s = ccnm.Solver(A=38, matter=ccnm.PNM, rho=0.16, nmax=1)
        s.generate_interaction()
        s.setup_t_amplitudes()
        return s
    want = solver()
    want.t2_intermediate(ccnm.PREC_BF16X3)
    n = want.dims["t2_unique"]
    s = solver()
    assert 8 * s.dims["vpppp_unique"] * 1.2 < 16 * n
    monkeypatch.setenv("CCGPU_FORCE_NOMEM", str(16 * n))
    for _ in range(2):
        with pytest.raises(RuntimeError, match="hipMalloc of .* bytes failed"):
            s.t2_intermediate(ccnm.PREC_BF16X3)
    monkeypatch.delenv("CCGPU_FORCE_NOMEM")
    s.t2_intermediate(ccnm.PREC_BF16X3)
    r = want.debug_fetch("R", n)
    assert np.all(np.isfinite(r)) and np.any(r != 0)
    assert np.array_equal(s.debug_fetch("R", n), r)


def test_network_after_a_refused_allocation(ccnm, monkeypatch):
    """A minibatch and a training set that the card has no room for leave the
    network as it was: the steps before and after are those of one that was
    never refused."""
    s = ccnm.Solver(A=14, matter=ccnm.PNM, rho=0.16, nmax=1)
    s.generate_interaction()
    s.setup_t_amplitudes()
    s.ccd_iter()
    nets = [ccnm.WarmStart(seed=3) for _ in range(2)]
    n = s.dims["t2_unique"]
    for net in nets:
        net.add_solve(s)
        net.train(2, batch=64, seed=5)
    monkeypatch.setenv("CCGPU_FORCE_NOMEM", str(4 * n))
    with pytest.raises(RuntimeError, match="hipMalloc of .* bytes failed"):
        nets[1].add_solve(s)
    with pytest.raises(RuntimeError, match="hipMalloc of .* bytes failed"):
        nets[1].train(1, batch=1 << 20, seed=5)
    monkeypatch.delenv("CCGPU_FORCE_NOMEM")
    for net in nets:
        net.train(2, batch=64, seed=6)
        net.add_solve(s)
        net.train(2, batch=128, seed=7)
    assert np.array_equal(nets[0].params, nets[1].params)


def pnm66_n3(ccnm):
    s = ccnm.Solver(A=66, matter=ccnm.PNM, rho=0.16, nmax=3)   # 11.5 MB of amplitudes
    s.generate_interaction()
    s.setup_t_amplitudes()
    return s


def test_amplitudes_into_every_kind_of_memory(ccnm):
    """ccgpu_get_t2_unique into pageable, pinned and device memory, and into
    none, which is an error: the route through pinned halves is for host memory."""
    rt = C.CDLL("libamdhip64.so.7")
    s = pnm66_n3(ccnm)
    want = s.t2_unique()
    get = ccnm.lib().ccgpu_get_t2_unique
    got = np.empty_like(want)
    for alloc, free in (("hipMalloc", "hipFree"), ("hipHostMalloc", "hipHostFree")):
        p = C.c_void_p()
        args = (C.byref(p), C.c_size_t(want.nbytes)) + ((C.c_uint(0),) if alloc == "hipHostMalloc" else ())
        assert getattr(rt, alloc)(*args) == 0
        assert get(s.h, C.cast(p, C.POINTER(C.c_double))) == 0
        assert rt.hipMemcpy(C.c_void_p(got.ctypes.data), p, C.c_size_t(want.nbytes), C.c_int(4)) == 0
        assert getattr(rt, free)(p) == 0
        assert np.any(want != 0) and np.array_equal(got, want), alloc
        got[:] = 0
    assert get(s.h, C.POINTER(C.c_double)()) != 0
    assert np.array_equal(s.t2_unique(), want)


def test_amplitudes_of_a_handle_on_a_second_gpu(ccnm):
    """Large copies to host memory from handles on two devices of one process."""
    rt = C.CDLL("libamdhip64.so.7")
    n = C.c_int()
    assert rt.hipGetDeviceCount(C.byref(n)) == 0
    if n.value < 2:
        pytest.skip("one GPU")
    got = []
    try:
        for dev in (0, 1):
            assert rt.hipSetDevice(dev) == 0
            got.append(pnm66_n3(ccnm))
        for dev in (1, 0):   # also with the other device current
            assert rt.hipSetDevice(dev) == 0
            a, b = (s.t2_unique() for s in got)
            assert np.any(a != 0) and np.array_equal(a, b)
    finally:
        rt.hipSetDevice(0)


def test_generating_again_takes_no_more_device_memory(ccnm):
    """A scan over the constants of the interaction on one handle: its tables
    (of the lattice's size: 20 kB of radial functions at |n_i|<=2, side factors,
    parity images of the orbitals) are written again, not added."""
    s = ccnm.Solver(A=2, matter=ccnm.PNM, rho=0.16, nmax=2)
    def generate(k):
        s.set_chiral(ccnm.NNLO, 450.0, ci=(-0.74, -0.49 - 1e-3 * k, -0.65, 0.96))
        s.set_3nf(0)
        s.generate_interaction(ccnm.INT_CHIRAL)
    generate(0)
    before = device_memory_free()
    for k in range(1, 513):
        generate(k)
    assert before - device_memory_free() < 4 << 20


def test_low_precision_solve_tunes_only_lists_that_it_launches(ccnm):
    """A BF16x3 solve contracts X and the hh ladder on its own lists, the ring in
    one launch, and its FP64 iterations outside the pp ladder on tiles that need
    no tuning: no time goes to shapes of the lists these replace."""
    s = ccnm.Solver(A=14, matter=ccnm.PNM, rho=0.16, nmax=2, twist=(0.31, 1.27, 2.03))
    s.generate_interaction()
    s.setup_t_amplitudes()
    seen = len(ccnm.autotune_report())
    r = s.ccd_iter(precision=ccnm.PREC_BF16X3, fp32_switch=1e-3)
    assert r["converged"] and r["fp32_iterations"] < r["iterations"]
    tuned = {x.split(":")[0].strip() for x in ccnm.autotune_report()[seen:].split(";") if x.strip()}
    assert "fam10/kind6" in tuned   # X under BF16x3
    dead = {f"fam{f}/kind0" for f in (0, 2, 3, 4)} | {f"fam{f}/kind6" for f in (13, 14)}
    assert not tuned & dead, tuned


@pytest.mark.parametrize("A,matter,nmax", [(28, "snm", 2), (54, "pnm", 3)])
def test_residual_launches_give_the_same_bits(ccnm, monkeypatch, A, matter, nmax):
    """Below 400 k amplitudes an FP64 residual runs in merged launches on one
    stream, above it on three; CCGPU_FORK=0 keeps one stream, CCGPU_TIMING=1 one
    launch after another: the same tiles and sums, so the same bits."""
    s = ccnm.Solver(A=A, matter=ccnm.PNM if matter == "pnm" else ccnm.SNM, rho=0.16, nmax=nmax)
    assert (s.dims["t2_unique"] < 400000) == (nmax == 2)
    s.generate_interaction()
    got = []
    for env in (None, "CCGPU_FORK", "CCGPU_TIMING"):
        with monkeypatch.context() as m:
            if env:
                m.setenv(env, "0" if env == "CCGPU_FORK" else "1")
            s.setup_t_amplitudes()
            s.ccd_iter(subspace=4, diis_step=4, tol=1e-30, maxit=3)
            got.append(s.t2_unique())
    assert np.any(got[0] != 0)
    for t in got[1:]:
        assert np.array_equal(t, got[0])
