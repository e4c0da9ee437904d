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
