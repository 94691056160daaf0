"""The per-term kernels (stencil, projection, fused KB pass, KB scatter) on cells small enough for the
whole-orbital kernels, which a launch shape set by hand selects: few orbitals of many projectors, where the
KB scatter and the fused KB pass take another form, against the CPU oracle.

Tolerances as elsewhere: 1e-12 relative on H psi and one FP64 Taylor step (sums of a few hundred products),
1e-6 on a step of the complex-FP32 chain."""
import numpy as np
import pytest

from salmon2_amd import system

pytestmark = pytest.mark.gpu

A = np.array([0.013, -0.021, 0.007])


def rel(a, b):
    a, b = np.asarray(a), np.asarray(b)
    return float(np.abs(a - b).max() / np.abs(b).max())


def per_term(s):
    """Handle of s with the per-term kernels, phase table of A."""
    import torch

    assert torch.cuda.is_available(), "GPU tests need a visible MI355X"
    from salmon2_amd.hip import Handle

    h = Handle(s, stream=torch.cuda.current_stream())
    h._set_shape(0, 0)
    h.update_kvector(A)
    return h


def check_step(oracle_lib, s, what):
    import torch

    h = per_term(s)
    O = oracle_lib.Oracle(s)
    O.update_kvector(A)
    psi = torch.from_numpy(s.psi).cuda()
    out, work = torch.zeros_like(psi), torch.zeros_like(psi)
    ny = s.ny
    h.hpsi(psi, out)
    assert rel(out.cpu().numpy()[..., :ny, :], O.hpsi(A, s.psi)[..., :ny, :]) <= 1e-12
    ref = O.taylor(A, s.psi)[0][..., :ny, :]
    for prec, tol in (("fp64", 1e-12), ("mixed", 1e-6)):
        if prec == "mixed" and s.n_hamil < 2:
            continue
        h.set_precision(prec)
        h.taylor(s.zc(), psi, out, work)
        e = rel(out.cpu().numpy()[..., :ny, :], ref)
        print(f"[parity] per-term {what} {prec}: {e:.2e}", flush=True)
        assert e <= tol
    h.close()


# 4 and 5 orbitals: the last count of the scatter's plain form and the first of the other; two spins
# make two orbital blocks of each
@pytest.mark.parametrize("no,nspin", [(1, 1), (2, 2), (3, 2), (4, 1), (5, 1), (9, 1)])
@pytest.mark.parametrize("lmax,rcut", [(2, 3.6), (3, 2.2)])
def test_few_orbitals(oracle_lib, no, nspin, lmax, rcut):
    print(f"[gpu] per-term few orbitals no={no} nspin={nspin} lmax={lmax}", flush=True)
    s = system.make_si_system(n=(13, 12, 11), no=no, nspin=nspin, lmax=lmax, rcut=rcut, nkgrid=(1, 1, 2), seed=311)
    check_step(oracle_lib, s, f"no={no} nspin={nspin} lmax={lmax}")


@pytest.mark.parametrize("nos", [(3, 4), (4, 6)])
def test_batch_few_orbitals(oracle_lib, nos):
    """A batch with d projectors whose members all take the plain scatter, and one with a member that does not."""
    from salmon2_amd.batch import BatchRunner

    nt = 3
    print(f"[gpu] per-term batch of {nos} orbitals, lmax 2", flush=True)
    systems = [system.make_si_system(n=12 + i, no=no, lmax=2, seed=331 + i, nt=nt) for i, no in enumerate(nos)]
    br = BatchRunner(systems, nt)
    br.run(nt)
    got = br.results(nt)
    br.close()
    for s, g in zip(systems, got):
        _, cur, dip, rne = oracle_lib.Oracle(s).rt_run(nt=nt, psi=s.psi)
        for k, ref in (("curr", cur), ("dip", dip), ("rne", rne)):
            assert rel(g[k], ref) <= 1e-9, k


@pytest.mark.parametrize("whole", [True, False])
@pytest.mark.parametrize("nk,lmax", [((1, 1, 1), 0), ((1, 3, 5), 3), ((1, 2, 8), 2), ((1, 2, 8), 3), ((1, 1, 17), 1)])
def test_phase_table_blocks(oracle_lib, nk, lmax, whole):
    """The phase table by projector (below 128 atoms x k: 8 x 15) and by atom (from 8 x 16 on), as H psi reads it:
    its per-point form in the projections and its per-entry form in the scatter and the shared points."""
    import torch

    from salmon2_amd.hip import Handle

    print(f"[gpu] phase table k={nk} lmax={lmax} whole={whole}", flush=True)
    s = system.make_si_system(n=(12, 11, 13), no=1, lmax=lmax, rcut=3.6, nkgrid=nk, seed=347)
    h = Handle(s, stream=torch.cuda.current_stream())
    if not whole:
        h._set_shape(0, 0)
    O = oracle_lib.Oracle(s)
    psi = torch.from_numpy(s.psi).cuda()
    out = torch.zeros_like(psi)
    cur = torch.zeros(3, dtype=torch.float64, device="cuda")
    for a in (A, -2.0 * A):
        h.update_kvector(a)
        O.update_kvector(a)
        h.hpsi(psi, out)
        ref = O.hpsi(a, s.psi)[..., : s.ny, :]
        assert rel(out.cpu().numpy()[..., : s.ny, :], ref) <= 1e-12
    h.current_next(a, psi, cur, A)  # the table of A built ahead
    h.update_kvector(A)
    O.update_kvector(A)
    h.hpsi(psi, out)
    assert rel(out.cpu().numpy()[..., : s.ny, :], O.hpsi(A, s.psi)[..., : s.ny, :]) <= 1e-12
    h.close()


# points covered by up to two and up to ten (atom, point) pairs, and up to 16 projectors per atom
@pytest.mark.parametrize("kw", [
    dict(n=12, no=4, nkgrid=(1, 1, 2), rcut=3.6, seed=23),
    dict(n=12, no=4, nkgrid=(1, 1, 2), rcut=5.3, seed=23),
    dict(n=12, no=9, rcut=5.3, lmax=2, seed=23),
    dict(n=14, no=5, nkgrid=(1, 1, 2), seed=59, lmax=3),
    dict(n=12, no=17, rcut=5.3, lmax=3, seed=61),
])
def test_covered_points(oracle_lib, kw):
    import torch

    print(f"[gpu] per-term covered points {kw}", flush=True)
    s = system.make_si_system(**kw)
    check_step(oracle_lib, s, str(kw))
    h = per_term(s)
    psi = torch.from_numpy(s.psi).cuda()
    cur = torch.zeros((s.nspin, 3), dtype=torch.float64, device="cuda")
    h.current(A, psi, cur)
    O = oracle_lib.Oracle(s)
    O.update_kvector(A)
    assert rel(cur.cpu().numpy(), O.current(A, s.psi)) <= 1e-9
    h.close()


@pytest.mark.parametrize("n_hamil", [1, 2, 3, 5, 6])
def test_orders(oracle_lib, n_hamil):
    """Chains of 0 .. 5 fused KB passes."""
    print(f"[gpu] per-term order {n_hamil}", flush=True)
    check_step(oracle_lib, system.make_si_system(n=12, no=4, nkgrid=(1, 1, 2), rcut=3.6, seed=29, n_hamil=n_hamil),
               f"order {n_hamil}")


@pytest.mark.parametrize("lmax", [1, 3])
def test_prepared_projection(lmax):
    """current_next's projection of psi is the one that the next step uses, bit for bit, and is discarded under
    any other field than the one it was formed for."""
    import torch

    from salmon2_amd.hip import Handle

    print(f"[gpu] per-term prepared projection lmax={lmax}", flush=True)
    s = system.make_si_system(n=12, no=4, nkgrid=(1, 1, 2), lmax=lmax, seed=7)
    h = Handle(s, stream=torch.cuda.current_stream())
    h._set_shape(0, 0)
    psi = torch.from_numpy(s.psi).cuda()
    cur = torch.zeros(3 * s.nspin, dtype=torch.float64, device="cuda")
    B = np.array([0.02, -0.01, 0.0])

    def step():
        out, work = torch.zeros_like(psi), torch.zeros_like(psi)
        h.prof_start(64)
        h.taylor(s.zc(), psi, out, work)
        n = h.prof_read("proj")[1]
        h.prof_end()
        return n, out

    h.update_kvector(A)
    n, plain = step()
    assert n == 1  # the first term's projection; the others are fused with the KB pass before
    h.update_kvector(B)
    h.current_next(B, psi, cur, A)
    h.update_kvector(A)
    n, out = step()
    assert n == 0 and torch.equal(out, plain)
    h.current_next(A, psi, cur, B)
    h.update_kvector(A)
    n, out = step()
    assert n == 1 and torch.equal(out, plain)
    h.close()


@pytest.mark.parametrize("name,kw", [("tiny", dict()), ("c1", dict()), ("c1", dict(scf=True, pc=True))])
def test_fused_current_equals_unfused(name, kw):
    """The RT step with current_next's gather and without it, bit for bit."""
    from salmon2_amd.rt import RTPropagator

    print(f"[gpu] per-term current_next {name} {kw}", flush=True)
    s = system.config(name)
    r = []
    for fuse in (False, True):
        p = RTPropagator(s, fuse_current=fuse, **kw)
        p.h._set_shape(0, 0)
        r.append((p.run(8), p.psi_a.cpu().numpy()))
        p.close()
    for k in ("curr", "dip", "rne"):
        assert np.array_equal(r[0][0][k], r[1][0][k]), k
    assert np.array_equal(r[0][1], r[1][1])
