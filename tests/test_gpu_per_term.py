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
