"""Whole-orbital kernels of small grids (one block per orbital, the orbital in LDS): H psi, the Taylor
step of orders 1 to 6, the corrector from a given H psi, the current and the device-side gate against
the CPU oracle, at the shapes where the split can go wrong: the smallest extents, columns that do not
fill the waves, a last z chunk of one plane, every launch class, points covered by several spheres, no
projectors, more than four projectors per atom, padded and unpadded rows, two spins, and the largest
orbital that fits (and the first that does not, which takes the per-term kernels).

Tolerances as elsewhere for FP64: 1e-12 relative on H psi and one Taylor step (a few hundred roundings
of 1e-16 per point), 1e-9 on the current (a sum with cancellation)."""
import numpy as np
import pytest

from salmon2_amd import system

pytestmark = pytest.mark.gpu

CASES = {
    "8x8x8": dict(n=8, no=3, nkgrid=(1, 1, 2)),
    "4x5x6_noproj": dict(n=(4, 5, 6), no=2, with_projectors=False),
    "12cube_many": dict(n=12, no=33, nkgrid=(2, 2, 4)),          # over 512 orbitals: blocks share a CU
    "13x11x9": dict(n=(13, 11, 9), no=3, nkgrid=(1, 1, 2)),      # 143 columns, a last chunk of one plane
    "15x17x14_spin": dict(n=(15, 17, 14), no=3, nspin=2, nkgrid=(1, 2, 1)),
    "16cube_nopad": dict(n=16, no=4, pad=0),
    "12cube_pad3": dict(n=12, no=3, pad=3),
    "18cube": dict(n=18, no=2),                                  # nine planes per thread
    "24x24x9": dict(n=(24, 24, 9), no=2),                        # 576 columns: one z chunk
    "32x28x4": dict(n=(32, 28, 4), no=2, ncell=(2, 2, 1), rcut=1.5),  # 896 columns
    "24x16x20": dict(n=(24, 16, 20), no=2),                      # 7680 points, the most that one block takes
    "24x16x21": dict(n=(24, 16, 21), no=2),                      # one plane more: the per-term kernels
    "overlap_rc3.6": dict(n=12, no=3, rcut=3.6),                 # most touched points covered twice
    "selfimage_rc5.3": dict(n=12, no=2, rcut=5.3),               # points covered up to ten times
    "spdf_14cube": dict(n=14, no=3, lmax=3, nkgrid=(1, 1, 2)),   # 16 projectors per atom
    "spd_2cells": dict(n=(10, 11, 20), no=3, ncell=(1, 1, 2), lmax=2),  # 16 atoms on 8 waves
}


def rel(a, b):
    a, b = np.asarray(a), np.asarray(b)
    return float(np.abs(a - b).max() / np.abs(b).max())


@pytest.fixture(scope="module")
def torch_dev():
    import torch

    assert torch.cuda.is_available(), "GPU tests need a visible MI355X"
    from salmon2_amd import hip

    hip.load()
    return torch


@pytest.mark.parametrize("name", list(CASES))
def test_small_grid(torch_dev, oracle_lib, name):
    torch = torch_dev
    from salmon2_amd.hip import Handle

    print(f"[gpu] small grid case={name}", flush=True)
    s = system.make_si_system(seed=101, **CASES[name])
    A = np.array([0.013, -0.021, 0.007])
    h = Handle(s, stream=torch.cuda.current_stream())
    h.update_kvector(A)
    O = oracle_lib.Oracle(s)
    O.update_kvector(A)
    psi = torch.from_numpy(s.psi).cuda()
    out, work = torch.zeros_like(psi), torch.zeros_like(psi)
    ny = s.ny

    def got(t):
        a = t.cpu().numpy()
        assert np.all(a[..., ny:, :] == 0), "padding row written"
        return a[..., :ny, :]

    h.hpsi(psi, out)
    ref = O.hpsi(A, s.psi)
    assert rel(got(out), ref[..., :ny, :]) <= 1e-12
    h.taylor(s.zc(), psi, out, work)
    ref_t, _, _ = O.taylor(A, s.psi)
    assert rel(got(out), ref_t[..., :ny, :]) <= 1e-12
    assert rel(got(work), ref[..., :ny, :]) <= 1e-12
    assert np.array_equal(psi.cpu().numpy(), s.psi)
    # the corrector: the same step after V_local changed by dv, from the H psi of the step above
    rng = np.random.default_rng(7)
    dv = 0.2 * rng.standard_normal(s.vlocal.shape)
    h.set_vlocal(s.vlocal + dv)
    h.taylor_reuse(s.zc(), psi, out, work, torch.from_numpy(dv).cuda())
    first = got(out).copy()
    h.taylor(s.zc(), psi, out, work)
    assert rel(first, got(out)) <= 1e-12
    h.set_vlocal(s.vlocal)
    # the current, alone and with the next field's table prepared
    B = np.array([0.02, 0.001, -0.01])
    cur = torch.zeros((s.nspin, 3), dtype=torch.float64, device="cuda")
    h.current(B, psi, cur)
    ref_c = O.current(B, s.psi)
    assert rel(cur.cpu().numpy(), ref_c) <= 1e-9
    two = torch.zeros_like(cur)
    h.current_next(B, psi, two, B)
    assert torch.equal(cur, two)
    h.update_kvector(B)
    h.taylor(s.zc(), psi, out, work)
    O.update_kvector(B)
    assert rel(got(out), O.taylor(B, s.psi)[0][..., :ny, :]) <= 1e-12
    # the device-side gate: a set flag leaves the outputs alone
    flag = torch.ones(1, dtype=torch.int32, device="cuda")
    out.fill_(3.0)
    h.set_skip(flag)
    h.taylor(s.zc(), psi, out, work)
    h.hpsi(psi, out)
    h.set_skip(None)
    assert bool((out == 3.0).all())
    h.close()


@pytest.mark.parametrize("n_hamil", [1, 2, 3, 6])
def test_small_grid_orders(torch_dev, oracle_lib, n_hamil):
    torch = torch_dev
    from salmon2_amd.hip import Handle

    print(f"[gpu] small grid order {n_hamil}", flush=True)
    s = system.make_si_system(n=(13, 12, 14), no=3, seed=103, n_hamil=n_hamil)
    A = np.array([0.012, -0.02, 0.007])
    h = Handle(s, stream=torch.cuda.current_stream())
    h.update_kvector(A)
    psi = torch.from_numpy(s.psi).cuda()
    out = torch.zeros_like(psi)
    work = torch.full_like(psi, 5.0)
    h.taylor(s.zc(), psi, out, work)
    O = oracle_lib.Oracle(s)
    O.update_kvector(A)
    ref, _, _ = O.taylor(A, s.psi)
    assert rel(out.cpu().numpy()[..., : s.ny, :], ref[..., : s.ny, :]) <= 1e-12
    if n_hamil == 1:  # sshtpsi is written from order 2 on
        assert bool((work == 5.0).all())
    h.close()
