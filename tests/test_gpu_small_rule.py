"""Grids that fit the whole-orbital kernels, on both sides of the rules that leave them to the per-term kernels
(many orbitals of many projector values, spread over many atoms): which form runs, its result against
the CPU oracle, and the RT step with and without the current's prepared projection, bit for bit.

Tolerances as elsewhere for FP64: 1e-12 relative on H psi and one Taylor step, 1e-9 on the current."""
import numpy as np
import pytest

from salmon2_amd import system

pytestmark = pytest.mark.gpu

A = np.array([0.013, -0.021, 0.007])


def rel(a, b):
    a, b = np.asarray(a), np.asarray(b)
    return float(np.abs(a - b).max() / np.abs(b).max())


def counts(h, call):
    """launches of the projections (0: the call ran the whole-orbital kernels)"""
    h.prof_start(64)
    call()
    n = h.prof_read("proj")[1] + h.prof_read("proj_current")[1]
    h.prof_end()
    return n


# 10^3 points under 16 projectors of 5.3 bohr on each of 8 atoms: about 73 000 values
@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("no,whole", [(16, True), (64, True), (256, False)])  # x 4 k-points
def test_step_and_hpsi(oracle_lib, order, no, whole):
    import torch

    from salmon2_amd.hip import Handle

    print(f"[gpu] small rule step, H psi: order {order}, {4 * no} orbitals", flush=True)
    s = system.make_si_system(n=10, lmax=3, rcut=5.3, nkgrid=(1, 2, 2), seed=401, n_hamil=order, no=no)
    h = Handle(s, stream=torch.cuda.current_stream())
    h.update_kvector(A)
    O = oracle_lib.Oracle(s)
    O.update_kvector(A)
    psi = torch.from_numpy(s.psi).cuda()
    out, work = torch.zeros_like(psi), torch.zeros_like(psi)
    assert (counts(h, lambda: h.taylor(s.zc(), psi, out, work)) == 0) == whole
    ref = O.taylor(A, s.psi)[0]
    assert rel(out.cpu().numpy()[..., : s.ny, :], ref[..., : s.ny, :]) <= 1e-12
    assert (counts(h, lambda: h.hpsi(psi, out)) == 0) == whole
    assert rel(out.cpu().numpy()[..., : s.ny, :], O.hpsi(A, s.psi)[..., : s.ny, :]) <= 1e-12
    h.close()


@pytest.mark.parametrize("no,whole", [(16, True), (100, False)])  # x 16 k-points
def test_current(oracle_lib, no, whole):
    import torch

    from salmon2_amd.hip import Handle

    print(f"[gpu] small rule current: {16 * no} orbitals of 12 x 12 x 24", flush=True)
    s = system.make_si_system(ncell=(1, 1, 2), n=(12, 12, 24), lmax=3, rcut=4.0, no=no, nkgrid=(1, 4, 4), seed=403)
    h = Handle(s, stream=torch.cuda.current_stream())
    h.update_kvector(A)
    psi = torch.from_numpy(s.psi).cuda()
    cur, two = (torch.zeros((1, 3), dtype=torch.float64, device="cuda") for _ in range(2))
    h.current(A, psi, cur)
    h.current_next(A, psi, two, A)
    O = oracle_lib.Oracle(s)
    O.update_kvector(A)
    ref = O.current(A, s.psi)
    assert rel(cur.cpu().numpy(), ref) <= 1e-9
    assert rel(two.cpu().numpy(), ref) <= 1e-9
    h._set_shape(0, 0)  # the per-term kernels
    h.current(A, psi, two)
    assert torch.equal(cur, two) != whole
    h.close()


@pytest.mark.parametrize("kw", [
    dict(n=10, lmax=3, rcut=5.3, no=64, nkgrid=(1, 4, 4)),                          # per-term step, whole-orbital current
    dict(ncell=(1, 1, 2), n=(10, 20, 30), no=160, nkgrid=(1, 4, 4)),                # whole-orbital step, per-term current
    dict(ncell=(1, 1, 2), n=(12, 12, 24), lmax=3, rcut=4.0, no=100, nkgrid=(1, 4, 4)),  # both per term
])
def test_fused_current_equals_unfused(kw):
    from salmon2_amd.rt import RTPropagator

    print(f"[gpu] small rule current_next {kw}", flush=True)
    s = system.make_si_system(seed=405, nt=3, **kw)
    r = []
    for fuse in (False, True):
        p = RTPropagator(s, fuse_current=fuse)
        r.append((p.run(3), p.psi_a.cpu().numpy()))
        p.close()
    for k in ("curr", "dip", "rne"):
        assert np.array_equal(r[0][0][k], r[1][0][k]), k
    assert np.array_equal(r[0][1], r[1][1])
