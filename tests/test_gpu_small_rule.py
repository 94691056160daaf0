"""Grids that fit the whole-orbital kernels, at the edges of the rules that leave them to the per-term kernels
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


def values(s):
    """projector values of one orbital"""
    return int(sum(int(s.mps[ia]) * int((np.asarray(s.ia_tbl) == ia + 1).sum()) for ia in range(s.natom)))


def counts(h, call):
    """launches of the projections (0: the call ran the whole-orbital kernels)"""
    h.prof_start(64)
    call()
    n = h.prof_read("proj")[1] + h.prof_read("proj_current")[1]
    h.prof_end()
    return n


# 10^3 points under 16 projectors of 5.3 bohr: about 73 000 values, 8 atoms
@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("past", [0, 1])
def test_step_and_hpsi_edges(oracle_lib, order, past):
    import torch

    from salmon2_amd.hip import Handle

    kw = dict(n=10, lmax=3, rcut=5.3, nkgrid=(1, 2, 2), seed=401, n_hamil=order)
    w = values(system.make_si_system(no=1, **kw)) * 8
    for what, lim in (("step", int(94e6 * order / w) // 4), ("hpsi", int(196e6 / w) // 4)):
        no = lim + past
        print(f"[gpu] small rule {what} order {order}: {4 * no} orbitals of {w // 8} values", flush=True)
        s = system.make_si_system(no=no, **kw)
        h = Handle(s, stream=torch.cuda.current_stream())
        h.update_kvector(A)
        O = oracle_lib.Oracle(s)
        O.update_kvector(A)
        psi = torch.from_numpy(s.psi).cuda()
        out, work = torch.zeros_like(psi), torch.zeros_like(psi)
        if what == "step":
            n = counts(h, lambda: h.taylor(s.zc(), psi, out, work))
            ref = O.taylor(A, s.psi)[0]
        else:
            n = counts(h, lambda: h.hpsi(psi, out))
            ref = O.hpsi(A, s.psi)
        assert (n > 0) == bool(past)
        assert rel(out.cpu().numpy()[..., : s.ny, :], ref[..., : s.ny, :]) <= 1e-12
        h.close()


@pytest.mark.parametrize("no", [91, 92])  # 16 k: 8.49 and 8.58 million points
def test_current_edge(oracle_lib, no):
    import torch

    from salmon2_amd.hip import Handle

    print(f"[gpu] small rule current: {16 * no} orbitals of 18^3", flush=True)
    s = system.make_si_system(n=18, no=no, nkgrid=(1, 4, 4), seed=403)
    h = Handle(s, stream=torch.cuda.current_stream())
    h.update_kvector(A)
    psi = torch.from_numpy(s.psi).cuda()
    cur, two = (torch.zeros((1, 3), dtype=torch.float64, device="cuda") for _ in range(2))
    out = torch.zeros_like(psi)
    work = torch.zeros_like(psi)
    # its 11 600 values keep the step whole for any number of orbitals
    assert counts(h, lambda: h.taylor(s.zc(), psi, out, work)) == 0
    h.current(A, psi, cur)
    h.current_next(A, psi, two, A)
    assert torch.equal(cur, two)
    O = oracle_lib.Oracle(s)
    O.update_kvector(A)
    assert rel(cur.cpu().numpy(), O.current(A, s.psi)) <= 1e-9
    h.close()


@pytest.mark.parametrize("kw", [
    dict(n=10, lmax=3, rcut=5.3, no=41, nkgrid=(1, 4, 4)),  # per-term step, whole-orbital current
    dict(n=18, no=92, nkgrid=(1, 4, 4)),                    # whole-orbital step, per-term current
    dict(n=18, lmax=2, no=115, nkgrid=(1, 4, 4)),           # both per term
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
