"""Projection and fused KB kernels at the edges of their blocks: orbital counts around 16 and 64, spheres
of fewer points than a wave's chunk and of odd remainders, one to sixteen projectors per atom, against
the CPU oracle (H psi, one Taylor step, the current, which weights the projections by position).

Tolerances as elsewhere: 1e-12 relative on H psi and the step (sums of a few hundred FP64 products), 1e-9 on
the current (a sum with cancellation), 1e-6 on a step of the complex-FP32 chain."""
import numpy as np
import pytest

from salmon2_amd import system

pytestmark = pytest.mark.gpu


def rel(a, b):
    a, b = np.asarray(a), np.asarray(b)
    return float(np.abs(a - b).max() / np.abs(b).max())


@pytest.mark.parametrize("no", [1, 15, 17, 64, 65])
@pytest.mark.parametrize("lmax,rcut", [(0, 1.2), (1, 1.0), (1, 2.8), (2, 1.7), (3, 2.2)])
def test_projection_blocks(oracle_lib, no, lmax, rcut):
    import torch

    from salmon2_amd import hip

    print(f"[gpu] projections no={no} lmax={lmax} rcut={rcut}", flush=True)
    s = system.make_si_system(n=(13, 12, 11), no=no, lmax=lmax, rcut=rcut, nkgrid=(1, 1, 2), seed=307)
    A = np.array([0.013, -0.021, 0.007])
    h = hip.Handle(s, stream=torch.cuda.current_stream())
    h._set_shape(0, 0)  # the per-term kernels
    h.update_kvector(A)
    O = oracle_lib.Oracle(s)
    O.update_kvector(A)
    psi = torch.from_numpy(s.psi).cuda()
    out, work = torch.zeros_like(psi), torch.zeros_like(psi)
    ny = s.ny
    h.hpsi(psi, out)
    assert rel(out.cpu().numpy()[..., :ny, :], O.hpsi(A, s.psi)[..., :ny, :]) <= 1e-12
    ref = O.taylor(A, s.psi)[0][..., :ny, :]
    for prec, tol in (("fp64", 1e-12), ("mixed", 1e-6)):
        h.set_precision(prec)
        h.taylor(s.zc(), psi, out, work)
        assert rel(out.cpu().numpy()[..., :ny, :], ref) <= tol
    cur = torch.zeros(3 * s.nspin, dtype=torch.float64, device="cuda")
    h.current(A, psi, cur)
    assert rel(cur.cpu().numpy(), np.asarray(O.current(A, s.psi)).ravel()) <= 1e-9
    h.close()
