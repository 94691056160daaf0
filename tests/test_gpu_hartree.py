"""The Hartree passes (half spectrum, folded columns) and the potential update against the CPU oracle at the
extents where their split can go wrong: the smallest, odd and even ones on each axis (self-paired output at
n/2 or not), column counts that do not fill a block, rows above 128 points (four columns per block), the
largest extent taken, one and two spin channels.

Tolerance 1e-12 relative as for the other potential calls: sums of at most 256 terms per pass, five passes."""
import numpy as np
import pytest

from salmon2_amd import system

pytestmark = pytest.mark.gpu


def rel(a, b):
    a, b = np.asarray(a), np.asarray(b)
    return float(np.abs(a - b).max() / np.abs(b).max())


@pytest.mark.parametrize("n", [(4, 4, 4), (4, 5, 6), (13, 8, 7), (7, 13, 9), (16, 11, 20), (56, 50, 42), (129, 6, 5),
                               (6, 130, 8), (5, 6, 131), (256, 4, 4), (4, 256, 5), (6, 4, 256)])
@pytest.mark.parametrize("nspin", [1, 2])
def test_hartree_extents(oracle_lib, n, nspin):
    import torch

    assert torch.cuda.is_available(), "GPU tests need a visible MI355X"
    from salmon2_amd.hip import Handle

    print(f"[gpu] hartree {n} nspin={nspin}", flush=True)
    s = system.make_si_system(n=n, no=1, with_projectors=False, host_orbitals=False, nspin=nspin, seed=3)
    rng = np.random.default_rng(9)
    shape = (s.nz, s.ny, s.nx)
    rho = 0.02 + 0.1 * rng.random((nspin,) + shape)
    vmix = rng.standard_normal((nspin,) + shape)
    h = Handle(s, stream=torch.cuda.current_stream())
    h.set_poisson(s.al)
    d = {k: torch.from_numpy(np.ascontiguousarray(v)).cuda() for k, v in dict(rho=rho, vpsl=s.vlocal[0], vmix=vmix).items()}
    tot = d["rho"].sum(dim=0)
    vh = torch.full(shape, float("nan"), dtype=torch.float64, device="cuda")
    v = torch.full((nspin,) + shape, float("nan"), dtype=torch.float64, device="cuda")
    h.hartree(tot, vh)
    h.update_potential(d["rho"], d["vpsl"], vmix=d["vmix"], vout=v)
    ref = oracle_lib.hartree(rho.sum(axis=0), s.al)
    e1 = rel(vh.cpu().numpy(), ref)
    vxc = oracle_lib.xc_pz(rho[0])[0][None] if nspin == 1 else oracle_lib.xc_pz_sp(rho)[0]
    e2 = rel(v.cpu().numpy(), 0.5 * (vmix + s.vlocal[0] + ref + vxc))
    # in place: the density's own array receives the potential
    h.hartree(tot, tot)
    e3 = rel(tot.cpu().numpy(), ref)
    print(f"[parity] hartree {n} nspin={nspin}: {e1:.2e}, potential {e2:.2e}", flush=True)
    assert max(e1, e2, e3) <= 1e-12
    h.close()
