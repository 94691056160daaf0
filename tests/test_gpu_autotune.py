"""The launch-shape autotuner: what later calls run is what it timed, and its choice handed to
set_launch_shape (as a host that stores it does) leaves every result as it is, bit for bit."""
import numpy as np
import pytest

from salmon2_amd import system

pytestmark = pytest.mark.gpu

A = np.array([0.013, -0.021, 0.007])


def _step(h, s, psi):
    import torch

    out, work, hp = (torch.zeros_like(psi) for _ in range(3))
    h.taylor(s.zc(), psi, out, work)
    h.hpsi(psi, hp)
    return out, work, hp


@pytest.mark.parametrize("kw,whole", [
    (dict(n=(12, 11, 13), no=3), True),                                # an orbital per block
    (dict(n=(26, 20, 31), no=3), False),                               # too large for that
    (dict(n=10, lmax=3, rcut=5.3, no=64, nkgrid=(1, 4, 4)), False),    # fits, but too many orbitals
])
def test_autotune_then_step(oracle_lib, kw, whole):
    import torch

    from salmon2_amd.hip import Handle

    print(f"[gpu] autotune then step {kw}", flush=True)
    s = system.make_si_system(seed=501, **kw)
    h = Handle(s, stream=torch.cuda.current_stream())
    h.update_kvector(A)
    psi = torch.from_numpy(s.psi).cuda()
    h._set_shape(0, 1)  # a shape set by hand before does not keep the rule out
    plane, nzt, ms = h.autotune(reps=2)
    assert ms > 0.0
    if whole:
        assert (plane, nzt) == (-1, 0)
    first = _step(h, s, psi)
    h.prof_start(64)
    h.taylor(s.zc(), psi, torch.zeros_like(psi), torch.zeros_like(psi))
    n = h.prof_read("hpsi_taylor1")[1]
    h.prof_end()
    assert (n == 0) == whole
    h._set_shape(plane, nzt)
    for a, b in zip(first, _step(h, s, psi)):
        assert torch.equal(a, b)
    O = oracle_lib.Oracle(s)
    O.update_kvector(A)
    ref = O.taylor(A, s.psi)[0][..., : s.ny, :]
    e = np.abs(first[0].cpu().numpy()[..., : s.ny, :] - ref).max() / np.abs(ref).max()
    assert e <= 1e-12
    h.close()


# (extents, order, whether some launch of the step is a persistent one): rows of up to 64 points take one block per
# tile in every term up to order 4; above that the last term is persistent, and rows above 64 points always are
@pytest.mark.parametrize("ns,order,persistent", [
    (((12, 11, 13), (20, 16, 24)), 4, False),
    (((12, 11, 13), (20, 16, 24)), 5, True),
    (((12, 11, 13), (66, 8, 9)), 4, True),
    (((66, 8, 9), (130, 6, 10), (13, 8, 9)), 2, True),
    (((66, 8, 9), (128, 6, 10), (13, 8, 9)), 5, True),
])
def test_batch_autotune(oracle_lib, ns, order, persistent):
    """The batched step on either side of its persistent form, before and after tuning: the tuner's grid choice
    where there is one to make, and every member's series against the oracle (1e-9, the series bar)."""
    from salmon2_amd.batch import BatchRunner

    print(f"[gpu] batch autotune {ns} order {order}", flush=True)
    nt = 3
    systems = [system.make_si_system(ncell=(6, 1, 1) if n[0] > 64 else (1, 1, 1), n=n, no=3, rcut=1.8, n_hamil=order,
                                     seed=510 + i, nt=nt) for i, n in enumerate(ns)]
    br = BatchRunner(systems, nt)
    refs = []
    for s in systems:
        _, cur, dip, rne = oracle_lib.Oracle(s).rt_run(nt=nt, psi=s.psi)
        refs.append(dict(curr=cur, dip=dip, rne=rne))
    for tuned in (False, True):
        if tuned:
            choice, ms = br.batch.autotune(reps=2)
            assert ms > 0.0 and (choice % 100 != 99 or any(n[0] > 64 for n in ns)) == persistent
            br.reset()
        br.run(nt)
        for g, ref in zip(br.results(nt), refs):
            for k in ref:
                e = np.abs(np.asarray(g[k]) - ref[k]).max() / np.abs(ref[k]).max()
                assert e <= 1e-9, (tuned, k, e)
    br.close()
