"""H psi and one Taylor step on grids whose planes are cut into tiles with ragged edges: numbers of planes
that are no multiple of four, z chunks of uneven length, rows above 64 points (tiles on x and y, with a
last tile of few points), the longest rows, and the shapes beside them that take the other tile forms.
Every grid is above what one block holds, so that the per-term kernels run.

Tolerances as elsewhere: FP64 1e-12 relative (a few hundred roundings of 1e-16 per point); the complex-FP32
chain 1e-6 (its terms are small beside psi, whose rounding it does not take part in)."""
import numpy as np
import pytest

from salmon2_amd import system

pytestmark = pytest.mark.gpu

CASES = {
    "17x31x23": dict(n=(17, 31, 23), no=3, nkgrid=(1, 1, 2)),      # 15 rows of 17 points: 31 = 2 * 15 + 1
    "30x25x18_spin": dict(n=(30, 25, 18), no=2, nspin=2),
    "64x13x11": dict(n=(64, 13, 11), no=2, ncell=(2, 1, 1)),       # the longest undivided row
    "32x32x14": dict(n=(32, 32, 14), no=2),
    "65x9x17": dict(n=(65, 9, 17), no=2, ncell=(2, 1, 1)),         # two x tiles of 33 and 32 points
    "97x12x9_spin": dict(n=(97, 12, 9), no=2, nspin=2, ncell=(3, 1, 1)),
    "100x18x6_pad0": dict(n=(100, 18, 6), no=3, ncell=(3, 1, 1), pad=0),
    "131x6x16_pad3": dict(n=(131, 6, 16), no=2, ncell=(3, 1, 1), pad=3),
    "256x8x5": dict(n=(256, 8, 5), no=2, ncell=(4, 1, 1)),         # the longest row
    "80x4x26_many": dict(n=(80, 4, 26), no=65, ncell=(2, 1, 1), nkgrid=(1, 1, 2)),  # y halo wraps twice
    "70x14x12_noproj": dict(n=(70, 14, 12), no=2, with_projectors=False),
}


def rel(a, b):
    a, b = np.asarray(a), np.asarray(b)
    return float(np.abs(a - b).max() / np.abs(b).max())


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("chunks", [0, 1, 3])
def test_stencil_tiles(oracle_lib, name, chunks):
    import torch

    from salmon2_amd import hip

    print(f"[gpu] stencil tiles case={name} chunks={chunks}", flush=True)
    s = system.make_si_system(seed=211, **CASES[name])
    A = np.array([0.021, -0.013, 0.017])
    h = hip.Handle(s, stream=torch.cuda.current_stream())
    if chunks:
        h._set_shape(0, chunks)  # row tiles, that many z chunks
    h.update_kvector(A)
    O = oracle_lib.Oracle(s)
    O.update_kvector(A)
    psi = torch.from_numpy(s.psi).cuda()
    out, work = torch.zeros_like(psi), torch.zeros_like(psi)
    ny = s.ny
    h.hpsi(psi, out)
    ref = O.hpsi(A, s.psi)
    g = out.cpu().numpy()
    assert np.all(g[..., ny:, :] == 0), "padding row written"
    assert rel(g[..., :ny, :], ref[..., :ny, :]) <= 1e-12
    ref_t = O.taylor(A, s.psi)[0]
    for prec, tol in (("fp64", 1e-12), ("mixed", 1e-6)):
        h.set_precision(prec)
        out.zero_()
        h.taylor(s.zc(), psi, out, work)
        g = out.cpu().numpy()
        assert np.all(g[..., ny:, :] == 0), "padding row written"
        e = rel(g[..., :ny, :], ref_t[..., :ny, :])
        print(f"[parity] {name} {prec}: {e:.2e}", flush=True)
        assert e <= tol


@pytest.mark.parametrize("name", ["17x31x23", "65x9x17"])
@pytest.mark.parametrize("n_hamil", [1, 2, 3, 5, 6])
def test_stencil_tiles_orders(oracle_lib, name, n_hamil):
    """The last term's sum over 0 to 5 earlier terms (order 4 above), the planes in one chunk and in two."""
    import torch

    from salmon2_amd import hip

    print(f"[gpu] stencil tiles case={name} order {n_hamil}", flush=True)
    s = system.make_si_system(seed=223, n_hamil=n_hamil, **CASES[name])
    A = np.array([0.021, -0.013, 0.017])
    O = oracle_lib.Oracle(s)
    O.update_kvector(A)
    ref = O.taylor(A, s.psi)[0][..., : s.ny, :]
    for chunks in (0, 2):
        h = hip.Handle(s, stream=torch.cuda.current_stream())
        h._set_shape(0, chunks)
        h.update_kvector(A)
        psi = torch.from_numpy(s.psi).cuda()
        out, work = torch.zeros_like(psi), torch.zeros_like(psi)
        h.taylor(s.zc(), psi, out, work)
        assert rel(out.cpu().numpy()[..., : s.ny, :], ref) <= 1e-12


@pytest.mark.parametrize("n_hamil", [2, 4, 5])
def test_batch_ragged_planes(oracle_lib, n_hamil):
    """A batch whose members have numbers of planes that are no multiple of four, against the oracle."""
    from salmon2_amd.batch import BatchRunner

    print(f"[gpu] batch of ragged planes, order {n_hamil}", flush=True)
    nt = 3
    grids = [(17, 31, 23), (30, 25, 18), (12, 13, 9), (32, 32, 14)]
    systems = [system.make_si_system(n=n, no=2 + i, seed=230 + i, nt=nt, n_hamil=n_hamil, nkgrid=(1, 1, 1 + i % 2))
               for i, n in enumerate(grids)]
    br = BatchRunner(systems, nt)
    br.run(nt)
    got = br.results(nt)
    br.close()
    for s, g in zip(systems, got):
        _, cur, dip, rne = oracle_lib.Oracle(s).rt_run(nt=nt, psi=s.psi)
        for k, ref in (("curr", cur), ("dip", dip), ("rne", rne)):
            assert rel(g[k], ref) <= 1e-9, k
