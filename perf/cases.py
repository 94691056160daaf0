"""Performance cases of the real-time propagation framework.

``listed()`` names the workloads whose speed matters, ``draw(rng)`` gives further ones of the same
ranges.  ``prepare`` builds what a program holds before the call (system, handle, orbitals on the
GPU), ``run`` is one pass through the public entry points, ``work`` the bytes and operations a pass
cannot do without, and ``exact`` the same pass in plain torch at 64 bits.

Kinds of case
  step       one real-time step of ``rt.RTPropagator`` (Taylor propagation, density, current, dipole,
             and with scf the potential update; predictor-corrector or aetrs)
  hpsi       H psi alone, as an eigen-energy evaluation or a ground-state solver calls it
  potential  Hartree + exchange-correlation + local potential from a density
  batch      one step of several uneven systems together (``batch.BatchRunner``)
  predict    the learned midpoint predictor: features, network, potential
  train      one minibatch of the predictor's training, with its gradients
"""
import functools
import math

import numpy as np
import torch

from salmon2_amd import batch as _batch
from salmon2_amd import hip as _hip
from salmon2_amd import learned as _learned
from salmon2_amd import rt as _rt
from salmon2_amd import system as _system

NT = 2000          # rows of the field tables
T0 = NT // 4       # passes start inside the pulse, as in a continued run
SCALES = (0.05, 2.0, 0.1)  # feature and target scales of the predictor
LR = 1e-3


def _step(name, cell, n, no, k, **kw):
    c = dict(name=name, kind="step", cx=cell[0], cy=cell[1], cz=cell[2], nx=n[0], ny=n[1], nz=n[2], no=no, kx=k[0],
             ky=k[1], kz=k[2], nspin=1, lmax=1, scf=False, pc=False, precision="fp64", propagator="middlepoint")
    c.update(kw)
    return c


def listed():
    one = (1, 1, 1)
    return [
        # the smallest run in use: one cell at Gamma, where launches and latency count
        _step("gamma-8-atoms", one, (16, 16, 16), 16, one),
        # bulk Si as SALMON's own benchmark input has it (12^3 points, 4^3 k), the method's default step
        _step("bulk-8-atoms-64k", one, (12, 12, 12), 16, (4, 4, 4), scf=True, pc=True),
        # spin-polarised material on an odd grid with the aetrs propagator
        _step("spin-odd-aetrs", one, (15, 17, 14), 16, (2, 2, 2), nspin=2, scf=True, propagator="aetrs"),
        # the 64-atom benchmark supercell: self-consistent predictor-corrector in FP64
        _step("64-atoms-pc", (2, 2, 2), (32, 32, 32), 128, (2, 2, 2), scf=True, pc=True),
        # a 64-atom supercell on a ragged grid in mixed precision
        _step("64-atoms-ragged-mixed", (2, 2, 2), (30, 27, 26), 128, (1, 1, 2), scf=True, pc=True, precision="mixed"),
        # the largest: 216 atoms, 432 orbitals at 4 k, mixed precision with a fixed potential
        _step("216-atoms-mixed", (3, 3, 3), (48, 48, 48), 432, (2, 2, 1), precision="mixed"),
        # an elongated cell (rows wider than 64 points) with d projectors
        _step("rod-64-atoms-spd", (8, 1, 1), (96, 14, 12), 128, (1, 2, 2), lmax=2),
        # H psi of the 64-atom supercell at Gamma
        dict(name="hpsi-64-atoms", kind="hpsi", cx=2, cy=2, cz=2, nx=32, ny=32, nz=32, no=128, kx=1, ky=1, kz=1, nspin=1,
             lmax=1),
        # the potential update alone, on a grid with three different extents
        dict(name="potential-56x50x42", kind="potential", cx=4, cy=4, cz=3, nx=56, ny=50, nz=42, nspin=1),
        # many small uneven systems served together
        dict(name="batch-8-systems", kind="batch", count=8, pick=20261205),
        # the learned predictor at the benchmark grid: inference, and a training minibatch
        dict(name="predict-32", kind="predict", nx=32, ny=32, nz=32),
        dict(name="train-32", kind="train", nx=32, ny=32, nz=32, samples=4),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any cell, grid, orbital and k-point count of the listed ones' ranges."""
    u = rng.random()
    if u < 0.1:
        n = [4 * rng.randint(3, 10) for _ in range(3)]
        kind = "predict" if rng.random() < 0.5 else "train"
        c = dict(kind=kind, nx=n[0], ny=n[1], nz=n[2])
        if kind == "train":
            c["samples"] = rng.randint(1, 6)
        return c
    if u < 0.18:
        return dict(kind="batch", count=rng.randint(2, 8), pick=rng.randrange(1 << 20))
    cell = rng.choice([(1, 1, 1), (1, 1, 2), (2, 1, 1), (2, 2, 1), (2, 2, 2), (4, 1, 1), (1, 2, 4), (8, 1, 1), (3, 2, 2)])
    # spacings of 0.6 to 0.95 bohr, odd extents among them
    n = [max(8, int(round(_system.SI_A * m / rng.uniform(0.6, 0.95)))) for m in cell]
    if u < 0.26:
        return dict(kind="potential", cx=cell[0], cy=cell[1], cz=cell[2], nx=n[0], ny=n[1], nz=n[2],
                    nspin=rng.choice([1, 1, 2]))
    points = n[0] * n[1] * n[2]
    kpt = rng.choice([(1, 1, 1), (1, 1, 2), (2, 1, 1), (2, 2, 1), (2, 2, 2), (4, 4, 4)])
    nspin = rng.choice([1, 1, 1, 2])
    total = math.exp(rng.uniform(math.log(6e4), math.log(4e7)))
    no = max(3, min(256, int(total / (points * kpt[0] * kpt[1] * kpt[2] * nspin))))
    lmax = rng.choice([1, 1, 1, 2, 3])
    common = dict(cx=cell[0], cy=cell[1], cz=cell[2], nx=n[0], ny=n[1], nz=n[2], no=no, kx=kpt[0], ky=kpt[1], kz=kpt[2],
                  nspin=nspin, lmax=lmax)
    if u < 0.36:
        return dict(kind="hpsi", **common)
    form = rng.choice(["fixed", "pc", "pc", "plain", "aetrs"])
    return dict(kind="step", scf=form != "fixed", pc=form == "pc", precision=rng.choice(["fp64", "fp64", "mixed"]),
                propagator="aetrs" if form == "aetrs" else "middlepoint", **common)


# ---------------------------------------------------------------------------- inputs
@functools.lru_cache(maxsize=32)
def _crystal(cell, n, no, k, nspin, lmax, projectors=True):
    """The crystal without its orbitals (the same for every seed: the seed gives the orbitals)."""
    return _system.make_si_system(ncell=cell, n=n, no=no, nkgrid=k, seed=77, dt=0.08, nt=NT, A0=0.01, nspin=nspin, lmax=lmax,
                                  with_projectors=projectors, host_orbitals=False)


def _system_of(c):
    return _crystal((c["cx"], c["cy"], c["cz"]), (c["nx"], c["ny"], c["nz"]), c["no"], (c["kx"], c["ky"], c["kz"]),
                    c["nspin"], c["lmax"])


def _batch_of(c):
    """Uneven systems: 8 to 64 atoms, 8 to 64 orbitals, 1 to 8 k-points, extents of 12 to 36."""
    r = np.random.default_rng(c["pick"])
    out = []
    for _ in range(c["count"]):
        cell = [(1, 1, 1), (1, 1, 2), (2, 2, 1), (2, 2, 2)][r.integers(4)]
        n = tuple(int(r.choice([g for g in range(12, 37, 4) if 0.55 <= _system.SI_A * m / g <= 0.95])) for m in cell)
        k = [(1, 1, 1), (2, 1, 1), (2, 2, 1), (2, 2, 2)][r.integers(4)]
        out.append(_crystal(cell, n, int(r.choice([8, 16, 32, 64])), k, 1, 1))
    return out


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _lowpass(n, al, cut, device="cuda"):
    """exp(-|G|^2 / (2 cut^2)) on the reciprocal grid (nz, ny, nx)."""
    g2 = 0.0
    for d, m in ((2, n[2]), (1, n[1]), (0, n[0])):
        g = torch.fft.fftfreq(m, 1.0 / m, dtype=torch.float64, device=device) * (2.0 * math.pi / float(al[d]))
        g2 = g2 + (g * g).reshape([-1 if i == 2 - d else 1 for i in range(3)])
    return torch.exp(-g2 / (2.0 * cut * cut))


def _orbitals(s, seed):
    """Smooth normalised random orbitals in the padded layout (nk, no, nspin, nz, ly, nx)."""
    g = _generator(seed)
    low = _lowpass((s.nx, s.ny, s.nz), s.al, 1.5)
    psi = torch.zeros((s.nk, s.no, s.nspin, s.nz, s.ly, s.nx), dtype=torch.complex128, device="cuda")
    for ik in range(s.nk):
        z = torch.randn((s.no, s.nspin, s.nz, s.ny, s.nx, 2), generator=g, dtype=torch.float64, device="cuda")
        w = torch.fft.ifftn(torch.view_as_complex(z) * low, dim=(2, 3, 4))
        del z
        w /= torch.sqrt(w.abs().square().sum(dim=(2, 3, 4), keepdim=True) * s.hvol)
        psi[ik, :, :, :, : s.ny, :] = w
        del w
    return psi


def _field(n, al, seed, cut=1.2):
    """A smooth real random field on the grid, zero mean, unit deviation."""
    z = torch.randn((n[2], n[1], n[0]), generator=_generator(seed), dtype=torch.float64, device="cuda")
    f = torch.fft.ifftn(torch.fft.fftn(z) * _lowpass(n, al, cut)).real
    return ((f - f.mean()) / f.std()).contiguous()


def _net_inputs(c, seed):
    n = (c["nx"], c["ny"], c["nz"])
    return n, [m * 0.64 for m in n]


# a layer of the predictor: output channels, input channels, level of the grid it works on
_LAYERS = [(16, 16, 0), (16, 16, 0), (32, 16, 1), (32, 32, 1), (64, 32, 2), (64, 64, 2), (32, 96, 1), (32, 32, 1), (16, 48, 0),
           (16, 16, 0)]


def _net_params(seed):
    """He-normal weights, small biases, in the network's flat order."""
    r = np.random.default_rng(seed)
    parts = []
    for co, ci, _ in _LAYERS:
        parts.append(r.standard_normal(27 * co * ci) * math.sqrt(2.0 / (27 * ci)))
        parts.append(0.05 * r.standard_normal(co))
    parts.append(r.standard_normal(17) * 0.25)
    return np.concatenate(parts).astype(np.float32)


def _net_samples(c, seed):
    n, al = _net_inputs(c, seed)
    out = []
    for i in range(c["samples"]):
        x = torch.stack([_field(n, al, seed * 1000 + 10 * i + j).reshape(-1) for j in range(4)], dim=1).float().contiguous()
        out.append((x, _field(n, al, seed * 1000 + 10 * i + 5).reshape(-1).float().contiguous()))
    return out


def _histories(c, seed):
    """Four successive potentials and Vpsl."""
    n, al = _net_inputs(c, seed)
    base = 2.0 * _field(n, al, seed * 100)
    v = [base + SCALES[0] * _field(n, al, seed * 100 + 1 + j) for j in range(4)]
    return v, base - 1.0


def _density(c, s, seed):
    """Channel densities (nspin, nz, ny, nx), positive, about Si's valence density."""
    n = (c["nx"], c["ny"], c["nz"])
    return torch.stack([0.03 / c["nspin"] * torch.exp(0.8 * _field(n, s.al, seed * 10 + j)) for j in range(c["nspin"])])


def prepare(case, seed):
    kind = case["kind"]
    torch.cuda.set_device(0)
    if kind == "step":
        s = _system_of(case)
        p = _rt.RTPropagator(s, psi=_orbitals(s, seed), scf=case["scf"], pc=case["pc"], precision=case["precision"],
                             propagator=case["propagator"])
        p.setup_outputs(NT)
        p.itt = T0
        return dict(kind=kind, p=p)
    if kind == "hpsi":
        s = _system_of(case)
        h = _hip.Handle(s, stream=torch.cuda.current_stream())
        h.update_kvector(_ac(s)[T0])
        psi = _orbitals(s, seed)
        return dict(kind=kind, h=h, psi=psi, out=torch.zeros_like(psi))
    if kind == "potential":
        s = _crystal((case["cx"], case["cy"], case["cz"]), (case["nx"], case["ny"], case["nz"]), 1, (1, 1, 1),
                     case["nspin"], 1, False)
        h = _hip.Handle(s, stream=torch.cuda.current_stream())
        h.set_poisson(s.al)
        rho = _density(case, s, seed)
        return dict(kind=kind, h=h, rho=rho, vpsl=torch.from_numpy(s.vlocal[0]).cuda(), v=torch.zeros_like(rho))
    if kind == "batch":
        systems = _batch_of(case)
        r = _batch.BatchRunner(systems, NT, psi=[_orbitals(s, seed * 100 + i) for i, s in enumerate(systems)])
        r.batch.set_time(T0 + 1)
        return dict(kind=kind, r=r, itt=T0)
    n, al = _net_inputs(case, seed)
    pred = _learned.Predictor(*n, stream=torch.cuda.current_stream(), scales=SCALES)
    pred.net.set_params(_net_params(seed))
    if kind == "predict":
        v, vpsl = _histories(case, seed)
        return dict(kind=kind, pred=pred, v=v, vpsl=vpsl, out=torch.zeros_like(vpsl))
    data = _net_samples(case, seed)
    return dict(kind=kind, pred=pred, data=data, loss=torch.zeros(len(data), dtype=torch.float32, device="cuda"))


def run(state):
    kind = state["kind"]
    if kind == "step":
        p = state["p"]
        if p.itt >= NT:
            p.itt = T0
        p.step()
        out = dict(psi=p.psi_a, rho=p.rho, curr=p.curr_t[p.itt - 1], dip=p.dip_t[p.itt - 1])
        if p.scf:
            out["v"] = p.vcur
        return out
    if kind == "hpsi":
        state["h"].hpsi(state["psi"], state["out"])
        return state["out"]
    if kind == "potential":
        state["h"].update_potential(state["rho"], state["vpsl"], vout=state["v"])
        return state["v"]
    if kind == "batch":
        r = state["r"]
        if state["itt"] >= NT:
            r.batch.set_time(T0 + 1)
            state["itt"] = T0
        r.run(1)
        i = state["itt"]
        state["itt"] = i + 1
        state["odd"] = not state.get("odd", False)
        # the orbital buffers alternate by step
        return [dict(psi=b["psi_b" if state["odd"] else "psi_a"], rho=b["rho"], curr=b["curr"][i], dip=b["dip"][i])
                for b in r.buf]
    pred = state["pred"]
    if kind == "predict":
        pred.predict(state["v"], state["vpsl"], state["out"])
        return dict(vpred=state["out"], nn=pred.nn)
    for i, (x, t) in enumerate(state["data"]):
        pred.net.train_sample(x, t, state["loss"][i : i + 1])
    grads = pred.net.get_grads()
    pred.net.adam_step(LR, len(state["data"]))
    return dict(loss=state["loss"], grads=grads)


# ---------------------------------------------------------------------------- work
def _step_work(s, applications):
    """Orbitals read and written once; 158 operations per point and orbital of a stencil application,
    8 of a Taylor update, 21 per projector and sphere point (src/io/flops.f90:119,138-139,162)."""
    po = float(s.ngrid) * s.norb
    per_atom = s.nlma / max(1, s.natom)
    kb = 21.0 * per_atom * float(np.sum(s.mps)) * s.norb
    return 32.0 * po, applications * (166.0 * po + kb)


def work(case):
    kind = case["kind"]
    if kind in ("step", "hpsi"):
        s = _system_of(case)
        # predictor-corrector: the corrector's first application follows from the predictor's
        times = 1 if kind == "hpsi" else 7 if case["pc"] else 8 if case["propagator"] == "aetrs" else 4
        b, f = _step_work(s, times)
        return dict(bytes=b + 24.0 * s.nspin * s.ngrid, flops=f)
    if kind == "potential":
        n = case["nx"] * case["ny"] * case["nz"]
        return dict(bytes=8.0 * n * (2 * case["nspin"] + 1), flops=n * (10.0 * math.log2(n) + 60.0 * case["nspin"]))
    if kind == "batch":
        w = [_step_work(s, 4) for s in _batch_of(case)]
        return dict(bytes=sum(x[0] for x in w), flops=sum(x[1] for x in w))
    n = case["nx"] * case["ny"] * case["nz"]
    flops = sum(2.0 * 27 * co * ci * (n >> (3 * lv)) for co, ci, lv in _LAYERS)
    par = sum(27 * co * ci + co for co, ci, _ in _LAYERS) + 17
    if kind == "predict":
        return dict(bytes=48.0 * n + 2.0 * par, flops=flops)
    return dict(bytes=case["samples"] * 20.0 * n + 32.0 * par, flops=3.0 * case["samples"] * flops)


# ---------------------------------------------------------------------------- 64-bit values
def _ac(s):
    """A(t) = -A0 sin^2(pi t / tw) cos(omega t) along x, rows 0 .. NT + 1."""
    t = np.arange(NT + 2) * s.dt
    p = s.pulse
    a = np.where(t < p.tw, -p.A0 * np.sin(np.pi * t / p.tw) ** 2 * np.cos(p.omega * t), 0.0)
    return a[:, None] * np.asarray(p.epdir)[None, :]


class _Exact:
    """The step's operators in plain torch complex128; psi (nk, no, nspin, nz, ny, nx)."""

    def __init__(self, s):
        self.s = s
        dev = "cuda"
        self.dims = {0: -1, 1: -2, 2: -3}
        self.atoms = []
        for ia in range(s.natom):
            m = int(s.mps[ia])
            rows = np.nonzero(s.ia_tbl == ia + 1)[0]
            j = s.jxyz[ia, :m].astype(np.int64) - 1
            self.atoms.append((torch.from_numpy(j[:, 0] + s.nx * (j[:, 1] + s.ny * j[:, 2])).to(dev),
                               torch.from_numpy(np.ascontiguousarray(s.rxyz[ia, :m])).to(dev),
                               torch.from_numpy(np.ascontiguousarray(s.uv[rows, :m])).to(dev),
                               torch.from_numpy(np.ascontiguousarray(s.rinv_uvu[rows])).to(dev)))

    def kvector(self, a):
        """Phase factors conj(e^{i(k+A)r}) uv of every k and atom, and k + A."""
        self.kac = self.s.vec_k + np.asarray(a)[None, :]
        self.z = [[torch.exp(-1j * (r @ torch.from_numpy(k).to(r.device))) * uv for _, r, uv, _ in self.atoms]
                  for k in self.kac]

    def hpsi_k(self, psi, v, ik):
        """H of the orbitals (no, nspin, nz, ny, nx) of one k-point."""
        s, k = self.s, self.kac[ik]
        out = psi * (v + s.coef_lap0 + 0.5 * float(k @ k))
        for d in range(3):
            for n in range(1, 5):
                up, dn = torch.roll(psi, -n, self.dims[d]), torch.roll(psi, n, self.dims[d])
                out += (-0.5 * s.coef_lap[d, n - 1] - 1j * k[d] * s.coef_nab[d, n - 1]) * up
                out += (-0.5 * s.coef_lap[d, n - 1] + 1j * k[d] * s.coef_nab[d, n - 1]) * dn
        flat, res = psi.reshape(s.no * s.nspin, -1), torch.view_as_real(out).reshape(s.no * s.nspin, -1, 2)
        for (idx, _, _, rinv), z in zip(self.atoms, self.z[ik]):
            c = (flat[:, idx] @ z.conj().T.contiguous()) * rinv
            res.index_add_(1, idx, torch.view_as_real(c @ z))
        return torch.view_as_complex(res).reshape(psi.shape)

    def taylor(self, psi, v, dt):
        out = torch.empty_like(psi)
        for ik in range(self.s.nk):
            h, z = psi[ik], 1.0
            acc = h.clone()
            for n in range(1, self.s.n_hamil + 1):
                h = self.hpsi_k(h, v, ik)
                z = z * (-1j * dt) / n
                acc += z * h
            out[ik] = acc
        return out

    def density(self, psi):
        s = self.s
        w = torch.from_numpy(np.ascontiguousarray(s.rocc.transpose(1, 2, 0) * s.wtk[:, None, None])).to(psi.device)
        rho = torch.zeros(psi.shape[2:], dtype=torch.float64, device=psi.device)
        for ik in range(s.nk):
            rho += (psi[ik].abs().square() * w[ik][:, :, None, None, None]).sum(dim=0)
        return rho

    def current(self, psi, a):
        """Kinetic part with the field a, nonlocal part with the current phase factors."""
        s = self.s
        out = torch.zeros((s.nspin, 3), dtype=torch.float64, device=psi.device)
        for ik in range(s.nk):
            p = psi[ik]
            norm = p.abs().square().sum(dim=(2, 3, 4))
            w = torch.from_numpy(np.ascontiguousarray(s.rocc[:, ik, :].T * s.wtk[ik])).to(psi.device)
            j = torch.zeros((s.no, s.nspin, 3), dtype=torch.float64, device=psi.device)
            for d in range(3):
                t = sum(s.coef_nab[d, n - 1] * (p.conj() * torch.roll(p, -n, self.dims[d])).sum(dim=(2, 3, 4))
                        for n in range(1, 5))
                j[..., d] = (s.vec_k[ik, d] + a[d]) * norm + 2.0 * t.imag
            flat = p.reshape(s.no * s.nspin, -1)
            for (idx, r, _, rinv), z in zip(self.atoms, self.z[ik]):
                g = flat[:, idx]
                u = (g @ z.conj().T.contiguous()) * rinv
                for d in range(3):
                    ur = g @ (z * r[:, d]).conj().T.contiguous()
                    j[..., d] += 2.0 * (ur.conj() * u).imag.sum(dim=1).reshape(s.no, s.nspin)
            out += (j * w[:, :, None]).sum(dim=0)
        return out / s.ngrid

    def dipole(self, rho):
        s = self.s
        tot, out = rho.sum(dim=0), []
        for d, n in enumerate((s.nx, s.ny, s.nz)):
            pos = torch.arange(1, n + 1, dtype=torch.float64, device=rho.device) - (0.0 if n % 2 else 0.5)
            out.append(-(tot * pos.reshape([-1 if i == 2 - d else 1 for i in range(3)])).sum() * float(s.hgs[d]) * s.hvol)
        return torch.stack(out + [tot.sum() * s.hvol])


def _exact_potential(rho, vpsl, al):
    """Vpsl + Hartree + PZ81 (unpolarised or spin-polarised) of channel densities (nspin, nz, ny, nx)."""
    n = (rho.shape[3], rho.shape[2], rho.shape[1])
    g2 = 0.0
    for d in range(3):
        g = torch.fft.fftfreq(n[d], 1.0 / n[d], dtype=torch.float64, device=rho.device) * (2.0 * math.pi / float(al[d]))
        g2 = g2 + (g * g).reshape([-1 if i == 2 - d else 1 for i in range(3)])
    coef = torch.where(g2 > 0, 4.0 * math.pi / torch.where(g2 > 0, g2, torch.ones_like(g2)), torch.zeros_like(g2))
    vh = torch.fft.ifftn(torch.fft.fftn(rho.sum(dim=0)) * coef).real
    return vpsl + vh + _pz(rho)


def _pz(rho):
    """PZ81 potential per channel: v = e + rho de/drho (nspin = 1), the polarised form for 2."""
    cx = 0.75 * (3.0 / (2.0 * math.pi)) ** (2.0 / 3.0)

    def corr(rs, low, high):
        g, b1, b2 = low
        a, b, c, d = high
        q, ln = torch.sqrt(rs), torch.log(rs)
        e1 = g / (1.0 + b1 * q + b2 * rs)
        v1 = e1 * (1.0 + 7.0 / 6.0 * b1 * q + 4.0 / 3.0 * b2 * rs) / (1.0 + b1 * q + b2 * rs)
        e2 = a * ln + b + c * rs * ln + d * rs
        v2 = a * ln + (b - a / 3.0) + 2.0 / 3.0 * c * rs * ln + (2.0 * d - c) / 3.0 * rs
        return torch.where(rs > 1.0, e1, e2), torch.where(rs > 1.0, v1, v2)

    low_u, high_u = (-0.1423, 1.0529, 0.3334), (0.0311, -0.048, 0.002, -0.0116)
    low_p, high_p = (-0.0843, 1.3981, 0.2611), (0.01555, -0.0269, 0.0007, -0.0048)
    if rho.shape[0] == 1:
        t = rho[0] + 1e-10
        rs = (3.0 / (4.0 * math.pi * t)) ** (1.0 / 3.0)
        ec, vc = corr(rs, low_u, high_u)
        ex = -cx / rs
        # v = e + rho de/drho with the offset density in de/drho
        de = ex / (3.0 * t) + (vc - ec) / t
        return (ex + ec + rho[0] * de)[None]
    tot = rho.sum(dim=0)
    rs = (3.0 / (4.0 * math.pi * tot)) ** (1.0 / 3.0)
    zeta = (rho[0] - rho[1]) / tot
    f = ((1 + zeta) ** (4.0 / 3.0) + (1 - zeta) ** (4.0 / 3.0) - 2.0) / (2.0 ** (4.0 / 3.0) - 2.0)
    ecu, vcu = corr(rs, low_u, high_u)
    ecp, vcp = corr(rs, low_p, high_p)
    df = 4.0 / 3.0 * ((1 + zeta) ** (1.0 / 3.0) - (1 - zeta) ** (1.0 / 3.0)) / (2.0 ** (4.0 / 3.0) - 2.0)
    out = []
    for sg, z in ((1.0, 1 + zeta), (-1.0, 1 - zeta)):
        out.append(-4.0 / 3.0 * cx / rs * z ** (1.0 / 3.0) + vcu + f * (vcp - vcu) + (ecp - ecu) * (sg - zeta) * df)
    return torch.stack(out)


def _padded(s, psi):
    out = torch.zeros((s.nk, s.no, s.nspin, s.nz, s.ly, s.nx), dtype=psi.dtype, device=psi.device)
    out[:, :, :, :, : s.ny, :] = psi
    return out


def _exact_step(s, psi, scf=False, pc=False, aetrs=False):
    """The pass of a fresh state: step T0 -> T0 + 1."""
    ac, e = _ac(s), _Exact(s)
    psi = psi[:, :, :, :, : s.ny, :].contiguous()
    v = torch.from_numpy(np.ascontiguousarray(s.vlocal)).cuda()
    vpsl = v[0]
    if scf:
        v = _exact_potential(e.density(psi), vpsl, s.al)
    now, mid = ac[T0 + 1], 0.5 * (ac[T0 + 1] + ac[T0])
    if aetrs:
        e.kvector(now)
        psi = e.taylor(psi, v, s.dt / 2)
        e.kvector(ac[T0 + 2])  # the extrapolated potential of a run's first step is V itself
        psi = e.taylor(psi, v, s.dt / 2)
    else:
        e.kvector(mid)
        if pc:
            rho = e.density(e.taylor(psi, v, s.dt))
            v = 0.5 * (v + _exact_potential(rho, vpsl, s.al))
        psi = e.taylor(psi, v, s.dt)
    rho = e.density(psi)
    cur = e.current(psi, now)
    out = dict(psi=_padded(s, psi), rho=rho, curr=cur, dip=e.dipole(rho))
    if scf:
        v = _exact_potential(rho, vpsl, s.al)
        out["v"] = v if s.nspin == 2 else v[0]
    return out


def _exact_net(w, x, shape):
    """The network in float64 without rounding; x (points, 4), w the flat parameters."""
    nz, ny, nx = shape
    taps = [(z, y, q) for z in (-1, 0, 1) for y in (-1, 0, 1) for q in (-1, 0, 1)]
    off = 0
    layers = []
    for co, ci, _ in _LAYERS:
        layers.append((w[off : off + 27 * co * ci].reshape(27, co, ci), w[off + 27 * co * ci : off + 27 * co * ci + co]))
        off += 27 * co * ci + co
    head = w[off : off + 17]

    def conv(t, i):
        k, b = layers[i]
        y = sum(torch.roll(t, (-dz, -dy, -dx), (0, 1, 2)) @ k[j].T for j, (dz, dy, dx) in enumerate(taps))
        return torch.relu(y + b)

    def pool(t):
        a, b, c, m = t.shape
        return t.reshape(a // 2, 2, b // 2, 2, c // 2, 2, m).mean(dim=(1, 3, 5))

    def up(t):
        return t.repeat_interleave(2, 0).repeat_interleave(2, 1).repeat_interleave(2, 2)

    h = torch.cat([x.double(), torch.zeros((x.shape[0], 12), dtype=torch.float64, device=x.device)], 1).reshape(nz, ny, nx, 16)
    e1 = conv(conv(h, 0), 1)
    e2 = conv(conv(pool(e1), 2), 3)
    e3 = conv(conv(pool(e2), 4), 5)
    d2 = conv(conv(torch.cat([up(e3), e2], 3), 6), 7)
    d1 = conv(conv(torch.cat([up(d2), e1], 3), 8), 9)
    return (d1 @ head[:16] + head[16]).reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        s = _system_of(case)
        return _exact_step(s, _orbitals(s, seed), case["scf"], case["pc"], case["propagator"] == "aetrs")
    if kind == "hpsi":
        s = _system_of(case)
        e = _Exact(s)
        e.kvector(_ac(s)[T0])
        psi = _orbitals(s, seed)[:, :, :, :, : s.ny, :].contiguous()
        v = torch.from_numpy(np.ascontiguousarray(s.vlocal)).cuda()
        return _padded(s, torch.stack([e.hpsi_k(psi[ik], v, ik) for ik in range(s.nk)]))
    if kind == "potential":
        s = _crystal((case["cx"], case["cy"], case["cz"]), (case["nx"], case["ny"], case["nz"]), 1, (1, 1, 1),
                     case["nspin"], 1, False)
        return _exact_potential(_density(case, s, seed), torch.from_numpy(s.vlocal[0]).cuda(), s.al)
    if kind == "batch":
        out = []
        for i, s in enumerate(_batch_of(case)):
            d = _exact_step(s, _orbitals(s, seed * 100 + i))
            out.append(dict(psi=d["psi"], rho=d["rho"], curr=d["curr"].reshape(-1), dip=d["dip"]))
        return out
    shape = (case["nz"], case["ny"], case["nx"])
    w = torch.from_numpy(_net_params(seed)).cuda().double()
    if kind == "predict":
        v, vpsl = _histories(case, seed)
        x = torch.stack([(v[0] - v[1]) / SCALES[0], (v[1] - v[2]) / SCALES[0], (v[2] - v[3]) / SCALES[0],
                         (v[0] - vpsl) / SCALES[1]], dim=-1).reshape(-1, 4)
        nn = _exact_net(w, x, shape)
        return dict(vpred=v[0] + 0.5 * (v[0] - v[1]) + SCALES[2] * nn.reshape(shape), nn=nn)
    w.requires_grad_(True)
    losses = []
    for x, t in _net_samples(case, seed):
        loss = torch.mean((_exact_net(w, x, shape) - t.double()) ** 2)
        loss.backward()
        losses.append(loss.detach())
    return dict(loss=torch.stack(losses), grads=w.grad)
