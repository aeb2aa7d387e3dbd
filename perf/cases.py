"""Performance cases of the multislice engine: the work its users have it do,
through the package's public entry points.

`listed()` gives the fixed cases, `draw(rng)` further ones of the same ranges.
`prepare(case, seed)` makes what a program holds before the call (specimen,
handle, potentials and probes), `run(state)` one pass of it, `work(case)` the
bytes and operations the pass cannot do without, and `exact(case, seed)` the
pass's outputs in 64-bit torch arithmetic.

Specimens are those of the benchmark and the tests (diamond-cubic silicon,
SrTiO3, random atoms); every atom is moved by a seeded Gaussian of 0.08 A per
axis, a frozen phonon.
"""
import math

import numpy as np
import torch

from cudamultislice_amd import MultisliceSimulation, fparams
from cudamultislice_amd import structures as S
from cudamultislice_amd.diff import DiffEngine, MultisliceIntensity
from cudamultislice_amd.serve import FD, Job, serve

THERMAL = 0.08  # A per axis
CS_TEM = 1.2e7  # A
F = np.float32


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # plane-wave TEM runs, whole: binning, tables, every slice, exit wave
        # (and CTF images).  A unit-test sized run, where latency counts ...
        dict(name="tem_64", kind="tem", nx=64, ny=64, ps=0.2, cx=2, cy=2, cz=2, dz=1.0, kV=200.0, projected=False,
             images=0),
        # ... the small benchmark run (Si 4x4x10, exit wave and CTF image) ...
        dict(name="tem_256", kind="tem", nx=256, ny=256, ps=0.084844, cx=4, cy=4, cz=10, dz=1.0, kV=200.0,
             projected=False, images=1),
        # ... the run at scale (Si 14x14x92, 252 slices, 8 defoci) ...
        dict(name="tem_1024", kind="tem", nx=1024, ny=1024, ps=0.07424, cx=14, cy=14, cz=92, dz=2.0, kV=300.0,
             projected=False, images=8),
        # ... and the GUI's smallest camera preset, whose sides (2 3 167 and
        # 4 167) have no radix plan
        dict(name="tem_1002x668", kind="tem", nx=1002, ny=668, ps=0.03, cx=5, cy=3, cz=6, dz=2.0, kV=200.0,
             projected=False, images=1),
        # finite-difference multislice on one handle (the reference's default
        # method): 200 steps through the middle of the specimen
        dict(name="fd_256", kind="fd", nx=256, ny=256, ps=0.084844, cx=4, cy=4, cz=4, kV=200.0, steps=200),
        # one probe position, frozen phonons, CBED and ADF: the reference's
        # own STEM/TDS loop
        dict(name="cbed_512", kind="cbed", nx=512, ny=512, ps=0.078125, cx=10, cy=10, cz=10, dz=2.0, configs=2),
        # batched STEM: a line scan on a small grid with the projected
        # potential and a PACBED map (odd probe count) ...
        dict(name="stem_128_odd", kind="stem", nx=128, ny=128, ps=0.15625, cx=5, cy=5, cz=8, dz=2.0, probes=37,
             configs=1, sigma=0.0, projected=True, graph=False, pacbed=True),
        # ... and a part of the headline scan (512^2, SrTiO3 10x10x50, 99
        # slices, frozen phonons, graph replay)
        dict(name="stem_512", kind="stem", nx=512, ny=512, ps=0.078125, cx=10, cy=10, cz=50, dz=2.0, probes=512,
             configs=2, sigma=0.08, projected=False, graph=True, pacbed=False),
        # gradients of an intensity loss with respect to the potential: a
        # small reconstruction step, and the benchmark's
        dict(name="train_128", kind="train", nx=128, ny=128, slices=6, probes=3, keep=0),
        dict(name="train_1024", kind="train", nx=1024, ny=1024, slices=100, probes=64, keep=10),
        # intensities only (evaluation of a reconstruction)
        dict(name="infer_512", kind="infer", nx=512, ny=512, slices=60, probes=24, keep=0),
        # a serving mix: grids 256 to 1024, plane waves and probes, both methods
        dict(name="serve_16", kind="serve", jobs=16, mix=1, top=1024, slices=60, atoms=10000, probes=48),
    ]


def _between(rng, a, b):
    """an integer of [a, b], spread over its logarithm"""
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.choice(["tem", "tem", "gui", "fd", "cbed", "stem", "stem", "train", "infer", "serve"])
    if kind in ("tem", "gui"):
        n = rng.choice([64, 128, 256, 512, 1024])
        nx, ny = n, rng.choice([n, n, max(64, n // 2)])
        if kind == "gui":  # camera presets and other sides without a plan
            nx, ny = rng.choice([(1002, 668), (2004, 1336), (rng.randint(60, 900), rng.randint(60, 900))])
        cells = rng.randint(2, max(2, min(10, n // 64)))
        ps = round((cells * 5.43 + rng.uniform(0.0, 4.0)) / min(nx, ny), 6)
        return dict(kind="tem", nx=nx, ny=ny, ps=ps, cx=max(2, int(ps * nx / 5.43)), cy=max(2, int(ps * ny / 5.43)),
                    cz=_between(rng, 2, 24 if kind == "tem" else 6), dz=rng.choice([1.0, 1.5, 2.0]),
                    kV=rng.choice([80.0, 200.0, 300.0]), projected=rng.random() < 0.3, images=rng.choice([0, 1, 3, 8]))
    if kind == "fd":
        n = rng.choice([64, 128, 256, 512])
        c = rng.randint(2, 5)
        return dict(kind=kind, nx=n, ny=rng.choice([n, n, n // 2]), ps=round((c * 5.43 + rng.uniform(0, 3)) / n, 6),
                    cx=c, cy=c, cz=rng.randint(2, 6), kV=rng.choice([100.0, 200.0, 300.0]),
                    steps=_between(rng, 20, 200))
    if kind == "cbed":
        n = rng.choice([128, 256, 512])
        c = rng.randint(4, 10)
        return dict(kind=kind, nx=n, ny=n, ps=round((c * 3.905 + rng.uniform(0, 2)) / n, 6), cx=c, cy=c,
                    cz=_between(rng, 3, 20), dz=rng.choice([1.0, 2.0]), configs=rng.randint(1, 4))
    if kind == "stem":
        n = rng.choice([128, 256, 512])
        c = rng.randint(5, 10)
        return dict(kind=kind, nx=n, ny=n, ps=round((c * 3.905 + rng.uniform(0, 1)) / n, 6), cx=c, cy=c,
                    cz=_between(rng, 4, 40), dz=2.0, probes=_between(rng, 5, 400), configs=rng.randint(1, 2),
                    sigma=rng.choice([0.0, 0.08]), projected=rng.random() < 0.3, graph=rng.random() < 0.5,
                    pacbed=rng.random() < 0.3)
    if kind in ("train", "infer"):
        n = rng.choice([64, 128, 256, 512])
        return dict(kind=kind, nx=n, ny=rng.choice([n, n, 2 * n]), slices=_between(rng, 3, 60),
                    probes=_between(rng, 1, 48), keep=rng.choice([0, 0, 5, 10]))
    return dict(kind="serve", jobs=rng.randint(3, 16), mix=rng.randint(2, 10 ** 6), top=rng.choice([256, 512, 1024]),
                slices=_between(rng, 20, 60), atoms=_between(rng, 1000, 10000), probes=_between(rng, 16, 48))


# ---------------------------------------------------------------- inputs
def _specimen(c, seed):
    cell = S.silicon if c["kind"] in ("tem", "fd") else S.srtio3
    Z, x, y, z = cell(c["cx"], c["cy"], c["cz"])
    rng = np.random.default_rng(seed)
    return (Z,) + tuple((v + rng.normal(0.0, THERMAL, v.size)).astype(F) for v in (x, y, z))


def _positions(c, seed):
    rng = np.random.default_rng(seed + 7)
    return tuple(rng.integers(0, c[n], c["probes"]).astype(np.int32) for n in ("nx", "ny"))


def _defoci(c):
    return np.linspace(-800.0, 600.0, c["images"]).astype(F) if c["images"] > 1 else np.array([-500.0], F)


PS_DIFF, KV_DIFF, DZ_DIFF = 0.1, 300.0, 2.0  # the differentiable benchmark's sampling


def _diff_inputs(c, seed):
    """Potentials of light atoms (2 to 90 V A, 0.45 A wide), 25 mrad probes on
    a raster and noisy measured intensities."""
    g = torch.Generator("cuda").manual_seed(seed)
    nx, ny, ns, B = c["nx"], c["ny"], c["slices"], c["probes"]
    kx, ky = (torch.fft.fftfreq(n, PS_DIFF, dtype=torch.float64, device="cuda") for n in (nx, ny))
    k2 = kx[None, :] ** 2 + ky[:, None] ** 2
    blur = torch.exp(-2 * (math.pi * 0.2) ** 2 * k2).float()
    V = torch.empty(ns, ny, nx, device="cuda")
    for i in range(ns):
        hit = (torch.rand(ny, nx, device="cuda", generator=g) < 0.12 * PS_DIFF ** 2).float()
        V[i] = torch.fft.ifft2(torch.fft.fft2(hit * 2500.0) * blur).real.clamp_(min=0.0)
    lam = float(_physics(KV_DIFF)[0])
    side = max(1, math.ceil(math.sqrt(B)))
    psi = torch.empty(B, ny, nx, dtype=torch.complex64, device="cuda")
    for b in range(B):
        px, py = (b % side + 0.5) / side * nx * PS_DIFF, (b // side + 0.5) / side * ny * PS_DIFF
        k = (k2 < (0.025 / lam) ** 2) * torch.exp(-2j * math.pi * (kx[None, :] * px + ky[:, None] * py))
        w = torch.fft.ifft2(k)
        psi[b] = (w / w.abs().square().sum().sqrt()).to(torch.complex64)
    target = psi.abs().square() * (1.0 + 0.3 * torch.randn(B, ny, nx, device="cuda", generator=g))
    return V, psi, target


def _serving_jobs(c, seed):
    """Jobs of the uneven mix: the kinds and sizes follow the case, atoms and
    probe positions the seed."""
    shape = np.random.default_rng(c["mix"])
    rng = np.random.default_rng(seed)
    jobs = []
    for k in range(c["jobs"]):
        n = int(shape.choice([v for v in (256, 512, 1024) if v <= c["top"]]))
        ns = int(shape.integers(20, c["slices"] + 1))
        method = k % 2
        nprobe = 0 if k % 4 < 2 else int(shape.integers(16, max(17, c["probes"] + 1)))
        lateral, thick = n * 0.1 - 4.0, max(3.0, ns * (2.0 if method != FD else 0.06))
        nat = int(min(shape.integers(c["atoms"] // 2, c["atoms"] + 1), 0.05 * lateral * lateral * thick))
        Z, x, y, z = S.jittered_atoms(max(1, nat), (lateral, lateral, thick), seed=seed + k)
        pos = [rng.integers(0, n, nprobe).astype(np.int32) for _ in range(2)] if nprobe else (None, None)
        jobs.append(Job(n, Z, x, y, z, ns, method, *pos))
    return jobs


SERVE = dict(kV=300.0, ps=0.1, dz=2.0, aperture=25.0, adf=(20.0, 200.0))


def _handle(c, seed):
    sim = MultisliceSimulation(0)
    sim.set_atoms(*_specimen(c, seed))
    sim.GetParameterisation()
    return sim


def prepare(case, seed):
    c = case
    st = {"case": c, "seed": seed}
    if c["kind"] in ("train", "infer"):
        V, psi, target = _diff_inputs(c, seed)
        st.update(V=V.requires_grad_(c["kind"] == "train"), psi=psi, target=target,
                  engine=DiffEngine(c["nx"], c["ny"], PS_DIFF, KV_DIFF, DZ_DIFF, c["slices"], c["probes"], c["keep"]))
    elif c["kind"] == "serve":
        st["jobs"] = _serving_jobs(c, seed)
    else:
        st["sim"] = sim = _handle(c, seed)
        if c["kind"] in ("stem", "cbed"):
            sim.ApplyMicroscopeParameters(300.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 25.0)
            i = sim.info()
            sim.STEMSetCalculationVariables(c["ps"], 0.0, c["nx"], c["ny"], i["MaximumX"] - i["MinimumX"],
                                            i["MaximumY"] - i["MinimumY"], i["MaximumZ"] - i["MinimumZ"])
            sim.PreCalculateFrequencies()
            if c["kind"] == "stem":
                sim.set_potential_mode(int(c["projected"]))
                st["pos"] = _positions(c, seed)
    return st


# ---------------------------------------------------------------- one pass
def _setup(sim, c, df, Cs, off):
    sim.UploadBinnedAtoms()
    sim.ApplyMicroscopeParameters(c["kV"], df, 0.0, 0.0, Cs, 0.0, 0.0, 20.0)
    i = sim.info()
    sim.SetCalculationVariables(c["ps"], df, c["nx"], c["ny"], i["MaximumX"] - i["MinimumX"],
                                i["MaximumY"] - i["MinimumY"], i["MaximumZ"] - i["MinimumZ"], off, off)
    sim.PreCalculateFrequencies()


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "tem":
        sim, dfs = state["sim"], _defoci(c)
        sim.set_potential_mode(int(c["projected"]))
        _setup(sim, c, float(dfs[0]), CS_TEM, 2.0)
        sim.InitialiseWavefunctions(c["dz"])
        for it in range(1, sim.GetSlices(True) + 1):
            sim.MultisliceStepConv(it)
        out = {"exit": sim.GetExitWave()}
        if c["images"] == 1:
            out["image"] = sim.SimulateImage(1.0)
        elif c["images"] > 1:
            out["image"] = sim.ctf_sweep(dfs)
        return out
    if kind == "fd":
        sim = state["sim"]
        _setup(sim, c, 0.0, 0.0, 0.0)
        sim.InitialiseWavefunctions()
        i = sim.info()
        first = int(0.5 * (i["MaximumZ"] - i["MinimumZ"]) / i["dzFD"])
        for it in range(first, first + c["steps"]):
            sim.MultisliceStep(it)
        return {"exit": sim.GetExitWave()}
    if kind == "cbed":
        sim = state["sim"]
        sim.set_tds(state["seed"], THERMAL)
        sim.AllocTDS()
        adf = []
        for _ in range(c["configs"]):
            sim.UploadBinnedAtomsTDS()
            sim.STEMInitialiseWavefunctions(c["nx"] // 2 + 3, c["ny"] // 2 - 5)
            sim.set_conventional_dz(c["dz"])
            for it in range(1, sim.GetSlices(True) + 1):
                sim.MultisliceStepConv(it)
            sim.AddTDSWaves()
            adf.append(sim.adf(20.0, 200.0))
        return {"adf": np.array(adf, F), "tds": sim.GetTDS()}
    if kind == "stem":
        return state["sim"].stem_batched(*state["pos"], c["dz"], nconfig=c["configs"], seed=state["seed"],
                                         sigma=c["sigma"], adf=(20.0, 200.0), use_graph=c["graph"],
                                         pacbed=c["pacbed"])
    if kind == "train":
        V = state["V"]
        V.grad = None
        out = MultisliceIntensity.apply(V, state["psi"], state["engine"])
        ((out - state["target"]) ** 2).sum().backward()
        return {"intensity": out.detach(), "grad": V.grad}
    if kind == "infer":
        return {"intensity": state["engine"].forward(state["V"], state["psi"], keep=False)}
    serve(state["jobs"], **SERVE)
    return [j.result.get("exit", j.result.get("adf")) for j in state["jobs"]]


# ---------------------------------------------------------------- work
def _fft_flops(nx, ny):
    return 5.0 * nx * ny * math.log2(nx * ny)


def _potential_flops(atoms, ps, samples, slices_per_atom):
    """10 operations for each sample of the potential inside the 5 A^2 cutoff"""
    return 10.0 * atoms * slices_per_atom * (math.pi * 5.0 / ps ** 2) * samples * 0.6


def work(case):
    c = case
    kind = c["kind"]
    if kind == "serve":
        b = f = 0.0
        for j in _serving_jobs(c, 1):
            w = max(1, j.nprobe)
            f += w * j.nslices * (6 if j.method == FD else 2) * _fft_flops(j.n, j.n)
            f += _potential_flops(j.Z.size, 0.1, 1 if j.method == FD else 20, 3.2 if j.method != FD else j.nslices)
            b += 16 * j.Z.size + (4 * w if j.nprobe else 8 * j.n ** 2)
        return {"bytes": b, "flops": f}
    nx, ny = c["nx"], c["ny"]
    np_, fft = float(nx * ny), _fft_flops(nx, ny)
    if kind in ("train", "infer"):
        ns, B = c["slices"], c["probes"]
        b = ns * np_ * 4 + B * np_ * 12
        f = B * ns * (2 * fft + 12 * np_)
        if kind == "train":
            b += ns * np_ * 4 + B * np_ * 8
            f += B * ns * (2 * fft + 30 * np_)
        return {"bytes": b, "flops": f}
    atoms = c["cx"] * c["cy"] * c["cz"] * (8 if kind in ("tem", "fd") else 5)
    thick = c["cz"] * (5.43 if kind in ("tem", "fd") else 3.905) + 3.0
    if kind == "fd":
        return {"bytes": atoms * 16 + np_ * 8,
                "flops": c["steps"] * (6 * fft + 40 * np_)
                + _potential_flops(atoms * 4.5 / thick, c["ps"], 1, c["steps"])}
    ns = math.ceil(thick / c["dz"])
    waves = c.get("probes", 1) * c.get("configs", 1)
    f = waves * ns * (2 * fft + 12 * np_) + c.get("configs", 1) * _potential_flops(
        atoms, c["ps"], 1 if c.get("projected") else 20, 1 if c.get("projected") else (c["dz"] + 4.5) / c["dz"])
    b = atoms * 16.0
    if kind == "tem":
        b += np_ * (8 + 4 * c["images"])
        f += c["images"] * (fft + 60 * np_)
    elif kind == "cbed":
        b += np_ * 4
        f += waves * fft
    else:
        b += 12.0 * c["probes"] + (np_ * 4 if c["pacbed"] else 0)
        f += waves * fft / 2
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------- 64-bit values
# Quantities are 64-bit; what the method decides in 32 bits (bins, slice
# positions, the r^2 < 5 A^2 cutoff, frequencies, step sizes) is decided so.
def _physics(kV):
    """wavelength (A) and interaction constant (rad / V A)"""
    pi, V, e, rest = F(3.1415926), F(kV), F(1.6e-19), F(9.11e-31) * F(9e16)
    E = e * V * F(1000)
    lam = F(6.63e-34) * F(3e8) / np.sqrt(E * (F(2) * F(9.11e-31) * F(9e16) + E)) * F(1e10)
    sig = (F(2) * pi / (lam * V * F(1000))) * ((rest + E) / (F(2) * F(9.11e-31) * F(9e16) + E))
    return lam, sig


def _fd_step(kV, ps, nx, ny, stem):
    """stable finite-difference slice thickness"""
    pi, (lam, s2), V2 = F(3.1415926), _physics(kV), F(kV) * F(1000)
    p1, p2 = F(nx) / (F(2) * (F(ps) * F(nx))), F(ny) / (F(2) * (F(ps) * F(ny)))
    ke = F(0.666666) * (p1 * p1 + p2 * p2)
    a = (ke * ke * F(16) * pi * pi * pi * pi) - (F(32) * pi * pi * pi * ke * s2 * V2 / lam) + (
        F(16) * pi * pi * s2 * s2 * V2 * V2 / (lam * lam))
    b = F(16) * pi * pi * (ke - (s2 * V2 / (pi * lam)) - (F(1) / (F(4) * lam * lam)))
    step = (-b + np.sqrt(b * b - F(4) * a * F(3))) / (F(2) * a)
    step = F(0.99 * float(np.sqrt(step)))
    return F(0.06) if stem and step > 0.06 else step


class _Grid:
    """frequencies, band limit and k-space factors"""

    def __init__(self, kV, ps, nx, ny):
        self.nx, self.ny, self.ps = nx, ny, F(ps)
        self.lam, self.sigma = _physics(kV)
        kx, ky = self._k(nx), self._k(ny)
        half = [k[n // 2 - 1] * F(1) / F(2) for k, n in ((kx, nx), (ky, ny))]
        self.kmax = float(np.sqrt(min(F(float(h) ** 2) for h in half)))
        self.kx = torch.from_numpy(kx).cuda().double()[None, :]
        self.ky = torch.from_numpy(ky).cuda().double()[:, None]
        self.k2 = self.kx ** 2 + self.ky ** 2
        self.k = self.k2.sqrt()

    def _k(self, n):
        i = np.arange(n)
        return np.where(i > n // 2, i - n, i).astype(F) / (self.ps * F(n))

    def propagator(self, dz):
        return (self.k < self.kmax) * torch.exp(-1j * 3.14159265 * float(F(dz)) * float(self.lam) * self.k2)

    def band(self):
        return (self.k <= self.kmax).double()

    def probe(self, aperture, px, py, norm=None):
        """probe of the aperture (mrad) at pixel (px, py), over sum |psi|"""
        a = float(F(float(F(aperture)) * 0.001 / float(self.lam)))
        w = torch.fft.ifft2((self.k < a) * torch.exp(2j * 3.14159265 * float(self.ps) * (self.kx * px + self.ky * py)),
                            norm="forward")
        return w / (w.abs().sum() if norm is None else norm)

    def annulus(self, w, inner, outer):
        """sum |F(w)|^2 / N over inner <= lambda |k| < outer (mrad), per wave"""
        lo, hi = (float(F(v) * F(1e-3) / self.lam) for v in (inner, outer))
        return (torch.fft.fft2(w, norm="ortho").abs().square() * ((self.k >= lo) & (self.k < hi))).sum((-2, -1))


def _k0(x):
    """modified Bessel function K0 by the polynomials of Abramowitz and Stegun
    9.8.1, 9.8.5 and 9.8.6, which define the projected potential"""
    def poly(t, cs):
        r = torch.zeros_like(t)
        for v in reversed(cs):
            r = r * t + v
        return r
    s, u = x.clamp(max=2.0), x.clamp(min=2.0)
    i0 = poly((s / 3.75) ** 2, (1.0, 3.5156229, 3.0899424, 1.2067492, 0.2659732, 0.0360768, 0.0045813))
    small = -(s / 2).log() * i0 + poly((s / 2) ** 2, (-0.57721566, 0.42278420, 0.23069756, 0.03488590, 0.00262698,
                                                      0.00010750, 0.00000740))
    large = torch.exp(-u) / u.sqrt() * poly(2 / u, (1.25331414, -0.07832358, 0.02189568, -0.01062446, 0.00587872,
                                                    -0.00251540, 0.00053208))
    return torch.where(x <= 2.0, small, large)


class _Atoms:
    """atoms relative to the margins of their bounding box, by 1 A slab"""

    def __init__(self, Z, x, y, z, moved=(0, 0, 0)):
        lo, hi = [F(v.min() - F(2)) for v in (x, y, z)], [F(v.max() + F(2)) for v in (x, y, z)]
        x, y, z = ((v + d).astype(F) for v, d in zip((x, y, z), moved))
        self.H = hi[2] - lo[2]
        slab = np.floor(hi[2] - z).astype(np.int64)
        order = np.argsort(slab, kind="stable")
        self.slab = slab[order]
        self.xyz = [torch.from_numpy((v - m)[order]).cuda() for v, m in zip((x, y, z), lo)]
        fp = torch.from_numpy(fparams()).cuda().double()[torch.from_numpy(Z[order].astype(np.int64) - 1).cuda()]
        self.a, self.b, self.c, self.d = fp[:, 0:6:2], fp[:, 1:6:2], fp[:, 6:12:2], fp[:, 7:12:2]

    def slices(self, conventional_dz):
        return int(math.ceil(self.H / F(conventional_dz)))

    def potential(self, g, mode, z, dz=1.0, off=0.0):
        """real potential on the grid: 'integrated' over the 20 samples of the
        slice from z down to z - dz, 'projected' Bessel form of its atoms, or
        the 'plane' z"""
        z, dz, reach = F(z), F(dz), math.sqrt(5.0)
        top = self.H - z
        lo, hi = ((int(np.floor(top)), int(np.floor(top + dz)) - 1) if mode == "projected" else
                  (int(np.floor(top)) - 3, int(np.floor(top)) + 3))
        at = np.searchsorted(self.slab, [max(lo, 0), hi + 1])
        V = torch.zeros(g.ny * g.nx, dtype=torch.float64, device="cuda")
        w = int(reach / float(g.ps)) + 2
        step = max(1, 12_000_000 // (2 * w + 1) ** 2)
        for s in range(int(at[0]), int(at[1]), step):
            i = slice(s, min(s + step, int(at[1])))
            ax, ay, az = (v[i] for v in self.xyz)
            offs = torch.arange(-w, w + 1, device="cuda")
            ix, iy = (((v.double() - off) / float(g.ps)).round().long()[:, None] + offs for v in (ax, ay))
            dx, dy = ((((j.double() * float(g.ps) + off).float() - v[:, None])) for j, v in ((ix, ax), (iy, ay)))
            ok = ((ix >= 0) & (ix < g.nx))[:, None, :] & ((iy >= 0) & (iy < g.ny))[:, :, None]
            rxy = ((dy.double() ** 2)[:, :, None] + (dx * dx).double()[:, None, :]).float()
            n, jy, jx = torch.nonzero(ok & (rxy < 5.0), as_tuple=True)
            if not n.numel():
                continue
            flat, rxy = iy[n, jy] * g.nx + ix[n, jx], rxy[n, jy, jx]
            ca, cb, cc, cd = ([p[i][:, q][n] for q in range(3)] for p in (self.a, self.b, self.c, self.d))
            pi = 3.141592654
            if mode == "projected":
                r = rxy.double().sqrt().clamp(min=0.25)
                v = sum(300.8242834 * ca[q] * _k0(2 * pi * cb[q].sqrt() * r) +
                        150.4121417 * cc[q] / cd[q] * torch.exp(-pi * pi / cd[q] * r * r) for q in range(3))
            else:
                amp = [266.5157269 * cc[q] * cd[q] ** -1.5 for q in range(3)]
                dec = [2 * pi * cb[q].sqrt() for q in range(3)]
                wid = [pi * pi / cd[q] for q in range(3)]
                samples = [z] if mode == "plane" else [F(z - F(F(m) * dz) / F(20)) for m in range(1, 21)]
                v = torch.zeros_like(rxy, dtype=torch.float64)
                for zs in samples:
                    dd = (float(zs) - az.double()).float()[n]
                    r2 = (dd.double() ** 2 + rxy.double()).float()
                    r = r2.double().sqrt().clamp(min=0.25)
                    t = sum(150.4121417 * ca[q] * torch.exp(-dec[q] * r) for q in range(3)) / r
                    t += sum(amp[q] * torch.exp(-wid[q] * r * r) for q in range(3))
                    v += torch.where(r2 < 5.0, t, 0.0)
                if mode == "integrated":
                    v *= float(dz) / 20
            V.index_add_(0, flat, v)
        return V.view(g.ny, g.nx)

    def transmission(self, g, it, dz, projected, off=0.0):
        mode = "projected" if projected else "integrated"
        return torch.exp(1j * float(g.sigma) * self.potential(g, mode, self.H - F(dz) * F(it), dz, off))


def _conventional(atoms, g, w, dz, ns, projected=False, off=0.0):
    P = g.propagator(dz)
    for it in range(1, ns + 1):
        w = torch.fft.ifft2(P * torch.fft.fft2(w * atoms.transmission(g, it, dz, projected, off)))
    return w


def _finite_differences(atoms, g, w, dz, its):
    def filtered(v, m):
        return torch.fft.ifft2(m * torch.fft.fft2(v))
    dzf, lam, pi = float(dz), float(g.lam), 3.14159
    band, lap, al = g.band(), -4 * pi * pi * g.k2, 2 * pi * float(dz) / float(g.lam)
    before, now = w, filtered(w, g.propagator(dz))
    for it in its:
        V = filtered(atoms.potential(g, "plane", atoms.H - dz * F(it)), band).real
        u = 2 * now - dzf ** 2 * filtered(now, lap) - dzf ** 2 * 4 * pi * float(g.sigma) * V / lam * now
        before, now = now, filtered((u - (1 - 1j * al) * before) / (1 + 1j * al), band)
    return now


def _ctf_images(g, w, dfs, Cs, aperture):
    k = torch.fft.fft2(w, norm="ortho")
    lam, lim = float(g.lam), float((F(aperture) * F(0.001) / g.lam) ** 2)
    for df in dfs:
        chi = 3.1415926 * lam * g.k2 * (0.5 * Cs * lam * lam * g.k2 + float(df))
        yield torch.fft.ifft2((g.k2 < lim) * torch.exp(-1j * chi) * k, norm="ortho").abs().square()


def _philox(seed, config, n, axis):
    """first two words of Philox4x64-10 at counters (atom, config, axis, 0)"""
    def mulhi(a, b):
        m = np.uint64(0xFFFFFFFF)
        s = np.uint64(32)
        al, ah, bl, bh = a & m, a >> s, b & m, b >> s
        mid = (al * bl >> s) + (ah * bl & m) + (al * bh & m)
        return ah * bh + (ah * bl >> s) + (al * bh >> s) + (mid >> s)
    M0, M1 = np.uint64(0xD2E7470EE14C6C93), np.uint64(0xCA5A826395121157)
    c = [np.arange(n, dtype=np.uint64)] + [np.full(n, v, np.uint64) for v in (config, axis, 0)]
    k0, k1 = seed, 0x4D534C
    for _ in range(10):
        c = [mulhi(M1, c[2]) ^ c[1] ^ np.uint64(k0), M1 * c[2], mulhi(M0, c[0]) ^ c[3] ^ np.uint64(k1), M0 * c[0]]
        k0, k1 = (k0 + 0x9E3779B97F4A7C15) % 2 ** 64, (k1 + 0xBB67AE8584CAA73B) % 2 ** 64
    return c[0], c[1]


def _phonons(seed, config, n, sigma):
    """displacements of one frozen-phonon configuration"""
    out = []
    for axis in range(3):
        a, b = _philox(seed, config, n, axis)
        u1, u2 = ((a >> np.uint64(11)).astype(float) + 1) / 2 ** 53, (b >> np.uint64(11)).astype(float) / 2 ** 53
        out.append((float(F(sigma)) * np.sqrt(-2 * np.log(u1)) * np.cos(2 * np.pi * u2)).astype(F))
    return out


def _exact_diff(c, seed):
    V, psi, target = _diff_inputs(c, seed)
    g = _Grid(KV_DIFF, PS_DIFF, c["nx"], c["ny"])
    P, sig, ns = g.propagator(DZ_DIFF), float(g.sigma), c["slices"]
    inten = torch.empty(target.shape, dtype=torch.float64, device="cuda")
    grad = torch.zeros(V.shape, dtype=torch.float64, device="cuda")
    chunk = max(1, int(24e9 / (ns * c["nx"] * c["ny"] * 16)))
    for b in range(0, c["probes"], chunk):
        w, kept = psi[b:b + chunk].to(torch.complex128), []
        for i in range(ns):
            if c["kind"] == "train":
                kept.append(w)
            w = torch.fft.ifft2(P * torch.fft.fft2(torch.exp(1j * sig * V[i].double()) * w))
        inten[b:b + chunk] = w.abs().square()
        if c["kind"] == "infer":
            continue
        G = 4 * (inten[b:b + chunk] - target[b:b + chunk].double()) * w
        for i in range(ns - 1, -1, -1):
            G = torch.fft.ifft2(P.conj() * torch.fft.fft2(G)) * torch.exp(-1j * sig * V[i].double())
            grad[i] -= sig * (G.conj() * kept.pop()).imag.sum(0)
    return {"intensity": inten, "grad": grad} if c["kind"] == "train" else {"intensity": inten}


def exact(case, seed):
    c = case
    kind = c["kind"]
    if kind in ("train", "infer"):
        return _exact_diff(c, seed)
    if kind == "serve":
        out = []
        for j in _serving_jobs(c, seed):
            g, atoms = _Grid(SERVE["kV"], SERVE["ps"], j.n, j.n), _Atoms(j.Z, j.x, j.y, j.z)
            w = torch.ones(j.n, j.n, dtype=torch.complex128, device="cuda")
            if j.nprobe:
                w = torch.stack([g.probe(SERVE["aperture"], int(a), int(b)) for a, b in zip(j.posx, j.posy)])
            if j.method == FD:
                step = _fd_step(SERVE["kV"], SERVE["ps"], j.n, j.n, j.nprobe > 0)
                w = _finite_differences(atoms, g, w, step, range(1, j.nslices + 1))
            else:
                w = _conventional(atoms, g, w, SERVE["dz"], j.nslices)
            out.append(g.annulus(w, *SERVE["adf"]) if j.nprobe else w)
        return out
    spec = _specimen(c, seed)
    nx, ny = c["nx"], c["ny"]
    if kind in ("tem", "fd"):
        g, atoms = _Grid(c["kV"], c["ps"], nx, ny), _Atoms(*spec)
        w = torch.ones(ny, nx, dtype=torch.complex128, device="cuda")
        if kind == "fd":
            step = _fd_step(c["kV"], c["ps"], nx, ny, False)
            first = int(0.5 * float(atoms.H) / float(step))
            return {"exit": _finite_differences(atoms, g, w, step, range(first, first + c["steps"]))}
        out = {"exit": _conventional(atoms, g, w, c["dz"], atoms.slices(c["dz"]), c["projected"], 2.0)}
        if c["images"]:
            im = torch.stack(list(_ctf_images(g, out["exit"], _defoci(c), CS_TEM, 20.0)))
            out["image"] = im[0] if c["images"] == 1 else im
        return out
    g = _Grid(300.0, c["ps"], nx, ny)
    if kind == "cbed":
        adf, tds = [], torch.zeros(ny, nx, dtype=torch.float64, device="cuda")
        for cfg in range(c["configs"]):
            atoms = _Atoms(*spec, _phonons(seed, cfg, spec[0].size, THERMAL))
            w = _conventional(atoms, g, g.probe(25.0, nx // 2 + 3, ny // 2 - 5), c["dz"], atoms.slices(c["dz"]))
            tds += torch.fft.fftshift(torch.fft.fft2(w).abs())
            adf.append(g.annulus(w, 20.0, 200.0))
        return {"adf": torch.stack(adf), "tds": tds}
    px, py = _positions(c, seed)
    adf = torch.zeros(c["probes"], dtype=torch.float64, device="cuda")
    pac = torch.zeros(ny, nx, dtype=torch.float64, device="cuda")
    norm = torch.fft.ifft2((g.k < float(F(0.025 / float(g.lam)))).to(torch.complex128), norm="forward").abs().sum()
    for cfg in range(c["configs"]):
        moved = _phonons(seed, cfg, spec[0].size, c["sigma"]) if c["sigma"] > 0 else (0, 0, 0)
        atoms = _Atoms(*spec, moved)
        ns = atoms.slices(c["dz"])
        t = [atoms.transmission(g, it, c["dz"], c["projected"]) for it in range(1, ns + 1)]
        P = g.propagator(c["dz"])
        for b in range(0, c["probes"], 128):
            w = torch.stack([g.probe(25.0, int(a), int(q), norm) for a, q in zip(px[b:b + 128], py[b:b + 128])])
            for v in t:
                w = torch.fft.ifft2(P * torch.fft.fft2(w * v))
            adf[b:b + 128] += g.annulus(w, 20.0, 200.0) / c["configs"]
            if c["pacbed"]:
                pac += torch.fft.fft2(w).abs().square().sum(0) / (c["configs"] * c["probes"])
    return {"adf": adf, "pacbed": pac} if c["pacbed"] else {"adf": adf}
