"""Workloads by which the framework's speed is measured.

Each case is one call (or one short chain of calls) that a user's program
makes through the public entry points: the drop-in shot, one pattern on a
detector by the direct sum, a wavelength spectrum, a batch of molecules or
orientations, the non-uniform FFT forms of these, a gradient step and the
detector chain. Sizes are those of the benchmark configurations and of the
tests, spread over their ranges; molecules are C/N/O/S balls of protein
density (5 nm radius at 5000 atoms), detectors 75 um or 20 um pixels.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import spsim
from spsim_amd import _lib
from spsim_amd import device as dv
from spsim_amd import torch_ops as to

DEV = "cuda"

# Cromer-Mann rows of the elements used here: a1..a4, b1..b4 (A^2), c.
ROWS = {6: (2.31, 1.02, 1.5886, 0.865, 20.8439, 10.2075, 0.5687, 51.6512, 0.2156),
        7: (12.2126, 3.1322, 2.0125, 1.1663, 0.0057, 9.8933, 28.9975, 0.5826, -11.529),
        8: (3.0485, 2.2868, 1.5463, 0.867, 13.2771, 5.7011, 0.3239, 32.9089, 0.2508),
        16: (6.9053, 5.2034, 1.4379, 1.5863, 1.4679, 22.2151, 0.2536, 56.172, 0.8669)}


def listed():
    return [
        # one small shot through the drop-in C API, host arrays in and out: where calls and launches count
        {"name": "shot_small", "kind": "shot", "natoms": 500, "nx": 64, "ny": 64, "pixel": 3e-4, "distance": 0.1,
         "wavelength": 0.2e-9, "bin": 1},
        # one small protein on a quarter-megapixel quadrant, amplitudes kept: the ordinary single call
        {"name": "grid_256", "kind": "grid", "natoms": 5000, "nx": 256, "ny": 256, "pixel": 75e-6, "distance": 0.1,
         "wavelength": 0.2e-9, "shift": 0.0, "rot": False, "b": False, "keep_F": True},
        # an off-centre rectangular detector of odd sizes, the molecule turned: no symmetry anywhere
        {"name": "grid_offcentre", "kind": "grid", "natoms": 3001, "nx": 333, "ny": 217, "pixel": 75e-6,
         "distance": 0.1, "wavelength": 0.15e-9, "shift": 1.3e-3, "rot": True, "b": False, "keep_F": True},
        # a large assembly with a B factor on every atom, a megapixel: the largest single pattern
        {"name": "grid_1024_b", "kind": "grid", "natoms": 100_000, "nx": 1024, "ny": 1024, "pixel": 75e-6,
         "distance": 0.1, "wavelength": 0.15e-9, "shift": 0.0, "rot": False, "b": True, "keep_F": True},
        # molecules of very different sizes, one orientation each, in one plan
        {"name": "batch_mixed", "kind": "batch", "nmol": 16, "natoms": 2000, "natoms_max": 100_000, "npat": 16,
         "n": 512, "pixel": 75e-6, "distance": 0.1, "wavelength": 0.2e-9},
        # one molecule in many orientations at long wavelength: a single-particle data set
        {"name": "batch_orientations", "kind": "batch", "nmol": 1, "natoms": 50_000, "natoms_max": 50_000, "npat": 8,
         "n": 1024, "pixel": 20e-6, "distance": 0.05, "wavelength": 1.3e-9},
        # a few per cent of bandwidth: the wavelength spectrum of one pattern
        {"name": "spectrum_512", "kind": "spectrum", "natoms": 20_000, "n": 512, "pixel": 75e-6, "distance": 0.1,
         "wavelength": 0.2e-9, "bandwidth": 0.02, "samples": 5},
        # refinement: intensities, Poisson likelihood and gradients of positions and B factors
        {"name": "fit_512", "kind": "fit", "natoms": 20_000, "n": 512, "pixel": 75e-6, "distance": 0.1,
         "wavelength": 0.2e-9},
        # the large single pattern by the non-uniform FFT
        {"name": "nufft_1024", "kind": "nufft", "natoms": 100_000, "n": 1024, "pixel": 75e-6, "distance": 0.1,
         "wavelength": 0.15e-9, "b": False, "eps": 1e-6},
        # orientations of one molecule over one set of NUFFT grids
        {"name": "nufft_orientations", "kind": "nufft_batch", "natoms": 50_000, "npat": 8, "n": 1024, "pixel": 20e-6,
         "distance": 0.05, "wavelength": 1.3e-9, "eps": 1e-6},
        # many molecules through the NUFFT in one call
        {"name": "nufft_molecules", "kind": "nufft_molecules", "nmol": 24, "natoms": 2000, "natoms_max": 50_000,
         "n": 512, "pixel": 75e-6, "distance": 0.1, "wavelength": 0.2e-9, "eps": 1e-6},
        # detector chain of a stack of patterns, 4 x 4 binning, binned outputs only
        {"name": "chain_binned", "kind": "chain", "npat": 64, "nx": 1024, "ny": 1024, "bin": 4, "binned": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["shot", "grid", "grid", "batch", "spectrum", "fit", "nufft", "nufft_batch", "nufft_molecules",
                       "chain"])
    optics = rng.choice([{"pixel": 75e-6, "distance": 0.1, "wavelength": 0.2e-9},
                         {"pixel": 75e-6, "distance": 0.1, "wavelength": 0.15e-9},
                         {"pixel": 20e-6, "distance": 0.05, "wavelength": 1.3e-9}])
    if kind == "shot":
        n = 2 * _log(rng, 24, 80)
        return {"kind": kind, "natoms": _log(rng, 200, 4000), "nx": n, "ny": max(32, n - 2 * rng.randrange(0, 8)),
                "pixel": 3e-4, "distance": 0.1, "wavelength": 0.2e-9, "bin": rng.choice([1, 2])}
    if kind == "grid":
        nx = _log(rng, 96, 900)
        return {"kind": kind, "natoms": _log(rng, 1000, 60_000), "nx": nx,
                "ny": nx if rng.random() < 0.5 else max(64, nx - rng.randrange(1, nx // 2)), **optics,
                "shift": rng.choice([0.0, 0.0, 0.7e-3]), "rot": rng.random() < 0.5, "b": rng.random() < 0.5,
                "keep_F": rng.random() < 0.5}
    if kind == "batch":
        nmol = rng.choice([1, 8, 24])
        lo = _log(rng, 1500, 6000)
        return {"kind": kind, "nmol": nmol, "natoms": lo, "natoms_max": lo if nmol == 1 else 6 * lo,
                "npat": nmol if nmol > 1 else rng.choice([5, 16, 40]), "n": rng.choice([255, 384, 512]), **optics}
    if kind == "spectrum":
        return {"kind": kind, "natoms": _log(rng, 1000, 20_000), "n": _log(rng, 128, 512), **optics,
                "bandwidth": rng.choice([0.005, 0.02, 0.06]), "samples": rng.choice([3, 5, 11])}
    if kind == "fit":
        return {"kind": kind, "natoms": _log(rng, 1000, 20_000), "n": _log(rng, 128, 512), **optics}
    if kind == "nufft":
        return {"kind": kind, "natoms": _log(rng, 2000, 100_000), "n": _log(rng, 200, 1024), **optics,
                "b": rng.random() < 0.4, "eps": rng.choice([1e-6, 1e-6, 1e-4])}
    if kind == "nufft_batch":
        return {"kind": kind, "natoms": _log(rng, 2000, 50_000), "npat": rng.choice([3, 7]), "n": _log(rng, 200, 1024),
                **optics, "eps": 1e-6}
    if kind == "nufft_molecules":
        lo = _log(rng, 1000, 5000)
        return {"kind": kind, "nmol": rng.choice([6, 20]), "natoms": lo, "natoms_max": 8 * lo, "n": _log(rng, 200, 512),
                **optics, "eps": 1e-6}
    n = _log(rng, 128, 1024)
    b = rng.choice([1, 2, 4, 5])
    return {"kind": "chain", "npat": rng.choice([1, 9, 40]), "nx": n // b * b, "ny": max(b, (n * 3 // 4) // b * b),
            "bin": b, "binned": rng.random() < 0.6}


# ---- inputs ---------------------------------------------------------------


def _molecule(natoms, rng, with_b):
    """Atoms uniform in a ball of protein density; (Z, positions in m, B or None)."""
    radius = 5e-9 * (natoms / 5000.0) ** (1.0 / 3.0)
    pos = np.empty((0, 3))
    while len(pos) < natoms:
        c = rng.uniform(-radius, radius, size=(2 * natoms + 64, 3))
        pos = np.concatenate([pos, c[(c * c).sum(1) <= radius * radius]])
    Z = rng.choice(np.array([6, 7, 8, 16], np.int32), size=natoms, p=[0.62, 0.17, 0.20, 0.01])
    B = rng.uniform(10.0, 40.0, size=natoms).astype(np.float32) if with_b else None
    return Z.astype(np.int32), pos[:natoms].astype(np.float32), B


def _sizes(case):
    """Atom counts of the case's molecules, evenly spaced in their logarithm."""
    k, lo, hi = case["nmol"], case["natoms"], case.get("natoms_max", case["natoms"])
    return [int(round(lo * (hi / lo) ** (i / max(1, k - 1)))) for i in range(k)]


def _rotations(count, rng):
    q = rng.normal(size=(count, 4))
    w, x, y, z = (q / np.linalg.norm(q, axis=1, keepdims=True)).T
    return np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                     2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                     2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], 1).reshape(count, 3, 3)


def _f32(v):
    return np.float32(v).item()


def _geometry(case):
    nx, ny = case.get("nx", case.get("n")), case.get("ny", case.get("n"))
    return nx, ny, _f32(nx * case["pixel"]), _f32(ny * case["pixel"]), _f32(case.get("shift", 0.0))


def _q_list(case):
    """The detector's Ewald-sphere q list [ny*nx, 3], FP32, on the GPU."""
    nx, ny, width, height, shift = _geometry(case)
    return dv.hkl_detector(nx, ny, width, height, case["distance"], case["wavelength"], center_x=shift,
                           center_y=-0.5 * shift, device=DEV)


def _molecules(case, seed, with_b=False):
    rng = np.random.default_rng(seed)
    mols = [_molecule(n, rng, with_b) for n in (_sizes(case) if "nmol" in case else [case["natoms"]])]
    return mols, _rotations(case.get("npat", case.get("nmol", 1)), rng)


class _Plan:
    """A batched plan, kept by the program for as long as it runs patterns."""

    def __init__(self, case, mols, rots):
        vp = lambda a: a.ctypes.data_as(C.c_void_p)  # noqa: E731
        n, npat = case["n"], case["npat"]
        offs = np.concatenate([[0], np.cumsum([len(m[0]) for m in mols])]).astype(np.int32)
        Z = np.concatenate([m[0] for m in mols])
        pos = np.ascontiguousarray(np.concatenate([m[1] for m in mols]))
        which = np.ascontiguousarray(np.arange(npat) % len(mols), np.int32)
        R = np.ascontiguousarray(rots.reshape(npat, 9))
        q = np.ascontiguousarray(_q_list(case).cpu().numpy())
        self.handle = C.c_void_p()
        _lib.check(_lib.load().spsim_hip_batch_create(vp(q), n, n, len(mols), vp(offs), vp(Z), vp(pos), None, None, 0,
                                                      npat, vp(which), vp(R), None, 0.0, None, C.byref(self.handle)),
                   "spsim_hip_batch_create")

    def __del__(self):
        if self.handle:
            torch.cuda.synchronize()
            _lib.load().spsim_hip_batch_destroy(self.handle)


def _chain_params(case):
    nx, ny, b = case["nx"], case["ny"], case["bin"]
    return dv.detector_params(nx=nx, ny=ny, bin_x=b, bin_y=b, width=_f32(nx * 20e-6), height=_f32(ny * 20e-6),
                              distance=0.05, pixel_width=20e-6, pixel_height=20e-6, beam_intensity=1e25,
                              quantum_efficiency=0.15, wavelength=1.3e-9, electron_hole_production_energy=5.8e-19,
                              dark_current=0.1, exposure_time=1e-13, readout_noise=10.0, linear_full_well=2e5,
                              maximum_value=65535.0)


def _intensities(case, seed):
    """Speckle: exponentially distributed around a mean that falls steeply from the beam outwards."""
    nx, ny, npat = case["nx"], case["ny"], case["npat"]
    g = torch.Generator(device=DEV).manual_seed(seed)
    y = torch.linspace(-1, 1, ny, device=DEV)[:, None]
    x = torch.linspace(-1, 1, nx, device=DEV)[None, :]
    mean = 2e6 / (1.0 + 400.0 * (x * x + y * y)) ** 2 + 20.0
    u = torch.rand((npat, ny, nx), device=DEV, generator=g)
    return (-torch.log1p(-u * 0.999999) * mean).reshape(npat, ny * nx).contiguous()


def _counts(case, seed, q, mols):
    """Counts that a refinement fits: Poisson draws around another conformation's pattern."""
    (Z, pos, B), rng = mols[0], np.random.default_rng(seed + 77)
    moved = (pos + rng.normal(0, 2e-11, size=pos.shape)).astype(np.float32)
    I0 = _intensity64(_sum64(q.double(), (Z, moved, B))).float()
    K = torch.full_like(I0, 10.0 / (40.0 * case["natoms"]))  # about ten photons on an average pixel
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.poisson(K * I0, generator=g), K


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "chain":
        s.update(det=_chain_params(case), I=_intensities(case, seed), seed=seed)
        return s
    mols, rots = _molecules(case, seed, with_b=kind == "fit" or case.get("b", False))
    if kind == "shot":
        o = spsim.set_defaults()
        d, e = o.detector, o.experiment
        d.nx, d.ny, d.nz = case["nx"], case["ny"], 1
        d.pixel_width = d.pixel_height = case["pixel"]
        _, _, d.width, d.height, _ = _geometry(case)
        d.distance, e.wavelength = case["distance"], case["wavelength"]
        d.binning_x = d.binning_y = case["bin"]
        e.beam_intensity = 2e23
        d.quantum_efficiency, d.electron_hole_production_energy = 0.5, 5.8e-19
        d.readout_noise, d.dark_current, e.exposure_time = 3.0, 0.1, 1e-13
        d.linear_full_well, d.maximum_value = 2e5, 65535.0
        o.verbosity_level = 0
        s.update(opts=o, mol=spsim.get_molecule_from_atoms(mols[0][0], mols[0][1]), seed=seed)
        return s
    s["ff"] = dv.form_factor_table(device=DEV)
    if kind == "batch":
        s["plan"] = _Plan(case, mols, rots)
        s["I"] = torch.empty((case["npat"], case["n"] ** 2), dtype=torch.float32, device=DEV)
        return s
    s["q"] = _q_list(case)
    if kind == "fit":
        Z, pos, B = mols[0]
        s["layout"] = to.SpeciesLayout(Z, torch.device(DEV))
        s["pos"] = torch.from_numpy(pos).to(DEV).requires_grad_()
        s["B"] = torch.from_numpy(B).to(DEV).requires_grad_()
        s["y"], s["K"] = _counts(case, seed, s["q"], mols)
        return s
    if kind == "nufft_molecules":
        s["mols"] = dv.DeviceMolecules([dv.pack_atoms(Z, pos) for Z, pos, _ in mols], DEV)
    else:
        s["atoms"] = dv.DeviceAtoms(dv.pack_atoms(*mols[0][:2], atom_b=mols[0][2]), DEV)
    s["rots"] = rots
    if kind == "spectrum":
        s["samples"] = dv.spectrum_samples(case["wavelength"], case["bandwidth"], case["samples"])
    return s


# ---- one pass --------------------------------------------------------------


def _shot(s):
    o, n = s["opts"], s["case"]["nx"] * s["case"]["ny"]
    spsim.sp_srand(s["seed"] % (1 << 31))
    pat = spsim.simulate_shot(s["mol"], o)
    d = o.detector
    nb = (d.nx // d.binning_x) * (d.ny // d.binning_y)
    out = {"ints": spsim.float_array(pat.ints, n), "F": spsim.float_array(C.cast(pat.F, C.POINTER(C.c_float)), 2 * n)}
    for k in ("thomson_correction", "solid_angle", "photons_per_pixel", "photon_count", "electrons_per_pixel"):
        out[k] = spsim.float_array(getattr(d, k), n)
    for k in ("real_output", "noiseless_output"):
        out[k] = spsim.float_array(getattr(d, k), nb)
    spsim.free_diffraction_pattern(pat)
    spsim.free_output_in_options(o)
    return out


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "shot":
        return _shot(s)
    if kind == "grid":
        F, I = dv.structure_factor_grid(s["q"], case["nx"], case["ny"], s["atoms"], s["ff"], want_F=case["keep_F"],
                                        R=s["rots"][0] if case["rot"] else None)
        return {"F": F, "I": I} if case["keep_F"] else {"I": I}
    if kind == "batch":
        _lib.check(_lib.load().spsim_hip_batch_run(s["plan"].handle, None, C.c_void_p(s["I"].data_ptr()), 0,
                                                   C.c_void_p(torch.cuda.current_stream().cuda_stream)),
                   "spsim_hip_batch_run")
        return {"I": s["I"]}
    if kind == "spectrum":
        F, I = dv.structure_factor_spectrum(s["q"], s["atoms"], s["ff"], *s["samples"])
        return {"F": F, "I": I}
    if kind == "fit":
        s["pos"].grad = s["B"].grad = None
        I = to.intensity(s["pos"], s["q"], s["layout"], s["ff"], atom_b=s["B"])
        loss = to.poisson_nll(I, s["y"], s["K"])
        loss.backward()
        return {"loss": loss.detach().float(), "I": I.detach(), "pos_grad": s["pos"].grad, "b_grad": s["B"].grad}
    if kind == "nufft":
        F, I, _ = dv.structure_factor_nfft(s["q"], s["atoms"], s["ff"], eps=case["eps"])
        return {"F": F, "I": I}
    if kind == "nufft_batch":
        _, I, _ = dv.structure_factor_nfft_batch(s["q"], s["atoms"], s["ff"], s["rots"], eps=case["eps"], want_F=False)
        return {"I": I}
    if kind == "nufft_molecules":
        _, I = dv.structure_factor_nfft_molecules(s["q"], s["mols"], s["ff"], rots=s["rots"], eps=case["eps"],
                                                  want_F=False)
        return {"I": I}
    if case["binned"]:
        return dv.detector_chain_binned(s["det"], s["I"], npatterns=case["npat"], seed=s["seed"])
    return dv.detector_chain(s["det"], s["I"], npatterns=case["npat"], seed=s["seed"],
                             outputs=("photons", "count", "real_output", "noiseless_output"))


def work(case):
    """Inputs read once, outputs written once; one complex exponential and
    weight (about 16 operations) per atom and per output pixel, which every
    method of evaluating the sums has to form."""
    kind = case["kind"]
    if kind == "chain":
        raw = case["npat"] * case["nx"] * case["ny"]
        nb = raw // case["bin"] ** 2
        out = 2 * nb if case["binned"] else 2 * raw + 2 * nb
        return {"bytes": 4 * (raw + out), "flops": 8 * raw}
    nx, ny = case.get("nx", case.get("n")), case.get("ny", case.get("n"))
    npix, npat = nx * ny, case.get("npat", case.get("nmol", 1))
    atoms = sum(_sizes(case)) if "nmol" in case else case["natoms"]
    per_pixel = {"shot": 12 + 5 * 4 + 8 // case.get("bin", 1) ** 2, "grid": 12 if case.get("keep_F") else 4,
                 "spectrum": 12, "nufft": 12, "fit": 4 + 8}.get(kind, 4)
    b = 12 * npix + 16 * atoms + per_pixel * npix * npat
    f = 16 * (atoms + npix * npat)
    if kind == "fit":
        b, f = b + 4 * atoms + 16 * atoms, 2 * f
    return {"bytes": b, "flops": f}


# ---- the same outputs in 64 bits ---------------------------------------------


def _detector64(case):
    """The FP32 q list of the detector, from its FP64 geometry, widened again."""
    nx, ny, width, height, shift = _geometry(case)
    distance, lam = _f32(case["distance"]), _f32(case["wavelength"])
    x = ((np.arange(nx) - (nx - 1.0) / 2.0) / nx) * width - shift
    y = ((np.arange(ny) - (ny - 1.0) / 2.0) / ny) * height - _f32(-0.5 * shift)
    px, py = np.meshgrid(x, y)
    p = np.sqrt(px * px + py * py + distance * distance)
    q = np.stack([px / p, py / p, distance / p - 1.0], -1).reshape(-1, 3) * (1.0 / lam)
    return torch.from_numpy(q.astype(np.float32)).to(DEV).double()


def _factor(z, s2):
    c = [_f32(v) for v in ROWS[int(z)]]
    return sum(c[i] * torch.exp(-c[4 + i] * s2) for i in range(4)) + c[8]


def _sum64(q, mol, R=None, scales=(1.0,), weights=(1.0,)):
    """F at every q: the direct sum in FP64, in chunks of pixels and atoms."""
    Z, pos, B = mol
    r = torch.from_numpy(pos).to(DEV).double()
    if R is not None:
        r = r @ torch.from_numpy(np.ascontiguousarray(R)).to(DEV)  # (R q).r = q.(R^T r)
    Zt = torch.from_numpy(Z).to(DEV)
    Bt = None if B is None else torch.from_numpy(B).to(DEV).double()
    F = torch.zeros((len(q), 2), dtype=torch.float64, device=DEV)
    s2 = (q * q).sum(1) * 2.5e-21
    for z in np.unique(Z):
        idx = torch.nonzero(Zt == int(z)).flatten()
        f = _factor(z, s2)
        for part in idx.split(16384):
            rt = r[part].T.contiguous()
            for p0 in range(0, len(q), 8192):
                t = q[p0:p0 + 8192] @ rt
                e = None if Bt is None else torch.exp(-s2[p0:p0 + 8192, None] * Bt[part][None, :])
                for sc, w in zip(scales, weights):
                    ph = t * sc if sc != 1.0 else t
                    ph = (ph - torch.round(ph)) * (2.0 * math.pi)
                    re, im = torch.cos(ph), torch.sin(ph)
                    if e is not None:
                        re, im = re * e, im * e
                    F[p0:p0 + 8192, 0] += w * f[p0:p0 + 8192] * re.sum(1)
                    F[p0:p0 + 8192, 1] -= w * f[p0:p0 + 8192] * im.sum(1)
    return F


def _intensity64(F):
    return (F * F).sum(1)


def _gradients64(q, mol, F, g):
    """dL/dr and dL/dB for dL/dI = g, by the closed form, in FP64."""
    Z, pos, B = mol
    r = torch.from_numpy(pos).to(DEV).double()
    Bt = torch.from_numpy(B).to(DEV).double()
    Zt = torch.from_numpy(Z).to(DEV)
    s2 = (q * q).sum(1) * 2.5e-21
    gp, gb = torch.zeros_like(r), torch.zeros_like(Bt)
    for z in np.unique(Z):
        idx = torch.nonzero(Zt == int(z)).flatten()
        A = 2.0 * g[:, None] * _factor(z, s2)[:, None] * F  # (Ar, Ai)
        for part in idx.split(4096):
            for p0 in range(0, len(q), 16384):
                sl = slice(p0, p0 + 16384)
                t = r[part] @ q[sl].T.contiguous()
                t = (t - torch.round(t)) * (2.0 * math.pi)
                e = torch.exp(-Bt[part][:, None] * s2[sl][None, :])
                c, s = torch.cos(t) * e, torch.sin(t) * e
                u = s * A[sl, 0] + c * A[sl, 1]
                gp[part] -= 2.0 * math.pi * (u @ q[sl])
                gb[part] -= (c * A[sl, 0] - s * A[sl, 1]) @ s2[sl]
    return gp, gb


def _chain64(p, photons, nx, ny, bins):
    """Noiseless binned output of per-pixel photons [npat, ny*nx]."""
    gain = _f32(p.quantum_efficiency) * (1.98644521e-25 / p.wavelength / p.electron_hole_production_energy)
    gain *= p.maximum_value / p.linear_full_well
    v = (photons * gain).reshape(-1, ny // bins, bins, nx // bins, bins)
    return v.sum((2, 4)).reshape(len(photons), -1)


def _solid_angle64(p):
    x = ((torch.arange(p.nx, dtype=torch.float64, device=DEV) - (p.nx - 1.0) / 2.0) / p.nx) * p.width
    y = ((torch.arange(p.ny, dtype=torch.float64, device=DEV) - (p.ny - 1.0) / 2.0) / p.ny) * p.height
    tan = torch.sqrt(x[None, :] ** 2 + y[:, None] ** 2) / p.distance
    return (p.pixel_width * p.pixel_height / p.distance ** 2 * torch.cos(torch.atan(tan)) ** 3).reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "chain":
        p, I = _chain_params(case), _intensities(case, seed).double()
        photons = (2.81794e-15 ** 2) * _solid_angle64(p) * I * p.beam_intensity
        out = {"real_output": None, "noiseless_output": _chain64(p, photons, case["nx"], case["ny"], case["bin"])}
        return out if case["binned"] else {"photons": photons, "count": None, **out}
    mols, rots = _molecules(case, seed, with_b=kind == "fit" or case.get("b", False))
    q = _detector64(case)
    if kind == "shot":
        F = _sum64(q, mols[0])
        I = _intensity64(F)
        nx, ny, width, height, _ = _geometry(case)
        p = dv.detector_params(nx=nx, ny=ny, width=width, height=height, distance=case["distance"],
                               pixel_width=case["pixel"], pixel_height=case["pixel"], wavelength=case["wavelength"],
                               beam_intensity=2e23, quantum_efficiency=0.5, electron_hole_production_energy=5.8e-19,
                               linear_full_well=2e5, maximum_value=65535.0)
        om = _solid_angle64(p)
        th = torch.full_like(om, 2.81794e-15 ** 2)
        ph = th * om * I * p.beam_intensity
        res = {"ints": I, "F": F.reshape(-1), "thomson_correction": th, "solid_angle": om, "photons_per_pixel": ph,
               "noiseless_output": _chain64(p, ph[None], nx, ny, case["bin"])[0]}
        res = {k: v.cpu().numpy() for k, v in res.items()}
        noisy = {k: None for k in ("photon_count", "electrons_per_pixel", "real_output")}
        return {k: {**res, **noisy}[k] for k in ("ints", "F", "thomson_correction", "solid_angle", "photons_per_pixel",
                                                 "photon_count", "electrons_per_pixel", "real_output",
                                                 "noiseless_output")}
    if kind in ("batch", "nufft_batch", "nufft_molecules"):
        return {"I": torch.stack([_intensity64(_sum64(q, mols[i % len(mols)], R)) for i, R in enumerate(rots)])}
    if kind == "fit":
        F = _sum64(q, mols[0])
        I = _intensity64(F)
        y, K = _counts(case, seed, q.float(), mols)
        y, K = y.double(), K.double()
        lam = torch.clamp(K * I, min=1e-30)
        loss = (lam - torch.where(y > 0, y * torch.log(lam), torch.zeros_like(y))).sum()
        gp, gb = _gradients64(q, mols[0], F, K * (1.0 - y / lam))
        return {"loss": loss, "I": I, "pos_grad": gp, "b_grad": gb}
    if kind == "spectrum":
        lam, bw, ns = case["wavelength"], case["bandwidth"], case["samples"]
        k = lam * (1 - bw / 2) + np.arange(ns) / (ns - 1.0) * lam * bw
        w = np.exp(-0.5 * ((k - lam) / (lam * bw / 4)) ** 2)
        F = _sum64(q, mols[0], scales=lam / k, weights=w / w.sum())
    else:
        F = _sum64(q, mols[0], R=rots[0] if case.get("rot") else None)
    I = _intensity64(F)
    return {"F": F, "I": I} if case.get("keep_F", True) else {"I": I}
