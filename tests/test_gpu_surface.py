"""Interpolation over the detector surface (csrc/hip/surface.hip), which large
patterns on a smooth list take with the automatic tile, against the FP64 oracle
and against the direct kernels (an explicit tile).

Tolerance: the interpolation's own error is below 3e-8 of |F| (normwise), the
FP32 sums' error 1e-7 of F and 2e-7 of I, as for the direct kernels: 4e-7
leaves a factor of two."""
import numpy as np
import pytest

import oracle
from spsim_amd import device as dv
from spsim_amd import workloads as wl
from tests.conftest import oracle_threads, rel_l2

pytestmark = pytest.mark.gpu

TOL = 4e-7


def _run(gpu, hkl, nx, ny, Z, pos, atom_b=None, amp=None, B=0.0, R=None, tile=None):
    import torch

    atoms = dv.DeviceAtoms(dv.pack_atoms(Z, pos, atom_b=atom_b, amp=amp), gpu)
    q = torch.from_numpy(np.ascontiguousarray(hkl, np.float32)).to(gpu)
    F, I = dv.structure_factor_grid(q, nx, ny, atoms, dv.form_factor_table(device=gpu), B=B, R=R, tile=tile)
    torch.cuda.synchronize()
    F = F.cpu().numpy()
    return F[:, 0] + 1j * F[:, 1], I.cpu().numpy()


def _list(nx, ny, pixel=75e-6, distance=0.1, wavelength=0.2e-9, cx=0.0, cy=0.0, spherical=0):
    return oracle.hkl_detector(nx, ny, np.float32(nx * pixel).item(), np.float32(ny * pixel).item(), distance, cx, cy,
                               spherical, wavelength)


# (nx, ny, atoms, radius, list, per-atom B, rotation): the shortest sides, odd
# and unequal ones, one that ends inside every tile, a long wavelength (fewest
# nodes), a wide angle (most nodes), a molecule far from the origin
CASES = [
    (64, 64, 60_000, 4e-9, {"pixel": 3e-4}, False, False),
    (65, 67, 50_000, 5e-9, {}, True, True),
    (333, 217, 4_000, 5e-9, {"cx": 1.3e-3, "wavelength": 0.15e-9}, False, True),
    (129, 257, 9_000, 6e-9, {}, True, False),
    (400, 400, 3_000, 5e-9, {"pixel": 20e-6, "distance": 0.05, "wavelength": 1.3e-9}, False, True),
    (512, 512, 3_000, 14e-9, {"pixel": 150e-6}, True, True),
    (300, 300, 3_000, 4e-9, {"spherical": 1}, False, False),
]


@pytest.mark.parametrize("nx,ny,natoms,radius,geometry,with_b,rotated", CASES)
def test_interpolated_pattern_vs_f64_and_direct(gpu, nx, ny, natoms, radius, geometry, with_b, rotated):
    rng = np.random.default_rng(nx * 1000 + ny)
    Z, pos, b = wl.random_molecule(natoms, radius, rng, atom_b_range=(5.0, 40.0))
    pos = (pos + np.array([3e-9, -2e-9, 1e-9])).astype(np.float32)
    Z[: natoms // 50] = 1
    b = b if with_b else None
    R = wl.uniform_rotations(1, rng)[0] if rotated else None
    hkl = _list(nx, ny, **geometry)
    F, I = _run(gpu, hkl, nx, ny, Z, pos, atom_b=b, B=2.0, R=R)
    Fd, Id = _run(gpu, hkl, nx, ny, Z, pos, atom_b=b, B=2.0, R=R, tile=dv.make_tile(1, 256, 0))
    assert not np.array_equal(I, Id)  # the interpolation ran
    # the corners, the edges and a random sample
    sub = np.unique(np.concatenate([[0, nx - 1, nx * ny - nx, nx * ny - 1], np.arange(0, nx * ny, 7 * nx),
                                    rng.choice(nx * ny, 1500, replace=False)]))
    F_ref, I_ref = oracle.sf_f64(hkl[sub], Z, pos, atom_b=b, B=2.0, R=R, threads=oracle_threads())
    e, ed = rel_l2(I[sub], I_ref), rel_l2(Id[sub], I_ref)
    ef = np.linalg.norm(F[sub] - F_ref) / np.linalg.norm(F_ref)
    print(f"{nx}x{ny}: I {e:.2e} (direct {ed:.2e}), F {ef:.2e}", flush=True)
    assert e < TOL and ef < TOL
    assert np.linalg.norm(F - Fd) / np.linalg.norm(Fd) < 2 * TOL


@pytest.mark.parametrize("scale", [0.3, 1.0, 2.5, (2.0, 0.5, 1.0), np.nan])
def test_matrices_that_are_not_rotations(gpu, scale):
    """q' = R q for any matrix: the node counts follow its length, in single
    patterns and plans, and a non-finite one gives the direct kernel's bits."""
    import ctypes as C

    import torch

    from spsim_amd import _lib
    from tests.test_gpu_batch import make_plan

    rng = np.random.default_rng(21)
    n, natoms = 256, 6_000
    Z, pos, _ = wl.random_molecule(natoms, 4e-9, rng)
    R = wl.uniform_rotations(1, rng)[0] @ np.diag(np.broadcast_to(scale, 3).astype(np.float64))
    hkl = _list(n, n)
    F, I = _run(gpu, hkl, n, n, Z, pos, R=R)
    Fd, Id = _run(gpu, hkl, n, n, Z, pos, R=R, tile=dv.make_tile(1, 256, 0))
    if not np.isfinite(R).all():
        assert np.array_equal(I, Id, equal_nan=True)
        return
    print(f"scale {scale}: {rel_l2(I, Id):.2e}", flush=True)
    assert not np.array_equal(I, Id) and rel_l2(I, Id) < 2 * TOL
    # the same molecule in a plan, once more unrotated: one node count serves both
    plan, *_ = make_plan([(Z, pos)], np.stack([np.eye(3), R]), np.zeros(2, np.int32), hkl, n, n)
    try:
        Ip = torch.empty((2, n * n), dtype=torch.float32, device=gpu)
        _lib.check(_lib.load().spsim_hip_batch_run(plan, None, C.c_void_p(Ip.data_ptr()), 0, None), "run")
        torch.cuda.synchronize()
    finally:
        _lib.load().spsim_hip_batch_destroy(plan)
    _, I_one = _run(gpu, hkl, n, n, Z, pos)
    assert rel_l2(Ip[1].cpu().numpy(), Id) < 2 * TOL
    assert rel_l2(Ip[0].cpu().numpy(), I_one) < 2 * TOL


@pytest.mark.parametrize("what", ["pixel", "noise", "nan pixel", "wide B", "infinite weight", "huge molecule"])
def test_rough_inputs_keep_the_direct_sum(gpu, what):
    """Lists and molecules that do not vary smoothly over the detector give
    the direct kernel's results bit for bit."""
    rng = np.random.default_rng(5)
    n, natoms = 200, 6_000
    Z, pos, b = wl.random_molecule(natoms, 5e-9, rng, atom_b_range=(5.0, 40.0))
    hkl, amp, B = _list(n, n).copy(), None, 0.0
    if what == "pixel":
        hkl[123 * n + 77, 1] *= np.float32(1.001)
    elif what == "noise":
        hkl = (hkl * (1.0 + 1e-4 * rng.normal(size=hkl.shape))).astype(np.float32)
    elif what == "nan pixel":
        hkl[31, 2] = np.nan
    elif what == "wide B":
        b = b * np.float32(1e4)
    elif what == "infinite weight":
        amp = np.ones(natoms, np.float32)
        amp[10] = np.inf
    else:
        pos = pos * np.float32(300.0)
    F, I = _run(gpu, hkl, n, n, Z, pos, atom_b=b, amp=amp, B=B)
    Fd, Id = _run(gpu, hkl, n, n, Z, pos, atom_b=b, amp=amp, B=B, tile=dv.make_tile(8, 256, 0))
    assert np.array_equal(I, Id, equal_nan=True) and np.array_equal(F, Fd, equal_nan=True)


def test_interpolated_pattern_repeats_and_captures(gpu):
    """The same bits on every call, with the workspace used by other calls in
    between, and on every replay of a captured graph."""
    import torch

    rng = np.random.default_rng(8)
    n = 256
    Z, pos, _ = wl.random_molecule(5_000, 5e-9, rng)
    atoms = dv.DeviceAtoms(dv.pack_atoms(Z, pos), gpu)
    ff = dv.form_factor_table(device=gpu)
    q = torch.from_numpy(_list(n, n)).to(gpu)
    small = torch.from_numpy(_list(128, 128)).to(gpu)
    F0, I0 = dv.structure_factor_grid(q, n, n, atoms, ff)
    dv.structure_factor_grid(small, 128, 128, atoms, ff)
    F1, I1 = dv.structure_factor_grid(q, n, n, atoms, ff)
    torch.cuda.synchronize()
    assert torch.equal(I0, I1) and torch.equal(F0, F1)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        dv.structure_factor_grid(q, n, n, atoms, ff, F=F1, I=I1, stream=stream)
    stream.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        dv.structure_factor_grid(q, n, n, atoms, ff, F=F1, I=I1, stream=torch.cuda.current_stream())
    for _ in range(3):
        I1.fill_(float("nan"))
        F1.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(I0, I1) and torch.equal(F0, F1)
        dv.structure_factor_grid(small, 128, 128, atoms, ff)


@pytest.mark.parametrize("with_b", [False, True])
def test_plan_mixes_interpolated_and_direct_patterns(gpu, with_b):
    """A batched plan on a 96 x 80 detector: molecules that are interpolated,
    one too wide for it (direct kernels) and an empty one, each at its own
    rotation, against the FP64 oracle; graph replays bit for bit; and the same
    plan with a tile asked for, which takes the direct kernels throughout."""
    import ctypes as C

    import torch

    from spsim_amd import _lib
    from tests.test_gpu_batch import make_plan

    rng = np.random.default_rng(17)
    nx, ny = 96, 80
    q = _list(nx, ny, pixel=3e-4, cx=1e-3)
    mols, Bs = [], []
    for natoms, radius in ((900, 3e-9), (2500, 4e-9), (400, 2e-7), (0, 0.0)):
        Z, pos, b = (wl.random_molecule(natoms, radius, rng, atom_b_range=(5.0, 40.0)) if natoms else
                     (np.zeros(0, np.int32), np.zeros((0, 3), np.float32), np.zeros(0, np.float32)))
        mols.append((Z, pos))
        Bs.append(b)
    pm = np.array([1, 2, 0, 3, 1, 0], np.int32)
    rots = wl.uniform_rotations(len(pm), rng)
    L = _lib.load()
    plan, *_ = make_plan(mols, rots, pm, q, nx, ny, atom_b=np.concatenate(Bs) if with_b else None, b_global=3.0)
    try:
        stream = torch.cuda.Stream()
        sp = C.c_void_p(stream.cuda_stream)
        I = torch.full((len(pm), nx * ny), float("nan"), dtype=torch.float32, device=gpu)
        F = torch.full((len(pm), nx * ny, 2), float("nan"), dtype=torch.float32, device=gpu)
        torch.cuda.synchronize()
        run = lambda g: _lib.check(L.spsim_hip_batch_run(plan, C.c_void_p(F.data_ptr()), C.c_void_p(I.data_ptr()), g,
                                                         sp), "run")
        run(0)
        stream.synchronize()
        first, Fh = I.cpu().numpy().copy(), F.cpu().numpy()
        for p, m in enumerate(pm):
            Z, pos = mols[m]
            if not len(Z):
                assert np.all(first[p] == 0) and np.all(Fh[p] == 0)
                continue
            Fr, Ir = oracle.sf_f64(q, Z, pos, atom_b=Bs[m] if with_b else None, B=3.0, R=rots[p],
                                   threads=oracle_threads())
            assert rel_l2(first[p], Ir) < TOL, p
            assert np.linalg.norm(Fh[p, :, 0] + 1j * Fh[p, :, 1] - Fr) / np.linalg.norm(Fr) < TOL, p
        for _ in range(3):
            I.fill_(float("nan"))
            torch.cuda.synchronize()
            run(1)
            stream.synchronize()
            assert np.array_equal(I.cpu().numpy(), first)
        _lib.check(L.spsim_hip_batch_set_tile(plan, C.byref(dv.make_tile(1, 256, 0))), "set_tile")
        run(0)
        stream.synchronize()
        direct = I.cpu().numpy()
        same = [np.array_equal(direct[p], first[p]) for p in range(len(pm))]
        assert same == [False, True, False, True, False, False]
        assert rel_l2(direct, first) < 2 * TOL
    finally:
        L.spsim_hip_batch_destroy(plan)


@pytest.mark.parametrize("bandwidth,samples,with_b", [(0.02, 5, False), (0.01, 11, True), (0.05, 3, False)])
def test_interpolated_spectrum_vs_f64(gpu, bandwidth, samples, with_b):
    """The wavelength spectrum on a flat list of n x n vectors, in the fitted
    and the per-sample form (3 samples), a molecule off the origin."""
    import torch

    rng = np.random.default_rng(samples)
    n, natoms = 160, 12_000
    Z, pos, b = wl.random_molecule(natoms, 6e-9, rng, atom_b_range=(5.0, 40.0))
    pos = (pos + np.array([1e-9, 2e-9, -1e-9])).astype(np.float32)
    b = b if with_b else None
    hkl = _list(n, n, pixel=1.5e-4)
    R = wl.uniform_rotations(1, rng)[0]
    atoms = dv.DeviceAtoms(dv.pack_atoms(Z, pos, atom_b=b), gpu)
    q, ff = torch.from_numpy(hkl).to(gpu), dv.form_factor_table(device=gpu)
    sc, w = dv.spectrum_samples(0.2e-9, bandwidth, samples)
    F, I = dv.structure_factor_spectrum(q, atoms, ff, sc, w, R=R)
    _, Id = dv.structure_factor_spectrum(q, atoms, ff, sc, w, R=R, tile=dv.make_tile(2, 256, 0))
    torch.cuda.synchronize()
    assert not torch.equal(I, Id)
    sub = np.sort(rng.choice(n * n, 1200, replace=False))
    F_ref, I_ref = oracle.sf_spectrum_f64(hkl[sub], Z, pos, sc, w, atom_b=b, R=R)
    Fh = F.cpu().numpy()[sub]
    e = rel_l2(I.cpu().numpy()[sub], I_ref)
    print(f"spectrum {bandwidth} {samples}: I {e:.2e} (direct {rel_l2(Id.cpu().numpy()[sub], I_ref):.2e})", flush=True)
    assert e < TOL
    assert np.linalg.norm(Fh[:, 0] + 1j * Fh[:, 1] - F_ref) / np.linalg.norm(F_ref) < TOL


def test_flat_volume_keeps_the_direct_spectrum(gpu):
    """A flat list of n^2 vectors that is no detector (a 64^3 volume's 512^2)
    gives the direct kernel's bits."""
    import torch

    rng = np.random.default_rng(3)
    Z, pos, _ = wl.random_molecule(1_000, 4e-9, rng)
    atoms, ff = dv.DeviceAtoms(dv.pack_atoms(Z, pos), gpu), dv.form_factor_table(device=gpu)
    volume = dv.hkl_detector_3d(64, 64, 64, 5e-3, 5e-3, 5e-3, 0.1, 0.2e-9, device=gpu)
    sc, w = dv.spectrum_samples(0.2e-9, 0.02, 5)
    _, I = dv.structure_factor_spectrum(volume, atoms, ff, sc, w)
    _, Id = dv.structure_factor_spectrum(volume, atoms, ff, sc, w, tile=dv.make_tile(2, 256, 0))
    torch.cuda.synchronize()
    assert torch.equal(I, Id)


@pytest.mark.parametrize("n,natoms,radius,with_b,want_b,listing", [
    (150, 25_000, 6e-9, True, True, "detector"),
    (257, 9_000, 5e-9, False, False, "detector"),
    (200, 13_000, 5e-9, True, False, "off centre"),
    (131, 30_000, 4e-9, False, True, "detector"),
    (512, 2_000, 4e-9, True, True, "volume"),
])
def test_adjoint_by_nodes_vs_f64(gpu, n, natoms, radius, with_b, want_b, listing):
    """Gradients of a loss with random dL/dI on square detectors, given F,
    against FP64 sums; a 64^3 volume of 512^2 vectors takes the direct kernel.
    The sums are FP32 (1e-7 of each term); 2e-6 allows for their cancellation."""
    import ctypes as C

    import torch

    from spsim_amd import _lib

    rng = np.random.default_rng(n)
    Z, pos, b = wl.random_molecule(natoms, radius, rng, atom_b_range=(5.0, 40.0))
    pos = (pos + np.array([2e-9, -1e-9, 1e-9])).astype(np.float32)
    if listing == "volume":
        hkl = oracle.hkl_3d(64, 64, 64, 5e-3, 5e-3, 5e-3, 0.1, 0.2e-9)
    else:
        hkl = _list(n, n, pixel=1.5e-4, cx=2e-3 if listing == "off centre" else 0.0)
    npix = n * n
    packed = dv.pack_atoms(Z, pos, atom_b=b if with_b else None)
    atoms = dv.DeviceAtoms(packed, gpu)
    q, ff = torch.from_numpy(hkl).to(gpu), dv.form_factor_table(device=gpu)
    F, _ = dv.structure_factor(q, atoms, ff, B=3.0)
    g = rng.normal(size=npix).astype(np.float32)
    gI = torch.from_numpy(g).to(gpu)
    gp = torch.full((natoms, 3), float("nan"), device=gpu)
    gb = torch.full((natoms,), float("nan"), device=gpu) if want_b else None
    vp = lambda t: None if t is None else C.c_void_p(t.data_ptr())
    segs = np.ascontiguousarray(packed.segs)
    _lib.check(_lib.load().spsim_hip_sf_adjoint(vp(q), npix, vp(atoms.atoms), vp(atoms.b),
                                                segs.ctypes.data_as(C.c_void_p), atoms.nsegs, natoms, vp(ff), 3.0,
                                                vp(F), vp(gI), vp(gp), vp(gb), None), "adjoint")
    Fh = F.cpu().numpy().astype(np.float64)
    some = np.sort(rng.choice(natoms, 24, replace=False))
    rp, rb = oracle.sf_grad_given_f_f64(hkl, Fh[:, 0] + 1j * Fh[:, 1], Z, pos, g, some, atom_b=b if with_b else None,
                                        B=3.0, threads=oracle_threads())
    at = {int(o): i for i, o in enumerate(packed.perm)}
    rows = [at[int(j)] for j in some]
    e = rel_l2(gp.cpu().numpy()[rows], rp)
    print(f"adjoint {n}: positions {e:.2e}", flush=True)
    assert e < 2e-6
    if want_b:
        assert rel_l2(gb.cpu().numpy()[rows], rb) < 2e-6


def _nfft_both(gpu, q, Z, pos, b, rots, ff):
    """Orientations through the NUFFT entry point on a square list, and on the
    same list with one vector more, which only the grids take."""
    import torch

    atoms = dv.DeviceAtoms(dv.pack_atoms(Z, pos, atom_b=b), gpu)
    longer = np.concatenate([q, q[-1:]])
    F, I, info = dv.structure_factor_nfft_batch(torch.from_numpy(q).to(gpu), atoms, ff, rots, B=2.0)
    _, Ig, info_g = dv.structure_factor_nfft_batch(torch.from_numpy(longer).to(gpu), atoms, ff, rots, B=2.0)
    assert {k: info[k] for k in info if k != "staged"} == {k: info_g[k] for k in info_g if k != "staged"}
    return F.cpu().numpy(), I.cpu().numpy(), Ig.cpu().numpy()[:, :-1]


@pytest.mark.parametrize("with_b", [False, True])
def test_nfft_orientations_by_the_surface(gpu, with_b):
    """Orientations of one molecule through the NUFFT's entry point on a square
    list are interpolated, with the error of direct sums; the grids' sizes are
    reported all the same."""
    rng = np.random.default_rng(31)
    n, natoms = 320, 400
    Z, pos, b = wl.random_molecule(natoms, 4e-9, rng, atom_b_range=(5.0, 10.0))
    pos = (pos + np.array([2e-9, 0, -1e-9])).astype(np.float32)
    b = b if with_b else None
    q = _list(n, n)
    rots = wl.uniform_rotations(3, rng)
    F, I, Ig = _nfft_both(gpu, q, Z, pos, b, rots, dv.form_factor_table(device=gpu))
    for p in range(3):
        Fr, Ir = oracle.sf_f64(q, Z, pos, atom_b=b, B=2.0, R=rots[p], threads=oracle_threads())
        assert rel_l2(I[p], Ir) < TOL, p
        assert np.linalg.norm(F[p, :, 0] + 1j * F[p, :, 1] - Fr) / np.linalg.norm(Fr) < TOL, p
        assert 1e-7 < rel_l2(Ig[p], I[p]) < 2e-5


@pytest.mark.parametrize("what", ["scaled B", "rough", "small"])
def test_nfft_orientations_that_keep_the_grids(gpu, what):
    """Scaled matrices with per-atom B (whose factors the grids take at R q),
    rough lists and few terms: the grids' values."""
    rng = np.random.default_rng(32)
    n, natoms = (64, 300) if what == "small" else (320, 400)
    Z, pos, b = wl.random_molecule(natoms, 4e-9, rng, atom_b_range=(5.0, 10.0))
    q = _list(n, n)
    rots = wl.uniform_rotations(2, rng)
    if what == "scaled B":
        rots = 0.9 * rots
    if what == "rough":
        q = (q * (1.0 - 1e-4 * rng.uniform(size=q.shape))).astype(np.float32)
    _, I, Ig = _nfft_both(gpu, q, Z, pos, b if what == "scaled B" else None, rots, dv.form_factor_table(device=gpu))
    assert rel_l2(I, Ig) < 1e-7


@pytest.mark.parametrize("with_b,rotated", [(False, True), (True, False)])
def test_nfft_molecules_split_between_surface_and_grids(gpu, with_b, rotated):
    """Molecules in one call: two that are interpolated, one too wide for it (the
    grids) and an empty one; twice, the second time in a workspace that holds
    everything."""
    import torch

    rng = np.random.default_rng(33)
    n = 256
    q = _list(n, n)
    mols = []
    for natoms, radius in ((900, 3e-9), (200, 2.5e-7), (0, 0.0), (1500, 5e-9)):
        mols.append(wl.random_molecule(natoms, radius, rng, atom_b_range=(5.0, 10.0)) if natoms else
                    (np.zeros(0, np.int32), np.zeros((0, 3), np.float32), np.zeros(0, np.float32)))
    rots = wl.uniform_rotations(len(mols), rng) if rotated else None
    dm = dv.DeviceMolecules([dv.pack_atoms(Z, pos, atom_b=b if with_b else None) for Z, pos, b in mols], gpu)
    ff = dv.form_factor_table(device=gpu)
    qs = torch.from_numpy(q).to(gpu)
    out = []
    for _ in range(2):
        F, I = dv.structure_factor_nfft_molecules(qs, dm, ff, rots, B=1.0)
        torch.cuda.synchronize()
        out.append(I.cpu().numpy())
    assert np.array_equal(out[0], out[1])
    for m, (Z, pos, b) in enumerate(mols):
        if not len(Z):
            assert not out[0][m].any()
            continue
        _, Ir = oracle.sf_f64(q, Z, pos, atom_b=b if with_b else None, B=1.0, R=rots[m] if rotated else None,
                              threads=oracle_threads())
        e = rel_l2(out[0][m], Ir)
        print(f"molecule {m}: {e:.2e}", flush=True)
        assert TOL < e < 2e-5 if m == 1 else e < TOL, m


@pytest.mark.parametrize("shape,n,natoms,geometry,with_b,rotated", [
    ("ball", (640, 640), 30_011, {}, False, False),
    ("ball", (700, 610), 30_000, {"cx": 1.1e-3, "wavelength": 0.15e-9}, True, True),
    ("rod", (800, 800), 20_001, {"pixel": 60e-6}, True, False),
    ("dense", (720, 720), 24_000, {}, False, True),
    ("unordered", (640, 640), 30_011, {}, False, False),
    ("pieces", (640, 640), 30_011, {}, False, False),
])
def test_sums_by_cells(gpu, shape, n, natoms, geometry, with_b, rotated):
    """Large patterns, whose node sums go by cells: octants and plain nodes, atom
    counts that end within every piece, a rod (empty cells), nearly all atoms
    in a few cells, and species that are not in order or in many pieces (no cells). The same bits
    on every call and replay."""
    import torch

    nx, ny = n
    rng = np.random.default_rng(natoms)
    Z, pos, b = wl.random_molecule(natoms, 13e-9, rng, atom_b_range=(5.0, 40.0))
    if shape == "rod":
        pos = pos * np.array([1.2, 0.1, 0.1], np.float32)
    if shape == "dense":
        pos[: natoms - 200] *= np.float32(0.1)
    atoms = dv.DeviceAtoms(dv.pack_atoms(Z, pos, atom_b=b if with_b else None), gpu)
    if shape == "unordered":
        atoms.segs = torch.flip(atoms.segs.reshape(-1, 4), [0]).contiguous()
    if shape == "pieces":  # more segments than species
        pieces = [[i, min(100, int(s + c) - i), int(z), 0] for s, c, z, _ in atoms.segs.reshape(-1, 4).tolist()
                  for i in range(int(s), int(s + c), 100)]
        atoms.segs, atoms.nsegs = torch.tensor(pieces, dtype=torch.int32, device=gpu), len(pieces)
    R = wl.uniform_rotations(1, rng)[0] if rotated else None
    ff = dv.form_factor_table(device=gpu)
    q = _list(nx, ny, **geometry)
    qs = torch.from_numpy(q).to(gpu)
    run = lambda **kw: dv.structure_factor_grid(qs, nx, ny, atoms, ff, B=1.0, R=R, **kw)
    F, I = run()
    _, Id = run(tile=dv.make_tile(1, 256, 0))
    torch.cuda.synchronize()
    first, Fh, Id = I.cpu().numpy(), F.cpu().numpy(), Id.cpu().numpy()
    sub = np.unique(np.concatenate([[0, nx - 1, nx * ny - nx, nx * ny - 1], rng.choice(nx * ny, 400, replace=False)]))
    Fr, Ir = oracle.sf_f64(q[sub], Z, pos, atom_b=b if with_b else None, B=1.0, R=R, threads=oracle_threads())
    e, ed = rel_l2(first[sub], Ir), rel_l2(Id[sub], Ir)
    print(f"{shape}: I {e:.2e} (direct {ed:.2e})", flush=True)
    assert e < TOL and np.linalg.norm(Fh[sub, 0] + 1j * Fh[sub, 1] - Fr) / np.linalg.norm(Fr) < TOL
    assert not np.array_equal(first, Id) and rel_l2(first, Id) < 2 * TOL
    stream = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        run(F=F, I=I, stream=torch.cuda.current_stream())
    for _ in range(2):
        I.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(I.cpu().numpy(), first)


@pytest.mark.parametrize("n,natoms,with_b,rotated,geometry", [
    (400, 16_000, True, False, {}), (401, 16_000, False, True, {}), (400, 16_001, True, True, {"cx": 1e-3}),
    (2000, 700, True, False, {})])
def test_flat_square_list_by_quads_keeps_the_bits(gpu, n, natoms, with_b, rotated, geometry):
    """A large flat list of n x n vectors, mirror-symmetric (one quad per lane) or not,
    against the same tile asked for: every bit of F and I, odd sides and one
    atom range (2000^2) included; and with a NaN among the vectors."""
    import torch

    rng = np.random.default_rng(n + natoms)
    Z, pos, b = wl.random_molecule(natoms, 6e-9, rng, atom_b_range=(5.0, 40.0))
    atoms = dv.DeviceAtoms(dv.pack_atoms(Z, pos, atom_b=b if with_b else None), gpu)
    ff = dv.form_factor_table(device=gpu)
    R = wl.uniform_rotations(1, rng)[0] if rotated else None
    q = _list(n, n, **geometry)
    tile = dv.make_tile(2 if n * n >= 4 * 256 * 256 else 1, 256, 0)  # the library's default
    for nan in (False, True):
        if nan:
            q = q.copy()
            q[n * 7 + 5, 1] = np.nan
        qs = torch.from_numpy(q).to(gpu)
        F, I = dv.structure_factor(qs, atoms, ff, B=1.0, R=R)
        Ft, It = dv.structure_factor(qs, atoms, ff, B=1.0, R=R, tile=tile)
        torch.cuda.synchronize()
        assert np.array_equal(F.cpu().numpy(), Ft.cpu().numpy(), equal_nan=True)
        assert np.array_equal(I.cpu().numpy(), It.cpu().numpy(), equal_nan=True)


@pytest.mark.parametrize("entry", ["grid", "spectrum", "nfft"])
def test_empty_segments_change_nothing(gpu, entry):
    """A segment without atoms does not take part in the choice of path, whatever
    its species' form factor."""
    import torch

    rng = np.random.default_rng(41)
    n, natoms = 256, 6_000
    Z, pos, _ = wl.random_molecule(natoms, 4e-9, rng)
    table = dv.default_form_factors().copy()
    table[98] = np.nan
    ff, q = dv.form_factor_table(table, device=gpu), torch.from_numpy(_list(n, n)).to(gpu)
    sc, w = dv.spectrum_samples(0.2e-9, 0.02, 5)
    got = []
    for empty in (False, True):
        atoms = dv.DeviceAtoms(dv.pack_atoms(Z, pos), gpu)
        if empty:
            last = torch.tensor([[natoms, 0, 98, 0]], dtype=torch.int32, device=gpu)
            atoms.segs, atoms.nsegs = torch.cat([atoms.segs.reshape(-1, 4), last]).contiguous(), atoms.nsegs + 1
        if entry == "grid":
            got.append(dv.structure_factor_grid(q, n, n, atoms, ff)[1])
        elif entry == "spectrum":
            got.append(dv.structure_factor_spectrum(q, atoms, ff, sc, w)[1])
        else:
            got.append(dv.structure_factor_nfft(q, atoms, ff)[1])
    torch.cuda.synchronize()
    assert bool(torch.isfinite(got[0]).all()) and torch.equal(got[0], got[1])


def _ends(natoms, radius, rng):
    """Two clusters of carbon at the ends of the x axis: every phase is the steepest."""
    pos = np.zeros((natoms, 3))
    pos[:, 0] = np.where(np.arange(natoms) % 2, radius, -radius) * (1 - 1e-3 * rng.uniform(size=natoms))
    return np.full(natoms, 6, np.int32), pos.astype(np.float32)


@pytest.mark.parametrize("entry", ["grid", "plan"])
@pytest.mark.parametrize("n,width,radius", [(512, 0.0384, 6e-8), (1024, 0.04, 8e-8)])
def test_atoms_at_the_ends_of_the_molecule(gpu, entry, n, width, radius):
    """240 to 330 radians from the middle of the detector to its edge, with all atoms at
    the ends: the nodes serve the steepest phase as well as a ball's average one."""
    import ctypes as C

    import torch

    from spsim_amd import _lib
    from tests.test_gpu_batch import make_plan

    rng = np.random.default_rng(51)
    Z, pos = _ends(1_500, radius, rng)
    hkl = oracle.hkl_detector(n, n, np.float32(width).item(), np.float32(width).item(), 0.2, 0.0, 0.0, 0, 0.15e-9)
    if entry == "grid":
        F, I = _run(gpu, hkl, n, n, Z, pos)
    else:
        plan, *_ = make_plan([(Z, pos)], np.eye(3)[None], np.zeros(1, np.int32), hkl, n, n)
        try:
            It = torch.empty((1, n * n), dtype=torch.float32, device=gpu)
            Ft = torch.empty((1, n * n, 2), dtype=torch.float32, device=gpu)
            _lib.check(_lib.load().spsim_hip_batch_run(plan, C.c_void_p(Ft.data_ptr()), C.c_void_p(It.data_ptr()), 0,
                                                       None), "run")
            torch.cuda.synchronize()
        finally:
            _lib.load().spsim_hip_batch_destroy(plan)
        Fh = Ft.cpu().numpy()[0]
        F, I = Fh[:, 0] + 1j * Fh[:, 1], It.cpu().numpy()[0]
    sub = np.sort(rng.choice(n * n, 3000, replace=False))
    Fr, Ir = oracle.sf_f64(hkl[sub], Z, pos, threads=oracle_threads())
    e, ef = rel_l2(I[sub], Ir), np.linalg.norm(F[sub] - Fr) / np.linalg.norm(Fr)
    print(f"{entry} {n}: I {e:.2e}, F {ef:.2e}", flush=True)
    assert e < TOL and ef < TOL


def test_sharp_form_factors(gpu):
    """A form factor of one wide Gaussian (200 A^2, exponents up to 42 on this detector)
    and a constant, on a molecule of 0.2 nm, whose phases need few nodes."""
    import torch

    rng = np.random.default_rng(52)
    n, natoms = 1500, 150
    Z, pos, _ = wl.random_molecule(natoms, 2e-10, rng)
    Z[:] = 6
    table = dv.default_form_factors().copy()
    table[6] = [4.0, 0, 0, 0, 200.0, 0, 0, 0, 2.0]
    hkl = oracle.hkl_detector(n, n, np.float32(0.1).item(), np.float32(0.1).item(), 0.05, 0.0, 0.0, 0, 1e-10)
    atoms, ff = dv.DeviceAtoms(dv.pack_atoms(Z, pos), gpu), dv.form_factor_table(table, device=gpu)
    q = torch.from_numpy(hkl).to(gpu)
    _, I = dv.structure_factor_grid(q, n, n, atoms, ff)
    _, Id = dv.structure_factor_grid(q, n, n, atoms, ff, tile=dv.make_tile(1, 256, 0))
    torch.cuda.synchronize()
    assert not torch.equal(I, Id)
    sub = np.sort(rng.choice(n * n, 3000, replace=False))
    _, Ir = oracle.sf_f64(hkl[sub], Z, pos, ff=table, threads=oracle_threads())
    e = rel_l2(I.cpu().numpy()[sub], Ir)
    print(f"sharp: I {e:.2e} (direct {rel_l2(Id.cpu().numpy()[sub], Ir):.2e})", flush=True)
    assert e < TOL
