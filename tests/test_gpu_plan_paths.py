"""Each of the paths that a plan or a call may take, made to run: the direct kernels with
automatic atom ranges, sums by cells beside plain node sums and direct patterns in
one plan of several groups, and what a call does without the memory for the
interpolation. Tolerance as in test_gpu_surface."""
import ctypes as C
import os
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

import oracle
from spsim_amd import _lib
from spsim_amd import device as dv
from spsim_amd import workloads as wl
from tests.conftest import oracle_threads, rel_l2
from tests.test_gpu_batch import make_plan

pytestmark = pytest.mark.gpu

TOL = 4e-7


def _run(gpu, plan, npat, npix, graph=0):
    import torch

    stream = torch.cuda.Stream()
    I = torch.full((npat, npix), float("nan"), dtype=torch.float32, device=gpu)
    F = torch.full((npat, npix, 2), float("nan"), dtype=torch.float32, device=gpu)
    torch.cuda.synchronize()
    _lib.check(_lib.load().spsim_hip_batch_run(plan, C.c_void_p(F.data_ptr()), C.c_void_p(I.data_ptr()), graph,
                                               C.c_void_p(stream.cuda_stream)), "run")
    stream.synchronize()
    Fh = F.cpu().numpy()
    return Fh[..., 0] + 1j * Fh[..., 1], I.cpu().numpy()


def test_direct_plan_splits_a_large_molecule(gpu):
    """One molecule of 60,000 atoms among 400-atom ones with the plan's own tile asked
    for: the direct kernels with the automatic item bound, split tiles among them,
    against FP64, against the same plan unsplit, and against a plan without a tile
    (interpolated: other bits in every pattern)."""
    rng = np.random.default_rng(32)
    mols = [wl.random_molecule(60_000, 6e-9, rng)[:2]] + [wl.random_molecule(400, 1.5e-9, rng)[:2] for _ in range(7)]
    pm, rots, n = np.arange(8, dtype=np.int32), wl.uniform_rotations(8, rng), 128
    q = oracle.hkl_detector(n, n, n * 75e-6, n * 75e-6, 0.1, 0, 0, 0, 0.2e-9)
    L = _lib.load()
    plan, *_ = make_plan(mols, rots, pm, q, n, n)
    try:
        _, smooth = _run(gpu, plan, 8, n * n)
        tile, blocks = _lib.Tile(), C.c_int()
        _lib.check(L.spsim_hip_batch_get_tile(plan, C.byref(tile), C.byref(blocks)), "get_tile")
        _lib.check(L.spsim_hip_batch_set_tile(plan, C.byref(tile)), "set_tile")
        bound, split = C.c_int(), C.c_int()
        L.spsim_hip_batch_describe(plan, None, C.byref(bound), C.byref(split))
        assert 0 < bound.value < 60_000 and split.value > 0
        _, direct = _run(gpu, plan, 8, n * n)
        _, replayed = _run(gpu, plan, 8, n * n, graph=1)
        assert np.array_equal(direct, replayed)
        assert not any(np.array_equal(a, b) for a, b in zip(direct, smooth))
        sub = np.sort(rng.choice(n * n, 1024, replace=False))
        for p, (Z, pos) in enumerate(mols):
            ref = oracle.sf_f64(q[sub], Z, pos, R=rots[p], threads=oracle_threads())[1]
            assert rel_l2(direct[p, sub], ref) < TOL and rel_l2(smooth[p, sub], ref) < TOL, p
        _lib.check(L.spsim_hip_batch_set_item_atoms(plan, -1), "no split")
        _, whole = _run(gpu, plan, 8, n * n)
        assert not np.array_equal(whole[0], direct[0]) and rel_l2(whole, direct) < TOL
    finally:
        L.spsim_hip_batch_destroy(plan)


@pytest.mark.parametrize("nx,ny,cx,with_b", [(640, 640, 0.0, False), (700, 610, 1.1e-3, True)])
def test_plan_with_cells_in_several_groups(gpu, nx, ny, cx, with_b):
    """Two molecules that are summed by cells, in eighteen patterns (whose buffers do not
    fit one group's 256 MB), one by plain node sums and one too wide for the
    interpolation, in turn: every pattern against FP64 on a sample of pixels and
    on the outermost ones, and the same bits again by a graph."""
    rng = np.random.default_rng(nx)
    q = oracle.hkl_detector(nx, ny, np.float32(nx * 75e-6).item(), np.float32(ny * 75e-6).item(), 0.1, cx, 0.0, 0,
                            0.15e-9)
    mols, Bs = [], []
    for natoms, radius in ((30_011, 13e-9), (400, 2e-7), (2_000, 4e-9), (24_000, 11e-9)):
        Z, pos, b = wl.random_molecule(natoms, radius, rng, atom_b_range=(5.0, 40.0))
        mols.append((Z, (pos + np.array([2e-9, -1e-9, 1e-9])).astype(np.float32)))
        Bs.append(b)
    pm = np.array([0, 1, 2, 3] + [0, 3] * 8 + [2], np.int32)
    rots = wl.uniform_rotations(len(pm), rng)
    plan, *_ = make_plan(mols, rots, pm, q, nx, ny, atom_b=np.concatenate(Bs) if with_b else None, b_global=1.0)
    try:
        F, I = _run(gpu, plan, len(pm), nx * ny)
        _, again = _run(gpu, plan, len(pm), nx * ny, graph=1)
        assert np.array_equal(I, again)
        u, v = np.meshgrid(np.linspace(-1, 1, nx), np.linspace(-1, 1, ny))
        outer = np.flatnonzero((u * u + v * v).ravel() > 1.6)
        for p, m in enumerate(pm):
            Z, pos = mols[m]
            for pixels in (rng.choice(nx * ny, 300, replace=False), rng.choice(outer, 300, replace=False)):
                pixels = np.sort(pixels)
                Fr, Ir = oracle.sf_f64(q[pixels], Z, pos, atom_b=Bs[m] if with_b else None, B=1.0, R=rots[p],
                                       threads=oracle_threads())
                e = np.linalg.norm(F[p, pixels] - Fr) / np.linalg.norm(Fr)
                # the outermost pixels' own norm: the atoms' terms (sqrt(N) of them add
                # up) are as large there, so are the sums' errors
                assert e < TOL and rel_l2(I[p, pixels], Ir) < 2 * TOL, (p, m, e)
    finally:
        _lib.load().spsim_hip_batch_destroy(plan)


# (pixels per side, atoms, their cube's edge) of calls whose interpolation takes a
# workspace of more than a hundredth of the card, and their other path less: by 102
# bytes an atom, or, on the NUFFT's lists, by 12 bytes a pixel for the look at the list
LARGE = {"grid": (64, 45_000_000, 6e-9), "adjoint": (64, 45_000_000, 6e-9), "nfft": (0, 300, 1.5e-9),
         "molecules": (0, 300, 1.5e-9)}


def _large_call(gpu, kind):
    import torch

    n, natoms, edge = LARGE[kind]
    if n == 0:  # the workspace is allocated with a quarter more than it is asked for
        n = int(np.sqrt(1.01 * torch.cuda.get_device_properties(gpu).total_memory / 1500))
    g = torch.Generator(device=gpu).manual_seed(3)
    atoms = torch.rand((natoms, 4), generator=g, device=gpu)
    atoms[:, :3] = (atoms[:, :3] - 0.5) * edge
    atoms[:, 3] = 1.0
    ff = dv.form_factor_table(device=gpu)
    width = 0.0192 if n == 64 else 0.1
    q = dv.hkl_detector(n, n, width, width, 0.1, 0.2e-9, device=gpu)
    segs = np.array([[0, natoms, 6, 0]], np.int32)
    vp = lambda t: None if t is None else C.c_void_p(t.data_ptr())
    host = lambda a: a.ctypes.data_as(C.c_void_p)
    dsegs = torch.from_numpy(segs).to(gpu)
    I = torch.full((n * n,), float("nan"), device=gpu)
    some = lambda: I[:: max(1, n * n // 100_003)].cpu().numpy()
    L = _lib.load()
    if kind == "grid":
        def call(tile):
            _lib.check(L.spsim_hip_sf_grid(vp(q), n, n, vp(atoms), None, vp(dsegs), 1, natoms, vp(ff), 0.0, None, None,
                                           vp(I), tile, None), kind)
            return some()
        return call(None), call(C.byref(dv.make_tile(8, 256, 0)))
    if kind == "nfft":
        _lib.check(L.spsim_hip_sf_nfft(vp(q), n * n, vp(atoms), None, vp(dsegs), 1, natoms, vp(ff), 0.0, None, 1e-6, None,
                                       vp(I), None, None), kind)
        return (some(),)
    if kind == "molecules":
        off, soff = np.array([0, natoms], np.int32), np.array([0, 1], np.int32)
        _lib.check(L.spsim_hip_sf_nfft_molecules(vp(q), n * n, 1, vp(atoms), None, host(off), vp(dsegs), host(soff),
                                                 vp(ff), 0.0, None, 1e-6, None, vp(I), None), kind)
        return (some(),)
    F = torch.randn((n * n, 2), generator=g, device=gpu)
    gI = torch.randn((n * n,), generator=g, device=gpu)
    gp = torch.full((natoms, 3), float("nan"), device=gpu)
    _lib.check(L.spsim_hip_sf_adjoint(vp(q), n * n, vp(atoms), None, host(segs), 1, natoms, vp(ff), 0.0, vp(F), vp(gI),
                                      vp(gp), None, None), kind)
    return (gp[:: natoms // 10_000].cpu().numpy(),)


@pytest.mark.parametrize("kind", LARGE)
def test_without_memory_for_the_interpolation(gpu, kind, tmp_path):
    """The same call in a process whose largest allocation is one hundredth of the
    card: the direct kernels' bits, or the grids' values, instead of a failure."""
    import torch

    free = _large_call(gpu, kind)
    torch.cuda.empty_cache()
    _lib.load().spsim_hip_release()
    out = tmp_path / "out.npz"
    code = (f"import numpy as np, torch\nfrom tests.test_gpu_plan_paths import _large_call\n"
            f"print('{kind}', flush=True)\n"
            f"np.savez({str(out)!r}, *_large_call(torch.device('cuda', 0), '{kind}'))\n")
    r = subprocess.run([sys.executable, "-c", code], cwd=Path(__file__).resolve().parents[1], capture_output=True,
                       text=True, timeout=100, env=dict(os.environ, GPU_SINGLE_ALLOC_PERCENT="1"))
    assert r.returncode == 0, r.stdout + r.stderr
    with np.load(out) as f:
        short = [f[k] for k in f.files]
    assert not np.array_equal(short[0], free[0])  # another path ran
    e = rel_l2(short[0], free[0])
    print(f"{kind}: {e:.2e}", flush=True)
    if kind == "grid":
        assert np.array_equal(short[0], short[1]) and np.array_equal(short[1], free[1]) and e < 2 * TOL
    else:
        assert e < (2e-6 if kind == "adjoint" else 2e-5)
