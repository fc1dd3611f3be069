"""Calls that share the library workspace, issued on several streams and by several
threads without a wait in between, give bit for bit what each gives alone."""
import ctypes as C
import threading

import numpy as np
import pytest

import oracle
from spsim_amd import _lib
from spsim_amd import device as dv
from spsim_amd import workloads as wl

pytestmark = pytest.mark.gpu


def _input(gpu, kind, n, natoms, seed, cx=0.0):
    """A call of one kind and the arrays it needs: run(stream, F, I)."""
    import torch

    rng = np.random.default_rng(seed)
    Z, pos, _ = wl.random_molecule(natoms, 4e-9, rng)
    packed = dv.pack_atoms(Z, pos)
    atoms, ff = dv.DeviceAtoms(packed, gpu), dv.form_factor_table(device=gpu)
    hkl = oracle.hkl_detector(n, n, np.float32(0.04).item(), np.float32(0.04).item(), 0.1, cx, 0.0, 0, 0.2e-9)
    q = torch.from_numpy(hkl).to(gpu)
    sc, w = dv.spectrum_samples(0.2e-9, 0.02, 5)
    calls = {
        "grid": lambda s, F, I: dv.structure_factor_grid(q, n, n, atoms, ff, F=F, I=I, stream=s),
        "pattern": lambda s, F, I: dv.structure_factor(q, atoms, ff, F=F, I=I, stream=s),
        "spectrum": lambda s, F, I: dv.structure_factor_spectrum(q, atoms, ff, sc, w, F=F, I=I, stream=s),
        "nfft": lambda s, F, I: dv.structure_factor_nfft(q, atoms, ff, F=F, I=I, stream=s),
        "bridge": lambda s, F, I: _bridge(hkl, n, packed, F, I),
    }
    return calls[kind], n * n


def _bridge(hkl, n, packed, F, I):
    """The drop-in library's host-array call, into host copies of F and I."""
    Fh, Ih = np.zeros((n * n, 2), np.float32), np.zeros(n * n, np.float32)
    vp = lambda a: a.ctypes.data_as(C.c_void_p)
    atoms, segs, ff = (np.ascontiguousarray(a) for a in (packed.atoms, packed.segs, dv.default_form_factors()))
    fn = _lib.load().spsim_bridge_structure_factor_grid
    assert fn(vp(hkl), n, n, vp(atoms), None, vp(segs), len(segs), len(atoms), vp(ff), C.c_float(0.0), vp(Fh),
              vp(Ih)) == 0
    F.copy_(torch_from(Fh))
    I.copy_(torch_from(Ih))


def torch_from(a):
    import torch

    return torch.from_numpy(a)


def _outputs(gpu, npix):
    import torch

    return (torch.full((npix, 2), float("nan"), dtype=torch.float32, device=gpu),
            torch.full((npix,), float("nan"), dtype=torch.float32, device=gpu))


def _alone(gpu, run, npix):
    import torch

    F, I = _outputs(gpu, npix)
    run(None, F, I)
    torch.cuda.synchronize()
    return F, I


# (kind, n, atoms, x offset): several atom ranges, one (few atoms), and for the
# pattern mirror-symmetric lists (by quads) beside one that is not
STREAMS = [
    [("grid", 512, 4_000, 0.0), ("grid", 300, 6_000, 1e-3)],
    [("grid", 1500, 400, 0.0), ("grid", 2048, 300, 2e-3)],
    [("pattern", 2600, 400, 0.0), ("pattern", 2500, 420, 1e-3)],
    [("spectrum", 1024, 300, 0.0), ("grid", 1024, 500, 0.0), ("nfft", 300, 900, 0.0)],
]


@pytest.mark.parametrize("cases", STREAMS, ids=lambda c: "+".join(k[0] for k in c))
def test_streams_share_the_workspace(gpu, cases):
    import torch

    runs = [_input(gpu, *c[:3], seed=i, cx=c[3]) for i, c in enumerate(cases)]
    want = [_alone(gpu, *r) for r in runs]
    streams = [torch.cuda.Stream() for _ in runs]
    for _ in range(3):
        got = [_outputs(gpu, npix) for _, npix in runs]
        torch.cuda.synchronize()
        for _ in range(4):
            for (run, _), s, (F, I) in zip(runs, streams, got):
                run(s, F, I)
        torch.cuda.synchronize()
        for (F, I), (Fw, Iw) in zip(got, want):
            assert torch.equal(F, Fw) and torch.equal(I, Iw)


def test_threads_share_the_workspace(gpu):
    """Threads on the default stream, on streams of their own and in the drop-in
    library's host-array calls; one of them releases the library's buffers."""
    import torch

    cases = [("grid", 512, 4_000, 0.0, False), ("grid", 1500, 400, 0.0, True), ("pattern", 300, 5_000, 1e-3, True),
             ("nfft", 256, 900, 0.0, True), ("bridge", 256, 5_000, 0.0, False), ("bridge", 100, 3_000, 0.0, False)]
    runs = [_input(gpu, *c[:3], seed=i, cx=c[3]) for i, c in enumerate(cases)]
    want = [_alone(gpu, *r) for r in runs]
    streams = [torch.cuda.Stream() if c[4] else None for c in cases]
    got = [_outputs(gpu, npix) for _, npix in runs]
    torch.cuda.synchronize()
    failed = []

    def work(i):
        try:
            for k in range(6):
                runs[i][0](streams[i], *got[i])
                if i == 0 and k == 3:
                    _lib.load().spsim_hip_release()
        except Exception as e:  # noqa: BLE001  (reported by the test's thread)
            failed.append((i, repr(e)))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(cases))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not failed
    for (F, I), (Fw, Iw) in zip(got, want):
        assert torch.equal(F, Fw) and torch.equal(I, Iw)


def _replays(graph, F, I, want, between):
    import torch

    for _ in range(3):
        F.fill_(float("nan"))
        I.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(F, want[0]) and torch.equal(I, want[1])
        between()
        torch.cuda.synchronize()


@pytest.mark.parametrize("kind,n,natoms", [("grid", 1500, 400), ("pattern", 2600, 400), ("spectrum", 1024, 300)])
def test_captured_calls_of_one_atom_range_need_no_workspace(gpu, kind, n, natoms):
    """They take the direct kernels, as with an explicit tile, and their graphs
    replay after the library's buffers are released."""
    import torch

    run, npix = _input(gpu, kind, n, natoms, 1)
    eager = _alone(gpu, run, npix)  # the workspace is large enough
    F, I = _outputs(gpu, npix)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        run(torch.cuda.current_stream(), F, I)
    _lib.load().spsim_hip_release()
    graph.replay()
    torch.cuda.synchronize()
    direct = F.clone(), I.clone()
    close = float(torch.linalg.norm(eager[1] - I) / torch.linalg.norm(I))
    assert torch.equal(eager[1], I) if kind == "pattern" else 0 < close < 8e-7
    _replays(graph, F, I, direct, lambda: _alone(gpu, run, npix))


def test_captured_workspace_outlives_growth(gpu):
    """A graph's calls of several atom ranges keep their buffer when a later call
    needs a larger one."""
    import torch

    run, npix = _input(gpu, "grid", 512, 4_000, 1)
    large, large_pix = _input(gpu, "grid", 1600, 3_000, 2)
    _lib.load().spsim_hip_release()
    want = _alone(gpu, run, npix)
    F, I = _outputs(gpu, npix)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        run(torch.cuda.current_stream(), F, I)
    before = torch.cuda.mem_get_info()[0]
    F2, I2 = _outputs(gpu, large_pix)
    large(None, F2, I2)
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info()[0] < before  # the buffer has grown
    ones = torch.ones(64 << 20, dtype=torch.float32, device=gpu)  # would take up what was freed
    _replays(graph, F, I, want, lambda: (large(None, F2, I2), ones.fill_(1.0)))
    assert bool((ones == 1.0).all())
    del graph
    _lib.load().spsim_hip_release()
