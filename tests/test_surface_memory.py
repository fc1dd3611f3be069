"""Workspace that an interpolated pattern asks for (surf_single_bytes, a host function
of the library: no GPU needed)."""
import ctypes as C

import pytest

from spsim_amd import _lib


def single_bytes(nx, ny, natoms, nsegs, spectrum):
    f = getattr(_lib.load(), "_ZN5spsim17surf_single_bytesEiiiib")
    f.restype = C.c_size_t
    f.argtypes = [C.c_int] * 4 + [C.c_bool]
    return f(nx, ny, natoms, nsegs, spectrum)


@pytest.mark.parametrize("n,natoms", [(512, 20_000), (512, 40_000), (1024, 100_000), (2048, 1_000_000)])
def test_spectra_ask_for_no_cells(n, natoms):
    """A spectrum's atoms are never sorted into cells: it takes an atom record of 48
    bytes, 12 bytes a pixel, the two axes' tables and the node sums, and nothing
    beside; from 1e10 terms on a plain pattern also takes the cells' buffers (two of
    4 Mi sums, 24 bytes each, and 54 bytes an atom)."""
    plain, spectrum = single_bytes(n, n, natoms, 8, False), single_bytes(n, n, natoms, 8, True)
    m = min(512, int(0.6 * n) // 4 * 4)  # most nodes per axis
    slots = max(1 << 20, m * m + 2 * 512 + 2048)
    need = 48 * natoms + 12 * n * n + 2 * 16 * m * n + 48 * m * m + 24 * slots + 32 * m * n
    assert need <= spectrum <= need + (1 << 16)
    cells = n * n * natoms >= 10**10
    assert plain - spectrum >= 2 * 24 * (4 << 20) + 54 * natoms if cells else plain == spectrum
