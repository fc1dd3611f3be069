"""A simulate_shot that fails leaves the random state where the calls it stands for leave
it: no orientation is drawn without a q list, and no shot number is taken without a
pattern, so that the next shot's orientation and noise are the same."""
import numpy as np
import pytest

import spsim
from tests.test_gpu_dropin import make_opts, molecule


def test_no_orientation_without_a_list():
    """A detector beyond the largest (2^28 pixels), where no device is reached."""
    opts = make_opts(20_000)
    opts.random_orientation = 1
    opts.detector.binning_x = opts.detector.binning_y = 100
    _, _, mol = molecule(5)
    spsim.sp_srand(7)
    first = spsim.p_drand48()
    spsim.sp_srand(7)
    assert spsim.simulate_shot(mol, opts) is None
    assert spsim.p_drand48() == first


@pytest.mark.gpu
@pytest.mark.parametrize("cuda", [0, 1])
def test_no_shot_number_without_a_pattern(gpu, cuda):
    """A molecule that is refused (atomic number 120) takes an orientation, as
    apply_orientation_to_HKL_list does before the pattern, but no shot number."""
    opts = make_opts(48)
    opts.random_orientation, opts.use_cuda = 1, cuda
    d, e = opts.detector, opts.experiment
    e.beam_intensity, d.quantum_efficiency, d.readout_noise = 1e25, 0.5, 2.0
    Z, pos, mol = molecule(300)
    bad = spsim.get_molecule_from_atoms(np.where(np.arange(300) == 10, 120, Z).astype(np.int32), pos)
    n = 48 * 48

    def shot():
        pat = spsim.simulate_shot(mol, opts)
        got = [spsim.float_array(pat.ints, n), spsim.float_array(d.photon_count, n), spsim.float_array(d.real_output, n)]
        spsim.free_diffraction_pattern(pat)
        spsim.free_output_in_options(opts)
        return got

    spsim.sp_srand(3)
    for _ in range(3):  # the refused molecule's orientation, of three uniforms
        spsim.p_drand48()
    want = shot()
    spsim.sp_srand(3)
    assert spsim.simulate_shot(bad, opts) is None
    for a, b in zip(shot(), want):
        np.testing.assert_array_equal(a, b)
