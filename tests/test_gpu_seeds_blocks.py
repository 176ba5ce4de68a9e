"""FOD seeding at the edges of its blocks: coefficient counts around whole
orders, seed counts around a wavefront, totals that select nothing."""

import numpy as np
import pytest

import oracle
import tractography_amd as tg

from test_gpu_seeds import _device_seeds, _states

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [1, 14, 15, 16, 28, 29, 44])
@pytest.mark.parametrize("n", [1, 65, 3000])
def test_seeds_bit_exact_for_every_coefficient_count(runtime, K, n):
    rng = np.random.default_rng(K)
    fod = 0.1 * rng.standard_normal((5, 6, 7, K)).astype(np.float32)
    fod[..., 0] = np.abs(fod[..., 0]) + 0.05
    fod[0] = 0
    fod[0, ..., 0] = -1000  # every weight underflows to zero
    inline, voxels, affine = tg.seeds.sparse_fod(tg.Nifti1Image(fod, np.diag([2.0, 1.0, 1.0, 1.0])))
    states = _states(n, K)
    got, got_states = _device_seeds(runtime, 0, K, inline, voxels, affine, states)
    ref, ref_states = oracle.seeds_from_fod(0, K, inline, voxels, affine, states, threads=8)
    np.testing.assert_array_equal(got, ref)
    np.testing.assert_array_equal(got_states, ref_states)
