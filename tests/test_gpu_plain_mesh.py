"""Plain tracking against a boundary mesh: the candidate lists that spare a
step its traversal change no result, wherever they decide."""

import numpy as np
import pytest

import bench
import fixtures
import oracle
import tractography_amd as tg

from test_gpu_plain import _compare_tracks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_seeds", [1, 65, 1500])
@pytest.mark.parametrize("reach", [0.05, 0.1, 0.1001, 2.0])
def test_lists_that_decide_some_steps(runtime, reach, n_seeds, oracle_threads):
    # Steps of 0.1: lists of a shorter reach never decide, of about that
    # length by the rounding of a step, of a longer one always.
    shell, seeds, _, _ = fixtures.shell_scene(n_seeds=n_seeds, seed=12)
    mesh = tg.domain.Mesh(shell.boundary.vertices, shell.boundary.faces, cell_size=0.7, reach=reach)
    cfg = bench.sphere32_transport(seed=3, n_seeds=1)
    field = tg.field.Image(tg.Nifti1Image(cfg["fod"], np.eye(4)))
    algorithm = tg.algorithm.Transport(tg.local.RealSymmetricSphericalHarmonics(45), step_size=0.1, gamma=1.0)
    got = tg.tracking.track(algorithm, mesh, field, seeds, [0], n_seeds, 0.25, 40.0, runtime)
    ref = oracle.track(mesh, field, algorithm, seeds, [0], n_seeds, 0.25, 40.0, threads=oracle_threads)
    _compare_tracks(got, ref)
    np.testing.assert_array_equal(got.hits, ref["hits"])
