"""Plain tracking by wavefronts that share a step, and launches that hand
their last streamlines over to them: bit-exact at the sizes where the form of
the launch changes."""

import numpy as np
import pytest

import bench
import fixtures
import oracle
import tractography_amd as tg

from test_gpu_plain import _compare_tracks

pytestmark = pytest.mark.gpu


def _both(runtime, algorithm, domain, field, *args, threads):
    return (tg.tracking.track(algorithm, domain, field, *args, runtime),
            oracle.track(domain, field, algorithm, *args, threads=threads))


SPLIT = 32768  # seeds up to which a launch is split wavefronts throughout


@pytest.fixture(scope="module")
def scene():
    cfg = bench.sphere32_transport(seed=4, n_seeds=270_001)
    field = tg.field.Image(tg.Nifti1Image(cfg["fod"], np.eye(4)))
    domain = tg.domain.Image(tg.Nifti1Image(cfg["mask"], np.eye(4)))
    return cfg["seeds"], field, domain


def _algorithm(name, K=45):
    model = tg.local.RealSymmetricSphericalHarmonics(K)
    if name == "transport":
        return tg.algorithm.Transport(model, step_size=0.2, gamma=1.0)
    return tg.algorithm.Diffusion(model, step_size=0.2, gamma=1.0, noise_variance=0.1, seed=3)


@pytest.mark.parametrize("name", ["transport", "diffusion"])
@pytest.mark.parametrize("n", [1, 64, 65, SPLIT, SPLIT + 1, 150_000, 270_001])
def test_mask_domain(runtime, scene, name, n, oracle_threads):
    # 270,001 seeds end in three launches: all lanes, half of them, split.
    seeds, field, domain = scene
    algorithm = _algorithm(name)
    rng = [algorithm.get_rng_seed() for _ in range(-(-n // 1000))]
    _compare_tracks(*_both(runtime, algorithm, domain, field, seeds[:n], rng, 1000, 0.5, 12.0,
                           threads=oracle_threads))


@pytest.mark.parametrize("name", ["transport", "diffusion"])
@pytest.mark.parametrize("n", [65, SPLIT + 1])
def test_mesh_domain(runtime, scene, name, n, oracle_threads):
    _, field, _ = scene
    mesh, seeds, _, _ = fixtures.shell_scene(n_seeds=n, seed=13)
    algorithm = _algorithm(name)
    rng = [algorithm.get_rng_seed()]
    got, ref = _both(runtime, algorithm, mesh, field, seeds, rng, n, 0.5, 16.0, threads=oracle_threads)
    _compare_tracks(got, ref)
    np.testing.assert_array_equal(got.hits, ref["hits"])


@pytest.mark.parametrize("n", [100, SPLIT + 100])
def test_fewer_coefficients(runtime, scene, n, oracle_threads):
    seeds, field, domain = scene
    fod = tg.field.Image(tg.Nifti1Image(np.ascontiguousarray(field.values[..., :15]), np.eye(4)))
    algorithm = _algorithm("diffusion", 15)
    _compare_tracks(*_both(runtime, algorithm, domain, fod, seeds[:n], [algorithm.get_rng_seed()], n, 0.5, 10.0,
                           threads=oracle_threads))
