"""Lane groups of the fast path (several lanes per streamline): the same tracks
as one lane per streamline, and the FP64 oracle's."""

import numpy as np
import pytest

import bench
import deviation
import oracle
import tractography_amd as tg

pytestmark = pytest.mark.gpu

# A launch of more seeds runs one lane per streamline when an update has few
# candidates.
MANY = 65537


@pytest.fixture(scope="module")
def scene():
    cfg = bench.sphere32_transport(seed=5, n_seeds=MANY)
    field = tg.field.Image(tg.Nifti1Image(cfg["fod"], np.eye(4)))
    domain = tg.domain.Image(tg.Nifti1Image(cfg["mask"], np.eye(4)))
    return cfg["seeds"], field, domain


@pytest.fixture(scope="module")
def fast_runtime():
    return tg.HipRuntime(path="fast")


def _prefix_equal(few, many):
    n = len(few.lengths)
    np.testing.assert_array_equal(few.lengths, many.lengths[:n])
    np.testing.assert_array_equal(few.steps, many.steps[:n])
    np.testing.assert_array_equal(few.points, many.points[: len(few.points)])


@pytest.mark.parametrize("n_samples", [1, 7, 8, 9, 16])
@pytest.mark.parametrize("n", [1, 9, 3001])
def test_probabilistic_groups_equal_single_lanes(fast_runtime, scene, n_samples, n):
    # Candidates below, at and past a whole share per lane; seeds below and
    # past a wavefront's eight groups. Same sums, choices and noise states.
    seeds, field, domain = scene
    algorithm = tg.algorithm.Probabilistic(tg.local.RealSymmetricSphericalHarmonics(45), n_samples=n_samples,
                                           max_angle=0.4, seed=7, step_size=0.2)
    rng = [algorithm.get_rng_seed() for _ in range(MANY // 1000 + 1)]
    args = (1000, 0.5, 15.0, fast_runtime)
    few = tg.tracking.track(algorithm, domain, field, seeds[:n], rng, *args)
    many = tg.tracking.track(algorithm, domain, field, seeds, rng, *args)
    _prefix_equal(few, many)


@pytest.mark.parametrize("n_samples", [17, 63, 64, 65])
def test_probabilistic_groups_follow_the_fp64_oracle(fast_runtime, n_samples, oracle_threads):
    # The tolerance and the field of the Probabilistic path's own test; 65
    # candidates run one lane per streamline.
    cfg = bench.brain145_diffusion(seed=1, n_seeds=300, shape=(49, 58, 49))
    field = tg.field.Image(tg.Nifti1Image(cfg["fod"], np.eye(4)))
    domain = tg.domain.Image(tg.Nifti1Image(cfg["mask"], np.eye(4)))
    algorithm = tg.algorithm.Probabilistic(tg.local.RealSymmetricSphericalHarmonics(45), n_samples=n_samples, seed=3,
                                           step_size=0.1)
    rng = [algorithm.get_rng_seed()]
    args = (cfg["seeds"], rng, 300, 0.25, 30.0)
    ref = oracle.track(domain, field, algorithm, *args, precision=64, threads=oracle_threads)
    fast = tg.tracking.track(algorithm, domain, field, *args, fast_runtime)
    r = deviation.report(fast.lengths, fast.steps, fast.points, ref, jump=1e-2)
    assert r["max_deviation"] <= 1e-3
    assert r["compared_fraction"] > 0.5


@pytest.mark.parametrize("n", [1, 9, 300])
@pytest.mark.parametrize("options", [{}, {"max_iterations": 0}, {"max_iterations": 1}, {"tolerance": 0.02},
                                     {"max_step_size": 0.05}])
def test_deterministic_groups_follow_the_fp64_oracle(fast_runtime, runtime, options, n, oracle_threads):
    # Updates that end before, in and after the first iteration, next to one
    # another in a wavefront; held to twice the plain path's own FP32
    # deviation, as the Deterministic path's own test.
    cfg = bench.brain145_diffusion(seed=1, n_seeds=n, shape=(49, 58, 49))
    field = tg.field.Image(tg.Nifti1Image(cfg["fod"], np.eye(4)))
    domain = tg.domain.Image(tg.Nifti1Image(cfg["mask"], np.eye(4)))
    algorithm = tg.algorithm.Deterministic(tg.local.RealSymmetricSphericalHarmonics(45), step_size=0.1, **options)
    args = (cfg["seeds"], [0], n, 0.25, 30.0)
    ref = oracle.track(domain, field, algorithm, *args, precision=64, threads=oracle_threads)
    fast = tg.tracking.track(algorithm, domain, field, *args, fast_runtime)
    plain = tg.tracking.track(algorithm, domain, field, *args, runtime)
    rf = deviation.report(fast.lengths, fast.steps, fast.points, ref, jump=1e-2)
    rp = deviation.report(plain.lengths, plain.steps, plain.points, ref, jump=1e-2)
    assert rf["max_deviation"] <= max(1e-3, 2.0 * rp["max_deviation"])
    assert rf["compared_fraction"] > 0.8 * rp["compared_fraction"]
