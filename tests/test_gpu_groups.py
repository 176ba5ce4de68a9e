"""Lane groups of the fast path (several lanes per streamline): the same tracks
as one lane per streamline, and the FP64 oracle's."""

import numpy as np
import pytest

import bench
import deviation
import fixtures
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


def _few_equal_many(runtime, domain, field, seeds, model, n_samples):
    # The many in one chunk, one lane per streamline; the few by groups.
    algorithm = tg.algorithm.Probabilistic(model, n_samples=n_samples, max_angle=0.4, seed=7, step_size=0.2)
    rng = [algorithm.get_rng_seed() for _ in range(MANY // 1000 + 1)]
    args = (1000, 0.5, 15.0, runtime)
    few = tg.tracking.track(algorithm, domain, field, seeds[:3001], rng, *args)
    assert runtime.fast_form() == "groups"
    many = tg.tracking.track(algorithm, domain, field, seeds, rng, *args)
    assert runtime.fast_form() == "lanes"
    _prefix_equal(few, many)
    np.testing.assert_array_equal(few.hits, many.hits[: len(few.hits)])
    return few


@pytest.mark.parametrize("n_samples", [7, 16])
@pytest.mark.parametrize("kind", ["mesh", "dti", "dti mesh", "order 12", "order 12 mesh"])
def test_probabilistic_groups_equal_single_lanes_on(fast_runtime, scene, kind, n_samples):
    # The other instances of the group kernel: the boundary asked once per
    # group, the tensor model, the order-12 polynomial.
    seeds, field, domain = scene
    model = tg.local.RealSymmetricSphericalHarmonics(45)
    if "dti" in kind:
        rng = np.random.default_rng(3)
        e = rng.standard_normal((32, 32, 32, 3))
        e /= np.linalg.norm(e, axis=-1, keepdims=True)
        tensor = 0.3e-3 * np.eye(3) + 1.4e-3 * e[..., :, None] * e[..., None, :]
        rows = np.stack([tensor[..., i, j] for i, j in ((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))], axis=-1)
        field = tg.field.Image(tg.Nifti1Image(rows.astype(np.float32), np.eye(4)))
        model = tg.local.DiffusionTensorImaging()
    elif "order 12" in kind:
        rng = np.random.default_rng(4)
        directions = bench.smooth_direction_fields(rng, (32, 32, 32), sigma=3.0)
        _, weights = bench._random_fibres(rng, 32**3, base_directions=directions)
        fod = bench.fod_from_fibres(directions, weights, lmax=12).reshape(32, 32, 32, 91)
        field = tg.field.Image(tg.Nifti1Image(fod.astype(np.float32), np.eye(4)))
        model = tg.local.RealSymmetricSphericalHarmonics(91)
    if "mesh" in kind:
        domain, seeds, _, _ = fixtures.shell_scene(n_seeds=MANY, seed=15)
    few = _few_equal_many(fast_runtime, domain, field, seeds, model, n_samples)
    assert few.steps.sum() > 10_000
    if "mesh" in kind:
        assert np.mean(few.hits != np.iinfo(np.uint32).max) > 0.05


@pytest.mark.parametrize("name", ["probabilistic", "deterministic"])
def test_group_boundary_tests_equal_the_traversal(fast_runtime, scene, name):
    # Candidate lists that decide, that every segment outruns, and none: the
    # same hits, hence the same tracks.
    _, field, _ = scene
    model = tg.local.RealSymmetricSphericalHarmonics(45)
    geometry = np.random.default_rng(16)
    outer, inner = (13.0, 14.0, 12.0), (5.0, 6.0, 5.0)
    vertices, faces, centre, radii = bench.shell_domain(geometry, (32, 32, 32), outer, inner, 30, 36, 1.0)
    seeds = bench.seeds_in_shell(geometry, centre, radii, np.asarray(outer) + 2.0, 1500)
    results = []
    for cell_size, reach in [(0.5, 0.15), (1.0, 0.09), (1.0, 0.0)]:
        if name == "probabilistic":
            algorithm = tg.algorithm.Probabilistic(model, n_samples=20, seed=5, step_size=0.1)
        else:
            algorithm = tg.algorithm.Deterministic(model, step_size=0.1)
        domain = tg.domain.Mesh(vertices, faces, cell_size=cell_size, reach=reach)
        results.append(tg.tracking.track(algorithm, domain, field, seeds, [3], 1500, 0.25, 30.0, fast_runtime))
        assert fast_runtime.fast_form() == "groups"
    assert np.mean(results[0].hits != np.iinfo(np.uint32).max) > 0.05
    for r in results[:-1]:
        _prefix_equal(r, results[-1])
        np.testing.assert_array_equal(r.hits, results[-1].hits)


def test_deterministic_groups_on_a_mesh_follow_the_fp64_oracle(fast_runtime, runtime, oracle_threads):
    # Held as the mask domain's above.
    cfg = bench.brain145_diffusion(seed=1, n_seeds=1, shape=(32, 32, 32))
    field = tg.field.Image(tg.Nifti1Image(cfg["fod"], np.eye(4)))
    mesh, seeds, _, _ = fixtures.shell_scene(n_seeds=600, seed=17)
    algorithm = tg.algorithm.Deterministic(tg.local.RealSymmetricSphericalHarmonics(45), step_size=0.1)
    args = (seeds, [0], 600, 0.25, 20.0)
    ref = oracle.track(mesh, field, algorithm, *args, precision=64, threads=oracle_threads)
    fast = tg.tracking.track(algorithm, mesh, field, *args, fast_runtime)
    plain = tg.tracking.track(algorithm, mesh, field, *args, runtime)
    rf = deviation.report(fast.lengths, fast.steps, fast.points, ref, jump=1e-2)
    rp = deviation.report(plain.lengths, plain.steps, plain.points, ref, jump=1e-2)
    assert rf["max_deviation"] <= max(1e-3, 2.0 * rp["max_deviation"])
    assert rf["compared_fraction"] > 0.8 * rp["compared_fraction"]
    same = (fast.lengths == ref["lengths"]) & (fast.steps == ref["steps"])
    assert np.mean(fast.hits[same] == ref["hits"][same]) > 0.99
