"""Fast tracking by wavefronts that share a step, and launches that hand their
last streamlines over to them: the same tracks and the same memory reads as one
lane per streamline, which a fixed grid keeps (and which other tests hold to the
FP64 oracle, as they do launches of few seeds)."""

import numpy as np
import pytest

import bench
import fixtures
import tractography_amd as tg

pytestmark = pytest.mark.gpu

SPLIT = 32768  # seeds up to which a mask-domain launch is split throughout


@pytest.fixture(scope="module")
def scene():
    cfg = bench.sphere32_transport(seed=6, n_seeds=70_001)
    field = tg.field.Image(tg.Nifti1Image(cfg["fod"], np.eye(4)))
    domain = tg.domain.Image(tg.Nifti1Image(cfg["mask"], np.eye(4)))
    return cfg["seeds"], field, domain


def _algorithm(name):
    model = tg.local.RealSymmetricSphericalHarmonics(45)
    if name == "transport":
        return tg.algorithm.Transport(model, step_size=0.2, gamma=1.0)
    return tg.algorithm.Diffusion(model, step_size=0.2, gamma=1.0, noise_variance=0.1, seed=3)


def _one_lane(blocks=1024):
    runtime = tg.HipRuntime(path="fast")
    runtime.set_fast_grid(blocks)
    runtime.set_fast_repack(2**31 - 1)
    return runtime


def _equal(algorithm, domain, field, seeds, split, reads=True):
    tracks = []
    for runtime in (split, _one_lane()):
        tracks.append(tg.tracking.track(algorithm, domain, field, seeds, [11], len(seeds), 0.5, 15.0, runtime))
        tracks[-1].reads = runtime.fast_reads()
    got, ref = tracks
    np.testing.assert_array_equal(got.lengths, ref.lengths)
    np.testing.assert_array_equal(got.steps, ref.steps)
    np.testing.assert_array_equal(got.hits, ref.hits)
    np.testing.assert_array_equal(got.points, ref.points)
    if reads:
        assert got.reads == ref.reads


@pytest.mark.parametrize("name", ["transport", "diffusion"])
@pytest.mark.parametrize("n", [1, 63, 65, SPLIT - 1])
def test_mask_domain(scene, name, n):
    seeds, field, domain = scene
    _equal(_algorithm(name), domain, field, seeds[:n].copy(), tg.HipRuntime(path="fast"))


@pytest.mark.parametrize("name", ["transport", "diffusion"])
def test_mask_image_other_than_the_fields(scene, name):
    # The mask on a grid and an affine of its own, and seeds that leave it.
    seeds, field, _ = scene
    mask = np.zeros((40, 36, 44), dtype=np.uint8)
    mask[2:-2, 2:-2, 2:-2] = 1
    affine = np.diag([0.75, 0.8, 0.7, 1.0])
    domain = tg.domain.Image(tg.Nifti1Image(mask, affine))
    few = seeds[:1000].copy()
    few[3, :3] = 1e6
    few[4, 4:7] = 0.0
    _equal(_algorithm(name), domain, field, few, tg.HipRuntime(path="fast"))


@pytest.mark.parametrize("name", ["transport", "diffusion"])
@pytest.mark.parametrize("n", [65, 3001])
def test_mesh_domain(scene, name, n):
    _, field, _ = scene
    mesh, seeds, _, _ = fixtures.shell_scene(n_seeds=n, seed=14)
    _equal(_algorithm(name), mesh, field, seeds, tg.HipRuntime(path="fast"))


# Launches handed over in the first, a middle or the last generation, and a
# small grid's (what a launch reads then depends on when each one ends).
@pytest.mark.parametrize("n, blocks, repack", [(SPLIT, 0, 16384), (70_001, 0, 16384), (70_001, 0, 1), (5000, 4, 16),
                                               (300, 1, 1)])
def test_last_streamlines(scene, n, blocks, repack):
    seeds, field, domain = scene
    runtime = tg.HipRuntime(path="fast")
    runtime.set_fast_grid(blocks)
    runtime.set_fast_repack(repack)
    for name in ("transport", "diffusion"):
        _equal(_algorithm(name), domain, field, seeds[:n].copy(), runtime, reads=False)
