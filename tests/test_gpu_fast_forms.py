"""Which form of the fast path a tracking launch takes (tgk_runtime_fast_form),
and that the settings of the persistent kernel (grid, launch shape, repack
threshold) reach that kernel and change no result."""

import numpy as np
import pytest

import bench
import fixtures
import tractography_amd as tg
from tractography_amd import autotune

pytestmark = pytest.mark.gpu

SH45 = tg.local.RealSymmetricSphericalHarmonics(45)


@pytest.fixture(scope="module")
def scene():
    cfg = bench.sphere32_transport(seed=8, n_seeds=70_000)
    field = tg.field.Image(tg.Nifti1Image(cfg["fod"], np.eye(4)))
    domain = tg.domain.Image(tg.Nifti1Image(cfg["mask"], np.eye(4)))
    return cfg["seeds"], field, domain


def _diffusion(seed=58):
    return tg.algorithm.Diffusion(SH45, step_size=0.1, gamma=1.0, noise_variance=0.1, seed=seed)


def _track(runtime, algorithm, domain, field, seeds, max_length=60.0):
    return tg.tracking.track(algorithm, domain, field, seeds, [7], len(seeds), 0.25, max_length, runtime)


def _equal(got, ref):
    np.testing.assert_array_equal(got.lengths, ref.lengths)
    np.testing.assert_array_equal(got.steps, ref.steps)
    np.testing.assert_array_equal(got.hits, ref.hits)
    np.testing.assert_array_equal(got.points.view(np.uint32), ref.points.view(np.uint32))


@pytest.mark.parametrize("case", ["transport", "diffusion", "mesh"])
def test_every_launch_shape_of_the_persistent_kernel(scene, case):
    # On two blocks, so that lanes are refilled and generations are cut short
    # in every shape, and on the default grid; against the split form.
    seeds, field, domain = scene
    seeds = seeds[:2000].copy()
    algorithm = tg.algorithm.Transport(SH45, step_size=0.1, gamma=1.0) if case == "transport" else _diffusion()
    if case == "mesh":
        domain, seeds, _, _ = fixtures.shell_scene(n_seeds=2000, seed=13)
    default = tg.HipRuntime(path="fast")
    ref = _track(default, algorithm, domain, field, seeds)
    assert default.fast_form() == "split"
    for shape in range(len(tg.runtime.fast_shapes())):
        for grid, repack in ((2, 1 << 30), (2, 64), (0, 1 << 30)):
            runtime = tg.HipRuntime(path="fast")
            runtime.set_fast_shape(shape)
            runtime.set_fast_grid(grid)
            runtime.set_fast_repack(repack)
            _equal(_track(runtime, algorithm, domain, field, seeds), ref)
            assert runtime.fast_form() == ("split" if shape == 0 and grid == 0 else "lanes")


def test_forms_by_seeds_and_settings(scene):
    seeds, field, domain = scene
    runtime = tg.HipRuntime(path="fast")

    def form(n, algorithm=_diffusion(), dom=domain, fld=field):
        _track(runtime, algorithm, dom, fld, seeds[:n].copy(), 2.0)
        return runtime.fast_form()

    assert [form(n) for n in (1, 32768, 32769)] == ["split", "split", "lanes"]
    mesh, _, _, _ = fixtures.shell_scene(n_seeds=1, seed=13)
    assert [form(n, dom=mesh) for n in (65536, 65537)] == ["split", "lanes"]
    assert [form(100, tg.algorithm.Probabilistic(SH45, n_samples=k, step_size=0.2, seed=1)) for k in (64, 65)] == [
        "groups", "lanes"]
    assert [form(65537, tg.algorithm.Probabilistic(SH45, n_samples=k, step_size=0.2, seed=1)) for k in (16, 17)] == [
        "lanes", "groups"]
    assert form(100, tg.algorithm.Deterministic(SH45, step_size=0.2)) == "groups"
    # Settings keep few seeds on the kernel they are settings of, unless they
    # are marked as chosen for launches that fill the GPU.
    runtime.set_fast_shape(2)
    runtime.set_fast_repack(64)
    assert form(100) == "lanes"
    runtime.set_fast_tuned(True)
    assert [form(n) for n in (32768, 32769)] == ["split", "lanes"]
    runtime.set_fast_shape(0)
    runtime.set_fast_grid(4)
    assert form(100) == "lanes"


def test_probabilistic_generations(scene):
    # More candidates than groups take: one lane per streamline, cut short and
    # resumed four times over.
    seeds, field, domain = scene
    algorithm = tg.algorithm.Probabilistic(SH45, n_samples=65, step_size=0.1, seed=52)
    whole, cut = tg.HipRuntime(path="fast"), tg.HipRuntime(path="fast")
    whole.set_fast_repack(1 << 30)
    cut.set_fast_repack(8)
    ref = _track(whole, algorithm, domain, field, seeds[:2000].copy(), 20.0)
    got = _track(cut, algorithm, domain, field, seeds[:2000].copy(), 20.0)
    assert whole.fast_form() == cut.fast_form() == "lanes"
    _equal(got, ref)


def test_tuner_times_the_shapes_it_chooses_from(scene, monkeypatch):
    # A sample small enough for the split form, which has no shape.
    seeds, field, domain = scene
    runtime = tg.HipRuntime(path="fast")
    time_fast, forms = autotune.time_fast, []

    def recorded(*args, **kwargs):
        result = time_fast(*args, **kwargs)
        forms.append(runtime.fast_form())
        return result

    monkeypatch.setattr(autotune, "time_fast", recorded)
    tuned = autotune.tune_fast(_diffusion(), domain, field, seeds[:1000], runtime=runtime, save_at=0.25,
                               maximum_streamline_length=10.0, grid_factors=(1.0,), repacks=(1 << 30,), repeats=1,
                               cache=False)
    assert forms[:5] == ["lanes"] * 5
    # What is tuned is for launches that fill the GPU.
    autotune.apply(runtime, {**tuned, "blocks": 512})
    _track(runtime, _diffusion(), domain, field, seeds[:1000].copy(), 10.0)
    assert runtime.fast_form() == "split"
