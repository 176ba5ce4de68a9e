"""Timed cases of the tracking engine: what a user's program has it do, from a
handful of seeds in a phantom to a million streamlines of a whole brain.

A case names a product and its options:

``tractogram``  ``tg.tractogram`` on prepared field and domain objects, host
                seeds in, ragged streamlines out, transfers included; the
                program gathers them in an array of its own.
``device``      the same tracking on buffers that stay in HBM: the C entry
                points ``tgk_track_device`` and ``tgk_compact_device``.
``seeds``       seeds drawn from a FOD on the device
                (``tgk_seeds_from_fod_device``).
``connectome``  boundary-seeded tracks to vertex-pair weights in host arrays
                (the C entry point ``tgk_connectome``).
``tod``         ``tg.tod`` from boundary seeds, the normalised orientation image.

Volumes are synthetic: one to three fibres per voxel that follow smooth random
direction fields (or independent random directions, ``fibres="random"``),
projected to spherical harmonics and normalised to unit integral, inside an
ellipsoid; tensors for DTI. Seeds are uniform in the ellipsoid with uniform
directions, or between two nested closed surfaces for mesh domains.
"""

from __future__ import annotations

import ctypes
import functools
import math

import numpy as np
import torch

import tractography_amd as tg
from tractography_amd import _native

BRAIN = (145, 174, 145)
SEMI_AXES = (60.0, 75.0, 60.0)  # of the domain ellipsoid in a BRAIN volume


def _case(name, kind, shape, n, **options):
    case = {
        "name": name, "kind": kind, "nx": shape[0], "ny": shape[1], "nz": shape[2], "n": n, "path": "fast",
        "model": "sh", "coefficients": 45, "algorithm": "diffusion", "fibres": "smooth", "step_size": 0.1,
        "save_at": 0.25, "max_length": 300.0, "triangles": 0, "batch_size": 50000, "method": "valu",
    }
    case.update(options)
    return case


def listed():
    return [
        # A first look at a phantom: a few dozen seeds on the default path.
        # Launches, copies and the chain of dependent steps are all there is.
        _case("phantom_plain", "tractogram", (16, 15, 14), 64, path="plain", algorithm="transport", fibres="random",
              save_at=1.0, max_length=20.0),
        # The 32^3 sphere of 10k Transport seeds (the benchmark's smallest
        # configuration), on the default path and on the fast one: far fewer
        # streamlines than lanes, each up to 3000 dependent steps.
        _case("sphere32_plain", "tractogram", (32, 32, 32), 10000, path="plain", algorithm="transport",
              fibres="random", save_at=1.0),
        _case("sphere32_fast", "tractogram", (32, 32, 32), 10000, algorithm="transport", fibres="random",
              save_at=1.0),
        # A whole-brain tractogram on the default path.
        _case("brain_sh_plain", "device", BRAIN, 300000, path="plain"),
        # The benchmark's headline: a million streamlines tracked and
        # compacted in HBM.
        _case("brain_sh_fast", "device", BRAIN, 1000000),
        # Whole-brain DTI.
        _case("brain_dti_fast", "device", BRAIN, 500000, model="dti", coefficients=6, algorithm="transport"),
        # Termination against two surfaces instead of a mask, default path.
        _case("shell_plain", "device", (97, 116, 97), 200000, path="plain", triangles=40000),
        # The sampling algorithm with its own defaults (64 candidates, step
        # 0.25) and the peak-following one.
        _case("probabilistic_fast", "device", (97, 116, 97), 150000, algorithm="probabilistic", step_size=0.25,
              save_at=0.5),
        _case("deterministic_fast", "device", (97, 116, 97), 100000, algorithm="deterministic", save_at=0.5),
        # Seeding from the FOD itself, the default method.
        _case("seeds_valu", "seeds", (97, 116, 97), 1000000, path="plain"),
        # The two boundary-seeded products.
        _case("connectome_fast", "connectome", (97, 116, 97), 300000),
        _case("tod_fast", "tod", (97, 116, 97), 300000),
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


# The most seeds of a drawn case by algorithm, on the fast and the plain path:
# what keeps it below the largest listed one.
_MOST_SEEDS = {
    "transport": (600000, 200000), "diffusion": (600000, 200000), "probabilistic": (150000, 30000),
    "deterministic": (100000, 20000),
}


def draw(rng):
    kind = rng.choice(["tractogram", "tractogram", "device", "device", "seeds", "connectome", "tod"])
    edge = _log_uniform(rng, 14, 120)
    shape = tuple(max(8, int(edge * rng.uniform(0.8, 1.2))) for _ in range(3))
    path = rng.choice(["plain", "fast"])
    model = rng.choice(["sh", "sh", "sh", "dti"])
    algorithm = rng.choice(["transport", "diffusion", "diffusion", "probabilistic", "deterministic"])
    options = {
        "path": path, "model": model, "coefficients": 6 if model == "dti" else rng.choice([15, 28, 45, 45, 45]),
        "algorithm": algorithm, "fibres": rng.choice(["smooth", "smooth", "random"]),
        "step_size": rng.choice([0.1, 0.1, 0.2, 0.25, 0.5]), "save_at": rng.choice([0.25, 0.5, 1.0]),
        "max_length": round(rng.uniform(20.0, 300.0), 1), "batch_size": rng.choice([1000, 50000, 50000, 100003]),
    }
    most = _MOST_SEEDS[algorithm][0 if path == "fast" else 1]
    if kind == "tractogram":
        most = min(most, 20000)
        options["save_at"] = 1.0
    elif kind == "seeds":
        options["method"] = rng.choice(["valu", "valu", "mfma"])
        if options["method"] == "mfma" and model == "sh":
            options["coefficients"] = rng.choice([15, 45, 45, 91])
        most = 2000000
    elif kind in ("connectome", "tod"):
        most = min(most, 300000)
        options["fibres"] = "smooth"
    elif path == "fast" and kind == "device" and model == "sh" and algorithm in ("transport", "diffusion"):
        options["coefficients"] = rng.choice([45, 45, 45, 91])
        if options["coefficients"] == 91:
            most = 200000
    if kind in ("tractogram", "device") and min(shape) >= 24 and rng.random() < 0.25:
        options["triangles"] = _log_uniform(rng, 400, 60000)
    case = _case("", kind, shape, _log_uniform(rng, 50, most), **options)
    del case["name"]
    return case


# ------------------------------------------------------------- volumes ---


def _coefficient_degrees(K):
    degrees = []
    l = 0
    while len(degrees) < K:
        degrees.extend([l] * (2 * l + 1))
        l += 2
    return degrees[:K]


def _sh_basis(x, y, z, K):
    """Real symmetric SH values (K, ...) of unit vectors, MRtrix order (index
    l(l+1)/2 + m over even l), in the inputs' precision."""
    lmax = max(_coefficient_degrees(K))
    out = [None] * ((lmax + 1) * (lmax + 2) // 2)
    # sin^m theta (cos, sin)(m phi) by powers of x + i y; the Legendre part
    # divided by sin^m theta by the normalised three-term recurrence in l.
    cm, sm = torch.ones_like(x), torch.zeros_like(x)
    p_mm = math.sqrt(1.0 / (4.0 * math.pi))
    for m in range(lmax + 1):
        if m > 0:
            p_mm *= -math.sqrt((2 * m + 1) / (2 * m))
            cm, sm = cm * x - sm * y, cm * y + sm * x
        before, now = None, torch.full_like(z, p_mm)
        for l in range(m, lmax + 1):
            if l == m + 1:
                before, now = now, math.sqrt(2 * m + 3) * z * now
            elif l > m + 1:
                a = math.sqrt((4 * l * l - 1) / (l * l - m * m))
                b = math.sqrt(((l - 1) ** 2 - m * m) / (4 * (l - 1) ** 2 - 1))
                before, now = now, a * (z * now - b * before)
            if l % 2 == 0:
                centre = l * (l + 1) // 2
                if m == 0:
                    out[centre] = now
                else:
                    out[centre + m] = math.sqrt(2.0) * now * cm
                    out[centre - m] = math.sqrt(2.0) * now * sm
    return torch.stack(out[:K])


def _kernel_weights(K, sharpness=4.0):
    """Funk-Hecke weights of the fibre kernel exp(sharpness (t^2 - 1))."""
    t, w = np.polynomial.legendre.leggauss(200)
    k = np.exp(sharpness * (t * t - 1.0))
    return [2 * math.pi * float(np.sum(w * k * np.polynomial.legendre.Legendre.basis(l)(t)))
            for l in _coefficient_degrees(K)]


def _directions(g, shape, n, fibres):
    """n unit vectors per voxel, (n, 3, X, Y, Z): independent, or Gaussian
    noise blurred over four voxels."""
    d = torch.randn((n, 3, *shape), generator=g, device="cuda")
    if fibres == "smooth":
        for axis, size in enumerate(shape):
            i = torch.arange(size, device="cuda", dtype=torch.float32)
            blur = torch.exp(-0.5 * ((i[:, None] - i[None, :]) / 4.0) ** 2)
            blur /= blur.sum(dim=1, keepdim=True)
            d = torch.movedim(torch.tensordot(d, blur, dims=([2 + axis], [1])), -1, 2 + axis)
    return d / torch.linalg.vector_norm(d, dim=1, keepdim=True)


def _ellipsoid(shape):
    semi = [a * s / b for a, s, b in zip(SEMI_AXES, shape, BRAIN)]
    axes = [((torch.arange(s, device="cuda") - (s - 1) / 2.0) / a) ** 2 for s, a in zip(shape, semi)]
    return axes[0][:, None, None] + axes[1][None, :, None] + axes[2][None, None, :] <= 1.0


def _volume(case, g):
    """(X, Y, Z, K) float32 coefficients and the mask, on the GPU."""
    shape = (case["nx"], case["ny"], case["nz"])
    mask = _ellipsoid(shape)
    if case["model"] == "dti":
        e = _directions(g, shape, 1, case["fibres"])[0]
        low, delta = 0.3e-3, 1.4e-3
        e = torch.where(mask, e, torch.zeros_like(e))
        flat = torch.where(mask, low, 0.8e-3)
        rows = [flat + delta * e[i] * e[i] for i in range(3)]
        rows += [delta * e[i] * e[j] for i, j in ((0, 1), (0, 2), (1, 2))]
        return torch.stack(rows, dim=-1).contiguous(), mask
    K = case["coefficients"]
    d = _directions(g, shape, 3, case["fibres"])
    weights = torch.empty((3, *shape), device="cuda").exponential_(generator=g)
    count = torch.randint(1, 4, shape, generator=g, device="cuda")
    for i in range(3):
        weights[i] *= i < count
    weights /= weights.sum(dim=0)
    kernel = torch.tensor(_kernel_weights(K), device="cuda", dtype=torch.float32)
    fod = torch.empty((*shape, K), device="cuda")
    for x in range(0, shape[0], 16):  # slabs: the basis of three fibres is large
        part = slice(x, x + 16)
        acc = sum(_sh_basis(d[i, 0, part], d[i, 1, part], d[i, 2, part], K) * weights[i, part] for i in range(3))
        acc *= kernel[:, None, None, None]
        fod[part] = torch.movedim(acc / (math.sqrt(4.0 * math.pi) * acc[:1]), 0, -1)
    fod *= mask[..., None]
    return fod, mask


def _homogeneous(points, g):
    d = torch.randn(points.shape, generator=g, device="cuda")
    seeds = torch.zeros((len(points), 8), device="cuda")
    seeds[:, :3] = points
    seeds[:, 3] = 1.0
    seeds[:, 4:7] = d / torch.linalg.vector_norm(d, dim=1, keepdim=True)
    return seeds


def _seeds_in_mask(mask, n, g):
    voxels = torch.nonzero(mask)
    index = torch.randint(0, len(voxels), (n,), generator=g, device="cuda")
    return _homogeneous(voxels[index] + torch.rand((n, 3), generator=g, device="cuda") - 0.5, g)


class _Shell:
    """Two nested closed surfaces about the volume centre: ellipsoids of the
    domain's semi-axes and of half of them, displaced radially by a random
    quadratic form."""

    def __init__(self, case, rng):
        shape = (case["nx"], case["ny"], case["nz"])
        self.centre = (np.array(shape) - 1) / 2.0
        semi = np.array(SEMI_AXES) * np.array(shape) / np.array(BRAIN)
        self.semi = (semi, 0.5 * semi)
        self.forms = []
        for _ in range(2):
            q = rng.standard_normal((3, 3))
            self.forms.append((q + q.T) * 0.03 * semi.min() / np.linalg.norm(q + q.T, 2))
        rings = max(6, int(round(math.sqrt(case["triangles"] / 2))))
        parts = [self._surface(i, rings, rings) for i in range(2)]
        self.vertices = np.vstack([v for v, _ in parts])
        self.faces = np.vstack([parts[0][1], parts[1][1][:, ::-1] + len(parts[0][0])])

    def radius(self, i, u):
        return 1.0 / np.sqrt(((u / self.semi[i]) ** 2).sum(axis=1)) + np.einsum("ni,ij,nj->n", u, self.forms[i], u)

    def _surface(self, i, rings, segments):
        theta = math.pi * np.arange(1, rings) / rings
        phi = 2.0 * math.pi * np.arange(segments) / segments
        ring = np.stack([np.outer(np.sin(theta), np.cos(phi)), np.outer(np.sin(theta), np.sin(phi)),
                         np.repeat(np.cos(theta)[:, None], segments, axis=1)], axis=-1).reshape(-1, 3)
        u = np.vstack([[0.0, 0.0, 1.0], ring, [0.0, 0.0, -1.0]])
        vertices = self.centre + self.radius(i, u)[:, None] * u
        a = 1 + np.arange((rings - 2) * segments).reshape(rings - 2, segments)
        d = np.roll(a, -1, axis=1)
        b, c = a + segments, d + segments
        first, last = a[0], b[-1]
        faces = np.concatenate([
            np.stack([np.zeros(segments, dtype=int), first, np.roll(first, -1)], axis=1),
            np.stack([a.ravel(), b.ravel(), c.ravel()], axis=1),
            np.stack([a.ravel(), c.ravel(), d.ravel()], axis=1),
            np.stack([np.full(segments, len(u) - 1), np.roll(last, -1), last], axis=1),
        ])
        return vertices, faces

    def seeds(self, n, rng):
        kept, count = [], 0
        while count < n:
            q = rng.uniform(-1.1, 1.1, (4 * (n - count) + 1024, 3)) * self.semi[0]
            r = np.linalg.norm(q, axis=1)
            u = q / np.maximum(r, 1e-9)[:, None]
            q = q[(r > self.radius(1, u) + 0.5) & (r < self.radius(0, u) - 0.5)]
            kept.append(q + self.centre)
            count += len(q)
        return np.concatenate(kept)[:n].astype(np.float32)


# ------------------------------------------------------------ programs ---


@functools.lru_cache(maxsize=None)
def _runtime(path):
    """A program makes a runtime once and keeps it."""
    return tg.HipRuntime(path=path)


def _algorithm(case, seed):
    if case["model"] == "dti":
        model = tg.local.DiffusionTensorImaging()
    else:
        model = tg.local.RealSymmetricSphericalHarmonics(case["coefficients"])
    step = case["step_size"]
    if case["algorithm"] == "transport":
        return tg.algorithm.Transport(model, step_size=step, gamma=1.0)
    if case["algorithm"] == "diffusion":
        return tg.algorithm.Diffusion(model, step_size=step, gamma=1.0, noise_variance=0.1, seed=seed)
    if case["algorithm"] == "probabilistic":
        return tg.algorithm.Probabilistic(model, seed=seed, step_size=step)
    return tg.algorithm.Deterministic(model, step_size=step)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    rng = np.random.default_rng(seed)
    runtime = _runtime(case["path"])
    volume, mask = _volume(case, g)
    state = {"case": case, "seed": seed, "runtime": runtime}
    if case["kind"] == "seeds":
        inside = mask & (volume != 0).any(dim=-1)
        voxels = torch.nonzero(inside).to(torch.float32)
        state["fod"] = volume[inside].contiguous()
        state["voxels"] = torch.cat([voxels, torch.ones_like(voxels[:, :1])], dim=1).contiguous()
        state["affine"] = torch.eye(4, device="cuda")
        states = rng.integers(0, 2**32 - 1, (case["n"], 2), dtype=np.uint32)
        state["states"] = torch.from_numpy(states.view(np.int32)).cuda()
        state["seeds"] = torch.empty((case["n"], 8), device="cuda")
        state["model"] = 1 if case["model"] == "dti" else 0
        state["method"] = tg.seeds.METHODS[case["method"]]
        _native.check(_native.lib().tgk_seeds_prepare(runtime.handle, state["model"], case["coefficients"],
                                                      state["method"]))
        return state

    affine = np.eye(4)
    state["field"] = tg.field.Image(tg.Nifti1Image(volume.cpu().numpy(), affine))
    state["field"].upload(runtime)
    del volume
    if case["triangles"]:
        # Culling cells of half a voxel that certify segments of 1.5 steps.
        shell = _Shell(case, rng)
        state["domain"] = tg.domain.Mesh(shell.vertices, shell.faces, cell_size=0.5, reach=1.5 * case["step_size"])
        points = torch.from_numpy(shell.seeds(case["n"], rng)).cuda()
        seeds = _homogeneous(points, g)
    else:
        state["domain"] = tg.domain.Image(tg.Nifti1Image(mask.to(torch.uint8).cpu().numpy(), affine))
        seeds = None
        if case["kind"] in ("tractogram", "device"):
            seeds = _seeds_in_mask(mask, case["n"], g)
    # Boundary-seeded products sample the domain's surface: its mesh and the
    # bounding volumes over it belong to the domain object.
    domain = state["domain"].upload(runtime, with_boundary=case["kind"] in ("connectome", "tod"))
    state["domain_handle"] = domain
    n = case["n"]
    points = tg.tracking.point_capacity(case["max_length"], case["save_at"])
    if case["kind"] == "connectome":
        state["boundary_handle"] = tg.domain._mesh_handle_for(state["domain"], runtime)
        state["rows"] = np.zeros(9 * n, dtype=np.int32)
        state["cols"] = np.zeros(9 * n, dtype=np.int32)
        state["weights"] = np.zeros(9 * n, dtype=np.float32)
    elif case["kind"] == "tractogram":
        state["seeds"] = seeds.cpu().numpy()
        state["points"] = np.zeros((n * points, 3), dtype=np.float32)
    elif case["kind"] == "device":
        algorithm = _algorithm(case, seed)
        batches = [algorithm.get_rng_seed() for _ in range(-(-n // case["batch_size"]))]
        state.update(
            seeds=seeds, n_points=points, descriptor=algorithm.descriptor(),
            rng=torch.from_numpy(np.array(batches, dtype=np.uint32).view(np.int32)).cuda(),
            lengths=torch.empty(n, dtype=torch.int32, device="cuda"),
            steps=torch.empty(n, dtype=torch.int32, device="cuda"),
            hits=torch.empty(n, dtype=torch.int32, device="cuda"),
            offsets=torch.empty(n + 1, dtype=torch.int64, device="cuda"),
            dense=torch.empty(n * points * 3, device="cuda"),
            points=torch.zeros(n * points * 3, device="cuda"),
        )
        _native.check(_native.lib().tgk_track_prepare(
            runtime.handle, domain.handle, state["field"].upload(runtime).handle, ctypes.byref(state["descriptor"]),
            runtime.path_id, n))
    return state


def run(state):
    case, runtime = state["case"], state["runtime"]
    kind = case["kind"]
    if kind == "tractogram":
        result = tg.tractogram(
            state["field"], state["seeds"], state["domain"], _algorithm(case, state["seed"]), save_at=case["save_at"],
            maximum_streamline_length=case["max_length"], batch_size=case["batch_size"], runtime=runtime)
        data = result.streamlines.data
        state["points"][: len(data)] = data
        return {"points": state["points"], "lengths": result.streamlines.lengths}
    if kind == "tod":
        image = tg.tod(state["field"], case["n"], state["domain"], _algorithm(case, state["seed"]),
                       maximum_streamline_length=case["max_length"], runtime=runtime)
        return image.dataobj
    lib = _native.lib()
    if kind == "seeds":
        _native.check(lib.tgk_seeds_from_fod_device(
            runtime.handle, state["model"], case["coefficients"], state["fod"].data_ptr(), state["voxels"].data_ptr(),
            len(state["voxels"]), state["affine"].data_ptr(), state["states"].data_ptr(), case["n"], state["method"],
            state["seeds"].data_ptr()))
        return {"seeds": state["seeds"], "states": state["states"]}
    if kind == "connectome":
        algorithm = _algorithm(case, state["seed"])
        _native.check(lib.tgk_connectome(
            runtime.handle, state["domain_handle"].handle, state["boundary_handle"].handle,
            state["field"].upload(runtime).handle, algorithm.descriptor(), runtime.path_id, algorithm.get_rng_seed(),
            case["n"], int(case["max_length"] / case["step_size"]), 0.0, _native.ptr(state["rows"]),
            _native.ptr(state["cols"]), _native.ptr(state["weights"])))
        return {k: state[k] for k in ("rows", "cols", "weights")}
    n, n_points = case["n"], state["n_points"]
    _native.check(lib.tgk_track_device(
        runtime.handle, state["domain_handle"].handle, state["field"].upload(runtime).handle,
        ctypes.byref(state["descriptor"]), runtime.path_id, state["seeds"].data_ptr(), 0, n, state["rng"].data_ptr(),
        case["batch_size"], n_points, float(np.float32(case["save_at"])), state["lengths"].data_ptr(),
        state["steps"].data_ptr(), state["hits"].data_ptr(), state["dense"].data_ptr()))
    _native.check(lib.tgk_compact_device(
        runtime.handle, runtime.path_id, state["dense"].data_ptr(), n, n_points, state["lengths"].data_ptr(),
        state["offsets"].data_ptr(), state["points"].data_ptr()))
    return {k: state[k] for k in ("points", "offsets", "lengths", "steps", "hits")}


# ---------------------------------------------------------------- work ---


def _mean_steps(case):
    """Expected orientation updates of a streamline: the paths are close to
    diffusive walks that leave an ellipsoid of mean semi-axis r after about
    2 r voxels, cut at the maximum length (1248 of 3000 steps in the
    145 x 174 x 145 volume)."""
    r = sum(a * case[k] / b for a, k, b in zip(SEMI_AXES, ("nx", "ny", "nz"), BRAIN)) / 3.0
    mean = 2.0 * r * (1.0 - math.exp(-case["max_length"] / (2.0 * r)))
    return max(1.0, mean / case["step_size"])


def work(case):
    n, K = case["n"], case["coefficients"]
    voxels = case["nx"] * case["ny"] * case["nz"]
    if case["kind"] == "seeds":
        # The coefficients of each seed's voxel, its state in and out and its
        # row; one product with the 1000 directions and its running sum.
        return {"bytes": n * (4.0 * K + 16 + 16 + 32), "flops": n * 1000.0 * (2 * K + 2)}
    steps = n * _mean_steps(case)
    # An evaluation: value and gradient, or the value alone, as one
    # contraction each, and what turns it into a direction.
    full, value = 6.0 * K + 60, 2.0 * K + 30
    per_step = {"transport": full, "diffusion": full + 20, "probabilistic": 64 * (value + 20),
                "deterministic": 5 * full + value}[case["algorithm"]]
    # A row and a mask value each time the voxel changes, about every 0.65
    # voxel of arc length.
    moved = steps * min(1.0, case["step_size"] / 0.65) * (4.0 * K + 1)
    if case["kind"] == "connectome":
        return {"bytes": moved + n * 9 * 12.0, "flops": steps * per_step}
    if case["kind"] == "tod":
        return {"bytes": moved + voxels * 45 * 4.0, "flops": steps * (per_step + 150)}
    points = n + steps * case["step_size"] / case["save_at"]
    return {"bytes": moved + points * 12 + n * (32 + 12.0), "flops": steps * per_step}


# --------------------------------------------------------------- exact ---


def _randu(x, c):
    """One draw of every stream (uint32 halves held in int64): the draw, and
    the advanced state x A + c as a 64-bit multiply with carry."""
    draw = ((x ^ c) >> 8).to(torch.float64) * 2.0**-24
    a = 4294883355
    low = x * (a & 0xFFFF) + c
    high = x * (a >> 16) + (low >> 16)
    return draw, ((high & 0xFFFF) << 16) | (low & 0xFFFF), high >> 16


def exact(case, seed):
    """Seeds drawn from a FOD, in 64 bits on the same noise streams.

    The other products have no such value: a path reads the nearest voxel, so
    where it passes within a rounding of a voxel's face it goes on in another
    cell, and its points, its length and what is summed along it are those of
    another path."""
    if case["kind"] != "seeds":
        return None
    g = torch.Generator(device="cuda").manual_seed(seed)
    rng = np.random.default_rng(seed)
    volume, mask = _volume(case, g)
    inside = mask & (volume != 0).any(dim=-1)
    voxels = torch.nonzero(inside)
    rows = volume[inside]
    states = torch.from_numpy(rng.integers(0, 2**32 - 1, (case["n"], 2), dtype=np.uint32).astype(np.int64)).cuda()

    i = torch.arange(1000, dtype=torch.float64, device="cuda")
    z = 1.0 - 2.0 * i / 999.0
    r = torch.sqrt(torch.clamp(1.0 - z * z, min=0.0))
    angle = i * (2.0 * math.pi / ((math.sqrt(5.0) + 1.0) / 2.0))
    directions = torch.stack([r * torch.cos(angle), r * torch.sin(angle), z], dim=1)
    if case["model"] == "dti":
        x, y, z = directions.T
        basis = torch.stack([x * x, y * y, z * z, 2 * x * y, 2 * x * z, 2 * y * z])
    else:
        basis = _sh_basis(*directions.T, case["coefficients"])

    out = torch.zeros((case["n"], 8), dtype=torch.float64, device="cuda")
    for first in range(0, case["n"], 1 << 15):
        x, c = states[first : first + (1 << 15)].T
        pick, x, c = _randu(x, c)
        # The voxel is a draw of single precision by definition.
        index = (pick.to(torch.float32) * np.float32(len(voxels))).to(torch.int64).clamp(max=len(voxels) - 1)
        part = out[first : first + (1 << 15)]
        for axis in range(3):
            jitter, x, c = _randu(x, c)
            part[:, axis] = voxels[index, axis] + (jitter - 0.5)
        values = rows[index].to(torch.float64) @ basis
        if case["model"] != "dti":
            values = torch.where(values * 100.0 < 30.0, torch.log1p(torch.exp(100.0 * values)) / 100.0, values)
        sums = torch.cumsum(torch.clamp(values, min=0.0), dim=1)
        target, x, c = _randu(x, c)
        above = sums > (target * sums[:, -1])[:, None]
        chosen = directions[torch.argmax(above.to(torch.uint8), dim=1)]
        part[:, 3] = 1.0
        part[:, 4:7] = torch.where(above[:, -1:], chosen, torch.tensor([0.0, 0.0, 1.0], dtype=torch.float64,
                                                                       device="cuda"))
    return {"seeds": out, "states": None}
