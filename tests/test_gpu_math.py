"""The device's branch-free elementary functions against the host's: every
mantissa where a quotient is formed without the division's special cases, and
the arguments that are left to the shared code."""

import numpy as np
import pytest

import oracle
import tractography_amd as tg
from tractography_amd import _native

pytestmark = pytest.mark.gpu


def _device(runtime, fn, x, y=None):
    x = np.ascontiguousarray(x, dtype=np.float32)
    y = np.ascontiguousarray(x if y is None else y, dtype=np.float32)
    out = np.empty_like(x)
    _native.check(_native.lib().tgk_math(runtime.handle, fn, _native.ptr(x), _native.ptr(y), len(x), _native.ptr(out)))
    return out


def _same(got, ref):
    nan = np.isnan(ref)
    np.testing.assert_array_equal(np.isnan(got), nan)
    np.testing.assert_array_equal(got[~nan].view(np.uint32), ref[~nan].view(np.uint32))


@pytest.mark.parametrize("exponent", [0, 126, 127, 253])
def test_log_of_every_mantissa(runtime, exponent):
    # Subnormals, [1/2, 1), [1, 2) and the last binade but one.
    x = (np.arange(1 << 23, dtype=np.uint32) | np.uint32(exponent << 23)).view(np.float32)
    _same(_device(runtime, 5, x), oracle.math32(5, x))


@pytest.mark.parametrize("fn", [0, 1, 3, 4, 5])
def test_special_arguments(runtime, fn):
    tiny, big = np.float32(1e-45), np.finfo(np.float32).max
    x = np.array([0.0, tiny, 1e-38, 0.5, np.nextafter(np.float32(0.5), np.float32(1)), 1.0, 89.0, 89.1, 104.0, 104.1,
                  2.0**20, 2.0**20 + 1, 1e30, big, np.inf, np.nan], dtype=np.float32)
    x = np.concatenate([x, -x])
    _same(_device(runtime, fn, x), oracle.math32(fn, x))


def test_special_arguments_of_atan2(runtime):
    v = np.array([0.0, 1e-45, 1e-38, 0.41421356, 0.41421357, 1.0, 2.0, 1e38, 3e38, np.inf, np.nan], dtype=np.float32)
    v = np.concatenate([v, -v])
    y, x = (a.ravel() for a in np.meshgrid(v, v))
    _same(_device(runtime, 2, y, x), oracle.math32(2, y, x))


def test_softplus_over_its_range(runtime):
    # log(1 + exp(100 v)) / 100 as the models form it, below and above the
    # bound where it is left out, and where the exponential no longer counts.
    v = np.linspace(-1.2, 1.1, 400_001).astype(np.float32)
    v = np.concatenate([v, np.array([-1e30, -np.inf, 1e30, np.inf, np.nan, 0.0, -0.0, 1.0634723, 1.0634724], np.float32)])
    params = np.zeros((len(v), 1), dtype=np.float32)
    params[:, 0] = v
    o = np.tile(np.array([0.0, 0.6, 0.8], np.float32), (len(v), 1))
    got = np.empty((len(v), 3), np.float32)
    _native.check(_native.lib().tgk_evaluate(runtime.handle, 0, 1, _native.ptr(params), _native.ptr(o), len(v),
                                             _native.ptr(got)))
    ref = oracle.evaluate(0, 1, params, o)
    _same(got[:, 0], np.ascontiguousarray(ref[:, 0]))
