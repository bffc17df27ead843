"""The float-weight selectors (FP32, DIRECT, TILED) on the matrix cores, and
windows of a multiple of 64 spectra on every kernel.

Every weight reaches the matrix unit as three bfloat16 slices that add up to
it, so only FP32 accumulation rounds: an output is a sum of squares of sums
of 2A exact products, each sum of relative error at most 2A 2^-24 of the sum
of magnitudes, far inside the 1e-5 floored bar of the split kernel.
"""
import numpy as np
import pytest

import oracle as O
from beamform_project_amd import api
from helpers import F, incoherent_floor, rel_err_floored
from test_gpu_fixed_grid import fp64_reference, random_case, run_gpu

pytestmark = pytest.mark.gpu

K = api.Kernel


def tiled_weights(w, A, B):
    tiles = -(-B // 32)
    p = np.zeros((tiles * 32, F, A, 2), np.float32)
    p[:B] = w.reshape(B, F, A, 2)
    return np.ascontiguousarray(p.reshape(tiles, 32, F, A, 2).transpose(2, 0, 3, 1, 4))


# T around tiles of 16, stages of 64 and windows; B around 8-beam columns and
# 32/64-beam groups; S of every window scheme (10; 12, 20, 100: four windows
# side by side; 64, 320: one window at a time; 7: the FMA kernel)
@pytest.mark.parametrize("T,A,B,S", [
    (161, 32, 33, 0), (79, 64, 65, 0), (95, 128, 9, 0), (65, 256, 17, 0),
    (171, 64, 16, 10), (130, 64, 8, 12), (203, 32, 40, 20), (401, 64, 31, 100),
    (63, 64, 24, 64), (129, 256, 8, 64), (641, 64, 128, 320), (319, 128, 33, 320),
    (2049, 64, 1, 320), (2063, 32, 3, 64), (70, 64, 32, 7), (40, 64, 3, 320),
])
def test_float_weights_vs_fp64(T, A, B, S):
    x, w = random_case(T, A, B, seed=T + A + B)
    ref = fp64_reference(x, w, T, A, B, S)
    floor = incoherent_floor(x, A, S or 1)
    dims = api.Dimensions(T, F, A, B)
    got = run_gpu(K.FP32, x, w, dims, S)
    assert rel_err_floored(got, ref, floor) <= 1e-5
    if S in (0, 320):
        assert np.array_equal(run_gpu(K.DIRECT, x, w, dims, S), got)
    if S in (0, 10, 320):
        assert np.array_equal(run_gpu(K.TILED, x, tiled_weights(w, A, B), dims, S), got)


@pytest.mark.parametrize("kernel,tol", [(K.SPLIT_F16, 1e-5), (K.F16, 2e-3)])
@pytest.mark.parametrize("T,A,B,S", [(1, 64, 9, 64), (64, 32, 40, 64), (65, 128, 12, 64),
                                     (1285, 64, 100, 320), (961, 256, 45, 320),
                                     (17, 256, 1, 64), (195, 256, 48, 64), (195, 256, 49, 64),
                                     (700, 256, 9, 128),
                                     # four windows side by side where that pads little, one
                                     # by one where it pads much, on both sides of the line
                                     (256, 64, 20, 64), (197, 32, 9, 64), (180, 32, 9, 64),
                                     (1010, 128, 17, 64), (468, 64, 120, 128),
                                     (430, 64, 120, 128), (515, 256, 50, 64)])
def test_long_windows_vs_fp64(kernel, tol, T, A, B, S):
    x, w = random_case(T, A, B, seed=3 * T + B)
    got = run_gpu(kernel, x, w, api.Dimensions(T, F, A, B), S)
    ref = fp64_reference(x, w, T, A, B, S)
    assert rel_err_floored(got, ref, incoherent_floor(x, A, S)) <= tol


@pytest.mark.parametrize("kernel,tol", [(K.SPLIT_F16, 1e-5), (K.F16, 2e-3)])
@pytest.mark.parametrize("T,A,B,S", [(163, 128, 32, 20), (163, 128, 33, 20), (410, 64, 12, 100),
                                     (301, 256, 9, 20), (4095, 256, 2, 20), (4097, 256, 2, 20),
                                     (4097, 256, 33, 100)])
def test_stage_lengths_vs_fp64(kernel, tol, T, A, B, S):
    """Windows of a multiple of 20 on both sides of the rule for their stages."""
    x, w = random_case(T, A, B, seed=5 * T + B)
    got = run_gpu(kernel, x, w, api.Dimensions(T, F, A, B), S)
    ref = fp64_reference(x, w, T, A, B, S)
    assert rel_err_floored(got, ref, incoherent_floor(x, A, S)) <= tol


def test_weights_outside_half_range():
    """Weights far outside fp16's range, and infinities and NaN, behave as
    float weights do."""
    T, A, B, S = 128, 64, 8, 0
    x, w = random_case(T, A, B, seed=5)
    w = w.reshape(B, F, A, 2).copy()
    scale = np.float32(2.0) ** np.array([0, 30, -30, 17, -17, 50, -50, 5], np.float32)
    w *= scale[:, None, None, None]
    got = run_gpu(K.FP32, x, w, api.Dimensions(T, F, A, B), S)
    ref = fp64_reference(x, w, T, A, B, S)
    floor = incoherent_floor(x, A) * scale.astype(np.float64) ** 2
    assert float(np.max(np.abs(got - ref) / np.maximum(np.abs(ref), floor))) <= 1e-5
    x[:, :, 7] = 0x11  # one antenna at 1 + 1j, which meets the odd weights
    w[1, :, 7] = np.inf
    w[2, :, 7, 0] = np.nan
    # a NaN whose payload sits in the low bits only
    w[3, :, 7, 0] = np.array([0x7F800001], np.uint32).view(np.float32)[0]
    got = run_gpu(K.FP32, x, w, api.Dimensions(T, F, A, B), S)
    assert not np.isfinite(got[:, :, 1]).any()
    assert np.isnan(got[:, :, 2]).all() and np.isnan(got[:, :, 3]).all()
    assert np.isfinite(got[:, :, [0, 4, 5, 6, 7]]).all()


@pytest.mark.parametrize("T,A,B,S", [(163, 64, 8, 10), (167, 64, 8, 12), (137, 64, 40, 20),
                                     (203, 32, 17, 100), (171, 128, 9, 64), (330, 256, 9, 320),
                                     (81, 256, 9, 16), (39, 64, 8, 10), (40, 64, 3, 7)])
def test_infinite_weight_in_a_short_last_window(T, A, B, S):
    """An infinite weight that every spectrum meets with a voltage of 1 + 1j
    gives an infinite power in every window, a last one cut short by T too;
    the other beams are as without it."""
    x, w = random_case(T, A, B, seed=T + B)
    w = w.reshape(B, F, A, 2).copy()
    x[:, :, 7] = 0x11
    dims = api.Dimensions(T, F, A, B)
    want = run_gpu(K.FP32, x, w, dims, S)
    w[1, :, 7] = (np.inf, 0.0)
    got = run_gpu(K.FP32, x, w, dims, S)
    assert np.isposinf(got[:, :, 1]).all()
    got[:, :, 1] = want[:, :, 1]
    assert np.array_equal(got, want)
