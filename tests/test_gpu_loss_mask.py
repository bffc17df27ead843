"""Loss masks on the GPU (include/beamformer/formats.hpp:22-32: one validity
byte per [t][f] frame, 0 = lost; the reference defines but never applies
them).  A masked launch must equal, bit for bit, an unmasked launch on a
copy of the payload whose lost frames are zeroed (int4 zero contributes
exactly nothing, and every tile shape sums in the same order); an all-valid
mask must change nothing; the FP32 selectors refuse a mask.
"""
import numpy as np
import pytest

import oracle as O
from beamform_project_amd import _capi, api
from helpers import F

pytestmark = pytest.mark.gpu
K = api.Kernel


def run(kernel, x, w, dims, S, mask=None):
    W = api.integrated_time_count(dims.n_time, S) if S else dims.n_time
    dx, dw = api.DeviceArray.from_numpy(x), api.DeviceArray.from_numpy(w)
    out = api.DeviceArray.empty((W, F, dims.n_beams), np.float32)
    dm = api.DeviceArray.from_numpy(mask) if mask is not None else None
    if S and mask is not None:
        api.launch_packed_integrated_beamformer_masked(kernel, None, dx, dm, dw, out, dims, S)
    elif S:
        api.launch_packed_integrated_beamformer(kernel, None, dx, dw, out, dims, S)
    elif mask is not None:
        api.launch_packed_beamformer_masked(kernel, None, dx, dm, dw, out, dims)
    else:
        api.launch_packed_beamformer(kernel, None, dx, dw, out, dims)
    api.device_synchronize()
    return out.to_numpy()


@pytest.mark.parametrize("A,B,S,T,kernel", [
    (64, 40, 10, 437, K.SPLIT_F16),
    (32, 16, 0, 150, K.F16),
    (128, 24, 320, 700, K.SPLIT_F16),
    (256, 9, 12, 100, K.SPLIT_F16),
    (64, 128, 10, 320, K.AUTO),
    # windows side by side and one by one; stages of five tiles and of one
    (64, 20, 64, 256, K.SPLIT_F16), (64, 20, 64, 180, K.SPLIT_F16),
    (128, 40, 20, 250, K.SPLIT_F16), (128, 9, 100, 250, K.F16), (256, 60, 128, 300, K.SPLIT_F16),
    # one wave per block of 8 beams
    (256, 9, 64, 195, K.SPLIT_F16), (256, 9, 64, 195, K.F16),
    (256, 45, 320, 700, K.SPLIT_F16), (256, 48, 128, 128, K.F16),
])
def test_masked_equals_zeroed_payload(A, B, S, T, kernel):
    rng = np.random.default_rng(A * 1000 + B)
    x = O.make_noise(T, F, A, 5 + A).reshape(T, F, A)
    w = (rng.standard_normal((B, F, A, 2)) * 0.5).astype(np.float32)
    mask = (rng.random((T, F)) > 0.15).astype(np.uint8)
    mask[20:40] = 0          # a run of lost frames across all channels
    mask[:, 7] = 0           # a dead channel
    zeroed = x * mask[:, :, None]
    dims = api.Dimensions(T, F, A, B)
    got = run(kernel, x, w, dims, S, mask)
    want = run(kernel, zeroed, w, dims, S)
    assert np.array_equal(got, want)
    assert np.all(got[..., 7, :] == 0)
    # every frame valid: identical to the unmasked launch on the payload
    ones = np.ones((T, F), np.uint8)
    assert np.array_equal(run(kernel, x, w, dims, S, ones), run(kernel, x, w, dims, S))


def test_masks_need_an_mfma_kernel():
    T, A, B = 32, 64, 8
    x = np.zeros((T, F, A), np.uint8)
    w = np.zeros((B, F, A, 2), np.float32)
    with pytest.raises(_capi.InvalidArgument, match="MFMA kernels"):
        run(K.FP32, x, w, api.Dimensions(T, F, A, B), 0, np.ones((T, F), np.uint8))
    with pytest.raises(_capi.InvalidArgument, match="loss_mask"):
        api.launch_packed_beamformer_masked(K.SPLIT_F16, None, api.DeviceArray.from_numpy(x),
                                            None, api.DeviceArray.from_numpy(w),
                                            api.DeviceArray.empty((T, F, B), np.float32),
                                            api.Dimensions(T, F, A, B))
