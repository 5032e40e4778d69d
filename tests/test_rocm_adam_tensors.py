"""rlt_rocm_adam_step over tensors that follow each other in memory, which one pass takes together, and over the same tensors lying apart and off 16-byte boundaries: the
arithmetic of an element is the same, so every value is, bit for bit; and the squared gradient norm against 64-bit sums."""
import ctypes as C

import numpy as np
import pytest

import helpers
from helpers import capi

pytestmark = pytest.mark.gpu
COUNTS = {"ragged": [5, 1, 1023, 1024, 1025, 3, 256], "network": [17 * 256, 256, 256 * 256, 256, 6 * 256, 6], "many": [130] * 37, "one": [1], "sixteen workgroups": [16 * 1024], "seventeen": [16 * 1024 + 1], "large": [1_500_001, 7]}


def step(rocm, counts, apart, parameters, arrays):
    """Two steps; apart: a tensor starts `apart` floats behind the end of the one before."""
    starts, at = [], apart
    for n in counts:
        starts.append(at)
        at += n + apart
    device = []
    for a in arrays:
        spread, k = np.full(at, 7, np.float32), 0
        for s, n in zip(starts, counts):
            spread[s:s + n] = a[k:k + n]
            k += n
        device.append(rocm.array(spread))
    tensors = (capi.AdamTensor * len(counts))(*[capi.AdamTensor(*[d.offset(s) for d in device], n, 1 + i % 2) for i, (s, n) in enumerate(zip(starts, counts))])
    age, norm = rocm.array(np.array([3], np.uint32)), rocm.zeros((1,))
    for k in range(2):
        rocm.call("adam_step", tensors, len(counts), C.byref(parameters), age.ptr, 0.25, norm.ptr if k else None)
    rocm.sync()
    assert age.numpy()[0] == 5
    out = [d.numpy() for d in device]
    between = np.ones(at, bool)
    for s, n in zip(starts, counts):
        between[s:s + n] = False
    assert all(np.all(o[between] == 7) for o in out)
    return [np.concatenate([o[s:s + n] for s, n in zip(starts, counts)]) for o in out], float(norm.numpy()[0])


@pytest.mark.parametrize("decay", [False, True])
@pytest.mark.parametrize("counts", sorted(COUNTS))
def test_neighbouring_tensors_are_stepped_as_separate_ones(rocm, counts, decay):
    print("case", counts, decay, flush=True)
    counts = COUNTS[counts]
    rng = np.random.default_rng(sum(counts))
    arrays = [rng.standard_normal(sum(counts)).astype(np.float32) for _ in range(5)]
    arrays[3] = arrays[3] ** 2
    parameters = capi.adam_parameters()
    parameters.weight_decay, parameters.bias_lr_factor = 0.1, 0.5
    parameters.enable_weight_decay = parameters.enable_bias_lr_factor = int(decay)
    joined, norm = step(rocm, counts, 0, parameters, arrays)
    for apart in (1, 4):
        got, apart_norm = step(rocm, counts, apart, parameters, arrays)
        assert all(np.array_equal(a, b) for a, b in zip(joined, got)), apart
        assert abs(apart_norm - norm) <= 1e-5 * norm
    exact = float(np.sum(arrays[1].astype(np.float64) ** 2))
    assert abs(norm - exact) <= 1e-5 * exact       # positive summands: n * 2^-24 is the bound of a serial sum, a thread's share is a few of them
