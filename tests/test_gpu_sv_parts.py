"""backprojection_sv with its images split into parts (few views): part edges against the FP64 oracle at
the bars of test_gpu_sv.py (fp32 1e-5, fp64 1e-7 relative L2), view by view."""
import numpy as np
import pytest
import torch

import ctlib_amd
from ctlib_amd import phantom
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,tol", [(np.float32, 1e-5), (np.float64, 1e-7)])
@pytest.mark.parametrize("size", [(70, 31), (33, 63), (65, 64), (64, 95), (40, 200), (130, 513)], ids=str)
def test_parts(dev, size, dtype, tol):
    width, height = size
    side = max(size)
    o = phantom.fan_options(12, 90, width, height, 3.38 / side, 5.3 / 90, 5.95, 4.906, 0, Ang0=0.1, binshift=0.01)
    y = np.random.default_rng(width).random((2, 1, 12, 90)).astype(dtype)
    print(f"[case] sv {size} {dtype.__name__}", flush=True)
    got = ctlib_amd.backprojection_sv(torch.from_numpy(y).to(dev), torch.from_numpy(o)).cpu().numpy()
    ref = O.apply("backprojection_sv", o.astype(np.float64), y[:, 0].astype(np.float64))
    for b in range(2):
        for v in range(12):
            err = np.linalg.norm(got[b, v] - ref[b, v]) / np.linalg.norm(ref[b, v])
            assert err <= tol, (b, v, err)
