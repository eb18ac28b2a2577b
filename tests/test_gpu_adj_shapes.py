"""projection_t and backprojection at the edges of the bin -> pixel kernel's launch shapes.

The kernel shares one lookup among 1, 2 or 4 slices (batch 1, 2, 3 and more; four only up to 1022
bins) and tiles a line in runs of 8 edges, slots of 32 and up to 16 waves; an edge count of a whole
number of tiles takes its last edge apart.  Each case is compared with the FP64 oracle at the bars
of the parity tests (fp32 1e-5, fp64 1e-7 relative L2), slice by slice, so that a slice that read
its neighbour's table would show.
"""
import math

import numpy as np
import pytest
import torch

import ctlib_amd
from ctlib_amd import abi, phantom
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TOL = {np.float32: 1e-5, np.float64: 1e-7}

# width, height, bins: one slot and less, tile edges and their neighbours, several waves per line, the
# largest lines; bins on both sides of the four-slice limit
SIZES = [(5, 9, 7), (32, 31, 40), (33, 64, 50), (127, 129, 150), (256, 256, 300), (257, 200, 300), (511, 512, 600),
         (512, 512, 1022), (512, 513, 1023), (640, 640, 700), (1024, 1000, 1100), (1024, 1024, 1022), (2048, 2047, 1500)]


def options(st, width, height, dets, views):
    side = max(width, height)
    if st == 2:
        return phantom.para_options(views, dets, width, height, 1.0 / side, 1.45 / dets, Ang0=0.1, binshift=0.3 / dets)
    return phantom.fan_options(views, dets, width, height, 3.38 / side, (5.3 if st == 0 else 0.98) / dets, 5.95, 4.906,
                               st, Ang0=0.1, binshift=0.002)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("batch", [1, 2, 3, 5])
@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_launch_shapes(dev, size, batch, dtype):
    width, height, dets = size
    st = (SIZES.index(size) + batch) % 3
    views = 12 if width < 600 else 6
    o = options(st, width, height, dets, views)
    rng = np.random.default_rng(width * 7 + batch)
    y = rng.random((batch, 1, views, dets)).astype(dtype)
    y *= (10.0 ** np.arange(batch))[:, None, None, None].astype(dtype)  # a neighbour's value would stand out
    ot = torch.from_numpy(o)
    for op in ("projection_t", "backprojection"):
        print(f"[case] {op} st={st} {size} batch={batch} {dtype.__name__}", flush=True)
        got = getattr(ctlib_amd, op)(torch.from_numpy(y).to(dev), ot).cpu().numpy()[:, 0]
        ref = O.apply(op, o.astype(np.float64), y[:, 0].astype(np.float64))
        for b in range(batch):
            err = np.linalg.norm(got[b] - ref[b]) / np.linalg.norm(ref[b])
            assert err <= TOL[dtype], (op, st, b, err)


def test_fan_ea_without_polynomial(dev):
    """A fan too wide for the polynomial arctangent (atanf), X-axis views only, four slices."""
    o = phantom.fan_options(16, 300, 128, 128, 0.01, 2.3 / 300, 1.0, 1.0, 1, Ang0=0.1, dAng=0.01)
    assert abi.plan_export(o, "ea_atan")[7] == 0
    y = np.random.default_rng(1).random((4, 1, 16, 300)).astype(np.float32)
    for op in ("projection_t", "backprojection"):
        print(f"[case] wide fan {op}", flush=True)
        got = getattr(ctlib_amd, op)(torch.from_numpy(y).to(dev), torch.from_numpy(o)).cpu().numpy()[:, 0]
        ref = O.apply(op, o.astype(np.float64), y[:, 0].astype(np.float64))
        assert np.linalg.norm(got - ref) / np.linalg.norm(ref) <= 1e-5
        assert math.isfinite(float(got.sum()))
