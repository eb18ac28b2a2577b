"""backprojection_t (weighted line -> bin) at the edges of its launch shapes, against the FP64 oracle.

fp64 batches of pairs share one slice's weights and addresses (lines up to 512 pixels, up to 895 bins);
lines fill a wave's 4, 8 or 16 pixels per lane or end within them; bins end on either side of a slot of
64.  Bars of the parity tests (fp32 1e-5, fp64 1e-7 relative L2), slice by slice on slices of very
different size.
"""
import numpy as np
import pytest
import torch

import ctlib_amd
from ctlib_amd import phantom
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TOL = {np.float32: 1e-5, np.float64: 1e-7}
SIZES = [(5, 9, 7), (64, 33, 64), (256, 256, 255), (257, 255, 300), (512, 512, 895), (512, 300, 896), (513, 512, 512),
         (1024, 1024, 700)]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("batch", [1, 2, 3, 9])
@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_launch_shapes(dev, size, batch, dtype):
    width, height, dets = size
    batch = min(batch, 4) if width > 600 else batch
    st = (SIZES.index(size) + batch) % 3
    views = 10 if width < 600 else 6
    side = max(width, height)
    if st == 2:
        o = phantom.para_options(views, dets, width, height, 1.0 / side, 1.45 / dets, Ang0=0.1, binshift=0.3 / dets)
    else:
        o = phantom.fan_options(views, dets, width, height, 3.38 / side, (5.3 if st == 0 else 0.98) / dets, 5.95, 4.906,
                                st, Ang0=0.1, binshift=0.002)
    rng = np.random.default_rng(width + batch)
    x = rng.random((batch, 1, height, width)).astype(dtype)
    x *= (10.0 ** np.arange(batch))[:, None, None, None].astype(dtype)
    for op in ("backprojection_t", "backprojection_t_true"):
        print(f"[case] {op} st={st} {size} batch={batch} {dtype.__name__}", flush=True)
        got = getattr(ctlib_amd, op)(torch.from_numpy(x).to(dev), torch.from_numpy(o)).cpu().numpy()[:, 0]
        ref = O.apply(op, o.astype(np.float64), x[:, 0].astype(np.float64))
        for b in range(batch):
            err = np.linalg.norm(got[b] - ref[b]) / np.linalg.norm(ref[b])
            assert err <= TOL[dtype], (op, st, b, err)
