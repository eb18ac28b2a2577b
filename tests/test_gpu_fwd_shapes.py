"""projection and the residual step at the edges of the line -> bin kernel's launch shapes.

The kernel shares one lookup among 1, 2 or 4 slices (four with packed tables, where few of the last
group's slots stay empty), gives a wave up to 7 or 12 slots of 64 bin edges, splits a view's edges over
2 or 4 waves beyond that, and takes the last edge of a detector of whole slots apart; lines come in
classes of 256, 512, 1024 and 2048 pixels.  Unsplit launches (one line chunk) form the residual tables
and row sums in their epilogue.  Each case against the FP64 oracle at the bars of the parity tests (fp32
1e-5, fp64 1e-7 relative L2), slice by slice on slices of very different size.
"""
import numpy as np
import pytest
import torch

import ctlib_amd
from ctlib_amd import _C, phantom
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TOL = {np.float32: 1e-5, np.float64: 1e-7}

# width, height, bins
SIZES = [(5, 9, 7), (64, 64, 63), (64, 33, 64), (255, 256, 255), (256, 256, 447), (257, 256, 448), (256, 256, 449),
         (512, 512, 512), (512, 513, 767), (300, 512, 768), (512, 512, 769), (1024, 700, 895), (512, 512, 1024),
         (1024, 1024, 1536), (1025, 512, 1537), (2048, 1100, 2046)]


def options(st, width, height, dets, views):
    side = max(width, height)
    if st == 2:
        return phantom.para_options(views, dets, width, height, 1.0 / side, 1.45 / dets, Ang0=0.1, binshift=0.3 / dets)
    return phantom.fan_options(views, dets, width, height, 3.38 / side, (5.3 if st == 0 else 0.98) / dets, 5.95, 4.906,
                               st, Ang0=0.1, binshift=0.002)


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("batch", [1, 2, 3, 5, 9])
@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_launch_shapes(dev, size, batch, dtype):
    width, height, dets = size
    if batch == 9 and width > 600:
        batch = 4
    st = (SIZES.index(size) + batch) % 3
    views = 14 if width < 600 else 6
    o = options(st, width, height, dets, views)
    ot = torch.from_numpy(o)
    rng = np.random.default_rng(width * 7 + batch)
    scale = (10.0 ** np.arange(batch))[:, None, None, None].astype(dtype)  # a neighbour's value would stand out
    x = rng.random((batch, 1, height, width)).astype(dtype) * scale
    m = rng.random((batch, 1, views, dets)).astype(dtype) * scale
    xd, md = torch.from_numpy(x).to(dev), torch.from_numpy(m).to(dev)
    o64 = o.astype(np.float64)
    y = O.apply("projection", o64, x[:, 0].astype(np.float64))
    r = y - m[:, 0]
    g = O.apply("projection_t", o64, r)
    for chunks in (0, 1):
        print(f"[case] st={st} {size} batch={batch} {dtype.__name__} chunks={chunks}", flush=True)
        _C.set_plan_chunks(ot, dev.index or 0, chunks, chunks)
        try:
            got = ctlib_amd.projection(xd, ot).cpu().numpy()[:, 0]
            gy, gg = (t.cpu().numpy()[:, 0] for t in ctlib_amd.residual_step(xd, md, ot))
            rows, gl = _C.residual_loss_step(xd, md, ot)
        finally:
            _C.set_plan_chunks(ot, dev.index or 0, 0, 0)
        rows, gl = rows.cpu().numpy(), gl.cpu().numpy()[:, 0]
        for b in range(batch):
            assert rel(got[b], y[b]) <= TOL[dtype], (chunks, st, b, rel(got[b], y[b]))
            assert rel(gy[b], y[b]) <= TOL[dtype], (chunks, st, b)
            assert rel(gg[b], g[b]) <= TOL[dtype], (chunks, st, b, rel(gg[b], g[b]))
            assert rel(gl[b], g[b]) <= TOL[dtype], (chunks, st, b)
            assert rel(rows[b], (r[b] ** 2).sum(-1)) <= TOL[dtype], (chunks, st, b)
