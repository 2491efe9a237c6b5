"""Connected components joined by runs, and equal-bin histograms: the sizes at
which runs cross 64-voxel boundaries, rows of one voxel, every connectivity in
1-D .. 4-D, and edges that are not equal bins.  Integers: exact."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1,), (64,), (200,), (5, 63), (7, 65), (130, 1), (3, 200),
                                   (4, 5, 67), (9, 1, 130), (2, 64, 64), (3, 4, 5, 33),
                                   (2, 2, 2, 2, 9)])
@pytest.mark.parametrize("density", [0.3, 0.6, 0.97, 1.0])
def test_label_every_connectivity(gpu, shape, density):
    from cucim_amd.skimage.measure import label
    from oracle import skimage as osk

    rng = np.random.default_rng(len(shape) * 100 + shape[-1])
    x = (rng.random(shape) < density) * rng.integers(1, 3, shape)
    for dt in (np.uint8, np.int32):
        xd = torch.from_numpy(x.astype(dt)).cuda()
        for conn in range(1, len(shape) + 1):
            got, num = label(xd, return_num=True, connectivity=conn)
            exp = osk.label(x, connectivity=conn)
            exp = exp[0] if isinstance(exp, tuple) else exp
            np.testing.assert_array_equal(got.cpu().numpy(), exp)
            assert num == exp.max()


@pytest.mark.parametrize("nbins", [1, 2, 7, 256, 1024, 1025, 4096, 5000])
@pytest.mark.parametrize("kind", ["uniform", "crowded", "wide", "edges"])
def test_histogram_bins(gpu, nbins, kind):
    from cucim_amd.skimage.exposure.exposure import _counts

    rng = np.random.default_rng(nbins)
    x = rng.random(20011).astype(np.float32)
    if kind == "crowded":
        x = (x ** 9).astype(np.float32)
    e = np.linspace(float(x.min()), float(x.max()), nbins + 1)
    if kind == "wide":  # bins of unequal width: the search
        e = np.sort(rng.random(nbins + 1)) ** 3
    if kind == "edges":  # values on the edges, and outside
        x = np.concatenate([e, e - 1e-9, e + 1e-9, [np.nan, -1, 2]])
    got = _counts(torch.from_numpy(x).cuda(), nbins, e).cpu().numpy()
    v = x.astype(np.float64)
    v = v[(v >= e[0]) & (v <= e[-1])]
    i = np.minimum(np.searchsorted(e, v, side="right") - 1, nbins - 1)
    np.testing.assert_array_equal(got, np.bincount(i, minlength=nbins))
