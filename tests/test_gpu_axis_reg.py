"""The line kernels of strided axes (the register kernel where its rule takes
the array, else the LDS kernel), the fused filter over stacks and the vector
conversions: bit for bit what the element-wise kernel and the separate passes
give, at tile edges, odd strides, unaligned arrays and with non-finite
values."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _view(shape, off, seed, special=False):
    """A float32 tensor that starts `off` elements into its storage."""
    g = torch.Generator().manual_seed(seed)
    n = int(np.prod(shape))
    t = torch.randn(n + off, generator=g)
    if special and n > 40:
        t[off + n // 2] = float("inf")
        t[off + n // 3] = float("nan")
    return t.cuda()[off:].view(shape)


@pytest.mark.parametrize("shape,axis", [((7, 32), 0), ((33, 257), 0), ((300, 513), 0),
                                        ((2, 40, 33), 1), ((5, 9, 70), 0), ((3, 640, 655), 1),
                                        ((1, 1, 40), 0), ((600, 4099), 0), ((1030, 1021), 0),
                                        ((2, 3, 17, 45), 2)])
@pytest.mark.parametrize("K,origin", [(1, 0), (3, 1), (4, 0), (8, -2), (13, 0), (18, 3), (33, 0)])
@pytest.mark.parametrize("mode", ["reflect", "mirror", "nearest", "wrap", "constant"])
def test_strided_axis_equals_gather(gpu, shape, axis, K, origin, mode):
    from cucim_amd.skimage._vendored import ndimage as ndi

    x = _view(shape, K % 2, K * 7 + axis, special=True)
    w = np.random.default_rng(K).standard_normal(K).astype(np.float32)
    if K > 4:
        w[1] = 0  # a zero tap is skipped, also on inf and NaN
    kw = dict(axis=axis, mode=mode, cval=1.5, origin=origin)
    a = ndi.correlate1d(x, w, **kw)
    b = ndi.correlate1d(x, w, algorithm="elementwise", **kw)
    assert torch.equal(a.view(torch.int32)[~b.isnan()], b.view(torch.int32)[~b.isnan()])
    assert torch.equal(a.isnan(), b.isnan())


# float32 arrays that the register kernel takes (an axis stride that is no whole
# number of 16-byte words, at least 32; 2^20 elements or more): both of its
# heights, ragged tiles and strips, lines shorter than the kernel, one line more
# than a strip holds, and the fewest lines for each kernel length
@pytest.mark.parametrize("shape,axis,K,origin", [
    ((33, 387, 1413), 0, 13, 0), ((33, 387, 1413), 1, 33, 5), ((201, 387, 413), 0, 7, -1),
    ((70, 257, 1031), 1, 25, 0), ((1025, 3, 517), 0, 17, 2), ((5, 700, 401), 0, 33, 0),
    ((2, 3, 180001), 0, 13, 0), ((2, 3, 180001), 1, 18, -3), ((1, 1, 1 << 20 | 1), 0, 5, 0),
    ((4099, 257), 0, 33, 0), ((32000, 33), 0, 13, 0), ((16200, 65), 0, 25, 0),
    ((8130, 129), 0, 33, -8), ((4, 8000, 33), 1, 4, 0)])
@pytest.mark.parametrize("mode", ["reflect", "mirror", "nearest", "wrap", "constant"])
def test_register_kernel_equals_gather(gpu, shape, axis, K, origin, mode):
    from cucim_amd.skimage._vendored import ndimage as ndi

    assert np.prod(shape) >= 1 << 20
    x = _view(shape, 0, K + axis, special=True)
    w = np.random.default_rng(K).standard_normal(K).astype(np.float32)
    kw = dict(axis=axis, mode=mode, cval=1.5, origin=origin)
    a = ndi.correlate1d(x, w, **kw)
    b = ndi.correlate1d(x, w, algorithm="elementwise", **kw)
    assert torch.equal(a.isnan(), b.isnan())
    assert torch.equal(a.view(torch.int32)[~b.isnan()], b.view(torch.int32)[~b.isnan()])


@pytest.mark.parametrize("shape", [(1, 5, 9), (3, 33, 240), (4, 17, 515), (2, 1, 300)])
@pytest.mark.parametrize("sigma", [0.6, 1.5, (1.0, 2.0, 4.0), (0, 1.5, 2.0)])
@pytest.mark.parametrize("mode", ["nearest", "reflect", "constant"])
def test_stack_gaussian_equals_passes(gpu, monkeypatch, shape, sigma, mode):
    from cucim_amd.skimage._vendored import _ndimage_filters as F

    x = _view(shape, 1, 5)
    a = F.gaussian_filter(x, sigma, mode=mode, cval=0.5)
    y = x.clone()
    F.gaussian_filter(y, sigma, mode=mode, cval=0.5, output=y)  # in place
    t = torch.empty(shape[::-1], device="cuda").permute(2, 1, 0)
    F.gaussian_filter(x.transpose(1, 2).contiguous().transpose(1, 2), sigma, mode=mode, cval=0.5,
                      output=t)
    monkeypatch.setattr(F, "FUSED_2D", False)
    b = F.gaussian_filter(x, sigma, mode=mode, cval=0.5)
    for got in (a, y, t):
        assert torch.equal(got, b)


# slices of the fused launch's two row counts (8 up to 2^22 elements, 16 above),
# whole and ragged tiles, kernels longer than a slice, and stacks that the rule
# leaves to the line kernels
_STACKS = [((20, 448, 512), 13, True), ((33, 386, 413), 33, True), ((600, 100, 225), 9, True),
           ((700, 24, 333), 25, True), ((3000, 40, 24), 5, True), ((4000, 32, 40), 33, True),
           ((4000, 5, 129), 25, True), ((300, 64, 512), (5, 33), True),
           ((4000, 4, 260), 13, False), ((1500, 7, 300), 33, False), ((200, 10, 400), 33, False),
           ((2000, 18, 300), 33, False), ((300, 27, 512), (5, 33), False)]


@pytest.mark.parametrize("shape,K,fused", _STACKS)
@pytest.mark.parametrize("mode", ["reflect", "mirror", "nearest", "wrap", "constant"])
def test_stack_rule(gpu, monkeypatch, shape, K, fused, mode):
    """The fused launch gives the separate passes' bits whether the rule takes
    it or not."""
    from cucim_amd import _array
    from cucim_amd import _lib as L
    from cucim_amd.skimage._vendored import _ndimage_filters as F

    x = _view(shape, 0, 3, special=True)
    rng = np.random.default_rng(1)
    K0, K1 = K if isinstance(K, tuple) else (K, K)
    w = [None] + [rng.standard_normal(k).astype(np.float32) for k in (K0, K1)]
    t = [F._get_taps(v, v.size // 2, np.float32) for v in w[1:]]
    out = torch.empty_like(x)
    m = F._util._mode_code(mode)
    rc = L.lib().hc_separable2d_slices(_array.hc_array(x), _array.hc_array(out), t[0].struct,
                                       t[1].struct, m, m, 0.5, _array.stream())
    assert rc == L.OK
    assert F._stack_pays(*shape, K0, K1, shape[2] % 4 == 0) == fused
    a = F._run_1d_correlates(x, (0, 1, 2), w, None, mode, 0.5)
    monkeypatch.setattr(F, "FUSED_2D", False)
    b = F._run_1d_correlates(x, (0, 1, 2), w, None, mode, 0.5)
    for got in (a, out):
        assert torch.equal(got.isnan(), b.isnan())
        assert torch.equal(got.view(torch.int32)[~b.isnan()], b.view(torch.int32)[~b.isnan()])


@pytest.mark.parametrize("n", [1, 7, 8, 9, 2047, 100003])
@pytest.mark.parametrize("off", [0, 1, 3])
def test_unsigned_to_float(gpu, n, off):
    from cucim_amd.skimage.util import img_as_float32

    rng = np.random.default_rng(n)
    for dt, top in ((np.uint8, 255), (np.uint16, 65535)):
        x = rng.integers(0, top + 1, n + off).astype(dt)
        got = img_as_float32(torch.from_numpy(x).cuda()[off:]).cpu().numpy()
        exp = x[off:].astype(np.float32) * np.float32(1.0 / top)
        np.testing.assert_array_equal(got, exp)
