"""Float32 3 x 3 eigenvalues (the angle from a float estimate, corrected in double)
against numpy in float64, over magnitudes from denormal cubes to 1e15 and the
cases where two or three eigenvalues meet; and the float32 vesselness's
1 - e^x at exponents from 1e-16 to 200 and infinity.

The result is rounded to float32 once (2^-24 of itself); the closed form in
double adds 1e-16 of the largest eigenvalue, and sqrt(2^-52) = 1.5e-8 of it
where two eigenvalues meet (the sine of the angle is the root of a rounded
difference): 2^-23 of the largest eigenvalue bounds both."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _matrices(kind, n, rng):
    if kind == "random":
        m = rng.standard_normal((n, 3, 3))
    elif kind == "rank1":
        v = rng.standard_normal((n, 3))
        m = v[:, :, None] * v[:, None, :]
    elif kind == "pair":  # two equal eigenvalues, rotated
        q = np.linalg.qr(rng.standard_normal((n, 3, 3)))[0]
        d = np.stack([np.ones(n), np.ones(n), rng.uniform(-2, 2, n)], 1)
        m = q @ (d[:, :, None] * q.transpose(0, 2, 1))
    elif kind == "diagonal":
        m = np.stack([np.diag(v) for v in rng.integers(-2, 3, (n, 3)).astype(float)])
    else:  # traceless: eigenvalues of opposite sign
        m = rng.standard_normal((n, 3, 3))
        m -= np.eye(3) * np.trace(m, axis1=1, axis2=2)[:, None, None] / 3
    return m + m.transpose(0, 2, 1)


@pytest.mark.parametrize("scale", [1e-30, 1e-12, 1.0, 1e6, 1e15])
@pytest.mark.parametrize("kind", ["random", "rank1", "pair", "diagonal", "traceless"])
def test_eigenvalues_against_double(gpu, kind, scale):
    from cucim_amd.skimage.feature import hessian_matrix_eigvals

    rng = np.random.default_rng(3)
    m = (_matrices(kind, 999, rng) * scale).astype(np.float32)
    el = [torch.from_numpy(np.ascontiguousarray(m[:, i, j])).cuda().view(3, 3, 111)
          for i, j in ((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))]
    got = hessian_matrix_eigvals(el)
    got = torch.stack(list(got)).cpu().numpy().reshape(3, -1).astype(np.float64)
    exp = np.linalg.eigvalsh(m.astype(np.float64))[:, ::-1].T
    top = np.abs(exp).max(0)
    assert (np.abs(got - exp) <= 2.0 ** -23 * top + 1e-44).all()


def _eigenvalues(m, dtype):
    """The closed form of symmetric float32 matrices in `dtype`, descending
    and rounded to float32."""
    a, d, f, b, e, c = (m[:, i, j].astype(dtype)
                        for i, j in ((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2)))
    ta, tb, tc = 2 * a - b - c, 2 * b - a - c, 2 * c - a - b
    x2 = -ta * tb * tc + 9 * (tc * (d * d) + tb * (f * f) + ta * (e * e)) - 54 * (d * e * f)
    x1 = a * a + b * b + c * c - a * b - a * c - b * c + 3 * (d * d + e * e + f * f)
    th = np.arctan2(np.sqrt(np.maximum(4 * x1 * x1 * x1 - x2 * x2, 0)), x2) / 3
    t, mid, third = 2 * np.sqrt(x1) / 3, (a + b + c) / 3, np.arccos(dtype(-1)) / 3
    lam = np.stack([mid - t * np.cos(th), mid + t * np.cos(third - th),
                    mid + t * np.cos(third + th)])
    return np.sort(lam, axis=0)[::-1].astype(np.float32)


def test_eigenvalues_of_equal_pairs_round_as_in_double(gpu):
    """Where two eigenvalues meet, an error of the angle's sine, the root of a
    rounded difference, moves some results to the next float: as many of them
    as the closed form in double does (a tenth more for the order of its
    roundings), against 80 bits.  A sine from the rounded cosine moves half as
    many again."""
    from cucim_amd.skimage.feature import hessian_matrix_eigvals

    if np.finfo(np.longdouble).nmant < 63:
        pytest.skip("needs 80-bit long double")
    m = _matrices("pair", 60000, np.random.default_rng(8)).astype(np.float32)
    el = [torch.from_numpy(np.ascontiguousarray(m[:, i, j])).cuda().view(30, 40, 50)
          for i, j in ((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))]
    got = torch.stack(list(hessian_matrix_eigvals(el))).cpu().numpy().reshape(3, -1)
    exact = _eigenvalues(m, np.longdouble)
    moved = np.count_nonzero(_eigenvalues(m, np.float64) != exact)
    assert 0 < np.count_nonzero(got != exact) <= 1.1 * moved


def test_eigenvalues_of_zero_and_nan(gpu):
    from cucim_amd.skimage.feature import hessian_matrix_eigvals

    el = [torch.zeros((2, 2, 2), device="cuda") for _ in range(6)]
    assert all(bool((v == 0).all()) for v in hessian_matrix_eigvals(el))
    el[1][0, 0, 0] = float("nan")
    for v in hessian_matrix_eigvals(el):
        assert bool(v[0, 0, 0].isnan()) and int(v.isnan().sum()) == 1


def _closed_form(a, b, c, d, e, f):
    """The closed form in float64 of [[a, d, f], [d, b, e], [f, e, c]], its
    results in float32 after the descending compare-swaps."""
    with np.errstate(all="ignore"):
        a, b, c, d, e, f = (np.float64(v) for v in (a, b, c, d, e, f))
        ta, tb, tc = 2 * a - b - c, 2 * b - a - c, 2 * c - a - b
        x2 = -ta * tb * tc + 9 * (tc * (d * d) + tb * (f * f) + ta * (e * e)) - 54 * (d * e * f)
        x1 = (a * a + b * b + c * c - a * b - a * c - b * c
              + 3 * (d * d + e * e + f * f))
        x1 = np.fmax(x1, 0.0)
        if x2 == 0:
            phi = np.pi / 2
        else:
            phi = np.arctan(np.sqrt(np.fmax(4 * x1 ** 3 - x2 * x2, 0.0)) / x2)
            if x2 < 0:
                phi += np.pi
        m, t = (a + b + c) / 3, 2 / 3 * np.sqrt(x1)
        l1 = np.float32(m - t * np.cos(phi / 3))
        l2 = np.float32(m + t * np.cos((phi - np.pi) / 3))
        l3 = np.float32(m + t * np.cos((phi + np.pi) / 3))
        v1, v2, v3 = l3, l2, l1
        if v1 > v2:
            v1, v2 = v2, v1
        if v1 > v3:
            v1, v3 = v3, v1
        if v2 > v3:
            v2, v3 = v3, v2
        return v3, v2, v1


def test_eigenvalues_with_infinite_elements(gpu):
    """One element infinite, of either sign, in any place: what the closed
    form with a double arctangent gives, infinities and NaN alike."""
    from cucim_amd.skimage.feature import hessian_matrix_eigvals

    cases = []
    for base in ((1, 2, 3, 0.5, -0.1, 0.1), (0, 0, 0, 0, 0, 0), (1, 2, 3, 0, 0, 0),
                 (-1, 4, -2, 0.3, 0, 0.7)):
        for k in range(6):
            for v in (float("inf"), -float("inf")):
                m = list(base)
                m[k] = v
                cases.append(m)
    m = np.array(cases, np.float32)
    assert m.shape == (48, 6)
    el = [torch.from_numpy(np.ascontiguousarray(m[:, i])).cuda().view(2, 4, 6)
          for i in (0, 3, 5, 1, 4, 2)]  # 00 01 02 11 12 22
    got = torch.stack(list(hessian_matrix_eigvals(el))).cpu().numpy().reshape(3, -1).T
    exp = np.array([_closed_form(*r) for r in m], np.float32)
    exp.sort(axis=1)
    got = np.sort(got, axis=1)
    np.testing.assert_array_equal(got, exp)
    assert np.isinf(exp).any() and np.isnan(exp).any()


def _gamma_factor(shape):
    """An image whose midrange is 0 (nothing is subtracted before its Hessian),
    its r_g, computed as the kernels do, and where the voxel's eigenvalues are
    such that with alpha -> 0 and beta -> infinity the vesselness is exactly
    its gamma factor 1 - e^(-r_g / 2 gamma^2)."""
    from cucim_amd.skimage.feature import hessian_matrix, hessian_matrix_eigvals

    x = np.random.default_rng(0).uniform(-0.9, 0.9, shape).astype(np.float32)
    x.flat[0], x.flat[1] = -1, 1
    xd = torch.from_numpy(x).cuda()
    H = hessian_matrix(xd, sigma=1.5, mode="reflect", use_gaussian_derivatives=True)
    l = torch.stack(list(hessian_matrix_eigvals(H))).cpu().numpy().reshape(len(shape), -1)
    s = np.take_along_axis(l, np.argsort(np.abs(l), axis=0, kind="stable"), 0)
    a = np.abs(s)
    ok = (s[1:] > 1e-4).all(0) & (a[0] > 1e-6) & (a[1:] > 1.001 * a[:-1]).all(0)
    rg = s[0] * s[0]
    for v in s[1:]:  # fma
        rg = (v.astype(np.longdouble) ** 2 + rg.astype(np.longdouble)).astype(np.float32)
    assert np.count_nonzero(ok) > 10000
    return xd, rg, ok


def _ulps(got, exact):
    return np.abs(got - exact) / np.spacing(exact.astype(np.float32)).astype(np.float64)


@pytest.mark.parametrize("shape", [(48, 50, 52), (300, 310)])
def test_vesselness_one_minus_exp(gpu, shape):
    """expm1 in float: 0.89 ulp at most over all its arguments (measured), so
    1 here."""
    from cucim_amd.skimage.filters import frangi

    x, rg, ok = _gamma_factor(shape)
    top = float(np.sqrt(rg[ok].max()))
    for g in (1e6 * top, 1e3 * top, 10 * top, top, top / 2, top / 4, top / 20):
        out = frangi(x, sigmas=[1.5], alpha=1e-6, beta=1e6, gamma=g, black_ridges=True,
                     mode="reflect").cpu().numpy().reshape(-1)[ok]
        e = rg[ok] * np.float32(-1.0 / (2.0 * g * g))
        assert _ulps(out, -np.expm1(e.astype(np.float64))).max() <= 1.0
    kw = dict(sigmas=[1.5], alpha=1e-6, beta=1e6, gamma=1e-30, black_ridges=True)
    out = frangi(x, **kw).cpu().numpy().reshape(-1)
    assert (out[ok] == 1).all()  # exponents of -inf
    x[(shape[0] // 2,) * len(shape)] = float("nan")
    assert np.isnan(frangi(x, **kw).cpu().numpy()).any()


@pytest.mark.parametrize("shape", [(48, 50, 52), (300, 310)])
def test_first_sigma_in_double(gpu, shape):
    """The first sigma's vesselness, once gamma is known from its maximum, is
    computed in double and rounded once: half an ulp (and 2^-52 over the
    exponent, which is above 1e-6 where it is looked at)."""
    from cucim_amd.skimage.filters import frangi

    x, rg, ok = _gamma_factor(shape)
    out = frangi(x, sigmas=[1.5], alpha=1e-6, beta=1e6, gamma=None, black_ridges=True,
                 mode="reflect").cpu().numpy().reshape(-1)
    gsq = 2 * (np.sqrt(np.float64(rg.max())) / 2) ** 2
    e = -rg.astype(np.float64) / gsq
    ok &= e < -1e-6
    assert _ulps(out[ok], -np.expm1(e[ok])).max() <= 0.501
