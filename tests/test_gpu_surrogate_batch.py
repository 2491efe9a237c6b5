"""The matrix-core weight and input gradients over batches of patches against
float64 autograd, and a training step over stacked patches against the same
step patch by patch.

A float32 sum of n products differs from the exact one by at most
n 2^-24 sum |products| (one rounding of half an ulp per addition, the products
of the matrix core being exact or rounded once), which bounds every element
here; the 512 partial sums add at most 512 more roundings."""

import numpy as np
import pytest
import torch
import torch.nn.functional as Fnn

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


def _conv(x, w, b=None):
    """x: (B, D, H, W, ci), w: (27, ci, co), float64."""
    ci, co = w.shape[1:]
    k = w.view(3, 3, 3, ci, co).permute(4, 3, 0, 1, 2)
    return Fnn.conv3d(x.permute(0, 4, 1, 2, 3), k, b).permute(0, 2, 3, 4, 1)


def _grads(x, w, dy):
    x, w = x.clone().requires_grad_(True), w.clone().requires_grad_(True)
    b = torch.zeros(w.shape[2], dtype=torch.float64, requires_grad=True)
    _conv(x, w, b).backward(dy)
    return x.grad, w.grad, b.grad


@pytest.mark.parametrize("ci,co,act", [(24, 24, 1), (1, 24, 1), (24, 1, 0), (24, 1, 2)])
@pytest.mark.parametrize("shape", [(2, 3, 3, 3), (3, 5, 11, 19), (3, 29, 59, 117)])
def test_batched_forward(gpu, ci, co, act, shape):
    """Batches through both block heights (the last shape has enough blocks
    for eight planes), one element past 16-byte alignment on the output."""
    from cucim_amd import _array
    from cucim_amd import _lib as L

    lib, st = L.lib(), _array.stream()
    g = torch.Generator().manual_seed(7)
    x = torch.randn(shape + (ci,), generator=g).to(torch.bfloat16)
    w = torch.randn((27, ci, co), generator=g) / (27 * ci) ** 0.5
    b = torch.randn(co, generator=g) * 0.1
    wq = w.to(torch.bfloat16).double()
    ref = _conv(x.double(), wq, b.double())
    mag = _conv(x.double().abs(), wq.abs(), b.double().abs())
    out_t = torch.bfloat16 if co == 24 else torch.float32
    out = torch.empty(ref.numel() + 1, dtype=out_t, device="cuda")[1:].view(ref.shape)
    pre = torch.empty(ref.numel() + 1, device="cuda")[1:].view(ref.shape)
    wd, bd, xd = w.cuda(), b.cuda(), x.cuda()
    packed = torch.empty(lib.hc_cnn3d_packed_size(ci, co), dtype=torch.uint8, device="cuda")
    L.check(lib.hc_cnn3d_pack(wd.data_ptr(), packed.data_ptr(), ci, co, st))
    L.check(lib.hc_cnn3d_conv(_array.hc_array(xd), _array.hc_array(out), packed.data_ptr(),
                              bd.data_ptr(), act, pre.data_ptr(), st))
    p = pre.double().cpu()
    # the products of bfloat16 values are exact in float32
    assert bool(((p - ref).abs() <= (27 * ci + 1) * EPS * mag).all())
    if act == 1:
        # the hardware exp and reciprocal (1e-6 relative), then one bf16 rounding
        exp = Fnn.gelu(p, approximate="tanh")
        assert bool(((out.double().cpu() - exp).abs() <= 2.0 ** -8 * exp.abs() + 1e-5).all())
    else:
        assert torch.equal(out.cpu(), (pre.clamp(0, 1) if act == 2 else pre).cpu())


@pytest.mark.parametrize("ci,co,act", [(24, 24, 1), (1, 24, 1), (24, 1, 0)])
@pytest.mark.parametrize("shape", [(1, 5, 11, 19), (3, 29, 59, 117)])
def test_bias_is_added_to_the_finished_sum(gpu, ci, co, act, shape):
    """Products 1 and -1 of the first and the last tap cancel exactly, so a
    bias of 2^-30 comes back whole; added before the products, 1 + 2^-30
    would round it away."""
    from cucim_amd import _array
    from cucim_amd import _lib as L

    lib, st = L.lib(), _array.stream()
    x = torch.ones(shape + (ci,), dtype=torch.bfloat16, device="cuda")
    w = torch.zeros((27, ci, co), device="cuda")
    w[0, 0], w[26, ci - 1] = 1, -1
    b = 2.0 ** -30 * torch.arange(1, co + 1, device="cuda")
    oshape = (shape[0],) + tuple(s - 2 for s in shape[1:]) + (co,)
    out = torch.empty(oshape, dtype=torch.bfloat16 if co == 24 else torch.float32, device="cuda")
    pre = torch.empty(oshape, device="cuda")
    packed = torch.empty(lib.hc_cnn3d_packed_size(ci, co), dtype=torch.uint8, device="cuda")
    L.check(lib.hc_cnn3d_pack(w.data_ptr(), packed.data_ptr(), ci, co, st))
    L.check(lib.hc_cnn3d_conv(_array.hc_array(x), _array.hc_array(out), packed.data_ptr(),
                              b.data_ptr(), act, pre.data_ptr(), st))
    assert torch.equal(pre, b.expand(oshape))


@pytest.mark.parametrize("ci,co", [(24, 24), (1, 24), (24, 1)])
@pytest.mark.parametrize("shape", [(1, 3, 3, 3), (2, 4, 10, 18), (3, 5, 11, 19), (1, 20, 3, 35),
                                   (2, 13, 27, 9)])
def test_batched_gradients(gpu, ci, co, shape):
    from cucim_amd import _array
    from cucim_amd import _lib as L

    lib, st = L.lib(), _array.stream()
    g = torch.Generator().manual_seed(sum(shape) * 31 + ci)
    B, D, H, W = shape
    x = torch.randn(shape + (ci,), generator=g).to(torch.bfloat16)
    w = torch.randn((27, ci, co), generator=g) / 25
    dy = torch.randn((B, D - 2, H - 2, W - 2, co), generator=g)
    ref = _grads(x.double(), w.double(), dy.double())
    mag = _grads(x.double().abs(), w.double().abs(), dy.double().abs())
    xd, wd, dyd = x.cuda(), w.cuda(), dy.cuda()
    n = lib.hc_cnn3d_wgrad_work(ci, co)
    work = torch.full((n,), float("nan"), device="cuda")
    dw, db = torch.ones((27, ci, co), device="cuda"), torch.ones(co, device="cuda")
    L.check(lib.hc_cnn3d_wgrad_batch(xd.data_ptr(), dyd.data_ptr(), dw.data_ptr(), db.data_ptr(),
                                     B, D, H, W, ci, co, work.data_ptr(), n, st))
    terms = B * (D - 2) * (H - 2) * (W - 2) + 512 + 1
    for got, r, m in ((dw, ref[1], mag[1]), (db, ref[2], mag[2])):
        err = (got.double().cpu() - 1 - r).abs()  # both accumulate (here: onto ones)
        assert bool((err <= terms * EPS * (m + 1)).all())
    if ci == 1:
        rc = lib.hc_cnn3d_dgrad_batch(dyd.data_ptr(), wd.data_ptr(), None, xd.data_ptr(), B, D, H,
                                      W, ci, co, st)
        assert rc == L.ERR_UNSUPPORTED
        return
    pre = torch.randn(shape + (ci,), generator=g)
    for p in (None, pre):
        dx = torch.full(shape + (ci,), float("nan"), device="cuda")
        pd = None if p is None else p.cuda()
        L.check(lib.hc_cnn3d_dgrad_batch(dyd.data_ptr(), wd.data_ptr(),
                                         None if p is None else pd.data_ptr(), dx.data_ptr(), B,
                                         D, H, W, ci, co, st))
        r, m = ref[0], mag[0]
        slack = 0.0
        if p is not None:
            q = p.double().requires_grad_(True)
            Fnn.gelu(q, approximate="tanh").sum().backward()
            # the derivative through the hardware exp and reciprocal: 1e-5
            # absolute, as the elementwise kernel's test allows
            slack = 1e-5 * m
            r, m = r * q.grad, m * q.grad.abs()
        err = (dx.double().cpu() - r).abs()
        assert bool((err <= (27 * co + 2) * EPS * m + slack).all())


@pytest.mark.parametrize("ci,co", [(24, 24), (1, 24), (24, 1)])
@pytest.mark.parametrize("shape", [(1, 3, 3, 3), (2, 4, 10, 18), (2, 5, 11, 21), (1, 20, 3, 35)])
def test_gradients_of_infinite_values_hold_their_own_terms(gpu, ci, co, shape):
    """An infinite activation, gradient or weight makes those sums infinite or
    NaN that contain it, and no others (the blocks are padded with zeros).
    The reference adds the same terms in float64, tap by tap."""
    from cucim_amd import _array
    from cucim_amd import _lib as L

    lib, st = L.lib(), _array.stream()
    B, D, H, W = shape
    OD, OH, OW = D - 2, H - 2, W - 2
    g = torch.Generator().manual_seed(11)
    x0 = torch.randn(shape + (ci,), generator=g).to(torch.bfloat16)
    w0 = torch.randn((27, ci, co), generator=g) / 25
    dy0 = torch.randn((B, OD, OH, OW, co), generator=g)

    def reference(x, w, dy):
        dw, dx = torch.zeros_like(w), torch.zeros_like(x)
        f = dy.reshape(-1, co)
        for t in range(27):
            cut = (slice(None), slice(t // 9, t // 9 + OD), slice(t // 3 % 3, t // 3 % 3 + OH),
                   slice(t % 3, t % 3 + OW))
            dw[t] = (x[cut].reshape(-1, ci)[:, :, None] * f[:, None, :]).sum(0)
            dx[cut] += (dy[..., None, :] * w[t]).sum(-1)
        return dw, f.sum(0), dx

    mag = reference(x0.double().abs(), w0.double().abs(), dy0.double().abs())
    work = torch.empty(lib.hc_cnn3d_wgrad_work(ci, co), device="cuda")
    for where in ("x last", "x first", "dy", "w"):
        x, w, dy = x0.clone(), w0.clone(), dy0.clone()
        if where == "x last":
            x[-1, -1, -1, -1, 0] = float("inf")
        elif where == "x first":
            x[0, 0, 0, 0, ci - 1] = float("nan")
        elif where == "dy":
            dy[0, OD - 1, OH // 2, OW - 1, co - 1] = -float("inf")
        else:
            w[13, ci - 1, 0] = float("inf")
        dw_r, db_r, dx_r = reference(x.double(), w.double(), dy.double())
        xd, wd, dyd = x.cuda(), w.cuda(), dy.cuda()
        dw, db = torch.zeros((27, ci, co), device="cuda"), torch.zeros(co, device="cuda")
        L.check(lib.hc_cnn3d_wgrad_batch(xd.data_ptr(), dyd.data_ptr(), dw.data_ptr(),
                                         db.data_ptr(), B, D, H, W, ci, co, work.data_ptr(),
                                         work.numel(), st))
        terms = B * OD * OH * OW + 512
        res = [(dw, dw_r, mag[0], terms), (db, db_r, mag[1], terms)]
        if ci > 1:
            dx = torch.empty(shape + (ci,), device="cuda")
            L.check(lib.hc_cnn3d_dgrad_batch(dyd.data_ptr(), wd.data_ptr(), None, dx.data_ptr(),
                                             B, D, H, W, ci, co, st))
            res.append((dx, dx_r, mag[2], 27 * co + 2))
        for got, ref, m, n in res:
            got = got.double().cpu()
            fin = ref.isfinite()
            assert torch.equal(got[~fin].nan_to_num(7.0), ref[~fin].nan_to_num(7.0)), where
            assert bool(((got[fin] - ref[fin]).abs() <= n * EPS * m[fin]).all()), where


def test_wgrad_work_is_checked(gpu):
    from cucim_amd import _array
    from cucim_amd import _lib as L

    lib = L.lib()
    x = torch.zeros((1, 3, 3, 3, 24), dtype=torch.bfloat16, device="cuda")
    f = torch.zeros(27 * 24 * 24 + 24, device="cuda")
    n = lib.hc_cnn3d_wgrad_work(24, 24)
    assert lib.hc_cnn3d_wgrad_work(24, 8) < 0
    for elems, ptr in ((n - 1, f.data_ptr()), (n, f.data_ptr() + 4)):
        rc = lib.hc_cnn3d_wgrad_batch(x.data_ptr(), f.data_ptr(), f.data_ptr(), f.data_ptr(), 1, 3,
                                      3, 3, 24, 24, ptr, elems, _array.stream())
        assert rc == L.ERR_VALUE


def test_step_batches_like_single_patches(gpu, monkeypatch):
    """Patches of two shapes in one step: stacked, or one by one."""
    from cucim_amd import surrogate as S

    g = torch.Generator().manual_seed(5)
    xs = [torch.rand((e, e, e + 1, 1), generator=g).to(torch.bfloat16).cuda()
          for e in (14, 14, 14, 12, 13)]
    ts = [torch.rand(tuple(s - 10 for s in x.shape[:3]), generator=g).cuda() for x in xs]
    got = []
    for most in (S._BATCH_VOXELS, 1):
        monkeypatch.setattr(S, "_BATCH_VOXELS", most)
        assert len(list(S._batches(xs, ts))) == (3 if most > 1 else 5)
        m = S.FrangiSurrogate(seed=3)
        loss = m.train_step(xs, ts)
        got.append((float(loss), [t.clone() for t in m._gw + m._gb]))
    assert abs(got[0][0] - got[1][0]) <= 1e-5 * got[1][0]
    for a, b in zip(got[0][1], got[1][1]):
        assert float((a - b).norm()) <= 1e-5 * float(b.norm())
    assert np.isfinite(got[0][0])


def _step(S, xs, ts):
    m = S.FrangiSurrogate(seed=3)
    loss = m.train_step(xs, ts)
    return float(loss), [t.clone() for t in m._gw + m._gb]


def test_targets_that_are_not_dense(gpu):
    """A crop of a larger label volume, alone and among patches of its shape,
    gives what its dense copy gives; so does a target with a channel axis."""
    from cucim_amd import surrogate as S

    g = torch.Generator().manual_seed(9)
    xs = [torch.rand((14, 13, 15, 1), generator=g).to(torch.bfloat16).cuda() for _ in range(3)]
    labels = [torch.rand((14, 13, 15), generator=g).cuda() for _ in range(3)]
    crops = [t[5:-5, 5:-5, 5:-5] for t in labels]
    assert not any(t.is_contiguous() for t in crops)
    for n in (1, 3):
        exp = _step(S, xs[:n], [t.contiguous() for t in crops[:n]])
        for ts in (crops, [t[..., None] for t in crops]):
            got = _step(S, xs[:n], ts[:n])
            # the loss is added by atomics, in any order
            assert abs(got[0] - exp[0]) <= 1e-6 * exp[0]
            assert all(torch.equal(a, b) for a, b in zip(got[1], exp[1]))


def test_targets_that_do_not_fit_are_refused(gpu):
    from cucim_amd import surrogate as S

    x = torch.zeros((13, 13, 13, 1), dtype=torch.bfloat16, device="cuda")
    t = torch.zeros((3, 3, 3), device="cuda")
    m = S.FrangiSurrogate(seed=3)
    before = [w.clone() for w in m.w]
    for bad in (t.double(), t.to(torch.bfloat16), t[:2], torch.zeros((4, 3, 3), device="cuda"),
                t.cpu()):
        for xs, ts in (([x], [bad]), ([x, x], [t, bad])):
            with pytest.raises(ValueError):
                m.train_step(xs, ts)
    assert all(torch.equal(a, b) for a, b in zip(before, m.w))
