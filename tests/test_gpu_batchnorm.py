"""GPU parity of spatial batch normalisation in training mode (hk_batch_norm_fwd / _bwd) against the oracle's
restatement of cuDNN's documented arithmetic: outputs, saved and running statistics, all three gradients."""
import numpy as np
import pytest

import helpers
import oracle

pytestmark = pytest.mark.gpu

SHAPES = [(8, 16, 14, 14), (2, 3, 5, 7), (32, 64, 8, 8), (1, 4, 1, 1), (4, 7, 33, 1), (64, 256, 4, 4), (3, 5, 9)]


@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16", "fp64"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_forward_and_backward(hk, cuda, dtype, shape):
    import torch
    g = helpers.rng(sum(shape))
    C = shape[1]
    pt = "fp64" if dtype == "fp64" else "fp32"             # parameters and statistics: fp32 for 16-bit data
    rnd = lambda a, d: a.astype(np.float64) if d == "fp64" else oracle.round_to(a.astype(np.float32), d)
    x = rnd(g.standard_normal(shape) * 2 + 3, dtype)       # a mean well away from zero
    scale = rnd(g.uniform(0.5, 1.5, C), pt); bias = rnd(g.standard_normal(C), pt)
    rm = rnd(g.standard_normal(C), pt); rv = rnd(g.uniform(0.5, 2.0, C), pt)
    dy = rnd(g.standard_normal(shape), dtype)
    momentum, eps = 0.1, 1e-5
    ey, erm, erv, emean, einv = oracle.batch_norm_fwd(x, scale, bias, rm, rv, momentum, eps)
    tx = helpers.to_torch(x, dtype, cuda); ts = helpers.to_torch(scale, pt, cuda); tb = helpers.to_torch(bias, pt, cuda)
    trm = helpers.to_torch(rm, pt, cuda); trv = helpers.to_torch(rv, pt, cuda)
    ty = torch.empty_like(tx); smean = torch.empty_like(ts); sinv = torch.empty_like(ts)
    hk.batch_norm_fwd(tx, ts, tb, ty, momentum, eps, trm, trv, smean, sinv)
    torch.cuda.synchronize()
    m = x.size // C
    helpers.assert_close(ty, ey, dtype, "y")
    helpers.assert_close(smean, emean, pt, "save_mean", scale=float(np.sqrt(np.mean(x.astype(np.float64) ** 2))))
    if m > 1:
        helpers.assert_close(sinv, einv, pt, "save_invstd", rtol=1e-4 if pt == "fp32" else None)
        helpers.assert_close(trv, erv, pt, "running_var", rtol=1e-4 if pt == "fp32" else None)
    helpers.assert_close(trm, erm, pt, "running_mean", scale=1.0)
    # backward from the statistics as saved
    sm = helpers.to_numpy(smean).astype(np.float64); si = helpers.to_numpy(sinv).astype(np.float64)
    edx, eds, edb = oracle.batch_norm_bwd(dy, x, scale, sm, si)
    tdy = helpers.to_torch(dy, dtype, cuda)
    dx = torch.empty_like(tx); ds = torch.empty_like(ts); db = torch.empty_like(ts)
    hk.batch_norm_bwd(tdy, tx, ts, dx, ds, db, smean, sinv)
    torch.cuda.synchronize()
    helpers.assert_close(dx, edx, dtype, "dx", rtol=2e-2 if dtype in ("bf16", "fp16") else (1e-4 if dtype == "fp32" else None))
    helpers.assert_close(ds, eds, pt, "dscale", rtol=1e-4 if pt == "fp32" else None)
    helpers.assert_close(db, edb, pt, "dbias", rtol=1e-4 if pt == "fp32" else None)


def test_properties_at_size(hk, cuda):
    """[128, 256, 28, 28] bf16: per channel the output has mean bias and variance scale^2 var / (var + eps);
    the gradient of x sums to zero over every channel."""
    import torch
    N, C, H, W = 128, 256, 28, 28
    x = (torch.randn(N, C, H, W, device=cuda) * 1.5 + 0.5).bfloat16()
    scale = torch.rand(C, device=cuda) + 0.5; bias = torch.randn(C, device=cuda)
    y = torch.empty_like(x); sm = torch.empty(C, device=cuda); si = torch.empty(C, device=cuda)
    hk.batch_norm_fwd(x, scale, bias, y, 0.1, 1e-5, None, None, sm, si)
    torch.cuda.synchronize()
    yf = y.float()
    assert torch.allclose(yf.mean(dim=(0, 2, 3)), bias, atol=2e-2)
    assert torch.allclose(yf.var(dim=(0, 2, 3), unbiased=False), scale ** 2, rtol=3e-2)
    assert torch.allclose(sm, x.float().mean(dim=(0, 2, 3)), atol=1e-4)
    dy = torch.randn_like(yf).bfloat16()
    dx = torch.empty_like(x); ds = torch.empty(C, device=cuda); db = torch.empty(C, device=cuda)
    hk.batch_norm_bwd(dy, x, scale, dx, ds, db, sm, si)
    torch.cuda.synchronize()
    assert torch.allclose(db, dy.float().sum(dim=(0, 2, 3)), rtol=1e-4, atol=1e-2)
    per_channel = dx.float().sum(dim=(0, 2, 3)).abs()
    assert float(per_channel.max()) < 2e-2 * float(dx.float().abs().sum(dim=(0, 2, 3)).max())


def test_refused_and_empty(hk, cuda):
    import torch
    x = torch.zeros(2, 3, 4, 4, device=cuda)
    p = torch.ones(3, device=cuda)
    with pytest.raises(hk.HkError) as e:
        hk.batch_norm_fwd(x.long(), p, p, x.long(), 0.1, 1e-5, None, None, None, None)
    assert e.value.code == -2
    import ctypes
    rc = hk.lib().hk_batch_norm_fwd(6, ctypes.c_void_p(x.data_ptr()), ctypes.c_void_p(p.data_ptr()),
                                    ctypes.c_void_p(p.data_ptr()), ctypes.c_void_p(x.data_ptr()), ctypes.c_double(0.1),
                                    ctypes.c_double(1e-5), None, None, None, None, ctypes.c_int64(2),
                                    ctypes.c_int64(3), ctypes.c_int64(16), None, ctypes.c_size_t(0), None)
    assert rc == -4                                       # no workspace
    e0 = torch.empty(0, 3, 4, 4, device=cuda)
    hk.batch_norm_fwd(e0, p, p, e0.clone(), 0.1, 1e-5, None, None, None, None)
    c0 = torch.empty(2, 0, 4, 4, device=cuda)             # no channel at all: nothing to do, forward and backward
    hk.batch_norm_fwd(c0, p[:0], p[:0], c0.clone(), 0.1, 1e-5, None, None, None, None)
    hk.batch_norm_bwd(c0, c0, p[:0], c0.clone(), p[:0].clone(), p[:0].clone(), p[:0], p[:0])
    # a constant channel: variance 0, output = bias, finite statistics
    c = torch.full((4, 2, 8, 8), 3.0, device=cuda)
    y = torch.empty_like(c); sm = torch.empty(2, device=cuda); si = torch.empty(2, device=cuda)
    hk.batch_norm_fwd(c, torch.ones(2, device=cuda), torch.full((2,), 0.25, device=cuda), y, 0.1, 1e-5, None, None, sm, si)
    torch.cuda.synchronize()
    assert (y == 0.25).all() and (sm == 3.0).all() and torch.allclose(si, torch.full((2,), 1e-5 ** -0.5, device=cuda))


@pytest.mark.parametrize("shape", [(0, 8, 4, 4), (4, 0, 4, 4), (4, 8, 0, 4)])
def test_batch_norm_empty_shapes(hk, cuda, shape):
    """An array without elements (no samples, no channels, no pixels) returns at once, forward and backward, and
    needs no workspace; running statistics are left as they are."""
    import torch
    N, C = shape[0], shape[1]
    x = torch.empty(shape, dtype=torch.float32, device=cuda)
    y = torch.empty_like(x)
    scale = torch.ones(C, device=cuda); bias = torch.zeros(C, device=cuda)
    rm = torch.full((C,), 3.0, device=cuda); rv = torch.full((C,), 5.0, device=cuda)
    sm = torch.empty(C, device=cuda); si = torch.empty(C, device=cuda)
    assert hk.batch_norm_workspace_bytes(x) == 0
    hk.batch_norm_fwd(x, scale, bias, y, 0.1, 1e-5, rm, rv, sm, si)
    dx = torch.empty_like(x); ds = torch.empty(C, device=cuda); db = torch.empty(C, device=cuda)
    hk.batch_norm_bwd(y, x, scale, dx, ds, db, sm, si)
    torch.cuda.synchronize()
    assert bool((rm == 3.0).all()) and bool((rv == 5.0).all())


# planes around one vector, odd planes, channels on both sides of what a workgroup's registers hold (65536 16-bit, 32768
# 32-bit elements; half of that backward), many and few of them, several splits per channel
RUNS = [(3, 5, 8), (3, 5, 9), (7, 3, 15), (16, 1100, 17), (64, 4, 196), (1, 2, 32768), (1, 2, 65537), (5, 3, 13121),
        (64, 8, 3136), (3, 700, 3969), (300, 2, 1021), (2, 1, 300007), (40, 1500, 49), (2048, 3, 20)]


@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("shift", [0, 1])
def test_planes_of_any_length(hk, cuda, dtype, shift):
    """Against the formulas in fp64 on the GPU; base addresses on and off the 16-byte grid; in place as well."""
    import torch
    dt = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}[dtype]

    def placed(a):
        buf = torch.full((a.numel() + 32,), 7.0, dtype=dt, device=cuda)
        view = buf[8 + shift:8 + shift + a.numel()].view(a.shape)
        view.copy_(a)
        return buf, view

    def clean(buf, view):
        return bool((buf[:8 + shift] == 7.0).all()) and bool((buf[8 + shift + view.numel():] == 7.0).all())

    gen = torch.Generator(device="cuda").manual_seed(17)
    for N, C, HW in RUNS:
        shape, m = (N, C, HW), N * HW
        rand = lambda *s: torch.randn(*s, generator=gen, device=cuda)
        _, x = placed((rand(N, C, HW) * 2 + 3).to(dt))
        _, dy = placed(rand(N, C, HW).to(dt))
        scale, bias = rand(C).abs() + 0.5, rand(C)
        rm, rv = rand(C), rand(C).abs() + 0.5
        rm0, rv0 = rm.double(), rv.double()
        yb, y = placed(torch.zeros(shape, device=cuda))
        sm, si = torch.empty(C, device=cuda), torch.empty(C, device=cuda)
        hk.batch_norm_fwd(x, scale, bias, y, 0.1, 1e-5, rm, rv, sm, si)
        torch.cuda.synchronize()
        xd, dyd = x.double(), dy.double()
        mean = xd.mean((0, 2)); var = ((xd - mean[:, None]) ** 2).mean((0, 2))
        inv = (var + 1e-5).rsqrt()
        ey = (xd - mean[:, None]) * (scale.double() * inv)[:, None] + bias.double()[:, None]
        num = lambda t: t.cpu().numpy()
        helpers.assert_close(y.contiguous(), num(ey), dtype, "y %s" % (shape,))
        helpers.assert_close(sm, num(mean), "fp32", "save_mean")
        helpers.assert_close(si, num(inv), "fp32", "save_invstd")
        helpers.assert_close(rm, num(0.9 * rm0 + 0.1 * mean), "fp32", "running_mean", scale=1.0)
        helpers.assert_close(rv, num(0.9 * rv0 + 0.1 * var * m / max(m - 1, 1)), "fp32", "running_var")
        assert clean(yb, y), shape
        xb, x2 = placed(x)
        hk.batch_norm_fwd(x2, scale, bias, x2, 0.1, 1e-5, None, None, None, None)
        torch.cuda.synchronize()
        assert torch.equal(x2, y) and clean(xb, x2), shape
        smd, sid = sm.double()[:, None], si.double()[:, None]
        xhat = (xd - smd) * sid
        eb, es = dyd.sum((0, 2)), (dyd * xhat).sum((0, 2))
        edx = scale.double()[:, None] * sid * (dyd - eb[:, None] / m - xhat * es[:, None] / m)
        db_, dx = placed(torch.zeros(shape, device=cuda))
        ds, db = torch.empty(C, device=cuda), torch.empty(C, device=cuda)
        hk.batch_norm_bwd(dy, x, scale, dx, ds, db, sm, si)
        torch.cuda.synchronize()
        helpers.assert_close(dx.contiguous(), num(edx), dtype, "dx %s" % (shape,), rtol=1e-4 if dtype == "fp32" else None)
        # sums of m terms of both signs: the rounding error is that of the terms
        helpers.assert_close(ds, num(es), "fp32", "dscale", scale=float(np.sqrt(m)))
        helpers.assert_close(db, num(eb), "fp32", "dbias", scale=float(np.sqrt(m)))
        assert clean(db_, dx), shape
        gb, g2 = placed(dy)
        hk.batch_norm_bwd(g2, x, scale, g2, None, None, sm, si)
        torch.cuda.synchronize()
        assert torch.equal(g2, dx) and clean(gb, g2), shape


# one workgroup per channel, several with a second launch, element by element
@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("shape", [(3, 6, 121), (64, 6, 196), (64, 6, 3136), (3, 6, 3)])
def test_channels_that_hold_a_nan_or_an_infinity(hk, cuda, dtype, shape):
    """Their variance, saved and running, and every output are NaN and their mean is not finite, whatever the channel's
    size; the channels beside them are as if alone."""
    import torch
    dt = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}[dtype]
    gen = torch.Generator(device="cuda").manual_seed(23)
    clean = torch.randn(shape, generator=gen, device="cuda").to(dt)
    dirty = clean.clone()
    dirty[-1, 1, shape[2] // 2] = float("nan")
    dirty[0, 2, 0] = float("inf")
    dirty[-1, 3, -1] = -float("inf")
    dirty[0, 4, 1], dirty[-1, 4, 2] = float("inf"), -float("inf")
    C, hit = shape[1], torch.tensor([False, True, True, True, True, False], device="cuda")
    scale, bias = torch.rand(C, generator=gen, device="cuda") + 0.5, torch.randn(C, generator=gen, device="cuda")
    out = []
    for x in (clean, dirty):
        y = torch.empty_like(x)
        rm, rv, sm, si = (torch.full((C,), v, device="cuda") for v in (0.0, 1.0, 7.0, 7.0))
        hk.batch_norm_fwd(x, scale, bias, y, 0.1, 1e-5, rm, rv, sm, si)
        torch.cuda.synchronize()
        out.append((y.transpose(0, 1), rm, rv, sm, si))
    for k, (a, b) in enumerate(zip(*out)):
        assert torch.equal(a[~hit], b[~hit]), k
    y, rm, rv, sm, si = (t[hit] for t in out[1])
    assert bool(torch.isnan(y).all()) and bool(torch.isnan(rv).all()) and bool(torch.isnan(si).all())
    assert not bool(torch.isfinite(rm).any()) and not bool(torch.isfinite(sm).any())


@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("shape", [(64, 513, 25), (10, 600, 1041), (40, 530, 144), (3, 700, 2003), (38, 587, 576), (30, 65, 2001),
                                   (13, 65, 9001)])
def test_many_channels(hk, cuda, dtype, shape):
    """More channels than run at once in their smallest number of vectors a thread, and one to three rounds of loads a slice."""
    import torch
    dt = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}[dtype]
    gen = torch.Generator(device="cuda").manual_seed(23)
    x = (torch.randn(shape, generator=gen, device=cuda) * 2 + 3).to(dt)
    dy = torch.randn(shape, generator=gen, device=cuda).to(dt)
    C, m = shape[1], shape[0] * shape[2]
    scale, bias = torch.rand(C, generator=gen, device=cuda) + 0.5, torch.randn(C, generator=gen, device=cuda)
    rm, rv = torch.zeros(C, device=cuda), torch.ones(C, device=cuda)
    y, dx = torch.empty_like(x), torch.empty_like(x)
    mean, invstd, ds, db = (torch.empty(C, device=cuda) for _ in range(4))
    hk.batch_norm_fwd(x, scale, bias, y, 0.1, 1e-5, rm, rv, mean, invstd)
    hk.batch_norm_bwd(dy, x, scale, dx, ds, db, mean, invstd)
    xd, gd = x.double(), dy.double()
    mu = xd.mean((0, 2))
    var = xd.var((0, 2), unbiased=False)
    istd = 1 / torch.sqrt(var + 1e-5)
    v = lambda t: t.double()[None, :, None]
    xhat = (xd - v(mu)) * v(istd)
    sdy, sdyx = gd.sum((0, 2)), (gd * xhat).sum((0, 2))
    host = lambda t: t.cpu().numpy()
    helpers.assert_close(mean, host(mu), "fp32", "mean", scale=3.0)
    helpers.assert_close(invstd, host(istd), "fp32", "invstd")
    helpers.assert_close(rv, host(0.9 + 0.1 * var * m / (m - 1)), "fp32", "running_var")
    # the rounding of what is stored, and fp32's of the terms that each element is the sum of: the statistics' own (2^-22), and
    # one for every operation
    ulp = {"fp32": 2.0 ** -23, "bf16": 2.0 ** -8, "fp16": 2.0 ** -10}[dtype]
    tiny = 2.0 ** -24 if dtype == "fp16" else 0.0
    # (the mean's rounding is that of terms of a standard deviation)
    ey, size = xhat * v(scale) + v(bias), (xhat.abs() + 1) * v(scale) + v(bias).abs()
    assert bool(((y.double() - ey).abs() <= ulp * ey.abs() + 2.0 ** -20 * size + tiny).all())
    # sums over m terms: their rounding error is that of the terms
    helpers.assert_close(db, host(sdy), "fp32", "dbias", scale=float(np.sqrt(m)))
    helpers.assert_close(ds, host(sdyx), "fp32", "dscale", scale=float(np.sqrt(m)))
    # (of a sum, the terms'; of xhat, the saved mean's as well, which is of fp32)
    k = v(scale) * v(istd)
    edx = k * (gd - v(sdy / m) - xhat * v(sdyx / m))
    size = k * (gd.abs() + v(gd.abs().mean((0, 2))) + (xhat.abs() + v(mu * istd)) * v((gd * xhat).abs().mean((0, 2))))
    assert bool(((dx.double() - edx).abs() <= ulp * edx.abs() + 2.0 ** -20 * size + tiny).all())


@pytest.mark.parametrize("shape", [(4, 800, 2300), (4, 800, 2310), (20, 800, 533), (20, 833, 621), (20, 832, 621), (4, 900, 3584), (4, 900, 3592)])
def test_many_channels_of_two_or_four_vectors_a_thread(hk, cuda, shape):
    """16-bit backward: both sides of the widths that take four."""
    test_many_channels(hk, cuda, "bf16", shape)
