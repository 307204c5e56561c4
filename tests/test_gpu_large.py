"""Arrays of more than 2^31 elements: every index computation past the 32-bit range.  The inputs are drawn on the
GPU; the kernels run on the whole array; the oracle checks a sample of rows (rows are independent) that holds the
first rows, the rows on either side of element 2^31 and the last rows, and column results are checked against
float64 sums taken in slices."""
import numpy as np
import pytest

import helpers
import oracle

pytestmark = pytest.mark.gpu

COLS = 2048
ROWS = (1 << 20) + 5                      # 2^31 + 10240 elements
EDGE = (1 << 31) // COLS                  # the row that starts at element 2^31


def _sample(rows, edge):
    return np.array([0, 1, 2, edge - 1, edge, edge + 1, rows - 2, rows - 1])


def _randn(torch, shape, seed, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.bfloat16) * scale


def _column_sums(torch, fn, rows, step=1 << 16):
    """float64 sum over rows of fn(lo, hi) -> [hi - lo, cols] float64, in slices."""
    total = None
    for lo in range(0, rows, step):
        part = fn(lo, min(rows, lo + step)).sum(0)
        total = part if total is None else total + part
    return total.cpu().numpy()


def test_rmsnorm_forward_backward_past_2_31_elements(hk, cuda):
    import torch
    x, dz = _randn(torch, (ROWS, COLS), 1), _randn(torch, (ROWS, COLS), 2)
    w = (torch.rand(COLS, device=cuda) * 0.4 + 0.8).to(torch.bfloat16)
    z, dx = torch.empty_like(x), torch.empty_like(x)
    mu, rs = torch.empty(ROWS, device=cuda), torch.empty(ROWS, device=cuda)
    dg, db = torch.empty_like(w), torch.empty_like(w)
    hk.dropout_add_ln_fwd(x, None, w, None, z, None, mu, rs, 1e-6, True)
    hk.dropout_add_ln_bwd(dz, None, x, mu, rs, w, dx, None, dg, db, True)
    torch.cuda.synchronize()
    sel = _sample(ROWS, EDGE)
    xs, dzs, ws = helpers.to_numpy(x[sel]), helpers.to_numpy(dz[sel]), helpers.to_numpy(w)
    ez, _, _, ers = oracle.dropout_add_ln_fwd(xs, None, ws, None, 1e-6, True)
    helpers.assert_close(z[sel], ez, "bf16", "z")
    helpers.assert_close(rs[sel], ers, "fp32", "rsigma")
    rs_sel = helpers.to_numpy(rs[sel])
    edx, _, _ = oracle.dropout_add_ln_bwd(dzs, None, xs, np.zeros(len(sel)), rs_sel, ws, True)
    helpers.assert_close(dx[sel], edx, "bf16", "dx")
    want = _column_sums(torch, lambda lo, hi: dz[lo:hi].double() * x[lo:hi].double() * rs[lo:hi].double()[:, None],
                        ROWS)
    helpers.assert_close(dg, want, "bf16", "dgamma over 2^20 rows")
    helpers.assert_close(db, _column_sums(torch, lambda lo, hi: dz[lo:hi].double(), ROWS), "bf16", "dbeta")


def test_softmax_past_2_31_elements(hk, cuda):
    import torch
    x, dy = _randn(torch, (ROWS, COLS), 3, 2.0), _randn(torch, (ROWS, COLS), 4)
    y, dx = torch.empty_like(x), torch.empty_like(x)
    hk.softmax_fwd(x, y, -1)
    hk.softmax_bwd(y, dy, dx, -1)
    torch.cuda.synchronize()
    sel = _sample(ROWS, EDGE)
    helpers.assert_close(y[sel], oracle.softmax_fwd(helpers.to_numpy(x[sel])), "bf16", "softmax")
    helpers.assert_close(dx[sel], oracle.softmax_bwd(helpers.to_numpy(y[sel]), helpers.to_numpy(dy[sel])), "bf16",
                         "softmax gradient")


def test_cross_entropy_past_2_31_elements(hk, cuda):
    import torch
    rows, cols = 67110, 32000              # 2 147 520 000 elements
    edge = (1 << 31) // cols
    x = _randn(torch, (rows, cols), 5, 2.0)
    labels = torch.randint(0, cols, (rows,), device=cuda)
    labels[::11] = -100
    loss = torch.empty(rows, dtype=torch.bfloat16, device=cuda)
    grad = _randn(torch, (rows,), 6)
    dx = torch.empty_like(x)
    hk.sce_sparse_fwd(x, labels, loss, -100)
    hk.sce_sparse_bwd(x, labels, grad, dx, -100)
    torch.cuda.synchronize()
    sel = _sample(rows, edge)
    xs, ls = helpers.to_numpy(x[sel]), labels[sel].cpu().numpy()
    helpers.assert_close(loss[sel], oracle.sce_sparse_fwd(xs, ls, -100), "bf16", "loss")
    helpers.assert_close(dx[sel], oracle.sce_sparse_bwd(xs, ls, helpers.to_numpy(grad[sel]), -100), "bf16", "dlogits")
    # every row of the gradient sums to zero (softmax sums to one, minus the one-hot), ignored rows are zero
    row_sums = torch.stack([dx[lo:lo + 4096].float().sum(1).abs().max() for lo in range(0, rows, 4096)]).max().item()
    assert row_sums <= 0.05
    assert (dx[::11] == 0).all()


def test_elementwise_and_broadcast_past_2_31_elements(hk, cuda):
    import torch
    x = _randn(torch, (ROWS, COLS), 7)
    per_row = _randn(torch, (ROWS, 1), 8)
    out = torch.empty_like(x)
    sel = _sample(ROWS, EDGE)
    hk.binary("sub", x, per_row, out)
    torch.cuda.synchronize()
    want = helpers.to_numpy(x[sel]).astype(np.float64) - helpers.to_numpy(per_row[sel]).astype(np.float64)
    helpers.assert_close(out[sel], want, "bf16", "x - per-row value")
    hk.unary("exp", x, out)
    torch.cuda.synchronize()
    helpers.assert_close(out[sel], np.exp(helpers.to_numpy(x[sel]).astype(np.float64)), "bf16", "exp")
    hk.broadcast(per_row, out, scalar=0.5)
    torch.cuda.synchronize()
    assert torch.equal(out[sel], (per_row[sel] * 0.5).expand(len(sel), COLS))
    assert torch.equal(out[:, COLS - 1], (per_row[:, 0] * 0.5))          # the last column of every row


def test_reduce_past_2_31_elements(hk, cuda):
    import torch
    x = _randn(torch, (ROWS, COLS), 9)
    rows_out = torch.empty(ROWS, dtype=torch.bfloat16, device=cuda)
    cols_out = torch.empty(COLS, dtype=torch.bfloat16, device=cuda)
    hk.reduce(x, rows_out, [1], "sum")
    hk.reduce(x, cols_out, [0], "mean")
    torch.cuda.synchronize()
    sel = _sample(ROWS, EDGE)
    helpers.assert_close(rows_out[sel], helpers.to_numpy(x[sel]).astype(np.float64).sum(1), "bf16", "row sums")
    want = _column_sums(torch, lambda lo, hi: x[lo:hi].double(), ROWS) / ROWS
    # a mean of 2^20 standard normal draws is ~1e-3: compare on the scale of one draw's share
    helpers.assert_close(cols_out, want, "bf16", "column means", scale=1e-3)
    nrm = torch.empty(ROWS, dtype=torch.bfloat16, device=cuda)
    hk.norm(x, nrm, 1, 2)
    torch.cuda.synchronize()
    helpers.assert_close(nrm[sel], np.sqrt((helpers.to_numpy(x[sel]).astype(np.float64) ** 2).sum(1)), "bf16", "2-norm")


def test_batch_norm_past_2_31_elements(hk, cuda):
    import torch
    n, c, hw = 33, 64, 1024 * 1024 + 8       # 2 214 609 920 elements
    x = _randn(torch, (n, c, hw), 10, 1.5) + 0.25
    y = torch.empty_like(x)
    scale, bias = torch.rand(c, device=cuda) + 0.5, torch.randn(c, device=cuda)
    rm, rv = torch.zeros(c, device=cuda), torch.ones(c, device=cuda)
    sm, si = torch.empty(c, device=cuda), torch.empty(c, device=cuda)
    hk.batch_norm_fwd(x, scale, bias, y, 0.1, 1e-5, rm, rv, sm, si)
    torch.cuda.synchronize()
    mean = torch.stack([x[:, ch].double().mean() for ch in range(c)])
    var = torch.stack([((x[:, ch].double() - mean[ch]) ** 2).mean() for ch in range(c)])
    helpers.assert_close(sm, mean.cpu().numpy(), "fp32", "saved mean", scale=1.0)
    helpers.assert_close(si, (1.0 / torch.sqrt(var + 1e-5)).cpu().numpy(), "fp32", "saved inverse deviation")
    for img, ch in ((0, 0), (15, 31), (16, 0), (32, 63)):       # image 15/16: either side of element 2^31
        want = (x[img, ch].double() - mean[ch]) / torch.sqrt(var[ch] + 1e-5) * scale[ch].double() + bias[ch].double()
        got = y[img, ch].double()
        assert ((got - want).abs() <= 1e-2 * (want.abs() + 1.0)).all()


# the last, partial vector of such a plane ends past element 2^31
LONGEST_PLANE = (1 << 31) - 3


def _guarded(torch, n, cuda):
    buf = torch.full((n + 64,), 7.0, dtype=torch.bfloat16, device=cuda)
    return buf, buf[32:32 + n]


def test_softmax_over_planes_that_end_below_2_31_elements(hk, cuda):
    import torch
    n = LONGEST_PLANE
    x = _randn(torch, (2 * n,), 11, 2.0).view(1, 2, n)
    dy = _randn(torch, (2 * n,), 12).view(1, 2, n)
    yb, y = _guarded(torch, 2 * n, cuda)
    hk.softmax_fwd(x, y.view(1, 2, n), 1)
    db, dx = _guarded(torch, 2 * n, cuda)
    hk.softmax_bwd(y.view(1, 2, n), dy, dx.view(1, 2, n), 1)
    torch.cuda.synchronize()
    for buf in (yb, db):
        assert bool((buf[:32] == 7.0).all()) and bool((buf[-32:] == 7.0).all())
    y, dx = y.view(2, n), dx.view(2, n)
    for lo in (0, n // 2, n - 1000):
        at = slice(lo, lo + 1000)
        helpers.assert_close(y[:, at].contiguous(), torch.softmax(x[0, :, at].double(), 0).cpu().numpy(), "bf16", "softmax")
        yd = y[:, at].double()
        want = yd * (dy[0, :, at].double() - (yd * dy[0, :, at].double()).sum(0))
        helpers.assert_close(dx[:, at].contiguous(), want.cpu().numpy(), "bf16", "softmax gradient")


def test_batch_norm_of_a_plane_that_ends_below_2_31_elements(hk, cuda):
    import torch
    n = LONGEST_PLANE
    x = _randn(torch, (n,), 13, 2.0).add_(3.0)
    total = squares = 0.0
    for part in x.split(1 << 28):
        d = part.double()
        total += float(d.sum())
        squares += float(((d - 3.0) ** 2).sum())
    mean = total / n
    var = squares / n - (mean - 3.0) ** 2
    scale, bias = torch.full((1,), 1.5, device=cuda), torch.full((1,), 0.25, device=cuda)
    sm, si = torch.empty(1, device=cuda), torch.empty(1, device=cuda)
    yb, y = _guarded(torch, n, cuda)
    hk.batch_norm_fwd(x.view(1, 1, n), scale, bias, y.view(1, 1, n), 0.1, 1e-5, None, None, sm, si)
    db, dx = _guarded(torch, n, cuda)
    dy = _randn(torch, (n,), 14)
    hk.batch_norm_bwd(dy.view(1, 1, n), x.view(1, 1, n), scale, dx.view(1, 1, n), None, None, sm, si)
    torch.cuda.synchronize()
    for buf in (yb, db):
        assert bool((buf[:32] == 7.0).all()) and bool((buf[-32:] == 7.0).all())
    inv = (var + 1e-5) ** -0.5
    helpers.assert_close(sm, np.array([mean]), "fp32", "save_mean")
    helpers.assert_close(si, np.array([inv]), "fp32", "save_invstd")
    mean_dy = mean_dyx = 0.0
    for lo in range(0, n, 1 << 28):
        d, xhat = dy[lo:lo + (1 << 28)].double(), (x[lo:lo + (1 << 28)].double() - mean) * inv
        mean_dy += float(d.sum()) / n
        mean_dyx += float((d * xhat).sum()) / n
    for lo in (0, n // 2, n - 1000):
        at = slice(lo, lo + 1000)
        xhat = (x[at].double() - mean) * inv
        helpers.assert_close(y[at], (xhat * 1.5 + 0.25).cpu().numpy(), "bf16", "batch norm")
        want = 1.5 * inv * (dy[at].double() - mean_dy - xhat * mean_dyx)
        helpers.assert_close(dx[at], want.cpu().numpy(), "bf16", "batch norm gradient")


def _batch_norm_time(torch, hk, cuda, N, C, HW):
    """us of a forward and a backward, the best of three."""
    x, y = torch.ones((N, C, HW), dtype=torch.bfloat16, device=cuda), torch.empty((N, C, HW), dtype=torch.bfloat16, device=cuda)
    scale, bias, sm, si = (torch.ones(C, device=cuda) for _ in range(4))
    workspace = torch.empty(hk.batch_norm_workspace_bytes(x) // 4 + 1, device=cuda)
    best = [1e9, 1e9]
    for _ in range(4):
        at = [torch.cuda.Event(enable_timing=True) for _ in range(3)]
        at[0].record()
        hk.batch_norm_fwd(x, scale, bias, y, 0.1, 1e-5, None, None, sm, si, workspace=workspace)
        at[1].record()
        hk.batch_norm_bwd(x, x, scale, y, None, None, sm, si, workspace=workspace)
        at[2].record()
        torch.cuda.synchronize()
        best = [min(b, at[i].elapsed_time(at[i + 1]) * 1e3) for i, b in enumerate(best)]
    return best


# channels of the two-launch form and of one workgroup
@pytest.mark.parametrize("half,C,HW", [(90, 1024, 112 * 112), (16, 168000, 28 * 28)])
def test_batch_norm_past_2_31_elements_is_no_slower_by_element(hk, cuda, half, C, HW):
    """Twice the array costs about twice the time: the same kernels take it past element 2^31 (element by element it
    was eight times)."""
    import torch
    assert half * C * HW < (1 << 31) < 2 * half * C * HW
    small, large = _batch_norm_time(torch, hk, cuda, half, C, HW), _batch_norm_time(torch, hk, cuda, 2 * half, C, HW)
    assert large[0] < 3 * small[0] and large[1] < 3 * small[1], (small, large)


# of both forms, whole vectors and ragged planes, and a plane of more than 2^31 elements
@pytest.mark.parametrize("N,C,HW", [(180, 1024, 112 * 112), (32, 90000, 28 * 28 + 1), (2, 1, (1 << 31) + 5)])
def test_batch_norm_past_2_31_elements_of_every_form(hk, cuda, N, C, HW):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(21)
    x, dy = (_randn(torch, (N, C, HW), 31 + k, 2.0) for k in range(2))
    x += 3.0
    scale, bias = (torch.rand(C, generator=gen, device=cuda) + 0.5 for _ in range(2))
    y, dx = torch.empty_like(x), torch.empty_like(x)
    sm, si, ds, db = (torch.empty(C, device=cuda) for _ in range(4))
    hk.batch_norm_fwd(x, scale, bias, y, 0.1, 1e-5, None, None, sm, si)
    hk.batch_norm_bwd(dy, x, scale, dx, ds, db, sm, si)
    torch.cuda.synchronize()
    m = N * HW
    for c in sorted({0, 1 % C, C // 2, C - 1}):
        def mean_of(fn):
            total = 0.0
            for n in range(N):
                for lo in range(0, HW, 1 << 28):
                    at = slice(lo, min(HW, lo + (1 << 28)))
                    total += float(fn(x[n, c, at].double(), dy[n, c, at].double()).sum())
            return total / m
        mean = mean_of(lambda a, g: a)
        inv = (mean_of(lambda a, g: (a - mean) ** 2) + 1e-5) ** -0.5
        helpers.assert_close(sm[c:c + 1], np.array([mean]), "fp32", "save_mean")
        helpers.assert_close(si[c:c + 1], np.array([inv]), "fp32", "save_invstd")
        mean, inv = float(sm[c]), float(si[c])
        mg, mgx = mean_of(lambda a, g: g), mean_of(lambda a, g: g * (a - mean) * inv)
        # sums of m terms of both signs: the rounding error is that of the terms
        helpers.assert_close(db[c:c + 1], np.array([mg * m]), "fp32", "dbias", scale=float(np.sqrt(m)))
        helpers.assert_close(ds[c:c + 1], np.array([mgx * m]), "fp32", "dscale", scale=float(np.sqrt(m)))
        for n in sorted({0, 1, N // 2, N - 1}):
            for at in (slice(0, 700), slice(HW - 700, HW)):
                xhat = (x[n, c, at].double() - mean) * inv
                helpers.assert_close(y[n, c, at], (xhat * float(scale[c]) + float(bias[c])).cpu().numpy(), "bf16", "y")
                want = float(scale[c]) * inv * (dy[n, c, at].double() - mg - xhat * mgx)
                helpers.assert_close(dx[n, c, at], want.cpu().numpy(), "bf16", "dx")


@pytest.mark.parametrize("cols", [64, 61, 1000, 1021])
def test_rows_2_31_elements_apart(hk, cuda, cols):
    """Steps between rows that 32 bits do not hold, on one level and as one of three, against the same rows side by side."""
    import torch
    far = (1 << 31) + 8
    block = 3 * 5 * 1024
    base = torch.empty(far + block, dtype=torch.bfloat16, device=cuda)

    def check(shape, strides):
        def far_copy(t, off):
            v = base.as_strided(shape, strides, off)
            v.copy_(t)
            return v
        g = torch.Generator(device=cuda).manual_seed(cols)
        x, dy = (torch.randn(shape, generator=g, device=cuda).to(torch.bfloat16) for _ in range(2))
        y, dx = torch.empty_like(x), torch.empty_like(x)
        hk.softmax_fwd(x, y, -1)
        hk.softmax_bwd(y, dy, dx, -1)
        fy, fdx = torch.empty_like(x), torch.empty_like(x)
        hk.softmax_fwd(far_copy(x, 0), fy, -1)
        assert torch.equal(fy, y), shape
        hk.softmax_bwd(far_copy(y, 0), dy, fdx, -1)
        assert torch.equal(fdx, dx), shape
        fout = base.as_strided(shape, strides, 0)
        hk.softmax_fwd(x, fout, -1)
        assert torch.equal(fout, y), shape
        rows = x.numel() // cols
        w = torch.rand(cols, generator=g, device=cuda).to(torch.bfloat16)
        mu, rs, z = torch.empty(rows, device=cuda), torch.empty(rows, device=cuda), torch.empty_like(x)
        fmu, frs, fz = torch.empty(rows, device=cuda), torch.empty(rows, device=cuda), torch.empty_like(x)
        hk.layer_norm_fwd(x, w, w, z, mu, rs, 1e-5)
        hk.layer_norm_fwd(far_copy(x, 0), w, w, fz, fmu, frs, 1e-5)
        helpers.assert_close(fz, helpers.to_numpy(z).astype(np.float64), "bf16", "z")
        helpers.assert_close(frs, helpers.to_numpy(rs).astype(np.float64), "fp32", "rstd")
        dg, db, fdg, fdb = (torch.empty_like(w) for _ in range(4))
        hk.layer_norm_bwd(dy, x, w, w, mu, rs, dx, dg, db, 1e-5)
        hk.layer_norm_bwd(far_copy(dy, 0), x, w, w, mu, rs, fdx, fdg, fdb, 1e-5)
        for got, want, what in ((fdx, dx, "dx"), (fdg, dg, "dgamma"), (fdb, db, "dbeta")):
            helpers.assert_close(got, helpers.to_numpy(want).astype(np.float64), "bf16", what)

    check((2, cols), (far, 1))
    if cols % 8 == 0:
        check((3, 2, 5, cols), (5 * cols, far, cols, 1))
        check((2, 5, 3, cols), (far, cols, 5 * cols, 1))


def test_cross_entropy_rows_2_31_elements_apart(hk, cuda):
    """As above: per token losses, their gradient from gradients of their own, labels by row number."""
    import torch
    cols, far = 200, (1 << 31) + 8
    base = torch.empty(far + 3 * 5 * cols, dtype=torch.bfloat16, device=cuda)
    for shape, strides in (((2, cols), (far, 1)), ((3, 2, 5, cols), (5 * cols, far, cols, 1)), ((2, 5, 3, cols), (far, cols, 5 * cols, 1))):
        g = torch.Generator(device=cuda).manual_seed(7)
        x = torch.randn(shape, generator=g, device=cuda).to(torch.bfloat16)
        labels = torch.randint(0, cols, shape[:-1], generator=g, device=cuda)
        labels.view(-1)[1] = -100
        dloss = torch.rand(shape[:-1], generator=g, device=cuda).to(torch.bfloat16)
        loss, floss = torch.empty_like(dloss), torch.empty_like(dloss)
        dx, fdx = torch.empty_like(x), torch.empty_like(x)
        hk.sce_sparse_fwd(x, labels, loss, -100)
        hk.sce_sparse_bwd(x, labels, dloss, dx, -100)
        fx = base.as_strided(shape, strides, 0)
        fx.copy_(x)
        hk.sce_sparse_fwd(fx, labels, floss, -100)
        hk.sce_sparse_bwd(fx, labels, dloss, fdx, -100)
        assert torch.equal(floss, loss) and torch.equal(fdx, dx), shape


def test_gradients_of_rows_2_31_elements_apart(hk, cuda):
    """Gradients that are written so far apart, on one level and as one of three, against the same side by side; logits beside them
    or as far apart in another order."""
    import torch
    cols, far = 200, (1 << 31) + 8
    room = 3 * 5 * cols
    base = torch.empty(far + 2 * room, dtype=torch.bfloat16, device=cuda)
    for shape, strides in (((2, cols), (far, 1)), ((3, 2, 5, cols), (5 * cols, far, cols, 1)), ((2, 5, 3, cols), (far, cols, 5 * cols, 1)),
                           ((5, 3, 2, cols), (cols, 5 * cols, far, 1))):
        g = torch.Generator(device=cuda).manual_seed(11)
        x, dy = (torch.randn(shape, generator=g, device=cuda).to(torch.bfloat16) for _ in range(2))
        labels = torch.randint(0, cols, shape[:-1], generator=g, device=cuda)
        labels.view(-1)[1] = -100
        dloss = torch.rand(shape[:-1], generator=g, device=cuda).to(torch.bfloat16)
        y, dx = torch.empty_like(x), torch.empty_like(x)
        out = base.as_strided(shape, strides, room)
        hk.softmax_fwd(x, y, -1)
        hk.softmax_bwd(y, dy, dx, -1)
        hk.softmax_bwd(y, dy, out, -1)
        assert torch.equal(out, dx), shape
        hk.sce_sparse_bwd(x, labels, dloss, dx, -100)
        hk.sce_sparse_bwd(x, labels, dloss, out, -100)
        assert torch.equal(out, dx), shape
        fx = base.as_strided(shape, strides, 0)
        fx.copy_(x)
        out.zero_()
        hk.sce_sparse_bwd(fx, labels, dloss, out, -100)
        assert torch.equal(out, dx), shape
