"""Rows of any length and alignment through the register kernels: row lengths at the edges of a vector, of a lane
group and of a workgroup, bases that lie off the 16-byte grid by one element, and row pitches that are no multiple of
a vector.  The outputs sit inside guarded buffers: nothing outside a row may be written."""
import numpy as np
import pytest

import helpers
import oracle

pytestmark = pytest.mark.gpu

ES = {"fp32": 4, "bf16": 2, "fp16": 2}
GUARD = 16


def _placed(cuda, a, dtype, offset, pitch, fill=None):
    """(whole buffer, [rows, cols] view): `a` (or, without it, `fill`) laid `offset` elements into a buffer of rows
    `pitch` apart, with guard elements of value 7 around and between the rows."""
    import torch
    rows, cols = a.shape
    dt = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}[dtype]
    buf = torch.full((GUARD + rows * pitch + GUARD,), 7.0, dtype=dt, device=cuda)
    view = torch.as_strided(buf, (rows, cols), (pitch, 1), GUARD + offset)
    view.copy_(helpers.to_torch(a, dtype, cuda) if fill is None else torch.full_like(view, fill))
    return buf, view


def _guards_untouched(buf, view):
    import torch
    keep = buf.clone()
    inside = torch.as_strided(keep, view.shape, view.stride(), view.storage_offset())
    inside.fill_(7.0)
    return bool((keep == 7.0).all())


# vectors per row around 1, 8, 16, 32, 64, 128, 192, 256 and the workgroup widths above, and one element off each
def _lengths(dtype):
    vec = 16 // ES[dtype]
    out = set()
    for v in (1, 2, 8, 16, 32, 64, 96, 128, 192, 256, 300, 512):
        out.update((v * vec, v * vec + 1, v * vec + vec - 1))
    return sorted(out)


@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("shift", [0, 1])
def test_softmax_any_length(hk, cuda, dtype, shift):
    import torch
    rows = 37
    for cols in _lengths(dtype):
        pitch = cols + (0 if shift == 0 else 5)
        x = helpers.draw(3000 + cols, (rows, cols), dtype=dtype)
        dy = helpers.draw(4000 + cols, (rows, cols), dtype=dtype)
        ey = oracle.softmax_fwd(x)
        _, tx = _placed(cuda, x, dtype, shift, pitch)
        yb, ty = _placed(cuda, x, dtype, shift, pitch, 0.0)
        hk.softmax_fwd(tx, ty)
        torch.cuda.synchronize()
        helpers.assert_close(ty.contiguous(), ey, dtype, "softmax y %d" % cols)
        assert _guards_untouched(yb, ty), cols
        y = helpers.to_numpy(ty.contiguous())
        _, tdy = _placed(cuda, dy, dtype, shift, pitch)
        db, tdx = _placed(cuda, x, dtype, shift, pitch, 0.0)
        hk.softmax_bwd(ty, tdy, tdx)
        torch.cuda.synchronize()
        # dx = y (dy - sum dy y): a difference of terms of the size of y dy, which `scale` names
        helpers.assert_close(tdx.contiguous(), oracle.softmax_bwd(y, dy), dtype, "softmax dx %d" % cols,
                             scale=float(np.sqrt(np.mean(np.square(y * dy)))),
                             ordinary_rtol=helpers.SOFTMAX_GRADIENT_ORDINARY_RTOL)
        assert _guards_untouched(db, tdx), cols
        # in place: the row's last vector overlaps the one before it
        hk.softmax_fwd(tx, tx)
        torch.cuda.synchronize()
        assert torch.equal(tx.contiguous(), ty.contiguous()), cols


# entries around one lane's share, a wavefront's and half a wavefront's slices and the most of both; planes around a
# vector and a workgroup's vectors
DIM_SHAPES = [(2, d, n) for d in (2, 3, 7, 8, 9, 16, 17, 21, 33, 128, 129, 150, 255, 256, 257) for n in (7, 8, 9, 67)] + \
             [(1, 5, 1), (1, 5, 3), (3, 21, 515), (2, 40, 1031), (300, 11, 49), (1, 256, 600)]


@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("shift", [0, 1])
def test_softmax_over_a_leading_dimension(hk, cuda, dtype, shift):
    import torch
    dt = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}[dtype]
    low = torch.finfo(dt).min
    for shape in DIM_SHAPES:
        n = int(np.prod(shape))
        x, dy = (helpers.to_torch(helpers.draw(s + n, shape, dtype=dtype), dtype, cuda) for s in (10, 20))
        x[0, :, -1] = low                         # masked: all of a column, all but one entry, -inf, NaN
        if shape[2] > 3:
            x[0, 1:, 0] = low
            x[0, 0, 1] = -float("inf")
            x[-1, :, 2] = -float("inf")
            x[-1, 0, 3] = float("nan")

        def placed(a):
            buf = torch.full((n + 32,), 7.0, dtype=dt, device=cuda)
            view = buf[8 + shift:8 + shift + n].view(shape)
            view.copy_(a)
            return buf, view

        def clean(buf):
            return bool((buf[:8 + shift] == 7.0).all()) and bool((buf[8 + shift + n:] == 7.0).all())

        (_, tx), (_, tdy) = placed(x), placed(dy)
        (yb, ty), (db, tdx) = placed(torch.zeros_like(x)), placed(torch.zeros_like(x))
        hk.softmax_fwd(tx, ty, 1)
        torch.cuda.synchronize()
        ey = torch.softmax(x.double(), 1)
        assert torch.equal(torch.isnan(ty), torch.isnan(ey)), shape
        helpers.assert_close(ty.nan_to_num().contiguous(), ey.nan_to_num().cpu().numpy(), dtype, "softmax y %s" % (shape,))
        y = ty.nan_to_num()
        (_, ty2) = placed(y)
        hk.softmax_bwd(ty2, tdy, tdx, 1)
        torch.cuda.synchronize()
        yd = y.double() * dy.double()
        edx = yd - y.double() * yd.sum(1, keepdim=True)
        helpers.assert_close(tdx.contiguous(), edx.cpu().numpy(), dtype, "softmax dx %s" % (shape,),
                             scale=float(yd.square().mean().sqrt()), ordinary_rtol=helpers.SOFTMAX_GRADIENT_ORDINARY_RTOL)
        assert clean(yb) and clean(db), shape
        (xb, x2), (gb, g2) = placed(x), placed(dy)
        hk.softmax_fwd(x2, x2, 1)                 # in place
        hk.softmax_bwd(ty2, g2, g2, 1)
        torch.cuda.synchronize()
        assert torch.equal(x2.nan_to_num(), ty.nan_to_num()) and torch.equal(g2, tdx) and clean(xb) and clean(gb), shape


# (shape, axes, permutation of the dense array or None): runs of every length around a vector and the widths of the
# lane groups and workgroups, few and many of them, rows that several workgroups share; rows shorter than a vector;
# rows on two levels; columns that are no whole number of vectors, over few and many rows
REDUCTIONS = [((b, c, n), (0, 2), None) for b, c, n in
              [(2, 3, 8), (9, 5, 7), (8, 16, 1), (8, 33, 40), (8, 33, 63), (7, 33, 9), (8, 40, 127), (8, 40, 129),
               (64, 3, 1000), (300, 20, 31), (5, 300, 257), (3, 2, 70001), (64, 1030, 130), (2, 1, 400003)]]
REDUCTIONS += [((45, n), (1,), None) for n in list(range(2, 18)) + [31, 63, 65, 127, 129, 255, 257, 511, 513, 1021, 4099]]
REDUCTIONS += [((3, 70001), (1,), None), ((1, 600011), (1,), None), ((70001, 3), (1,), None)]
REDUCTIONS += [((4, 6, 50), (2,), (1, 0, 2)), ((5, 4, 6, 50), (1, 3), (0, 2, 1, 3)), ((5, 4, 6, 50), (0, 3), (2, 0, 1, 3))]
REDUCTIONS += [((r, c), (0,), None) for r in (2, 7, 9, 300) for c in (3, 8, 9, 15, 513, 1025)]
REDUCTIONS += [((3, 41, 77), (1,), None), ((2, 3000, 1001), (1,), None)]


@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("shift", [0, 1])
def test_reduce_any_extent(hk, cuda, dtype, shift):
    """Whole numbers of -3..3: their sums are exact in fp32 in any order, so the result is the rounded exact sum."""
    import torch
    dt = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}[dtype]
    for k, (shape, axes, perm) in enumerate(REDUCTIONS):
        a = np.random.default_rng(5000 + k).integers(-3, 4, shape).astype(np.float32)
        buf = torch.zeros(GUARD + a.size, dtype=dt, device=cuda)
        x = torch.as_strided(buf, shape, torch.empty(shape).stride(), shift)
        x.copy_(torch.from_numpy(a).to(dt))
        if perm is not None:
            x, a = x.permute(perm), a.transpose(perm)
        kept = [n for i, n in enumerate(a.shape) if i not in axes]
        for op, expected in (("sum", a.sum(axes, dtype=np.float64)), ("max", a.max(axes))):
            # with the scratch asked for, and (where rows lie off the 16-byte grid) without any
            for workspace in [None] + ([torch.empty(1, device=cuda)] if shift else []):
                out = torch.full((GUARD + int(np.prod(kept)) + GUARD,), 77.0, dtype=dt, device=cuda)
                view = out[GUARD:-GUARD].view(kept)
                hk.reduce(x, view, list(axes), op, workspace=workspace)
                torch.cuda.synchronize()
                what = (shape, axes, op, workspace is None)
                assert torch.equal(view.float().cpu().double(), torch.from_numpy(
                    oracle.round_to(np.asarray(expected, np.float32), dtype).astype(np.float64))), what
                assert bool((out[:GUARD] == 77.0).all()) and bool((out[-GUARD:] == 77.0).all()), what


@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("cols", [3, 40, 41, 130, 1001, 2047, 2048, 4097])
def test_softmax_of_lowest_values(hk, cuda, dtype, cols):
    """Scores masked with the type's lowest value (whole threads' share of a row, and whole rows), -inf, +inf and NaN."""
    import torch
    dt = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}[dtype]
    low = torch.finfo(dt).min
    x = helpers.to_torch(helpers.draw(9000 + cols, (8, cols), dtype=dtype), dtype, cuda)
    x[0, 2:] = low
    x[1, : cols - 2] = -float("inf")
    x[2, :] = low
    x[3, :] = low
    x[3, 1] = low / 1.25
    x[4, :] = -float("inf")
    x[5, cols // 2] = float("nan")
    x[6, cols - 1] = float("inf")
    y = torch.empty_like(x)
    hk.softmax_fwd(x, y)
    torch.cuda.synchronize()
    want = torch.softmax(x.double(), -1)
    assert torch.equal(torch.isnan(y), torch.isnan(want))
    ok = [0, 1, 2, 3, 7]
    helpers.assert_close(y[ok], want[ok].cpu().numpy(), dtype, "softmax y")
    hk.softmax_fwd(x, x)
    torch.cuda.synchronize()
    assert torch.equal(x[ok], y[ok])


# vectors per row around 1, a wavefront, the widths of the workgroups, and (65536 16-bit / 32768 32-bit elements)
# past what a workgroup holds: whole vectors, one element more, one fewer
def _class_counts(dtype):
    vec = 16 // ES[dtype]
    out = {v * vec + k for v in (1, 2, 63, 64, 65, 256, 512, 1000) for k in (0, 1, vec - 1)}
    out.update(range(1, 2 * vec))
    out.update((4096 * vec, 4096 * vec + 1, 8192 * vec - 1, 8192 * vec, 8192 * vec + 1, 9000 * vec + 3, 12289 * vec - 1))
    return sorted(out)


@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("shift", [0, 1])
def test_cross_entropy_any_length(hk, cuda, dtype, shift):
    import torch
    rows, ignored = 9, -100
    for cols in _class_counts(dtype):
        pitch = cols + (0 if shift == 0 else 5)
        x = helpers.draw(6000 + cols, (rows, cols), dtype=dtype)
        lab = np.array([0, cols - 1, ignored, cols // 2, cols - min(cols, 5), 1 % cols, -7, ignored, max(cols - 2, 0)], np.int64)
        g = helpers.draw(7000 + cols, (rows,), dtype=dtype)
        _, tx = _placed(cuda, x, dtype, shift, pitch)
        tl, tg = torch.from_numpy(lab).to(cuda), helpers.to_torch(g, dtype, cuda)
        loss = torch.empty(rows, dtype=tx.dtype, device=cuda)
        hk.sce_sparse_fwd(tx, tl, loss, ignored)
        db, dx = _placed(cuda, x, dtype, shift, pitch, 0.0)
        hk.sce_sparse_bwd(tx, tl, tg, dx, ignored)
        torch.cuda.synchronize()
        inside = (lab >= 0) | (lab == ignored)     # -7 is no class: the loss is NaN, the gradient has no one-hot term
        el = oracle.sce_sparse_fwd(x[inside], lab[inside], ignored)
        helpers.assert_close(loss[torch.from_numpy(inside).to(cuda)], el, dtype, "loss %d" % cols)
        assert bool(torch.isnan(loss[~torch.from_numpy(inside).to(cuda)]).all())
        edx = oracle.sce_sparse_bwd(x[inside], lab[inside], g[inside], ignored)
        helpers.assert_close(dx.contiguous()[torch.from_numpy(inside).to(cuda)], edx, dtype, "dlogits %d" % cols)
        want = torch.softmax(tx[6].double(), -1) * tg[6].double()
        helpers.assert_close(dx[6].contiguous(), want.cpu().numpy(), dtype, "dlogits of no class %d" % cols)
        assert _guards_untouched(db, dx), cols
        hk.sce_sparse_bwd(tx, tl, tg, tx, ignored)     # in place
        torch.cuda.synchronize()
        assert torch.equal(tx.contiguous(), dx.contiguous()), cols


@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("cols", [40, 41, 1001, 4096, 50257, 70001])
def test_cross_entropy_of_lowest_values(hk, cuda, dtype, cols):
    """Logits masked with the type's lowest value (whole threads' share of a row, and whole rows), -inf, +inf and NaN."""
    import torch
    dt = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}[dtype]
    low = torch.finfo(dt).min
    x = helpers.to_torch(helpers.draw(8000 + cols, (8, cols), dtype=dtype), dtype, cuda)
    x[0, 3:] = low
    x[1, : cols - 2] = -float("inf")
    x[2, :] = low
    x[3, :] = low
    x[3, 5] = low / 1.25
    x[4, :] = -float("inf")
    x[5, cols // 2] = float("nan")
    x[6, cols - 1] = float("inf")
    lab = torch.tensor([1, cols - 1, 7, 5, 0, 0, 0, cols - 1], device=cuda)
    g = torch.ones(8, dtype=dt, device=cuda)
    loss, dx = torch.empty(8, dtype=dt, device=cuda), torch.empty_like(x)
    hk.sce_sparse_fwd(x, lab, loss, -100)
    hk.sce_sparse_bwd(x, lab, g, dx, -100)
    torch.cuda.synchronize()
    p = torch.softmax(x.double(), -1)
    want = torch.nn.functional.cross_entropy(x.double(), lab, reduction="none")
    p[torch.arange(8, device=cuda), lab] -= 1
    for r in range(8):
        assert bool(torch.isnan(loss[r])) == bool(torch.isnan(want[r])), r
        assert torch.equal(torch.isnan(dx[r]), torch.isnan(p[r])), r
    ok = [0, 1, 2, 3, 7]
    helpers.assert_close(loss[ok], want[ok].cpu().numpy(), dtype, "loss")
    helpers.assert_close(dx[ok], p[ok].cpu().numpy(), dtype, "dlogits")


# one of every launch of the kernels above: many fp32 planes (runs of 128 and 256 lanes, of 64 where planes are whole lines), 16-bit ones with blocks left over
# after the runs that stay on one XCD, more than 16 slices, 64 MiB and more of them in up to 6 slices and in 13, 7 slices and more
# of less, and few positions with up to and more than 64 entries
@pytest.mark.parametrize("dtype,outer,dim,inner", [("fp32", 1, 9, 4 * 524288 + 3), ("fp32", 1, 9, 4 * 524288), ("fp32", 2, 32, 1048577), ("bf16", 8, 21, 40961),
                                                   ("fp16", 8, 21, 40960), ("bf16", 16, 150, 8191), ("fp32", 4, 129, 8003),
                                                   ("bf16", 4, 65, 355), ("fp32", 2, 250, 203), ("fp16", 5, 256, 15),
                                                   ("bf16", 8, 21, 200001), ("fp16", 8, 100, 42001), ("bf16", 16, 60, 20001), ("fp32", 16, 60, 10001),
                                                   ("bf16", 5, 8, 4111), ("fp32", 3, 57, 5877), ("bf16", 2, 17, 8)])
def test_softmax_dim_launches(hk, cuda, dtype, outer, dim, inner):
    import torch
    dt = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}[dtype]
    gen = torch.Generator(device=cuda).manual_seed(dim * 1000003 + inner)
    guard = lambda: torch.full((outer * dim * inner + 2 * GUARD,), 7.0, dtype=dt, device=cuda)
    x, dy = (torch.randn(outer, dim, inner, generator=gen, device=cuda).to(dt) for _ in range(2))
    yb, db = guard(), guard()
    y, dx = (b[GUARD:-GUARD].view(outer, dim, inner) for b in (yb, db))
    hk.softmax_fwd(x, y, 1)
    hk.softmax_bwd(y, dy, dx, 1)
    torch.cuda.synchronize()
    assert bool((yb[:GUARD] == 7).all() and (yb[-GUARD:] == 7).all() and (db[:GUARD] == 7).all() and (db[-GUARD:] == 7).all())
    # every element against 64 bits: half a unit in the last place of the stored type (8, 11 and 24 bits), and roundings of
    # 2^-24: 12 for the exponents (arguments up to 16, half a unit of which is 16 of these, times log 2) of the element
    # and of the sum, dim additions, exp2 and the quotient; dx carries the dot product's error, dim roundings at most
    unit = {"fp32": 2.0 ** -24, "bf16": 2.0 ** -8, "fp16": 2.0 ** -11}[dtype]
    for o in range(outer):
        want = torch.softmax(x[o].double(), 0)
        assert bool(((y[o].double() - want).abs() <= want * (unit + (28 + dim) * 2.0 ** -24) + 2.0 ** -25 * (dtype == "fp16")).all()), o
        yo, do = y[o].double(), dy[o].double()
        dot = (yo * do).sum(0, keepdim=True)
        want = yo * (do - dot)
        terms = yo * (do.abs() + (yo * do.abs()).sum(0, keepdim=True))
        assert bool(((dx[o].double() - want).abs() <= want.abs() * unit + terms * (dim + 4) * 2.0 ** -24 +
                     2.0 ** -25 * (dtype == "fp16")).all()), o


@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
def test_softmax_dim_of_every_length(hk, cuda, dtype):
    """Every number of entries, with the fewest positions, some more, the most that count as few, and one more: the plans
    name kernels that are built."""
    import torch
    dt = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}[dtype]
    vec, cus = 16 // ES[dtype], torch.cuda.get_device_properties(0).multi_processor_count
    unit = {"fp32": 2.0 ** -24, "bf16": 2.0 ** -8, "fp16": 2.0 ** -11}[dtype]
    gen = torch.Generator(device=cuda).manual_seed(3)
    for dim in range(1, 257):
        for vectors in {3, 16 * cus, 16 * cus + 1, min(64 * cus, 3072 * cus // dim), min(64 * cus, 3072 * cus // dim) + 1}:
            x, dy = (torch.randn(1, dim, vectors * vec - 1, generator=gen, device=cuda).to(dt) for _ in range(2))
            y, dx = torch.empty_like(x), torch.empty_like(x)
            hk.softmax_fwd(x, y, 1)
            hk.softmax_bwd(y, dy, dx, 1)
            # against fp32: both round each of dim terms and their quotient, and the argument of the exponential (up to 16)
            # half a unit of 2^-20; dx the same of its terms
            eps = (2 * dim + 64) * 2.0 ** -24
            want = torch.softmax(x.float(), 1)
            assert bool(((y.float() - want).abs() <= want * (unit + eps) + 2.0 ** -25).all()), (dim, vectors)
            yf, df = y.float(), dy.float()
            dot = (yf * df).sum(1, keepdim=True)
            terms = yf * (df.abs() + (yf * df.abs()).sum(1, keepdim=True))
            assert bool(((dx.float() - yf * (df - dot)).abs() <= terms * (unit + eps) + 2.0 ** -25).all()), (dim, vectors)


def _norm_lengths(dtype):
    vec = 16 // ES[dtype]
    out = {v * vec + k for v in (1, 2, 8, 16, 32, 64, 65, 128, 192, 256, 300, 512, 1024) for k in (0, 1, vec - 1)}
    return sorted(out | {8192, 4097 * vec + 1})


@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("is_rms", [True, False])
def test_norm_any_length(hk, cuda, dtype, shift, is_rms):
    """Forward with a residual (in place of it, and without), backward with an upstream gradient and a second output,
    with the scratch that the library asks for and without any."""
    import torch
    eps = 1e-6
    for cols in _norm_lengths(dtype):
        rows = 37 if cols < 3000 else 5
        pitch = cols + (0 if shift == 0 else 5)
        x0, res, dz, dxin = (helpers.draw(s + cols, (rows, cols), dtype=dtype) for s in (100, 200, 300, 400))
        gamma = helpers.draw(500 + cols, (cols,), "uniform", 0.5, 1.5, dtype)
        beta = None if is_rms else helpers.draw(600 + cols, (cols,), "normal", 0.0, 0.1, dtype)
        place = lambda a, fill=None: _placed(cuda, a, dtype, shift, pitch, fill)
        vector = lambda a: None if a is None else _placed(cuda, a[None], dtype, shift, cols)[1][0]
        tg, tb = vector(gamma), vector(beta)
        tx0, tres = place(x0)[1], place(res)[1]
        zb, tz = place(x0, 0.0)
        xb, tx = place(x0, 0.0)
        tmu, trs = torch.empty(rows, device=cuda), torch.empty(rows, device=cuda)
        hk.dropout_add_ln_fwd(tx0, tres, tg, tb, tz, tx, tmu, trs, eps, is_rms)
        torch.cuda.synchronize()
        ez, ex, emu, ers = oracle.dropout_add_ln_fwd(x0, res, gamma, beta, eps, is_rms)
        helpers.assert_close(tz.contiguous(), ez, dtype, "z %d" % cols)
        helpers.assert_close(tx.contiguous(), ex, dtype, "x %d" % cols)
        helpers.assert_close(trs, ers, "fp32", "rsigma %d" % cols)
        helpers.assert_close(tmu, emu, "fp32", "mu %d" % cols, scale=1.0)
        assert _guards_untouched(zb, tz) and _guards_untouched(xb, tx), cols
        z2b, z2 = place(x0, 0.0)
        hk.dropout_add_ln_fwd(tx0, tres, tg, tb, z2, tres, tmu, trs, eps, is_rms)     # the sum in place of the residual
        torch.cuda.synchronize()
        assert torch.equal(z2.contiguous(), tz.contiguous()) and torch.equal(tres.contiguous(), tx.contiguous()), cols
        hk.dropout_add_ln_fwd(tx, None, tg, tb, z2, None, tmu, trs, eps, is_rms)      # no residual
        torch.cuda.synchronize()
        x = helpers.to_numpy(tx.contiguous())
        ez, _, _, _ = oracle.dropout_add_ln_fwd(x, None, gamma, beta, eps, is_rms)
        helpers.assert_close(z2.contiguous(), ez, dtype, "z %d" % cols)

        mu32, rs32 = helpers.to_numpy(tmu), helpers.to_numpy(trs)
        edx, edg, edb = oracle.dropout_add_ln_bwd(dz, dxin, x, mu32, rs32, gamma, is_rms)
        tdz, tdxin = place(dz)[1], place(dxin)[1]
        for workspace in (None, torch.empty(1, device=cuda)) if cols % (16 // ES[dtype]) or shift else (None,):
            db, dx = place(x0, 0.0)
            rb, dr = place(x0, 0.0)
            (gb, dg), (bb, dbeta) = (_placed(cuda, gamma[None], dtype, shift, cols, 0.0) for _ in range(2))
            hk.dropout_add_ln_bwd(tdz, tdxin, tx, tmu, trs, tg, dx, dr, dg[0], dbeta[0], is_rms, workspace=workspace)
            torch.cuda.synchronize()
            what = "%d %s" % (cols, workspace is None)
            helpers.assert_close(dx.contiguous(), edx, dtype, "dx0 " + what)
            assert torch.equal(dr.contiguous(), dx.contiguous())
            helpers.assert_close(dg[0].contiguous(), edg, dtype, "dgamma " + what)
            helpers.assert_close(dbeta[0].contiguous(), edb, dtype, "dbeta " + what)
            for b, v in ((db, dx), (rb, dr), (gb, dg), (bb, dbeta)):
                assert _guards_untouched(b, v), what
        # in place of the upstream gradient
        hk.dropout_add_ln_bwd(tdz, tdxin, tx, tmu, trs, tg, tdxin, None, None, None, is_rms)
        torch.cuda.synchronize()
        helpers.assert_close(tdxin.contiguous(), edx, dtype, "dx0 %d" % cols)


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("cols", [9, 67, 1021, 3001, 8191])
def test_layer_norm_bwd_any_length_modes(hk, cuda, dtype, cols):
    """The plain backward from (mean, variance) in the data type, and the one that rebuilds x_hat from the output."""
    import torch
    rows, eps = 300, 1e-5
    x, dy = (helpers.draw(s + cols, (rows, cols), dtype=dtype) for s in (700, 800))
    gamma = helpers.draw(900 + cols, (cols,), "uniform", 0.5, 1.5, dtype)
    beta = helpers.draw(950 + cols, (cols,), "normal", 0.0, 0.1, dtype)
    y64, mean, var, rstd = oracle.layernorm_fwd(x, gamma, beta, eps)
    tx, tg, tb, tdy = (helpers.to_torch(v, dtype, cuda) for v in (x, gamma, beta, dy))
    tdx, tdg, tdb = torch.empty_like(tx), torch.empty_like(tg), torch.empty_like(tg)
    # sums over 300 rows: their rounding error is that of the terms
    many = float(np.sqrt(rows))
    mean_s, var_s = oracle.round_to(mean, dtype), oracle.round_to(var, dtype)
    edx, edg, edb = oracle.layernorm_bwd(dy, x, gamma, mean_s, 1.0 / np.sqrt(var_s.astype(np.float64) + eps), eps)
    hk.layer_norm_bwd(tdy, tx, tg, tb, helpers.to_torch(mean_s, dtype, cuda), helpers.to_torch(var_s, dtype, cuda), tdx,
                      tdg, tdb, eps, stat_kind=0)
    torch.cuda.synchronize()
    for got, want, what in ((tdx, edx, "dx"), (tdg, edg, "dgamma"), (tdb, edb, "dbeta")):
        helpers.assert_close(got, want, dtype, what, scale=None if what == "dx" else many)
    y, rstd32 = oracle.round_to(y64, dtype), rstd.astype(np.float32)
    edx, edg, edb = oracle.layernorm_bwd_memeff(dy, y, gamma, beta, rstd32, eps)
    hk.layer_norm_bwd(tdy, helpers.to_torch(y, dtype, cuda), tg, tb, None, helpers.to_torch(rstd32, "fp32", cuda), tdx,
                      tdg, tdb, eps, memory_efficient=True)
    torch.cuda.synchronize()
    for got, want, what in ((tdx, edx, "dx"), (tdg, edg, "dgamma"), (tdb, edb, "dbeta")):
        helpers.assert_close(got, want, dtype, what, scale=None if what == "dx" else many)


@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("is_rms", [True, False])
@pytest.mark.parametrize("shift", [0, 1])
def test_norm_bwd_without_options(hk, cuda, dtype, is_rms, shift):
    """Several rows to a wavefront (short rows, more of them than one step of the other kernels' workgroups takes) at
    the edges of a lane group, and the longer rows' folds of one, several and many groups, dx in place of dz."""
    import torch
    vec, many_rows = 16 // ES[dtype], torch.cuda.get_device_properties(0).multi_processor_count * 16
    shapes = [(many_rows + k, v * vec + j) for k, v in ((1, 1), (300, 15), (77, 16), (1, 17), (33, 31))
              for j in (0, 1, vec - 1)] + [(many_rows, 9 * vec + 1), (many_rows + 1, 32 * vec), (3 * many_rows, 8 * vec + 3)] + \
             [(1, 3 * vec), (600, 40 * vec + 1), (900, 128 * vec), (513, 129 * vec + 3), (300, 300 * vec + 1)]
    for rows, cols in shapes:
        pitch = cols + (0 if shift == 0 else 5)
        x, dz = (helpers.draw(s + cols, (rows, cols), dtype=dtype) for s in (1100, 1200))
        gamma = helpers.draw(1300 + cols, (cols,), "uniform", 0.5, 1.5, dtype)
        mean = None if is_rms else x.astype(np.float64).mean(-1).astype(np.float32)
        centred = x.astype(np.float64) - (0 if is_rms else mean[:, None])
        rs = (1.0 / np.sqrt(np.square(centred).mean(-1) + 1e-5)).astype(np.float32)
        edx, edg, edb = oracle.dropout_add_ln_bwd(dz, None, x, np.zeros_like(rs) if is_rms else mean, rs, gamma, is_rms)
        tx = _placed(cuda, x, dtype, shift, pitch)[1]
        zb, tz = _placed(cuda, dz, dtype, shift, pitch)
        tg = _placed(cuda, gamma[None], dtype, shift, cols)[1][0]
        (gb, dg), (bb, db) = (_placed(cuda, gamma[None], dtype, shift, cols, 0.0) for _ in range(2))
        tmean = None if is_rms else helpers.to_torch(mean, "fp32", cuda)
        hk.dropout_add_ln_bwd(tz, None, tx, tmean, helpers.to_torch(rs, "fp32", cuda), tg, tz, None, dg[0],
                              None if is_rms else db[0], is_rms)
        torch.cuda.synchronize()
        what = "%d x %d" % (rows, cols)
        helpers.assert_close(tz.contiguous(), edx, dtype, "dx0 " + what)
        # column sums over `rows` terms: their rounding error is that of the terms
        helpers.assert_close(dg[0].contiguous(), edg, dtype, "dgamma " + what, scale=float(np.sqrt(rows)))
        if not is_rms:
            helpers.assert_close(db[0].contiguous(), edb, dtype, "dbeta " + what, scale=float(np.sqrt(rows)))
        for b, v in ((zb, tz), (gb, dg), (bb, db)):
            assert _guards_untouched(b, v), what


def _highest_rows(torch, cuda, seed, cols, dt):
    """Six rows: one element of the type's highest value, two of them, all of them, one above a second highest, highest
    beside lowest, and +inf beside the highest.  softmax is 1 / count at the row's maximum but for the last, all NaN."""
    x = torch.from_numpy(helpers.draw(seed, (6, cols))).to(dt).to(cuda)
    high = torch.finfo(dt).max
    x[0, cols // 2] = high
    x[1, 0] = x[1, cols - 1] = high
    x[2, :] = high
    x[3, :] = high / 1.25
    x[3, 1] = high
    x[4, :] = -high
    x[4, cols - 2] = high
    x[5, :] = high
    x[5, 1] = float("inf")
    return x


# rows that some lanes of a wavefront, a wavefront and a workgroup hold, whole vectors and ragged ones
@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("cols", [3, 40, 41, 130, 1001, 2047, 2048, 4097, 9000])
def test_softmax_of_highest_values(hk, cuda, dtype, cols):
    """Finite scores whose product with log2(e) is past fp32."""
    import torch
    dt = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}[dtype]
    x = _highest_rows(torch, cuda, 9100 + cols, cols, dt)
    y = torch.empty_like(x)
    hk.softmax_fwd(x, y)
    torch.cuda.synchronize()
    want = torch.softmax(x.double(), -1)
    assert bool(torch.isnan(y[5]).all()) and bool(torch.isnan(want[5]).all())
    helpers.assert_close(y[:5], want[:5].cpu().numpy(), dtype, "softmax y")
    hk.softmax_fwd(x, x)
    torch.cuda.synchronize()
    assert torch.equal(x[:5], y[:5])


@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("dim,inner", [(3, 9), (21, 8), (21, 67), (150, 40), (256, 33), (257, 9)])
def test_softmax_of_highest_values_over_a_leading_dimension(hk, cuda, dtype, dim, inner):
    """The rows above as columns, ordinary ones between them."""
    import torch
    dt = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}[dtype]
    x = torch.from_numpy(helpers.draw(9200 + dim, (2, dim, inner))).to(dt).to(cuda)
    x[1, :, :6] = _highest_rows(torch, cuda, 9300 + dim, dim, dt).t()
    y = torch.empty_like(x)
    hk.softmax_fwd(x, y, 1)
    torch.cuda.synchronize()
    want = torch.softmax(x.double(), 1)
    assert torch.equal(torch.isnan(y), torch.isnan(want))
    helpers.assert_close(y.nan_to_num(), want.nan_to_num().cpu().numpy(), dtype, "softmax y")


# a wavefront's and a workgroup's rows, 16-bit rows kept packed, streamed ones; whole vectors and ragged ones
@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("cols", [40, 41, 1001, 4096, 40001, 50257, 70001])
def test_cross_entropy_of_highest_values(hk, cuda, dtype, cols):
    import torch
    dt = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}[dtype]
    x = _highest_rows(torch, cuda, 8100 + cols, cols, dt)
    lab = torch.tensor([cols // 2, cols - 1, 7, 1, cols - 2, 0], device=cuda)
    g = torch.ones(6, dtype=dt, device=cuda)
    loss, dx = torch.empty(6, dtype=dt, device=cuda), torch.empty_like(x)
    stats = torch.empty(3, 6, device=cuda)
    hk.sce_sparse_fwd(x, lab, loss, -100)
    hk.sce_sparse_bwd(x, lab, g, dx, -100)
    hk.vocab_parallel_ce_stats(x, lab, stats, 0, -100)
    torch.cuda.synchronize()
    p = torch.softmax(x.double(), -1)
    want = torch.nn.functional.cross_entropy(x.double(), lab, reduction="none")
    p[torch.arange(6, device=cuda), lab] -= 1
    assert bool(torch.isnan(loss[5])) and bool(torch.isnan(dx[5]).all()) and bool(torch.isnan(stats[1, 5]))
    helpers.assert_close(loss[:5], want[:5].cpu().numpy(), dtype, "loss")
    helpers.assert_close(dx[:5], p[:5].cpu().numpy(), dtype, "dlogits")
    top = x[:5].double().max(-1).values
    assert torch.equal(stats[0, :5].double(), top)
    helpers.assert_close(stats[1, :5], (x[:5].double() - top[:, None]).exp().sum(-1).cpu().numpy(), "fp32", "stats")


@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("is_rms", [True, False])
def test_pre_norm_sum_without_a_residual(hk, cuda, dtype, shift, is_rms):
    """x_out is written whether a residual is added or not: then it is the input, in a buffer of its own and in place."""
    import torch
    eps = 1e-6
    for cols in (3, 40, 41, 256, 520, 1021, 4096, 4099, 40000):
        rows, pitch = 5, cols + (0 if shift == 0 else 5)
        x0 = helpers.draw(150 + cols, (rows, cols), dtype=dtype)
        gamma = helpers.draw(550 + cols, (cols,), "uniform", 0.5, 1.5, dtype)
        place = lambda a, fill=None: _placed(cuda, a, dtype, shift, pitch, fill)
        tg = helpers.to_torch(gamma, dtype, cuda)
        _, tx0 = place(x0)
        zb, tz = place(x0, 0.0)
        xb, tx = place(x0, 0.0)
        mu, rs = torch.empty(rows, device=cuda), torch.empty(rows, device=cuda)
        hk.dropout_add_ln_fwd(tx0, None, tg, None, tz, tx, mu, rs, eps, is_rms)
        torch.cuda.synchronize()
        assert torch.equal(tx.contiguous(), tx0.contiguous()), cols
        helpers.assert_close(tz.contiguous(), oracle.dropout_add_ln_fwd(x0, None, gamma, None, eps, is_rms)[0], dtype,
                             "z %d" % cols)
        assert _guards_untouched(zb, tz) and _guards_untouched(xb, tx), cols
        z2, before = torch.empty_like(tz.contiguous()), tx0.clone()
        hk.dropout_add_ln_fwd(tx0, None, tg, None, z2, tx0, mu, rs, eps, is_rms)
        torch.cuda.synchronize()
        assert torch.equal(tx0.contiguous(), before) and torch.equal(z2, tz.contiguous()), cols


@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
def test_rows_that_need_no_scratch(hk, cuda, dtype):
    """A row of the most whole vectors that one workgroup takes, and a partial one more, on the 16-byte grid."""
    import torch
    dt = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}[dtype]
    vec = 16 // ES[dtype]
    for cols in [32768 * vec + k for k in range(vec)]:
        a = np.random.default_rng(cols).integers(-3, 4, cols)
        x, out = torch.from_numpy(a).to(dt).to(cuda), torch.empty(1, dtype=dt, device=cuda)
        assert hk.reduce_workspace_bytes(hk.dtype_code(x), [cols], [1], [0]) == 0, cols
        hk.reduce(x, out, [0], "sum", workspace=torch.empty(1, device=cuda))
        torch.cuda.synchronize()
        assert float(out) == float(oracle.round_to(np.asarray([a.sum()], np.float32), dtype)[0]), cols


# a wavefront's rows, a workgroup's, rows kept packed (16-bit) and streamed ones, whole vectors and ragged
@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("cols", [5, 40, 41, 1031, 4096, 40001, 70001])
def test_cross_entropy_gradient_at_every_edge_column(hk, cuda, dtype, shift, cols):
    """Equal logits, the label on each of the first and last 20 columns: 1 / cols, less one at the label and nowhere else."""
    import torch
    dt = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}[dtype]
    lab = torch.tensor(sorted(set(range(min(cols, 20))) | set(range(max(cols - 20, 0), cols))), device=cuda)
    rows = len(lab)
    pitch = cols + (0 if shift == 0 else 5)
    _, x = _placed(cuda, np.zeros((rows, cols), np.float32), dtype, shift, pitch)
    db, dx = _placed(cuda, np.zeros((rows, cols), np.float32), dtype, shift, pitch, 3.0)
    hk.sce_sparse_bwd(x, lab, torch.ones(rows, dtype=dt, device=cuda), dx, -100)
    torch.cuda.synchronize()
    want = np.full((rows, cols), 1.0 / cols)
    want[np.arange(rows), lab.cpu().numpy()] -= 1.0
    helpers.assert_close(dx.contiguous(), want, dtype, "dlogits")
    assert _guards_untouched(db, dx)


@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("cols", [5, 40, 41, 1001, 4096, 40001, 70001])
def test_shard_statistics_keep_a_nan(hk, cuda, dtype, cols):
    """A column shard of nothing but -inf adds nothing to the row's sum; one that holds a NaN as well, or nothing else,
    makes it NaN."""
    import torch
    dt = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}[dtype]
    x = torch.full((3, cols), -float("inf"), dtype=dt, device=cuda)
    x[1, cols // 2] = float("nan")
    x[2, :] = float("nan")
    stats = torch.full((3, 3), 7.0, device=cuda)
    hk.vocab_parallel_ce_stats(x, torch.zeros(3, dtype=torch.int64, device=cuda), stats, 0, -100)
    torch.cuda.synchronize()
    assert float(stats[1, 0]) == 0.0 and bool(torch.isnan(stats[1, 1:]).all()), stats


# 16-bit rows with a part in LDS: the most vectors of four and two rows per compute unit (6592, 12224) and of a
# gradient row with exponentials in registers (8128), one more each, and the first rows past registers alone (4097)
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("vectors", [4097, 4160, 6592, 6593, 8128, 8129, 8448, 8449, 12224, 12225])
def test_cross_entropy_rows_with_a_tail(hk, cuda, dtype, shift, vectors):
    import torch
    rows = 5
    for cols in (8 * vectors, 8 * vectors - 7):
        pitch = cols + (0 if shift == 0 else 5)
        x = helpers.draw(9100 + cols, (rows, cols), dtype=dtype)
        _, tx = _placed(cuda, x, dtype, shift, pitch)
        lab = torch.tensor([0, cols - 1, -100, 32768, cols - 9], device=cuda)     # the first and last column, one in the tail
        g = torch.tensor([1.0, -2.0, 3.0, 0.5, 1.5], dtype=tx.dtype, device=cuda)
        loss = torch.empty(rows, dtype=tx.dtype, device=cuda)
        db, dx = _placed(cuda, x, dtype, shift, pitch, 3.0)
        hk.sce_sparse_fwd(tx, lab, loss, -100)
        hk.sce_sparse_bwd(tx, lab, g, dx, -100)
        torch.cuda.synchronize()
        p = torch.softmax(tx.double(), -1)
        want = torch.logsumexp(tx.double(), -1) - tx.double().gather(1, lab.clamp(min=0)[:, None])[:, 0]
        p[torch.arange(rows, device=cuda), lab.clamp(min=0)] -= 1
        want[2] = 0
        p[2] = 0
        helpers.assert_close(loss, want.cpu().numpy(), dtype, "loss %d" % cols)
        helpers.assert_close(dx.contiguous(), (p * g.double()[:, None]).cpu().numpy(), dtype, "dlogits %d" % cols)
        assert _guards_untouched(db, dx), cols
        hk.sce_sparse_bwd(tx, lab, g, tx, -100)     # in place
        torch.cuda.synchronize()
        assert torch.equal(tx.contiguous(), dx.contiguous()), cols


# the same in as many rows as take a plan of their own: more than two and than four per compute unit, three rows' longest and one
# vector more, past registers, the longest and one more
@pytest.mark.parametrize("vectors", [6593, 7680, 7681, 8192, 8193, 12224, 12225])
def test_cross_entropy_of_many_rows_with_a_tail(hk, cuda, vectors):
    import torch
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    cols = 8 * vectors - 3
    x = helpers.to_torch(helpers.draw(9150 + cols, (5, cols), dtype="bf16"), "bf16", cuda)
    lab = torch.tensor([0, cols - 1, -100, 32768, cols - 9], device=cuda)
    want = torch.logsumexp(x.double(), -1) - x.double().gather(1, lab.clamp(min=0)[:, None])[:, 0]
    want[2] = 0
    for times in (2 * cus // 5, 2 * cus // 5 + 1, 4 * cus // 5 + 1):
        loss = torch.full((5 * times,), 5.0, dtype=torch.bfloat16, device=cuda)
        hk.sce_sparse_fwd(x.repeat(times, 1), lab.repeat(times), loss, -100)
        torch.cuda.synchronize()
        loss = loss.view(times, 5)
        helpers.assert_close(loss[0], want.cpu().numpy(), "bf16", "loss %d" % times)
        assert torch.equal(loss, loss[:1].expand(times, 5)), times


# operands whose rows start on different boundaries: x on even ones, on odd ones, on both in turn (an odd pitch), the others
# the other way round; one vector, the edges of a lane group's and of a wavefront's shares, a workgroup
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("x_at,other_at", [((0, 6), (1, 6)), ((1, 6), (0, 6)), ((0, 5), (1, 5)), ((1, 5), (0, 6)), ((0, 6), (0, 5))])
def test_rows_on_different_boundaries(hk, cuda, dtype, x_at, other_at):
    import torch
    rows = 21
    for cols in (8, 9, 15, 16, 17, 63, 64, 65, 128, 257, 512, 519, 1024, 2047, 2048, 2055, 4096, 8190):
        x, dy = (helpers.draw(s + cols, (rows, cols), dtype=dtype) for s in (9500, 9600))
        at = lambda a, where, fill=None: _placed(cuda, a, dtype, where[0], cols + where[1], fill)
        tx = at(x, x_at)[1]
        yb, ty = at(x, other_at, 0.0)
        hk.softmax_fwd(tx, ty)
        tdy = at(dy, other_at)[1]
        yx = at(x, x_at)[1]
        yx.copy_(ty)
        db, dx = at(x, other_at, 0.0)
        hk.softmax_bwd(yx, tdy, dx)
        torch.cuda.synchronize()
        assert _guards_untouched(yb, ty) and _guards_untouched(db, dx), cols
        helpers.assert_close(ty.contiguous(), oracle.softmax_fwd(x), dtype, "softmax y %d" % cols)
        y = helpers.to_numpy(ty.contiguous())
        helpers.assert_close(dx.contiguous(), oracle.softmax_bwd(y, dy), dtype, "softmax dx %d" % cols,
                             scale=float(np.sqrt(np.mean(np.square(y * dy)))),
                             ordinary_rtol=helpers.SOFTMAX_GRADIENT_ORDINARY_RTOL)
        gamma = helpers.draw(9700 + cols, (cols,), "uniform", 0.5, 1.5, dtype)
        tg = _placed(cuda, gamma[None], dtype, other_at[0], cols)[1][0]
        for is_rms in (True, False):
            zb, tz = at(x, other_at, 0.0)
            xb, tsum = at(x, x_at, 0.0)
            mu, rs = torch.empty(rows, device=cuda), torch.empty(rows, device=cuda)
            hk.dropout_add_ln_fwd(tx, tdy, tg, None, tz, tsum, mu, rs, 1e-6, is_rms)
            torch.cuda.synchronize()
            ez, ex, _, ers = oracle.dropout_add_ln_fwd(x, dy, gamma, None, 1e-6, is_rms)
            helpers.assert_close(tz.contiguous(), ez, dtype, "z %d" % cols)
            helpers.assert_close(tsum.contiguous(), ex, dtype, "x %d" % cols)
            helpers.assert_close(rs, ers, "fp32", "rsigma %d" % cols)
            assert _guards_untouched(zb, tz) and _guards_untouched(xb, tsum), cols


# whole vectors that start on odd boundaries, where a start one element earlier needs a vector more: rows with lanes to spare
# for it and without, a wavefront's longest (few rows and many), workgroups, and the most that a workgroup holds
@pytest.mark.parametrize("rows,cols", [(33, 64), (33, 192), (33, 512), (9, 2048), (1100, 2048), (9, 4096), (7, 8192), (600, 8192),
                                       (5, 12288), (5, 16384), (3, 24576), (3, 32768), (3, 40960), (3, 65536)])
@pytest.mark.parametrize("pitch", [1, 8])
def test_whole_vectors_on_odd_boundaries(hk, cuda, rows, cols, pitch):
    import torch
    x, dy = (helpers.draw(s + cols + rows, (rows, cols), dtype="bf16") for s in (9800, 9900))
    at = lambda a, fill=None: _placed(cuda, a, "bf16", 1, cols + pitch, fill)
    tx, tdy = at(x)[1], at(dy)[1]
    yb, ty = at(x, 0.0)
    db, dx = at(x, 0.0)
    hk.softmax_fwd(tx, ty)
    hk.softmax_bwd(ty, tdy, dx)
    torch.cuda.synchronize()
    assert _guards_untouched(yb, ty) and _guards_untouched(db, dx)
    helpers.assert_close(ty.contiguous(), torch.softmax(tx.double(), -1).cpu().numpy(), "bf16", "softmax y")
    yd, dd = ty.double(), tdy.double()
    helpers.assert_close(dx.contiguous(), (yd * (dd - (yd * dd).sum(-1, keepdim=True))).cpu().numpy(), "bf16", "softmax dx",
                         scale=float((yd * dd).square().mean().sqrt()))
    g, b = (helpers.to_torch(helpers.draw(s, (cols,), "uniform", 0.5, 1.5, "bf16"), "bf16", cuda) for s in (9701, 9702))
    xd = tx.double()
    mean, var = xd.mean(-1, keepdim=True), xd.var(-1, unbiased=False, keepdim=True)
    mu, rs = torch.empty(rows, device=cuda), torch.empty(rows, device=cuda)
    zb, tz = at(x, 0.0)
    hk.layer_norm_fwd(tx, g, b, tz, mu, rs, 1e-5)
    torch.cuda.synchronize()
    helpers.assert_close(tz.contiguous(), ((xd - mean) / (var + 1e-5).sqrt() * g.double() + b.double()).cpu().numpy(), "bf16", "z")
    helpers.assert_close(rs, (1 / (var + 1e-5).sqrt())[:, 0].cpu().numpy(), "fp32", "rsigma")
    assert _guards_untouched(zb, tz)
    zb, tz = at(x, 0.0)
    hk.dropout_add_ln_fwd(tx, None, g, None, tz, None, mu, rs, 1e-5, True)
    torch.cuda.synchronize()
    want = 1 / (xd.square().mean(-1, keepdim=True) + 1e-5).sqrt()
    helpers.assert_close(tz.contiguous(), (xd * want * g.double()).cpu().numpy(), "bf16", "z")
    helpers.assert_close(rs, want[:, 0].cpu().numpy(), "fp32", "rsigma")
    assert _guards_untouched(zb, tz)


@pytest.mark.parametrize("what,rows,cols", [("softmax_bwd", 256, 32768), ("softmax_fwd", 256, 65536), ("layer_norm", 256, 65536),
                                            ("rms_norm", 256, 65536), ("layer_norm", 40000, 256), ("rms_norm", 40000, 256)])
def test_whole_vectors_on_odd_boundaries_cost_no_more(hk, cuda, what, rows, cols):
    """A row of whole vectors against the row one vector shorter, which has one to spare: it took 1.6 times as long, and 8 to 17
    times where the vector more did not fit a workgroup.  Without the shift a gradient's accesses lie off 4 bytes, for which it takes 1.33 times as long (11.5 against 8.6 us at 256 x 32768); the others take the same time."""
    import torch

    def time_of(n, calls=20):
        x, y, z = (torch.randn(rows * (n + 1) + 1, device=cuda).bfloat16()[1:].view(rows, n + 1)[:, :n] for _ in range(3))
        g, m, r = torch.ones(n, device=cuda).bfloat16(), torch.empty(rows, device=cuda), torch.empty(rows, device=cuda)
        run = {"softmax_fwd": lambda: hk.softmax_fwd(x, y), "softmax_bwd": lambda: hk.softmax_bwd(x, y, z),
               "layer_norm": lambda: hk.layer_norm_fwd(x, g, g, y, m, r, 1e-5),
               "rms_norm": lambda: hk.dropout_add_ln_fwd(x, None, g, None, y, None, m, r, 1e-5, True)}[what]
        best = 1e9
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            run()
            a.record()
            for _ in range(calls):
                run()
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b) * 1e3 / calls)
        return best

    for _ in range(5):   # (a time that something else lengthened is taken again)
        whole, shorter = time_of(cols), time_of(cols - 8)
        if whole < 1.5 * shorter:
            break
    assert whole < 1.5 * shorter, (whole, shorter)
