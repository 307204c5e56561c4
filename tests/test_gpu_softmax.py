"""GPU parity of Softmax forward / backward against the oracle (hk_softmax_*)."""
import numpy as np
import pytest

import helpers
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("shape,dim", [((7, 64), -1), ((3, 5, 2048), -1), ((33, 1000), 1), ((4, 7), -1),
                                       ((2, 3, 4096), 2), ((2, 20000), -1), ((1, 70000), -1),
                                       ((4, 6, 10), 1), ((5, 33, 7, 3), 1), ((16, 8), 0)])
def test_softmax_fwd_bwd(hk, cuda, dtype, shape, dim):
    import torch
    x = helpers.draw(201, shape, "normal", 0.0, 3.0, dtype)
    ey = oracle.softmax_fwd(x, dim)
    tx = helpers.to_torch(x, dtype, cuda)
    ty = torch.empty_like(tx)
    hk.softmax_fwd(tx, ty, dim)
    torch.cuda.synchronize()
    helpers.assert_close(ty, ey, dtype, "y")
    sums = ty.float().sum(dim % len(shape)).cpu().numpy()
    assert np.max(np.abs(sums - 1.0)) <= (2e-2 if dtype != "fp32" else 1e-5)

    y = helpers.to_numpy(ty)                      # backward consumes the stored y
    dy = helpers.draw(202, shape, dtype=dtype)
    edx = oracle.softmax_bwd(y, dy, dim)
    tdy = helpers.to_torch(dy, dtype, cuda)
    tdx = torch.empty_like(tx)
    hk.softmax_bwd(ty, tdy, tdx, dim)
    torch.cuda.synchronize()
    helpers.assert_close(tdx, edx, dtype, "dx", ordinary_rtol=helpers.SOFTMAX_GRADIENT_ORDINARY_RTOL)


def test_softmax_special_rows(hk, cuda):
    import torch
    cols = 2048
    x = np.zeros((4, cols), dtype=np.float32)
    x[0, :] = 5.0                       # all equal -> uniform
    x[1, :] = -np.inf; x[1, 17] = 0.0   # one finite logit -> one-hot
    x[2, :] = -80.0; x[2, 5] = 80.0     # dominant logit
    x[3, :] = helpers.draw(9, (cols,)) + 1000.0   # large common offset
    tx = helpers.to_torch(x, "fp32", cuda)
    ty = torch.empty_like(tx)
    hk.softmax_fwd(tx, ty)
    torch.cuda.synchronize()
    y = ty.cpu().numpy()
    assert np.allclose(y[0], 1.0 / cols, rtol=1e-6)
    assert y[1, 17] == 1.0 and y[1].sum() == 1.0
    assert y[2, 5] == 1.0 and y[2].sum() == 1.0
    ref = oracle.softmax_fwd(x[3][None, :])[0]
    assert np.max(np.abs(y[3] - ref)) <= 1e-5 * ref.max()


def test_softmax_full_size_bf16(hk, cuda):
    """[4, 32, 2048, 2048] bf16: GPU on everything, oracle on sampled rows."""
    import torch
    g = torch.Generator(device="cpu").manual_seed(201)
    shape = (4, 32, 2048, 2048)
    tx = (torch.randn(shape, generator=g, dtype=torch.float32) * 3.0).to(torch.bfloat16).to(cuda)
    ty = torch.empty_like(tx)
    hk.softmax_fwd(tx, ty)
    tdy = torch.randn(shape, generator=g, dtype=torch.float32).to(torch.bfloat16).to(cuda)
    tdx = torch.empty_like(tx)
    hk.softmax_bwd(ty, tdy, tdx)
    torch.cuda.synchronize()
    rows = 4 * 32 * 2048
    sel = torch.from_numpy(helpers.sample_rows(3, rows, 64)).to(cuda)
    x2, y2, dy2, dx2 = (t.view(rows, 2048)[sel] for t in (tx, ty, tdy, tdx))
    ey = oracle.softmax_fwd(helpers.to_numpy(x2))
    helpers.assert_close(y2, ey, "bf16", "y")
    edx = oracle.softmax_bwd(helpers.to_numpy(y2), helpers.to_numpy(dy2))
    helpers.assert_close(dx2, edx, "bf16", "dx")
    # size-independent properties on the whole tensor
    s = ty.view(rows, 2048).float().sum(1)
    assert float((s - 1).abs().max()) <= 2e-2
    assert float(tdx.view(rows, 2048).float().sum(1).abs().max()) <= 5e-2


# planes and positions on either side of the launches' limits
@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("shape", [(16384, 5, 8), (16385, 5, 8), (20000, 3, 12), (20000, 3, 16), (5000, 3, 28), (5000, 3, 32),
                                   (2674, 4, 49), (2675, 4, 49), (2674, 5, 49), (40, 2, 9),
                                   (6145, 3, 8), (131, 4, 1000), (132, 4, 1000)])
def test_short_and_narrow_planes(hk, cuda, dtype, shape):
    import torch
    x, dy = (helpers.to_torch(helpers.draw(40 + k, shape, dtype=dtype), dtype, cuda) for k in range(2))
    y, dx = torch.empty_like(x), torch.empty_like(x)
    hk.softmax_fwd(x, y, 1)
    hk.softmax_bwd(y, dy, dx, 1)
    torch.cuda.synchronize()
    helpers.assert_close(y, torch.softmax(x.double(), 1).cpu().numpy(), dtype, "y")
    yd = y.double()
    want = yd * (dy.double() - (yd * dy.double()).sum(1, keepdim=True))
    # dx = y (dy - sum y dy): seven roundings (2^-24) of terms of up to three times their rms stay after the difference
    # cancelled to the 1e-3 rms from which the strict figure counts, 1.3e-3 of it in fp32
    helpers.assert_close(dx, want.cpu().numpy(), dtype, "dx", scale=float((yd * dy.double()).square().mean().sqrt()),
                         ordinary_rtol=helpers.SOFTMAX_GRADIENT_ORDINARY_RTOL,
                         strict_rtol=helpers.SOFTMAX_GRADIENT_STRICT_RTOL if dtype == "fp32" else None)


def test_short_planes_cost_their_bytes(hk, cuda):
    """The same array as planes of 8 and of 64 positions: one thread per position takes 3.4 (backward 2.2) times as long for
    the short ones, whose every vector has a cache line to itself; vectors of neighbouring positions took 6.8 (6.4)."""
    import torch

    def replay_time(shape, calls=10):
        x, y, dx = (torch.rand(shape, device=cuda).bfloat16() for _ in range(3))
        times = []
        for fn in (lambda: hk.softmax_fwd(x, y, 1), lambda: hk.softmax_bwd(y, x, dx, 1)):
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                fn()
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                for _ in range(calls):
                    fn()
            best = 1e9
            for _ in range(5):
                a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                a.record()
                graph.replay()
                b.record()
                torch.cuda.synchronize()
                best = min(best, a.elapsed_time(b) * 1e3 / calls)
            times.append(best)
        return times

    short, long = replay_time((32000, 64, 8)), replay_time((4000, 64, 64))
    assert short[0] < 5 * long[0] and short[1] < 4 * long[1], (short, long)


@pytest.mark.parametrize("width", [1, 8, 24, 40, 64, 100, 256])
@pytest.mark.parametrize("cols", [64, 256, 1024, 2048, 4096])
def test_forced_widths(hk, cuda, width, cols):
    """Any width may be asked for, on rows of one level and of two: it is rounded to one that exists."""
    import torch
    x = helpers.draw(50 + cols, (6, 4, cols), dtype="bf16")
    base = helpers.to_torch(x, "bf16", cuda)
    y, y2 = torch.empty_like(base), torch.empty(4, 6, cols, dtype=base.dtype, device=cuda)
    hk.tune_set("softmax_threads", width)
    try:
        hk.softmax_fwd(base, y)
        hk.softmax_fwd(base.transpose(0, 1), y2)
        torch.cuda.synchronize()
    finally:
        hk.tune_set("softmax_threads", 0)
    want = torch.softmax(base.double(), -1)
    helpers.assert_close(y, want.cpu().numpy(), "bf16", "y")
    helpers.assert_close(y2, want.transpose(0, 1).contiguous().cpu().numpy(), "bf16", "y of a view")


@pytest.mark.parametrize("dtype,shape", [
    # slices of 4 to 16 entries, in runs of half and of a quarter of a wavefront's vectors, whole and odd planes, streamed
    # and through the cache, elements formed again or kept: the edges of the rules on entries and on the array's bytes
    ("bf16", (68, 32, 2048)), ("bf16", (70, 33, 1984)), ("fp16", (33, 48, 4099)), ("bf16", (33, 49, 4099)),
    ("bf16", (34, 80, 4096)), ("fp16", (34, 81, 4100)), ("bf16", (32, 96, 4224)), ("bf16", (9, 97, 16383)),
    ("bf16", (60, 112, 4601)), ("bf16", (60, 128, 4608)), ("fp16", (9, 129, 8185)), ("bf16", (7, 160, 12001)),
    ("bf16", (6, 161, 8192)), ("fp16", (6, 192, 8190)), ("bf16", (5, 193, 8192)), ("bf16", (6, 208, 21001)),
    ("bf16", (4, 224, 8777)), ("fp16", (4, 225, 8192)), ("bf16", (3, 256, 11001)), ("bf16", (20, 256, 4992)),
    ("bf16", (6, 26, 90001)), ("bf16", (6, 40, 60001)), ("bf16", (3000, 21, 403)), ("fp32", (9, 48, 8193)), ("fp32", (2, 9, 1048577)),
    ("fp32", (3, 21, 700001)), ("fp32", (3, 32, 699904)), ("fp32", (3, 8, 700001)),
    ("fp32", (9, 64, 8193)), ("fp32", (7, 128, 4100)), ("fp32", (5, 129, 5001)), ("fp32", (4, 256, 4099)),
    ("fp32", (700, 150, 85))])
def test_dimension_shapes(hk, cuda, dtype, shape):
    import torch
    g = torch.Generator(device=cuda).manual_seed(sum(shape))
    tt = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}[dtype]
    x = (torch.randn(shape, generator=g, device=cuda) * 3.0).to(tt)
    x[:, :, 0] = torch.finfo(tt).min           # nothing but the lowest value: uniform
    x[:, 1:, 1] = -float("inf")                # one finite entry: one-hot
    dy = torch.randn(shape, generator=g, device=cuda).to(tt)
    y, dx = torch.empty_like(x), torch.empty_like(x)
    hk.softmax_fwd(x, y, 1)
    hk.softmax_bwd(y, dy, dx, 1)
    ey = torch.softmax(x.double(), 1)
    d = dy.double()
    s = y.double()
    edx = s * (d - (s * d).sum(1, keepdim=True))
    # the rounding of what is stored (twice half an ulp, for a value that fp32 puts on the other side of a tie), and fp32's:
    # forward, exponents of up to 32 in magnitude are rounded to 2^-20 and x times the rounded log2(e) is off by 2^-20, times
    # ln 2, and the exponential and the sum by 2^-22 each: 2^-19 of the result; backward, of the products that the bracket is the
    # difference of, of which there are up to 256
    ulp = {"fp32": 2.0 ** -19, "bf16": 2.0 ** -8, "fp16": 2.0 ** -10}[dtype]
    tiny = 2.0 ** -24 if dtype == "fp16" else 0.0   # fp16 results below its smallest normal number
    assert bool(((y.double() - ey).abs() <= ulp * ey + tiny).all()), shape
    size = s * (d.abs() + (s * d.abs()).sum(1, keepdim=True))
    assert bool(((dx.double() - edx).abs() <= ulp * edx.abs() + 2.0 ** -19 * size + tiny).all()), shape


@pytest.mark.parametrize("dtype,shape", [
    # fp32 in two slices of 128 lanes: the edges of the planes' length and of the vectors per compute unit
    ("fp32", (105, 21, 10001)), ("fp32", (104, 9, 10001)), ("fp32", (4, 24, 262145)), ("fp32", (4, 32, 262145)), ("fp32", (5, 25, 209713)),
    ("fp32", (4, 26, 262144)), ("fp32", (16, 28, 65533)),
    # 16 bits: what is streamed and what is stored through the cache, on both sides of 24, 32, 48 and 64 MiB
    ("bf16", (37, 24, 18999)), ("fp16", (46, 40, 18999)), ("bf16", (16, 56, 15001)), ("bf16", (20, 64, 14001)), ("bf16", (14, 128, 15001)),
    ("fp16", (12, 176, 14001)), ("bf16", (14, 250, 8001)), ("bf16", (8, 90, 14400)), ("bf16", (16, 90, 14400)), ("bf16", (6, 200, 14001))])
def test_dimension_shapes_at_the_edges_of_the_rules(hk, cuda, dtype, shape):
    test_dimension_shapes(hk, cuda, dtype, shape)
