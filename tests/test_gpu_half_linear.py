"""GPU parity of the fused linear layer on bf16 / fp16 tensors as they are:
equal to widening them, running the fp32 layer and casting its output back,
bit for bit (the widening is exact, the cast rounds to nearest even), at the
edges of its tiles, odd leading dimensions (rows off every wider boundary),
special values, and with views and mixed types, which take the cast path.
"""
import numpy as np
import pytest

import raclib as rl

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DTYPES = [torch.bfloat16, torch.float16]


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm device")
    import rac_amd
    rac_amd.load()
    yield
    torch.cuda.synchronize()


def data(shape, seed, dt, scale=1.0):
    return (torch.from_numpy(rl.gen_normal(shape, seed=seed)).cuda() * scale).to(dt)


def widened(x, w, b, act, iters):
    from rac_amd import ext
    bf = b.float() if b is not None else torch.empty(0, device="cuda")
    out, pre = ext.fused_linear_forward(x.float(), w.float(), bf, act, iters=iters, mode=ext.MODE_FAST, return_pre=True)
    return out.to(x.dtype), pre


def same(a, b):
    return torch.equal(a.isnan(), b.isnan()) and torch.equal(torch.nan_to_num(a, 0.0), torch.nan_to_num(b, 0.0))


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("act,iters", [(0, 24), (1, 24), (2, 24), (3, 24), (3, 16), (3, 11)])
@pytest.mark.parametrize("shape", [(1, 31, 4), (7, 130, 63), (17, 33, 65), (100, 257, 17), (130, 2050, 70),
                                   (500, 1027, 129), (2049, 2177, 34)])
def test_half_linear_equals_widened(shape, act, iters, dt):
    from rac_amd import ext
    M, N, K = shape
    print(f"half linear shape={shape} act={act} iters={iters} dtype={dt}", flush=True)
    x, w, b = data((M, K), 1, dt), data((N, K), 2, dt, K ** -0.5), data((N,), 3, dt)
    for bias in (b, None):
        ref, rpre = widened(x, w, bias, act, iters)
        arg = bias if bias is not None else torch.empty(0, device="cuda", dtype=dt)
        got, pre = ext.fused_linear_forward(x, w, arg, act, iters=iters, mode=ext.MODE_FAST, return_pre=True)
        assert got.dtype == dt and pre.dtype == torch.float32
        assert torch.equal(pre, rpre) and torch.equal(got, ref)
    assert torch.equal(ext.linear_forward(x, w, b, mode=ext.MODE_FAST), widened(x, w, b, 0, 24)[0])


@pytest.mark.parametrize("dt", DTYPES)
def test_half_linear_specials_and_routes(dt):
    """Infinite, NaN, subnormal and overflowing values; leading dimensions,
    transposed views, rows 2 bytes off a boundary, mixed types, another MAC
    and fewer than 4 features."""
    from rac_amd import ext
    print(f"half linear specials dtype={dt}", flush=True)
    x, w, b = data((2, 9, 21), 4, dt), data((37, 21), 5, dt), data((37,), 6, dt)
    x[0, 0, 3], x[0, 1, 4], x[1, 2, 5], x[1, 3] = float("inf"), float("nan"), 1e-7, 6e4
    ref = widened(x, w, b, 0, 24)[0]
    assert same(ext.fused_linear_forward(x, w, b, 0, mode=ext.MODE_FAST), ref)
    wt = w.t().contiguous().t()
    off = torch.zeros(2 * 9 * 21 + 1, device="cuda", dtype=dt)
    off[1:] = x.reshape(-1)
    xo = off[1:].view(2, 9, 21)
    assert same(ext.fused_linear_forward(xo, wt, b, 0, mode=ext.MODE_FAST), ref)
    assert same(ext.fused_linear_forward(x, w.float(), b, 0, mode=ext.MODE_FAST), ref)
    assert same(ext.fused_linear_forward(x, w, b.float(), 0, mode=ext.MODE_FAST), ref)
    cx = ext.fused_linear_forward(x, w, b, 1, iters=8, mode=ext.MODE_CORDIC)
    assert cx.dtype == dt and cx.shape == (2, 9, 37)
    assert same(ext.linear_forward(x[..., :3], w[:, :3], b, mode=ext.MODE_FAST),
                widened(x[..., :3], w[:, :3], b, 0, 24)[0])
    assert ext.linear_forward(x[:0], w, b, mode=ext.MODE_FAST).shape == (0, 9, 37)
    with pytest.raises(RuntimeError):
        ext.linear_forward(x, w, b[:5], mode=ext.MODE_FAST)
    with pytest.raises(RuntimeError):
        ext.linear_forward(x, w[:, :20], b, mode=ext.MODE_FAST)
