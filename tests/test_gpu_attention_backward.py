"""GPU parity of the attention core's native backward (ext.attention_backward)
against the same gradients composed from the RAC products and torch, whole
and in chunks of query rows, causal (which skips the half past the diagonal)
and not, at sizes around the products' tiles: 32x32 and the few-column ones in
the first test, the larger ones in test_attention_backward_large_tiles.

The products have the composition's bits for equal dS; dS itself sums each
row in another order.  A row sum of T terms dP P with sum |dP P| <= max |dP|
(P sums to 1) moves by at most ~T 2^-24 max |dP|, so dS by that times P, and
dQ = s dS K, dK = s dS^T Q by at most T 2^-24 max|dP| max|K or Q| each (P's
rows, and its columns up to T of them, sum to at most T); dV has no dS.
"""
import pytest

import raclib as rl

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm device")
    import rac_amd
    rac_amd.load()
    yield
    torch.cuda.synchronize()


def inputs(B, H, T, D):
    return [torch.from_numpy(rl.gen_normal((B, H, T, D), seed=s)).to(DEV) for s in (1, 2, 3, 4)]


def composed(q, k, v, P, g, mode):
    from rac_amd import ext
    B, H, T, D = q.shape
    q3, k3, v3, g3, P3 = (t.reshape(B * H, *t.shape[2:]) for t in (q, k, v, g, P))
    kw = dict(iters=16, mode=mode)
    dV = ext.bmm(P3, g3, trans_a=True, **kw)
    dP = ext.bmm(g3, v3, trans_b=True, **kw)
    dS = P3 * (dP - (dP * P3).sum(-1, keepdim=True))
    s = ext.attention_scale(D)
    return (ext.bmm(dS, k3, alpha=s, **kw).view_as(q), ext.bmm(dS, q3, trans_a=True, alpha=s, **kw).view_as(q),
            dV.view_as(q), float(dP.abs().max()))


@pytest.mark.parametrize("mode", ["fast", "cordic"])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("shape,rows", [((1, 2, 5, 8), 5), ((2, 3, 33, 20), 33), ((1, 2, 130, 64), 64),
                                        ((1, 2, 257, 33), 100), ((1, 1, 600, 128), 192), ((1, 2, 1030, 16), 1030)])
def test_attention_backward(shape, rows, causal, mode):
    from rac_amd import ext
    B, H, T, D = shape
    m = {"fast": ext.MODE_FAST, "cordic": ext.MODE_CORDIC}[mode]
    print(f"attention backward shape={shape} rows={rows} causal={causal} mode={mode}", flush=True)
    q, k, v, g = inputs(*shape)
    _, P = ext.attention(q, k, v, None, causal, iters=16, mode=m, return_probs=True)
    want = composed(q, k, v, P, g, m)
    # buffers full of NaN: nothing unwritten is read, everything is written
    dq, dk, dv = (torch.full_like(q, float("nan")) for _ in range(3))
    for t0 in range(0, T, rows):
        Pc = P[:, :, t0:t0 + rows].contiguous()
        junk = torch.full_like(Pc, float("nan"))         # the workspace's memory, most likely
        del junk
        ext.attention_backward(q, k, v, Pc, g, causal, dq, dk, dv, row0=t0, accumulate=t0 > 0, iters=16, mode=m)
    eps = T * 2.0 ** -24 * want[3]
    if rows >= T:
        assert torch.equal(dv, want[2])
    else:           # the chunks add in turn
        assert float((dv - want[2]).abs().max()) <= T * 2.0 ** -24 * float(g.abs().max()) * T ** 0.5
    assert float((dq - want[0]).abs().max()) <= 2 * eps * float(k.abs().max())
    assert float((dk - want[1]).abs().max()) <= 2 * eps * float(q.abs().max()) * T ** 0.5


# 256 CUs give the causal products 64x64 tiles (the first three shapes and the
# last two; 32x64 the fourth and fifth), and dP 64x64, 32x64, 64x128, 32x64,
# 32x32, 128x128 and 32x32 ones; the chunks' first rows are on no tile's edge
@pytest.mark.parametrize("shape,rows", [((1, 16, 1030, 100), 1030), ((1, 16, 1030, 100), 333), ((1, 32, 1000, 64), 1000),
                                        ((1, 8, 1030, 128), 1030), ((1, 8, 1030, 128), 500),
                                        ((1, 4, 2000, 600), 2000), ((1, 8, 1030, 516), 500)])
def test_attention_backward_large_tiles(shape, rows):
    test_attention_backward(shape, rows, True, "fast")


@pytest.mark.parametrize("value", [float("inf"), float("nan"), 2.0 ** 100])
@pytest.mark.parametrize("which", [0, 1, 2, 3])
def test_attention_backward_unbounded_operands(which, value):
    """An operand the zero half would turn into NaN: every k is taken, and the
    gradients are NaN where the composition's are."""
    from rac_amd import ext
    q, k, v, g = inputs(1, 2, 70, 24)
    _, P = ext.attention(q, k, v, None, True, iters=16, mode=ext.MODE_FAST, return_probs=True)
    ops = [q, k, v, g]
    ops[which] = ops[which].clone()
    ops[which][0, 1, 60, 3] = value
    want = composed(*ops[:3], P, ops[3], ext.MODE_FAST)
    got = [torch.empty_like(q) for _ in range(3)]
    ext.attention_backward(*ops[:3], P, ops[3], True, *got)
    for a, b in zip(got, want):
        assert torch.equal(a.isnan(), b.isnan())


def test_attention_backward_overflowing_differences():
    """Operands whose products are finite but whose dP - rowsum(dP P) is not:
    0 times it is NaN past the diagonal too, so nothing may be skipped.  dP is
    +-1.125 * 2^127 in alternate columns: row 0's sum is dP[0, 0] and
    dP[0, 1] - dP[0, 0] overflows."""
    from rac_amd import ext
    q, k, v, g = inputs(1, 1, 8, 4096)
    big = 1.5 * 2.0 ** 57
    v = torch.full_like(v, big)
    v[:, :, 1::2] = -big
    g = torch.full_like(g, big)
    _, P = ext.attention(q, k, v, None, True, iters=16, mode=ext.MODE_FAST, return_probs=True)
    want = composed(q, k, v, P, g, ext.MODE_FAST)
    assert want[1].isnan().any()
    got = [torch.empty_like(q) for _ in range(3)]
    ext.attention_backward(q, k, v, P, g, True, *got)
    for a, b in zip(got, want):
        assert torch.equal(a.isnan(), b.isnan())
