"""GPU parity of the row kernels' layouts (16-byte groups or single values, a
workgroup or a wave per row) against the oracle in the kernels' summation
order, bit for bit: row lengths at the edges of the register tiles and of the
wave layouts, row counts on both sides of the rule that gives a wave a row,
zero maxima of either sign, NaN and infinities.
"""
import numpy as np
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


def case(rows, n):
    x = rl.gen_normal((rows, n), seed=rows + n, std=2.0)
    x[0] = 0.0
    x[0, 0] = -0.0
    if rows > 2:
        x[1] = -np.abs(x[1])
        x[1, n // 2] = -np.inf
        x[2, n - 1] = np.nan
    return x


def dev(x, offset=0):
    buf = torch.empty(x.size + offset, device=DEV)[offset:].view(x.shape)   # offset: not 16-byte aligned
    return buf.copy_(torch.from_numpy(x))


def same(got, want):
    assert np.array_equal(got.cpu().numpy(), want, equal_nan=True)


WIDTHS = [1, 2, 3, 4, 63, 65, 101, 255, 256, 257, 511, 516, 767, 768, 769, 772, 1001, 1023, 1024, 1025, 2047, 4095, 4097]


@pytest.mark.parametrize("n", WIDTHS)
@pytest.mark.parametrize("rows", [3, 1030])
@pytest.mark.parametrize("iters", [8, 11, 16])
def test_softmax_layouts(n, rows, iters):
    from rac_amd import ext
    if rows > 3 and n > 1100:
        pytest.skip("one layout there; the small row count covers it")
    x = case(rows, n)
    same(ext.softmax(dev(x), iters), rl.orc_softmax_lanes(x, iters))


@pytest.mark.parametrize("rows,n", [(8200, 770), (8200, 1021), (4100, 1022)])
def test_wide_rows_of_a_wave(rows, n):
    from rac_amd import ext
    x = case(rows, n)
    g, b = rl.gen_normal(n, seed=4), rl.gen_normal(n, seed=5)
    same(ext.softmax(dev(x), 16), rl.orc_softmax_lanes(x, 16))
    same(ext.rmsnorm(dev(x), dev(g), 1e-6), rl.orc_rmsnorm_lanes(x, g, 1e-6))
    same(ext.layernorm(dev(x), dev(g), dev(b), 1e-6), rl.orc_layernorm_lanes(x, g, b, 1e-6))


@pytest.mark.parametrize("n", WIDTHS)
@pytest.mark.parametrize("rows", [3, 1030])
def test_norm_layouts(n, rows):
    from rac_amd import ext
    x = case(rows, n)
    g, b = rl.gen_normal(n, seed=4), rl.gen_normal(n, seed=5)
    same(ext.rmsnorm(dev(x), dev(g), 1e-6), rl.orc_rmsnorm_lanes(x, g, 1e-6))
    same(ext.layernorm(dev(x), dev(g), dev(b), 1e-6), rl.orc_layernorm_lanes(x, g, b, 1e-6))


@pytest.mark.parametrize("T", [5, 64, 101, 300, 513, 770])
def test_masked_softmax_layouts(T):
    from rac_amd import ext
    s = rl.gen_normal((1030 // T + 1 if T < 300 else 4, T, T), seed=T)
    s[0, 0] = 0.0
    mask = rl.gen_normal((T, T), seed=T + 1)
    for causal, m in ((True, None), (True, mask), (False, mask), (False, None)):
        got = ext.softmax_masked_(dev(s), None if m is None else dev(m), causal, 16)
        for b in range(s.shape[0]):
            same(got[b], rl.orc_softmax_lanes(s[b], 16, causal=causal, mask=m, zero_guard=True))


@pytest.mark.parametrize("rows,n", [(3, 260), (1030, 500), (3, 2000), (1030, 768)])
def test_unaligned_rows(rows, n):
    """Rows off a 16-byte boundary take the single-value layout; its order of
    the sums differs from the aligned rows' by at most n roundings each."""
    from rac_amd import ext
    x = rl.gen_normal((rows, n), seed=n, std=2.0)
    tol = n * 2.0 ** -23
    for f in (lambda t: ext.softmax(t, 16), lambda t: ext.rmsnorm(t, None, 1e-6)):
        a, u = f(dev(x)).cpu().numpy(), f(dev(x, 1)).cpu().numpy()
        assert np.max(np.abs(a - u) / np.maximum(np.abs(a), 1e-30)) <= tol
