"""GPU parity of the decode attention's matrix-core form (d_head 32, 64, 128)
at cache lengths around its 16-position groups, the rounds of its 16 waves and
its lanes' rounds of 1024 positions, bit for bit against the oracle's
composition; and with special keys and values next to the row's end.
"""
import numpy as np
import pytest

import raclib as rl
from test_gpu_decoder import orc_decode_attention

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

F32 = np.float32


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm device")
    import rac_amd
    rac_amd.load()
    yield
    torch.cuda.synchronize()


def run(q, K, V, n, heads, scale, iters):
    from rac_amd import ext
    t = [torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in (q, K, V)]
    pos = torch.tensor([n - 1], dtype=torch.int32, device="cuda")
    out = ext.decode_attention(*t, pos, heads, float(scale), iters)
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("dh", [32, 64, 128])
@pytest.mark.parametrize("t_cap,lengths", [(2048, (15, 16, 31, 32, 255, 257, 511, 513, 1023, 1025, 2047, 2048)),
                                           (8192, (1, 1024, 2049, 4111, 8191, 8192))])
def test_decode_attention_lengths(dh, t_cap, lengths):
    heads, kv = 3, 1
    K, V = (rl.gen_normal((kv, t_cap, dh), seed=s + dh) for s in (1, 2))
    q = rl.gen_normal((heads * dh,), seed=3)
    scale = F32(1) / np.sqrt(F32(dh))
    for n in lengths:
        print(f"decode attention dh={dh} t_cap={t_cap} n={n}", flush=True)
        assert np.array_equal(run(q, K, V, n, heads, scale, 24), orc_decode_attention(q, K, V, n, heads, scale, 24)), n


@pytest.mark.parametrize("n", [1, 5, 16, 21])
def test_decode_attention_special_rows(n):
    """Values past the row are never seen, an infinite one in its last position
    is, a NaN key makes the head NaN, and a zero query takes the first key's
    signed zero as its maximum."""
    heads, kv, dh, t_cap = 2, 1, 64, 64
    K, V = (rl.gen_normal((kv, t_cap, dh), seed=s) for s in (1, 2))
    q = rl.gen_normal((heads * dh,), seed=3)
    q[:dh] = 0.0
    K[:, n:], V[:, n:] = np.nan, np.inf
    scale = F32(0.125)
    print(f"decode attention special n={n}", flush=True)
    assert np.array_equal(run(q, K, V, n, heads, scale, 8), orc_decode_attention(q, K, V, n, heads, scale, 8))
    V[:, n - 1, 5] = np.inf
    got = run(q, K, V, n, heads, scale, 24).reshape(heads, dh)
    assert np.all(np.isinf(got[:, 5])) and np.all(np.isfinite(np.delete(got, 5, 1)))
    K[:, n // 2, 7] = np.nan
    assert np.all(np.isnan(run(q, K, V, n, heads, scale, 24)))


@pytest.mark.parametrize("dh", [32, 64, 128, 80])
@pytest.mark.parametrize("n", [3, 5, 16, 21, 40, 1030])
def test_decode_attention_negative_underflow(n, dh):
    """Equal probabilities times the smallest negative subnormal underflow to
    -0 at every position: the group's positions past the row leave it so."""
    heads, kv, t_cap = 2, 1, 1040
    K = rl.gen_normal((kv, t_cap, dh), seed=1)
    V = np.full((kv, t_cap, dh), -1e-45, F32)
    print(f"decode attention underflow n={n} dh={dh}", flush=True)
    got = run(np.zeros(heads * dh, F32), K, V, n, heads, F32(0.125), 24)
    assert np.all(got.view(np.uint32) == 0x80000000)


@pytest.mark.parametrize("dh", [32, 64, 128])
@pytest.mark.parametrize("which", ["q", "k", "v", "out"])
def test_decode_attention_alignment(dh, which):
    """Any 4-byte boundary of the queries, either cache and the output gives
    the bits of the 16-byte one, and writes the output's elements alone."""
    from rac_amd import ext
    heads, kv, t_cap, n = 4, 2, 300, 277
    K, V = (rl.gen_normal((kv, t_cap, dh), seed=s) for s in (1, 2))
    q = rl.gen_normal((heads * dh,), seed=3)
    want = orc_decode_attention(q, K, V, n, heads, F32(0.125), 24)
    pos = torch.tensor([n - 1], dtype=torch.int32, device="cuda")
    for off in (1, 2, 3):
        print(f"decode attention alignment dh={dh} {which} off={off}", flush=True)
        t = {"q": torch.from_numpy(q), "k": torch.from_numpy(K), "v": torch.from_numpy(V),
             "out": torch.zeros(heads * dh)}
        buf = torch.full((t[which].numel() + 4,), float("nan"), device="cuda")
        t = {name: x.cuda() for name, x in t.items()}
        view = buf[off:off + t[which].numel()].view(t[which].shape)
        view.copy_(t[which])
        t[which] = view
        ext.decode_attention(t["q"], t["k"], t["v"], pos, heads, 0.125, 24, out=t["out"])
        assert np.array_equal(t["out"].cpu().numpy(), want)
        assert torch.isnan(buf[:off]).all() and torch.isnan(buf[off + view.numel():]).all()
