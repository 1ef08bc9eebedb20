"""GPU parity of the native causal prefill attention (ext.prefill_attention)
against its stages run one by one over a masked score matrix, at sizes around
the products' tiles: score tiles past the diagonal are left unwritten there
(the workspace is filled with NaN first), and must not reach the result.

The stages have the same operations per element: products in the same order
of k, the same softmax over the same row (masked scores weigh 0), so the
results are equal bit for bit.
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


@pytest.mark.parametrize("nkv,rep,T,start,dh", [
    (4, 8, 500, 0, 64), (2, 1, 129, 0, 128), (4, 2, 33, 31, 64), (1, 8, 3, 200, 16), (2, 4, 1, 64, 64),
    (8, 1, 127, 1, 32), (3, 3, 65, 0, 20), (2, 2, 2, 0, 4), (1, 1, 3, 1, 2), (2, 8, 1023, 2, 64)])
def test_prefill_attention_matches_its_stages(nkv, rep, T, start, dh):
    from rac_amd import ext
    t_cap, total = start + T + 5, start + T
    q = torch.from_numpy(rl.gen_normal((nkv, rep * T, dh), seed=1)).to(DEV)
    kc, vc = (torch.from_numpy(rl.gen_normal((nkv, t_cap, dh), seed=s)).to(DEV) for s in (2, 3))
    kc[:, total:] = vc[:, total:] = float("nan")                    # past the prompt: not read
    scale = ext.attention_scale(dh)
    s = ext.bmm(q, kc[:, :total], trans_b=True, alpha=scale, iters=16, mode=ext.MODE_FAST)
    t = torch.arange(T, device=DEV).repeat(rep).view(rep * T, 1)
    s.masked_fill_(torch.arange(total, device=DEV).view(1, total) > start + t, float("-inf"))
    p = ext.softmax(s.view(-1, total), 16).view(nkv, rep * T, total)
    want = ext.bmm(p, vc[:, :total], iters=16, mode=ext.MODE_FAST)
    for _ in range(2):
        # the allocator hands this block to the call as its workspace
        torch.full((nkv * rep * T * total,), float("nan"), device=DEV)
        got = ext.prefill_attention(q, kc, vc, T, start, scale, 16)
        assert torch.isfinite(got).all()
        assert torch.equal(got, want)


def test_prefill_attention_composed_form():
    """RACDecoder's form for more query rows than the native call takes: the
    same result."""
    from types import SimpleNamespace

    from rac_amd import ext
    from rac_amd.decoder import RACDecoder
    nkv, rep, T, start, dh = 2, 3, 37, 11, 16
    kc, vc = (torch.from_numpy(rl.gen_normal((nkv, 64, dh), seed=s)).to(DEV) for s in (2, 3))
    dec = SimpleNamespace(cfg=SimpleNamespace(n_kv_heads=nkv, n_heads=nkv * rep, d_head=dh, d_model=nkv * rep * dh),
                          k_cache=[kc], v_cache=[vc], scale=ext.attention_scale(dh), iters=16)
    q = torch.from_numpy(rl.gen_normal((T, nkv * rep * dh), seed=1)).to(DEV)
    qg = q.view(T, nkv, rep, dh).permute(1, 2, 0, 3).reshape(nkv, rep * T, dh).contiguous()
    want = RACDecoder._prefill_attention_composed(dec, 0, qg, start, T)
    assert torch.equal(RACDecoder._prefill_attention(dec, 0, q, start, T), want)
