"""GPU parity of the FAST GEMM's matrix-core tiles at their edges.

Every output is one fmaf chain over k in order (rac_kernels.hip:204-219, mode
FAST), so each result must equal the oracle's bit for bit whatever tile a
launch takes: sizes one short of and one past the 32 / 64 / 128 tiles, K
around the K-tiles of 16 / 32 / 64 and their four-k loads, the smallest the
matrix cores take (4 k, 4 rows) and what falls below, and odd leading
dimensions, whose rows start off the 16-byte grid.
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


def run(A, B, C0, M, N, K, ta, tb, alpha, beta):
    import rac_amd
    lib = rac_amd.load()
    Ad, Bd, Cd = (torch.from_numpy(np.ascontiguousarray(t)).to(DEV) for t in (A, B, C0))
    rc = lib.rac_gemm_dev(Ad.data_ptr(), Bd.data_ptr(), Cd.data_ptr(), M, N, K, ta, tb, alpha, beta, 24, 0,
                          torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib.rac_last_error()
    torch.cuda.synchronize()
    return Cd.cpu().numpy()


SHAPES = [(17, 17, 4), (17, 33, 3), (20, 18, 1), (801, 3913, 1), (2050, 2041, 3), (31, 32, 63), (33, 65, 64), (32, 31, 65), (63, 129, 15),
          (65, 64, 129), (127, 200, 16), (128, 257, 17), (129, 8200, 37), (300, 5633, 31), (500, 2049, 70),
          (1000, 777, 131), (2047, 2177, 19), (2049, 4095, 33),
          # few rows or columns: one, the 2 and 3 of a thin operand, 16; blocks
          # of 32 and of 64, with both K-tiles
          (1, 1, 5), (1, 31, 130), (2, 3, 70), (3, 2100, 129), (16, 33, 127), (5, 8300, 65), (2, 16500, 131),
          (33, 1, 64), (2100, 3, 129), (31, 16, 257), (8300, 2, 65), (16500, 7, 131)]


# few k: the VALU tiles up to 16, one K-tile with all its 16-k groups or some,
# the 16-k tiles of many outputs, short K-tiles of a transposed A's few rows
SHAPES += [(300, 301, 15), (300, 299, 16), (299, 300, 17), (679, 1739, 32), (679, 1739, 33), (1167, 3867, 16),
           (1167, 3868, 47), (2049, 1030, 64), (12, 300, 32), (13, 301, 33), (301, 7, 17), (4, 62, 48)]
# few rows or columns of short K (the few-row kernels) and one past it
SHAPES += [(1, 62, 200), (1, 2050, 511), (1, 2050, 1027), (3, 6874, 255), (3, 6874, 257), (4, 62, 512), (9, 301, 513),
           (550, 12, 210), (2036, 2, 511), (16, 16, 256), (7, 16, 40), (1, 513, 4090)]


@pytest.mark.parametrize("layout", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("shape", SHAPES)
def test_fast_tile_edges(shape, layout):
    M, N, K = shape
    ta, tb = layout
    print(f"fast tile shape={shape} layout={layout}", flush=True)
    A, B = rl.gen_normal((K, M) if ta else (M, K), seed=M + K), rl.gen_normal((N, K) if tb else (K, N), seed=N + K)
    C0 = rl.gen_normal((M, N), seed=5)
    for alpha, beta in ((1.0, 0.0), (0.75, -1.5)):
        ref = rl.orc_matmul(A, B, M, N, K, 24, 0, ta=ta, tb=tb, alpha=alpha, beta=beta, C0=C0)
        assert np.array_equal(run(A, B, C0, M, N, K, ta, tb, alpha, beta), ref)


@pytest.mark.parametrize("shape", [(4, 40, 9), (5, 21, 64), (16, 100, 4), (3, 40, 9), (40, 3, 20), (2, 2, 2)])
def test_few_rows_of_a_transposed_operand(shape):
    """op(A) = A^T with few rows, op(B) = B with few columns."""
    M, N, K = shape
    print(f"fast tile transposed shape={shape}", flush=True)
    A, B, C0 = rl.gen_normal((K, M), seed=1), rl.gen_normal((K, N), seed=2), np.zeros((M, N), np.float32)
    assert np.array_equal(run(A, B, C0, M, N, K, 1, 0, 1.0, 0.0), rl.orc_matmul(A, B, M, N, K, 24, 0, ta=1))


@pytest.mark.parametrize("layout", [(0, 0), (0, 1), (1, 0)])
def test_fast_tile_specials(layout):
    """Subnormal, infinite and NaN operands next to the edges: nothing read
    past an edge reaches an output."""
    ta, tb = layout
    M, N, K = 67, 70, 66
    print(f"fast tile specials layout={layout}", flush=True)
    A, B = rl.gen_normal((M, K), seed=3), rl.gen_normal((K, N), seed=4)
    A[-1, ::7] = [np.inf, 1e-45, -np.inf, 3e38, np.nan, 2.0 ** -126, -0.0, 1e-40, 1.0, -3e-39]
    B[::5, -1] = 2.0 ** 100
    B[-1, 3] = np.nan
    A2, B2 = (A.T.copy() if ta else A), (B.T.copy() if tb else B)
    got = run(A2, B2, np.zeros((M, N), np.float32), M, N, K, ta, tb, 1.0, 0.0)
    ref = rl.orc_matmul(A2, B2, M, N, K, 24, 0, ta=ta, tb=tb)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[~np.isnan(ref)], ref[~np.isnan(ref)])


UNDERFLOW = [(17, 17, 4), (20, 18, 1), (31, 32, 63), (33, 65, 80), (63, 129, 15), (129, 8200, 37), (300, 5633, 31),
             (500, 2049, 70), (1000, 777, 131), (2049, 4095, 33), (1, 31, 130), (3, 2100, 129), (16, 33, 127),
             (2100, 3, 129), (2, 2, 2), (2, 3, 70), (1, 62, 35), (4, 62, 270), (16, 300, 33)]


@pytest.mark.parametrize("layout", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("shape", UNDERFLOW)
def test_fast_tile_negative_underflow(shape, layout):
    """Products that all underflow negatively: every fmaf of the chain rounds
    to -0, and the k that a tile adds past K must leave it so."""
    M, N, K = shape
    ta, tb = layout
    print(f"fast tile underflow shape={shape} layout={layout}", flush=True)
    A = np.full((K, M) if ta else (M, K), -1e-30, np.float32)
    B = np.full((N, K) if tb else (K, N), 1e-30, np.float32)
    got = run(A, B, np.zeros((M, N), np.float32), M, N, K, ta, tb, 1.0, 0.0)
    assert (got.view(np.uint32) == 0x80000000).all()


@pytest.mark.parametrize("shape", [(3, 70, 37), (33, 65, 80), (301, 5632, 130)])
def test_half_linear_negative_underflow(shape):
    """The same through the 16-bit linear layer."""
    from rac_amd import ext
    M, N, K = shape
    x = torch.full((M, K), -1e-30, device=DEV, dtype=torch.bfloat16)
    w = torch.full((N, K), 1e-30, device=DEV, dtype=torch.bfloat16)
    out = ext.fused_linear_forward(x, w, None, 0, mode=ext.MODE_FAST)
    assert (out.view(torch.int16) == -0x8000).all()


@pytest.mark.parametrize("act", [0, 1, 2, 3])
@pytest.mark.parametrize("shape", [(18, 35, 70), (130, 2050, 40), (700, 1027, 36), (1, 3, 40), (1, 11009, 64), (3, 2035, 70),
                                   (550, 2, 33)])
def test_fast_tile_fused_epilogue(shape, act):
    """Bias, the kept pre-activation and the activation: those of the plain
    product's output."""
    from rac_amd import ext
    M, N, K = shape
    print(f"fast tile fused shape={shape} act={act}", flush=True)
    x, w, b = (torch.from_numpy(rl.gen_normal(s, seed=i)).to(DEV) for i, s in enumerate([(M, K), (N, K), (N,)]))
    out, pre = ext.fused_linear_forward(x, w, b, act, iters=16, mode=ext.MODE_FAST, return_pre=True)
    ref = rl.orc_matmul(x.cpu().numpy(), w.cpu().numpy(), M, N, K, 24, 0, tb=1) + b.cpu().numpy()
    assert np.array_equal(pre.cpu().numpy(), ref)
    want = [pre, ext.relu(pre), ext.gelu(pre), ext.silu(pre, iters=16)][act]
    assert torch.equal(out, want)
