"""Rows beyond whole tiles in the same launch as the whole ones: against the product in float64 and, bit for bit, against the same rows
in a product small enough for 64 x 64 tiles; one row and a full tile of rows beyond, columns that fill no tile, every epilogue."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from bare_cuda_4gib_amd.csrc import ops as _ops
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the shapes are chosen for 256 CUs")
    return _ops


def rnd(*shape, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).bfloat16()


SHAPES = [(257, 11264, 512, 128), (270, 11268, 576, 128), (320, 11012, 2048, 128),      # 128 x 128 and 64 x 256
          (519, 22020, 1024, 256), (513, 28676, 576, 256)]                              # 256 x 256 and 64 x 256


@pytest.mark.parametrize("m,n,k,rows", SHAPES)
def test_rows_beyond(ops, m, n, k, rows):
    assert ops.tiled_tile(m, n, k) == (rows, rows) and ops.tiled_tile(65, 1028, k) == (64, 64) and ops.tiled_cut(m, n, k) == (n, None, True)
    x, w = rnd(m, k, seed=1).to(DEV), rnd(n, k, seed=2).to(DEV)
    got = ops.gemm_fast(x, w, torch.float32)
    assert (got.double() - x.double() @ w.double().T).abs().max() < 2.0 * k * 2.0 ** -24 * math.sqrt(k)    # k float additions of terms around 1
    for c in (0, n // 64 * 32, n - 1028):
        cols = w[c:c + 1028].contiguous()
        for a in list(range(0, m - 65, 65)) + [m - 65]:
            assert torch.equal(ops.gemm_fast(x[a:a + 65].contiguous(), cols, torch.float32), got[a:a + 65, c:c + 1028])
    onto = rnd(m, n, seed=3).float().to(DEV)
    assert torch.equal(ops.gemm_fast(x, w, accumulate_into=onto.clone()), onto + got)
    assert torch.equal(ops.gemm_fast(x, w, torch.bfloat16), got.bfloat16())


@pytest.mark.parametrize("m,half,k,rows", [(270, 5632, 2048, 128), (519, 14336, 576, 256)])
def test_gated_rows_beyond(ops, m, half, k, rows):
    assert ops.tiled_tile(m, 2 * half, k) == (rows, rows) and ops.tiled_tile(65, 2048, k) == (64, 64) and ops.tiled_cut(m, 2 * half, k) == (2 * half, None, True)
    x = (rnd(m, k, seed=4) * 0.2).to(DEV)
    gate, up = ((rnd(half, k, seed=s) * 0.2).to(DEV).view(half // 8, 8, k) for s in (5, 6))
    w = torch.stack([gate, up], 1).view(2 * half, k)           # every 16 rows: eight gate rows, then the eight up rows of the same outputs
    got = ops.gemm_swiglu(x, w, interleaved=True)
    for c in (0, half - 1024):
        few_cols = w[2 * c:2 * c + 2048].contiguous()
        for a in (0, m // 2, m - 65):
            assert torch.equal(ops.gemm_swiglu(x[a:a + 65].contiguous(), few_cols, interleaved=True), got[a:a + 65, c:c + 1024])


@pytest.mark.parametrize("nh,nkv,d,m,k,rows", [(32, 32, 128, 270, 512, 128), (172, 86, 64, 519, 512, 256)])
@pytest.mark.parametrize("page", [64, 16])
def test_qkv_rows_beyond(ops, nh, nkv, d, m, k, rows, page):
    """Queries, and the pages that keys and values are written to: the bits of the same rows a few at a time."""
    n = (nh + 2 * nkv) * d
    assert ops.tiled_tile(m, n, k, qkv=True) == (rows, rows) and ops.tiled_tile(65, n, k, qkv=True) != (rows, rows)
    assert ops.tiled_cut(m, n, k, qkv=True) == (n, None, True)
    x, w = rnd(m, k, seed=7).to(DEV), (rnd(n, k, seed=8) * 0.2).to(DEV)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)      # noqa: E731
    pages = -(-m // page) + 1
    slots = [5 + i for i in range(m)]
    table = ops.rope_table(i32([3 * i for i in range(m)]), d, 10000.0)
    caches = [[torch.zeros(pages, nkv, *shape, dtype=torch.bfloat16, device=DEV) for shape in ((page, d), (d, page))] for _ in range(2)]
    q = ops.gemm_qkv_rope_tiled(x, w, table, i32(slots), *caches[0], nh, nkv, d)
    for a in range(0, m, 65):
        b = min(a + 65, m)
        few = ops.gemm_qkv_rope_tiled(x[a:b].contiguous(), w, table[a:b].contiguous(), i32(slots[a:b]), *caches[1], nh, nkv, d)
        assert torch.equal(few, q[a:b])
    assert all(torch.equal(one, two) for one, two in zip(*caches))
