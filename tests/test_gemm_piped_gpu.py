"""The tiles whose waves read fragments slices ahead (256 x 128 from three steps of k on, 128 x 128 from ten): against the product in float64 and, bit
for bit, against the same rows in a product small enough for 64 x 64 tiles, at walks over k shorter than, as long as and longer than
their rings, odd and even, at edges in both directions."""
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


@pytest.mark.parametrize("m,n,tile,steps", [(m, n, (256, 128), s) for m, n in [(1793, 4090), (2036, 4082)] for s in (3, 4, 5, 6, 7, 14)] +
                         [(m, n, (128, 128), s) for m, n in [(1793, 2044), (2036, 2040)] for s in (10, 11, 12, 13)])
def test_short_walks(ops, m, n, tile, steps):
    k = 64 * steps
    assert ops.tiled_tile(m, n, k) == tile and ops.tiled_tile(65, n, k) == (64, 64) and ops.tiled_cut(m, n, k) == (n, None, False)
    x, w = rnd(m, k, seed=1).to(DEV), rnd(n, k, seed=2).to(DEV)
    onto = rnd(m, n, seed=3).float().to(DEV)
    got, added = ops.gemm_fast(x, w, torch.float32), ops.gemm_fast(x, w, accumulate_into=onto.clone())
    want = x.double() @ w.double().T
    assert (got.double() - want).abs().max() < 2.0 * k * 2.0 ** -24 * math.sqrt(k)      # k float additions of terms around 1
    assert torch.equal(onto + got, added)
    assert torch.equal(got.bfloat16(), ops.gemm_fast(x, w, torch.bfloat16))
    for a in (0, m // 2, m - 65):
        assert torch.equal(ops.gemm_fast(x[a:a + 65].contiguous(), w, torch.float32), got[a:a + 65])


@pytest.mark.parametrize("m,n,k,parts,tile", [(129, 136, 640, 5, 128), (300, 2048, 5632, 4, 128), (66, 130, 192, 3, 128), (257, 264, 1536, 8, 256),
                                              (511, 392, 128, 2, 256), (700, 4096, 1024, 4, 256)])
def test_parts_of_k(ops, m, n, k, parts, tile):
    x, w = rnd(m, k, seed=4).to(DEV), rnd(n, k, seed=5).to(DEV)
    out = torch.full((parts, m, n), float("nan"), device=DEV)
    ops.library.call("bc4g_gemm_mfma_parts_large", x.data_ptr(), ops.pack_weight(w).data_ptr(), 1, out.data_ptr(), m, n, k, parts, tile,
                     torch.cuda.current_stream().cuda_stream)
    step = k // parts
    for p in range(parts):
        want = x[:, p * step:(p + 1) * step].double() @ w[:, p * step:(p + 1) * step].double().T
        assert (out[p].double() - want).abs().max() < 2.0 * step * 2.0 ** -24 * math.sqrt(step)


@pytest.mark.parametrize("m,n,k,parts,tile", [(270, 2048, 5632, 4, 128), (512, 4096, 14336, 4, 256), (700, 2048, 5632, 4, 256), (1000, 2048, 2560, 2, 128),
                                              (257, 2048, 2048, 1, 64), (256, 2048, 2048, 2, 64)])
def test_an_adding_product_and_the_norm_behind_it(ops, m, n, k, parts, tile):
    """As many parts as the weight's plan says, against float64: the sums to k float additions of terms around k ** -0.5, the norm to a rounding."""
    plan = ops.plan_for(n, k)
    assert plan.parts_tiles(m) == (parts, tile) and plan.parts(m) == parts
    if parts == 1:
        return
    x, w = rnd(m, k, seed=6).to(DEV), (rnd(n, k, seed=7) * k ** -0.5).to(DEV)
    onto, g = rnd(m, n, seed=8).float().to(DEV), rnd(n, seed=9).float().to(DEV)
    want = onto.double() + x.double() @ w.double().T
    left = ops.gemm_parts_accumulate_norm(x, w, onto, g, 1e-5)
    assert (onto.double() - want).abs().max() < 2.0 * k * 2.0 ** -24
    normed = want / (want.square().mean(1, keepdim=True) + 1e-5).sqrt() * g.double()
    assert ((left.tensor.double() - normed).abs() <= 2.0 ** -8 * normed.abs() + 1e-4).all()


@pytest.mark.parametrize("m,k,tile", [(600, 2048, (128, 64)), (633, 1088, (128, 64)), (1800, 2048, (128, 128)), (1921, 832, (128, 128)), (3200, 1088, (128, 128))])
def test_qkv(ops, m, k, tile):
    """Queries, and the pages that keys and values are written to: the bits of the same rows a few at a time."""
    nh, nkv, d, page = 32, 4, 64, 64
    n = (nh + 2 * nkv) * d
    assert ops.tiled_tile(m, n, k, qkv=True) == tile and ops.tiled_tile(65, n, k, qkv=True) != tile
    x, w = rnd(m, k, seed=10).to(DEV), (rnd(n, k, seed=11) * 0.2).to(DEV)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)      # noqa: E731
    slots = [5 + i for i in range(m)]
    table = ops.rope_table(i32([3 * i for i in range(m)]), d, 10000.0)
    caches = [[torch.zeros(-(-m // page) + 1, nkv, *shape, dtype=torch.bfloat16, device=DEV) for shape in ((page, d), (d, page))] for _ in range(2)]
    q = ops.gemm_qkv_rope_tiled(x, w, table, i32(slots), *caches[0], nh, nkv, d)
    for a in range(0, m, 65):
        b = min(a + 65, m)
        few = ops.gemm_qkv_rope_tiled(x[a:b].contiguous(), w, table[a:b].contiguous(), i32(slots[a:b]), *caches[1], nh, nkv, d)
        assert torch.equal(few, q[a:b])
    assert all(torch.equal(one, two) for one, two in zip(*caches))
