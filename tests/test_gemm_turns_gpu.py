"""The tiled products whose waves take turns, and outputs whose columns are cut between two tiles: against the product in
float64 and, bit for bit, against the smallest tile (65 rows take it), at the shortest walks over k, an odd and an even number of
steps, and at edges in both directions."""
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
    return _ops


def rnd(*shape, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).bfloat16()


# columns cut between two tiles: the first tile and its columns, the tile of the others
CUT = [(1430, 11276, 1536, (256, 256), 10752, (64, 64)), (1025, 4100, 14336, (128, 128), 3584, (64, 64)), (2900, 6156, 2048, (256, 256), 5376, (128, 128))]
CUT_QKV = [(78, 13, 128, 1280, 1024, 13056, (64, 64)), (48, 16, 80, 2821, 2048, 5376, (128, 128)), (24, 24, 128, 2055, 2048, 7168, (128, 64))]


@pytest.mark.parametrize("m,n,k,tile", [
    (3860, 3852, 64, (256, 256)), (3860, 3852, 128, (256, 256)), (3841, 3841, 320, (256, 256)),       # one row, one column in the last tile
    (2036, 6132, 64, (256, 192)), (2036, 6132, 320, (256, 192)),
    (2036, 2040, 128, (128, 128)), (1921, 2036, 320, (128, 128)),
    # the shortest walks that the groups in turns take (above: the kernel whose waves go together), of an even and an odd number of steps
    (3860, 3852, 640, (256, 256)), (3841, 3841, 704, (256, 256)), (3860, 3852, 1088, (256, 256)), (3841, 3841, 1152, (256, 256)),
    (2036, 6132, 384, (256, 192)), (2036, 6132, 704, (256, 192)), (2036, 2040, 640, (128, 128)), (1921, 2036, 704, (128, 128)),
    (1290, 11276, 1536, (256, 256)),                                       # (ten rows beyond whole tiles, beside them)
    *((m, n, k, tile) for m, n, k, tile, _, _ in CUT)])
def test_turns_and_cut_columns(ops, m, n, k, tile):
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the shapes are chosen for 256 CUs")
    assert ops.tiled_tile(m, n, k) == tile and ops.tiled_tile(65, n, k) == (64, 64)
    cut = next((c[4:] for c in CUT if c[:3] == (m, n, k)), (n, None))
    assert ops.tiled_cut(m, n, k) == (*cut, (m, n, k) == (1290, 11276, 1536))
    x, w = rnd(m, k, seed=1).to(DEV), rnd(n, k, seed=2).to(DEV)
    want = x.double() @ w.double().T
    bound = 2.0 * k * 2.0 ** -24 * math.sqrt(k)            # k float additions of terms around 1
    got = ops.gemm_fast(x, w, torch.float32)
    assert (got.double() - want).abs().max() < bound
    few = x[:65].contiguous()
    assert torch.equal(ops.gemm_fast(few, w, torch.float32), got[:65])
    last = x[m - 65:].contiguous()
    assert torch.equal(ops.gemm_fast(last, w, torch.float32), got[m - 65:])
    assert torch.equal(ops.gemm_fast(x, w, torch.bfloat16), got.bfloat16())
    base, bias = torch.randn(m, n, device=DEV), torch.randn(n, device=DEV)
    assert torch.equal(ops.gemm_fast(x, w, accumulate_into=base.clone(), bias=bias), base + (got + bias))
    half = n // 32 * 16                                     # gate and up rows in blocks of eight
    rows = torch.stack([w[:half].view(-1, 8, k), w[half:2 * half].view(-1, 8, k)], dim=1).reshape(2 * half, k).contiguous()
    act = ops.gemm_swiglu(x, rows, interleaved=True)
    assert torch.equal(ops.gemm_swiglu(few, rows, interleaved=True), act[:65])
    gate, up = want[:, :half], want[:, half:2 * half]
    exact = gate / (1 + torch.exp(-gate)) * up
    assert ((act.double() - exact).abs() <= 2.0 ** -8 * exact.abs() + 3 * bound * (1 + gate.abs() + up.abs())).all()


@pytest.mark.parametrize("nh,nkv,d,m,k,first,second", CUT_QKV)
def test_cut_qkv(ops, nh, nkv, d, m, k, first, second):
    """Queries, and the pages that keys and values are written to: the bits of the same rows a few at a time."""
    n, page = (nh + 2 * nkv) * d, 64
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the shapes are chosen for 256 CUs")
    assert ops.tiled_cut(m, n, k, qkv=True) == (first, second, False) and ops.tiled_cut(129, n, k, qkv=True) == (n, None, False)
    x, w = rnd(m, k, seed=7).to(DEV), (rnd(n, k, seed=8) * 0.2).to(DEV)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)      # noqa: E731
    slots = [5 + i for i in range(m)]
    table = ops.rope_table(i32([3 * i for i in range(m)]), d, 10000.0)
    caches = [[torch.zeros(-(-m // page) + 1, nkv, *shape, dtype=torch.bfloat16, device=DEV) for shape in ((page, d), (d, page))] for _ in range(2)]
    w = ops.StreamedWeight(w)
    q = ops.gemm_qkv_rope_tiled(x, w, table, i32(slots), *caches[0], nh, nkv, d)
    for a in range(0, m, 129):
        b = min(a + 129, m)
        few = ops.gemm_qkv_rope_tiled(x[a:b].contiguous(), w, table[a:b].contiguous(), i32(slots[a:b]), *caches[1], nh, nkv, d)
        assert torch.equal(few, q[a:b])
    assert all(torch.equal(one, two) for one, two in zip(*caches))
