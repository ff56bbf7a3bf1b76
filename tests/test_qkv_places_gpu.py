"""Where the tiled q|k|v product puts keys and values: without a rotation every number is the plain product's, bit for bit, at the slot its row names --
for head and page sizes that are and are not powers of two, caches in fragment order and plain ones, places that follow each other, from multiples of
four on and not, and places in any order."""
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


def in_fragment_order(k, v, page, d):
    """[pages, kv, page, d] keys and [pages, kv, d, page] values as the matrix-core caches keep them (common.h)."""
    pages, kv = k.shape[:2]
    kf = k.view(pages, kv, page // 16, 16, d // 8, 8).permute(0, 1, 2, 4, 3, 5).reshape(k.shape)
    vf = v.view(pages, kv, d // 16, 16, page // 16, 4, 4).permute(0, 1, 4, 2, 5, 3, 6).reshape(v.shape)
    return kf.contiguous(), vf.contiguous()


@pytest.mark.parametrize("order", ["from 0", "from 2", "pages", "any", "mixed"])
@pytest.mark.parametrize("heads, kv, d, page, m, k", [(2, 1, 16, 16, 65, 192), (4, 2, 48, 32, 130, 64), (3, 3, 80, 24, 300, 128), (8, 1, 128, 64, 270, 2048),
                                                      (2, 2, 256, 16, 513, 640), (32, 4, 64, 64, 2049, 576), (6, 3, 96, 48, 700, 1088), (4, 2, 64, 1, 90, 64)])
def test_keys_and_values_lie_where_their_rows_say(ops, order, heads, kv, d, page, m, k):
    torch.manual_seed(m)
    n = (heads + 2 * kv) * d
    x, w = torch.randn(m, k, device=DEV).bfloat16(), ops.StreamedWeight((torch.randn(n, k, device=DEV) * k ** -0.5).bfloat16())
    pages = -(-(m + 3) // page) + 1
    if order == "any":
        slots = torch.randperm(pages * page)[:m]
    elif order == "pages":
        slots = (torch.randperm(pages)[:, None] * page + torch.arange(page)).reshape(-1)[:m]
    else:
        slots = torch.arange(m) + (2 if order == "from 2" else 0)
        if order == "mixed":            # (every fourth run of four broken)
            first = slots[5:m - 1:16].clone()
            slots[5:m - 1:16], slots[6:m:16] = slots[6:m:16].clone()[:len(first)], first
    kc, vc = torch.zeros(pages, kv, page, d, dtype=torch.bfloat16, device=DEV), torch.zeros(pages, kv, d, page, dtype=torch.bfloat16, device=DEV)
    q = ops.gemm_qkv_rope_tiled(x, w, None, slots.int().to(DEV), kc, vc, heads, kv, d)
    plain = ops.gemm_fast(x, w, torch.bfloat16)
    assert torch.equal(q, plain[:, :heads * d])
    kw, vw = torch.zeros_like(kc), torch.zeros_like(vc)
    where = slots.to(DEV)
    kw[where // page, :, where % page] = plain[:, heads * d:(heads + kv) * d].view(m, kv, d)
    vw[where // page, :, :, where % page] = plain[:, (heads + kv) * d:].view(m, kv, d)
    if page % 16 == 0:
        kw, vw = in_fragment_order(kw, vw, page, d)
    assert torch.equal(kc, kw) and torch.equal(vc, vw)
