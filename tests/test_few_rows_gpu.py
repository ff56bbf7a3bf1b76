"""Products of at most eight rows in the weight-streaming kernel: eight k-steps a batch, and two workgroups a block."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from bare_cuda_4gib_amd.csrc import ops as o
    return o


@pytest.mark.parametrize("m", [1, 2, 7, 8])
@pytest.mark.parametrize("n, k", [(8, 1024), (24, 1032), (2048, 2048), (2040, 5632), (2048, 1016), (2056, 1024), (3072, 264), (3088, 4096), (1024, 64), (3000, 1024), (2048, 3072), (2040, 3080), (3072, 2056)])
def test_eight_rows_are_the_first_of_more(ops, monkeypatch, m, n, k):
    """Every row's sums are the same bits as in a step of 16 rows (other batches, whole blocks) and as with a block a workgroup."""
    torch.manual_seed(n + m)
    a = torch.randn(16, k, device=DEV).to(torch.bfloat16)
    w = ops.StreamedWeight((torch.randn(n, k, device=DEV) * k ** -0.5).to(torch.bfloat16))
    base, bias = torch.randn(16, n, device=DEV), torch.randn(n, device=DEV)
    sums = {dt: ops.gemm_fast(a, w, dt) for dt in (torch.float32, torch.bfloat16)}
    added = ops.gemm_fast(a, w, accumulate_into=base.clone(), bias=bias)
    for blocks in (ops.HALF_BLOCKS, 0):
        monkeypatch.setattr(ops, "HALF_BLOCKS", blocks)
        assert ops.half_blocks(m, n, k) == (blocks > 0 and n <= 2048 and k >= 1024)
        for dt, want in sums.items():
            assert torch.equal(ops.gemm_fast(a[:m].contiguous(), w, dt), want[:m])
        assert torch.equal(ops.gemm_fast(a[:m].contiguous(), w, accumulate_into=base[:m].clone(), bias=bias), added[:m])
    assert float((sums[torch.float32].double() - a.double() @ w.rows.double().T).abs().max()) <= k * 2.0 ** -24 * 16


@pytest.mark.parametrize("m", [1, 5, 8])
@pytest.mark.parametrize("n, k", [(2048, 5632), (1000, 1024)])
def test_norm_prepared_by_half_blocks(ops, monkeypatch, m, n, k):
    """What two workgroups a block leave for the norm after them serves the products after it with the same bits."""
    torch.manual_seed(m)
    a = torch.randn(m, k, device=DEV).to(torch.bfloat16)
    w = ops.StreamedWeight((torch.randn(n, k, device=DEV) * k ** -0.5).to(torch.bfloat16))
    g, base = 1 + 0.1 * torch.randn(n, device=DEV), torch.randn(m, n, device=DEV)
    after = ops.StreamedWeight((torch.randn(16 * 700, n, device=DEV) * n ** -0.5).to(torch.bfloat16))
    made = []
    for blocks in (ops.HALF_BLOCKS, 0):
        monkeypatch.setattr(ops, "HALF_BLOCKS", blocks)
        res = base.clone()
        pre = ops.gemm_accumulate_emit(a, w, res, g, 1e-5)
        assert pre.parts.dim() == (3 if blocks else 2)
        made.append((res, pre.xb, pre.parts.sum(-1) if blocks else pre.parts, ops.gemm_prenormed(pre, after, ops.EPI_STORE_F32),
                     ops.gemm_prenormed(pre, after, ops.EPI_SWIGLU)))
    for one, other in zip(*made):
        assert torch.equal(one, other)
