"""Where a norm that a product could absorb is prepared before it, the bits of both ways, and the fused norm's staging with a float scale."""
import pytest
import torch


def test_wide_outputs_leave_the_norm_of_five_rows_and_more_to_its_own_kernel():
    from bare_cuda_4gib_amd.csrc import ops
    wide, narrow = ops.compute_plan(16384, 2048), ops.compute_plan(16376, 2048)
    assert [m for m in range(10) if wide.norms_apart(m)] == [5, 6, 7, 8, 9] and not any(narrow.norms_apart(m) for m in range(10))
    assert wide.fuses_norm(8) and wide.wants_prepared(5, swiglu=True)          # (what the kernels take, and who prepares, stay as they were)


def test_narrow_rows_are_prepared_for_wider_outputs_alone():
    from bare_cuda_4gib_amd.csrc import ops
    assert [n for n in (16384, 24568, 24576, 128256) if ops.compute_plan(n, 1016).norms_apart(8)] == [24576, 128256]
    assert ops.compute_plan(16384, 1024).norms_apart(8)


@pytest.mark.gpu
@pytest.mark.parametrize("k", [8, 504, 512, 520, 1024, 1032, 2048])
@pytest.mark.parametrize("rows", [1, 4, 5, 8])
def test_a_float_scale_gives_the_bits_of_the_same_scale_in_bfloat16(k, rows):
    from bare_cuda_4gib_amd.csrc import ops
    torch.manual_seed(k + rows)
    x, w = torch.randn(rows, k, device="cuda:0"), ops.StreamedWeight(torch.randn(48, k, device="cuda:0").bfloat16())
    g = torch.randn(k, device="cuda:0").bfloat16()
    one = ops.gemm_normed(x, None, rows, g, 1e-5, w, ops.EPI_STORE_F32)
    assert torch.equal(one, ops.gemm_normed(x, None, rows, g.float(), 1e-5, w, ops.EPI_STORE_F32))


@pytest.mark.gpu
@pytest.mark.parametrize("k", [8, 504, 512, 520, 2048, 4096, 4104, 6136])       # (one wave's pieces: 512 elements, eight of them a round)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_a_norm_prepared_before_a_product_gives_the_bits_of_one_inside_it(k, dtype):
    from bare_cuda_4gib_amd.csrc import ops
    torch.manual_seed(k)
    x, w = torch.randn(11, k, device="cuda:0"), ops.StreamedWeight(torch.randn(48, k, device="cuda:0").bfloat16())
    g = torch.randn(k, device="cuda:0").to(dtype)
    for rows in (None, torch.tensor([10, 0, 3, 3, 7], dtype=torch.int32, device="cuda:0")):
        at, n = (x, 5) if rows is not None else (x[:8].contiguous(), 8)
        pre = ops.rmsnorm_prepare(at, rows, n, g, 1e-5)
        for epilogue in (ops.EPI_STORE_F32, ops.EPI_STORE_BF16, ops.EPI_SWIGLU):
            assert torch.equal(ops.gemm_prenormed(pre, w, epilogue), ops.gemm_normed(at, rows, n, g, 1e-5, w, epilogue))


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [4, 5, 8])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_a_wide_output_has_the_bits_of_the_norm_inside_it_at_any_number_of_rows(rows, dtype):
    """The head's rows, a feed-forward's behind a sandwich's add, and one with xIELU: where the norm is made moves no bit."""
    from types import SimpleNamespace
    from bare_cuda_4gib_amd.csrc import ops
    from bare_cuda_4gib_amd.parts.lazy import Normed
    from bare_cuda_4gib_amd.parts.linear import absorbs_norm, linear, linear_swiglu, linear_xielu
    from bare_cuda_4gib_amd.parts.norm import RMSNorm
    torch.manual_seed(rows)
    k, n = 1024, 16384
    norm = RMSNorm(k, 1e-5)
    norm.bind({"weight": (1 + torch.randn(k, device="cuda:0") / 8).to(dtype)}, SimpleNamespace(act_dtype=torch.bfloat16))
    x, w = torch.randn(12, k, device="cuda:0"), ops.StreamedWeight((torch.randn(n, k, device="cuda:0") / 32).bfloat16())
    some = torch.tensor([11, 2, 0, 5, 1, 9, 4, 7][:rows], dtype=torch.int32, device="cuda:0")
    few, pq = x[:rows].contiguous(), torch.tensor([0.3, -0.2], device="cuda:0")
    inside = lambda at, at_rows, epilogue: ops.gemm_normed(at, at_rows, rows, norm.weight, norm.eps, w, epilogue)      # noqa: E731
    assert torch.equal(linear(Normed(x, norm, rows=some, n_rows=rows), w, out_dtype=torch.float32), inside(x, some, ops.EPI_STORE_F32))
    assert torch.equal(linear(Normed(few, norm), w, out_dtype=torch.bfloat16), inside(few, None, ops.EPI_STORE_BF16))
    assert torch.equal(linear_swiglu(Normed(few, norm), w, interleaved=True), inside(few, None, ops.EPI_SWIGLU))
    assert torch.equal(linear_xielu(Normed(few, norm), w, pq, torch.bfloat16), ops.xielu(inside(few, None, ops.EPI_STORE_BF16), pq))
    # (a sandwich's add leaves what the product absorbs)
    assert absorbs_norm(norm, w, rows)
    left = ops.rmsnorm_add(few.clone(), torch.zeros_like(few), torch.ones(k, device="cuda:0"), 1e-5, next_norm=(norm.weight, norm.eps, torch.bfloat16), prepare=True)
    assert torch.equal(linear(Normed(few, norm, pre=left), w, out_dtype=torch.float32), inside(few, None, ops.EPI_STORE_F32))
