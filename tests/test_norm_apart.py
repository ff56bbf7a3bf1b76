"""Where a norm that a product could absorb is run before it, and the fused norm's staging with a float scale."""
import pytest
import torch


def test_wide_outputs_leave_the_norm_of_five_rows_and_more_to_its_own_kernel():
    from bare_cuda_4gib_amd.csrc import ops
    wide, narrow = ops.compute_plan(16384, 2048), ops.compute_plan(16376, 2048)
    assert [m for m in range(10) if wide.norms_apart(m)] == [5, 6, 7, 8, 9] and not any(narrow.norms_apart(m) for m in range(10))
    assert wide.fuses_norm(8) and wide.wants_prepared(5, swiglu=True)          # (what the kernels take, and who prepares, stay as they were)


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
