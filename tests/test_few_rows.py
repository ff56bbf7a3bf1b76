"""What the entries of products refuse or leave to others before anything is launched: runs without a GPU."""
import ctypes

import pytest
import torch

from bare_cuda_4gib_amd.csrc import library, ops
from bare_cuda_4gib_amd.errors import KernelError

ROOM = ctypes.create_string_buffer(64)
AT = ctypes.addressof(ROOM)            # (an address that is not looked at)


@pytest.mark.parametrize("rows", [9, 16, 17, 64])
def test_parts_of_half_blocks_are_of_eight_rows(rows):
    """More rows are shared out over workgroups that count a row's parts in single numbers: pairs would be read from other rows."""
    with pytest.raises(KernelError, match="half blocks leave parts of at most 8 rows"):
        library.call("bc4g_gemm_skinny_prenormed", AT, AT, 1, rows, 1, 1e-5, AT, AT, 0, rows, 64, 64, None)
    with pytest.raises(KernelError, match="half blocks leave parts of at most 8 rows"):
        library.call("bc4g_gemm_skinny_qkv", AT, None, 0, 1e-5, AT, 1, rows, 1, AT, AT, AT, AT, AT, AT, rows, 64, 2, 1, 16, 16, 1e4, 64, 0, None)


@pytest.mark.parametrize("units, most", [(256, 128), (304, 128), (64, 32), (32, 16)])
def test_half_blocks_leave_a_block_for_every_other_cu(monkeypatch, units, most):
    """As the float32 products' rule has it: two workgroups share a block where the blocks are at most half the CUs."""
    monkeypatch.setattr(ops, "compute_units", lambda: units, raising=False)
    for blocks in (1, 16, 17, 32, 33, 128, 129):
        assert ops.half_blocks(8, 16 * blocks, 2048) == (blocks <= most)
    assert not ops.half_blocks(9, 16, 2048) and not ops.half_blocks(8, 16, 1016)


@pytest.mark.parametrize("k", [1024, 4096])
def test_rings_leave_many_rows_of_wide_outputs_to_the_streaming_kernel(k):
    """Two groups of rows of more than one and a half blocks of outputs a CU are more workgroups than run at once."""
    edge = 16 * (3 * ops.compute_units() // 2)
    assert ops.skinny_rings(33, edge, k) and ops.skinny_rings(64, edge, k) and ops.skinny_rings(32, edge + 1, k)
    assert not ops.skinny_rings(33, edge + 1, k) and not ops.skinny_rings(64, 2 * edge, k)
    assert not ops.skinny_rings(8, 2048, k + 32)


def test_rings_leave_wide_outputs_of_a_short_k_to_the_streaming_kernel():
    """Workgroups of one or two stages each, many of them: by rows, blocks a CU, k and what follows the sums."""
    block = 16 * ops.compute_units()
    for m in (1, 8):
        for epilogue in (ops.EPI_STORE_BF16, ops.EPI_STORE_F32, ops.EPI_SQUARED_RELU, ops.EPI_ACCUM_F32):
            assert not ops.skinny_rings(m, 3 * block + 1, 64, epilogue) and not ops.skinny_rings(m, 30 * block, 512, epilogue)
            assert ops.skinny_rings(m, 3 * block, 512, epilogue) and ops.skinny_rings(m, 30 * block, 832, epilogue)
            assert ops.skinny_rings(m, 30 * block, 768, epilogue) == (epilogue == ops.EPI_ACCUM_F32)
        assert not ops.skinny_rings(m, 8 * block, 512, ops.EPI_STORE_F32, True) and ops.skinny_rings(m, 8 * block, 576, ops.EPI_STORE_F32, True)
        assert not ops.skinny_rings(m, 4 * block, 1024, ops.EPI_STORE_F32, True) and ops.skinny_rings(m, 5 * block, 1024, ops.EPI_STORE_F32, True)
        assert not ops.skinny_rings(m, 8 * block, 512, ops.EPI_SWIGLU) and ops.skinny_rings(m, 8 * block, 512, ops.EPI_SWIGLU, True)
    for m in (9, 16):
        for epilogue in (ops.EPI_STORE_BF16, ops.EPI_SWIGLU):
            assert not ops.skinny_rings(m, 2 * block + 16, 1024, epilogue) and ops.skinny_rings(m, 2 * block, 512, epilogue)
            assert ops.skinny_rings(m, 8 * block, 1088, epilogue)
        assert ops.skinny_rings(m, 8 * block, 576, ops.EPI_ACCUM_F32) and ops.skinny_rings(m, 8 * block, 576, ops.EPI_SWIGLU, True)
        assert not ops.skinny_rings(m, 8 * block, 512, ops.EPI_ACCUM_F32) and not ops.skinny_rings(m, 8 * block, 512, ops.EPI_SWIGLU, True)
    assert ops.skinny_rings(17, 2 * block + 16, 512)


def test_rings_leave_small_weights_of_two_stages_a_wave_to_the_streaming_kernel():
    cus = ops.compute_units()
    for k in (576, 768, 1024):
        n = 16 * (640 * cus // k)
        for m in (1, 8, 17, 32):
            assert not ops.skinny_rings(m, n, k) and ops.skinny_rings(m, n + 1, k) and ops.skinny_rings(m, n, k, ops.EPI_ACCUM_F32)
        assert ops.skinny_rings(33, n, k) and ops.skinny_rings(9, n, k) and not ops.skinny_rings(9, 8 * cus, k)
    assert ops.skinny_rings(1, 768, 512) and ops.skinny_rings(1, 768, 1088)
    for m in (17, 32, 64):
        assert not ops.skinny_rings(m, 2048, 512, ops.EPI_STORE_F32, True) and ops.skinny_rings(m, 2048, 512, ops.EPI_STORE_F32)
    assert ops.skinny_rings(16, 2048, 512, ops.EPI_STORE_F32, True)


@pytest.mark.parametrize("rows, k", [(1, 12288), (4, 12352), (5, 6144), (16, 3072)])
def test_rows_too_long_for_the_fused_norm(rows, k):
    """Rounded up to four they do not fit the staging buffer: refused whichever kernel would take them (one row of 12,288 fits beside the rings)."""
    with pytest.raises(KernelError, match="do not fit the staging buffer"):
        at = -(-AT // 16) * 16
        library.call("bc4g_gemm_skinny_normed", at, None, at, 1, 1e-5, at, at, 1, rows, 64, k, None)


@pytest.mark.parametrize("k", [6, (1 << 24) + 4])
def test_float32_products_leave_what_their_kernels_refuse_to_the_plain_one(k):
    row = torch.empty(1, k)
    assert ops.gemm_f32(row, row) is None


def test_a_float32_product_asks_every_device_for_its_scratch_memory(monkeypatch):
    """How much it is follows from the device's compute units: what one device said does not answer for another."""
    wants = iter([4096, 65536])

    def call(name, m, n, k, place, launches):
        assert name == "bc4g_gemm_f32_scratch" and (m, n, k) == (2991, 1237, 1760) and not launches
        place._obj.value = next(wants)
    monkeypatch.setattr(ops.library, "call", call)
    try:
        assert [ops._gemm_f32_scratch(2991, 1237, 1760, device) for device in (0, 1, 0, 1)] == [4096, 65536, 4096, 65536]
    finally:
        ops._gemm_f32_scratch.cache_clear()
