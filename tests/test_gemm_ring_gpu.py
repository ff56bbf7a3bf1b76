"""The few-row product through rings in LDS against the streaming kernel, which takes the same operands where x lies off a 16-byte
boundary: the same bits from either, at the edges of the row counts, blocks of outputs and parts of k that a workgroup and its waves take."""
import dataclasses

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ROWS = [1, 2, 8, 9, 15, 16, 17, 31, 32, 33, 48, 64]


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from bare_cuda_4gib_amd.csrc import ops as _ops
    with _ops.weights_pass():             # (weights of 6 MB and more past the caches, as in the steps of a large model)
        yield _ops


def off_by_eight(x):
    """x at an address that is 8 bytes past a boundary of 16."""
    past = 8 // x.element_size()
    room = torch.empty(x.numel() + past, dtype=x.dtype, device=x.device)
    room[past:] = x.reshape(-1)
    moved = room[past:].view(x.shape)
    assert x.data_ptr() % 16 == 0 and moved.data_ptr() % 16 == 8
    return moved


def operands(ops, m, n, k, seed=0):
    torch.manual_seed(seed + m)
    return torch.randn(m, k, device=DEV).bfloat16(), ops.StreamedWeight((torch.randn(n, k, device=DEV) * k ** -0.5).bfloat16())


# outputs of a few blocks, of fewer than half the CUs, of fewer than all, of one and a half and two a CU and beyond, ragged; k of one step, of fewer
# and more steps than waves, of parts shorter than a ring and longer
@pytest.mark.parametrize("n, k", [(16, 64), (1000, 448), (2048, 1088), (2040, 5632), (3648, 2048), (6144, 576), (8184, 2560), (11264, 192)])
@pytest.mark.parametrize("m", ROWS)
def test_stored_and_added(ops, m, n, k):
    x, w = operands(ops, m, n, k)
    if not ops.streams_weights(m, n, k):
        pytest.skip("goes to the tiled kernel")
    bias, base = torch.randn(n, device=DEV), torch.randn(m, n, device=DEV)
    other = off_by_eight(x)
    got = ops.gemm_fast(x, w, torch.float32)
    want = x.double() @ w.rows.double().T
    assert (got.double() - want).abs().max() < 4 * k ** 0.5 * 2.0 ** -24 * (x.double().abs() @ w.rows.double().abs().T).max()
    assert torch.equal(got, ops.gemm_fast(other, w, torch.float32))
    assert torch.equal(ops.gemm_fast(x, w, torch.bfloat16), ops.gemm_fast(other, w, torch.bfloat16))
    assert torch.equal(ops.gemm_fast(x, w, torch.bfloat16, squared_relu=True), ops.gemm_fast(other, w, torch.bfloat16, squared_relu=True))
    for b in (None, bias):
        assert torch.equal(ops.gemm_fast(x, w, accumulate_into=base.clone(), bias=b), ops.gemm_fast(other, w, accumulate_into=base.clone(), bias=b))
    if n % 16 == 0:
        for act in ("silu", "gelu_tanh"):
            assert torch.equal(ops.gemm_swiglu(x, w, True, act), ops.gemm_swiglu(other, w, True, act))


@pytest.mark.parametrize("g_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n, k", [(64, 64), (2048, 1024), (1000, 1024), (4096, 320), (6400, 128)])
@pytest.mark.parametrize("m", ROWS)
def test_norms_prepared_and_finished(ops, m, n, k, g_dtype):
    """Parts of whole blocks and of half blocks, of one block (a norm kernel's), of up to 256 blocks and beyond."""
    x, w = operands(ops, m, n, k)
    g, base, bias = (1 + 0.1 * torch.randn(n, device=DEV)).to(g_dtype), torch.randn(m, n, device=DEV), torch.randn(n, device=DEV)
    made = []
    for a in (x, off_by_eight(x)):
        res = base.clone()
        made.append((res, ops.gemm_accumulate_emit(a, w, res, g, 1e-5, bias=bias)))
    (res, pre), (res2, pre2) = made
    assert torch.equal(res, res2) and torch.equal(pre.xb, pre2.xb) and torch.equal(pre.parts, pre2.parts)
    if n % 64:
        return
    after = ops.StreamedWeight((torch.randn(1600, n, device=DEV) * n ** -0.5).bfloat16())
    pq = torch.tensor([0.3, 0.2], device=DEV)
    one_part = ops.rmsnorm_prepare(res, None, m, g, 1e-5)
    for left in (pre, one_part):
        shifted = ops.Prenormed(off_by_eight(left.xb), left.parts, left.eps)
        for epilogue in (ops.EPI_STORE_BF16, ops.EPI_STORE_F32, ops.EPI_SWIGLU, ops.EPI_SQUARED_RELU):
            assert torch.equal(ops.gemm_prenormed(left, after, epilogue), ops.gemm_prenormed(shifted, after, epilogue))
        if left.parts.dim() == 2:
            assert torch.equal(ops.gemm_xielu(left.xb, after, pq, pre=left), ops.gemm_xielu(shifted.xb, after, pq, pre=shifted))


@pytest.mark.parametrize("n", [64, 2048])
@pytest.mark.parametrize("m", [65, 67, 72, 73, 77, 81, 97])
def test_norms_of_more_rows_than_one_launch_takes(ops, monkeypatch, m, n):
    """Rows from the 65th on go into a launch of their own, whose parts end with them and not with a whole part of all rows."""
    x, w = operands(ops, m, n, 512)
    after = ops.StreamedWeight((torch.randn(1600, n, device=DEV) * n ** -0.5).bfloat16())
    for weight in (w, after):
        monkeypatch.setitem(ops._PLANS, tuple(weight.shape), dataclasses.replace(ops.plan_for(*weight.shape), stream_rows=128))
    g, base = 1 + 0.1 * torch.randn(n, device=DEV), torch.randn(m, n, device=DEV)
    pre = ops.gemm_accumulate_emit(x, w, base.clone(), g, 1e-5)
    both = ops.gemm_prenormed(pre, after, ops.EPI_STORE_F32)
    for rows in (slice(0, 64), slice(64, m)):
        own = ops.Prenormed(pre.xb[rows].contiguous(), pre.parts[:, rows].contiguous(), pre.eps)
        assert torch.equal(both[rows], ops.gemm_prenormed(own, after, ops.EPI_STORE_F32))


@pytest.mark.parametrize("heads, kv_heads, head_dim, page", [(4, 2, 16, 16), (32, 4, 64, 64), (32, 8, 128, 64), (48, 48, 64, 24)])
@pytest.mark.parametrize("m", ROWS)
def test_rotated_and_cached(ops, m, heads, kv_heads, head_dim, page):
    n, k = (heads + 2 * kv_heads) * head_dim, 768
    x, w = operands(ops, m, n, k)
    pos = torch.randint(0, 4000, (m,), dtype=torch.int32, device=DEV)
    slots = torch.randperm(8 * page, device=DEV)[:m].to(torch.int32)
    made = []
    for a in (x, off_by_eight(x)):
        kc, vc = torch.zeros(8, kv_heads, page, head_dim, dtype=torch.bfloat16, device=DEV), torch.zeros(8, kv_heads, head_dim, page, dtype=torch.bfloat16, device=DEV)
        q = ops.gemm_qkv_rope(a, None, 0.0, w, pos, slots, kc, vc, heads, kv_heads, head_dim, head_dim, 1e4)
        plain = ops.gemm_qkv_rope(a, None, 0.0, w, pos, None, None, None, heads, kv_heads, head_dim, 0, 1e4, write_kv=False)
        made.append((q, kc, vc, plain))
    assert all(torch.equal(one, other) for one, other in zip(*made))
    want = (x.float() @ w.rows[:heads * head_dim].float().T)
    assert (made[0][3].float() - want).abs().max() < 2.0 ** -8 * want.abs().max()


# parts of k that end inside a piece of 1 KB, waves without a part; one workgroup a CU and several, with as many rows as then fit beside the rings and more
@pytest.mark.parametrize("g_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n, k", [(16, 2048), (1000, 2240), (2048, 2112), (4064, 5632), (4128, 2496), (8192, 3008), (4800, 4096)])
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 8, 9])
def test_norm_fused(ops, m, n, k, g_dtype):
    _, w = operands(ops, m, n, k)
    x, g = 3 * torch.randn(m + 2, k, device=DEV), (1 + 0.1 * torch.randn(k, device=DEV)).to(g_dtype)
    if not ops.gemm_normed_supported(x, m, g, w):
        pytest.skip("the norm runs apart")
    rows = torch.tensor([m + 1 - r for r in range(m)], dtype=torch.int32, device=DEV)
    other, first = off_by_eight(x), x[:m].clone()
    # against float64: the operands are bfloat16(x * g), the sums and the rows' scales float32
    turned, scale = (first * g.float()).bfloat16().double(), torch.rsqrt((first.double() ** 2).mean(1, keepdim=True) + 1e-5)
    want = turned @ w.rows.double().T * scale
    bound = 4 * k ** 0.5 * 2.0 ** -24 * (turned.abs() @ w.rows.double().abs().T * scale).max() + 2.0 ** -21 * want.abs().max()
    assert (ops.gemm_normed(first, None, m, g, 1e-5, w, ops.EPI_STORE_F32).double() - want).abs().max() < bound
    epilogues = [ops.EPI_STORE_F32, ops.EPI_STORE_BF16, ops.EPI_SQUARED_RELU] + ([ops.EPI_SWIGLU] if n % 16 == 0 else [])
    for e in epilogues:
        assert torch.equal(ops.gemm_normed(x, rows, m, g, 1e-5, w, e), ops.gemm_normed(other, rows, m, g, 1e-5, w, e))
        assert torch.equal(ops.gemm_normed(first, None, m, g, 1e-5, w, e), ops.gemm_normed(off_by_eight(first), None, m, g, 1e-5, w, e))
    if n % 64 == 0 and n >= 192:
        kv = n // 64 // 3
        made = []
        for a in (first, off_by_eight(first)):
            kc, vc = torch.zeros(2, kv, 16, 64, dtype=torch.bfloat16, device=DEV), torch.zeros(2, kv, 64, 16, dtype=torch.bfloat16, device=DEV)
            at = torch.arange(m, dtype=torch.int32, device=DEV) * 3
            made.append((ops.gemm_qkv_rope(a, g, 1e-5, w, at, at, kc, vc, n // 64 - 2 * kv, kv, 64, 64, 1e4), kc, vc))
        assert all(torch.equal(one, two) for one, two in zip(*made))
