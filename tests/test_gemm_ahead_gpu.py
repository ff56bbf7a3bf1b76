"""The 64 x 64 tile, whose fragments are read a step ahead: against the product in float64 at walks over k shorter than, as long as and
longer than its ring of four stages, odd and even, at edges in both directions."""
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
    with _ops.weights_pass():             # (weights of 6 MB and more past the caches, as in the steps of a large model)
        yield _ops


def rnd(*shape, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).bfloat16()


@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13])      # (up to nine by the kernel without a step ahead)
@pytest.mark.parametrize("m,n", [(65, 52), (129, 130)])
def test_short_walks(ops, steps, m, n):
    k = 64 * steps
    assert ops.tiled_tile(m, n, k) == (64, 64)
    x, w = rnd(m, k, seed=1).to(DEV), rnd(n, k, seed=2).to(DEV)
    want = x.double() @ w.double().T
    bound = 2.0 * k * 2.0 ** -24 * math.sqrt(k)            # k float additions of terms around 1
    got = ops.gemm_fast(x, w, torch.float32)
    assert (got.double() - want).abs().max() < bound
    onto = rnd(m, n, seed=3).float().to(DEV)
    assert torch.equal(ops.gemm_fast(x, w, accumulate_into=onto.clone()), onto + got)


@pytest.mark.parametrize("m,n,k,parts", [(33, 256, 640, 5), (64, 320, 1536, 8), (130, 96, 256, 2)])
def test_parts_of_k(ops, m, n, k, parts):
    x, w = rnd(m, k, seed=4).to(DEV), rnd(n, k, seed=5).to(DEV)
    out = torch.full((parts, m, n), float("nan"), device=DEV)
    ops.library.call("bc4g_gemm_mfma_parts", x.data_ptr(), ops.pack_weight(w).data_ptr(), 1, out.data_ptr(), m, n, k, parts,
                     torch.cuda.current_stream().cuda_stream)
    step = k // parts
    for p in range(parts):
        want = x[:, p * step:(p + 1) * step].double() @ w[:, p * step:(p + 1) * step].double().T
        assert (out[p].double() - want).abs().max() < 2.0 * step * 2.0 ** -24 * math.sqrt(step)


@pytest.mark.parametrize("m,n,k", [(33, 11264, 2048), (64, 11250, 2048), (64, 9600, 4096)])
def test_weights_past_the_caches(ops, m, n, k):
    """One tile of rows of a large weight, which is read past the caches, against the same rows among more of them: the same bits."""
    assert not ops.streams_weights(m, n, k) and ops.tiled_tile(m, n, k) == (64, 64) and n * k * 2 >= 6 << 20
    x, w = rnd(65, k, seed=6).to(DEV), (rnd(n, k, seed=7) * k ** -0.5).to(DEV)
    few = x[:m].contiguous()
    got = ops.gemm_fast(few, w, torch.float32)
    assert torch.equal(got, ops.gemm_fast(x, w, torch.float32)[:m])
    assert torch.equal(ops.gemm_fast(few, w, torch.bfloat16), ops.gemm_fast(x, w, torch.bfloat16)[:m])
    assert (got.double() - few.double() @ w.double().T).abs().max() < 2.0 * k * 2.0 ** -24
    if n % 16 == 0:
        assert torch.equal(ops.gemm_swiglu(few, w, True), ops.gemm_swiglu(x, w, True)[:m])
