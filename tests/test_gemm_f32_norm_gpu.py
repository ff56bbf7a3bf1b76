"""The float32 products of few rows that prepare an RMSNorm, finish one, rotate and write the cache (gemm_f32.hip) against float64.

Tolerance: a float32 sum of k products is off by at most k 2^-24 sum |x w|; the factor of a norm comes from a sum of squares of at most
(16 + 16 + blocks / 16) steps, half of whose relative error it inherits, and a few roundings of its own."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
U = 2.0 ** -24
EPS = 1e-5


@pytest.fixture(scope="module")
def ops():
    from bare_cuda_4gib_amd.csrc import ops as o
    with o.weights_pass():                # (weights of 6 MB and more past the caches, as in the steps of a large model)
        yield o


def held(got, want, bound, what):
    assert got.dtype == torch.float32 and tuple(got.shape) == tuple(want.shape), what
    assert torch.isfinite(got).all() and float(((got.double() - want).abs() / bound).max()) <= 1.0, what


def prepared(ops, m, n, seed, k=36):
    """(residual after an adding product, the norm's scale, what the product left) for m rows of n columns."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    x, w = torch.randn(m, k, generator=gen, device=DEV), torch.randn(n, k, generator=gen, device=DEV)
    residual, bias = torch.randn(m, n, generator=gen, device=DEV), torch.randn(n, generator=gen, device=DEV)
    g = 1.0 + 0.2 * torch.randn(n, generator=gen, device=DEV)
    want = ops.gemm_f32(x, w, accumulate_into=residual.clone(), bias=bias)
    few = ops.gemm_f32_emit(x[m - 1:].clone(), w, residual[m - 1:].clone(), g, EPS, bias=bias)
    pre = ops.gemm_f32_emit(x, w, residual, g, EPS, bias=bias)
    assert torch.equal(residual, want) and torch.equal(pre.xb, want * g) and torch.equal(few.xb, pre.xb[m - 1:])
    return residual, g, pre, few


@pytest.mark.parametrize("n", [96, 2048])
def test_rows_on_both_sides_of_few(ops, n):
    """64 rows finish the norm behind the product's sums, 65 run it before the product: a row's bits are others, its bound is the same."""
    gen = torch.Generator(device=DEV).manual_seed(n)
    f = lambda *shape: torch.randn(*shape, generator=gen, device=DEV)      # noqa: E731
    x, w, start, g, after = f(65, 36), f(n, 36), f(65, n), 1.0 + 0.2 * f(n), 0.1 * f(42, n)
    residual = start[:64].clone()
    pre = ops.gemm_f32_emit(x[:64].contiguous(), w, residual, g, EPS)
    many = ops.gemm_f32(x, w, accumulate_into=start.clone())
    assert ops.gemm_f32_emit(x, w, start, g, EPS) is None and not ops.gemm_f32_finishes_norm(65, after) and torch.equal(many[:64], residual)
    r = residual.double()
    normed = r * torch.rsqrt((r * r).mean(-1, keepdim=True) + EPS) * g.double()
    z, size = normed @ after.double().T, normed.abs() @ after.double().abs().T
    rel = (n + 2 + 40 + n / 256) * U
    held(ops.gemm_f32_prenormed(pre, after), z, rel * size, "64 rows")
    held(ops.gemm_f32(ops.rmsnorm(many, g, EPS, torch.float32), after)[:64], z, rel * size, "65 rows")


# Rows at the edges of the forms (8, 16 and 32 a workgroup); columns that end inside a block of 16 and inside its half, few enough for
# eight outputs a workgroup and too many, and more than the 4,096 whose parts a product asks for together.
@pytest.mark.parametrize("m", [1, 7, 8, 9, 16, 17, 33, 64])
@pytest.mark.parametrize("n", [4, 24, 96, 2048, 2052, 4112, 5000])
@pytest.mark.parametrize("act", [None, "silu", "gelu_tanh"])
def test_a_norm_between_two_products(ops, m, n, act):
    residual, g, pre, few = prepared(ops, m, n, m + n)
    gen = torch.Generator(device=DEV).manual_seed(n)
    w = torch.randn(2 * 21, n, generator=gen, device=DEV) * 0.1
    got = ops.gemm_f32_prenormed(pre, w, act)
    r = residual.double()
    normed = r * torch.rsqrt((r * r).mean(-1, keepdim=True) + EPS) * g.double()
    z, size = normed @ w.double().T, normed.abs() @ w.double().abs().T
    rel = (n + 2 + 40 + n / 256) * U
    if act is None:
        held(got, z, rel * size, "stored")
    else:
        gate, up = z[:, :21], z[:, 21:]
        f = torch.nn.functional.silu(gate) if act == "silu" else torch.nn.functional.gelu(gate, approximate="tanh")
        bound = 1.2 * rel * size[:, :21] * up.abs() + f.abs() * rel * size[:, 21:] + 16 * U * (gate * up).abs()
        held(got, f * up, 1.01 * bound + 1e-30, act)
    assert torch.equal(ops.gemm_f32_prenormed(few, w, act), got[m - 1:]), "a row's bits must not depend on the rows beside it"


@pytest.mark.parametrize("m", [1, 8, 9, 17, 64])
@pytest.mark.parametrize("heads,kv_heads,d,n", [(4, 2, 16, 64), (3, 3, 32, 100), (5, 1, 80, 132), (32, 4, 64, 2048)])
@pytest.mark.parametrize("normed,rotates,writes", [(True, True, True), (False, True, True), (True, False, True), (True, True, False)])
def test_qkv(ops, m, heads, kv_heads, d, n, normed, rotates, writes):
    """Against the product, then the kernel that rotates and writes the cache (its own tests hold that one against the reference)."""
    residual, g, pre, _ = prepared(ops, m, n, m + n)
    gen = torch.Generator(device=DEV).manual_seed(d)
    total = (heads + 2 * kv_heads) * d
    w = torch.randn(total, n, generator=gen, device=DEV) * 0.1
    x = pre.xb if normed else residual
    positions = torch.randint(0, 2000, (m,), generator=gen, device=DEV, dtype=torch.int32)
    slots = torch.randperm(6 * 16, generator=gen, device=DEV)[:m].to(torch.int32)
    theta, page = 10000.0, 16
    caches = [torch.zeros((6, kv_heads, page, d), device=DEV), torch.zeros((6, kv_heads, d, page), device=DEV)]
    wanted = [c.clone() for c in caches]
    table = ops.rope_table(positions, d, theta, double=True) if rotates else None
    q = ops.gemm_f32_qkv(x, w, table, slots if writes else None, *(caches if writes else (None, None)), heads, kv_heads, d, write_kv=writes,
                         pre=pre if normed else None)
    qkv = ops.gemm_f32_prenormed(pre, w) if normed else ops.gemm_f32(x, w)
    ops.rope_kv_write(qkv, positions, slots if writes else None, *(wanted if writes else (None, None)), heads, kv_heads, d, d if rotates else 0, theta,
                      write_kv=writes)
    # (the same sums; a rotation rounds two products and their sum, fused or not)
    size = qkv.abs().max().item()
    torch.testing.assert_close(q, qkv[:, :heads * d], rtol=0, atol=4 * U * size)
    for got, want in zip(caches, wanted):
        torch.testing.assert_close(got, want, rtol=0, atol=4 * U * size)


def test_refusals(ops):
    from bare_cuda_4gib_amd.errors import KernelError
    x, w = torch.randn(65, 64, device=DEV), torch.randn(96, 64, device=DEV)
    g = torch.ones(96, device=DEV)
    assert ops.gemm_f32_emit(x, w, torch.zeros(65, 96, device=DEV), g, EPS) is None
    assert ops.gemm_f32_emit(x[:3, :63].contiguous(), w[:, :63].contiguous(), torch.zeros(3, 96, device=DEV), g, EPS) is None
    with pytest.raises(KernelError):
        ops.gemm_f32_emit(x[:3].contiguous(), w, torch.zeros(4, 96, device=DEV), g, EPS)
    with pytest.raises(KernelError):
        ops.gemm_f32_qkv(x[:3].contiguous(), w, None, None, None, None, 4, 2, 32, write_kv=False)


@pytest.mark.parametrize("m", [1, 8, 9, 16, 17, 32, 33])
def test_large_weights_as_small_ones(ops, m):
    """A weight that is read past the caches against its halves, which are not: the same bits in every column."""
    gen = torch.Generator(device=DEV).manual_seed(m)
    f = lambda *shape: torch.randn(*shape, generator=gen, device=DEV)      # noqa: E731
    n, k = 816, 2052
    assert n * k * 4 >= 6 << 20 > n // 2 * k * 4
    x, w, add, g = f(m, k), 0.1 * f(n, k), f(m, n), 1.0 + 0.2 * f(k)
    halves = [w[:n // 2].contiguous(), w[n // 2:].contiguous()]
    assert torch.equal(ops.gemm_f32(x, w), torch.cat([ops.gemm_f32(x, h) for h in halves], 1))
    added = [ops.gemm_f32(x, h, accumulate_into=a.clone(memory_format=torch.contiguous_format)) for h, a in zip(halves, add.chunk(2, 1))]
    assert torch.equal(ops.gemm_f32(x, w, accumulate_into=add.clone()), torch.cat(added, 1))
    pre = ops.gemm_f32_emit(f(m, 36), f(k, 36), f(m, k), g, EPS)
    assert torch.equal(ops.gemm_f32_prenormed(pre, w), torch.cat([ops.gemm_f32_prenormed(pre, h) for h in halves], 1))
    order = torch.cat([torch.arange(0, n // 4), torch.arange(n // 2, 3 * n // 4)])
    gates = torch.cat([ops.gemm_f32_prenormed(pre, w[(order + d).to(w.device)].contiguous(), "silu") for d in (0, n // 4)], 1)
    assert torch.equal(ops.gemm_f32_prenormed(pre, w, "silu"), gates)
