"""The float32 matrix-core products (gemm_f32.hip) against float64.

Tolerance: a float32 sum of k products, in any order, is off by at most k 2^-24 sum |x w| (rounded up here by a few units for
the product, the norm's factor and the activation)."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
U = 2.0 ** -24


@pytest.fixture(scope="module")
def ops():
    from bare_cuda_4gib_amd.csrc import ops as o
    return o


def operands(m, n, k, seed):
    gen = torch.Generator().manual_seed(seed)
    return torch.randn(m, k, generator=gen), torch.randn(n, k, generator=gen) * 0.1


def held(got, want, bound, what):
    assert got.dtype == torch.float32 and tuple(got.shape) == tuple(want.shape), what
    off = ((got.cpu().double() - want).abs() / bound).max()
    assert torch.isfinite(got).all() and float(off) <= 1.0, f"{what}: {float(off):.2f} times the bound"


# The kernel that streams the weights, which takes all of these: rows at the edges of its forms (8, 16 and 32 a workgroup) and beyond,
# k at the edges of a step (32) and of the shares it is added up in, n at the edges of a block.
@pytest.mark.parametrize("m", [1, 7, 8, 9, 16, 17, 33, 64, 65, 129, 300])
@pytest.mark.parametrize("n,k", [(1, 4), (16, 32), (130, 176), (301, 260), (64, 2048), (129, 288), (4098, 36), (2100, 64), (24, 5632)])
def test_products(ops, m, n, k):
    x, w = operands(m, n, k, m + n + k)
    xd, wd = x.to(DEV), w.to(DEV)
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    got = ops.gemm_f32(xd, wd)
    held(got, want, (k + 2) * U * size, "stored")
    base, bias = torch.randn(m, n), torch.randn(n)
    acc = base.to(DEV)
    ops.gemm_f32(xd, wd, accumulate_into=acc, bias=bias.to(DEV))
    held(acc, want + base.double() + bias.double(), (k + 4) * U * (size + base.double().abs() + bias.double().abs()), "added")
    for first, rows in ((m - 1, 1), (0, (m + 1) // 2)):
        assert torch.equal(ops.gemm_f32(xd[first:first + rows].clone(), wd), got[first:first + rows]), "a row's bits must not depend on the rows beside it"


# The tiled kernel, every form of it: rows and outputs that end inside a tile, shares of one step of k and of several, the last of
# them short.  (The tiles are those of 256 CUs.)
TILED = [((1001, 11266, 544), (128, 128)), ((100, 11266, 96), (128, 128)), ((65, 11262, 544), (64, 128)), ((127, 8198, 1056), (64, 128)),
         ((511, 2102, 2048), (64, 128)), ((130, 11266, 288), (64, 64)), ((193, 3002, 2080), (64, 64)), ((300, 2046, 5632), (64, 64))]


@pytest.mark.parametrize("sizes,tile", TILED)
@pytest.mark.parametrize("epilogue", ["store", "add", "add with bias", "silu", "gelu_tanh"])
def test_tiles(ops, sizes, tile, epilogue):
    """Against float64, and bit for bit against the kernel that streams the weights, to which few of the rows go."""
    m, n, k = sizes
    assert ops.gemm_f32_tile(m, n, k) == tile and ops.gemm_f32_tile(8, n, k) == (0, 0)
    torch.manual_seed(m)
    x, w = torch.randn(m, k, device=DEV), torch.randn(n, k, device=DEV) * 0.1
    z, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    base, bias = torch.randn(m, n, device=DEV), torch.randn(n, device=DEV) if epilogue == "add with bias" else None

    def product(rows):
        if epilogue.startswith("add"):
            return ops.gemm_f32(x[rows].clone(), w, accumulate_into=base[rows].clone(), bias=bias)
        return ops.gemm_f32(x[rows].clone(), w, act=None if epilogue == "store" else epilogue)

    got = product(slice(0, m))
    if epilogue in ("silu", "gelu_tanh"):
        gate, up = z[:, :n // 2], z[:, n // 2:]
        want = (torch.nn.functional.silu(gate) if epilogue == "silu" else torch.nn.functional.gelu(gate, approximate="tanh")) * up
        bound = (1.2 * (k + 2) * U * size[:, :n // 2] * up.abs() + (want / up).abs() * (k + 2) * U * size[:, n // 2:] + 16 * U * (gate * up).abs()) * 1.01 + 1e-30
    else:
        added = (base.double() + (bias.double() if bias is not None else 0.0)) if epilogue.startswith("add") else torch.zeros_like(z)
        want, bound = z + added, (k + 4) * U * (size + added.abs() + (base.double().abs() if bias is not None else 0.0))
    held(got, want.cpu(), bound.cpu(), epilogue)
    for rows in ([0, 1, 63, 64], [m // 2, m - 2, m - 1]):
        assert torch.equal(product(torch.tensor(rows, device=DEV)), got[rows]), "a row's bits must not depend on the rows beside it"


@pytest.mark.parametrize("act", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("m,n,k", [(3, 2 * 88, 64), (8, 2 * 7, 100), (20, 2 * 2100, 36), (70, 2 * 70, 64), (200, 2 * 3000, 96)])
def test_gated(ops, act, m, n, k):
    x, w = operands(m, n, k, m + n)
    z, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    gate, up = z[:, :n // 2], z[:, n // 2:]
    f = torch.nn.functional.silu(gate) if act == "silu" else torch.nn.functional.gelu(gate, approximate="tanh")
    # (both activations' slopes stay below 1.2; tanhf and expf are good to a few units)
    bound = 1.2 * (k + 2) * U * size[:, :n // 2] * up.abs() + f.abs() * (k + 2) * U * size[:, n // 2:] + 16 * U * (gate.abs() * up.abs())
    held(ops.gemm_f32(x.to(DEV), w.to(DEV), act=act), f * up, bound * 1.01 + 1e-30, act)
    assert torch.equal(ops.gemm_f32(x[1:2].to(DEV), w.to(DEV), act=act)[0], ops.gemm_f32(x.to(DEV), w.to(DEV), act=act)[1])
    held(ops.gemm_swiglu(x.to(DEV), w.to(DEV), act=act), f * up, bound * 1.01 + 1e-30, act)


def test_what_it_refuses_goes_to_the_plain_product(ops):
    from bare_cuda_4gib_amd.parts.linear import linear
    x, w = operands(3, 40, 64, 1)
    xd, wd = x.to(DEV), w.to(DEV)
    assert ops.gemm_f32(xd.bfloat16(), wd) is None and ops.gemm_f32(xd[:, :63].contiguous(), wd[:, :63].contiguous()) is None
    shifted = torch.empty(3 * 64 + 1, device=DEV)[1:].view(3, 64).copy_(xd)
    assert ops.gemm_f32(shifted, wd) is None
    torch.testing.assert_close(linear(shifted, wd).cpu().double(), x.double() @ w.double().T, rtol=1e-5, atol=1e-5 * math.sqrt(64))
    x[1, 5] = float("inf")
    got = linear(x.to(DEV), wd).cpu()
    assert torch.isinf(got[1]).all() and torch.isfinite(got[[0, 2]]).all()
