"""The float32 products of parts (gemm_f32.hip) where they can go wrong beside what test_gemm_f32_gpu.py asks: products cut into quarters of k, tiles of
33 to 64 rows, a k that ends inside a pair of shares, and operands that three bfloat16 cannot hold.

Tolerance: a float32 sum of k products, in any order, is off by at most k 2^-24 sum |x w|."""
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


def operands(m, n, k, seed, scale=1.0):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    f = lambda *shape: torch.randn(*shape, generator=gen, device=DEV)      # noqa: E731
    return f(m, k) * scale, f(n, k) * 0.1


def quarters(ops, m, n, k):
    """Whether the product is cut into quarters: it then wants room for their sums beside x's parts."""
    return ops._gemm_f32_scratch(m, n, k) == -(-m // 16) * (k // 32) * 3072 + 16 * m * n


# Every tile cut into quarters (rows and columns that end inside one, a last quarter that is short or empty, outputs that are no whole 16 bytes),
# and tiles at the fewest rows.
@pytest.mark.parametrize("m,n,k", [(100, 2560, 2048), (193, 2050, 2080), (300, 2046, 5632), (256, 2048, 1056), (700, 642, 4128), (129, 1030, 14336),
                                   (120, 8190, 7168), (33, 11264, 2048), (64, 11262, 544)])
@pytest.mark.parametrize("epilogue", ["store", "add with bias", "silu"])
def test_quarters(ops, m, n, k, epilogue):
    x, w = operands(m, n, k, m + k)
    base, bias = torch.randn(m, n, device=DEV), torch.randn(n, device=DEV)
    assert ops.gemm_f32_tile(m, n, k) != (0, 0) and quarters(ops, m, n, k) == (m != 64)

    def product(rows):
        if epilogue == "add with bias":
            return ops.gemm_f32(x[rows].clone(), w, accumulate_into=base[rows].clone(), bias=bias)
        return ops.gemm_f32(x[rows].clone(), w, act=None if epilogue == "store" else epilogue)

    got, z, size = product(slice(0, m)), x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    if epilogue == "silu":
        gate, up = z[:, :n // 2], z[:, n // 2:]
        want = torch.nn.functional.silu(gate) * up
        bound = 1.25 * (k + 18) * U * (size[:, :n // 2] * up.abs() + gate.abs() * size[:, n // 2:]) + 1e-30
    elif epilogue == "store":
        want, bound = z, (k + 2) * U * size
    else:
        want, bound = z + base.double() + bias.double(), (k + 4) * U * (size + base.double().abs() + bias.double().abs())
    assert float(((got.double() - want).abs() / bound).max()) <= 1.0
    for rows in ([0], [m // 2, m - 1], list(range(min(m, 12)))):
        assert torch.equal(product(torch.tensor(rows, device=DEV)), got[rows]), "a row's bits must not depend on the rows beside it"


@pytest.mark.parametrize("m", [3, 8, 12, 40, 100, 1000])
def test_what_parts_cannot_hold(ops, m):
    """Rows with an infinity, a NaN, the largest float and floats near the smallest normal one: as plain float gives them, the others' bits unmoved."""
    n, k = 96, 256
    x, w = operands(m, n, k, m)
    plain = ops.gemm_f32(x, w)
    x[0, 5] = float("inf")
    x[1, 200] = float("nan")
    x[2] *= 2.0 ** -118
    got = ops.gemm_f32(x, w)
    assert torch.equal(torch.isposinf(got[0]), w[:, 5] > 0) and torch.equal(torch.isneginf(got[0]), w[:, 5] < 0)
    assert bool(torch.isnan(got[1]).all()) and torch.equal(got[3:], plain[3:])
    z, size = x[2].double() @ w.double().T, x[2].double().abs() @ w.double().abs().T
    assert float(((got[2].double() - z).abs() / ((k + 2) * U * size)).max()) <= 1.0
    x[0] = 0.0
    x[0, 7], x[1], w[3, 7] = torch.finfo(torch.float32).max, 1.0, 0.5
    got = ops.gemm_f32(x, w)
    assert float(got[0, 3]) == torch.finfo(torch.float32).max / 2 and bool(torch.isfinite(got[1]).all())


def small_and_large(seed, m, n, k, x_exp, w_exp):
    gen = torch.Generator().manual_seed(seed)
    at = lambda rows, exp: (torch.randn(rows, k, generator=gen, dtype=torch.float64) * 2.0 ** exp).float()      # noqa: E731
    return at(m, x_exp), at(n, w_exp)


# Operands down to the smallest denormals beside large ones, whichever of the two is small: every bit of an operand counts, however small it is.
@pytest.mark.parametrize("m,n,k", [(3, 96, 256), (8, 96, 256), (8, 8200, 256), (12, 96, 256), (40, 96, 260), (100, 96, 256), (1000, 96, 256), (300, 2050, 1056)])
@pytest.mark.parametrize("x_exp,w_exp", [(-112, 60), (-122, 60), (-125, 70), (-140, 75), (70, -125), (60, -140), (-70, -60), (-75, -70)])
def test_small_operands(ops, m, n, k, x_exp, w_exp):
    x, w = small_and_large(m + k, m, n, k, x_exp, w_exp)
    got = ops.gemm_f32(x.to(DEV), w.to(DEV)).double().cpu()
    z, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    # (a sum below the smallest normal float is rounded to multiples of 2^-149, each share's at most)
    assert float(((got - z).abs() / ((k + 2) * U * size + 20 * 2.0 ** -149)).max()) <= 1.0


@pytest.mark.parametrize("m", [3, 8, 12, 40, 100])
def test_what_is_left_of_small_operands_that_cancel(ops, m):
    """Products that take each other off but for the last bits of a small operand, and a sum of tiny products: neither is nothing."""
    n, k = 32, 256
    x, w = torch.zeros(m, k), torch.zeros(n, k)
    x[:, 3], x[:, 200], w[:, 3], w[:, 200] = 2.0 ** -120 * (1 + 2.0 ** -23), -(2.0 ** -120), 2.0 ** 100, 2.0 ** 100
    assert bool((ops.gemm_f32(x.to(DEV), w.to(DEV)) == 2.0 ** -43).all())
    x, w = torch.full((m, k), 2.0 ** -70), torch.full((n, k), 2.0 ** -70)
    assert bool((ops.gemm_f32(x.to(DEV), w.to(DEV)) == 2.0 ** -132).all())


@pytest.mark.parametrize("m", [3, 8, 12, 40, 100])
def test_large_operands_and_sums(ops, m):
    """Beyond what the parts hold: operands up to the largest float, sums that are finite and such as are not."""
    n, k = 40, 256
    x, w = small_and_large(m, m, n, k, 100, 15)
    x[0, 5], w[:, 5] = torch.finfo(torch.float32).max, 0.25
    x[1] = 2.0 ** 100
    w[7] = 2.0 ** 30
    got = ops.gemm_f32(x.to(DEV), w.to(DEV)).double().cpu()
    z, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    live = size < 2.0 ** 127
    assert float(((got - z).abs() / ((k + 2) * U * size))[live].max()) <= 1.0 and bool(torch.isposinf(got[1, 7])) and not bool(live[1, 7])


INVALID = [(3, 96, 256), (8, 2048, 2080), (8, 11264, 512), (16, 90, 260), (40, 2050, 2048), (100, 2560, 2048), (300, 2046, 1056), (1000, 2562, 1056)]


@pytest.mark.parametrize("m,n,k", INVALID)
@pytest.mark.parametrize("epilogue", ["store", "add with bias", "silu"])
def test_invalid_and_infinite_sums(ops, m, n, k, epilogue):
    """What float arithmetic gives of them, in every kernel: a NaN, infinities of both signs and beside zeros, sums beyond the parts' range and
    beyond float's.  The finite ones have the same bits whatever rows are beside them, and so have the rows without any of these."""
    x, w = operands(m, n, k, m + n)
    base, bias = torch.randn(m, n, device=DEV), torch.randn(n, device=DEV)

    def product(rows):
        if epilogue == "add with bias":
            return ops.gemm_f32(x[rows].clone(), w, accumulate_into=base[rows].clone(), bias=bias)
        return ops.gemm_f32(x[rows].clone(), w, act=None if epilogue == "store" else epilogue)

    every = torch.arange(m, device=DEV)
    before = product(every)
    x[0, k // 2], x[1, k - 1] = float("nan"), -float("inf")
    x[m - 1] *= 2.0 ** 90
    w[n - 1, k - 1] = 0.0
    got = product(every)
    w_last = w[:, k - 1]
    assert bool(torch.isnan(got[0]).all())
    if epilogue != "silu":
        assert bool(torch.isnan(got[1, n - 1])) and torch.equal(torch.isposinf(got[1]), w_last < 0) and torch.equal(torch.isneginf(got[1]), w_last > 0)
        z, size = x[m - 1].double() @ w.double().T, x[m - 1].double().abs() @ w.double().abs().T
        assert float(((got[m - 1].double() - z).abs() / ((k + 4) * U * size)).max()) <= 1.0
    others = every[2:m - 1]
    assert torch.equal(got[others, :-1], before[others, :-1])
    for rows in ([m - 1], [0, m - 1], [1, 0, m - 1]):
        assert torch.equal(product(torch.tensor(rows, device=DEV))[-1], got[m - 1])
    w[:, k // 3] = float("inf")                             # every sum of every row
    x[2:m - 1, k // 3] = 1.0
    got = product(every)
    assert bool((torch.isposinf(got) | torch.isnan(got))[2:m - 1].all())


@pytest.mark.parametrize("m,n,k", [(1000, 11264, 2048), (256, 2048, 5632), (64, 11264, 2048), (8, 2048, 5632)])
@pytest.mark.parametrize("what", ["all NaN", "an infinity a row", "one infinity"])
def test_invalid_rows_do_not_hold_up_the_others(ops, m, n, k, what):
    """A product with them takes a few times what it takes without (before they were added up by whole waves: 30 to 160 times)."""
    x, w = operands(m, n, k, 1)
    bad = x.clone()
    if what == "all NaN":
        bad[:] = float("nan")
    else:
        bad[:m if what == "an infinity a row" else 1, k // 2] = float("inf")

    def fastest(y):
        best = math.inf
        for _ in range(6):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record(), ops.gemm_f32(y, w), b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        return best
    assert fastest(bad) < 12.0 * fastest(x)


@pytest.mark.parametrize("kind", ["normal", "one sign", "one value", "every other share small", "every other share small, one sign"])
@pytest.mark.parametrize("m,n,k", [(8, 96, 2048), (16, 96, 14336), (64, 96, 5632), (300, 96, 14336)])
def test_error_of_lopsided_operands(ops, m, n, k, kind):
    """The matrix cores round sums down, and what cures that -- every other share of k is added up negated -- counts on shares alike: whatever the
    operands, the error's root mean square is at most twice that of plain float additions in the same sixteen shares."""
    gen = torch.Generator().manual_seed(k)
    x, w = torch.randn(m, k, generator=gen), torch.randn(n, k, generator=gen)
    share = -(-k // 512) * 32
    if kind == "one value":
        x[:], w[:] = 1.0 / 3.0, 1.0 / 7.0
    if kind.startswith("every other"):
        x = torch.where(torch.arange(k) // share % 2 == 1, x * 2.0 ** -12, x)
    if kind.endswith("one sign"):
        x, w = x.abs(), w.abs()
    z = x.double() @ w.double().T
    got = ops.gemm_f32(x.to(DEV), w.to(DEV)).double().cpu()
    rows, plain = min(m, 16), 0.0
    for first in range(0, k, share):
        part = torch.zeros(rows, n)
        for i in range(first, min(k, first + share)):
            part = (part.double() + x[:rows, i:i + 1].double() * w[:, i].double()).float()
        plain = part if first == 0 else plain + part
    rms = lambda t: float(t.double().square().mean().sqrt())      # noqa: E731
    assert rms(got - z) <= 2.0 * max(rms(plain.double() - z[:rows]), 2.0 ** -26 * rms(z))


def test_too_little_scratch_memory_is_refused(ops):
    """Before anything is launched, whoever worked the size out."""
    m, n, k = 300, 2048, 5632
    x, w = operands(m, n, k, 3)
    wants, out = ops._gemm_f32_scratch(m, n, k), torch.zeros(m, n, device=DEV)
    scratch = torch.empty(wants, dtype=torch.uint8, device=DEV)
    many = lambda nbytes: ops.library.call("bc4g_gemm_f32_many", x.data_ptr(), w.data_ptr(), None, out.data_ptr(), scratch.data_ptr(), nbytes, 0,      # noqa: E731
                                           m, n, k, torch.cuda.current_stream().cuda_stream)
    with pytest.raises(ops.KernelError, match="scratch memory"):
        many(wants - 1)
    assert not bool(out.any())
    many(wants)
    assert torch.equal(out, ops.gemm_f32(x, w))


@pytest.mark.parametrize("m,n,k", [(12600, 642, 14336), (25001, 322, 14336)])
@pytest.mark.parametrize("epilogue", ["store", "add with bias", "silu"])
def test_rows_in_blocks(ops, m, n, k, epilogue):
    """So many that their parts would pass what a product may take: blocks of rows, one after the other, with the bits of few rows."""
    assert -(-m // 16) * (k // 32) * 3072 > ops.PRODUCT_SCRATCH_BYTES[4] >= ops._gemm_f32_scratch(m, n, k) > 0
    x, w = operands(m, n, k, m)
    base, bias = torch.randn(m, n, device=DEV), torch.randn(n, device=DEV)

    def product(rows):
        if epilogue == "add with bias":
            return ops.gemm_f32(x[rows].contiguous(), w, accumulate_into=base[rows].clone(), bias=bias)
        return ops.gemm_f32(x[rows].contiguous(), w, act=None if epilogue == "store" else epilogue)

    got = product(slice(0, m))
    for first in list(range(0, m - 5, 1021)) + [m - 5]:
        assert torch.equal(product(slice(first, first + 5)), got[first:first + 5])


def without_scratch(ops, x, w, epilogue, out, bias=None):
    (m, k), n = x.shape, w.shape[0]
    ops.library.call("bc4g_gemm_f32", x.data_ptr(), w.data_ptr(), bias.data_ptr() if bias is not None else None, out.data_ptr(),
                     {"store": 0, "add with bias": 1, "silu": 2, "gelu_tanh": 3}[epilogue], m, n, k, torch.cuda.current_stream().cuda_stream)
    return out


# Callers without scratch memory: tiles of each size whose waves split x themselves, rows and columns that end inside one, k that ends inside a pair.
@pytest.mark.parametrize("m,n,k", [(1000, 2562, 1056), (1793, 2050, 544), (300, 8190, 96), (129, 11262, 2080), (700, 1030, 4128), (65, 28672, 64), (40, 2048, 2048)])
@pytest.mark.parametrize("epilogue", ["store", "add with bias", "silu", "gelu_tanh"])
def test_without_scratch_memory(ops, m, n, k, epilogue):
    x, w = operands(m, n, k, m + 2 * k)
    base, bias = torch.randn(m, n, device=DEV), torch.randn(n, device=DEV) if epilogue == "add with bias" else None
    x[m - 2, k - 3], x[m // 2, 1] = float("nan"), float("inf")
    out = base.clone() if bias is not None else torch.full((m, n if epilogue == "store" else n // 2), -7.0, device=DEV)
    got = without_scratch(ops, x, w, epilogue, out, bias)
    want = ops.gemm_f32(x, w, accumulate_into=base.clone(), bias=bias) if bias is not None else ops.gemm_f32(x, w, act=None if epilogue == "store" else epilogue)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(got.nan_to_num(), want.nan_to_num())


def test_many_rows_without_scratch_memory_go_to_tiles(ops):
    """They take up to twice the time of a product with it (the few rows' kernel, where they went in between: 2.5 times)."""
    x, w = operands(1000, 11264, 2048, 5)
    out = torch.empty(1000, 11264, device=DEV)

    def fastest(f):
        best = math.inf
        for _ in range(8):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record(), f(), b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        return best
    assert fastest(lambda: without_scratch(ops, x, w, "store", out)) < 2.0 * fastest(lambda: ops.gemm_f32(x, w))
