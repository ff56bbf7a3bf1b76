"""The kernels of a layer normed on both sides in a decode step, against the launches each takes the place of: the same bits."""
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from bare_cuda_4gib_amd.csrc import ops as o
    return o


def single_rows(slots):
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)      # noqa: E731
    n = len(slots)
    return SimpleNamespace(n_tokens=n, n_seqs=n, seq_slots=list(slots), seq_slots_dev=i32(slots), row_seq=i32(list(range(n))),
                           seq_start=list(range(n + 1)), seq_start_dev=i32(list(range(n + 1))))


@pytest.mark.parametrize("hidden", [8, 1000, 2048, 2056, 4096, 5120, 8192, 8200, 77])
@pytest.mark.parametrize("y_dtype, w_dtype, out_dtype", [(torch.float32, torch.float32, torch.bfloat16), (torch.bfloat16, torch.bfloat16, torch.float32),
                                                         (torch.float32, torch.float32, torch.float32)])
def test_add_and_the_norm_after_it(ops, hidden, y_dtype, w_dtype, out_dtype):
    torch.manual_seed(hidden)
    x, y = torch.randn(5, hidden, device=DEV), (torch.randn(5, hidden, device=DEV) * 3).to(y_dtype)
    w, g = torch.randn(hidden, device=DEV), torch.randn(hidden, device=DEV).to(w_dtype)
    yd = y.double()
    want = x.double() + yd * torch.rsqrt((yd * yd).mean(1, keepdim=True) + 1e-3) * w.double()
    alone, both = x.clone(), x.clone()
    assert ops.rmsnorm_add(alone, y, w, 1e-3) is alone
    made = ops.rmsnorm_add(both, y, w, 1e-3, next_norm=(g, 1e-5, out_dtype))
    # (a few roundings of 2^-24 of each term, which are below 8 * 4 here)
    assert float((alone.double() - want).abs().max()) <= 32 * 4 * 2.0 ** -24
    assert torch.equal(alone, both)
    assert (made is None) == (hidden in (8200, 77))
    if made is not None:
        assert torch.equal(made, ops.rmsnorm(alone, g, 1e-5, out_dtype))


def beside(t):
    """The same values one element beside a 16-byte boundary: what only the scalar kernels take."""
    room = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    room[1:] = t.reshape(-1)
    return room[1:].view(t.shape)


@pytest.mark.parametrize("y_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("hidden", [8, 1000, 2048, 2056, 5120, 8192])
def test_rows_held_in_registers_add_what_the_scalar_kernel_adds(ops, hidden, y_dtype):
    torch.manual_seed(hidden)
    x, y, w = torch.randn(5, hidden, device=DEV), (torch.randn(5, hidden, device=DEV) * 3).to(y_dtype), torch.randn(hidden, device=DEV)
    scalar = beside(x)
    ops.rmsnorm_add(scalar, y, w, 1e-3)
    ops.rmsnorm_add(x, y, w, 1e-3)
    assert torch.equal(x, scalar)


@pytest.mark.parametrize("g_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("hidden", [8, 512, 520, 2048, 5120, 6136])
def test_norm_prepared_by_the_add_is_the_norm_a_product_absorbs(ops, hidden, g_dtype):
    """Float products of 8 rows: a sum of squares that differs in its last bit would show in them."""
    torch.manual_seed(hidden)
    w, g = (torch.randn(64, hidden, device=DEV) * hidden ** -0.5).to(torch.bfloat16), torch.randn(hidden, device=DEV).to(g_dtype)
    for _ in range(20):
        x, y = torch.randn(8, hidden, device=DEV), torch.randn(8, hidden, device=DEV)
        pre = ops.rmsnorm_add(x, y, g.float(), 1e-5, next_norm=(g, 1e-6, torch.bfloat16), prepare=True)
        got = ops.gemm_prenormed(pre, w, ops.EPI_STORE_F32)
        assert torch.equal(got, ops.gemm_normed(x, None, 8, g, 1e-6, w, ops.EPI_STORE_F32))


@pytest.mark.parametrize("g_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows", [1, 5, 8, 9, 20])
@pytest.mark.parametrize("hidden, inter", [(64, 200), (1000, 520), (2048, 8192), (4096, 1024)])
def test_feedforward_behind_the_add_gives_what_its_launches_one_by_one_give(ops, hidden, inter, rows, g_dtype):
    """A sandwich layer's second half: the sum added to the stream under its norm, and the product with the activation
    that reads the stream's next norm, which absorbs that norm for few rows."""
    from bare_cuda_4gib_amd.parts.feedforward import DenseXIELU
    from bare_cuda_4gib_amd.parts.lazy import Normed
    from bare_cuda_4gib_amd.parts.linear import linear
    from bare_cuda_4gib_amd.parts.norm import RMSNorm
    from bare_cuda_4gib_amd.parts.block import SandwichBlock
    torch.manual_seed(rows)
    rt = SimpleNamespace(act_dtype=torch.bfloat16, device=torch.device(DEV))
    bf16 = lambda *shape: (torch.randn(*shape, device=DEV) * shape[-1] ** -0.5).to(torch.bfloat16)      # noqa: E731
    norms = [RMSNorm(hidden, 1e-5) for _ in range(4)]
    for norm in norms:
        norm.bind({"weight": (1 + torch.randn(hidden, device=DEV) * 0.2).to(g_dtype)}, rt)
    first, behind, second, last = norms
    ffn = DenseXIELU(hidden, inter)
    ffn.bind({"up": bf16(inter, hidden) * 2, "down": bf16(hidden, inter), "act": torch.tensor([0.4, -0.8], device=DEV)}, rt)
    start, sums = torch.randn(rows, hidden, device=DEV), torch.randn(rows, hidden, device=DEV) * 3

    class Mixer:
        adds_one_product = True

        def forward(self, h, ctx, cache, y, writes):
            y.tensor = sums.clone()

    ctx = SimpleNamespace(n_tokens=rows, handoff=SimpleNamespace(reading_next=None))
    x = start.clone()
    SandwichBlock(Mixer(), first, behind, ffn, second, last).forward(x, ctx, None)
    want = start.clone()
    want_sums = beside(sums)
    behind.add_to(want, want_sums)
    z = linear(Normed(want, second), ffn.w_up, out_dtype=torch.bfloat16)
    y = linear(ops.xielu(z, ffn.pq, out=z), ffn.w_down, out_dtype=torch.float32)
    last.add_to(want, beside(y))
    assert torch.equal(x, want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("hidden", [8, 1032, 2048, 2056, 4096])
@pytest.mark.parametrize("taps, bias", [(2, True), (3, False), (4, True), (4, False)])
def test_norm_and_convolution(ops, dtype, hidden, taps, bias):
    torch.manual_seed(taps)
    slots = [4, 0, 2]
    x = torch.randn(3, hidden, device=DEV)
    g, w = 1 + torch.randn(hidden, device=DEV) * 0.1, torch.randn(taps, hidden, device=DEV)
    b = torch.randn(hidden, device=DEV) if bias else None
    state = torch.randn(6, taps - 1, hidden, device=DEV).to(dtype)
    ctx, other = single_rows(slots), state.clone()
    got = ops.rmsnorm_conv(x, g, 1e-5, dtype, w, state, ctx, bias=b)
    h = ops.rmsnorm(x, g, 1e-5, dtype)
    want = ops.causal_conv(h, w, other, ctx, out_bias=b, add_input=True)
    assert torch.equal(got, want) and torch.equal(state, other)
    two = SimpleNamespace(**{**vars(ctx), "n_seqs": 2})
    assert ops.rmsnorm_conv(x, g, 1e-5, dtype, w, state, two) is None and ops.rmsnorm_conv(x, g, 1e-5, dtype, w[:1], state, ctx) is None


@pytest.mark.parametrize("channels", [8, 2560])
@pytest.mark.parametrize("taps", [2, 3, 4, 5])
@pytest.mark.parametrize("in_bias, out_bias, add", [(True, True, False), (False, False, True), (True, False, True)])
def test_convolution_of_single_rows(ops, channels, taps, in_bias, out_bias, add):
    torch.manual_seed(channels + taps)
    slots = [3, 1, 0]
    wide = torch.randn(3, 2 * channels, device=DEV).to(torch.bfloat16)
    x, w = wide[:, channels:], torch.randn(taps, channels, device=DEV)
    bi, bo = (torch.randn(channels, device=DEV) if on else None for on in (in_bias, out_bias))
    state = torch.randn(5, taps - 1, channels, device=DEV).to(torch.bfloat16)
    before = state.clone()
    got = ops.causal_conv(x, w, state, single_rows(slots), in_bias=bi, out_bias=bo, add_input=add)
    v = (x.float() + bi).to(torch.bfloat16) if in_bias else x
    rows = torch.cat([before[slots], v.unsqueeze(1)], dim=1)
    want = (rows.double() * w.double()).sum(1) + (bo.double() if out_bias else 0) + (x.double() if add else 0)
    # (stored as bfloat16: half a unit of the last of 8 bits, and the sums' own roundings)
    assert bool(((got.double() - want).abs() <= want.abs() * 2.0 ** -8 + 1e-5).all())
    before[slots] = rows[:, 1:]
    assert torch.equal(state, before)


@pytest.mark.parametrize("m", [1, 8, 16, 17, 33, 64])
@pytest.mark.parametrize("n, k", [(24, 40), (5120, 1024), (8, 2048)])
def test_product_with_the_activation(ops, m, n, k):
    from bare_cuda_4gib_amd.parts.linear import linear_xielu
    torch.manual_seed(m)
    a = torch.randn(m, k, device=DEV).to(torch.bfloat16)
    w = ops.StreamedWeight((torch.randn(n, k, device=DEV) * k ** -0.5 * 2).to(torch.bfloat16))
    pq = torch.tensor([0.4, -0.8], device=DEV)
    got = linear_xielu(a, w, pq, torch.bfloat16)
    assert torch.equal(got, ops.xielu(ops.gemm_fast(a, w), pq))
