"""A sandwich layer's last add made by the kernel with the next layer's norm and convolution: the bits of the two kernels one after the
other, at widths below, at and beyond a workgroup's pieces; and what the layers do where that kernel does not take the step."""
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from bare_cuda_4gib_amd.csrc import ops as _ops
    return _ops


def _ctx(n, handoff=None):
    slots = list(range(n))[::-1]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)      # noqa: E731
    return SimpleNamespace(n_tokens=n, n_seqs=n, seq_slots=slots, seq_slots_dev=i32(slots), seq_start=list(range(n + 1)), seq_start_dev=i32(list(range(n + 1))),
                           row_seq=i32(list(range(n))), seq_ctx=[5] * n, seq_ctx_dev=i32([5] * n), handoff=handoff, positions=i32([5] * n))


@pytest.mark.parametrize("hidden", [8, 64, 2040, 2048, 2056, 4096])
@pytest.mark.parametrize("taps,rows", [(2, 1), (3, 5), (4, 8)])
@pytest.mark.parametrize("dtype,g_dtype", [(torch.bfloat16, torch.float32), (torch.float32, torch.bfloat16)])
def test_add_norm_conv_gives_the_bits_of_two_kernels(ops, hidden, taps, rows, dtype, g_dtype):
    torch.manual_seed(hidden + taps)
    f = lambda *shape: torch.randn(*shape, device=DEV)      # noqa: E731
    x, y, aw, g, w, b = f(rows, hidden), f(rows, hidden) * 3, f(hidden), f(hidden).to(g_dtype), f(taps, hidden), f(hidden)
    state = f(rows, taps - 1, hidden).to(dtype)
    ctx = _ctx(rows)
    one, two, s1, s2 = x.clone(), x.clone(), state.clone(), state.clone()
    ops.rmsnorm_add(one, y, aw, 1e-5, next_norm=(g, 1e-6, dtype))       # (the kernel that holds a row, also for narrow ones)
    want = ops.rmsnorm_conv(one, g, 1e-6, dtype, w, s1, ctx, bias=b)
    got = ops.rmsnorm_conv(two, g, 1e-6, dtype, w, s2, ctx, bias=b, adds=(y, aw, 1e-5))
    assert torch.equal(one, two) and torch.equal(want, got) and torch.equal(s1, s2)


@pytest.mark.parametrize("hidden,rows", [(2048, 8), (4104, 3), (96, 2)])      # (4,104: beyond the kernel's width)
def test_blocks_that_leave_their_last_output_to_the_next(ops, hidden, rows):
    from bare_cuda_4gib_amd.parts.block import SandwichBlock
    from bare_cuda_4gib_amd.parts.conv import CausalConv
    from bare_cuda_4gib_amd.parts.lazy import NormHandoff
    from bare_cuda_4gib_amd.parts.norm import RMSNorm
    torch.manual_seed(hidden)
    rt = SimpleNamespace(act_dtype=torch.bfloat16, device=torch.device(DEV))
    mats = [torch.randn(hidden, hidden, device=DEV) * hidden ** -0.5 for _ in range(3)]

    class Mixer:
        adds_one_product = True

        def __init__(self, m):
            self.m = m

        def forward(self, h, ctx, cache, y, writes):
            y.tensor = (h.float() @ self.m).contiguous()

    def block(m):
        norms = [RMSNorm(hidden, 1e-5, offset=1.0) for _ in range(2)]
        for norm in norms:
            norm.bind({"weight": torch.randn(hidden, device=DEV) * 0.1}, rt)
        conv = CausalConv(hidden, 3)
        conv.bind({"weight": torch.randn(hidden, 3, device=DEV) * 0.3}, rt)
        return SandwichBlock(Mixer(m), *norms, mixer_conv=conv)

    blocks = [block(m) for m in mats]
    tails = [torch.randn(rows, 2, hidden, device=DEV).bfloat16() for _ in blocks]
    start = torch.randn(rows, hidden, device=DEV)

    def run(handed):
        handoff = NormHandoff()
        x, states = start.clone(), [t.clone() for t in tails]
        ctx = _ctx(rows, handoff)
        for i, b in enumerate(blocks):
            handoff.begin_entry(b, blocks[i + 1] if handed and i + 1 < len(blocks) else None, rows)
            b.forward(x, ctx, SimpleNamespace(mixer=None, conv=SimpleNamespace(tail=states[i])))
        return x, states

    (a, sa), (b, sb) = run(False), run(True)
    assert torch.equal(a, b) and all(torch.equal(p, q) for p, q in zip(sa, sb))
