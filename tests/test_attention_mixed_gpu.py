"""Prompt portions and decoded tokens in one launch: the work list of a step with both, run against the plain float kernel and against the
two launches that serve the same step where a context is too long to share; requests without cached tokens, of one row and a whole tile of rows,
walks cut into up to eight parts, a window, groups of 1 to 20 heads."""
import math
import random
import types

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
REQUESTS = [(700, 1), (0, 270), (256, 2), (33, 5), (1000, 1), (511, 130), (4090, 1), (0, 1), (31, 1), (300, 16)]


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from bare_cuda_4gib_amd.csrc import ops as _ops
    return _ops


@pytest.mark.parametrize("nh,nkv,d,page", [(32, 4, 64, 64), (4, 4, 16, 16), (8, 1, 128, 16), (40, 2, 80, 32), (2, 1, 256, 16)])
@pytest.mark.parametrize("window", [0, 300])
def test_portions_and_tokens_together(ops, nh, nkv, d, page, window, monkeypatch):
    requests = list(REQUESTS)
    random.Random(nh).shuffle(requests)
    gen = torch.Generator().manual_seed(d)
    start, pages = [0], [-(-(c + n) // page) for c, n in requests]
    for _, n in requests:
        start.append(start[-1] + n)
    total, order = sum(pages), torch.randperm(sum(pages) + 1, generator=gen).tolist()
    table = torch.zeros(len(requests), max(pages), dtype=torch.int32)
    for s, n in enumerate(pages):
        table[s, :n] = torch.tensor([order.pop() for _ in range(n)], dtype=torch.int32)
    kc, vc = (torch.randn(total + 1, nkv, *shape, generator=gen).bfloat16().to(DEV) for shape in ((page, d), (d, page)))
    qkv = torch.randn(start[-1], (nh + 2 * nkv) * d, generator=gen).bfloat16().to(DEV)
    dev = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    batch = types.SimpleNamespace(n_seqs=len(requests), n_tokens=start[-1], seq_start=start, seq_ctx=[c for c, _ in requests],
                                  max_q_len=max(n for _, n in requests))
    ctx = types.SimpleNamespace(**vars(batch), seq_start_dev=dev(start), seq_ctx_dev=dev(batch.seq_ctx), max_kv_len=max(c + n for c, n in requests),
                                row_seq=dev([s for s, (_, n) in enumerate(requests) for _ in range(n)]), cache_passes=False,
                                positions=dev([c + i for c, n in requests for i in range(n)]))
    scale = 1.0 / math.sqrt(d)

    def run():
        arrays, notes = ops.attention_plan(batch, nh, nkv, d, window)
        junk = torch.full((8 * start[-1] * nh * (d + 2),), float("nan"), device=DEV)      # (what a merge may read and nobody wrote would show)
        del junk
        return ops.attention(qkv, *ops.cache_from_plain(kc, vc), table.to(DEV), ctx, ({k: dev(v) for k, v in arrays.items()}, notes), nh, nkv, d, window,
                             scale), notes
    together, notes = run()
    assert notes["together"] and notes["apart"] and notes["most_parts"] > 1
    plain = ops.attention_generic(qkv, kc, vc, table.to(DEV), ctx.row_seq, ctx.positions, nh, nkv, d, window, scale)
    monkeypatch.setattr(ops, "ATTENTION_TOGETHER_CONTEXT", 4000)
    apart, notes = run()
    assert notes["apart"] and not notes["together"]
    # weights and outputs are rounded to bfloat16 in both: 2 ** -9 of a value each, of 16 to 256 values a head.  By head and row, as outputs shrink with
    # the context: of the row at 4,090 tokens, cut into the most parts, any one tile of 32 keys is 2 to 5 times this bound (in 64 bits, 150 rows).
    for got, want, what in ((together, plain, "plain"), (together, apart, "two launches")):
        off, size = ((t.float().view(start[-1], nh, d).abs().amax(2)) for t in (got.float() - want.float(), want))
        assert float((off / (2.0 ** -6 * size + 1e-6)).max()) <= 1.0, what
