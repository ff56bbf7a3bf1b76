"""Decode attention whose last part merges: the bits of the merge kernels, whichever part ends last, launch after launch and from a captured
graph, with the counters zero again behind every launch."""
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


# (requests, heads, key/value heads, head size, rows a request, longest context): one group of heads and several, tiles of several tokens, heads of
# 64, 128 and 256, heads that no tile is full of, and parts without any key (short contexts beside the longest)
CASES = [(1, 32, 4, 64, 1, 2000), (8, 32, 4, 64, 1, 600), (3, 32, 8, 128, 1, 4000), (2, 4, 2, 16, 3, 300), (5, 40, 2, 64, 1, 900), (1, 8, 4, 256, 2, 700),
         (16, 8, 1, 128, 1, 3000)]


@pytest.mark.parametrize("n_splits", [2, 3, 8, 9, 17, 64])
@pytest.mark.parametrize("S, heads, kv_heads, d, rows, longest", CASES)
def test_the_last_part_merges(ops, S, heads, kv_heads, d, rows, longest, n_splits):
    gen = torch.Generator().manual_seed(S * 131 + n_splits)
    page, group = 64, heads // kv_heads
    width = -(-longest // page)
    pages = S * width
    draw = lambda *shape: torch.randn(*shape, generator=gen).bfloat16().to(DEV)      # noqa: E731
    kc, vc, q = draw(pages, kv_heads, page, d), draw(pages, kv_heads, d, page), draw(S * rows, heads * d)
    table = torch.randperm(pages, generator=gen).view(S, width).int().to(DEV)
    ctx = torch.tensor([longest - rows if s == 0 else int(torch.randint(0, longest - rows, (1,), generator=gen)) for s in range(S)], dtype=torch.int32, device=DEV)
    start = (torch.arange(S + 1, dtype=torch.int32) * rows).to(DEV)
    tpt = ops.attention_tile_tokens(heads, kv_heads)
    tiles_each = -(-rows // tpt)
    tiles = (torch.arange(S + 1, dtype=torch.int32) * tiles_each).to(DEV)
    n_tiles = S * tiles_each
    arrived = torch.zeros(n_tiles * kv_heads * -(-group // 16), dtype=torch.int32, device=DEV)

    def run(counters):
        return ops.attention_mfma(q, kc, vc, table, start, ctx, tiles, n_tiles, heads, kv_heads, d, 0, d ** -0.5, n_splits, 1, 1,
                                  single_rows=rows == 1 and tiles_each == 1, arrived=counters)
    want = run(None)
    for _ in range(3):
        assert torch.equal(run(arrived), want) and not arrived.any()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            got = [run(arrived) for _ in range(4)]
        for _ in range(3):
            for one in got:
                one.zero_()
            graph.replay()
            stream.synchronize()
            assert all(torch.equal(one, want) for one in got) and not arrived.any()


# more parts than are asked for together; more outputs a tile than threads: 8 heads of 128, 4 of 256
@pytest.mark.parametrize("heads, kv_heads, d, n_splits, used", [(8, 8, 64, 8, True), (8, 8, 64, 9, False), (8, 1, 64, 8, True), (4, 1, 128, 8, True), (8, 1, 128, 2, False),
                                                                (1, 1, 256, 8, True), (2, 1, 256, 2, False)])
def test_counters_are_left_alone_where_a_kernel_merges(ops, heads, kv_heads, d, n_splits, used):
    gen = torch.Generator().manual_seed(d + n_splits)
    draw = lambda *shape: torch.randn(*shape, generator=gen).bfloat16().to(DEV)      # noqa: E731
    kc, vc, q = draw(8, kv_heads, 64, d), draw(8, kv_heads, d, 64), draw(1, heads * d)
    table, rows = torch.arange(8, dtype=torch.int32, device=DEV).view(1, 8), torch.arange(2, dtype=torch.int32, device=DEV)
    arrived = torch.full((kv_heads,), 0 if used else 77, dtype=torch.int32, device=DEV)
    run = lambda counters: ops.attention_mfma(q, kc, vc, table, rows, rows[1:] * 500, rows, 1, heads, kv_heads, d, 0, d ** -0.5, n_splits, 1, 1,      # noqa: E731
                                              single_rows=True, arrived=counters)
    assert torch.equal(run(arrived), run(None)) and (arrived == (0 if used else 77)).all()


@pytest.mark.parametrize("n_splits", [2, 8])
@pytest.mark.parametrize("heads, kv_heads, d", [(8, 2, 64), (32, 4, 64), (4, 4, 128)])
def test_short_requests_beside_others(ops, heads, kv_heads, d, n_splits):
    """A mixed step: tiles of the short requests alone, rows of the others left as another launch made them."""
    gen = torch.Generator().manual_seed(heads + n_splits)
    new, lengths, width = [1, 70, 2, 1, 33, 1], [900, 0, 40, 1500, 64, 3], 26
    S, rows = len(new), sum(new)
    draw = lambda *shape: torch.randn(*shape, generator=gen).bfloat16().to(DEV)      # noqa: E731
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)      # noqa: E731
    kc, vc, q = draw(S * width, kv_heads, 64, d), draw(S * width, kv_heads, d, 64), draw(rows, heads * d)
    table = torch.randperm(S * width, generator=gen).view(S, width).int().to(DEV)
    starts, tiles, tpt = [0], [0], ops.attention_tile_tokens(heads, kv_heads)
    for n in new:
        starts.append(starts[-1] + n)
        tiles.append(tiles[-1] + (-(-n // tpt) if n <= tpt else 0))
    row_seq = i32([s for s, n in enumerate(new) for _ in range(n)])
    others, arrived = draw(rows, heads * d), torch.zeros(tiles[-1] * kv_heads, dtype=torch.int32, device=DEV)

    def run(counters):
        return ops.attention_mfma(q, kc, vc, table, i32(starts), i32(lengths), i32(tiles), tiles[-1], heads, kv_heads, d, 0, d ** -0.5, n_splits, 1, 1,
                                  out=others.clone(), row_seq=row_seq, arrived=counters)
    want = run(None)
    long_rows = torch.tensor([n > tpt for n in new], device=DEV)[row_seq.long()]
    assert torch.equal(want[long_rows], others[long_rows]) and not torch.equal(want[~long_rows], others[~long_rows])
    for _ in range(3):
        assert torch.equal(run(arrived), want) and not arrived.any()


def test_too_few_counters_are_refused(ops):
    from bare_cuda_4gib_amd.errors import KernelError
    z = lambda *shape: torch.zeros(*shape, dtype=torch.int32, device=DEV)      # noqa: E731
    kc = torch.zeros(4, 2, 64, 64, dtype=torch.bfloat16, device=DEV)
    q = torch.zeros(2, 8 * 64, dtype=torch.bfloat16, device=DEV)
    tiles = torch.arange(3, dtype=torch.int32, device=DEV)
    with pytest.raises(KernelError, match="counters are fewer"):
        ops.attention_mfma(q, kc, kc.view(4, 2, 64, 64), z(2, 2), tiles, z(2), tiles, 2, 8, 2, 64, 0, 0.125, 2, 1, 1, arrived=z(3))


def test_counters_go_up_with_the_batch(ops):
    assert ops.attention_counters(8, 32, 4) == {"arrived": [0] * 32} and ops.attention_counters(33, 32, 4) == {} == ops.attention_counters(0, 32, 4)
    assert ops.attention_counters(1, 64, 2) == {"arrived": [0] * 4}


@pytest.mark.parametrize("n_splits", [1, 3])
@pytest.mark.parametrize("counted", [False, True])
@pytest.mark.parametrize("S, heads, kv_heads, d", [(16, 32, 8, 64), (8, 32, 8, 128), (4, 8, 8, 256), (5, 16, 16, 80)])
def test_past_the_caches_as_through_them(ops, S, heads, kv_heads, d, n_splits, counted):
    """Keys and values read past the caches, and tables with room for much more than the contexts, with the last part merging and with a kernel behind it."""
    gen = torch.Generator().manual_seed(S + d)
    page, width = 64, 4
    draw = lambda *shape: torch.randn(*shape, generator=gen).bfloat16().to(DEV)      # noqa: E731
    kc, vc, q = draw(S * width, kv_heads, page, d), draw(S * width, kv_heads, d, page), draw(S, heads * d)
    table = torch.randperm(S * width, generator=gen).view(S, width).int().to(DEV)
    ctx = torch.randint(1, width * page, (S,), generator=gen).int().to(DEV)
    rows = torch.arange(S + 1, dtype=torch.int32, device=DEV)
    room = -(-(32 << 20) // (S * page * kv_heads * d * 4))
    wide = torch.full((S, room), -1, dtype=torch.int32, device=DEV)
    wide[:, :width] = table
    arrived = torch.zeros(S * kv_heads, dtype=torch.int32, device=DEV) if counted else None
    run = lambda t, past: ops.attention_mfma(q, kc, vc, t, rows, ctx, rows, S, heads, kv_heads, d, 0, d ** -0.5, n_splits, 1, 1, single_rows=True,      # noqa: E731
                                             arrived=arrived, past_caches=past)
    want = run(table, False)
    assert room > width and all(torch.equal(run(t, past), want) for t in (table, wide) for past in (False, True))
    assert arrived is None or not arrived.any()
