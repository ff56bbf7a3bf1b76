"""Latent attention of single decoded rows whose keys are cut into parts, beside requests too short to have a key in every part; and the
cache row of sizes beside what a thread holds at once: against the same in float64."""
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
PAGE = 64


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from bare_cuda_4gib_amd.csrc import ops as _ops
    return _ops


def _i32(x):
    return torch.tensor(x, dtype=torch.int32, device=DEV)


@pytest.mark.parametrize("rank,rot,heads", [(512, 64, 16), (256, 64, 5), (64, 32, 20), (96, 32, 16)])
@pytest.mark.parametrize("lengths", [[1, 700, 33, 32], [2050, 31], [1], [65, 64, 63]])
@pytest.mark.parametrize("window", [0, 70])
def test_parts_without_a_key(ops, rank, rot, heads, lengths, window):
    gen = torch.Generator().manual_seed(rank + sum(lengths))
    row, n = rank + rot, len(lengths)
    pages = [-(-x // PAGE) for x in lengths]
    cache = torch.randn(sum(pages), PAGE, row, generator=gen).bfloat16()
    q, sink = torch.randn(n, heads, row, generator=gen), torch.randn(heads, generator=gen)
    order = torch.randperm(sum(pages), generator=gen).tolist()
    table = torch.zeros(n, max(pages), dtype=torch.int32)
    for s in range(n):
        table[s, :pages[s]] = torch.tensor(order[sum(pages[:s]):sum(pages[:s + 1])], dtype=torch.int32)
    ctx = SimpleNamespace(seq_start=list(range(n + 1)), n_seqs=n, max_kv_len=max(lengths), captured=False, row_seq=_i32(list(range(n))),
                          positions=_i32([x - 1 for x in lengths]), seq_start_dev=_i32(list(range(n + 1))), seq_ctx_dev=_i32([x - 1 for x in lengths]))
    scale = row ** -0.5
    got = ops.attention_latent(q.to(DEV), cache.to(DEV), sink.to(DEV), table.to(DEV), ctx, heads, rank, rot, PAGE, window, scale).cpu()
    for s, length in enumerate(lengths):
        first = max(0, length - window) if window else 0
        keys = torch.cat([cache[p] for p in table[s, :pages[s]].tolist()])[first:length].double()
        scores = (q[s].bfloat16().double() @ keys.T) * scale
        p = torch.softmax(torch.cat([scores, sink.double()[:, None]], 1), 1)[:, :-1]
        want = p @ keys[:, :rank]
        # weights rounded to bfloat16 (2^-9 of each), and scores in float: a sum of weights of at most one times the largest value
        assert (got[s].double() - want).abs().max() < 2.0 ** -8 * keys[:, :rank].abs().max()


@pytest.mark.parametrize("rank,rot,dims,heads", [(512, 64, 64, 16), (1000, 8, 4, 3), (1, 2, 2, 1), (130, 200, 130, 7), (24, 0, 0, 2)])
@pytest.mark.parametrize("halves", [False, True])
def test_cache_rows_of_any_size(ops, rank, rot, dims, heads, halves):
    gen = torch.Generator().manual_seed(rank)
    t, plain, eps = 5, 8, 1e-5
    q, dkv = torch.randn(t, heads * (plain + rot), generator=gen), torch.randn(t, rank + rot, generator=gen)
    g, angle = torch.randn(rank, generator=gen), torch.randn(t, max(dims // 2, 1), generator=gen)
    angles = torch.stack([angle.cos(), angle.sin()], -1).contiguous()
    cache, slots = torch.zeros(2, 4, rank + rot), [6, 0, 3, 5, 1]
    q_lat = torch.zeros(t, heads, rank + rot)
    on = [x.to(DEV) for x in (q, dkv, g, angles, cache, q_lat)]
    ops.latent_prepare(on[0], on[1], on[2], eps, on[3] if dims else None, _i32(slots), on[4], on[5], heads, plain, rot, rank, dims, halves=halves)

    def turned(u):                                   # [t, ..., rot]
        a = u.double().clone()
        i = torch.arange(dims // 2)
        x, y = (i, i + dims // 2) if halves else (2 * i, 2 * i + 1)
        shape = (t,) + (1,) * (u.dim() - 2) + (dims // 2,)
        c, s = (angles[:, :dims // 2, k].double().view(shape) for k in (0, 1))
        a[..., x], a[..., y] = u[..., x].double() * c - u[..., y].double() * s, u[..., y].double() * c + u[..., x].double() * s
        return a

    lat = dkv[:, :rank].double()
    rows = torch.cat([lat / torch.sqrt((lat * lat).mean(1, keepdim=True) + eps) * g.double(), turned(dkv[:, rank:])], 1)
    bound = 2.0 ** -20 * 8                           # a few float roundings of numbers up to 8
    assert (on[4].cpu().view(8, -1)[slots].double() - rows).abs().max() < bound
    if rot:
        want = turned(q.view(t, heads, plain + rot)[..., plain:])
        assert (on[5].cpu()[..., rank:].double() - want).abs().max() < bound


@pytest.mark.parametrize("t", [1, 8, 17, 32, 33])
@pytest.mark.parametrize("rank,rot,plain,heads", [(512, 64, 128, 16), (80, 24, 40, 3), (64, 0, 32, 2), (100, 8, 8, 1), (64, 6, 16, 2)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_absorbed_queries_beside_the_cache_rows(ops, t, rank, rot, plain, heads, dtype):
    """The two launches' bits, whether one takes their place or not (33 rows, float32, heads off 16 bytes: not), with queries and latent as
    parts of one product's rows."""
    gen = torch.Generator().manual_seed(t)
    n_q = heads * (plain + rot)
    qd = torch.randn(t, n_q + rank + rot, generator=gen).to(dtype).to(DEV)
    g, w = torch.randn(rank, generator=gen).to(DEV), torch.randn(heads, rank, plain, generator=gen).to(dtype).to(DEV)
    angles = torch.randn(t, max(rot // 2, 1), 2, generator=gen).to(DEV)
    slots = _i32(list(range(t))[::-1])
    q, dkv = qd[:, :n_q], qd[:, n_q:]
    out = []
    for together in (False, True):
        cache, q_lat = torch.zeros(1, t, rank + rot, dtype=dtype, device=DEV), torch.zeros(t, heads, rank + rot, device=DEV)
        ops.latent_prepare(q, dkv, g, 1e-5, angles if rot else None, slots, cache, q_lat, heads, plain, rot, rank, rot, absorb=w if together else None)
        if not together:
            ops.heads_gemm(q.unflatten(1, (heads, plain + rot)), w, q_lat, k=plain, n=rank)
        out.append((cache, q_lat))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


@pytest.mark.parametrize("m,n,k,heads", [(1000, 500, 136, 9), (8193, 64, 8, 8), (515, 512, 128, 16)])      # two blocks of rows a wave, the last in part
def test_products_per_head_of_many_rows_give_the_bits_of_few(ops, m, n, k, heads):
    assert -(-m // 16) * -(-n // 64) * heads >= 4096
    gen = torch.Generator().manual_seed(m)
    a = torch.randn(m, heads, k, generator=gen).bfloat16().to(DEV)
    w, gate = torch.randn(heads, n, k, generator=gen).bfloat16().to(DEV), torch.randn(m, heads, generator=gen).to(DEV)
    out, few = torch.empty(m, heads, n, device=DEV), torch.empty(100, heads, n, device=DEV)
    ops.heads_gemm(a, w, out, k=k, n=n, gate=gate)
    for first in (0, m // 2, m - 100):
        ops.heads_gemm(a[first:first + 100].contiguous(), w, few, k=k, n=n, gate=gate[first:first + 100].contiguous())
        assert torch.equal(out[first:first + 100], few)


@pytest.mark.parametrize("t", [1, 17, 32])
def test_absorbed_queries_with_nothing_else_to_write(ops, t):
    """rot 0 and neither cache nor queries' latent: the product alone, by the entry point itself."""
    from bare_cuda_4gib_amd.csrc import library
    gen = torch.Generator().manual_seed(t)
    heads, plain, rank = 3, 40, 80
    q, w = torch.randn(t, heads * plain, generator=gen).bfloat16().to(DEV), torch.randn(heads, rank, plain, generator=gen).bfloat16().to(DEV)
    got, want = torch.zeros(t, heads, rank, device=DEV), torch.zeros(t, heads, rank, device=DEV)
    ops.heads_gemm(q.unflatten(1, (heads, plain)), w, want, k=plain, n=rank)
    library.call("bc4g_latent_prepare", q.data_ptr(), None, 1, None, 1e-5, None, None, None, got.data_ptr(), t, heads, plain, 0, rank, 0, heads * plain, 0, 0,
                 None, None, None, 0, 0, w.data_ptr(), ops._stream())
    assert torch.equal(got, want)
