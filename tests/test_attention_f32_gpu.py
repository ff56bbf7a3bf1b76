"""The float32 matrix-core attention (attention_f32.hip) against float64 and against the plain kernel.

Tolerance: that of the plain float kernel's own test at these sizes, rtol 1e-4 and atol 1e-5."""
import math
import types

import pytest
import torch

from test_kernels_gpu import DEV, close, paged_case, plain_result

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from bare_cuda_4gib_amd.csrc import ops as o
    return o


def context(case):
    starts, ctx = case["seq_start"], case["seq_ctx"]
    dev = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)      # noqa: E731
    return types.SimpleNamespace(n_seqs=len(ctx), n_tokens=starts[-1], seq_start=starts, seq_ctx=ctx, seq_start_dev=dev(starts), seq_ctx_dev=dev(ctx),
                                 max_q_len=max(b - a for a, b in zip(starts, starts[1:])), max_kv_len=max(c + b - a for c, a, b in zip(ctx, starts, starts[1:])),
                                 row_seq=case["row_seq"], positions=case["positions"])


def run(ops, case, window):
    nh, nkv, d = case["nh"], case["nkv"], case["d"]
    assert ops.attention_f32_takes(case["qkv"], case["kc"], case["vc"], d)
    return ops.attention(case["qkv"], case["kc"], case["vc"], case["table"], context(case), None, nh, nkv, d, window, 1.0 / math.sqrt(d))


SHAPES = [  # query heads, key/value heads, head size, page: every register form, pages smaller and larger than a tile, no power of two
    (4, 2, 16, 16), (3, 3, 32, 4), (6, 2, 48, 32), (32, 4, 64, 64), (8, 1, 128, 12), (32, 1, 16, 16), (2, 2, 112, 128)]
# (cached, new): a row alone, prompts with rows at the edges of a wave's 16 and a group's 64, portions, long contexts of one token
SEQS = [[(0, 33), (40, 1), (17, 2), (0, 1), (64, 70), (129, 1)], [(0, 1)], [(700, 1), (127, 1), (0, 16), (15, 17)], [(250, 65), (0, 128)]]


@pytest.mark.parametrize("nh,nkv,d,page", SHAPES)
@pytest.mark.parametrize("window", [0, 20, 130])
@pytest.mark.parametrize("seqs", SEQS)
def test_against_float64(ops, nh, nkv, d, page, window, seqs):
    case = paged_case(seqs, nh, nkv, d, page, torch.float32, seed=3)          # (pages that nobody owns hold NaN)
    got = run(ops, case, window)
    close(got, plain_result(case, window), rtol=1e-4, atol=1e-5, what="float32 on the matrix cores")
    if len(seqs) > 1:                      # a request alone: the same bits
        alone = paged_case(seqs, nh, nkv, d, page, torch.float32, seed=3)
        s = len(seqs) - 1
        a, b = alone["seq_start"][s], alone["seq_start"][s + 1]
        alone.update(qkv=alone["qkv"][a:b].contiguous(), table=alone["table"][s:].contiguous(), row_seq=alone["row_seq"][a:b] * 0,
                     positions=alone["positions"][a:b], seq_start=[0, b - a], seq_ctx=alone["seq_ctx"][s:])
        assert torch.equal(run(ops, alone, window), got[a:b])


@pytest.mark.parametrize("new", [1, 2, 40])
def test_values_that_are_not_finite_stay_with_the_rows_that_see_them(ops, new):
    """An infinite value at the last position: rows before it, which share a tile with it, come out as if it were not there."""
    case = paged_case([(20, new)], 8, 2, 64, 64, torch.float32, seed=5)
    clean = run(ops, case, 0)
    page = int(case["table"][0, 0])
    case["vc"][page, :, :, (20 + new - 1) % 64] = float("inf")
    got = run(ops, case, 0)
    assert not torch.isfinite(got[-1]).any()
    torch.testing.assert_close(got[:-1], clean[:-1], rtol=1e-5, atol=1e-6)
    case["vc"][page, :, :, 3] = float("nan")                                  # seen by every row
    assert torch.isnan(run(ops, case, 0)).all()
