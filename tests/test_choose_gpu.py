"""A step's tokens chosen in one launch (ops.choose) against the host's law."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


class Fixed:
    def __init__(self, u):
        self.u = u

    def uniform(self):
        return self.u


@pytest.fixture(scope="module")
def ops():
    from bare_cuda_4gib_amd.csrc import ops as o
    return o


def check(ops, logits, temps, us, ks, ps):
    from bare_cuda_4gib_amd.sampling import SamplingParams, sample_token
    on_device = torch.from_numpy(logits).to(DEV)
    got = ops.choose(on_device, temps, us, ks, ps).cpu().tolist()
    want = [sample_token(row, SamplingParams(temperature=t, top_k=k, top_p=p), Fixed(u)) for row, t, u, k, p in zip(logits, temps, us, ks, ps)]
    # (a boundary may move by one token where u falls within a rounding of it: none of these draws does)
    assert got == want, [(i, g, w) for i, (g, w) in enumerate(zip(got, want)) if g != w]
    assert ops.choose(on_device, temps, us, ks, ps).cpu().tolist() == got


# vocabularies at the edges of what is held in LDS, none a multiple of four among them, smaller than a workgroup, and beyond one reading
@pytest.mark.parametrize("vocab", [1, 37, 1024, 32000, 32767, 32768, 32769, 50257, 128256])
# how far the logits spread: a few candidates, buckets of hundreds, of more than are put in order, and rows flatter than the buckets resolve
@pytest.mark.parametrize("spread", [8.0, 2.0, 0.4, 0.01])
def test_every_kind_of_row(ops, vocab, spread):
    rng = np.random.default_rng(vocab)
    options = [(0.0, 0, 1.0), (0.8, 0, 1.0), (0.7, 1, 1.0), (0.7, 40, 1.0), (1.0, 0, 0.9), (1.2, 100, 0.95), (1.0, 3000, 1.0), (1.5, 9000, 0.7),
               (1.0, 0, 0.01), (1.0, 0, 0.9999999), (0.3, vocab - 1, 0.5), (1.0, 10 * vocab, 0.999)]
    logits = (rng.standard_normal((len(options), vocab)) * spread).astype(np.float32)
    check(ops, logits, [o[0] for o in options], rng.random(len(options)).tolist(), [o[1] for o in options], [o[2] for o in options])


@pytest.mark.parametrize("vocab", [524288, 524289, 1100003])
@pytest.mark.parametrize("spread", [2.0, 0.4])
def test_vocabularies_whose_counts_have_words_of_their_own(ops, vocab, spread):
    rng = np.random.default_rng(vocab)
    options = [(0.0, 0, 1.0), (0.8, 0, 1.0), (0.7, 40, 1.0), (1.0, 0, 0.9), (1.2, 100, 0.95), (1.5, 9000, 0.7)]
    logits = (rng.standard_normal((len(options), vocab)) * spread).astype(np.float32)
    check(ops, logits, [o[0] for o in options], rng.random(len(options)).tolist(), [o[1] for o in options], [o[2] for o in options])


def test_ties_and_ends(ops):
    """Rows of few distinct weights (tokens told apart by id, buckets of more tokens than are put in order), u at its ends, weights that
    vanish, and more rows than go in one launch."""
    rng = np.random.default_rng(5)
    logits = np.repeat(rng.integers(0, 4, (140, 1)), 3000, axis=1).astype(np.float32)
    logits[:, ::7] += 1.0
    logits[:20, 1500:] = -np.inf
    logits[20:40, :] = rng.integers(0, 3, (20, 3000)).astype(np.float32) * 30.0
    ks = [(0, 5, 400, 2000)[i % 4] for i in range(140)]
    ps = [1.0 if i % 3 == 0 and ks[i] else (0.3, 0.999)[i % 2] for i in range(140)]
    us = [(0.0, 0.999999999, 0.5, float(rng.random()))[i // 4 % 4] for i in range(140)]
    check(ops, logits, [0.9] * 140, us, ks, ps)


@pytest.mark.parametrize("rows", [64, 65, 257])
@pytest.mark.parametrize("kind", ["greedy and plain", "plain", "limited"])
def test_any_number_of_rows_is_one_launch(ops, monkeypatch, rows, kind):
    """Options in the launch's arguments, and beyond them uploaded: every row what it is by itself, and one launch for all."""
    rng = np.random.default_rng(rows)
    logits = (rng.standard_normal((rows, 2001)) * 3).astype(np.float32)
    temps = [0.0 if kind == "greedy and plain" and i % 3 == 0 else 0.7 + 0.01 * (i % 40) for i in range(rows)]
    ks, ps = ([(0, 1, 40, 5000)[i % 4] for i in range(rows)], [(1.0, 0.9)[i // 4 % 2] for i in range(rows)]) if kind == "limited" else ([0] * rows, [1.0] * rows)
    us = rng.random(rows).tolist()
    launched = []
    call = ops.library.call
    monkeypatch.setattr(ops.library, "call", lambda name, *a, **k: (launched.append(name), call(name, *a, **k))[1])
    check(ops, logits, temps, us, ks, ps)
    assert launched == ["bc4g_choose" if rows <= 64 else "bc4g_choose_listed"] * 2         # (check asks twice)


def test_what_it_refuses(ops):
    logits = torch.zeros(2, 8, device=DEV)
    for bad in (dict(temperature=[1.0]), dict(top_k=[1, 2, 3])):
        with pytest.raises(Exception, match="choose"):
            ops.choose(logits, **dict(dict(temperature=[1.0, 1.0], u=[0.5, 0.5], top_k=[0, 0], top_p=[0.9, 0.9]), **bad))
    with pytest.raises(Exception, match="choose"):
        ops.choose(logits.bfloat16(), [1.0] * 2, [0.5] * 2, [0] * 2, [0.9] * 2)
