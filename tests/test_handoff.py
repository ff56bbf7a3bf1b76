"""What a block leaves to the next one: a sublayer's output is added exactly once whoever comes next, and is never dropped in silence.
The parts are plain stand-ins, on the CPU."""
from types import SimpleNamespace

import pytest
import torch

from bare_cuda_4gib_amd.errors import EngineError
from bare_cuda_4gib_amd.parts.block import AddingReader, SandwichBlock
from bare_cuda_4gib_amd.parts.lazy import NormHandoff


class Norm:
    def forward(self, x, ctx=None):
        return x * 0.5

    def add_to(self, x, y):
        x += 0.25 * y

    def added_by_the_reader(self, y):
        return y, self, 0.0


class Conv:
    def cache_spec(self):
        return None

    def forward(self, h, ctx, view, add_input=False):
        return h + 1.0

    def behind(self, norm, x, ctx, view, adds=None):
        if adds is not None:
            adds[1].add_to(x, adds[0])
        return self.forward(norm.forward(x), ctx, view)


class ConvOfItsOwn(Conv):
    def behind(self, norm, x, ctx, view):
        return self.forward(norm.forward(x), ctx, view)


class Mixer:
    adds_one_product = True

    def __init__(self, by):
        self.by = by

    def forward(self, h, ctx, cache, y, writes):
        y.tensor = h * self.by


class ForwardOfItsOwn(SandwichBlock):
    def forward(self, x, ctx, cache, writes=True):
        x += self.mixer_norm.forward(x)


class NoInit(SandwichBlock):
    def __init__(self):
        self.mixer, self.mixer_norm, self.mixer_post_norm, self.mixer_conv, self.ffn = Mixer(0.3), Norm(), Norm(), Conv(), None


def block(cls=SandwichBlock, conv=Conv, by=2.0):
    return cls(Mixer(by), Norm(), Norm(), mixer_conv=conv())


def run(blocks, handed):
    handoff = NormHandoff()
    ctx = SimpleNamespace(n_tokens=3, n_seqs=3, handoff=handoff)
    x = torch.arange(12.0).view(3, 4)
    handoff.begin_step()
    for i, b in enumerate(blocks):
        handoff.begin_entry(b, blocks[i + 1] if handed and i + 1 < len(blocks) else None, 3)
        b.forward(x, ctx, SimpleNamespace(mixer=None, conv=None))
    handoff.end_step()
    return x


def test_every_output_is_added_once_whoever_reads_next():
    plain = [block(by=b) for b in (2.0, 3.0, 5.0)]
    assert all(b.first_reader(3) is not None for b in plain)
    same = plain[1]
    for chain in (plain, [plain[0], block(ForwardOfItsOwn), plain[2]], [plain[0], block(conv=ConvOfItsOwn), plain[2]], [plain[0], NoInit(), plain[2]],
                  [same, same, same]):
        assert torch.equal(run(chain, True), run(chain, False))


def test_an_output_that_nobody_added_ends_the_step():
    takes, other = block(), block()
    reader = takes.first_reader(3)[0]
    assert isinstance(reader, AddingReader)

    def owing():
        handoff = NormHandoff()
        handoff.begin_step()
        handoff.begin_entry(other, takes, 3)
        handoff.owe(reader, "y")
        return handoff

    handoff = owing()
    handoff.begin_entry(takes, None, 3)
    assert handoff.take(reader) == "y" and handoff.take(reader) is None
    handoff.end_step()
    for wrong in (lambda h: h.end_step(), lambda h: h.begin_entry(other, None, 3), lambda h: h.owe(reader, "z"),
                  lambda h: (h.begin_entry(takes, takes, 3), h.begin_entry(takes, None, 3)), lambda h: (h.begin_entry(takes, None, 3), h.end_step())):
        handoff = owing()
        with pytest.raises(EngineError, match="did not add it"):
            wrong(handoff)
        handoff.end_step()                        # (nothing is left of it)
