"""Large weights are loaded past the caches by models whose weights do not stay there: which models those are, for which launches, and the same bits."""
import threading

import pytest
import torch

from bare_cuda_4gib_amd.config import architecture_for
from bare_cuda_4gib_amd.csrc import ops
from bare_cuda_4gib_amd.engine import Model, Runtime
from bare_cuda_4gib_amd.engine import model as model_file

RAW = dict(architectures=["LlamaForCausalLM"], model_type="llama", vocab_size=256, hidden_size=64, num_attention_heads=4, num_key_value_heads=2,
           head_dim=16, intermediate_size=176, rope_theta=10000.0, rms_norm_eps=1e-5, max_position_embeddings=128, num_hidden_layers=2)
BODY = 2 * (64 * 128 + 64 * 64 + 3 * 64 * 176 + 2 * 64) + 64          # numbers of two layers and the last norm


def bound(tied):
    arch = architecture_for(RAW)
    model = Model(arch.describe(arch.config_class.from_dict(dict(RAW, tie_word_embeddings=tied))))
    tensors = {name: torch.zeros(spec.shape) for name, spec in model.expected_weights().items() if not spec.optional}
    model.bind(tensors, Runtime(torch.device("cpu"), torch.float32))
    return model


@pytest.mark.parametrize("tied", [False, True])
def test_the_weights_a_step_reads_decide(monkeypatch, tied):
    """The output head counts, also where it is the embedding table; a table of its own, from which a step reads single rows, does not."""
    total = 4 * (BODY + 256 * 64)
    for most, stays in ((total, True), (total - 1, False)):
        monkeypatch.setattr(model_file, "WEIGHTS_STAY_BYTES", most)
        assert bound(tied).weights_stay is stays


def test_a_thread_s_launches_inside_the_block():
    """However large a weight is, by itself it is loaded through the caches: a narrow model's wide head, a 32-bit matrix."""
    assert not ops.weight_passes(32000, 768) and not ops.weight_passes(1536, 1024, 4)
    seen = []
    with ops.weights_pass():
        assert ops.weight_passes(32000, 768) and ops.weight_passes(1536, 1024, 4) and not ops.weight_passes(1536, 2044)
        other = threading.Thread(target=lambda: seen.append(ops.weight_passes(32000, 768)))
        other.start(), other.join()
    assert seen == [False] and not ops.weight_passes(32000, 768)
    with pytest.raises(ZeroDivisionError):
        with ops.weights_pass():
            1 / 0
    assert not ops.weight_passes(32000, 768)


@pytest.mark.parametrize("stays", [False, True])
def test_a_step_says_so_for_its_own_launches(monkeypatch, stays):
    model = bound(False)
    model.weights_stay, model.rt = stays, Runtime(torch.device("cuda:0"), torch.float32)
    monkeypatch.setattr(model, "_forward", lambda ctx: ops.weight_passes(32000, 768))
    assert model.forward(None) is not stays and not ops.weight_passes(32000, 768)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 8, 16, 24, 32, 40])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_the_same_bits_either_way(m, dtype):
    gen = torch.Generator(device="cuda:0").manual_seed(m)
    x, w = (torch.randn(n, 1088, generator=gen, device="cuda:0").to(dtype) for n in (m, 8208))
    product = (lambda: ops.gemm_f32(x, w)) if dtype == torch.float32 else (lambda: ops.gemm_fast(x, w, torch.float32))
    through = product()
    with ops.weights_pass():
        past = product()
    assert torch.equal(past, through)
