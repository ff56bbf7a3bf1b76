"""Which decode steps read their keys and values past the caches: those whose requests may reach far enough, whatever room their block tables have."""
import pytest
import torch

from bare_cuda_4gib_amd.cache import CacheManager, FixedState, PagedKV
from bare_cuda_4gib_amd.config import architecture_for
from bare_cuda_4gib_amd.csrc import ops
from bare_cuda_4gib_amd.engine import Executor, Model, Runtime, StepEntry
from bare_cuda_4gib_amd.engine import executor as executor_file

RAW = dict(architectures=["LlamaForCausalLM"], model_type="llama", vocab_size=256, hidden_size=64, num_attention_heads=4, num_key_value_heads=2,
           head_dim=16, intermediate_size=176, rope_theta=10000.0, rms_norm_eps=1e-5, max_position_embeddings=4096, tie_word_embeddings=False,
           num_hidden_layers=2)


def executor(device, dtype, **sizes):
    arch = architecture_for(RAW)
    model = Model(arch.describe(arch.config_class.from_dict(RAW)))
    tensors = {name: torch.zeros(spec.shape, dtype=dtype) for name, spec in model.expected_weights().items() if not spec.optional}
    model.bind(tensors, Runtime(torch.device(device), dtype))
    return Executor(model, page_tokens=64, **sizes)


def test_bytes_a_request_s_next_token_reads():
    streams = {"all": PagedKV(2, 16), "last": PagedKV(4, 8, window=100), "state": FixedState((7,))}
    cache = CacheManager(streams, page_tokens=16, num_pages=4, max_requests=2, max_tokens=4096, dtype=torch.bfloat16, device="cpu")
    token = 2 * 2 * 16 * 2, 2 * 4 * 8 * 2
    for length, kept in ((0, 0), (1, 1), (99, 99), (100, 99), (4000, 99)):
        assert cache.bytes_read(length) == length * token[0] + kept * token[1]


def test_the_reach_of_the_requests_decides_and_not_the_room(monkeypatch):
    """Two layers of 128 numbers a token in 32 bits: a request reads 512 bytes a token."""
    runs = {most: executor("cpu", torch.float32, num_pages=200, max_requests=3, max_tokens=most) for most in (128, 4096)}
    for run in runs.values():
        weights = run.model.cached_weight_bytes
        assert weights > 0 and run.model.weights_stay
        for r in range(3):
            run.admit(r)
        run.cache.reserve([(r, 100) for r in range(3)])
        for r in range(3):
            run.cache.advance(r, 99)
        step = [StepEntry(r, [1], [0]) for r in range(3)]
        for limit, passes in ((weights + 3 * 100 * 512, True), (weights + 3 * 100 * 512 + 1, False)):
            monkeypatch.setattr(executor_file, "CACHE_HOLDS_BYTES", limit)
            assert run.build_context(step).cache_passes is passes
            assert not run.build_context([StepEntry(0, [1, 2], [1])]).cache_passes


@pytest.mark.gpu
def test_a_captured_step_plans_for_its_bucket(monkeypatch):
    asked = []
    call = ops.library.call

    def watched(name, *args, **more):
        if name == "bc4g_attention_mfma_counted":
            asked.append(args[-2])
        return call(name, *args, **more)
    monkeypatch.setattr(ops.library, "call", watched)
    # (the middle of a bucket: 128 tokens of the first, of up to 256, and 384 of the one after it)
    for most, tokens, reach, past in ((300, 20, 128, 0), (4096, 20, 128, 0), (300, 20, 127, 1), (4096, 20, 127, 1), (600, 300, 384, 0), (4096, 300, 383, 1)):
        run = executor("cuda:0", torch.bfloat16, num_pages=80, max_requests=2, max_tokens=most)
        monkeypatch.setattr(executor_file, "CACHE_HOLDS_BYTES", run.model.cached_weight_bytes + 2 * reach * 256 + 1)
        for r in range(2):
            run.admit(r)
            run.step([StepEntry(r, [3] * (tokens + r), [])])
        asked.clear()
        run.step([StepEntry(r, [1], [0]) for r in range(2)])
        assert run.captures == 1 and asked == [past] * 4            # (once outside the capture and once inside, two layers)
