"""Steps of single new tokens whose layers are one launch (``parts.chain``), through the engine."""
import functools

import pytest
import torch

from tiny import make_folder

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    from qwen_engine_amd.engine import load_model
    return load_model(make_folder(tmp_path_factory.mktemp("chain"), "F", std=0.05), dtype="bfloat16", device=DEV)


def runner_of(model, **kw):
    from qwen_engine_amd.engine import ModelRunner
    kw = dict(dict(page_size=16, num_pages=600, max_requests=16, debug_poison=True), **kw)
    return ModelRunner(model, **kw)


def prompt_of(n, seed=0):
    return torch.randint(0, 400, (n,), generator=torch.Generator().manual_seed(seed)).tolist()


@pytest.mark.parametrize("graphs", [True, False])
def test_a_step_that_fails_on_the_device_is_told_and_leaves_nothing_to_share(model, monkeypatch, graphs):
    from qwen_engine_amd.engine import StepEntry
    from qwen_engine_amd.kernels import ops
    runner = runner_of(model, use_graphs=graphs, prefix_sharing=True, keep_freed_prefixes=True)
    tokens = prompt_of(47)
    runner.add_request("a")
    runner.step([StepEntry("a", tokens, [])])
    runner.add_request("b")
    assert runner.cache.match_prefix("b", tokens) == 32
    runner.step([StepEntry("b", tokens[32:], [])])
    assert runner.cache.num_kept == 0 and len(runner.cache._shared) == 2
    real = ops.decode_chain
    monkeypatch.setattr(ops, "decode_chain", functools.partial(real, absent=2, limit_us=3000))
    with pytest.raises(ops.KernelError, match="waited"):       # the step waits for its tokens: it fails itself
        runner.step([StepEntry("a", [5], [0])], greedy=True)
    assert runner.cache.get("a").num_tokens == 47 and not runner.cache._shared
    runner.free_request("a")
    logits = runner.step([StepEntry("b", [7], [0])])           # its logits are asked for later
    torch.cuda.synchronize()
    assert bool(torch.isnan(logits).all())
    with pytest.raises(ops.KernelError, match="waited"):
        runner.check()
    runner.check()
    runner.free_request("b")
    runner.cache.check_invariants()
    assert runner.cache.num_kept == 0
    # a request that ends before anybody has looked
    runner.add_request("c")
    runner.step([StepEntry("c", tokens, [])])
    runner.step([StepEntry("c", [5], [0])])
    torch.cuda.synchronize()
    runner.free_request("c")
    assert runner.cache.num_kept == 0
    with pytest.raises(ops.KernelError, match="waited"):
        runner.step([StepEntry("d", [5], [0])])
    # and all is well again
    monkeypatch.setattr(ops, "decode_chain", real)
    runner._graphs.clear()
    runner.add_request("e")
    assert runner.cache.match_prefix("e", tokens) == 0
    runner.step([StepEntry("e", tokens, [])])
    assert bool(torch.isfinite(runner.step([StepEntry("e", [5], [0])])).all())
    runner.check()


def test_the_engine_says_that_a_step_failed(model, monkeypatch):
    from qwen_engine_amd import EngineConfig
    from qwen_engine_amd.engine import LLMEngine
    from qwen_engine_amd.kernels import ops
    monkeypatch.setattr(ops, "decode_chain", functools.partial(ops.decode_chain, absent=1, limit_us=3000))
    for temperature in (0.0, 0.7):
        engine = LLMEngine(model, None, EngineConfig(dtype="bfloat16", block_size=16, max_model_len=256))
        engine.submit([prompt_of(20)], max_new_tokens=4, temperature=temperature, ignore_eos=True)
        with pytest.raises(ops.KernelError, match="waited"):
            engine.run()
