"""Steps of single new tokens whose layers are one launch (``parts.chain``), through the engine."""
import functools
import random

import pytest
import torch

from plain import qwen3_plain as P
from tiny import TINY, make_folder
import traces

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


TOL = 2e-2       # of the largest logit, as for the other bfloat16 models of this size (test_replay_gpu.py)


@pytest.fixture(scope="module")
def folder(tmp_path_factory):
    return make_folder(tmp_path_factory.mktemp("chain"), "F", std=0.05)


@pytest.fixture(scope="module")
def plain(folder):
    """Logits of the plain implementation."""
    cfg, w = P.read_folder(folder)
    return lambda tokens: P.forward_logits(cfg, w, tokens, act_dtype=torch.bfloat16)


@pytest.fixture(scope="module")
def model(folder):
    from qwen_engine_amd.engine import load_model
    return load_model(folder, dtype="bfloat16", device=DEV)


@pytest.fixture
def launches(monkeypatch):
    """The rows of every launch of whole steps (those that are recorded count when they are recorded)."""
    from qwen_engine_amd.kernels import ops
    real, rows = ops.decode_chain, []
    monkeypatch.setattr(ops, "decode_chain", lambda h, *a, **kw: (rows.append(h.shape[0]), real(h, *a, **kw))[1])
    return rows


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


@pytest.mark.parametrize("graphs", [True, False])
def test_steps_of_one_to_nine_requests(model, plain, launches, graphs):
    """Up to eight single tokens go in one launch, nine one by one; a row's bits do not follow how many stand beside it, up to eight."""
    from qwen_engine_amd.engine import StepEntry
    lengths = [130, 7, 300, 16, 257, 64, 500, 1, 90]
    prompts = [prompt_of(n + 2, seed=n) for n in lengths]
    want = [plain(p) for p in prompts]
    runner, first = runner_of(model, use_graphs=graphs), {}
    for rows in (1, 2, 3, 5, 8, 9):
        for i in range(rows):
            runner.add_request(i)
            runner.step([StepEntry(i, prompts[i][:lengths[i]], [])])
        before = len(launches)
        for at in range(2):
            logits = runner.step([StepEntry(i, prompts[i][lengths[i] + at:][:1], [0]) for i in range(rows)])
            for i in range(rows):
                ref = want[i][lengths[i] + at]
                assert float((logits[i].cpu() - ref).abs().max()) <= TOL * float(want[i].abs().max()), (rows, i, at)
                if rows <= 8:
                    assert torch.equal(first.setdefault((i, at), logits[i]), logits[i]), (rows, i, at)
        assert set(launches[before:]) == ({rows} if rows <= 8 else set())
        for i in range(rows):
            runner.free_request(i)
    runner.check()


def test_traces(folder, plain, launches, tmp_path):
    """Tokens one by one, portions beside them, pages used again, random cuttings, through the replay program's own function."""
    cfg = TINY["F"][0]
    requests = {f"r{i}": prompt_of(n, seed=n) for i, n in enumerate((350, 66, 257, 129, 480, 90))}
    ref = {rid: plain(tokens) for rid, tokens in requests.items()}
    cuttings = [(traces.tail_decoded(requests), 16), (traces.portions(requests), 16), (traces.mixed(requests, seed=7), 16)]
    for seed in range(6):
        rng = random.Random(seed)
        cuttings.append((traces.mixed(requests, seed=seed, max_live=rng.randint(1, 4), tail=rng.choice([1, 5, 12, 40])), rng.choice([16, 32, 64])))
    for k, (trace, page) in enumerate(cuttings):
        out = str(tmp_path / str(k))
        traces.run_in_process(trace, folder, "bfloat16", out, page)
        bad, _ = traces.first_mismatch(traces.collect(trace, out, cfg["vocab_size"]), ref, TOL)
        assert bad is None, f"cutting {k}, pages of {page}: first wrong logits at (request, position, relative error) {bad}"
    assert {1, 2, 3, 4} <= set(launches) and max(launches) <= 8


@pytest.mark.parametrize("start", [1010, 2038, 2550])
def test_across_the_positions_where_the_recorded_step_and_the_segments_change(model, plain, launches, start):
    """Recorded steps are kept for positions up to multiples of 1024, and a token's keys are cut otherwise from 2560 on."""
    from qwen_engine_amd.engine import StepEntry
    tokens = prompt_of(start + 24, seed=start)
    want = plain(tokens)[start:]
    runner = runner_of(model, use_graphs=True)
    runner.add_request("r")
    runner.step([StepEntry("r", tokens[:start], [])])
    got = torch.cat([runner.step([StepEntry("r", tokens[i:i + 1], [0])]) for i in range(start, len(tokens))]).cpu()
    assert float((got - want).abs().max()) <= TOL * float(want.abs().max())
    assert len(launches) >= (2 if start == 2550 else 4) and set(launches) == {1}          # one or two recorded steps, each run once before


def test_requests_that_share_pages(model, launches):
    """Keys that other requests read too are asked for in another way: the bits are the same."""
    from qwen_engine_amd.engine import StepEntry
    prefix, results = prompt_of(400, seed=1), []
    tails = [prompt_of(n, seed=n) for n in (5, 40, 17, 90)]
    for sharing in (True, False):
        runner, rows = runner_of(model, prefix_sharing=sharing), []
        for i, tail in enumerate(tails):
            runner.add_request(i)
            at = runner.cache.match_prefix(i, prefix + tail) if sharing else 0
            assert at == (400 if sharing and i else 0)
            rest = (prefix + tail)[at:]
            if at == 0:
                runner.step([StepEntry(i, rest[:400], [])])     # (the same steps on both sides)
                rest = rest[400:]
            runner.step([StepEntry(i, rest, [])])
        for token in range(20):
            rows.append(runner.step([StepEntry(i, [token], [0]) for i in range(4)]))
        results.append(torch.cat(rows))
    assert set(launches) == {4} and torch.equal(*results)
