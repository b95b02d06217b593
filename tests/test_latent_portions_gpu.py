"""Latent attention of prompts in portions through the step function: expanded keys in steps run as they come and in recorded ones,
against the plain implementations, over pages whose unwritten and returned places are not numbers."""
import pytest
import torch

import qwen_engine_amd  # noqa: F401
from plain import safurax_plain as S, zarorax_plain as Z
import safurax_tiny
import zarorax_tiny

pytestmark = pytest.mark.gpu

# heads of 64 + 32 numbers (a size that the kernels of expanded keys take) on a latent of 128; the second layer's sizes others
ZX = {"architecture": "Zarorax", "vocab": 300, "width": 128, "postln_alpha": 2.0, "norm": {"eps": 1e-5}, "canon": {"taps": 3},
      "layers": [{"type": "latent_attention", "mlp": {"kind": "dense", "ff": 256},
                  "mixer": {"heads": 4, "dim": 64, "rot_dim": 32, "vdim": 64, "kv_rank": 128, "q_rank": 96, "scale": 0.1,
                            "rot": {"base": 10000.0, "dims": 32}}},
                 {"type": "latent_attention_2", "mlp": {"kind": "dense", "ff": 192},
                  "mixer": {"heads": 3, "dim": 64, "rot_dim": 64, "vdim": 128, "kv_rank": 200, "scale": 0.09,
                            "rot": {"base": 5000.0, "dims": 64}}}]}
# windows (one that ends inside a page, and a wider one on the same latent), sinks, gates a head; heads without a rotated part
SX = {"architecture": "Safurax", "vocab": 300, "width": 128, "embedding": {"scale": 1.0}, "norm": {"eps": 1e-5},
      "layers": [{"type": "latent_attention_2", "mlp": {"kind": "dense", "ff": 256},
                  "mixer": {"heads": 4, "dim": 64, "rot_dim": 32, "vdim": 64, "kv_rank": 128, "scale": 0.12,
                            "rot": {"base": 10000.0, "dims": 32}, "mask": {"size": 201}}},
                 {"type": "latent_attention", "mlp": {"kind": "dense", "ff": 192},
                  "mixer": {"heads": 4, "dim": 64, "vdim": 64, "kv_rank": 128, "q_rank": 64, "scale": 0.13}},
                 {"type": "latent_attention_2", "mlp": {"kind": "dense", "ff": 192},
                  "mixer": {"heads": 2, "dim": 64, "rot_dim": 32, "vdim": 64, "kv_rank": 128, "scale": 0.12, "kv_from": 0,
                            "rot": {"base": 10000.0, "dims": 32}, "mask": {"size": 330}}}]}
MODELS = {"zarorax": (ZX, Z, zarorax_tiny), "safurax": (SX, S, safurax_tiny)}
PAGE = 16


@pytest.fixture(scope="module", params=sorted(MODELS))
def model(request, tmp_path_factory):
    from qwen_engine_amd.engine import load_model
    cfg, plain, tiny = MODELS[request.param]
    folder = tiny.write_folder(str(tmp_path_factory.mktemp(request.param) / "model"), cfg, tiny.random_tensors(cfg, 31))
    g = torch.Generator().manual_seed(8)
    prompts = [torch.randint(0, cfg["vocab"], (n,), generator=g).tolist() for n in (1100, 1090, 700)]
    read, tensors = plain.read_folder(folder)
    return load_model(folder, dtype="bfloat16"), prompts, [plain.forward(read, tensors, p).float() for p in prompts]


def runner_of(model, **kw):
    from qwen_engine_amd.engine import ModelRunner
    return ModelRunner(model, page_size=PAGE, num_pages=240, max_requests=3, debug_poison=True, **kw)


def expanded(ctx):
    return [v for k, v in ctx.memo.items() if k[0] == "latent_attention.expansion" and v is not None]


def expanded_of(ctx):
    return [k for k, v in ctx.memo.items() if k[0] == "latent_attention.expansion" and v is not None]


def close(got, rows, want):
    """Logits [n, vocab] against the plain ones of those rows, relative to the request's largest: a few roundings to bfloat16 a layer."""
    err = (got.float().cpu() - want[rows]).abs().amax(dim=1) / want.abs().max()
    assert not torch.isnan(err).any() and float(err.max()) < 3e-2, err


def test_recorded_portions_see_expanded_keys_wherever_they_stand(model):
    """Portions of 256 rows: one recorded step for the places of 257 to 512 keys and one for 513 to 1024, replayed at several
    places of each and for other requests; the steps run as they come beside them; a last portion of other length."""
    from qwen_engine_amd.engine import StepEntry
    weights, prompts, want = model
    logits = {}
    for use_graphs in (False, True):
        runner = runner_of(weights, use_graphs=use_graphs)
        for i, (p, skip) in enumerate(zip(prompts[:2], (0, 40))):           # (the second request's portions begin 40 tokens later)
            runner.add_request(i)
            at = 0
            for n in ([skip] if skip else []) + [256] * 4 + [len(p) - skip - 1024]:
                rows = runner.step([StepEntry(i, p[at:at + n], [n - 1])])
                at += n
                close(rows, [at - 1], want[i])
                logits[use_graphs, i, at] = rows
            runner.free_request(i)
        if use_graphs:
            recorded = {max(k for k in key[3] if k): r for key, r in runner._graphs.items() if key[0] == "portion" and key[1] == 256}
            assert runner.graph_steps_of["portion"] == 8 and sorted(recorded) == [256, 512, 1024, 2048]
            for keys, r in recorded.items():
                plans = expanded(r["ctx"])
                assert plans
                for (_, latent, dim, rot, v_dim, heads, window), e in zip(expanded_of(r["ctx"]), plans):
                    taken = 64 * e["owner"].shape[0]
                    assert taken == -(-(min(keys, window + 255) if window else keys) // 64) * 64
                    # (what the recording keeps counts: the expanded keys and values of a layer at the least)
                    assert r["bytes"] >= 2 * taken * heads * (dim + v_dim)
    for (graphs, i, at), rows in logits.items():
        if graphs:
            close(rows, [0], logits[False, i, at].float().cpu())


def test_long_portions_and_single_tokens_in_one_step(model):
    """Two portions whose keys are expanded, single tokens between and behind them whose maps stay folded, in one step and the next."""
    from qwen_engine_amd.engine import StepEntry
    weights, prompts, want = model
    a, b, c = prompts
    runner = runner_of(weights, use_graphs=False)
    for i in range(3):
        runner.add_request(i)
    runner.step([StepEntry(0, a[:300], []), StepEntry(1, b[:17], []), StepEntry(2, c[:5], [])])
    for step in ([(2, 5, 305), (1, 17, 18), (0, 300, 700)], [(0, 700, 701), (1, 18, 500), (2, 305, 306)],
                 [(1, 500, 501), (2, 306, 700), (0, 701, 1100)]):
        entries = [StepEntry(i, prompts[i][x:y], [0, y - x - 1] if y - x > 1 else [0]) for i, x, y in step]
        ctx = runner.build_context(entries)
        runner._begin_new_requests(ctx.seqs)
        rows = weights.forward(ctx, runner.bindings)
        for e in entries:
            runner.cache.commit(e.req_id, e.tokens)
        runner._poison_pages()
        long = [(s.q_start, s.q_start + s.q_len) for s in ctx.seqs if s.q_len > 1]
        assert expanded(ctx) and all(e["ranges"] == long for e in expanded(ctx))
        at = 0
        for (i, x, y), e in zip(step, entries):
            close(rows[at:at + len(e.want)], [x + w for w in e.want], want[i])
            at += len(e.want)


def test_recorded_steps_of_a_portion_beside_single_tokens(model):
    """A prompt in portions beside a request that decodes: recorded (where the model's steps of that kind are) and as they come."""
    from qwen_engine_amd.engine import StepEntry
    weights, prompts, want = model
    for use_graphs in (False, True):
        runner = runner_of(weights, use_graphs=use_graphs)
        for i in range(2):
            runner.add_request(i)
        runner.step([StepEntry(0, prompts[0][:50], [])])
        for k in range(4):
            rows = runner.step([StepEntry(0, prompts[0][50 + k:51 + k], [0]), StepEntry(1, prompts[1][250 * k:250 * (k + 1)], [249])])
            close(rows[:1], [50 + k], want[0])
            close(rows[1:], [250 * (k + 1) - 1], want[1])
