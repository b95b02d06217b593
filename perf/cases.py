"""The work whose speed counts: a serving step in the forms in which programs ask the engine for it.

A case is a set of requests that pass through ``ModelRunner``: requests are admitted, what the cache keeps of their
history is taken over, their prompts run in one step (or one after another in portions, beside the tokens of the
requests that came before), and every request then decodes a number of new tokens.  The tokens that are fed are given
with the inputs, so that the logits of a pass do not hang on near ties; the logits of every step are its outputs.

    design, sizes, layers, dtype    the model: layer sizes of the Qwen3 family or of another design, as ``bench.py`` has them
    requests, prompt, new           how many, the mean prompt length, the tokens each decodes after it
    history                         tokens of every request that the cache keeps from an earlier turn
    ragged                          lengths from half to one and a half times the mean instead of equal ones
    portion                         0: all prompts in one step; else arrivals, in portions of so many tokens
"""
import math
import zlib

import torch

import qwen_engine_amd  # noqa: F401
from qwen_engine_amd.config import config_from_dict
from qwen_engine_amd.engine import ModelRunner, StepEntry
from qwen_engine_amd.parts import DecoderModel, Runtime, expected_tensors

PAGE = 16
DESIGN_VOCAB = 32768
CLUSTERS = 64            # kinds of tokens that a mixture's router tells apart


def _case(name, design="qwen3", sizes="0.6b", layers=28, dtype="bfloat16", requests=1, history=0, prompt=16, new=0,
          ragged=False, portion=0):
    return {"name": name, "design": design, "sizes": sizes, "layers": layers, "dtype": dtype, "requests": requests,
            "history": history, "prompt": prompt, "new": new, "ragged": ragged, "portion": portion}


def listed():
    return [
        # one conversation with the small model: every kernel is at its floor and launches count
        _case("decode_1", history=2032, prompt=9, new=32),
        # the benchmark's decode point: eight conversations of some 4096 tokens
        _case("decode_8", requests=8, history=4032, prompt=16, new=32),
        # a full batch of a large model, contexts of all lengths
        _case("decode_64_large", sizes="8b", layers=8, requests=64, history=1024, prompt=7, new=16, ragged=True),
        # requests that arrive while others decode: single tokens beside a prompt's portion
        _case("arrivals", requests=16, prompt=320, new=24, ragged=True, portion=512),
        # the benchmark's prompt
        _case("prompt_2048", prompt=2048),
        # a further portion of a long document
        _case("portion_deep", history=7680, prompt=512),
        # several prompts of odd lengths in one step of a large model, and one very long prompt
        _case("prompts_large", sizes="32b", layers=3, requests=3, prompt=601, ragged=True),
        _case("prompt_8192_large", sizes="8b", layers=8, prompt=8192),
        # the 32-bit mode, as it is used to check a model
        _case("float32", layers=4, dtype="float32", requests=2, prompt=333, new=8, ragged=True),
        # latent attention and routed experts: a prompt with some tokens after it
        _case("latent_experts", design="zarorax", sizes="medium", layers=6, prompt=2048, new=4),
        # recurrences beside attention whose heads talk: eight prompts, tokens after them
        _case("recurrences", design="potatar", sizes="medium", layers=4, requests=8, prompt=235, new=12, ragged=True),
        # state spaces and matrix memories beside attention: one prompt, an answer after it
        _case("state_spaces", design="vuzinex", sizes="medium", layers=4, prompt=1000, new=24),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["prompt", "prompt", "decode", "decode", "arrivals", "float32", "design", "design"])
    sizes, layers = rng.choice([("0.6b", 28), ("0.6b", 28), ("8b", rng.randint(2, 8)), ("32b", rng.randint(2, 3))])
    if kind == "prompt":
        n = rng.randint(1, 4)
        c = _case("", sizes=sizes, layers=layers, requests=n, prompt=max(1, _log_uniform(rng, 24, 4096) // n),
                  history=rng.choice([0, PAGE * _log_uniform(rng, 4, 384 // n)]), ragged=n > 1)
    elif kind == "decode":
        n = _log_uniform(rng, 1, 64)
        c = _case("", sizes=sizes, layers=layers, requests=n, history=PAGE * _log_uniform(rng, 4, min(512, 8192 // n)),
                  prompt=rng.randint(1, 16), new=rng.randint(12, 32), ragged=n > 1 and rng.random() < 0.5)
    elif kind == "arrivals":
        c = _case("", sizes=sizes, layers=layers, requests=rng.randint(3, 16), prompt=_log_uniform(rng, 60, 480),
                  new=rng.randint(12, 32), ragged=True, portion=512)
    elif kind == "float32":
        c = _case("", layers=rng.randint(2, 4), dtype="float32", requests=rng.randint(1, 4),
                  prompt=_log_uniform(rng, 8, 400), new=rng.randint(2, 8), ragged=True)
    else:
        n = rng.choice([1, 1, rng.randint(2, 8)])
        c = _case("", design=rng.choice(["zarorax", "potatar", "vuzinex"]), sizes=rng.choice(["small", "medium"]),
                  layers=rng.randint(4, 6), requests=n, prompt=max(1, _log_uniform(rng, 24, 3000) // n),
                  new=rng.randint(0, 16), ragged=n > 1)
    del c["name"]
    return c


# ---- the model and the requests of a case ------------------------------------------------------------------------
QWEN3 = {
    "0.6b": dict(hidden_size=1024, intermediate_size=3072, num_attention_heads=16, tie_word_embeddings=True),
    "8b": dict(hidden_size=4096, intermediate_size=12288, num_attention_heads=32, tie_word_embeddings=False),
    "32b": dict(hidden_size=5120, intermediate_size=25600, num_attention_heads=64, tie_word_embeddings=False),
}
# (width, size of a head: 16 heads in every mixer, 4 of keys and values; rotated numbers of a latent query, ranks of the
# latents of keys and queries, width of an expert)
SIZES = {"small": (1024, 64, 32, 256, 384, 768), "medium": (2048, 128, 64, 512, 768, 1024)}


def _qwen3(case):
    return dict(architectures=["Qwen3ForCausalLM"], vocab_size=151936, num_hidden_layers=case["layers"], num_key_value_heads=8,
                head_dim=128, max_position_embeddings=40960, rms_norm_eps=1e-6, rope_theta=1e6, **QWEN3[case["sizes"]])


def _zarorax(case):
    """A dense layer, then mixtures; queries through a latent of their own and direct ones in turn."""
    width, dim, rot, rank, q_rank, ff = SIZES[case["sizes"]]
    layers = []
    for i in range(case["layers"]):
        mixer = {"heads": 16, "dim": dim, "rot_dim": rot, "vdim": dim, "kv_rank": rank, "scale": (dim + rot) ** -0.5,
                 "rot": {"base": 10000.0, "dims": rot}, **({} if i % 2 else {"q_rank": q_rank})}
        moe = {"kind": "moe", "expert": {"ff": ff, "limit": 7.0},
               "router": {"experts": 32, "top": 4, "groups": {"count": 4, "keep": 2}}}
        layers.append({"type": "latent_attention_2" if i % 2 else "latent_attention", "mixer": mixer,
                       "mlp": moe if i else {"kind": "dense", "ff": 3 * width}})
    return {"architecture": "Zarorax", "vocab": DESIGN_VOCAB, "width": width, "postln_alpha": 2.0, "norm": {"eps": 1e-5},
            "canon": {"taps": 4}, "layers": layers}


def _potatar(case):
    """Attention in chunks, talking heads beside linear attention, attention, the recurrence over shifted tokens."""
    width, dim = SIZES[case["sizes"]][:2]
    mlp = {"kind": "dense", "ff": 4 * width}
    heads = {"heads": 16, "kv_heads": 4, "dim": dim, "vdim": dim, "scale": dim ** -0.5, "mask": {"size": 1024}}
    plain = {"type": "attention", "mlp": mlp,
             "mixer": dict(heads, rot={"base": 10000.0, "dims": dim // 2}, v_mix=True)}
    both = {"type": "parallel", "mlp": mlp,
            "mixer": {"left": dict(heads, bias_max=1024, bias_rows=32), "left_scale": 1.0, "right_scale": 1.0,
                      "right": {"heads": 16, "dim": dim, "vdim": dim, "decay": [1.0 - 2.0 ** (-3 - i / 3) for i in range(16)]}}}
    wkv = {"type": "wkv", "mlp": None, "mixer": {"heads": 16, "dim": dim, "decay_rank": 64}}
    return {"architecture": "Potatar", "vocab": DESIGN_VOCAB, "width": width, "postln_alpha": 2.0, "logit_softcap": 30.0,
            "norm": {"eps": 1e-5}, "layers": [[plain, both, plain, wkv][i % 4] for i in range(case["layers"])]}


def _vuzinex(case):
    """Attention in chunks beside a matrix memory, the state space, attention beside gated linear attention, the state
    space."""
    width, dim = SIZES[case["sizes"]][:2]
    mlp = {"kind": "dense", "ff": 4 * width * 2 // 3 // 128 * 128}
    heads = {"heads": 16, "kv_heads": 4, "dim": dim, "vdim": dim, "scale": dim ** -0.5}
    banded = {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 2048}
    yarn = {"factor": 4.0, "original": 2048, "fast": 32.0, "slow": 1.0}
    rec = {"heads": 16, "dim": dim, "vdim": dim}
    one = {"type": "parallel", "mlp": mlp,
           "mixer": {"left": dict(heads, mask={"size": 1024}, rot={"base": 1e6, "dims": dim, "scaling": banded}),
                     "right": dict(rec, gate_cap=15.0), "left_scale": 1.0, "right_scale": 0.5}}
    two = {"type": "parallel_2", "mlp": mlp,
           "mixer": {"left": dict(heads, rot={"base": 10000.0, "dims": dim, "scaling": yarn}),
                     "right": dict(rec, tau=16.0, decay_rank=16), "left_scale": 1.0, "right_scale": 0.5}}
    ssm = {"type": "mamba2", "mlp": None,
           "mixer": {"heads": width // 32, "vdim": 64, "state": 128, "groups": 1, "conv": 4, "norm_groups": 1}}
    return {"architecture": "Vuzinex", "vocab": DESIGN_VOCAB, "width": width, "norm": {"eps": 1e-5}, "residual_mult": 0.8,
            "logit_scale": 0.5, "embedding": {"scale": 8.0, "bigram": {"buckets": 4093, "mul_prev": 23, "mul_cur": 41}},
            "loop": None, "layers": [[one, ssm, two, ssm][i % 4] for i in range(case["layers"])]}


def _config(case):
    return {"qwen3": _qwen3, "zarorax": _zarorax, "potatar": _potatar, "vuzinex": _vuzinex}[case["design"]](case)


def _vocab(config):
    return config["vocab_size"] if "vocab_size" in config else config["vocab"]


def _lengths(case):
    """(history, prompt) of every request; the golden section spreads ragged lengths over their range."""
    out = []
    for i in range(case["requests"]):
        f = 0.5 + (0.31 + 0.618034 * i) % 1.0 if case["ragged"] else 1.0
        out.append((int(case["history"] * f) // PAGE * PAGE, max(1, int(case["prompt"] * f))))
    return out


def _schedule(case):
    """The steps of a pass: lists of (request, first place after its history, tokens, whether logits are wanted)."""
    lengths, new = _lengths(case), case["new"]
    if not case["portion"]:
        first = [(i, 0, p, True) for i, (_, p) in enumerate(lengths)]
        return [first] + [[(i, p + s, 1, True) for i, (_, p) in enumerate(lengths)] for s in range(new)]
    steps, done = [], {}                      # done: request -> tokens it has decoded
    waiting = [(i, at, min(case["portion"], p - at), at + case["portion"] >= p)
               for i, (_, p) in enumerate(lengths) for at in range(0, p, case["portion"])]
    while waiting or any(d < new for d in done.values()):
        step = [(i, lengths[i][1] + d, 1, True) for i, d in done.items() if d < new]
        for i, *_ in step:
            done[i] += 1
        if waiting:
            step.append(waiting.pop(0))
            if step[-1][3]:
                done[step[-1][0]] = 0
        steps.append(step)
    return steps


def _generator(seed, name, device):
    return torch.Generator(device=device).manual_seed(zlib.crc32(f"{seed}:{name}".encode()) + (seed << 32))


def _tokens(case, seed, vocab):
    g = _generator(seed, "tokens", "cpu")
    return [torch.randint(0, vocab, (h + p + case["new"],), generator=g).tolist() for h, p in _lengths(case)]


def _weights(case, seed, config, device):
    """{name: tensor} in the case's type.  Matrices as the engine's own random weights are (0.02 wide), but for those
    that write into a pre-norm stream (a layer changes the stream of a trained model and does not replace it); gains,
    biases, decays and gates where trained models have them."""
    dtype = getattr(torch, case["dtype"])
    out = {}
    for name, info in expected_tensors(config_from_dict(config).to_model_spec()).items():
        if info.optional:
            continue
        g, shape = _generator(seed, name, device), tuple(info.shape)
        normal = lambda std: torch.randn(shape, generator=g, device=device) * std
        uniform = lambda lo, hi: torch.rand(shape, generator=g, device=device) * (hi - lo) + lo
        last = name.rsplit(".", 1)[-1]
        if name == "embed" and case["design"] in ("zarorax", "potatar"):
            t = normal(1.0)                                    # (designs that norm after the sum: rows of order one)
        elif name == "model.embed_tokens.weight":
            t = normal(0.3)
        elif name.endswith(("o_proj.weight", "down_proj.weight")):
            t = normal(0.02 * (2 * case["layers"]) ** -0.5)
        elif name.endswith(".router"):
            continue
        elif name.endswith(("q.norm", "q_norm.weight", "k.norm", "k_norm.weight")):
            t = 1.4 + normal(0.1)                              # scores two wide: some keys matter, most do not
        elif name.endswith("mlp.act"):
            t = torch.tensor([0.6, 0.3, 0.1, 0.0], device=device) + normal(0.05)
        elif name.endswith("talk"):
            t = torch.eye(shape[0], device=device) + normal(0.1)
        elif last == "rel" or last == "sink":
            t = normal(0.5)
        elif last.startswith("canon") or name.endswith("mix.conv"):
            t = normal(0.2)
        elif ".mu." in name or last == "vmix":
            t = uniform(0.2, 0.8)
        elif last == "w0":
            t = uniform(-6.0, -1.0)                            # decays from 0.998 to 0.69 a token
        elif last == "u":
            t = normal(0.3)
        elif name.endswith("right.f.b"):
            t = uniform(3.0, 6.0)                              # forget gates that open wide
        elif name.endswith("a2.b"):
            t = normal(1.0)
        elif last == "A_log":
            t = torch.log(uniform(1.0, 16.0))
        elif last == "dt_bias":
            step = torch.exp(uniform(math.log(1e-3), math.log(0.1)))
            t = torch.log(torch.expm1(step))
        elif info.init == "ones":
            t = 1.0 + normal(0.1)
        elif info.init == "zeros":
            t = normal(0.1)
        else:
            t = normal(0.02)
        out[name] = t.to(dtype)
    routers = [n for n in expected_tensors(config_from_dict(config).to_model_spec()) if n.endswith(".router")]
    if routers:
        # A trained router tells kinds of tokens apart: rows of the embedding lie around centres, and every kind has
        # experts of its own, in two groups.  (Routers drawn at random leave near ties, where the last bit of a sum
        # decides between two experts.)
        width = out["embed"].shape[1]
        centres = torch.randn(CLUSTERS, width, generator=_generator(seed, "centres", device), device=device)
        kinds = torch.arange(out["embed"].shape[0], device=device) % CLUSTERS
        out["embed"] = ((centres[kinds] + 0.7 * out["embed"].float()) / 1.22).to(dtype)
        for name in routers:
            layer = config["layers"][int(name[1:name.index(".")])]["mlp"]["router"]
            experts, top, groups = layer["experts"], layer["top"], layer["groups"]
            g = _generator(seed, name, "cpu")
            want = torch.rand(CLUSTERS, experts, generator=g) * 0.5
            for c in range(CLUSTERS):
                first = torch.randperm(groups["count"], generator=g)[:groups["keep"]]
                per = experts // groups["count"]
                for k in range(top):
                    free = [e for e in range(per) if want[c, first[k % len(first)] * per + e] < 1.0]
                    e = free[int(torch.randint(0, len(free), (1,), generator=g))]
                    want[c, first[k % len(first)] * per + e] = 3.0 + 0.3 * float(torch.rand(1, generator=g))
            out[name] = (want.to(device).t() @ centres * (1.22 / width)).to(dtype)
    return out


def prepare(case, seed):
    device = torch.device("cuda:0")
    config = _config(case)
    tokens = _tokens(case, seed, _vocab(config))
    weights = _weights(case, seed, config, device)
    if case["design"] == "vuzinex":           # (its projections are put together on the host, as tensors come from a file)
        weights = {name: t.cpu() for name, t in weights.items()}
    model = DecoderModel(config_from_dict(config).to_model_spec())
    model.load(weights, Runtime(device, getattr(torch, case["dtype"])))
    del weights
    lengths = _lengths(case)
    pages = sum((h + 2 * (p + case["new"])) // PAGE + 4 for h, p in lengths)
    keeps = case["history"] > 0
    runner = ModelRunner(model, page_size=PAGE, num_pages=pages, max_requests=case["requests"],
                         prefix_sharing=keeps, keep_freed_prefixes=keeps)
    if keeps:                                 # the earlier turns: their pages stay for the requests that go on from them
        for i in range(case["requests"]):
            runner.add_request(i)
        at = [0] * case["requests"]
        while any(a < h for a, (h, _) in zip(at, lengths)):
            step, room = [], 4096
            for i, (h, _) in enumerate(lengths):
                n = min(h - at[i], room, 2048)
                if n > 0:
                    step.append(StepEntry(i, tokens[i][at[i]:at[i] + n], []))
                    at[i] += n
                    room -= n
            runner.step(step)
        for i in range(case["requests"]):
            runner.free_request(i)
    steps = [[StepEntry(i, tokens[i][lengths[i][0] + a:lengths[i][0] + a + n], [n - 1] if want else [])
              for i, a, n, want in step] for step in _schedule(case)]
    kept = [tokens[i][:h + 1] for i, (h, _) in enumerate(lengths)]
    return {"runner": runner, "steps": steps, "kept": kept, "keeps": keeps}


def run(state):
    runner, live, out = state["runner"], set(), []
    for step in state["steps"]:
        for e in step:
            if e.req_id not in live:
                live.add(e.req_id)
                runner.add_request(e.req_id)
                if state["keeps"]:
                    runner.cache.match_prefix(e.req_id, state["kept"][e.req_id])
        logits = runner.step(step)
        if logits.shape[0]:
            out.append(logits)
    for i in live:
        runner.free_request(i)
    return out


# ---- what a pass cannot do without -------------------------------------------------------------------------------
def _pairs(first, n, size=None):
    """(query, key) pairs of n queries from position ``first``, with all keys or those of their chunk of ``size``."""
    return sum((p % size if size else p) + 1 for p in range(first, first + n))


def _attention(config):
    """Per layer: (numbers a pair of query and key costs, numbers a key keeps, chunk or None)."""
    if "layers" not in config:
        d, h, g = config["head_dim"], config["num_attention_heads"], config["num_key_value_heads"]
        return [(2 * h * d, 2 * g * d, None)] * config["num_hidden_layers"]
    out = []
    for layer in config["layers"]:
        m = layer["mixer"]
        m = m.get("left", m)
        if layer["type"] in ("wkv", "mamba2"):
            out.append((0, 0, None))
        elif "kv_rank" in m:
            out.append((m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"]), m["kv_rank"] + m["rot_dim"], None))
        else:
            out.append((m["heads"] * (m["dim"] + m["vdim"]), m["kv_heads"] * (m["dim"] + m["vdim"]),
                        m["mask"]["size"] if m.get("mask") else None))
    return out


def work(case):
    config = _config(case)
    size = torch.finfo(getattr(torch, case["dtype"])).bits // 8
    vocab, lengths, attention = _vocab(config), _lengths(case), _attention(config)
    dense = experts = head = top = count = 0
    for name, info in expected_tensors(config_from_dict(config).to_model_spec()).items():
        n = math.prod(info.shape)
        if info.shape and info.shape[0] == vocab:
            head = n
        elif ".mlp.e" in name:
            experts += n
        elif len(info.shape) == 2 and name != "bigram":
            dense += n
    for layer in config.get("layers", ()):
        if layer["mlp"] and layer["mlp"]["kind"] == "moe":
            count, top = layer["mlp"]["router"]["experts"], layer["mlp"]["router"]["top"]
    moved = flops = 0.0
    for step in _schedule(case):
        tokens = sum(n for _, _, n, _ in step)
        rows = sum(1 for *_, want in step if want)
        used = min(1.0, tokens * top / count) if count else 0.0
        moved += size * (dense + used * experts + (head if rows else 0)) + 4.0 * rows * vocab
        flops += 2.0 * tokens * (dense + (experts * top / count if count else 0)) + 2.0 * rows * head
        for i, a, n, _ in step:
            for pair, key, chunk in attention:
                first = lengths[i][0] + a
                flops += 2.0 * pair * _pairs(first, n, chunk)
                seen = first + n - (first // chunk * chunk if chunk else 0)
                moved += size * key * (seen + n)
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    """Two to four times what was measured between the engine's logits and the same in 64 bits: 0.013 at the large
    models' sizes and with matrix memories (a sum over many keys of values that cancel), 0.004 at the small model's
    with all its layers, 0.003 in the designs that norm after the sum; 7e-6 with 32-bit weights, caches and sums.  The
    largest single difference was five times as much."""
    if case["dtype"] == "float32":
        rel = 3e-5
    elif case["design"] in ("zarorax", "potatar"):
        rel = 0.012
    else:
        rel = 0.015 if case["sizes"] == "0.6b" else 0.03
    return {"rel": rel, "max": 10 * rel}


# ---- the same in 64 bits -----------------------------------------------------------------------------------------
def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + eps)


def _sigmoid(x):
    return torch.sigmoid(x)


def _silu(x):
    return x * torch.sigmoid(x)


def _rotate(x, freqs, halves, gain=1.0):
    """x [T, heads, D]: pairs (i, i + n) or (2 i, 2 i + 1) turned by position times frequency."""
    n = len(freqs)
    a = torch.arange(x.shape[0], device=x.device, dtype=x.dtype)[:, None, None] * torch.tensor(freqs, device=x.device, dtype=x.dtype)
    c, s = torch.cos(a) * gain, torch.sin(a) * gain
    i = slice(0, n) if halves else slice(0, 2 * n, 2)
    j = slice(n, 2 * n) if halves else slice(1, 2 * n, 2)
    out = x.clone()
    out[..., i] = x[..., i] * c - x[..., j] * s
    out[..., j] = x[..., j] * c + x[..., i] * s
    return out


def _frequencies(base, dims):
    return [base ** (-2.0 * i / dims) for i in range(dims // 2)]


def _attend(q, k, v, scale, chunk=None, sink=None, bias=None, talk=None):
    """q [T, H, D], k and v [T, G, ...] -> [T, H * Dv]; bias [H, distance], talk [H, H] over the heads' scores."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    k, v = (t.repeat_interleave(H // G, dim=1).transpose(0, 1).contiguous() for t in (k, v))
    out = torch.empty(T, H, v.shape[2], dtype=q.dtype, device=q.device)
    block = min(chunk or 512, 512)
    for a in range(0, T, block):
        b = min(T, a + block)
        lo = a // chunk * chunk if chunk else 0
        s = torch.matmul(q[a:b].transpose(0, 1), k[:, lo:b].transpose(1, 2)) * scale
        d = torch.arange(a, b, device=q.device)[:, None] - torch.arange(lo, b, device=q.device)[None, :]
        if bias is not None:
            s = s + bias[:, d.clamp(min=0)]
        if talk is not None:
            s = torch.matmul(talk, s.reshape(H, -1)).view(s.shape)
        s = s.masked_fill(d < 0, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink.view(H, 1, 1).expand(H, b - a, 1)], dim=2)
        p = torch.softmax(s, dim=-1)[..., :b - lo]
        out[a:b] = torch.matmul(p, v[:, lo:b]).transpose(0, 1)
    return out.reshape(T, -1)


def _convolve(x, w):
    """Causal, a filter per channel: x [T, C], w [C, taps]."""
    taps = w.shape[1]
    padded = torch.cat([x.new_zeros(taps - 1, x.shape[1]), x])
    return sum(w[:, j] * padded[j:j + x.shape[0]] for j in range(taps))


def _recur(q, k, v, keep, bonus=None):
    """S <- keep_t S + k_t v_t^T, o_t = S^T q_t, per head; with a bonus o_t = (S before + bonus k_t v_t^T)^T r_t."""
    T, H, D = q.shape
    S = q.new_zeros(H, D, v.shape[2])
    out = q.new_empty(T, H, v.shape[2])
    keep = keep.unsqueeze(-1)
    for t in range(T):
        kv = k[t].unsqueeze(2) * v[t].unsqueeze(1)
        if bonus is None:
            S = S * keep[t] + kv
            out[t] = torch.bmm(q[t].unsqueeze(1), S)[:, 0]
        else:
            out[t] = torch.bmm(q[t].unsqueeze(1), S + bonus.unsqueeze(2) * kv)[:, 0]
            S = S * keep[t] + kv
    return out


class _Exact:
    """One sequence after another through a model in 64 bits; ``t(name)`` is a weight."""

    def __init__(self, config, weights):
        self.c, self.w = config, weights

    def t(self, name):
        return self.w[name].double()

    def mul(self, x, name):
        return x @ self.t(name).t()

    # Qwen3
    def qwen3(self, tokens, rows):
        c, t, mul = self.c, self.t, self.mul
        T, D, H, G, eps = len(tokens), c["head_dim"], c["num_attention_heads"], c["num_key_value_heads"], c["rms_norm_eps"]
        freqs = _frequencies(c["rope_theta"], D)
        x = self.w["model.embed_tokens.weight"][tokens].double()
        for i in range(c["num_hidden_layers"]):
            p = f"model.layers.{i}."
            h = _rms(x, eps) * t(p + "input_layernorm.weight")
            heads = lambda n, g: mul(h, f"{p}self_attn.{n}_proj.weight").view(T, g, D)
            q = _rotate(_rms(heads("q", H), eps) * t(p + "self_attn.q_norm.weight"), freqs, True)
            k = _rotate(_rms(heads("k", G), eps) * t(p + "self_attn.k_norm.weight"), freqs, True)
            x = x + mul(_attend(q, k, heads("v", G), D ** -0.5), p + "self_attn.o_proj.weight")
            h = _rms(x, eps) * t(p + "post_attention_layernorm.weight")
            x = x + mul(_silu(mul(h, p + "mlp.gate_proj.weight")) * mul(h, p + "mlp.up_proj.weight"), p + "mlp.down_proj.weight")
        x = _rms(x[rows], eps) * t("model.norm.weight")
        return mul(x, "model.embed_tokens.weight" if c["tie_word_embeddings"] else "lm_head.weight")

    # Zarorax
    def zarorax(self, tokens, rows):
        c, t, mul, T = self.c, self.t, self.mul, len(tokens)
        eps, alpha = c["norm"]["eps"], c["postln_alpha"]
        x = t("embed")[tokens]
        for i, layer in enumerate(c["layers"]):
            p, m = f"l{i}.", layer["mixer"]
            h = x + _convolve(x, t(p + "canon1"))
            direct = layer["type"] == "latent_attention_2"
            q = mul(h, p + "mix.q") if direct else mul(_rms(mul(h, p + "mix.dq"), eps) * t(p + "mix.dq.norm"), p + "mix.uq")
            q = q.view(T, m["heads"], m["dim"] + m["rot_dim"])
            kv = mul(h, p + "mix.dkv")
            latent = _rms(kv[:, :m["kv_rank"]], eps) * t(p + "mix.dkv.norm")
            freqs = _frequencies(m["rot"]["base"], m["rot"]["dims"])
            q = torch.cat([q[..., :m["dim"]], _rotate(q[..., m["dim"]:], freqs, False)], dim=-1)
            k_rot = _rotate(kv[:, None, m["kv_rank"]:], freqs, False).expand(T, m["heads"], m["rot_dim"])
            k = torch.cat([mul(latent, p + "mix.uk").view(T, m["heads"], m["dim"]), k_rot], dim=-1)
            y = _attend(q, k, mul(latent, p + "mix.uv").view(T, m["heads"], m["vdim"]), m["scale"])
            if direct:
                y = y * _sigmoid(mul(h, p + "mix.g"))
            x = _rms(alpha * x + mul(y, p + "mix.o"), eps) * t(p + "norm1")
            if layer["mlp"]["kind"] == "dense":
                z = mul(x, p + "mlp.up")
                a = t(p + "mlp.act")
                y = mul(a[0] * _rms(z, eps) + a[1] * _rms(z * z, eps) + a[2] * _rms(z ** 3, eps) + a[3], p + "mlp.down")
            else:
                y = self._mixture(x, p + "mlp.", layer["mlp"])
            x = _rms(alpha * x + y, eps) * t(p + "norm2")
        return mul(_rms(x[rows], eps) * t("final.norm"), "head")

    def _mixture(self, x, p, mlp):
        r, limit = mlp["router"], mlp["expert"]["limit"]
        s = torch.softmax(self.mul(x, p + "router"), dim=-1)
        g = s.view(len(x), r["groups"]["count"], -1)
        best = g.amax(dim=-1).topk(r["groups"]["keep"], dim=-1).indices
        kept = torch.zeros(g.shape[:2], dtype=torch.bool, device=x.device).scatter_(1, best, True)
        value, chosen = g.masked_fill(~kept.unsqueeze(-1), -1.0).reshape(s.shape).topk(r["top"], dim=-1)
        out = torch.zeros_like(x)
        for e in range(r["experts"]):
            rows, place = (chosen == e).nonzero(as_tuple=True)
            if len(rows):
                gate = self.mul(x[rows], f"{p}e{e}.gate").clamp(max=limit)
                up = self.mul(x[rows], f"{p}e{e}.up").clamp(-limit, limit)
                y = self.mul(gate * _sigmoid(1.702 * gate) * (up + 1.0), f"{p}e{e}.down")
                out.index_add_(0, rows, y * value[rows, place].unsqueeze(1))
        return out

    # Potatar
    def potatar(self, tokens, rows):
        c, t, mul, T = self.c, self.t, self.mul, len(tokens)
        eps, alpha, first = c["norm"]["eps"], c["postln_alpha"], None
        x = t("embed")[tokens]
        for i, layer in enumerate(c["layers"]):
            p, m = f"l{i}.mix.", layer["mixer"]
            if layer["type"] == "attention":
                H, G, D, Dv = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
                proj = lambda n: mul(x, p + n) + t(f"{p}{n}.b")
                freqs = _frequencies(m["rot"]["base"], m["rot"]["dims"])
                q = _rotate((_rms(proj("q"), eps) * t(p + "q.norm")).view(T, H, D), freqs, True)
                k = _rotate((_rms(proj("k"), eps) * t(p + "k.norm")).view(T, G, D), freqs, True)
                v = _rms(proj("v").view(T, G, Dv), eps)
                first = v if first is None else first
                v = v if first is v else (1.0 - t(p + "vmix")) * v + t(p + "vmix") * first
                y = mul(_attend(q, k, v, m["scale"], m["mask"]["size"]), p + "o") + t(p + "o.b")
            elif layer["type"] == "parallel":
                y = m["left_scale"] * self._talking(x, p + "left.", m["left"], eps) + \
                    m["right_scale"] * self._linear(x, p + "right.", m["right"], eps)
            else:
                y = self._shifted(x, p, m, eps)
            x = _rms(alpha * x + y, eps) * t(f"l{i}.norm1")
            if layer["mlp"] is not None:
                z = mul(x, f"l{i}.mlp.up")
                y = mul(0.5 * z * (1.0 + torch.erf(z / math.sqrt(2.0))), f"l{i}.mlp.down")
                x = _rms(alpha * x + y, eps) * t(f"l{i}.norm2")
        logits = mul(_rms(x[rows], eps) * t("final.norm"), "head")
        return c["logit_softcap"] * torch.tanh(logits / c["logit_softcap"])

    def _talking(self, x, p, m, eps):
        t, T, H, G, D = self.t, len(x), m["heads"], m["kv_heads"], m["dim"]
        q = (self.mul(x, p + "q") + t(p + "q.b")).view(T, H, D)
        k = (self.mul(x, p + "k") + t(p + "k.b")).view(T, G, D)
        table = t(p + "rel")
        n, half, far = len(table), len(table) // 2, float(m["bias_max"])
        row = [d if d < half else min(n - 1, half + int(math.floor(math.log(d / half) / math.log(far / half) * (n - half))))
               for d in range(m["mask"]["size"])]
        bias = table[torch.tensor(row, device=x.device)].t()
        y = _attend(_rms(q, eps) * t(p + "q.norm"), _rms(k, eps) * t(p + "k.norm"), k, m["scale"], m["mask"]["size"],
                    bias=bias, talk=t(p + "talk"))
        return self.mul(y, p + "o") + t(p + "o.b")

    def _linear(self, x, p, m, eps):
        T, H = len(x), m["heads"]
        q, k, v = (_silu(self.mul(x, p + n)).view(T, H, -1) for n in "qkv")
        keep = torch.tensor(m["decay"], dtype=x.dtype, device=x.device).view(1, H, 1).expand(T, H, m["dim"])
        y = _recur(q, k, v, keep).reshape(T, -1)
        return self.mul(_rms(y, eps) * self.t(p + "norm") * _sigmoid(self.mul(x, p + "g")), p + "o")

    def _shifted(self, x, p, m, eps):
        t, mul, T, H = self.t, self.mul, len(x), m["heads"]
        before = torch.cat([torch.zeros_like(x[:1]), x[:-1]])
        blend = lambda s: x + (before - x) * t(p + "mu." + s)
        r, k, v = (mul(blend(s), p + s).view(T, H, -1) for s in "rkv")
        decay = torch.exp(-torch.exp(mul(torch.tanh(mul(blend("w"), p + "w1")), p + "w2") + t(p + "w0"))).view(T, H, -1)
        y = _rms(_recur(r, k, v, decay, t(p + "u")), eps).reshape(T, -1) * t(p + "norm")
        return mul(y * _silu(mul(blend("g"), p + "g")), p + "o")

    # Vuzinex
    def vuzinex(self, tokens, rows):
        c, t, mul = self.c, self.t, self.mul
        eps, mult, pair = c["norm"]["eps"], c["residual_mult"], c["embedding"]["bigram"]
        norm = lambda z, n: _rms(z, eps) * (1.0 + t(n))
        second = [pair["buckets"]] + [(a * pair["mul_prev"] + b * pair["mul_cur"]) % pair["buckets"] for a, b in zip(tokens, tokens[1:])]
        x = t("embed")[tokens] * c["embedding"]["scale"] + t("bigram")[second]
        for i, layer in enumerate(c["layers"]):
            p, m = f"l{i}.", layer["mixer"]
            h = norm(x, p + "norm1")
            if layer["type"] == "mamba2":
                y = self._state_space(h, p + "mix.", m, eps)
            else:
                one = layer["type"] == "parallel"
                left = (self._sink_attention if one else self._gated_attention)(h, p + "mix.left.", m["left"], eps)
                right = (self._memory if one else self._gated_linear)(h, p + "mix.right.", m["right"], eps)
                y = m["left_scale"] * left + m["right_scale"] * right
            x = x + mult * norm(y, p + "norm1b")
            if layer["mlp"] is not None:
                h = norm(x, p + "norm2")
                y = _silu(mul(h, p + "mlp.gate") + t(p + "mlp.gate.b")) * (mul(h, p + "mlp.up") + t(p + "mlp.up.b"))
                x = x + mult * norm(mul(y, p + "mlp.down") + t(p + "mlp.down.b"), p + "norm2b")
        return mul(norm(x[rows], "final.norm"), "embed") * c["logit_scale"]

    def _sink_attention(self, h, p, m, eps):
        rot, sc, T = m["rot"], m["rot"]["scaling"], len(h)
        freqs = []
        for f in _frequencies(rot["base"], rot["dims"]):
            s = (sc["original"] * f / (2.0 * math.pi) - sc["low"]) / (sc["high"] - sc["low"])
            freqs.append(f / sc["factor"] if s < 0 else f if s > 1 else (1.0 - s) * f / sc["factor"] + s * f)
        q, k, v = (self.mul(h, p + n).view(T, g, -1) for n, g in (("q", m["heads"]), ("k", m["kv_heads"]), ("v", m["kv_heads"])))
        y = _attend(_rotate(q, freqs, False), _rotate(k, freqs, False), v, m["scale"], m["mask"]["size"], sink=self.t(p + "sink"))
        return self.mul(y, p + "o")

    def _gated_attention(self, h, p, m, eps):
        rot, sc, t, T = m["rot"], m["rot"]["scaling"], self.t, len(h)
        dims, base = rot["dims"], rot["base"]
        at = lambda turns: dims * math.log(sc["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))
        lo, hi = max(math.floor(at(sc["fast"])), 0), min(math.ceil(at(sc["slow"])), dims - 1)
        freqs = []
        for i, f in enumerate(_frequencies(base, dims)):
            r = min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0)
            freqs.append(f / sc["factor"] * r + f * (1.0 - r))
        gain = 0.1 * math.log(sc["factor"]) + 1.0
        q, k, v = ((self.mul(h, p + n) + t(f"{p}{n}.b")).view(T, g, -1)
                   for n, g in (("q", m["heads"]), ("k", m["kv_heads"]), ("v", m["kv_heads"])))
        q = _rotate(_rms(q, eps) * t(p + "q.norm"), freqs, False, gain)
        k = _rotate(_rms(k, eps) * t(p + "k.norm"), freqs, False, gain)
        return self.mul(_attend(q, k, v, m["scale"]) * _sigmoid(self.mul(h, p + "g")), p + "o")

    def _memory(self, h, p, m, eps):
        t, T, H, cap = self.t, len(h), m["heads"], m["gate_cap"]
        q, k, v = (self.mul(h, p + n).view(T, H, -1) for n in "qkv")
        q = q * m["dim"] ** -0.5
        write, forget = (cap * torch.tanh((self.mul(h, p + n) + t(f"{p}{n}.b")) / cap) for n in "if")
        forget = torch.nn.functional.logsigmoid(forget)
        S, n, top = h.new_zeros(H, m["dim"], m["vdim"]), h.new_zeros(H, m["dim"]), h.new_zeros(H)
        out = h.new_empty(T, H, m["vdim"])
        for i in range(T):
            new = torch.maximum(forget[i] + top, write[i])
            a, b = torch.exp(forget[i] + top - new).unsqueeze(1), torch.exp(write[i] - new).unsqueeze(1)
            S = a.unsqueeze(2) * S + (b * k[i]).unsqueeze(2) * v[i].unsqueeze(1)
            n, top = a * n + b * k[i], new
            down = torch.maximum((n * q[i]).sum(dim=-1).abs(), torch.exp(-top)) + 1e-6
            out[i] = torch.bmm(q[i].unsqueeze(1), S)[:, 0] / down.unsqueeze(1)
        return self.mul(_rms(out, eps).reshape(T, -1) * t(p + "norm") * _sigmoid(self.mul(h, p + "g")), p + "o")

    def _gated_linear(self, h, p, m, eps):
        t, T, H = self.t, len(h), m["heads"]
        q, k, v = (self.mul(h, p + n).view(T, H, -1) for n in "qkv")
        z = self.mul(self.mul(h, p + "a1"), p + "a2") + t(p + "a2.b")
        keep = torch.exp(torch.nn.functional.logsigmoid(z) / m["tau"]).view(T, H, -1)
        y = _rms(_recur(q * m["dim"] ** -0.5, k, v, keep), eps) * t(p + "norm")
        return self.mul(y.reshape(T, -1) * _silu(self.mul(h, p + "g")), p + "o")

    def _state_space(self, h, p, m, eps):
        t, T, H, N, G = self.t, len(h), m["heads"], m["state"], m["groups"]
        inner = H * m["vdim"]
        z, xbc, dt = torch.split(self.mul(h, p + "in"), [inner, inner + 2 * G * N, H], dim=-1)
        x, B, C = torch.split(_silu(_convolve(xbc, t(p + "conv")) + t(p + "conv.b")), [inner, G * N, G * N], dim=-1)
        dt = torch.nn.functional.softplus(dt + t(p + "dt_bias"))
        x = x.reshape(T, H, -1)
        B, C = (a.reshape(T, G, N).repeat_interleave(H // G, dim=1) for a in (B, C))
        keep = torch.exp(-torch.exp(t(p + "A_log")) * dt).unsqueeze(-1).expand(T, H, N)
        y = _recur(C, B * dt.unsqueeze(-1), x, keep) + t(p + "D").view(1, H, 1) * x
        y = _rms((y.reshape(T, inner) * _silu(z)).view(T, m["norm_groups"], -1), eps).reshape(T, inner)
        return self.mul(y * t(p + "norm"), p + "o")


def exact(case, seed):
    device = torch.device("cuda:0" if torch.cuda.is_available() else "cpu")
    config, lengths = _config(case), _lengths(case)
    tokens = _tokens(case, seed, _vocab(config))
    model = _Exact(config, _weights(case, seed, config, device))
    places = [[] for _ in lengths]             # per request: where logits are wanted, in order
    for step in _schedule(case):
        for i, a, n, want in step:
            if want:
                places[i].append(lengths[i][0] + a + n - 1)
    logits = [getattr(model, case["design"])(tokens[i], places[i]) for i in range(len(lengths))]
    taken, out = [0] * len(lengths), []
    for step in _schedule(case):
        rows = []
        for i, _, _, want in step:
            if want:
                rows.append(logits[i][taken[i]])
                taken[i] += 1
        if rows:
            out.append(torch.stack(rows))
    return out
