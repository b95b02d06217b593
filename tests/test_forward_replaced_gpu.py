"""A program that puts a loop of its own in the place of the model's forward: recorded steps bring the block tables up to date all the same."""
import pytest
import torch

from tiny import make_folder
from qwen_engine_amd.parts import DecoderModel
from qwen_engine_amd.parts.base import add_pending

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _plain_loop(self, ctx, bindings):
    """The steps of the forward pass one by one; of ctx it knows what the layers are given."""
    from qwen_engine_amd.kernels import ops
    h, pending = ops.embedding(ctx.token_ids, self.embed), None
    for i, entry in enumerate(self.spec.schedule):
        pending = self.blocks[entry.layer].forward(h, pending, ctx, bindings[i])
    add_pending(h, pending)
    if not ctx.logit_rows.shape[0]:
        return torch.empty((0, self.spec.vocab_size), device=h.device)
    return ops.gemm(self.final_norm.forward(h, ctx.rt, rows=ctx.logit_rows), self.head, out_dtype=torch.float32)


def _run(folder, seen, use_graphs=True):
    from qwen_engine_amd.engine import ModelRunner, StepEntry, load_model
    model = load_model(folder, dtype="bfloat16", device=DEV)
    if seen == "wrapped":                    # (a trace: the model's own forward inside)
        real = model.forward
        model.forward = lambda ctx, bindings: real(ctx, bindings)
    elif seen == "derived":
        model.__class__ = type("Mine", (DecoderModel,), {"forward": _plain_loop})
    elif seen == "loop":
        model.forward = lambda ctx, bindings: _plain_loop(model, ctx, bindings)
    runner = ModelRunner(model, page_size=16, num_pages=200, max_requests=16, debug_poison=True, use_graphs=use_graphs)
    tokens = torch.randint(0, 400, (500,), generator=torch.Generator().manual_seed(1)).tolist()
    out = []
    for i in range(10):
        runner.add_request(i)
    out.append(runner.step([StepEntry(0, tokens[:256], [255])]))               # a portion, recorded
    for i in range(1, 10):
        out.append(runner.step([StepEntry(i, tokens[:7 + 3 * i], [0])]))
    for t in range(20):                                                         # single tokens that pass into new pages
        out.append(runner.step([StepEntry(i, [tokens[300 + t + i]], [0]) for i in range(9)]))
    for t in range(3):                                                          # and beside a portion
        out.append(runner.step([StepEntry(i, [tokens[350 + t + i]], [0]) for i in range(9)] + [StepEntry(9, tokens[:40], [39])]))
    counts = dict(runner.graph_steps_of)
    torch.cuda.synchronize()
    return [x.cpu() for x in out], counts


@pytest.mark.parametrize("seen", ["wrapped", "loop", "derived"])
def test_recorded_steps_with_another_forward(tmp_path, seen):
    folder = make_folder(tmp_path, "F", std=0.05)
    want, counts = _run(folder, None)
    assert counts["decode"] and counts["mixed"] and counts["portion"]
    got, same = _run(folder, seen)
    assert same == counts
    for a, b in zip(want, got):
        assert bool(b.isfinite().all())
        # (other kernels, with the roundings of 16 bits in other places; a page that is missed is NaN, or another request's)
        assert float((a - b).abs().max()) <= 2e-2 * float(a.abs().max())
    if seen == "wrapped":
        assert all(torch.equal(a, b) for a, b in zip(want, got))
