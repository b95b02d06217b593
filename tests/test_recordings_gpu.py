"""One recording a shape, whether a step's caller wants the logits or the picks."""
import pytest
import torch

from tiny import make_folder

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    from qwen_engine_amd.engine import load_model
    return load_model(make_folder(tmp_path_factory.mktemp("rec"), "F", std=0.05), dtype="bfloat16", device=DEV)


@pytest.fixture
def runner(model):
    from qwen_engine_amd.engine import ModelRunner
    return ModelRunner(model, page_size=16, num_pages=400, max_requests=16)


TOKENS = torch.randint(0, 400, (900,), generator=torch.Generator().manual_seed(2)).tolist()


@pytest.mark.parametrize("first", [False, True])
@pytest.mark.parametrize("kind", ["decode", "mixed", "portion"])
def test_logits_and_picks_in_turn(runner, kind, first):
    """Steps of one shape that ask for logits and for picks in turn: recorded again once at the most, where the first did not ask for picks.  Pairs of
    equal requests run the same tokens in both ways."""
    from qwen_engine_amd.engine import StepEntry
    for i in range(4):
        runner.add_request(i)
        runner.step([StepEntry(i, TOKENS[:20], [])])
    state = lambda: (runner.graph_steps_of[kind], runner.graphs_recorded, len(runner._graphs))
    before = state()
    for turn in range(6):
        greedy = first ^ bool(turn % 2)
        if kind == "portion":
            runner.add_request("p")
            entries = [StepEntry("p", TOKENS[100:356], [255])]
        else:
            entries = [StepEntry(i, [TOKENS[400 + turn // 2]], [0]) for i in ((0, 1) if turn % 2 else (2, 3))]
            if kind == "mixed":
                runner.add_request("p")
                entries.append(StepEntry("p", TOKENS[100:140], [39]))
        got = runner.step(entries, greedy=greedy)
        picks = got if greedy else got.argmax(1).tolist()
        if turn % 2:
            assert picks == last
        last = picks
        if kind != "decode":
            runner.free_request("p")
    steps, recorded, kept = (b - a for a, b in zip(before, state()))
    assert (steps, recorded, kept) == (6, 1 if first else 2, 1)


def test_a_portion_that_wants_nothing(runner):
    from qwen_engine_amd.engine import StepEntry
    for turn in range(4):
        runner.add_request("p")
        got = runner.step([StepEntry("p", TOKENS[:256], [])], greedy=bool(turn % 2))
        assert len(got) == 0
        runner.free_request("p")
    recorded, steps = runner.graphs_recorded, runner.graph_steps_of["portion"]
    assert (recorded, steps) == (1, 4)
