"""How a product's kernel is chosen and remembered (kernels/blaslt.py), with the library, the kernels and their times stood in for."""
import json
from types import SimpleNamespace

import pytest
import torch

from dinfer_amd.kernels import blaslt, tiles

ALGORITHMS = [SimpleNamespace(data=bytes([i] * 16)) for i in range(3)]


@pytest.fixture
def choices(monkeypatch, tmp_path):
    """blaslt with nothing chosen, a plan file of its own, and all candidates equally fast."""
    for name in ("_plans", "_ends", "_settings"):
        monkeypatch.setattr(blaslt, name, dict(getattr(blaslt, name)))
    blaslt._plans.clear()
    blaslt._ends.clear()
    for name in ("_stored", "_stored_path"):
        monkeypatch.setattr(blaslt, name, None)
    monkeypatch.setattr(blaslt, "_stored_dirty", False)
    monkeypatch.setattr(tiles, "shapes", lambda: [(96, 64, 384, False), (128, 128, 256, True), (256, 256, 192, True)])
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    ran = []
    monkeypatch.setattr(blaslt.ops, "gemm_tile", lambda a, w, out, m, shape, **_: ran.append(shape))

    def tune(handle, plan, *rest):
        plan.index, plan.tuned, plan.algo = 1, True, plan.candidates[1]

    monkeypatch.setattr(blaslt, "_tune", tune)
    monkeypatch.setattr(blaslt, "_least_of_three", lambda a, m, run: 10.0)
    monkeypatch.setattr(blaslt, "_in_trains", lambda w, forms, alone: [10.0] * len(forms), raising=False)
    blaslt.configure(tuning="measured", plan_file=str(tmp_path / "first.json"))
    return SimpleNamespace(ran=ran, folder=tmp_path)


A, W, OUT = (torch.zeros(s, dtype=torch.bfloat16) for s in ((320, 512), (1024, 512), (320, 512)))


def _end():
    return blaslt.with_end(A, W, OUT, 320, "gated", 300, lambda w: None)


def _product():
    plan = blaslt._plans.setdefault("p", SimpleNamespace(asked=False, tuned=False, candidates=ALGORITHMS, algo=ALGORITHMS[0], index=0,
                                                         tile=None, tiles=[]))
    key = (torch.device("cpu"), 320, 512, 512, 512, 512, 512, torch.bfloat16, True, False)
    if not plan.tuned:
        blaslt._choose(None, plan, key, A, W, OUT, None, blaslt._zero)
    return plan


def test_a_plan_file_named_later_is_asked_and_written(choices):
    """Shapes that were met before anything was measured, under one plan file, are looked up in the next one, and what is measured then is
    written there."""
    assert not _end() and not _product().tuned
    second = choices.folder / "second.json"
    blaslt.configure(plan_file=str(second))
    with blaslt.measuring():
        _end()
        _product()
    assert len(json.loads(second.read_text())) == 2
    assert not (choices.folder / "first.json").exists()


def test_a_plan_file_named_later_is_read(choices):
    assert not _end() and not _product().tuned
    second = choices.folder / "second.json"
    skey = ",".join(map(str, (320, 1024, 512, 512, 512, 512, "gated")))
    second.write_text(json.dumps({skey: {"tile": [256, 256]}, "320,512,512,512,512,512,bf16,0": {"index": 2, "algo": ALGORITHMS[2].data.hex()}}))
    blaslt.configure(plan_file=str(second))
    assert _end() and choices.ran == [2]
    assert _product().index == 2


def test_no_tile_where_nothing_could_be_timed(choices, monkeypatch):
    """Launches that all fail while they are timed leave the pass of its own, and no choice in the file."""
    monkeypatch.setattr(blaslt, "_least_of_three", lambda a, m, run: float("inf"))
    with blaslt.measuring():
        assert not _end()
    assert not choices.ran and not (choices.folder / "first.json").exists()


@pytest.mark.parametrize("alone,trains,tile", [
    ((10.0, 11.0, 11.2), (10.0, 10.5, 11.0), None),      # the tiles lose by less than a single launch's error: the product and its pass
    ((10.0, 9.9, 9.8), (10.0, 9.9, 9.9), None),          # they win by less than trains repeat
    ((10.0, 11.0, 11.2), (10.0, 9.8, 9.4), 2),           # they win in trains, the second of them
    ((10.0, 11.0, 11.2), (10.0, 9.4, 9.3), 1)])          # both alike: the first
def test_ends_are_chosen_as_they_run_in_a_step(choices, monkeypatch, alone, trains, tile):
    """By trains, without an allowance for either side, and the product and its pass where they are as fast; the forms are the pass first, then the
    tiles in the order of their estimate."""
    left = list(alone)
    monkeypatch.setattr(blaslt, "_least_of_three", lambda a, m, run: left.pop(0))
    monkeypatch.setattr(blaslt, "_in_trains", lambda w, forms, alone: list(trains), raising=False)
    monkeypatch.setattr(tiles, "candidates", lambda m, n, k, gated: [1, 2])
    with blaslt.measuring():
        assert _end() == (tile is not None)
    stored = json.loads((choices.folder / "first.json").read_text())
    assert [v["tile"] for v in stored.values()] == [None if tile is None else list(tiles.shapes()[tile][:2])]
    assert choices.ran == ([] if tile is None else [tile])


@pytest.mark.parametrize("alone,forms,tile", [
    ((10.0, 13.0, 14.0), 0, None), ((13.0, 10.0, 14.0), 0, 1),      # one is far ahead: no trains
    ((10.0, 11.0, 12.0), 2, 1), ((10.0, 11.0, 11.4), 3, 1),         # the second tile only where it is near the first
    ((float("inf"), 11.0, 12.0), 0, 1), ((10.0, float("inf"), 11.0), 2, 2)])     # what failed is left out
def test_trains_only_of_forms_that_may_win(choices, monkeypatch, alone, forms, tile):
    left, tried = list(alone), []
    monkeypatch.setattr(blaslt, "_least_of_three", lambda a, m, run: left.pop(0))
    monkeypatch.setattr(blaslt, "_in_trains", lambda w, f, alone: (tried.append(len(f)), [10.0, 9.0, 9.0][:len(f)])[1])
    monkeypatch.setattr(tiles, "candidates", lambda m, n, k, gated: [1, 2])
    with blaslt.measuring():
        assert _end() == (tile is not None)
    assert tried == ([forms] if forms else []) and choices.ran == ([] if tile is None else [tile])


def test_a_timed_run_finds_its_own_rows_in_the_caches(monkeypatch):
    """Of an activation buffer as long as the engine's budget only the product's rows are read before a timed run."""
    read = []

    class Buffer:
        device = "cpu"

        def __getitem__(self, rows):
            return SimpleNamespace(sum=lambda: read.append(rows))

        def sum(self):
            read.append(slice(None))

    monkeypatch.setattr(torch.cuda, "Event", lambda **_: SimpleNamespace(record=lambda: None, synchronize=lambda: None, elapsed_time=lambda _: 1.0))
    monkeypatch.setattr(blaslt, "flush_caches", lambda dev: None)
    assert blaslt._least_of_three(Buffer(), 64, lambda: None) == 1.0
    assert read == [slice(None, 64)] * 3


def test_what_was_chosen_names_the_tiles_that_run(choices, monkeypatch):
    """No library algorithm is named for a product that a tile runs, and products with their ends are listed."""
    import bench
    plan = _product()
    plan.tuned, plan.tile = True, blaslt._Tile(1)
    blaslt._plans[torch.device("cpu"), 2048, 512, 512, 512, 512, 512, torch.bfloat16, True, False] = blaslt._plans.pop("p")
    end = blaslt._ends[torch.device("cpu"), 2048, 1024, 512, 512, 512, 512, "gated"] = blaslt._End()
    end.tuned, end.tile = True, blaslt._Tile(2)
    assert bench.gemm_summary(blaslt.chosen()) == {"shapes": 2, "measured": 2, "algorithm_of": {
        "2048x512x512": "128x128", "2048x1024x512 gated": "256x256"}}


def test_the_warm_up_measures_on_rows_that_differ(choices, monkeypatch):
    """Rows that are all alike take the matrix cores less power, and the kernels that they bound seem faster than in any real step."""
    from dinfer_amd.engine import runner
    monkeypatch.setattr(blaslt, "available", lambda: True)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: None)
    steps = []
    made_up = SimpleNamespace(
        options=SimpleNamespace(gemm_tuning="measured", max_num_seqs=4, max_model_len=600), dtype=torch.bfloat16, group_specs=[None], max_tokens=1024,
        num_blocks=100, page_size=16, max_rows=4, device=None, model=SimpleNamespace(spec=SimpleNamespace(vocab_size=500)),
        reserve=lambda *a: True, finish=lambda rid: None, step=steps.append)
    monkeypatch.setattr(blaslt, "worth_measuring_met", 0)
    runner.ModelRunner.warm_up(made_up)
    tokens = [t for e in steps[0] for t in e.tokens]
    assert len(tokens) == 1024 and set(tokens) == set(range(500))
