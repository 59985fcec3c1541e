"""Whole models whose recurrences have sizes that long portions take chunk by chunk (csrc/chunked.hip): long prompts cut in every
way against each other and the plain float64 implementations, and steps padded up to the counts of a captured graph, with
portions of fewer and of more rows than the chunked form begins at."""
import pytest
import torch

import test_gpu_fanulix as fanulix
import test_gpu_karopel as karopel

pytestmark = pytest.mark.gpu

# a delta rule of 64 x 32; a retention of 64 x 64 and a state space of 64 x 32 (heads of 128 beside them)
MODELS = [(karopel, "C3"), (fanulix, "F6")]


@pytest.fixture(scope="module")
def models(tmp_path_factory):
    import json

    from dinfer_amd.weights.safetensors_io import write_safetensors
    out = {}
    for mod, name in MODELS:
        cfg, page, seed = mod.CONFIGS[name]
        d = tmp_path_factory.mktemp(name)
        w = mod.plain.random_weights(cfg, seed)
        (d / "config.json").write_text(json.dumps(cfg))
        write_safetensors(d / "model.safetensors", {k: v.to(torch.bfloat16) for k, v in w.items()}, metadata={"format": "pt"})
        out[name] = (d, cfg, karopel.plain.as_float64(w) if mod is karopel else w, page)
    return out


def logits(mod, models, name, dtype, ids, parts):
    r = mod.make_runner(models, name, dtype)
    rows = mod.replay(r, [([("x", p, list(range(len(p))))], []) for p in parts])
    return torch.stack([rows[("x", i)] for i in range(len(ids))])


@pytest.mark.parametrize("mod,name", MODELS)
def test_long_prompts_cut_in_32bit(models, mod, name):
    """Portions of 128 rows and more take other sums than shorter ones, so the bits are not the same; the logits are to the last
    few, as they are for short prompts (2e-5 of the largest there, and of a state space beside it 5e-5)."""
    _, cfg, w, _ = models[name]
    ids = mod.tokens_for(cfg, 400, 8)
    want = logits(mod, models, name, "float32", ids, [[t] for t in ids])
    for sizes in ([400], [200], [128, 1, 271], [127], [64, 300]):
        got = logits(mod, models, name, "float32", ids, mod.cut(ids, sizes))
        err = (got - want).abs().max().item() / want.abs().max().item()
        assert err < (2e-5 if mod is karopel else 5e-5), f"portions of {sizes}: {err}"


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("mod,name", MODELS)
def test_padded_portion_steps(models, mod, name, dtype):
    """The same counts come up until their graph is captured and replayed: lone portions and portions beside others, each step
    padded or not as its counts ask, portions just under and above the rows that go chunk by chunk."""
    _, cfg, w, _ = models[name]
    r = mod.make_runner(models, name, dtype, graph=True)
    toks, steps, n = {}, [], 0
    for _ in range(4):
        for sizes in ([120, 3], [135, 1], [127, 2, 1], [100], [130], [128, 129]):
            es = []
            for k in sizes:
                n += 1
                rid = f"r{n}"
                toks[rid] = mod.tokens_for(cfg, k, n)
                es.append((rid, toks[rid], [k - 1]))
            steps.append((es, [e[0] for e in es]))
    rows = mod.replay(r, steps)
    assert r.portion_replays > 0
    mod.compare_rows(rows, cfg, w, toks, dtype, f"{name} padded steps")
