"""Latent layers whose sizes have the keys' side (128 + 64 a head, values of 128, a latent of 512) through the engine: the steps that take
it, against the plain float64 models and against the queries' side. A head gate and layers on another's cache (Kudurax), a query latent
and no gate (Verorax), a gate for every entry (Dumovik)."""
import json
import random

import pytest
import torch

import plain_dumovik
import plain_kudurax
import plain_verorax

pytestmark = pytest.mark.gpu


def mixer(heads, **more):
    return dict(type="latent_attention", mixer=dict(heads=heads, dim=128, rot_dim=64, vdim=128, kv_rank=512, scale=192 ** -0.5,
                                                    rot=dict(base=10000.0, dims=64), **more))


def dense(layer, ff=96):
    return dict(layer, mlp=dict(kind="dense", ff=ff))


CONFIGS = {
    "kudurax": dict(architecture="Kudurax", vocab=160, width=64, embedding=dict(scale=5.0), norm=dict(eps=1e-5), layers=[
        dense(mixer(3)), dense(mixer(2, kv_from=0)), dense(mixer(3))]),
    "verorax": dict(architecture="Verorax", vocab=160, width=64, norm=dict(eps=1e-6), layers=[dense(mixer(3, q_rank=40)), dense(mixer(2, q_rank=33))]),
    "dumovik": dict(architecture="Dumovik", vocab=160, width=64, norm=dict(eps=1e-5), layers=[dense(mixer(3)), dense(mixer(2))]),
}


def plain_logits(name, cfg, w, ids):
    if name == "kudurax":
        return plain_kudurax.forward(cfg, w, ids)
    plain = plain_verorax if name == "verorax" else plain_dumovik
    return plain.forward(ids, plain.as_float64(w), cfg)


@pytest.fixture(scope="module")
def models(tmp_path_factory):
    from dinfer_amd.weights.safetensors_io import write_safetensors
    out = {}
    for name, cfg in CONFIGS.items():
        d = tmp_path_factory.mktemp(name)
        w = {"kudurax": plain_kudurax, "verorax": plain_verorax, "dumovik": plain_dumovik}[name].random_weights(cfg, 7)
        (d / "config.json").write_text(json.dumps(cfg))
        write_safetensors(d / "model.safetensors", w, metadata={"format": "pt"})
        rng = random.Random(3)
        ids = {k: [rng.randrange(160) for _ in range(n)] for k, n in (("a", 340), ("b", 640), ("c", 330), ("d", 150))}
        out[name] = (d, cfg, ids, {k: plain_logits(name, cfg, w, x) for k, x in ids.items()})
    return out


@pytest.fixture
def launched(monkeypatch):
    """The keys' side's launches of the last step, call by call."""
    from dinfer_amd.kernels.latent import Expanded
    seen, inner = [], Expanded.attention

    def attention(self, launches, *a, **kw):
        seen.append(launches)
        return inner(self, launches, *a, **kw)
    monkeypatch.setattr(Expanded, "attention", attention)
    return seen


def make_runner(models, name, graph=False, rows=1024, page=16):
    from dinfer_amd.config import EngineOptions
    from dinfer_amd.engine.runner import ModelRunner
    opt = EngineOptions(dtype="bfloat16", max_model_len=1024, max_num_seqs=4, max_num_batched_tokens=1024, block_size=page,
                        num_blocks=2048 // page, max_logits_rows=rows, decode_exempt_from_budget=False, hip_graph=graph)
    return ModelRunner.from_dir(models[name][0], opt)


# (request, tokens) a step: from nothing, behind histories, single rows beside, requests that end and whose pages are taken again
STEPS = [[("a", 300)], [("a", 1), ("b", 400)], [("b", 200), ("a", 1), ("c", 290)], [("a", 1), ("b", 1), ("c", 1)], [("a", 30), ("c", 9)],
         [("d", 140), ("b", 3)], [("d", 5), ("b", 30)]]
TAKEN = [True, True, True, False, False, False, False]      # ([("d", 140), ("b", 3)]: fewer than 128 rows a request)


def run(r, launched, ids, steps, want_all=True):
    """{(request, position): logits} and per step whether the keys' side ran."""
    from dinfer_amd.engine.batch import Entry
    at, rows, taken = {}, {}, []
    for step in steps:
        entries = []
        for k, n in step:
            start = at.get(k, 0)
            assert r.reserve(k, start, n)
            entries.append(Entry(k, ids[k][start:start + n], start, list(range(n)) if want_all else [n - 1]))
            at[k] = start + n
        del launched[:]
        logits = r.step(entries).double().cpu()
        taken.append(len(launched))
        i = 0
        for e in entries:
            for x in e.want:
                rows[(e.req_id, e.start + x)] = logits[i]
                i += 1
            r.advance(e.req_id, at[e.req_id])
            if at[e.req_id] == len(ids[e.req_id]):
                r.finish(e.req_id)
        r.cache.check()
    for k in at:
        if r.cache.has(k):
            r.finish(k)
    return rows, taken


def error(rows, wants):
    got, want = (torch.stack([f(k) for k in rows]) for f in (lambda k: rows[k], lambda k: wants[k[0]][k[1]]))
    scale = want.std(dim=-1, keepdim=True)
    return ((got - want).abs() / scale).max().item(), ((got - want).pow(2).mean() / want.pow(2).mean()).sqrt().item()


@pytest.mark.parametrize("page", [16, 8])
@pytest.mark.parametrize("name", list(CONFIGS))
def test_steps_that_take_the_keys_side(models, launched, name, page):
    _, _, ids, want = models[name]
    r = make_runner(models, name, page=page)
    rows, taken = run(r, launched, ids, STEPS)
    layers = len(CONFIGS[name]["layers"])
    assert taken == [layers if t else 0 for t in TAKEN]
    for c, _ in r.model._choices:
        c.weigh = lambda starts, counts: None
    other, none = run(r, launched, ids, STEPS)
    assert not any(none) and other.keys() == rows.keys()
    (most, rms), (most_q, rms_q) = error(rows, want), error(other, want)
    # roundings to 8 bits add up to 0.01 or so of the logits; a wrong operand, head or gate is off by several tenths and more
    assert most < 0.2 and most_q < 0.2 and rms < 0.03 and rms < 1.2 * rms_q + 1e-3, (most, rms, most_q, rms_q)


@pytest.mark.parametrize("name", list(CONFIGS))
def test_requests_dealt_to_several_launches(models, launched, name):
    """Scratch that holds one long request or two short ones: the same bits."""
    _, _, ids, _ = models[name]
    steps = [[("a", 200), ("b", 300), ("c", 250)], [("c", 80), ("a", 140), ("b", 340)]]
    r = make_runner(models, name)
    once, _ = run(r, launched, ids, steps)
    assert all(len(l) == 1 for l in launched)
    for c, _ in r.model._choices:
        c.chunks = 45
    parts, taken = run(r, launched, ids, steps)
    assert all(taken) and [l[:2] for l in launched[0]] == [(0, 2), (2, 1)]
    assert all(torch.equal(once[k], parts[k]) for k in once)


@pytest.mark.parametrize("name", list(CONFIGS))
def test_long_steps_between_replays(models, launched, name):
    """Steps of the same counts replay a captured graph; those that gain by their lengths are launched one by one between the replays, at
    other lengths each time, and the replays after them are as exact as before."""
    _, _, ids, want = models[name]
    r = make_runner(models, name, graph=True, rows=4)
    r.model._weights = 10 ** 9         # (as if the layers' weights kept the device busy: so small a model is never worth launching)
    steps = []
    for long_one in (300, 400, 520):
        steps += [[("b", long_one)], [("b", 20), ("c", 12)], [("c", 12), ("b", 20)], [("b", 1), ("c", 1)], [("b", 20), ("c", 12)]]
    replays = []
    for i in range(3):
        rows, taken = run(r, launched, ids, steps[5 * i:5 * i + 5], want_all=False)
        assert [t > 0 for t in taken] == [True, False, False, False, False]
        most, rms = error(rows, want)
        assert most < 0.2 and rms < 0.03, (i, most, rms)
        replays.append(r.portion_replays)
    assert replays[0] < replays[1] < replays[2]


def test_a_small_models_prompts_stay_in_the_graphs(models, launched):
    _, _, ids, want = models["kudurax"]
    r = make_runner(models, "kudurax", graph=True, rows=4)
    for _ in range(4):
        rows, taken = run(r, launched, ids, [[("a", 130)], [("a", 128)]], want_all=False)
        most, rms = error(rows, want)
        assert most < 0.2 and rms < 0.03 and not any(taken)
    assert r.portion_replays >= 2
