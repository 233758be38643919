"""Decode steps of whole models at widths where neighbouring launches are one: what each hands to the next, against the oracle in 64 bits and against
the same model with the launches apart."""
import pytest
import torch

from oracle import ref_hybrid, ref_latent
from tests import hybrid_helpers as hh, latent_helpers as lh

pytestmark = pytest.mark.gpu

# every neighbour: mixer before feed-forward, feed-forward before mixer, mixer before mixer, a mixer and a feed-forward before the logits
MIX = hh.parallel(hh.left(8, 2, 128, 128, 1000, bands=(8.0, 64, 1.0, 4.0)), hh.right(32, 64, 128, groups=2, norm_groups=2), (0.5, 0.9))
GLA = hh.gla(8, 128, 256)
CONFIGS = {
    "streams": hh.config(4160, 4096, 4, [(MIX, 2560), (GLA, None), (MIX, None), (GLA, 2560)]),
    "streams_end": hh.config(4160, 4096, 3, [(GLA, 2560), (MIX, None)]),
    # a width whose readers make the row themselves, one of them after a mixer without a feed-forward
    "connect": hh.config(12320, 2048, 4, [(hh.parallel(hh.left(32, 8, 128, 128, 1000), hh.right(64, 64, 128, norm_groups=2)), None),
                                          (hh.parallel(hh.left(32, 8, 128, 128, 90), hh.right(64, 64, 128)), 6160)]),
    "finish": lh.config(12320, 4096, [(lh.mixer(32, 128, 64, 128, 512, 512), 8192)] * 2, loop=(0, 2, 2), side=256),
}

# what a mistake in the wiring would exchange
WRONG = {"streams": [("l0.hc1.out", "l0.hc2.out"), ("l0.hc2.mix", "l1.hc1.mix"), ("l0.hc2.in", "l1.hc1.in"), ("l0.norm1", "l0.norm2"), ("l2.norm1", "l3.norm1"),
                     ("l3.norm2", "final.norm")],
         "connect": [("l0.hc1.out", "l1.hc1.out"), ("l1.hc1.mix", "l1.hc2.mix"), ("l1.norm1", "l1.norm2")],
         "finish": [("l0.norm1", "l1.norm1"), ("l0.side.norm", "l1.side.norm"), ("l1.norm1", "final.norm")]}


@pytest.fixture(scope="module")
def made():
    """name -> (model, weights), one at a time."""
    kept = {}

    def get(name):
        if name not in kept:
            kept.clear()
            torch.cuda.empty_cache()
            cfg, H = CONFIGS[name], lh if name == "finish" else hh
            from triforce_amd.models import registry
            c = registry.config_from_dict(cfg)
            sd = H.weights(cfg, 5, sharp=1.0)
            kept[name] = registry.model_class(cfg["architecture"]).from_state_dict(c, sd), {k: v.cuda().double() for k, v in sd.items()}
        return kept[name]
    yield get
    kept.clear()


def _steps(model, prompts, then, graphs):
    from triforce_amd.utils.batch_infer import BatchInferenceEngine
    e = BatchInferenceEngine(model, model.make_cache(sum(map(len, prompts)) + 16 * len(prompts), max_batch=len(prompts)), use_graphs=graphs)
    names = list(range(len(prompts)))
    e.step([(s, p, []) for s, p in zip(names, prompts)])
    return torch.stack([e.decode(names, ids).clone() for ids in then], 1).float()                # [rows, steps, vocab]


@pytest.mark.parametrize("name, rows", [("streams", 1), ("streams", 2), ("streams", 3), ("streams", 20), ("streams_end", 2), ("connect", 1), ("connect", 2),
                                        ("finish", 1), ("finish", 2), ("finish", 3), ("finish", 20)])
def test_decode_steps(made, monkeypatch, name, rows):
    from triforce_amd import ops_hybrid as oh, ops_latent as ol
    model, sd = made(name)
    cfg, R = CONFIGS[name], ref_latent if name == "finish" else ref_hybrid
    prompts = [lh.tokens_of(cfg, 3 + 5 * s % 11, s + 1) for s in range(rows)]
    then = torch.tensor([lh.tokens_of(cfg, rows, 100 + t) for t in range(3)])
    calls = []
    for cls, method in ((oh.Streams, "result"), (oh.Scaled, "_product"), (oh.Connect, "_product"), (ol.Finish, "product")):
        monkeypatch.setattr(cls, method, lambda *a, _f=getattr(cls, method), _n=cls.__name__, **kw: (calls.append(_n), _f(*a, **kw))[1])
    got = _steps(model, prompts, then, False)
    runs = {"streams": ("Streams", "Scaled", 6), "streams_end": ("Streams", "Scaled", 3), "connect": ("Connect", "Connect", 3 if rows == 1 else 0),
            "finish": ("Finish", "Finish", 4 if rows <= 2 else 0)}[name]
    for n in set(runs[:2]):
        assert calls.count(n) == 3 * runs[2]
    assert torch.equal(got, _steps(model, prompts, then, True))
    monkeypatch.setattr(oh.Streams, "takes", staticmethod(lambda *a: False))
    monkeypatch.setattr(oh.Connect, "takes", staticmethod(lambda *a: False))
    monkeypatch.setattr(ol.Finish, "takes", staticmethod(lambda *a: False))
    monkeypatch.setattr(ol, "token_side_pays", lambda *a: False)
    apart = _steps(model, prompts, then, False)
    worst = 0.0
    with torch.device("cuda"):
        for s in sorted({0, rows // 2, rows - 1}):
            toks, n = torch.tensor(prompts[s] + then[:, s].tolist()), len(prompts[s])
            want = R.forward(cfg, sd, toks)[n:]
            # as in the helpers' bound: three times what rounding the operands of every product does to the oracle
            may = 3 * lh.error(R.forward(cfg, sd, toks, operand=lambda x: x.to(torch.bfloat16).double())[n:], want)
            assert lh.error(got[s], want) <= may and lh.error(apart[s], want) <= may, (s, may)
            worst = max(worst, may)
            for a, b in WRONG[name] if rows == 1 else ():         # each of these in the oracle is more than the tests let pass
                assert lh.error(R.forward(cfg, dict(sd, **{a: sd[b], b: sd[a]}), toks)[n:], want) > 2 * may, (a, b)
    assert lh.error(got.flatten(0, 1), apart.flatten(0, 1)) <= 2 * worst
