"""Kemurax without a GPU: configuration, registry, checkpoint names, cache manager, rotation, weight layouts, and the oracle's own
sensitivity to every mechanism (a test that cannot see a fault proves nothing)."""
import copy
import ctypes
import json

import pytest
import torch

from oracle import ref_hybrid as R
from tests import hybrid_helpers as H
from triforce_amd.models import registry, zoo
from triforce_amd.models.cache import HybridCache
from triforce_amd.models.config_kemurax import KemuraxConfig
from triforce_amd.models.hybrid_core import AttentionGeom, HybridWeights, StateSpaceGeom
from triforce_amd.models.rotary import RotarySpec, RotaryTable, rotary_frequencies


# ---- configuration, registry, weights ---------------------------------------------------------------------------------------
@pytest.mark.parametrize("name", sorted(H.CONFIGS))
def test_config_round_trip(name):
    c = registry.config_from_dict(H.CONFIGS[name])
    assert isinstance(c, KemuraxConfig) and c.num_hidden_layers == len(H.CONFIGS[name]["layers"])
    assert KemuraxConfig.from_dict(c.to_dict()).to_dict() == c.to_dict()


@pytest.mark.parametrize("change, message", [
    (lambda d: d["layers"][0].update(type="other"), "mixer type"), (lambda d: d["layers"][0]["mlp"].update(kind="moe"), "feed-forward"),
    (lambda d: d["layers"][0]["mixer"]["left"].update(kv_heads=4), "kv_heads"), (lambda d: d["layers"][0]["mixer"]["left"]["rot"].update(dims=32), "dims"),
    (lambda d: d["layers"][0]["mixer"]["left"]["rot"]["scaling"].pop("low"), "low"), (lambda d: d["layers"][0]["mixer"]["left"]["mask"].update(size=0), "mask"),
    (lambda d: d["layers"][0]["mixer"]["right"].update(groups=3), "groups"), (lambda d: d["layers"][0]["mixer"]["right"].update(norm_groups=5), "norm_groups"),
    (lambda d: d["layers"][1]["mixer"].update(tau=0), "tau"), (lambda d: d.update(streams=0), "streams")])
def test_config_refuses_what_it_does_not_know(change, message):
    d = copy.deepcopy(H.CONFIGS["mixed"])
    change(d)
    with pytest.raises(ValueError, match=message):
        KemuraxConfig.from_dict(d)


def test_registry_and_command_line(tmp_path):
    from triforce_amd.models.modeling_llama import LlamaForCausalLM
    from triforce_amd.utils import cli
    (tmp_path / "config.json").write_text(json.dumps(H.CONFIGS["ones"]))
    arch = registry.architecture_of(str(tmp_path))
    assert registry.model_class(arch).__name__ == "KemuraxForCausalLM" and registry.libraries_of(arch) == ("tile", "hybrid")
    assert registry.libraries_of("Befidra") == ("tile", "latent") and registry.libraries_of("LlamaForCausalLM") == ("core",)
    assert type(zoo.config("kemurax-7B")).__name__ == type(zoo.config("kemurax-tiny")).__name__ == "KemuraxConfig"
    assert cli.parse("generate", ["--target", "kemurax-tiny"]).target == "kemurax-tiny"
    with pytest.raises(NotImplementedError, match="generate"):
        cli.load_causal_lm(LlamaForCausalLM, "random:1", "kemurax-tiny", "cpu")


def test_weights_name_missing_and_misshapen_tensors():
    d = H.CONFIGS["mixed"]
    sd = H.weights(d, 1)
    W = HybridWeights(KemuraxConfig.from_dict(d), "cpu", torch.float32)
    with pytest.raises(KeyError, match="l0.mix.left.g"):
        W.load_state_dict({k: v for k, v in sd.items() if k != "l0.mix.left.g"})
    with pytest.raises(KeyError, match="l2.hc2.mix"):
        W.load_state_dict({k: v for k, v in sd.items() if k != "l2.hc2.mix"})
    assert not any(k.startswith("l1.mlp") or k.startswith("l1.hc2") or k == "l1.norm2" for k in W.shapes())
    bad = dict(sd)
    bad["l0.mix.right.in"] = sd["l0.mix.right.in"][:-1]
    with pytest.raises(ValueError, match="l0.mix.right.in"):
        W.load_state_dict(bad)


def test_decay_rank_comes_from_the_tensors():
    d = copy.deepcopy(H.CONFIGS["mixed"])
    sd = H.weights(d, 1)
    for L in d["layers"]:
        L["mixer"].pop("rank", None)
    W = HybridWeights(KemuraxConfig.from_dict(d), "cpu", torch.float32).load_state_dict(sd)
    assert [L.mixer.geom.rank for L in W.layers if L.spec.mixer.type == "gla"] == [32, 64]


def test_input_projection_columns():
    """Every part sits where the geometry says, heads in their padded strides, zeros between."""
    d = H.CONFIGS["mixed"]
    sd = H.weights(d, 2)
    W = HybridWeights(KemuraxConfig.from_dict(d), "cpu", torch.float32).load_state_dict(sd)
    m, w = W.layers[0].mixer, W.layers[0].mixer.w_in.w
    a, s = m.left.geom, m.right.geom
    assert isinstance(a, AttentionGeom) and isinstance(s, StateSpaceGeom) and w.shape[0] == a.width + s.width
    assert torch.equal(w[a.q_off + 3 * a.D + 5, :88], sd["l0.mix.left.q"][3 * 24 + 5])
    assert torch.equal(w[a.v_off + a.V + 39, :88], sd["l0.mix.left.v"][40 + 39])
    assert bool((w[a.q_off + 24:a.q_off + 32] == 0).all()) and bool((w[:, 88:] == 0).all())
    p = sd["l0.mix.right.in"]                                        # z 96 | x 96 | B 40 | C 40 | dt 4
    assert torch.equal(w[s.gate_off + 2 * s.V + 7, :88], p[2 * 24 + 7])
    assert torch.equal(w[s.x_off + 3 * s.V + 1, :88], p[96 + 3 * 24 + 1])
    assert torch.equal(w[s.x_off + s.b_col + s.N + 2, :88], p[192 + 20 + 2])
    assert torch.equal(w[s.x_off + s.c_col + 19, :88], p[232 + 19]) and torch.equal(w[s.dt_off + 3, :88], p[272 + 3])
    c = sd["l0.mix.right.conv"]
    assert torch.equal(m.right.conv_w[:, 3 * s.V + 1], c[3 * 24 + 1]) and torch.equal(m.right.conv_w[:, s.c_col + s.N], c[136 + 20])
    assert m.cache_width() == 2 * (32 + 64) and m.state_shapes() == {"state": (4, 32, 32), "ring": (3, s.channels)}
    assert W.layers[1].mixer.cache_width() == 0 and W.layers[1].mixer.state_shapes() == {"state": (3, 32, 64)}


def test_interleaved_gate_and_up():
    from triforce_amd.ops_tile import interleave_glu
    gate, up = torch.arange(32.0).view(32, 1), 100 + torch.arange(32.0).view(32, 1)
    w = interleave_glu(gate, up).view(-1)
    assert w[:24].tolist() == list(range(8)) + list(range(100, 108)) + list(range(8, 16)) and w[56:].tolist() == list(range(124, 132))


@pytest.mark.parametrize("rot", [dict(dims=16, base=10000.0), dict(dims=32, base=500.0, scaling=dict(factor=4.0, original=64, low=1.0, high=4.0)),
                                 dict(dims=48, base=20.0, scaling=dict(factor=8.0, original=40, low=0.5, high=1.5)), dict(dims=2, base=100.0)])
def test_rotary_tables_against_the_oracle(rot):
    spec = RotarySpec(**rot, kind="bands")
    f, m = rotary_frequencies(spec)
    assert f == pytest.approx(R.frequencies(rot), rel=1e-14) and m == 1.0
    t, n = RotaryTable(spec, 700, "cpu"), rot["dims"]
    x = torch.randn(700, 1, n + 3)
    y = R.rotate(x.double(), torch.arange(700), rot)[:, 0]
    u, v = x[:, 0, :n // 2], x[:, 0, n // 2:n]
    assert torch.allclose(u * t.cos - v * t.sin, y[:, :n // 2].float(), atol=2e-6)
    assert torch.allclose(v * t.cos + u * t.sin, y[:, n // 2:n].float(), atol=2e-6)
    assert torch.equal(x[:, 0, n:].double(), y[:, n:])


def test_bands_keep_short_waves_and_stretch_long_ones():
    rot = dict(dims=64, base=10000.0, scaling=dict(factor=8.0, original=256, low=1.0, high=4.0))
    plain, f = R.frequencies(dict(rot, scaling=None)), R.frequencies(rot)
    turns = [256 * x / 6.283185307179586 for x in plain]
    assert all(a == b for a, b, t in zip(f, plain, turns) if t > 4) and all(a == b / 8 for a, b, t in zip(f, plain, turns) if t < 1)
    mid = [(a, b) for a, b, t in zip(f, plain, turns) if 1 < t < 4]
    assert mid and all(b / 8 < a < b for a, b in mid)


def test_bad_arguments_are_refused_before_any_launch():
    from triforce_amd import hip
    L = hip.hybrid_lib()
    assert L.tfh_recurrence(ctypes.byref(hip.TfhRecurrence()), 0, None) == -22
    assert L.tfh_step(None, None, 1, 8, 1, 1, 1e-5, 0, None) == -22
    assert L.tfh_step(ctypes.byref(hip.TfhAttnStep()), None, 1, 8, 1, 1, 1e-5, 0, None) == -22
    assert L.tfh_connect(None, None, 0, None, None, 0, 0, None, None, 1, 1, 1, 17, 1, 1, 32, 8, 1, 32, 32, 1e-5, 0, None) == -34   # streams
    assert L.tfh_glu(1, 1, 1, 12, 0, None) == -22
    for rows in (1, 3, 64):
        for heads, kv in ((1, 1), (32, 8), (34, 2)):
            for n in (1, 64, 5000, 131072):
                s = L.tfh_attn_step_pick_nsplit(rows, heads, kv, n)
                assert 1 <= s <= 256 and (s == 1 or s <= -(-n // 64))


# ---- cache manager ----------------------------------------------------------------------------------------------------------
class _Model:
    device, dtype = torch.device("cpu"), torch.float32

    def cache_widths(self):
        return [64, 0, 96]

    def state_shapes(self):
        return [{"state": (2, 32, 32), "ring": (3, 128)}, {"state": (1, 32, 64)}, {}]

    def prepare_positions(self, n):
        pass

    @staticmethod
    def segment_tokens(tokens):
        return 64


def test_step_splits_by_rows():
    """Splits per row of the decode step: one workgroup per CU for a row alone (two cost 5 to 12 %), two for more, above 16 splits in whole
    sixteens; more than 64 rows, which share nothing, take three (four cost 5 % at 128 rows of 1 000 keys)."""
    from triforce_amd import hip
    L = hip.hybrid_lib()
    pick = [L.tfh_attn_step_pick_nsplit(rows, 32, 8, 8256) for rows in (1, 2, 3, 4, 5, 8, 12, 16, 64, 65, 128, 1000)]
    assert pick == [32, 32, 16, 16, 12, 8, 5, 4, 4, 3, 3, 3]
    assert [L.tfh_attn_step_pick_nsplit(1, 16, g, 100000) for g in (1, 2, 4)] == [256, 128, 64]
    assert [L.tfh_attn_step_pick_nsplit(2, 32, 8, n) for n in (64, 65, 700)] == [1, 2, 11]


def test_step_splits_by_form():
    """The rule for heads of 128 in bfloat16 is theirs alone: others take their splits as they come, eight from 16 rows on, and from 32 on three
    where two workgroups or fewer fit a CU."""
    from triforce_amd import hip
    L = hip.hybrid_lib()
    for rows in (1, 2, 3, 16, 64, 65):
        for n in (1, 64, 5000, 131072):
            assert L.tfh_attn_step_splits(rows, 32, 8, 128, 128, n, 0) == L.tfh_attn_step_pick_nsplit(rows, 32, 8, n)
    rows = (1, 2, 3, 5, 8, 15, 16, 31, 32, 64, 65, 128)
    assert [L.tfh_attn_step_splits(r, 32, 8, 64, 64, 100000, 0) for r in rows] == [64, 32, 21, 12, 8, 4, 4, 4, 4, 4, 4, 4]
    for D, dtype in ((96, 0), (64, 1)):
        assert [L.tfh_attn_step_splits(r, 32, 8, D, D, 100000, dtype) for r in rows] == [64, 32, 21, 12, 8, 4, 8, 8, 4, 4, 4, 4]
    for D, dtype in ((256, 0), (160, 0), (128, 1), (96, 1)):
        assert [L.tfh_attn_step_splits(r, 32, 8, D, D, 100000, dtype) for r in rows] == [64, 32, 21, 12, 8, 4, 8, 8, 3, 3, 3, 3]
    assert [L.tfh_attn_step_splits(20, 32, 8, 96, 96, n, 0) for n in (1, 65, 449)] == [1, 2, 8]
    assert L.tfh_attn_step_splits(1 << 30, 1 << 15, 1 << 15, 96, 96, 100, 1) == 2


def test_cache_pages_and_seats():
    c = HybridCache(_Model(), max_budget=200, max_batch=3)
    assert [None if r is None else tuple(r.shape) for r in c.rows] == [(384, 64), None, (384, 96)]
    assert [tuple(s["state"].shape) for s in c.states[:2]] == [(3, 2, 32, 32), (3, 1, 32, 64)] and c.states[0]["ring"].shape == (3, 3, 128)
    c.extend([("a", 64), ("b", 1)])
    seats = dict(c.seat)
    assert sorted(seats.values()) == [0, 1]
    g = c.generation
    c.extend([("a", 1)])
    assert c.seat == seats and c.generation > g                  # (a page was handed out)
    c.release("a")
    c.extend([("c", 5), ("d", 5)])
    assert c.seat["b"] == seats["b"] and sorted(c.seat.values()) == [0, 1, 2] and seats["a"] in (c.seat["c"], c.seat["d"])
    with pytest.raises(IndexError):
        c.extend([("e", 1)])                                     # no seat
    lens, table, seat = c.tables(["d", "b"])
    assert lens.tolist() == [5, 1] and seat.tolist() == [c.seat["d"], c.seat["b"]] and table[0, 0] == c.pages["d"][0]
    c.reset()
    assert c.tokens == 0 and not c.seat and len(c.free_seats) == 3


def test_prefill_plan_segments_pasts_and_seats():
    c = HybridCache(_Model(), 400, 4)
    b = c.plan_prefill([("a", 130, [129]), ("b", 64, []), ("c", 1, [0])])
    assert b.seq.tolist() == [[0, 130, 0, c.seat["a"]], [130, 64, 0, c.seat["b"]], [194, 1, 0, c.seat["c"]]]
    assert b.seg.tolist() == [[0, 64, 0, 0], [64, 64, 0, 0], [128, 2, 0, 0], [130, 64, 1, 0], [194, 1, 2, 0]]
    assert b.span.tolist() == [[0, 3], [3, 1], [4, 1]] and b.max_segs == 3 and b.max_new == 130 and b.want.tolist() == [129, 194]
    b = c.plan_prefill([("c", 2, []), ("a", 5, [0])])
    assert b.pos.tolist() == [1, 2, 130, 131, 132, 133, 134] and [r[2] for r in b.seq.tolist()] == [1, 130] and b.max_segs == 1
    assert b.slot.tolist() == c.cache_rows("c", 1, 2).tolist() + c.cache_rows("a", 130, 5).tolist()
    assert b.table[1, :3].tolist() == c.pages["a"]


def test_segments_fill_the_chip_and_are_whole_chunks():
    from types import SimpleNamespace

    from triforce_amd.models.modeling_kemurax import KemuraxForCausalLM
    layer = lambda n: SimpleNamespace(mixer=SimpleNamespace(recurrence_units=lambda: n))
    model = SimpleNamespace(weights=SimpleNamespace(layers=[layer(64), layer(96)]))
    cut = lambda n: KemuraxForCausalLM.segment_tokens(model, n)
    assert [cut(n) for n in (1, 256, 2048, 4096, 4100)] == [256, 256, 256, 512, 576]
    assert all(cut(n) % 64 == 0 and (n < 4096 or -(-n // cut(n)) * 64 <= 512) for n in range(1, 20000, 331))


# ---- oracle -----------------------------------------------------------------------------------------------------------------
def _twist(cfg, sd, what):
    cfg, sd = copy.deepcopy(cfg), dict(sd)
    L0, L1 = cfg["layers"][0]["mixer"], cfg["layers"][1]["mixer"]

    def zero(n):
        sd[n] = torch.zeros_like(sd[n])
    if what == "chunk one longer":
        L0["left"]["mask"]["size"] += 1
    elif what == "no bands":
        L0["left"]["rot"]["scaling"] = None
    elif what == "rotation of all entries":
        L0["left"]["rot"]["dims"] = L0["left"]["dim"]
    elif what == "no output gate":
        zero("l0.mix.left.g")
    elif what == "key norm":
        sd["l0.mix.left.k.norm"] = torch.ones_like(sd["l0.mix.left.k.norm"])
    elif what == "key heads swapped":
        sd["l0.mix.left.k"] = sd["l0.mix.left.k"].roll(24, dims=0)
    elif what == "score scale":
        L0["left"]["scale"] *= 1.05
    elif what == "sides swapped":
        L0["left_scale"], L0["right_scale"] = L0["right_scale"], L0["left_scale"]
    elif what == "convolution one late":
        sd["l0.mix.right.conv"] = sd["l0.mix.right.conv"].roll(1, dims=1)
    elif what == "no convolution bias":
        zero("l0.mix.right.conv.b")
    elif what == "no step bias":
        zero("l0.mix.right.dt_bias")
    elif what == "decay of the next head":
        sd["l0.mix.right.A_log"] = sd["l0.mix.right.A_log"].roll(1)
    elif what == "no skip":
        zero("l0.mix.right.D")
    elif what == "norm parts":
        L0["right"]["norm_groups"] = 1
    elif what == "groups swapped":
        w = sd["l0.mix.right.in"].clone()
        w[192:232] = w[192:232].roll(20, dims=0)
        sd["l0.mix.right.in"] = w
    elif what == "tau":
        L1["tau"] *= 1.1
    elif what == "no decay bias":
        zero("l1.mix.a2.b")
    elif what == "no gate of the linear attention":
        zero("l1.mix.g")
    elif what == "mix transposed":
        sd["l2.hc1.mix"] = sd["l2.hc1.mix"].T.contiguous()
    elif what == "streams read in another order":
        sd["l2.hc2.in"] = sd["l2.hc2.in"].flip(0)
    elif what == "streams written in another order":
        sd["l3.hc1.out"] = sd["l3.hc1.out"].flip(0)
    elif what == "embedding norm":
        zero("embed.norm")
    elif what == "eps":
        cfg["norm"]["eps"] = 1e-5
    elif what == "no feed-forward":
        cfg["layers"][0]["mlp"] = None
    return cfg, sd


FAULTS = ["chunk one longer", "no bands", "rotation of all entries", "no output gate", "key norm", "key heads swapped", "score scale", "sides swapped",
          "convolution one late", "no convolution bias", "no step bias", "decay of the next head", "no skip", "norm parts", "groups swapped", "tau",
          "no decay bias", "no gate of the linear attention", "mix transposed", "streams read in another order",
          "streams written in another order", "embedding norm", "eps", "no feed-forward"]


@pytest.mark.parametrize("what", FAULTS)
def test_a_fault_in_a_mechanism_shows(what):
    """The fault is planted in the oracle; the bound is ten times what the fp32 device tests allow."""
    cfg = H.CONFIGS["mixed"]
    sd = H.weights(cfg, 5)
    toks = H.tokens_of(cfg, 60, 6)
    good = H.oracle_logits(cfg, sd, toks)
    bad = H.oracle_logits(*_twist(cfg, sd, what), toks)
    assert H.error(bad[40:], good[40:]) > 10 * H.F32


def test_chunks_count_from_the_sequence_start():
    cfg = H.CONFIGS["mixed"]["layers"][0]["mixer"]["left"]           # chunk 37
    g = torch.Generator().manual_seed(1)
    sd = {k[len("l0.mix.left."):]: v for k, v in H.weights(H.CONFIGS["mixed"], 3).items() if k.startswith("l0.mix.left.")}
    h = torch.randn(80, 88, generator=g)
    a = R.attention(h, sd, cfg, 1e-3)
    b = h.clone()
    b[:37] = torch.randn(37, 88, generator=g)
    assert torch.allclose(R.attention(b, sd, cfg, 1e-3)[37:], a[37:], atol=1e-6)         # the first chunk is out of sight from 37 on
    assert not torch.allclose(R.attention(b, sd, cfg, 1e-3)[36], a[36], atol=1e-3)
    assert torch.allclose(R.attention(h[37:], sd, cfg, 1e-3, positions=torch.arange(37, 80)), a[37:], atol=1e-6)


def test_recurrences_against_their_closed_forms():
    g = torch.Generator().manual_seed(2)
    r = lambda *s: torch.randn(*s, generator=g, dtype=torch.float64)
    T, Hn, N, V = 9, 2, 5, 4
    q, k, v, alpha = r(T, Hn, N), r(T, Hn, N), r(T, Hn, V), torch.sigmoid(r(T, Hn, N))
    o = R.channel_decay_recurrence(q, k, v, alpha)
    G = alpha.log().cumsum(0)
    want = torch.stack([sum(((q[t] * k[j] * (G[t] - G[j]).exp()).sum(-1, keepdim=True)) * v[j] for j in range(t + 1)) for t in range(T)])
    assert torch.allclose(o, want)
    dt, A, D = torch.rand(T, Hn, generator=g, dtype=torch.float64), r(Hn), r(Hn)
    y = R.scalar_decay_recurrence(v, k, q, dt, A, D)
    G = (-A.exp() * dt).cumsum(0)
    want = torch.stack([sum(((q[t] * k[j]).sum(-1) * (G[t] - G[j]).exp() * dt[j])[:, None] * v[j] for j in range(t + 1)) + D[:, None] * v[t]
                        for t in range(T)])
    assert torch.allclose(y, want)


def test_oracle_is_causal_and_remembers():
    cfg = H.CONFIGS["mixed"]
    sd = H.weights(cfg, 7)
    toks = H.tokens_of(cfg, 50, 8)
    a = H.oracle_logits(cfg, sd, toks)
    b = H.oracle_logits(cfg, sd, toks[:49] + [(toks[49] + 1) % cfg["vocab"]])
    assert torch.equal(a[:49], b[:49]) and not torch.equal(a[49], b[49])
    c = H.oracle_logits(cfg, sd, [(toks[0] + 1) % cfg["vocab"]] + toks[1:])
    assert H.error(c[40:], a[40:]) > 10 * H.F32                      # token 0 reaches past its chunk through the states
