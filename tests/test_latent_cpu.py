"""Befidra without a GPU: configuration, registry, checkpoint names, cache manager, command lines, and the oracle's own
sensitivity to every mechanism (a test that cannot see a fault proves nothing)."""
import copy
import ctypes
import json
import math
import os
import re

import pytest
import torch

from oracle import ref_latent as R
from tests import latent_helpers as H
from triforce_amd.models import registry, zoo
from triforce_amd.models.cache import LatentCache
from triforce_amd.models.config_befidra import BefidraConfig
from triforce_amd.models.latent_core import LatentWeights
from triforce_amd.models.rotary import RotaryTable, rotary_frequencies

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


# ---- library --------------------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("header, prefix, signatures, lib", [("triforce_tile.h", "tfl_", "TILE_SIGNATURES", "tile_lib"),
                                                             ("triforce_latent.h", "tfl_", "LATENT_SIGNATURES", "latent_lib"),
                                                             ("triforce_hybrid.h", "tfh_", "HYBRID_SIGNATURES", "hybrid_lib")])
def test_libraries_export_what_their_headers_declare(header, prefix, signatures, lib):
    from triforce_amd import hip
    src = re.sub(r"/\*.*?\*/", "", open(os.path.join(ROOT, "include", header)).read(), flags=re.S)
    names = set(re.findall(r"\b(%s[a-z0-9_]+)\s*\(" % prefix, src))
    assert names == set(getattr(hip, signatures))
    loaded = getattr(hip, lib)()
    assert all(hasattr(loaded, n) for n in names)


@pytest.mark.parametrize("header, name", [("triforce_tile.h", "TflGemm"), ("triforce_hybrid.h", "TfhRecurrence"),
                                          ("triforce_hybrid.h", "TfhAttnStep"), ("triforce_hybrid.h", "TfhRecStep")])
def test_structures_match_the_headers(header, name):
    from triforce_amd import hip
    src = open(os.path.join(ROOT, "include", header)).read()
    body = re.sub(r"/\*.*?\*/", "", re.search(r"typedef struct %s \{(.*?)\} %s;" % (name, name), src, re.S).group(1), flags=re.S)
    kinds = {"float": ctypes.c_float, "int64_t": ctypes.c_int64, "int32_t": ctypes.c_int}
    fields = []
    for decl in body.split(";"):
        m = re.match(r"^(?:const )?(void|float|int64_t|int32_t)\s*(.*)$", decl.strip(), re.S)
        if m:
            fields += [(f.strip().lstrip("* ").strip(), ctypes.c_void_p if "*" in f else kinds[m.group(1)]) for f in m.group(2).split(",")]
    assert fields == getattr(hip, name)._fields_


def test_bad_arguments_are_refused_before_any_launch():
    from triforce_amd import hip
    L, T = hip.latent_lib(), hip.tile_lib()
    a = hip.TflGemm()
    assert T.tfl_gemm(ctypes.byref(a), 0, 0, None) == -22
    a.wp = a.x = a.out_f = 1 << 20
    a.rows, a.n, a.k, a.groups, a.n_real, a.ld_f, a.ld_x = 1, 16, 32, 1, 16, 16, 32
    a.k = 40
    assert T.tfl_gemm(ctypes.byref(a), 0, 0, None) == -22
    assert L.tfl_attn_decode(1, 1, 1, 1, 1, 1, 1, None, 0, 1, 1, 48, 32, 1.0, 1, 0, None) == -22        # latent not padded
    assert L.tfl_attn_decode(1, 1, 1, 1, 1, 1, 1, None, 0, 1, 1, 64, 32, 1.0, 4, 0, None) == -28        # no workspace
    def beside(rows=1, heads=20, splits=8, workers=16, panels=2, ws=1 << 30, **kw):
        for key, v in dict(dict(rows=rows, n=4096, k=2048, groups=1, chunk_major=1, ld_x=8, x_oct=8, ld_f=4096, out_t=None), **kw).items():
            setattr(a, key, v)
        a.wp = a.x = a.out_f = 1 << 20
        return L.tfl_attn_decode_beside(1, 1, 1, 1, 1, 1, 1, 1, ws, rows, heads, 1.0, splits, workers, panels, ctypes.byref(a), None)
    assert beside(ws=20 * 8 * 514 - 1) == -28
    for bad in (dict(rows=33, workers=200), dict(rows=0), dict(heads=16), dict(heads=33), dict(splits=1), dict(splits=129), dict(workers=1),
                dict(workers=256), dict(panels=1), dict(panels=5), dict(n=4100), dict(k=2056), dict(groups=2), dict(chunk_major=0), dict(ld_x=12),
                dict(x_oct=4), dict(ld_f=4092), dict(out_t=1 << 20)):
        assert beside(**bad) == -22, bad
    def value(splits=8, ws=1 << 30, **kw):
        for key, v in dict(dict(rows=1, n=128, k=512, groups=20, chunk_major=0, ld_t=8, t_oct=8, ld_gate=2560), **kw).items():
            setattr(a, key, v)
        a.wp = a.gate = a.out_t = 1 << 20
        return L.tfl_latent_value(1, ws, splits, ctypes.byref(a), None)
    assert value(ws=20 * 8 * 514 - 1) == -28
    for bad in (dict(rows=5), dict(rows=0), dict(splits=1), dict(splits=129), dict(k=480), dict(n=24), dict(groups=0), dict(chunk_major=1), dict(ld_t=4),
                dict(t_oct=4), dict(ld_gate=2558), dict(ld_gate=2552)):
        assert value(**bad) == -22, bad
    for rows in (1, 3, 64):
        for heads in (1, 16, 33, 128):
            for n in (1, 64, 5000, 131072):
                s = L.tfl_attn_decode_pick_nsplit(rows, heads, n)
                assert 1 <= s <= 256 and (s == 1 or s <= math.ceil(n / 128))


def test_rows_inside_a_product_are_read_in_pieces_of_16_bytes():
    """The entries that make a product's rows, streams or scales refuse an address that is not one of theirs before any launch."""
    from triforce_amd import hip
    L, Y = hip.latent_lib(), hip.hybrid_lib()
    at = 1 << 20

    def gemm(**kw):
        a = hip.TflGemm()
        for key, v in dict(dict(wp=at, x=at, rows=1, n=16384, k=4096, groups=1, chunk_major=1, ld_x=8, x_oct=8, ld_f=16384, n_real=16384, ld_t=8, t_oct=8, out_f=at,
                                out_t=at, out_t2=at, norm_w=at, ss_out=at, ss_in=at, ss_n=256, ss_ld=1024, k_real=4096, n_raw=2048, n_scaled=512), **kw).items():
            setattr(a, key, v)
        return ctypes.byref(a)

    def rows(cls, **kw):
        f = cls()
        for name, kind in cls._fields_:
            setattr(f, name, dict(ld_y=4096, width=4096, width_real=4096, streams=4, eps=1e-5, x_out=2 * at).get(name, at))
        for key, v in kw.items():
            setattr(f, key, v)
        return ctypes.byref(f)
    epi = hip.TFL_EPI
    for off in (4, 8):
        for key in ("y", "y_w", "step", "norm_w", "x", "x_out"):
            assert L.tfl_finish_gemm(rows(hip.TflFinish, **{key: at + off}), gemm(), epi["f32"], None) == -22, key
        for key in ("out_f", "out_t", "out_t2", "norm_w", "wp"):
            assert L.tfl_finish_gemm(rows(hip.TflFinish), gemm(**{key: at + off}), epi["in"], None) == -22, key
        for key in ("y", "norm_w", "x", "x_out"):
            assert Y.tfh_connect_gemm(rows(hip.TfhConnect, **{key: at + off}), gemm(), epi["glu"], None) == -22, key
        assert Y.tfh_connect_gemm(rows(hip.TfhConnect), gemm(out_t=at + off), epi["glu"], None) == -22
        for key in ("norm_w", "x", "x_out"):
            assert Y.tfh_streams_gemm(rows(hip.TfhConnect, **{key: at + off}), gemm(n=4096), None) == -22, key
        for key in ("wp", "x", "out_t"):
            assert Y.tfh_streams_gemm(rows(hip.TfhConnect), gemm(n=4096, **{key: at + off}), None) == -22, key
        for key in ("wp", "x", "ss_in", "out_t"):
            assert Y.tfh_scaled_gemm(gemm(**{key: at + off}), epi["glu"], None) == -22, key
        for places in (1, 2, 5, 10):
            args = [at, at, at, 8, 8, at, 256, at, 100, at, 4096, at, 1 << 30, 1, 4096, 256, 256, 4096, None]
            args[{1: 0, 2: 1, 5: 2, 10: 11}[places]] += off
            assert L.tfl_token_side(*args) == -22, places


def test_large_sides_stay_panels():
    """Where it was measured the slower way, and more than the kernel takes: any side of a model's configuration is one."""
    from triforce_amd import ops_latent as ol
    for rows, width, side, want in ((1, 4096, 256, True), (10, 4096, 256, True), (11, 4096, 256, False), (1, 4096, 512, False), (1, 8192, 512, False), (10, 8192, 256, True),
                                    (4, 6144, 256, True), (8, 6144, 256, False), (1, 2048, 256, False), (10, 2048, 128, True), (4, 1024, 128, True), (8, 1024, 128, False),
                                    (10, 1024, 64, True), (1, 2048, 1024, False), (1, 2048, 4128, False)):
        assert ol.token_side_pays(rows, width, side) == want, (rows, width, side)


def test_decode_splits_by_form():
    """Two pages: one split where the merge costs more than the second page; float32 (one workgroup of 16 heads per CU): single pages only
    where they are no more rounds of 256 workgroups than pairs."""
    from triforce_amd import hip
    _, L = hip.tile_lib(), hip.latent_lib()
    splits = L.tfl_attn_decode_splits
    for rows in (1, 7, 64, 128):
        for heads in (1, 16, 33, 128):
            assert [splits(rows, heads, 512, 64, n, 0) for n in (1, 64, 65, 128)] == [1, 1, 1, 1]
            for n in (129, 1024, 1025, 40000):
                assert splits(rows, heads, 512, 64, n, 0) == L.tfl_attn_decode_pick_nsplit(rows, heads, n) == max(1, min(
                    256 // (rows * (-(-heads // 32))), -(-n // 64) if n <= 1024 else -(-n // 128), 256))
    assert [splits(rows, 16, 256, 32, 128, 0) for rows in (1, 64, 65, 128)] == [2, 2, 1, 1]
    assert [splits(rows, 32, 256, 32, 128, 0) for rows in (1, 32, 33)] == [2, 2, 1]
    assert [splits(rows, 16, 512, 64, 128, 1) for rows in (1, 128, 129)] == [2, 2, 1]
    assert [splits(rows, 32, 512, 64, 768, 1) for rows in (10, 11, 12, 21, 22)] == [12, 6, 6, 6, 11]
    assert splits(0, 16, 512, 64, 128, 0) == splits(1, 0, 512, 64, 128, 0) == splits(1, 16, 512, 64, 0, 0) == 1
    assert splits(1 << 30, 1 << 20, 512, 64, 1 << 30, 1) == 1


def test_plan_of_attention_beside_a_product():
    """Whatever the sizes: a plan's groups of panels and its workers share 256 CUs, two workers a row at least, splits the kernel takes."""
    from triforce_amd import ops_latent as ol
    seen = set()
    for rows in (0, 1, 5, 8, 17, 32, 33):
        for heads in (16, 17, 20, 32, 33):
            for pages in (0, 1, 31, 64, 500, 1500, 2016, 100000, 1 << 21):
                for n, k in ((4096, 11008), (4096, 2016), (4080, 11008), (8192, 8192), (8208, 8192), (6160, 2080)):
                    plan = ol.beside_plan(rows, heads, 512, 64, pages, n, k)
                    if plan is None:
                        continue
                    workers, each, splits, later = plan
                    assert not later or rows <= 4
                    assert 1 <= rows <= 32 and 16 < heads <= 32 and 256 <= n // 16 <= 512 and k >= 2048 and 2 <= each <= 4
                    assert workers >= 2 * rows and workers + -(-n // 16 // each) <= 256 and 2 <= splits <= 128
                    seen.add((each, n))
    assert {(2, 4096), (3, 4096), (4, 4096), (4, 8192)} <= seen
    assert ol.beside_plan(1, 20, 512, 32, 64, 4096, 11008) is None and ol.beside_plan(1, 20, 256, 64, 64, 4096, 11008) is None


# rows, pages in all -> panels each: the division that was the fastest, mostly by 3 % or more (32 heads, 4 096 x 11 008; rows half to all as long as the longest)
@pytest.mark.parametrize("rows,pages,each", [(1, 4, 2), (1, 64, 2), (1, 192, 2), (2, 114, 2), (4, 204, 2), (8, 54, 2), (8, 258, 2), (12, 438, 2), (16, 592, 2),
                                             (24, 596, 2), (24, 1192, 2), (32, 32, 2), (32, 784, 2), (32, 1184, 2), (12, 870, 2), (24, 1788, 3)])
def test_plan_picks_what_was_measured_fastest(rows, pages, each):
    from triforce_amd import ops_latent as ol
    assert ol.beside_plan(rows, 32, 512, 64, pages, 4096, 11008)[1] == each


# the same with the longest row known, others as long, half or an eighth as long; apart (0) where the product's part of the CUs is far the longer side
@pytest.mark.parametrize("rows,pages,longest,n,k,each", [
    (20, 1449, 96, 4096, 11008, 2), (14, 980, 70, 4096, 11008, 2), (26, 1040, 40, 4096, 11008, 2), (32, 503, 100, 4096, 11008, 2), (12, 1733, 192, 4096, 11008, 3),
    (8, 1539, 256, 4096, 11008, 3), (32, 2319, 96, 4096, 11008, 3), (28, 4044, 192, 4096, 11008, 4), (8, 2306, 512, 4096, 11008, 4),
    (26, 1250, 300, 4096, 11008, 4), (32, 1478, 300, 4096, 11008, 4), (24, 155, 8, 8192, 16384, 0), (24, 155, 8, 4096, 16384, 0), (24, 1163, 64, 4096, 16384, 2)])
def test_plan_for_a_known_longest_row(rows, pages, longest, n, k, each):
    from triforce_amd import ops_latent as ol
    plan = ol.beside_plan(rows, 32, 512, 64, pages, n, k, longest)
    assert plan is None if each == 0 else plan[1] == each


def test_carried_columns():
    """What query to latent carries of that product: one amount for its k that leaves a product the attention runs beside, or none, and as picked where it was
    measured."""
    from triforce_amd import ops_latent as ol
    for rows in (0, 1, 2, 7, 16, 17, 32):
        for heads in (16, 17, 32, 33):
            for pages in (0, 1, 64, 500, 2016, 1 << 21):
                for n, k in ((4096, 11008), (4096, 5120), (4096, 6144), (4096, 14336), (8192, 8192), (6160, 8224)):
                    for longest in (None, max(1, pages // 2)):
                        c = ol.carry_plan(rows, heads, 512, 64, pages, n, k, longest)
                        assert c in (0, 4096 if k < 7168 else 5120)
                        if c:
                            assert 1 <= rows <= 16 and 16 < heads <= 32 and pages >= 1 and ol.beside_plan(rows, heads, 512, 64, pages, n, k - c, longest)
    assert ol.carry_plan(1, 32, 256, 64, 64, 4096, 11008) == ol.carry_plan(1, 32, 512, 32, 64, 4096, 11008) == 0
    pick = [ol.carry_plan(rows, 32, 512, 64, pages, 4096, 11008, longest) for rows, pages, longest in
            ((1, 63, 63), (2, 112, 63), (4, 204, 63), (8, 396, 63), (16, 810, 63), (1, 7, 7), (16, 90, 7), (2, 560, 313), (8, 1950, 313))]
    assert pick == [5120, 5120, 5120, 5120, 0, 5120, 5120, 0, 0]


def test_plan_of_a_product_cut_over_k():
    """Whatever the sizes: panels in eights over 4 ranges, 3 where n is wide, and the workers share 256 CUs, two workers a row at least; picked where it was measured
    the faster way."""
    from triforce_amd import ops_latent as ol
    for rows in (1, 16, 17, 25, 32, 33):
        for heads in (16, 17, 32, 33):
            for pages in (0, 1, 40, 500, 2016, 100000, 1 << 21):
                for n, k in ((4096, 11008), (4096, 4064), (4080, 11008), (8192, 8192), (8208, 8192), (6160, 4128), (4096, 14368)):
                    for longest in (None, max(1, pages // 3)):
                        plan = ol.parts_plan(rows, heads, 512, 64, pages, n, k, longest)
                        if plan is None:
                            continue
                        workers, parts, splits = plan
                        assert 17 <= rows <= 32 and 16 < heads <= 32 and 4096 <= n <= 8192 and 4096 <= k <= 14336 and parts == (4 if n <= 6144 else 3)
                        assert workers >= 2 * rows and workers + parts * -(-n // 128) == 256 and 2 <= splits <= 128
    assert ol.parts_plan(20, 32, 256, 64, 64, 4096, 11008) is None and ol.parts_plan(20, 32, 512, 32, 64, 4096, 11008) is None
    pick = [(ol.parts_plan(rows, 32, 512, 64, pages, 4096, 11008, longest) or (0, 0))[1] for rows, pages, longest in
            ((17, 70, 5), (17, 629, 47), (20, 1457, 94), (24, 596, 32), (32, 130, 5), (32, 784, 32), (32, 1546, 63), (32, 2312, 94))]
    assert pick == [4, 4, 0, 4, 4, 4, 0, 0]


@pytest.mark.parametrize("heads, n, k", [(32, 4096, 11008), (20, 4096, 11008), (17, 4096, 6144), (20, 4096, 14336), (24, 6144, 8192), (32, 5120, 13824),
                                         (32, 8192, 8192), (32, 4096, 4096)])
def test_a_growing_answer_asks_for_few_forms(heads, n, k):
    """Every form of a decode step is a graph of its own, captured in the middle of an answer: what the product beside the attention shares with its neighbours adds one
    form at most to those of its place on the chip alone, whatever the rows."""
    from triforce_amd import ops_latent as ol
    from triforce_amd.models.latent_core import LatentLayer
    layer = object.__new__(LatentLayer)
    layer.geom, layer.ff = type("Geometry", (), dict(H=heads, C=512, R=64, V=128)), k
    layer.w_out = type("Weight", (), dict(chunk_major=True, dtype=torch.bfloat16, n=n, k=k + heads * 128))
    for rows in (1, 2, 3, 4, 6, 8, 12, 16, 17, 20, 21, 24, 28, 32):
        pages = range(1, min(32768, 200000 // rows) // 64 + 1)
        plain = {ol.beside_plan(rows, heads, 512, 64, rows * c, n, k, c) for c in pages}
        forms = {layer.beside(rows, rows * c, c) for c in pages}
        assert len(forms) <= min(5, len(plain) + 1), (rows, forms)


def test_a_step_says_how_long_its_longest_sequence_is():
    """With the token that it adds: a page's last and its first."""
    from triforce_amd.utils.batch_infer import _DecodeStep
    asked = []

    class Model:
        def decode_form(self, rows, pages, longest):
            asked.append((rows, pages, longest))
            raise StopIteration

    class Known:
        page, length = 64, {"a": 63, "b": 64, "c": 200}
    step = object.__new__(_DecodeStep)
    step.model, step.cache, step.use_graph, step.graphs = Model(), Known(), True, {}
    step.form = step.model.decode_form
    step.buf = type("Buffers", (), dict(B=2, batch=type("Batch", (), {})()))()
    for seqs in (["a", "b"], ["a", "a"], ["c", "new"]):
        with pytest.raises(StopIteration):
            step(seqs, None)
    assert asked == [(2, 3, 2), (2, 2, 1), (2, 5, 4)]


# ---- configuration and registry -------------------------------------------------------------------------------------------
@pytest.mark.parametrize("name", sorted(H.CONFIGS))
def test_config_round_trip_and_layer_order(name):
    d = H.CONFIGS[name]
    c = registry.config_from_dict(d)
    assert isinstance(c, BefidraConfig)
    assert BefidraConfig.from_dict(c.to_dict()).to_dict() == c.to_dict()
    assert [(i, t or 0, f) for i, t, f in c.layer_runs()] == R.layer_runs(d)


def test_layer_runs_of_a_loop():
    c = registry.config_from_dict(H.CONFIGS["mixed"])
    assert [(i, t, f) for i, t, f in c.layer_runs()] == \
        [(0, None, False), (1, 0, True), (2, 0, False), (1, 1, True), (2, 1, False), (1, 2, True), (2, 2, False)]


@pytest.mark.parametrize("change, message", [
    (lambda d: d["layers"][0].update(type="other"), "mixer type"), (lambda d: d["layers"][0]["mlp"].update(kind="gated"), "feed-forward"),
    (lambda d: d.update(loop=dict(start=1, stop=9, times=1)), "loop"), (lambda d: d["layers"][0]["mixer"]["rot"].update(dims=3), "even"),
    (lambda d: d["layers"][0]["mixer"]["rot"]["scaling"].pop("fast"), "fast"), (lambda d: d["layers"][0]["mixer"].update(heads=0), "heads")])
def test_config_refuses_what_it_does_not_know(change, message):
    d = copy.deepcopy(H.CONFIGS["mixed"])
    change(d)
    with pytest.raises(ValueError, match=message):
        BefidraConfig.from_dict(d)


def test_registry_chooses_by_config(tmp_path):
    assert registry.architecture_of({"architectures": ["LlamaForCausalLM"]}) == "LlamaForCausalLM"
    assert registry.architecture_of({}) == "LlamaForCausalLM"
    with pytest.raises(NotImplementedError):
        registry.architecture_of({"architecture": "Nobody"})
    (tmp_path / "config.json").write_text(json.dumps(H.CONFIGS["plain"]))
    assert registry.model_class(registry.architecture_of(str(tmp_path))).__name__ == "BefidraForCausalLM"
    assert type(zoo.config("befidra-7B")).__name__ == "BefidraConfig" and type(zoo.config("llama-68M")).__name__ == "LlamaConfig"


def test_speculative_scripts_refuse_and_generate_parses():
    from triforce_amd.models.modeling_llama import LlamaForCausalLM
    from triforce_amd.utils import cli
    with pytest.raises(NotImplementedError, match="generate"):
        cli.load_causal_lm(LlamaForCausalLM, "random:1", "befidra-tiny", "cpu")
    a = cli.parse("generate", ["--greedy", "--batch", "3"])
    assert (a.temp, a.top_p, a.batch, a.target) == (1.0, 1e-9, 3, "befidra-tiny")


def test_weights_name_missing_and_misshapen_tensors():
    d = H.CONFIGS["plain"]
    sd = H.weights(d, 1)
    W = LatentWeights(BefidraConfig.from_dict(d), "cpu", torch.float32)
    with pytest.raises(KeyError, match="l0.mix.g"):
        W.load_state_dict({k: v for k, v in sd.items() if k != "l0.mix.g"})
    sd["l1.mix.uv"] = sd["l1.mix.uv"][:-1]
    with pytest.raises(ValueError, match="l1.mix.uv"):
        W.load_state_dict(sd)


def test_packed_tiles_hold_the_matrix():
    from triforce_amd.ops_latent import pack_tiles
    w = torch.arange(48 * 64).float().view(48, 64)
    p = pack_tiles(w)
    for n, k in ((0, 0), (17, 33), (47, 63), (30, 8)):
        assert p[n // 16, k // 32, (k % 32) // 8, n % 16, k % 8] == w[n, k]


@pytest.mark.parametrize("rot", [dict(dims=16, base=10000.0), dict(dims=16, base=500.0, scaling=dict(factor=4.0, original=64, fast=8.0, slow=1.0)),
                                 dict(dims=2, base=100.0, scaling=dict(factor=2.0, original=32, fast=1.0, slow=1.0))])
def test_rotary_tables_against_the_oracle(rot):
    from triforce_amd.models.config_befidra import RotarySpec
    spec = RotarySpec(**rot)
    f, m = rotary_frequencies(spec)
    fo, mo = R.frequencies(rot)
    assert f == pytest.approx(fo, rel=1e-14) and m == pytest.approx(mo)
    t = RotaryTable(spec, 700, "cpu")
    x = torch.randn(700, rot["dims"])
    y = R.rotate(x.double(), torch.arange(700), rot)
    u, v = x[:, 0::2], x[:, 1::2]
    assert torch.allclose(u * t.cos - v * t.sin, y[:, 0::2].float(), atol=1e-6)
    assert torch.allclose(v * t.cos + u * t.sin, y[:, 1::2].float(), atol=1e-6)


# ---- cache manager --------------------------------------------------------------------------------------------------------
class _Model:
    device, dtype = torch.device("cpu"), torch.float32
    asked = 0

    def cache_widths(self):
        return [64, 96, 64]

    def prepare_positions(self, n):
        self.asked = n


def test_cache_pages_grow_are_freed_and_used_again():
    m = _Model()
    c = LatentCache(m, max_budget=200, max_batch=3)
    assert m.asked == 200 and c.n_pages == 4 + 2 and [r.shape for r in c.rows] == [(384, 64), (384, 96), (384, 64)]
    c.extend([("a", 64), ("b", 1)])
    assert len(c.pages["a"]) == 1 and len(c.pages["b"]) == 1
    c.extend([("a", 1)])
    assert len(c.pages["a"]) == 2
    rows = c.cache_rows("a", 0, 65).tolist()
    assert rows[:64] == [c.pages["a"][0] * 64 + j for j in range(64)] and rows[64] == c.pages["a"][1] * 64
    assert c.cache_rows("a", 63, 2).tolist() == rows[63:65]
    gone = set(c.pages["a"])
    c.release("a")
    c.extend([("c", 100)])
    assert set(c.pages["c"]) == gone and c.tokens == 101
    with pytest.raises(IndexError):
        c.extend([("b", 100)])                                   # 201 tokens
    assert c.tokens == 101 and c.length["b"] == 1, "a refused step changes nothing"
    c.extend([("b", 1), ("d", 98)])                              # the whole budget, three part-filled pages
    with pytest.raises(IndexError):
        LatentCache(_Model(), 200, 1).extend([("a", 1), ("b", 1)])
    c.reset()
    assert c.tokens == 0 and len(c.free) == c.n_pages


def test_cache_never_runs_out_of_pages_inside_its_budget():
    g = torch.Generator().manual_seed(3)
    for budget, batch in ((1, 1), (64, 64), (65, 5), (500, 70), (1000, 130)):
        c = LatentCache(_Model(), budget, batch)
        for _ in range(300):
            if c.length and torch.rand(1, generator=g) < 0.1:
                c.release(sorted(c.length)[int(torch.randint(len(c.length), (1,), generator=g))])
            left = budget - c.tokens
            if left == 0:
                c.release(sorted(c.length)[0])
                continue
            n = min(left, int(torch.randint(1, 3 if batch > 50 else 70, (1,), generator=g)))
            name = int(torch.randint(batch, (1,), generator=g))
            c.extend([(name, n)])
        owned = [p for ps in c.pages.values() for p in ps] + c.free
        assert sorted(owned) == list(range(c.n_pages))


def test_prefill_plan_positions_slots_and_keys():
    c = LatentCache(_Model(), 400, 4)
    b = c.plan_prefill([("a", 70, [69]), ("b", 3, range(3))])
    assert not b.decode and b.key_rows is None and b.max_new == 70
    assert b.pos.tolist() == list(range(70)) + [0, 1, 2] and b.seq.tolist() == [[0, 70, 0, 70], [70, 3, 70, 3]]
    assert b.want.tolist() == [69, 70, 71, 72]
    b = c.plan_prefill([("b", 2, []), ("a", 5, [0])])
    assert b.pos.tolist() == [3, 4, 70, 71, 72, 73, 74] and b.seq.tolist() == [[0, 2, 0, 5], [2, 5, 5, 75]]
    assert b.key_rows.tolist() == c.cache_rows("b", 0, 5).tolist() + c.cache_rows("a", 0, 75).tolist()
    assert b.slot.tolist() == c.cache_rows("b", 3, 2).tolist() + c.cache_rows("a", 70, 5).tolist()
    assert b.want.tolist() == [2]
    lens, table, seats = c.tables(["b", "a"])
    assert lens.tolist() == [5, 75] and table[1, :2].tolist() == c.pages["a"]


# ---- oracle ---------------------------------------------------------------------------------------------------------------
def _twist(cfg, sd, what):
    cfg, sd = copy.deepcopy(cfg), dict(sd)
    if what == "one pass less":
        cfg["loop"]["times"] -= 1
    elif what == "no yarn":
        cfg["layers"][0]["mixer"]["rot"]["scaling"] = None
    elif what == "no step":
        sd["loop.step"] = torch.zeros_like(sd["loop.step"])
    elif what == "steps swapped":
        sd["loop.step"] = sd["loop.step"].flip(0)
    elif what == "no gate":
        sd["l0.mix.g"] = torch.zeros_like(sd["l0.mix.g"])
    elif what == "no feed-forward":
        cfg["layers"][0]["mlp"] = None
    elif what == "side part of the neighbour":
        n = cfg["token_side"]["dim"]
        sd["side.embed"] = sd["side.embed"].roll(n, dims=1)
    elif what == "key rotation off by one":
        sd["l2.mix.dkv"] = sd["l2.mix.dkv"].roll(1, dims=0)
    elif what == "scale":
        cfg["layers"][2]["mixer"]["scale"] *= 1.05
    elif what == "eps":
        cfg["norm"]["eps"] = 1e-6
    elif what == "query norm":
        sd["l0.mix.dq.norm"] = torch.ones_like(sd["l0.mix.dq.norm"])
    return cfg, sd


@pytest.mark.parametrize("what", ["one pass less", "no yarn", "no step", "steps swapped", "no gate", "no feed-forward",
                                  "side part of the neighbour", "key rotation off by one", "scale", "eps", "query norm"])
def test_a_fault_in_a_mechanism_shows(what):
    """The fault is planted in the oracle; the bound is ten times what the fp32 device tests allow."""
    cfg = H.CONFIGS["mixed"]
    sd = H.weights(cfg, 5)
    toks = H.tokens_of(cfg, 40, 6)
    good = H.oracle_logits(cfg, sd, toks)
    bad = H.oracle_logits(*_twist(cfg, sd, what), toks)
    assert H.error(bad[20:], good[20:]) > 10 * 5e-5


def test_oracle_is_causal_and_position_dependent():
    cfg = H.CONFIGS["mixed"]
    sd = H.weights(cfg, 7)
    toks = H.tokens_of(cfg, 30, 8)
    a = H.oracle_logits(cfg, sd, toks)
    b = H.oracle_logits(cfg, sd, toks[:29] + [(toks[29] + 1) % cfg["vocab"]])
    assert torch.equal(a[:29], b[:29]) and not torch.equal(a[29], b[29])
    c = H.oracle_logits(cfg, sd, toks[1:])
    assert H.error(c[5:], a[6:]) > 1e-2                        # (the first token is gone and every position moved)


def test_trace_command_line():
    from triforce_amd.utils import trace
    a = trace.parse(["--model", "m", "--out", "o", "--max-tokens", "9", "--dtype", "float32"])
    assert (a.model, a.out, a.max_tokens, a.dtype) == ("m", "o", 9, "float32")
    with pytest.raises(SystemExit):
        trace.parse(["--model", "m", "--out", "o", "--max-tokens", "9", "--dtype", "float16"])


def test_trace_replay_protocol(tmp_path):
    """Steps in order, a file only where something is wanted, a line after every step."""
    from triforce_amd.utils import trace
    calls, lines = [], []

    class Engine:
        def step(self, entries, end):
            calls.append((entries, end))
            n = sum(len(w) for _, _, w in entries)
            return torch.arange(float(n * 4)).view(n, 4) if n else None
    steps = [{"step": 0, "entries": [{"id": "a", "tokens": [1, 2], "want": [1]}], "end": []},
             {"step": 1, "entries": [{"id": "a", "tokens": [3], "want": []}], "end": ["a"]}]
    trace.replay(Engine(), [json.dumps(s) + "\n" for s in steps] + ["\n"], str(tmp_path), lines.append)
    assert lines == ["done 0", "done 1"] and calls[1] == ([("a", [3], [])], ["a"])
    assert (tmp_path / "0.f32").stat().st_size == 16 and not (tmp_path / "1.f32").exists()
