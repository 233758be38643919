"""Latent attention of single tokens with a product beside it in the same launch, against fp64 and against the two launched apart."""
import pytest
import torch

from tests.test_gpu_latent import Geom, _paged, f, octets, rnd

pytestmark = pytest.mark.gpu
SCALE = 1.5 * 576 ** -0.5


def _block(rows, n, k0, k, seed):
    from triforce_amd import ops_latent as ol
    act = rnd(rows, k0 + k, seed=seed, dtype=torch.bfloat16)
    w = rnd(n, k0 + k, seed=seed + 1, dtype=torch.bfloat16, scale=(k0 + k) ** -0.5)
    wt = ol.TileWeight(w, packed_only=True)
    assert wt.chunk_major
    return act, w, wt, rnd(rows, n, seed=seed + 2)


# lens, heads, n, k0, k, (workers, panels each, splits): as many workers as splits and fewer, two panels and four, a last workgroup with
# fewer panels, rows of no key, one row, the borders of 16 and 32 rows
CASES = [([500], 20, 4096, 64, 2048, None), ([1], 32, 4096, 32, 4096, None), ([0], 17, 4096, 32, 4096, None),
         ([0, 1], 20, 4096, 4096, 3072, None), ([64, 65, 63, 4000, 0, 128, 129, 700], 20, 4096, 4096, 11008, None),
         ([2000] * 16, 20, 4096, 96, 2176, None), ([129] * 17, 32, 4096, 96, 2176, (170, 3, 20)),
         ([7 * b * b for b in range(32)], 20, 4096, 4096, 2048, (170, 3, 10)), ([1030, 5], 20, 4112, 32, 2080, (4, 2, 2)),
         ([1030, 5, 300], 20, 4112, 32, 2080, (6, 3, 3)), ([1030, 5, 300], 18, 6160, 32, 2080, (200, 4, 128)),
         ([3000] * 20, 18, 4112, 32, 2048, (40, 4, 2))]


@pytest.mark.parametrize("lens,heads,n,k0,k,plan", CASES, ids=[f"{len(c[0])}x{c[1]}-{c[2]}x{c[4]}-{c[5]}" for c in CASES])
def test_attention_beside_a_product(lens, heads, n, k0, k, plan):
    from triforce_amd import ops_latent as ol
    rows = len(lens)
    cache, table, keys = _paged(lens, 512, 64, torch.bfloat16, 5)
    q = rnd(rows, heads, 576, seed=1, dtype=torch.bfloat16)
    klen = torch.tensor(lens, dtype=torch.int32, device=q.device)
    act, w, wt, x = _block(rows, n, k0, k, 7)
    g = Geom(heads, 32, 64, 32, 512, 32)
    plan = plan or (128, 2, max(2, min(128, 256 // rows)))
    got = x.clone()
    out = ol.attn_decode_beside(q, cache, table, klen, g, SCALE, plan + (False,), octets(act), wt, got, k0)
    down = act[:, k0:].double() @ w[:, k0:].double().T
    # fp32 sums of exact products: error below (chunks of 32 + waves) ulp of the sum of magnitudes
    mag = act[:, k0:].double().abs() @ w[:, k0:].double().abs().T + x.double().abs()
    assert bool(((got.double() - (x.double() + down)).abs() <= mag * 2.0 ** -23 * 16).all())
    for b, v in enumerate(lens):
        if v == 0:
            assert bool((out[b] == 0).all())
            continue
        kb = f(keys[b])
        want = torch.softmax(f(q[b]) @ kb.T * SCALE, -1) @ kb[:, :512]
        torch.testing.assert_close(f(out[b]), want, atol=1e-2, rtol=1e-2)
    apart = f(ol.attn_decode(q, cache, table, klen, g, SCALE, max(max(lens), 1)))
    torch.testing.assert_close(f(out), apart, atol=2.0 ** -8, rtol=2.0 ** -7)          # two roundings to bfloat16 of nearly equal sums
    xt = ol.add_linear(octets(act), wt, got, want_copy=True, k=k0)
    total = x.double() + act.double() @ w.double().T
    mag += act.double().abs() @ w.double().abs().T
    assert bool(((got.double() - total).abs() <= mag * 2.0 ** -23 * 16).all())
    assert torch.equal(xt.permute(1, 0, 2).reshape(rows, n), got.bfloat16())


# as many splits as the kernel takes, rows of one and of none beside them, an odd number of rows; V of one panel and of eight
@pytest.mark.parametrize("lens,heads,V,plan", [([4000], 20, 128, (128, 2, 128)), ([0], 17, 16, (128, 2, 128)), ([130, 0, 1, 700], 20, 48, (128, 2, 64)),
                                               ([8000], 32, 128, (128, 2, 128)), ([65] * 4, 20, 128, (8, 3, 2)), ([3000, 2500, 7], 20, 128, (170, 3, 113))])
def test_value_of_unmerged_splits(lens, heads, V, plan):
    from triforce_amd import ops_latent as ol
    rows = len(lens)
    cache, table, keys = _paged(lens, 512, 64, torch.bfloat16, 5)
    q = rnd(rows, heads, 576, seed=1, dtype=torch.bfloat16)
    klen = torch.tensor(lens, dtype=torch.int32, device=q.device)
    act, w, wt, x = _block(rows, 4096, 32, 2048, 7)
    g = Geom(heads, 32, 64, V, 512, 32)
    raw, w_uv = rnd(rows, heads * V + 16, seed=3), rnd(heads, V, 512, seed=4, dtype=torch.bfloat16, scale=512 ** -0.5)
    value = ol.TileWeight(w_uv, packed_only=True)
    got, want = ol.empty_act(rows, heads * V, torch.bfloat16, q.device), ol.empty_act(rows, heads * V, torch.bfloat16, q.device)
    splits = ol.attn_decode_beside(q, cache, table, klen, g, SCALE, plan + (True,), octets(act), wt, x.clone(), 32)
    ol.latent_to_value(splits, value, raw, 16, got, g)
    merged = ol.attn_decode_beside(q, cache, table, klen, g, SCALE, plan + (False,), octets(act), wt, x.clone(), 32)
    ol.latent_to_value(merged, value, raw, 16, want, g)
    flat, gate = (f(t.permute(1, 0, 2).reshape(rows, heads, V)) for t in (got, want)), torch.sigmoid(raw[:, 16:]).view(rows, heads, V)
    got, want = flat
    exact = torch.einsum("rhc,hvc->rhv", f(merged), f(w_uv)) * gate
    size = torch.einsum("rhc,hvc->rhv", f(merged).abs(), f(w_uv).abs()) * gate
    # the merged row is rounded to bfloat16 either way, from sums in another order (now and then to the neighbour, 2^-8 of an entry), and the result
    assert ((got - exact).abs() <= 2.0 ** -8 * exact.abs() + 2.0 ** -8 * size / 8 + 1e-6).all()
    assert ((got - want).abs() <= 2.0 ** -7 * want.abs() + 2.0 ** -8 * size / 8 + 1e-6).all()


@pytest.mark.parametrize("plan", [(128, 2, 64), (170, 3, 85)])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), -float("inf")])
def test_values_that_are_not_finite(bad, plan):
    """A query and a cached row with such a value give what the two launches apart give, and other rows and heads what they give without."""
    from triforce_amd import ops_latent as ol
    lens, heads, V = [700, 130, 64, 300], 32, 32
    cache, table, keys = _paged(lens, 512, 64, torch.bfloat16, 5)
    q = rnd(4, heads, 576, seed=1, dtype=torch.bfloat16)
    klen = torch.tensor(lens, dtype=torch.int32, device=q.device)
    act, w, wt, x = _block(4, 4096, 1024, 2048, 7)
    g, octs = Geom(heads, 32, 64, V, 512, 32), octets(act)
    raw, value = rnd(4, heads * V, seed=3), ol.TileWeight(rnd(heads, V, 512, seed=4, dtype=torch.bfloat16, scale=512 ** -0.5), packed_only=True)

    def run(q, cache, later):
        got, sums = ol.empty_act(4, heads * V, torch.bfloat16, q.device), x.clone()
        o = ol.attn_decode_beside(q, cache, table, klen, g, SCALE, plan + (later,), octs, wt, sums, 1024)
        ol.latent_to_value(o, value, raw, 0, got, g)
        return (None if later else o), got.permute(1, 0, 2).reshape(4, heads, V), sums
    clean = {later: run(q, cache, later) for later in (False, True)}
    q2, cache2 = q.clone(), cache.clone()
    q2[0, 3, 17] = bad                                     # one head of row 0, and every head of row 2 through its first page
    cache2[int(table[2, 0]) * 64 + 5, 11] = bad
    apart = ol.attn_decode(q2, cache2, table, klen, g, SCALE, max(lens))
    spoilt = torch.zeros(4, heads, dtype=torch.bool, device=q.device)
    spoilt[0, 3] = spoilt[2] = True
    for later in (False, True):
        merged, values, sums = run(q2, cache2, later)
        assert torch.equal(sums, clean[later][2]) and torch.equal(values[~spoilt], clean[later][1][~spoilt])
        if merged is not None:
            assert torch.equal(merged[~spoilt], clean[later][0][~spoilt])
            assert torch.equal(merged.isnan(), apart.isnan()) and torch.equal(merged.isinf(), apart.isinf())
            together = values.isnan()
        else:
            assert torch.equal(values.isnan(), together)


def test_replays_in_a_graph():
    """Lengths that change between replays: the deal of the splits is made on the device."""
    from triforce_amd import ops_latent as ol
    lens = [700, 64, 1, 2000]
    cache, table, keys = _paged(lens, 512, 64, torch.bfloat16, 6)
    q = rnd(4, 20, 576, seed=1, dtype=torch.bfloat16)
    klen = torch.tensor(lens, dtype=torch.int32, device=q.device)
    act, w, wt, x = _block(4, 4096, 4096, 2048, 9)
    octs, g = octets(act), Geom(20, 32, 64, 32, 512, 32)
    plan = (128, 2, 64, False)
    keep = torch.zeros_like(x)
    run = lambda into: ol.attn_decode_beside(q, cache, table, klen, g, SCALE, plan, octs, wt, into, 4096)      # noqa: E731
    run(keep)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = run(keep)
    for short in ([700, 64, 1, 2000], [1, 0, 1, 1999], [65, 33, 0, 64], [700, 64, 1, 2000]):
        klen.copy_(torch.tensor(short, dtype=torch.int32))
        keep.zero_()
        graph.replay()
        fresh = torch.zeros_like(x)
        want = run(fresh)
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(keep, fresh)


def _model():
    from tests import latent_helpers as lh
    from triforce_amd.models.config_befidra import BefidraConfig
    from triforce_amd.models.modeling_befidra import BefidraForCausalLM
    cfg = lh.config(96, 4096, [(lh.mixer(17, 32, 64, 32, 64, 512), 11008)])
    return BefidraForCausalLM(BefidraConfig.from_dict(cfg)).init_random(3)


def _filled(model, budget, lens, graphs):
    from triforce_amd.utils.batch_infer import BatchInferenceEngine
    e = BatchInferenceEngine(model, model.make_cache(budget, max_batch=len(lens)), use_graphs=graphs)
    e.kv_cache.extend([(s, n) for s, n in enumerate(lens)])
    for s, n in enumerate(lens):
        for block in e.kv_cache.rows:
            block[e.kv_cache.cache_rows(s, 0, n).long().cuda()] = rnd(n, block.shape[1], seed=s, dtype=block.dtype)
    return e


@pytest.mark.parametrize("lens", [[200], [700, 90, 300, 64, 1, 500, 250, 63], [130 * b for b in range(1, 33)]], ids=lambda v: str(len(v)))
def test_steps_do_not_depend_on_the_room_in_the_cache(lens):
    """A server's cache is larger than its load: the same launches, and the same bits, as in a cache that is full."""
    model = _model()
    tight, roomy = (_filled(model, n, lens, True) for n in (sum(lens) + 8 * len(lens), 400000))
    names, ids = list(range(len(lens))), torch.arange(len(lens)) % 96
    for t in range(3):
        assert torch.equal(tight.decode(names, ids + t), roomy.decode(names, ids + t))
    forms = [list(e._steps[len(lens)].graphs) for e in (tight, roomy)]
    assert forms[0] == forms[1] and forms[0][0][0] is not None


def test_a_graph_for_each_form_of_the_step():
    """Few pages and many in turn, by replays and eagerly: the same logits, and a graph for each form, whichever rows are live."""
    model = _model()
    lens = [60 + 3 * b for b in range(8)] + [16000 - 16 * b for b in range(8)]          # (on either side of a change of the division)
    graphs, eager = (_filled(model, sum(lens) + 1000, lens, g) for g in (True, False))
    few, many = list(range(8)), list(range(8, 16))
    for t, names in enumerate((few, many, few, few, many, few)):
        ids = (torch.arange(8) * 7 + t) % 96
        assert torch.equal(graphs.decode(names, ids), eager.decode(names, ids)), t
    forms = list(graphs._steps[8].graphs)
    assert forms == [model.decode_form(8, sum(n // 64 + 1 for n in ls), max(ls) // 64 + 1) for ls in (lens[:8], lens[8:])] and len(set(forms)) == 2
