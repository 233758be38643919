"""Kernels at the sizes where their variants change: edges of tiles, remainders, both sides of a dispatch rule.  Each against plain
torch on the CPU or in float64, with a bound that follows from the types."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# sets - 1 winners: one, around a wave, around the 1 024 threads of the sort, several per thread; many ties, infinities, both zeros
@pytest.mark.parametrize("H,C,sets", [(1, 2, 2), (2, 65, 65), (3, 130, 64), (2, 200, 66), (2, 1100, 1025), (2, 2600, 1026), (1, 4000, 2500),
                                      (1, 9000, 8193), (2, 15616, 512), (1, 20000, 1), (1, 32768, 3000)])
@pytest.mark.parametrize("ties", [False, True])
def test_retrieval_topk_against_stable_sort(H, C, sets, ties):
    from triforce_amd import ops
    g = torch.Generator().manual_seed(C + sets)
    s = torch.randn(H, C, generator=g)
    s = (s * 2).round() / 2 if ties else s
    s = s.half()
    s[:, C // 2] = float("inf")
    s[:, C // 3] = float("-inf")
    got = ops.retrieval_topk(s.to(DEV), sets).cpu().long()
    v = s.float()
    v = torch.where((v == 0) & torch.signbit(v), torch.full_like(v, -1e-30), v)       # the keys' order: -0 below +0
    want = torch.argsort(-v[:, 1:].double(), dim=1, stable=True)[:, :sets - 1] + 1
    assert torch.equal(got, torch.cat([torch.zeros(H, 1, dtype=torch.long), want], 1))


# keys of the deciding bin: as many as are ranked against each other, one more, all (a second and a third digit); both sides of 8 and of 16 keys a thread
@pytest.mark.parametrize("C", [8193, 8194, 16385, 16386])
@pytest.mark.parametrize("crowd", [256, 257, 8000])
@pytest.mark.parametrize("equal", [True, False])
def test_retrieval_topk_of_a_crowded_bin(C, crowd, equal):
    from triforce_amd import ops
    g = torch.Generator().manual_seed(C + crowd)
    s = torch.rand(2, C, generator=g) * 0.9                                           # below the bin of 1 to 1 + 1/32
    for h in range(2):
        at = torch.randperm(C - 1, generator=g)[:crowd + 10] + 1
        s[h, at[:crowd]] = 1.0 + (0 if equal else 1) * torch.randint(0, 32, (crowd,), generator=g) / 1024.0
        s[h, at[crowd:]] = 2.0 + torch.arange(10)
    for sets in (12, 12 + crowd // 2, 11 + crowd):                                    # one of the bin, half of it, all
        got = ops.retrieval_topk(s.half().to(DEV), sets).cpu().long()
        want = torch.argsort(-s.half()[:, 1:].double(), dim=1, stable=True)[:, :sets - 1] + 1
        assert torch.equal(got, torch.cat([torch.zeros(2, 1, dtype=torch.long), want], 1))


# few rows and more, heads of whole 16-byte pieces and not, rows and bases that start on one and not, more pieces than a workgroup's threads; both cache layouts
@pytest.mark.parametrize("H,D", [(1, 16), (3, 48), (33, 128), (2, 8), (5, 40), (3, 2)])
@pytest.mark.parametrize("shift,pad", [(0, 0), (0, 4), (1, 7), (8, 8)])
@pytest.mark.parametrize("token_major", [False, True])
@pytest.mark.parametrize("rows", [63, 64, 70])
def test_rope_append_in_pieces(H, D, shift, pad, token_major, rows):
    from triforce_amd import ops
    from oracle import ref_ops as R
    g = torch.Generator().manual_seed(H * D + shift)
    T = rows + 7
    wide = torch.randn(rows, shift + 3 * H * D + pad, generator=g).half()
    qkv = wide.to(DEV)[:, shift:shift + 3 * H * D]
    cos, sin = torch.randn(40, D, generator=g).half(), torch.randn(40, D, generator=g).half()
    pos = torch.randint(0, 40, (rows,), generator=g)
    q, k, v = wide[:, shift:shift + 3 * H * D].view(rows, 3, H, D).unbind(1)
    for rotate in (True, False):
        kl, vl = (torch.zeros((T, H, D) if token_major else (H, T, D), dtype=torch.float16, device=DEV) for _ in "kv")
        if token_major:
            kl, vl = kl.permute(1, 0, 2), vl.permute(1, 0, 2)
        got = ops.rope_append(qkv, cos.to(DEV), sin.to(DEV), pos.to(DEV), kl, vl, 4, H, D, rotate_k=rotate)
        assert torch.equal(got.cpu(), R.apply_rope(q, cos, sin, pos))
        assert torch.equal(kl[:, 4:4 + rows].permute(1, 0, 2).cpu(), R.apply_rope(k, cos, sin, pos) if rotate else k)
        assert torch.equal(vl[:, 4:4 + rows].permute(1, 0, 2).cpu(), v)
        assert not kl[:, :4].any() and not kl[:, 4 + rows:].any() and not vl[:, :4].any() and not vl[:, 4 + rows:].any()


# chunks: fewer than a workgroup's groups, one step and a bit, an even and an odd number of steps, one workgroup per CU; both layouts
@pytest.mark.parametrize("H,C,token_major", [(3, 5, False), (5, 17, True), (32, 257, False), (40, 700, False), (32, 8200, False), (2, 3001, True)])
def test_retrieval_score_chunks_of_eight(H, C, token_major):
    from triforce_amd import ops
    g = torch.Generator(device=DEV).manual_seed(C)
    k = torch.randn(C * 8 + 3, H, 128, generator=g, device=DEV, dtype=torch.float16)
    k = k.transpose(0, 1) if token_major else k.transpose(0, 1).contiguous()
    q = torch.randn(H, 128, generator=g, device=DEV, dtype=torch.float16)
    got = ops.retrieval_score(k, q, C, 8)
    acc = torch.zeros(H, C, 128, device=DEV)
    for r in range(8):
        acc += k[:, :C * 8].reshape(H, C, 8, 128)[:, :, r].float()
    mean = (acc * 0.125).half().double()
    want = (mean * q[:, None].double()).sum(-1)
    # 128 fp32 products and sums, then one rounding to fp16
    bound = (mean * q[:, None].double()).abs().sum(-1) * 128 * 2.0 ** -24 + want.abs() * 2.0 ** -11 + 2.0 ** -24
    assert ((got.double() - want).abs() <= bound).all()


# three and four rounds of chunks and a little (the general kernel, up to its 2 048 workgroups), whole rounds, nearly four
@pytest.mark.parametrize("H,C,token_major", [(32, 769, False), (32, 800, True), (32, 768, False), (32, 921, False), (32, 1000, False), (40, 600, False), (40, 801, False),
                                             (64, 450, True), (7, 3700, False)])
def test_retrieval_score_rounds(H, C, token_major):
    test_retrieval_score_chunks_of_eight(H, C, token_major)


def _attention64(q, k, v, scale):
    """Causal attention of the last rows in float64: q (n, H, D), k / v (H, m, D) -> out and sum of weight x |value|, per head."""
    n, m = q.shape[0], k.shape[1]
    hidden = torch.arange(m, device=q.device)[None] > torch.arange(m - n, m, device=q.device)[:, None]
    out, size = [], []
    for h in range(q.shape[1]):
        w = torch.softmax((q[:, h].double() @ k[h].double().T * scale).masked_fill(hidden, float("-inf")), -1)
        out.append(w @ v[h].double())
        size.append(w @ v[h].double().abs())
    return torch.stack(out, 1), torch.stack(size, 1)


# row blocks of 128: one row more, whole, one short; slabs of 64 keys: partial and whole; one split (output written by the kernel) and
# several (merged); scores that rise with the key (the running maximum moves in every slab); rows H * D apart
@pytest.mark.parametrize("n,past,H,token_major,rising", [(129, 0, 8, False, False), (256, 63, 8, False, True), (383, 1, 3, True, False), (200, 2000, 8, True, False),
                                                         (1000, 129, 16, False, False), (2049, 0, 32, False, True), (4096, 5, 8, False, False),
                                                         (130, 9000, 5, False, False)])
def test_prefill_attention_blocks_and_splits(n, past, H, token_major, rising):
    from triforce_amd import ops
    g = torch.Generator(device=DEV).manual_seed(n)
    m, D, scale = past + n, 128, 0.08837890625
    k, v = (torch.randn(m + 7, H, D, generator=g, device=DEV, dtype=torch.float16) for _ in range(2))
    q = torch.randn(n, H, D, generator=g, device=DEV, dtype=torch.float16)
    if rising:
        k = (k + q.mean(0) * 20 * torch.linspace(0, 1, m + 7, device=DEV)[:, None, None]).half()
    k[m:], v[m:] = float("nan"), float("nan")                   # behind the keys: never read
    kc, vc = (t.transpose(0, 1) if token_major else t.transpose(0, 1).contiguous() for t in (k, v))
    got = ops.attn_prefill(q, kc, vc, m, scale).view(n, H, D).double()
    want, size = _attention64(q, kc[:, :m], vc[:, :m], scale)
    # weights are rounded to fp16 (2^-11 of each, numerator and sum are not rounded alike), scores and sums are fp32
    bound = 2.0 ** -10 * size + 2.0 ** -11 * want.abs() + 1e-6
    assert ((got - want).abs() <= bound).all()


# keys and values on either side of 256 MB (8 heads: 65 536 keys), row blocks that are no multiple of eight, splits
@pytest.mark.parametrize("n,past,H", [(1100, 64436, 8), (1100, 64437, 8), (2500, 63100, 8), (1409, 20000, 32)])
def test_prefill_attention_order_of_row_blocks(n, past, H):
    from triforce_amd import ops
    g = torch.Generator(device=DEV).manual_seed(n)
    k, v = (torch.randn(H, past + n, 128, generator=g, device=DEV, dtype=torch.float16) for _ in range(2))
    q = torch.randn(n, H, 128, generator=g, device=DEV, dtype=torch.float16)
    got = ops.attn_prefill(q, k, v, past + n, 0.088).view(n, H, 128).double()
    for rows in (slice(0, 64), slice(n - 140, n)):              # (the first rows and those of the last blocks)
        seen = past + n - (n - rows.stop)
        want, size = _attention64(q[rows], k[:, :seen], v[:, :seen], 0.088)
        assert ((got[rows] - want).abs() <= 2.0 ** -10 * size + 2.0 ** -11 * want.abs() + 1e-6).all()
    assert torch.isfinite(got).all()


# row blocks of 256 (640 MB of keys and values, whole rounds of 256 workgroups; 900 MB, more than half a last round): one ragged block and two, tiles of one key, of 63 and whole ones,
# rows H * D apart; scores that rise with the key
@pytest.mark.parametrize("n,past,H,token_major,rising", [(130, 2431, 512, False, False), (256, 2560, 512, True, True), (257, 4934, 256, True, False),
                                                         (511, 4672, 256, False, True), (3850, 37111, 32, False, False),
                                                         (3300, 54310, 32, True, True), (257, 9100, 200, False, False)])
def test_prefill_attention_wide_blocks(n, past, H, token_major, rising):
    from triforce_amd import ops
    g = torch.Generator(device=DEV).manual_seed(n)
    m = past + n
    k, v = (torch.randn(*((m + 7, H) if token_major else (H, m + 7)), 128, generator=g, device=DEV, dtype=torch.float16) for _ in range(2))
    kc, vc = (t.transpose(0, 1) if token_major else t for t in (k, v))
    q = torch.randn(n, H, 128, generator=g, device=DEV, dtype=torch.float16)
    some = [0, 7, H - 1]
    if rising:
        for h in some:
            kc[h] += (q[:, h].mean(0) * 20 * torch.linspace(0, 1, m + 7, device=DEV)[:, None]).half()
    kc[:, m:], vc[:, m:] = float("nan"), float("nan")           # behind the keys: never read
    got = ops.attn_prefill(q, kc, vc, m, 0.088).view(n, H, 128)
    assert torch.isfinite(got).all()
    for rows in {(0, min(70, n)), (max(0, n // 2 - 40), n // 2 + 40), (n - min(n, 140), n)}:
        seen = m - (n - rows[1])
        want, size = _attention64(q[rows[0]:rows[1], some], kc[some, :seen], vc[some, :seen], 0.088)
        assert ((got[rows[0]:rows[1], some].double() - want).abs() <= 2.0 ** -10 * size + 2.0 ** -11 * want.abs() + 1e-6).all()       # (as above)


# a value that is not finite spoils the rows that see it, and by hidden weights of 0 no others than those whose 64 rows walk its tile of 64 keys
@pytest.mark.parametrize("n,past,H", [(256, 2560, 512), (511, 4672, 256), (3850, 37111, 32), (3300, 54310, 32)])
def test_prefill_attention_reach_of_a_value_that_is_not_finite(n, past, H):
    from triforce_amd import ops
    g = torch.Generator(device=DEV).manual_seed(n)
    k, v = (torch.randn(H, past + n, 128, generator=g, device=DEV, dtype=torch.float16) for _ in range(2))
    q = torch.randn(n, H, 128, generator=g, device=DEV, dtype=torch.float16)
    plain = ops.attn_prefill(q, k, v, past + n, 0.088).view(n, H, 128).clone()
    at = past + torch.linspace(0, n - 1, H, device=DEV).long()  # a key of the chunk for each head
    v[torch.arange(H, device=DEV), at, 5] = float("inf")
    got = ops.attn_prefill(q, k, v, past + n, 0.088).view(n, H, 128)
    row = torch.arange(n, device=DEV)[:, None]
    walked = 64 * ((past + torch.clamp(64 * (row // 64 + 1), max=n) + 63) // 64)
    assert not torch.isfinite(got[..., 5])[past + row >= at].any()
    clean = at[None] >= walked
    assert clean.any() and torch.equal(got[clean], plain[clean])


# every key alike, rows that do not see all of their last slab: a hidden score of minus infinity times 0 is no number
@pytest.mark.parametrize("n,past,H", [(130, 0, 8), (200, 2000, 8), (2049, 0, 32)])
def test_prefill_attention_scale_of_zero(n, past, H):
    from triforce_amd import ops
    g = torch.Generator(device=DEV).manual_seed(n)
    k, v = (torch.randn(H, past + n, 128, generator=g, device=DEV, dtype=torch.float16) for _ in range(2))
    q = torch.randn(n, H, 128, generator=g, device=DEV, dtype=torch.float16)
    got = ops.attn_prefill(q, k, v, past + n, 0.0).view(n, H, 128).double()
    want, size = _attention64(q, k, v, 0.0)
    assert ((got - want).abs() <= 2.0 ** -10 * size + 2.0 ** -11 * want.abs() + 1e-6).all()


def test_prefill_attention_rows_far_apart():
    """Cache rows 2^25 elements apart: past the 32-bit offsets of a slab, so the chunk goes block by block."""
    from triforce_amd import ops
    g = torch.Generator(device=DEV).manual_seed(5)
    n, m, D, gap = 130, 131, 128, 1 << 25
    store = torch.empty((m - 1) * gap + 2 * D, device=DEV, dtype=torch.float16)
    k, v = (store.as_strided((1, m, D), (D, gap, 1), at) for at in (0, D))
    k.normal_(generator=g)
    v.normal_(generator=g)
    q = torch.randn(n, 1, D, generator=g, device=DEV, dtype=torch.float16)
    got = ops.attn_prefill(q, k, v, m, 0.088).view(n, 1, D).double()
    want, size = _attention64(q, k, v, 0.088)
    assert ((got - want).abs() <= 2.0 ** -10 * size + 2.0 ** -11 * want.abs() + 1e-6).all()


def _bf(g, *shape, std=1.0):
    return (torch.randn(*shape, generator=g, device=DEV) * std).to(torch.bfloat16)


def _near(got, want, size, k, out_bits=0):
    """fp32 sums of k exact products (k * 2^-24 of their magnitudes), and the output's own rounding."""
    bound = size * k * 2.0 ** -24 + (want.abs() * 2.0 ** -out_bits if out_bits else 0) + 1e-6
    assert ((got.double() - want).abs() <= bound).all()


# panels of 16 outputs over 256 workgroups: whole shares, 4 / 8 / 12 rows left over (full and ragged), a share of one panel more, the
# widest; chunks: fewer than the waves, odd, one per wave and more; batch rows around one and two row blocks
@pytest.mark.parametrize("panels", [256, 257, 319, 330, 391, 460, 512, 700, 1076, 2000, 2048])
@pytest.mark.parametrize("rows,k", [(1, 32), (3, 544), (16, 288), (17, 256), (32, 96), (33, 800)])
def test_wide_gemm_shares(panels, rows, k):
    from triforce_amd import ops_latent as ol, ops_tile as ot
    g = torch.Generator(device=DEV).manual_seed(panels * 100 + rows)
    n = 16 * panels
    w, h = _bf(g, n, k, std=k ** -0.5), _bf(g, k // 8, rows, 8)
    x = ot.act_rows(h)
    wt = ot.TileWeight(w)
    wt.packed, wt.chunk_major = ot.pack_tiles(w, True), True            # (the layout that weights of a longer k come in)
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    _near(ot.linear_f32(h, wt, n - 5), want[:, :n - 5], size[:, :n - 5], k)
    res = torch.randn(rows, n, generator=g, device=DEV)
    got = res.clone()
    copy = ol.add_linear(h, wt, got, want_copy=True)
    _near(got, want + res.double(), size + res.double().abs(), k + 1)
    assert torch.equal(ot.act_rows(copy), got.to(torch.bfloat16))
    # gate | up: the outputs of one panel are an octet; errors of gate and up carry over with slopes below 1.13 and |gate|
    out = ot.act_rows(ot.gelu_glu_linear(h, wt)).double()
    v, s = (t.view(rows, panels, 2, 8) for t in (want, size))
    glu = torch.nn.functional.gelu(v[:, :, 0], approximate="tanh") * v[:, :, 1]
    bound = (1.13 * s[:, :, 0] * v[:, :, 1].abs() + s[:, :, 1] * v[:, :, 0].abs()) * (k + 16) * 2.0 ** -24 + glu.abs() * 2.0 ** -8 + 1e-6
    assert ((out - glu.reshape(rows, -1)).abs() <= bound.reshape(rows, -1)).all()
    # raw outputs with sums of squares in front, gelu behind: the left-over rows lie behind, or the raw part reaches into them
    q_norm = 1.0 + 0.1 * torch.randn(64, generator=g, device=DEV)
    for n_raw in (128, 16 * (panels - 1)):
        act = ot.empty_act(rows, n - n_raw, torch.bfloat16, DEV)
        raw, ss, xq = ol.input_projection(h, wt, n_raw, q_norm, act, 0)
        _near(raw, want[:, :n_raw], size[:, :n_raw], k)
        sums = raw.double().square().view(rows, -1, 16).sum(-1)
        assert ((ss.double() - sums).abs() <= sums * 16 * 2.0 ** -24).all()
        assert torch.equal(ot.act_rows(xq), (raw[:, :64] * q_norm).to(torch.bfloat16))
        tail = torch.nn.functional.gelu(want[:, n_raw:], approximate="tanh")
        _near(ot.act_rows(act), tail, size[:, n_raw:] * 1.13, k + 16, out_bits=8)


# rests that are taken as a panel of their own, in some epilogues only, and the last that are not
@pytest.mark.parametrize("panels,rows,k", [(384, 3, 96), (385, 17, 64), (640, 16, 96), (704, 33, 64), (705, 2, 64), (960, 17, 64), (961, 1, 96), (1984, 5, 64)])
def test_wide_gemm_rests(panels, rows, k):
    test_wide_gemm_shares(panels, rows, k)


# what the packing rule says is what the kernel does: the two forms sum in different orders, so the layout's own form is the one whose
# bits a weight that was packed by the rule has; and both forms read either layout
@pytest.mark.parametrize("panels,raw", [(255, 0), (256, 0), (257, 16), (257, 4112), (330, 4096), (330, 4112), (452, 7232), (2047, 0), (2048, 0), (2049, 0), (2300, 64)])
def test_weight_layout_follows_the_kernel(panels, raw):
    from triforce_amd import ops_latent as ol, ops_tile as ot
    g = torch.Generator(device=DEV).manual_seed(panels)
    n, k, rows = 16 * panels, 2048, 3
    w, h = _bf(g, n, k, std=k ** -0.5), _bf(g, k // 8, rows, 8)
    x = ot.act_rows(h)
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    rule, other = ot.TileWeight(w, packed_only=True, raw=raw), ot.TileWeight(w, packed_only=True, raw=raw)
    other.chunk_major = not rule.chunk_major
    other.packed = ot.pack_tiles(w, True) if other.chunk_major else ot.pack_tiles(w.unsqueeze(0))
    q_norm = torch.ones(16, device=DEV)

    def outputs(wt):
        if raw:
            act = ot.empty_act(rows, max(n - raw, 16), torch.bfloat16, DEV)
            return ol.input_projection(h, wt, raw, q_norm, act, 0)[0]
        return ot.linear_f32(h, wt, n)
    a, b = outputs(rule), outputs(other)
    for got in (a, b):
        _near(got, want[:, :got.shape[1]], size[:, :got.shape[1]], k)
    assert rule.chunk_major == ot.shares_panels(n, k, raw) == (not torch.equal(a, b))          # (same bits: the same form on both layouts)
    if not raw:                                                  # the other epilogues of more panels than the form takes
        wt = rule if rule.chunk_major else other
        res = torch.randn(rows, n, generator=g, device=DEV)
        got = res.clone()
        ol.add_linear(h, wt, got)
        _near(got, want + res.double(), size + res.double().abs(), k + 1)
        v, s = (t.view(rows, panels, 2, 8) for t in (want, size))
        glu = torch.nn.functional.gelu(v[:, :, 0], approximate="tanh") * v[:, :, 1]
        bound = (1.13 * s[:, :, 0] * v[:, :, 1].abs() + s[:, :, 1] * v[:, :, 0].abs()) * (k + 16) * 2.0 ** -24 + glu.abs() * 2.0 ** -8 + 1e-6
        assert ((ot.act_rows(ot.gelu_glu_linear(h, wt)).double() - glu.reshape(rows, -1)).abs() <= bound.reshape(rows, -1)).all()


# weights of products without the one-workgroup-per-CU form: panel by panel, whatever their size; chunk-major ones give the same bits
def test_query_and_token_weights_in_both_layouts():
    from types import SimpleNamespace as NS
    from triforce_amd import ops_latent as ol, ops_tile as ot
    g = torch.Generator(device=DEV).manual_seed(6)
    geom, rows = NS(H=32, N=128, R=64, C=64, Q=2048, q_real=2048, c_real=64, row=128), 5
    raw = torch.randn(rows, 2048 + 128, generator=g, device=DEV)
    ss = raw.view(rows, -1, 16).square().sum(-1).contiguous()
    angle = torch.rand(50, 32, generator=g, device=DEV)
    rope = NS(cos=angle.cos().contiguous(), sin=angle.sin().contiguous(), half=32, max_pos=50)
    at = torch.arange(rows, dtype=torch.int32, device=DEV)
    wq, wg, h = _bf(g, 32 * 192, 2048), _bf(g, 4096, 2048), _bf(g, 256, rows, 8)
    table, ids = _bf(g, 9, 4096), torch.arange(rows, device=DEV)
    out = []
    for chunk_major in (False, True):
        a, b = ot.TileWeight(wq, per_panel=True), ot.TileWeight(wg, per_panel=True)
        assert not a.chunk_major and not b.chunk_major and ot.TileWeight(wg).chunk_major
        if chunk_major:
            for t, w in ((a, wq), (b, wg)):
                t.packed, t.chunk_major = ot.pack_tiles(w, True), True
        cache = torch.zeros(128, 128, dtype=torch.bfloat16, device=DEV)
        qn, q = ol.query_and_append(h, raw, ss, a, geom, torch.ones(64, device=DEV), 1e-5, rope, at, at, cache)
        out.append((qn, q[..., 64:], cache, ol.token_gate_linear(h, b, table, ids, 4096)))
    assert all(torch.equal(a, b) for a, b in zip(*out))


# seven panels per CU in two row blocks, whole and with rows left over: right, and no slower than the wider eight-panel form
def test_wide_gemm_of_seven_panels():
    from triforce_amd import ops_tile as ot
    g = torch.Generator(device=DEV).manual_seed(7)
    k, rows, spans = 4096, 33, {}
    for panels in (1700, 1792, 1900):
        h, ws, out = _bf(g, k // 8, rows - 1, 8), [], torch.empty(rows - 1, 16 * panels, device=DEV)
        for _ in range(2):                                       # (470 MB: from memory each time)
            w = _bf(g, 16 * panels, k, std=k ** -0.5)
            ws.append(ot.TileWeight(w, packed_only=True))
        assert ws[0].chunk_major
        h33 = _bf(g, k // 8, rows, 8)
        x = ot.act_rows(h33)
        _near(ot.linear_f32(h33, ws[1], 16 * panels), x.double() @ w.double().T, x.double().abs() @ w.double().abs().T, k)
        spans[panels] = []
        for i in range(12):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for j in range(4):
                ot.linear_f32(h, ws[j % 2], 16 * panels, out)
            b.record()
            b.synchronize()
            spans[panels].append(a.elapsed_time(b))
    assert min(spans[1700]) < min(spans[1900]) and min(spans[1792]) < min(spans[1900]), spans


@pytest.mark.parametrize("n", [1, 64, 65, 200])
def test_set_pages(n):
    from triforce_amd import hip, ops_tile as ot
    table = torch.zeros(7, 40, dtype=torch.int32, device=DEV)[:, :37]
    places = torch.randperm(7 * 37, generator=torch.Generator().manual_seed(n))[:n].tolist()
    ot.set_pages(table, [(p // 37, p % 37, 1000 + p) for p in places])
    want = torch.zeros(7 * 37, dtype=torch.int32)
    for p in places:
        want[p] = 1000 + p
    assert torch.equal(table.cpu(), want.view(7, 37))
    for bad in ((7, 0, 1), (0, 37, 1), (-1, 0, 1)):
        with pytest.raises(hip.TriforceHipError):
            ot.set_pages(table, [bad])


# the merge by waves (rows x heads from 128 on, at most 64 splits) and by workgroups; splits without a page, idle rows
@pytest.mark.parametrize("rows,H,nsplit", [(4, 32, 2), (5, 32, 16), (4, 33, 17), (9, 16, 64), (4, 32, 65), (1, 32, 30), (130, 1, 3)])
def test_latent_decode_merge(rows, H, nsplit):
    from types import SimpleNamespace
    from triforce_amd import ops_latent as ol
    g = torch.Generator(device=DEV).manual_seed(rows * nsplit)
    C, R, pages = 512, 64, 24
    geom = SimpleNamespace(H=H, C=C, R=R)
    lens = torch.tensor([0 if b % 7 == 6 else 1 + (b * 389) % (64 * 6) for b in range(rows)], dtype=torch.int32)
    table = torch.randint(0, pages, (rows, 6), generator=torch.Generator().manual_seed(1), dtype=torch.int32)
    cache, q = _bf(g, pages * 64, C + R), _bf(g, rows, H, C + R)
    got = ol.attn_decode(q, cache, table.to(DEV), lens.to(DEV), geom, 0.05, 384, nsplit=nsplit).double()
    for b in range(rows):
        n = int(lens[b])
        if n == 0:
            assert not got[b].any()
            continue
        k = cache.view(pages, 64, C + R)[table[b].long().to(DEV)].reshape(-1, C + R)[:n].double()
        w = torch.softmax(q[b].double() @ k.T * 0.05, -1)
        want = w @ k[:, :C]
        # weights as two bfloat16 (2^-16), fp32 scores of 576 products, fp32 sums, one rounding to bfloat16
        bound = (2.0 ** -15 + 1e-4) * (w @ k[:, :C].abs()) + 2.0 ** -8 * want.abs() + 1e-6
        assert ((got[b] - want).abs() <= bound).all()


# rows in a workgroup's registers (16 waves up to 256 rows, four waves beyond) and the general form (wider than 4 096)
@pytest.mark.parametrize("rows,width,real", [(1, 32, 30), (3, 4096, 4096), (256, 1056, 1040), (257, 4096, 4090), (300, 96, 96), (5, 4128, 4100)])
@pytest.mark.parametrize("dtype,y32,parts", [(torch.bfloat16, False, "ys"), (torch.bfloat16, True, "y"), (torch.float32, True, "es"), (torch.bfloat16, False, "")])
def test_finish_rows(rows, width, real, dtype, y32, parts):
    from triforce_amd import ops_latent as ol
    g = torch.Generator(device=DEV).manual_seed(rows + width)

    def rand(*s):
        t = torch.randn(*s, generator=g, device=DEV)
        t[..., real:] = 0
        return t
    x, w, yw, step = rand(rows, width), rand(width), rand(width), rand(width)
    y, embed, ids = rand(rows, width).to(torch.float32 if y32 else dtype), rand(50, width).to(dtype), torch.randint(0, 50, (rows,), generator=g, device=DEV)
    want = embed[ids].double() if "e" in parts else x.double()
    if "y" in parts:
        want = want + y.double() / torch.sqrt(y.double().square().sum(-1, keepdim=True) / real + 1e-5) * yw.double()
    if "s" in parts:
        want = want + step.double()
    h = ol.finish(x, w, 1e-5, real, dtype, **(dict(embed=embed, ids=ids) if "e" in parts else {}), **(dict(y=y, y_w=yw) if "y" in parts else {}),
                  step=step if "s" in parts else None)
    assert ((x.double() - want).abs() <= 2e-6 * (1 + want.abs())).all()
    normed = want / torch.sqrt(want.square().sum(-1, keepdim=True) / real + 1e-5) * w.double()
    assert ((h.double() - normed).abs() <= (2.0 ** -8 if dtype == torch.bfloat16 else 0) * normed.abs() + 4e-6 * (1 + normed.abs())).all()


# narrow rows (one wave up to 256, four up to 1 024) and many middling ones (the general form again)
@pytest.mark.parametrize("rows,width", [(1, 256), (5, 264), (300, 248), (300, 1024), (300, 1032), (1024, 2048), (1025, 2048), (1030, 2056)])
def test_finish_narrow_rows(rows, width):
    from triforce_amd import ops_latent as ol
    g = torch.Generator(device=DEV).manual_seed(rows + width)
    x, w, y, yw = (torch.randn(*s, generator=g, device=DEV) for s in ((rows, width), (width,), (rows, width), (width,)))
    want = x.double() + y.double() / torch.sqrt(y.double().square().mean(-1, keepdim=True) + 1e-5) * yw.double()
    h = ol.finish(x, w, 1e-5, width, torch.float32, y=y, y_w=yw)
    assert ((x.double() - want).abs() <= 2e-6 * (1 + want.abs())).all()
    normed = want / torch.sqrt(want.square().mean(-1, keepdim=True) + 1e-5) * w.double()
    assert ((h.double() - normed).abs() <= 4e-6 * (1 + normed.abs())).all()


def test_finish_narrow_rows_cost_less():
    """4 000 rows of 192 against 4 000 of 1 024: with the wide rows' sixteen quads a workgroup they took 0.8 of their time."""
    from triforce_amd import ops_latent as ol
    spans = []
    for width in (192, 1024):
        x, y, w = torch.randn(4000, width, device=DEV), torch.randn(4000, width, device=DEV).bfloat16(), torch.ones(width, device=DEV)
        ol.finish(x, w, 1e-5, width, torch.bfloat16, y=y, y_w=w)
        graph, a, b = torch.cuda.CUDAGraph(), torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        with torch.cuda.graph(graph):
            for _ in range(20):
                ol.finish(x, w, 1e-5, width, torch.bfloat16, y=y, y_w=w)
        times = []
        for _ in range(5):
            a.record()
            graph.replay()
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        spans.append(min(times))
    assert spans[0] < 0.7 * spans[1], spans


# splits dealt over unequal rows (2 to 64 rows), one row and more than 64 rows (the same number each); idle rows, rows right behind a
# chunk's edge; the sized attention and the general one
@pytest.mark.parametrize("rows,nsplit", [(1, 7), (2, 1), (5, 3), (33, 4), (64, 2), (65, 3)])
@pytest.mark.parametrize("D", [128, 96])
def test_step_splits_over_rows(rows, nsplit, D):
    from triforce_amd import ops_hybrid as oh
    g = torch.Generator(device=DEV).manual_seed(rows * 10 + nsplit)
    H, G, chunk, pages = 8, 2, 640, 40
    lens = [0 if b % 9 == 5 else (chunk * (1 + b % 2) + 1 if b % 4 == 3 else 1 + (b * 331) % 1200) for b in range(rows)]
    width = 2 * H * D + 2 * G * D
    raw = torch.randn(rows, width, generator=g, device=DEV)
    pool = _bf(g, pages * 64, G * 2 * D)
    norm = torch.ones(D, device=DEV)
    angle = torch.arange(2000, device=DEV)[:, None] * 0.01 * torch.arange(1, 9, device=DEV)

    def operand(which, splits):
        own = torch.stack([torch.randperm(pages, generator=torch.Generator().manual_seed(b))[:22].to(torch.int32) for b in which])
        table = torch.arange(22 * len(which), dtype=torch.int32).view(len(which), 22).to(DEV)          # pages of its own: the step writes
        cache = pool.view(pages, 64, -1)[own.reshape(-1).long().to(DEV)].reshape(-1, G * 2 * D).clone()
        attn = dict(q_norm=norm, k_norm=norm, cos=angle.cos().float().contiguous(), sin=angle.sin().float().contiguous(), cache=cache, table=table,
                    q_off=0, k_off=H * D, v_off=H * D + G * D, gate_off=H * D + 2 * G * D, half=8, max_pos=2000, H=H, G=G, D=D, D_real=D, V=D, chunk=chunk,
                    scale=0.1, out_scale=1.0)
        klen = torch.tensor([lens[b] for b in which], dtype=torch.int32, device=DEV)
        step = oh.MixerStep(raw[list(which)].contiguous(), klen, 1e-5, torch.bfloat16, attn=attn, max_keys=1300, nsplit=splits)
        return step.run().operand().permute(1, 0, 2).reshape(len(which), -1).double()
    got = operand(range(rows), nsplit)
    for b in range(rows):
        alone = operand([b], 1)[0]
        if lens[b] == 0:
            assert not got[b].any()
        # the same fp32 sums in another order, then one rounding to bfloat16 each
        assert ((got[b] - alone).abs() <= 2.0 ** -7 * alone.abs() + 1e-5).all()
        if lens[b] == 0:
            continue
        # and against plain attention: the new token's key and value behind the row's pages, its chunk alone
        n, at = lens[b], (lens[b] - 1) // chunk * chunk
        own = torch.randperm(pages, generator=torch.Generator().manual_seed(b))[:22]
        old = pool.view(pages, 64, -1)[own.to(DEV)].reshape(-1, G * 2 * D)[at:n - 1]

        def turned(x):                                           # norm, then pairs (e, e + 8) by the position's angle
            x = x / torch.sqrt(x.square().mean(-1, keepdim=True) + 1e-5)
            c, s = angle[n - 1].cos(), angle[n - 1].sin()
            return torch.cat([x[:, :8] * c - x[:, 8:16] * s, x[:, 8:16] * c + x[:, :8] * s, x[:, 16:]], 1).bfloat16().double()
        q, k = turned(raw[b, :H * D].view(H, D)), turned(raw[b, H * D:H * D + G * D].view(G, D))
        v = raw[b, H * D + G * D:H * D + 2 * G * D].view(G, D).bfloat16().double()
        keys = torch.cat([old[:, :G * D].double().view(-1, G, D), k[None]])
        vals = torch.cat([old[:, G * D:].double().view(-1, G, D), v[None]])
        gate = torch.sigmoid(raw[b, H * D + 2 * G * D:].double()).view(H, D)
        for h in range(H):
            w = torch.softmax(keys[:, h // (H // G)] @ q[h] * 0.1, 0)
            want, size = gate[h] * (w @ vals[:, h // (H // G)]), gate[h] * (w @ vals[:, h // (H // G)].abs())
            # the result's rounding to bfloat16; an entry of q or k that rounds the other way moves a score by 2^-8 * 4 * 4 * 0.1 at most
            assert ((got[b, h * D:h * D + D] - want).abs() <= 2.0 ** -8 * want.abs() + (2.0 ** -15 + 0.00625) * size + 1e-6).all()


# float32 on the bfloat16 matrix cores: below and above a tile of 256 x 128, waves without rows, parts of k of unequal length and empty ones
@pytest.mark.parametrize("rows,n,k,splits", [(1, 16, 32, 1), (17, 272, 96, 2), (128, 256, 64, 3), (129, 528, 1056, 5), (257, 48, 4096, 8), (700, 2064, 1536, 0),
                                             (64, 2304, 4096, 1), (300, 16, 32, 0)])
def test_split_float32_product(rows, n, k, splits):
    from triforce_amd import ops_tile as ot
    g = torch.Generator(device=DEV).manual_seed(rows + n)
    wide = torch.randn(rows, k + 36, generator=g, device=DEV)
    w = torch.randn(n, k, generator=g, device=DEV) * torch.exp2(torch.randint(-12, 12, (n, 1), generator=g, device=DEV).float())
    for x in (wide[:, :k], wide[:, 4:k + 4], wide[:, 1:k + 1]):                       # a copy where rows are not 16-byte aligned
        want = x.double() @ w.double().T
        # six sums per 32 columns, each rounded once: a walk of 6 k / 32 steps of at most 2^-24 (and the sum of the parts) of the size that
        # a product of independent values has; a lost lower plane would leave 2^-17 of it
        size = x.double().norm() * w.double().norm(dim=1) / k ** 0.5
        err = (ot.split_linear(x, w, splits).double() - want).norm(dim=0) / size
        assert err.max() <= 2.0 ** -24 * (6 * k / 32) ** 0.5 + 2.0 ** -22


# row tiles of up to 64 rows and of more, waves with some of their panels and with none, one step and two of a tile or part
@pytest.mark.parametrize("k,splits", [(32, 1), (64, 2), (64, 1), (352, 3), (4096, 0)])
@pytest.mark.parametrize("rows,n", [(16, 16), (64, 304), (65, 208), (192, 256), (193, 80), (330, 1040)])
def test_split_float32_ragged_tiles(rows, n, k, splits):
    from triforce_amd import ops_tile as ot
    g = torch.Generator(device=DEV).manual_seed(rows + n + k)
    x, w = torch.randn(rows, k, generator=g, device=DEV), torch.randn(n, k, generator=g, device=DEV)
    got, want = ot.split_linear(x, w, splits).double(), x.double() @ w.double().T
    # every result for itself: six sums per 32 columns, a walk of at most 2^-24 a step of the size of what has been added up
    assert ((got - want).abs() / (x.double().abs() @ w.double().abs().T)).max() <= 5 * 2.0 ** -24 * (1 + (k / 32 / 3) ** 0.5)
    x[rows - 1, k - 1], w[n - 1, 0] = float("inf"), -float("inf")
    odd, rest = ot.split_linear(x, w, splits).double(), (slice(0, rows - 1), slice(0, n - 1))
    assert torch.equal(odd[rest], got[rest]) and not torch.isfinite(odd[rows - 1]).any() and not torch.isfinite(odd[:, n - 1]).any()


# more tiles than CUs: whole rounds of whole tiles and the steps of the others shared by an XCD's CUs; k of no whole eights of steps, ragged last
# tiles, XCDs with one shared tile and with none, few sharers
@pytest.mark.parametrize("rows,n,k", [(1040, 7680, 1024), (1100, 7664, 1056), (700, 12320, 1536), (896, 9472, 2048), (2050, 4112, 4064)])
def test_split_float32_shared_tiles(rows, n, k):
    from triforce_amd import hip
    from triforce_amd import ops_tile as ot
    size_of = hip.tile_lib().tfl_split_gemm_ws_floats
    assert size_of(rows, n, k, 0) not in [size_of(rows, n, k, s) for s in range(1, 9)]
    g = torch.Generator(device=DEV).manual_seed(rows + n)
    x, w = torch.randn(rows, k, generator=g, device=DEV), torch.randn(n, k, generator=g, device=DEV)
    want, size = x.double() @ w.double().T, x.double().norm() * w.double().norm(dim=1) / k ** 0.5
    got = ot.split_linear(x, w)
    assert ((got.double() - want).norm(dim=0) / size).max() <= 2.0 ** -24 * (6 * k / 32) ** 0.5 + 2.0 ** -22         # (as above)
    assert ((got.double() - want).abs() / (x.double().abs() @ w.double().abs().T)).max() <= 5 * 2.0 ** -24 * (1 + (k / 32 / 3) ** 0.5)
    assert torch.equal(got, ot.split_linear(x, w))
    x[rows - 1, 5], x[3, k - 1], w[n - 1, k // 2] = float("inf"), float("nan"), -float("inf")
    got, plain = ot.split_linear(x, w), ot.split_linear(x, w, 1)
    assert torch.equal(torch.isnan(got), torch.isnan(plain)) and torch.equal(got[torch.isinf(plain)], plain[torch.isinf(plain)])
    assert torch.isfinite(got[torch.isfinite(plain)]).all()


# whole tiles of a product that would be cut in three parts of k otherwise: their running sums are as short
def test_split_float32_shared_tiles_are_as_exact_as_parts():
    from triforce_amd import ops_tile as ot
    x, w = _factors("absolute", 700, 12320, 4096)
    want = x.double() @ w.double().T
    far = [(ot.split_linear(x, w, s).double() - want).norm() for s in (0, 3, 1)]
    assert far[0] <= 1.02 * far[1] and far[1] < 0.5 * far[2]


# products that stand alone (a row of x with one entry): every bit of both factors counts, in every place of a step of 32
@pytest.mark.parametrize("splits", [1, 2])
def test_split_float32_single_products(splits):
    from triforce_amd import ops_tile as ot
    g = torch.Generator(device=DEV).manual_seed(splits)
    k, n = 64, 512
    a = torch.rand(k, generator=g, device=DEV) + 1
    w = (torch.rand(n, k, generator=g, device=DEV) + 1) * (torch.randint(0, 2, (n, k), generator=g, device=DEV) * 2 - 1)
    a[::2], w[::3] = 1.0 + 65535 * 2.0 ** -23, 1.0 + 65535 * 2.0 ** -23               # (what cutting loses most of)
    got, want = ot.split_linear(torch.diag(a), w, splits).double(), a.double()[:, None] * w.double().T
    # left out: ml + lm of 2^-25 each and ll; the small products' sum and the last addition are rounded, 2^-24 and less
    assert ((got - want).abs() <= 2.25 * 2.0 ** -24 * want.abs()).all()


def _factors(kind, rows, n, k):
    g = torch.Generator(device=DEV).manual_seed(k)
    x, w = torch.randn(rows, k, generator=g, device=DEV), torch.randn(n, k, generator=g, device=DEV)
    if kind == "uniform":
        return torch.rand(rows, k, generator=g, device=DEV) + 1, torch.rand(n, k, generator=g, device=DEV) + 1
    return {"normal": (x, w), "absolute": (x.abs(), w.abs()), "mean one": (x + 1, w + 1), "mixed": (x.abs(), w)}[kind]


# sums of one sign and of a mean: what a running sum swallows does not average out
@pytest.mark.parametrize("k,splits", [(15104, 1), (15104, 0), (4096, 1), (1024, 3)])
@pytest.mark.parametrize("kind", ["normal", "absolute", "mean one", "uniform", "mixed"])
def test_split_float32_sums(k, splits, kind):
    from triforce_amd import ops_tile as ot
    x, w = _factors(kind, 160, 256, k)
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    # k / 32 roundings of a running sum, 2^-24 of it each and independent; five of them for the largest of 40 960 results
    assert ((ot.split_linear(x, w, splits).double() - want).abs() / size).max() <= 5 * 2.0 ** -24 * (1 + (k / 32 / 3) ** 0.5)


# where these products are taken, they are no further off than the library's on the fp32 instruction
@pytest.mark.parametrize("rows,n,k", [(512, 1136, 15104), (272, 4112, 4096), (1030, 4096, 1024), (1152, 512, 65536)])
@pytest.mark.parametrize("kind", ["normal", "absolute", "mean one", "uniform", "mixed"])
def test_split_float32_against_the_instruction(rows, n, k, kind):
    from triforce_amd import ops_tile as ot
    x, w = _factors(kind, rows, n, k)
    want, library = x.double() @ w.double().T, torch.nn.functional.linear(x, w)
    got = ot.linear_rows(x, w)
    assert torch.equal(got, ot.split_linear(x, w))
    assert (got.double() - want).norm() <= (library.double() - want).norm()


# few results of a long k, and a short k: the library's; on the other side of either line the split kernel's, in parts that fit an XCD
@pytest.mark.parametrize("rows,n,k,split", [(256, 1136, 15104, False), (1024, 512, 8192, False), (1040, 512, 8192, True), (1030, 65536, 64, False),
                                            (700, 65536, 96, True), (700, 1536, 6144, True)])
def test_float32_products_by_shape(rows, n, k, split):
    from triforce_amd import ops_tile as ot
    x, w = _factors("normal", rows, n, k)
    got = ot.linear_rows(x, w)
    assert torch.equal(got, ot.split_linear(x, w) if split else torch.nn.functional.linear(x, w))
    want, size = x[:64].double() @ w[-48:].double().T, x[:64].double().norm(dim=1)[:, None] * w[-48:].double().norm(dim=1)
    assert ((got[:64, -48:].double() - want).abs() <= 2e-6 * size).all()


# every pair of scales, down to denormal factors: results of ordinary size from a tiny factor and a huge one, tiny and huge results
@pytest.mark.parametrize("splits", [1, 2])
def test_split_float32_scales(splits):
    from triforce_amd import ops_tile as ot
    g = torch.Generator(device=DEV).manual_seed(splits)
    k = 64
    scales = torch.tensor([-147, -140, -126, -120, -112, -100, -64, -24, 0, 30, 64, 79, 81, 100, 106, 120], device=DEV)
    x, w = torch.randn(256, k, generator=g, device=DEV, dtype=torch.float64), torch.randn(256, k, generator=g, device=DEV, dtype=torch.float64)
    x, w = ((t * torch.exp2(scales.repeat(16)[:, None].double())).float() for t in (x, w))
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    got = ot.split_linear(x, w, splits).double()
    ok = size < 2.0 ** 127                                       # (above, a partial sum may overflow in one order and not in another)
    assert torch.isfinite(got[ok]).all() and not torch.isnan(got[want.abs() > 2.0 ** 129]).any()
    assert ((got - want).abs()[ok] <= (k * 2.0 ** -24 * size + k * 2.0 ** -149)[ok]).all()


@pytest.mark.parametrize("splits", [1, 2])
def test_split_float32_extremes(splits):
    from triforce_amd import ops_tile as ot
    g = torch.Generator(device=DEV).manual_seed(splits)
    x, w = torch.randn(200, 64, generator=g, device=DEV), torch.randn(272, 64, generator=g, device=DEV).bfloat16().float()
    x[3, 5], x[4, 6], x[5, 7], x[6, 8], x[6, 9] = float("inf"), -float("inf"), float("nan"), float("inf"), -float("inf")
    x[130], x[131], x[132], x[133] = 0, x[131] * 1e-30, x[132] * 1e-36, x[133] * 1e36
    x[134, 1:] *= 1e-38
    w[7, 3], w[8, 3] = float("inf"), float("nan")
    want = x.double() @ w.double().T
    got = ot.split_linear(x, w, splits).double()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    assert torch.equal(got[torch.isinf(want)], want[torch.isinf(want)])
    ok = torch.isfinite(want)
    bound = 64 * 2.0 ** -24 * (x.double().abs().nan_to_num(0, 0, 0) @ w.double().abs().nan_to_num(0, 0, 0).T) + 64 * 2.0 ** -149
    assert ((got - want).abs()[ok] <= bound[ok]).all()

@pytest.mark.parametrize("rows,n,k", [(700, 8192, 4096), (300, 4096, 15104)])                    # whole k, parts of it
def test_split_float32_strange_rows_cost_no_walk(rows, n, k):
    """Results that are not finite are computed again by whole waves, rows with a NaN not at all; a thread for each result took 5 and
    38 times as long as the whole product here."""
    from triforce_amd import ops_tile as ot
    x, w = torch.randn(rows, k, device=DEV), torch.randn(n, k, device=DEV)

    def fastest():
        spans = []
        for _ in range(5):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            ot.split_linear(x, w)
            b.record()
            b.synchronize()
            spans.append(a.elapsed_time(b))
        return min(spans)
    plain = fastest()
    x[rows // 2, 7] = float("inf")
    assert fastest() < 4 * plain
    x[:, k - 3] = float("nan")
    assert fastest() < 1.5 * plain

def test_large_float32_products_that_something_follows():
    """Gradients, tangents, transforms, autocast and other shapes go through the library, which takes part in them."""
    from torch.autograd import forward_ad
    from triforce_amd import ops_tile as ot
    F = torch.nn.functional
    g = torch.Generator(device=DEV).manual_seed(4)
    w, x = torch.randn(4096, 4096, generator=g, device=DEV), torch.randn(256, 4096, generator=g, device=DEV)
    wt = ot.TileWeight(w)
    assert torch.equal(wt.matmul(x), ot.split_linear(x, w))                    # (nothing follows: the kernel)
    assert wt.matmul(x.view(256, 1, 4096)).shape == (256, 1, 4096)
    y = wt.matmul(x.clone().requires_grad_())
    assert y.requires_grad and torch.equal(y, F.linear(x, w))
    with torch.no_grad():
        assert torch.equal(wt.matmul(x.clone().requires_grad_()), ot.split_linear(x, w))
    with forward_ad.dual_level():
        t = forward_ad.unpack_dual(wt.matmul(forward_ad.make_dual(x, torch.ones_like(x)))).tangent
    assert torch.equal(t, F.linear(torch.ones_like(x), w))
    both = torch.func.vmap(wt.matmul)(torch.stack([x, 2 * x]))
    assert both.shape == (2, 256, 4096) and torch.allclose(both[0], F.linear(x, w), rtol=1e-4, atol=1e-3)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert wt.matmul(x).dtype == torch.bfloat16
    with pytest.raises(RuntimeError):
        ot.linear_rows(x[:, :4064], w)



def _flash_want(q, k, v, lo, hi, scale):
    """float64 attention of q [n, d] with keys lo .. hi of every row: (result, the same sums with |v|)."""
    s = (q.double() @ k.double().T) * scale
    at = torch.arange(k.shape[0], device=DEV)
    s = s.masked_fill((at < lo[:, None]) | (at > hi[:, None]), -float("inf"))
    p = torch.softmax(s, 1)
    return p @ v.double(), p @ v.double().abs()


# around a wave's 16 and 32 rows, a workgroup's 128, a tile's 64 keys; chunks that begin inside a tile and inside a workgroup; strange
# values behind the last key
@pytest.mark.parametrize("news,pasts,chunk", [([1], [0], 8192), ([127, 33], [1, 64], 8192), ([129, 16], [63, 500], 8192), ([300], [190], 100),
                                              ([257, 128, 2], [0, 127, 1000], 640), ([65], [0], 1)])
@pytest.mark.parametrize("H,G", [(8, 2), (3, 3)])
def test_chunked_prefill_tiles(news, pasts, chunk, H, G):
    from types import SimpleNamespace as NS
    from triforce_amd import ops_hybrid as oh
    g = torch.Generator(device=DEV).manual_seed(sum(news) + H)
    geom = NS(q_off=0, gate_off=H * 128, H=H, G=G, D=128, V=128, row=G * 256, chunk=chunk, scale=0.11)
    y, out = _bf(g, sum(news), 2 * H * 128), torch.full((sum(news), H * 128), 9.0, dtype=torch.bfloat16, device=DEV)
    pages = [(n + p + 63) // 64 for n, p in zip(news, pasts)]
    cache = _bf(g, (sum(pages) + 1) * 64, G * 256)
    own = torch.randperm(sum(pages), generator=torch.Generator().manual_seed(1)).to(torch.int32)
    table, seq, at, tok = torch.zeros(len(news), max(pages), dtype=torch.int32), [], 0, 0
    for b, (n, p) in enumerate(zip(news, pasts)):
        table[b, :pages[b]] = own[at:at + pages[b]]
        cache.view(-1, 64, G * 256)[int(own[at + pages[b] - 1]), (n + p - 1) % 64 + 1:] = float("nan")
        seq.append([tok, n, p, 0])
        at, tok = at + pages[b], tok + n
    batch = NS(table=table.to(DEV), seq=torch.tensor(seq, dtype=torch.int32, device=DEV), max_new=max(news))
    oh.attn_prefill(y, geom, cache, batch, out, 0.7)
    for b, (t0, n, p, _) in enumerate(seq):
        rows = cache.view(-1, 64, G * 256)[table[b, :pages[b]].long().to(DEV)].reshape(-1, G * 256)[:n + p]
        hi = p + torch.arange(n, device=DEV)
        for h in range(H):
            kv = h // (H // G)
            want, size = _flash_want(y[t0:t0 + n, 128 * h:128 * h + 128], rows[:, 128 * kv:128 * kv + 128], rows[:, 128 * (G + kv):128 * (G + kv) + 128],
                                     hi // chunk * chunk, hi, 0.11)
            s = 0.7 * torch.sigmoid(y[t0:t0 + n, 128 * (H + h):128 * (H + h) + 128].double())
            # every weight rounded to bfloat16 (2^-9 of it), the result too
            assert ((out[t0:t0 + n, 128 * h:128 * h + 128].double() - s * want).abs() <= 2.0 ** -8 * s * (want.abs() + size) + 1e-6).all()


# as above; the last one: long enough, and a whole round, for workgroups of 256 rows
@pytest.mark.parametrize("news,pasts,H", [([1], [0], 8), ([127, 33], [1, 64], 8), ([129, 16], [63, 500], 3), ([257, 128, 2], [0, 127, 1000], 8), ([300, 40], [16400, 16400], 52)])
@pytest.mark.parametrize("half", [32, 5, 0])
def test_latent_prefill_tiles(news, pasts, H, half):
    from types import SimpleNamespace as NS
    from triforce_amd import ops_latent as ol
    g = torch.Generator(device=DEV).manual_seed(sum(news) + H)
    tq, tk = sum(news), sum(news) + sum(pasts)
    geom = NS(H=H, N=128, R=64, V=128, C=64)
    q, kv, ck, gate = _bf(g, tq, H * 192), _bf(g, tk, H * 256), _bf(g, tk, 128), _bf(g, tq, H * 128)
    out = torch.full((tq, H * 128), 9.0, dtype=torch.bfloat16, device=DEV)
    angle = torch.rand(20000, max(half, 1), generator=g, device=DEV)
    rope = NS(cos=angle.cos().contiguous(), sin=angle.sin().contiguous(), half=half, max_pos=20000)
    seq, pos, a, b = [], [], 0, 0
    for n, p in zip(news, pasts):
        seq.append([a, n, b, n + p])
        pos += range(p, p + n)
        a, b = a + n, b + n + p
    pos = torch.tensor(pos, dtype=torch.int32, device=DEV)
    ol.attn_prefill(q, kv, ck, torch.tensor(seq, dtype=torch.int32, device=DEV), max(news), pos, rope, gate, out, geom, 0.08)
    turned = q.view(tq, H, 192).clone()
    even, odd = q.view(tq, H, 192)[..., 128:128 + 2 * half:2].float(), q.view(tq, H, 192)[..., 129:129 + 2 * half:2].float()
    cos, sin = rope.cos[pos.long(), None, :half], rope.sin[pos.long(), None, :half]
    turned[..., 128:128 + 2 * half:2], turned[..., 129:129 + 2 * half:2] = (even * cos - odd * sin).bfloat16(), (odd * cos + even * sin).bfloat16()
    for t0, n, k0, nk in seq:
        hi = nk - n + torch.arange(n, device=DEV)
        for h in sorted({0, H // 2, H - 1}):
            k = torch.cat([kv[k0:k0 + nk, 128 * h:128 * h + 128], ck[k0:k0 + nk, 64:]], 1)
            want, size = _flash_want(turned[t0:t0 + n, h], k, kv[k0:k0 + nk, 128 * (H + h):128 * (H + h) + 128], hi * 0, hi, 0.08)
            s = torch.sigmoid(gate[t0:t0 + n, 128 * h:128 * h + 128].double())
            assert ((out[t0:t0 + n, 128 * h:128 * h + 128].double() - s * want).abs() <= 2.0 ** -8 * s * (want.abs() + size) + 1e-6).all()


# more keys than the caches hold and more than one round of workgroups: sequence by sequence, in blocks of 128 and of 256 rows; heads that
# do not divide over the XCDs; blocks of 256 rows for a few rows behind many keys
@pytest.mark.parametrize("news,pasts,H", [([700, 130, 257], [6000, 5500, 5000], 40), ([700, 130, 257], [6000, 5500, 5000], 39),
                                          ([700, 130, 257, 513], [4200, 3500, 3000, 2500], 64), ([222, 130], [1500, 1700], 128)])
def test_latent_prefill_by_sequence(news, pasts, H):
    test_latent_prefill_tiles(news, pasts, H, 32)


# the same over the paged cache, where the kernel itself adds up the visible keys: on either side of its line, chunks that hide most of
# them, more sequences than a wave has lanes
@pytest.mark.parametrize("news,pasts,chunk,H,G", [([700, 130, 257, 513], [2500, 1000, 2000, 2300], 8192, 32, 32), ([700, 130, 257, 513], [4000, 3000, 2500, 2300], 8192, 23, 23),
                                                  ([700, 130, 257, 513], [4000, 3000, 2500, 2300], 600, 32, 32), ([130] + [1, 3] * 35, [1900] * 71, 8192, 8, 2),
                                                  ([700, 130, 257, 513], [3000, 1500, 1400, 691], 8192, 32, 32), ([700, 130, 257, 513], [3000, 1500, 1400, 692], 8192, 32, 32)])
def test_chunked_prefill_by_sequence(news, pasts, chunk, H, G):
    test_chunked_prefill_tiles(news, pasts, chunk, H, G)


# more pages in a split than the 64 whose ids a wave holds (tiles at 64 and 65 pages, two fetches of ids, none), and merges of more splits than the
# ones that are asked for first
@pytest.mark.parametrize("nsplit", [1, 2, 40])
@pytest.mark.parametrize("D", [64, 128])
def test_step_over_many_pages(nsplit, D):
    from triforce_amd import ops_hybrid as oh
    g = torch.Generator(device=DEV).manual_seed(D + nsplit)
    lens, pages, H, G = [4096, 4097, 8450, 70], 133, 4, 1
    raw = torch.randn(4, 2 * H * D + 2 * G * D, generator=g, device=DEV)
    cache = _bf(g, 4 * pages * 64, G * 2 * D)
    table = torch.randperm(4 * pages, generator=torch.Generator().manual_seed(D)).to(torch.int32).view(4, pages).to(DEV)
    norm = torch.ones(D, device=DEV)
    angle = torch.arange(8500, device=DEV)[:, None] * 0.01 * torch.arange(1, 9, device=DEV)
    before = cache.clone().view(-1, 64, G * 2 * D)
    attn = dict(q_norm=norm, k_norm=norm, cos=angle.cos().float().contiguous(), sin=angle.sin().float().contiguous(), cache=cache, table=table, q_off=0,
                k_off=H * D, v_off=H * D + G * D, gate_off=H * D + 2 * G * D, half=8, max_pos=8500, H=H, G=G, D=D, D_real=D, V=D, chunk=0, scale=0.1,
                out_scale=1.0)
    step = oh.MixerStep(raw, torch.tensor(lens, dtype=torch.int32, device=DEV), 1e-5, torch.bfloat16, attn=attn, max_keys=pages * 64, nsplit=nsplit)
    got = step.run().operand().permute(1, 0, 2).reshape(4, -1).double()

    def turned(x, at):                                           # norm, then pairs (e, e + 8) by the position's angle
        x = x / torch.sqrt(x.square().mean(-1, keepdim=True) + 1e-5)
        c, s = angle[at].cos(), angle[at].sin()
        return torch.cat([x[:, :8] * c - x[:, 8:16] * s, x[:, 8:16] * c + x[:, :8] * s, x[:, 16:]], 1).bfloat16().double()
    for b, n in enumerate(lens):
        old = before[table[b].long()].reshape(-1, G * 2 * D)[:n - 1].double()
        q, k = turned(raw[b, :H * D].view(H, D), n - 1), turned(raw[b, H * D:H * D + G * D].view(G, D), n - 1)
        v = raw[b, H * D + G * D:H * D + 2 * G * D].view(G, D).bfloat16().double()
        keys, vals = torch.cat([old[:, :D], k]), torch.cat([old[:, D:], v])
        gate = torch.sigmoid(raw[b, H * D + 2 * G * D:].double()).view(H, D)
        w = torch.softmax(q @ keys.T * 0.1, 1)
        want, size = gate * (w @ vals), gate * (w @ vals.abs())
        # the result's rounding to bfloat16; an entry of q or k that rounds the other way moves a score by 2^-8 * 4 * 4 * 0.1 at most
        assert ((got[b].view(H, D) - want).abs() <= 2.0 ** -8 * want.abs() + (2.0 ** -15 + 0.00625) * size + 1e-6).all()
        at = table[b, (n - 1) // 64].long()
        assert torch.equal(cache.view(-1, 64, 2 * D)[at, (n - 1) % 64, D:], v[0].bfloat16())


# rows of more quads than threads: the first of a thread is asked for ahead, the others are not
@pytest.mark.parametrize("streams", [1, 4])
@pytest.mark.parametrize("width", [4104, 8192])
def test_connect_of_wide_rows(streams, width):
    from triforce_amd import ops_hybrid as oh
    g = torch.Generator(device=DEV).manual_seed(width + streams)
    x, y, w = (torch.randn(*n, generator=g, device=DEV) for n in ((3, streams, width), (3, width), (width,)))
    u, out, mix = (torch.randn(*n, generator=g, device=DEV) for n in ((streams,), (streams,), (streams, streams)))
    got = x.clone()
    h = oh.connect(got, u, w, 1e-4, width, torch.bfloat16, y=y, out=out, mix=mix)
    want = torch.matmul(mix.double().T, x.double()) + out.double()[None, :, None] * y.double()[:, None]
    # at most 2 * streams float32 sums of terms up to 4 * 4: 8 * 16 * 2^-24 each
    torch.testing.assert_close(got, want.float(), atol=1e-4, rtol=1e-5)
    v = torch.matmul(u.double(), want)
    v = v / torch.sqrt(v.square().mean(-1, keepdim=True) + 1e-4) * w.double()
    assert ((h.double() - v).abs() <= 2.0 ** -8 * v.abs() + 1e-4).all()          # the result's rounding to bfloat16, and the sums above
