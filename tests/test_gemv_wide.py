"""The one-workgroup-per-CU products of csrc/gemv_wide.hip at the edges of their shares, against float64 with the rounding points of the path and bit for bit
against the panel form, and the rule that picks them."""
import os
import subprocess
import sys

import pytest
import torch

DEV = "cuda:0"
EPS = 1e-5


def test_the_rule_takes_whole_shares_only_where_panels_stay_whole():
    from triforce_amd import hip
    takes = hip.lib().tf_wide_gemm_takes
    for mode, n, k, want in [(0, 4096, 4096, 1), (0, 4096, 11008, 1), (0, 8192, 2048, 1), (0, 5120, 5120, 0), (0, 5120, 13824, 0), (0, 7168, 7168, 1),
                             (0, 7152, 7168, 0), (0, 7168, 4096, 0), (0, 7680, 4096, 0), (0, 8192, 2560, 1), (0, 4080, 4096, 0), (0, 4096, 2016, 0),
                             (3, 12288, 4096, 1), (3, 15360, 5120, 1), (3, 9216, 4096, 0),
                             (1, 22016, 4096, 1), (1, 27648, 5120, 1), (1, 4352, 4096, 0), (1, 8176, 4096, 0), (1, 8192, 2048, 1), (2, 4352, 4096, 0), (2, 5136, 4096, 1), (2, 4096, 4096, 1),
                             (2, 32000, 4096, 1), (2, 32768, 4096, 1), (2, 33024, 4096, 0),
                             (2, 32000, 768, 0), (1, 5504, 4096, 0)]:
        assert takes(mode, n, k) == want, (mode, n, k)
    for bad in [(-1, 4096, 4096), (4, 4096, 4096), (0, 4100, 4096), (0, 4096, 4100), (0, 0, 4096), (0, 4096, 0)]:
        assert takes(*bad) == -22


def test_a_line_that_was_asked_for_is_the_line():
    """Rows from which activations are octet-major: TRIFORCE_ACT_PACKED_MIN_ROWS where it is set, upwards too, whatever form the weights have."""
    show = "from triforce_amd import ops; print([[n for n in range(1, 40) if ops.act_packed(n, wide)][:1] for wide in (False, True)])"
    for line, want in ((None, "[[17], [4]]"), ("33", "[[33], [33]]"), ("9", "[[9], [9]]"), ("17", "[[17], [17]]"), ("2", "[[2], [2]]")):
        env = {k: v for k, v in os.environ.items() if not k.startswith("TRIFORCE_ACT")}
        env.update({} if line is None else {"TRIFORCE_ACT_PACKED_MIN_ROWS": line})
        assert subprocess.run([sys.executable, "-c", show], env=env, capture_output=True, text=True, check=True).stdout.strip() == want, line


def _rnd(g, *shape, std=1.0):
    return (torch.randn(*shape, generator=g, device=DEV) * std).half()


def _block(ops, x, packed):
    return ops.Act.from_rows(x, x.shape[0] + 3) if packed else x


def _rows(y):
    return y if isinstance(y, torch.Tensor) else y.rows()


def _normed(x, ln):
    inv = 1.0 / torch.sqrt(x.float().square().mean(-1, keepdim=True) + EPS)
    return ln * (x.float() * inv).half()


def _sums(ops, x):
    ss = ops.ss_buffer(x.shape[1], DEV)
    ss.fill_(float("nan"))                                     # (rows that are not there are not read)
    ss[:, :x.shape[0]] = x.float().view(x.shape[0], -1, 16).square().sum(-1).T
    return ss


def _product(h, w):
    """The product in 64 bits, and how far its fp16 may be: fp32 sums, their rounding, two operand elements on the neighbouring fp16 (the norm's own sum)."""
    want, size = h.double() @ w.double().T, h.double().abs() @ w.double().abs().T
    most = float(h.abs().max()) * w.double().abs().max(1).values
    return want, size * w.shape[1] * 2.0 ** -24 + want.abs() * 2.0 ** -11 + 2 * most * 2.0 ** -10 + 2.0 ** -24


def _near(got, want, bound):
    excess = (got.double() - want).abs() - bound
    assert bool((excess <= 0).all()), float(excess.max())


# batch rows: one, one block full, two blocks, the last row of them; chunks: as many for each wave, 65 (the last wave has 2), 129
ROWS_K = [(1, 2048), (7, 4128), (16, 2080), (17, 2048), (32, 4096)]


@pytest.mark.gpu
@pytest.mark.parametrize("M,K", ROWS_K)
@pytest.mark.parametrize("N", [4096, 7168, 8192])             # one panel a workgroup, two on 224 CUs, two
@pytest.mark.parametrize("packed", [False, True])
def test_residual(M, K, N, packed):
    from triforce_amd import ops
    K += 5120 if N == 7168 else 0                              # (a part of the CUs: from 7 168 on)
    g = torch.Generator(device=DEV).manual_seed(N + M)
    w, x, res = _rnd(g, N, K, std=K ** -0.5), _rnd(g, M, K), _rnd(g, M, N)
    pl = ops.PackedLinear(w, wide="residual")
    assert pl.wide == "residual"
    want, bound = _product(x, w)
    _near(_rows(ops.linear(_block(ops, x, packed), pl)), want, bound)
    assert torch.equal(_rows(ops.linear(_block(ops, x, packed), pl)), ops.linear(x, ops.PackedLinear(w)))
    ss, y = torch.full((N // 16, 32), float("nan"), device=DEV), _block(ops, res.clone(), packed)
    ops.linear(_block(ops, x, packed), pl, resid=y, out=y, ss_out=ss)
    got, total = _rows(y), want + res.double()
    _near(got, total, bound + total.abs() * 2.0 ** -11 + 2.0 ** -24)
    own = got.double().view(M, -1, 16).square().sum(-1).T
    assert bool(((ss[:, :M].double() - own).abs() <= own * 16 * 2.0 ** -24).all())
    pl.w.mul_(2.0)                                             # exact in fp16: re-packed in place
    before = pl.parts[0].data_ptr()
    assert pl.refresh_().parts[0].data_ptr() == before
    _near(_rows(ops.linear(_block(ops, x, packed), pl)), 2 * want, 2 * bound)


@pytest.mark.gpu
@pytest.mark.parametrize("M,K", ROWS_K)
# pairs of panels: one workgroup's rest of 4 rows (ragged), whole shares, rests of 8 (full and ragged), a share of one more on fewer CUs, the widest
@pytest.mark.parametrize("I", [4128, 4096, 5120, 11008, 13824, 16384])
def test_swiglu(M, K, I):
    from triforce_amd import ops
    g = torch.Generator(device=DEV).manual_seed(I + M)
    w, x, ln = _rnd(g, 2 * I, K, std=K ** -0.5), _rnd(g, M, K), (1 + 0.1 * torch.randn(K, generator=g, device=DEV)).half()
    pl = ops.PackedLinear(w, split=2, wide="swiglu")
    assert pl.wide == "swiglu"
    want, bound = _product(_normed(x, ln), w)
    (a, u), (ea, eu) = want.chunk(2, 1), bound.chunk(2, 1)
    # silu' is below 1.1 and |silu(a)| at most |a|; roundings of silu and of the product, and expf
    unit = torch.nn.functional.silu(a) * u
    most = 1.1 * ea * (u.abs() + eu) + a.abs() * eu + unit.abs() * 2.0 ** -9 + 2.0 ** -23 * (1 + u.abs())
    for packed in (False, True):
        for ss in (None, _sums(ops, x)):
            got = _rows(ops.mlp_act(_block(ops, x, packed), pl, ln=ln, eps=EPS, ss_in=ss))
            _near(got, unit, most)
            if M <= 16 or I > 3200:                            # (the panel form cuts K into eight for two row blocks of few panels)
                assert torch.equal(got, ops.mlp_act(x, ops.PackedLinear(w, split=2), ln=ln, eps=EPS, ss_in=ss))


@pytest.mark.gpu
@pytest.mark.parametrize("M,K", ROWS_K)
@pytest.mark.parametrize("N", [4096, 5136, 8208, 9984, 21504, 32000, 32768])  # whole shares, rests of 8 beside one panel, 4 and 12 rows, a share of one more, the widest
def test_logits(M, K, N):
    from triforce_amd import ops
    g = torch.Generator(device=DEV).manual_seed(N + M)
    w, x, ln = _rnd(g, N, K, std=K ** -0.5), _rnd(g, M, K), (1 + 0.1 * torch.randn(K, generator=g, device=DEV)).half()
    pl = ops.PackedLinear(w, wide="logits")
    assert pl.wide == "logits"
    want, bound = _product(x, w)
    got = ops.linear(x, pl, out_f32=True)
    assert got.dtype == torch.float32 and torch.equal(got, got.half().float())          # an fp16 product, then the cast
    _near(got, want, bound)
    want, bound = _product(_normed(x, ln), w)
    for ss in (None, _sums(ops, x)):
        y = ops.linear(_block(ops, x, ss is None), pl, out_f32=True, ln=ln, eps=EPS, ss_in=ss)
        _near(y, want, bound)
        if N > 8192:                                           # (up to 512 panels: eight parts of K there)
            assert torch.equal(y, ops.linear(x, ops.PackedLinear(w), out_f32=True, ln=ln, eps=EPS, ss_in=ss))
    wide = torch.full((M, N + 5), 7.0, device=DEV)
    ops.linear(x, pl, out_f32=True, out=wide[:, 2:N + 2])                               # rows at any stride: nothing beside them is written
    assert torch.equal(wide[:, 2:N + 2], got) and bool((wide[:, :2] == 7).all()) and bool((wide[:, N + 2:] == 7).all())


@pytest.mark.gpu
@pytest.mark.parametrize("M,K", ROWS_K)
@pytest.mark.parametrize("H,D", [(32, 128), (40, 128), (20, 128), (64, 64), (56, 128)])   # 3 panels a workgroup, 4 on 240 CUs, 2 on 240, heads of 64, 6 on 224
@pytest.mark.parametrize("rotate_k", [True, False])
def test_qkv(M, K, H, D, rotate_k):
    from triforce_amd import ops
    g = torch.Generator(device=DEV).manual_seed(H + M)
    w, x, ln = _rnd(g, 3 * H * D, K, std=K ** -0.5), _rnd(g, M, K), (1 + 0.1 * torch.randn(K, generator=g, device=DEV)).half()
    pl = ops.PackedLinear(w, rope=(H, D), wide="qkv")
    assert pl.wide == "qkv"
    a = torch.outer(torch.arange(300, device=DEV).float(), 100.0 ** (-torch.arange(0, D, 2, device=DEV) / D))
    cos, sin = (torch.cat([t, t], 1).half() for t in (a.cos(), a.sin()))
    pos = torch.randint(0, 300, (M,), generator=g, device=DEV)
    want, bound = ([t.view(M, H, D) for t in p.chunk(3, 1)] for p in _product(_normed(x, ln), w))
    c, s = cos[pos].double()[:, None], sin[pos].double()[:, None]

    def turned(v, e):
        other, eo = (torch.cat([t[..., D // 2:], t[..., :D // 2]], -1) for t in (v, e))
        sign = torch.cat([-torch.ones(D // 2), torch.ones(D // 2)]).to(DEV).double()
        return v * c + sign * other * s, (e * c.abs() + eo * s.abs()) + ((v * c).abs() + (other * s).abs()) * 2.0 ** -10 + 2.0 ** -23
    for ss, dev in ((None, None), (_sums(ops, x), torch.tensor([9], dtype=torch.int32, device=DEV))):
        k, v = (torch.full((H, 64, D), 5.0, device=DEV).half() for _ in range(2))
        q = ops.qkv_rope(_block(ops, x, ss is None), pl, ln, EPS, cos, sin, pos, k, v, 0 if dev is not None else 9, H, D, rotate_k=rotate_k, slot0_dev=dev,
                         ss_in=ss)
        _near(q, *turned(want[0], bound[0]))
        _near(k[:, 9:9 + M].transpose(0, 1), *(turned(want[1], bound[1]) if rotate_k else (want[1], bound[1])))
        _near(v[:, 9:9 + M].transpose(0, 1), want[2], bound[2])
        if 3 * H * D > 8192:
            k2, v2 = (torch.full((H, 64, D), 5.0, device=DEV).half() for _ in range(2))
            q2 = ops.qkv_rope(x, ops.PackedLinear(w, rope=(H, D)), ln, EPS, cos, sin, pos, k2, v2, 9, H, D, rotate_k=rotate_k, ss_in=ss)
            assert torch.equal(q, q2) and torch.equal(k, k2) and torch.equal(v, v2)
        for t in (k, v):
            assert bool((t[:, :9] == 5).all()) and bool((t[:, 9 + M:] == 5).all())


@pytest.mark.gpu
def test_a_row_that_is_not_finite_stays_its_own():
    from triforce_amd import ops
    g = torch.Generator(device=DEV).manual_seed(3)
    w, x, ln = _rnd(g, 8192, 2048, std=2048 ** -0.5), _rnd(g, 5, 2048), torch.ones(2048, device=DEV).half()
    pl = ops.PackedLinear(w, wide="logits")
    good = ops.linear(x, pl, out_f32=True, ln=ln, eps=EPS)
    x[2, 7], x[4] = float("inf"), 0.0
    got = ops.linear(x, pl, out_f32=True, ln=ln, eps=EPS)
    assert torch.equal(got[[0, 1, 3]], good[[0, 1, 3]]) and bool(got[2].isnan().any()) and bool((got[4] == 0).all())


# What the form does not have goes to the panel form, not to a library, and gives its bits; eagerly, in a captured graph, and after the weight has changed.
CALLS = {
    "residual": [lambda o, w, x, ln, r: o.linear(x, w, ln=ln, eps=EPS), lambda o, w, x, ln, r: o.linear(x, w, out_f32=True),
                 lambda o, w, x, ln, r: o.linear(x, w, resid=r[:, :w.N], out=r.clone()[:, 1:w.N + 1]),
                 lambda o, w, x, ln, r: o.linear(_beside(x), w)],
    "logits": [lambda o, w, x, ln, r: o.linear(x, w), lambda o, w, x, ln, r: o.linear(x, w, ln=ln, eps=EPS, resid=r[:, :w.N].contiguous())],
    "swiglu": [lambda o, w, x, ln, r: o.mlp_act(x, w), lambda o, w, x, ln, r: o.mlp_act(o.Act.from_rows(x), w).rows(),
               lambda o, w, x, ln, r: o.mlp_act(_beside(x), w, ln=ln, eps=EPS)],
    "qkv": [lambda o, w, x, ln, r: o.linear(x, w), lambda o, w, x, ln, r: _turned(o, w, x)],
}


def _beside(x):
    """x at 8 bytes behind a boundary of 16."""
    return torch.cat([x[:, :4], x, x[:, :4]], 1)[:, 4:-4]


def _turned(ops, w, x):
    H, D = w.rope
    cos = torch.ones(64, D, device=DEV).half()
    k, v = torch.zeros(H, 64, D, device=DEV).half(), torch.zeros(H, 64, D, device=DEV).half()
    q = ops.qkv_rope(x, w, None, 0.0, cos, cos * 0.5, torch.arange(x.shape[0], device=DEV), k, v, 3, H, D)
    return torch.cat([q.flatten(), k.flatten(), v.flatten()])


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 7, 32])
@pytest.mark.parametrize("use", sorted(CALLS))
def test_other_calls_of_a_wide_weight(monkeypatch, use, M):
    from triforce_amd import ops, ops_rows
    monkeypatch.setattr(ops_rows, "linear", lambda *a, **k: pytest.fail("library product"))
    monkeypatch.setattr(ops_rows, "glu_linear", lambda *a, **k: pytest.fail("product of many rows"))
    g = torch.Generator(device=DEV).manual_seed(M)
    kw = dict(swiglu=dict(split=2), qkv=dict(rope=(32, 128))).get(use, {})
    N, K = {"residual": 4096, "logits": 32000, "swiglu": 22016, "qkv": 12288}[use], 4096
    w, x, ln, r = _rnd(g, N, K, std=K ** -0.5), _rnd(g, M, K), (1 + 0.1 * torch.randn(K, generator=g, device=DEV)).half(), _rnd(g, M, N + 8)
    for call in CALLS[use]:
        pl, plain = ops.PackedLinear(w, wide=use, **kw), ops.PackedLinear(w, **kw)
        assert pl.wide == use and plain.wide is None
        want = call(ops, plain, x, ln, r)
        for eager_first in (False, True):
            graph = torch.cuda.CUDAGraph()
            if eager_first:
                assert torch.equal(call(ops, pl, x, ln, r), want)
                assert pl.panels() is pl.panels() is not pl
            with torch.cuda.graph(graph):
                out = call(ops, pl, x, ln, r)
            for _ in range(3):
                out.zero_()
                graph.replay()
                assert torch.equal(out, want) and torch.equal(call(ops, pl, x, ln, r), want)
        w.mul_(0.5)
        pl.refresh_(), plain.refresh_()
        want = call(ops, plain, x, ln, r)
        graph.replay()
        assert torch.equal(call(ops, pl, x, ln, r), want) and torch.equal(out, want)
        w.mul_(2.0)
