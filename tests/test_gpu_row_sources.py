"""Row kernels that run inside the wide product that reads their rows, against float64 with the rounding points of the path and against the two launched apart."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EPS = 1e-5


def _f32(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=DEV) * std


def _near(got, h, w, slack=0.0):
    """A product of bfloat16 h, of which a few elements may be the neighbouring one (the norm's own sum in another order)."""
    want, size = h.double() @ w.double().T, h.double().abs() @ w.double().abs().T
    most = float(h.abs().max()) * w.double().abs().max(1).values
    bound = size * w.shape[1] * 2.0 ** -24 + 4 * most * 2.0 ** -7 + want.abs() * slack + 1e-6
    excess = (got.double() - want).abs() - bound
    assert bool((excess <= 0).all()), float(excess.max())


def _rms(v, width):
    return v / torch.sqrt(v.square().sum(-1, keepdim=True) / width + EPS)


# panels of 16 outputs: rests of 4 rows (full, ragged), 8 and 12, whole shares, a share of one more on fewer CUs, the widest; widths of whole and of ragged
# quads a thread; real widths below the padded one
@pytest.mark.parametrize("rows", [1, 2])
@pytest.mark.parametrize("panels,n_raw", [(800, 256), (1024, 4096), (1076, 6272), (1100, 6272), (1200, 512), (1280, 20480), (1500, 512), (2000, 128), (2048, 512)])
@pytest.mark.parametrize("width,real", [(4096, 4096), (4064, 4050), (2048, 2048)])
@pytest.mark.parametrize("with_step", [False, True])
def test_finish_inside_the_input_projection(rows, panels, n_raw, width, real, with_step):
    from triforce_amd import ops_latent as ol, ops_tile as ot
    g = torch.Generator(device=DEV).manual_seed(panels + rows)
    n = 16 * panels
    w = _f32(g, n, width, std=width ** -0.5).bfloat16()
    w[:, real:] = 0
    wt = ol.TileWeight(w, packed_only=True, raw=n_raw)
    if not ol.Finish.takes(rows, width, wt, "in", n_raw):
        assert not wt.chunk_major                             # (sums of squares reach into the left-over rows: the other layout)
        return
    x, y, y_w, norm = _f32(g, rows, width), _f32(g, rows, width + 8)[:, :width], 1 + 0.1 * _f32(g, width), 1 + 0.1 * _f32(g, width)
    step = _f32(g, width, std=0.1) if with_step else None
    for t in (x, y, y_w, norm, step):
        if t is not None:
            t[..., real:] = 0
    q_norm = 1 + 0.1 * _f32(g, 64)
    before = x.clone()
    f = ol.Finish(x, norm, EPS, real, y, y_w, step)
    act = ot.empty_act(rows, max(8, n - n_raw), torch.bfloat16, DEV)
    raw, ss, xq = ol.input_projection(f, wt, n_raw, q_norm, act, 0)
    assert torch.equal(x, before)
    total = x.double() + _rms(y.double(), real) * y_w.double() + (0 if step is None else step.double())
    # the scale of y is off by a few roundings, its product and the two sums by one each: 8 of them, of terms no larger than the magnitudes' sum
    mag = (x.double().abs() + (_rms(y.double(), real) * y_w.double()).abs() + (0 if step is None else step.double().abs())) * 2.0 ** -21 + 1e-30
    assert bool(((f.out.double() - total).abs() <= mag).all())
    h = (_rms(f.out.double(), real) * norm.double()).bfloat16()
    _near(raw, h, w[:n_raw])
    assert bool(((ss.double() - raw.double().square().view(rows, -1, 16).sum(-1)).abs() <= ss.double() * 16 * 2.0 ** -24).all())
    assert torch.equal(ot.act_rows(xq), (raw[:, :64] * q_norm).bfloat16())
    if n > n_raw:
        z = h.double() @ w[n_raw:].double().T
        got, tail = ot.act_rows(act).double(), torch.nn.functional.gelu(z, approximate="tanh")
        assert bool(((got - tail).abs() <= tail.abs() * 2.0 ** -8 + 4 * 1.13 * float(h.abs().max()) * float(w.abs().max()) * 2.0 ** -7 + 1e-5).all())
    apart = x.clone()
    h2 = ol.finish(apart, norm, EPS, real, torch.bfloat16, y=y, y_w=y_w, step=step, octets=True)
    assert bool(((f.out.double() - apart.double()).abs() <= 2 * mag).all())
    raw2, _, _ = ol.input_projection(h2, wt, n_raw, q_norm, torch.empty_like(act), 0)
    _near(raw, ot.act_rows(h2), w[:n_raw])
    assert float((raw - raw2).abs().max()) <= 0.1
    again = ol.input_projection(ol.Finish(x, norm, EPS, real, y, y_w, step), wt, n_raw, q_norm, torch.empty_like(act), 0)
    assert torch.equal(again[0], raw)


@pytest.mark.parametrize("rows", [1, 2])
@pytest.mark.parametrize("n,n_real", [(32000, 32000), (16384, 16380), (32768, 32765), (20000, 19999)])
def test_finish_inside_the_logits(rows, n, n_real):
    from triforce_amd import ops_latent as ol, ops_tile as ot
    g = torch.Generator(device=DEV).manual_seed(n + rows)
    w = _f32(g, n, 4096, std=0.02).bfloat16()
    wt = ol.TileWeight(w, packed_only=True)
    assert ol.Finish.takes(rows, 4096, wt, "f32") and not ol.Finish.takes(3, 4096, wt, "f32")
    x, y, y_w, norm = _f32(g, rows, 4096), _f32(g, rows, 4096), 1 + 0.1 * _f32(g, 4096), 1 + 0.1 * _f32(g, 4096)
    got = ol.finish_logits(ol.Finish(x, norm, EPS, 4096, y, y_w), wt, n_real)
    assert got.shape == (rows, n_real)
    h = ol.finish(x, norm, EPS, 4096, torch.bfloat16, y=y, y_w=y_w)
    _near(got, h, w[:n_real])


@pytest.mark.parametrize("panels", [800, 1024, 1172, 1200, 1376, 1500, 2000, 2048])
@pytest.mark.parametrize("streams", [1, 3, 4])
@pytest.mark.parametrize("width,real", [(4096, 4096), (4064, 4050), (2048, 2048)])
def test_connect_inside_its_products(panels, streams, width, real):
    from triforce_amd import ops_hybrid as oh, ops_tile as ot
    g = torch.Generator(device=DEV).manual_seed(panels + streams)
    n = 16 * panels
    w = _f32(g, n, width, std=width ** -0.5).bfloat16()
    w[:, real:] = 0
    wt = oh.TileWeight(w, packed_only=True)
    assert wt.chunk_major
    x, y, norm = _f32(g, 1, streams, width), _f32(g, 1, width + 8)[:, :width], 1 + 0.1 * _f32(g, width)
    for t in (x, y, norm):
        t[..., real:] = 0
    u_in, out, mix = _f32(g, streams), _f32(g, streams), torch.eye(streams, device=DEV) + _f32(g, streams, streams, std=0.2)
    before = x.clone()
    for epi in ("f32", "glu"):
        assert oh.Connect.takes(x, wt, epi) and not oh.Connect.takes(x.expand(2, -1, -1), wt, epi)
        f = oh.Connect(x, u_in, norm, EPS, real, y, out, mix)
        got = oh.linear_of(f, wt, n - 5) if epi == "f32" else ot.act_rows(oh.gelu_glu_of(f, wt))
        assert torch.equal(x, before)
        new = torch.einsum("st,rsw->rtw", mix.double(), x.double()) + out.double()[None, :, None] * y.double()[:, None]
        mag = torch.einsum("st,rsw->rtw", mix.double().abs(), x.double().abs()) + out.double().abs()[None, :, None] * y.double().abs()[:, None]
        assert bool(((f.out.double() - new).abs() <= mag * 6 * 2.0 ** -24).all())          # five roundings at most, of partial sums
        u = torch.einsum("s,rsw->rw", u_in.double(), f.out.double())
        h = (_rms(u, real) * norm.double()).bfloat16()
        apart = x.clone()
        h2 = oh.connect(apart, u_in, norm, EPS, real, torch.bfloat16, y=y, out=out, mix=mix, octets=True)
        assert torch.equal(f.out, apart)
        if epi == "f32":
            _near(got, h, w[:n - 5])
            _near(got, ot.act_rows(h2), w[:n - 5])
            none = oh.Connect(x, u_in, norm, EPS, real, y, out, mix, keep=False)
            assert none.out is None and torch.equal(oh.linear_of(none, wt, n - 5), got)
        else:
            two = ot.act_rows(oh.gelu_glu_of(h2, wt)).double()
            gate, up = (h.double() @ w.double().T).view(1, panels, 2, 8).unbind(2)
            want = (torch.nn.functional.gelu(gate, approximate="tanh") * up).reshape(1, -1)
            slip = 4 * float(h.abs().max()) * float(w.abs().max()) * 2.0 ** -7
            bound = want.abs() * 2.0 ** -7 + slip * (1.13 * up.abs() + gate.abs() + 1).reshape(1, -1)
            assert bool(((got.double() - want).abs() <= bound).all()) and bool(((got.double() - two).abs() <= 2 * bound).all())
