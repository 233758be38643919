"""Residual streams brought on by the product in front of them, and the norm's scale behind the product that reads them, against float64 and the launches apart."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EPS = 1e-5


def _f32(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=DEV) * std


def _weight(g, n, k):
    from triforce_amd import ops_hybrid as oh
    w = _f32(g, n, k, std=k ** -0.5).bfloat16()
    wt = oh.TileWeight(w, packed_only=True)
    assert wt.chunk_major
    return w, wt


# rows: one, the borders of 16 and 32, more than a block; widths of one panel a CU, of two (full and ragged); panels behind it: rests of 4, 8, 12 rows, whole ones
@pytest.mark.parametrize("rows,streams,width,real,k,n", [
    (1, 4, 4096, 4096, 4096, 18752), (2, 3, 4096, 4080, 2048, 22016), (8, 4, 4096, 4096, 11008, 32000), (15, 1, 4096, 4096, 2080, 4160),
    (16, 4, 4096, 4096, 8192, 12320), (17, 2, 4096, 4096, 4096, 18752), (32, 4, 4096, 4090, 4096, 22016), (33, 4, 4096, 4096, 4096, 8192),
    (65, 3, 4096, 4096, 2048, 32768), (3, 4, 8192, 8192, 4096, 16400), (20, 4, 7232, 7180, 2048, 6160)])
def test_streams_between_two_products(rows, streams, width, real, k, n):
    from triforce_amd import ops_hybrid as oh, ops_tile as ot
    g = torch.Generator(device=DEV).manual_seed(rows + n)
    (w, wt), (after, at) = _weight(g, width, k), _weight(g, n, width)
    act = _f32(g, rows, k).bfloat16()
    x, norm = _f32(g, rows, streams, width), 1 + 0.1 * _f32(g, width)
    w[real:] = 0
    wt.packed = ot.pack_tiles(w.unsqueeze(0), True)
    for t in (x, norm):
        t[..., real:] = 0
    u_in, out, mix = _f32(g, streams), _f32(g, streams), torch.eye(streams, device=DEV) + _f32(g, streams, streams, std=0.2)
    octs = act.view(rows, k // 8, 8).transpose(0, 1).contiguous()
    y = oh.linear_f32(octs, wt, width)
    for epi in ("f32", "glu"):
        if not oh.Streams.takes(x, wt, at, epi):
            assert epi == "glu" and rows > 32 and n == 4160   # (a narrow gate | up of many rows)
            continue
        got = x.clone()
        s = oh.Streams(got, out, mix, u_in, norm, EPS, real).result(octs, wt)
        new = torch.einsum("st,rsw->rtw", mix.double(), x.double()) + out.double()[None, :, None] * y.double()[:, None]
        mag = torch.einsum("st,rsw->rtw", mix.double().abs(), x.double().abs()) + out.double().abs()[None, :, None] * y.double().abs()[:, None]
        # five roundings at most, of partial sums, and y's own sum, which the two forms may take in another order
        size = act.double().abs() @ w.double().abs().T
        assert bool(((got.double() - new).abs() <= mag * 6 * 2.0 ** -24 + out.double().abs()[None, :, None] * size[:, None] * 2.0 ** -20).all())
        u = torch.einsum("s,rsw->rw", u_in.double(), got.double())
        wide = torch.einsum("s,rsw->rw", u_in.double().abs(), got.double().abs()) * 6 * 2.0 ** -24
        h, have = u * norm.double(), ot.act_rows(s.h).double()
        assert bool(((have - h).abs() <= h.abs() * 2.0 ** -8 + wide * norm.double().abs() + 1e-30).all())
        sums = u.square().view(rows, -1, 16).sum(-1)
        assert bool(((s.ss.double() - sums).abs() <= sums * 2.0 ** -19 + 1e-6).all())
        inv = 1 / torch.sqrt(s.ss.double().sum(-1, keepdim=True) / real + EPS)
        z, amount = (have @ after.double().T) * inv, (have.abs() @ after.double().abs().T) * inv
        bound = amount * 2.0 ** -19 + 1e-30                   # fp32 sums of exact products, a few roundings of the scale
        if epi == "f32":
            res = oh.linear_of(s, at, n - 3)
            assert res.shape == (rows, n - 3) and bool(((res.double() - z[:, :n - 3]).abs() <= bound[:, :n - 3]).all())
            # the launches apart: bfloat16 of the normed input instead of the input
            old = oh.linear_f32(oh.connect(x.clone(), u_in, norm, EPS, real, torch.bfloat16, y=y, out=out, mix=mix, octets=True), at, n - 3)
            size = (h.abs() * inv) @ after[:n - 3].double().abs().T
            assert bool(((res - old).double().abs() <= size * 2.0 ** -7 + 1e-6).all())
            none = x.clone()
            again = oh.Streams(none, out, mix, u_in, norm, EPS, real, keep=False).result(octs, wt)
            assert torch.equal(none, x) and torch.equal(again.h, s.h) and torch.equal(oh.linear_of(again, at, n - 3), res)
        else:
            res = ot.act_rows(oh.gelu_glu_of(s, at)).double()
            (gate, up), (gb, ub) = (t.view(rows, n // 16, 2, 8).unbind(2) for t in (z, bound))
            want = torch.nn.functional.gelu(gate, approximate="tanh") * up
            slack = want.abs() * 2.0 ** -8 + (1.13 * gb + 2e-6) * up.abs() + gate.abs() * ub + 1e-6
            assert bool(((res - want.reshape(rows, -1)).abs() <= slack.reshape(rows, -1)).all())


def test_what_is_refused():
    from triforce_amd import hip, ops_hybrid as oh
    g = torch.Generator(device=DEV).manual_seed(1)
    w, wt = _weight(g, 4096, 4096)
    five, narrow = torch.zeros(1, 5, 4096, device=DEV), torch.zeros(1, 4, 2048, device=DEV)
    assert not oh.Streams.takes(five, wt, wt, "f32") and not oh.Streams.takes(narrow, wt, wt, "f32")
    L = hip.hybrid_lib()
    assert L.tfh_streams_gemm_takes(1, 4, 4112, 4096) == L.tfh_streams_gemm_takes(1, 4, 7200, 4096) == 0 and L.tfh_streams_gemm_takes(1, 4, 12288, 4096) == 0 and L.tfh_scaled_gemm_takes(1, 2048, 0) == 0
