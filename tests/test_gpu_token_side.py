"""The per-layer token input with the gate's K cut over the grid, against float64 and against the two products of panels."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# fewer chunks of the width than parts, ragged parts, one per wave and more; sides of one chunk, fewer than the waves, as many, more; real sizes below the padded ones
@pytest.mark.parametrize("rows", [1, 2, 7, 10, 11, 16])
@pytest.mark.parametrize("width,real", [(4096, 4096), (192, 180), (2080, 2080), (8224, 8223)])
@pytest.mark.parametrize("side,side_real", [(32, 20), (64, 64), (256, 256), (256, 250), (544, 544)])
def test_token_side(monkeypatch, rows, width, real, side, side_real):
    from triforce_amd import ops_latent as ol, ops_tile as ot
    monkeypatch.setattr(ol, "token_side_pays", lambda *a: rows <= 10)      # (the kernels at all of these, not only where they are the faster way)
    g = torch.Generator(device=DEV).manual_seed(rows * width + side)

    def rnd(*shape, std=1.0):
        return (torch.randn(*shape, generator=g, device=DEV) * std).bfloat16()
    wg, wp = rnd(side, width, std=width ** -0.5), rnd(width, side, std=side ** -0.5)
    gate, proj = ol.TileWeight(wg, per_panel=True, packed_only=True), ol.TileWeight(wp, packed_only=True)
    x, tables = rnd(width // 8, rows, 8), rnd(100, side_real + 30)
    table = tables[:, 7:7 + side_real]
    ids = torch.randint(0, 100, (rows,), generator=g, device=DEV)
    ids[0] = 99
    got = ol.token_side(x, gate, proj, table, ids, side_real, real)
    assert got.shape == (rows, real)
    xr = ot.act_rows(x).double()
    z, size = xr @ wg.double().T, xr.abs() @ wg.double().abs().T
    e = table[ids].double()
    inner = torch.nn.functional.gelu(z[:, :side_real], approximate="tanh") * e
    want = inner @ wp[:real, :side_real].double().T
    # fp32 sums, gelu with a slope below 1.13, one rounding to bfloat16, the second product's sum
    off = (1.13 * size[:, :side_real] * (width + 16) * 2.0 ** -24 + 1e-6) * e.abs() + inner.abs() * 2.0 ** -8
    bound = off @ wp[:real, :side_real].double().abs().T + inner.abs() @ wp[:real, :side_real].double().abs().T * side * 2.0 ** -24 + 1e-6
    assert bool(((got.double() - want).abs() <= bound).all())
    apart = ot.linear_f32(ol.token_gate_linear(x, gate, table, ids, side_real), proj, real)
    assert bool(((got.double() - apart.double()).abs() <= 2 * bound).all())
    assert torch.equal(got, ol.token_side(x, gate, proj, table, ids, side_real, real))
    if rows > 1:                                              # a row that is not finite stays its own
        x[:, 1] = float("nan")
        spoiled = ol.token_side(x, gate, proj, table, ids, side_real, real)
        assert bool(spoiled[1].isnan().all()) and torch.equal(spoiled[0], got[0]) and torch.equal(spoiled[2:], got[2:])


def test_ids_outside_the_table_are_its_ends():
    from triforce_amd import ops_latent as ol
    g = torch.Generator(device=DEV).manual_seed(1)
    w = torch.randn(64, 256, generator=g, device=DEV).bfloat16()
    gate, proj = ol.TileWeight(w, per_panel=True, packed_only=True), ol.TileWeight(w.T.contiguous(), packed_only=True)
    x, table = torch.randn(32, 3, 8, generator=g, device=DEV).bfloat16(), torch.randn(9, 64, generator=g, device=DEV).bfloat16()
    a = ol.token_side(x, gate, proj, table, torch.tensor([-5, 3, 100], device=DEV), 64, 256)
    assert torch.equal(a, ol.token_side(x, gate, proj, table, torch.tensor([0, 3, 8], device=DEV), 64, 256))


def test_bad_arguments_are_refused():
    from triforce_amd import hip
    f = hip.latent_lib().tfl_token_side
    ok = [1 << 20, 1 << 20, 1 << 20, 8, 8, 1 << 20, 64, 1 << 20, 9, 1 << 20, 256, 1 << 20, 8 * 64 * 3, 3, 256, 64, 64, 256, None]
    for at, v in ((0, None), (2, None), (4, 4), (6, 63), (8, 0), (10, 255), (13, 0), (13, 17), (14, 250), (15, 48), (16, 65), (17, 257)):
        bad = list(ok)
        bad[at] = v
        assert f(*bad) == -22, at
    ok[12] -= 1
    assert f(*ok) == -28
