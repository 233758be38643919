"""Token gate and latent to value of 17 to 64 rows, whose blocks of 16 rows go to workgroups of their own where the panels are few, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [16, 17, 33, 64, 65])
@pytest.mark.parametrize("n,k", [(32, 4096), (1024, 2080), (1056, 64)])
def test_token_gate(rows, n, k):
    from triforce_amd import ops_latent as ol
    g = torch.Generator(device="cuda").manual_seed(rows + n)
    x, w, table = (torch.randn(*s, generator=g, device="cuda").bfloat16() for s in ((rows, k), (n, k), (50, n)))
    w = (w * k ** -0.5).bfloat16()
    ids = torch.randint(0, 50, (rows,), generator=g, device="cuda")
    octs = x.view(rows, k // 8, 8).transpose(0, 1).contiguous()
    real = n - 3 if n == 1056 else n
    got = ol.token_gate_linear(octs, ol.TileWeight(w, packed_only=True, per_panel=True), table[:, :real], ids, real)
    z = x.double() @ w.double().T
    e = table.double()[ids]
    want = torch.nn.functional.gelu(z, approximate="tanh") * e
    # fp32 sums of exact products, a slope of gelu below 1.13, one rounding to bfloat16
    size = (x.double().abs() @ w.double().abs().T) * 2.0 ** -23 * 16
    bound = want.abs() * 2.0 ** -8 + (1.13 * size + 2e-6) * e.abs() + 1e-30
    assert bool(((got.double() - want).abs() <= bound)[:, :real].all()) and bool((got[:, real:] == 0).all())


@pytest.mark.parametrize("rows,H,V", [(17, 32, 128), (64, 16, 96), (65, 20, 128), (33, 32, 160)])
def test_latent_to_value(rows, H, V):
    from tests.test_gpu_latent import Geom
    from triforce_amd import ops_latent as ol
    g = torch.Generator(device="cuda").manual_seed(rows)
    o, w = (torch.randn(*s, generator=g, device="cuda").bfloat16() for s in ((rows, H, 512), (H, V, 512)))
    w = (w * 512 ** -0.5).bfloat16()
    raw = torch.randn(rows, 32 + H * V, generator=g, device="cuda")
    act = ol.empty_act(rows, H * V + 64, torch.bfloat16, "cuda").fill_(3)
    geom = Geom(H, 32, 64, V, 512, 32)
    ol.latent_to_value(o, ol.TileWeight(w, packed_only=True), raw, 32, act, geom)
    o64, w64 = o.double().transpose(0, 1).contiguous(), w.double().transpose(1, 2).contiguous()
    z, size = (torch.bmm(a, b).transpose(0, 1).reshape(rows, H * V) for a, b in ((o64, w64), (o64.abs(), w64.abs())))
    s = torch.sigmoid(raw[:, 32:].double())
    got = ol.act_rows(act).double()
    assert bool(((got[:, :H * V] - z * s).abs() <= (z * s).abs() * 2.0 ** -7 + size * 2.0 ** -23 * 16 + 1e-30).all()) and bool((got[:, H * V:] == 3).all())


# float32 at the same borders, and the last rows and panels for which every block of 16 rows has a CU
@pytest.mark.parametrize("rows", [16, 17, 64, 65])
def test_token_gate_float32(rows):
    from triforce_amd import ops_latent as ol
    g = torch.Generator(device="cuda").manual_seed(rows)
    n, k = 96, 2080
    x, w, table = (torch.randn(*s, generator=g, device="cuda") for s in ((rows, k), (n, k), (50, n)))
    w *= k ** -0.5
    ids = torch.randint(0, 50, (rows,), generator=g, device="cuda")
    got = ol.token_gate_linear(x.view(rows, k // 8, 8).transpose(0, 1).contiguous(), ol.TileWeight(w, packed_only=True, per_panel=True), table, ids, n)
    z, e = x.double() @ w.double().T, table.double()[ids]
    size = (x.double().abs() @ w.double().abs().T) * k * 2.0 ** -24              # fp32 products and sums, a slope of gelu below 1.13
    assert bool(((got.double() - torch.nn.functional.gelu(z, approximate="tanh") * e).abs() <= (1.13 * size + 2e-6) * e.abs() + 1e-6).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,H", [(1, 20), (32, 16), (33, 16), (48, 10), (48, 11), (17, 32), (64, 8), (65, 8)])
def test_latent_to_value_where_the_blocks_part(rows, H, dtype):
    from tests.test_gpu_latent import Geom
    from triforce_amd import ops_latent as ol
    g, V, C = torch.Generator(device="cuda").manual_seed(rows), 128, 512
    o, w = (torch.randn(*s, generator=g, device="cuda").to(dtype) for s in ((rows, H, C), (H, V, C)))
    w = (w * C ** -0.5).to(dtype)
    raw = torch.randn(rows, H * V, generator=g, device="cuda")
    act = ol.empty_act(rows, H * V, dtype, "cuda")
    ol.latent_to_value(o, ol.TileWeight(w, packed_only=True), raw, 0, act, Geom(H, 32, 64, V, C, 32))
    o64, w64 = o.double().transpose(0, 1).contiguous(), w.double().transpose(1, 2).contiguous()
    z, size = (torch.bmm(a, b).transpose(0, 1).reshape(rows, H * V) for a, b in ((o64, w64), (o64.abs(), w64.abs())))
    want = z * torch.sigmoid(raw.double())
    # sums in fp32 (C of them), the sigmoid's roundings, one rounding of the result
    assert bool(((ol.act_rows(act).double() - want).abs() <= want.abs() * (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -20) + size * C * 2.0 ** -24).all())
