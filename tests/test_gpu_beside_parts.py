"""Latent attention of 17 to 32 rows with a product cut over k beside it, whose sums the next product adds."""
import pytest
import torch

from tests.test_gpu_attn_beside import SCALE, _block
from tests.test_gpu_latent import Geom, _paged, f, octets, rnd

pytestmark = pytest.mark.gpu


# rows, heads, n, k0, k, (workers, parts, splits): fewer chunks than waves, ranges of unequal chunks, a last workgroup with fewer panels, rows without keys
@pytest.mark.parametrize("lens,heads,n,k0,k,plan", [
    ([129] * 17, 32, 4096, 96, 2176, (160, 3, 18)), ([7 * b * b for b in range(32)], 20, 4096, 4096, 11008, (128, 4, 8)),
    ([500 + b for b in range(24)], 17, 4112, 2048, 160, (128, 2, 10)), ([0] * 8 + [64] * 12, 32, 8192, 4096, 4096, (64, 3, 6)),
    ([90 * b for b in range(32)], 32, 5120, 4096, 2080, (64, 1, 4)), ([1] * 18, 32, 6160, 1952, 128, (60, 4, 2))])
def test_attention_beside_parts_of_a_product(lens, heads, n, k0, k, plan):
    from triforce_amd import ops_latent as ol
    rows = len(lens)
    cache, table, keys = _paged(lens, 512, 64, torch.bfloat16, 5)
    q = rnd(rows, heads, 576, seed=1, dtype=torch.bfloat16)
    klen = torch.tensor(lens, dtype=torch.int32, device=q.device)
    act, w, wt, x = _block(rows, n, k0, k, 7)
    g = Geom(heads, 32, 64, 32, 512, 32)
    out, sums = ol.attn_decode_beside_parts(q, cache, table, klen, g, SCALE, plan, octets(act), wt, k0, k0 + k)
    assert sums.shape == (plan[1], rows, n)
    a, b = act[:, k0:].double(), w[:, k0:].double()
    mag = a.abs() @ b.abs().T
    assert bool(((sums.double().sum(0) - a @ b.T).abs() <= mag * 2.0 ** -23 * 16).all())          # (as tests/test_gpu_attn_beside.py)
    apart = f(ol.attn_decode(q, cache, table, klen, g, SCALE, max(max(lens), 1)))
    torch.testing.assert_close(f(out), apart, atol=2.0 ** -8, rtol=2.0 ** -7)          # two roundings to bfloat16 of nearly equal sums
    got = x.clone()
    xt = ol.add_linear(octets(act), wt, got, want_copy=True, k=k0, also=sums)
    total = x.double() + act.double() @ w.double().T
    mag = act.double().abs() @ w.double().abs().T + x.double().abs()
    assert bool(((got.double() - total).abs() <= mag * 2.0 ** -23 * 16).all())
    assert torch.equal(xt.permute(1, 0, 2).reshape(rows, n), got.bfloat16())
    again, more = ol.attn_decode_beside_parts(q, cache, table, klen, g, SCALE, plan, octets(act), wt, k0, k0 + k)
    assert torch.equal(again, out) and torch.equal(more, sums)


@pytest.mark.parametrize("rows,n,parts", [(17, 4160, 2), (32, 4096, 4), (33, 5120, 3), (20, 8192, 1)])
def test_sums_that_a_product_adds(rows, n, parts):
    """Whatever the form of the product: rests of rows, several row blocks."""
    from triforce_amd import ops_latent as ol
    act, w, wt, x = _block(rows, n, 0, 2048, 3)
    also = rnd(parts, rows, n, seed=9)
    got, want = x.clone(), x.clone()
    ol.add_linear(octets(act), wt, got, also=also)
    ol.add_linear(octets(act), wt, want)
    mag = act.double().abs() @ w.double().abs().T + x.double().abs() + also.double().abs().sum(0)
    assert bool(((got.double() - want.double() - also.double().sum(0)).abs() <= mag * 2.0 ** -23 * 16).all())
