"""Latent decode attention in half pages: edges of half pages, pages and the window of 64 page ids, idle rows and heads, scores that outgrow the
reference of the weights, stale cache rows."""
import pytest
import torch

from tests.test_gpu_latent import Geom

pytestmark = pytest.mark.gpu


# lens, heads, splits: one key, a half page, one more, a page, one more; a split of more than 64 pages; an idle row; 16 heads, two groups of heads
@pytest.mark.parametrize("lens,heads,nsplit", [([1, 32, 33, 64, 65], 32, 1), ([96, 97, 128, 2, 31], 20, 2), ([4100, 0, 4096, 63], 32, 1), ([8300], 17, 2),
                                               ([700, 3], 16, 3), ([1000, 129], 40, 4)])
@pytest.mark.parametrize("rising", [0.0, 1.0, 40.0])
def test_half_pages(lens, heads, nsplit, rising):
    from triforce_amd import ops_latent as ol
    g = torch.Generator(device="cuda").manual_seed(len(lens) + heads)
    rows, pages = len(lens), [(n + 63) // 64 for n in lens]
    own = torch.randperm(sum(pages) + 1, generator=torch.Generator().manual_seed(1)).to(torch.int32)
    cache = torch.randn((sum(pages) + 1) * 64, 576, generator=g, device="cuda").to(torch.bfloat16)
    q = torch.randn(rows, heads, 576, generator=g, device="cuda").to(torch.bfloat16)
    table, at, paged = torch.zeros(rows, max(pages), dtype=torch.int32), 0, cache.view(-1, 64, 576)
    for b, n in enumerate(lens):
        table[b, :pages[b]] = own[at:at + pages[b]]
        at += pages[b]
        for k, p in enumerate(table[b, :pages[b]].tolist()):   # a page's scores lie up to 40 times the mean square of q above the last one's
            paged[p] += (q[b].float().mean(0) * rising * k).to(torch.bfloat16)
        if n % 64:
            paged[int(table[b, pages[b] - 1]), n % 64:] = float("nan")
    klen = torch.tensor(lens, dtype=torch.int32, device="cuda")
    out = ol.attn_decode(q, cache, table.cuda(), klen, Geom(heads, 128, 64, 128, 512, 32), 0.07, max(lens), nsplit=nsplit)
    for b, n in enumerate(lens):
        if n == 0:
            assert (out[b] == 0).all()
            continue
        keys = paged[table[b, :pages[b]].long().cuda()].reshape(-1, 576)[:n].double()
        w = torch.softmax(q[b].double() @ keys.T * 0.07, -1)
        want, size = w @ keys[:, :512], w @ keys[:, :512].abs()
        # scores: fp32 sums of 576 products, 2^-24 of each; weights as two bfloat16: 2^-17; sums of n in fp32; the result rounded to bfloat16
        spread = (q[b].double().abs() @ keys.abs().T * 0.07).amax(-1, keepdim=True) * 576 * 2.0 ** -24
        bound = 2.0 ** -8 * want.abs() + (2.0 ** -16 + n * 2.0 ** -24 + 2 * spread) * size + 1e-6
        assert ((out[b].double() - want).abs() <= bound).all()
