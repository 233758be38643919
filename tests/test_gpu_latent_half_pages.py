"""Latent decode attention in half pages: edges of half pages, pages and the window of 64 page ids, idle rows and heads, scores that outgrow the
reference of the weights, latents of the largest and the smallest size, stale cache rows."""
import pytest
import torch

from tests.test_gpu_latent import Geom

pytestmark = pytest.mark.gpu

SCALE = 0.0625


def offsets(n, heads):
    """What head h adds to its score of key j, [n, heads]: level; once far above (2^100 and more) in the first and in the second half of a page; just
    above the room that a reference leaves (5.5); a little more with every page; two rises in one split; falling; low in the
    first half page, by 2^144 and by 2^98."""
    j = torch.arange(n)
    mid = n // 2 // 64 * 64
    kinds = [torch.zeros(n), 80.0 * (j == mid + 5), 6.0 * (j >= mid + 40), 80.0 * (j == mid + 63), 3.0 * (j // 64), 20.0 * (j >= mid // 2) + 40.0 * (j >= mid),
             -30.0 * (j >= 32), -100.0 * (j < 32), 5.0 * (j == mid), 68.0 * (j >= 32)]
    return torch.stack([kinds[h % len(kinds)] for h in range(heads)], 1)


# Every score is exact: small whole numbers over the latents, a column of the rotated part for each head's own.
def rows_of(lens, heads, latent, q_latent):
    g = torch.Generator().manual_seed(len(lens) + heads)
    q = torch.zeros(len(lens), heads, 576)
    q[:, :, :512] = torch.randint(-1, 2, (len(lens), heads, 512), generator=g) * q_latent
    q[:, torch.arange(heads), 512 + torch.arange(heads)] = 1.0
    keys = []
    for n in lens:
        k = torch.zeros(n, 576)
        k[:, :512] = latent(g, n)
        k[:, 512:512 + heads] = offsets(n, heads) / SCALE + torch.randint(-16, 17, (n, heads), generator=g)
        keys.append(k.to(torch.bfloat16))
    return q.to(torch.bfloat16), keys


def check(lens, heads, nsplit, latent, q_latent=1):
    from triforce_amd import ops_latent as ol
    q, keys = rows_of(lens, heads, latent, q_latent)
    pages = [(n + 63) // 64 for n in lens]
    own = torch.randperm(sum(pages) + 1, generator=torch.Generator().manual_seed(1)).to(torch.int32)
    paged, table, at = torch.full(((sum(pages) + 1), 64, 576), float("nan"), dtype=torch.bfloat16), torch.zeros(len(lens), max(pages), dtype=torch.int32), 0
    for b, n in enumerate(lens):
        table[b, :pages[b]] = own[at:at + pages[b]]
        at += pages[b]
        for p in range(pages[b]):
            part = keys[b][64 * p:64 * p + 64]
            paged[int(table[b, p]), :len(part)] = part
    klen = torch.tensor(lens, dtype=torch.int32, device="cuda")
    out = ol.attn_decode(q.cuda(), paged.view(-1, 576).cuda(), table.cuda(), klen, Geom(heads, 128, 64, 128, 512, 32), SCALE, max(lens), nsplit=nsplit)
    for b, n in enumerate(lens):
        if n == 0:
            assert (out[b] == 0).all()
            continue
        k = keys[b].cuda().double()
        s = q[b].cuda().double() @ k.T * SCALE
        w, below = torch.softmax(s, -1), s.amax(-1, keepdim=True) - s
        v = k[:, :512]
        # a weight: score and reference and their difference in fp32 (2^-24 of each, in powers of two), its exponential, two bfloat16 (2^-17); sums of n
        # and up to n rescales and the merge in fp32; a weight below 2^-126 is 0 and the largest is 2^-8 or more; the result rounded to bfloat16; in denormals, sums of 32 keys rounded to 2^-149 eight times for
        # either half of the weights, which are 2^-8 and more, and the result to 2^-133
        err = 2.0 ** -16 + (below + s.abs().amax(-1, keepdim=True) + 6) * 2.0 ** -22 + (n + 16) * 2.0 ** -23
        bound = 2.0 ** -8 * (w @ v).abs() + (w * err + 2.0 ** -117) @ v.abs() + n * 2.0 ** -143 + 2.0 ** -133
        got = out[b].double()
        assert torch.isfinite(got).all()
        assert ((got - w @ v).abs() <= bound).all()


# lens, heads, splits: one key, a half page, one more, a page, one more; a split of more than 64 pages; an idle row; 16 heads, two groups of heads
@pytest.mark.parametrize("lens,heads,nsplit", [([1, 32, 33, 64, 65], 32, 1), ([96, 97, 128, 2, 31], 20, 2), ([4100, 0, 4096, 63], 32, 1), ([8300], 17, 2),
                                               ([700, 3], 16, 3), ([1000, 129], 40, 4), ([700, 1000, 129], 32, 1)])
def test_half_pages(lens, heads, nsplit):
    check(lens, heads, nsplit, lambda g, n: torch.randint(-16, 17, (n, 512), generator=g) * 0.25)


# 2 000 keys whose scores rise: as large as sums of 2 000 weights of 1 allow, and the smallest that bfloat16 holds whole
@pytest.mark.parametrize("power", [20, 112, -126])
@pytest.mark.parametrize("lens,heads,nsplit", [([2000, 40], 32, 1), ([2000, 700], 18, 4)])
def test_latents_of_any_size(lens, heads, nsplit, power):
    check(lens, heads, nsplit, lambda g, n: (1 + torch.randint(0, 64, (n, 512), generator=g) / 64) * (2.0 * torch.randint(0, 2, (n, 512), generator=g) - 1) * 2.0 ** power,
          q_latent=0)
