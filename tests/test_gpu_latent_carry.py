"""Query to latent with another product's panels beside it, in one launch (tfl_gemm_carry)."""
import pytest
import torch

from triforce_amd import ops_latent as ol

pytestmark = pytest.mark.gpu


class Geom:
    def __init__(self, H, N, C, R):
        self.H, self.N, self.C, self.R = H, N, C, R


@pytest.mark.parametrize("rows,H,N,C,R,n,k,k0,k1", [
    (1, 32, 128, 512, 64, 4096, 8192, 4096, 8192),
    (2, 17, 32, 512, 64, 4096, 4096, 4064, 4096),             # one chunk: seven waves have none
    (3, 20, 160, 512, 64, 5120, 8192, 3072, 8192),            # five chunks over four waves, 320 carried panels
    (15, 32, 128, 64, 0, 4112, 2048, 0, 2048),                # a head of one pair of pairs, 257 carried panels
    (16, 1, 96, 192, 32, 8192, 2560, 32, 2528),
    (16, 32, 128, 512, 64, 4096, 11008, 4864, 11008),
])
def test_carry(rows, H, N, C, R, n, k, k0, k1):
    gen = torch.Generator(device="cuda").manual_seed(rows + k)
    make = lambda *s: torch.randn(*s, generator=gen, device="cuda").bfloat16()                                     # noqa: E731
    g = Geom(H, N, C, R)
    qn, w, wide, act = make(rows, H, N), ol.TileWeight(make(H, C, N), packed_only=True), make(n, k), make(rows, k)
    x = torch.randn(rows, n, generator=gen, device="cuda")
    wt = ol.TileWeight(wide, packed_only=True)
    if not wt.chunk_major:                                    # (panels that the rule for whole products leaves panel by panel)
        wt.chunk_major, wt.packed = True, ol.pack_tiles(wide.unsqueeze(0), True)
    octs = act.view(rows, k // 8, 8).transpose(0, 1).contiguous()
    want, got = (torch.full((rows, H, C + R), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    ol.query_to_latent(qn, w, want, g)
    have = x.clone()
    ol.query_to_latent(qn, w, got, g, ol.part_of(octs, wt, have, k0, k1))
    if H * C // 16 > 512:
        assert torch.equal(got, want)                         # the same sums in the same order
    q64, w64 = qn.double().cpu().transpose(0, 1).contiguous(), w_rows(w, H, C, N).transpose(1, 2).contiguous()
    exact, mag = (torch.bmm(a, b).transpose(0, 1) for a, b in ((q64, w64), (q64.abs(), w64.abs())))
    # one rounding to bfloat16 of fp32 sums of exact products: error below (chunks of 32 + waves) ulp of the sum of magnitudes
    bound = 2.0 ** -8 * exact.abs() + mag * 2.0 ** -23 * 16
    assert ((got[..., :C].double().cpu() - exact).abs() <= bound).all() and (got[..., C:] == 7).all()
    a64, w64 = act[:, k0:k1].double(), wide[:, k0:k1].double()
    mag = x.double().abs() + a64.abs() @ w64.abs().T
    assert ((have.double() - (x.double() + a64 @ w64.T)).abs() <= mag * 2.0 ** -23 * 16).all()
    again = x.clone()
    ol.query_to_latent(qn, w, got, g, ol.part_of(octs, wt, again, k0, k1))
    assert torch.equal(again, have)


def w_rows(w, H, C, N):
    """[H, C, N] in float64 of a panel-major packed weight."""
    p = w.packed.view(H, C // 16, N // 32, 4, 16, 8).double().cpu()                     # panel, chunk, quarter of a chunk, row, entry
    return p.permute(0, 1, 4, 2, 3, 5).reshape(H, C, N)
