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
