"""A workspace of the decode attention may begin at any float: the same bits from every entry, and nothing written beside it."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("H, sq, sk, nsplit", [(4, 1, 300, 3), (8, 7, 4103, 8), (5, 16, 700, 2), (3, 18, 1500, 5), (32, 32, 2100, 1), (2, 9, 5000, 20)])
def test_any_float_is_a_beginning(D, H, sq, sk, nsplit):
    from triforce_amd import hip
    L = hip.lib()
    g = torch.Generator(device=DEV).manual_seed(sk)
    q, k, v = (torch.randn(*s, generator=g, device=DEV).half() for s in ((sq, H, D), (H, sk, D), (H, sk, D)))
    tickets = torch.zeros(128, dtype=torch.int32, device=DEV)
    floats = L.tf_attn_decode_ws_floats(H, sq, D, nsplit)
    stream = torch.cuda.current_stream().cuda_stream

    def run(entry, first):
        out, block = torch.full((sq, H * D), 3.0, device=DEV).half(), torch.full((floats + 8,), 5.0, device=DEV)
        ws = block[first:first + floats]
        same = [D, sk * D, sq, sk, None, H, D, D ** -0.5, nsplit, ws.data_ptr(), floats]
        head = [t.data_ptr() for t in (q, k, v, out)]
        rc = L.tf_attn_decode(*head, *same, stream) if entry == "plain" else \
            L.tf_attn_decode_fused(*head, *same, tickets.data_ptr(), stream) if entry == "fused" else \
            L.tf_attn_decode_act(*head, H * D, 8, *same, tickets.data_ptr() if entry == "act" else None, stream)
        assert rc == 0
        assert bool((block[:first] == 5).all()) and bool((block[first + floats:] == 5).all()) and bool((tickets == 0).all())
        return out
    want = run("plain", 0)
    s = torch.einsum("qhd,hkd->hqk", q.cpu().float(), k.cpu().float()) * D ** -0.5
    s.masked_fill_(torch.arange(sk)[None] > sk - sq + torch.arange(sq)[:, None], float("-inf"))
    exact = torch.einsum("hqk,hkd->qhd", s.softmax(-1), v.cpu().float()).reshape(sq, H * D)
    assert float((want.cpu().float() - exact).abs().max()) < 4e-3                  # (fp16 results up to 4, an fp16 part of each weight)
    for entry in ("plain", "fused", "act", "act2"):
        for first in (0, 1, 2, 3):
            assert torch.equal(run(entry, first), want), (entry, first)
