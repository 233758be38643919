"""Lengths, positions and cache rows of a decode step made by the step's first launch, against the launch of their own."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _prep(rows, columns, gen):
    lens = torch.randint(-1, columns * 64 + 3, (rows,), generator=gen, device="cuda", dtype=torch.int32)          # idle rows, and rows past their table
    table = torch.randint(0, 1000, (rows, columns + 2), generator=gen, device="cuda", dtype=torch.int32)[:, :columns]
    return [lens, table, *(torch.full((rows,), 77, dtype=torch.int32, device="cuda") for _ in range(3))]


# widths of every form of the row kernels, one row and more than a workgroup's threads of them
@pytest.mark.parametrize("rows,width,dtype", [(1, 4096, torch.bfloat16), (33, 256, torch.bfloat16), (300, 1024, torch.float32), (1100, 2048, torch.bfloat16),
                                              (70, 4096, torch.float32), (5, 8192, torch.bfloat16), (300, 4096, torch.bfloat16)])
def test_first_launch(rows, width, dtype):
    from triforce_amd import ops_hybrid as oh, ops_latent as ol
    gen = torch.Generator(device="cuda").manual_seed(rows + width)
    embed, ids = torch.randn(100, width, generator=gen, device="cuda").to(dtype), torch.randint(0, 100, (rows,), generator=gen, device="cuda")
    w, step, ew = (torch.randn(width, generator=gen, device="cuda") for _ in range(3))
    for streams in (0, 1, 3, 7, 16):
        mine, other = _prep(rows, 5, gen), None
        other = [mine[0].clone(), mine[1]] + [t.clone() for t in mine[2:]]
        shape = (rows, streams, width) if streams else (rows, width)
        x, y = (torch.full(shape, 3.0, device="cuda") for _ in range(2))
        if streams:
            u = torch.randn(streams, generator=gen, device="cuda")
            call = lambda into, prep: oh.connect(into, u, w, 1e-5, width, dtype, embed=embed, ids=ids, embed_w=ew, octets=True, prep=prep)          # noqa: E731
        else:
            call = lambda into, prep: ol.finish(into, w, 1e-5, width, dtype, embed=embed, ids=ids, step=step, octets=True, prep=prep)               # noqa: E731
        h = call(x, mine)
        want = call(y, None)
        ol.decode_prep(*other)
        assert torch.equal(h, want) and torch.equal(x, y) and all(torch.equal(a, b) for a, b in zip(mine, other))
