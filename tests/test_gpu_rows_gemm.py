"""Products of many rows in 16 bits (csrc/rows_gemm.h): every tile at its edges, with and without parts of k, and the calls that stay torch's.

The reference is float64 on the same operands.  A result is the fp32 sum of k exact products, rounded once: |error| <= u |y| + k 2^-23 (|x| . |w|),
u half an ulp of the type.  The silu unit rounds gate, up, the activation and the product: against float64 of the kernel's own rounded sums two
roundings are left.  The gelu unit rounds its product: the sums' own error comes in by slopes of at most 1.13 and |up|."""
import pytest
import torch
import torch.nn.functional as F

from triforce_amd import hip, ops_rows

pytestmark = pytest.mark.gpu
TILES = [(256, 256), (224, 256), (192, 256), (160, 256), (128, 256), (64, 128), (96, 64), (64, 64)]
UNIT = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _operands(rows, n, k, dtype, seed=0, ld=None):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(rows, ld or k, generator=g, device="cuda").to(dtype)[:, :k]
    return x, (torch.randn(n, k, generator=g, device="cuda") * k ** -0.5).to(dtype)


def _check_plain(y, x, w):
    want, k = x.double() @ w.double().T, x.shape[1]
    bound = UNIT[y.dtype] * want.abs() + k * 2.0 ** -23 * (x.double().abs() @ w.double().abs().T) + 2.0 ** -24
    assert bool(((y.double() - want).abs() <= bound).all())


def _launch(x, w, form, shape, splits, pad=8):
    """The entry point on a block of a larger one: (result, everything around it)."""
    rows, n, k = x.shape[0], w.shape[0], x.shape[1]
    n_out = n if form == ops_rows.PLAIN else n // 2
    out = torch.full((rows + 1, n_out + pad), 7.0, dtype=x.dtype, device="cuda")
    ws = torch.full((splits * rows * n + 4,), 7.0, device="cuda")
    f = hip.lib().tf_rows_gemm if x.dtype == torch.float16 else hip.tile_lib().tfl_rows_gemm
    hip.check(f(x.data_ptr(), x.stride(0), w.data_ptr(), out.data_ptr(), out.stride(0), ws.data_ptr(), ws.numel() - 4, rows, n, k, form, shape, splits,
                torch.cuda.current_stream().cuda_stream), "rows_gemm")
    assert bool((out[rows] == 7).all()) and bool((out[:, n_out:] == 7).all()) and bool((ws[splits * rows * n:] == 7).all())
    return out[:rows, :n_out]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", range(len(TILES)))
def test_every_tile_at_its_edges(shape, dtype):
    r, c = TILES[shape]
    unit = ops_rows.SILU_HALVES if dtype == torch.float16 else ops_rows.GELU_EIGHTS
    for rows, n, k, splits in ((1, 32, 64, 1), (r, c, 128, 1), (r + 1, c + 32, 192, 1), (r - 1, 2 * c - 32, 256, 2), (2 * r + 15, c + 64, 704, 4),
                               (3 * r - 16, 11 * c + 32, 320, 1), (17 * r, 32, 192, 3)):
        x, w = _operands(rows, n, k, dtype, seed=rows + n, ld=k + 8)
        y = _launch(x, w, ops_rows.PLAIN, shape, splits)
        _check_plain(y, x, w)
        got = _launch(x, w, unit, shape, splits).double()
        if unit == ops_rows.SILU_HALVES:
            z, u = y.double().chunk(2, 1)
            want = F.silu(z).to(dtype).double() * u
            bound = 3.1 * UNIT[dtype] * want.abs()
        else:
            z, u = (x.double() @ w.double().T).view(rows, n // 16, 2, 8).unbind(2)
            dz, du = (k * 2.0 ** -23 * (x.double().abs() @ w.double().abs().T)).view(rows, n // 16, 2, 8).unbind(2)
            act = F.gelu(z, approximate="tanh")
            want = (act * u).reshape(rows, n // 2)
            bound = 1.01 * UNIT[dtype] * want.abs() + (1.13 * u.abs() * dz + act.abs() * du + 1e-6 * (act * u).abs()).reshape(rows, n // 2)
        assert bool(((got - want).abs() <= bound + 2.0 ** -24).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_more_tiles_than_a_round_of_workgroups(dtype):
    for shape, rows, n, k in ((0, 4100, 8208, 128), (4, 2100, 9008, 192), (7, 1900, 5008, 64)):
        x, w = _operands(rows, n, k, dtype)
        _check_plain(ops_rows.product(x, w, plan=(shape, 1)), x, w)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_its_own_choice(dtype):
    for rows, n, k in ((33, 4096, 4096), (130, 12288, 4096), (513, 4096, 11008), (700, 6144, 1536), (1500, 2080, 576)):
        x, w = _operands(rows, n, k, dtype)
        assert ops_rows.takes(x, w)
        _check_plain(ops_rows.linear(x, w), x, w)


def test_infinities_and_nan_stay_in_their_rows():
    x, w = _operands(300, 512, 320, torch.float16)
    x = x.clone()
    clean = ops_rows.product(x, w)
    x[17, 3], x[40, 300] = float("inf"), float("nan")
    for splits in (1, 2):
        y = ops_rows.product(x, w, plan=(4, splits))
        assert bool(y[40].isnan().all()) and not bool(y[17].isfinite().any())
        rest = [i for i in range(300) if i not in (17, 40)]
        assert float((y[rest].double() - clean[rest].double()).abs().max()) < 4e-3 and bool(y[rest].isfinite().all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("plan", [(0, 1), (4, 1), (4, 2), (7, 1), (7, 3)])
def test_values_that_are_not_finite_through_the_units(dtype, plan):
    """Infinities, NaN and sums beyond the type's range: as the library's product and the unit's own launch treat them, and other rows untouched."""
    from triforce_amd import ops, ops_hybrid
    unit = ops_rows.SILU_HALVES if dtype == torch.float16 else ops_rows.GELU_EIGHTS
    x, w = _operands(300, 512, 320, dtype)
    plain, clean = ops_rows.product(x, w, plan=plan), ops_rows.product(x, w, unit, plan=plan)
    bad = x.clone()
    big = 6e4 if dtype == torch.float16 else 3e38
    bad[17, 3], bad[40, 300], bad[90, 5], bad[200] = float("inf"), float("nan"), -float("inf"), big * torch.sign(x[200])
    rows = [17, 40, 90, 200]
    rest = [i for i in range(300) if i not in rows]
    y, got = ops_rows.product(bad, w, plan=plan), ops_rows.product(bad, w, unit, plan=plan)
    assert torch.equal(y[rest], plain[rest]) and torch.equal(got[rest], clean[rest])
    assert bool(y[40].isnan().all()) and not bool((y[17].isfinite() | y[90].isfinite()).any()) and bool(got[40].isnan().all())
    library = F.linear(bad, w)
    apart = ops.silu_mul(library) if unit == ops_rows.SILU_HALVES else ops_hybrid.glu(library)
    for a, b in ((y[[17, 40, 90]], library[[17, 40, 90]]), (got[[17, 40, 90]], apart[[17, 40, 90]])):
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isposinf(), b.isposinf()) and torch.equal(a.isneginf(), b.isneginf())
    # the unit of the kernel's own sums, where they leave the type's range or do not
    own = ops.silu_mul(y) if unit == ops_rows.SILU_HALVES else ops_hybrid.glu(y)
    assert torch.equal(got[200].isnan(), own[200].isnan()) and torch.equal(got[200].isinf(), own[200].isinf())


def test_what_the_kernel_does_not_take_is_torchs():
    for dtype in (torch.float16, torch.bfloat16):
        x, w = _operands(96, 256, 256, dtype)
        odd = [(x.t().contiguous().t(), w), (x, w.t().contiguous().t()), (x[:, :200], w[:, :200].contiguous()), (x, w[:250]), (x[0], w), (x[None], w),
               (x[:1].expand(96, 256), w), (torch.cat([x, x], 1)[:, 4:260], w)]
        for a, b in odd:
            assert not ops_rows.takes(a, b)
            assert torch.equal(ops_rows.linear(a, b), F.linear(a, b))
        p = torch.nn.Parameter(w.clone())
        y = ops_rows.linear(x, p)
        y.sum().backward()
        assert p.grad is not None
        with torch.inference_mode():
            assert ops_rows.takes(x, p)
        v = torch.func.vmap(lambda a: ops_rows.linear(a, w))(x.view(2, 48, 256))
        assert torch.allclose(v.reshape(96, 256).float(), F.linear(x, w).float(), atol=0.05)


def test_captured_with_parts_of_k():
    x, w = _operands(200, 4096, 11008, torch.float16)
    assert ops_rows._plan(torch.float16, 200, 4096, 11008)[1] > 1
    want = ops_rows.linear(x, w)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = ops_rows.linear(x, w)
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
        assert torch.equal(ops_rows.linear(x, w), want)


def test_products_that_are_the_librarys(monkeypatch):
    """linear at sizes that were timed (the rule itself: test_sizes_of_the_kernel_and_of_the_library)."""
    taken = []
    monkeypatch.setattr(ops_rows, "product", lambda x, w, form=ops_rows.PLAIN, plan=None: taken.append((x.shape[0], w.shape[0], form)) or F.linear(x, w))
    wide, narrow = (torch.zeros(n, 4096, dtype=torch.float16, device="cuda") for n in (32000, 768))
    for rows in (40, 128, 700):
        x = torch.zeros(rows, 4096, dtype=torch.float16, device="cuda")
        ops_rows.linear(x, wide)
        ops_rows.linear(x, narrow)
        ops_rows.glu_linear(x, wide, ops_rows.SILU_HALVES)
        assert ops_rows.glu_linear(x, wide, ops_rows.GELU_EIGHTS) is None
    assert taken == [(40, 32000, 0), (40, 32000, 1), (128, 32000, 1), (700, 32000, 0), (700, 768, 0), (700, 32000, 1)]
