"""Tensor-level wrappers over the C ABI that the batch-served model families share (include/triforce_tile.h): padding and packing
of weights, activation blocks, the skinny GEMM, the set-up of a decode step.

Same rules as ops.py: torch owns the memory and the stream, every function validates its tensors and enqueues hand-written
gfx950 kernels on torch's current stream; no CPU path exists.  The element type is bfloat16 or float32 and follows the tensors.
"""
import ctypes

import torch

from . import hip, ops_rows

PAGE = hip.TFL_PAGE
_CODE = {torch.bfloat16: 0, torch.float32: 1}


def pad32(n):
    return (n + 31) // 32 * 32


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _p(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def _need(*ts):
    for t in ts:
        if t is not None:
            if not t.is_cuda:
                raise hip.TriforceHipError("triforce_amd ops need HIP device tensors (no CPU fallback)")
            assert t.is_contiguous() or t.stride(-1) == 1


def _f32(*ts):
    assert all(t is None or t.dtype == torch.float32 for t in ts)


def _i32(*ts):
    assert all(t is None or t.dtype == torch.int32 for t in ts)


def grow(t, *shape):
    """Zero-pad the trailing edge of every dimension to ``shape``."""
    if tuple(t.shape) == tuple(shape):
        return t
    out = torch.zeros(*shape, dtype=t.dtype, device=t.device)
    out[tuple(slice(0, n) for n in t.shape)] = t
    return out


def pack_tiles(w, chunk_major=False):
    """[.., n, k] -> MFMA operand order [.., n/16, k/32, 4 (k octet), 16 (row), 8]: one 16x32 tile is one wavefront load.
    ``chunk_major``: the tiles as [.., k/32, n/16]."""
    n, k = w.shape[-2:]
    assert n % 16 == 0 and k % 32 == 0
    lead = w.shape[:-2]
    d = len(lead)
    order = (d + 2, d) if chunk_major else (d, d + 2)
    return w.reshape(*lead, n // 16, 16, k // 32, 4, 8).permute(*range(d), *order, d + 3, d + 1, d + 4).contiguous()


def shares_panels(n, k, raw=0):
    """Does the one-workgroup-per-CU form of the skinny kernel (share_gemm in csrc/tile_gemm.hip) take n outputs in bfloat16, the first
    ``raw`` of them with sums of squares?  A panel or more per CU and at most eight; left-over panels are dealt in fours of rows, where
    sums of squares need whole ones.  k from 2 048 on: a shorter one is over before the form's look-ahead pays (4 096 x 256 at 32
    rows 4.6 us with a workgroup per panel, 6.4 with one per CU; 6 144 x 1 536 10.0 and 11.1)."""
    panels = n // 16
    whole, left = panels // 256, panels % 256
    return k >= 2048 and 256 <= panels <= 2048 and (left == 0 or left > 192 or 256 * whole * 16 >= raw)


class TileWeight:
    """A (groups of) [n, k] weight(s): packed for the skinny kernel and, unless ``packed_only``, row-major for the prefill's products
    of many rows (linear_rows).  Weights of the one-workgroup-per-CU form are packed chunk-major, the layout it streams; the workgroup-per-panel form
    reads that one too, but up to 10 % slower (128 256 x 4 096 at 8 rows 171 -> 181 us, a projection of 17 216 with 16 480 raw 27.4 -> 30.1
    at one row), so its weights stay panel by panel.  ``raw``: outputs of an input projection that come with sums of squares; ``per_panel``:
    the weight of a product that only the workgroup-per-panel form has (query, token gate)."""

    def __init__(self, w, packed_only=False, raw=0, per_panel=False):
        w3 = w if w.dim() == 3 else w.unsqueeze(0)
        self.groups, self.n, self.k = w3.shape
        self.chunk_major = self.groups == 1 and w.dtype == torch.bfloat16 and not per_panel and shares_panels(self.n, self.k, raw)
        self.packed = pack_tiles(w3, self.chunk_major)
        self.w = None if packed_only else w.contiguous()
        self.dtype, self.device = w.dtype, w.device

    def nbytes(self):
        return sum(t.numel() * t.element_size() for t in (self.packed, self.w) if t is not None)

    def matmul(self, x):
        """x . W^T over many rows (prefill)."""
        assert self.groups == 1 and x.dtype == self.dtype
        return linear_rows(x, self.w)

    def glu_matmul(self, x):
        """gelu_tanh(gate) * up of x . W^T over many rows in bfloat16, the weight interleave_glu(gate, up); None where it is not one launch."""
        assert self.groups == 1 and x.dtype == self.dtype
        return ops_rows.glu_linear(x, self.w, ops_rows.GELU_EIGHTS)


def empty_act(rows, k, dtype, device):
    """Octet-major activation block [k/8, rows, 8] (include/triforce_tile.h); a 2-D tensor is a row-major one."""
    return torch.empty(k // 8, rows, 8, dtype=dtype, device=device)


def act_rows(x):
    """Row-major copy of an activation block."""
    return x if x.dim() == 2 else x.permute(1, 0, 2).reshape(x.shape[1], -1)


def _lay(x):
    """(rows, k, ld, oct) of an activation block."""
    if x.dim() == 3:
        assert x.shape[2] == 8 and x.is_contiguous()
        return x.shape[1], 8 * x.shape[0], 8, 8 * x.shape[1]
    return x.shape[0], x.shape[1], x.stride(0), 8


def _tail(x, k):
    """The columns from k on."""
    return x[k // 8:] if x.dim() == 3 else x[:, k:]


def part_of(act, wt, x, k0, k1):
    """x (fp32) += act . W^T over the columns k0 .. k1 - 1 of both, as a product that another launch carries (_gemm, tfl_attn_decode_beside): the octet-major
    block act, chunk-major weights.  The tensors have to outlive the launch's enqueueing only."""
    _need(act, x)
    _f32(x)
    assert act.dim() == 3 and act.is_contiguous() and act.dtype == wt.dtype == torch.bfloat16 and wt.chunk_major
    rows = act.shape[1]
    assert act.shape[0] == wt.k // 8 and x.shape == (rows, wt.n) and x.is_contiguous() and 0 <= k0 < k1 <= wt.k and k0 % 32 == 0 and k1 % 32 == 0
    a = hip.TflGemm()
    a.wp, a.x, a.out_f = wt.packed.data_ptr() + 2 * k0 * wt.n, act[k0 // 8:].data_ptr(), x.data_ptr()
    a.rows, a.n, a.k, a.groups, a.chunk_major, a.ld_f = rows, wt.n, k1 - k0, 1, 1, x.stride(0)
    a.ld_x, a.x_oct, a.t_oct = 8, 8 * rows, 8
    return a


def _gemm(wt, x, epi, rows, carried=None, **kw):
    a = hip.TflGemm()
    a.wp, a.x = wt.packed.data_ptr(), x.data_ptr()
    a.rows, a.n, a.k, a.groups = rows, wt.n, wt.k, wt.groups
    a.x_oct = a.t_oct = 8
    a.chunk_major = int(wt.chunk_major)
    for name, v in kw.items():
        setattr(a, name, v.data_ptr() if isinstance(v, torch.Tensor) else v)
    if carried is not None:
        assert wt.dtype == torch.bfloat16 and epi == "latent"
        hip.check(hip.tile_lib().tfl_gemm_carry(ctypes.byref(a), ctypes.byref(carried), _stream()), "tfl_gemm_carry")
        return
    hip.check(hip.tile_lib().tfl_gemm(ctypes.byref(a), _CODE[wt.dtype], hip.TFL_EPI[epi], _stream()), "tfl_gemm " + epi)


def linear_f32(x, wt, n_real, out=None):
    """fp32 x . W^T: x [rows, k] of the weight's type."""
    _need(x)
    rows, k, ld, octet = _lay(x)
    assert x.dtype == wt.dtype and k == wt.k
    if out is None:
        out = torch.empty(rows, n_real, dtype=torch.float32, device=x.device)
    assert out.dtype == torch.float32 and out.shape[0] == rows and out.shape[1] >= n_real and out.stride(1) == 1
    _gemm(wt, x, "f32", rows, ld_x=ld, x_oct=octet, out_f=out, ld_f=out.stride(0), n_real=n_real)
    return out


def gelu_glu_linear(x, wt):
    """gelu_tanh(gate) * up of one product; wt: interleave_glu(gate, up) packed.  Returns an octet-major block."""
    _need(x)
    rows, k, ld, octet = _lay(x)
    assert x.dtype == wt.dtype and k == wt.k and wt.n % 16 == 0
    out = empty_act(rows, wt.n // 2, wt.dtype, x.device)
    _gemm(wt, x, "glu", rows, ld_x=ld, x_oct=octet, out_t=out, ld_t=8, t_oct=8 * rows)
    return out


def interleave_glu(gate, up):
    """[n, k] twice -> [2n, k] in blocks of 8 gate rows | 8 up rows (both halves of an output octet meet in one 16-row panel)."""
    n, k = gate.shape
    return torch.stack([gate.view(n // 8, 8, k), up.view(n // 8, 8, k)], 1).reshape(2 * n, k)


def linear_rows(x, w):
    """x . W^T over many rows (prefill), w [n, k] contiguous: in 16 bits ops_rows.linear, in float32 the library GEMM, and for large products
    split_linear.  Its tiles are 256 x 128: from 256 rows and 2^32 multiply-adds on it is the faster one (256 x 4 096 x 4 096 87 -> 68 us, 2 048 x 2 048 x 1 024
    68 -> 65, 700 x 22 016 x 4 096 917 -> 590), below that it leaves CUs idle (300 x 6 144 x 1 536 47 -> 52, 64 x 22 016 x 4 096
    117 -> 124), as with few results of a long k, whose parts are eight at most (2^19 results: 385 x 1 136 x 15 104 117 -> 135, 512 x 1 136
    160 -> 143), and with k below 96 the cut and the results are all there is (1 030 x 65 536 x 64 111 -> 127).  At k = 96 the two are as fast on the
    whole (300 x 151 552 144 -> 103, 700 x 65 536 100 -> 92, 1 030 x 65 536 143 -> 153, 262 144 x 1 024 505 -> 602), but the library is three times as far off
    (normals 1.8e-7 against 5.8e-8), so it starts there.  Up to k = 65 536 its error is a tenth to a half of the library's; at 2^20, with as few parts,
    the two are equal."""
    rows, (n, k) = x.shape[0], w.shape
    if x.dtype == w.dtype == torch.float32 and x.dim() == 2 and x.shape[1] == k and 256 <= rows <= 1 << 24 and rows * n * k >= 1 << 32 \
            and rows * n > 1 << 19 and n % 16 == 0 and k % 32 == 0 and 96 <= k <= 1 << 16 and x.device == w.device and ops_rows.unwatched(x, w) \
            and w.is_contiguous() and w.data_ptr() % 16 == 0:
        return split_linear(x, w)
    return ops_rows.linear(x, w)


def split_linear(x, w, splits=0):
    """x . W^T in float32 precision on the bfloat16 matrix cores: x [rows, k], w [n, k] contiguous."""
    _need(x, w)
    _f32(x, w)
    (rows, k), n = x.shape, w.shape[0]
    assert w.shape[1] == k and w.is_contiguous()
    if x.stride(1) != 1 or x.stride(0) % 4 or x.stride(0) < k or x.data_ptr() % 16:
        x = x.clone(memory_format=torch.contiguous_format)
    L = hip.tile_lib()
    out = torch.empty(rows, n, dtype=torch.float32, device=x.device)
    ws = torch.empty(L.tfl_split_gemm_ws_floats(rows, n, k, splits), dtype=torch.float32, device=x.device)
    hip.check(L.tfl_split_gemm(_p(w), _p(x), x.stride(0), _p(out), n, _p(ws), ws.numel(), rows, n, k, splits, _stream()), "tfl_split_gemm")
    return out


def set_pages(table, entries):
    """table[row, column] = page for every (row, column, page) of a host list; the entries travel as kernel arguments."""
    _need(table)
    _i32(table)
    for at in range(0, len(entries), hip.TFL_MAX_ENTRIES):
        part = entries[at:at + hip.TFL_MAX_ENTRIES]
        flat = (ctypes.c_int32 * (3 * len(part)))(*(v for e in part for v in e))
        hip.check(hip.tile_lib().tfl_set_pages(_p(table), table.stride(0), table.shape[0], table.shape[1], flat, len(part), _stream()), "tfl_set_pages")


def decode_prep_of(lens, table, pos, slot, klen):
    """decode_prep() as an argument of a step's first launch (ops_latent.finish, ops_hybrid.connect)."""
    _need(lens, table, pos, slot, klen)
    _i32(lens, table, pos, slot, klen)
    rows = lens.numel()
    assert table.shape[0] == rows and table.stride(1) == 1 and pos.numel() == rows and slot.numel() == rows and klen.numel() == rows
    return hip.TflDecodePrep(_p(lens), _p(table), _p(pos), _p(slot), _p(klen), table.stride(0), table.shape[1], rows)


def decode_prep(lens, table, pos, slot, klen):
    _need(lens, table, pos, slot, klen)
    _i32(lens, table, pos, slot, klen)
    rows = lens.numel()
    assert table.shape[0] == rows and pos.numel() == rows and slot.numel() == rows and klen.numel() == rows
    hip.check(hip.tile_lib().tfl_decode_prep(_p(lens), _p(table), table.stride(0), table.shape[1], _p(pos), _p(slot), _p(klen), rows,
                                               _stream()), "tfl_decode_prep")
