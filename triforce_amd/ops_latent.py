"""Tensor-level wrappers over the latent-attention C ABI (include/triforce_latent.h, on top of ops_tile.py).

Same rules as ops.py: torch owns the memory and the stream, every function validates its tensors and enqueues hand-written
gfx950 kernels on torch's current stream; no CPU path exists.  The element type is bfloat16 or float32 and follows the
tensors.  Call these as ``ops_latent.<name>(...)``.
"""
import ctypes
import functools

import torch

from . import hip
from .ops_tile import (_CODE, PAGE, TileWeight, _f32, _gemm, _i32, _lay, _need, _p, _stream, _tail, act_rows, decode_prep, decode_prep_of, empty_act, linear_rows,  # noqa: F401
                       linear_f32, pack_tiles, pad32, part_of)

class Finish:
    """finish() of decode rows that the product which reads them makes for itself (tfl_finish_gemm): stands for its activation block; ``out`` is the
    updated residual."""

    def __init__(self, x, norm_w, eps, width, y, y_w, step=None):
        _need(x, norm_w, y, y_w, step)
        _f32(x, norm_w, y, y_w, step)
        rows, wp = x.shape
        assert x.is_contiguous() and norm_w.numel() == wp == y_w.numel() and y.shape == (rows, wp) and y.stride(1) == 1 and (step is None or step.numel() == wp)
        self.out, self.dtype, self.is_cuda, self.shape = torch.empty_like(x), torch.bfloat16, True, (rows, wp)
        self.device, self.keep = x.device, (x, norm_w, y, y_w, step)
        f = self.c = hip.TflFinish()
        f.y, f.y_w, f.step, f.norm_w, f.x, f.x_out = y.data_ptr(), y_w.data_ptr(), None if step is None else step.data_ptr(), norm_w.data_ptr(), x.data_ptr(), self.out.data_ptr()
        f.ld_y, f.width, f.width_real, f.eps = y.stride(0), wp, width, eps

    @staticmethod
    def takes(rows, wp, wt, epi, n_raw=0):
        """Does the product of wt with this epilogue ("in", "f32") make ``rows`` rows itself?"""
        return wt.chunk_major and wt.dtype == torch.bfloat16 and wt.k == wp and hip.latent_lib().tfl_finish_gemm_takes(rows, wp, wt.n, wt.k, hip.TFL_EPI[epi], n_raw) == 1

    def product(self, wt, epi, **kw):
        a = hip.TflGemm()
        a.wp, a.rows, a.n, a.k, a.groups, a.x_oct, a.t_oct, a.ld_x, a.chunk_major = wt.packed.data_ptr(), self.shape[0], wt.n, wt.k, 1, 8, 8, 8, 1
        for name, v in kw.items():
            setattr(a, name, v.data_ptr() if isinstance(v, torch.Tensor) else v)
        hip.check(hip.latent_lib().tfl_finish_gemm(ctypes.byref(self.c), ctypes.byref(a), hip.TFL_EPI[epi], _stream()), "tfl_finish_gemm " + epi)


def input_projection(h, wt, n_raw, q_norm, act, act_off):
    """All projections of the layer's one norm (h, act: activation blocks, h also a Finish).  Returns (raw fp32 [rows, n_raw], per-panel sums of
    squares, the first len(q_norm) outputs times q_norm as an octet-major block); gelu of the outputs behind n_raw goes to the
    columns of act from act_off on."""
    inside = isinstance(h, Finish)
    _need(None if inside else h, act)
    rows, k, ld, octet = (*h.shape, 8, 8) if inside else _lay(h)
    act_rows_, act_k, act_ld, act_oct = _lay(act)
    assert h.dtype == wt.dtype == act.dtype and k == wt.k and act_rows_ == rows and act_k >= act_off + wt.n - n_raw and act_off % 8 == 0
    raw = torch.empty(rows, n_raw, dtype=torch.float32, device=h.device)
    ss = torch.empty(rows, n_raw // 16, dtype=torch.float32, device=h.device)
    _f32(q_norm)
    xq = empty_act(rows, q_norm.numel(), wt.dtype, h.device)
    tail = _tail(act, act_off) if wt.n > n_raw else act
    to = dict(out_f=raw, ld_f=n_raw, ss_out=ss, ss_ld=n_raw // 16, n_raw=n_raw, out_t=tail, ld_t=act_ld, t_oct=act_oct, out_t2=xq, norm_w=q_norm,
              n_scaled=q_norm.numel())
    if inside:
        h.product(wt, "in", **to)
    else:
        _gemm(wt, h, "in", rows, ld_x=ld, x_oct=octet, **to)
    return raw, ss, xq


def finish_logits(h, wt, n_real):
    """linear_f32 of a Finish."""
    assert h.dtype == wt.dtype
    out = torch.empty(h.shape[0], n_real, dtype=torch.float32, device=h.device)
    h.product(wt, "f32", out_f=out, ld_f=n_real, n_real=n_real)
    return out


def query_and_append(xq, raw, ss, wt, g, kv_norm, eps, rope, pos, slot, cache):
    """Second stage of a decode step: the weighted query latent xq up-projected and scaled by its norm (returned as unrotated
    [rows, H, N] and [rows, H, C + R] with the rotated part filled in), raw's key latent normalised / rotated into the cache rows
    ``slot``.  g: LatentGeom."""
    _need(xq, raw, ss, cache, pos, slot)
    _i32(pos, slot)
    _f32(raw, ss, kv_norm)
    rows, k, ld, octet = _lay(xq)
    assert k == g.Q and xq.dtype == wt.dtype and raw.shape[0] == rows
    assert wt.n == g.H * (g.N + g.R) and wt.k == g.Q and cache.dtype == wt.dtype and cache.shape[1] == g.C + g.R and cache.is_contiguous()
    assert pos.numel() == rows and slot.numel() == rows and raw.stride(0) == raw.shape[1] >= g.Q + g.C + g.R
    qn = torch.empty(rows, g.H, g.N, dtype=wt.dtype, device=raw.device)
    q = torch.empty(rows, g.H, g.C + g.R, dtype=wt.dtype, device=raw.device)
    kv = raw[:, g.Q:]
    _gemm(wt, xq, "query", rows, ld_x=ld, x_oct=octet, ss_in=ss, ss_n=g.Q // 16, ss_ld=ss.shape[1],
          k_real=g.q_real, eps=eps, out_t=q, out_t2=qn, pos=pos, cos=rope.cos, sin=rope.sin, half=rope.half, max_pos=rope.max_pos,
          H=g.H, N=g.N, R=g.R, C=g.C, c_real=g.c_real, kv_raw=kv, ld_kv=raw.stride(0), kv_norm_w=kv_norm, cache=cache,
          cache_rows=cache.shape[0], slot=slot)
    return qn, q


def query_to_latent(qn, wt, q, g, carried=None):
    """q[:, h, :C] = qn[:, h] . Wuk_h (wt: groups of [C, N]).  ``carried``: a product (part_of) in the same launch."""
    _need(qn, q)
    rows = qn.shape[0]
    assert (wt.groups, wt.n, wt.k) == (g.H, g.C, g.N) and qn.dtype == q.dtype == wt.dtype
    _gemm(wt, qn, "latent", rows, carried, ld_x=g.H * g.N, x_group=g.N, out_t=q, H=g.H, C=g.C, R=g.R)
    return q


def latent_to_value(ol, wt, raw, gate_off, act, g):
    """Columns h*V .. of the activation block act = (ol[:, h] . Wuv_h^T) * sigmoid(gate).  ``ol``: a tensor, or Splits that it merges."""
    _need(ol.ws if isinstance(ol, Splits) else ol, raw, act)
    rows, (act_rows_, act_k, act_ld, act_oct) = ol.shape[0], _lay(act)
    assert (wt.groups, wt.n, wt.k) == (g.H, g.V, g.C) and ol.dtype == act.dtype == wt.dtype and act_rows_ == rows and act_k >= g.H * g.V
    assert raw.shape[1] >= gate_off + g.H * g.V
    if isinstance(ol, Splits):
        a = hip.TflGemm()
        a.wp, a.gate, a.out_t, a.ld_gate, a.ld_t, a.t_oct = wt.packed.data_ptr(), raw[:, gate_off:].data_ptr(), act.data_ptr(), raw.stride(0), act_ld, act_oct
        a.rows, a.n, a.k, a.groups, a.chunk_major = rows, wt.n, wt.k, wt.groups, int(wt.chunk_major)
        hip.check(hip.latent_lib().tfl_latent_value(_p(ol.ws), ol.ws.numel(), ol.nsplit, ctypes.byref(a), _stream()), "tfl_latent_value")
        return
    _gemm(wt, ol, "gated", rows, ld_x=g.H * g.C, x_group=g.C, gate=raw[:, gate_off:], ld_gate=raw.stride(0), out_t=act,
          ld_t=act_ld, t_oct=act_oct)


def add_linear(act, wt, x, want_copy=False, k=None, also=None):
    """x (fp32) += act . W^T, over the first ``k`` columns of both if given (chunk-major weights); returns the sum as an octet-major
    block of act's type when ``want_copy``.  ``also``: fp32 [parts][rows][n] to be added too (attn_decode_beside_parts)."""
    _need(act, x, also)
    _f32(x, also)
    rows, have, ld, octet = _lay(act)
    assert act.dtype == wt.dtype and have == wt.k and x.shape == (rows, wt.n) and x.is_contiguous()
    assert k is None or (wt.chunk_major and 0 < k <= have and k % 32 == 0)
    assert also is None or (also.shape[1:] == x.shape and also.is_contiguous() and 1 <= also.shape[0] <= 4)
    xt = empty_act(rows, wt.n, wt.dtype, x.device) if want_copy else None
    _gemm(wt, act, "residual", rows, ld_x=ld, x_oct=octet, out_f=x, ld_f=x.stride(0), k=have if k is None else k,
          **(dict(out_t=xt, ld_t=8, t_oct=8 * rows) if want_copy else {}), **(dict(also=also, n_also=also.shape[0]) if also is not None else {}))
    return xt


def token_gate_linear(x, wt, table, ids, n_real):
    """gelu(x . W^T) * table[ids]: x an activation block, table a column slice [vocab, n_real] of the token-side embedding."""
    _need(x, table, ids)
    rows, k, ld, octet = _lay(x)
    assert ids.dtype == torch.int64 and ids.numel() == rows and k == wt.k and x.dtype == table.dtype == wt.dtype and table.shape[1] == n_real
    out = torch.empty(rows, wt.n, dtype=wt.dtype, device=x.device)
    _gemm(wt, x, "token", rows, ld_x=ld, x_oct=octet, out_t=out, ld_t=wt.n, ids=ids, tok_table=table, ld_tok=table.stride(0),
          vocab=table.shape[0], n_real=n_real)
    return out


TOKEN_SIDE_ROWS = 10


def token_side_pays(rows, width, side):
    """Is the gate's K cut over the grid the faster way?  Every workgroup of the projection then reads all parts of all rows, which has to be little beside what the gate
    gains by more CUs.  us of the two launches, panels -> parts, at 1 / 4 / 10 rows: side 64 of 1 024 6.3 / 6.3 / 6.3 -> 5.6 / 5.8 / 6.2, of 4 096 8.4 / 8.4 / 8.9 -> 6.2 / 6.4 / 6.6;
    128 of 1 024 6.4 / 6.7 / 6.8* -> 6.0 / 6.4 / 7.2, of 8 192 11.9 / 12.1 / 13.2 -> 7.8 / 8.6 / 10.2; 256 of 2 048 7.6* / 7.9* / 8.2* -> 7.2 / 8.0 / 9.5, of 4 096 9.1 / 9.4 / 9.9 ->
    7.4 / 8.2 / 9.7, of 6 144 11.8 / 12.2 / 13.1* -> 9.5 / 11.2 / 14.2; 512 of 4 096 9.4* / 9.7* / 10.2* -> 9.6 / 10.9 / 13.9, 1 024 10.4* / 10.7* / 11.0* -> 15.2 / 16.8 / 24.0 (*: stays
    panels).  Eight steps of six layer runs, side 256 of 4 096, 1 row 4 296 -> 4 187, 8 4 968 -> 4 925, 12 the same, 16 5 378 -> 5 402."""
    if rows > TOKEN_SIDE_ROWS or side > 256 or (side > 128 and width < 4096):
        return False
    rounds = 1 if width <= 4096 or width % 4096 == 0 else 2          # (of the projection's workgroups over the CUs, and one that is half empty)
    return 8 * rows * side * rounds <= 5 * width


def token_side(x, gate, proj, table, ids, n_real, width):
    """linear_f32(token_gate_linear(x, gate, table, ids, n_real), proj, width), for a few rows of bfloat16 with the gate's K cut over the grid (tfl_token_side)."""
    rows, k, ld, octet = _lay(x)
    if x.dtype != torch.bfloat16 or not token_side_pays(rows, k, gate.n) or proj.chunk_major or gate.chunk_major:
        return linear_f32(token_gate_linear(x, gate, table, ids, n_real), proj, width)
    _need(x, table, ids)
    assert ids.dtype == torch.int64 and ids.numel() == rows and k == gate.k == proj.n and gate.n == proj.k and x.dtype == table.dtype == gate.dtype == proj.dtype
    assert table.shape[1] == n_real and ids.is_contiguous()
    L = hip.latent_lib()
    out = torch.empty(rows, width, dtype=torch.float32, device=x.device)
    ws = torch.empty(L.tfl_token_side_ws_floats(rows, gate.n), dtype=torch.float32, device=x.device)
    hip.check(L.tfl_token_side(_p(gate.packed), _p(proj.packed), _p(x), ld, octet, _p(table), table.stride(0), _p(ids), table.shape[0], _p(out), out.stride(0), _p(ws),
                               ws.numel(), rows, gate.k, gate.n, n_real, width, _stream()), "tfl_token_side")
    return out


def finish(x, norm_w, eps, width, dtype, embed=None, ids=None, y=None, y_w=None, step=None, octets=False, prep=None):
    """Residual bookkeeping between two layers and the next norm; see tfl_finish.  x fp32 [rows, padded width] is updated in
    place; returns h in ``dtype``, row-major or (``octets``) octet-major.  ``prep``: decode_prep() of these tensors in the same launch (embed, no y)."""
    _need(x, norm_w, embed, ids, y, y_w, step)
    _f32(x, norm_w, y_w, step)
    rows, wp = x.shape
    assert x.is_contiguous() and norm_w.numel() == wp and (step is None or step.numel() == wp)
    assert embed is None or (embed.dtype == dtype and embed.shape[1] == wp and embed.is_contiguous() and ids.numel() == rows
                             and ids.dtype == torch.int64)
    assert y is None or (y.shape == (rows, wp) and y_w.numel() == wp and y.dtype in (dtype, torch.float32) and y.stride(1) == 1)
    h = empty_act(rows, wp, dtype, x.device) if octets else torch.empty(rows, wp, dtype=dtype, device=x.device)
    _, _, ld, octet = _lay(h)
    if prep is not None:
        assert embed is not None and y is None
        d = decode_prep_of(*prep)
        hip.check(hip.latent_lib().tfl_finish_first(_p(embed), _p(ids), embed.shape[0], _p(step), _p(norm_w), _p(x), _p(h), ld, octet, rows, wp, width, float(eps),
                                                    ctypes.byref(d), _CODE[dtype], _stream()), "tfl_finish_first")
        return h
    hip.check(hip.latent_lib().tfl_finish(_p(embed), _p(ids), 0 if embed is None else embed.shape[0], _p(y),
                                          int(y is not None and y.dtype == torch.float32), 0 if y is None else y.stride(0), _p(y_w),
                                          _p(step), _p(norm_w), _p(x), _p(h), ld, octet, rows, wp, width, float(eps), _CODE[dtype], _stream()),
              "tfl_finish")
    return h


def residual(d, x, want_copy):
    """x += d; returns x in d's type when ``want_copy``."""
    _need(d, x)
    _f32(x)
    assert d.shape == x.shape and d.is_contiguous() and x.is_contiguous()
    xt = torch.empty_like(d) if want_copy else None
    hip.check(hip.latent_lib().tfl_residual(_p(d), _p(x), _p(xt), d.numel(), _CODE[d.dtype], _stream()), "tfl_residual")
    return xt


def token_gate(s, table, ids, n_real):
    _need(s, table, ids)
    assert s.dtype == table.dtype and table.shape[1] == n_real and ids.dtype == torch.int64 and ids.numel() == s.shape[0]
    out = torch.empty(s.shape[0], s.shape[1], dtype=s.dtype, device=s.device)
    hip.check(hip.latent_lib().tfl_token_gate(_p(s), s.stride(0), _p(table), table.stride(0), _p(ids), table.shape[0], _p(out),
                                              s.shape[0], s.shape[1], n_real, _CODE[s.dtype], _stream()), "tfl_token_gate")
    return out


def prepare(y, g, up_off, n_up, q_norm, kv_norm, eps, rope, pos, slot, cache, act, act_off, want_rows):
    """Prefill half of the input projection (tfl_prepare): returns (cq, packed cache rows or None)."""
    _need(y, pos, slot, cache, act)
    _i32(pos, slot)
    _f32(q_norm, kv_norm)
    rows = y.shape[0]
    assert y.stride(1) == 1 and pos.numel() == rows and slot.numel() == rows and cache.dtype == y.dtype == act.dtype
    assert cache.shape[1] == g.C + g.R and cache.is_contiguous() and act.shape[1] >= act_off + n_up
    cq = torch.empty(rows, g.Q, dtype=y.dtype, device=y.device)
    ck = torch.empty(rows, g.C + g.R, dtype=y.dtype, device=y.device) if want_rows else None
    hip.check(hip.latent_lib().tfl_prepare(_p(y), y.stride(0), g.Q, g.q_real, g.C, g.c_real, g.R, up_off, n_up, _p(q_norm), _p(kv_norm),
                                           float(eps), _p(rope.cos), _p(rope.sin), rope.half, rope.max_pos, _p(pos), _p(slot),
                                           _p(cache), cache.shape[0], _p(cq), _p(ck), _p(act[:, act_off:]) if n_up else None,
                                           act.stride(0), rows, _CODE[y.dtype], _stream()), "tfl_prepare")
    return cq, ck


def gather_rows(cache, src):
    _need(cache, src)
    _i32(src)
    out = torch.empty(src.numel(), cache.shape[1], dtype=cache.dtype, device=cache.device)
    hip.check(hip.latent_lib().tfl_gather_rows(_p(cache), cache.shape[0], _p(src), _p(out), src.numel(), cache.shape[1],
                                               _CODE[cache.dtype], _stream()), "tfl_gather_rows")
    return out


def attn_prefill(q, kv, ck, seq, max_new, pos, rope, gate, out, g, scale):
    """q [tq, H*(N+R)], kv [tk, H*(N+V)], ck [tk, C+R], seq int32 [nseq, 4], gate / out [tq, >= H*V] views."""
    _need(q, kv, ck, seq, pos, gate, out)
    _i32(seq, pos)
    tq, tk = q.shape[0], kv.shape[0]
    assert q.dtype == kv.dtype == ck.dtype == gate.dtype == out.dtype and q.is_contiguous() and kv.is_contiguous() and ck.is_contiguous()
    assert q.shape[1] == g.H * (g.N + g.R) and kv.shape[1] == g.H * (g.N + g.V) and ck.shape == (tk, g.C + g.R)
    assert pos.numel() == tq and gate.shape[0] == tq and out.shape[0] == tq and seq.shape[1] == 4 and seq.is_contiguous()
    assert gate.shape[1] >= g.H * g.V and out.shape[1] >= g.H * g.V
    hip.check(hip.latent_lib().tfl_attn_prefill(_p(q), _p(kv), _p(ck), _p(seq), seq.shape[0], int(max_new), _p(pos), _p(rope.cos),
                                                _p(rope.sin), rope.half, rope.max_pos, _p(gate), gate.stride(0), _p(out), out.stride(0),
                                                tq, tk, g.H, g.N, g.R, g.V, g.C, float(scale), _CODE[q.dtype], _stream()),
              "tfl_attn_prefill")


def attn_decode(q, cache, table, klen, g, scale, max_len, nsplit=None):
    """q [rows, H, C+R] against the paged cache -> [rows, H, C].  max_len sizes the split (klen is on the device)."""
    _need(q, cache, table, klen)
    _i32(table, klen)
    rows = q.shape[0]
    assert q.dtype == cache.dtype and q.is_contiguous() and q.shape[1:] == (g.H, g.C + g.R) and cache.shape[1] == g.C + g.R
    assert cache.is_contiguous() and cache.shape[0] % PAGE == 0 and table.shape[0] == rows and table.stride(1) == 1 and klen.numel() == rows
    L = hip.latent_lib()
    if nsplit is None:
        nsplit = L.tfl_attn_decode_splits(rows, g.H, g.C, g.R, int(max_len), _CODE[q.dtype])
    n_ws = L.tfl_attn_decode_ws_floats(rows, g.H, g.C, nsplit)
    ws = torch.empty(n_ws, dtype=torch.float32, device=q.device) if n_ws else None
    out = torch.empty(rows, g.H, g.C, dtype=q.dtype, device=q.device)
    hip.check(L.tfl_attn_decode(_p(q), _p(cache), cache.shape[0] // PAGE, _p(table), table.stride(0), _p(klen), _p(out), _p(ws), n_ws,
                                rows, g.H, g.C, g.R, float(scale), nsplit, _CODE[q.dtype], _stream()), "tfl_attn_decode")
    return out


def _value_merges(rows, H, nsplit, parts):
    """Does latent_to_value merge the splits of attn_decode_beside itself (latent_value_kernel) or a launch in front of it?  us of a layer's attention,
    value and output product, launch -> itself: one row 35.5 -> 33.9 (64 pages), 37.7 -> 37.5 (192), the same from there on; two 36.2 -> 35.4 (72 pages),
    39.6 -> 39.8 (192); three rows the same to 1 %; four rows of 32 heads, whose merge is a wave for 128 columns (launch_merge: from 128 heads
    on, up to 64 splits), 39.9 -> 39.0 with 64 splits a row (144 pages), with 85 49.8 -> 51.2 (576 pages).  Over 672 points of 1 to 4 rows 1.001 of the
    better one, at most 1.04."""
    return rows == 1 or (rows == 2 and parts <= 72) or (rows <= 4 and rows * H >= 128 and nsplit <= 64)


@functools.lru_cache(maxsize=1024)
def beside_plan(rows, H, C, R, pages, n, k, longest=None):
    """(workers, panels each, splits, does latent_to_value merge them) of attn_decode_beside for rows that hold ``pages`` pages in all, the longest
    ``longest`` of them (not known: rows half to all as long as it), and a product of n outputs of k, None where the two are better launched apart."""
    each, nsplit, parts = ctypes.c_int32(), ctypes.c_int32(), ctypes.c_int32()
    to = ctypes.byref(each), ctypes.byref(nsplit), ctypes.byref(parts)
    L = hip.latent_lib()
    workers = L.tfl_attn_beside_plan(rows, H, C, R, pages, n, k, *to) if longest is None else L.tfl_attn_beside_plan_of(rows, H, C, R, pages, longest, n, k, *to)
    return (workers, each.value, nsplit.value, _value_merges(rows, H, nsplit.value, parts.value)) if workers > 0 else None


@functools.lru_cache(maxsize=1024)
def carry_plan(rows, H, C, R, pages, n, k, longest=None):
    """Columns of such a product, from the last on, that query_to_latent carries (0: none); what is left goes beside the attention as its own beside_plan says."""
    return hip.latent_lib().tfl_latent_carry(rows, H, C, R, pages, _longest(rows, pages, longest), n, k)


def _longest(rows, pages, longest):
    """As tfl_attn_beside_plan takes it where nobody knows: rows half to all as long as it."""
    return longest if longest is not None else pages if rows <= 1 else (4 * pages - 1) // (3 * rows) + 1


@functools.lru_cache(maxsize=1024)
def parts_plan(rows, H, C, R, pages, n, k, longest=None):
    """(workers, parts, splits) of attn_decode_beside_parts, None where beside_plan's division, or the two apart, are the faster way."""
    workers, nsplit = ctypes.c_int32(), ctypes.c_int32()
    parts = hip.latent_lib().tfl_beside_parts(rows, H, C, R, pages, _longest(rows, pages, longest), n, k, ctypes.byref(workers), ctypes.byref(nsplit))
    return (workers.value, parts, nsplit.value) if parts else None


class Splits:
    """What attn_decode_beside leaves to latent_to_value: unmerged splits of [rows, H, C]."""

    def __init__(self, ws, nsplit, shape, dtype):
        self.ws, self.nsplit, self.shape, self.dtype, self.is_cuda = ws, nsplit, shape, dtype, ws.is_cuda


def attn_decode_beside(q, cache, table, klen, g, scale, plan, act, wt, x, k0, k1=None):
    """attn_decode of bfloat16 rows of 512 + 64 with x += act . W^T over the columns from k0 on (to k1) in the same launch.  Splits as the plan says."""
    product = part_of(act, wt, x, k0, wt.k if k1 is None else k1)
    _need(q, cache, table, klen)
    _i32(table, klen)
    rows, (workers, each, nsplit, later) = q.shape[0], plan
    assert q.dtype == cache.dtype == torch.bfloat16 and product.rows == rows and q.is_contiguous() and q.shape[1:] == (g.H, 576) and (g.C, g.R) == (512, 64)
    assert cache.is_contiguous() and cache.shape[1] == 576 and cache.shape[0] % PAGE == 0
    assert table.shape[0] == rows and table.stride(1) == 1 and klen.numel() == rows
    L = hip.latent_lib()
    ws = torch.empty(L.tfl_attn_decode_ws_floats(rows, g.H, g.C, nsplit), dtype=torch.float32, device=q.device)
    out = None if later else torch.empty(rows, g.H, g.C, dtype=q.dtype, device=q.device)
    hip.check(L.tfl_attn_decode_beside(_p(q), _p(cache), cache.shape[0] // PAGE, _p(table), table.stride(0), _p(klen), _p(out), _p(ws), ws.numel(), rows, g.H,
                                       float(scale), nsplit, workers, each, ctypes.byref(product), _stream()), "tfl_attn_decode_beside")
    return Splits(ws, nsplit, (rows, g.H, g.C), q.dtype) if later else out


def attn_decode_beside_parts(q, cache, table, klen, g, scale, plan, act, wt, k0, k1):
    """attn_decode_beside of 17 to 32 rows with the product cut over k too: (attention, the parts' sums fp32 [parts][rows][n]) for add_linear.  plan: parts_plan."""
    _need(q, cache, table, klen)
    _i32(table, klen)
    rows, (workers, parts, nsplit) = q.shape[0], plan
    sums = torch.empty(parts, rows, wt.n, dtype=torch.float32, device=q.device)
    product = part_of(act, wt, sums[0], k0, k1)
    product.n_real = wt.n
    assert q.dtype == cache.dtype == torch.bfloat16 and product.rows == rows and q.is_contiguous() and q.shape[1:] == (g.H, 576) and (g.C, g.R) == (512, 64)
    assert cache.is_contiguous() and cache.shape[1] == 576 and cache.shape[0] % PAGE == 0
    assert table.shape[0] == rows and table.stride(1) == 1 and klen.numel() == rows
    L = hip.latent_lib()
    ws = torch.empty(L.tfl_attn_decode_ws_floats(rows, g.H, g.C, nsplit), dtype=torch.float32, device=q.device)
    out = torch.empty(rows, g.H, g.C, dtype=q.dtype, device=q.device)
    hip.check(L.tfl_attn_decode_beside_parts(_p(q), _p(cache), cache.shape[0] // PAGE, _p(table), table.stride(0), _p(klen), _p(out), _p(ws), ws.numel(), rows, g.H,
                                             float(scale), nsplit, workers, parts, ctypes.byref(product), _stream()), "tfl_attn_decode_beside_parts")
    return out, sums
