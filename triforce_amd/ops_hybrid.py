"""Tensor-level wrappers over the hybrid C ABI (include/triforce_hybrid.h, on top of ops_tile.py): residual streams, chunked
grouped-query attention, linear recurrences.

Same rules as ops.py: torch owns the memory and the stream, every function validates its tensors and enqueues hand-written
gfx950 kernels on torch's current stream; no CPU path exists.  The element type is bfloat16 or float32 and follows the tensors.
Geometry arguments (``g``) are models.hybrid_core.AttentionGeom / StateSpaceGeom / LinearAttentionGeom.
"""
import ctypes

import torch

from . import hip
from .ops_tile import (_CODE, PAGE, TileWeight, _f32, _i32, _lay, _need, _p, _stream, decode_prep, decode_prep_of, empty_act, gelu_glu_linear,  # noqa: F401
                       grow, interleave_glu, linear_f32, pad32)

CHUNK = 64                     # tokens a recurrence takes at a time in prefill (TFH_CHUNK)


def _lib():
    return hip.hybrid_lib()


def connect(x, u_in, norm_w, eps, width, dtype, embed=None, ids=None, embed_w=None, y=None, out=None, mix=None, keep=True, octets=False,
            prep=None):
    """Residual streams between two sublayers; see tfh_connect.  x fp32 [rows, streams, padded width] is updated in place (unless
    not ``keep``); returns the sublayer's normed input in ``dtype``, row-major or (``octets``) octet-major.  ``prep``: decode_prep() of these tensors in the same
    launch (embed, kept)."""
    _need(x, u_in, norm_w, embed, ids, embed_w, y, out, mix)
    _f32(x, u_in, norm_w, embed_w, out, mix)
    rows, streams, wp = x.shape
    assert x.is_contiguous() and norm_w.numel() == wp and u_in.numel() == streams
    assert embed is None or (embed.dtype == dtype and embed.shape[1] == wp and embed.is_contiguous() and ids.numel() == rows
                             and ids.dtype == torch.int64 and embed_w.numel() == wp and y is None)
    assert y is None or (y.shape == (rows, wp) and y.dtype in (dtype, torch.float32) and y.stride(1) == 1 and out.numel() == streams
                         and mix.shape == (streams, streams) and mix.is_contiguous())
    h = empty_act(rows, wp, dtype, x.device) if octets else torch.empty(rows, wp, dtype=dtype, device=x.device)
    _, _, ld, octet = _lay(h)
    if prep is not None:
        assert embed is not None and y is None and keep
        d = decode_prep_of(*prep)
        hip.check(_lib().tfh_connect_first(_p(embed), _p(ids), embed.shape[0], _p(embed_w), _p(u_in), _p(norm_w), _p(x), streams, _p(h), ld, octet, rows, wp, width,
                                           float(eps), ctypes.byref(d), _CODE[dtype], _stream()), "tfh_connect_first")
        return h
    hip.check(_lib().tfh_connect(_p(embed), _p(ids), 0 if embed is None else embed.shape[0], _p(embed_w), _p(y),
                                 int(y is not None and y.dtype == torch.float32), 0 if y is None else y.stride(0), _p(out), _p(mix), _p(u_in),
                                 _p(norm_w), _p(x), streams, int(keep), _p(h), ld, octet, rows, wp, width, float(eps), _CODE[dtype], _stream()),
              "tfh_connect")
    return h


class Connect:
    """connect() of decode rows that the product which reads them makes for itself (tfh_connect_gemm): stands for its activation block; ``out`` holds the
    updated streams."""

    def __init__(self, x, u_in, norm_w, eps, width, y, out, mix, keep=True):
        _need(x, u_in, norm_w, y, out, mix)
        _f32(x, u_in, norm_w, y, out, mix)
        rows, streams, wp = x.shape
        assert x.is_contiguous() and norm_w.numel() == wp and u_in.numel() == streams == out.numel() and mix.shape == (streams, streams) and mix.is_contiguous()
        assert y.shape == (rows, wp) and y.stride(1) == 1
        self.out, self.rows, self.dtype, self.device = torch.empty_like(x) if keep else None, rows, torch.bfloat16, x.device
        self.keep = (x, u_in, norm_w, y, out, mix)
        f = self.c = hip.TfhConnect()
        for name, t in (("y", y), ("out", out), ("mix", mix), ("in", u_in), ("norm_w", norm_w), ("x", x), ("x_out", self.out)):
            setattr(f, name, None if t is None else t.data_ptr())
        f.ld_y, f.streams, f.width, f.width_real, f.eps = y.stride(0), streams, wp, width, eps

    @staticmethod
    def takes(x, wt, epi):
        """Does the product of wt with this epilogue ("f32", "glu") make the rows of x itself?"""
        rows, streams, wp = x.shape
        return wt.chunk_major and wt.dtype == torch.bfloat16 and wt.k == wp and _lib().tfh_connect_gemm_takes(rows, streams, wp, wt.n, wt.k, hip.TFL_EPI[epi]) == 1

    def _product(self, wt, epi, **kw):
        assert wt.dtype == self.dtype
        a = hip.TflGemm()
        a.wp, a.rows, a.n, a.k, a.groups, a.x_oct, a.t_oct, a.ld_x, a.chunk_major = wt.packed.data_ptr(), self.rows, wt.n, wt.k, 1, 8, 8, 8, 1
        for name, v in kw.items():
            setattr(a, name, v.data_ptr() if isinstance(v, torch.Tensor) else v)
        hip.check(_lib().tfh_connect_gemm(ctypes.byref(self.c), ctypes.byref(a), hip.TFL_EPI[epi], _stream()), "tfh_connect_gemm " + epi)

    def linear(self, wt, n_real):
        """linear_f32 of the rows."""
        out = torch.empty(self.rows, n_real, dtype=torch.float32, device=self.device)
        self._product(wt, "f32", out_f=out, ld_f=n_real, n_real=n_real)
        return out

    def gelu_glu(self, wt):
        """gelu_glu_linear of the rows."""
        out = empty_act(self.rows, wt.n // 2, wt.dtype, self.device)
        self._product(wt, "glu", out_t=out, ld_t=8, t_oct=8 * self.rows)
        return out


class Streams:
    """Where a sublayer's last product takes its result (tfh_streams_gemm): into the residual streams x (in place; not kept unless ``keep``), and on as the
    next sublayer's input."""

    def __init__(self, x, out, mix, u_in, norm_w, eps, width, keep=True):
        _need(x, u_in, norm_w, out, mix)
        _f32(x, u_in, norm_w, out, mix)
        rows, streams, wp = x.shape
        assert x.is_contiguous() and norm_w.numel() == wp and u_in.numel() == streams == out.numel() and mix.shape == (streams, streams) and mix.is_contiguous()
        self.keep, self.rows, self.eps, self.width = (x, u_in, norm_w, out, mix), rows, eps, width
        f = self.c = hip.TfhConnect()
        for name, t in (("out", out), ("mix", mix), ("in", u_in), ("norm_w", norm_w), ("x", x), ("x_out", x if keep else None)):
            setattr(f, name, None if t is None else t.data_ptr())
        f.streams, f.width, f.width_real, f.eps = streams, wp, width, eps

    @staticmethod
    def takes(x, wt, after, epi):
        """Do the product of wt into the streams x and the one of ``after`` with this epilogue ("f32", "glu") behind it have these forms?"""
        rows, streams, wp = x.shape
        L = _lib()
        return (wt.chunk_major and after.chunk_major and wt.dtype == after.dtype == torch.bfloat16 and wt.n == wp == after.k
                and L.tfh_streams_gemm_takes(rows, streams, wt.n, wt.k) == 1 and L.tfh_scaled_gemm_takes(rows, after.n, hip.TFL_EPI[epi]) == 1)

    def result(self, act, wt):
        """The input (a Scaled) that comes out of the streams behind act . W^T."""
        _need(act)
        rows, k, ld, octet = _lay(act)
        assert act.dtype == wt.dtype and k == wt.k and rows == self.rows
        h = empty_act(rows, wt.n, wt.dtype, act.device)
        ss = torch.empty(rows, wt.n // 16, dtype=torch.float32, device=act.device)
        a = hip.TflGemm()
        a.wp, a.x, a.out_t, a.ss_out = wt.packed.data_ptr(), act.data_ptr(), h.data_ptr(), ss.data_ptr()
        a.rows, a.n, a.k, a.groups, a.chunk_major, a.ld_x, a.x_oct, a.ld_t, a.t_oct, a.ss_ld = rows, wt.n, wt.k, 1, 1, ld, octet, 8, 8 * rows, wt.n // 16
        hip.check(_lib().tfh_streams_gemm(ctypes.byref(self.c), ctypes.byref(a), _stream()), "tfh_streams_gemm")
        return Scaled(h, ss, self.width, self.eps)


class Scaled:
    """An activation block whose rows still miss their norm's scale, which the next product makes of their sums of squares (tfh_scaled_gemm)."""

    def __init__(self, h, ss, width, eps):
        self.h, self.ss, self.width, self.eps, self.dtype, self.device = h, ss, width, eps, h.dtype, h.device

    def _product(self, wt, epi, **kw):
        rows, k, ld, octet = _lay(self.h)
        assert wt.dtype == self.dtype and k == wt.k and wt.chunk_major
        a = hip.TflGemm()
        a.wp, a.x, a.ss_in = wt.packed.data_ptr(), self.h.data_ptr(), self.ss.data_ptr()
        a.rows, a.n, a.k, a.groups, a.chunk_major, a.ld_x, a.x_oct, a.t_oct = rows, wt.n, wt.k, 1, 1, ld, octet, 8
        a.ss_n = a.ss_ld = self.ss.shape[1]
        a.k_real, a.eps = self.width, self.eps
        for name, v in kw.items():
            setattr(a, name, v.data_ptr() if isinstance(v, torch.Tensor) else v)
        hip.check(_lib().tfh_scaled_gemm(ctypes.byref(a), hip.TFL_EPI[epi], _stream()), "tfh_scaled_gemm " + epi)

    def linear(self, wt, n_real):
        """linear_f32 of the rows."""
        out = torch.empty(self.h.shape[1], n_real, dtype=torch.float32, device=self.device)
        self._product(wt, "f32", out_f=out, ld_f=n_real, n_real=n_real)
        return out

    def gelu_glu(self, wt):
        """gelu_glu_linear of the rows."""
        rows = self.h.shape[1]
        out = empty_act(rows, wt.n // 2, wt.dtype, self.device)
        self._product(wt, "glu", out_t=out, ld_t=8, t_oct=8 * rows)
        return out


def linear_of(h, wt, n_real):
    """linear_f32 of an activation block, a Connect or a Scaled."""
    return h.linear(wt, n_real) if isinstance(h, (Connect, Scaled)) else linear_f32(h, wt, n_real)


def gelu_glu_of(h, wt):
    """gelu_glu_linear of an activation block, a Connect or a Scaled."""
    return h.gelu_glu(wt) if isinstance(h, (Connect, Scaled)) else gelu_glu_linear(h, wt)


def result_of(act, wt, to):
    """A sublayer's result: fp32 act . W^T, or with ``to`` (Streams) the next sublayer's input."""
    return linear_f32(act, wt, wt.n) if to is None else to.result(act, wt)


def qkv_prepare(y, g, q_norm, k_norm, eps, rope, pos, slot, cache):
    """Norm and rotation of new queries (in place) and keys; keys and values into the cache rows ``slot``."""
    _need(y, pos, slot, cache)
    _i32(pos, slot)
    _f32(q_norm, k_norm)
    rows = y.shape[0]
    assert y.stride(1) == 1 and pos.numel() == rows and slot.numel() == rows and cache.dtype == y.dtype and cache.is_contiguous()
    assert cache.shape[1] == g.row and q_norm.numel() == g.D and k_norm.numel() == g.D
    hip.check(_lib().tfh_qkv_prepare(_p(y), y.stride(0), g.q_off, g.k_off, g.v_off, _p(q_norm), _p(k_norm), _p(rope.cos), _p(rope.sin), rope.half,
                                     rope.max_pos, _p(pos), _p(slot), _p(cache), cache.shape[0], rows, g.H, g.G, g.D, g.d_real, g.V, float(eps),
                                     _CODE[y.dtype], _stream()), "tfh_qkv_prepare")


def attn_prefill(y, g, cache, batch, out, out_scale):
    """New tokens' attention over the paged cache; y [tokens, >= all projections] holds queries and gates, out [tokens, >= H*V]."""
    _need(y, cache, batch.table, batch.seq, out)
    _i32(batch.table, batch.seq)
    q, gate = y[:, g.q_off:], y[:, g.gate_off:]
    assert y.dtype == cache.dtype == out.dtype and cache.is_contiguous() and cache.shape[1] == g.row and cache.shape[0] % PAGE == 0
    assert batch.seq.shape[1] == 4 and batch.seq.is_contiguous() and batch.table.stride(1) == 1 and out.shape[0] == y.shape[0]
    assert q.shape[1] >= g.H * g.D and gate.shape[1] >= g.H * g.V and out.shape[1] >= g.H * g.V
    hip.check(_lib().tfh_attn_prefill(_p(q), y.stride(0), _p(cache), cache.shape[0] // PAGE, _p(batch.table), batch.table.stride(0), _p(batch.seq),
                                      batch.seq.shape[0], int(batch.max_new), _p(gate), y.stride(0), _p(out), out.stride(0), y.shape[0], g.H, g.G,
                                      g.D, g.V, g.chunk, float(g.scale), float(out_scale), _CODE[y.dtype], _stream()), "tfh_attn_prefill")


def conv_prepare(y, g, w, b, dt_bias, ring, batch):
    """Short convolution over x | B | C and the step sizes: (xbc [tokens, channels], dt fp32 [tokens, H]); the ring takes the last
    inputs.  w fp32 [taps, channels]."""
    _need(y, w, b, dt_bias, ring, batch.seq)
    _f32(w, b, dt_bias, ring)
    taps, channels = w.shape
    assert y.stride(1) == 1 and w.is_contiguous() and ring.shape[1:] == (taps, channels) and ring.is_contiguous() and channels == g.channels
    assert b.numel() == channels and dt_bias.numel() == g.H
    xbc = torch.empty(y.shape[0], channels, dtype=y.dtype, device=y.device)
    dt = torch.empty(y.shape[0], g.H, dtype=torch.float32, device=y.device)
    hip.check(_lib().tfh_conv_prepare(_p(y), y.stride(0), g.x_off, g.dt_off, _p(w), _p(b), taps, channels, _p(dt_bias), g.H, _p(ring), ring.shape[0],
                                      _p(xbc), _p(dt), _p(batch.seq), batch.seq.shape[0], int(batch.max_new), y.shape[0], _CODE[y.dtype],
                                      _stream()), "tfh_conv_prepare")
    return xbc, dt


def decay_prepare(z, bias, inv_tau, batch):
    """Log decays per key channel, summed up inside chunks of CHUNK new tokens: fp32 [tokens, channels]."""
    _need(z, bias, batch.seq)
    _f32(bias)
    assert z.stride(1) == 1 and bias.numel() == z.shape[1]
    out = torch.empty(z.shape, dtype=torch.float32, device=z.device)
    hip.check(_lib().tfh_decay_prepare(_p(z), z.stride(0), _p(bias), float(inv_tau), _p(out), _p(batch.seq), batch.seq.shape[0],
                                       int(batch.max_new), z.shape[0], z.shape[1], _CODE[z.dtype], _stream()), "tfh_decay_prepare")
    return out


def recurrence(q, k, v, g, state, batch, gcum=None, dt=None, nega=None, skip=None, gate=None, q_scale=1.0):
    """Packed new tokens through S = decay S + k v^T, o = S^T q (tfh_recurrence): returns o [tokens, H*V]; ``state`` fp32
    [seats, H, N, V] goes on from the sequences' pasts."""
    _need(q, k, v, gcum, dt, nega, skip, gate, state, batch.seq, batch.seg, batch.span)
    _i32(batch.seq, batch.seg, batch.span)
    _f32(gcum, dt, nega, skip, state)
    tokens, nseg = v.shape[0], batch.seg.shape[0]
    groups = g.H // g.per_group
    assert q.dtype == k.dtype == v.dtype and q.shape == k.shape == (tokens, groups * g.N) and v.shape == (tokens, g.H * g.V)
    assert state.shape[1:] == (g.H, g.N, g.V) and state.is_contiguous() and batch.seg.is_contiguous() and batch.span.is_contiguous()
    assert (gcum is None) != (dt is None) and (gcum is None or (gcum.shape == (tokens, g.H * g.N) and gcum.is_contiguous() and g.per_group == 1))
    assert dt is None or (dt.shape == (tokens, g.H) and dt.is_contiguous() and nega.numel() == g.H)
    assert gate is None or (gate.dtype == v.dtype and gate.shape == v.shape and gate.stride(1) == 1)
    out = torch.empty(tokens, g.H * g.V, dtype=v.dtype, device=v.device)
    part = decay = None
    if batch.max_segs > 1:
        part = torch.empty(nseg, g.H, g.N, g.V, dtype=torch.float32, device=v.device)
        decay = torch.empty(nseg, g.H * (g.N if gcum is not None else 1), dtype=torch.float32, device=v.device)
    a = hip.TfhRecurrence()
    for name, t in (("q", q), ("k", k), ("v", v), ("gcum", gcum), ("dt", dt), ("nega", nega), ("skip", skip), ("gate", gate), ("state", state),
                    ("part", part), ("decay", decay), ("out", out), ("seq", batch.seq), ("seg", batch.seg), ("span", batch.span)):
        setattr(a, name, None if t is None else t.data_ptr())
    a.ld_q, a.ld_k, a.ld_v, a.ld_gate, a.ld_out = q.stride(0), k.stride(0), v.stride(0), 0 if gate is None else gate.stride(0), out.stride(0)
    a.nseq, a.nseg, a.max_segs, a.tokens, a.seats = batch.seq.shape[0], nseg, batch.max_segs, tokens, state.shape[0]
    a.H, a.per_group, a.N, a.V, a.q_scale = g.H, g.per_group, g.N, g.V, q_scale
    hip.check(_lib().tfh_recurrence(ctypes.byref(a), _CODE[v.dtype], _stream()), "tfh_recurrence")
    return out


def group_norm(src, w, groups, size, g, out, eps, scale=1.0, gate=None, shared_w=False):
    """``groups`` parts of ``size`` real values of each row / rms * w * scale [* silu(gate)] into ``out`` [rows, >= H*V]."""
    _need(src, w, gate, out)
    _f32(w)
    assert src.stride(1) == 1 and src.shape[1] == g.H * g.V and groups * size == g.H * g.v_real and w.numel() == (size if shared_w else groups * size)
    assert gate is None or (gate.dtype == src.dtype and gate.shape == src.shape and gate.stride(1) == 1)
    assert out.shape[0] == src.shape[0] and out.shape[1] >= g.H * g.V and src.dtype in (out.dtype, torch.float32)
    hip.check(_lib().tfh_group_norm(_p(src), src.stride(0), _p(gate), 0 if gate is None else gate.stride(0), int(src.dtype == torch.float32), _p(w),
                                    int(shared_w), _p(out), out.stride(0), 8, src.shape[0], groups, size, g.v_real, g.V, float(eps), float(scale),
                                    _CODE[out.dtype], _stream()), "tfh_group_norm")


def glu(s):
    """[rows, 2n] in blocks of 8 gate | 8 up columns -> gelu_tanh(gate) * up."""
    _need(s)
    assert s.is_contiguous()
    out = torch.empty(s.shape[0], s.shape[1] // 2, dtype=s.dtype, device=s.device)
    hip.check(_lib().tfh_glu(_p(s), _p(out), s.shape[0], out.shape[1], _CODE[s.dtype], _stream()), "tfh_glu")
    return out


class MixerStep:
    """One decode step of a layer's mixer: the two launches share their arguments and workspace.  ``attn`` / ``rec``: what the
    layer has of each (dicts of tensors and numbers named like the fields of TfhAttnStep / TfhRecStep)."""

    def __init__(self, raw, klen, eps, dtype, attn=None, rec=None, max_keys=0, nsplit=None):
        _need(raw, klen)
        _f32(raw)
        _i32(klen)
        rows = raw.shape[0]
        assert raw.stride(1) == 1 and klen.numel() == rows
        self.raw, self.klen, self.eps, self.dtype, self.rows, self.keep = raw, klen, float(eps), dtype, rows, [attn, rec]
        self.attn = self.rec = None
        if attn is not None:
            a = self.attn = self._fill(hip.TfhAttnStep(), attn)
            assert attn["cache"].dtype == dtype and attn["cache"].is_contiguous() and attn["table"].stride(1) == 1 and attn["table"].shape[0] == rows
            a.n_pages, a.table_ld = attn["cache"].shape[0] // PAGE, attn["table"].stride(0)
            a.nsplit = nsplit or _lib().tfh_attn_step_splits(rows, a.H, a.G, a.D, a.V, min(max_keys, a.chunk + PAGE) if a.chunk else max_keys,
                                                             _CODE[dtype])
            ws = torch.empty(_lib().tfh_attn_step_ws_floats(rows, a.H, a.V, a.nsplit), dtype=torch.float32, device=raw.device)
            a.ws = ws.data_ptr()
            self.keep.append(ws)
        if rec is not None:
            r = self.rec = self._fill(hip.TfhRecStep(), rec)
            _i32(rec["seat"])
            assert rec["seat"].numel() == rows and rec["state"].shape[1:] == (r.H, r.N, r.V) and rec["state"].is_contiguous()
            r.seats = rec["state"].shape[0]
            o = torch.empty(rows, r.H, r.V, dtype=torch.float32, device=raw.device)
            r.out = o.data_ptr()
            self.keep.append(o)

    @staticmethod
    def _fill(s, values):
        for name, v in values.items():
            if isinstance(v, torch.Tensor):
                _need(v)
                v = v.data_ptr()
            setattr(s, name, v)
        return s

    def _refs(self):
        return tuple(None if s is None else ctypes.byref(s) for s in (self.attn, self.rec))

    def run(self):
        hip.check(_lib().tfh_step(*self._refs(), _p(self.raw), self.raw.stride(0), _p(self.klen), self.rows, self.eps, _CODE[self.dtype], _stream()),
                  "tfh_step")
        return self

    def operand(self):
        """Octet-major [attention | recurrence] block of the output projection."""
        k = sum(s.H * s.V for s in (self.attn, self.rec) if s is not None)
        act = empty_act(self.rows, k, self.dtype, self.raw.device)
        hip.check(_lib().tfh_step_out(*self._refs(), _p(self.raw), self.raw.stride(0), _p(act), 8, 8 * self.rows, self.rows, self.eps,
                                      _CODE[self.dtype], _stream()), "tfh_step_out")
        return act
