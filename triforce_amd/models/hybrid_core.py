"""Weights and the per-layer compute of a decoder with several residual streams and hybrid mixers (chunked attention beside a
state-space recurrence, or gated linear attention) on the HIP ops (ops_hybrid).

Decode form of a layer (one token per sequence, any number of sequences): [input projections] [mixer: attention splits and state updates side by side]
[merge, norms, gates] [output projection] [gated unit] [down] and, in front of the input projections and of the gated unit, [streams, norm].  In bfloat16
with up to four streams the two are no launches of their own where the width is 4 096, or 7 232 to 8 192 in 64s (ops_hybrid.Streams: the product in front of
them brings the streams on, the one behind scales), nor, with one sequence, where it is 2 048 to 4 064 (ops_hybrid.Connect: the product behind makes its row).
Prefill form: products of many rows (ops_rows) between the row kernels, the paged attention and the segmented recurrence.
"""
import zlib

import torch

from .. import ops_hybrid as oh
from ..ops_tile import TileWeight, grow


def _heads(w, heads, size, padded, width):
    """[heads * size, k] -> [heads * padded, width], zero rows behind every head."""
    return grow(w.view(heads, size, w.shape[1]), heads, padded, width).reshape(heads * padded, width)


def _head_cols(w, heads, size, padded, width):
    """[n, heads * size] -> [width, heads * padded], zero columns behind every head."""
    return grow(w.view(w.shape[0], heads, size), width, heads, padded).reshape(width, heads * padded)


def _units(g):
    """Workgroups of a recurrence per segment."""
    return g.H * -(-g.V // 64)


class AttentionGeom:
    """Padded sizes of one attention and the columns of its parts in the layer's input projection."""

    def __init__(self, m):
        p = oh.pad32
        self.H, self.G, self.D, self.V, self.d_real, self.chunk, self.scale = m.heads, m.kv_heads, p(m.dim), p(m.vdim), m.dim, m.chunk, m.scale
        self.q_off = 0
        self.k_off = self.H * self.D
        self.v_off = self.k_off + self.G * self.D
        self.gate_off = self.v_off + self.G * self.V
        self.width = self.gate_off + self.H * self.V

    row = property(lambda s: s.G * (s.D + s.V))                   # one cached row


class StateSpaceGeom:
    """Scalar-decay recurrence: H heads in groups that share B and C, state N x V, behind ``base`` other columns."""

    def __init__(self, m, base):
        p = oh.pad32
        self.H, self.per_group, self.N, self.V, self.v_real, self.norm_groups = m.heads, m.heads // m.groups, p(m.state), p(m.vdim), m.vdim, m.norm_groups
        inner, gn = self.H * self.V, m.groups * self.N
        self.gate_off, self.x_off = base, base + inner
        self.b_col, self.c_col, self.channels = inner, inner + gn, inner + 2 * gn
        self.dt_off = self.x_off + self.channels
        self.width = self.dt_off + p(m.heads) - base


class LinearAttentionGeom:
    """Per-channel decay recurrence: a state of N x V per head."""
    per_group = 1

    def __init__(self, m, rank):
        p = oh.pad32
        self.H, self.N, self.V, self.v_real, self.rank = m.heads, p(m.dim), p(m.vdim), m.vdim, p(rank)
        self.norm_groups = m.heads
        self.q_off, self.k_off = 0, self.H * self.N
        self.v_off = 2 * self.H * self.N
        self.gate_off = self.v_off + self.H * self.V
        self.a_off = self.gate_off + self.H * self.V
        self.width = self.a_off + self.rank


class Connection:
    """How one sublayer reads and writes the residual streams (fp32)."""

    def __init__(self, get, name):
        self.u_in, self.out, self.mix = (get(f"{name}.{k}").float().contiguous() for k in ("in", "out", "mix"))


class ChunkedAttention:
    def __init__(self, spec, get, W):
        self.spec, g = spec, AttentionGeom(spec)
        self.geom = g
        self.rows_in = [_heads(get("q"), g.H, spec.dim, g.D, W), _heads(get("k"), g.G, spec.dim, g.D, W), _heads(get("v"), g.G, spec.vdim, g.V, W),
                        _heads(get("g"), g.H, spec.vdim, g.V, W)]
        self.cols_out = _head_cols(get("o"), g.H, spec.vdim, g.V, W)
        self.q_norm, self.k_norm = (grow(get(f"{n}.norm").float(), g.D) for n in ("q", "k"))

    def step(self, batch, rope, cache_rows, out_scale):
        g = self.geom
        return dict(q_norm=self.q_norm, k_norm=self.k_norm, cos=rope.cos, sin=rope.sin, cache=cache_rows, table=batch.table, q_off=g.q_off,
                    k_off=g.k_off, v_off=g.v_off, gate_off=g.gate_off, half=rope.half, max_pos=rope.max_pos, H=g.H, G=g.G, D=g.D, D_real=g.d_real,
                    V=g.V, chunk=g.chunk, scale=g.scale, out_scale=out_scale)

    def prefill(self, y, act, batch, rope, cache_rows, eps, out_scale):
        oh.qkv_prepare(y, self.geom, self.q_norm, self.k_norm, eps, rope, batch.pos, batch.slot, cache_rows)
        oh.attn_prefill(y, self.geom, cache_rows, batch, act, out_scale)


class StateSpace:
    def __init__(self, spec, get, W, base):
        self.spec, g = spec, StateSpaceGeom(spec, base)
        self.geom = g
        H, V, N, G = spec.heads, spec.vdim, spec.state, spec.groups

        def parts(t, k):                                          # x | B | C of a [channels, ...] tensor
            x, B, C = t.split([H * V, G * N, G * N])
            return [_heads(x, H, V, g.V, k), _heads(B, G, N, g.N, k), _heads(C, G, N, g.N, k)]
        z, xbc, dt = get("in").split([H * V, H * V + 2 * G * N, H])
        self.rows_in = [_heads(z, H, V, g.V, W)] + parts(xbc, W) + [grow(dt, oh.pad32(H), W)]
        self.cols_out = _head_cols(get("o"), H, V, g.V, W)
        self.conv_w = torch.cat(parts(get("conv").float(), spec.conv)).t().contiguous()          # [taps, channels]
        self.conv_b = torch.cat(parts(get("conv.b").float().unsqueeze(1), 1)).reshape(-1).contiguous()
        self.dt_bias, self.skip, self.norm_w = (get(n).float().contiguous() for n in ("dt_bias", "D", "norm"))
        self.nega = (-torch.exp(get("A_log").float())).contiguous()

    def state_shapes(self):
        g = self.geom
        return {"state": (g.H, g.N, g.V), "ring": (self.spec.conv, g.channels)}

    def step(self, batch, states, out_scale):
        g = self.geom
        return dict(conv_w=self.conv_w, conv_b=self.conv_b, ring=states["ring"], dt_bias=self.dt_bias, nega=self.nega, skip=self.skip,
                    norm_w=self.norm_w, state=states["state"], seat=batch.seat, x_off=g.x_off, dt_off=g.dt_off, gate_off=g.gate_off,
                    taps=self.spec.conv, channels=g.channels, H=g.H, per_group=g.per_group, N=g.N, V=g.V, V_real=g.v_real,
                    norm_groups=g.norm_groups, q_scale=1.0, out_scale=out_scale)

    def prefill(self, y, act, batch, states, eps, out_scale):
        g = self.geom
        xbc, dt = oh.conv_prepare(y, g, self.conv_w, self.conv_b, self.dt_bias, states["ring"], batch)
        yz = oh.recurrence(xbc[:, g.c_col:], xbc[:, g.b_col:g.c_col], xbc[:, :g.b_col], g, states["state"], batch, dt=dt, nega=self.nega,
                           skip=self.skip, gate=y[:, g.gate_off:g.gate_off + g.H * g.V])
        oh.group_norm(yz, self.norm_w, g.norm_groups, g.H * g.v_real // g.norm_groups, g, act, eps, scale=out_scale)


class ParallelMixer:
    """Chunked attention and a state-space recurrence on one input: one input projection, one output projection (their scales go on
    its operand)."""

    def __init__(self, spec, get, W, dtype):
        self.spec = spec
        self.left = ChunkedAttention(spec.left, lambda n: get("left." + n), W)
        self.right = StateSpace(spec.right, lambda n: get("right." + n), W, self.left.geom.width)
        self.w_in = TileWeight(torch.cat([t.to(dtype) for t in self.left.rows_in + self.right.rows_in]))
        self.w_out = TileWeight(torch.cat([self.left.cols_out.to(dtype), self.right.cols_out.to(dtype)], 1))
        for part in (self.left, self.right):
            del part.rows_in, part.cols_out

    @staticmethod
    def shapes(m, d, rank=None):
        a, s = m.left, m.right
        inner, gn = s.heads * s.vdim, s.groups * s.state
        return {"left.q": (a.heads * a.dim, d), "left.k": (a.kv_heads * a.dim, d), "left.v": (a.kv_heads * a.vdim, d), "left.q.norm": (a.dim,),
                "left.k.norm": (a.dim,), "left.g": (a.heads * a.vdim, d), "left.o": (d, a.heads * a.vdim),
                "right.in": (2 * inner + 2 * gn + s.heads, d), "right.conv": (inner + 2 * gn, s.conv), "right.conv.b": (inner + 2 * gn,),
                "right.dt_bias": (s.heads,), "right.A_log": (s.heads,), "right.D": (s.heads,), "right.norm": (inner,), "right.o": (d, inner)}

    def cache_width(self):
        return self.left.geom.row

    def state_shapes(self):
        return self.right.state_shapes()

    def recurrence_units(self):
        return _units(self.right.geom)

    def decode(self, h, batch, rope, cache_rows, states, eps, to=None):
        raw = oh.linear_of(h, self.w_in, self.w_in.n)
        step = oh.MixerStep(raw, batch.klen, eps, h.dtype, attn=self.left.step(batch, rope, cache_rows, self.spec.left_scale),
                            rec=self.right.step(batch, states, self.spec.right_scale), max_keys=batch.max_len)
        return oh.result_of(step.run().operand(), self.w_out, to)

    def prefill(self, h, batch, rope, cache_rows, states, eps):
        y = self.w_in.matmul(h)
        act = torch.empty(h.shape[0], self.w_out.k, dtype=h.dtype, device=h.device)
        self.left.prefill(y, act, batch, rope, cache_rows, eps, self.spec.left_scale)
        self.right.prefill(y, act[:, self.left.geom.H * self.left.geom.V:], batch, states, eps, self.spec.right_scale)
        return self.w_out.matmul(act)


class LinearAttentionMixer:
    """Gated linear attention with a decay per key channel."""

    def __init__(self, spec, get, W, dtype):
        a1, a2 = get("a1"), get("a2")
        self.spec, g = spec, LinearAttentionGeom(spec, a1.shape[0])
        self.geom = g
        self.w_in = TileWeight(torch.cat([t.to(dtype) for t in (
            _heads(get("q"), g.H, spec.dim, g.N, W), _heads(get("k"), g.H, spec.dim, g.N, W), _heads(get("v"), g.H, spec.vdim, g.V, W),
            _heads(get("g"), g.H, spec.vdim, g.V, W), grow(a1, g.rank, W))]))
        self.w_out = TileWeight(_head_cols(get("o"), g.H, spec.vdim, g.V, W).to(dtype))
        self.a2 = _heads(a2, g.H, spec.dim, g.N, g.rank).to(dtype).contiguous()
        self.a2_b = _heads(get("a2.b").float().unsqueeze(1), g.H, spec.dim, g.N, 1).reshape(-1).contiguous()
        self.norm_w = get("norm").float().contiguous()
        self.q_scale = spec.dim ** -0.5

    @staticmethod
    def shapes(m, d, rank=None):
        n, v, r = m.heads * m.dim, m.heads * m.vdim, m.rank if rank is None else rank
        return {"q": (n, d), "k": (n, d), "v": (v, d), "g": (v, d), "o": (d, v), "norm": (m.vdim,), "a1": (r, d), "a2": (n, r), "a2.b": (n,)}

    def cache_width(self):
        return 0

    def state_shapes(self):
        g = self.geom
        return {"state": (g.H, g.N, g.V)}

    def recurrence_units(self):
        return _units(self.geom)

    def decode(self, h, batch, rope, cache_rows, states, eps, to=None):
        g = self.geom
        raw = oh.linear_of(h, self.w_in, self.w_in.n)
        rec = dict(a2=self.a2, a2_b=self.a2_b, norm_w=self.norm_w, state=states["state"], seat=batch.seat, gate_off=g.gate_off, q_off=g.q_off,
                   k_off=g.k_off, v_off=g.v_off, a_off=g.a_off, rank=g.rank, H=g.H, per_group=1, N=g.N, V=g.V, V_real=g.v_real,
                   norm_groups=g.norm_groups, inv_tau=1.0 / self.spec.tau, q_scale=self.q_scale, out_scale=1.0)
        return oh.result_of(oh.MixerStep(raw, batch.klen, eps, h.dtype, rec=rec).run().operand(), self.w_out, to)

    def prefill(self, h, batch, rope, cache_rows, states, eps):
        g = self.geom
        y = self.w_in.matmul(h)
        z = torch.nn.functional.linear(y[:, g.a_off:g.a_off + g.rank], self.a2)
        gcum = oh.decay_prepare(z, self.a2_b, 1.0 / self.spec.tau, batch)
        o = oh.recurrence(y[:, :g.k_off], y[:, g.k_off:g.v_off], y[:, g.v_off:g.gate_off], g, states["state"], batch, gcum=gcum,
                          q_scale=self.q_scale)
        act = torch.empty(h.shape[0], self.w_out.k, dtype=h.dtype, device=h.device)
        oh.group_norm(o, self.norm_w, g.H, g.v_real, g, act, eps, gate=y[:, g.gate_off:g.a_off], shared_w=True)
        return self.w_out.matmul(act)


MIXERS = {"parallel": ParallelMixer, "gla": LinearAttentionMixer}


class GatedFeedForward:
    """gelu(gate) * up, down; gate and up rows interleaved in eights (ops_tile.interleave_glu)."""

    def __init__(self, ff, get, W, dtype):
        F = oh.pad32(ff)
        self.w_gu = TileWeight(oh.interleave_glu(grow(get("gate").to(dtype), F, W), grow(get("up").to(dtype), F, W)))
        self.w_down = TileWeight(grow(get("down").to(dtype), W, F))

    def decode(self, h, to=None):
        return oh.result_of(oh.gelu_glu_of(h, self.w_gu), self.w_down, to)

    def prefill(self, h):
        act = self.w_gu.glu_matmul(h)
        return self.w_down.matmul(oh.glu(self.w_gu.matmul(h)) if act is None else act)


def one_plus(w, n):
    """Norm weights are stored as their distance from one."""
    return grow(1.0 + w.float(), n)


class HybridLayer:
    """One layer's weights in the forms the kernels take."""

    def __init__(self, spec, width, get, dtype):
        W = oh.pad32(width)
        self.spec = spec
        self.mixer = MIXERS[spec.mixer.type](spec.mixer, lambda n: get("mix." + n), W, dtype)
        self.norm1, self.hc1 = one_plus(get("norm1"), W), Connection(get, "hc1")
        self.ff = None
        if spec.ff:
            self.ff = GatedFeedForward(spec.ff, lambda n: get("mlp." + n), W, dtype)
            self.norm2, self.hc2 = one_plus(get("norm2"), W), Connection(get, "hc2")

    def weights(self):
        m = [self.mixer.w_in, self.mixer.w_out]
        return m + ([self.ff.w_gu, self.ff.w_down] if self.ff else [])


class HybridWeights:
    """Device-resident weights of the whole model in ``dtype`` (norm weights, stream factors, convolutions, decays fp32)."""

    def __init__(self, cfg, device, dtype):
        self.cfg, self.device, self.dtype = cfg, torch.device(device), dtype
        self.layers = []
        self.embed = self.logits = self.embed_norm = self.final_norm = self.final_in = None
        self.capture = None       # list -> the forward appends the sum of the streams after every layer (comparisons)

    def shapes(self, sd=None):
        """Tensor name -> shape of a checkpoint (``sd``: where sizes that only tensors tell are looked up)."""
        c, d, S = self.cfg, self.cfg.hidden_size, self.cfg.streams
        out = {"embed": (c.vocab_size, d), "embed.norm": (d,), "final.norm": (d,)}
        for i, s in enumerate(c.layers):
            p = f"l{i}."
            a1 = None if sd is None else sd.get(p + "mix.a1")
            out.update({p + "mix." + n: shape for n, shape in MIXERS[s.mixer.type].shapes(s.mixer, d, None if a1 is None else a1.shape[0]).items()})
            out[p + "norm1"] = (d,)
            if s.ff:
                out.update({p + "norm2": (d,), p + "mlp.gate": (s.ff, d), p + "mlp.up": (s.ff, d), p + "mlp.down": (d, s.ff)})
            for q in ("hc1", "hc2") if s.ff else ("hc1",):
                out.update({f"{p}{q}.in": (S,), f"{p}{q}.out": (S,), f"{p}{q}.mix": (S, S)})
        return out

    def _build(self, get):
        c, d = self.cfg, oh.pad32(self.cfg.hidden_size)
        embed = grow(get("embed").to(self.dtype), c.vocab_size, d)
        self.embed = embed.contiguous()
        self.logits = TileWeight(grow(embed, oh.pad32(c.vocab_size), d), packed_only=True)
        self.embed_norm, self.final_norm = one_plus(get("embed.norm"), d), one_plus(get("final.norm"), d)
        self.final_in = torch.ones(c.streams, dtype=torch.float32, device=self.device)
        self.layers = [HybridLayer(s, c.hidden_size, lambda n, i=i: get(f"l{i}." + n), self.dtype) for i, s in enumerate(c.layers)]
        return self

    def load_state_dict(self, sd):
        want = self.shapes(sd)
        missing = [n for n in want if n not in sd]
        if missing:
            raise KeyError(f"checkpoint lacks {missing[:4]}{' ...' if len(missing) > 4 else ''}")
        for n, s in want.items():
            if tuple(sd[n].shape) != s:
                raise ValueError(f"{n}: shape {tuple(sd[n].shape)}, the configuration says {s}")
        return self._build(lambda n: sd[n].to(self.device))

    def init_random(self, seed):
        """Gaussian weights with 1 / sqrt(fan-in) scale, unit norms, streams that mean the plain residual sum, decays between fast and
        slow; one generator per tensor (order does not matter)."""
        want, S = self.shapes(), self.cfg.streams

        def get(n):
            s, leaf = want[n], n.rsplit(".", 1)[-1]
            if ".hc" in n:
                w = {"in": torch.ones(S) / S, "out": torch.ones(S), "mix": torch.eye(S)}[leaf]
                return w.to(self.device)
            if leaf in ("norm1", "norm2") or n in ("embed.norm", "final.norm") or n.endswith("conv.b"):
                return torch.zeros(s, device=self.device)
            if leaf in ("norm", "D"):
                return torch.ones(s, device=self.device)
            if leaf == "A_log":
                return torch.log(torch.linspace(1.0, 16.0, s[0], device=self.device))
            if leaf == "dt_bias":
                return torch.linspace(-6.0, -2.0, s[0], device=self.device)
            if n.endswith("a2.b"):
                return torch.full(s, 2.0, device=self.device)
            g = torch.Generator(device=self.device)
            g.manual_seed((seed * 1000003 + zlib.crc32(n.encode())) % (2 ** 31))
            std = 0.02 if n == "embed" else s[1] ** -0.5
            return torch.randn(s, generator=g, device=self.device, dtype=torch.float32) * std
        return self._build(get)

    def nbytes(self):
        return self.embed.numel() * self.embed.element_size() + sum(w.nbytes() for L in self.layers for w in L.weights()) + self.logits.nbytes()
