"""Kemurax on the HIP ops: several residual streams; layers mix tokens by gated linear attention, or by chunked grouped-query
attention and a state-space recurrence side by side.

Same surface as the other target models (``from_pretrained`` / ``from_state_dict`` / ``init_random``, ``model(input_ids=,
kv_cache=).logits`` for one sequence), plus ``forward_batch`` for a batch of sequences that is described by a
``models.cache.PagedBatch``.  Residual streams, norms, rotation, softmax, gates, decays and recurrent states are fp32; matrix
products run in the model's dtype (bfloat16, or float32 throughout) with fp32 accumulation.
"""
import torch

from .. import ops_hybrid as oh
from .config_kemurax import KemuraxConfig
from .hybrid_core import HybridWeights
from .llama_core import CausalLMOutput, load_checkpoint_state_dict, parse_random_spec
from .rotary import RotaryTable


class KemuraxForCausalLM:
    supports_speculation = False                   # a recurrent state cannot be rolled back to an accepted prefix: served autoregressively
    prepares_steps = True                          # a decode step's first launch takes PagedBatch.prep

    def __init__(self, config: KemuraxConfig, device="cuda:0", dtype=torch.bfloat16):
        if dtype not in (torch.bfloat16, torch.float32):
            raise ValueError(f"dtype must be bfloat16 or float32, got {dtype}")
        self.config, self.device, self.dtype = config, torch.device(device), dtype
        self.vocab_size = config.vocab_size
        self.weights = HybridWeights(config, self.device, dtype)
        self._rope = {}
        self.max_positions = 0

    # -- construction ------------------------------------------------------------------------
    @classmethod
    def from_pretrained(cls, name_or_path, torch_dtype=torch.bfloat16, device_map="cuda:0", config=None, **_):
        """Local checkpoint directory, or ``random:<seed>`` with an explicit ``config``."""
        seed = parse_random_spec(name_or_path)
        if seed is not None:
            assert config is not None, "random:<seed> needs config="
            return cls(config, device_map, torch_dtype).init_random(seed)
        m = cls(config or KemuraxConfig.from_pretrained(name_or_path), device_map, torch_dtype)
        m.weights.load_state_dict(load_checkpoint_state_dict(name_or_path))
        return m

    @classmethod
    def from_state_dict(cls, config, sd, device="cuda:0", dtype=torch.bfloat16):
        m = cls(config, device, dtype)
        m.weights.load_state_dict(sd)
        return m

    def init_random(self, seed):
        self.weights.init_random(seed)
        return self

    def eval(self):
        return self

    # -- cache, and the sizes it asks for ----------------------------------------------------
    def make_cache(self, max_budget, max_batch=64):
        from .cache import HybridCache
        return HybridCache(self, max_budget=max_budget, max_batch=max_batch)

    def cache_widths(self):
        """Elements of one cached row per layer (0: the layer keeps nothing per token)."""
        return [L.mixer.cache_width() for L in self.weights.layers]

    def state_shapes(self):
        """What a sequence keeps per layer whatever its length."""
        return [L.mixer.state_shapes() for L in self.weights.layers]

    def segment_tokens(self, tokens):
        """Tokens per segment of the recurrences in a forward over ``tokens`` new tokens: long enough that the smallest of them
        fills the chip once (two workgroups per CU, one per head, 64 value columns and segment)."""
        units = min(L.mixer.recurrence_units() for L in self.weights.layers)
        return max(4, -(-tokens * units // (512 * oh.CHUNK))) * oh.CHUNK

    def prepare_positions(self, n):
        """Rotary tables for positions 0 .. n-1 (called by the cache: captured graphs keep the tables' addresses)."""
        if n > self.max_positions:
            self.max_positions = n
            specs = {s.mixer.left.rot.key(): s.mixer.left.rot for s in self.config.layers if s.mixer.type == "parallel"}
            self._rope = {k: RotaryTable(s, n, self.device) for k, s in specs.items()}

    def _rope_of(self, spec):
        return self._rope[spec.mixer.left.rot.key()] if spec.mixer.type == "parallel" else None

    # -- forward -----------------------------------------------------------------------------
    @torch.inference_mode()
    def __call__(self, input_ids, kv_cache=None, graph_cache=None, position_ids=None, **_):
        return self.forward(input_ids, kv_cache)

    def forward(self, input_ids, kv_cache, graph_cache=None, position_ids=None, last_rows=None):
        """One sequence (the cache's default one), ``input_ids`` (1, n): appends n tokens, logits (1, rows, V) of the trailing
        ``last_rows`` (default: all)."""
        n = input_ids.shape[1]
        batch = kv_cache.plan_prefill([(kv_cache.DEFAULT, n, range(0 if last_rows is None else max(0, n - last_rows), n))])
        return CausalLMOutput(self.forward_batch(input_ids.reshape(-1).to(self.device), batch, kv_cache).unsqueeze(0))

    @torch.inference_mode()
    def forward_batch(self, ids, batch, cache):
        """ids int64 [tokens of the batch]; returns fp32 logits [wanted tokens, V] (None when nothing is wanted)."""
        W, eps, width = self.weights, self.config.eps, self.config.hidden_size
        x = torch.empty(ids.numel(), self.config.streams, oh.pad32(width), dtype=torch.float32, device=self.device)
        first = dict(embed=W.embed, ids=ids, embed_w=W.embed_norm)
        y = hc = None

        def read(x, connection, norm, wt, epi):
            """The last sublayer's result into the streams, the next sublayer's input, which goes through wt, out of them: (input, streams)."""
            if batch.decode and hc is not None and W.capture is None and oh.Connect.takes(x, wt, epi):
                h = oh.Connect(x, connection.u_in, norm, eps, width, y, hc.out, hc.mix)
                return h, h.out
            before = dict(first, prep=batch.prep) if hc is None else dict(y=y, out=hc.out, mix=hc.mix)
            return oh.connect(x, connection.u_in, norm, eps, width, self.dtype, octets=batch.decode, **before), x
        fused = batch.decode and W.capture is None and batch.want is None

        def goes(hc, wt, following):
            """Where the sublayer that ends with wt takes its result if that is the next one's input already (ops_hybrid.Streams)."""
            if not fused:
                return {}
            connection, norm, after, epi = following
            ok = oh.Streams.takes(x, wt, after, epi)
            return dict(to=oh.Streams(x, hc.out, hc.mix, connection, norm, eps, width, keep=after is not W.logits)) if ok else {}
        last = (W.final_in, W.final_norm, W.logits, "f32")
        for i, L in enumerate(W.layers):
            following = (W.layers[i + 1].hc1.u_in, W.layers[i + 1].norm1, W.layers[i + 1].mixer.w_in, "f32") if i + 1 < len(W.layers) else last
            h, x = (y, x) if isinstance(y, oh.Scaled) else read(x, L.hc1, L.norm1, L.mixer.w_in, "f32")
            if W.capture is not None and i > 0:
                W.capture.append(x.sum(1)[:, :width])
            run = L.mixer.decode if batch.decode else L.mixer.prefill
            to = goes(L.hc1, L.mixer.w_out, following if L.ff is None else (L.hc2.u_in, L.norm2, L.ff.w_gu, "glu"))
            y, hc = run(h, batch, self._rope_of(L.spec), cache.rows[i], cache.states[i], eps, **to), L.hc1
            if L.ff is not None:
                h, x = (y, x) if isinstance(y, oh.Scaled) else read(x, L.hc2, L.norm2, L.ff.w_gu, "glu")
                y, hc = (L.ff.decode if batch.decode else L.ff.prefill)(h, **goes(L.hc2, L.ff.w_down, following)), L.hc2
        if isinstance(y, oh.Scaled):
            return y.linear(W.logits, self.vocab_size)
        if batch.want is not None and batch.want.numel() == 0:
            return None
        if batch.want is not None:
            x, y = x[batch.want], y[batch.want]
        if batch.decode and W.capture is None and oh.Connect.takes(x, W.logits, "f32"):
            return oh.Connect(x, W.final_in, W.final_norm, eps, width, y, hc.out, hc.mix, keep=False).linear(W.logits, self.vocab_size)
        h = oh.connect(x, W.final_in, W.final_norm, eps, width, self.dtype, y=y, out=hc.out, mix=hc.mix, keep=W.capture is not None)
        if W.capture is not None:
            W.capture.append(x.sum(1)[:, :width])
        return oh.linear_f32(h, W.logits, self.vocab_size)
