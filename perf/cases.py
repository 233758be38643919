"""The work that programs have this framework do, as cases that can be timed and checked.

Three model families are served.  The Llama targets (fp16) run the speculative loop on one GPU: the prompt in chunks, the build of
the retrieval cache, then per step a few draft forwards, a few verifies against the retrieval cache and one verify against the whole
cache.  Befidra and Kemurax (bfloat16, float32 for traces that are compared digit by digit) are served in batches: prompts packed
into forwards, then lockstep decoding through one captured graph.

A model here has four layers of its real size instead of 32 or 40: weights and caches are still several times what the chip's caches
hold, and every layer is like the others.  Weights are random with the spread that trained ones have; cached keys and values have the
spread that the model's own projections give.
"""
import json
import math

import torch
import torch.nn.functional as F

from triforce_amd.models import registry, zoo

LAYERS = 4
START, RECENT_BUDGET = 16, 256                      # the draft's window: sinks, sinks + recent + gamma
CHUNK = 8                                           # keys per retrieval chunk
STEPS = 8                                           # lockstep tokens of one decode case: what is between two scheduler decisions
VOCAB = 32000


# ---- the cases ------------------------------------------------------------------------------------------------------------------
def listed():
    return [
        # one token drafted by the 68M model, the launch that a speculative step has most of
        dict(name="draft step", path="draft", tokens=3),
        # six drafted tokens checked against the retrieval cache of 4096 keys per head
        dict(name="retrieval verify", path="retrieval", model="llama-7B-128K", gamma=6, budget=4096),
        # the same tokens checked against a 122K-token context: what bounds the speculative loop
        dict(name="full verify 122k", path="verify", model="llama-7B-128K", gamma=6, context=124928),
        # the retrieval cache chosen out of that context for one query, every layer
        dict(name="retrieval build 122k", path="build", model="llama-7B-128K", context=124928, budget=4096),
        # a prompt of ordinary length, and the late part of a long one
        dict(name="llama prompt 3100", path="prompt", model="llama-7B-128K", tokens=3100, past=0),
        dict(name="llama prompt 4096 at 60k", path="prompt", model="llama-7B-128K", tokens=4096, past=61440),
        # one user's answer, and a server's full batch, with contexts of unequal length (the longest is given)
        dict(name="befidra decode 1", path="decode", model="befidra-7B", dtype="bfloat16", batch=1, context=4000),
        dict(name="befidra decode 32", path="decode", model="befidra-7B", dtype="bfloat16", batch=32, context=4000),
        # prompts of several users in one forward
        dict(name="befidra prompts 6", path="prompts", model="befidra-7B", dtype="bfloat16", batch=6, tokens=4000, past=0),
        # a batch of middle size whose contexts reach over the attention's chunk of 8192
        dict(name="kemurax decode 8", path="decode", model="kemurax-7B", dtype="bfloat16", batch=8, context=9000),
        # a document: two forwards, the second one goes on from the first one's states
        dict(name="kemurax prompt 8000", path="prompts", model="kemurax-7B", dtype="bfloat16", batch=1, tokens=8000, past=0),
        # a trace in 32 bits throughout
        dict(name="kemurax float32 700", path="prompts", model="kemurax-7B", dtype="float32", batch=2, tokens=700, past=0),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    path = rng.choice(["draft", "retrieval", "verify", "build", "prompt", "decode", "decode", "prompts", "prompts"])
    llama = rng.choice(["llama-7B-128K", "llama-7B-128K", "llama-13B-128K"])
    if path == "draft":
        return dict(path=path, tokens=rng.randint(1, 8))
    if path == "retrieval":
        return dict(path=path, model=llama, gamma=rng.randint(2, 16), budget=CHUNK * _log(rng, 32, 1536))
    if path == "verify":
        return dict(path=path, model="llama-7B-128K", gamma=rng.randint(2, 16), context=_log(rng, 1000, 124928))
    if path == "build":
        context = CHUNK * _log(rng, 512, 15616)
        return dict(path=path, model="llama-7B-128K", context=context, budget=CHUNK * min(_log(rng, 32, 1536), context // CHUNK // 2))
    if path == "prompt":
        return dict(path=path, model="llama-7B-128K", tokens=_log(rng, 129, 4096), past=rng.choice([0, _log(rng, 100, 61440)]))
    model, dtype = rng.choice(["befidra-7B", "kemurax-7B"]), rng.choice(["bfloat16", "bfloat16", "bfloat16", "float32"])
    if path == "decode":
        batch = _log(rng, 1, 32)
        return dict(path=path, model=model, dtype=dtype, batch=batch, context=_log(rng, 100, min(32768, 200000 // batch)))
    batch = _log(rng, 1, 12)
    tokens = _log(rng, max(40, 3 * batch), 1200 if dtype == "float32" else 6000)
    return dict(path=path, model=model, dtype=dtype, batch=batch, tokens=tokens, past=rng.choice([0, 0, _log(rng, 50, 6000 // batch)]))


def _contexts(case):
    """Cached tokens of every sequence of a decode case: between half of the context and all of it."""
    c = case["context"]
    return [c - c * (b * 7 % 16) // 32 for b in range(case["batch"])]


def _prompts(case):
    """New tokens of every sequence: unequal parts of the total."""
    parts = [1 + b * 5 % 7 for b in range(case["batch"])]
    n = [max(1, case["tokens"] * p // sum(parts)) for p in parts]
    n[0] += case["tokens"] - sum(n)
    return n


# ---- inputs: made from the seed alone -------------------------------------------------------------------------------------------
class _Draw:
    def __init__(self, seed, dtype):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)
        self.dtype = dtype

    def normal(self, *shape, std=1.0, dtype=None):
        return torch.empty(*shape, dtype=dtype or self.dtype, device="cuda").normal_(0.0, std, generator=self.g)

    def near_one(self, n, dtype=None):
        return (1.0 + self.normal(n, std=0.1, dtype=torch.float32)).to(dtype or self.dtype)

    def ids(self, *shape):
        return torch.randint(0, VOCAB, shape, generator=self.g, device="cuda")


def _dict(name, layers=LAYERS):
    d = json.loads(json.dumps(zoo.CONFIGS[name]))
    if "layers" in d:
        d["layers"] = d["layers"][:layers]
        if d.get("loop"):                           # the loop runs the middle layers twice
            d["loop"] = dict(start=1, stop=3, times=2)
    else:
        d["num_hidden_layers"] = min(layers, d["num_hidden_layers"])
    return d


def _llama_weights(d, r):
    W, I = d["hidden_size"], d["intermediate_size"]
    sd = {"model.embed_tokens.weight": r.normal(VOCAB, W, std=0.02), "lm_head.weight": r.normal(VOCAB, W, std=3.0 * W ** -0.5),
          "model.norm.weight": r.near_one(W)}
    for i in range(d["num_hidden_layers"]):
        p = f"model.layers.{i}."
        for n, s in (("self_attn.q_proj", (W, W)), ("self_attn.k_proj", (W, W)), ("self_attn.v_proj", (W, W)), ("self_attn.o_proj", (W, W)),
                     ("mlp.gate_proj", (I, W)), ("mlp.up_proj", (I, W)), ("mlp.down_proj", (W, I))):
            sd[p + n + ".weight"] = r.normal(*s, std=s[1] ** -0.5)
        for n in ("input_layernorm", "post_attention_layernorm"):
            sd[p + n + ".weight"] = r.near_one(W)
    return sd


def _befidra_weights(d, r):
    W, side = d["width"], d["token_side"]["dim"]
    sd = {"embed": r.normal(VOCAB, W, std=0.02), "final.norm": r.near_one(W), "loop.step": r.normal(d["loop"]["times"], W, std=0.1),
          "side.embed": r.normal(VOCAB, len(d["layers"]) * side)}
    for i, L in enumerate(d["layers"]):
        m, ff = L["mixer"], L["mlp"]["ff"]
        H, N, R, V, Q, C = (m[k] for k in ("heads", "dim", "rot_dim", "vdim", "q_rank", "kv_rank"))
        for n, s in (("mix.dq", (Q, W)), ("mix.uq", (H * (N + R), Q)), ("mix.dkv", (C + R, W)), ("mix.uk", (H * N, C)), ("mix.uv", (H * V, C)),
                     ("mix.g", (H * V, W)), ("mix.o", (W, H * V)), ("mlp.up", (ff, W)), ("mlp.down", (W, ff)), ("side.gate", (side, W)),
                     ("side.proj", (W, side))):
            sd[f"l{i}.{n}"] = r.normal(*s, std=s[1] ** -0.5)
        for n, s in (("norm1", W), ("mix.dq.norm", Q), ("mix.dkv.norm", C), ("side.norm", W)):
            sd[f"l{i}.{n}"] = r.near_one(s, torch.float32)
    return sd


def _kemurax_weights(d, r):
    W, S, f32 = d["width"], d["streams"], torch.float32
    sd = {"embed": r.normal(VOCAB, W, std=0.02), "embed.norm": r.normal(W, std=0.1, dtype=f32), "final.norm": r.normal(W, std=0.1, dtype=f32)}
    for i, L in enumerate(d["layers"]):
        p, ff, m = f"l{i}.", L["mlp"]["ff"], L["mixer"]
        mats = [("mlp.gate", (ff, W)), ("mlp.up", (ff, W)), ("mlp.down", (W, ff))]
        if L["type"] == "gla":
            n, v = m["heads"] * m["dim"], m["heads"] * m["vdim"]
            mats += [("mix.q", (n, W)), ("mix.k", (n, W)), ("mix.v", (v, W)), ("mix.g", (v, W)), ("mix.o", (W, v)), ("mix.a1", (m["rank"], W)),
                     ("mix.a2", (n, m["rank"]))]
            sd[p + "mix.a2.b"] = 2.0 + r.normal(n, std=0.5, dtype=f32)
            sd[p + "mix.norm"] = r.near_one(m["vdim"], f32)
        else:
            a, s = m["left"], m["right"]
            inner, gn = s["heads"] * s["vdim"], s["groups"] * s["state"]
            mats += [("mix.left.q", (a["heads"] * a["dim"], W)), ("mix.left.k", (a["kv_heads"] * a["dim"], W)),
                     ("mix.left.v", (a["kv_heads"] * a["vdim"], W)), ("mix.left.g", (a["heads"] * a["vdim"], W)),
                     ("mix.left.o", (W, a["heads"] * a["vdim"])), ("mix.right.in", (2 * inner + 2 * gn + s["heads"], W)),
                     ("mix.right.o", (W, inner))]
            sd.update({p + "mix.left.q.norm": r.near_one(a["dim"], f32), p + "mix.left.k.norm": r.near_one(a["dim"], f32),
                       p + "mix.right.conv": r.normal(inner + 2 * gn, s["conv"], std=s["conv"] ** -0.5, dtype=f32),
                       p + "mix.right.conv.b": r.normal(inner + 2 * gn, std=0.1, dtype=f32),
                       p + "mix.right.dt_bias": torch.linspace(-6.0, -2.0, s["heads"], device="cuda"),
                       p + "mix.right.A_log": torch.log(torch.linspace(1.0, 16.0, s["heads"], device="cuda")),
                       p + "mix.right.D": r.near_one(s["heads"], f32), p + "mix.right.norm": r.near_one(inner, f32)})
        for n, s in mats:
            sd[p + n] = r.normal(*s, std=s[1] ** -0.5)
        for n in ("1", "2"):
            sd[p + "norm" + n] = r.normal(W, std=0.1, dtype=f32)
            sd[p + f"hc{n}.in"] = 1.0 / S + r.normal(S, std=0.05, dtype=f32)
            sd[p + f"hc{n}.out"] = r.near_one(S, f32)
            sd[p + f"hc{n}.mix"] = torch.eye(S, device="cuda") + r.normal(S, S, std=0.05, dtype=f32)
    return sd


def _inputs(case, seed):
    """Everything that is drawn, the same for the framework and for the check: (config dict, weights, the case's own inputs)."""
    path = case["path"]
    r = _Draw(seed, getattr(torch, case.get("dtype", "float16")))
    d = _dict(case.get("model", "llama-68M"))
    if path == "build":
        H, D = d["num_attention_heads"], d["hidden_size"] // d["num_attention_heads"]
        return d, None, dict(q=r.normal(LAYERS, H, D, std=1.3), cache=_llama_rows(d, case["context"], r))
    if path in ("draft", "retrieval", "verify", "prompt"):
        sd = _llama_weights(d, r)
        n = {"draft": case.get("tokens"), "prompt": case.get("tokens")}.get(path) or case["gamma"] + 1
        past = {"draft": START + _recent(6), "retrieval": case.get("budget"), "verify": case.get("context"), "prompt": case.get("past")}[path]
        return d, sd, dict(ids=r.ids(1, n), cache=_llama_rows(d, past, r))
    sd = (_befidra_weights if "token_side" in d else _kemurax_weights)(d, r)
    past = _contexts(case) if path == "decode" else [case["past"]] * case["batch"]
    new = [STEPS] * case["batch"] if path == "decode" else _prompts(case)
    x = dict(past=past, new=new, ids=[r.ids(n) for n in new])
    if "token_side" in d:
        runs = _befidra_runs(d)
        width = [d["layers"][i]["mixer"]["kv_rank"] + d["layers"][i]["mixer"]["rot_dim"] for i, _, _ in runs]
        x["rows"] = [[r.normal(p, w) for p in past] for w in width]
        return d, sd, x
    x["rows"], x["states"] = [], []
    for L in d["layers"]:
        m, B = L["mixer"], case["batch"]
        if L["type"] == "gla":
            x["rows"].append(None)
            x["states"].append(dict(state=r.normal(B, m["heads"], m["dim"], m["vdim"], dtype=torch.float32, std=3.0)))
            continue
        a, s = m["left"], m["right"]
        x["rows"].append([r.normal(p, a["kv_heads"] * (a["dim"] + a["vdim"])) for p in past])
        channels = s["heads"] * s["vdim"] + 2 * s["groups"] * s["state"]
        x["states"].append(dict(state=r.normal(B, s["heads"], s["state"], s["vdim"], dtype=torch.float32, std=0.3),
                                ring=r.normal(B, s["conv"], channels, dtype=torch.float32)))
    return d, sd, x


def _llama_rows(d, past, r):
    L, H = d["num_hidden_layers"], d["num_attention_heads"]
    shape = (L, H, past, d["hidden_size"] // H)
    return r.normal(*shape), r.normal(*shape)


def _recent(gamma):
    return RECENT_BUDGET - START - gamma


# ---- what a program has in hand ---------------------------------------------------------------------------------------------------
@torch.inference_mode()
def prepare(case, seed):
    d, sd, x = _inputs(case, seed)
    if "ids" in x and isinstance(x["ids"], list):
        return _prepare_batch(case, d, sd, x)
    from triforce_amd.models.cache import FlashSimpleCache, RetrievalCache, StreamingLLMEvictionCache
    from triforce_amd.models.modeling_llama import LlamaForCausalLM
    from triforce_amd.models.modeling_llama_68m import LlamaForCausalLM as Draft
    from triforce_amd.utils.graph_infer import GraphInferenceEngine
    path, gamma = case["path"], case.get("gamma", 6)
    k, v = x["cache"]
    if path == "build":
        model = LlamaForCausalLM(registry.config_from_dict(d))
        full = FlashSimpleCache(model, case["context"])
        full.k.copy_(k)
        full.v.copy_(v)
        full.seq_len = case["context"]
        return dict(case=case, q=x["q"], full=full, small=RetrievalCache(model, max_budget=case["budget"], prefill=case["context"], chunk_size=CHUNK,
                                                                        gamma=gamma))
    draft_dict = d if path == "draft" else _dict("llama-68M")
    target = LlamaForCausalLM(zoo.config("tiny")).init_random(seed) if path == "draft" else LlamaForCausalLM.from_state_dict(
        registry.config_from_dict(d), sd)
    draft = Draft(registry.config_from_dict(draft_dict), "cuda:0")
    if path == "draft":
        draft.weights.load_state_dict(sd)
    else:
        draft.init_random(seed)
    budget = {"draft": 64, "retrieval": case.get("budget")}.get(path, 64)
    full = FlashSimpleCache(target, {"verify": case.get("context", 0) + 32, "prompt": case.get("past", 0) + case.get("tokens", 0)}.get(path, 64))
    small = RetrievalCache(target, max_budget=budget, prefill=budget, gamma=gamma, chunk_size=CHUNK)
    window = StreamingLLMEvictionCache(draft, start_size=START, recent_size=_recent(gamma), gamma=gamma)
    engine = GraphInferenceEngine(target, full, small, draft, window)
    if path != "prompt":
        engine.initialize_cuda_graph(gamma, probs=True, temperature=0.6, top_p=0.9, verbose=False, capture_target=path == "verify")
    cache = {"draft": window, "retrieval": small}.get(path, full)
    cache.k[:, :, :k.shape[2]] = k
    cache.v[:, :, :k.shape[2]] = v
    s = dict(case=case, engine=engine, cache=cache, ids=x["ids"], at=k.shape[2])
    if path == "retrieval":                         # where the tokens stand: behind the whole prompt, which is longer than the budget
        s["pos"] = torch.arange(20000, 20000 + gamma + 1, device="cuda").unsqueeze(0)
    return s


def _prepare_batch(case, d, sd, x):
    from triforce_amd.utils.batch_infer import BatchInferenceEngine
    dtype = getattr(torch, case["dtype"])
    torch.backends.cuda.matmul.allow_tf32 = False   # float32 means float32
    cfg = registry.config_from_dict(d)
    model = registry.model_class(d["architecture"]).from_state_dict(cfg, sd, dtype=dtype)
    B, past, new = case["batch"], x["past"], x["new"]
    cache = model.make_cache(sum(past) + sum(new) + 64, max_batch=B)
    s = dict(case=case, engine=BatchInferenceEngine(model, cache), past=past, names=list(range(B)))
    if case["path"] == "decode":
        s["ids"] = [torch.stack([i[t] for i in x["ids"]]) for t in range(STEPS)]
    else:
        s["entries"] = [(b, i.tolist(), [new[b] - 1]) for b, i in enumerate(x["ids"])]
    s["new_rows"] = torch.zeros(1, dtype=torch.int64, device="cuda")
    run(s)                                          # an earlier request: the graph is captured, pages were in other hands
    s["new_rows"] = torch.cat([cache.cache_rows(b, past[b], new[b]) for b in range(B)]).to(torch.int64).cuda()
    for block, rows in zip(cache.rows, x["rows"]):
        for b in range(B):
            if rows is not None and past[b]:
                block[cache.cache_rows(b, 0, past[b]).to(torch.int64).cuda()] = rows[b]
    for have, given in zip(getattr(cache, "states", ()), x.get("states", ())):
        for n, t in given.items():                  # seats are handed out in order
            have[n][:B].copy_(t)
    return s


# ---- one pass -----------------------------------------------------------------------------------------------------------------------
@torch.inference_mode()
def run(s):
    case = s["case"]
    path = case["path"]
    if path in ("decode", "prompts"):
        return _run_batch(s)
    if path == "build":
        for i in range(s["q"].shape[0]):
            s["small"].init_graph_cache(s["full"], s["q"][i:i + 1], i)
        return dict(k=s["small"].k[:, :, :case["budget"]], v=s["small"].v[:, :, :case["budget"]])
    engine, cache, ids, at = s["engine"], s["cache"], s["ids"], s["at"]
    if path == "draft":
        out = engine.graph_draft_inference(ids, gamma_offset=ids.shape[1] - 1)
    elif path == "retrieval":
        out = engine.graph_verify(ids, s["pos"])
    else:
        cache.seq_len = at                          # the same tokens again, behind the same context
        out = engine.inference(ids)
    n = ids.shape[1]
    return dict(out=out, k=cache.k[:, :, at:at + n], v=cache.v[:, :, at:at + n])


def _run_batch(s):
    engine, cache = s["engine"], s["engine"].kv_cache
    engine.clear_kv()
    if any(s["past"]):
        cache.extend([(b, n) for b, n in zip(s["names"], s["past"]) if n])
    if s["case"]["path"] == "decode":
        logits = [engine.decode(s["names"], ids).clone() for ids in s["ids"]]
    else:
        logits = engine.step(s["entries"])
    out = dict(logits=logits, rows=[c.index_select(0, s["new_rows"]) for c in cache.rows if c is not None])
    if hasattr(cache, "states"):                    # these go on from pass to pass where there is a past, as in a longer answer
        out["states"] = [t for d in cache.states for t in d.values()]
    return out


# ---- what a pass cannot do without ------------------------------------------------------------------------------------------------
def work(case):
    path = case["path"]
    d = _dict(case.get("model", "llama-68M"))
    if "layers" not in d:
        W, I, L = d["hidden_size"], d["intermediate_size"], d["num_hidden_layers"]
        if path == "build":                         # all keys once, the chosen keys and values read and written
            return dict(bytes=L * W * 2 * (case["context"] + 4 * case["budget"]), flops=L * W * 3 * case["context"])
        per_layer = 4 * W * W + 3 * W * I
        n = case["tokens"] if "tokens" in case else case["gamma"] + 1
        past = {"draft": START + _recent(6), "retrieval": case.get("budget"), "verify": case.get("context"), "prompt": case.get("past")}[path]
        rows = {"draft": 1, "prompt": n - 128 * (-(-n // 128) - 1)}.get(path, n)
        weights = L * per_layer + VOCAB * W
        flops = 2 * n * L * per_layer + 2 * rows * VOCAB * W + L * 4 * W * (n * past + n * (n + 1) // 2)
        return dict(bytes=2 * (weights + L * 2 * W * (past + 2 * n)) + 4 * rows * VOCAB, flops=flops)
    size = 4 if case["dtype"] == "float32" else 2
    past = _contexts(case) if path == "decode" else [case["past"]] * case["batch"]
    new = [STEPS] * case["batch"] if path == "decode" else _prompts(case)
    tokens, wanted = sum(new), sum(new) if path == "decode" else case["batch"]
    passes = STEPS if path == "decode" else 1       # every decoded token needs all weights again
    W = d["width"]
    params, cached, flops = VOCAB * W, 0, 2 * wanted * VOCAB * W
    if "token_side" in d:
        for i, _, _ in _befidra_runs(d):
            m, ff, side = d["layers"][i]["mixer"], d["layers"][i]["mlp"]["ff"], d["token_side"]["dim"]
            H, N, R, V, Q, C = (m[k] for k in ("heads", "dim", "rot_dim", "vdim", "q_rank", "kv_rank"))
            p = W * (Q + C + R + 2 * H * V + 2 * ff + 2 * side) + H * (N + R) * Q + H * (N + V) * C
            pairs = sum(a * n + n * (n + 1) // 2 for a, n in zip(past, new))
            params, flops = params + p, flops + 2 * tokens * p + 2 * pairs * H * (N + R + V)
            cached += (C + R) * (sum(sum(range(a + 1, a + n + 1)) for a, n in zip(past, new)) if path == "decode" else sum(past) + tokens) + (C + R) * tokens
        return dict(bytes=size * (passes * params + cached) + 4 * wanted * VOCAB, flops=flops)
    state = 0
    for L in d["layers"]:
        m, ff = L["mixer"], L["mlp"]["ff"]
        if L["type"] == "gla":
            n, v = m["heads"] * m["dim"], m["heads"] * m["vdim"]
            p, N, V, H = W * (2 * n + 3 * v + m["rank"] + 3 * ff) + n * m["rank"], m["dim"], m["vdim"], m["heads"]
        else:
            a, s = m["left"], m["right"]
            inner, gn = s["heads"] * s["vdim"], s["groups"] * s["state"]
            p = W * (a["heads"] * (a["dim"] + 2 * a["vdim"]) + a["kv_heads"] * (a["dim"] + a["vdim"]) + 3 * inner + 2 * gn + s["heads"] + 3 * ff)
            N, V, H = s["state"], s["vdim"], s["heads"]
            seen = [[min(j, j % a["mask"]["size"]) + 1 for j in range(b, b + n)] for b, n in zip(past, new)]
            row = a["kv_heads"] * (a["dim"] + a["vdim"])
            flops += 2 * a["heads"] * (a["dim"] + a["vdim"]) * sum(map(sum, seen))
            cached += row * (tokens + (sum(map(sum, seen)) if path == "decode" else sum(min(b, b % a["mask"]["size"]) for b in past)))
        params, flops = params + p, flops + 2 * tokens * p + 4 * tokens * H * N * V
        state += case["batch"] * H * N * V * (2 * passes if any(past) else 1)
    return dict(bytes=size * (passes * params + cached) + 4 * (wanted * VOCAB + state), flops=flops)


# ---- how far another correct implementation may be ------------------------------------------------------------------------------
def tolerance(case):
    """About four times what is seen against 64 bits (below), by what the operands of the products are rounded to.  The build copies
    rows whose choice is defined down to the rounding of the scores."""
    if case["path"] == "build":
        return "exact"
    if case.get("dtype") == "float32":
        return {"rel": 2e-5, "max": 2e-3}
    if case.get("dtype") == "bfloat16":
        return {"rel": 0.025, "max": 0.4}
    return {"rel": 0.014, "max": 0.3}


# ---- the same in 64 bits ----------------------------------------------------------------------------------------------------------
def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _gelu(z):
    return F.gelu(z, approximate="tanh")


def _attend(q, k, v, scale, first, chunk=0):
    """Causal attention: q (n, H, D) at positions first .. on k (m, G, D), v (m, G, V) at positions 0 .. m - 1."""
    n, H, m = q.shape[0], q.shape[1], k.shape[0]
    k, v = (t.repeat_interleave(H // t.shape[1], 1).transpose(0, 1).contiguous() for t in (k, v))
    kt, out, at = k.transpose(1, 2).contiguous(), [], torch.arange(m, device="cuda")
    step = max(1, (1 << 27) // (H * m))
    for a in range(0, n, step):
        i = torch.arange(first + a, first + min(n, a + step), device="cuda")[:, None]
        hidden = (at[None] > i) if not chunk else (at[None] > i) | (at[None] // chunk != i // chunk)
        s = torch.matmul(q[a:a + step].transpose(0, 1).contiguous(), kt) * scale
        out.append(torch.matmul(torch.softmax(s.masked_fill_(hidden, float("-inf")), -1), v))
    return torch.cat(out, 1).transpose(0, 1)


def _halves(x, c, s):
    """Rotation of entries i and i + n of x (tokens, heads, 2n)."""
    u, w = x.chunk(2, -1)
    return torch.cat([u * c - w * s, w * c + u * s], -1)


def _llama_tables(d, pos):
    """cos / sin as the model defines them: angles in float32, values kept as float16."""
    D, base = d["hidden_size"] // d["num_attention_heads"], d.get("rope_theta", 10000.0)
    e, mscale = torch.arange(0, D, 2).float() / D, 1.0
    inv, y = 1.0 / (base ** e), d.get("rope_scaling")
    if y:
        def edge(turns):
            return D * math.log(y["original_max_position_embeddings"] / (turns * 2 * math.pi)) / (2 * math.log(base))
        low, high = max(math.floor(edge(32)), 0), min(math.ceil(edge(1)), D - 1)
        keep = 1 - torch.clamp((torch.arange(D // 2).float() - low) / (high - low), 0, 1)
        freq = base ** e
        inv = 1.0 / (y["factor"] * freq) * (1 - keep) + 1.0 / freq * keep
        mscale = 0.1 * math.log(y["factor"]) + 1.0
    a = torch.outer(pos.cpu().float(), inv)
    return [(f(a) * mscale).half().double().cuda().unsqueeze(1) for f in (torch.cos, torch.sin)]


def _llama_exact(case, d, sd, x):
    H, eps = d["num_attention_heads"], d["rms_norm_eps"]
    ids, (ck, cv), path = x["ids"][0], x["cache"], case["path"]
    n, past = ids.numel(), x["cache"][0].shape[2]
    D = d["hidden_size"] // H
    scale = float(1 / torch.sqrt(torch.tensor(D, dtype=torch.float16)))
    first = 20000 if path == "retrieval" else past
    cos, sin = _llama_tables(d, torch.arange(first, first + n))
    on_read = _llama_tables(d, torch.arange(past + n)) if path == "draft" else None     # the draft's cache keeps keys unrotated
    h, new_k, new_v = sd["model.embed_tokens.weight"][ids].double(), [], []
    for i in range(d["num_hidden_layers"]):
        def w(name):
            return sd[f"model.layers.{i}.{name}.weight"].double()
        u = _rms(h, eps) * w("input_layernorm")
        q, k, v = ((u @ w(f"self_attn.{c}_proj").T).view(n, H, D) for c in "qkv")
        q, k = _halves(q, cos, sin), k if on_read else _halves(k, cos, sin)
        new_k.append(k.transpose(0, 1))
        new_v.append(v.transpose(0, 1))
        k, v = (torch.cat([c[i].transpose(0, 1).double(), t]) for c, t in ((ck, k), (cv, v)))
        h = h + _attend(q, _halves(k, *on_read) if on_read else k, v, scale, past).reshape(n, H * D) @ w("self_attn.o_proj").T
        u = _rms(h, eps) * w("post_attention_layernorm")
        h = h + (F.silu(u @ w("mlp.gate_proj").T) * (u @ w("mlp.up_proj").T)) @ w("mlp.down_proj").T
    out = None                                      # after top-p a value may be in or out by its last digit
    if path in ("verify", "prompt"):
        rows = n - 128 * (-(-n // 128) - 1) if path == "prompt" else n
        out = (_rms(h[-rows:], eps) * sd["model.norm.weight"].double() @ sd["lm_head.weight"].double().T).unsqueeze(0)
    return dict(out=out, k=torch.stack(new_k), v=torch.stack(new_v))


def _befidra_runs(d):
    n, a, b, times = len(d["layers"]), *(d["loop"][k] for k in ("start", "stop", "times"))
    return [(i, None, False) for i in range(a)] + [(i, t, i == a) for t in range(times) for i in range(a, b)] + [(i, None, False) for i in range(b, n)]


def _frequencies(rot, bands):
    n, base, s = rot["dims"], rot["base"], rot.get("scaling")
    f = [base ** (-2.0 * i / n) for i in range(n // 2)]
    if s is None:
        return f, 1.0
    if bands:
        keep = [min(max((s["original"] * w / (2 * math.pi) - s["low"]) / (s["high"] - s["low"]), 0.0), 1.0) for w in f]
        return [w * k + w / s["factor"] * (1 - k) for w, k in zip(f, keep)], 1.0

    def edge(turns):
        return n * math.log(s["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))
    low, high = max(math.floor(edge(s["fast"])), 0), min(math.ceil(edge(s["slow"])), n - 1)
    ramp = [min(max((i - low) / max(high - low, 0.001), 0.0), 1.0) for i in range(n // 2)]
    return [w / s["factor"] * r + w * (1 - r) for w, r in zip(f, ramp)], 0.1 * math.log(s["factor"]) + 1.0


def _turns(rot, pos, bands):
    f, m = _frequencies(rot, bands)
    a = pos.double()[:, None] * torch.tensor(f, dtype=torch.float64, device="cuda")
    return (m * a.cos()).unsqueeze(1), (m * a.sin()).unsqueeze(1)


def _pairs(x, c, s):
    """Rotation of neighbouring entries."""
    u, w = x[..., 0::2], x[..., 1::2]
    return torch.stack([u * c - w * s, w * c + u * s], -1).flatten(-2)


def _befidra_exact(d, sd, x):
    eps, side, past, new = d["norm"]["eps"], d["token_side"]["dim"], x["past"], x["new"]
    ids, pos = torch.cat(x["ids"]), torch.cat([torch.arange(p, p + n, device="cuda") for p, n in zip(past, new)])
    h, rows = sd["embed"][ids].double(), []
    for r, (i, t, first) in enumerate(_befidra_runs(d)):
        def w(name):
            return sd[f"l{i}.{name}"].double()
        m = d["layers"][i]["mixer"]
        H, N, V, C, T = m["heads"], m["dim"], m["vdim"], m["kv_rank"], ids.numel()
        if first:
            h = h + sd["loop.step"][t].double()
        u = _rms(h, eps) * w("norm1")
        cos, sin = _turns(m["rot"], pos, False)
        q = (_rms(u @ w("mix.dq").T, eps) * w("mix.dq.norm") @ w("mix.uq").T).view(T, H, -1)
        q = torch.cat([q[..., :N], _pairs(q[..., N:], cos, sin)], -1)
        kv = u @ w("mix.dkv").T
        own = torch.cat([_rms(kv[:, :C], eps) * w("mix.dkv.norm"), _pairs(kv[:, C:].unsqueeze(1), cos, sin).squeeze(1)], -1)
        rows.append(own)
        o, at = [], 0
        for b, (p, n) in enumerate(zip(past, new)):
            c = torch.cat([x["rows"][r][b].double(), own[at:at + n]])
            k = torch.cat([(c[:, :C] @ w("mix.uk").T).view(-1, H, N), c[:, None, C:].expand(-1, H, -1)], -1)
            o.append(_attend(q[at:at + n], k, (c[:, :C] @ w("mix.uv").T).view(-1, H, V), m["scale"], p))
            at += n
        o = torch.cat(o).reshape(T, H * V) * torch.sigmoid(u @ w("mix.g").T)
        h = h + o @ w("mix.o").T + _gelu(u @ w("mlp.up").T) @ w("mlp.down").T
        e = sd["side.embed"][ids][:, i * side:(i + 1) * side].double()
        h = h + _rms((_gelu(h @ w("side.gate").T) * e) @ w("side.proj").T, eps) * w("side.norm")
    return _rms(h, eps) * sd["final.norm"].double(), rows, None


def _scalar_recurrence(v, k, q, dt, log, S, chunk=256):
    """S = exp(log) S + dt k v^T, o = S^T q: v (T, H, V), k / q (T, H, N), dt / log (T, H), S (H, N, V)."""
    out = []
    for a in range(0, v.shape[0], chunk):
        vv, kk, qq = (t[a:a + chunk].transpose(0, 1).contiguous() for t in (v, k * dt[..., None], q))
        g = log[a:a + chunk].cumsum(0).T
        p = torch.exp((g[:, :, None] - g[:, None, :]).clamp(max=0.0)).tril() * (qq @ kk.transpose(1, 2).contiguous())
        out.append((p @ vv + (qq * g.exp()[..., None]) @ S).transpose(0, 1))
        S = S * g[:, -1].exp()[:, None, None] + (kk * (g[:, -1:] - g).exp()[..., None]).transpose(1, 2).contiguous() @ vv
    return torch.cat(out), S


def _channel_recurrence(v, k, q, log, S, chunk=64):
    """S = diag(exp(log)) S + k v^T, o = S^T q: log (T, H, N)."""
    out = []
    for a in range(0, v.shape[0], chunk):
        vv, kk, qq, g = (t[a:a + chunk].transpose(0, 1).contiguous() for t in (v, k, q, log))
        g = g.cumsum(1)
        p = ((qq * g.exp()) @ (kk * (-g).exp()).transpose(1, 2).contiguous()).tril()
        out.append((p @ vv + (qq * g.exp()) @ S).transpose(0, 1))
        S = S * g[:, -1].exp()[..., None] + (kk * (g[:, -1:] - g).exp()).transpose(1, 2).contiguous() @ vv
    return torch.cat(out), S


def _kemurax_exact(d, sd, x):
    eps, past, new = d["norm"]["eps"], x["past"], x["new"]
    ids, pos = torch.cat(x["ids"]), torch.cat([torch.arange(p, p + n, device="cuda") for p, n in zip(past, new)])
    T, rows, states = ids.numel(), [], []
    spans = [(p, sum(new[:b]), n) for b, (p, n) in enumerate(zip(past, new))]

    def norm(t, name):
        return _rms(t, eps) * (1.0 + sd[name].double())
    h = norm(sd["embed"][ids].double(), "embed.norm").expand(d["streams"], -1, -1)
    for i, L in enumerate(d["layers"]):
        def w(name):
            return sd[f"l{i}.{name}"].double()

        def connect(h, n, sublayer):
            y = sublayer(norm(torch.einsum("s,std->td", w(f"hc{n}.in"), h), f"l{i}.norm{n}"))
            return torch.einsum("st,sxd->txd", w(f"hc{n}.mix"), h) + w(f"hc{n}.out")[:, None, None] * y

        def start(name, b, p):                      # a sequence without a past starts from nothing
            s = x["states"][i][name][b].double()
            return s if p else torch.zeros_like(s)

        def linear(u, m):
            H, N, V = m["heads"], m["dim"], m["vdim"]
            q, k, v = (u @ w("mix.q").T).view(T, H, N) * N ** -0.5, (u @ w("mix.k").T).view(T, H, N), (u @ w("mix.v").T).view(T, H, V)
            log = (F.logsigmoid(u @ w("mix.a1").T @ w("mix.a2").T + w("mix.a2.b")) / m["tau"]).view(T, H, N)
            got = [_channel_recurrence(v[a:a + n], k[a:a + n], q[a:a + n], log[a:a + n], start("state", b, p)) for b, (p, a, n) in enumerate(spans)]
            states.append(torch.stack([S for _, S in got]))
            o = _rms(torch.cat([o for o, _ in got]), eps) * w("mix.norm")
            return (o.reshape(T, H * V) * F.silu(u @ w("mix.g").T)) @ w("mix.o").T

        def parallel(u, m):
            a, s = m["left"], m["right"]
            H, G, D, V = (a[k] for k in ("heads", "kv_heads", "dim", "vdim"))
            cos, sin = _turns(a["rot"], pos, True)
            q, k = (_halves(_rms((u @ w(f"mix.left.{n}").T).view(T, -1, D), eps) * w(f"mix.left.{n}.norm"), cos, sin) for n in "qk")
            v, o = (u @ w("mix.left.v").T).view(T, G, V), []
            rows.append(torch.cat([k.reshape(T, -1), v.reshape(T, -1)], -1))
            for b, (p, f, n) in enumerate(spans):
                c = torch.cat([x["rows"][i][b].double(), rows[-1][f:f + n]])
                o.append(_attend(q[f:f + n], c[:, :G * D].reshape(-1, G, D), c[:, G * D:].reshape(-1, G, V), a["scale"], p, a["mask"]["size"]))
            left = (torch.cat(o).reshape(T, H * V) * torch.sigmoid(u @ w("mix.left.g").T)) @ w("mix.left.o").T
            H, V, N, G, taps = (s[k] for k in ("heads", "vdim", "state", "groups", "conv"))
            inner, gn = H * V, G * N
            z, xbc, dt = (u @ w("mix.right.in").T).split([inner, inner + 2 * gn, H], 1)
            dt, o, ends, rings = F.softplus(dt + w("mix.right.dt_bias")), [], [], []
            for b, (p, f, n) in enumerate(spans):
                ring = start("ring", b, p)
                seen = torch.cat([ring[[(p - taps + 1 + j) % taps for j in range(taps - 1)]], xbc[f:f + n]])
                for j in range(min(n, taps)):       # slot position % taps holds that position's input
                    ring[(p + n - 1 - j) % taps] = xbc[f + n - 1 - j]
                rings.append(ring)
                c = F.silu(sum(seen[j:j + n] * w("mix.right.conv")[:, j] for j in range(taps)) + w("mix.right.conv.b"))
                v, B, C = (t.reshape(n, -1, size) for t, size in zip(c.split([inner, gn, gn], 1), (V, N, N)))
                y, S = _scalar_recurrence(v, B.repeat_interleave(H // G, 1), C.repeat_interleave(H // G, 1), dt[f:f + n],
                                          -w("mix.right.A_log").exp() * dt[f:f + n], start("state", b, p))
                o.append(y + w("mix.right.D")[:, None] * v)
                ends.append(S)
            states.extend([torch.stack(ends), torch.stack(rings) if min(new) >= taps or all(past) else None])
            y = torch.cat(o).reshape(T, inner) * F.silu(z)
            y = _rms(y.view(T, s["norm_groups"], -1), eps).reshape(T, inner) * w("mix.right.norm")
            return m["left_scale"] * left + m["right_scale"] * (y @ w("mix.right.o").T)
        h = connect(h, 1, lambda u: (linear if L["type"] == "gla" else parallel)(u, L["mixer"]))
        h = connect(h, 2, lambda u: (_gelu(u @ w("mlp.gate").T) * (u @ w("mlp.up").T)) @ w("mlp.down").T)
    return norm(h.sum(0), "final.norm"), rows, states


@torch.inference_mode()
def exact(case, seed):
    d, sd, x = _inputs(case, seed)
    if case["path"] == "build":
        return None                                 # a choice and a copy
    if not isinstance(x["ids"], list):
        return _llama_exact(case, d, sd, x)
    h, rows, states = (_befidra_exact if "token_side" in d else _kemurax_exact)(d, sd, x)
    ends = torch.tensor(x["new"]).cumsum(0)
    if case["path"] == "decode":
        at = [torch.tensor([int(e) - n + t for e, n in zip(ends, x["new"])]) for t in range(STEPS)]
        logits = [h[i.cuda()] @ sd["embed"].double().T for i in at]
    else:
        logits = h[(ends - 1).cuda()] @ sd["embed"].double().T
    out = dict(logits=logits, rows=rows)
    return out if states is None else dict(out, states=states)
