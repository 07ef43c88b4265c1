"""Work that users of the engine have it do, as cases that can be timed and checked.

Every case is one or more calls of the engine's step function on a model of a published layer size with random weights
(as bench.py makes them) and seeded token ids:

  prompt   whole prompts read in one step, or one long prompt in portions of ``portion`` tokens, as the scheduler cuts it;
           the logits of each prompt's last token come back
  decode   one further token for each of ``requests`` requests whose contexts are in the cache already
  mixed    decoded tokens beside prompts in one step, what continuous batching makes of a serving load

``tokens`` is the mean length of the contexts (decode) or prompts; several requests have ragged lengths around it. The
sizes are bench.py's (batch 1 to 64, prompts of 20 to 2,048 tokens and more, layer sizes 0.6B and 8B, bfloat16) and
the float32 engine that replays and checks run. The engine of a model is made once for a process, as a server does.
"""
import math

import torch

from minivllm_amd.config import EngineConfig
from minivllm_amd.config.shapes import named_shape
from minivllm_amd.engine.executor import Executor
from minivllm_amd.engine.step import SeqStep
from minivllm_amd.models import config_from_dict, expected_tensors
from minivllm_amd.weights.device_random import DeviceRandomSource

MODELS = {"qwen3-0.6b": "0.6b", "qwen3-8b": "8b", "dutilix-0.6b": "dutilix-0.6b", "bolapel-0.6b": "bolapel-0.6b",
          "sorulix-0.6b": "sorulix-0.6b", "furanex-0.6b": "furanex-0.6b"}
# tokens the cache of an engine holds: four times the largest case of its model
CACHE_TOKENS = {"qwen3-0.6b": 360448, "qwen3-8b": 98304}
PAGE = 16


def listed():
    return [
        # one user chatting: the shortest step there is, bound by launches
        dict(name="chat decode", model="qwen3-0.6b", dtype="bfloat16", kind="decode", requests=1, tokens=300),
        # a loaded server between prompts: 64 ragged contexts
        dict(name="busy decode", model="qwen3-0.6b", dtype="bfloat16", kind="decode", requests=64, tokens=1100),
        # one request's prompt at the benchmark's size
        dict(name="prompt", model="qwen3-0.6b", dtype="bfloat16", kind="prompt", requests=1, tokens=2048, portion=8192),
        # continuous batching: 17 decoding requests while three short prompts arrive
        dict(name="mixed step", model="qwen3-0.6b", dtype="bfloat16", kind="mixed", requests=17, tokens=700, prompts=3,
             prompt_tokens=150),
        # the larger model serving a small batch: bound by the bytes of its weights
        dict(name="8b decode", model="qwen3-8b", dtype="bfloat16", kind="decode", requests=8, tokens=1024),
        # the larger model reading a batch of documents: the largest case
        dict(name="8b prompts", model="qwen3-8b", dtype="bfloat16", kind="prompt", requests=3, tokens=1333, portion=8192),
        # scores checked in full precision, as the trace tool's replays and tests do
        dict(name="float32 prompt", model="qwen3-0.6b", dtype="float32", kind="prompt", requests=1, tokens=200, portion=8192),
        # recurrent layers, latent attention and routed experts: a prompt, and a small batch decoding
        dict(name="dutilix prompt", model="dutilix-0.6b", dtype="bfloat16", kind="prompt", requests=1, tokens=2048, portion=8192),
        dict(name="dutilix decode", model="dutilix-0.6b", dtype="bfloat16", kind="decode", requests=8, tokens=1024),
        # a prompt longer than a step's budget, its state carried from portion to portion
        dict(name="bolapel prompt", model="bolapel-0.6b", dtype="bfloat16", kind="prompt", requests=1, tokens=2600, portion=2048),
        # two ragged prompts in a step
        dict(name="sorulix prompts", model="sorulix-0.6b", dtype="bfloat16", kind="prompt", requests=2, tokens=800, portion=8192),
        # experts named by token id, residual streams and latent attention
        dict(name="furanex prompt", model="furanex-0.6b", dtype="bfloat16", kind="prompt", requests=1, tokens=1000, portion=8192),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    model = rng.choice(["qwen3-0.6b"] * 4 + ["qwen3-8b"] * 2 + ["dutilix-0.6b"] * 2 + ["bolapel-0.6b", "sorulix-0.6b", "furanex-0.6b"])
    case = dict(model=model, dtype="bfloat16", kind=rng.choice(["prompt", "prompt", "decode", "decode", "mixed"]))
    if model == "qwen3-0.6b" and rng.random() < 0.15:
        return dict(case, dtype="float32", kind="prompt", requests=1, tokens=_log_uniform(rng, 16, 400), portion=8192)
    if case["kind"] == "prompt":
        requests = rng.choice([1, 1, 1, 2, 3, 5])
        most = 4000 if model.startswith("qwen3") else 2600
        portion = rng.choice([8192, 2048]) if requests == 1 else 8192
        return dict(case, requests=requests, tokens=_log_uniform(rng, 20, most) // requests + 1, portion=portion)
    requests = _log_uniform(rng, 1, 64 if model == "qwen3-0.6b" else 16)
    case.update(requests=requests, tokens=_log_uniform(rng, 20, 1100 if requests > 32 else 1900))
    if case["kind"] == "mixed":
        case.update(prompts=rng.randint(1, 4), prompt_tokens=_log_uniform(rng, 16, 300))
    return case


# --------------------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------------------
def _lengths(count, mean):
    """``count`` ragged lengths around ``mean``, the same for every seed."""
    if count == 1:
        return [mean]
    return [max(1, int(mean * (0.25 + 1.5 * ((0.618034 * (i + 1)) % 1.0)))) for i in range(count)]


def _requests(case, seed):
    """Token ids per request (a [n] list) and how many of its last tokens belong to the measured step."""
    vocab = named_shape(MODELS[case["model"]]).get("vocab_size") or named_shape(MODELS[case["model"]])["vocab"]
    if case["kind"] == "prompt":
        lens = [(n, n) for n in _lengths(case["requests"], case["tokens"])]
    else:
        lens = [(n + 1, 1) for n in _lengths(case["requests"], case["tokens"])]
        if case["kind"] == "mixed":
            lens += [(n, n) for n in _lengths(case["prompts"], case["prompt_tokens"])]
    gen = torch.Generator().manual_seed(int(seed))
    return [(torch.randint(0, vocab, (n,), generator=gen).tolist(), last) for n, last in lens]


class _Weights(DeviceRandomSource):
    """Random weights whose sizes are those of a trained model where it matters for how rounding grows from layer to
    layer: embeddings of unit size, and sublayers that add to the residual stream a part of what is there (projections
    and norms at a sublayer's end are small), not many times it."""

    def read(self, name):
        t = super().read(name)
        if name in ("embed", "model.embed_tokens.weight"):
            return (t.float() / self.std).to(t.dtype)
        if name.endswith((".o", ".down", "o_proj.weight", "down_proj.weight")):
            return t * 0.25
        if name.endswith(("norm1b", "norm2b")):
            return t * 0.125
        return t


def _model(case):
    raw = dict(named_shape(MODELS[case["model"]]), torch_dtype=case["dtype"])
    arch, cfg = config_from_dict(raw)
    stored = torch.float32 if case["dtype"] == "float32" else torch.bfloat16
    return raw, arch, cfg, _Weights(expected_tensors(arch, cfg), 1, stored, torch.device("cuda:0"),
                                    std=0.64 / cfg.hidden_size ** 0.5)


_engines = {}


class _Engine:
    def __init__(self, case):
        _, arch, cfg, source = _model(case)
        tokens = 8192 if case["dtype"] == "float32" else CACHE_TOKENS.get(case["model"], 98304)
        config = EngineConfig(model="", dtype=case["dtype"], max_model_len=4096, max_num_batched_tokens=8192,
                              max_num_batched_seqs=288, kv_cache_block_size=PAGE, kv_cache_num_blocks=tokens // PAGE)
        self.executor = Executor(config, model=(arch, cfg, source))
        self.manager = self.executor.new_cache_manager()
        self.next_id = 0


class _State:
    """Requests in the cache and the steps of one pass; gives its pages back when it goes."""

    def __init__(self, case, seed):
        key = (case["model"], case["dtype"])
        if key not in _engines:
            _engines[key] = _Engine(case)
        self.engine = engine = _engines[key]
        self.ids, self.steps = [], []
        ex, manager = engine.executor, engine.manager
        contexts, step = [], []
        for tokens, last in _requests(case, seed):
            rid, engine.next_id = engine.next_id, engine.next_id + 1
            self.ids.append(rid)
            manager.admit(rid)
            manager.reserve(rid, len(tokens))
            seq = manager.sequence(rid)
            share = dict(block_tables=[list(manager.block_table(rid, g)) for g in range(len(manager.groups))],
                         state_slot=seq.state_slot)
            n = len(tokens) - last
            if n:
                contexts.append(SeqStep(tokens=tokens[:n], start=0, want=[], **share))
            step.append(SeqStep(tokens=tokens[n:], start=n, want=[last - 1], **share))
        portion = case.get("portion", 1 << 30)
        if len(step) == 1 and len(step[0].tokens) > portion:
            s = step[0]
            for at in range(0, len(s.tokens), portion):
                part = s.tokens[at:at + portion]
                last = at + len(part) == len(s.tokens)
                self.steps.append([SeqStep(tokens=part, start=at, block_tables=s.block_tables, state_slot=s.state_slot,
                                           want=[len(part) - 1] if last else [])])
        else:
            self.steps.append(step)
        while contexts:                                     # contexts into the cache, up to 8,192 tokens a step
            batch = []
            while contexts and sum(len(s.tokens) for s in batch) + len(contexts[0].tokens) <= 8192:
                batch.append(contexts.pop(0))
            ex.step(batch)

    def __del__(self):
        for rid in self.ids:
            if rid in self.engine.manager:
                self.engine.manager.release(rid)


def prepare(case, seed):
    return _State(case, seed)


def run(state):
    logits = None
    for step in state.steps:
        logits = state.engine.executor.step(step)
    return logits


# --------------------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------------------
def work(case):
    raw, arch, cfg, source = _model(case)
    item = 4 if case["dtype"] == "float32" else 2
    requests = _requests(case, 0)
    n = sum(last for _, last in requests)                   # tokens computed
    wanted = len(requests)
    head_in_embed = not any(name in ("head", "lm_head.weight") for name in source.names())
    nbytes, flops = 0.0, 0.0
    for name in source.names():
        shape = source.shape(name)
        size = math.prod(shape)
        if name in ("embed", "model.embed_tokens.weight", "head", "lm_head.weight"):
            if head_in_embed or "head" in name:
                nbytes += size * item
                flops += 2.0 * wanted * size
            else:
                nbytes += n * shape[1] * item
        elif ".mlp.e" in name:                              # an expert: the share of tokens that use it
            router = raw["layers"][int(name[1:name.index(".")])]["mlp"]["router"]
            nbytes += size * item * min(1.0, n * router["top"] / router["experts"])
            flops += 2.0 * n * size * router["top"] / router["experts"]
        elif len(shape) == 2 and not source.is_integer(name) and not name.endswith(".conv"):
            nbytes += size * item
            flops += 2.0 * n * size
        elif not source.is_integer(name):
            nbytes += size * item
    pairs = sum(last * (len(t) - last) + last * (last + 1) / 2 for t, last in requests)
    keys = sum(len(t) for t, _ in requests)
    layers = raw.get("layers") or [dict(type="attention", mixer=dict(heads=cfg.num_attention_heads, kv_heads=cfg.num_key_value_heads,
                                                                    dim=cfg.head_dim, vdim=cfg.head_dim))] * cfg.num_hidden_layers
    for layer in layers:
        mixers = [layer["mixer"]] if "left" not in layer["mixer"] else [layer["mixer"]["left"], layer["mixer"]["right"]]
        for m in mixers:
            if layer["type"] == "latent_attention":
                nbytes += keys * (m["kv_rank"] + m["rot_dim"]) * item
                flops += 2.0 * pairs * m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"])
            elif layer["type"] == "attention" or (layer["type"] == "parallel" and "decay" not in m):
                share = 1.0
                if "mask" in m and len(requests) == 1:      # attention in chunks: a query sees its own
                    share = min(1.0, m["mask"]["size"] / len(requests[0][0]))
                nbytes += share * keys * m.get("kv_heads", m["heads"]) * (m["dim"] + m["vdim"]) * item
                flops += 2.0 * share * pairs * m["heads"] * (m["dim"] + m["vdim"])
            else:                                           # a matrix state per head: read, written, four products a token
                dv = m.get("vdim", m["dim"])
                nbytes += 2.0 * len(requests) * m["heads"] * m["dim"] * dv * 4
                flops += 8.0 * n * m["heads"] * m["dim"] * dv
    return {"bytes": nbytes + wanted * cfg.vocab_size * 4.0, "flops": flops}


def tolerance(case):
    # four times what the engine's logits are off the 64-bit ones (float32 2e-6, bfloat16 up to 5e-3 on these weights)
    return {"rel": 1e-5} if case["dtype"] == "float32" else {"rel": 0.02}


# --------------------------------------------------------------------------------------
# the same logits in 64 bits, as plain torch computes them
# --------------------------------------------------------------------------------------
def exact(case, seed):
    raw, _, _, source = _model(case)
    requests = [tokens for tokens, _ in _requests(case, seed)]
    device = torch.device("cuda:0")
    ids = torch.zeros((len(requests), max(len(t) for t in requests)), dtype=torch.long, device=device)
    for i, tokens in enumerate(requests):                   # shorter ones are padded behind their end
        ids[i, :len(tokens)] = torch.tensor(tokens, device=device)
    lens = [len(t) for t in requests]
    layers = case["model"].split("-")[0]
    with torch.no_grad():
        return _FORWARD[layers](raw, lambda name: source.read(name).double(), ids, lens, source)


def _rms(x, eps, weight=None):
    y = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps)
    return y if weight is None else y * weight


def _silu(x):
    return x * torch.sigmoid(x)


def _unit(x):
    return x * torch.rsqrt(x.pow(2).sum(-1, keepdim=True) + 1e-6)


def _last(x, lens):
    return torch.stack([x[i, n - 1] for i, n in enumerate(lens)])


def _rotate(x, dims, freqs, factor=1.0, neighbours=False):
    """x [B, n, heads, d] at positions 0..n-1."""
    angle = torch.arange(x.shape[1], device=x.device, dtype=torch.float64)[:, None] * freqs[None, :]
    c, s = (factor * angle.cos())[None, :, None, :], (factor * angle.sin())[None, :, None, :]
    a, b = (x[..., 0:dims:2], x[..., 1:dims:2]) if neighbours else (x[..., :dims // 2], x[..., dims // 2:dims])
    turned = (a * c - b * s, b * c + a * s)
    turned = torch.stack(turned, -1).flatten(-2) if neighbours else torch.cat(turned, -1)
    return torch.cat([turned, x[..., dims:]], -1)


def _frequencies(dims, base, device, scaling=None):
    i = torch.arange(dims // 2, dtype=torch.float64, device=device)
    f = base ** (-2.0 * i / dims)
    if not scaling:
        return f, 1.0
    turns = lambda t: dims * math.log(scaling["original"] / (2 * math.pi * t)) / (2 * math.log(base))
    lo, hi = max(math.floor(turns(scaling["fast"])), 0), min(math.ceil(turns(scaling["slow"])), dims - 1)
    r = ((i - lo) / max(hi - lo, 0.001)).clamp(0, 1)
    return f / scaling["factor"] * r + f * (1 - r), 0.1 * math.log(scaling["factor"]) + 1.0


def _attend(q, k, v, lens, weigh):
    """Causal attention of padded sequences, [B, n, heads, d]; ``weigh`` turns a head's scores [n, n] (minus infinity or
    zero weight left to it) into weights."""
    out = torch.zeros(q.shape[:3] + v.shape[3:], dtype=q.dtype, device=q.device)
    rep = q.shape[2] // k.shape[2]
    for b, n in enumerate(lens):
        hidden = torch.ones((n, n), dtype=torch.bool, device=q.device).triu(1)
        for h in range(q.shape[2]):
            p = weigh(q[b, :n, h] @ k[b, :n, h // rep].T.contiguous(), hidden, h)
            out[b, :n, h] = p @ v[b, :n, h // rep]
    return out


def _softmax(scale):
    return lambda s, hidden, h: torch.softmax((s * scale).masked_fill_(hidden, -math.inf), -1)


def _qwen3(raw, w, ids, lens, source):
    H, G, d, eps = raw["num_attention_heads"], raw["num_key_value_heads"], raw["head_dim"], raw["rms_norm_eps"]
    B, n = ids.shape
    embed = w("model.embed_tokens.weight")
    x = embed[ids]
    freqs, _ = _frequencies(d, raw["rope_theta"], ids.device)
    for i in range(raw["num_hidden_layers"]):
        p, a = f"model.layers.{i}.", f"model.layers.{i}.self_attn."
        h = _rms(x, eps, w(p + "input_layernorm.weight"))
        q = _rotate(_rms((h @ w(a + "q_proj.weight").T).view(B, n, H, d), eps, w(a + "q_norm.weight")), d, freqs)
        k = _rotate(_rms((h @ w(a + "k_proj.weight").T).view(B, n, G, d), eps, w(a + "k_norm.weight")), d, freqs)
        v = (h @ w(a + "v_proj.weight").T).view(B, n, G, d)
        x = x + _attend(q, k, v, lens, _softmax(d ** -0.5)).flatten(2) @ w(a + "o_proj.weight").T
        h = _rms(x, eps, w(p + "post_attention_layernorm.weight"))
        x = x + (_silu(h @ w(p + "mlp.gate_proj.weight").T) * (h @ w(p + "mlp.up_proj.weight").T)) @ w(p + "mlp.down_proj.weight").T
    head = embed if raw.get("tie_word_embeddings") else w("lm_head.weight")
    return _rms(_last(x, lens), eps, w("model.norm.weight")) @ head.T


def _pair(h, w, p):
    return (_silu(h @ w(p + "gate").T) * (h @ w(p + "up").T)) @ w(p + "down").T


def _bolapel(raw, w, ids, lens, source):
    eps, x = raw["norm"]["eps"], w("embed")[ids]
    B, n = ids.shape
    kept = {}
    for i, layer in enumerate(raw["layers"]):
        p, m, a = f"l{i}.", layer["mixer"], f"l{i}.mix."
        H, D = m["heads"], m["dim"]
        h = _rms(x, eps, w(p + "norm1"))
        before = torch.cat([torch.zeros_like(h[:, :1]), h[:, :-1]], 1)
        h = h + (before - h) * w(p + "shift")
        if layer["type"] == "attention":
            G, src = m["kv_heads"], m.get("kv_from", i)
            freqs, _ = _frequencies(m["rot"]["dims"], m["rot"]["base"], ids.device)
            if src == i:
                k = _rms((h @ w(a + "k").T).view(B, n, G, D), eps, w(a + "k.norm"))
                kept[i] = _rotate(k, m["rot"]["dims"], freqs), (h @ w(a + "v").T).view(B, n, G, -1)
            q = _rotate(_rms((h @ w(a + "q").T).view(B, n, H, D), eps, w(a + "q.norm")), m["rot"]["dims"], freqs)
            bias, chunk = w(a + "pb"), torch.arange(n, device=ids.device) // m["mask"]["size"]

            def weigh(s, hidden, head):
                other = chunk[:s.shape[0], None] != chunk[None, :s.shape[0]]
                return torch.sigmoid(s * m["scale"] + bias[head]).masked_fill_(hidden | other, 0.0)
            o = _attend(q, *kept[src], lens, weigh) * torch.sigmoid(h @ w(a + "g").T)[..., None]
            y = o.flatten(2) @ w(a + "o").T
        else:
            r, k, v = ((h @ w(a + c).T).view(B, n, H, D) for c in "rkv")
            decay = torch.exp(-math.exp(-0.5) * torch.sigmoid(torch.tanh(h @ w(a + "w1").T) @ w(a + "w2").T + w(a + "w0"))).view(B, n, H, D)
            u = _unit(k)
            au = torch.sigmoid(h @ w(a + "a").T + w(a + "a.b")).view(B, n, H, D) * u
            S = torch.zeros((B, H, D, D), dtype=x.dtype, device=x.device)
            o = torch.empty_like(r)
            for t in range(n):
                read = (u[:, t, :, :, None] * S).sum(2)
                S = decay[:, t, :, :, None] * S - au[:, t, :, :, None] * read[:, :, None] + k[:, t, :, :, None] * v[:, t, :, None]
                o[:, t] = (r[:, t, :, :, None] * S).sum(2)
            y = (_rms(o, eps).flatten(2) * w(a + "norm") * torch.sigmoid(h @ w(a + "g").T)) @ w(a + "o").T
        x = x + _rms(y, eps, w(p + "norm1b"))
        x = x + _rms(_pair(_rms(x, eps, w(p + "norm2")), w, p + "mlp."), eps, w(p + "norm2b"))
    cap = raw["logit_softcap"]
    return cap * torch.tanh(_rms(_last(x, lens), eps, w("final.norm")) @ w("head").T / cap)


def _convolved(x, taps):
    ext = torch.cat([torch.zeros_like(x[:, :taps.shape[1] - 1]), x], 1)
    return _silu(sum(ext[:, j:j + x.shape[1]] * taps[:, j] for j in range(taps.shape[1])))


def _delta_rule(q, k, v, decay, beta):
    """S <- decay S; S <- S + k (beta (v - S^T k))^T; o = S^T q; [B, n, H, ...], decay per head or per key channel."""
    S = torch.zeros(q.shape[0], q.shape[2], q.shape[3], v.shape[3], dtype=q.dtype, device=q.device)
    o = torch.empty_like(v)
    for t in range(q.shape[1]):
        S = decay[:, t, :, :, None] * S
        u = beta[:, t, :, None] * (v[:, t] - (k[:, t, :, :, None] * S).sum(2))
        S = S + k[:, t, :, :, None] * u[:, :, None]
        o[:, t] = (q[:, t, :, :, None] * S).sum(2)
    return o


def _latent(h, w, a, m, eps, lens, freqs, factor, neighbours):
    (B, n), H, D, R, Dr = h.shape[:2], m["heads"], m["dim"], m["kv_rank"], m["rot_dim"]
    q = (_rms(h @ w(a + "dq").T, eps, w(a + "dq.norm")) @ w(a + "uq").T).view(B, n, H, D + Dr)
    down = h @ w(a + "dkv").T
    c = _rms(down[..., :R], eps, w(a + "dkv.norm"))
    kr = _rotate(down[..., None, R:], Dr, freqs, factor, neighbours).expand(B, n, H, Dr)
    q = torch.cat([q[..., :D], _rotate(q[..., D:], Dr, freqs, factor, neighbours)], -1)
    k = torch.cat([(c @ w(a + "uk").T).view(B, n, H, D), kr], -1)
    return _attend(q, k, (c @ w(a + "uv").T).view(B, n, H, -1), lens, _softmax(m["scale"]))


def _experts(h, w, p, count, chosen, weights):
    """h [T, width]; chosen, weights [T, top]."""
    y = torch.zeros_like(h)
    for e in range(count):
        t, slot = (chosen == e).nonzero(as_tuple=True)
        if t.numel():
            y.index_add_(0, t, _pair(h[t], w, f"{p}e{e}.") * weights[t, slot][:, None])
    return y


def _dutilix(raw, w, ids, lens, source):
    eps, x = raw["norm"]["eps"], w("embed")[ids]
    B, n = ids.shape
    for i, layer in enumerate(raw["layers"]):
        p, m, a = f"l{i}.", layer["mixer"], f"l{i}.mix."
        H, D = m["heads"], m["dim"]
        h = _rms(x, eps, w(p + "norm1"))
        if layer["type"] == "latent_attention":
            freqs, factor = _frequencies(m["rot"]["dims"], m["rot"]["base"], ids.device)
            y = _latent(h, w, a, m, eps, lens, freqs, factor, False).flatten(2) * torch.sigmoid(h @ w(a + "g").T)
        elif layer["type"] == "delta":
            G = m["kv_heads"]
            q, k, v = (_convolved(h @ w(a + c).T, w(a + c + ".conv")) for c in "qkv")
            q, k = _unit(q.view(B, n, G, D)) * D ** -0.5, _unit(k.view(B, n, G, D))
            decay = torch.exp(-torch.exp(w(a + "A_log")) * torch.nn.functional.softplus(h @ w(a + "a").T + w(a + "dt_bias")))
            o = _delta_rule(q.repeat_interleave(H // G, 2), k.repeat_interleave(H // G, 2), v.view(B, n, H, -1), decay[..., None],
                            torch.sigmoid(h @ w(a + "b").T))
            y = (_rms(o, eps, w(a + "norm")) * _silu(h @ w(a + "g").T).view(o.shape)).flatten(2)
        else:
            cap = m["gate_cap"]
            q, k, v = ((h @ w(a + c).T).view(B, n, H, -1) for c in "qkv")
            li = cap * torch.tanh((h @ w(a + "i").T + w(a + "i.b")) / cap)
            lf = torch.nn.functional.logsigmoid(cap * torch.tanh((h @ w(a + "f").T + w(a + "f.b")) / cap))
            v1 = torch.cat([v, torch.ones_like(v[..., :1])], -1)
            S = torch.zeros(B, H, D, v1.shape[3], dtype=x.dtype, device=x.device)
            top, o = torch.zeros(B, H, dtype=x.dtype, device=x.device), torch.empty_like(v)
            for t in range(n):
                now = torch.maximum(lf[:, t] + top, li[:, t])
                S = torch.exp(lf[:, t] + top - now)[..., None, None] * S \
                    + (torch.exp(li[:, t] - now)[..., None] * k[:, t])[..., None] * v1[:, t, :, None]
                top = now
                y = (q[:, t, :, :, None] * D ** -0.5 * S).sum(2)
                o[:, t] = y[..., :-1] / (torch.maximum(y[..., -1:].abs(), torch.exp(-top)[..., None]) + 1e-6)
            y = _rms(o, eps).flatten(2) * w(a + "norm") * torch.sigmoid(h @ w(a + "g").T)
        x = x + y @ w(a + "o").T
        h, mlp = _rms(x, eps, w(p + "norm2")), layer["mlp"]
        if mlp["kind"] == "dense":
            x = x + _pair(h, w, p + "mlp.")
            continue
        r, flat = mlp["router"], h.flatten(0, 1)
        score = torch.softmax(flat @ w(p + "mlp.router").T, -1)
        choice = (score + w(p + "mlp.correction")).view(-1, r["groups"]["count"], r["experts"] // r["groups"]["count"])
        closed = torch.ones(choice.shape[:2], dtype=torch.bool, device=x.device)
        closed.scatter_(1, choice.amax(-1).topk(r["groups"]["keep"], -1).indices, False)
        chosen = choice.masked_fill(closed[..., None], -math.inf).flatten(1).topk(r["top"], -1).indices
        weights = score.gather(1, chosen)
        x = x + _experts(flat, w, p + "mlp.", r["experts"], chosen, weights / (weights.sum(-1, keepdim=True) + 1e-20)).view(x.shape)
    return _rms(_last(x, lens), eps, w("final.norm")) @ w("head").T * raw["logit_scale"]


def _sorulix(raw, w, ids, lens, source):
    eps, embed = raw["norm"]["eps"], w("embed")
    x = embed[ids]
    B, n = ids.shape
    at = torch.arange(n, device=ids.device, dtype=torch.float64)
    for i, layer in enumerate(raw["layers"]):
        p, m, a = f"l{i}.", layer["mixer"], f"l{i}.mix."
        h = _rms(x, eps, 1 + w(p + "norm1"))
        if layer["type"] == "parallel":
            m, r, a, b = layer["mixer"]["left"], layer["mixer"]["right"], a + "left.", a + "right."
            H, G, D = m["heads"], m["kv_heads"], m["dim"]
            temp = 1 + m["q_temp"]["coef"] * torch.log((at + 1).div(m["q_temp"]["every"], rounding_mode="floor") + 1)
            q = (_rms(h @ w(a + "q").T, eps, w(a + "q.norm")) * temp[None, :, None]).view(B, n, H, D)
            k = _rms(h @ w(a + "k").T, eps, w(a + "k.norm")).view(B, n, G, D)
            cap = m["softcap"]

            def weigh(s, hidden, head):
                t = at[:s.shape[0]]
                s = cap * torch.tanh(s * m["scale"] / cap) - 2.0 ** (-8.0 * (head + 1) / H) * (t[:, None] - t[None, :])
                s = s.masked_fill(hidden, -math.inf)
                top = s.amax(-1, keepdim=True).clamp(min=0)
                e = torch.exp(s - top)
                return e / (torch.exp(-top) + e.sum(-1, keepdim=True))
            left = _attend(q, k, (h @ w(a + "v").T).view(B, n, G, -1), lens, weigh).flatten(2) @ w(a + "o").T
            q, k, v = (_silu(h @ w(b + c).T).view(B, n, r["heads"], -1) for c in "qkv")
            decay = torch.tensor(r["decay"], dtype=torch.float64, device=x.device)[None, :, None, None]
            S = torch.zeros(B, r["heads"], r["dim"], r["vdim"], dtype=x.dtype, device=x.device)
            o = torch.empty_like(v)
            for t in range(n):
                S = decay * S + k[:, t, :, :, None] * v[:, t, :, None]
                o[:, t] = (q[:, t, :, :, None] * S).sum(2)
            right = (_rms(o.flatten(2), eps, w(b + "norm")) * torch.sigmoid(h @ w(b + "g").T)) @ w(b + "o").T
            x = x + 0.5 * (_rms(left, eps, w(a + "out")) + _rms(right, eps, w(b + "out")))
        else:
            H, G, D = m["heads"], m["kv_heads"], m["dim"]
            q, k, v = (_convolved(h @ w(a + c).T, w(a + c + ".conv")) for c in "qkv")
            z = (h @ w(a + "a1").T @ w(a + "a2").T + w(a + "dt_bias")).view(B, n, H, D)
            decay = torch.exp(-torch.exp(w(a + "A_log"))[:, None] * torch.nn.functional.softplus(z))
            q, k = _unit(q.view(B, n, G, D)) * D ** -0.5, _unit(k.view(B, n, G, D))
            o = _delta_rule(q.repeat_interleave(H // G, 2), k.repeat_interleave(H // G, 2), v.view(B, n, H, -1), decay,
                            torch.sigmoid(h @ w(a + "b").T))
            gate = torch.sigmoid(h @ w(a + "g1").T @ w(a + "g2").T).view(o.shape)
            x = x + (_rms(o, eps, w(a + "norm")) * gate).flatten(2) @ w(a + "o").T
        h, f, limit = _rms(x, eps, 1 + w(p + "norm2")), p + "mlp.", layer["mlp"]["limit"]
        g = (h @ w(f + "gate").T + w(f + "gate.b")).clamp(max=limit)
        u = (h @ w(f + "up").T + w(f + "up.b")).clamp(-limit, limit)
        x = x + (g * torch.sigmoid(1.702 * g) * (u + 1)) @ w(f + "down").T + w(f + "down.b")
    return _rms(_last(x, lens), eps, 1 + w("final.norm")) @ embed.T


def _furanex(raw, w, ids, lens, source):
    eps, embed = raw["norm"]["eps"], w("embed")
    xs = (embed[ids] * raw["embedding"]["scale"])[None].repeat(raw["streams"], 1, 1, 1)
    B, n = ids.shape
    first = None
    for i, layer in enumerate(raw["layers"]):
        p, m, a = f"l{i}.", layer["mixer"], f"l{i}.mix."
        H, D = m["heads"], m["dim"]
        for part in (1, 2):
            h = _rms(torch.einsum("s,sbnw->bnw", w(f"{p}hc{part}.in"), xs), eps, w(f"{p}norm{part}"))
            if part == 2:
                flat, top = h.flatten(0, 1), layer["mlp"]["router"]["top"]
                chosen = source.read(p + "mlp.table")[ids.flatten()].long()
                y = _experts(flat, w, p + "mlp.", layer["mlp"]["router"]["experts"], chosen, torch.full(chosen.shape, 1.0 / top, dtype=xs.dtype, device=xs.device))
                y = (y + _pair(flat, w, p + "mlp.shared.")).view(h.shape)
            elif layer["type"] == "latent_attention":
                freqs, factor = _frequencies(m["rot_dim"], m["rot"]["base"], ids.device, m["rot"]["scaling"])
                o = _latent(h, w, a, m, eps, lens, freqs, factor, True) * torch.sigmoid(h @ w(a + "g").T)[..., None]
                y = o.flatten(2) @ w(a + "o").T
            else:
                G = m["kv_heads"]
                freqs, factor = _frequencies(m["rot"]["dims"], m["rot"]["base"], ids.device, m["rot"]["scaling"])
                q = _rms(_rotate((h @ w(a + "q").T).view(B, n, H, D), m["rot"]["dims"], freqs, factor), eps)
                k = _rms(_rotate((h @ w(a + "k").T).view(B, n, G, D), m["rot"]["dims"], freqs, factor), eps)
                v = (h @ w(a + "v").T).view(B, n, G, -1)
                if first is None:
                    first = v
                else:
                    share = w(a + "vmix")
                    v = (1 - share) * v + share * first
                y = _attend(q, k, v, lens, _softmax(m["scale"])).flatten(2) @ w(a + "o").T
            xs = torch.einsum("st,sbnw->tbnw", w(f"{p}hc{part}.mix"), xs) + w(f"{p}hc{part}.out")[:, None, None, None] * y[None]
    return _rms(_last(xs.sum(0), lens), eps, w("final.norm")) @ embed.T


_FORWARD = {"qwen3": _qwen3, "bolapel": _bolapel, "dutilix": _dutilix, "sorulix": _sorulix, "furanex": _furanex}
