"""What this framework is measured on: one step of a served model, through the model API that the engine drives.

A case is a decode step (one new token for each of `rows` sequences, replayed from a HIP graph as the engine
replays it) or a prefill step (`rows` prompts packed into one eager forward, some behind a cached prefix).  The
models are the decoders of the game (`qwen*`, `mistral*`: paged K/V, bf16 or fp8 weights) and three of the
fp32-stream families, which between them hold differential, windowed and latent attention, gated delta rule,
selective state space and retention, table-routed experts, and dense feed-forwards of both forms.  Depth is cut
(`layers`) where a full model adds nothing but preparation: every layer of a model has the same shapes.

The outputs are a step's logits, the paged K/V caches of the decoders and the state tables of the recurrent
families.  `exact` computes a step in float64 from the model's equations, without the package.
"""

import dataclasses
import functools
import math
import zlib

import numpy as np
import torch

from byzantine_consensus_llm_agents_amd.models import build_model
from byzantine_consensus_llm_agents_amd.models.config import MabivikConfig, MofidraConfig, VagozenConfig, get_model_config
from byzantine_consensus_llm_agents_amd.models.transformer import AttnMeta
from byzantine_consensus_llm_agents_amd.ops import get_ops

BLOCK = 16             # tokens of a KV page (the engine's default)
CHUNK = 16384          # tokens of one prefill step (the engine's default)
FP8_MAX = 448.0
FAMILIES = {"mofidra": MofidraConfig, "mabivik": MabivikConfig, "vagozen": VagozenConfig}


def _case(name, model, mode, rows, length, layers=4, width=0, cached=0, quant=""):
    """rows: sequences; length: mean context (decode) or mean new prompt tokens (prefill); cached: prefix tokens
    already in the cache, per prompt."""
    c = {"model": model, "mode": mode, "rows": rows, "length": length, "layers": layers, "width": width,
         "cached": cached, "quant": quant}
    return {"name": name, **c} if name else c


def listed():
    return [
        # one game of four agents on the small model: the smallest step there is, all launches and latency
        _case("qwen2.5-0.5b decode 4", "qwen2.5-0.5b", "decode", 4, 500, layers=24),
        # one game of 8 honest + 2 Byzantine agents on the default model: weights are streamed for ten rows
        _case("qwen3-14b decode 10", "qwen3-14b", "decode", 10, 1100, layers=16),
        # a 16 + 4 game on the fp8 model
        _case("mistral-22b fp8 decode 20", "mistral-22b", "decode", 20, 1500, layers=12, quant="fp8"),
        # a dozen games decoding together, and the large pool of a serving process (odd row counts: rows finish
        # one by one)
        _case("qwen3-8b decode 101", "qwen3-8b", "decode", 101, 1000, layers=12),
        _case("qwen3-14b decode 448", "qwen3-14b", "decode", 448, 1050, layers=8),
        # the prompts of one game's round: a shared system prompt is cached, the history is new
        _case("qwen3-8b prefill 10x450", "qwen3-8b", "prefill", 10, 450, layers=12, cached=380),
        # a full prefill chunk of the default model
        _case("qwen3-14b prefill 16x1000", "qwen3-14b", "prefill", 16, 1000, layers=8),
        # the fp32-stream families at the two layer sizes of the family benchmark: a batch of prompts, a decode batch
        _case("mofidra prefill 8x1000", "mofidra", "prefill", 8, 1000, width=2048),
        _case("mofidra decode 64", "mofidra", "decode", 64, 1000, width=4096),
        _case("mabivik prefill 8x1000", "mabivik", "prefill", 8, 1000, width=4096),
        _case("mabivik decode 64", "mabivik", "decode", 64, 1000, width=2048),
        _case("vagozen prefill 3x700", "vagozen", "prefill", 3, 700, width=2048),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A decode step of 1 to 512 rows or a prefill step of 40 to 12000 tokens, of any of the models."""
    decoders = [("qwen2.5-0.5b", 24, ""), ("qwen3-8b", 12, ""), ("qwen3-14b", 8, ""), ("mistral-22b", 8, "fp8")]
    mode = rng.choice(["decode", "prefill"])
    family = rng.random() < 0.45
    if mode == "decode":
        rows = _log_int(rng, 1, 200 if family else 512)
        length = _log_int(rng, 40, min(2500, (100000 if family else 450000) // rows))
        cached = 0
    else:
        tokens = _log_int(rng, 40, 12000)
        rows = _log_int(rng, 1, min(24, tokens // 20))
        length = min(tokens // rows, 3000)
        cached = 0 if family or rng.random() < 0.5 else 16 * rng.randint(1, 60)
    if family:
        return _case("", rng.choice(sorted(FAMILIES)), mode, rows, length, width=rng.choice([2048, 4096]))
    model, layers, quant = rng.choice(decoders)
    return _case("", model, mode, rows, length, layers=layers, cached=cached, quant=quant)


def tolerance(case):
    # measured against float64 (2-norm of the error over an output): bf16 decoders and families 0.5 to 1.1 %, the
    # fp8 decoder 1.8 % (a rounding that falls the other way in e4m3 is 6 % of one value)
    return {"rel": 0.03, "max": 0.4} if case["quant"] else {"rel": 0.025, "max": 0.3}


# ---------------------------------------------------------------------------------------------- sizes
def _lengths(case):
    """[(tokens resident before the step, new tokens)] per sequence: lengths are spread around their mean."""
    out = []
    for i in range(case["rows"]):
        n = max(2, int(round(case["length"] * (0.7 + 0.6 * ((0.5 + 0.61803 * i) % 1.0)))))
        out.append((n - 1, 1) if case["mode"] == "decode" else (case["cached"], n))
    return out


def _family_dict(case):
    """config.json of a family model: the layer sizes of the family benchmark."""
    W = case["width"]
    H, G, ff, vocab = (16, 4, 8192, 32768) if W == 2048 else (32, 8, 12288, 32768)
    base = {"width": W, "vocab": vocab, "norm": {"eps": 1e-5}}
    if case["model"] == "mofidra":
        mixer = {"heads": H, "kv_heads": G, "dim": 64, "vdim": 128, "scale": 0.125, "diff": 0.5, "rot": {"dims": 64, "base": 1e6}}
        return {**base, "architecture": "Mofidra", "embedding": {"scale": 1.0},
                "layers": [{"type": "attention", "mixer": mixer, "mlp": {"kind": "dense", "ff": ff}}] * case["layers"]}
    latent = {"heads": H, "dim": 128, "rot_dim": 64, "vdim": 128, "q_rank": 768, "kv_rank": 128, "scale": 0.072}
    if case["model"] == "mabivik":
        latent.update(mask={"size": 512}, rot={"dims": 64, "base": 1e6, "scaling": {"factor": 8.0, "original": 8192,
                                                                                    "fast": 32.0, "slow": 1.0}})
        ssm = {"heads": 2 * W // 128, "vdim": 128, "state": 128, "groups": 2, "norm_groups": 2, "conv": 4}
        delta = {"heads": H, "kv_heads": H // 2, "dim": 128, "vdim": 128, "conv": 4}
        mlp = {"kind": "moe", "expert": {"ff": ff // 4}, "router": {"experts": 8, "top": 2}}
        kinds = [("latent_attention", latent), ("mamba2", ssm), ("delta", delta), ("latent_attention", dict(latent, kv_from=0))]
        return {**base, "architecture": "Mabivik", "embedding": {"scale": 1.0}, "logit_scale": 1.0, "token_side": {"dim": 256},
                "layers": [{"type": k, "mixer": m, "mlp": mlp} for k, m in kinds]}
    att = {"heads": H, "kv_heads": G, "dim": 128, "vdim": 128, "scale": 0.088, "mask": {"size": 512, "keep_first": 16},
           "rot": {"dims": 128, "base": 1e6, "scaling": {"factor": 4.0, "original": 8192, "fast": 32.0, "slow": 1.0}}}
    ret = {"heads": H // 2, "dim": 128, "vdim": 256, "decay": [1.0 - 2.0 ** (-5 - i % 8) for i in range(H // 2)],
           "rot": {"dims": 128, "base": 1e6}}
    latent["rot"] = {"dims": 64, "base": 1e6}
    kinds = [("attention", att), ("retention", ret), ("latent_attention", latent), ("retention", ret)]
    return {**base, "architecture": "Vagozen", "logit_scale": 0.5, "loop": {"start": 2, "stop": 4, "times": 2},
            "layers": [{"type": k, "mixer": m, "mlp": {"kind": "dense", "ff": ff, "limit": 7.0}} for k, m in kinds]}


def _layer_order(cfg):
    """Layer of every layer run."""
    n, loop = len(cfg["layers"]), cfg.get("loop")
    if not loop:
        return list(range(n))
    return list(range(loop["start"])) + list(range(loop["start"], loop["stop"])) * loop["times"] + list(range(loop["stop"], n))


def _config(case):
    if case["model"] in FAMILIES:
        return FAMILIES[case["model"]].from_dict(_family_dict(case), case["model"])
    return dataclasses.replace(get_model_config(case["model"]), num_layers=case["layers"])


def work(case):
    """Weights read once, the cache and state a step needs read once, what it adds and the logits written once."""
    seqs = _lengths(case)
    T, n = sum(q for _, q in seqs), len(seqs)

    def pairs(window=0, keep=0):  # (query, key) pairs and keys read
        p = k = 0
        for a, q in seqs:
            k += a + q if not window else min(a + q, q + window - 1 + keep)
            first = np.arange(a, a + q) + 1
            p += int((np.minimum(first, window + keep) if window else first).sum())
        return p, k

    if case["model"] not in FAMILIES:
        c, L = _config(case), case["layers"]
        h, qs, kv, inter = c.hidden_size, c.q_size, c.kv_size, c.intermediate_size
        w_qkv, w_rest = h * (qs + 2 * kv), qs * h + 3 * h * inter
        p, k = pairs()
        wb = 1 if case["quant"] else 2
        head = c.vocab_size * h
        flops = 2 * L * T * w_qkv + 2 * ((L - 1) * T + n) * w_rest + 2 * n * head + 4 * L * qs * p
        return {"bytes": L * (w_qkv + w_rest) * wb + 2 * head + 2 * T * h + L * 4 * kv * (k + T) + 2 * n * c.vocab_size, "flops": flops}
    cfg = _family_dict(case)
    W, V = cfg["width"], cfg["vocab"]
    order = _layer_order(cfg)
    bytes_, flops = 2 * V * W + 2 * T * W + 4 * n * V, 2 * n * V * W
    seen = set()
    for r, li in enumerate(order):
        m, f, kind = cfg["layers"][li]["mixer"], cfg["layers"][li]["mlp"], cfg["layers"][li]["type"]
        mask = m.get("mask") or {}
        p, k = pairs(mask.get("size", 0), mask.get("keep_first", 0))
        after = n if r == len(order) - 1 else T    # past the last mixer only the rows with logits matter
        H = m["heads"]
        if kind == "attention":
            qd = m["dim"] * (2 if case["model"] == "mofidra" else 1)
            w_in, w_out, cache = W * (H * qd + m["kv_heads"] * (qd + m["vdim"])), W * H * m["vdim"], m["kv_heads"] * (qd + m["vdim"])
            flops += 2 * H * p * (qd + m["vdim"] * (2 if case["model"] == "mofidra" else 1))
        elif kind == "latent_attention":
            d, rd, vd, rank = m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
            own = "kv_from" not in m
            w_in = W * (m["q_rank"] + (rank + rd if own else 0)) + m["q_rank"] * H * (d + rd) + H * d * rank
            w_out = H * vd * (rank + W) + (W * H * vd if case["model"] == "mabivik" else 0)
            cache = rank + rd
            flops += 2 * H * p * (2 * rank + rd)
        else:
            d, vd = m.get("state", m.get("dim")), m["vdim"]
            if kind == "mamba2":
                w_in = W * (2 * H * vd + 2 * m["groups"] * d + H)
            elif kind == "delta":
                w_in = W * (2 * m["kv_heads"] * d + 2 * H * vd + 2 * H)
            else:
                w_in = W * (2 * H * d + 2 * H * vd)
            w_out, cache = W * H * vd, 0
            flops += T * H * d * vd * (7 if kind == "delta" else 5)
            bytes_ += 4 * n * H * d * vd * (2 if case["mode"] == "decode" else 1)
        bytes_ += 2 * cache * (k + T)
        flops += 2 * T * w_in + 2 * after * w_out
        w = w_in + w_out
        if f["kind"] == "moe":
            ff = f["expert"]["ff"]
            w += 3 * W * ff * min(f["router"]["experts"], f["router"]["top"] * after)
            flops += 6 * after * W * ff * f["router"]["top"]
        else:
            n_mat = 2 if case["model"] == "mofidra" else 3
            w += n_mat * W * f["ff"]
            flops += 2 * n_mat * after * W * f["ff"]
        if cfg.get("token_side"):
            w += 2 * W * cfg["token_side"]["dim"]
            flops += 4 * after * W * cfg["token_side"]["dim"]
        if li not in seen:     # a looped layer's weights have to be read once
            bytes_ += 2 * w
            seen.add(li)
    return {"bytes": bytes_, "flops": flops}


# ---------------------------------------------------------------------------------------------- inputs
class _Weights:
    """Checkpoint tensors by name, each drawn from its own generator when it is asked for."""

    def __init__(self, shapes, scale, seed, device):
        self.shapes, self.scale, self.seed, self.device = shapes, scale, seed, device

    def __contains__(self, name):
        return name in self.shapes

    def __getitem__(self, name):
        g = torch.Generator(device=self.device).manual_seed((zlib.crc32(name.encode()) << 20) + self.seed % (1 << 20))
        shape, (mean, std) = self.shapes[name], self.scale(name, self.shapes[name])
        if name.endswith("mlp.table"):     # experts of a token: distinct entries
            return torch.rand(shape[0], 8, generator=g, device=self.device).argsort(-1)[:, :shape[1]].to(torch.int32)
        t = torch.empty(shape, dtype=torch.bfloat16, device=self.device)
        return t.normal_(mean, std, generator=g)


def _decoder_weights(case, seed, device):
    c = _config(case)
    h, hd = c.hidden_size, c.head_dim
    shapes = {"model.embed_tokens.weight": (c.vocab_size, h), "model.norm.weight": (h,)}
    if not c.tie_embeddings:
        shapes["lm_head.weight"] = (c.vocab_size, h)
    for i in range(c.num_layers):
        p = f"model.layers.{i}."
        shapes.update({p + "self_attn.q_proj.weight": (c.q_size, h), p + "self_attn.k_proj.weight": (c.kv_size, h),
                       p + "self_attn.v_proj.weight": (c.kv_size, h), p + "self_attn.o_proj.weight": (h, c.q_size),
                       p + "mlp.gate_proj.weight": (c.intermediate_size, h), p + "mlp.up_proj.weight": (c.intermediate_size, h),
                       p + "mlp.down_proj.weight": (h, c.intermediate_size), p + "input_layernorm.weight": (h,),
                       p + "post_attention_layernorm.weight": (h,)})
        if c.qkv_bias:
            shapes.update({p + "self_attn.q_proj.bias": (c.q_size,), p + "self_attn.k_proj.bias": (c.kv_size,),
                           p + "self_attn.v_proj.bias": (c.kv_size,)})
        if c.qk_norm:
            shapes.update({p + "self_attn.q_norm.weight": (hd,), p + "self_attn.k_norm.weight": (hd,)})

    # a layer adds a fraction of the stream, as a trained one does; a smaller one under fp8, where two correct
    # implementations round single activations apart by 6 % (the tolerance has to tell a mistake from that)
    down, out = (0.0025 / c.num_layers, 0.01) if case["quant"] else (0.01 / c.num_layers, 0.02)

    def scale(name, shape):
        if "norm" in name:
            return 1.0, 0.1
        if name == "model.embed_tokens.weight":
            return 0.0, 0.02 if c.tie_embeddings else 1.0
        return 0.0, down if name.endswith("down_proj.weight") else out if name.endswith("o_proj.weight") else 0.02
    return _Weights(shapes, scale, seed, device)


def _family_weights(case, model, seed, device):
    def scale(name, shape):
        last = name.split(".")[-1]
        if case["model"] == "mofidra" and "norm" in name:
            return 0.0, 0.1                                # stored as an offset from one
        if last == "alpha":
            return 0.7, 0.05
        if last in ("lq1", "lk1", "lq2", "lk2"):
            return 0.0, 0.1
        if last in ("b", "step") and len(shape) == 1 or name == "loop.step":
            return 0.0, 0.1
        if last == "norm" or last.startswith("norm"):
            return 1.0, 0.2
        if last.startswith("ls"):
            return 0.6, 0.15
        if last == "A_log":
            return -1.0, 0.5
        if last in ("dt_bias", "D"):
            return 0.0, 0.5
        if last == "conv":
            return 0.0, 0.4
        if name in ("embed", "side.embed"):
            return 0.0, 0.7
        return 0.0, shape[-1] ** -0.5
    return _Weights(model.tensor_shapes(), scale, seed, device)


def _tokens(case, seed, vocab):
    """Token ids of every sequence, the resident ones too (a decoder's cache is drawn instead of computed)."""
    r = np.random.RandomState(seed % (1 << 31))
    return [r.randint(0, vocab, a + q).astype(np.int32) for a, q in _lengths(case)]


def _pages(case, seed):
    """[sequence, page] -> physical block, in no order; block 0 stays free."""
    blocks = [-(-(a + q) // BLOCK) for a, q in _lengths(case)]
    order = np.random.RandomState(seed % (1 << 31) + 1).permutation(sum(blocks)) + 1
    table, at = np.zeros((len(blocks), max(blocks)), dtype=np.int32), 0
    for i, b in enumerate(blocks):
        table[i, :b] = order[at:at + b]
        at += b
    return table, sum(blocks) + 1


def _resident(case, seed, layer, c, blocks, device):
    """The K and V pages [blocks, heads, BLOCK, dim] that a decoder's cache holds before the step."""
    g = torch.Generator(device=device).manual_seed(seed * 1009 + layer)
    shape = (blocks, c.num_kv_heads, BLOCK, c.head_dim)
    return tuple(torch.empty(shape, dtype=torch.bfloat16, device=device).normal_(generator=g) for _ in range(2))


def _meta(seqs, table, model, device, state=None, rows=None):
    """The device tables of one packed step over `seqs` = [(resident tokens, new tokens)]."""
    i32 = torch.int32
    decode = all(q == 1 for _, q in seqs)
    starts = np.concatenate([[0], np.cumsum([q for _, q in seqs])])
    owner = np.repeat(np.arange(len(seqs)), [q for _, q in seqs])
    pos = np.concatenate([np.arange(a, a + q) for a, q in seqs])
    tile_rows = getattr(model, "prefill_tile_rows", None) or model.ops.prefill_tile_rows(model.hd, False, table.shape[1])
    tiles = [] if decode else [(a + q - (starts[i + 1] - t), i, t, min(t + tile_rows, starts[i + 1]))
                               for i, (a, q) in enumerate(seqs) for t in range(starts[i], starts[i + 1], tile_rows)]
    tiles.sort(key=lambda t: -t[0])   # the deepest tiles first

    def dev(x, dtype=i32):
        return torch.as_tensor(np.ascontiguousarray(x)).to(device=device, dtype=dtype)
    return AttnMeta(
        positions=dev(pos), slots=dev(table[owner, pos // BLOCK].astype(np.int64) * BLOCK + pos % BLOCK), block_tables=dev(table),
        seq_lens=dev([a + q for a, q in seqs]), q_start=dev(starts), max_q_len=max(q for _, q in seqs), decode=decode,
        logits_idx=None if decode else dev(starts[1:] - 1, torch.int64),
        tiles=dev(np.array([t[1:] for t in tiles]).reshape(-1, 3)), tile_rows=tile_rows,
        single=torch.zeros(0, 2, dtype=i32, device=device) if getattr(model, "split_single_rows", False) else None,
        state=state, state_rows=dev(np.arange(len(seqs)) if rows is None else rows), token_seq=dev(owner))


@functools.lru_cache(maxsize=None)
def _ops():
    return get_ops("hip")


def prepare(case, seed):
    device = torch.device("cuda", torch.cuda.current_device())
    ops, c = _ops(), _config(case)
    model = build_model(c, ops, device, torch.bfloat16, quant=case["quant"] or None)
    family = case["model"] in FAMILIES
    model.load_hf_state_dict(_family_weights(case, model, seed, device) if family else _decoder_weights(case, seed, device))
    seqs, (table, blocks) = _lengths(case), _pages(case, seed)
    ids = _tokens(case, seed, c.vocab_size)
    k, v = model.alloc_kv(blocks, BLOCK, torch.bfloat16)
    state = model.alloc_state(len(seqs)) if getattr(model, "has_seq_state", False) else None
    if not family:
        for layer in range(c.num_layers):
            kp, vp = _resident(case, seed, layer, c, blocks, device)
            k[layer].copy_(kp)
            v[layer].copy_(vp.transpose(2, 3))
    elif case["mode"] == "decode":     # the contexts of the rows come through the model, a chunk of sequences at a time
        for part in _groups([(0, a) for a, _ in seqs], CHUNK):
            m = _meta([(0, seqs[i][0]) for i in part], table[part], model, device, state, rows=part)
            model.forward(torch.as_tensor(np.concatenate([ids[i][:-1] for i in part])).to(device), m, k, v)
    tokens = torch.as_tensor(np.concatenate([t[a:] for t, (a, _) in zip(ids, seqs)])).to(device)
    s = {"model": model, "tokens": tokens, "meta": _meta(seqs, table, model, device, state), "k": k, "v": v,
         "state": model.state_tensors(state) if state is not None else [], "graph": None, "caches": not family}
    if case["mode"] == "decode":       # captured once, as the engine captures a decode bucket
        ops.prepare_device(device)
        saved = [t.clone() for t in s["state"]]
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            model.forward(tokens, s["meta"], k, v)
        torch.cuda.current_stream().wait_stream(side)
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            s["logits"] = model.forward(tokens, s["meta"], k, v)
        for t, old in zip(s["state"], saved):
            t.copy_(old)
    return s


def run(s):
    if s["graph"] is not None:
        s["graph"].replay()
        logits = s["logits"]
    else:
        logits = s["model"].forward(s["tokens"], s["meta"], s["k"], s["v"])
    out = {"logits": logits, "state": s["state"]}
    if s["caches"]:
        out["k"], out["v"] = s["k"], s["v"]
    return out


def _groups(seqs, most):
    """Indices of consecutive sequences, at most `most` tokens (or one sequence) together."""
    out, used = [], 0
    for i, (a, q) in enumerate(seqs):
        if not out or used + a + q > most:
            out.append([])
            used = 0
        out[-1].append(i)
        used += a + q
    return out


# ---------------------------------------------------------------------------------------------- float64
F64 = torch.float64


def exact(case, seed):
    if not torch.cuda.is_available():
        return None
    with torch.no_grad():
        if case["model"] not in FAMILIES:
            return {"logits": _decoder_exact(case, seed), "state": [], "k": None, "v": None}
        logits, state = _family_exact(case, seed)
        return {"logits": logits, "state": state}


def _unit_rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _turn(x, pos, freqs, amp=1.0, pairs=False):
    """x [T, heads, d], the first 2 * len(freqs) features turned by pos * freqs: in halves, or in neighbouring pairs."""
    n = freqs.numel()
    ang = pos.to(F64)[:, None, None] * freqs
    c, s = torch.cos(ang) * amp, torch.sin(ang) * amp
    y = x.clone()
    if pairs:
        a, b = x[..., 0:2 * n:2], x[..., 1:2 * n:2]
        y[..., 0:2 * n:2], y[..., 1:2 * n:2] = a * c - b * s, b * c + a * s
    else:
        a, b = x[..., :n], x[..., n:2 * n]
        y[..., :n], y[..., n:2 * n] = a * c - b * s, b * c + a * s
    return y


def _fp8(x):
    """Row-wise e4m3 values, as float64."""
    xf = x.float()
    scale = xf.abs().amax(-1, keepdim=True).clamp(min=1e-12) / FP8_MAX
    return (xf / scale).clamp(-FP8_MAX, FP8_MAX).to(torch.float8_e4m3fn).to(F64) * scale.to(F64)


def _decoder_exact(case, seed):
    device = torch.device("cuda", torch.cuda.current_device())
    c, w = _config(case), _decoder_weights(case, seed, device)
    seqs, (table, blocks) = _lengths(case), _pages(case, seed)
    table = torch.as_tensor(table).to(device).long()
    ids = _tokens(case, seed, c.vocab_size)
    tokens = torch.as_tensor(np.concatenate([t[a:] for t, (a, _) in zip(ids, seqs)])).to(device).long()
    pos = torch.as_tensor(np.concatenate([np.arange(a, a + q) for a, q in seqs])).to(device)
    starts = np.concatenate([[0], np.cumsum([q for _, q in seqs])])
    H, G, hd, eps = c.num_heads, c.num_kv_heads, c.head_dim, c.rms_eps
    freqs = c.rope_theta ** (-torch.arange(0, hd, 2, dtype=F64, device=device) / hd)

    def linear(x, name):
        m = w[name]
        y = _fp8(x) @ _fp8(m).T if case["quant"] else x @ m.to(F64).T
        bias = name.replace(".weight", ".bias")
        return y + w[bias].to(F64) if bias in w else y

    def norm(x, name):
        return _unit_rms(x, eps) * w[name].to(F64)

    x = w["model.embed_tokens.weight"][tokens].to(F64)
    for i in range(c.num_layers):
        p = f"model.layers.{i}."
        h = norm(x, p + "input_layernorm.weight")
        q, k, v = (linear(h, p + f"self_attn.{n}_proj.weight").view(-1, heads, hd) for n, heads in (("q", H), ("k", G), ("v", G)))
        if c.qk_norm:
            q, k = norm(q, p + "self_attn.q_norm.weight"), norm(k, p + "self_attn.k_norm.weight")
        q, k = _turn(q, pos, freqs), _turn(k, pos, freqs)
        kp, vp = _resident(case, seed, i, c, blocks, device)
        att = torch.empty_like(q)
        for b, (a, n) in enumerate(seqs):
            lo, hi = int(starts[b]), int(starts[b + 1])
            pages = table[b, :-(-a // BLOCK)] if a else table[b, :0]
            kk, vv = (torch.cat([t[pages].transpose(1, 2).reshape(-1, G, hd)[:a].to(F64), new[lo:hi]])
                      for t, new in ((kp, k), (vp, v)))
            att[lo:hi] = _attend(q[lo:hi], kk, vv, hd ** -0.5, _causal(a, n, device))
        x = x + linear(att.reshape(-1, H * hd), p + "self_attn.o_proj.weight")
        h = norm(x, p + "post_attention_layernorm.weight")
        g, u = linear(h, p + "mlp.gate_proj.weight"), linear(h, p + "mlp.up_proj.weight")
        x = x + linear(torch.nn.functional.silu(g) * u, p + "mlp.down_proj.weight")
    x = norm(x[torch.as_tensor(starts[1:] - 1).to(device)], "model.norm.weight")
    head = "model.embed_tokens.weight" if c.tie_embeddings else "lm_head.weight"
    return x @ w[head].to(F64).T


def _causal(a, n, device, window=0, keep=0):
    """[n, a + n]: the keys that the queries at positions a .. a + n - 1 see."""
    i, j = torch.arange(a, a + n, device=device)[:, None], torch.arange(a + n, device=device)[None]
    see = j <= i
    return see & ((i - j < window) | (j < keep)) if window else see


def _attend(q, k, v, scale, see):
    """q [n, H, d], k [m, G, d], v [m, G, e] -> [n, H, e]; head h reads key head h // (H / G)."""
    n, H, d = q.shape
    G = k.shape[1]
    qg = q.view(n, G, H // G, d).permute(1, 2, 0, 3).reshape(G, H // G * n, d).contiguous()
    s = torch.matmul(qg, k.permute(1, 2, 0).contiguous()).view(G, H // G, n, -1) * scale
    s = torch.softmax(s.masked_fill_(~see, -math.inf), -1).view(G, H // G * n, -1)
    o = torch.matmul(s, v.permute(1, 0, 2).contiguous())
    return o.view(G, H // G, n, -1).permute(2, 0, 1, 3).reshape(n, H, -1)


def _ramp(rot, device):
    """(frequencies, factor of cos and sin) of a rotary embedding whose low frequencies may be scaled down."""
    dims, base = rot["dims"], float(rot["base"])
    f = base ** (-2.0 * torch.arange(dims // 2, dtype=F64, device=device) / dims)
    s = rot.get("scaling")
    if not s:
        return f, 1.0

    def turns(t):
        return dims * math.log(s["original"] / (2.0 * math.pi * t)) / (2.0 * math.log(base))
    lo, hi = max(math.floor(turns(s["fast"])), 0), min(math.ceil(turns(s["slow"])), dims - 1)
    r = ((torch.arange(dims // 2, dtype=F64, device=device) - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
    return f / s["factor"] * r + f * (1.0 - r), 0.1 * math.log(s["factor"]) + 1.0


class _Packed:
    """The sequences of one group, one after the other."""

    def __init__(self, ids, device):
        self.n = [len(t) for t in ids]
        self.starts = np.concatenate([[0], np.cumsum(self.n)])
        self.tokens = torch.as_tensor(np.concatenate(ids)).to(device).long()
        self.pos = torch.as_tensor(np.concatenate([np.arange(n) for n in self.n])).to(device)
        self.seq = torch.as_tensor(np.repeat(np.arange(len(ids)), self.n)).to(device)
        self.device = device

    def spans(self):
        return [(int(a), int(b)) for a, b in zip(self.starts[:-1], self.starts[1:])]

    def padded(self, x):
        """[T, ...] -> [longest, sequences, ...]"""
        out = torch.zeros((max(self.n), len(self.n)) + x.shape[1:], dtype=x.dtype, device=self.device)
        out[self.pos, self.seq] = x
        return out

    def conv(self, u, w, bias=None):
        """y_t = sum_j w[:, j] u_(t - taps + 1 + j) (+ bias) inside every sequence, then silu."""
        y = torch.zeros_like(u) if bias is None else bias.expand_as(u).clone()
        taps = w.shape[1]
        for j in range(taps):
            back = taps - 1 - j
            src = torch.arange(u.shape[0], device=self.device) - back
            y += w[:, j] * u[src.clamp(min=0)] * (self.pos >= back)[:, None]
        return torch.nn.functional.silu(y)

    def scan(self, q, k, v, decay, beta, delta):
        """S <- decay S, then S += k (beta v)^T (delta: k (beta (v - S^T k))^T); o = S^T q.  q, k [T, H, d], v [T, H, e],
        decay, beta [T, H].  Returns o [T, H, e] and the last states [sequences, H, d, e]."""
        qp, kp, vp, gp, bp = (self.padded(t) for t in (q, k, v, decay, beta))
        last = torch.as_tensor(self.n).to(self.device)
        S = torch.zeros(len(self.n), *k.shape[1:], v.shape[-1], dtype=F64, device=self.device)
        out = torch.empty_like(vp)
        for t in range(max(self.n)):
            new = S * gp[t, ..., None, None]
            u = vp[t]
            if delta:
                u = u - (new * kp[t, ..., None]).sum(-2)
            new.addcmul_(kp[t, ..., None], (u * bp[t, ..., None])[..., None, :])
            out[t] = (new * qp[t, ..., None]).sum(-2)
            S = torch.where((last > t).view(-1, 1, 1, 1), new, S)
        return out[self.pos, self.seq], S


def _family_exact(case, seed):
    device = torch.device("cuda", torch.cuda.current_device())
    cfg = _family_dict(case)
    model = build_model(_config(case), _ops(), device, torch.bfloat16)      # for the names and shapes of its checkpoint only
    w = _family_weights(case, model, seed, device)
    cached = functools.lru_cache(maxsize=None)(lambda name: w[name] if name.endswith("table") else w[name].to(F64))
    ids = _tokens(case, seed, cfg["vocab"])
    forward = {"mofidra": _mofidra, "mabivik": _mabivik, "vagozen": _vagozen}[case["model"]]
    parts = [forward(cfg, cached, _Packed([ids[i] for i in part], device))
             for part in _groups([(0, len(t)) for t in ids], 12288)]
    return torch.cat([p[0] for p in parts]), [torch.cat(s) if s[0] is not None else None for s in zip(*(p[1] for p in parts))]


def _last(seqs, x):
    return x[torch.as_tensor(seqs.starts[1:] - 1).to(x.device)]


def _mofidra(cfg, w, seqs):
    eps = cfg["norm"]["eps"]

    def norm(x, name):
        return _unit_rms(x, eps) * (1.0 + w(name))
    x = w("embed")[seqs.tokens] * cfg["embedding"]["scale"]
    for i, layer in enumerate(cfg["layers"]):
        p, m, T = f"l{i}.", layer["mixer"], x.shape[0]
        h = norm(x, p + "norm1")
        H, G, d, vd = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        freqs, _ = _ramp(m["rot"], x.device)
        q, k = ((h @ w(p + "mix." + n).T).view(T, heads, 2, d) for n, heads in (("q", H), ("k", G)))
        v = (h @ w(p + "mix.v").T).view(T, G, vd)
        lam = (torch.exp((w(p + "mix.lq1") * w(p + "mix.lk1")).sum()) - torch.exp((w(p + "mix.lq2") * w(p + "mix.lk2")).sum())
               + m["diff"])
        maps = []
        for j in range(2):
            qj, kj = _turn(q[:, :, j], seqs.pos, freqs), _turn(k[:, :, j], seqs.pos, freqs)
            maps.append(torch.cat([_attend(qj[a:b], kj[a:b], v[a:b], m["scale"], _causal(0, b - a, x.device))
                                   for a, b in seqs.spans()]))
        att = _unit_rms(maps[0] - lam * maps[1], eps) * (1.0 - m["diff"])
        ff = torch.nn.functional.gelu(h @ w(p + "mlp.up").T, approximate="tanh") @ w(p + "mlp.down").T
        x = x + att.reshape(T, H * vd) @ w(p + "mix.o").T + ff
    return norm(_last(seqs, x), "final.norm") @ w("head").T, []


def _latent_kv(w, q, m, h, seqs, eps, pairs):
    y, r = h @ w(q + "dkv").T, m["kv_rank"]
    freqs, amp = _ramp(m["rot"], h.device)
    return (_unit_rms(y[:, :r], eps) * w(q + "dkv.norm"), _turn(y[:, None, r:], seqs.pos, freqs, amp, pairs))


def _latent(w, q, m, h, seqs, eps, kv, pairs):
    """Per-head keys and values from the normed latent, one rotated key part for all heads."""
    T, H, d, rd, vd = h.shape[0], m["heads"], m["dim"], m["rot_dim"], m["vdim"]
    freqs, amp = _ramp(m["rot"], h.device)
    y = ((_unit_rms(h @ w(q + "dq").T, eps) * w(q + "dq.norm")) @ w(q + "uq").T).view(T, H, d + rd)
    qq = torch.cat([y[..., :d], _turn(y[..., d:], seqs.pos, freqs, amp, pairs)], -1)
    k = torch.cat([(kv[0] @ w(q + "uk").T).view(T, H, d), kv[1].expand(T, H, rd)], -1)
    v = (kv[0] @ w(q + "uv").T).view(T, H, vd)
    win = (m.get("mask") or {}).get("size", 0)
    return torch.cat([_attend(qq[a:b], k[a:b], v[a:b], m["scale"], _causal(0, b - a, h.device, win))
                      for a, b in seqs.spans()]).reshape(T, H * vd)


def _mabivik(cfg, w, seqs):
    eps, silu, softplus = cfg["norm"]["eps"], torch.nn.functional.silu, torch.nn.functional.softplus

    def norm(x, name):
        return torch.tanh(w(name + ".alpha") * x) * w(name) + w(name + ".b")
    x, kv, states = w("embed")[seqs.tokens] * cfg["embedding"]["scale"], {}, []
    for i, layer in enumerate(cfg["layers"]):
        p, q, m, kind, T = f"l{i}.", f"l{i}.mix.", layer["mixer"], layer["type"], x.shape[0]
        h, H, vd = norm(x, p + "norm1"), m["heads"], m["vdim"]
        if kind == "latent_attention":
            src = m.get("kv_from", i)
            if src == i:
                kv[i] = _latent_kv(w, q, m, h, seqs, eps, False)
            y = _latent(w, q, m, h, seqs, eps, kv[src], False) * torch.sigmoid(h @ w(q + "g").T)
        elif kind == "delta":
            G, d = m["kv_heads"], m["dim"]
            qq, kk, vv = (seqs.conv(h @ w(q + n).T, w(q + n + ".conv")) for n in "qkv")
            qq, kk = (t.view(T, G, d) / torch.sqrt((t.view(T, G, d) ** 2).sum(-1, keepdim=True) + 1e-6) for t in (qq, kk))
            qq, kk = (t.repeat_interleave(H // G, 1) for t in (qq * d ** -0.5, kk))
            decay = torch.exp(-torch.exp(w(q + "A_log")) * softplus(h @ w(q + "a").T + w(q + "dt_bias")))
            o, S = seqs.scan(qq, kk, vv.view(T, H, vd), decay, torch.sigmoid(h @ w(q + "b").T), True)
            states += [None, S]
            y = (_unit_rms(o, eps) * w(q + "norm") * silu(h @ w(q + "g").T).view(T, H, vd)).reshape(T, H * vd)
        else:
            N, G, inner, parts = m["state"], m["groups"], H * vd, m["norm_groups"]
            z, xbc, dt = (h @ w(q + "in").T).split([inner, inner + 2 * G * N, H], -1)
            xx, B, C = seqs.conv(xbc, w(q + "conv"), w(q + "conv.b")).split([inner, G * N, G * N], -1)
            B, C = (t.reshape(T, G, N).repeat_interleave(H // G, 1) for t in (B, C))
            xx, dt = xx.reshape(T, H, vd), softplus(dt + w(q + "dt_bias"))
            o, S = seqs.scan(C, B, xx, torch.exp(-torch.exp(w(q + "A_log")) * dt), dt, False)
            states += [None, S]
            o = (o + w(q + "D")[:, None] * xx).reshape(T, inner) * silu(z)
            y = _unit_rms(o.view(T, parts, inner // parts), eps).reshape(T, inner) * w(q + "norm")
        x = x + norm(y @ w(q + "o").T, p + "norm1b")
        h, f = norm(x, p + "norm2"), layer["mlp"]
        chosen = w(p + "mlp.table")[seqs.tokens].long()
        y = torch.zeros_like(x)
        for e in range(f["router"]["experts"]):
            t = (chosen == e).any(-1).nonzero()[:, 0]
            n = f"{p}mlp.e{e}."
            y[t] += (silu(h[t] @ w(n + "gate").T) * (h[t] @ w(n + "up").T)) @ w(n + "down").T / f["router"]["top"]
        x = x + norm(y, p + "norm2b")
        dim = cfg["token_side"]["dim"]
        side = w("side.embed")[seqs.tokens][:, i * dim:(i + 1) * dim]
        y = (torch.nn.functional.gelu(x @ w(p + "side.gate").T, approximate="tanh") * side) @ w(p + "side.proj").T
        x = x + _unit_rms(y, eps) * w(p + "side.norm")
    return norm(_last(seqs, x), "final.norm") @ w("head").T * cfg["logit_scale"], states


def _vagozen(cfg, w, seqs):
    eps, silu, loop = cfg["norm"]["eps"], torch.nn.functional.silu, cfg["loop"]

    def norm(x, name):
        return _unit_rms(x, eps) * w(name)
    x0 = w("embed")[seqs.tokens]
    x, states, opened = x0, [], 0
    for r, i in enumerate(_layer_order(cfg)):
        p, q, m, kind, T = f"l{i}.", f"l{i}.mix.", cfg["layers"][i]["mixer"], cfg["layers"][i]["type"], x.shape[0]
        if i == loop["start"]:      # a pass opens: its vector, from the second on the embedding too
            x = x + w("loop.step")[opened] + (x0 if opened else 0.0)
            opened += 1
        h, H, vd = norm(x, p + "norm1"), m["heads"], m["vdim"]
        freqs, amp = _ramp(m["rot"], x.device)
        if kind == "attention":
            G, d, mask = m["kv_heads"], m["dim"], m["mask"]
            qq, kk, vv = ((h @ w(q + n).T + w(q + n + ".b")).view(T, heads, -1) for n, heads in (("q", H), ("k", G), ("v", G)))
            qq, kk = _turn(qq, seqs.pos, freqs, amp, True), _turn(kk, seqs.pos, freqs, amp, True)
            y = torch.cat([_attend(qq[a:b], kk[a:b], vv[a:b], m["scale"], _causal(0, b - a, x.device, mask["size"], mask["keep_first"]))
                           for a, b in seqs.spans()]).reshape(T, H * vd)
        elif kind == "retention":
            d = m["dim"]
            qq, kk = (_turn((h @ w(q + n).T).view(T, H, d), seqs.pos, freqs, amp) for n in "qk")
            decay = torch.tensor(m["decay"], dtype=F64, device=x.device).expand(T, H)
            o, S = seqs.scan(qq, kk / math.sqrt(d), (h @ w(q + "v").T).view(T, H, vd), decay, torch.ones_like(decay), False)
            states.append(S)
            y = _unit_rms(o, eps).reshape(T, H * vd) * silu(h @ w(q + "g").T)
        else:
            y = _latent(w, q, m, h, seqs, eps, _latent_kv(w, q, m, h, seqs, eps, True), True)
        x = x + norm(y @ w(q + "o").T, p + "norm1b") * w(p + "ls1")
        h, f = norm(x, p + "norm2"), cfg["layers"][i]["mlp"]
        g, u = (h @ w(p + "mlp.gate").T).clamp(max=f["limit"]), (h @ w(p + "mlp.up").T).clamp(-f["limit"], f["limit"])
        x = x + norm((g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ w(p + "mlp.down").T, p + "norm2b") * w(p + "ls2")
    return norm(_last(seqs, x), "final.norm") @ w("embed").T * cfg["logit_scale"], states
