"""Performance cases: the work a serving program has this framework do.

Every case goes through the entry points such a program calls: the kernels'
tensor front end (``nanovllm_amd.kernels``), one decoder layer, the language
model head with the acceptance scan, one draft step and a whole prompt through
the target.  Shapes are the Qwen3-0.6B / 8B / 32B geometries of
``nanovllm_amd.synthetic`` with the batch sizes, draft lengths and context
ranges of the benchmark and of the kernel tests.

A case's ragged lengths follow from the case itself (``_lengths``), so that
``work`` counts them exactly; the seed makes the values, the page order and
the token ids.
"""
from __future__ import annotations

import math
import os
import random
import sys
import zlib
from types import SimpleNamespace

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "extend-nano-vllm_amd"))

from nanovllm_amd import kernels as K  # noqa: E402
from nanovllm_amd.context import reset_context, set_context  # noqa: E402
from nanovllm_amd.eagle3 import Eagle3Config, Eagle3ForCausalLM  # noqa: E402
from nanovllm_amd.layers import RMSNorm, init_random_  # noqa: E402
from nanovllm_amd.qwen3 import Qwen3DecoderLayer, Qwen3ForCausalLM, aux_concat  # noqa: E402
from nanovllm_amd.synthetic import QWEN3_PRESETS, default_aux_layers  # noqa: E402

BF16 = torch.bfloat16
BLOCK = 256                 # tokens per KV page
D = 128                     # head_dim of every preset
KV_HEADS = 8
EPS = 1e-6
THETA = 1000000.0
CHUNK_TOKENS = 16384        # the scheduler's token budget of one prefill step
HEADS = {"qwen3-0.6b": 16, "qwen3-8b": 32, "qwen3-32b": 64}


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # one request being served, 1024-token prompt and k = 8 drafts: the
        # smallest verify call there is, all latency
        dict(name="verify-one-8b", kind="verify", preset="qwen3-8b", batch=1, q=9, lo=1033,
             hi=1289, kv="bf16"),
        # the headline serving batch (k = 5, prompts of 256-2048 plus output)
        dict(name="verify-8b", kind="verify", preset="qwen3-8b", batch=64, q=6, lo=256, hi=2304,
             kv="bf16"),
        # the largest model at a large batch and long contexts: 2.7 GB of keys
        # and values in one call
        dict(name="verify-32b", kind="verify", preset="qwen3-32b", batch=128, q=8, lo=2048,
             hi=8192, kv="bf16"),
        # FP8 pages, long contexts
        dict(name="verify-fp8", kind="verify", preset="qwen3-0.6b", batch=128, q=5, lo=4096,
             hi=16384, kv="fp8"),
        # serving without drafts, one new token per sequence
        dict(name="decode-0.6b", kind="decode", preset="qwen3-0.6b", batch=32, q=1, lo=512,
             hi=4096, kv="bf16"),
        # attention of one prefill step: several ordinary prompts packed into
        # the token budget
        dict(name="prefill-8b", kind="prefill", preset="qwen3-8b", lo=256, hi=2048, cached=0,
             kv="bf16"),
        # long prompts of the largest model
        dict(name="prefill-32b", kind="prefill", preset="qwen3-32b", lo=2048, hi=8192, cached=0,
             kv="bf16"),
        # long prompts over FP8 pages whose first blocks come from the prefix
        # cache
        dict(name="prefill-fp8", kind="prefill", preset="qwen3-0.6b", lo=4096, hi=8192,
             cached=2048, kv="fp8"),
        # the head after a verify forward: final norm, logits of every row,
        # argmax and acceptance
        dict(name="head-8b", kind="head", preset="qwen3-8b", batch=64, q=6),
        # one decoder layer of the headline verify forward
        dict(name="layer-verify-8b", kind="layer", preset="qwen3-8b", mode="verify", batch=64, q=6,
             lo=256, hi=2304),
        # one EAGLE3 draft step at the headline batch, with its sampling
        dict(name="draft-8b", kind="draft", preset="qwen3-8b", batch=64, lo=256, hi=2304),
        # time to first token: one 1024-token prompt through the whole target
        dict(name="first-token-0.6b", kind="model", preset="qwen3-0.6b", lo=1024, hi=1024),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    most = [work(c) for c in listed()]
    while True:
        case = _draw(rng)
        w = work(case)
        if all(w[k] <= max(m[k] for m in most) for k in w):
            return case


def _draw(rng):
    kind = rng.choice(["verify", "verify", "decode", "decode", "prefill", "prefill", "prefill",
                       "head", "layer", "layer", "draft", "model"])
    preset = rng.choice(sorted(HEADS))
    kv = rng.choice(["bf16", "bf16", "fp8"])
    if kind in ("verify", "decode"):
        q = 1 if kind == "decode" else rng.randint(2, 9)
        batch = _log_int(rng, 1, 128 if kind == "verify" else 256)
        hi = _log_int(rng, 300, 16384)
        # at most the largest listed call's keys
        hi = max(300, min(hi, 2 * 600000 // batch - 256))
        return dict(kind=kind, preset=preset, batch=batch, q=q, lo=max(q, hi // rng.randint(2, 9)),
                    hi=hi, kv=kv)
    if kind == "prefill":
        hi = _log_int(rng, 64, 8192)
        cached = rng.choice([0, 0, 0, 256, 512, 1024, 2048])
        return dict(kind=kind, preset=preset, lo=max(1, hi // rng.randint(1, 8)), hi=hi,
                    cached=cached, kv=kv)
    if kind == "head":
        return dict(kind=kind, preset=rng.choice(["qwen3-0.6b", "qwen3-8b"]),
                    batch=_log_int(rng, 1, 64), q=rng.randint(2, 6))
    if kind == "layer":
        mode = rng.choice(["verify", "decode", "prefill"])
        hi = _log_int(rng, 300, 4096)
        q = dict(verify=rng.randint(2, 7), decode=1, prefill=0)[mode]
        batch = _log_int(rng, 1, 64) if mode != "prefill" else rng.randint(1, 3)
        if mode == "prefill":
            hi = min(hi, 4096 // batch)
        return dict(kind=kind, preset=rng.choice(["qwen3-0.6b", "qwen3-8b"]), mode=mode,
                    batch=batch, q=q, lo=max(q, hi // rng.randint(2, 9)), hi=hi)
    if kind == "draft":
        hi = _log_int(rng, 300, 4096)
        return dict(kind=kind, preset=rng.choice(["qwen3-0.6b", "qwen3-8b"]),
                    batch=_log_int(rng, 1, 64), lo=max(2, hi // rng.randint(2, 9)), hi=hi)
    n = _log_int(rng, 16, 2048)
    return dict(kind="model", preset="qwen3-0.6b", lo=n, hi=n)


# ---------------------------------------------------------------- lengths

def _rng(case):
    text = repr(sorted((k, v) for k, v in case.items() if k != "name"))
    return random.Random(zlib.crc32(text.encode()))


def _lengths(case):
    """(query rows, keys) of every sequence; a sequence's query rows are its
    last keys."""
    rng = _rng(case)
    lo, hi = case["lo"], case["hi"]
    kind = case["kind"]
    if kind == "prefill":
        rows = []
        while len(rows) < 256:
            n = rng.randint(lo, hi)
            if rows and sum(rows) + n > CHUNK_TOKENS:
                break
            rows.append(n)
        return rows, [n + case["cached"] for n in rows]
    if kind == "model":
        return [lo], [lo]
    n = case["batch"]
    keys = [rng.randint(lo, hi) for _ in range(n)]
    if kind == "layer" and case["mode"] == "prefill":
        return keys, list(keys)
    q = case.get("q", 1)
    if kind == "verify" or kind == "layer" and case["mode"] == "verify":
        keys.sort(reverse=True)      # the engine verifies longest sequences first
    return [q] * n, keys


def _pairs(rows, keys):
    """(query row, visible key) pairs under the bottom-right causal mask."""
    return sum(r * k - r * (r - 1) // 2 for r, k in zip(rows, keys))


def _cu(values):
    out = [0]
    for v in values:
        out.append(out[-1] + v)
    return out


# ---------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _i32(values):
    return torch.tensor(values, dtype=torch.int32).to("cuda")


def _normal(shape, gen, std=1.0, dtype=BF16):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, std, generator=gen)


def _pages(rows, keys, seed, gen, fp8=False):
    """A paged cache holding `keys` tokens per sequence in shuffled pages, as
    the engine stores it (one kv head's K rows then V rows per page), seen
    through the [blocks, block_size, heads, head_dim] views it hands out."""
    blocks = [-(-k // BLOCK) for k in keys]
    order = list(range(sum(blocks)))
    random.Random(seed).shuffle(order)
    table, at = [], 0
    for n in blocks:
        table.append(order[at:at + n] + [-1] * (max(blocks) - n))
        at += n
    shape = (sum(blocks), KV_HEADS, 2, BLOCK, D)
    if fp8:
        pages = torch.empty(shape, dtype=torch.float8_e4m3fn, device="cuda")
        step = max(1, (1 << 28) // (KV_HEADS * 2 * BLOCK * D))
        for b in range(0, shape[0], step):
            part = pages[b:b + step]
            part.copy_(_normal(part.shape, gen))
    else:
        pages = _normal(shape, gen)
    view = pages.permute(2, 0, 3, 1, 4)
    slots = []
    for t, r, k in zip(table, rows, keys):
        slots.extend(t[p // BLOCK] * BLOCK + p % BLOCK for p in range(k - r, k))
    positions = torch.tensor([p for r, k in zip(rows, keys) for p in range(k - r, k)],
                             dtype=torch.int64).to("cuda")
    return SimpleNamespace(k=view[0], v=view[1], table=_i32(table), rows=rows, keys=keys,
                           max_q=max(rows),
                           cu_q=_i32(_cu(rows)), cu_k=_i32(_cu(keys)), lens=_i32(keys),
                           slots=_i32(slots), positions=positions)


def _bound(case):
    """The longest context the program declares (its configured limit)."""
    return max(case["hi"], case.get("q", 1)) + case.get("cached", 0)


def _hf(preset, **changes):
    return SimpleNamespace(rms_norm_eps=EPS, rope_theta=THETA, attention_bias=False,
                           **dict(QWEN3_PRESETS[preset], **changes))


def _bf16_module(make, seed):
    """A module with random bf16 weights, built on the GPU as the engine does."""
    default = torch.get_default_dtype()
    torch.set_default_dtype(BF16)
    torch.set_default_device("cuda")
    try:
        m = make()
    finally:
        torch.set_default_device("cpu")
        torch.set_default_dtype(default)
    init_random_(m, int(seed) % (1 << 31))
    gen = _gen(seed + 1)
    for p in m.modules():
        if isinstance(p, RMSNorm):       # trained norm weights are spread around one
            p.weight.data.normal_(1.0, 0.1, generator=gen)
    return m.eval()


def prepare(case, seed):
    kind = case["kind"]
    gen = _gen(seed)
    s = SimpleNamespace(case=case, kind=kind)
    p = QWEN3_PRESETS[case["preset"]]
    h, hq = p["hidden_size"], p["num_attention_heads"]
    if kind == "head":
        t, v = case["batch"] * case["q"], p["vocab_size"]
        s.model = _bf16_module(
            lambda: Qwen3ForCausalLM(_hf(case["preset"], num_hidden_layers=0)), seed)
        # a trained model's rows point at a token; about 70% of the drafts
        # guess the token of the row before them
        tokens = torch.randint(0, v, (t,), generator=gen, device="cuda")
        s.hidden = _normal((t, h), gen, 0.5)
        s.residual = _normal((t, h), gen) + 15.0 * s.model.lm_head.weight[tokens]
        s.cu_q = _i32(list(range(0, t + 1, case["q"])))
        wrong = torch.rand(t, generator=gen, device="cuda") > 0.7
        s.ids = torch.where(wrong, torch.randint(0, v, (t,), generator=gen, device="cuda"),
                            tokens.roll(1))
        return s
    rows, keys = _lengths(case)
    t = sum(rows)
    if kind in ("verify", "decode", "prefill"):
        s.kv = _pages(rows, keys, seed, gen, case["kv"] == "fp8")
        s.q = _normal((t, hq, D), gen)
        s.scale = torch.ones(1, dtype=torch.float32, device="cuda")
        return s
    if kind == "layer":
        s.kv = _pages(rows, keys, seed, gen)
        s.layer = _bf16_module(lambda: Qwen3DecoderLayer(_hf(case["preset"])), seed)
        s.layer.self_attn.attn.k_cache, s.layer.self_attn.attn.v_cache = s.kv.k, s.kv.v
        s.hidden, s.residual = _normal((t, h), gen), _normal((t, h), gen)
        return s
    if kind == "draft":
        s.kv = _pages(rows, keys, seed, gen)
        config = Eagle3Config(
            hidden_size=h, intermediate_size=p["intermediate_size"], num_attention_heads=hq,
            num_key_value_heads=KV_HEADS, head_dim=D,
            max_position_embeddings=p["max_position_embeddings"], rms_norm_eps=EPS,
            rope_theta=THETA, attention_bias=False, target_vocab_size=p["vocab_size"],
            draft_vocab_size=p["vocab_size"], target_hidden_size=h, num_aux_hidden_states=3,
            norm_before_residual=True, torch_dtype=BF16)
        s.draft = _bf16_module(lambda: Eagle3ForCausalLM(config), seed)
        s.draft.layers[0].self_attn.attn.k_cache = s.kv.k
        s.draft.layers[0].self_attn.attn.v_cache = s.kv.v
        s.ids = torch.randint(0, p["vocab_size"], (t,), generator=gen, device="cuda")
        # a trained draft's rows point at a token
        tokens = torch.randint(0, p["vocab_size"], (t,), generator=gen, device="cuda")
        s.feedback = _normal((t, h), gen) + 40.0 * s.draft.lm_head.weight[tokens]
        return s
    # model
    s.model = _bf16_module(lambda: Qwen3ForCausalLM(_hf(case["preset"])), seed)
    s.aux_layers = default_aux_layers(case["preset"])
    s.kv = _pages(rows, keys, seed, gen)
    for layer in s.model.model.layers:
        k = torch.zeros(s.kv.k.shape[0], KV_HEADS, 2, BLOCK, D, dtype=BF16, device="cuda")
        k = k.permute(2, 0, 3, 1, 4)
        layer.self_attn.attn.k_cache, layer.self_attn.attn.v_cache = k[0], k[1]
    s.ids = torch.randint(0, p["vocab_size"], (t,), generator=gen, device="cuda")
    return s


# ---------------------------------------------------------------- one pass

def _context(s, prefill):
    kv = s.kv
    if prefill:
        set_context(True, kv.cu_q, kv.cu_k, kv.max_q, max(kv.keys) if s.kind == "model"
                    else _bound(s.case), kv.slots, None, kv.table)
    else:
        set_context(False, slot_mapping=kv.slots, context_lens=kv.lens, block_tables=kv.table,
                    max_seqlen_k=_bound(s.case))


@torch.inference_mode()
def run(s):
    kind, case = s.kind, s.case
    if kind == "head":
        hidden, residual = s.model.model.norm(s.hidden, s.residual)
        logits = s.model.compute_all_logits(hidden)
        argmax, accepted, bonus = K.argmax_accept(logits, s.cu_q, s.ids)
        return dict(logits=logits, residual=residual, argmax=argmax, accepted=accepted,
                    bonus=bonus)
    kv = s.kv
    scales = dict(k_scale=s.scale, v_scale=s.scale) if case.get("kv") == "fp8" else {}
    if kind == "decode":
        return K.paged_attention_decode(s.q, kv.k, kv.v, kv.lens, kv.table, D ** -0.5,
                                        max_seqlen_k=_bound(case), **scales)
    if kind in ("verify", "prefill"):
        return K.paged_attention_varlen(s.q, kv.k, kv.v, kv.cu_q, kv.cu_k, kv.max_q,
                                        _bound(case), D ** -0.5, kv.table, **scales)
    try:
        if kind == "layer":
            _context(s, case["mode"] != "decode")
            hidden, residual = s.layer(kv.positions, s.hidden, s.residual)
            return dict(hidden=hidden, residual=residual, k_cache=kv.k, v_cache=kv.v)
        if kind == "draft":
            _context(s, False)
            hidden, feedback = s.draft.forward_with_cache(s.ids, kv.positions, s.feedback)
            logits = s.draft.lm_head(hidden)
            return dict(hidden=hidden, feedback=feedback, logits=logits,
                        tokens=K.argmax_rows(logits, s.draft.d2t), k_cache=kv.k, v_cache=kv.v)
        _context(s, True)
        hidden, aux = s.model.forward_with_aux_hidden_states(s.ids, kv.positions, s.aux_layers)
        logits = s.model.compute_logits(hidden[kv.cu_q[1:].long() - 1])
        return dict(logits=logits, aux=aux_concat(aux))
    finally:
        reset_context()


# ---------------------------------------------------------------- work and tolerance

def _layer_work(p, t, rows, keys, inputs=1):
    """(bytes, flops) of one decoder layer over t rows: weights, K/V, rows."""
    h, i, hq = p["hidden_size"], p["intermediate_size"], p["num_attention_heads"]
    weights = (inputs * h * (hq + 2 * KV_HEADS) * D + hq * D * h + 3 * h * i)
    kv = sum(keys) * KV_HEADS * D * 2
    return 2 * (weights + kv), 2 * t * weights + 4 * hq * D * _pairs(rows, keys)


def work(case):
    kind, p = case["kind"], QWEN3_PRESETS[case["preset"]]
    h, hq, v = p["hidden_size"], p["num_attention_heads"], p["vocab_size"]
    if kind == "head":
        t = case["batch"] * case["q"]
        return {"bytes": 2 * (v * h + 3 * t * h + t * v) + 4 * t, "flops": 2 * t * v * h}
    rows, keys = _lengths(case)
    t = sum(rows)
    if kind in ("verify", "decode", "prefill"):
        esz = 1 if case["kv"] == "fp8" else 2
        return {"bytes": sum(keys) * KV_HEADS * D * 2 * esz + 2 * t * hq * D * 2,
                "flops": 4 * hq * D * _pairs(rows, keys)}
    if kind == "layer":
        b, f = _layer_work(p, t, rows, keys)
        return {"bytes": b + 2 * 4 * t * h, "flops": f}
    if kind == "draft":
        b, f = _layer_work(p, t, rows, keys, inputs=2)
        return {"bytes": b + 2 * (v * h + t * v + 4 * t * h), "flops": f + 2 * t * v * h}
    b, f = _layer_work(p, t, rows, keys)
    n = p["num_hidden_layers"]
    return {"bytes": n * b + 2 * (v * h + v + t * h + 3 * t * h), "flops": n * f + 2 * v * h}


def tolerance(case):
    """About four times what two correct bf16 implementations differ by."""
    kind = case["kind"]
    if kind in ("verify", "decode", "prefill"):
        # probabilities and the result rounded to bf16
        return {"rel": 1e-2, "max": 0.1}
    if kind == "head":
        # bf16 logits of bf16 rows; a row's best two may tie
        return {"rel": 1e-2, "max": 0.1, "differ": 0.01}
    if kind in ("layer", "draft"):
        # half a dozen bf16 roundings on the way
        return {"rel": 2e-2, "max": 0.25, "differ": 0.01}
    # every layer's rounding travels through all that follow
    return {"rel": 3e-2, "max": 0.5, "differ": 0.01}


# ---------------------------------------------------------------- 64-bit results

def _norm64(x, w, eps=EPS):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _rope64(x, positions):
    # the angles are float32 by definition
    freq = 1.0 / THETA ** (torch.arange(0, D, 2, dtype=torch.float32) / D)
    angle = (positions.float()[:, None] * freq.to(x.device)).double()[:, None]
    c, s = angle.cos(), angle.sin()
    a, b = x[..., :D // 2], x[..., D // 2:]
    return torch.cat((a * c - b * s, b * c + a * s), -1)


def _attend64(q, kv, rows, keys, new=None):
    """softmax(q k^T / sqrt(D)) v in float64 over the paged cache; `new` are
    (k, v) rows that take the place of each sequence's last cached rows."""
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    g = q.shape[1] // KV_HEADS
    at = 0
    for i, (r, n) in enumerate(zip(rows, keys)):
        ids = kv.table[i, :-(-n // BLOCK)].long()
        k = kv.k[ids].reshape(-1, KV_HEADS, D)[:n].double()
        v = kv.v[ids].reshape(-1, KV_HEADS, D)[:n].double()
        if new is not None:
            k[n - r:], v[n - r:] = new[0][at:at + r], new[1][at:at + r]
        for j in range(0, r, 1024):
            m = min(1024, r - j)
            see = n - r + j + m
            mask = (torch.arange(see, device=q.device)[None]
                    > torch.arange(n - r + j, see, device=q.device)[:, None])
            for h in range(KV_HEADS):
                qq = q[at + j:at + j + m, h * g:(h + 1) * g].double()
                sc = (qq.reshape(m * g, D) @ k[:see, h].t()).view(m, g, see) * D ** -0.5
                sc.masked_fill_(mask[:, None], -math.inf)
                o = torch.softmax(sc, -1).view(m * g, see) @ v[:see, h]
                out[at + j:at + j + m, h * g:(h + 1) * g] = o.view(m, g, D)
        at += r
    return out


def _self_attention64(m, x, kv, qk_norm):
    hq = m.num_heads
    qkv = x @ m.qkv_proj.weight.double().t()
    t = x.shape[0]
    q, k, v = (y.reshape(t, -1, D) for y in qkv.split([hq * D, KV_HEADS * D, KV_HEADS * D], -1))
    if qk_norm:
        q, k = _norm64(q, m.q_norm.weight), _norm64(k, m.k_norm.weight)
    q, k = _rope64(q, kv.positions), _rope64(k, kv.positions)
    o = _attend64(q, kv, kv.rows, kv.keys, (k, v))
    return o.reshape(t, -1) @ m.o_proj.weight.double().t()


def _mlp64(m, x):
    a, b = (x @ m.gate_up_proj.weight.double().t()).chunk(2, -1)
    return (torch.nn.functional.silu(a) * b) @ m.down_proj.weight.double().t()


def _layer64(layer, kv, hidden, residual):
    residual = hidden + residual
    x = _norm64(residual, layer.input_layernorm.weight)
    residual = residual + _self_attention64(layer.self_attn, x, kv, True)
    return _mlp64(layer.mlp, _norm64(residual, layer.post_attention_layernorm.weight)), residual


def _logits64(x, weight):
    return torch.cat([x @ w.double().t() for w in weight.split(16384)], -1)


@torch.inference_mode()
def exact(case, seed):
    kind = case["kind"]
    s = prepare(case, seed)
    if kind == "head":
        residual = s.hidden.double() + s.residual.double()
        logits = _logits64(_norm64(residual, s.model.model.norm.weight), s.model.lm_head.weight)
        return dict(logits=logits, residual=residual, argmax=None, accepted=None, bonus=None)
    kv = s.kv
    if kind in ("verify", "decode", "prefill"):
        return _attend64(s.q, kv, kv.rows, kv.keys)
    if kind == "layer":
        hidden, residual = _layer64(s.layer, kv, s.hidden.double(), s.residual.double())
        return dict(hidden=hidden, residual=residual, k_cache=None, v_cache=None)
    if kind == "draft":
        d = s.draft.layers[0]
        x = _norm64(s.draft.embed_tokens.weight[s.ids].double(), d.input_layernorm.weight)
        residual = _norm64(s.feedback.double(), d.hidden_norm.weight)
        x = torch.cat((x, residual), -1)
        residual = residual + _self_attention64(d.self_attn, x, kv, False)
        feedback = residual + _mlp64(d.mlp, _norm64(residual, d.post_attention_layernorm.weight))
        hidden = _norm64(feedback, s.draft.norm.weight)
        return dict(hidden=hidden, feedback=feedback,
                    logits=_logits64(hidden, s.draft.lm_head.weight), tokens=None, k_cache=None,
                    v_cache=None)
    m = s.model.model
    hidden = m.embed_tokens.weight[s.ids].double()
    residual, aux = torch.zeros_like(hidden), []
    for n, layer in enumerate(m.layers, start=1):
        hidden, residual = _layer64(layer, kv, hidden, residual)
        if n in s.aux_layers:
            aux.append(hidden + residual)
    last = _norm64((hidden + residual)[kv.cu_q[1:].long() - 1], m.norm.weight)
    return dict(logits=_logits64(last, s.model.lm_head.weight), aux=torch.cat(aux, -1))
