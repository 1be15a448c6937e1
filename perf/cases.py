"""Performance cases: the attention and Gated DeltaNet work of a serving engine.

Every case goes through the entry points that a nano_qwen user calls: the
``Attention`` layer, the fused q/k norm + rotary + store, ``gdn_core`` and
``ModelRunner`` with its captured decode graphs.  Lengths follow from the case
alone (``lens`` seeds them, so that a batch is ragged); the seed given to
``prepare`` makes the values and the block permutation.

Kinds:

* ``decode``       one layer's decode step: the new token's store and the attention
* ``graph``        a whole decode step replayed from its captured graph: per layer
                   the q/k norm + rotary + store and the gated decode
* ``prefill``      one layer's prefill: store and causal attention, over packed
                   K/V, or over the paged cache when a prefix is cached; with
                   ``norm`` the q/k norm + rotary + store and the output gate too
* ``gdn_prefill``  one Gated DeltaNet layer's core over packed prompts
* ``gdn_decode``   the same for one token per sequence
"""
import math
import random
from types import SimpleNamespace

import torch

from nano_qwen_amd.engine import ModelRunner
from nano_qwen_amd.layers import Attention, gdn_core, qk_norm_rope_store
from nano_qwen_amd.utils.context import set_context

BLOCK = 256
VOCAB = 512
EPS = 1e-6
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
DEVICE = "cuda"


# ------------------------------------------------------------------- cases

def listed():
    return [
        # one user's chat, token by token without graphs: latency is all
        dict(name="decode_one_user", kind="decode", batch=1, lo=777, hi=777, hq=32, hkv=8, d=128,
             dtype="bf16", kv="same", lens=1),
        # a few users of a Qwen3.5 engine: the runner replays the whole step's graph
        dict(name="decode_step_graph", kind="graph", batch=6, lo=150, hi=3000, hq=16, hkv=4, d=256, rot=64,
             layers=8, dtype="bf16", kv="same", lens=2),
        # a busy server's step, Qwen3-8B heads (the benchmark's headline shape)
        dict(name="decode_batch", kind="decode", batch=64, lo=1024, hi=4096, hq=32, hkv=8, d=128,
             dtype="bf16", kv="same", lens=3),
        # the largest batch, its contexts held as fp8
        dict(name="decode_batch_fp8", kind="decode", batch=128, lo=2048, hi=8192, hq=32, hkv=8, d=128,
             dtype="bf16", kv="fp8", lens=4),
        # few sequences with long contexts (documents, agents), 64 query heads
        dict(name="decode_long", kind="decode", batch=3, lo=20000, hi=32768, hq=64, hkv=8, d=128,
             dtype="bf16", kv="same", lens=5),
        # time to first token of one ordinary prompt
        dict(name="prefill_prompt", kind="prefill", batch=1, lo=1111, hi=1111, pre_lo=0, pre_hi=0, hit=1, hq=32,
             hkv=8, d=128, rot=0, norm=False, dtype="bf16", kv="same", lens=6),
        # a full prefill batch, half of its prompts behind a cached prefix
        dict(name="prefill_batch", kind="prefill", batch=16, lo=256, hi=2048, pre_lo=1, pre_hi=4, hit=2, hq=32,
             hkv=8, d=128, rot=0, norm=False, dtype="bf16", kv="same", lens=7),
        # the next turns of a few long chats: short questions behind cached fp8 histories
        dict(name="prefill_chat_fp8", kind="prefill", batch=4, lo=40, hi=400, pre_lo=16, pre_hi=32, hit=1, hq=32,
             hkv=8, d=128, rot=0, norm=False, dtype="bf16", kv="fp8", lens=8),
        # two long documents, as many tokens as one prefill step takes
        dict(name="prefill_long", kind="prefill", batch=2, lo=7900, hi=8192, pre_lo=0, pre_hi=0, hit=1, hq=32,
             hkv=8, d=128, rot=0, norm=False, dtype="bf16", kv="same", lens=9),
        # a Qwen3.5 full-attention layer's prefill: q/k norm, rotary, store, gated attention at head_dim 256
        dict(name="prefill_gated_d256", kind="prefill", batch=6, lo=200, hi=3000, pre_lo=0, pre_hi=0, hit=1, hq=16,
             hkv=4, d=256, rot=64, norm=True, dtype="bf16", kv="same", lens=10),
        # a Qwen3.5 linear-attention layer's prefill of a few prompts
        dict(name="gdn_prefill", kind="gdn_prefill", batch=3, lo=500, hi=4000, h=16, hv=32, dtype="bf16", lens=11),
        # and its decode step for a server's batch
        dict(name="gdn_decode", kind="gdn_decode", batch=48, h=16, hv=32, dtype="bf16", lens=12),
    ]


HEADS_128 = ((32, 8), (64, 8), (16, 8), (16, 4), (8, 2))
HEADS_256 = ((16, 4), (16, 2), (8, 2))
HEADS_GDN = ((16, 32), (16, 16), (8, 32), (4, 8))


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    most = [work(c) for c in listed()]
    most = {k: max(w[k] for w in most) for k in ("bytes", "flops")}
    while True:
        case = _draw(rng)
        w = work(case)
        if w["bytes"] <= most["bytes"] and w["flops"] <= most["flops"]:
            return case


def _draw(rng):
    kind = rng.choice(("decode", "decode", "graph", "prefill", "prefill", "prefill", "gdn_prefill", "gdn_decode"))
    dtype = rng.choice(("bf16", "bf16", "f16"))
    kv = rng.choice(("same", "same", "fp8"))
    d = rng.choice((128, 128, 256))
    hq, hkv = rng.choice(HEADS_128 if d == 128 else HEADS_256)
    rot = d // 4
    lens = rng.randrange(1 << 30)
    if kind == "decode":
        hi = _log(rng, 64, 32768)
        return dict(kind=kind, batch=_log(rng, 1, 128), lo=max(1, int(hi * rng.uniform(0.1, 1.0))), hi=hi, hq=hq,
                    hkv=hkv, d=d, dtype=dtype, kv=kv, lens=lens)
    if kind == "graph":
        hi = _log(rng, 64, 8192)
        return dict(kind=kind, batch=_log(rng, 1, 32), lo=max(1, int(hi * rng.uniform(0.1, 1.0))), hi=hi, hq=hq,
                    hkv=hkv, d=d, rot=rot, layers=rng.choice((4, 8)), dtype=dtype, kv=kv, lens=lens)
    if kind == "prefill":
        hi = _log(rng, 16, 8192)
        pre = rng.choice((0, 0, _log(rng, 1, 32)))
        norm = rng.random() < 0.4
        return dict(kind=kind, batch=_log(rng, 1, 16), lo=max(1, int(hi * rng.uniform(0.1, 1.0))), hi=hi,
                    pre_lo=(pre + 1) // 2, pre_hi=pre, hit=rng.choice((1, 2)), hq=hq, hkv=hkv, d=d,
                    rot=rot if norm else 0, norm=norm, dtype=dtype, kv=kv if pre else "same", lens=lens)
    h, hv = rng.choice(HEADS_GDN)
    if kind == "gdn_prefill":
        hi = _log(rng, 32, 8192)
        return dict(kind=kind, batch=_log(rng, 1, 16), lo=max(1, int(hi * rng.uniform(0.1, 1.0))), hi=hi, h=h, hv=hv,
                    dtype=dtype, lens=lens)
    return dict(kind=kind, batch=_log(rng, 1, 128), h=h, hv=hv, dtype=dtype, lens=lens)


def _lengths(case):
    """(new tokens, cached tokens before them) of each sequence."""
    r = random.Random(case["lens"])
    new = [r.randint(case["lo"], case["hi"]) for _ in range(case["batch"])]
    pre = [0] * len(new)
    if case.get("pre_hi"):    # one of every ``hit`` sequences has a cached prefix
        pre = [BLOCK * r.randint(case["pre_lo"], case["pre_hi"]) if i % case["hit"] == 0 else 0
               for i in range(len(new))]
    return new, pre


# ------------------------------------------------------------------ inputs

def _randn(gen, *shape, dtype=torch.float32, amp=1.0):
    x = torch.randn(shape, generator=gen, device=DEVICE, dtype=torch.float32)
    return (x.mul_(amp) if amp != 1.0 else x).to(dtype)


def _tables(counts, pool, seed):
    perm = torch.randperm(pool, generator=torch.Generator().manual_seed(seed)).to(torch.int32)
    tables = torch.full((len(counts), max(counts)), -1, dtype=torch.int32)
    at = 0
    for i, c in enumerate(counts):
        tables[i, :c] = perm[at:at + c]
        at += c
    return tables


def _slots(tables, pre, new):
    """Cache rows of each sequence's new tokens, packed."""
    out = []
    for i, (p, n) in enumerate(zip(pre, new)):
        t = torch.arange(p, p + n)
        out.append(tables[i].long()[t // BLOCK] * BLOCK + t % BLOCK)
    return torch.cat(out).to(torch.int32)


def _pool(case, lk, layers, seed, gen):
    """A runner whose pool holds keys and values for every sequence (and a
    tenth more blocks), with tables in a random block order."""
    counts = [(n + BLOCK - 1) // BLOCK for n in lk]
    blocks = math.ceil(1.1 * sum(counts))
    tables = _tables(counts, blocks, seed)
    dtype = DTYPES[case["dtype"]]
    runner = ModelRunner(block_size=BLOCK, max_num_seqs=case["batch"], device=DEVICE)
    attns = [Attention(case["hq"], case["d"], case["d"] ** -0.5, case["hkv"]) for _ in range(layers)]
    kv = torch.float8_e4m3fn if case["kv"] == "fp8" else dtype
    runner.allocate_kv_cache(torch.nn.ModuleList(attns), layers, blocks, case["hkv"], case["d"], dtype,
                             kv_cache_dtype=kv)
    shape = (blocks, BLOCK, case["hkv"], case["d"])
    for a in attns:
        for cache, scale in ((a.k_cache, a.k_scale), (a.v_cache, a.v_scale)):
            x = torch.randn(shape, generator=gen, device=DEVICE, dtype=torch.float32)
            if scale is None:
                cache.copy_(x)
            else:    # calibrated: the largest value of a head is e4m3's largest
                scale.copy_(x.abs().amax(dim=(0, 1, 3)) / 448.0)
                cache.copy_(_quantized(x, scale))
            del x
    return runner, attns, tables


def _quantized(x, scale):
    return (x.float() * (1.0 / scale)[:, None]).clamp_(-448.0, 448.0).to(torch.float8_e4m3fn)


def _norms(case, gen, dtype):
    def one():
        return SimpleNamespace(weight=_randn(gen, case["d"], dtype=dtype, amp=0.1), eps=EPS)
    return one(), one()


def _rotary(rot, positions):
    inv = 1e7 ** -(torch.arange(0, rot, 2, dtype=torch.float64, device=DEVICE) / rot)
    t = torch.arange(positions, dtype=torch.float64, device=DEVICE)[:, None] * inv
    table = torch.cat((t.cos(), t.sin()), dim=-1).float()[:, None, :].contiguous()
    return SimpleNamespace(cos_sin_cache=table, rotary_dim=rot)


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    with torch.inference_mode():
        return _PREPARE[case["kind"]](case, seed, gen)


def _prepare_decode(case, seed, gen):
    lens, _ = _lengths(case)
    dtype = DTYPES[case["dtype"]]
    runner, attns, tables = _pool(case, lens, 1, seed, gen)
    b, hq, hkv, d = case["batch"], case["hq"], case["hkv"], case["d"]
    slots = _slots(tables, [n - 1 for n in lens], [1] * b)
    return dict(case=case, runner=runner, attn=attns[0], q=_randn(gen, b, hq, d, dtype=dtype, amp=1.5),
                k=_randn(gen, b, hkv, d, dtype=dtype), v=_randn(gen, b, hkv, d, dtype=dtype),
                tables=tables.to(DEVICE), lens=torch.tensor(lens, dtype=torch.int32).to(DEVICE),
                slots=slots.to(DEVICE))


class _Step(torch.nn.Module):
    """The attention part of a decoder's layers.  The projections are not this
    framework's; a row of a table stands for the hidden state times them."""

    def __init__(self, case, attns, tables, q_norm, k_norm, rotary):
        super().__init__()
        self.hq, self.hkv, self.d = case["hq"], case["hkv"], case["d"]
        self.attns, self.tables = torch.nn.ModuleList(attns), tables
        self.q_norm, self.k_norm, self.rotary = q_norm, k_norm, rotary

    def forward(self, input_ids, positions):
        hidden = None
        for attn, table in zip(self.attns, self.tables):
            q, gate, k, v = _qgkv(table[input_ids], self.hq, self.hkv, self.d)
            q, k = qk_norm_rope_store(positions, q, k, v, self.q_norm, self.k_norm, self.rotary, attn)
            o = attn(q, k, v, kv_stored=True, gate=gate).reshape(-1, self.hq * self.d)
            hidden = o if hidden is None else hidden + o
        return hidden


def _qgkv(row, hq, hkv, d):
    """q_proj's output holds each head's query, then its gate."""
    q, gate = row[:, :2 * hq * d].view(-1, hq, 2 * d).chunk(2, dim=-1)
    k, v = row[:, 2 * hq * d:].view(-1, 2, hkv, d).unbind(1)
    return q, gate, k, v


def _prepare_graph(case, seed, gen):
    lens, _ = _lengths(case)
    dtype = DTYPES[case["dtype"]]
    runner, attns, tables = _pool(case, lens, case["layers"], seed, gen)
    width = 2 * (case["hq"] + case["hkv"]) * case["d"]
    rows = [_randn(gen, VOCAB, width, dtype=dtype) for _ in attns]
    q_norm, k_norm = _norms(case, gen, dtype)
    step = _Step(case, attns, rows, q_norm, k_norm, _rotary(case["rot"], case["hi"]))
    ids = torch.randint(0, VOCAB, (case["batch"],), generator=gen, device=DEVICE)
    runner.capture_cudagraph(step, case["hq"] * case["d"], case["hi"], dtype=dtype)
    slots = _slots(tables, [n - 1 for n in lens], [1] * len(lens))
    return dict(case=case, runner=runner, step=step, ids=ids,
                positions=torch.tensor([n - 1 for n in lens], device=DEVICE), tables=tables.to(DEVICE),
                lens=torch.tensor(lens, dtype=torch.int32).to(DEVICE), slots=slots.to(DEVICE))


def _prepare_prefill(case, seed, gen):
    new, pre = _lengths(case)
    dtype = DTYPES[case["dtype"]]
    runner, attns, tables = _pool(case, [p + n for p, n in zip(pre, new)], 1, seed, gen)
    t, hq, hkv, d = sum(new), case["hq"], case["hkv"], case["d"]
    state = dict(case=case, runner=runner, attn=attns[0], tables=tables.to(DEVICE) if any(pre) else None,
                 all_tables=tables, slots=_slots(tables, pre, new).to(DEVICE), max_q=max(new),
                 max_k=max(p + n for p, n in zip(pre, new)))
    for name, ls in (("cu_q", new), ("cu_k", [p + n for p, n in zip(pre, new)])):
        state[name] = torch.tensor([0] + ls).cumsum(0).to(torch.int32).to(DEVICE)
    if case["norm"]:
        q, gate, k, v = _qgkv(_randn(gen, t, 2 * (hq + hkv) * d, dtype=dtype), hq, hkv, d)
        q_norm, k_norm = _norms(case, gen, dtype)
        state.update(q=q, gate=gate, k=k.contiguous(), v=v.contiguous(), q_norm=q_norm, k_norm=k_norm,
                     rotary=_rotary(case["rot"], state["max_k"]),
                     positions=torch.cat([torch.arange(p, p + n) for p, n in zip(pre, new)]).to(DEVICE))
    else:
        state.update(q=_randn(gen, t, hq, d, dtype=dtype, amp=1.5), k=_randn(gen, t, hkv, d, dtype=dtype),
                     v=_randn(gen, t, hkv, d, dtype=dtype))
    return state


def _prepare_gdn(case, seed, gen):
    new = _lengths(case)[0] if case["kind"] == "gdn_prefill" else [1] * case["batch"]
    dtype = DTYPES[case["dtype"]]
    t, h, hv, n = sum(new), case["h"], case["hv"], case["batch"]
    channels = (2 * h + hv) * 128
    slots = n + 2
    dt = torch.exp(torch.rand(hv, generator=gen, device=DEVICE) * math.log(100.0) + math.log(1e-3))
    layer = SimpleNamespace(
        num_k_heads=h, num_v_heads=hv, head_k_dim=128, head_v_dim=128,
        conv1d=SimpleNamespace(weight=_randn(gen, channels, 1, 4, dtype=dtype, amp=0.5)),
        A_log=(1.0 + 15.0 * torch.rand(hv, generator=gen, device=DEVICE)).log(),
        dt_bias=dt + torch.log(-torch.expm1(-dt)),    # softplus(dt_bias) = dt, log-uniform in 0.001 .. 0.1
        norm=SimpleNamespace(weight=1.0 + _randn(gen, 128, amp=0.1), eps=EPS),
        conv_states=_randn(gen, slots, channels, 3, dtype=dtype),
        recurrent_states=_randn(gen, slots, hv, 128, 128, amp=0.1))
    where = torch.randperm(slots, generator=torch.Generator().manual_seed(seed))[:n].to(torch.int32)
    cu = None
    if case["kind"] == "gdn_prefill":
        cu = torch.tensor([0] + new).cumsum(0).to(torch.int32).to(DEVICE)
    return dict(case=case, layer=layer, qkv=_randn(gen, t, channels, dtype=dtype),
                z=_randn(gen, t, hv * 128, dtype=dtype), a=_randn(gen, t, hv, dtype=dtype),
                b=_randn(gen, t, hv, dtype=dtype), where=where.to(DEVICE), cu=cu)


_PREPARE = {"decode": _prepare_decode, "graph": _prepare_graph, "prefill": _prepare_prefill,
            "gdn_prefill": _prepare_gdn, "gdn_decode": _prepare_gdn}


# -------------------------------------------------------------------- pass

def _bytes_of(cache):
    return cache.view(torch.uint8) if cache.dtype == torch.float8_e4m3fn else cache


@torch.inference_mode()
def run(state):
    kind = state["case"]["kind"]
    if kind == "decode":
        attn = state["attn"]
        set_context(False, slot_mapping=state["slots"], context_lens=state["lens"], block_tables=state["tables"])
        return attn(state["q"], state["k"], state["v"]), _bytes_of(attn.k_cache), _bytes_of(attn.v_cache)
    if kind == "graph":
        set_context(False, slot_mapping=state["slots"], context_lens=state["lens"], block_tables=state["tables"])
        out = state["runner"].run_model(state["ids"], state["positions"], False)
        return out, _bytes_of(state["runner"].kv_cache)
    if kind == "prefill":
        attn, q, k, v, gate = state["attn"], state["q"], state["k"], state["v"], state.get("gate")
        set_context(True, state["cu_q"], state["cu_k"], state["max_q"], state["max_k"], state["slots"], None,
                    state["tables"])
        if gate is not None:
            q, k = qk_norm_rope_store(state["positions"], q, k, v, state["q_norm"], state["k_norm"],
                                      state["rotary"], attn)
            o = attn(q, k, v, kv_stored=True, gate=gate)
        else:
            o = attn(q, k, v)
        return o, _bytes_of(attn.k_cache), _bytes_of(attn.v_cache)
    layer = state["layer"]
    y = gdn_core(layer, state["qkv"], state["z"], state["a"], state["b"], state["where"], cu_seqlens=state["cu"])
    return y, layer.conv_states, layer.recurrent_states


# -------------------------------------------------------------------- work

def work(case):
    kind, item = case["kind"], 2
    if kind.startswith("gdn"):
        new = _lengths(case)[0] if kind == "gdn_prefill" else [1] * case["batch"]
        t, h, hv, n = sum(new), case["h"], case["hv"], case["batch"]
        channels = (2 * h + hv) * 128
        state = 4 * hv * 128 * 128 + item * 3 * channels
        moved = item * t * (channels + 2 * hv * 128 + 2 * hv) + n * state * (1 if kind == "gdn_prefill" else 2)
        # the recurrence: S k, S += u k^T, S q; and four taps of convolution
        return dict(bytes=moved, flops=t * (hv * 6 * 128 * 128 + 8 * channels))
    new, pre = _lengths(case)
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    kv = 2 * hkv * d * (1 if case["kv"] == "fp8" else item)    # a token's cached key and value
    if kind in ("decode", "graph"):
        b, layers = case["batch"], case.get("layers", 1)
        heads = 2 * hq + 2 * hkv + (hq if kind == "graph" else 0)    # q, o, k, v (and the gate)
        return dict(bytes=layers * (sum(new) * kv + b * (kv + item * heads * d + 8)),
                    flops=layers * 4 * hq * d * sum(new))
    t = sum(new)
    heads = 2 * hq + 2 * hkv + (hq if case["norm"] else 0)
    pairs = sum(n * p + n * (n + 1) // 2 for n, p in zip(new, pre))
    return dict(bytes=t * (item * heads * d + kv + 4) + sum(pre) * kv, flops=4 * hq * d * pairs)


def tolerance(case):
    # About four times what the kernels are off 64-bit results, measured: a 16-bit
    # output of products with 16-bit operands and 32-bit sums; with the q/k norm,
    # the gate or the delta rule before it, a few such roundings in a row.
    plain = case["kind"] in ("decode", "prefill") and not case.get("norm")
    return {"rel": (0.009 if plain else 0.022) / (1 if case["dtype"] == "bf16" else 7)}


# ------------------------------------------------------------ 64-bit result

def _attend(q, k, v, scale):
    """Causal attention of the last rows of a sequence, all in float64:
    q [n, hq, d], k and v [m, hkv, d]."""
    n, hq, d = q.shape
    m, hkv, _ = k.shape
    g = hq // hkv
    kt = k.permute(1, 2, 0).contiguous()
    vt = v.permute(1, 0, 2).contiguous()
    out = torch.empty_like(q)
    step = max(1, (1 << 27) // (hq * m))
    for lo in range(0, n, step):
        rows = q[lo:lo + step]
        r = rows.shape[0]
        s = torch.matmul(rows.view(r, hkv, g, d).permute(1, 0, 2, 3).reshape(hkv, r * g, d), kt).mul_(scale)
        last = torch.arange(m - n + lo, m - n + lo + r, device=DEVICE).repeat_interleave(g)
        s.masked_fill_(torch.arange(m, device=DEVICE)[None, :] > last[:, None], -math.inf)
        o = torch.matmul(torch.softmax(s, dim=-1), vt)
        out[lo:lo + r] = o.view(hkv, r, g, d).permute(1, 0, 2, 3).reshape(r, hq, d)
    return out


def _rows(cache, scale, table, n):
    """The first n cached rows of a sequence, in float64."""
    t = torch.arange(n, device=DEVICE)
    at = table.to(DEVICE).long()[t // BLOCK] * BLOCK + t % BLOCK
    flat = cache.view(-1, *cache.shape[2:])
    if scale is None:
        return flat[at].double()
    return flat.view(torch.uint8)[at].view(torch.float8_e4m3fn).double() * scale.double()[:, None]


def _put(cache, scale, slots, x):
    flat = cache.view(-1, *cache.shape[2:])
    if scale is None:
        flat[slots.long()] = x.to(cache.dtype)
    else:
        flat.view(torch.uint8)[slots.long()] = _quantized(x, scale).view(torch.uint8)


def _norm_rope(x, weight, positions, table, rot):
    x = x.double()
    x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * (1.0 + weight.double())
    c = table.view(-1, rot)[positions].double()[:, None, :]
    cos, sin = c[..., :rot // 2], c[..., rot // 2:]
    a, b = x[..., :rot // 2], x[..., rot // 2:rot]
    return torch.cat((a * cos - b * sin, b * cos + a * sin, x[..., rot:]), dim=-1)


def _cached(cache):
    return None if cache.dtype == torch.float8_e4m3fn else cache.double()


@torch.inference_mode()
def exact(case, seed):
    state = prepare(case, seed)
    return _EXACT[case["kind"]](case, state)


def _exact_decode(case, s):
    attn, lens = s["attn"], s["lens"].tolist()
    _put(attn.k_cache, attn.k_scale, s["slots"], s["k"])
    _put(attn.v_cache, attn.v_scale, s["slots"], s["v"])
    out = [_attend(s["q"][i:i + 1].double(), _rows(attn.k_cache, attn.k_scale, s["tables"][i], n),
                   _rows(attn.v_cache, attn.v_scale, s["tables"][i], n), attn.scale) for i, n in enumerate(lens)]
    return torch.stack(out), _cached(attn.k_cache), _cached(attn.v_cache)


def _exact_graph(case, s):
    step, lens, total = s["step"], s["lens"].tolist(), 0.0
    hq, hkv, d, rot = case["hq"], case["hkv"], case["d"], case["rot"]
    table = step.rotary.cos_sin_cache
    for attn, rows in zip(step.attns, step.tables):
        q, gate, k, v = _qgkv(rows[s["ids"]], hq, hkv, d)
        q = _norm_rope(q, step.q_norm.weight, s["positions"], table, rot)
        k = _norm_rope(k, step.k_norm.weight, s["positions"], table, rot)
        _put(attn.k_cache, attn.k_scale, s["slots"], k.to(DTYPES[case["dtype"]]))
        _put(attn.v_cache, attn.v_scale, s["slots"], v)
        o = torch.cat([_attend(q[i:i + 1], _rows(attn.k_cache, attn.k_scale, s["tables"][i], n),
                               _rows(attn.v_cache, attn.v_scale, s["tables"][i], n), attn.scale)
                       for i, n in enumerate(lens)])
        total = total + (o * torch.sigmoid(gate.double())).reshape(-1, hq * d)
    return total, None


def _exact_prefill(case, s):
    attn, q, k, v = s["attn"], s["q"].double(), s["k"], s["v"]
    if case["norm"]:
        table = s["rotary"].cos_sin_cache
        q = _norm_rope(q, s["q_norm"].weight, s["positions"], table, case["rot"])
        k = _norm_rope(k, s["k_norm"].weight, s["positions"], table, case["rot"]).to(v.dtype)
    _put(attn.k_cache, attn.k_scale, s["slots"], k)
    _put(attn.v_cache, attn.v_scale, s["slots"], v)
    cu_q, cu_k, out = s["cu_q"].tolist(), s["cu_k"].tolist(), []
    for i in range(case["batch"]):
        n = cu_k[i + 1] - cu_k[i]
        out.append(_attend(q[cu_q[i]:cu_q[i + 1]], _rows(attn.k_cache, attn.k_scale, s["all_tables"][i], n),
                           _rows(attn.v_cache, attn.v_scale, s["all_tables"][i], n), attn.scale))
    o = torch.cat(out)
    if case["norm"]:
        o = o * torch.sigmoid(s["gate"].double())
    return o, _cached(attn.k_cache), _cached(attn.v_cache)


def _exact_gdn(case, s):
    """The recurrence, token by token, for all sequences side by side."""
    layer, h, hv = s["layer"], case["h"], case["hv"]
    decode = s["cu"] is None
    n = case["batch"]
    cu = list(range(n + 1)) if decode else s["cu"].tolist()
    where = s["where"].long()
    x = s["qkv"].double()
    channels = x.shape[1]
    w = layer.conv1d.weight.double().view(channels, 4)
    conv, recurrent = layer.conv_states.double(), layer.recurrent_states.double()
    mixed = torch.empty_like(x)
    for i in range(n):
        past = conv[where[i]].t() if decode else torch.zeros(3, channels, dtype=x.dtype, device=DEVICE)
        ext = torch.cat((past, x[cu[i]:cu[i + 1]]))
        m = cu[i + 1] - cu[i]
        mixed[cu[i]:cu[i + 1]] = torch.nn.functional.silu(sum(ext[j:j + m] * w[:, j] for j in range(4)))
        conv[where[i]] = ext[-3:].t()
    t = x.shape[0]
    unit = lambda y: y * torch.rsqrt(y.square().sum(-1, keepdim=True) + 1e-6)    # noqa: E731
    q = unit(mixed[:, :h * 128].view(t, h, 128)).repeat_interleave(hv // h, 1) * 128 ** -0.5
    k = unit(mixed[:, h * 128:2 * h * 128].view(t, h, 128)).repeat_interleave(hv // h, 1)
    v = mixed[:, 2 * h * 128:].view(t, hv, 128)
    step = torch.nn.functional.softplus(s["a"].double() + layer.dt_bias.double())
    decay = torch.exp(-layer.A_log.double().exp() * step)
    beta = torch.sigmoid(s["b"].double())
    S = recurrent[where] if decode else torch.zeros(n, hv, 128, 128, dtype=x.dtype, device=DEVICE)
    y = torch.empty(t, hv, 128, dtype=x.dtype, device=DEVICE)
    starts = torch.tensor(cu[:-1], device=DEVICE)
    lens = [b - a for a, b in zip(cu, cu[1:])]
    order = sorted(range(n), key=lambda i: -lens[i])    # the live ones are always the first
    S, starts, lens = S[order], starts[order], sorted(lens, reverse=True)
    live = n
    for j in range(lens[0]):
        while lens[live - 1] <= j:
            live -= 1
        at, A = starts[:live] + j, S[:live]
        A.mul_(decay[at][:, :, None, None])
        u = beta[at][..., None] * (v[at] - torch.matmul(A, k[at][..., None])[..., 0])
        A.add_(u[..., None] * k[at][:, :, None, :])
        y[at] = torch.matmul(A, q[at][..., None])[..., 0]
    recurrent[where[order]] = S
    y = y * torch.rsqrt(y.square().mean(-1, keepdim=True) + layer.norm.eps) * layer.norm.weight.double()
    y = y * torch.nn.functional.silu(s["z"].double().view(t, hv, 128))
    return y.view(t, hv * 128), conv, recurrent


_EXACT = {"decode": _exact_decode, "graph": _exact_graph, "prefill": _exact_prefill,
          "gdn_prefill": _exact_gdn, "gdn_decode": _exact_gdn}
