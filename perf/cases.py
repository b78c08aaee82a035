"""Performance cases: the calls that a program serving a 24/8-head, 128-wide, 3072-hidden
model makes through this package's public entry points.

Six kinds of call, each over the range of sizes that serving meets:

* ``decode``   one paged-attention call: 1 to 64 sequences, contexts of 64 to 4096 tokens,
               one shared length or a length per row, block sizes 16, 32 and 64;
* ``prefill``  one causal attention call on the model's transposed views: 1 to 8 prompts
               of 16 to 4096 tokens, with or without the write into the paged pool;
* ``linear``   one projection (QKV, output, MLP gate/up and down): 1 to 16384 rows, packed
               INT4 or fp16 weights, with or without the RMSNorm before it;
* ``rope``     rotary embedding and pool write of 1 to 16384 new tokens;
* ``layer``    the attention block of one decode step for 1 to 64 sequences;
* ``step``     the attention blocks of a whole batch-1 decode step, as one HIP graph.

``exact`` computes the same values in 64 bits with plain torch operations.
"""

import math

import torch

import fast_infer_amd as fi

HQ, HKV, D = 24, 8, 128          # query heads, key/value heads, head width
HIDDEN = HQ * D                  # 3072
QKV = (HQ + 2 * HKV) * D         # 5120 columns of the fused QKV projection
MLP = 8192                       # MLP width: gate/up has 2 x 8192 columns
GROUP = 128                      # weights per INT4 scale
MAX_SEQ = 4096
EPS = 1e-5
SHAPES = {"qkv": (QKV, HIDDEN), "o": (HIDDEN, HIDDEN), "gate_up": (2 * MLP, HIDDEN),
          "down": (HIDDEN, MLP)}
DEV = "cuda"
MOST_LINEAR = 16384 * QKV * HIDDEN    # largest rows * columns * depth of a linear case
MOST_PREFILL = 4 * MAX_SEQ * MAX_SEQ  # largest batch * seq^2 of a prefill case


def listed():
    return [
        # interactive chat, one short conversation: launch latency and host time
        {"name": "decode_b1_ctx256", "kind": "decode", "batch": 1, "low": 256, "high": 256,
         "block": 64, "ragged": False},
        # a lightly loaded server with small blocks: odd batch, odd lengths
        {"name": "decode_b7_block16", "kind": "decode", "batch": 7, "low": 100, "high": 3001,
         "block": 16, "ragged": True},
        # a loaded server: the benchmark's headline decode call
        {"name": "decode_b32", "kind": "decode", "batch": 32, "low": 512, "high": 4096,
         "block": 64, "ragged": True},
        # the prompt of a chat turn
        {"name": "prefill_b1_s512", "kind": "prefill", "batch": 1, "seq": 512, "store": True},
        # a few prompts of a length that is no multiple of any tile, pool written elsewhere
        {"name": "prefill_b3_s1111", "kind": "prefill", "batch": 3, "seq": 1111, "store": False},
        # long documents: the benchmark's headline prefill call
        {"name": "prefill_b4_s4096", "kind": "prefill", "batch": 4, "seq": 4096, "store": True},
        # an unquantized projection for a batch of about a hundred sequences
        {"name": "linear_f16_o_m100", "kind": "linear", "rows": 100, "shape": "o",
         "packed": False, "norm": False},
        # the MLP's down projection of a 509-token prompt
        {"name": "linear_down_m509", "kind": "linear", "rows": 509, "shape": "down",
         "packed": True, "norm": False},
        # the QKV projection of four 4096-token prompts
        {"name": "linear_qkv_m16384", "kind": "linear", "rows": 16384, "shape": "qkv",
         "packed": True, "norm": False},
        # rotary embedding and pool write of the same prompts
        {"name": "rope_b4_t4096", "kind": "rope", "batch": 4, "tokens": 4096, "block": 64,
         "keep_k": True},
        # the attention block of a loaded server's decode step
        {"name": "layer_b64", "kind": "layer", "batch": 64, "low": 200, "high": 2300,
         "block": 64},
        # a single-stream decode step through 28 layers, replayed as one graph
        {"name": "step_b1_28layers", "kind": "step", "layers": 28, "context": 1024},
    ]


def _log(rng, low, high):
    """An integer from low to high, spread evenly over its logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    kind = rng.choice(["decode", "prefill", "linear", "linear", "rope", "layer"])
    if kind == "decode":
        ragged = rng.random() < 0.7
        high = _log(rng, 64, MAX_SEQ)
        low = _log(rng, min(64, high), high) if ragged else high
        return {"kind": kind, "batch": _log(rng, 1, 64), "low": low, "high": high,
                "block": rng.choice([16, 32, 64, 64]), "ragged": ragged}
    if kind == "prefill":
        seq = _log(rng, 16, MAX_SEQ)
        batch = _log(rng, 1, 8)
        while batch * seq * seq > MOST_PREFILL:
            batch -= 1
        return {"kind": kind, "batch": batch, "seq": seq, "store": rng.random() < 0.5}
    if kind == "linear":
        shape = rng.choice(sorted(SHAPES))
        n, k = SHAPES[shape]
        return {"kind": kind, "rows": _log(rng, 1, min(16384, MOST_LINEAR // (n * k))),
                "shape": shape, "packed": rng.random() < 0.75,
                "norm": k == HIDDEN and rng.random() < 0.4}
    if kind == "rope":
        tokens = _log(rng, 1, MAX_SEQ)
        return {"kind": kind, "batch": _log(rng, 1, min(64, 16384 // tokens)),
                "tokens": tokens, "block": rng.choice([16, 32, 64, 64]),
                "keep_k": rng.random() < 0.5}
    high = _log(rng, 64, 2300)
    return {"kind": kind, "batch": _log(rng, 1, 64), "low": _log(rng, min(64, high), high),
            "high": high, "block": rng.choice([16, 32, 64, 64])}


# -- inputs ------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, device=DEV, generator=g, dtype=torch.float16)


def _lengths(case):
    """Context lengths of a decode, layer or step case: a property of the case, so that its
    work is the same for every seed."""
    if case["kind"] == "step":
        return [case["context"]]
    low, high, batch = case["low"], case["high"], case["batch"]
    if low == high:
        return [high] * batch
    r = torch.Generator().manual_seed(1000003 * batch + 1009 * high + low)
    return torch.randint(low, high + 1, (batch,), generator=r).tolist()


def _paged(g, lengths, block):
    """A block table (shuffled pool blocks, -1 past each row's own) and the pool's size."""
    counts = [-(-n // block) for n in lengths]
    total = sum(counts)
    perm = torch.randperm(total, device=DEV, generator=g).int()
    table = torch.full((len(lengths), max(counts)), -1, dtype=torch.int32, device=DEV)
    at = 0
    for b, n in enumerate(counts):
        table[b, :n] = perm[at:at + n]
        at += n
    return table, total


def _weight(g, n, k, packed):
    """fp16 weights of deviation 0.02, or INT4 values with a scale per 128 of them."""
    if not packed:
        return _randn(g, n, k) * 0.02
    q = (_randn(g, n, k) * 2.5).round_().clamp_(-8, 7).to(torch.int8)
    bytes_ = (q[:, 0::2] & 15) | (q[:, 1::2] << 4)
    scales = torch.empty(n, k // GROUP, device=DEV, dtype=torch.float16)
    return bytes_, scales.uniform_(0.006, 0.01, generator=g)


def _tables():
    cos, sin = fi.precompute_freqs(D, MAX_SEQ, device=DEV)
    return cos.half(), sin.half()


def _attention_state(g, case, lengths):
    block = case.get("block", 64)
    table, blocks = _paged(g, lengths, block)
    return {"table": table, "block": block, "max": max(lengths), "lengths": lengths,
            "kc": _randn(g, blocks, block, HKV, D), "vc": _randn(g, blocks, block, HKV, D)}


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "decode":
        lengths = _lengths(case)
        s = _attention_state(g, case, lengths)
        s["q"] = _randn(g, case["batch"], HQ, D)
        s["ctx"] = (torch.tensor(lengths, dtype=torch.int32, device=DEV)
                    if case["ragged"] else None)
        s["ws"] = fi.paged_attention_workspace(case["batch"], HQ, HKV, s["max"], D, DEV)
    elif kind == "prefill":
        b, t = case["batch"], case["seq"]
        s = {"q": _randn(g, b, t, HQ, D).transpose(1, 2),
             "k": _randn(g, b, t, HKV, D).transpose(1, 2),
             "v": _randn(g, b, t, HKV, D).transpose(1, 2), "store": case["store"]}
        if case["store"]:
            s["table"], blocks = _paged(g, [t] * b, 64)
            s["kc"] = torch.zeros(blocks, 64, HKV, D, device=DEV, dtype=torch.float16)
            s["vc"] = torch.zeros_like(s["kc"])
    elif kind == "linear":
        n, k = SHAPES[case["shape"]]
        s = {"x": _randn(g, case["rows"], k), "w": _weight(g, n, k, case["packed"]),
             "norm": (1 + 0.1 * _randn(g, k)) if case["norm"] else None}
    elif kind == "rope":
        b, t = case["batch"], case["tokens"]
        table, blocks = _paged(g, [t] * b, case["block"])
        qkv = _randn(g, b, t, QKV)
        q, k, v = qkv.split([HQ * D, HKV * D, HKV * D], dim=-1)
        s = {"q": q.unflatten(-1, (HQ, D)), "k": k.unflatten(-1, (HKV, D)),
             "v": v.unflatten(-1, (HKV, D)), "table": table, "keep_k": case["keep_k"],
             "kc": torch.zeros(blocks, case["block"], HKV, D, device=DEV, dtype=torch.float16)}
        s["vc"] = torch.zeros_like(s["kc"])
        s["cos"], s["sin"] = _tables()
    elif kind == "layer":
        lengths = _lengths(case)
        s = _attention_state(g, case, lengths)
        s.update(_layer_weights(g))
        s["x"] = _randn(g, case["batch"], HIDDEN)
        s["ctx"] = torch.tensor(lengths, dtype=torch.int32, device=DEV)
        s["pos"] = s["ctx"] - 1
        s["ws"] = fi.paged_attention_workspace(case["batch"], HQ, HKV, s["max"], D, DEV)
        s["cos"], s["sin"] = _tables()
    else:
        s = _step_state(g, case)
    s["kind"] = kind
    return s


def _layer_weights(g):
    return {"norm": 1 + 0.1 * _randn(g, HIDDEN), "w_qkv": _weight(g, QKV, HIDDEN, True),
            "w_o": _weight(g, HIDDEN, HIDDEN, True)}


def _step_state(g, case):
    """Weights and pools of every layer, and the step captured into a graph after one eager
    step, as a latency-bound server keeps it."""
    first = _attention_state(g, case, _lengths(case))
    layers = [first]
    for _ in range(case["layers"] - 1):
        layers.append(dict(first, kc=_randn(g, *first["kc"].shape),
                           vc=_randn(g, *first["vc"].shape)))
    for layer in layers:
        layer.update(_layer_weights(g))
    s = {"layers": layers, "x": _randn(g, 1, HIDDEN)}
    s["ctx"] = torch.tensor([case["context"]], dtype=torch.int32, device=DEV)
    s["pos"] = s["ctx"] - 1
    s["ws"] = fi.paged_attention_workspace(1, HQ, HKV, case["context"], D, DEV)
    s["cos"], s["sin"] = _tables()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _step(s)
    torch.cuda.current_stream().wait_stream(side)
    s["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(s["graph"]):
        s["h"] = _step(s)
    return s


# -- the calls ---------------------------------------------------------------------------

def _block(x, layer, s):
    """The attention block of one decode step: norm and QKV projection, rotary embedding
    and pool write, paged attention, output projection."""
    batch = x.shape[0]
    qkv = fi.rms_norm_int4_matmul(x, layer["norm"], layer["w_qkv"], EPS)
    q, k, v = qkv.split([HQ * D, HKV * D, HKV * D], dim=-1)
    q, _ = fi.rope_store_kv(q.view(batch, 1, HQ, D), k.view(batch, 1, HKV, D),
                            v.view(batch, 1, HKV, D), s["cos"], s["sin"], 0, layer["kc"],
                            layer["vc"], layer["table"], start_positions=s["pos"],
                            return_k=False)
    o = fi.paged_attention(q[:, 0], layer["kc"], layer["vc"], layer["table"], layer["block"],
                           layer["max"], context_lens=s["ctx"], workspace=s["ws"])
    return fi.int4_matmul(o.view(batch, HIDDEN), layer["w_o"])


def _step(s):
    h = s["x"]
    for layer in s["layers"]:
        h = h + _block(h, layer, s)
    return h


def run(s):
    kind = s["kind"]
    if kind == "decode":
        return fi.paged_attention(s["q"], s["kc"], s["vc"], s["table"], s["block"], s["max"],
                                  context_lens=s["ctx"], workspace=s["ws"])
    if kind == "prefill":
        if not s["store"]:
            return fi.flash_attention(s["q"], s["k"], s["v"])
        o = fi.flash_attention(s["q"], s["k"], s["v"], k_cache=s["kc"], v_cache=s["vc"],
                               block_table=s["table"])
        return o, s["kc"], s["vc"]
    if kind == "linear":
        if s["norm"] is not None:
            return fi.rms_norm_int4_matmul(s["x"], s["norm"], s["w"], EPS)
        return fi.int4_matmul(s["x"], s["w"])
    if kind == "rope":
        q, k = fi.rope_store_kv(s["q"], s["k"], s["v"], s["cos"], s["sin"], 0, s["kc"],
                                s["vc"], s["table"], return_k=s["keep_k"])
        return q, k, s["kc"], s["vc"]
    if kind == "layer":
        return _block(s["x"], s, s), s["kc"], s["vc"]
    s["graph"].replay()
    return s["h"], [layer["kc"] for layer in s["layers"]]


# -- what a pass cannot do without ---------------------------------------------------------

def _attention_work(lengths, block):
    batch, tokens = len(lengths), sum(lengths)
    return (tokens * 2 * HKV * D * 2 + 2 * batch * HQ * D * 2
            + 4 * sum(-(-n // block) for n in lengths), 4 * tokens * HQ * D)


def _linear_work(m, n, k, packed):
    weight = n * k // 2 + n * (k // GROUP) * 2 if packed else n * k * 2
    return m * k * 2 + weight + m * n * 2, 2 * m * n * k


def _rope_work(batch, tokens, positions, keep_k):
    heads = 2 * HQ + (4 + (1 if keep_k else 0)) * HKV  # q, k and v read; q, pool and k written
    return batch * tokens * heads * D * 2 + positions * 2 * D * 2


def work(case):
    kind = case["kind"]
    if kind == "decode":
        nbytes, flops = _attention_work(_lengths(case), case["block"])
    elif kind == "prefill":
        b, t = case["batch"], case["seq"]
        nbytes = b * t * (2 * HQ + (4 if case["store"] else 2) * HKV) * D * 2
        flops = 4 * b * HQ * D * t * (t + 1) // 2
    elif kind == "linear":
        n, k = SHAPES[case["shape"]]
        nbytes, flops = _linear_work(case["rows"], n, k, case["packed"])
    elif kind == "rope":
        nbytes = _rope_work(case["batch"], case["tokens"], case["tokens"], case["keep_k"])
        flops = 0
    else:
        lengths = _lengths(case)
        batch = len(lengths)
        parts = [_attention_work(lengths, case.get("block", 64)),
                 _linear_work(batch, QKV, HIDDEN, True),
                 _linear_work(batch, HIDDEN, HIDDEN, True),
                 (_rope_work(batch, 1, batch, False), 0)]
        layers = case.get("layers", 1)
        nbytes = layers * sum(p[0] for p in parts)
        flops = layers * sum(p[1] for p in parts)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Relative errors of fp16 results, four times what was measured against ``exact``: 2.1e-4
    for a projection and 2.6e-4 for attention (the output rounded once, and attention's
    probabilities), 5.7e-4 for four chained calls, 1.2e-3 for 28 layers of them."""
    kind = case["kind"]
    if kind == "rope":
        return "exact"  # every implementation rounds at the same three points
    return {"rel": {"linear": 1e-3, "decode": 1e-3, "prefill": 1e-3, "layer": 2.4e-3,
                    "step": 5e-3}[kind]}


# -- the same values in 64 bits --------------------------------------------------------------

def _exact_weight(w):
    if not isinstance(w, tuple):
        return w.double()
    b, scales = w
    n, half = b.shape
    low, high = (b << 4) >> 4, b >> 4  # sign-extended nibbles
    q = torch.stack([low, high], dim=-1).view(n, 2 * half)
    # the weight that both forms stand for is fp16(q * scale)
    scaled = q.view(n, -1, GROUP).float() * scales.float().unsqueeze(-1)
    return scaled.half().double().view(n, 2 * half)


def _exact_norm(x, weight):
    x = x.double()
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * weight.double()


def _exact_rope(x, cos, sin):
    """x [rows, heads, D] at table rows cos, sin [rows, D]."""
    x = x.double()
    turned = torch.cat([-x[..., D // 2:], x[..., :D // 2]], dim=-1)
    return x * cos.double().unsqueeze(1) + turned * sin.double().unsqueeze(1)


def _exact_decode(q, kc, vc, table, block, lengths):
    out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
    for b, n in enumerate(lengths):
        blocks = table[b, :-(-n // block)].long()
        k = kc[blocks].flatten(0, 1)[:n].double().permute(1, 2, 0).contiguous()
        v = vc[blocks].flatten(0, 1)[:n].double().transpose(0, 1).contiguous()
        s = torch.matmul(q[b].double().view(HKV, HQ // HKV, D), k) * D ** -0.5
        out[b] = torch.matmul(s.softmax(-1), v).view(HQ, D)
    return out


def _exact_pool(pool, table, rows):
    """`pool` with rows [batch, tokens, HKV, D] at positions 0, 1, ... of each table row."""
    out = pool.clone()
    batch, tokens = rows.shape[:2]
    t = torch.arange(tokens, device=DEV)
    slots = table[:batch].long()[:, t // pool.shape[1]] * pool.shape[1] + t % pool.shape[1]
    out.view(-1, HKV, D)[slots.view(-1)] = rows.reshape(-1, HKV, D).to(out.dtype)
    return out


def _exact_prefill(q, k, v):
    batch, heads, seq, _ = q.shape
    out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
    mask = torch.ones(seq, seq, dtype=torch.bool, device=DEV).triu_(1)
    for b in range(batch):
        for h in range(heads):
            kv = h // (heads // k.shape[1])
            s = q[b, h].double() @ k[b, kv].double().t().contiguous() * D ** -0.5
            out[b, h] = s.masked_fill_(mask, -math.inf).softmax(-1) @ v[b, kv].double()
    return out


def _exact_block(x, layer, pos, lengths, cos, sin):
    """The attention block's output and its pools with this step's rows, in 64 bits."""
    batch = x.shape[0]
    qkv = _exact_norm(x, layer["norm"]) @ _exact_weight(layer["w_qkv"]).t()
    q, k, v = qkv.split([HQ * D, HKV * D, HKV * D], dim=-1)
    cos, sin = cos[pos.long()], sin[pos.long()]
    q = _exact_rope(q.view(batch, HQ, D), cos, sin)
    k = _exact_rope(k.view(batch, HKV, D), cos, sin)
    kc, vc, block = layer["kc"].double(), layer["vc"].double(), layer["block"]
    at = layer["table"][torch.arange(batch, device=DEV), pos.long() // block].long()
    kc[at, pos.long() % block] = k
    vc[at, pos.long() % block] = v.reshape(batch, HKV, D)
    o = _exact_decode(q, kc, vc, layer["table"], block, lengths)
    return o.view(batch, HIDDEN) @ _exact_weight(layer["w_o"]).t(), kc, vc


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "decode":
        return _exact_decode(s["q"], s["kc"], s["vc"], s["table"], s["block"], s["lengths"])
    if kind == "prefill":
        o = _exact_prefill(s["q"], s["k"], s["v"])
        if not s["store"]:
            return o
        return (o, _exact_pool(s["kc"].double(), s["table"], s["k"].transpose(1, 2)),
                _exact_pool(s["vc"].double(), s["table"], s["v"].transpose(1, 2)))
    if kind == "linear":
        x = s["x"].double() if s["norm"] is None else _exact_norm(s["x"], s["norm"])
        return x @ _exact_weight(s["w"]).t()
    if kind == "rope":
        b, t = case["batch"], case["tokens"]
        cos, sin = s["cos"][:t].repeat(b, 1), s["sin"][:t].repeat(b, 1)
        q = _exact_rope(s["q"].flatten(0, 1), cos, sin).view(b, t, HQ, D)
        k = _exact_rope(s["k"].flatten(0, 1), cos, sin).view(b, t, HKV, D)
        return (q, k if case["keep_k"] else None,
                _exact_pool(s["kc"].double(), s["table"], k),
                _exact_pool(s["vc"].double(), s["table"], s["v"]))
    if kind == "layer":
        return _exact_block(s["x"], s, s["pos"], s["lengths"], s["cos"], s["sin"])
    h, pools = s["x"].double(), []
    for layer in s["layers"]:
        o, kc, _ = _exact_block(h, layer, s["pos"], layer["lengths"], s["cos"], s["sin"])
        h = h + o
        pools.append(kc)
    return h, pools
