"""The serving engine's forward steps: what a request costs on the GPU.

A pass is one `DecoderModel.forward` on a paged K/V cache, as the engine calls it: a decode step of a
batch of sequences, replayed from a captured graph (the engine captures one per batch size), or a chunk
of prompt tokens, run eagerly.  The models have the layer shapes, formats and vocabularies of the
configurations that the repository serves and benchmarks (Llama-3-8B Q4_K_M and Q8_0, Mixtral-8x7B
Q4_K_M), on 8 and 4 layers, with random weights: every layer costs the same, and 8 layers (4 with
experts) are several times what the caches hold.
"""
import math
import zlib
from types import SimpleNamespace

import numpy as np
import torch

from localai_amd.models.decoder import DecoderModel, ForwardBatch

DEV = "cuda"
BLOCK = 32                  # tokens of a K/V page: the engine's default
F32, Q8_0, Q4_K, Q6_K = 0, 8, 12, 14
BLOCK_VALUES = {F32: 1, Q8_0: 32, Q4_K: 256, Q6_K: 256}
BLOCK_BYTES = {F32: 4, Q8_0: 34, Q4_K: 144, Q6_K: 210}

_DENSE = dict(layers=8, width=4096, heads=32, kv_heads=8, ffn=14336, vocab=128256, theta=500000.0, experts=0)
MODELS = {
    "llama3-8b-q4": dict(_DENSE, mix="Q4_K_M"),
    "llama3-8b-q8": dict(_DENSE, mix="Q8_0"),
    "mixtral-q4": dict(_DENSE, mix="Q4_K_M", layers=4, vocab=32000, theta=1e6, experts=8),
}
EXPERTS_USED = 2
EPS = 1e-5


# ------------------------------------------------------------------------------------------ cases

def _decode(model, batch, keys):
    """One token for each of `batch` sequences that hold about `keys` tokens each."""
    return {"model": model, "step": "decode", "batch": batch, "keys": keys}


def _prefill(model, prompts, rows, keys=0):
    """`rows` prompt tokens of `prompts` requests together, after `keys` cached tokens of each."""
    return {"model": model, "step": "prefill", "batch": prompts, "rows": rows, "keys": keys}


def listed():
    q4, q8, moe = "llama3-8b-q4", "llama3-8b-q8", "mixtral-q4"
    return [
        # a single user's chat: every token of an answer
        dict(_decode(q4, 1, 700), name="decode-1"),
        # a handful of users on the larger 8-bit files
        dict(_decode(q8, 4, 1500), name="decode-4-q8"),
        # a few users who each have a long document in their prompt
        dict(_decode(q4, 7, 8000), name="decode-7-long"),
        # a small team's server
        dict(_decode(q4, 19, 900), name="decode-19"),
        # a busy server, between two of the benchmark's concurrencies
        dict(_decode(q4, 50, 640), name="decode-50"),
        # the benchmark's batch: 256 streams, 128 prompt and up to 256 generated tokens
        dict(_decode(q4, 256, 256), name="decode-256"),
        # a sparse mixture of experts serving a small team
        dict(_decode(moe, 24, 500), name="decode-24-experts"),
        # a short question: the time to its first token
        dict(_prefill(q4, 1, 45), name="prefill-45"),
        # one prompt with a page of text
        dict(_prefill(q4, 1, 701), name="prefill-701"),
        # a chunk of a long document, behind what is cached of it
        dict(_prefill(q4, 1, 2048, 10007), name="prefill-2048-long"),
        # a burst of short prompts in one full chunk: the benchmark's arrivals
        dict(_prefill(q4, 64, 8192), name="prefill-8192"),
        # several prompts on the mixture of experts
        dict(_prefill(moe, 5, 1203), name="prefill-1203-experts"),
    ]


def _log_between(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    model = rng.choice(["llama3-8b-q4", "llama3-8b-q4", "llama3-8b-q4", "llama3-8b-q8", "mixtral-q4"])
    if rng.random() < 0.6:
        batch = _log_between(rng, 1, 256)
        return _decode(model, batch, _log_between(rng, 64, min(12000, 90000 // batch)))
    # (a chunk of prompts on the mixture of experts is held to what keeps it below the largest listed case)
    rows = _log_between(rng, 16, 3000 if model == "mixtral-q4" else 8000)
    prompts = min(_log_between(rng, 1, 64), max(1, rows // 8))
    keys = _log_between(rng, 32, 12000) if prompts == 1 and rows <= 2048 and rng.random() < 0.5 else 0
    return _prefill(model, prompts, rows, keys)


# ---------------------------------------------------------------------------------------- weights

def _tensors(m):
    """(name, shape, format) of every tensor of a model's file."""
    d, f, kv = m["width"], m["ffn"], m["width"] // m["heads"] * m["kv_heads"]
    L, mixed = m["layers"], m["mix"] == "Q4_K_M"
    low = Q4_K if mixed else Q8_0
    out = [("token_embd.weight", (m["vocab"], d), low)]
    for i in range(L):
        # the mix's rule: attn_v and ffn_down of the first and last eighth and of every third layer between in Q6_K
        more = Q6_K if mixed and (i < L // 8 or i >= 7 * L // 8 or (i - L // 8) % 3 == 2) else low
        b = "blk.%d." % i
        out += [(b + "attn_norm.weight", (d,), F32), (b + "attn_q.weight", (d, d), low), (b + "attn_k.weight", (kv, d), low),
                (b + "attn_v.weight", (kv, d), more), (b + "attn_output.weight", (d, d), low),
                (b + "ffn_norm.weight", (d,), F32)]
        if m["experts"]:
            E = m["experts"]
            out += [(b + "ffn_gate_inp.weight", (E, d), F32), (b + "ffn_gate_exps.weight", (E, f, d), low),
                    (b + "ffn_up_exps.weight", (E, f, d), low), (b + "ffn_down_exps.weight", (E, d, f), more)]
        else:
            out += [(b + "ffn_gate.weight", (f, d), low), (b + "ffn_up.weight", (f, d), low),
                    (b + "ffn_down.weight", (d, f), more)]
    out += [("output_norm.weight", (d,), F32), ("output.weight", (m["vocab"], d), Q6_K if mixed else Q8_0)]
    return out


def _half(x):
    return x.to(torch.float16).view(torch.uint8).view(-1, 2)


def _raw(model, name, shape, fmt):
    """The bytes of a tensor in its file format (uint8, on the GPU).  The embedding has a standard deviation of
    1, matrices of 0.02, those that write to the residual stream of 0.005 (0.002 with experts), so that a layer
    changes the stream by a part of it, as in trained models; scales vary from block to block."""
    g = torch.Generator(device=DEV).manual_seed(zlib.crc32((model + name).encode()))
    n = math.prod(shape)
    if fmt == F32:
        if name.endswith("norm.weight"):
            v = 1.0 + 0.1 * torch.randn(n, generator=g, device=DEV)
            v[::257] *= 3.0     # a few channels stand out, as in trained models
        else:
            # the routers: the same eight directions, for other experts in each layer (see _vocabulary)
            g.manual_seed(zlib.crc32(model.encode()))
            v = 0.06 * torch.randn(shape, generator=g, device=DEV).roll(int(name.split(".")[1]), 0).flatten()
        return v.view(torch.uint8)
    sd = 0.02
    if name == "token_embd.weight":
        sd = 1.0
    elif "attn_output" in name or "ffn_down" in name:
        sd = 0.002 if MODELS[model]["experts"] else 0.005
    nb = n // BLOCK_VALUES[fmt]
    size = BLOCK_BYTES[fmt]
    raw = torch.randint(0, 256, (nb, size), generator=g, device=DEV, dtype=torch.uint8)
    vary = 0.75 + 0.5 * torch.rand(nb, generator=g, device=DEV)
    if fmt == Q8_0:
        raw[:, :2] = _half(vary * (sd / 73.9))
        return raw.view(-1)
    if fmt == Q6_K:
        sc = torch.randint(32, 128, (nb, 16), generator=g, device=DEV)
        sc = torch.where(torch.rand(nb, 16, generator=g, device=DEV) < 0.5, sc, -sc)
        raw[:, 192:208] = sc.to(torch.int8).view(torch.uint8)
        raw[:, 208:] = _half(vary * (sd / (85.0 * 18.5)))
        return raw.view(-1)
    d = vary * (sd / (47.5 * 4.61))
    sc = torch.randint(32, 64, (nb, 8), generator=g, device=DEV)
    mn = (sc.float() * (7.5 / 8.0)).round().long()
    raw[:, 0:2], raw[:, 2:4] = _half(d), _half(d * 8.0)
    raw[:, 4:8] = (sc[:, :4] | ((sc[:, 4:] >> 4) << 6)).to(torch.uint8)
    raw[:, 8:12] = (mn[:, :4] | ((mn[:, 4:] >> 4) << 6)).to(torch.uint8)
    raw[:, 12:16] = ((sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)).to(torch.uint8)
    return raw.view(-1)


_LOADED = {}


def _model(name):
    """The model, loaded once for all requests as a server does.  The reader has what the loaders ask of
    a checkpoint's reader: architecture, metadata and tensors by name."""
    if name not in _LOADED:
        m = MODELS[name]
        kv = {"llama.context_length": 16384, "llama.embedding_length": m["width"], "llama.block_count": m["layers"],
              "llama.feed_forward_length": m["ffn"], "llama.attention.head_count": m["heads"],
              "llama.attention.head_count_kv": m["kv_heads"], "llama.rope.freq_base": m["theta"],
              "llama.rope.dimension_count": m["width"] // m["heads"], "llama.attention.layer_norm_rms_epsilon": EPS,
              "llama.vocab_size": m["vocab"]}
        if m["experts"]:
            kv.update({"llama.expert_count": m["experts"], "llama.expert_used_count": EXPERTS_USED})
        tensors = {n: SimpleNamespace(name=n, shape=s, ggml_type=t, data=_raw(name, n, s, t).cpu().numpy())
                   for n, s, t in _tensors(m)}
        reader = SimpleNamespace(architecture="llama", kv=kv, tensors=tensors)
        _LOADED[name] = DecoderModel(reader, torch.device(DEV), max_pos=16384)
    return _LOADED[name]


# ----------------------------------------------------------------------------------------- inputs

def _requests(case, seed):
    """Cached tokens and new tokens of every sequence, as two lists: ragged around the case's mean, and in
    another order for another seed, so that a case always needs as many pages."""
    B = case["batch"]
    share = np.random.default_rng([B, case["keys"]]).uniform(0.6, 1.4, B)
    share = share[np.random.default_rng([seed, 7]).permutation(B)]
    if case["step"] == "decode":
        return [max(1, int(round(case["keys"] * s))) if B > 1 else case["keys"] for s in share], [1] * B
    size = np.maximum(1, np.floor(share / share.sum() * case["rows"]).astype(int))
    size[np.argmax(share)] += case["rows"] - size.sum()
    return [case["keys"]] * B, [int(n) for n in size]


_CLEAR = {}


def _vocabulary(name):
    """The tokens that prompts are made of: all, or with experts those of which the second and third best experts
    are well apart.  A trained router is decided; of random ones some token's choice hangs on the last bit of a sum."""
    m = MODELS[name]
    if name not in _CLEAR:
        if not m["experts"]:
            _CLEAR[name] = np.arange(m["vocab"])
        else:
            spec = {n: (s, t) for n, s, t in _tensors(m)}
            x, r = (_weight(name, n, *spec[n]) for n in ("token_embd.weight", "blk.0.ffn_gate_inp.weight"))
            top = torch.topk((x * torch.rsqrt(x.square().mean(-1, keepdim=True))) @ r.t(), EXPERTS_USED + 1, -1)[0]
            margin = top[:, -2] - top[:, -1]
            _CLEAR[name] = torch.topk(margin, m["vocab"] // 16)[1].sort()[0].cpu().numpy()
    return _CLEAR[name]


def _layout(case, seed):
    """(cached, new, tokens, block table, pages in all) of a pass, on the host."""
    old, new = _requests(case, seed)
    rng = np.random.default_rng([seed, 8])
    pages = [-(-(o + n) // BLOCK) for o, n in zip(old, new)]
    order = rng.permutation(sum(pages)).astype(np.int32)
    bt = np.zeros((len(old), max(pages)), np.int32)
    at = 0
    for s, p in enumerate(pages):
        bt[s, :p] = order[at:at + p]
        at += p
    vocabulary = _vocabulary(case["model"])
    tokens = vocabulary[rng.integers(0, len(vocabulary), sum(new))].astype(np.int32)
    return old, new, tokens, bt, at


def _fill(case, seed, layer, k, v):
    """What earlier steps left in a layer's pages: rows as these weights give them."""
    g = torch.Generator(device=DEV).manual_seed(seed * 1009 + layer)
    k.normal_(0.0, 1.3, generator=g)
    v.normal_(0.0, 1.3, generator=g)


def prepare(case, seed):
    model, m = _model(case["model"]), MODELS[case["model"]]
    old, new, tokens, bt, pages = _layout(case, seed)
    decode = case["step"] == "decode"
    kv = model.new_kv_cache(pages, BLOCK)
    if max(old):
        for i in range(m["layers"]):
            _fill(case, seed, i, kv.k[i], kv.v[i])
    pos = np.concatenate([np.arange(o, o + n) for o, n in zip(old, new)]).astype(np.int32)
    seq = np.repeat(np.arange(len(old)), new)
    slots = bt[seq, pos // BLOCK] * BLOCK + pos % BLOCK

    def dev(a, dtype=np.int32):
        return torch.from_numpy(np.ascontiguousarray(a, dtype)).to(DEV)

    fb = ForwardBatch(tokens=dev(tokens), pos=dev(pos), slots=dev(slots), decode=decode, block_tables=dev(bt))
    ends = np.cumsum(new)
    state = {"model": model, "kv": kv, "batch": fb}
    if not decode:
        fb.cu_q = dev(np.concatenate([[0], ends]))
        fb.ctx_lens = dev(np.array(old) + np.array(new))
        fb.logits_idx = dev(ends - 1, np.int64)     # the last token of every prompt is the one sampled from
        fb.tiles, fb.tile_rows = model.prefill_tiles(new, torch.device(DEV))
        return state
    fb.seq_lens = dev(np.array(old) + 1)
    fb.max_len = 4096 if max(old) < 4096 else 16384     # the served context, not this batch's longest
    ws = model.decode_workspace(len(old), fb.max_len, BLOCK)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            model.forward(fb, kv, attn_workspace=ws)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        state["logits"] = model.forward(fb, kv, attn_workspace=ws)
    state.update(graph=graph, workspace=ws)
    return state


def run(state):
    """The logits that the next tokens are sampled from, and the K/V cache with the new rows."""
    if "graph" in state:
        state["graph"].replay()
        logits = state["logits"]
    else:
        logits = state["model"].forward(state["batch"], state["kv"])
    return {"logits": logits, "k": state["kv"].k, "v": state["kv"].v}


# ----------------------------------------------------------------------------- what a pass has to do

def work(case):
    m = MODELS[case["model"]]
    old, new = _requests(case, 0)
    T, B = sum(new), len(old)
    d, dh, E = m["width"], m["width"] // m["heads"], m["experts"]
    nbytes = flops = 0.0
    for name, shape, fmt in _tensors(m):
        size = math.prod(shape) / BLOCK_VALUES[fmt] * BLOCK_BYTES[fmt]
        if name == "token_embd.weight":
            nbytes += T * size / m["vocab"]
        elif "_exps." in name:      # the experts that some token is routed to; every token has two
            nbytes += size * (1.0 - (1.0 - EXPERTS_USED / E) ** T)
            flops += 2.0 * math.prod(shape) / E * EXPERTS_USED * T
        else:
            nbytes += size
            if len(shape) == 2:
                flops += 2.0 * math.prod(shape) * (B if name == "output.weight" else T)
    row = 2.0 * m["kv_heads"] * dh * 2      # the K and V of a token in a layer, in bf16
    keys = sum(old)
    pairs = sum(n * o + n * (n + 1) / 2 for o, n in zip(old, new))
    nbytes += m["layers"] * row * (keys + T) + 4.0 * B * m["vocab"]
    flops += m["layers"] * 4.0 * d * pairs
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # bf16 operands in 8 layers of 4 products after each other: logits measured 0.7 to 1.0 % off exact(); one or two
    # rows quantise their activations to 8 bits: 1.9 %
    return {"rel": 0.03, "max": 0.3}


# ------------------------------------------------------------------------ the same, in 64 bits

def _weight(model, name, shape, fmt):
    """A tensor of a model's file in float64, from the definition of its format."""
    raw = _raw(model, name, shape, fmt)
    if fmt == F32:
        return raw.view(torch.float32).double().view(shape)
    b = raw.view(-1, BLOCK_BYTES[fmt])

    def half(x):
        return x.contiguous().view(torch.float16).double()

    if fmt == Q8_0:
        w = half(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).double()
    elif fmt == Q4_K:
        s = b[:, 4:16]
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        q = b[:, 16:].view(-1, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).view(-1, 8, 32).double()
        w = (half(b[:, :2]) * sc)[:, :, None] * q - (half(b[:, 2:4]) * mn)[:, :, None]
    else:
        lo, hi = b[:, :128].view(-1, 2, 2, 32), b[:, 128:192].view(-1, 2, 1, 32)
        q = torch.cat([lo & 15, lo >> 4], 2)                                     # [blocks, half, quarter, 32]
        top = torch.cat([(hi >> (2 * i)) & 3 for i in range(4)], 2)
        q = (q | (top << 4)).double() - 32.0
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        w = (half(b[:, 208:]) * sc)[:, :, None] * q.reshape(-1, 16, 16)
    return w.reshape(shape)


def exact(case, seed):
    name, m = case["model"], MODELS[case["model"]]
    spec = {n: (s, t) for n, s, t in _tensors(m)}

    def w(n):
        return _weight(name, n, *spec[n])

    def norm(x, n):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w(n)

    old, new, tokens, bt, pages = _layout(case, seed)
    H, G, dh = m["heads"], m["kv_heads"], m["width"] // m["heads"]
    tok = torch.from_numpy(tokens).long().to(DEV)
    pos = torch.from_numpy(np.concatenate([np.arange(o, o + n) for o, n in zip(old, new)])).to(DEV)
    seq = torch.from_numpy(np.repeat(np.arange(len(old)), new)).to(DEV)
    table = torch.from_numpy(bt).long().to(DEV)
    page, place = table[seq, pos // BLOCK], pos % BLOCK
    angle = pos.double()[:, None] * m["theta"] ** (-torch.arange(0, dh, 2, device=DEV).double() / dh)
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]

    def turn(x):
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)

    x = w("token_embd.weight")[tok]
    ks, vs = [], []
    for i in range(m["layers"]):
        b = "blk.%d." % i
        h = norm(x, b + "attn_norm.weight")
        q = turn((h @ w(b + "attn_q.weight").t()).view(-1, H, dh))
        k = turn((h @ w(b + "attn_k.weight").t()).view(-1, G, dh))
        v = (h @ w(b + "attn_v.weight").t()).view(-1, G, dh)
        kp = torch.zeros(pages, G, BLOCK, dh, dtype=torch.bfloat16, device=DEV)
        vp = torch.zeros(pages, G, BLOCK // 8, dh, 8, dtype=torch.bfloat16, device=DEV)
        if max(old):
            _fill(case, seed, i, kp, vp)
        kp, vp = kp.double(), vp.double()
        kp[page, :, place] = k
        vp[page, :, place // 8, :, place % 8] = v
        ks.append(kp)
        vs.append(vp)
        out, at = torch.empty_like(q), 0
        for s, (o, n) in enumerate(zip(old, new)):
            mine = table[s, :-(-(o + n) // BLOCK)]
            kk = kp[mine].transpose(0, 1).reshape(G, -1, dh)[:, :o + n]
            vv = vp[mine].permute(1, 0, 2, 4, 3).reshape(G, -1, dh)[:, :o + n]
            for a in range(0, n, 512):
                e = min(n, a + 512)
                qq = q[at + a:at + e].view(e - a, G, H // G, dh)
                late = torch.arange(o + n, device=DEV)[None, :] > torch.arange(o + a, o + e, device=DEV)[:, None]
                for g in range(G):
                    sc = (qq[:, g].reshape(-1, dh) @ kk[g].t()).view(e - a, H // G, -1) / math.sqrt(dh)
                    p = torch.softmax(sc.masked_fill(late[:, None], -math.inf), -1)
                    out[at + a:at + e, g * (H // G):(g + 1) * (H // G)] = (p.view(-1, o + n) @ vv[g]).view(e - a, H // G, dh)
            at += n
        x = x + out.flatten(1) @ w(b + "attn_output.weight").t()
        h = norm(x, b + "ffn_norm.weight")
        if m["experts"]:
            p, pick = torch.topk(torch.softmax(h @ w(b + "ffn_gate_inp.weight").t(), -1), EXPERTS_USED, -1)
            p = p / p.sum(-1, keepdim=True)
            gate, up, down = (w(b + "ffn_%s_exps.weight" % n) for n in ("gate", "up", "down"))
            add = torch.zeros_like(x)
            for e in range(m["experts"]):
                rows, which = (pick == e).nonzero(as_tuple=True)
                y = torch.nn.functional.silu(h[rows] @ gate[e].t()) * (h[rows] @ up[e].t())
                add.index_add_(0, rows, (y @ down[e].t()) * p[rows, which, None])
            x = x + add
        else:
            y = torch.nn.functional.silu(h @ w(b + "ffn_gate.weight").t()) * (h @ w(b + "ffn_up.weight").t())
            x = x + y @ w(b + "ffn_down.weight").t()
    x = x[torch.from_numpy(np.cumsum(new) - 1).to(DEV)]
    return {"logits": norm(x, "output_norm.weight") @ w("output.weight").t(), "k": ks, "v": vs}
