"""Performance cases of the attention core, each through a public entry point.

Geometry is the decoder's (16 query heads, 8 KV heads, head_dim 128, blocks of
16 tokens) and the audio encoder's (14 heads of 64, 104-token windows).  A case
is one of four kinds of call:

decode   one token per sequence through ``PagedAttention`` with Qwen3's q/k
         prologue and the fused store, over the engine's paged pool (16-bit or
         FP8).  ``graph``: the layers are captured once in a HIP graph whose
         ``max_seqlen_k`` is the model's maximum (``bound``), as the engine's
         decode buckets are, and a pass replays it; otherwise an eager step
         with the batch's exact maximum.
tts      the talker's ``paged_attention_decode`` over its head-major pool, with
         int64 tables, the key mask and the current row, layers captured in a
         HIP graph.
prefill  one layer of an eager step through ``PagedAttention`` with the
         prologue and the fused store: new prompts, prompts that continue a
         cached prefix (chunked or streamed audio), and decoding sequences that
         share the step (continuous batching mixes them).
encoder  one layer of ``VarlenSelfAttention`` over packed audio windows.

Several layers of a decode pass have pools of their own, so the K/V rows are
read from memory as in a whole model's step rather than from a cache.
"""

from __future__ import annotations

import math
import random

import torch

HQ, HKV, D, BLOCK = 16, 8, 128, 16
EPS = 1e-6
MAX_POS = 32768
ENC_HEADS, ENC_DIM, ENC_WINDOW = 14, 64, 104
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
FP8_SCALE = 1.0 / 32.0  # value of one FP8 code unit, K and V


# --------------------------------------------------------------- the cases
def listed():
    return [
        # One user speaking: a decode step of a single 30 s utterance.
        decode("decode-1", 1, 430, 430, layers=8, graph=True),
        # The serving batch: 32 utterances of a few seconds to half a minute.
        decode("decode-32", 32, 60, 600, layers=6, graph=True),
        # A full server over an FP8 pool, the largest decode bucket in use.
        decode("decode-128-fp8", 128, 60, 600, layers=4, graph=True, kv="fp8"),
        # Long-form audio: contexts of thousands of tokens, eager step.
        decode("decode-8-long", 8, 4096, 16384, layers=2),
        # The talker speaking four replies of about two minutes.
        tts("tts-4", 4, 1500, layers=8),
        # A burst of new utterances (the packed prompt step).
        prefill("prefill-32", prompts=32, lo=50, hi=450),
        # One new utterance: the time to the first token of a single user.
        prefill("prefill-1", prompts=1, lo=420, hi=420),
        # A long recording transcribed in one prompt.
        prefill("prefill-1-long", prompts=1, lo=16384, hi=16384),
        # Streams that add a few seconds of audio to a cached context.
        prefill("prefill-4-prefix", prompts=4, lo=200, hi=300, plo=2048, phi=8192),
        # A continuous-batching step: 28 decoding sequences and 4 new prompts.
        prefill("mixed-32", prompts=4, lo=50, hi=450, decodes=28, dlo=60, dhi=600),
        # The encoder over a burst of 32 clips.
        encoder("encoder-32", 32, 2.0, 30.0),
        # The encoder over a single 30 s clip.
        encoder("encoder-1", 1, 30.0, 30.0),
    ]


def decode(name, batch, lo, hi, *, layers, graph=False, kv="bf16", dtype="bf16", bound=32768, mix=0):
    return {"name": name, "kind": "decode", "batch": batch, "lo": lo, "hi": hi, "layers": layers,
            "graph": graph, "kv": kv, "dtype": dtype, "bound": bound, "mix": mix}


def tts(name, batch, length, *, layers, dtype="bf16", mix=0):
    return {"name": name, "kind": "tts", "batch": batch, "lo": max(1, length * 3 // 4),
            "hi": length, "layers": layers, "dtype": dtype, "mix": mix}


def prefill(name, *, prompts, lo, hi, plo=0, phi=0, decodes=0, dlo=0, dhi=0, kv="bf16",
            dtype="bf16", mix=0):
    return {"name": name, "kind": "prefill", "prompts": prompts, "lo": lo, "hi": hi, "plo": plo,
            "phi": phi, "decodes": decodes, "dlo": dlo, "dhi": dhi, "kv": kv, "dtype": dtype,
            "mix": mix}


def encoder(name, clips, lo, hi, *, dtype="bf16", mix=0):
    return {"name": name, "kind": "encoder", "clips": clips, "lo": lo, "hi": hi, "dtype": dtype,
            "mix": mix}


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges; no case reads more K/V than the
    long-form decode or multiplies more than the long prompt."""
    kind = rng.choice(["decode", "tts", "prefill", "prefill", "prefill", "encoder"])
    mix = rng.randrange(1, 1 << 20)
    dtype = rng.choice(["bf16", "bf16", "f16"])
    kv = rng.choice([dtype, dtype, "fp8"])
    if kind == "decode":
        batch = _log(rng, 1, 160)
        hi = _log(rng, 64, min(16384, max(600, 90000 // batch)))
        lo = max(1, int(hi * rng.uniform(0.1, 1.0)))
        layers = max(2, min(8, 150000 // (batch * hi)))
        case = decode("", batch, lo, hi, layers=layers, graph=rng.random() < 0.6 or batch * hi < 4096,
                      kv=kv, dtype=dtype, mix=mix)
    elif kind == "tts":
        batch = _log(rng, 1, 16)
        case = tts("", batch, _log(rng, 100, 3000), layers=rng.randrange(4, 9), dtype=dtype, mix=mix)
    elif kind == "encoder":
        lo = rng.uniform(0.5, 20.0)
        case = encoder("", _log(rng, 1, 64), round(lo, 2), round(rng.uniform(lo, 30.0), 2),
                       dtype=dtype, mix=mix)
    else:
        form = rng.choice(["new", "prefix", "mixed"])
        if form == "new":
            prompts = _log(rng, 1, 48)
            hi = _log(rng, 24, int(16000 / prompts ** 0.75))
            case = prefill("", prompts=prompts, lo=max(1, int(hi * rng.uniform(0.1, 1.0))), hi=hi,
                           kv=kv, dtype=dtype, mix=mix)
        elif form == "prefix":
            prompts = _log(rng, 1, 12)
            hi = _log(rng, 8, 1200)
            phi = _log(rng, 64, int(12000 / prompts ** 0.25))
            case = prefill("", prompts=prompts, lo=max(1, int(hi * rng.uniform(0.2, 1.0))), hi=hi,
                           plo=max(1, int(phi * rng.uniform(0.1, 1.0))), phi=phi, kv=kv,
                           dtype=dtype, mix=mix)
        else:
            prompts = _log(rng, 1, 8)
            hi = _log(rng, 30, 1500)
            decodes = _log(rng, 1, 64)
            dhi = _log(rng, 60, int(6000 / decodes ** 0.4))
            case = prefill("", prompts=prompts, lo=max(1, int(hi * rng.uniform(0.2, 1.0))), hi=hi,
                           decodes=decodes, dlo=max(1, dhi // 8), dhi=dhi, kv=kv, dtype=dtype,
                           mix=mix)
    del case["name"]
    return case


# ------------------------------------------------------- lengths of a case
def _spread(rng, n, lo, hi):
    return [hi if n == 1 else rng.randint(lo, hi) for _ in range(n)]


def _lengths(case):
    """(new tokens, context tokens) of every sequence; the case alone says."""
    rng = random.Random(17 + case["mix"])
    if case["kind"] in ("decode", "tts"):
        return [(1, n) for n in _spread(rng, case["batch"], case["lo"], case["hi"])]
    if case["kind"] == "prefill":
        new = _spread(rng, case["prompts"], case["lo"], case["hi"])
        pre = _spread(rng, case["prompts"], case["plo"], case["phi"])
        seqs = [(n, n + p) for n, p in zip(new, pre)]
        seqs += [(1, n) for n in _spread(rng, case["decodes"], case["dlo"], case["dhi"])]
        rng.shuffle(seqs)
        return seqs
    from voiceagent_amd.audio import batcher
    secs = [case["hi"] if case["clips"] == 1 else rng.uniform(case["lo"], case["hi"])
            for _ in range(case["clips"])]
    toks = [batcher.num_audio_tokens(int(s * 100)) for s in secs]
    bounds = batcher.build_window_boundaries(toks, ENC_WINDOW)
    return [(b - a, b - a) for a, b in zip(bounds[:-1], bounds[1:])]


def work(case):
    seqs = _lengths(case)
    total = sum(n for n, _ in seqs)
    if case["kind"] == "encoder":
        width = ENC_HEADS * ENC_DIM
        return {"bytes": 4 * total * width * 2, "flops": sum(4 * width * n * n for n, _ in seqs)}
    kv_bytes = 1 if case.get("kv") == "fp8" else 2
    row = HKV * D
    layers = case.get("layers", 1)
    cached = sum(c - n for n, c in seqs) * 2 * row * kv_bytes
    rows = total * (2 * HQ * D + 2 * row) * 2 + total * 2 * row * kv_bytes
    pairs = sum(n * (c - n) + n * (n + 1) // 2 for n, c in seqs)
    return {"bytes": layers * (cached + rows), "flops": layers * 4 * HQ * D * pairs}


def tolerance(case):
    # 16-bit outputs and probabilities: two correct implementations differ by
    # about 2^-8 relative (2-norm).  FP8 pools come back as codes, of which a
    # new key's may fall on the other side of a rounding tie.
    return {"rel": 1e-2, "max": 0.25, "differ": 1e-3}


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(gen, *shape, std=1.0, dtype=torch.float32):
    return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32).mul_(std).to(dtype)


def _pool(gen, shape, std, dtype, kv):
    x = _randn(gen, *shape, std=std, dtype=torch.bfloat16 if kv == "fp8" else dtype)
    return (x.float() / FP8_SCALE).to(torch.float8_e4m3fn) if kv == "fp8" else x


def _tables(seed, ctx):
    """Block ids of every sequence from one shuffled free list, -1 padded."""
    need = [-(-n // BLOCK) for n in ctx]
    blocks = sum(need) + 8
    perm = torch.randperm(blocks, generator=torch.Generator().manual_seed(seed))
    table = torch.full((len(ctx), max(need)), -1, dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = perm[at:at + n]
        at += n
    return table, blocks


def _inputs(case, seed):
    """The tensors of a case, from the seed alone."""
    seqs, gen, dtype = _lengths(case), _gen(seed), DTYPES[case["dtype"]]
    total = sum(n for n, _ in seqs)
    cu = torch.tensor([0] + [n for n, _ in seqs]).cumsum(0)
    cuk = torch.tensor([0] + [c for _, c in seqs]).cumsum(0)
    s = {"seqs": seqs, "cu_q": cu.to("cuda", torch.int32), "cu_k": cuk.to("cuda", torch.int32)}
    if case["kind"] == "encoder":
        s["q"], s["k"], s["v"] = (_randn(gen, total, ENC_HEADS, ENC_DIM, std=sd, dtype=dtype)
                                  for sd in (1.5, 1.5, 1.0))
        return s
    layers, kv = case.get("layers", 1), case.get("kv", case["dtype"])
    table, blocks = _tables(seed, [c for _, c in seqs])
    pos = torch.cat([torch.arange(c - n, c) for n, c in seqs])
    owner = torch.cat([torch.full((n,), i) for i, (n, _) in enumerate(seqs)])
    s["slots_cpu"] = table[owner, pos // BLOCK].long() * BLOCK + pos % BLOCK
    s["table_cpu"] = table
    s["positions"] = pos.cuda()
    s["layers"] = []
    hnd = case["kind"] == "tts"
    shape = (blocks, HKV, BLOCK, D) if hnd else (blocks, BLOCK, HKV, D)
    for _ in range(layers):
        # The projections' output: q, k and v are views of one qkv tensor.
        qkv = _randn(gen, total, (HQ + 2 * HKV) * D, dtype=dtype)
        s["layers"].append({
            "q": qkv[:, :HQ * D].view(total, HQ, D),
            "k": qkv[:, HQ * D:(HQ + HKV) * D].view(total, HKV, D),
            "v": qkv[:, (HQ + HKV) * D:].view(total, HKV, D),
            "qw": (1.2 + _randn(gen, D, std=0.1)).to(dtype),
            "kw": (1.2 + _randn(gen, D, std=0.1)).to(dtype),
            "kp": _pool(gen, shape, 1.2, dtype, kv),
            "vp": _pool(gen, shape, 1.0, dtype, kv),
        })
    if hnd:
        width = -(-max(c for _, c in seqs) // 128) * 128
        mask = torch.rand(len(seqs), width, generator=gen, device="cuda") < 0.95
        mask[:, :width // 20] = False  # left padding
        s["mask"] = mask
    else:
        inv = 1.0 / (1e6 ** (torch.arange(0, D, 2, dtype=torch.float) / D))
        freqs = torch.outer(torch.arange(MAX_POS, dtype=torch.float), inv)
        s["cos_sin"] = torch.cat((freqs.cos(), freqs.sin()), dim=-1).cuda()
    return s


def prepare(case, seed):
    from voiceagent_amd import ops
    from voiceagent_amd.layers import AttentionContext, PagedAttention, VarlenSelfAttention

    s = _inputs(case, seed)
    s["case"] = case
    if case["kind"] == "encoder":
        s["layer"] = VarlenSelfAttention(ENC_HEADS, ENC_DIM, ENC_DIM ** -0.5)
        s["max_len"] = max(n for n, _ in s["seqs"])
        return s
    if case["kind"] == "tts":
        s["lens"] = torch.tensor([c for _, c in s["seqs"]], device="cuda")
        s["table"] = s["table_cpu"].clamp(min=0).long().cuda()
        s["kernel_seq_len"] = s["mask"].shape[1]
        for t in s["layers"]:
            for name in ("q", "k", "v"):
                t[name] = t[name].contiguous().unsqueeze(2)
    else:
        graph = case.get("graph", False)
        s["context"] = AttentionContext(
            cu_seqlens_q=s["cu_q"], cu_seqlens_k=s["cu_k"],
            max_seqlen_q=max(n for n, _ in s["seqs"]),
            max_seqlen_k=case["bound"] if graph else max(c for _, c in s["seqs"]),
            slot_mapping=s["slots_cpu"].to("cuda", torch.int32), block_tables=s["table_cpu"].cuda(),
            max_seqlen_k_exact=not graph)
        for t in s["layers"]:
            layer = t["layer"] = PagedAttention(HQ, D, D ** -0.5, HKV)
            layer.k_cache, layer.v_cache = t["kp"], t["vp"]
            if case["kv"] == "fp8":
                layer.k_scale = layer.v_scale = FP8_SCALE
            t["prologue"] = ops.QKPrologue(t["qw"], t["kw"], EPS, s["cos_sin"], s["positions"])
    if case["kind"] == "tts" or case.get("graph", False):
        stream = torch.cuda.Stream()
        ops.reserve_decode_workspace(torch.device("cuda", torch.cuda.current_device()), HQ, HKV, D,
                                     stream=stream)
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            _layers(s)  # warm-up, as before any capture
        stream.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"], stream=stream):
            s["out"] = _layers(s)
    return s


# -------------------------------------------------------------------- calls
def _layers(s):
    if s["case"]["kind"] == "tts":
        from voiceagent_amd.agent import paged_attention_decode
        return [paged_attention_decode(t["q"], t["kp"], t["vp"], s["table"], s["lens"], s["mask"],
                                       new_key=t["k"], new_value=t["v"],
                                       kernel_seq_len=s["kernel_seq_len"],
                                       kernel_page_count=s["table"].shape[1], validate=False)
                for t in s["layers"]]
    from voiceagent_amd.layers import attention_context
    with attention_context(s["context"]):
        return [t["layer"](t["q"], t["k"], t["v"], prologue=t["prologue"]) for t in s["layers"]]


def run(s):
    case = s["case"]
    if case["kind"] == "encoder":
        return s["layer"](s["q"], s["k"], s["v"], s["cu_q"], s["max_len"])
    if "graph" in s:
        s["graph"].replay()
        out = s["out"]
    else:
        out = _layers(s)
    codes = case.get("kv") == "fp8"
    return {"out": out,
            "k": [t["kp"].view(torch.uint8) if codes else t["kp"] for t in s["layers"]],
            "v": [t["vp"].view(torch.uint8) if codes else t["vp"] for t in s["layers"]]}


# ------------------------------------------------------------ 64-bit results
def _attend(q, k, v, diag, keep=None):
    """Rows of q [n, h, d] over k, v [c, hk, d]; row i sees keys <= diag + i
    (all of them for diag None); keep [c] drops masked keys."""
    n, h, d = q.shape
    c, hk, _ = k.shape
    out = torch.empty(n, h, d, dtype=torch.float64, device=q.device)
    kt = k.permute(1, 2, 0).contiguous()
    vt = v.permute(1, 0, 2).contiguous()
    step = max(1, min(n, (1 << 27) // (h * c)))
    for a in range(0, n, step):
        b = min(n, a + step)
        end = c if diag is None else min(c, diag + b)
        x = q[a:b].view(b - a, hk, h // hk, d).permute(1, 2, 0, 3).reshape(hk, -1, d)
        x = torch.matmul(x.contiguous(), kt[:, :, :end].contiguous()) * d ** -0.5
        x = x.view(hk, h // hk, b - a, end)
        if diag is not None:
            seen = (torch.arange(end, device=q.device)[None]
                    <= diag + torch.arange(a, b, device=q.device)[:, None])
            x = x.masked_fill(~seen, -math.inf)
        if keep is not None:
            x = x.masked_fill(~keep[:end], -math.inf)
        x = torch.softmax(x, dim=-1).view(hk, -1, end)
        x = torch.matmul(x, vt[:, :end].contiguous())
        out[a:b] = x.view(hk, h // hk, b - a, d).permute(2, 0, 1, 3).reshape(b - a, h, d)
    return out


def _normed(x, w, cos_sin):
    """Qwen3's per-head RMSNorm and half-split rotary embedding."""
    x = x.double()
    x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()
    cos, sin = (t[:, None] for t in cos_sin.double().chunk(2, dim=-1))
    a, b = x.chunk(2, dim=-1)
    return torch.cat((a * cos - b * sin, b * cos + a * sin), dim=-1)


def exact(case, seed):
    s = _inputs(case, seed)
    starts = [0]
    for n, _ in s["seqs"]:
        starts.append(starts[-1] + n)
    if case["kind"] == "encoder":
        q, k, v = (s[x].double() for x in ("q", "k", "v"))
        return torch.cat([_attend(q[a:b], k[a:b], v[a:b], None)
                          for a, b in zip(starts[:-1], starts[1:])])
    hnd, fp8 = case["kind"] == "tts", case.get("kv") == "fp8"
    slots, table = s["slots_cpu"].cuda(), s["table_cpu"].cuda().long()
    got = {"out": [], "k": [], "v": []}
    for t in s["layers"]:
        q, k, v = (t[x].double() for x in ("q", "k", "v"))
        if not hnd:
            rot = s["cos_sin"][s["positions"]]
            q, k = _normed(t["q"], t["qw"], rot), _normed(t["k"], t["kw"], rot)
        pools = []
        for name, new in (("kp", k), ("vp", v)):
            pool = t[name].permute(0, 2, 1, 3).contiguous() if hnd else t[name]
            pool = (pool.float().double() * FP8_SCALE if fp8 else pool.double()).view(-1, HKV, D)
            pool[slots] = new
            pools.append(pool)
        outs = []
        for i, (n, c) in enumerate(s["seqs"]):
            blocks = table[i, :-(-c // BLOCK)]
            idx = (blocks[:, None] * BLOCK + torch.arange(BLOCK, device="cuda")).view(-1)[:c]
            keep = s["mask"][i, :c] if hnd else None
            outs.append(_attend(q[starts[i]:starts[i + 1]], pools[0][idx], pools[1][idx], c - n, keep))
        out = torch.cat(outs)
        got["out"].append(out.unsqueeze(2) if hnd else out)
        for name, pool in zip(("k", "v"), pools):
            pool = pool.view(-1, BLOCK, HKV, D)
            got[name].append(None if fp8 else pool.permute(0, 2, 1, 3).contiguous() if hnd else pool)
    return got
