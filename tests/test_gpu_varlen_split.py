"""Varlen launches whose long items are cut into pieces over several
workgroups and merged (varlen_merge_kernel), at the sizes where the plan, the
block-id windows (64 tiles of 64 keys) and the piece edges can go wrong:
against the oracle (2e-2 for 16-bit inputs, the suite's bound) and against the
same launch without a workspace, which runs unsplit.  Each case says whether
its launch splits, as the host's rule and the device's plan do.  Both forms keep fp32
sums and differ in their order and in the reference maximum of P's 16-bit
rounding, so they agree to two 16-bit output roundings and P's: 2^-7 of the
largest |v| (under 5 for these N(0, 1) values)."""
import math

import pytest
import torch

from oracle import attention as oracle
from voiceagent_amd import _native as N
from voiceagent_amd import ops

pytestmark = pytest.mark.gpu


class Library:
    """The library as the wrappers call it, with the workspace of varlen launches
    held here: ``size`` is what the host's rule asked for, ``pieces()`` what the
    device's plan cut (its counts stand in the workspace's last 256 bytes).
    ``give`` says which workspace a launch gets: "fit", "none", one byte too
    "short", or "odd" (not on 16 bytes)."""

    def __init__(self, give):
        self.real, self.give, self.size, self.ws = N.lib(), give, None, None

    def __call__(self):
        return self

    def __getattr__(self, fn):
        return getattr(self.real, fn)

    def va_varlen_split_workspace_bytes(self, args):
        self.size = self.real.va_varlen_split_workspace_bytes(args)
        return 0

    def va_varlen_attention(self, args, stream):
        a = args._obj
        if self.size and self.give != "none":
            self.ws = torch.full((self.size + 16,), 0xAB, dtype=torch.uint8, device="cuda")
            a.workspace = self.ws.data_ptr() + (8 if self.give == "odd" else 0)
            a.workspace_bytes = self.size - (1 if self.give == "short" else 0)
        return self.real.va_varlen_attention(args, stream)

    def pieces(self):
        return int(self.ws[self.size - 256:self.size - 224].view(torch.int32).sum()) if self.size else 0


def _through(monkeypatch, give):
    lib = Library(give)
    monkeypatch.setattr(ops, "_FAST_LOADED", True)
    monkeypatch.setattr(ops, "_FAST", None)
    monkeypatch.setattr(N, "lib", lib)
    return lib


def _cu(lens):
    return torch.tensor([0] + lens, dtype=torch.int32).cumsum(0).to(torch.int32)


# (prefix, new tokens) per sequence
CASES = {
    "one_decode_past_the_id_window": [(64 * 64 + 5, 1)],
    "window_edges": [(64 * 64, 3), (64 * 64 - 1, 1), (64 * 128, 70)],
    "decodes_beside_prompts": [(n, 1) for n in (1, 15, 16, 17, 63, 64, 700, 2500, 4097)]
                              + [(0, 300), (0, 1), (0, 65), (33, 130)],
    "short_chunks_long_prefixes": [(3000, 8), (2049, 17), (1500, 64), (1, 2)],
    "long_prompt": [(0, 1100)],
    "with_empty_sequences": [(0, 0), (900, 1), (700, 0), (0, 270), (0, 0)],
    "many_sequences": [(130 + 7 * i, 1 + i % 3) for i in range(60)],
    "twenty_long_contexts": [(2000 + 37 * i, 1 + i % 3) for i in range(20)],
}
WHOLE = ("long_prompt", "many_sequences")  # nothing to gain: the host leaves them whole


@pytest.mark.parametrize("kv", ["bf16", "f16", "fp8"])
@pytest.mark.parametrize("hq,hkv,d,bs,i64,hnd", [(16, 8, 128, 16, False, False),
                                                 (32, 4, 128, 48, True, True),
                                                 (14, 14, 64, 8, False, False),
                                                 (16, 2, 64, 16, True, False)])
@pytest.mark.parametrize("name", list(CASES))
def test_split_launch(dev, monkeypatch, name, hq, hkv, d, bs, i64, hnd, kv):
    seqs = CASES[name]
    gen = torch.Generator().manual_seed(len(name) + hq + d + bs)
    dt = torch.float16 if kv == "f16" else torch.bfloat16
    ql, kl = [n for _, n in seqs], [p + n for p, n in seqs]
    need = [math.ceil(n / bs) for n in kl]
    nb, width = sum(need) + 3, max(need)
    perm = torch.randperm(nb, generator=gen).tolist()
    table = torch.full((len(seqs), width), -1, dtype=torch.int64 if i64 else torch.int32)
    at, slots = 0, []
    for s, m in enumerate(need):
        table[s, :m] = torch.tensor(perm[at:at + m])
        at += m
        slots += [int(table[s, j // bs]) * bs + j % bs for j in range(seqs[s][0], kl[s])]
    slots = torch.tensor(slots, dtype=torch.int32)
    shape = (nb, hkv, bs, d) if hnd else (nb, bs, hkv, d)
    layout = ops.LAYOUT_HND if hnd else ops.LAYOUT_NHD
    ks, vs = (0.05, 0.08) if kv == "fp8" else (1.0, 1.0)
    kp, vp = (torch.randn(shape, generator=gen) for _ in range(2))
    if kv == "fp8":
        kp, vp = oracle.quantize_fp8(kp, ks), oracle.quantize_fp8(vp, vs)
    else:
        kp, vp = kp.to(dt), vp.to(dt)
    q = torch.randn(sum(ql), hq, d, generator=gen).to(dt)
    k, v = (torch.randn(sum(ql), hkv, d, generator=gen).to(dt) for _ in range(2))
    cu_q, cu_k = _cu(ql), _cu(kl)
    print(f"{name} {hq}/{hkv}x{d} block {bs} {kv}", flush=True)

    def call():
        kd, vd = kp.to(dev), vp.to(dev)
        out = ops.varlen_attention(q.to(dev), k.to(dev), v.to(dev), cu_q.to(dev), cu_k.to(dev),
                                   max(ql), max(kl), scale=d ** -0.5, causal=True, k_cache=kd,
                                   v_cache=vd, block_tables=table.to(dev),
                                   slot_mapping=slots.to(dev), layout=layout, k_scale=ks,
                                   v_scale=vs)
        torch.cuda.synchronize()
        return out.float().cpu(), kd.cpu(), vd.cpu()

    out, kd, vd = call()
    ref = oracle.varlen_attention(q, k, v, cu_q, cu_k, d ** -0.5, True, k_cache=kp, v_cache=vp,
                                  block_tables=table, layout=layout, k_scale=ks, v_scale=vs)
    assert (out - ref).abs().max().item() <= 2e-2
    ek, ev = oracle.store_kvcache(k, v, kp, vp, slots, layout=layout, k_scale=ks, v_scale=vs)
    as_bytes = torch.uint8 if kv == "fp8" else torch.int16
    assert torch.equal(kd.view(as_bytes), ek.view(as_bytes))
    assert torch.equal(vd.view(as_bytes), ev.view(as_bytes))
    # The same launch with the workspace in hand: did it split?
    lib = _through(monkeypatch, "fit")
    again, _, _ = call()
    assert torch.equal(again, out)
    assert (lib.size > 0) == (lib.pieces() > 1) == (name not in WHOLE)
    # Without one, and with one that cannot be used: unsplit.
    monkeypatch.undo()
    _through(monkeypatch, "none")
    whole, _, _ = call()
    assert (whole - ref).abs().max().item() <= 2e-2
    assert (whole - out).abs().max().item() <= 5 * 2 ** -7
    for give in ("short", "odd"):
        monkeypatch.undo()
        lib = _through(monkeypatch, give)
        assert torch.equal(call()[0], whole)
        assert lib.ws is None or bool((lib.ws == 0xAB).all())


@pytest.mark.parametrize("hq,hkv,d,lens,splits", [
    (hq, hkv, d, lens, splits) for hq, hkv, d in [(14, 14, 64), (16, 8, 128)]
    for lens, splits in [([700], False), ([300, 1, 900, 64], False), ([1, 2, 1300], False)]] + [
    (14, 14, 64, [2500], True), (8, 8, 128, [2500], True), (8, 8, 128, [300, 1, 2200, 64], True)])
@pytest.mark.parametrize("causal", [False, True])
def test_split_launch_without_a_pool(dev, monkeypatch, hq, hkv, d, causal, lens, splits):
    gen = torch.Generator().manual_seed(sum(lens) + d)
    q = torch.randn(sum(lens), hq, d, generator=gen).to(torch.bfloat16)
    k, v = (torch.randn(sum(lens), hkv, d, generator=gen).to(torch.bfloat16) for _ in range(2))
    cu = _cu(lens)
    out = ops.varlen_attention(q.to(dev), k.to(dev), v.to(dev), cu.to(dev), cu.to(dev), max(lens),
                               max(lens), scale=d ** -0.5, causal=causal)
    ref = oracle.varlen_attention(q, k, v, cu, cu, d ** -0.5, causal)
    assert (out.float().cpu() - ref).abs().max().item() <= 2e-2
    lib = _through(monkeypatch, "fit")
    again = ops.varlen_attention(q.to(dev), k.to(dev), v.to(dev), cu.to(dev), cu.to(dev), max(lens),
                                 max(lens), scale=d ** -0.5, causal=causal)
    assert torch.equal(again, out)
    assert (lib.size > 0) == (lib.pieces() > 1) == splits


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,qlens,prefix", [
    (16, 8, [8, 17, 64, 2], [3000, 2049, 1500, 1]), (32, 4, [1, 70, 5], [4096, 2100, 900]),
    (8, 8, [130, 1], [1900, 64]), (8, 8, [2500], None), (8, 8, [300, 1, 2200], None)])
def test_split_launch_with_the_query_prologue(dev, monkeypatch, hq, hkv, qlens, prefix, dtype):
    # Each piece normalises and rotates its query rows itself: against the
    # oracle and against the prologue in a launch of its own.
    d, bs, eps = 128, 16, 1e-6
    gen = torch.Generator().manual_seed(hq + sum(qlens))
    klens = [p + n for p, n in zip(prefix or [0] * len(qlens), qlens)]
    T = sum(qlens)
    q = torch.randn(T, hq, d, generator=gen).to(dtype)
    k, v = (torch.randn(T, hkv, d, generator=gen).to(dtype) for _ in range(2))
    wq, wk = ((torch.rand(d, generator=gen) + 0.5).to(dtype) for _ in range(2))
    pos, cs = torch.randint(0, 4096, (T,), generator=gen), oracle.rope_cache(d, 4096, 1e6)
    cu_q, cu_k = _cu(qlens), _cu(klens)
    pro = ops.QKPrologue(wq.to(dev), wk.to(dev), eps, cs.to(dev), pos.to(dev))
    pool, paged = {}, {}
    if prefix:
        need = [math.ceil(n / bs) for n in klens]
        perm = torch.randperm(sum(need) + 3, generator=gen)
        table = torch.full((len(qlens), max(need)), -1, dtype=torch.int32)
        at = 0
        for s, m in enumerate(need):
            table[s, :m] = perm[at:at + m]
            at += m
        slots = torch.tensor([int(table[s, j // bs]) * bs + j % bs for s in range(len(qlens))
                              for j in range(prefix[s], klens[s])], dtype=torch.int32)
        kp, vp = (torch.randn(len(perm), bs, hkv, d, generator=gen).to(dtype) for _ in range(2))
        paged = dict(k_cache=kp, v_cache=vp, block_tables=table)

    def call(q, k, prologue=None):
        pool.update({n: t.to(dev) for n, t in paged.items()})
        if paged:
            pool["slot_mapping"] = slots.to(dev)
        return ops.varlen_attention(q, k, v.to(dev), cu_q.to(dev), cu_k.to(dev), max(qlens),
                                    max(klens), scale=d ** -0.5, causal=True, prologue=prologue,
                                    **pool)

    print(f"prologue, {hq}/{hkv} heads, {qlens} over {prefix}, {dtype}", flush=True)
    q2, k2 = ops.qk_norm_rope(q.to(dev), k.to(dev), pro)
    two = call(q2, k2)
    stored = [pool[n].clone() for n in ("k_cache", "v_cache")] if paged else []
    lib = _through(monkeypatch, "fit")
    out = call(q.to(dev), k2, pro)
    torch.cuda.synchronize()
    assert lib.size > 0 and lib.pieces() > 1
    for t, n in zip(stored, ("k_cache", "v_cache")):
        assert torch.equal(pool[n], t)
    rq, rk = oracle.qk_norm_rope(q, k, pos, wq, wk, eps, cs)
    ref = oracle.varlen_attention(rq, rk, v, cu_q, cu_k, d ** -0.5, True, **paged)
    assert (out.float().cpu() - ref).abs().max().item() <= 2e-2
    assert (out.float() - two.float()).abs().max().item() <= 2e-2


@pytest.mark.parametrize("kv", ["bf16", "fp8"])
@pytest.mark.parametrize("bs", [16, 8])
@pytest.mark.parametrize("dim", [0, 1, 2], ids=["block", "slot", "head"])
def test_pool_with_a_negative_stride(dev, monkeypatch, dim, bs, kv):
    # The C ABI takes pool strides of either sign: the pool lies reversed along
    # one dimension and is described from that dimension's last element.
    gen = torch.Generator().manual_seed(10 * bs + dim)
    hq, hkv, d, seqs = 16, 8, 128, [(700, 1), (130, 70), (0, 90), (33, 5)]
    ql, kl = [n for _, n in seqs], [p + n for p, n in seqs]
    need = [math.ceil(n / bs) for n in kl]
    nb = sum(need) + 1
    perm = torch.randperm(nb, generator=gen)
    table = torch.full((len(seqs), max(need)), -1, dtype=torch.int32)
    at = 0
    for s, m in enumerate(need):
        table[s, :m] = perm[at:at + m]
        at += m
    slots = torch.tensor([int(table[s, j // bs]) * bs + j % bs
                          for s, (p, n) in enumerate(seqs) for j in range(p, p + n)],
                         dtype=torch.int32)
    ks, vs = (0.05, 0.08) if kv == "fp8" else (1.0, 1.0)
    kp, vp = (torch.randn(nb, bs, hkv, d, generator=gen) for _ in range(2))
    if kv == "fp8":
        kp, vp = oracle.quantize_fp8(kp, ks), oracle.quantize_fp8(vp, vs)
    else:
        kp, vp = kp.to(torch.bfloat16), vp.to(torch.bfloat16)
    q = torch.randn(sum(ql), hq, d, generator=gen).to(torch.bfloat16)
    k, v = (torch.randn(sum(ql), hkv, d, generator=gen).to(torch.bfloat16) for _ in range(2))
    cu_q, cu_k = _cu(ql), _cu(kl)
    as_bytes = torch.uint8 if kv == "fp8" else torch.int16
    monkeypatch.setattr(ops, "_FAST_LOADED", True)
    monkeypatch.setattr(ops, "_FAST", None)
    real = N.lib()

    class Reversed:
        def __getattr__(self, fn):
            return self.launch if fn == "va_varlen_attention" else getattr(real, fn)

        def launch(self, args, stream):
            pool = args._obj.pool
            field = ("stride_block", "stride_slot", "stride_head")[dim]
            step = getattr(pool, field) * (1 if kv == "fp8" else 2)
            pool.k += ((nb, bs, hkv)[dim] - 1) * step
            pool.v += ((nb, bs, hkv)[dim] - 1) * step
            setattr(pool, field, -getattr(pool, field))
            return real.va_varlen_attention(args, stream)

    monkeypatch.setattr(N, "lib", Reversed)
    print(f"dimension {dim} reversed, block {bs} {kv}", flush=True)
    kd, vd = (p.view(as_bytes).flip(dim).view(p.dtype).to(dev) for p in (kp, vp))
    out = ops.varlen_attention(q.to(dev), k.to(dev), v.to(dev), cu_q.to(dev), cu_k.to(dev),
                               max(ql), max(kl), scale=d ** -0.5, causal=True, k_cache=kd,
                               v_cache=vd, block_tables=table.to(dev), slot_mapping=slots.to(dev),
                               k_scale=ks, v_scale=vs)
    torch.cuda.synchronize()
    ref = oracle.varlen_attention(q, k, v, cu_q, cu_k, d ** -0.5, True, k_cache=kp, v_cache=vp,
                                  block_tables=table, k_scale=ks, v_scale=vs)
    assert (out.float().cpu() - ref).abs().max().item() <= 2e-2
    ek, ev = oracle.store_kvcache(k, v, kp, vp, slots, k_scale=ks, v_scale=vs)
    assert torch.equal(kd.cpu().view(as_bytes).flip(dim), ek.view(as_bytes))
    assert torch.equal(vd.cpu().view(as_bytes).flip(dim), ev.view(as_bytes))


def test_loose_max_seqlen_q(dev):
    # max_seqlen_q is any bound of the lengths; the largest a launch takes is
    # 65535 * 16 query blocks of 128 rows, also where items of 64 rows would do.
    hq, hkv, d, lens = 16, 2, 128, [4, 1, 2]
    gen = torch.Generator().manual_seed(5)
    q = torch.randn(sum(lens), hq, d, generator=gen).to(torch.bfloat16)
    k, v = (torch.randn(sum(lens), hkv, d, generator=gen).to(torch.bfloat16) for _ in range(2))
    cu = _cu(lens)
    bound = 65535 * 16 * (128 * hkv // hq)
    out = ops.varlen_attention(q.to(dev), k.to(dev), v.to(dev), cu.to(dev), cu.to(dev), bound,
                               max(lens), scale=d ** -0.5, causal=True)
    ref = oracle.varlen_attention(q, k, v, cu, cu, d ** -0.5, True)
    assert (out.float().cpu() - ref).abs().max().item() <= 2e-2
    with pytest.raises(N.NativeError, match="max_seqlen_q"):
        ops.varlen_attention(q.to(dev), k.to(dev), v.to(dev), cu.to(dev), cu.to(dev), bound + 1,
                             max(lens), scale=d ** -0.5, causal=True)
