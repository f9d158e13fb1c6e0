"""Matrix-core decode at the edges of its tiles: contexts ending on either side
of a 16-token tile and of a wave's 64-tile block-id window, in pools whose
unattended rows hold NaN, with an unmapped block inside the context and the
current row in it holding infinities.  Against the oracle, 2e-2 as for every
16-bit decode test."""
import pytest
import torch

from oracle import attention as oracle
from voiceagent_amd import ops

pytestmark = pytest.mark.gpu
HQ, HKV, D, BS = 16, 8, 128, 16


def _case(lens, kv, gen):
    need = [-(-n // BS) for n in lens]
    nb = sum(need) + 2
    perm = torch.randperm(nb, generator=gen)
    table = torch.full((len(lens), max(need)), -1, dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = perm[at:at + n]
        at += n
    dt = torch.float16 if kv == "f16" else torch.bfloat16
    pools = [torch.randn(nb, BS, HKV, D, generator=gen) for _ in range(2)]
    pools = [oracle.quantize_fp8(p, 0.05) if kv == "fp8" else p.to(dt) for p in pools]
    return table, pools, dt


@pytest.mark.parametrize("kv", ["bf16", "f16", "fp8"])
@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("lens", [[1, 15, 16, 17, 31, 33, 127, 128, 129],
                                  [8191, 8192, 8193, 8209],      # 64 tiles of eight waves
                                  [4096 + 1] * 40,               # four-wave workgroups, two windows
                                  [n for n in range(1, 280, 7)]])
def test_tile_edges_over_nan_tails(dev, lens, exact, kv):
    gen = torch.Generator().manual_seed(sum(lens) + exact)
    table, (kp, vp), dt = _case(lens, kv, gen)
    q = torch.randn(len(lens), HQ, D, generator=gen).to(dt)
    ks = 0.05 if kv == "fp8" else 1.0
    ref = oracle.paged_decode(q, kp, vp, table, torch.tensor(lens, dtype=torch.int32), D ** -0.5,
                              k_scale=ks, v_scale=ks)
    # Every row no context covers becomes NaN.
    live = torch.zeros(kp.shape[0], BS, dtype=torch.bool)
    for i, n in enumerate(lens):
        pos = torch.arange(n)
        live[table[i, pos // BS].long(), pos % BS] = True
    kp, vp = kp.clone(), vp.clone()
    for p in (kp, vp):
        if kv == "fp8":
            p.view(torch.uint8)[~live] = 0x7F
        else:
            p[~live] = float("nan")
    # Four contexts of 8192 would be cut over the CUs: whole, each of a
    # workgroup's eight waves has 64 tiles and refills its window.
    split = 8704 if len(lens) == 4 else ops.SPLIT_EXACT if exact else 0
    print(f"{len(lens)} contexts up to {max(lens)}, {kv}", flush=True)
    out = ops.paged_decode(q.to(dev), kp.to(dev), vp.to(dev), table.to(dev),
                           torch.tensor(lens, dtype=torch.int32, device=dev),
                           max_seq_len=max(lens) if exact else 32768, scale=D ** -0.5,
                           split_tokens=split, k_scale=ks, v_scale=ks)
    assert (out.float().cpu() - ref).abs().max().item() <= 2e-2


@pytest.mark.parametrize("kv", ["bf16", "fp8"])
def test_current_row_of_an_unmapped_block_is_stored_and_not_attended(dev, kv):
    lens = [40, 100]
    gen = torch.Generator().manual_seed(9)
    table, (kp, vp), dt = _case(lens, kv, gen)
    slots = torch.tensor([int(table[i, (n - 1) // BS]) * BS + (n - 1) % BS
                          for i, n in enumerate(lens)], dtype=torch.int32)
    bad = table.clone()
    bad[0, 2] = -1  # the block of the first context's current row
    bad[1, 1] = kp.shape[0]
    q = torch.randn(2, HQ, D, generator=gen).to(dt)
    nk = torch.randn(2, HKV, D, generator=gen).to(dt)
    nv = torch.randn(2, HKV, D, generator=gen).to(dt)
    big = nv.clone()
    big[0] = float("inf")
    ks = 0.05 if kv == "fp8" else 1.0
    outs = []
    for v_row in (nv, big):
        kd, vd = kp.to(dev), vp.to(dev)
        out = ops.paged_decode(q.to(dev), kd, vd, bad.to(dev),
                               torch.tensor(lens, dtype=torch.int32, device=dev), max_seq_len=100,
                               scale=D ** -0.5, new_k=nk.to(dev), new_v=v_row.to(dev),
                               new_slots=slots.to(dev), k_scale=ks, v_scale=ks)
        torch.cuda.synchronize()
        ek, ev = oracle.store_kvcache(nk, v_row, kp, vp, slots, k_scale=ks, v_scale=ks)
        as_bytes = torch.uint8 if kv == "fp8" else torch.int16
        assert torch.equal(kd.cpu().view(as_bytes), ek.view(as_bytes))
        assert torch.equal(vd.cpu().view(as_bytes), ev.view(as_bytes))
        outs.append(out.float().cpu())
    assert torch.isfinite(outs[1]).all()
    assert torch.equal(outs[0], outs[1])
