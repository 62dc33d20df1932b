"""Decode steps of batches whose (sequence, KV group) pairs fill between half a
wave of workgroups and a whole one, at the edges of their split rule, against
attention in float64.

Bar: fp16 outputs of N(0, 1) inputs, |o| below 4: max-abs <= 2e-3, two fp16
roundings there; cache rows bit for bit.
"""
import math

import pytest

torch = pytest.importorskip("torch")

import nwd_attn as nw  # noqa: E402
from gpu_util import pos_tensor, randn_f16, say  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,Hkv,Dh,B,longest,splits", [
    (32, 8, 128, 17, 800, 1),   # the longest of one split
    (32, 8, 128, 17, 801, 2),
    (32, 8, 128, 17, 2304, 2),
    (32, 8, 128, 17, 2305, 5),
    (32, 8, 128, 31, 600, 1),
    (32, 8, 128, 30, 2500, 2),  # its two waves are nearly full
    (32, 8, 128, 24, 5000, 8),
    (32, 8, 128, 17, 6500, 4),  # waves times keys only a sixth less
    (24, 8, 128, 17, 400, 1),   # a group below four heads
    (24, 8, 128, 17, 401, 2),
    (32, 32, 96, 5, 1500, 3),   # one head per workgroup
    (32, 32, 96, 6, 1500, 2),   # three waves of a third are two of a half
    (16, 8, 256, 20, 2500, 5),
    (10, 2, 256, 65, 400, 1),   # head sizes past 128
    (10, 2, 256, 65, 401, 2),
    (14, 2, 64, 65, 300, 1),
    (14, 2, 64, 65, 3000, 2),   # not by waves at head size 64
])
def test_batched_step(H, Hkv, Dh, B, longest, splits):
    say(f"batched step H={H} Hkv={Hkv} D={Dh} B={B} longest={longest}")
    lens = [longest - (b * 37) % (longest // 2) for b in range(B)]
    cap = longest + 3
    q, kn, vn = randn_f16((B, H, Dh), 1), randn_f16((B, Hkv, Dh), 2), randn_f16((B, Hkv, Dh), 3)
    kc, vc = randn_f16((B, Hkv, cap, Dh), 4), randn_f16((B, Hkv, cap, Dh), 5)
    k, v = kc.clone(), vc.clone()
    out = torch.empty((B, H, Dh), dtype=torch.float16, device="cuda")
    with nw.AttnContext(H, Hkv, cap, head_dim=Dh, max_batch=B) as ctx:
        assert ctx.decode_splits(B, longest) == splits
        ctx.append_decode(q, kn, vn, k, v, pos_tensor([n - 1 for n in lens]), out, B, longest)
        assert ctx.device_status() == nw.NWD_OK
    for b, n in enumerate(lens):
        kc[b, :, n - 1], vc[b, :, n - 1] = kn[b], vn[b]
        qb = q[b].double().view(Hkv, H // Hkv, Dh)
        w = torch.softmax(torch.matmul(qb, kc[b, :, :n].double().transpose(1, 2).contiguous()) / math.sqrt(Dh), -1)
        want = torch.matmul(w, vc[b, :, :n].double()).view(H, Dh)
        assert float((out[b].double() - want).abs().max()) <= 2e-3, b
    assert torch.equal(k, kc) and torch.equal(v, vc)
