"""reshape_and_cache_tiers: one launch into both tiers' caches, against the two
reshape_and_cache calls it replaces, bit for bit."""

from __future__ import annotations

import pytest
import torch

from vllm_fastdecoder_amd import ops
from vllm_fastdecoder_amd.pinned import pinned_empty

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,KVH,D,BS,dtype", [
    (1, 8, 128, 16, torch.bfloat16), (33, 32, 128, 16, torch.float16), (5, 1, 80, 32, torch.float16),
    (17, 2, 20, 16, torch.bfloat16), (9, 3, 7, 16, torch.float16), (64, 4, 64, 16, torch.float32),
])
@pytest.mark.parametrize("gate", [None, 0, 1])
@pytest.mark.parametrize("native", [True, False])
def test_matches_two_calls(gpu, T, KVH, D, BS, dtype, gate, native, monkeypatch):
    if not native:
        monkeypatch.setattr(ops, "_NATIVE", False)
    g = torch.Generator().manual_seed(T + D)
    B, C = 8, 6
    qkv = torch.randn(T + 2, KVH, 2 * D, generator=g).to(dtype).to(gpu)
    key, value = qkv[..., :D], qkv[..., D:]  # strided rows, two more than slots
    slots = torch.randperm((B + C) * BS, generator=g)[:T].to(gpu)
    hbm = torch.where(slots < B * BS, slots, -1)
    host = torch.where(slots >= B * BS, slots - B * BS, -1)
    if T > 4:
        hbm[0], host[0] = -1, C * BS + 3     # past the host tier: not written
        hbm[1], host[1] = B * BS, -1         # past the HBM tier
    wg = None if gate is None else torch.full((1,), gate, dtype=torch.int32, device=gpu)

    def caches():
        kv = torch.zeros(B, BS, KVH, 2 * D, dtype=dtype, device=gpu)
        return kv, *(pinned_empty((C, KVH, BS, D), dtype, zero=True) for _ in range(2))

    kv, hk, hv = caches()
    ops.reshape_and_cache_tiers(key, value, kv[..., :D], kv[..., D:], hbm, hk, hv, host,
                                write_gate=wg)
    kv2, hk2, hv2 = caches()
    ops.reshape_and_cache(key, value, kv2[..., :D], kv2[..., D:], hbm, write_gate=wg)
    ops.reshape_and_cache(key, value, hk2.transpose(1, 2), hv2.transpose(1, 2), host, write_gate=wg)
    torch.cuda.synchronize()
    assert torch.equal(kv, kv2) and torch.equal(hk, hk2) and torch.equal(hv, hv2)
    assert bool(kv.any() or hk.any()) == (gate != 1)
