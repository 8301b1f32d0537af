"""Two-tier launches whose tasks divide their waves between the tiers
(wave_blocks in decode_tiled.h) and read only the valid tokens of a host block
(block_src): host shares from one block to all but one, rows up to the 256
blocks a task holds (past 64 blocks per wave the division does not apply),
stale host rows full of NaN. Bars of test_gpu_split_fused."""

from __future__ import annotations

import math

import pytest
import torch

import oracle
from tests.test_gpu_decode import assert_lse_close, assert_out_close
from vllm_fastdecoder_amd import ops
from vllm_fastdecoder_amd.pinned import pinned_empty

pytestmark = pytest.mark.gpu

# (HBM blocks, host blocks) of each row, and the tokens of its last host block
ROWS = [(1, 1, 1), (1, 40, 16), (40, 1, 3), (3, 3, 15), (20, 11, 7), (11, 20, 9), (192, 63, 5),
        (193, 63, 16), (63, 192, 1), (128, 128, 8), (0, 5, 2), (5, 0, 16), (0, 0, 16)]


@pytest.mark.parametrize("split", ["256", "32"])
@pytest.mark.parametrize("H,KVH,D,dtype", [(2, 2, 128, torch.float16), (4, 1, 128, torch.bfloat16),
                                           (2, 1, 256, torch.float16), (2, 2, 64, torch.float32)])
def test_tier_shares(gpu, H, KVH, D, dtype, split, monkeypatch):
    monkeypatch.setenv("FD_SPLIT_BLOCKS", split)
    BS, n = 16, len(ROWS)
    g = torch.Generator().manual_seed(D + H)
    G, C = sum(r[0] for r in ROWS), sum(r[1] for r in ROWS)
    W = max(a + b for a, b, _ in ROWS)
    pool_k = torch.randn(G + C, KVH, BS, D, generator=g).to(dtype)
    pool_v = torch.randn(G + C, KVH, BS, D, generator=g).to(dtype)
    bt_g, bt_c, full = (torch.zeros(n, W, dtype=torch.int32) for _ in range(3))
    lens_g, lens_c = [], []
    pg, pc = torch.randperm(G, generator=g).int(), torch.randperm(C, generator=g).int()
    for i, (a, b, last) in enumerate(ROWS):
        bt_g[i, :a], pg = pg[:a], pg[a:]
        bt_c[i, :b], pc = pc[:b], pc[b:]
        full[i, :a], full[i, a:a + b] = bt_g[i, :a], bt_c[i, :b] + G
        lens_g.append(a * BS)
        lens_c.append((b - 1) * BS + last if b else 0)
        if b and last < BS:
            pool_k[full[i, a + b - 1], :, last:] = float("nan")
            pool_v[full[i, a + b - 1], :, last:] = float("nan")
    lens = torch.tensor([x + y for x, y in zip(lens_g, lens_c)], dtype=torch.int32)
    q = torch.randn(n, H, D, generator=g).to(dtype)
    kv = torch.cat([pool_k[:G].transpose(1, 2), pool_v[:G].transpose(1, 2)], -1).contiguous().to(gpu)
    hk, hv = pinned_empty((C, KVH, BS, D), dtype), pinned_empty((C, KVH, BS, D), dtype)
    hk.copy_(pool_k[G:])
    hv.copy_(pool_v[G:])
    out = torch.empty(n, H, D, device=gpu)
    out, lse = ops.split_decode(
        q.to(gpu), kv[..., :D], kv[..., D:], bt_g.to(gpu),
        torch.tensor(lens_g, dtype=torch.int32, device=gpu), hk, hv, bt_c.to(gpu),
        torch.tensor(lens_c, dtype=torch.int32, device=gpu), 1 / math.sqrt(D), out=out)
    torch.cuda.synchronize()
    ref_out, ref_lse = oracle.decode_attn_host_layout_f64(q, pool_k, pool_v, full, lens,
                                                          1 / math.sqrt(D))
    nz = lens > 0
    assert_out_close(out, ref_out, 5e-5 if dtype == torch.float32 else 2e-3, mask=nz)
    assert_lse_close(lse, ref_lse, mask=nz)
    assert torch.all(out[~nz.to(gpu)] == 0) and torch.all(torch.isneginf(lse[:, ~nz.to(gpu)]))
