"""Two-tier launches: tasks that divide their waves between the tiers
(wave_blocks in decode_tiled.h), host blocks read only as far as they hold
tokens (block_src), and host workers that take the host tier alone
(balanced_task, decode_mm_tiers_kernel): host shares from one block to all but
one, rows up to the 256 blocks a task holds (past 64 blocks per wave the
division does not apply), stale host rows full of NaN, one worker taking every
part in turn. Bars of test_gpu_split_fused."""

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


def _run(gpu, H, KVH, D, dtype, rows, row_order=None, bad_row=None):
    BS, n = 16, len(rows)
    g = torch.Generator().manual_seed(D + H)
    G, C = sum(r[0] for r in rows), sum(r[1] for r in rows)
    W = max(a + b for a, b, _ in rows)
    pool_k = torch.randn(G + C, KVH, BS, D, generator=g).to(dtype)
    pool_v = torch.randn(G + C, KVH, BS, D, generator=g).to(dtype)
    bt_g, bt_c, full = (torch.zeros(n, max(W, 1), dtype=torch.int32) for _ in range(3))
    lens_g, lens_c = [], []
    pg, pc = torch.randperm(G, generator=g).int(), torch.randperm(C, generator=g).int()
    for i, (a, b, last) in enumerate(rows):
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
    if bad_row is not None:  # a host block id past the host cache
        bt_c[bad_row, 0] = C + 1
    out = torch.full((n, H, D), 7.0, device=gpu)
    lse = torch.full((H, n), 7.0, device=gpu)
    ops.split_decode(
        q.to(gpu), kv[..., :D], kv[..., D:], bt_g.to(gpu),
        torch.tensor(lens_g, dtype=torch.int32, device=gpu), hk, hv, bt_c.to(gpu),
        torch.tensor(lens_c, dtype=torch.int32, device=gpu), 1 / math.sqrt(D), out=out, lse=lse,
        row_order=row_order)
    torch.cuda.synchronize()
    ref_out, ref_lse = oracle.decode_attn_host_layout_f64(q, pool_k, pool_v, full, lens,
                                                          1 / math.sqrt(D))
    return out, lse, ref_out, ref_lse, lens


def _plan(H, KVH, D, dtype, rows):
    """The launch of _run's call (tables as wide as the longest row)."""
    W = max(a + b for a, b, _ in rows)
    return ops.split_plan_info(len(rows), H, KVH, D, 16, W, W, dtype)


def _check(got, dtype, rows=None):
    out, lse, ref_out, ref_lse, lens = got
    rows = list(range(len(lens))) if rows is None else rows
    nz = lens[rows] > 0
    out, lse = out.cpu()[rows], lse.cpu()[:, rows]
    assert_out_close(out, ref_out[rows], 5e-5 if dtype == torch.float32 else 2e-3, mask=nz)
    assert_lse_close(lse, ref_lse[:, rows], mask=nz)
    assert torch.all(out[~nz] == 0) and torch.all(torch.isneginf(lse[:, ~nz]))


@pytest.mark.parametrize("divided", ["1", "0"])
@pytest.mark.parametrize("split", ["256", "32"])
@pytest.mark.parametrize("H,KVH,D,dtype", [(2, 2, 128, torch.float16), (4, 1, 128, torch.bfloat16),
                                           (2, 1, 256, torch.float16), (2, 2, 64, torch.float32)])
def test_tier_shares(gpu, H, KVH, D, dtype, split, divided, monkeypatch):
    monkeypatch.setenv("FD_TIER_WAVES", divided)
    monkeypatch.setenv("FD_SPLIT_BLOCKS", split)
    _check(_run(gpu, H, KVH, D, dtype, ROWS), dtype)


@pytest.mark.parametrize("workers", ["1", "32"])
@pytest.mark.parametrize("H,KVH,D,dtype", [
    (2, 2, 128, torch.float16), (6, 2, 128, torch.bfloat16), (4, 1, 128, torch.bfloat16),
    (7, 1, 48, torch.float16), (16, 1, 64, torch.bfloat16), (10, 2, 80, torch.float16)])
def test_host_workers(gpu, H, KVH, D, dtype, workers, monkeypatch):
    """Rows of every tier share, one row, and 64 (the most the workers take);
    the same bits on a second call and in any order, from a workspace of the
    call's own size as from a larger one."""
    monkeypatch.setenv("FD_HOST_WGS", workers)
    for rows in (ROWS, ROWS[:1], ROWS * 5):
        wgs = _plan(H, KVH, D, dtype, rows)["host_workgroups"]
        assert wgs == (int(workers) if len(rows) <= 64 else 0), rows
    monkeypatch.setattr(ops, "WORKSPACE", ops._Workspace())
    first = _run(gpu, H, KVH, D, dtype, ROWS)
    _check(first, dtype)
    order = torch.randperm(len(ROWS), generator=torch.Generator().manual_seed(2)).int()
    again = _run(gpu, H, KVH, D, dtype, ROWS, row_order=order)
    assert torch.equal(again[0], first[0]) and torch.equal(again[1], first[1])
    ops.WORKSPACE.get(gpu, 1 << 24)
    again = _run(gpu, H, KVH, D, dtype, ROWS)
    assert torch.equal(again[0], first[0]) and torch.equal(again[1], first[1])
    _check(_run(gpu, H, KVH, D, dtype, [(30, 9, 4)]), dtype)
    _check(_run(gpu, H, KVH, D, dtype, [(i % 5, (3 * i) % 7, 1 + i % 16) for i in range(64)]), dtype)


def test_host_workers_leave_out_and_range_errors(gpu, monkeypatch):
    monkeypatch.setenv("FD_HOST_WGS", "32")
    monkeypatch.setattr(ops, "WORKSPACE", ops._Workspace())
    assert _plan(4, 1, 128, torch.bfloat16, ROWS)["host_workgroups"] == 32
    rows = list(range(len(ROWS)))
    order = torch.tensor([r if r not in (2, 5) else -1 for r in rows], dtype=torch.int32)
    got = _run(gpu, 4, 1, 128, torch.bfloat16, ROWS, row_order=order)
    _check(got, torch.bfloat16, [r for r in rows if r not in (2, 5)])
    assert torch.all(got[0][[2, 5]] == 7.0) and torch.all(got[1][:, [2, 5]] == 7.0)
    got = _run(gpu, 4, 1, 128, torch.bfloat16, ROWS, bad_row=4)
    _check(got, torch.bfloat16, [r for r in rows if r != 4])
    assert torch.isnan(got[0][4]).all() and torch.isnan(got[1][:, 4]).all()


@pytest.mark.parametrize("n", [13, 70])  # with host workers and past their 64 rows
@pytest.mark.parametrize("H,KVH,D,dtype", [
    (8, 2, 128, torch.bfloat16), (8, 2, 128, torch.float16), (16, 2, 96, torch.bfloat16),
    (4, 4, 128, torch.bfloat16), (34, 1, 64, torch.bfloat16)])
def test_weights_keep_fp32_precision(gpu, H, KVH, D, dtype, n):
    """An fp32 out over a pinned host tier, the matrix-core kernels included:
    within 4e-7 of 64 bits in the 2-norm (fp32 arithmetic: 1.5-2.5e-7 measured;
    bf16 weights kept to 16 bits: 2e-6)."""
    rows = [((3 * i) % 40 + 4, i % 9 + 1, i % 16 + 1) for i in range(n)]
    out, _, ref_out, _, _ = _run(gpu, H, KVH, D, dtype, rows)
    assert float((out.cpu().double() - ref_out).norm() / ref_out.norm()) < 4e-7
