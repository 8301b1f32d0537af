"""Decode launches whose rows are cut by their lengths on the device
(balanced_task in decode_tiled.h) against the float64 oracle, where that cut
can go wrong: one row and rows on both sides of a 64-lane group, empty and
one-token rows among long ones, rows longer than the 256 blocks a task holds,
parts forced down to the smallest size, every kernel family, one tier and two,
an order that leaves rows out, range errors, and the entry points with and
without arrival counters. Bars of test_gpu_decode: fp32 out 2e-3 (fp32 KV
5e-5), lse 1e-4 relative."""

from __future__ import annotations

import ctypes
import math

import pytest
import torch

import oracle
from tests.test_gpu_decode import assert_lse_close, assert_out_close
from tests.test_gpu_split_fused import run_fused, two_tier_case
from vllm_fastdecoder_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _case(lens, H, KVH, D, dtype, seed, spare=8):
    """Rows of the given lengths over a shuffled pool, host layout."""
    BS = 16
    g = torch.Generator().manual_seed(seed)
    nb = [-(-x // BS) for x in lens]
    pool = sum(nb) + 1
    perm = torch.randperm(pool, generator=g).to(torch.int32)
    bt = torch.zeros(len(lens), max(nb) + spare, dtype=torch.int32)
    pos = 0
    for i, k in enumerate(nb):
        bt[i, :k] = perm[pos:pos + k]
        pos += k
    q = torch.randn(len(lens), H, D, generator=g).to(dtype)
    kc = torch.randn(pool, KVH, BS, D, generator=g).to(dtype)
    vc = torch.randn(pool, KVH, BS, D, generator=g).to(dtype)
    return q, kc, vc, bt, torch.tensor(lens, dtype=torch.int32)


def _run(case, dev, out=None, lse=None, row_order=None):
    q, kc, vc, bt, lens = case
    n, H, D = q.shape
    out = torch.empty(n, H, D, device=dev) if out is None else out
    lse = torch.empty(H, n, device=dev) if lse is None else lse
    ops.decode_attn(q.to(dev), kc.to(dev), vc.to(dev), bt.to(dev), lens.to(dev),
                    1 / math.sqrt(D), out, lse, row_order=row_order)
    torch.cuda.synchronize()
    return out, lse


def _check(case, out, lse, rows=slice(None)):
    q, kc, vc, bt, lens = case
    ref_out, ref_lse = oracle.decode_attn_host_layout_f64(q, kc, vc, bt, lens,
                                                          1 / math.sqrt(q.shape[2]))
    tol = 5e-5 if q.dtype == torch.float32 else 2e-3
    nz = lens[rows] > 0
    out, lse = out[rows].cpu(), lse[:, rows].cpu()
    assert_out_close(out, ref_out[rows], tol, mask=nz)
    assert_lse_close(lse, ref_lse[:, rows], mask=nz)
    assert torch.all(out[~nz] == 0) and torch.all(torch.isneginf(lse[:, ~nz]))


def _lens(n, seed, hi=900):
    """Rows of 0 to hi tokens: empty, one-token and block-edge rows first."""
    g = torch.Generator().manual_seed(seed)
    lens = torch.randint(0, hi, (n,), generator=g).tolist()
    for k, x in enumerate((hi, 0, 1, 15, 16, 17)):
        if k < n:
            lens[k] = x
    return lens


@pytest.mark.parametrize("H,KVH,D,dtype", [
    (2, 2, 128, torch.float16), (4, 2, 128, torch.bfloat16), (2, 2, 64, torch.bfloat16),
    (2, 2, 80, torch.float16), (4, 2, 256, torch.bfloat16),       # VALU
    (8, 2, 128, torch.bfloat16), (14, 2, 64, torch.float16), (16, 1, 96, torch.bfloat16),  # mm
    (8, 2, 256, torch.bfloat16),                                  # mfma
    (2, 2, 128, torch.float32), (8, 2, 72, torch.float32), (20, 2, 256, torch.float32),  # f32
])
@pytest.mark.parametrize("n", [1, 7, 65])
def test_forced_cuts_match_oracle(gpu, H, KVH, D, dtype, n, monkeypatch):
    """Cuts wherever they can be made: about three parts per row and kv head."""
    monkeypatch.setenv("FD_BALANCE", str(3 * n * KVH))
    case = _case(_lens(n, n + D), H, KVH, D, dtype, seed=n)
    assert ops.balanced_parts(n, H, KVH, D, 16, case[3].shape[1], dtype) > 0
    out, lse = _run(case, gpu)
    _check(case, out, lse)


@pytest.mark.parametrize("n,want", [(1, 1), (2, 512), (63, 70), (64, 256), (65, 66), (130, 512),
                                    (512, 700)])
def test_row_counts_and_part_counts(gpu, n, want, monkeypatch):
    """From fewer parts than cut rows need (they stay whole) to parts of the
    smallest size; row counts around the 64-lane groups, up to the most the
    cut takes."""
    monkeypatch.setenv("FD_BALANCE", str(want))
    case = _case(_lens(n, n, hi=400 if n > 64 else 1500), 8, 1, 128, torch.bfloat16, seed=n)
    _check(case, *_run(case, gpu))


def test_rows_past_one_tasks_blocks(gpu, monkeypatch):
    """One part per row wanted, rows of more than 256 blocks: the parts stop at
    the 256 blocks a task can hold."""
    monkeypatch.setenv("FD_BALANCE", "2")
    case = _case([9000, 33, 4097, 0], 4, 1, 128, torch.float16, seed=5)
    _check(case, *_run(case, gpu))


@pytest.mark.parametrize("H,KVH,D,dtype,bar_out,bar_lse", [
    (8, 8, 128, torch.float16, 2.0e-7, 3.55e-8), (8, 4, 64, torch.bfloat16, 2.1e-7, 3.9e-8),
    (8, 2, 256, torch.bfloat16, 2.4e-7, 3.2e-8), (8, 2, 128, torch.float32, 2.05e-7, 3.8e-8)])
def test_merged_rows_keep_fp32_precision(gpu, H, KVH, D, dtype, bar_out, bar_lse, monkeypatch):
    """Rows of many parts, kernels whose weights are fp32 throughout: distances
    from 64 bits in the 2-norm (2^-24 is 6e-8; the last rounding of a number
    alone is up to 3e-8). Measured with the parts kept as sums: 1.7, 1.6, 2.2,
    1.9e-7 and 3.2, 3.5, 2.9, 3.7e-8; kept as normalised outputs and LSEs: 2.3,
    2.7, 2.7, 2.2e-7 and 3.9, 4.4, 3.5, 4.0e-8. The bars lie between."""
    monkeypatch.setenv("FD_BALANCE", str(16 * 8 * KVH))
    case = _case([1200 + 37 * i for i in range(8)], H, KVH, D, dtype, seed=D + H)
    out, lse = _run(case, gpu)
    q, kc, vc, bt, lens = case
    ref_out, ref_lse = oracle.decode_attn_host_layout_f64(q, kc, vc, bt, lens, 1 / math.sqrt(D))
    assert float((out.cpu().double() - ref_out).norm() / ref_out.norm()) < bar_out
    assert float((lse.cpu().double() - ref_lse).norm() / ref_lse.norm()) < bar_lse


@pytest.mark.parametrize("H,KVH,D,dtype", [(2, 2, 128, torch.float16), (8, 2, 128, torch.bfloat16),
                                           (8, 2, 256, torch.bfloat16), (2, 2, 128, torch.float32)])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_bad_values_of_a_weightless_part_show(gpu, H, KVH, D, dtype, bad, monkeypatch):
    """A V entry that is no number in a part whose weight underflows: as in a
    row of one task (and in 64 bits), its dimension is no number either."""
    q, kc, vc, bt, lens = _case([640], H, KVH, D, dtype, seed=6)
    q.fill_(1.0)
    kc.fill_(14.0)
    for b in bt[0, :8]:  # the row's first 128 tokens: scores about 300 lower
        kc[int(b)] = -14.0
    vc[int(bt[0, 3]), :, 5, 9] = bad
    for parts in ("0", str(8 * KVH)):
        monkeypatch.setenv("FD_BALANCE", parts)
        out, lse = _run((q, kc, vc, bt, lens), gpu)
        assert not torch.isfinite(out[..., 9]).any() and torch.isfinite(lse).all()
        keep = torch.arange(D) != 9
        assert torch.isfinite(out[..., keep]).all()


def test_chosen_by_the_plan(gpu):
    """A small grouped-query batch takes the cut by itself, and gives the same
    bits on every call (the counters are back at zero) and in any order; a
    batch of one row per CU does not take it."""
    case = _case([900, 2500, 64, 700, 3000], 32, 8, 128, torch.bfloat16, seed=9)
    assert ops.balanced_parts(5, 32, 8, 128, 16, case[3].shape[1], torch.bfloat16) > 0
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert ops.balanced_parts(cus // 8, 32, 8, 128, 16, 256, torch.bfloat16) == 0
    first = _run(case, gpu)
    _check(case, *first)
    for order in (None, torch.tensor([4, 1, 0, 3, 2], dtype=torch.int32)):
        again = _run(case, gpu, row_order=order)
        assert torch.equal(again[0], first[0]) and torch.equal(again[1], first[1])


def test_order_entries_outside_the_rows_are_skipped(gpu, monkeypatch):
    monkeypatch.setenv("FD_BALANCE", "64")
    case = _case([900, 500, 64, 700], 8, 2, 128, torch.bfloat16, seed=10)
    out = torch.full((4, 8, 128), 7.0, device=gpu)
    lse = torch.full((8, 4), 7.0, device=gpu)
    _run(case, gpu, out, lse, row_order=torch.tensor([3, -1, 0, 9], dtype=torch.int32))
    _check(case, out, lse, rows=[0, 3])
    assert torch.all(out[[1, 2]] == 7.0) and torch.all(lse[:, [1, 2]] == 7.0)


@pytest.mark.parametrize("H,KVH,D", [(8, 2, 128), (2, 2, 128), (8, 2, 256)])
def test_a_row_listed_twice_beside_a_skipped_entry(gpu, H, KVH, D, monkeypatch):
    """Each listing is cut and merged by itself; the launches after it are
    whole again."""
    monkeypatch.setenv("FD_BALANCE", "64")
    case = _case([900, 500, 64, 700, 0], H, KVH, D, torch.bfloat16, seed=13)
    for _ in range(3):
        out = torch.full((5, H, D), 7.0, device=gpu)
        lse = torch.full((H, 5), 7.0, device=gpu)
        _run(case, gpu, out, lse, row_order=torch.tensor([3, -1, 3, 0, 0], dtype=torch.int32))
        _check(case, out, lse, rows=[0, 3])
        rest = [1, 2, 4]
        assert torch.all(out[rest] == 7.0) and torch.all(lse[:, rest] == 7.0)
        _check(case, *_run(case, gpu))


def test_range_errors_stay_in_their_rows(gpu, monkeypatch):
    """A bad block id and a length past the table: NaN in those rows only."""
    monkeypatch.setenv("FD_BALANCE", "96")
    case = _case([900, 800, 700, 600], 8, 2, 128, torch.bfloat16, seed=11, spare=0)
    q, kc, vc, bt, lens = case
    bad_bt, bad_lens = bt.clone(), lens.clone()
    bad_bt[1, 40] = kc.shape[0]
    bad_lens[2] = bt.shape[1] * 16 + 1
    out, lse = _run((q, kc, vc, bad_bt, bad_lens), gpu)
    assert torch.isnan(out[[1, 2]]).all() and torch.isnan(lse[:, [1, 2]]).all()
    _check(case, out, lse, rows=[0, 3])


@pytest.mark.parametrize("H,KVH,dtype", [(4, 4, torch.float16), (8, 2, torch.bfloat16),
                                         (8, 2, torch.float32)])
def test_two_tiers(gpu, H, KVH, dtype, monkeypatch):
    """Cuts anywhere in a row's two block lists, both tiers ending in a partial
    block, against the launch that is not cut this way."""
    c = two_tier_case(9, H, KVH, 128, dtype, seed=3, dev=gpu, gpu_first=False)
    monkeypatch.setenv("FD_BALANCE", "0")
    ref_out, ref_lse = run_fused(c, gpu)
    monkeypatch.setenv("FD_BALANCE", str(30 * KVH))
    out, lse = run_fused(c, gpu)
    assert not torch.equal(out, ref_out)  # another cut: summed in another order
    torch.testing.assert_close(out, ref_out, atol=2e-5, rtol=0)
    torch.testing.assert_close(lse, ref_lse, atol=1e-5, rtol=1e-5)


def _c_call(case, dev, size, counters=None):
    """The C entry point without counters, or with the given ones, a
    workspace of `size` bytes full of ones."""
    q, kc, vc, bt, lens = (x.to(dev) for x in case)
    n, H, D = q.shape
    KVH = kc.shape[1]
    lib = _lib.load_lib()
    ws = torch.full((max(size, 1),), 0xFF, dtype=torch.uint8, device=dev)
    out, lse = torch.empty(n, H, D, device=dev), torch.empty(H, n, device=dev)
    args = (q.data_ptr(), q.stride(0), q.stride(1), kc.data_ptr(), vc.data_ptr(), kc.stride(0),
            kc.stride(1), kc.stride(2), kc.shape[0], bt.data_ptr(), bt.stride(0), bt.shape[1],
            lens.data_ptr(), None, n, H, KVH, D, 16, 1 / math.sqrt(D), _lib.FD_BF16,
            out.data_ptr(), out.stride(0), out.stride(1), _lib.FD_F32, lse.data_ptr(),
            lse.stride(0), ws.data_ptr() if size else None, ctypes.c_size_t(size),
            torch.cuda.current_stream().cuda_stream)
    if counters is None:
        _lib.check(lib.fd_paged_decode_partial(*args))
    else:
        _lib.check(lib.fd_paged_decode_counted(*args, 0, counters.data_ptr()))
    torch.cuda.synchronize()
    return out, lse


def test_entry_points_without_counters(gpu):
    """The C entry points that bring no counters: a workspace of the query's
    size, full of ones, gives the counted call's bits; one that only covers
    the cut by table width (here none) is still taken."""
    case = _case([900, 500, 64], 32, 8, 128, torch.bfloat16, seed=12, spare=0)
    ref = _run(case, gpu)
    need = ops.workspace_bytes(3, 32, 8, 128, 16, case[3].shape[1])
    assert need > 0
    for size in (need, 0):
        out, lse = _c_call(case, gpu, size)
        if size:
            assert torch.equal(out, ref[0]) and torch.equal(lse, ref[1])
        _check(case, out, lse)


@pytest.mark.parametrize("left", [1, 2, 1000])
def test_counts_an_earlier_launch_left_do_not_reach_the_next(gpu, left):
    """Every counter starts with arrivals in it, as launches that overlapped
    on them may leave."""
    case = _case([900, 500, 64], 32, 8, 128, torch.bfloat16, seed=12, spare=0)
    ref = _run(case, gpu)
    need = ops.workspace_bytes(3, 32, 8, 128, 16, case[3].shape[1])
    counters = torch.zeros(_lib.DECODE_COUNTERS // 2, dtype=torch.int64, device=gpu)
    counters += left
    for _ in range(2):
        out, lse = _c_call(case, gpu, need, counters)
        assert torch.equal(out, ref[0]) and torch.equal(lse, ref[1])


@pytest.mark.parametrize("native", [True, False])
def test_graphs_that_share_an_unreserved_workspace(gpu, native, monkeypatch):
    """Two graphs captured on one stream with no workspace reserved, so each
    with scratch of its own: the second is replayed first, then they are in
    turn with eager calls on that stream; every result is the eager one."""
    if not native:
        monkeypatch.setattr(ops, "_NATIVE", False)
    case = _case([900, 2500, 64, 700], 32, 8, 128, torch.bfloat16, seed=21)
    q, kc, vc, bt, lens = (x.to(gpu) for x in case)
    outs = [(torch.empty(4, 32, 128, device=gpu), torch.empty(32, 4, device=gpu)) for _ in range(3)]

    def step(k):
        ops.decode_attn(q, kc, vc, bt, lens, 1 / math.sqrt(128), *outs[k])
        kv = kc.transpose(1, 2), vc.transpose(1, 2)
        ops.paged_decode(q, *kv, bt, lens, 1 / math.sqrt(128), out=outs[k][0], lse=outs[k][1])

    step(2)
    torch.cuda.synchronize()
    ref = [t.clone() for t in outs[2]]
    side = torch.cuda.Stream(device=gpu)
    graphs = [torch.cuda.CUDAGraph() for _ in range(2)]
    for k, g in enumerate(graphs):
        with torch.cuda.graph(g, stream=side):
            step(k)
    for k in (1, 0, 1, 2, 1, 0):
        for t in (t for pair in outs for t in pair):
            t.fill_(7.0)
        if k < 2:
            graphs[k].replay()
        else:
            torch.cuda.synchronize()
            with torch.cuda.stream(side):
                step(2)
        torch.cuda.synchronize()
        assert torch.equal(outs[k][0], ref[0]) and torch.equal(outs[k][1], ref[1]), k


@pytest.mark.parametrize("native", [True, False])
def test_unreserved_graphs_keep_their_scratch(gpu, native, monkeypatch):
    """Two graphs captured on one stream without a reservation, rows cut by
    length: a larger eager call grows the stream's workspace, fresh tensors
    take whatever memory that freed, and both graphs replay at once on two
    streams. They write into none of those tensors and give the eager bits."""
    if not native:
        monkeypatch.setattr(ops, "_NATIVE", False)
    case = _case([900, 2500, 64, 700], 32, 8, 128, torch.bfloat16, seed=22)
    q, kc, vc, bt, lens = (x.to(gpu) for x in case)
    kv = kc.transpose(1, 2), vc.transpose(1, 2)
    outs = [(torch.empty(4, 32, 128, device=gpu), torch.empty(32, 4, device=gpu)) for _ in range(3)]

    def step(k, rep=1):
        out, lse = outs[k] if rep == 1 else (None, None)
        ops.paged_decode(q.repeat(rep, 1, 1), *kv, bt.repeat(rep, 1), lens.repeat(rep),
                         1 / math.sqrt(128), out=out, lse=lse)

    side, other = (torch.cuda.Stream(device=gpu) for _ in range(2))
    with torch.cuda.stream(side):
        step(2)
    torch.cuda.synchronize()
    ref = [t.clone() for t in outs[2]]
    graphs = [torch.cuda.CUDAGraph() for _ in range(2)]
    for k, g in enumerate(graphs):
        with torch.cuda.graph(g, stream=side):
            step(k)
    size = ops.workspace_bytes(4, 32, 8, 128, 16, bt.shape[1])
    with torch.cuda.stream(side):
        step(2, rep=4)
        assert ops.workspace_bytes(16, 32, 8, 128, 16, bt.shape[1]) > size
        markers = [torch.full((size + 4 * _lib.DECODE_COUNTERS,), 77, dtype=torch.uint8, device=gpu)
                   for _ in range(8)]
    torch.cuda.synchronize()
    for _ in range(3):
        for pair in outs[:2]:
            for t in pair:
                t.fill_(7.0)
        torch.cuda.synchronize()
        for s, g in zip((side, other), graphs):
            with torch.cuda.stream(s):
                g.replay()
        torch.cuda.synchronize()
        for pair in outs[:2]:
            assert torch.equal(pair[0], ref[0]) and torch.equal(pair[1], ref[1])
        assert all(bool((m == 77).all()) for m in markers)
