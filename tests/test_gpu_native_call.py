"""The native call path (csrc/torch/torch_call.cpp) against the checks and
ctypes calls of ops.py it stands in for: the same bits, the same refusals, and
the forms it leaves to Python."""

from __future__ import annotations

import pytest
import torch

from vllm_fastdecoder_amd import ops
from vllm_fastdecoder_amd.pinned import pinned_empty

pytestmark = pytest.mark.gpu

N, H, KVH, D, BS, POOL = 5, 8, 2, 64, 16, 40


def _inputs(dev, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(3)
    kv = torch.randn(POOL, BS, KVH, 2 * D, generator=g).to(dtype).to(dev)
    hk, hv = (pinned_empty((POOL, KVH, BS, D), dtype) for _ in range(2))
    hk.copy_(torch.randn(hk.shape, generator=g))
    hv.copy_(torch.randn(hv.shape, generator=g))
    return dict(
        q=torch.randn(N, H, 2 * D, generator=g).to(dtype).to(dev)[..., :D],  # strided rows
        k=kv[..., :D], v=kv[..., D:], hk=hk, hv=hv, kv=kv,
        bt=torch.stack([torch.randperm(POOL, generator=g)[:24] for _ in range(N)]).int().to(dev),
        lens=torch.tensor([70, 0, 16, 100, 1], dtype=torch.int32, device=dev),
        hbt=torch.stack([torch.randperm(POOL, generator=g)[:3] for _ in range(N)]).int().to(dev),
        hlens=torch.tensor([40, 0, 3, 0, 17], dtype=torch.int32, device=dev),
        order=torch.tensor([3, 0, 2, 4, 1], dtype=torch.int32, device=dev))


def _outcome(f):
    try:
        return [t.clone() for t in f()]
    except Exception as e:  # the same refusal either way
        return type(e), str(e)


def _both(f, monkeypatch):
    assert ops._native(), "the native call path must be built"
    native = _outcome(f)
    monkeypatch.setattr(ops, "_NATIVE", False)
    plain = _outcome(f)
    monkeypatch.undo()
    if isinstance(plain, tuple):
        assert native == plain
    else:
        assert len(native) == len(plain)
        for a, b in zip(native, plain):
            assert a.dtype == b.dtype and a.stride() == b.stride()
            torch.testing.assert_close(a, b, atol=0, rtol=0, equal_nan=True)
    return native


@pytest.mark.parametrize("form", [
    dict(), dict(order=True), dict(max_seqlen_k=100, total_tokens=187), dict(max_seqlen_k=60),
    dict(max_seqlen_k=-4), dict(total_tokens=-1), dict(out=torch.float32), dict(out=torch.float16),
    dict(lens_cpu=True), dict(bt64=True), dict(order64=True), dict(scale=1), dict(lens_step=True),
    dict(q_transposed=True), dict(grad=True), dict(param=True), dict(bt_width=0), dict(k_short=True),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_paged_decode_forms(gpu, form, dtype, monkeypatch):
    x = _inputs(gpu, dtype)
    q, bt, lens, k = x["q"], x["bt"], x["lens"], x["k"]
    if form.get("q_transposed"):
        q = torch.randn(H, N, D, device=gpu).to(dtype).transpose(0, 1)
    if form.get("grad"):
        q = q.clone().requires_grad_()
    if form.get("param"):
        q = torch.nn.Parameter(q.clone())
    if form.get("lens_cpu"):
        lens = lens.cpu()
    if form.get("lens_step"):
        lens = lens.repeat_interleave(2)[::2]
    if form.get("bt64"):
        bt = bt.long()
    if "bt_width" in form:
        bt = bt[:, :0]
    if form.get("k_short"):
        k = k[:-1]
    order = x["order"] if form.get("order") else None
    if form.get("order64"):
        order = x["order"].long()
    out = torch.empty(N, H, D, dtype=form["out"], device=gpu) if "out" in form else None
    _both(lambda: ops.paged_decode(q, k, x["v"], bt, lens, form.get("scale", 0.125), out=out,
                                   row_order=order, max_seqlen_k=form.get("max_seqlen_k"),
                                   total_tokens=form.get("total_tokens")), monkeypatch)


@pytest.mark.parametrize("form", [dict(), dict(order=True), dict(pageable=True), dict(hbm_host=True),
                                  dict(lens_cpu=True), dict(heads=True), dict(out=torch.float32)])
def test_split_decode_forms(gpu, form):
    """ops.split_decode (which the native path does not carry): every form it
    takes gives the plain form's result, every other is refused."""
    x = _inputs(gpu)
    hk, hv = x["hk"], x["hv"]

    def call(hk=hk, hv=hv, lens=x["lens"], order=None, out=None):
        return ops.split_decode(x["q"], x["k"], x["v"], x["bt"], lens, hk, hv, x["hbt"],
                                x["hlens"], 0.125, out=out, row_order=order)

    ref_out, ref_lse = (t.clone() for t in call())
    nz = (x["lens"] + x["hlens"]) > 0
    assert ref_out[nz].abs().max() > 0.1 and torch.isfinite(ref_lse[:, nz]).all()
    if form.get("pageable") or form.get("heads"):
        bad = (hk.clone(), hv.clone()) if form.get("pageable") else (hk[:, :1], hv[:, :1])
        with pytest.raises(RuntimeError, match="pinned" if form.get("pageable") else "kv heads"):
            call(*bad)
        return
    if form.get("hbm_host"):  # other kernels: 16-bit rounding apart
        out, lse = call(hk.to(gpu), hv.to(gpu))
        torch.testing.assert_close(out, ref_out, atol=2e-2, rtol=0)
        torch.testing.assert_close(lse, ref_lse, atol=1e-5, rtol=1e-5)
        return
    out = torch.empty(N, H, D, dtype=form["out"], device=gpu) if "out" in form else None
    out, lse = call(lens=x["lens"].cpu() if form.get("lens_cpu") else x["lens"],
                    order=x["order"] if form.get("order") else None, out=out)
    assert torch.equal(out.to(ref_out.dtype), ref_out) and torch.equal(lse, ref_lse)


@pytest.mark.parametrize("form", [dict(), dict(host=True), dict(pad=True), dict(gate=True),
                                  dict(dtype="fp8"), dict(wrong=True), dict(slots32=True)])
def test_cache_write_forms(gpu, form, monkeypatch):
    x = _inputs(gpu)
    g = torch.Generator().manual_seed(4)
    T = 7
    rows = torch.randn(2, T + (3 if form.get("pad") else 0), KVH, D + (8 if form.get("wrong") else 0),
                       generator=g).to(torch.bfloat16).to(gpu)
    slots = torch.tensor([5, -1, 33, 600, 99, 10 ** 9, 0], device=gpu)
    if form.get("slots32"):
        slots = slots.int()
    gate = torch.ones(1, dtype=torch.int32, device=gpu) if form.get("gate") else None

    def write():
        err = torch.zeros(1, dtype=torch.int32, device=gpu)
        if form.get("host"):
            k, v = (torch.zeros_like(t) for t in (x["hk"], x["hv"]))
            k, v = (pinned_empty(t.shape, t.dtype, zero=True) for t in (k, v))
            views = k.transpose(1, 2), v.transpose(1, 2)
        else:
            kv = torch.zeros_like(x["kv"])
            k, v = kv[..., :D], kv[..., D:]
            views = k, v
        ops.reshape_and_cache(rows[0], rows[1], *views, slots, form.get("dtype", "auto"),
                              error_count=err, write_gate=gate)
        torch.cuda.synchronize()
        return k.contiguous(), v.contiguous(), err

    got = _both(write, monkeypatch)
    if not form:
        assert int(got[2]) == 1 and bool(got[0].any())


def test_modes_and_wrappers_are_left_to_python(gpu):
    """Under a torch-function or dispatch mode, and for functorch wrappers, the
    native path takes nothing (Python's own path then meets the mode)."""
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    class Fn(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    native, x = ops._native(), _inputs(gpu)

    def call(q):
        return native.paged_decode(q, x["k"], x["v"], x["bt"], x["lens"], 0.125, None, None, None,
                                   None, None)

    assert call(x["q"]) is not None
    for mode in (Fn, Dispatch):
        with mode():
            assert call(x["q"]) is None
    seen = []
    torch.func.vmap(lambda q: (seen.append(call(q)), q)[1])(x["q"][None])
    assert seen == [None]
