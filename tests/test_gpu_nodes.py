"""The C++ autograd nodes (csrc/autograd.cpp), which eager calls take, against the
Python nodes, which tracers record: whole values over the forms a call can have, and
the ways autograd is used around a custom function."""

from __future__ import annotations

import pytest
import torch

from machinelearning_amd import flash_cuda as fc
from machinelearning_amd import prologue as pro

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _library():
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    assert fc.is_available(), fc.unavailable_reason()
    yield


def _qkv(B=2, T=70, H=4, Hkv=2, D=64, dtype=torch.bfloat16, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(B, T, h, D, device="cuda", generator=g).to(dtype) for h in (H, Hkv, Hkv, H)]


FORMS = {
    "causal": {}, "d128_residual": dict(D=128), "f32": dict(dtype=torch.float32),
    "f32_sinks": dict(dtype=torch.float32, window=20, sinks=3),
    "f16_sinks": dict(dtype=torch.float16, window=20, sinks=3),
    "blocks": dict(block=16), "noncausal": dict(causal=False), "gate": dict(gate=True),
    "gate_f32": dict(gate=True, dtype=torch.float32), "lse_only": dict(use="lse"),
    "both": dict(use="both"), "strided_do": dict(strided=True),
    "only_k": dict(needs="k"), "only_gate": dict(gate=True, needs="z"), "one_row": dict(T=1),
}


@pytest.mark.parametrize("form", list(FORMS))
def test_same_bits_as_the_python_node(form):
    f = FORMS[form]
    q, k, v, do = _qkv(T=f.get("T", 70), D=f.get("D", 64), dtype=f.get("dtype", torch.bfloat16))
    z = torch.randn(q.shape[:3], device="cuda") if f.get("gate") else None
    if f.get("strided"):
        do = torch.cat([do, do], -1)[..., ::2]
    dl = torch.randn(q.shape[0], q.shape[2], q.shape[1], device="cuda")
    args = (f.get("causal", True), f.get("window", 0), f.get("sinks", 0), q.shape[-1] ** -0.5)
    res = []
    for node in (fc._apply, fc._AttnFn.apply):
        xs = {n: t.detach().requires_grad_(n in f.get("needs", "qkvz"))
              for n, t in (("q", q), ("k", k), ("v", v), ("z", z)) if t is not None}
        o, lse = node(xs["q"], xs["k"], xs["v"], *args, xs.get("z"), f.get("block", 0))
        outs, gos = {"lse": ((lse,), (dl,)), "both": ((o, lse), (do, dl))}.get(
            f.get("use"), ((o,), (do,)))
        leaves = [t for t in xs.values() if t.requires_grad]
        res.append((o.detach(), lse.detach(), *torch.autograd.grad(outs, leaves, gos)))
    assert len(res[0]) == len(res[1])
    for a, b in zip(*res):
        assert a.dtype == b.dtype and a.stride() == b.stride() and torch.equal(a, b)


@pytest.mark.parametrize("norm,rope,dtype,out", [
    (True, True, torch.bfloat16, torch.bfloat16), (True, False, torch.float32, torch.bfloat16),
    (False, True, torch.float16, torch.float32), (False, False, torch.float32, torch.float32)])
def test_prologue_same_bits_as_the_python_node(norm, rope, dtype, out):
    x, _, _, _ = _qkv(dtype=dtype)
    g = torch.randn(x.shape, device="cuda").to(out)
    w = torch.randn(64, device="cuda") if norm else None
    cs = [torch.randn(70, 64, device="cuda") for _ in range(2)] if rope else [None, None]
    res = []
    for node in ("cpp", "python"):
        xr = x.detach().requires_grad_()
        wr = w.detach().requires_grad_() if norm else None
        if node == "cpp":
            y = pro.qk_norm_rope(xr, wr, *cs, 1e-6, out)
        else:
            y = pro._ProFn.apply(xr, wr, *cs, 1e-6, out)
        res.append((y.detach(), *torch.autograd.grad(y, [xr] + ([wr] if norm else []), g)))
    for a, b in zip(*res):
        assert a.dtype == b.dtype and torch.equal(a, b)


def test_no_grad_and_frozen_inputs_record_nothing():
    q, k, v, _ = _qkv()
    o, lse = fc.attn(q, k, v)
    assert o.grad_fn is None and not lse.requires_grad
    q.requires_grad_()
    with torch.no_grad():
        assert fc.attn(q, k, v)[0].grad_fn is None
    with torch.inference_mode():
        assert not fc.attn(q, k, v)[0].requires_grad
    assert fc.attn(q, k, v)[0].requires_grad


def test_second_differentiation_and_second_backward_are_refused():
    q, k, v, do = _qkv()
    q.requires_grad_()
    do.requires_grad_()
    for node in (fc._apply, fc._AttnFn.apply):
        o, _ = node(q, k, v, True, 0, 0, 0.125, None, 0)
        dq, = torch.autograd.grad(o, q, do, create_graph=True)
        with pytest.raises(RuntimeError, match="once_differentiable"):
            dq.sum().backward()
    o, _ = fc.attn(q, k, v)
    o.sum().backward()
    with pytest.raises(RuntimeError, match="second time"):
        o.sum().backward()


def test_saved_tensor_hooks_and_modified_inputs():
    q, k, v, do = _qkv()
    q.requires_grad_()
    want, = torch.autograd.grad(fc.attn(q, k, v)[0], q, do)
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(
            lambda t: (seen.append(tuple(t.shape)), t.cpu())[1], lambda t: t.cuda()):
        o, _ = fc.attn(q, k, v)
    assert {tuple(q.shape), tuple(k.shape)} <= set(seen) and len(seen) == 5   # q k v O LSE
    assert torch.equal(torch.autograd.grad(o, q, do)[0], want)
    o, _ = fc.attn(q, k, v)
    k.add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(o, q, do)


def test_transforms_are_refused_and_traces_run():
    q, k, v, _ = _qkv(B=1)
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda a: fc.attn(a, k, v)[0])(torch.stack([q, q]))
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda a: fc.attn(a, k, v)[0].float().sum())(q)
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(q, q)
        with pytest.raises(RuntimeError):
            fc.attn(dual, k, v)
    traced = torch.jit.trace(lambda a, b, c: fc.attn(a, b, c)[0], (q, k, v))
    q2, k2, v2, _ = _qkv(B=1, seed=3)
    assert torch.equal(traced(q2, k2, v2), fc.attn(q2, k2, v2)[0])


def test_without_the_cpp_nodes_everything_runs_on_the_python_ones(monkeypatch, caplog):
    """A missing or foreign _mi_torch.so costs host time, not the library: attention,
    prologue and decode run, with the same bits."""
    import sys
    import machinelearning_amd as pkg
    from machinelearning_amd.decode import attn_cached

    def step():
        q, k, v, do = _qkv()
        q.requires_grad_()
        o, lse = fc.attn(q, k, v)
        dq, = torch.autograd.grad(o, q, do)
        y = pro.qk_norm_rope(do, torch.ones(64, device="cuda"), None, None)
        with torch.no_grad():
            return [o.detach(), lse.detach(), dq, y, attn_cached(q, k, v, {}, False, True)]
    want = step()
    monkeypatch.delattr(pkg, "_mi_torch")
    monkeypatch.setitem(sys.modules, "machinelearning_amd._mi_torch", None)
    for name, value in (("_lib", None), ("_ext", None), ("_load_attempted", False)):
        monkeypatch.setattr(fc, name, value)
    with caplog.at_level("WARNING"):
        assert fc.is_available(), fc.unavailable_reason()
    assert fc._ext is None and "autograd nodes did not load" in caplog.text
    assert all(torch.equal(a, b) for a, b in zip(step(), want))


@pytest.mark.parametrize("node", ["attn", "prologue"])
def test_the_nodes_release_the_gil(node):
    """Other Python threads run while a node allocates and launches. The switch interval is
    set so long that the second thread, which wakes from a sleep, gets the GIL only
    where the call gives it up."""
    import sys
    import threading
    import time
    q, k, v, do = _qkv()
    call = {"attn": lambda: fc._ext.attn(q, k, v, None, True, 0, 0, 0.125, 0, False),
            "prologue": lambda: fc._ext.prologue(do, None, None, None, 1e-6, 2)}[node]
    call()
    turns, stop = [0], threading.Event()

    def other():
        while not stop.is_set():
            turns[0] += 1
            time.sleep(1e-4)
    thread = threading.Thread(target=other)
    interval = sys.getswitchinterval()
    try:
        sys.setswitchinterval(1000.0)
        thread.start()
        time.sleep(0.01)
        before = turns[0]
        kept = []                                # freeing a tensor may give the GIL up too
        for _ in range(8000):
            kept.append(call())
            if turns[0] > before:
                break
        gained = turns[0] - before
    finally:
        sys.setswitchinterval(interval)
        stop.set()
        thread.join()
    assert gained > 0
