"""The native autograd nodes against the Python nodes they stand for: same kernels on the
same operands, so outputs and gradients are bit-identical, and the same refusals."""

import sys
import threading
import time

import pytest
import torch

from soupsuck_amd import _lib, lora
from soupsuck_amd.bnb_compat import matmul_4bit, quantize_4bit
from soupsuck_amd.kernels.add_rmsnorm import add_rms_norm
from soupsuck_amd.kernels.rmsnorm import rms_norm
from soupsuck_amd.native import nodes

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _randn(*shape, dtype=torch.float16, seed=0):
    gen = torch.Generator().manual_seed(seed)
    return torch.randn(shape, generator=gen).to(dtype).to(DEV)


def _weight(n, k):
    return quantize_4bit(_randn(n, k, seed=9) * 0.02, blocksize=64, compress_statistics=True,
                         quant_type="nf4")


def _linear(t, n=192, k=128, biased=True):
    packed, state = _weight(n, k)
    bias = _randn(n, seed=3) if biased else None
    return [_randn(1, t, k, seed=1)], lambda x: matmul_4bit(x, packed, state, bias=bias)


def _linear_unbiased(t):
    return _linear(t, biased=False)


def _linear_plain_path(t):
    return _linear(t, n=96, k=80)       # K % 64 != 0: the Python node on both sides


def _norm(t):
    return ([_randn(t, 256, dtype=torch.float32), _randn(256, seed=2)],
            lambda x, w: rms_norm(x, w, 1e-6))


def _norm_rows(t):                       # rows of a wider matrix
    base = _randn(t, 512)
    return [base[:, :256]], lambda x: rms_norm(x, _randn(256, seed=2), 1e-6)


def _norm_add(t):
    return ([_randn(t, 256), _randn(t, 256, seed=4), _randn(256, seed=2)],
            lambda r, d, w: add_rms_norm(r, d, w, 1e-6))


def _norm_residual_only(t):              # no gradient reaches y: dw is zero
    args, fn = _norm_add(t)
    return args, lambda *a: fn(*a)[0]


def _qlora(t, p=0.0, dtype=torch.float16):
    packed, state = _weight(192, 128)
    return ([_randn(t, 128), _randn(16, 128, dtype=dtype, seed=5) * 0.1,
             _randn(192, 16, dtype=dtype, seed=6) * 0.1],
            lambda x, a, b: lora.qlora_projection(x, a, b, packed, state, None, 2.0, p))


def _qlora_dropout(t):
    return _qlora(t, 0.25, torch.float32)


def _run(make, t, python, wrap=None):
    args, fn = make(t)
    args = [a.detach().requires_grad_() for a in args]
    torch.manual_seed(11)
    if python:
        _lib.hooks["none"] = None    # any hook selects the Python nodes
    try:
        outs = fn(*args) if wrap is None else wrap(fn, args)
        outs = outs if isinstance(outs, tuple) else (outs,)
        grads = torch.autograd.grad(sum((o.float() * (i + 1)).sum() for i, o in enumerate(outs)),
                                    args)
    finally:
        _lib.hooks.pop("none", None)
    return [o.detach() for o in outs], grads


@pytest.mark.parametrize("t", [1, 67])
@pytest.mark.parametrize("make", [_linear, _linear_unbiased, _linear_plain_path, _norm, _norm_rows,
                                  _norm_add, _norm_residual_only, _qlora, _qlora_dropout])
def test_native_node_is_the_python_node(make, t):
    want = _run(make, t, python=True)

    def hooked(fn, args):
        with torch.autograd.graph.saved_tensors_hooks(lambda s: s.cpu(), lambda s: s.to(DEV)):
            return fn(*args)

    for got in (_run(make, t, python=False), _run(make, t, python=False, wrap=hooked)):
        for a, b in zip((*want[0], *want[1]), (*got[0], *got[1])):
            assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b)
    args, fn = make(t)
    with torch.no_grad():
        torch.manual_seed(11)
        outs = fn(*args)
    for a, b in zip(want[0], outs if isinstance(outs, tuple) else (outs,)):
        assert torch.equal(a, b) and not b.requires_grad


@pytest.mark.parametrize("make", [_linear, _norm, _norm_add, _qlora])
def test_native_node_refuses_what_the_python_node_refuses(make):
    args, fn = make(5)
    args = [a.detach().requires_grad_() for a in args]
    out = fn(*args)
    out = out[-1] if isinstance(out, tuple) else out
    seed = torch.ones_like(out, requires_grad=True)
    (first,) = torch.autograd.grad(out, args[0], seed, create_graph=True)
    with pytest.raises(RuntimeError, match="once_differentiable"):
        first.float().sum().backward()
    import torch.autograd.forward_ad as fwd

    with fwd.dual_level(), pytest.raises((RuntimeError, NotImplementedError)):
        fn(fwd.make_dual(args[0].detach(), torch.ones_like(args[0])),
           *[a.detach() for a in args[1:]])
    with pytest.raises((RuntimeError, ValueError)):
        torch.func.vmap(lambda x: fn(x, *[a.detach() for a in args[1:]]))(
            torch.stack([args[0].detach()] * 2))


def _native_call(name):
    """A call of one native entry point with no other Python code in it."""
    native, x = nodes(), _randn(32768, 128)
    if name == "row_norm":
        w = _randn(128, seed=2)
        return lambda: native.row_norm(x, None, w, 1e-6, False)
    packed, state = _weight(192, 128)
    second = state.state2
    weight = (packed, state.absmax, second.absmax, second.code, state.offset, 192, 128)
    if name == "nf4_linear":
        return lambda: native.nf4_linear(x, *weight, None)
    a, b = _randn(16, 128, seed=5), _randn(192, 16, seed=6)
    stream = _lib.stream(x.device)
    ws = lora._gemm_ws(32768, 192, 128, x.device, stream)[0]
    rank_ws = lora._qlora_rank_ws(32768, 192, 128, x.device, stream)
    return lambda: native.qlora(x, a, b, *weight, None, 2.0, None, ws, rank_ws)


@pytest.mark.parametrize("name", ["nf4_linear", "row_norm", "qlora"])
def test_other_threads_run_during_a_native_call(name):
    """The entry points give up the interpreter lock: with a switch interval longer than the
    test, another thread advances only where the calling one lets go of it."""
    call = _native_call(name)
    call()
    turns, stop = [0], threading.Event()

    def other():
        while not stop.is_set():
            turns[0] += 1
            time.sleep(0)

    thread = threading.Thread(target=other)
    interval = sys.getswitchinterval()
    sys.setswitchinterval(60.0)
    try:
        thread.start()          # start() waits for the thread's first turn
        before, kept = turns[0], []
        while turns[0] == before and len(kept) < 600:
            kept.append(call())     # kept: freeing a tensor may give up the lock too
        assert turns[0] > before
    finally:
        stop.set()
        sys.setswitchinterval(interval)
        thread.join()
    torch.cuda.synchronize()
