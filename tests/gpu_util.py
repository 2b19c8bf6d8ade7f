"""Helpers shared by the GPU parity tests (host-side conversions only)."""

import ctypes
from types import SimpleNamespace

import numpy as np
import torch

from oracle import nf4 as onf4
from soupsuck_amd import _lib


class _NtPlan(ctypes.Structure):
    _fields_ = [("cfg", ctypes.c_int), ("splits", ctypes.c_int64), ("k_split", ctypes.c_int64)]


def nt_plan(m, n, k, layout=0, split=True):
    """(configuration, splits) that the dense kernels take for an M x N x K product (ss::nt_plan in
    csrc/gemm_nt.hip; pure host code): layout bit 0 / 1 for a K-major A / B, split=False
    without scratch."""
    plan = _lib.load()._ZN2ss7nt_planElllim
    plan.restype = _NtPlan
    plan.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_int, ctypes.c_size_t]
    got = plan(m, n, k, layout, ctypes.c_size_t(-1).value if split else 0)
    return got.cfg, got.splits


def device_state(state, device):
    """QuantState-like namespace (bitsandbytes field names) from an oracle NF4State."""
    second = SimpleNamespace(
        blocksize=256, dtype=torch.float32, nested=False,
        code=torch.from_numpy(np.ascontiguousarray(state.code2)).to(device),
        absmax=torch.from_numpy(np.ascontiguousarray(state.absmax2)).to(device))
    packed = torch.from_numpy(np.ascontiguousarray(state.packed)).to(device).view(-1, 1)
    qs = SimpleNamespace(
        quant_type="nf4", blocksize=64, dtype=torch.float16, nested=True,
        shape=tuple(int(d) for d in state.shape),
        absmax=torch.from_numpy(np.ascontiguousarray(state.qabs)).to(device),
        state2=second,
        offset=torch.from_numpy(np.ascontiguousarray(state.offset)).to(device))
    return packed, qs


def random_weight(n, k, seed, scale=0.02):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((n, k), dtype=np.float32) * scale).astype(np.float16)


def quantized(n, k, seed):
    """(oracle state, decoded fp16 weight) of a seeded N(0, 0.02) weight."""
    state = onf4.quantize_nested(random_weight(n, k, seed))
    return state, state.decode()


def bits(t):
    return t.detach().contiguous().cpu().view(torch.int16).numpy()


def np16(t):
    return t.detach().cpu().numpy()


def rel_norm(actual, expected):
    a = np.asarray(actual, np.float64)
    e = np.asarray(expected, np.float64)
    return float(np.linalg.norm(a - e) / max(np.linalg.norm(e), 1e-300))
