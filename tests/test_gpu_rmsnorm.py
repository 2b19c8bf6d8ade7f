"""GPU parity of the standalone RMSNorm (ss_rmsnorm_fwd + the add-RMSNorm backward).

Bar (solution/tests/test_rmsnorm.py:10-11): y and the gradients within fp32
1e-5 / fp16 2e-3 (rtol = atol) of oracle/rmsnorm.py, evaluated with the
residual term zero (s = x exactly: adding an fp16/fp32 zero and casting back
is the identity up to the sign of zero, which the numeric comparison
ignores); fp16 outputs also differ from it on at most 1/1000 entries, by at
most two fp16 ulps (after the reference's half-store rule, :14-37: a flipped
rounding of q, then of w q); dgamma within the same
magnitude-scaled fp32 budget as the add-RMSNorm tests.  Cases: Qwen2.5-1.5B
hidden 1536 at 826 and 4096 rows, the reference's dtype grid, a 2-D
row-strided input, zero rows.
"""

import numpy as np
import pytest
import torch

from oracle import rmsnorm as ormsnorm
from soupsuck_amd.kernels.rmsnorm import rms_norm
from tests.gpu_util import np16

pytestmark = pytest.mark.gpu

F32_TOL = dict(rtol=1e-5, atol=1e-5)
F16_TOL = dict(rtol=2e-3, atol=2e-3)
NP = {torch.float16: np.float16, torch.float32: np.float32}


def _case(device, shape, xdt, wdt, out_dtype, train_weight, strided=False, seed=7):
    print(f"case rmsnorm shape={shape} x={xdt} w={wdt} out={out_dtype} dw={train_weight} "
          f"strided={strided}", flush=True)
    rng = np.random.default_rng(seed)
    h = shape[-1]
    x = rng.standard_normal(shape).astype(NP[xdt])
    w = (1 + 0.1 * rng.standard_normal(h)).astype(NP[wdt])
    if strided:
        big = torch.zeros((shape[0], h + 64), dtype=xdt)
        big[:, 8:8 + h] = torch.from_numpy(x)
        xt = big.to(device)[:, 8:8 + h].requires_grad_()
        assert not xt.is_contiguous()
    else:
        xt = torch.from_numpy(x).to(device).requires_grad_()
    wt = torch.from_numpy(w).to(device).requires_grad_(train_weight)
    y = rms_norm(xt, wt, 1e-6, out_dtype)
    zero = np.zeros_like(x)
    _, ey, rstd = ormsnorm.add_rmsnorm_forward(x, zero, w, 1e-6, out_dtype is not None)
    assert y.dtype == torch.from_numpy(ey).dtype
    all32 = xdt == torch.float32 and wdt == torch.float32 and out_dtype is None
    tol = F32_TOL if all32 else F16_TOL
    got = np16(y).astype(np.float64)
    np.testing.assert_allclose(got, ey.astype(np.float64), **tol)
    if ey.dtype == np.float16:
        ulp = np.spacing(np.abs(ey)).astype(np.float64)
        diff = np.abs(got - ey.astype(np.float64))
        # A last-bit difference of the fp32 rstd can flip the rounding of q, and
        # w q rounds again: at most two output ulps, on at most 1/1000 entries.
        assert (diff <= 2 * ulp).all()
        assert (diff > 0).sum() * 1000 <= diff.size
    gy = rng.standard_normal(shape).astype(ey.dtype)
    y.backward(torch.from_numpy(gy).to(device))
    exact = np.promote_types(x.dtype, w.dtype)
    dx, _, dg = ormsnorm.add_rmsnorm_backward(None, gy, x, w, rstd, x.dtype, x.dtype, exact)
    assert xt.grad.dtype == xt.dtype
    np.testing.assert_allclose(np16(xt.grad).astype(np.float64), dx.astype(np.float64),
                               **(F32_TOL if all32 else F16_TOL))
    if train_weight:
        gw = np16(wt.grad).astype(np.float64)
        if not all32:
            np.testing.assert_allclose(gw, dg, **F16_TOL)
        else:
            q = (x.astype(np.float64) * rstd[..., None]).astype(x.dtype).astype(np.float64)
            magnitude = np.abs(gy.astype(np.float64) * q).reshape(-1, h).sum(0)
            budget = 1e-5 * np.abs(dg) + 32 * np.finfo(np.float32).eps * magnitude
            assert np.all(np.abs(gw - dg) <= budget)


@pytest.mark.parametrize("rows", [826, 4096])
def test_qwen_hidden_fp16_fused_output(device, rows):
    _case(device, (rows, 1536), torch.float16, torch.float16, torch.float16, True)


@pytest.mark.parametrize("h", [3584, 6144])
def test_wide_rows_trained_weight(device, h):
    print(f"case rmsnorm h={h}", flush=True)
    _case(device, (300, h), torch.float16, torch.float16, torch.float16, True)


@pytest.mark.parametrize("xdt", [torch.float16, torch.float32])
@pytest.mark.parametrize("wdt", [torch.float16, torch.float32])
@pytest.mark.parametrize("out_dtype", [None, torch.float16])
@pytest.mark.parametrize("train_weight", [False, True])
def test_dtype_grid(device, xdt, wdt, out_dtype, train_weight):
    _case(device, (2, 5, 1000), xdt, wdt, out_dtype, train_weight)


def test_row_strided_input(device):
    _case(device, (37, 1536), torch.float16, torch.float32, None, True, strided=True)


def test_zero_rows_and_invalid_inputs(device):
    x = torch.empty((0, 64), device=device, dtype=torch.float16, requires_grad=True)
    w = torch.ones(64, device=device, dtype=torch.float16, requires_grad=True)
    y = rms_norm(x, w, 1e-6)
    y.sum().backward()
    assert y.shape == (0, 64) and torch.equal(w.grad, torch.zeros_like(w))
    with pytest.raises(ValueError):
        rms_norm(torch.zeros((4, 8), device=device, dtype=torch.bfloat16),
                 torch.ones(8, device=device), 1e-6)
    with pytest.raises(ValueError):
        rms_norm(torch.zeros((4, 8), device=device), torch.ones(4, device=device), 1e-6)
    with pytest.raises(ValueError):
        rms_norm(torch.zeros((4, 8), device=device), torch.ones(8, device=device), -1.0)


def test_patched_qwen2_rmsnorm_matches_eager(device):
    modeling = pytest.importorskip("transformers.models.qwen2.modeling_qwen2")
    from soupsuck_amd.patch import patch_qwen2_rmsnorm

    norm = modeling.Qwen2RMSNorm(1536, eps=1e-6).to(device)
    with torch.no_grad():
        norm.weight.copy_(1 + 0.1 * torch.randn(1536, device=device))
    x = torch.randn((3, 77, 1536), device=device, dtype=torch.float16, requires_grad=True)
    original = modeling.Qwen2RMSNorm.forward
    expected = original(norm, x)
    expected.float().sum().backward()
    gx_ref, gw_ref = x.grad.clone(), norm.weight.grad.clone()
    x.grad, norm.weight.grad = None, None
    assert patch_qwen2_rmsnorm(modeling)
    try:
        actual = norm(x)
        assert "RowNorm" in type(actual.grad_fn).__name__
        actual.float().sum().backward()
    finally:
        modeling.Qwen2RMSNorm.forward = original
    assert actual.dtype == expected.dtype
    torch.testing.assert_close(actual, expected, **F16_TOL)
    torch.testing.assert_close(x.grad, gx_ref, **F16_TOL)
    torch.testing.assert_close(norm.weight.grad, gw_ref, rtol=2e-3, atol=2e-2)
