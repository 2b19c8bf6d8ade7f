"""The skinny forward's row instances and the dense product's tiles at their edges: every
16-row count and its remainders, one to several iterations and splits, one to a few 64-deep
stages, remainders of each tile (the plan of every case is asserted), against the float64
product of the same fp16 operands.
Bar: the projections' gate (rtol = atol = 2e-3 on fp16, relative L2 <= 1e-3); fp32 outputs
within the fp32 sum's bound, K eps sum |a b| for a K-term sum in any order."""

import numpy as np
import pytest
import torch

from oracle import gemm as ogemm
from oracle import nf4 as onf4
from soupsuck_amd.bnb_compat import quantize_4bit
from soupsuck_amd.kernels.nf4 import dequantize_nf4
from soupsuck_amd.kernels.nf4_gemm import gemm_f16, nf4_matmul
from soupsuck_amd.lora import qlora_projection
from tests.gpu_util import device_state, np16, nt_plan, random_weight

pytestmark = pytest.mark.gpu


def _gate(actual, expected, what):
    ok, max_abs, rel = ogemm.gate(np16(actual).astype(np.float64), expected)
    assert ok, f"{what}: max_abs={max_abs:.3e} rel_l2={rel:.3e}"


# K = 128 k: one iteration (the code ring longer than the work), two, splits of two
# iterations with a shorter last one, and of four (K above 2560) with a shorter last one; N
# around the 128-row workgroup.
@pytest.mark.parametrize("n,k", [(40, 128), (128, 256), (136, 640), (64, 2432), (136, 2944)])
@pytest.mark.parametrize("t", [33, 48, 49, 64, 65, 81, 96, 101, 112, 113, 128])
def test_skinny_rows(device, t, n, k):
    state = onf4.quantize_nested(random_weight(n, k, 11))
    packed, qs = device_state(state, device)
    rng = np.random.default_rng(t * 7 + n + k)
    x = rng.standard_normal((t, k), dtype=np.float32).astype(np.float16)
    bias = (rng.standard_normal(n) * 0.1).astype(np.float16)
    xt, bt = torch.from_numpy(x).to(device), torch.from_numpy(bias).to(device)
    y = nf4_matmul(xt, packed, qs, bias=bt)
    _gate(y, ogemm.linear(x, state.decode(), bias), f"t={t} n={n} k={k}")
    # a row's result does not depend on the rows after it (they change the instance only
    # through its tile count): the first rows alone give the same bits in the same instance
    least = (t - 1) // 16 * 16 + 1
    if least > 32:
        assert torch.equal(nf4_matmul(xt[:least], packed, qs, bias=bt), y[:least])


# m, n, k, scratch for a split, then the plan: configuration (1 .. 7 for 64x64, 128x64, 128x128,
# 128x256, 256x160, 256x192, 256x256; 8 the ping-pong 256x256 of a K-major A) and splits.  Every
# configuration with M and N past a tile edge, unsplit and split with a shorter last split, the
# small ones also with one to four 64-deep stages (a stage ring longer than the work, equal,
# longer work) and on grids wider than the chip.
TILES = [
    (1, 8, 64, False, 1, 1), (65, 72, 128, False, 1, 1), (257, 264, 192, False, 1, 1),
    (129, 2064, 256, False, 1, 1), (1025, 8008, 64, False, 1, 1), (1000, 8960, 192, False, 2, 1),
    (2049, 4104, 128, False, 2, 1), (4100, 6408, 64, False, 2, 1), (300, 520, 1600, True, 1, 1),
    (827, 264, 4160, True, 1, 3), (513, 1544, 8256, True, 1, 1),
    (578, 3376, 256, False, 3, 1), (1170, 5128, 384, False, 4, 1), (1669, 5424, 384, False, 5, 1),
    (1950, 5128, 384, False, 6, 1), (2576, 5496, 576, False, 7, 1),
    (287, 1096, 5568, True, 3, 8), (259, 3824, 6016, True, 4, 5), (386, 3192, 9024, True, 5, 6),
    (1428, 1320, 11392, True, 6, 6), (775, 5168, 10240, True, 7, 3),
]
# m, n, k, K-major A, K-major B, configuration, splits
K_MAJOR = [
    (1096, 2736, 128, True, False, 3, 1), (2440, 2912, 256, True, False, 4, 1),
    (1861, 3784, 256, False, True, 4, 1), (1864, 3784, 256, True, True, 4, 1),
    (72, 2784, 4416, True, False, 3, 8), (68, 2784, 4416, False, True, 3, 8),
    (136, 5536, 5056, True, True, 4, 5), (1832, 3856, 64, True, False, 8, 1),
    (1832, 3856, 192, True, True, 8, 1),
]
# t, n, k of a QLoRA projection, then the plans of its forward (t x n x k, LoRA epilogue) and of
# its dX (t x k x n, rank-16 epilogue)
QLORA = [
    (1672, 3648, 384, (4, 1), (1, 1)), (1284, 6016, 448, (5, 1), (1, 1)),
    (1806, 5504, 384, (6, 1), (1, 1)), (2562, 5504, 576, (7, 1), (2, 1)),
    (265, 1216, 5632, (3, 8), (1, 1)), (261, 3648, 6016, (4, 5), (1, 1)),
    (642, 5504, 5312, (5, 2), (3, 1)),
    (1220, 384, 4928, (1, 1), (4, 1)), (1289, 448, 6016, (1, 1), (5, 1)),
    (1665, 384, 5888, (1, 1), (6, 1)), (2455, 576, 5760, (2, 1), (7, 1)),
    (385, 5632, 832, (3, 1), (3, 8)), (658, 5248, 5504, (3, 1), (5, 2)),
]


def _products(device, m, n, k):
    rng = np.random.default_rng(m + 3 * n + 5 * k)
    a = rng.standard_normal((m, k), dtype=np.float32).astype(np.float16)
    b = (rng.standard_normal((n, k), dtype=np.float32) * 0.05).astype(np.float16)
    ad, bd = torch.from_numpy(a).to(device), torch.from_numpy(b).to(device)
    exact = ad.double() @ bd.double().T
    bound = (k * 2.0 ** -24) * (ad.double().abs() @ bd.double().abs().T) + 1e-30
    return ad, bd, exact, bound


@pytest.mark.parametrize("m,n,k,split,cfg,splits", TILES)
def test_dense_tile_edges(device, m, n, k, split, cfg, splits):
    assert nt_plan(m, n, k, split=split) == (cfg, splits)
    ad, bd, exact, bound = _products(device, m, n, k)
    bias = (np.random.default_rng(n).standard_normal(n) * 0.1).astype(np.float16)
    got = gemm_f16(ad, bd, b_trans=True, out_dtype=torch.float32, split_k=split)
    assert bool(((got.double() - exact).abs() <= bound).all())
    half = gemm_f16(ad, bd, b_trans=True, bias=torch.from_numpy(bias).to(device), split_k=split)
    _gate(half, exact.cpu().numpy() + bias.astype(np.float64), f"{m}x{n}x{k}")
    # a wider destination's neighbours stay as they were
    wide = torch.full((m, n + 8), 7.0, device=device, dtype=torch.float16)
    gemm_f16(ad, bd, b_trans=True, out=wide[:, :n], split_k=split)
    assert bool((wide[:, n:] == 7.0).all())
    assert torch.equal(wide[:, :n], gemm_f16(ad, bd, b_trans=True, split_k=split))


@pytest.mark.parametrize("m,n,k,a_k_major,b_k_major,cfg,splits", K_MAJOR)
def test_k_major_tile_edges(device, m, n, k, a_k_major, b_k_major, cfg, splits):
    assert nt_plan(m, n, k, a_k_major + 2 * b_k_major) == (cfg, splits)
    ad, bd, exact, bound = _products(device, m, n, k)
    got = gemm_f16(ad.T.contiguous() if a_k_major else ad, bd.T.contiguous() if b_k_major else bd,
                   a_trans=a_k_major, b_trans=not b_k_major, out_dtype=torch.float32, split_k=True)
    assert bool(((got.double() - exact).abs() <= bound).all())


@pytest.mark.parametrize("t,n,k,forward,backward", QLORA)
def test_qlora_tile_edges(device, t, n, k, forward, backward):
    """The LoRA and rank-16 epilogues on every wide tile, unsplit and split.  Forward: the
    projections' gate against the composition with fp16 after each product; dX: relative L2
    1e-3 against the float64 gradient (fp16 rounding of dX and of dZ, 2^-12 each in the mean)."""
    assert nt_plan(t, n, k) == forward and nt_plan(t, k, n) == backward
    gen = torch.Generator().manual_seed(t + n + k)

    def randn(*shape, scale=1.0):
        return (torch.randn(shape, generator=gen) * scale).half().to(device)

    packed, state = quantize_4bit(randn(n, k, scale=0.02))
    w = dequantize_nf4(packed, state).double()
    x, g = randn(t, k).requires_grad_(), randn(t, n, scale=0.01)
    a, b = randn(16, k, scale=k ** -0.5).requires_grad_(), randn(n, 16, scale=0.01).requires_grad_()
    y = qlora_projection(x, a, b, packed, state, None, scaling=2.0)
    z = (x.detach().double() @ a.detach().double().T).half().double()
    lora = (z @ b.detach().double().T).half().float() * 2.0
    base = (x.detach().double() @ w.T).half().float()
    _gate(y.detach(), (base + lora.half().float()).half().cpu().numpy().astype(np.float64),
          f"forward t={t} n={n} k={k}")
    (dx,) = torch.autograd.grad(y, x, g)
    exact = g.double() @ w + (g.double() * 2.0 @ b.detach().double()) @ a.detach().double()
    assert float((dx.double() - exact).norm() / exact.norm()) <= 1e-3
