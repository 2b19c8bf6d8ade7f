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
# 128x256, 256x160, 256x192, 256x256; 8 the ping-pong 256x256) and splits.  Every configuration
# with M and N past a tile edge, unsplit and split with a shorter last split (8 is not split),
# the small ones also with one to four 64-deep stages (a stage ring longer than the work,
# equal, longer work) and on grids wider than the chip.
TILES = [
    (1, 8, 64, False, 1, 1), (65, 72, 128, False, 1, 1), (257, 264, 192, False, 1, 1),
    (129, 2064, 256, False, 1, 1), (1025, 8008, 64, False, 1, 1), (1000, 8960, 192, False, 5, 1),
    (2049, 4104, 128, False, 1, 1), (4100, 6408, 64, False, 8, 1), (300, 520, 1600, True, 1, 1),
    (827, 264, 4160, True, 2, 7), (513, 1544, 8256, True, 3, 3), (130, 5512, 256, False, 1, 1),
    (201, 5960, 192, False, 2, 1), (642, 4440, 128, False, 3, 1), (1235, 5704, 128, False, 4, 1),
    (1170, 5128, 384, False, 4, 1), (1665, 5480, 128, False, 5, 1), (1680, 4832, 256, False, 5, 1),
    (1547, 5928, 192, False, 6, 1), (1950, 5128, 384, False, 6, 1),
    (2564, 5456, 3008, False, 7, 1), (1732, 5848, 64, False, 8, 1), (2375, 6024, 64, False, 8, 1),
    (2576, 5496, 576, False, 8, 1), (12, 32, 2624, True, 1, 5), (2872, 8, 6016, True, 2, 8),
    (67, 4120, 4864, True, 3, 7), (134, 5544, 7488, True, 4, 5), (130, 5704, 11968, True, 5, 7),
    (2494, 544, 12096, True, 6, 8), (1026, 4088, 11648, True, 7, 3),
]
# m, n, k, K-major A, K-major B, configuration, splits
K_MAJOR = [
    (1205, 3208, 9536, False, True, 8, 3), (528, 5488, 128, True, False, 3, 1),
    (1480, 4768, 128, True, False, 4, 1), (1480, 4768, 128, False, True, 4, 1),
    (1480, 4768, 128, True, True, 4, 1), (72, 4584, 4160, True, False, 3, 6),
    (72, 4584, 4160, False, True, 3, 6), (72, 4584, 4160, True, True, 3, 6),
    (16, 8, 3904, False, True, 1, 7), (1288, 5400, 64, True, False, 8, 1),
    (1832, 3856, 192, True, True, 8, 1),
]
# t, n, k of a QLoRA projection, then the plans of its forward (t x n x k, LoRA epilogue) and of
# its dX (t x k x n, rank-16 epilogue)
QLORA = [
    (327, 4032, 192, (2, 1), (1, 7)), (534, 5568, 128, (3, 1), (1, 8)),
    (1217, 5760, 128, (4, 1), (1, 6)), (2372, 3904, 128, (5, 1), (2, 6)),
    (1567, 6016, 192, (6, 1), (2, 6)), (2314, 5696, 2624, (7, 1), (4, 1)),
    (1948, 5312, 128, (8, 1), (2, 7)), (278, 832, 3136, (1, 1), (1, 1)),
    (267, 1856, 5824, (3, 5), (1, 1)), (646, 5504, 5696, (5, 2), (5, 2)),
    (324, 192, 4352, (1, 8), (2, 1)), (514, 128, 5696, (1, 8), (3, 1)),
    (1409, 128, 5056, (1, 5), (4, 1)), (1665, 128, 5504, (2, 8), (5, 1)),
    (1561, 192, 6016, (2, 6), (6, 1)), (2330, 2880, 5184, (4, 1), (7, 1)),
    (2313, 128, 4480, (2, 6), (8, 1)), (273, 3328, 832, (2, 1), (2, 6)),
    (258, 5824, 1856, (1, 1), (3, 5)), (652, 5696, 5504, (5, 2), (5, 2)),
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
