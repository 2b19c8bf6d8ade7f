"""The skinny forward's row instances and the dense product's tiles at their edges: every
16-row count and its remainders, one to several iterations and splits, one to a few 64-deep
stages, remainders of each tile, against the float64 product of the same fp16 operands.
Bar: the projections' gate (rtol = atol = 2e-3 on fp16, relative L2 <= 1e-3); fp32 outputs
within the fp32 sum's bound, K eps sum |a b| for a K-term sum in any order."""

import numpy as np
import pytest
import torch

from oracle import gemm as ogemm
from oracle import nf4 as onf4
from soupsuck_amd.kernels.nf4_gemm import gemm_f16, nf4_matmul
from tests.gpu_util import device_state, np16, random_weight

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


# Sizes around each tile edge (64, 128, 160, 192, 256) with one to four 64-deep stages (a
# stage ring longer than the work, equal, longer work), and a split product's last shorter
# split; single-tile grids and ones wider than the chip.
@pytest.mark.parametrize("m,n,k,split", [
    (1, 8, 64, False), (65, 72, 128, False), (257, 264, 192, False), (129, 2064, 256, False),
    (1025, 8008, 64, False), (1000, 8960, 192, False), (2049, 4104, 128, False),
    (4100, 6408, 64, False), (300, 520, 1600, True), (827, 264, 4160, True),
    (513, 1544, 8256, True),
])
def test_dense_tile_edges(device, m, n, k, split):
    rng = np.random.default_rng(m + 3 * n + 5 * k)
    a = rng.standard_normal((m, k), dtype=np.float32).astype(np.float16)
    b = (rng.standard_normal((n, k), dtype=np.float32) * 0.05).astype(np.float16)
    bias = (rng.standard_normal(n) * 0.1).astype(np.float16)
    ad, bd = torch.from_numpy(a).to(device), torch.from_numpy(b).to(device)
    exact = ad.double() @ bd.double().T
    bound = (k * 2.0 ** -24) * (ad.double().abs() @ bd.double().abs().T) + 1e-30
    got = gemm_f16(ad, bd, b_trans=True, out_dtype=torch.float32, split_k=split)
    assert bool(((got.double() - exact).abs() <= bound).all())
    half = gemm_f16(ad, bd, b_trans=True, bias=torch.from_numpy(bias).to(device), split_k=split)
    _gate(half, exact.cpu().numpy() + bias.astype(np.float64), f"{m}x{n}x{k}")
    # a wider destination's neighbours stay as they were
    wide = torch.full((m, n + 8), 7.0, device=device, dtype=torch.float16)
    gemm_f16(ad, bd, b_trans=True, out=wide[:, :n], split_k=split)
    assert bool((wide[:, n:] == 7.0).all())
    assert torch.equal(wide[:, :n], gemm_f16(ad, bd, b_trans=True, split_k=split))
