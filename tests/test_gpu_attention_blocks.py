"""GPU parity of the attention kernels at the edges of their blocks and variants.

The kernels work in blocks of 128 queries / keys (64 for batches too small to fill
the chip and, on 16-row waves, for batches of short rows), 64-token tiles and 32-token halves, and find their (block, row) from the row
lengths (at most 64 rows) or from the grid (more rows).  Each case puts row ends on
both sides of those edges, for both block sizes, with and without GQA, and with the
signs of the softmax scale that the kernels treat apart.

Bar, as in test_gpu_attention.py (fp16 inputs, P and outputs, fp32 sums): against the
float64 oracle the output within atol = rtol = 2e-3 and the gradients within relative
L2 1e-2; two calls bit-identical.
"""

import numpy as np
import pytest
import torch

from oracle import attention as oattn
from soupsuck_amd import _lib
from soupsuck_amd.kernels.attention import packed_causal_attention

pytestmark = pytest.mark.gpu

EDGES = (1, 31, 32, 33, 63, 64, 65, 127, 128, 129, 161, 193, 257)
MANY = tuple(1 + (7 * i) % 40 for i in range(70))   # more rows than one wave has lanes


def _np(t):
    return t.detach()[0].transpose(0, 1).float().cpu().numpy()


@pytest.mark.parametrize("lengths,hq,hk,scale", [
    (EDGES, 6, 2, 128 ** -0.5),     # 64-token blocks
    (EDGES, 56, 8, 128 ** -0.5),    # 128-token blocks, 7:1 GQA
    (EDGES, 52, 52, 128 ** -0.5),   # 128-token blocks, dK / dV written directly
    (MANY, 4, 2, 128 ** -0.5),      # positions from the grid, 64-token blocks
    (MANY, 60, 10, 128 ** -0.5),    # positions from the grid, 128-token blocks
    ((40, 300), 4, 2, -0.07),
    ((40, 300), 4, 2, 0.0),
    # 16-row waves: all three steps, dQ and dK / dV, dK / dV alone, none; and few tokens
    ((1, 15, 16, 17, 31, 32) * 20, 12, 2, 128 ** -0.5),
    ((32, 33, 48, 47) * 10, 12, 12, 128 ** -0.5),
    ((32, 33, 48, 63, 64) * 10, 12, 12, 128 ** -0.5),
    ((64, 65, 127, 129, 191, 192) * 3, 12, 2, 128 ** -0.5),
    ((64, 65, 127, 129, 193) * 3, 12, 2, 128 ** -0.5),
    ((128, 65, 1), 12, 2, 128 ** -0.5),
    ((128, 129, 1), 12, 2, 128 ** -0.5),
    ((20, 32), 4, 2, -0.07),
    ((20, 32), 4, 2, 0.0),
])
def test_block_edges(device, lengths, hq, hk, scale):
    t = sum(lengths)
    print(f"case rows={len(lengths)} T={t} hq={hq} hk={hk} scale={scale}", flush=True)
    gen = torch.Generator().manual_seed(t + hq)

    def heads(h):
        x = torch.randn((1, t, h * 128), generator=gen).half().to(device)
        return x.view(1, t, h, 128).transpose(1, 2).requires_grad_()

    q, k, v = heads(hq), heads(hk), heads(hk)
    o = packed_causal_attention(q, k, v, lengths, scale)
    assert torch.equal(o, packed_causal_attention(q, k, v, lengths, scale))
    ref, _ = oattn.forward(_np(q), _np(k), _np(v), lengths, scale)
    got = o.detach()[0].float().cpu().numpy().astype(np.float64)
    np.testing.assert_allclose(got, ref, rtol=2e-3, atol=2e-3)
    g = torch.randn((1, t, hq, 128), generator=gen).half().to(device)
    grads = torch.autograd.grad(o, (q, k, v), g)
    refs = oattn.backward(_np(q), _np(k), _np(v), g[0].float().cpu().numpy(), lengths, scale)
    for name, x, ref_g in zip("qkv", grads, refs):
        norm = np.linalg.norm(ref_g)
        err = np.linalg.norm(_np(x).astype(np.float64) - ref_g)
        assert err <= 1e-2 * norm, f"d{name}: {err:.3e} of {norm:.3e}"


@pytest.mark.parametrize("lengths,hq,hk", [
    ((45, 100), 2, 1),             # 16-row waves
    ((45, 200), 2, 1),             # 64-token blocks
    ((130, 300), 2, 2),            # 64-token blocks, dK / dV written directly
    ((450,) * 10, 16, 16),         # 128-token blocks
])
def test_nan_query_reaches_only_what_it_attends_to(device, lengths, hq, hk):
    """A query row of NaN (head 0, token 10 of every packed row) makes its own output and dQ NaN
    and, as its P, dV of the keys it attends to; no other row of O, dQ or dV."""
    t = sum(lengths)
    print(f"case NaN rows={len(lengths)} T={t} hq={hq} hk={hk}", flush=True)
    gen = torch.Generator().manual_seed(t)

    def heads(h):
        x = torch.randn((1, t, h * 128), generator=gen).half().to(device)
        return x.view(1, t, h, 128).transpose(1, 2)

    q, k, v = heads(hq), heads(hk), heads(hk)
    starts = np.cumsum((0,) + lengths[:-1])
    for s in starts:
        q[0, 0, s + 10] = float("nan")
    q, k, v = (x.requires_grad_() for x in (q, k, v))
    o = packed_causal_attention(q, k, v, lengths, 128 ** -0.5)
    g = torch.randn((1, t, hq, 128), generator=gen).half().to(device)
    dq, _, dv = torch.autograd.grad(o, (q, k, v), g)

    def bad(x):   # [heads, tokens]
        return ~torch.isfinite(x.detach()).all(-1)[0].cpu().numpy()

    own = np.zeros((hq, t), bool)
    own[0, starts + 10] = True
    seen = np.zeros((hk, t), bool)
    for s in starts:
        seen[0, s:s + 11] = True
    np.testing.assert_array_equal(bad(o.transpose(1, 2)), own)
    np.testing.assert_array_equal(bad(dq), own)
    np.testing.assert_array_equal(bad(dv), seen)


@pytest.mark.parametrize("lengths,hq,hk", [((50, 65), 2, 1), ((230, 65), 2, 1),
                                                 ((700,) * 6, 16, 16)])
def test_reversed_token_axis(device, lengths, hq, hk):
    """The C entry points take any token stride: operands stored last token first (a negative
    stride from the last row) give the bits of the same operands stored forwards."""
    t = sum(lengths)
    print(f"case reversed rows={len(lengths)} T={t} hq={hq} hk={hk}", flush=True)
    gen = torch.Generator().manual_seed(t)
    cu = torch.tensor(np.cumsum((0,) + lengths), dtype=torch.int32, device=device)
    q, dout = (torch.randn((t, hq, 128), generator=gen).half().to(device) for _ in range(2))
    k, v = (torch.randn((t, hk, 128), generator=gen).half().to(device) for _ in range(2))
    size = _lib.load().ss_attn_varlen_bwd_workspace_size(hq, hk, t)
    ws = torch.empty(size, dtype=torch.uint8, device=device)
    stream = _lib.stream(device)

    def run(reverse):
        def operand(x):
            held = x.flip(0).contiguous() if reverse else x
            first = held[-1] if reverse else held[0]
            return held, (first.data_ptr(), -x.stride(0) if reverse else x.stride(0), x.stride(1))

        ins = [operand(x) for x in (q, k, v)]
        args = sum((a for _, a in ins), ())
        o, ovec = operand(torch.empty_like(q))
        lse = torch.empty((hq, t), device=device)
        sizes = (cu.data_ptr(), len(lengths), max(lengths), t, hq, hk, 128, 128 ** -0.5)
        _lib.call("ss_attn_varlen_fwd", *args, *sizes, *ovec, lse.data_ptr(), stream)
        g, gvec = operand(dout)
        outs = [operand(torch.empty_like(x)) for x in (q, k, v)]
        _lib.call("ss_attn_varlen_bwd", *args, *ovec, *gvec, lse.data_ptr(), *sizes,
                  *sum((a for _, a in outs), ()), ws.data_ptr(), size, stream)
        torch.cuda.synchronize()
        return [x.flip(0) if reverse else x for x in (o, *(held for held, _ in outs))] + [lse]

    for got, want in zip(run(True), run(False)):
        assert torch.equal(got, want)


@pytest.mark.parametrize("n,tail", [(2048, 2e-5), (2048, 1e-5), (100, 5e-5), (3000, 1e-6)])
def test_dominating_key_with_subnormal_tail(device, n, tail):
    """One key at P = 1 and n - 1 keys at P = tail, an fp16 subnormal (below 6.1e-5) that adds up
    to percents of the mass: the P.V product and the sum that O is divided by must both
    count it.  Bound on O: its own rounding, and a half step of the subnormal P (2^-25) for
    every key in the product and in the sum."""
    print(f"case dominating key n={n} tail={tail}", flush=True)
    gen = torch.Generator().manual_seed(n)
    q, k = torch.zeros((1, 2, n, 128)), torch.zeros((1, 1, n, 128))
    q[..., 0] = 8.0
    k[0, 0, 0, 0] = np.log(1 / tail) / 8 * 128 ** 0.5
    v = torch.rand((1, 1, n, 128), generator=gen) + 1.0
    v[:, :, 0] = -1.0
    q, k, v = (a.half().to(device) for a in (q, k, v))
    o = packed_causal_attention(q, k, v, (n,), 128 ** -0.5)
    ref, _ = oattn.forward(_np(q), _np(k), _np(v), (n,), 128 ** -0.5)
    err = np.abs(o[0].float().cpu().numpy().astype(np.float64) - ref).max()
    bound = 2.0 ** -11 * max(1.0, np.abs(ref).max()) + n * 2.0 ** -25 * (2.0 + np.abs(ref).max())
    assert err <= bound, f"{err:.3e} of {bound:.3e}"
