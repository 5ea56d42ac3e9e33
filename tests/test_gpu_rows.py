"""The one-launch tail of a block of separate modules (rmoe_combine) and the
SwiGLU of separate projections (rmoe_swiglu) against torch on the CPU: slot
counts around the eight rows requested at once, widths that end inside a
workgroup, with and without the shared row and the residual, infinities and
NaN."""

import numpy as np
import pytest

from helpers import dev_bf16, host_bf16
from oracle import moe_ref as M

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from runnel_amd import _lib
    _lib.load()
    return torch


@pytest.mark.parametrize("shared,residual", [(True, True), (True, False), (False, False)])
@pytest.mark.parametrize("T,k,H", [(1, 1, 8), (3, 8, 2048), (2, 9, 2056), (5, 64, 512)])
def test_combine(torch_cuda, T, k, H, shared, residual):
    """Within the fp32 sums' error and one bf16 rounding (8 significant bits:
    half a spacing of 2^(e - 7) is at most 2^-8 of a value in [2^e, 2^(e + 1)))
    of the sum; with a residual also of the final sum."""
    torch = torch_cuda
    from runnel_amd import native
    rng = np.random.default_rng(T * k + H)
    y, w = M.make_x(1, T * k, H).reshape(T, k, H), rng.random((T, k)).astype(np.float32)
    sh, res, g = M.make_x(2, T, H), M.make_x(3, T, H), M.make_x(4, T, 8)[:, :1].copy()
    out = native.combine(dev_bf16(y), torch.from_numpy(w).cuda(),
                         dev_bf16(sh) if shared else None, dev_bf16(g) if shared else None,
                         dev_bf16(res) if residual else None)
    f = lambda a: M.bf16_to_f32(a).astype(np.float64)
    terms = f(y) * w[..., None].astype(np.float64)
    ref, size = terms.sum(1), np.abs(terms).sum(1)
    if shared:
        s = f(sh) / (1.0 + np.exp(-f(g)))
        ref, size = ref + s, size + np.abs(s)
    tol = 2.0 ** -8 * np.abs(ref) + (k + 4) * 2.0 ** -23 * size
    if residual:
        ref = ref + f(res)
        tol = tol + 2.0 ** -8 * (np.abs(ref) + tol)
    assert (np.abs(f(host_bf16(out)) - ref) <= tol * 1.01 + 1e-30).all()


@pytest.mark.parametrize("n", [1, 7, 8, 2049, 5 * 512])
def test_swiglu(torch_cuda, n):
    torch = torch_cuda
    from runnel_amd import native
    up, gate = torch.randn(2, n).bfloat16()
    gate[0] = -float("inf") if n == 7 else gate[0]
    gate[n // 2] = float("nan") if n > 8 else gate[n // 2]
    up[n - 1] = float("inf")
    got = native.swiglu(up.cuda(), gate.cuda()).cpu().float().numpy()
    s = torch.nn.functional.silu(gate.float()).bfloat16().float().numpy()
    ref = M.round_bf16(s * up.float().numpy())
    # an ulp of the rounded silu either way, then the product's rounding
    ok = np.abs(got - ref) <= 2.0 ** -7 * np.abs(ref)
    assert (ok | (got == ref) | (np.isnan(got) & np.isnan(ref))).all()
    fin = np.isfinite(ref)
    assert (got[fin] == ref[fin]).mean() >= 0.99 or n < 100


def test_block_tail_under_forward_mode(torch_cuda):
    """A residual's forward-mode tangent passes through the block before
    packing (its other operands carry none)."""
    torch = torch_cuda
    from torch.autograd import forward_ad

    from runnel_amd import SparseMoeBlock
    blk = SparseMoeBlock(64, 64, 4, 2, shared_expert_intermediate_size=64, device="cuda")
    x, r, t = torch.randn(3, 5, 64, device="cuda").bfloat16()
    plain = blk(x, residual=r)
    with forward_ad.dual_level():
        out = forward_ad.unpack_dual(blk(x, residual=forward_ad.make_dual(r, t)))
        assert torch.equal(out.primal, plain)  # (zero weights: the residual itself)
        assert torch.equal(out.tangent, t)
