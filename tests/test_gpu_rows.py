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


def test_combine_non_finite(torch_cuda):
    """Infinities and NaN in a slot's row, the shared row, the gate and the
    residual reach the values they belong to and no others, as in the torch
    form (slots past the call's k, which the kernel's batch of eight reads
    again, add nothing)."""
    torch = torch_cuda
    from runnel_amd import native
    g = torch.Generator().manual_seed(5)
    T, k, H = 6, 3, 64
    y = torch.randn((T, k, H), generator=g).bfloat16()
    sh, res = torch.randn((2, T, H), generator=g).bfloat16()
    gate = torch.randn((T, 1), generator=g).bfloat16()
    w = torch.rand((T, k), generator=g)
    y[0, k - 1, 3], y[1, 0, 5], y[1, 1, 5] = float("inf"), float("inf"), -float("inf")
    sh[2, 7], res[3, 9], gate[4], gate[5] = float("nan"), -float("inf"), float("nan"), -float("inf")
    w[0, 1] = 0.0
    y[0, 1, 11] = float("inf")  # weight 0: NaN
    ref = (y.float() * w[..., None]).sum(1) + torch.sigmoid(gate.float()) * sh.float()
    ref = (res.float() + ref.bfloat16().float()).bfloat16().float()
    got = native.combine(*(t.cuda() for t in (y, w, sh, gate, res))).cpu().float()
    assert torch.equal(got.isnan(), ref.isnan())
    assert torch.equal(got.isinf(), ref.isinf())
    fin = ref.isfinite()
    assert ((got - ref)[fin].abs() <= 2.0 ** -6 * ref[fin].abs() + 2.0 ** -7).all()


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


def test_swiglu_function_keeps_the_torch_bits(torch_cuda):
    """Every bf16 gate against up values of every kind: the kernel behind
    switch_layers.swiglu gives the bits of silu(gate) * up (NaN for NaN)."""
    torch = torch_cuda
    from runnel_amd import native
    from runnel_amd.switch_layers import swiglu
    gate = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16).cuda()
    for u in (1.0, -0.7109375, 3.0e38, 1.0e-38, 0.0, -0.0, float("inf"), float("nan")):
        up = torch.full_like(gate, u)
        assert native.rows_ready(up, gate)
        got, ref = swiglu(up, gate), torch.nn.functional.silu(gate) * up
        same = (got.view(torch.int16) == ref.view(torch.int16)) | (got.isnan() & ref.isnan())
        assert same.all(), u


def test_swiglu_torch_form(torch_cuda):
    """Rows the kernel does not take: in autograd, not contiguous, not 16-byte
    aligned, of broadcasting shapes, with a forward-mode tangent."""
    torch = torch_cuda
    from torch.autograd import forward_ad

    from runnel_amd import native
    from runnel_amd.switch_layers import swiglu
    up, gate = torch.randn(2, 48, 64, device="cuda").bfloat16()
    form = lambda u, g: torch.nn.functional.silu(g) * u
    pad = torch.randn(2, 48 * 64 + 8, device="cuda").bfloat16()
    for u, g in ((up.t(), gate.t()), (pad[0, 1:3073], pad[1, 1:3073]), (up, gate[:1])):
        assert not native.rows_ready(u, g) or u.shape != g.shape
        assert torch.equal(swiglu(u, g), form(u, g))
    u, g = up.clone().requires_grad_(), gate.clone().requires_grad_()
    swiglu(u, g).sum().backward()
    u2, g2 = up.clone().requires_grad_(), gate.clone().requires_grad_()
    form(u2, g2).sum().backward()
    assert torch.equal(u.grad, u2.grad) and torch.equal(g.grad, g2.grad)
    with forward_ad.dual_level():
        out = swiglu(forward_ad.make_dual(up, gate), forward_ad.make_dual(gate, up))
        ref = form(forward_ad.make_dual(up, gate), forward_ad.make_dual(gate, up))
        assert torch.equal(forward_ad.unpack_dual(out).tangent,
                           forward_ad.unpack_dual(ref).tangent)


def test_replaced_calls_are_made(torch_cuda, monkeypatch):
    """A program that wraps QuantizedSwitchLinear or SwiGLU sees every one of
    their calls inside SwitchGLU, with the result unchanged."""
    torch = torch_cuda
    from runnel_amd import QuantizedSwitchLinear, SwiGLU, SwitchGLU
    sm = SwitchGLU(64, 128, 4, device="cuda")
    for p in (sm.gate_proj, sm.up_proj, sm.down_proj):
        w = torch.randn(4, p.output_dims, p.input_dims, device="cuda") * 0.1
        q = QuantizedSwitchLinear.from_float(w)
        p.weight, p.scales, p.biases = q.weight, q.scales, q.biases
    x = torch.randn(5, 64, device="cuda").bfloat16()
    idx = torch.randint(0, 4, (5, 2), device="cuda", dtype=torch.int32)
    ref = sm(x, idx)
    calls = []
    for cls in (QuantizedSwitchLinear, SwiGLU):
        own = cls.__call__

        def wrapped(self, *args, _own=own, _name=cls.__name__):
            calls.append(_name)
            return _own(self, *args)
        monkeypatch.setattr(cls, "__call__", wrapped)
    assert torch.equal(sm(x, idx), ref)
    assert sorted(calls) == ["QuantizedSwitchLinear"] * 3 + ["SwiGLU"]


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


def test_block_tail_torch_form(torch_cuda):
    """Before packing, a residual that is not contiguous, not 16-byte aligned
    or in autograd takes the torch form: the same values, and a gradient of
    ones."""
    torch = torch_cuda
    from runnel_amd import SparseMoeBlock, native
    blk = SparseMoeBlock(64, 64, 4, 2, shared_expert_intermediate_size=64, device="cuda")
    w = torch.randn((4, 64, 64), device="cuda") * 0.1
    for p in (blk.switch_mlp.gate_proj, blk.switch_mlp.up_proj, blk.switch_mlp.down_proj):
        q, s, b = native.quantize(w, 8)
        p.weight.copy_(q), p.scales.copy_(s), p.biases.copy_(b)
    x, r = torch.randn(2, 5, 64, device="cuda").bfloat16()
    plain = blk(x, residual=r).float()
    wide = torch.zeros((5, 72), device="cuda").bfloat16()
    wide[:, :64] = r
    odd = torch.zeros(5 * 64 + 8, device="cuda").bfloat16()
    odd[1:321] = r.reshape(-1)
    grad = r.clone().requires_grad_()
    for res in (wide[:, :64], odd[1:321].view(5, 64), grad):
        assert not native.rows_ready(res)
        out = blk(x, residual=res)
        # the fp32 sum in another order: a step of bf16 at each of two roundings
        assert ((out.float() - plain).abs() <= 2.0 ** -7 * (plain.abs() + r.float().abs())).all()
    out.sum().backward()
    assert torch.equal(grad.grad, torch.ones_like(grad))


def test_stream_handle_follows_the_current_stream(torch_cuda):
    torch = torch_cuda
    from runnel_amd import _lib
    for stream in (torch.cuda.default_stream(), torch.cuda.Stream()):
        with torch.cuda.stream(stream):
            for device in (None, 0, "cuda", "cuda:0", torch.device("cuda"), torch.device("cuda:0")):
                assert _lib.stream_handle(device) == stream.cuda_stream
