"""Quantize and dequantize at the edges of their work split: group counts
around a wave's 16 groups and a workgroup's 64, row ranges, outputs that are
not 16-byte aligned, and groups that hold NaN or infinity.  Bytes equal the
oracle's (whole numbers and bf16 bits, no tolerance)."""

import ctypes

import numpy as np
import pytest

from helpers import host_bf16, host_u32
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


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("rows,cols", [(1, 64), (5, 192), (1, 1024), (17, 64), (1, 4096),
                                       (13, 320), (3, 4160)])
def test_group_counts(torch_cuda, bits, rows, cols):
    torch = torch_cuda
    from runnel_amd import native
    w = (np.random.default_rng(rows * cols + bits).standard_normal((rows, cols)) * 0.02)
    w = w.astype(np.float32)
    wq, s, b = native.quantize(torch.from_numpy(w).cuda(), bits)
    rw, rs, rb = M.quantize(w, bits)
    assert np.array_equal(host_u32(wq), rw)
    assert np.array_equal(host_bf16(s), rs)
    assert np.array_equal(host_bf16(b), rb)
    ref = M.dequantize(rw, rs, rb, bits)
    got = native.dequantize(wq, s, b, bits).cpu().numpy()
    got16 = native.dequantize(wq, s, b, bits, out_dtype=torch.bfloat16)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
    assert np.array_equal(host_bf16(got16), M.f32_to_bf16(ref))


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("skip", [0, 1, 4])
def test_dequantize_row_range_unaligned(torch_cuda, bits, skip):
    """Rows 2..6 of a bank into outputs `skip` elements past an aligned
    address (both outputs in one call); nothing else is written."""
    torch = torch_cuda
    from runnel_amd import _lib, native
    rng = np.random.default_rng(bits + skip)
    w = (rng.standard_normal((9, 192)) * 0.5).astype(np.float32)
    words, s, b = M.quantize(w, bits)
    dev = (torch.from_numpy(words.view(np.int32)).cuda(),
           torch.from_numpy(s.view(np.int16)).cuda().view(torch.bfloat16),
           torch.from_numpy(b.view(np.int16)).cuda().view(torch.bfloat16))
    qw = native.qweight_struct(*dev, bits)
    n = 5 * 192
    f32 = torch.full((n + 8,), 7.0, device="cuda")
    b16 = torch.full((n + 8,), 7.0, device="cuda", dtype=torch.bfloat16)
    _lib.check(_lib.load().rmoe_dequantize(
        ctypes.byref(qw), 2, 5, f32[skip:].data_ptr(), b16[skip:].data_ptr(),
        _lib.stream_handle(f32.device)))
    ref = M.dequantize(words, s, b, bits)[2:7].reshape(-1)
    exp = np.full(n + 8, 7.0, np.float32)
    exp[skip:skip + n] = ref
    assert np.array_equal(f32.cpu().numpy(), exp)
    assert np.array_equal(host_bf16(b16), M.f32_to_bf16(exp))


@pytest.mark.parametrize("bits", [8, 4])
def test_quotients_at_half_integers(torch_cuda, bits):
    """Values within a few 2^-20 of a half-integer multiple of the scale,
    where the reciprocal's product may round the other way than the
    quotient: the codes are the quotient's."""
    torch = torch_cuda
    from runnel_amd import native
    rng = np.random.default_rng(bits)
    n = 2 ** bits - 1
    k = rng.integers(0, 2 * n + 1, (64, 512)) * 0.5 + rng.integers(-3, 4, (64, 512)) * 2.0 ** -20
    k[:, ::64], k[:, 1::64] = 0.0, n
    w = (k * np.exp2(rng.integers(-20, 20, (64, 1))) * rng.uniform(0.5, 1, (64, 1)))
    w = w.astype(np.float32)
    wq, s, b = native.quantize(torch.from_numpy(w).cuda(), bits)
    rw, rs, rb = M.quantize(w, bits)
    assert np.array_equal(host_u32(wq), rw)
    assert np.array_equal(host_bf16(s), rs)
    assert np.array_equal(host_bf16(b), rb)


@pytest.mark.parametrize("bits", [8, 4])
def test_nan_and_infinity(torch_cuda, bits):
    """The extremes are a sequential "larger than" scan from value 0: a NaN
    counts only as the first value, and any other NaN gets code 0."""
    torch = torch_cuda
    from runnel_amd import native
    w = (np.random.default_rng(3).standard_normal((1, 6 * 64)) * 0.02).astype(np.float32)
    w[0, 5] = np.nan              # group 0: ignored by the extremes
    w[0, 64] = np.nan             # group 1: NaN throughout
    w[0, 128 + 63] = np.inf       # group 2
    w[0, 192 + 10] = -np.inf      # group 3
    wq, s, b = native.quantize(torch.from_numpy(w).cuda(), bits)
    codes = M.unpack(host_u32(wq), bits).reshape(6, 64)
    s, b = host_bf16(s)[0], host_bf16(b)[0]
    clean = np.where(np.isfinite(w), w, np.float32(0.01))
    clean[0, 5] = clean[0, 6]
    rw, rs, rb = M.quantize(clean, bits)
    rcodes = M.unpack(rw, bits).reshape(6, 64)
    rcodes[0, 5] = 0
    for g in (0, 4, 5):
        assert np.array_equal(codes[g], rcodes[g])
        assert s[g] == rs[0, g] and b[g] == rb[0, g]
    for g, edge in ((1, np.nan), (2, np.inf), (3, -np.inf)):
        assert np.isnan(M.bf16_to_f32(s[g:g + 1]))[0]
        assert np.array_equal(M.bf16_to_f32(b[g:g + 1]), np.float32([edge]), equal_nan=True)
        assert not codes[g].any()


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("both", [False, True])
def test_dequantize_from_the_longest_split_on(torch_cuda, bits, both):
    """2^24 values and one group on either side: bf16 alone takes four steps a
    thread from there on; with an fp32 output a thread takes one."""
    torch = torch_cuda
    from runnel_amd import _lib, native
    for groups in (2 ** 18 - 1, 2 ** 18, 2 ** 18 + 1):
        g = torch.Generator().manual_seed(groups + bits)
        wq = torch.randint(-2 ** 31, 2 ** 31 - 1, (groups, 2 * bits), generator=g,
                           dtype=torch.int32)
        s, b = torch.randn((2, groups, 1), generator=g).bfloat16()
        dev = (wq.cuda(), s.cuda(), b.cuda())
        qw = native.qweight_struct(*dev, bits)
        b16 = torch.empty((groups, 64), dtype=torch.bfloat16, device="cuda")
        f32 = torch.empty((groups, 64), device="cuda") if both else None
        _lib.check(_lib.load().rmoe_dequantize(ctypes.byref(qw), 0, groups, _lib.ptr(f32),
                                               b16.data_ptr(), _lib.stream_handle(b16.device)))
        q = wq.view(torch.uint8)
        if bits == 4:
            q = torch.stack((q & 15, q >> 4), -1).reshape(groups, 64)
        # the product of a code and a bf16 scale fits fp32, so this rounds once
        ref = (q.float() * s.float()).double() + b.double()
        assert torch.equal(b16.cpu(), ref.float().bfloat16())
        assert f32 is None or torch.equal(f32.cpu(), ref.float())


@pytest.mark.parametrize("bits", [8, 4])
def test_quantize_a_whole_bank(torch_cuda, bits):
    """128 experts of 512 x 2048 (134 M values): every word, scale and bias
    equals the format's fp32 rules (correctly rounded division, halves to
    even), evaluated by torch on the CPU."""
    torch = torch_cuda
    from runnel_amd import native
    n = 2 ** bits - 1
    g = torch.Generator(device="cuda").manual_seed(bits)
    w = torch.randn((128, 512, 2048), generator=g, device="cuda") * 0.02
    wq, s, b = (t.cpu() for t in native.quantize(w, bits))
    w = w.cpu()
    for e in range(0, 128, 16):
        v = w[e:e + 16].reshape(-1, 64)
        hi, lo = v.amax(1), v.amin(1)
        mask = lo.abs() > hi.abs()
        scale = ((hi - lo) / n).clamp_min(1e-7)
        scale = torch.where(mask, scale, -scale)
        edge = torch.where(mask, lo, hi)
        q0 = (edge / scale).round()
        scale = torch.where(q0 != 0, edge / q0, scale).bfloat16()
        bias = torch.where(q0 == 0, torch.zeros_like(edge), edge).bfloat16()
        q = (v - bias.float()[:, None]).div_(scale.float()[:, None]).round_().clamp_(0, n)
        q = q.to(torch.uint8)
        if bits == 4:
            q = q[:, 0::2] | q[:, 1::2] << 4
        assert torch.equal(s[e:e + 16].reshape(-1).view(torch.int16), scale.view(torch.int16))
        assert torch.equal(b[e:e + 16].reshape(-1).view(torch.int16), bias.view(torch.int16))
        assert torch.equal(wq[e:e + 16].reshape(q.shape[0], -1).view(torch.uint8), q)
