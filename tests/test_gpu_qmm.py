"""Dense quantized products at prefill sizes on the matrix cores
(rmoe_gather_qmm without index arrays, 64 rows or more, bf16 out): the
reference's own prefill QMM datasets (native/src/quantized_qmm_probe.mm:
243-307, x bf16 [64, 2048] against an 8- or 4-bit [4096, 2048] weight) and
random shapes, against the oracle.

The matrix-core path rounds every dequantised weight to bf16 (the prefill
contract), so it is held tightly to x . bf16(w)^T, and to the reference's
fp32-weight oracle and its recorded checksum within the error that rounding
the weights and the outputs to bf16 can cause."""

import json
from pathlib import Path

import numpy as np
import pytest

from helpers import dev_bf16, dev_i32, host_bf16
from oracle import moe_ref as M

pytestmark = pytest.mark.gpu

GOLDEN = json.loads((Path(__file__).parent / "golden" / "reference_vectors.json").read_text())
U = 2.0 ** -8  # bf16 unit roundoff


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from runnel_amd import _lib
    _lib.load()
    return torch


def _bf16_weight_product(x_bits, w, s, b, bits):
    """float64 x . bf16(fl32(q s + b))^T and the weights' rounding error."""
    w64 = M.dequantize(w, s, b, bits, dtype=np.float64)
    wb = M.round_bf16(w64.astype(np.float32)).astype(np.float64)
    x = M.bf16_to_f32(x_bits).astype(np.float64)
    return x @ wb.T, x, w64, wb


def _check_contract(got_bits, ref64, x, wb):
    """Within one bf16 step of the bf16-weight product plus the fp32
    accumulation's error (order unknown), elementwise."""
    got = M.bf16_to_f32(got_bits).astype(np.float64)
    acc = (np.abs(x) @ np.abs(wb).T) * x.shape[1] * 2.0 ** -24
    tol = U * np.abs(ref64) + acc + 1e-30
    bad = np.abs(got - ref64) > 2 * tol
    return int(bad.sum()), got


@pytest.mark.parametrize("case", GOLDEN["qmm"], ids=lambda c: Path(c["source"]).stem)
def test_reference_qmm_dataset_on_the_matrix_cores(torch_cuda, case):
    torch = torch_cuda
    from runnel_amd import native
    bits = case["bits"]
    ds = M.qmm_dataset(bits, case["tokens"], case["outputs"], case["reduction_size"])
    y = native.gather_qmm(dev_bf16(ds["x"]), dev_i32(ds["w"]), dev_bf16(ds["scales"]),
                          dev_bf16(ds["biases"]), bits)
    torch.cuda.synchronize()
    ref64, x, w64, wb = _bf16_weight_product(ds["x"], ds["w"], ds["scales"], ds["biases"], bits)
    nbad, got = _check_contract(host_bf16(y), ref64, x, wb)
    assert nbad == 0
    # against the reference's fp32-weight oracle (whose checksum the CPU
    # tests pin to the recorded one): weight rounding moves each output by at
    # most sum_k |x| |w - bf16(w)|, the bf16 output by U |y|
    exp = ds["expected"].astype(np.float64)
    dw = np.abs(w64 - wb)
    bound = np.abs(x) @ dw.T + U * np.abs(exp) + (np.abs(x) @ np.abs(wb).T) * 2048 * 2.0 ** -24
    assert (np.abs(got - exp) <= bound * 1.01 + 1e-6).all()
    # the recorded checksum (3 decimals), within the summed bound
    assert abs(got.sum() - case["reference_checksum"]) <= bound.sum() + 5e-4
    # and far inside it in practice: the rounding errors mostly cancel
    print(f"q{bits}: checksum {got.sum():.3f} vs recorded {case['reference_checksum']:.3f} "
          f"(bound {bound.sum():.1f})", flush=True)


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("shape", [(64, 256, 128), (130, 768, 384), (300, 512, 2048)])
def test_dense_qmm_random_shapes(torch_cuda, bits, shape):
    """Partial row tiles (130, 300 rows), several column and K tiles."""
    torch = torch_cuda
    from runnel_amd import native
    Mr, N, K = shape
    rng = np.random.default_rng(Mr + N + K + bits)
    w = rng.standard_normal((N, K), dtype=np.float32) * np.float32(0.02)
    words, s, b = M.quantize(w, bits)
    xb = M.make_x(5 + Mr, Mr, K)
    y = native.gather_qmm(dev_bf16(xb), dev_i32(words), dev_bf16(s), dev_bf16(b), bits)
    torch.cuda.synchronize()
    ref64, x, _, wb = _bf16_weight_product(xb, words, s, b, bits)
    nbad, _ = _check_contract(host_bf16(y), ref64, x, wb)
    assert nbad == 0


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("Mr,N,K,E", [
    (32, 80, 256, 1), (40, 512, 2048, 1), (63, 130, 3072, 1),      # one matrix
    (64, 2048, 512, 8), (130, 1100, 256, 3), (530, 144, 512, 40),  # gathered
    (128, 520, 512, 1), (300, 64, 2048, 200), (128, 72, 4096, 5),
    # either side of the lines below which qmv_kernel takes the call
    (32, 1023, 256, 1), (32, 1025, 256, 1), (63, 153, 3072, 1), (63, 152, 3072, 1),
    (1030, 72, 1024, 40), (1100, 64, 2048, 200), (128, 264, 4096, 5), (128, 264, 4096, 103)])
def test_rows_sharing_experts(torch_cuda, bits, Mr, N, K, E):
    """Many rows a call, fp32 out: row groups that fill, exceed or just miss
    16, windows of 512 rows, column remainders, ids out of range (zero rows)
    and 1 to 16 slices of K.  Every product and sum is fp32, so each output is
    within K roundings of |x| . (|q - c| s + |b + c s|) of the 64-bit value
    (c the middle code), and in norm far closer."""
    torch = torch_cuda
    from runnel_amd import native
    rng = np.random.default_rng(Mr + N + K + bits)
    w = rng.standard_normal((E, N, K), dtype=np.float32) * np.float32(0.02)
    words, s, b = M.quantize(w, bits)
    X = max(1, Mr // 3) if E > 1 or Mr >= 64 else Mr
    xb = M.make_x(9 + Mr, X, K)
    dev = (dev_i32(words), dev_bf16(s), dev_bf16(b))
    if E == 1 and Mr < 64:
        lhs, rhs = np.arange(Mr), np.zeros(Mr, np.int64)
        y = native.gather_qmm(dev_bf16(xb), *(t[0] for t in dev), bits, out_dtype=torch.float32)
    else:
        lhs, rhs = rng.integers(0, X, Mr), rng.integers(0, E, Mr)
        lhs[5], rhs[Mr - 1], rhs[17] = -1, E, -3
        y = native.gather_qmm(dev_bf16(xb), *dev, bits,
                              rhs_indices=torch.from_numpy(rhs.astype(np.int32)).cuda(),
                              lhs_indices=torch.from_numpy(lhs.astype(np.int32)).cuda(),
                              out_dtype=torch.float32)
    got = y.cpu().numpy().astype(np.float64)
    ok = (lhs >= 0) & (rhs >= 0) & (rhs < E)
    assert not got[~ok].any()
    x = M.bf16_to_f32(xb).astype(np.float64)[lhs * ok]
    w64 = M.dequantize(words, s, b, bits, dtype=np.float64)
    s64 = np.repeat(M.bf16_to_f32(s).astype(np.float64), 64, -1)
    b64 = np.repeat(M.bf16_to_f32(b).astype(np.float64), 64, -1)
    c = 2 ** (bits - 1)
    size = np.abs(w64 - b64 - c * s64) + np.abs(b64 + c * s64)
    ref = np.zeros_like(got)
    bound = np.zeros_like(got)
    for e in np.unique(rhs[ok]):
        r = np.nonzero(ok & (rhs == e))[0]
        ref[r], bound[r] = x[r] @ w64[e].T, np.abs(x[r]) @ size[e].T
    err = np.abs(got - ref)
    assert (err <= K * 2.0 ** -24 * bound).all()
    assert np.linalg.norm(err) <= 4 * 2.0 ** -24 * np.linalg.norm(ref)


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("shift", [1, 2, 4])
def test_scales_at_any_address(torch_cuda, bits, shift):
    """Scales and biases 2, 4 and 8 bytes past a 16-byte boundary: only the
    last suit the kernel that many rows share; the products are the same to
    fp32 accuracy (K roundings; see test_rows_sharing_experts)."""
    torch = torch_cuda
    from runnel_amd import native
    rng = np.random.default_rng(bits)
    Mr, N, K, E = 128, 520, 1024, 4
    w = rng.standard_normal((E, N, K), dtype=np.float32) * np.float32(0.02)
    words, s, b = M.quantize(w, bits)
    xb = M.make_x(11, Mr, K)
    rhs = torch.from_numpy(rng.integers(0, E, Mr).astype(np.int32)).cuda()

    def moved(a):
        t = torch.empty(a.size + 8, dtype=torch.bfloat16, device="cuda")
        v = t[shift:shift + a.size].view(a.shape)
        v.copy_(dev_bf16(a))
        return v

    def product(sc, bi):
        return native.gather_qmm(dev_bf16(xb), dev_i32(words), sc, bi, bits, rhs_indices=rhs,
                                 out_dtype=torch.float32).double()
    ref, got = product(dev_bf16(s), dev_bf16(b)), product(moved(s), moved(b))
    assert torch.equal(got, ref) == (shift == 4)
    assert (got - ref).norm() <= 8 * 2.0 ** -24 * ref.norm()


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_non_finite_row_stays_alone(torch_cuda, bits, bad):
    """A row of x that holds a NaN or an infinity gives no finite output and
    leaves the rows that share its expert as they are."""
    torch = torch_cuda
    from runnel_amd import native
    rng = np.random.default_rng(7)
    w = rng.standard_normal((2, 512, 1024), dtype=np.float32) * np.float32(0.02)
    words, s, b = M.quantize(w, bits)
    x = dev_bf16(M.make_x(12, 128, 1024))
    rhs = (torch.arange(128, device="cuda") % 2).to(torch.int32)
    dev = (dev_i32(words), dev_bf16(s), dev_bf16(b))
    ref = native.gather_qmm(x, *dev, bits, rhs_indices=rhs)
    x[37, 500] = bad
    got = native.gather_qmm(x, *dev, bits, rhs_indices=rhs)
    assert not got[37].isfinite().any()
    keep = torch.arange(128, device="cuda") != 37
    assert torch.equal(got[keep], ref[keep])


@pytest.mark.parametrize("Mr,N,K,index", [
    (131072 + 600, 2048, 4096, "both"),   # qmv_rows_kernel, 2^15 threads a row
    (131072 + 600, 2048, 4096, "rhs"),    # and x in order
    (262144 + 48, 4096, 4096, "none"),    # the same on one matrix, 16 rows a group
    (262144 + 5, 2048, 128, "rhs"),       # qmv_kernel, 2^14 threads a row
])
def test_calls_of_more_than_one_launch(torch_cuda, Mr, N, K, index):
    """Products of 2^32 threads and more (K and N chosen for the most threads
    a row).  The rows repeat with a period of 4095, which divides no piece, so
    every piece has to find its own x rows, indices and output rows; a row's
    value does not depend on the others, so the repeats are equal bit for
    bit."""
    torch = torch_cuda
    from runnel_amd import native
    print(f"{Mr} x {N} x {K}, indices: {index}", flush=True)
    P, E = 4095, 1 if index == "none" else 3
    rng = np.random.default_rng(Mr + K)
    w = rng.standard_normal((E, N, K), dtype=np.float32) * np.float32(0.02)
    wq, s, b = native.quantize(torch.from_numpy(w).cuda(), 8)
    base = dev_bf16(M.make_x(31, P, K))
    at = torch.arange(Mr, device="cuda") % P
    rhs = (at % E).to(torch.int32)
    dt = torch.float32 if index == "none" else torch.bfloat16
    if index == "none":
        y = native.gather_qmm(base[at], wq[0], s[0], b[0], 8, out_dtype=dt)
    elif index == "rhs":
        y = native.gather_qmm(base[at], wq, s, b, 8, rhs_indices=rhs, out_dtype=dt)
    else:
        y = native.gather_qmm(base, wq, s, b, 8, rhs_indices=rhs,
                              lhs_indices=at.to(torch.int32), out_dtype=dt)
    torch.cuda.synchronize()
    first = y[:P]
    for r in range(P, Mr, P):
        assert torch.equal(y[r:r + P], first[:Mr - r]), r
    few = torch.arange(0, P, 97, device="cuda")
    wf = native.dequantize(wq, s, b, 8).double()
    ref = torch.stack([wf[int(rhs[i])] @ base[i].double() for i in few])
    err = (first[few].double() - ref).norm() / ref.norm()
    assert err <= (2.0 ** -8 if dt == torch.bfloat16 else 1e-6)
