"""INT8 x INT8 projections (h3_gemm_i8_256, kernels/gemm_integer.loom:444-485):
bits-8 activations and weights through the C ABI, bit for bit against the
oracle's G1 with bits = 8."""
import numpy as np
import pytest
import torch

import clef_i4
import oracle

pytestmark = pytest.mark.gpu

BF = oracle.f32_to_bf16
F = oracle.bf16_to_f32


def dev_bf16(a: np.ndarray) -> torch.Tensor:
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).view(torch.bfloat16).cuda()


def host_u16(t: torch.Tensor) -> np.ndarray:
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


def run(x, w, residual=None):
    n, k = w.shape
    qw = clef_i4.load_quantized_weight(dev_bf16(w), bits=8)
    a = clef_i4.prepare(dev_bf16(x), bits=8)
    got = clef_i4.project_prepared(a, qw, residual=None if residual is None else dev_bf16(residual))
    stride = oracle.activation_stride(k, 8)
    codes, scales, _ = oracle.prepare(x, stride, 8)
    w_tiled, w_scales = oracle.pack_weight(w, bits=8)
    assert np.array_equal(qw.codes.cpu().numpy().view(np.uint32), w_tiled), "packed int8 weight"
    want = oracle.gemm(codes, scales, w_tiled, w_scales, n, k, bits=8, residual=residual)
    return host_u16(got), want


@pytest.mark.parametrize("m,n,k", [(1, 256, 256), (17, 256, 768), (300, 768, 1024), (1100, 512, 2048),
                                   (64, 1024, 4096)])
def test_i8_gemm_matches_oracle(m, n, k):
    rng = np.random.default_rng(m + n + k)
    x = BF(rng.standard_normal((m, k)).astype(np.float32))
    w = BF((rng.standard_normal((n, k)) * 0.02).astype(np.float32))
    got, want = run(x, w)
    assert np.array_equal(got, want), f"{np.sum(got != want)} mismatches"


@pytest.mark.parametrize("m", [1, 255, 1030])
def test_i8_gemm_residual_matches_oracle(m):
    rng = np.random.default_rng(m)
    n, k = 256, 1024
    x = BF(rng.standard_normal((m, k)).astype(np.float32))
    w = BF((rng.standard_normal((n, k)) * 0.02).astype(np.float32))
    res = BF(rng.standard_normal((m, n)).astype(np.float32))
    got, want = run(x, w, res)
    assert np.array_equal(got, want)


# every INT8 kernel at its edges: dot products (m <= 4), split-K tiles of
# 32 x 32, 32 x 64 and 64 x 64 (fewer k-steps than waves, uneven, two rounds),
# the 128 x 128 ring (fewer k-steps than stages, as many, more, ragged rows),
# 128 x 128 and 256 x 256 two-stage tiles
@pytest.mark.parametrize("m,n,k,resid", [
    (4, 256, 256, True), (5, 256, 256, False), (33, 1024, 1280, True), (64, 2048, 768, False),
    (100, 4096, 512, True), (20, 12288, 512, False), (250, 4096, 2304, False), (130, 7168, 768, True),
    (300, 8192, 256, False), (300, 8192, 512, True), (257, 8192, 768, False), (385, 6144, 1280, True),
    (1000, 3072, 512, False), (1030, 4352, 512, True), (2100, 5120, 512, False),
    (8, 33024, 256, True), (32, 33024, 256, False), (33, 33024, 256, False)])  # wide N: 32 x 64, then 128 x 128
def test_i8_gemm_every_path(m, n, k, resid):
    """Sampled rows (block edges, a NaN row, an infinite value, the last row)
    against the oracle; two launches agree on every row."""
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn((m, k), generator=g, device="cuda", dtype=torch.bfloat16)
    w = torch.randn((n, k), generator=g, device="cuda", dtype=torch.bfloat16) * 0.02
    w[64:80] *= 1e-4
    w[96:98] = 0.0
    if m > 40:
        x[m - 5] = float("nan")
        x[37, 3] = float("inf")
    res = torch.randn((m, n), generator=g, device="cuda", dtype=torch.bfloat16) if resid else None
    q = clef_i4.load_quantized_weight(w, bits=8)
    a = clef_i4.prepare(x, bits=8)
    got = host_u16(clef_i4.project_prepared(a, q, residual=res))
    assert np.array_equal(got, host_u16(clef_i4.project_prepared(a, q, residual=res)))
    rows = sorted({0, 1 % m, m // 3, m - 1, min(37, m - 1), max(m - 5, 0), min(127, m - 1), min(128, m - 1),
                   min(255, m - 1), min(256, m - 1), m // 128 * 128 if m % 128 else m - 1})
    codes, scales, _ = oracle.prepare(host_u16(x[rows]), oracle.activation_stride(k, 8), 8)
    want = oracle.gemm(codes, scales, q.codes.cpu().numpy().view(np.uint32), q.scales.cpu().numpy(), n, k, bits=8,
                       residual=host_u16(res)[rows] if resid else None)
    nan = np.isnan(F(want))
    assert np.array_equal(nan, np.isnan(F(got[rows]))) and np.array_equal(got[rows][~nan], want[~nan])


def test_i8_gemm_extreme_codes_and_nonfinite_rows():
    """Constant rows give codes +-127 everywhere (the largest |acc|); huge
    scales saturate; NaN and Inf rows give zero codes with infinite scales."""
    m, n, k = 8, 256, 512
    x = np.zeros((m, k), dtype=np.float32)
    x[0] = 1.0
    x[1] = -3.0e38
    x[2, 5] = np.nan
    x[3, 7] = np.inf
    x[4] = np.linspace(-1, 1, k)
    x[5] = 3.0e38
    w = np.ones((n, k), dtype=np.float32)
    w[1::2] = -2.0e38
    got, want = run(BF(x), BF(w))
    assert np.array_equal(got, want)


@pytest.mark.parametrize("m", [1, 3, 8])
@pytest.mark.parametrize("n,k", [(256, 256), (512, 2304), (1024, 4096), (256, 12288)])
def test_i8_gemm_decode_rows_match_oracle(m, n, k):
    """Up to 4 rows: the v_dot4_i32_i8 kernel, k-steps of 128 k (2 to 96 of
    them over its 8 waves); 8 rows: the split-K tiles on the same k-steps; with
    and without the residual."""
    rng = np.random.default_rng(m * 100 + n + k)
    x = BF(rng.standard_normal((m, k)).astype(np.float32))
    w = BF((rng.standard_normal((n, k)) * 0.02).astype(np.float32))
    got, want = run(x, w)
    assert np.array_equal(got, want), f"{np.sum(got != want)} mismatches"
    res = BF(rng.standard_normal((m, n)).astype(np.float32))
    got, want = run(x, w, res)
    assert np.array_equal(got, want), f"residual: {np.sum(got != want)} mismatches"
