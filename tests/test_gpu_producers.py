"""Fused quantizer producers beyond SwiGLU (kernels/prepare_integer_register.loom):
the attention-gate producer and the named-RMSNorm producer, through the C ABI,
bit for bit against the oracle.
"""
import numpy as np
import pytest
import torch

import clef_i4
import oracle
from test_oracle import norm_test_rows, norm_test_weight

pytestmark = pytest.mark.gpu

BF = oracle.f32_to_bf16


def dev_bf16(a: np.ndarray) -> torch.Tensor:
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).view(torch.bfloat16).cuda()


def host_u16(t: torch.Tensor) -> np.ndarray:
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


def assert_prepared(p: clef_i4.Prepared, codes: np.ndarray, scales: np.ndarray, what: str):
    words = p.width * p.bits // 32
    got = p.codes.cpu().numpy().view(np.uint32)[:, :words]
    if not np.array_equal(got, codes[:, :words]):
        bad = np.argwhere(got != codes[:, :words])
        raise AssertionError(f"{what}: {len(bad)} code words differ, first at {tuple(bad[0])}")
    assert np.array_equal(p.scales.cpu().numpy().view(np.uint32), scales.view(np.uint32)), f"{what}: scales"


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("rows,width", [(1, 256), (17, 768), (5, 2048), (33, 5120), (3, 6144), (2, 17408)])
def test_attention_gate_matches_oracle(rows, width, bits):
    """h3_prepare_attention_gate (src/quantized.rs:440-468, 615-635); both the
    multi-row (width <= 4096) and the one-row-per-workgroup kernels."""
    rng = np.random.default_rng(rows * 7 + width + bits)
    x = BF(rng.standard_normal((rows, width)).astype(np.float32))
    q = BF((rng.standard_normal((rows, 2 * width)) * 3.0).astype(np.float32))
    q[0, 256:256 + 16] = BF(np.array([np.inf, -np.inf, np.nan, 0.0, -0.0, 100.0, -100.0, 1e-30] * 2,
                                     dtype=np.float32))
    stride = oracle.activation_stride(width, bits)
    codes, scales, _ = oracle.prepare_attention_gate(x, q, stride, bits)
    p = clef_i4.prepare_attention_gate(dev_bf16(x), dev_bf16(q), bits=bits, stride=stride)
    assert_prepared(p, codes, scales, f"attention gate rows={rows} width={width} bits={bits}")


@pytest.mark.parametrize("store", [False, True])
@pytest.mark.parametrize("exceptional", [False, True])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("rows", [1, 2, 7, 65, 129])
def test_norm_matches_oracle(rows, bits, exceptional, store):
    """h3_prepare_norm[_store] on the inputs of the reference's fused-norm test
    (src/quantized.rs:1567-1610): codes, scales and stored normalized rows."""
    x = norm_test_rows(rows)
    w = norm_test_weight(exceptional=exceptional)
    stride = 5120 + 512 // bits
    codes, scales, _, normalized = oracle.prepare_norm(x, w, stride, bits)
    p, norm = clef_i4.prepare_norm(dev_bf16(x), dev_bf16(w), bits=bits, stride=stride, store=store)
    assert_prepared(p, codes, scales, f"norm rows={rows} bits={bits}")
    if store:
        assert np.array_equal(host_u16(norm), normalized)


def test_attention_gate_projection_matches_oracle():
    """Engine::project_attention_gate: gated packing then the residual G1."""
    rng = np.random.default_rng(5)
    rows, width, n = 40, 2048, 512
    x = BF(rng.standard_normal((rows, width)).astype(np.float32))
    q = BF((rng.standard_normal((rows, 2 * width)) * 2.0).astype(np.float32))
    w = BF((rng.standard_normal((n, width)) * 0.02).astype(np.float32))
    res = BF(rng.standard_normal((rows, n)).astype(np.float32))
    stride = oracle.activation_stride(width)
    codes, scales, _ = oracle.prepare_attention_gate(x, q, stride)
    w_tiled, w_scales = oracle.pack_weight(w)
    want = oracle.gemm(codes, scales, w_tiled, w_scales, n, width, residual=res)
    qw = clef_i4.load_quantized_weight(dev_bf16(w))
    got = clef_i4.project_attention_gate(dev_bf16(x), dev_bf16(q), qw, dev_bf16(res))
    assert np.array_equal(host_u16(got), want)


@pytest.mark.parametrize("tokens,experts", [(1, 128), (31, 128), (33, 64), (4096, 128), (70, 32)])
def test_router_logits_within_f32_summation_bound(tokens, experts):
    """Router gate projection (src/omni.rs:764): each logit within the f32
    summation bound of the exact dot product (float64), plus half a bf16 step
    for the final rounding. The reference's WMMA summation order is not
    reproduced, so bits are compared only through this bound."""
    hidden = 2048
    rng = np.random.default_rng(tokens + experts)
    x = BF(rng.standard_normal((tokens, hidden)).astype(np.float32))
    w = BF((rng.standard_normal((experts, hidden)) * 0.02).astype(np.float32))
    got = oracle.bf16_to_f32(host_u16(clef_i4.router_logits(dev_bf16(x), dev_bf16(w)))).astype(np.float64)
    xf, wf = oracle.bf16_to_f32(x).astype(np.float64), oracle.bf16_to_f32(w).astype(np.float64)
    exact = xf @ wf.T
    bound = hidden * 2.0 ** -23 * (np.abs(xf) @ np.abs(wf).T) + np.abs(exact) * 2.0 ** -8 + 1e-30
    assert (np.abs(got - exact) <= bound).all()


def test_router_logits_one_hot_weights_are_exact():
    """With one-hot gate rows every logit is a single exact product, so the
    output is the selected input column bit for bit: pins the token/expert
    indexing and the tail of a partial 32-token block."""
    tokens, hidden, experts = 45, 256, 128
    rng = np.random.default_rng(9)
    x = BF(rng.standard_normal((tokens, hidden)).astype(np.float32))
    w = np.zeros((experts, hidden), dtype=np.uint16)
    cols = rng.permutation(hidden)[:experts]
    w[np.arange(experts), cols] = 0x3F80  # 1.0
    got = host_u16(clef_i4.router_logits(dev_bf16(x), dev_bf16(w)))
    assert np.array_equal(got, x[:, cols])


@pytest.mark.parametrize("tokens,hidden,experts", [(1, 64, 32), (33, 448, 128), (32, 512, 96), (65, 960, 64),
                                                   (300, 1024, 128), (5, 4096, 32)])
def test_router_logits_integer_inputs_are_exact(tokens, hidden, experts):
    """Small integer inputs make every f32 partial sum exact, so the logits
    equal bf16 of the integer dot product: fewer k-steps than the load ring
    holds, ring remainders, partial token blocks and each expert group count."""
    rng = np.random.default_rng(tokens * 7 + hidden)
    x = rng.integers(-4, 5, (tokens, hidden)).astype(np.float32)
    w = rng.integers(-3, 4, (experts, hidden)).astype(np.float32)
    got = host_u16(clef_i4.router_logits(dev_bf16(BF(x)), dev_bf16(BF(w))))
    assert np.array_equal(got, BF(x @ w.T))


@pytest.mark.parametrize("hidden,experts", [(64, 32), (448, 96), (960, 64), (1024, 128), (1088, 32), (1984, 128),
                                            (2048, 128)])
def test_router_logits_few_tokens_equal_many(hidden, experts):
    """The kernel for up to 256 tokens runs the same MFMA chain as the one for
    more: its logits equal the first rows of a 300-token call bit for bit, and
    those lie within the f32 summation bound of float64."""
    g = torch.Generator(device="cuda").manual_seed(hidden + experts)
    x = torch.randn((300, hidden), generator=g, device="cuda", dtype=torch.bfloat16)
    w = torch.randn((experts, hidden), generator=g, device="cuda", dtype=torch.bfloat16)
    many = clef_i4.router_logits(x, w).view(torch.int16)
    for n in (1, 15, 16, 17, 240, 256):
        assert torch.equal(clef_i4.router_logits(x[:n].contiguous(), w).view(torch.int16), many[:n]), n
    xd, wd = x.double(), w.double()
    bound = hidden * 2.0 ** -23 * (xd.abs() @ wd.abs().t()) + 2.0 ** -8 * (xd @ wd.t()).abs() + 1e-30
    assert bool(((many.view(torch.bfloat16).double() - xd @ wd.t()).abs() <= bound).all())


@pytest.mark.parametrize("producer,width,bits,extra", [
    (0, 256, 4, 0), (0, 1024, 4, 0), (0, 768, 8, 128), (0, 4096, 8, 0), (0, 5120, 4, 1024), (0, 12288, 8, 0),
    (1, 2048, 4, 256), (1, 17408, 4, 0), (1, 6144, 8, 0), (2, 1024, 8, 0), (2, 5120, 4, 0), (3, 5120, 4, 0),
    (3, 5120, 8, 0)])
def test_prepare_filled_writes_every_word(producer, width, bits, extra):
    """clef_i4_prepare_filled on a buffer of ones bits: padding words zero,
    codes and scales those of the entry it stands for; that entry itself
    leaves the padding words as they were."""
    rows = 19
    rng = np.random.default_rng(width + bits + producer)
    stride = clef_i4.activation_stride(width, bits) + extra
    words, used = stride * bits // 32, width * bits // 32
    x = dev_bf16(BF(rng.standard_normal((rows, width)).astype(np.float32)))
    second = None if producer == 0 else dev_bf16(BF(rng.standard_normal(
        {1: (rows, width), 2: (rows, 2 * width), 3: (width,)}[producer]).astype(np.float32)))
    stream = torch.cuda.current_stream().cuda_stream
    lib = clef_i4.lib()
    filled, plain = (torch.full((rows * (words + 1),), -1, dtype=torch.int32, device="cuda") for _ in range(2))
    p2 = None if second is None else second.data_ptr()
    assert lib.clef_i4_prepare_filled(x.data_ptr(), p2, producer, rows, width, stride, bits, filled.data_ptr(),
                                      stream) == 0
    args = (rows, width, stride, bits)
    if producer == 0:
        rc = lib.clef_i4_prepare(x.data_ptr(), *args, plain.data_ptr(), stream)
    elif producer == 3:
        rc = lib.clef_i4_prepare_norm(x.data_ptr(), p2, *args, 0, plain.data_ptr(), stream)
    else:
        fn = lib.clef_i4_prepare_swiglu if producer == 1 else lib.clef_i4_prepare_attention_gate
        rc = fn(x.data_ptr(), p2, *args, plain.data_ptr(), stream)
    assert rc == 0
    f, p = filled[: rows * words].view(rows, words), plain[: rows * words].view(rows, words)
    assert torch.equal(f[:, :used], p[:, :used]) and torch.equal(filled[rows * words:], plain[rows * words:])
    assert not f[:, used:].any() and bool((p[:, used:] == -1).all())
