"""Edge-case weights and activations through the batched product forms: the
dequantize-once product (spiral_amd/csrc/gemm_dense.hip), the fused GEMM in
ranges of k (gemm.hip) and MUL_MAT_ID's tiled form (moe_tile.hip).

 - Q4_0, Q8_0 and Q6_K block scales of exponent 0 and 31, code -128 and
   sub-scales over the whole int8 range, as in tests/test_gpu_specials.py and
   on its bars;
 - IEEE scales (the K-quants' d and dmin, IQ4's d): subnormal, infinite and
   NaN. The batched forms answer as the form that takes the same call with
   less memory or fewer tokens, infinities and NaN in the same places;
 - infinities and NaN in x reach the outputs of their own row only.
"""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from spiral_amd import lib, ops, synth
from test_gpu_specials import (FORMATS, TOL_BF16_OUT, TOL_F32_OUT, check_product, dev_bf16, dev_u8, moe_special_case,
                               run_mul_mat, special_weights)

pytestmark = pytest.mark.gpu

IEEE_FORMATS = [O.Q4_K, O.Q5_K, O.IQ4_NL, O.IQ4_XS]
IEEE_SCALES = np.array([0x7C00, 0xFC00, 0x7E00, 0x0001, 0x83FF, 0x0000, 0x8000, 0x7BFF], dtype=np.uint16)


def ieee_weights(qtype, n_rows, k, seed):
    """Every third row has a block whose d (and, in the K-quants, dmin) is one of
    IEEE_SCALES."""
    raw = synth.make_weights(qtype, n_rows, k, seed)
    blocks = raw.reshape(n_rows, k // O.BLOCK_ELEMS[qtype], O.BLOCK_BYTES[qtype])
    rng = np.random.default_rng(seed + 5)
    fields = (0, 2) if qtype in (O.Q4_K, O.Q5_K) else (0,)
    for r in range(0, n_rows, 3):
        h = int(IEEE_SCALES[(r // 3) % IEEE_SCALES.size])
        b, f = int(rng.integers(blocks.shape[1])), fields[(r // 3 // IEEE_SCALES.size) % len(fields)]
        blocks[r, b, f], blocks[r, b, f + 1] = h & 0xFF, h >> 8
    return raw


def packed(m, k):
    return -(-m // 16) * 16 * k * 2


def same(a, b, tol):
    """Equal in infinities and NaN, and to tol of the finite outputs' root mean
    square elsewhere. Returns how many are not finite."""
    a, b = a.double(), b.double()
    assert torch.equal(torch.isnan(a), torch.isnan(b))
    inf = torch.isinf(a) | torch.isinf(b)
    assert torch.equal(a[inf], b[inf])
    fin = torch.isfinite(a)
    assert fin.any()
    row = b[fin]
    assert float((a[fin] - row).abs().max()) <= tol * max(float(row.abs().max()), 1e-30)
    return int((~fin).sum())


@pytest.mark.parametrize("qtype", FORMATS)
@pytest.mark.parametrize("out_dtype,tol", [(torch.float32, TOL_F32_OUT), (torch.bfloat16, TOL_BF16_OUT)])
def test_dense_special_weights(cuda, qtype, out_dtype, tol):
    m, n, k = 2049, 2500, 512
    assert lib().spiral_mul_mat_workspace_bytes(qtype, n, k, m) == n * k * 2
    y, wb, x = run_mul_mat(cuda, qtype, n, k, m, 500, out_dtype)
    check_product(y, wb, x, tol)


@pytest.mark.parametrize("qtype", FORMATS)
@pytest.mark.parametrize("out_dtype,tol", [(torch.float32, TOL_F32_OUT), (torch.bfloat16, TOL_BF16_OUT)])
def test_split_special_weights(cuda, qtype, out_dtype, tol):
    m, n, k = 33, 40, 8192
    assert lib().spiral_mul_mat_workspace_bytes(qtype, n, k, m) == packed(m, k) + 4 * m * n * 4
    y, wb, x = run_mul_mat(cuda, qtype, n, k, m, 510, out_dtype)
    check_product(y, wb, x, tol)


@pytest.mark.parametrize("k", [256, 2560, 5120])
def test_tile_special_weights(cuda, k):
    n_expert, n, top_k = 4, 96, 2
    n_tokens = 60 if k < 2560 else 30  # 30 and 15 pairs an expert
    w, per, ids, x, deq = moe_special_case(cuda, O.Q4_0, n_expert, n, k, n_tokens, top_k, top_k, 90)
    y = ops.mul_mat_id(O.Q4_0, w, per, n_expert, n, k, dev_bf16(x, cuda), torch.from_numpy(ids).to(cuda),
                       out_dtype=torch.float32).cpu().numpy()
    for t in range(n_tokens):
        for s in range(top_k):
            check_product(y[t, s][None, :], deq[ids[t, s]], x[t, s][None, :], TOL_F32_OUT)


# The two orders of the sum are 1e-6 apart (fp32); rounded to bf16, one step of 2^-8.
@pytest.mark.parametrize("qtype", IEEE_FORMATS)
@pytest.mark.parametrize("m,n,k", [(2049, 2500, 512), (33, 40, 8192)])
@pytest.mark.parametrize("out_dtype,tol", [(torch.float32, 1e-5), (torch.bfloat16, 2.0 ** -7)])
def test_ieee_scales(cuda, qtype, m, n, k, out_dtype, tol):
    """Dequantized once and in ranges of k, against the fused GEMM in one."""
    w = ops.to_planar(qtype, dev_u8(ieee_weights(qtype, n, k, 520), cuda), n, k)
    x = dev_bf16(synth.make_x(m, k, 521), cuda)
    assert lib().spiral_mul_mat_workspace_bytes(qtype, n, k, m) > packed(m, k)
    y = ops.mul_mat(qtype, w, n, k, x, out_dtype=out_dtype)
    one = ops.mul_mat(qtype, w, n, k, x, out_dtype=out_dtype,
                      workspace=torch.empty(packed(m, k), dtype=torch.uint8, device=cuda))
    assert same(y, one, tol) > 0


@pytest.mark.parametrize("qtype", IEEE_FORMATS)
@pytest.mark.parametrize("glu", [False, True])
def test_tile_ieee_scales(cuda, qtype, glu):
    """The tiled form, against the same tokens four at a time (streaming form)."""
    n_expert, n, k, n_tokens = 3, 96, 512, 90
    w = torch.stack([ops.to_planar(qtype, dev_u8(ieee_weights(qtype, n, k, 530 + e), cuda), n, k)
                     for e in range(n_expert)])
    x = dev_bf16(synth.make_x(n_tokens, k, 540), cuda).view(n_tokens, 1, k)
    ids = (torch.arange(n_tokens, dtype=torch.int32, device=cuda) % n_expert)[:, None].contiguous()

    def call(xs, i):
        if glu:
            return ops.mul_mat_id_glu(qtype, w, w.stride(0), n_expert, n, k, xs, i, ops.GLU_SWIGLU,
                                      out_dtype=torch.float32)
        return ops.mul_mat_id(qtype, w, w.stride(0), n_expert, n, k, xs, i, out_dtype=torch.float32)

    y = call(x, ids)
    parts = torch.cat([call(x[t:t + 4].contiguous(), ids[t:t + 4].contiguous()) for t in range(0, n_tokens, 4)])
    assert same(y, parts, 0.0) > 0


@pytest.mark.parametrize("m,n,k", [(2049, 2500, 512), (33, 40, 8192)])
def test_special_activations(cuda, m, n, k):
    qtype = O.Q4_0
    w = ops.to_planar(qtype, dev_u8(synth.make_weights(qtype, n, k, 550), cuda), n, k)
    x = dev_bf16(synth.make_x(m, k, 551), cuda)
    clean = ops.mul_mat(qtype, w, n, k, x, out_dtype=torch.float32)
    bad = torch.tensor([0, 15, 16, m - 1], device=cuda)
    x[bad, torch.tensor([0, k - 1, 65, 130], device=cuda)] = torch.tensor(
        [float("inf"), float("nan"), float("-inf"), float("nan")], dtype=torch.bfloat16, device=cuda)
    y = ops.mul_mat(qtype, w, n, k, x, out_dtype=torch.float32)
    assert not torch.isfinite(y[bad]).any()
    rest = torch.ones(m, dtype=torch.bool, device=cuda)
    rest[bad] = False
    assert torch.equal(y[rest], clean[rest])


def test_tile_special_activations(cuda):
    qtype, n_expert, n, k, n_tokens = O.Q4_0, 3, 96, 512, 135  # 45 tokens an expert, tiles of 64
    w = torch.stack([ops.to_planar(qtype, dev_u8(synth.make_weights(qtype, n, k, 560 + e), cuda), n, k)
                     for e in range(n_expert)])
    x = dev_bf16(synth.make_x(n_tokens, k, 570), cuda).view(n_tokens, 1, k)
    ids = (torch.arange(n_tokens, dtype=torch.int32, device=cuda) % n_expert)[:, None].contiguous()
    clean = ops.mul_mat_id(qtype, w, w.stride(0), n_expert, n, k, x, ids, out_dtype=torch.float32)
    x[7, 0, 3], x[134, 0, k - 1] = float("nan"), float("inf")
    y = ops.mul_mat_id(qtype, w, w.stride(0), n_expert, n, k, x, ids, out_dtype=torch.float32)
    assert not torch.isfinite(y[[7, 134]]).any()
    rest = [t for t in range(n_tokens) if t not in (7, 134)]
    assert torch.equal(y[rest], clean[rest])
