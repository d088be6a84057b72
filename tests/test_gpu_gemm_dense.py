"""GPU parity of the many-row products that dequantize the weights once into
the workspace (spiral_amd/csrc/gemm_dense.hip): every tile the dispatch
chooses, ragged rows of x and of W, one to twenty k steps of 64 (the LDS
stages' prologue, their steady state and the F32 accumulator flushes), strided
and misaligned outputs, the fused fallback, and a matrix taken in two chunks.
Held to the product bars of tests/test_gpu_parity.py against float64, and the
F32 and bf16 errors to the fused form's.
"""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from spiral_amd import lib, ops, synth
from test_gpu_parity import REL_TOL, REL_TOL_EXACT_W, _mul_mat_case, dev_bf16, dev_u8, rel_err

pytestmark = pytest.mark.gpu

# One row or more past whole tiles in both directions; the tile widths follow
# from the sizes (128 x 128, 256 x 128, .. 256 x 256).
SHAPES = [
    (O.Q4_0, 257, 7001, 64),
    (O.Q4_0, 1300, 1501, 96 * 12),
    (O.Q8_0, 769, 5003, 128),
    (O.Q5_K, 1025, 7001, 256),
    (O.IQ4_NL, 1300, 7001, 192),
    (O.IQ4_XS, 1537, 7001, 256),
    (O.Q6_K, 2049, 7001, 256),
    (O.Q4_K, 513, 7001, 1024),
]


def takes_dense(qtype, m, n, k):
    return lib().spiral_mul_mat_workspace_bytes(qtype, n, k, m) == n * k * 2


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("qtype,m,n,k", SHAPES)
def test_dense_tiles(cuda, qtype, m, n, k, out_dtype):
    assert takes_dense(qtype, m, n, k)
    y, ref = _mul_mat_case(cuda, qtype, n, k, m, 200, out_dtype)
    assert rel_err(y, ref) <= (REL_TOL if out_dtype == torch.bfloat16 else REL_TOL_EXACT_W)


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_dense_strides_and_fallback(cuda, out_dtype):
    """x and y wider than k and n, y rows off 16-byte alignment; a workspace
    of the packed x alone still runs (the fused GEMM), and agrees."""
    qtype, m, n, k = O.Q8_0, 513, 5003, 128
    assert takes_dense(qtype, m, n, k)
    raw = synth.make_weights(qtype, n, k, 210)
    x = synth.make_x(m, k, 211)
    w = ops.to_planar(qtype, dev_u8(raw, cuda), n, k)
    xw = torch.full((m, k + 40), float("nan"), dtype=torch.bfloat16, device=cuda)
    xw[:, :k] = dev_bf16(x, cuda)
    ref = O.matmul_f64(O.dequant(qtype, raw, n, k), x)
    tol = REL_TOL if out_dtype == torch.bfloat16 else REL_TOL_EXACT_W
    off = 2  # elements: 4 or 8 bytes
    for ws in (None, torch.empty(-(-m // 16) * 16 * k * 2, dtype=torch.uint8, device=cuda)):
        flat = torch.full((m * (n + 13) + off,), 7.0, dtype=out_dtype, device=cuda)
        yw = flat[off:].view(m, n + 13)
        ops.mul_mat(qtype, w, n, k, xw[:, :k], out=yw[:, :n], workspace=ws)
        torch.cuda.synchronize()
        got = yw.float().cpu().numpy()
        assert rel_err(got[:, :n], ref) <= tol
        assert (got[:, n:] == 7.0).all() and (flat[:off] == 7.0).all()  # nothing written outside


def test_dense_chunks(cuda):
    """A matrix above the workspace's 256 MiB of bf16: rows on both sides of
    the chunk boundary (4352) and the last ones."""
    qtype, m, n, k = O.Q4_K, 1500, 8500, 16384
    assert lib().spiral_mul_mat_workspace_bytes(qtype, n, k, m) == 4352 * k * 2
    raw = synth.make_weights(qtype, n, k, 220)
    x = synth.make_x(m, k, 221)
    w = ops.to_planar(qtype, dev_u8(raw, cuda), n, k)
    y = ops.mul_mat(qtype, w, n, k, dev_bf16(x, cuda), out_dtype=torch.float32).cpu().numpy()
    rows = np.r_[0:4, 4348:4356, 8496:8500]
    sub = np.ascontiguousarray(raw.reshape(n, -1)[rows]).reshape(-1)
    ref = O.matmul_f64(O.dequant(qtype, sub, len(rows), k), x)
    assert rel_err(y[:, rows], ref) <= REL_TOL_EXACT_W


# F32 results sum in chains no longer than the fused form's quarters of k, so that
# rows of a few k steps are as exact. The errors are root mean squares over a
# million outputs or more, within 1 % of their expectation; one chain every 1024 k
# had 1.3 to 1.9 times the fused form's at k = 512 to 2048.
@pytest.mark.parametrize("m,n,k", [(513, 7001, 512), (513, 7001, 1024), (1025, 4097, 512), (1025, 4097, 1024),
                                   (2049, 4097, 512), (2049, 4097, 1536), (2049, 4097, 2048), (2049, 4097, 4096),
                                   (2049, 7001, 64), (2049, 7001, 128), (2049, 7001, 192), (2049, 7001, 256)])
def test_f32_error_at_most_the_fused_forms(cuda, m, n, k):
    qtype = O.Q4_0
    w = ops.to_planar(qtype, dev_u8(synth.make_weights(qtype, n, k, 230), cuda), n, k)
    x = dev_bf16(synth.make_x(m, k, 231), cuda)
    ref = x.double() @ ops.dequant(qtype, w, n, k).double().t()
    fused = ops.mul_mat(qtype, w, n, k, x, out_dtype=torch.float32,
                        workspace=torch.empty(-(-m // 16) * 16 * k * 2, dtype=torch.uint8, device=cuda))
    y = ops.mul_mat(qtype, w, n, k, x, out_dtype=torch.float32)
    assert torch.equal(y, fused) == (k < 192)  # shorter rows keep the fused form
    rms = [float((a.double() - ref).square().mean().sqrt()) for a in (y, fused)]
    assert rms[0] <= 1.02 * rms[1], rms


# A bf16 result is one fp32 chain over k, up to 7e-7 of the outputs from the exact
# sum; its rounding is 1.66e-3 from it, so the chain adds (7e-7 / 1.66e-3)^2 / 2 =
# 1e-7 of the error at most.
@pytest.mark.parametrize("m,n,k", [(513, 7001, 1024), (1025, 7001, 4096), (2049, 7001, 14336)])
def test_bf16_error_is_the_roundings(cuda, m, n, k):
    qtype = O.Q4_K
    w = ops.to_planar(qtype, dev_u8(synth.make_weights(qtype, n, k, 240), cuda), n, k)
    x = dev_bf16(synth.make_x(m, k, 241), cuda)
    ref = x.double() @ ops.dequant(qtype, w, n, k).double().t()
    fused = ops.mul_mat(qtype, w, n, k, x, workspace=torch.empty(-(-m // 16) * 16 * k * 2, dtype=torch.uint8, device=cuda))
    y = ops.mul_mat(qtype, w, n, k, x)
    assert not torch.equal(y, fused)
    rms = [float((a.double() - ref).square().mean().sqrt()) for a in (y, fused)]
    assert rms[0] <= (1 + 1e-6) * rms[1], rms


# 20 k steps: prologue, steady state with its load counts, F32 flushes (every 5
# steps) and tail. The sizes are the smallest that the tile estimate gives to
# 128 x 128, 256 x 128, x 160, x 192, x 224 and x 256 (F32 stops at 160).
@pytest.mark.parametrize("m,n", [(257, 5454), (257, 10883), (513, 10883), (513, 13628), (769, 12347), (769, 14360)])
@pytest.mark.parametrize("out_dtype,tol", [(torch.bfloat16, REL_TOL), (torch.float32, REL_TOL_EXACT_W)])
def test_dense_tiles_long_rows(cuda, m, n, out_dtype, tol):
    qtype, k = O.Q6_K, 1280
    assert takes_dense(qtype, m, n, k)
    w = ops.to_planar(qtype, dev_u8(synth.make_weights(qtype, n, k, 250), cuda), n, k)
    x = dev_bf16(synth.make_x(m, k, 251), cuda)
    y = ops.mul_mat(qtype, w, n, k, x, out_dtype=out_dtype)
    ref = x.double() @ ops.dequant(qtype, w, n, k).double().t()
    assert rel_err(y.float().cpu().numpy(), ref.cpu().numpy()) <= tol
