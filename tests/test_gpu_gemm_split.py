"""GPU parity of the fused GEMM with its k range split between workgroups
(spiral_amd/csrc/gemm.hip: k_splits): two to eight ranges, a k tail in the
last one, unequal ranges, ragged rows, strided and misaligned outputs, and a
workspace without room for the sums (one range). Held to the product bars of
tests/test_gpu_parity.py against the float64 oracle.
"""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from spiral_amd import lib, ops, synth
from test_gpu_parity import REL_TOL, REL_TOL_EXACT_W, _mul_mat_case, dev_bf16, dev_u8, rel_err

pytestmark = pytest.mark.gpu


def packed(m, k):
    return -(-m // 16) * 16 * k * 2


def splits(qtype, m, n, k):
    return (lib().spiral_mul_mat_workspace_bytes(qtype, n, k, m) - packed(m, k)) // (m * n * 4)


# (format, rows of x, n, k, ranges): 32-element blocks take a k tail of 32, 64 or 96.
SHAPES = [
    (O.Q4_0, 17, 300, 4096 + 96, 2),
    (O.Q8_0, 130, 64, 6 * 1024 + 32, 3),
    (O.IQ4_NL, 33, 20, 2048 * 8 + 64, 8),
    (O.Q6_K, 77, 1000, 2048 * 4 + 256, 4),
    (O.Q4_K, 200, 132, 2048 * 5 + 256, 5),
    (O.Q5_K, 128, 260, 4096, 2),
    (O.IQ4_XS, 47, 68, 2048 * 7, 7),
]


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("qtype,m,n,k,nz", SHAPES)
def test_split_ranges(cuda, qtype, m, n, k, nz, out_dtype):
    assert splits(qtype, m, n, k) == nz
    y, ref = _mul_mat_case(cuda, qtype, n, k, m, 300, out_dtype)
    assert rel_err(y, ref) <= (REL_TOL if out_dtype == torch.bfloat16 else REL_TOL_EXACT_W)


def test_unsplit_rules(cuda):
    """Columns that are no multiple of four, square projections, short rows and
    grids that fill the chip keep one range and the packed x alone."""
    for m, n, k in ((17, 301, 8192), (17, 4096, 4096), (77, 1024, 2048), (2000, 1024, 8192)):
        assert splits(O.Q4_0, m, n, k) == 0


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_split_strides_and_small_workspace(cuda, out_dtype):
    qtype, m, n, k = O.Q4_0, 40, 100, 4096
    assert splits(qtype, m, n, k) == 2
    raw = synth.make_weights(qtype, n, k, 310)
    x = synth.make_x(m, k, 311)
    w = ops.to_planar(qtype, dev_u8(raw, cuda), n, k)
    ref = O.matmul_f64(O.dequant(qtype, raw, n, k), x)
    tol = REL_TOL if out_dtype == torch.bfloat16 else REL_TOL_EXACT_W
    off = 2  # elements: 4 or 8 bytes past the allocation's alignment
    for ws in (None, torch.empty(packed(m, k), dtype=torch.uint8, device=cuda)):
        flat = torch.full((m * (n + 5) + off,), 7.0, dtype=out_dtype, device=cuda)
        yw = flat[off:].view(m, n + 5)
        ops.mul_mat(qtype, w, n, k, dev_bf16(x, cuda), out=yw[:, :n], workspace=ws)
        torch.cuda.synchronize()
        got = yw.float().cpu().numpy()
        assert rel_err(got[:, :n], ref) <= tol
        assert (got[:, n:] == 7.0).all() and (flat[:off] == 7.0).all()  # nothing written outside
