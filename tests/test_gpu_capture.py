"""The batched product forms recorded in a HIP graph: dequantized once, in ranges
of k, tiled and fused MUL_MAT_ID. Each graph is replayed several times on new
inputs, with eager calls between the replays, and every replay equals the eager
result bit for bit.
"""

import pytest
import torch

from oracle import oracle as O
from spiral_amd import lib, ops, synth
from test_gpu_parity import dev_bf16, dev_u8

pytestmark = pytest.mark.gpu


def replays(call, x, fresh):
    """Records call(out) over x, then replays it on fresh(seed) inputs."""
    out = call(None)  # eager: allocates and warms up
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(out)
    for seed in range(4):
        x.copy_(fresh(seed))
        out.fill_(float("nan"))
        graph.replay()
        got = out.clone()
        want = call(None)
        torch.cuda.synchronize()
        assert torch.equal(got, want)  # equal: no NaN is left


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("qtype,m,n,k", [(O.Q4_K, 1025, 4097, 512), (O.Q4_0, 33, 40, 8192), (O.Q6_K, 130, 100, 512)])
def test_mul_mat(cuda, qtype, m, n, k, out_dtype):
    w = ops.to_planar(qtype, dev_u8(synth.make_weights(qtype, n, k, 1), cuda), n, k)
    x = dev_bf16(synth.make_x(m, k, 2), cuda)
    ws = torch.empty(lib().spiral_mul_mat_workspace_bytes(qtype, n, k, m), dtype=torch.uint8, device=cuda)
    replays(lambda out: ops.mul_mat(qtype, w, n, k, x, out_dtype=out_dtype, out=out, workspace=ws), x,
            lambda seed: dev_bf16(synth.make_x(m, k, 10 + seed), cuda))


@pytest.mark.parametrize("glu", [False, True])
@pytest.mark.parametrize("tokens", [40, 90, 1100])  # streaming; tiled; tiled past 1024 pairs
def test_mul_mat_id(cuda, glu, tokens):
    qtype, e, n, k = O.Q4_K, 3, 96, 512
    w = torch.stack([ops.to_planar(qtype, dev_u8(synth.make_weights(qtype, n, k, 20 + i), cuda), n, k)
                     for i in range(e)])
    x = dev_bf16(synth.make_x(tokens, k, 3), cuda).view(tokens, 1, k)
    ids = (torch.arange(tokens, dtype=torch.int32, device=cuda) % e)[:, None].contiguous()
    ws = ops.mul_mat_id_workspace(e, tokens, 1, cuda)

    def call(out):
        if glu:
            return ops.mul_mat_id_glu(qtype, w, w.stride(0), e, n, k, x, ids, ops.GLU_SWIGLU,
                                      out_dtype=torch.float32, workspace=ws, out=out)
        return ops.mul_mat_id(qtype, w, w.stride(0), e, n, k, x, ids, out_dtype=torch.float32, workspace=ws, out=out)

    replays(call, x, lambda seed: dev_bf16(synth.make_x(tokens, k, 30 + seed), cuda).view(tokens, 1, k))
