"""GPU parity of MUL_MAT_ID's tiled form (spiral_amd/csrc/moe_tile.hip), which
takes batches of 24 routed tokens an expert or more (13 past k = 2304): every
format it has, rows
that are no multiple of its 96 (48 features with GLU), of 16 or of 4, one to five
super-blocks of k, experts of no tokens, of one, and of counts at the edges of
its token tiles (32, 64, 80 and over), per-slot inputs, ids routed nowhere, the
fused GLU form merged and split, every GLU variant. Up to k = 4096 equal bit for
bit to the same tokens in small calls (the streaming form, which ends there), and
to the oracle within the product bars at every k.
"""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from spiral_amd import ops
from test_gpu_parity import _moe_inputs, _moe_ref, check_moe, dev_bf16

pytestmark = pytest.mark.gpu

FORMATS = [O.Q4_0, O.Q4_K, O.Q5_K, O.IQ4_NL, O.IQ4_XS]


def ids_of(counts):
    """[tokens, 1] ids giving expert e counts[e] tokens, shuffled; the last
    entry counts the tokens routed nowhere."""
    ids = np.concatenate([np.full(c, e if e + 1 < len(counts) else -1) for e, c in enumerate(counts)])
    return np.random.default_rng(1).permutation(ids).astype(np.int32)[:, None]


def small_calls(call, x, ids, step):
    return torch.cat([call(x[t:t + step].contiguous(), ids[t:t + step].contiguous())
                      for t in range(0, ids.shape[0], step)])


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,k", [(96, 256), (100, 768), (198, 1280), (8, 512)])
@pytest.mark.parametrize("qtype", FORMATS)
def test_tile(cuda, qtype, n, k, out_dtype):
    ids = ids_of([32, 1, 0, 64, 81, 7])  # 178 pairs routed to 5 experts
    e, tokens = 5, ids.shape[0]
    w, per, raws, ids, x = _moe_inputs(cuda, qtype, e, n, k, tokens, 1, 1, 400, ids)
    xd, idd = dev_bf16(x, cuda), torch.from_numpy(ids).to(cuda)

    def call(xs, i):
        return ops.mul_mat_id(qtype, w, per, e, n, k, xs, i, out_dtype=out_dtype)

    y = call(xd, idd)
    assert torch.equal(y, small_calls(call, xd, idd, 10))
    got = y.float().cpu().numpy()
    assert not got[ids < 0].any()
    check_moe(got, _moe_ref(qtype, raws, n, k, ids, x), out_dtype == torch.float32)


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("F,k", [(48, 256), (50, 768), (132, 1024)])
@pytest.mark.parametrize("qtype", FORMATS)
def test_tile_glu(cuda, qtype, F, k, split):
    """Merged: equal to the product and the standalone GLU. Split: the same
    stacks' halves as two matrices; two tokens slots an expert pair."""
    e, tokens, top = 4, 160, 2
    n = 2 * F
    w, per, raws, ids, x = _moe_inputs(cuda, qtype, e, n, k, tokens, top, 1, 410)
    xd, idd = dev_bf16(x, cuda), torch.from_numpy(ids).to(cuda)
    prod = ops.mul_mat_id(qtype, w, per, e, n, k, xd, idd, out_dtype=torch.float32)
    want = ops.glu(prod, ops.GLU_SWIGLU)
    if not split:
        got = ops.mul_mat_id_glu(qtype, w, per, e, n, k, xd, idd, ops.GLU_SWIGLU, out_dtype=torch.float32)
    else:
        half = [torch.stack([ops.to_planar(qtype, torch.from_numpy(np.ascontiguousarray(
            r.reshape(n, -1)[i * F:(i + 1) * F]).reshape(-1)).to(cuda), F, k) for r in raws]) for i in range(2)]
        got = ops.mul_mat_id_glu_split(qtype, half[0], half[1], half[0].shape[1], e, F, k, xd, idd, ops.GLU_SWIGLU,
                                       out_dtype=torch.float32)
    torch.cuda.synchronize()
    assert torch.equal(got, want)


@pytest.mark.parametrize("qtype", FORMATS)
def test_tile_slots_and_many_tiles(cuda, qtype):
    """Per-slot inputs and an expert of several tiles; a base address of y that
    is only 4-byte aligned."""
    e, n, k, tokens, top = 3, 70, 512, 300, 2
    w, per, raws, ids, x = _moe_inputs(cuda, qtype, e, n, k, tokens, top, top, 420)
    xd, idd = dev_bf16(x, cuda), torch.from_numpy(ids).to(cuda)

    def call(xs, i):
        flat = torch.full((i.shape[0] * top * n + 1,), 7.0, dtype=torch.float32, device=cuda)
        ops.mul_mat_id(qtype, w, per, e, n, k, xs, i, out=flat[1:].view(i.shape[0], top, n))
        assert flat[0] == 7.0
        return flat[1:].view(i.shape[0], top, n)

    y = call(xd, idd)
    assert torch.equal(y, small_calls(call, xd, idd, 10))
    check_moe(y.cpu().numpy(), _moe_ref(qtype, raws, n, k, ids, x), True)


# Which form ran shows in the workspace: with at most 1024 pairs only the tiled
# form has the routing lists written there. Rows of up to 1152 k stay with the
# streaming form while its passes of 64 tokens hold the average expert with room
# (33 to 44 tokens; 65 to 89 with many rows), which is the faster one there.
@pytest.mark.parametrize("e,n,k,per,tiled", [
    (8, 96, 768, 23, False), (8, 96, 768, 24, True), (8, 96, 768, 32, True), (8, 96, 768, 33, False),
    (8, 96, 1024, 44, False), (8, 96, 768, 45, True), (8, 96, 768, 64, True), (8, 96, 768, 72, True),
    (8, 15000, 768, 64, True), (8, 15000, 768, 65, False), (8, 15000, 512, 89, False), (8, 15000, 512, 90, True),
    (8, 96, 1280, 40, True), (8, 96, 2560, 13, True), (8, 96, 2560, 12, False),
])
def test_form_by_tokens_an_expert(cuda, e, n, k, per, tiled):
    qtype, tokens = O.Q4_K, per * e
    w = torch.zeros((e, O.row_bytes(qtype, k) * n), dtype=torch.uint8, device=cuda)
    x = torch.ones((tokens, 1, k), dtype=torch.bfloat16, device=cuda)
    ids = (torch.arange(tokens, dtype=torch.int32, device=cuda) % e)[:, None].contiguous()
    ws = torch.full((4 * (e + 1 + tokens),), 0x5A, dtype=torch.uint8, device=cuda)
    y = ops.mul_mat_id(qtype, w, w.stride(0), e, n, k, x, ids, out_dtype=torch.float32, workspace=ws)
    torch.cuda.synchronize()
    assert bool((ws != 0x5A).any()) == tiled
    assert not y.any()
    if k <= 1152:  # the fused GLU form's passes take 32 tokens at most: tiled from 24 on
        ws.fill_(0x5A)
        ops.mul_mat_id_glu(qtype, w, w.stride(0), e, n, k, x, ids, ops.GLU_SWIGLU, workspace=ws)
        torch.cuda.synchronize()
        assert bool((ws != 0x5A).any()) == (per >= 24)


@pytest.mark.parametrize("per", [13, 16, 23])
@pytest.mark.parametrize("k", [2560, 4096, 5120])
@pytest.mark.parametrize("qtype", FORMATS)
def test_tile_long_rows(cuda, qtype, k, per):
    """13 to 23 tokens an expert, tiled past k = 2304; past 4096 the small calls
    run another kernel, whose sums are ordered otherwise."""
    e, n, tokens = 3, 100, 3 * per
    ids = (np.arange(tokens, dtype=np.int32) % e)[:, None]
    w, per_e, raws, ids, x = _moe_inputs(cuda, qtype, e, n, k, tokens, 1, 1, 430, ids)
    xd, idd = dev_bf16(x, cuda), torch.from_numpy(ids).to(cuda)
    ws = torch.zeros(4 * (e + 1 + tokens), dtype=torch.uint8, device=cuda)

    def call(xs, i, ws=None):
        return ops.mul_mat_id(qtype, w, per_e, e, n, k, xs, i, out_dtype=torch.float32, workspace=ws)

    y = call(xd, idd, ws)
    assert ws.any()  # the tiled form's routing lists
    if k <= 4096:
        assert torch.equal(y, small_calls(call, xd, idd, 10))
    check_moe(y.cpu().numpy(), _moe_ref(qtype, raws, n, k, ids, x), True)


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("swapped", [False, True])
@pytest.mark.parametrize("op", [ops.GLU_REGLU, ops.GLU_GEGLU, ops.GLU_SWIGLU, ops.GLU_GEGLU_ERF, ops.GLU_GEGLU_QUICK])
def test_tile_glu_variants(cuda, op, swapped, split):
    """Every activation, merged and split, halves swapped: the product and the
    standalone GLU bit for bit; bf16 output its rounding."""
    qtype, e, F, k, tokens, top = O.Q4_K, 4, 56, 512, 120, 2
    n = 2 * F
    w, per, raws, ids, x = _moe_inputs(cuda, qtype, e, n, k, tokens, top, 1, 440)
    xd, idd = dev_bf16(x, cuda), torch.from_numpy(ids).to(cuda)
    prod = ops.mul_mat_id(qtype, w, per, e, n, k, xd, idd, out_dtype=torch.float32)
    if split:
        half = [torch.stack([ops.to_planar(qtype, torch.from_numpy(np.ascontiguousarray(
            r.reshape(n, -1)[i * F:(i + 1) * F]).reshape(-1)).to(cuda), F, k) for r in raws]) for i in range(2)]
        want = ops.glu_split(prod[..., :F].contiguous(), prod[..., F:].contiguous(), op, swapped)
    else:
        want = ops.glu(prod, op, swapped)
    for dtype in (torch.float32, torch.bfloat16):
        if split:
            got = ops.mul_mat_id_glu_split(qtype, half[0], half[1], half[0].shape[1], e, F, k, xd, idd, op, swapped,
                                           out_dtype=dtype)
        else:
            got = ops.mul_mat_id_glu(qtype, w, per, e, n, k, xd, idd, op, swapped, out_dtype=dtype)
        torch.cuda.synchronize()
        assert torch.equal(got, want.to(dtype))
