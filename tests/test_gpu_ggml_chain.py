"""A ggml graph computed whole equals its nodes computed one call at a time, bit
for bit: get_rows and GLU leave a bf16 copy of their rows for the product behind
them, and products over one activation share its conversion
(spiral_amd/csrc/backend.hip). Covered: one row (GEMV), a few (small batch) and
many (GEMM); both GLU forms; batched rows; an activation that a product
overwrites; products that read something else than the node before them; a
product between them whose workspace takes the place of their copy.
"""

import numpy as np
import pytest
import torch

from spiral_amd import ggml, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def quant(buf, qtype, n, k, seed):
    t = buf.alloc(ggml.new_tensor(qtype, (k, n)))
    buf.set(t, synth.make_weights(qtype, n, k, seed).tobytes())
    return t


def place(nodes):
    mem = []
    for node in nodes:
        mem.append(torch.full((int(np.prod(node.ne[:4])),), 7.0, dtype=torch.float32, device="cuda"))
        node.data = mem[-1].data_ptr()
    torch.cuda.synchronize()
    return mem


def whole_and_single(nodes, mem):
    """Results of one graph, and of a call per node from the same start."""
    backend, got = ggml.Backend(0), []
    for groups in ([nodes], [[n] for n in nodes]):
        for m in mem:
            m.fill_(7.0)
        torch.cuda.synchronize()
        for g in groups:
            assert backend.graph_compute(g) == 0
        backend.synchronize()
        got.append([m.clone() for m in mem])
    return got


def ids_tensor(ids):
    dev = torch.tensor(ids, dtype=torch.int32, device="cuda")
    t = ggml.new_tensor(ggml.TYPE_I32, [len(ids)])
    t.data = dev.data_ptr()
    return t, dev


@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("tokens", [1, 5, 40])
@pytest.mark.parametrize("qtype", [O.Q4_K, O.Q4_0, O.Q6_K])
def test_block(cuda, qtype, tokens, split):
    h, f, vocab = 512, 768, 100
    buf = ggml.Buffer(8 << 20)
    embed, down = quant(buf, qtype, vocab, h, 1), quant(buf, qtype, h, f, 2)
    ids, keep = ids_tensor([(17 * i) % vocab for i in range(tokens)])
    x = ggml.get_rows(embed, ids)
    if split:
        gate, up = ggml.mul_mat(quant(buf, qtype, f, h, 3), x), ggml.mul_mat(quant(buf, qtype, f, h, 4), x)
        act = ggml.glu_split(gate, up)
        nodes = [x, gate, up, act, ggml.mul_mat(down, act)]
    else:
        both = ggml.mul_mat(quant(buf, qtype, 2 * f, h, 3), x)
        act = ggml.glu(both, ggml.GLU_SWIGLU_OAI)
        nodes = [x, both, act, ggml.mul_mat(down, act)]
    whole, single = whole_and_single(nodes, place(nodes))
    assert all(torch.equal(a, b) and not (a == 7.0).any() for a, b in zip(whole, single))


def test_other_activations_between(cuda):
    """Products in an order that drops and renews the copy: x, x, then the
    block's own input y, x again; a GLU whose rows no product reads."""
    qtype, h, n = O.Q4_0, 256, 320
    buf = ggml.Buffer(4 << 20)
    embed = quant(buf, qtype, 64, h, 1)
    w = [quant(buf, qtype, n, h, 2 + i) for i in range(4)]
    (ia, ka), (ib, kb) = ids_tensor([3, 9]), ids_tensor([60, 1])
    x, y = ggml.get_rows(embed, ia), ggml.get_rows(embed, ib)
    p = [ggml.mul_mat(w[0], x), ggml.mul_mat(w[1], x), ggml.mul_mat(w[2], y), ggml.mul_mat(w[3], x)]
    act = ggml.glu_split(p[0], p[2])
    nodes = [y, x, p[0], p[1], p[2], act, p[3]]
    whole, single = whole_and_single(nodes, place(nodes))
    assert all(torch.equal(a, b) for a, b in zip(whole, single))


def test_product_over_its_input(cuda):
    """A product written over the rows it read: the next product over those
    rows sees the new values."""
    qtype, h = O.Q8_0, 256
    buf = ggml.Buffer(4 << 20)
    embed, w0, w1 = quant(buf, qtype, 64, h, 1), quant(buf, qtype, h, h, 2), quant(buf, qtype, h, h, 3)
    ids, keep = ids_tensor([5])
    x = ggml.get_rows(embed, ids)
    a, b = ggml.mul_mat(w0, x), ggml.mul_mat(w1, x)
    nodes = [x, a, b]
    mem = place(nodes)
    a.data = x.data
    whole, single = whole_and_single(nodes, mem)
    assert torch.equal(whole[0], single[0]) and torch.equal(whole[2], single[2])
    assert not (whole[2] == 7.0).any()


def test_batched_rows(cuda):
    """Row ids in two dimensions, and a product batched over them."""
    qtype, h, n = O.Q4_K, 256, 96
    buf = ggml.Buffer(4 << 20)
    t = buf.alloc(ggml.new_tensor(qtype, (h, 50, 2)))
    buf.set(t, synth.make_weights(qtype, 100, h, 1).tobytes())
    w = quant(buf, qtype, n, h, 2)
    dev = torch.tensor([[1, 7, 49], [0, 3, 20]], dtype=torch.int32, device="cuda")
    ids = ggml.new_tensor(ggml.TYPE_I32, [3, 2])
    ids.data = dev.data_ptr()
    x = ggml.get_rows(t, ids)
    nodes = [x, ggml.mul_mat(w, x)]
    whole, single = whole_and_single(nodes, place(nodes))
    assert all(torch.equal(a, b) and not (a == 7.0).any() for a, b in zip(whole, single))


# A bf16 activation is read in place, so its product's workspace starts where the
# copy lies: the packed rows, the sums of two k ranges, the dequantized matrix;
# and a product of few rows, which takes no workspace.
@pytest.mark.parametrize("qtype,m,n,k", [(O.Q6_K, 40, 96, 512), (O.Q4_0, 17, 300, 4096 + 96),
                                         (O.Q4_0, 257, 7001, 64), (O.Q4_K, 5, 96, 512)])
@pytest.mark.parametrize("made", [False, True])
def test_bf16_product_between(cuda, qtype, m, n, k, made):
    """x, a bf16 activation's product, x again, with x given (converted by its
    first product) and made by get_rows (which leaves the copy)."""
    h, w_rows = 256, 64
    buf = ggml.Buffer(8 << 20)
    w0, w2 = quant(buf, O.Q4_K, w_rows, h, 1), quant(buf, O.Q4_K, w_rows, h, 2)
    w1 = quant(buf, qtype, n, k, 3)
    z_mem = torch.randn((m, k), device="cuda").to(torch.bfloat16)
    z = ggml.new_tensor(ggml.TYPE_BF16, (k, m))
    z.data = z_mem.data_ptr()
    if made:
        ids, keep = ids_tensor([(7 * i) % w_rows for i in range(40)])
        x = ggml.get_rows(w0, ids)
    else:
        x_mem = torch.randn((40, h), device="cuda")
        x = ggml.new_tensor(ggml.TYPE_F32, (h, 40))
        x.data = x_mem.data_ptr()
    nodes = [ggml.mul_mat(w0, x), ggml.mul_mat(w1, z), ggml.mul_mat(w2, x)]
    if made:
        nodes.insert(0, x)
    whole, single = whole_and_single(nodes, place(nodes))
    assert all(torch.equal(a, b) and not (a == 7.0).any() for a, b in zip(whole, single))
