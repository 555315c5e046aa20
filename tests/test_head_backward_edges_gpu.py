"""GPU: the cross-entropy backward's float4 stream at every mix of offsets of its two arrays, at lengths
that are no multiple of 4, and at rows of fewer than 4 logits: the float32 expression of the CPU loop
(train_bnn.c:358-378) evaluated by torch, bit for bit, and nothing written outside the array."""
import numpy as np
import pytest
import torch

import gen
from test_parity_gpu import assert_bits, dev, host

pytestmark = pytest.mark.gpu
GUARD = 7.25


@pytest.mark.parametrize("rows,V", [(1, 1), (5, 2), (7, 3), (1, 4), (3, 5), (9, 7), (5, 27), (3, 33), (2, 1001), (3, 4099)])
@pytest.mark.parametrize("offsets", [(0, 0), (1, 0), (0, 2), (3, 1), (31, 4)])
@pytest.mark.parametrize("zeroed", [False, True])
def test_offsets_and_ends(gpu, rows, V, offsets, zeroed):
    g = torch.Generator("cuda").manual_seed(rows * 100 + V)
    n = rows * V
    buf = torch.full((n + 96,), GUARD, device="cuda")
    d = buf[32 + offsets[0]:32 + offsets[0] + n]
    d.copy_(torch.randn(n, generator=g, device="cuda"))
    p = torch.rand(n + 8, generator=g, device="cuda")[offsets[1]:offsets[1] + n]
    t = torch.randint(0, V, (rows,), generator=g, device="cuda", dtype=torch.int32)
    hot = torch.nn.functional.one_hot(t.long(), V).float().reshape(-1)
    want = (torch.zeros_like(d) if zeroed else d.clone()) + (p - hot) * torch.tensor(1.0 / rows, device="cuda")
    f = gpu.crossentropy_softmax_backward_zeroed if zeroed else gpu.crossentropy_softmax_backward
    f(d, p, t, 1, rows, V)
    torch.cuda.synchronize()
    assert torch.equal(d.view(torch.int32), want.view(torch.int32))
    assert bool((buf[:32 + offsets[0]] == GUARD).all()) and bool((buf[32 + offsets[0] + n:] == GUARD).all())


@pytest.mark.parametrize("rows,V", [(64, 27), (7, 30), (8, 32), (5, 3)])
@pytest.mark.parametrize("zeroed", [False, True])
def test_targets_outside_the_row(gpu, oracle, rows, V, zeroed):
    """Through the unchecked entry points a target outside [0, V) is no element of any row: not of its
    neighbours in the flat array either (train_bnn.c:358-378 compares it with the row's own indexes)."""
    g = gen.rng(rows + V)
    p = gen.normal(g, (rows * V,))
    t = gen.tokens_uniform(g, rows, V)
    t[:5] = (-1, V, V + 1, -2, 0x7fffffff)
    want = np.zeros(rows * V, np.float32)
    oracle.crossentropy_softmax_backward(want, p, t, 1, rows, V)
    d, tp, tt = dev(np.zeros(rows * V, np.float32)), dev(p), dev(t)
    f = gpu.lib.ugk_crossentropy_softmax_backward_zeroed if zeroed else gpu.lib.ugk_crossentropy_softmax_backward
    assert f(d.data_ptr(), tp.data_ptr(), tt.data_ptr(), 1, rows, V) == 0
    assert_bits(host(d), want, "dlogits")
    assert np.array_equal(host(tt), t)
