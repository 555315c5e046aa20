"""GPU: the cross-entropy backward's float4 stream at every mix of offsets of its two arrays, at lengths
that are no multiple of 4, and at rows of fewer than 4 logits: the float32 expression of the CPU loop
(train_bnn.c:358-378) evaluated by torch, bit for bit, and nothing written outside the array."""
import pytest
import torch

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
