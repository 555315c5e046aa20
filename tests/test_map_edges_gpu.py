"""The elementwise kernels' float4 slots start at a cache line of the first output and the elements
around them go one by one, and few elements at a misaligned address take a thread each: results at
every mix of offsets and at sizes around the edges, and on both sides of each operator's line between
the two, are those of the same call on aligned copies (each element is computed alone, so bit for bit),
and nothing outside the arrays is written."""
import pytest
import torch

pytestmark = pytest.mark.gpu

GUARD = 7.25
SIZES = [1, 2, 3, 4, 5, 31, 32, 33, 35, 36, 127, 2049, 4096 + 31, 3 * 4096 + 2, 1 << 19, (1 << 19) + 1, (5 << 17) + 2,
         (3 << 18) + 3, (1 << 20) + 33]


def ops(ugk):
    """name -> (number of arrays, call)"""
    adam = (3, 3e-4, 0.9, 0.999, 1e-8, 0.0)
    return {
        "residual_forward": (3, lambda a, n: ugk.residual_forward(a[0], a[1], a[2], n)),
        "residual_backward": (3, lambda a, n: ugk.residual_backward(a[0], a[1], a[2], n)),
        "gelu_backward": (3, lambda a, n: ugk.gelu_backward(a[0], a[1], a[2], n)),
        "bayes_materialize": (4, lambda a, n: ugk.bayes_materialize(a[0], a[1], a[2], a[3], n)),
        "bayes_sample": (4, lambda a, n: ugk.bayes_sample(a[0], a[1], a[2], a[3], n, 0x5EED, 3)),
        "adamw_update": (4, lambda a, n: ugk.adamw_update(a[0], a[1], a[2], a[3], n, *adam)),
        "bayes_backward_philox": (4, lambda a, n: ugk.bayes_backward_philox(a[0], a[1], a[2], a[3], n, 0x5EED, 3)),
        "bbb_step_fused": (8, lambda a, n: ugk.bbb_step_fused(*a, n, 0x5EED, 3, 0.1, 1e-6, 0.3, 0.003, *adam[1:])),
    }


@pytest.mark.parametrize("name", ["residual_forward", "residual_backward", "gelu_backward", "bayes_materialize",
                                  "bayes_sample", "adamw_update", "bayes_backward_philox", "bbb_step_fused"])
@pytest.mark.parametrize("offsets", [(0, 0, 0, 0), (1, 1, 1, 1), (0, 2, 1, 3), (3, 0, 2, 1), (29, 4, 31, 2)])
def test_offsets_and_ends(gpu, name, offsets):
    k, call = ops(gpu)[name]
    offsets = (offsets * 2)[:k]
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    for n in SIZES:
        bufs = [torch.full((n + 128,), GUARD, device="cuda") for _ in range(k)]
        views = [b[32 + o:32 + o + n] for b, o in zip(bufs, offsets)]
        for v in views:
            v.copy_(torch.randn(n, generator=g, device="cuda").abs_())
        plain = [v.clone() for v in views]
        call(views, n)
        call(plain, n)
        torch.cuda.synchronize()
        for i, (b, v, p, o) in enumerate(zip(bufs, views, plain, offsets)):
            assert torch.equal(v.view(torch.int32), p.view(torch.int32)), (name, n, offsets, i)
            assert bool((b[:32 + o] == GUARD).all()) and bool((b[32 + o + n:] == GUARD).all()), (name, n, offsets, i)
