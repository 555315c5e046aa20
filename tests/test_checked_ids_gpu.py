"""GPU: the id check inside the ops' own kernels, over every kernel that reads ids: out-of-range ids (below,
at and beyond the bound; the first two rows, the middle and the last) are replaced in place, the others not written, the
outputs are those of the replaced ids, and the next synchronize names the op, once."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def planted(n, V, seed):
    g = torch.Generator(DEV).manual_seed(seed)
    ids = torch.randint(0, V, (n,), device=DEV, dtype=torch.int32, generator=g)
    bad = ids.clone()
    at = sorted({0, 1, n // 2, n - 1})
    for k, i in enumerate(at):
        bad[i] = (V, -1, 0x7fffffff, V + 7)[k]
    return g, bad, at


def reported(gpu, name):
    with pytest.raises(gpu.UgkError, match=name):
        gpu.synchronize()
    gpu.synchronize()


def same(a, b):
    return torch.equal(a.view(torch.int32), b.view(torch.int32))


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("rows,V", [(5, 2), (70, 27), (9, 100), (3, 900), (3, 4000), (3, 16000), (2, 32000), (3, 50257),
                                    (3, 51500), (1025, 51500)])
def test_head(gpu, rows, V, exact):
    g, bad, at = planted(rows, V, rows + V)
    want_ids = bad.clone()
    want_ids[at] = 0
    x = torch.randn(rows * V, device=DEV, generator=g)
    prev = gpu.softmax_exact()
    gpu.set_softmax_exact(exact)
    try:
        out = []
        for ids in (bad.clone(), want_ids.clone()):
            losses, probs = torch.empty(rows, device=DEV), torch.empty(rows * V, device=DEV)
            gpu.softmax_crossentropy(losses, probs, x, ids, 1, rows, V)
            out.append((losses, probs))
            if len(out) == 1:
                reported(gpu, "softmax_crossentropy")
            assert torch.equal(ids, want_ids)
        assert same(out[0][0], out[1][0]) and same(out[0][1], out[1][1])
    finally:
        gpu.set_softmax_exact(prev)
    for f in (gpu.crossentropy_softmax_backward, gpu.crossentropy_softmax_backward_zeroed):
        ids, d = bad.clone(), [torch.zeros(rows * V, device=DEV) for _ in range(2)]
        f(d[0], out[0][1], ids, 1, rows, V)
        reported(gpu, "crossentropy_softmax_backward")
        assert torch.equal(ids, want_ids)
        f(d[1], out[0][1], ids, 1, rows, V)
        gpu.synchronize()
        assert same(*d)


# few rows; the bucket table, with dwpe of few and of many sequences and rows in a second chunk; the fused
# forward with two rows per wavefront, an odd number of them
@pytest.mark.parametrize("B,T,C", [(1, 5, 7), (2, 9, 384), (1, 40, 2052), (20, 3, 64), (5, 257, 384), (20, 60, 30),
                                   (1, 70001, 16), (3, 1367, 384), (1, 2049, 1600)])
def test_encoder(gpu, B, T, C):
    V, n = 11, B * T
    g, bad, at = planted(n, V, n + C)
    r = lambda k: torch.randn(k, device=DEV, generator=g)
    wte, wpe, w, b, dout = r(V * C), r(T * C), r(C), r(C), r(n * C)
    zero = bad.clone()
    zero[at] = 0
    out = [torch.empty(n * C, device=DEV) for _ in range(4)]
    stat = [torch.empty(n, device=DEV) for _ in range(4)]
    for k, ids in enumerate((bad.clone(), zero.clone())):
        gpu.encoder_forward(out[k], ids, wte, wpe, B, T, C)
        if k == 0:
            reported(gpu, "encoder_forward")
        assert torch.equal(ids, zero)
    assert same(out[0], out[1])
    ids = bad.clone()
    gpu.encoder_layernorm_forward(out[1], out[2], stat[0], stat[1], ids, wte, wpe, w, b, B, T, C)
    reported(gpu, "encoder_layernorm_forward")
    assert torch.equal(ids, zero) and same(out[0], out[1])
    gpu.layernorm_forward(out[3], stat[2], stat[3], out[0], w, b, B, T, C)
    assert same(out[2], out[3]) and same(stat[0], stat[2]) and same(stat[1], stat[3])
    skip = bad.clone()
    skip[at] = -1
    ids, dwte, dwpe = bad.clone(), torch.zeros(V * C, device=DEV), torch.zeros(T * C, device=DEV)
    gpu.encoder_backward(dwte, dwpe, dout, ids, B, T, C)
    reported(gpu, "encoder_backward")
    assert torch.equal(ids, skip)
    keep = torch.ones(n, device=DEV)
    keep[at] = 0
    want = torch.zeros(V, C, device=DEV, dtype=torch.float64)
    want.index_add_(0, zero.long(), (dout.view(n, C) * keep[:, None]).double())
    assert (dwte.view(V, C).double() - want).abs().max() <= n * 2.0 ** -23 * want.abs().max().clamp(min=1)


def test_empty_table_is_refused(gpu):
    t = torch.zeros(4, device=DEV)
    ids = torch.zeros(4, device=DEV, dtype=torch.int32)
    assert gpu.lib.ugk_encoder_forward_checked(t.data_ptr(), ids.data_ptr(), t.data_ptr(), t.data_ptr(), 1, 1, 4, 0) == 1
    assert b"V must be > 0" in gpu.lib.ugk_last_error()
