"""GPU: the LayerNorm kernels that a row's width and the number of rows choose between, at the edges
of each: one wavefront per row (4 to 2,048 channels), a workgroup per row (to 8,192), the lane loops
(beyond, and below 4); widths that are no multiple of 4, whose last slot of four columns overlaps the
one before it; rows at any alignment; the few-row backward, which adds its column sums without partial
rows, on both sides of its rule (512 rows of 2^20 elements, 1,024 rows of 384 channels).

Against the CPU oracle with the bars of test_parity_gpu.py's ln_case; the fused pairs against the ops
in sequence, bit for bit; and nothing written outside the arrays."""
import numpy as np
import pytest
import torch

import gen
from test_fused_gpu import put
from test_parity_gpu import assert_bits, host, ln_case

pytestmark = pytest.mark.gpu

SHAPES = [  # rows, C, offset
    (9, 3, 0), (7, 5, 1), (70, 7, 0), (33, 255, 2), (530, 257, 0), (600, 771, 3), (40, 1301, 0), (530, 2047, 1),
    (520, 2048, 2), (5, 2049, 0), (64, 2052, 1), (40, 3001, 0), (515, 4096, 0), (30, 4097, 3), (129, 6144, 0),
    (60, 8191, 0), (128, 8192, 1), (4, 8193, 0),
    (512, 768, 1), (513, 768, 2), (1024, 384, 0), (1025, 384, 0), (1024, 385, 0), (512, 2048, 0), (257, 4096, 0),
]


@pytest.mark.parametrize("rows,C,offset", SHAPES)
def test_against_the_oracle(gpu, oracle, rows, C, offset):
    ln_case(gpu, oracle, 1, rows, C, seed=rows * 31 + C, offset=offset, reps=2)


@pytest.mark.parametrize("rows,C,offset", SHAPES)
def test_pairs_equal_the_ops_in_sequence(gpu, rows, C, offset):
    g = gen.rng(rows * 17 + C)
    n = rows * C
    x, y, dout, w, b = (gen.normal(g, (k,)) for k in (n, n, n, C, C))
    init = [gen.normal(g, (k,)) for k in (n, C, C, n, n)]
    tx, ty, tdo, tw, tb = (put(a, offset) for a in (x, y, dout, w, b))
    got = []
    for fused in (True, False):
        res, out, m, r = (put(np.zeros(k, np.float32), offset) for k in (n, n, rows, rows))
        di, dw, db, dx, dy = (put(a, offset) for a in init)
        if fused:
            gpu.residual_layernorm_forward(res, out, m, r, tx, ty, tw, tb, 1, rows, C)
            gpu.layernorm_residual_backward(di, dw, db, dx, dy, tdo, res, tw, m, r, 1, rows, C)
        else:
            gpu.residual_forward(res, tx, ty, n)
            gpu.layernorm_forward(out, m, r, res, tw, tb, 1, rows, C)
            gpu.layernorm_backward(di, dw, db, tdo, res, tw, m, r, 1, rows, C)
            gpu.residual_backward(dx, dy, di, n)
        got.append([host(t) for t in (res, out, m, r, di, dw, db, dx, dy)])
    for name, a, c in zip(("res", "out", "mean", "rstd", "dinp", "dweight", "dbias", "dx", "dy"), *got):
        assert_bits(a, c, name)


@pytest.mark.parametrize("rows,C,offset", [s for s in SHAPES if s[0] <= 130])
def test_writes_nothing_outside(gpu, rows, C, offset):
    n, guard = rows * C, 7.25

    def arr(k):
        return torch.full((k + 64,), guard, device="cuda")

    x, dout, w = (torch.randn(k, device="cuda") for k in (n, n, C))
    bufs = {k: arr(s) for k, s in (("out", n), ("mean", rows), ("rstd", rows), ("dinp", n), ("dw", C), ("db", C),
                                   ("dx", n), ("dy", n))}
    v = {k: t[16 + offset:16 + offset + t.numel() - 64] for k, t in bufs.items()}
    for t in v.values():
        t.zero_()
    gpu.layernorm_forward(v["out"], v["mean"], v["rstd"], x, w, w, 1, rows, C)
    gpu.layernorm_residual_backward(v["dinp"], v["dw"], v["db"], v["dx"], v["dy"], dout, x, w, v["mean"], v["rstd"], 1,
                                    rows, C)
    torch.cuda.synchronize()
    for k, t in bufs.items():
        lo, hi = 16 + offset, 16 + offset + t.numel() - 64
        assert bool((t[:lo] == guard).all()) and bool((t[hi:] == guard).all()), k
