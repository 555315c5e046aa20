"""GPU: the LayerNorm kernels that a row's width and the number of rows choose between, at the edges
of each: one wavefront per row (4 to 2,048 channels), a workgroup per row (to 8,192), the lane loops
(beyond, and below 4); widths that are no multiple of 4, whose last slot of four columns overlaps the
one before it; rows at any alignment; the few-row backward, which adds its column sums without partial
rows, on both sides of its rule (512 rows of 2^19 elements, or of 2^20 beyond 1,536 channels; 1,024 rows
of 2^18 elements, or of 3 2^16 off a 16-byte boundary); every number of float4 per lane above it.

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
    (512, 1024, 0), (512, 1028, 0), (512, 1540, 0), (1024, 256, 0), (1025, 256, 0), (1024, 260, 0), (768, 256, 1),
    (769, 256, 1), (600, 1280, 0), (600, 1600, 0), (600, 1792, 0), (200, 6144, 0), (300, 4099, 0), (140, 8191, 0),
    (2100, 771, 0),
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


def in_place_results(gpu, rows, C, offset, pair):
    """dinp (for the pair dx) over dout, and in an array of its own: [dinp or dx, dinp, dy, dweight, dbias] of both."""
    g = gen.rng(rows * 13 + C)
    n = rows * C
    x, dout, w, b, dw0, db0 = (gen.normal(g, (k,)) for k in (n, n, C, C, C, C))
    tx, tw, tb = (put(a, offset) for a in (x, w, b))
    out, m, r = (put(np.zeros(k, np.float32), offset) for k in (n, rows, rows))
    gpu.layernorm_forward(out, m, r, tx, tw, tb, 1, rows, C)
    got = []
    for same in (True, False):
        do = put(dout, offset)
        over = do if same else put(dout, offset)
        di, dy = put(np.zeros(n, np.float32), offset), put(dout, offset)
        dw, db = put(dw0, offset), put(db0, offset)
        if pair:
            gpu.layernorm_residual_backward(di, dw, db, over, dy, do, tx, tw, m, r, 1, rows, C)
        else:
            gpu.layernorm_backward(over, dw, db, do, tx, tw, m, r, 1, rows, C)
        got.append([host(t) for t in (over, di, dy, dw, db)])
    return got, x, dout, w, dw0, db0, host(m), host(r)


@pytest.mark.parametrize("rows,C,offset", [(256, 384, 0), (512, 768, 1), (300, 771, 0), (128, 8192, 0), (513, 768, 0),
                                           (70, 3, 0), (40, 8193, 0)])
@pytest.mark.parametrize("pair", [False, True])
def test_in_place(gpu, rows, C, offset, pair):
    """dinp (for the pair dx) over dout: a row's terms are those of dout as it was. Another kernel may
    take the call then, with its sums in another order, so the results agree to the bound of two orders
    of 32-bit additions (n terms: n 2^-24 of their absolute sum, each)."""
    got, x, dout, w, dw0, db0, m, r = in_place_results(gpu, rows, C, offset, pair)
    u, d64 = 2.0 ** -24, dout.reshape(rows, C).astype(np.float64)
    r64 = r.astype(np.float64)[:, None]
    xhat = np.abs((x.reshape(rows, C) - m.astype(np.float64)[:, None]) * r64)
    dn = np.abs(d64 * w)
    # of a row's two means, and of the rounding of dinp's and dx's own few terms
    means = 2 * C * u * (dn.mean(1, keepdims=True) + xhat * (dn * xhat).mean(1, keepdims=True))
    row = r64 * (means + 16 * u * (dn + dn.mean(1, keepdims=True) + xhat * (dn * xhat).mean(1, keepdims=True)))
    row += 8 * u * np.abs(d64)
    for k, bound in ((0, row), (1, row), (2, row), (3, 2 * rows * u * ((np.abs(d64) * xhat).sum(0) + np.abs(dw0))),
                     (4, 2 * rows * u * (np.abs(d64).sum(0) + np.abs(db0)))):
        diff = np.abs(got[0][k].astype(np.float64) - got[1][k]).reshape(bound.shape)
        assert (diff <= bound).all(), k


@pytest.mark.parametrize("rows,C,offset", [(256, 384, 0), (300, 771, 1), (70, 3, 0)])
@pytest.mark.parametrize("pair", [False, True])
def test_in_place_exact(gpu, rows, C, offset, pair):
    """The exact mode in place: the same bits."""
    prev = gpu.layernorm_exact()
    gpu.set_layernorm_exact(True)
    try:
        got = in_place_results(gpu, rows, C, offset, pair)[0]
    finally:
        gpu.set_layernorm_exact(prev)
    for k, (a, c) in enumerate(zip(*got)):
        assert_bits(a, c, str(k))


def test_column_sums_no_further_from_64_bits(gpu):
    """dweight and dbias of many rows off a 16-byte boundary (959 partial rows) are no further from the
    64-bit sums than the same terms in chains of 32 rows, 16 groups of 30 such chains and the groups,
    each in order, as the lane loops would add them."""
    rows, C, offset = 15345, 768, 2
    g = gen.rng(3)
    n = rows * C
    x, dout, w = (gen.normal(g, (k,)) for k in (n, n, C))
    tx, tw, td, tb = (put(a, offset) for a in (x, w, dout, w))
    out, m, r, di, dw, db = (put(np.zeros(k, np.float32), offset) for k in (n, rows, rows, n, C, C))
    gpu.layernorm_forward(out, m, r, tx, tw, tb, 1, rows, C)
    gpu.layernorm_backward(di, dw, db, td, tx, tw, m, r, 1, rows, C)
    x2, d2, m2, r2 = x.reshape(rows, C), dout.reshape(rows, C), host(m)[:, None], host(r)[:, None]
    terms = {"dweight": ((x2 - m2) * r2 * d2, (x2.astype(np.float64) - m2) * r2 * d2, host(dw)),
             "dbias": (d2, d2.astype(np.float64), host(db))}
    for k, (t, t64, got) in terms.items():
        pad = np.zeros((16 * 30 * 32, C), np.float32)
        pad[:rows] = t
        rung = pad.reshape(16, 30, 32, C)
        for axis in (2, 1, 0):  # np.add.accumulate over a leading axis is a float32 chain in order
            rung = np.add.accumulate(rung, axis=axis, dtype=np.float32).take(-1, axis=axis)
        want = t64.sum(0)
        off = [np.linalg.norm(a - want) / np.linalg.norm(want) for a in (got, rung)]
        print(k, off)
        assert off[0] <= off[1], k
