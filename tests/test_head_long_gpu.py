"""GPU: softmax over rows beyond 51,393 logits (row statistics by one workgroup per row, of 1,024 threads
below 1,024 rows and of 256 from there on, then a normalising pass): widths around its float4 slots,
special rows and both workgroup sizes, with the bars of test_head_gpu.py; all copies of a row get the same
bits."""
import numpy as np
import pytest
import torch

from test_head_gpu import DEV, bits_equal, check_forward, dev, head_inputs, host, special_rows

pytestmark = pytest.mark.gpu


def softmax(gpu, logits, targets):
    rows, V = logits.shape
    tp, tl = torch.empty(rows * V, device=DEV), torch.empty(rows, device=DEV)
    gpu.softmax_crossentropy(tl, tp, dev(logits), dev(targets), 1, rows, V)
    return host(tp).reshape(rows, V), host(tl)


@pytest.mark.parametrize("V", [51394, 51395, 51396, 51397, 60002, 131071, 200000])
def test_widths(gpu, oracle, V):
    logits, targets = head_inputs(V, 1, 3, V)
    logits = logits.reshape(3, V)
    targets[:] = [0, V - 1, V // 2]
    gp, gl = softmax(gpu, logits, targets)
    cp, cl = np.zeros_like(logits), np.zeros(3, np.float32)
    oracle.softmax_crossentropy(cl, cp, logits, targets, 1, 3, V)
    check_forward(gp, gl, cp, cl, logits, targets)


@pytest.mark.parametrize("V,copies", [(51397, 1), (51397, 160), (60002, 1)])
def test_special_rows(gpu, oracle, V, copies):
    logits = special_rows(V)
    k = logits.shape[0]
    targets = np.full(k, V // 2, np.int32)
    gp, gl = softmax(gpu, np.tile(logits, (copies, 1)), np.tile(targets, copies))
    for c in range(1, copies):
        assert bits_equal(gp[c * k:(c + 1) * k], gp[:k]) and bits_equal(gl[c * k:(c + 1) * k], gl[:k]), c
    gp, gl = gp[:k], gl[:k]
    cp, cl = np.zeros_like(logits), np.zeros(k, np.float32)
    oracle.softmax_crossentropy(cl, cp, logits, targets, 1, k, V)
    assert bits_equal(gp[0], cp[0]) and bits_equal(gp[1], cp[1])  # uniform rows: exact
    assert bits_equal(gp[3], cp[3]) and gl[3] == cl[3] == 0.0  # one finite logit
    assert np.isnan(gp[4]).all() and np.isnan(cp[4]).all()  # all below -1e30
    check_forward(gp, gl, cp, cl, logits, targets)
