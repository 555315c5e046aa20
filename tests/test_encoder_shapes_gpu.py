"""GPU: the encoder backward at the edges of its kernels, with the bit-exact checks of test_parity_gpu.py's
enc_case: batches on both sides of 16 sequences (how many dwpe rows a thread has in flight), buckets on
both sides of 1,024 rows (32- or 64-channel slices) and of 256 blocks of 64 rows (one or more rounds of
block sums), more than 8,192 rows (rounds of the slot scan), up to 1,024 rows (one launch), small buckets of every size up to 33 rows, and
widths around the slices and the three float4 a lane adds at a time."""
import numpy as np
import pytest
import torch

import gen
from test_parity_gpu import blocked_encoder_backward, dev, enc_case, host

pytestmark = pytest.mark.gpu


def counts_to_tokens(counts, seed):
    t = np.repeat(np.arange(len(counts), dtype=np.int32), counts)
    np.random.default_rng(seed).shuffle(t)
    return t


@pytest.mark.parametrize("B,T,C,V", [(16, 65, 96, 27), (17, 64, 100, 27), (32, 33, 33, 5), (65, 16, 64, 27), (128, 64, 384, 27),
                                     (33, 40, 13, 3)])
def test_batches(gpu, oracle, B, T, C, V):
    enc_case(gpu, oracle, B, T, C, V, gen.tokens_zipf(gen.rng(B), B * T, V), B + T, reps=2)


@pytest.mark.parametrize("C", [4, 31, 32, 33, 64, 100, 768, 772, 1600])
def test_bucket_sizes(gpu, oracle, C):
    counts = list(range(34)) + [63, 64, 65, 128, 129, 1024, 1025, 2500]
    inp = counts_to_tokens(counts, C)
    enc_case(gpu, oracle, 1, inp.size, C, len(counts), inp, C)


@pytest.mark.parametrize("B,T", [(1, 1), (1, 63), (1, 65), (4, 128), (1, 513), (8, 128), (25, 41)])
@pytest.mark.parametrize("C,V", [(5, 1), (64, 2), (384, 27), (768, 5000)])
def test_few_rows(gpu, oracle, B, T, C, V):
    """Up to 512 and 1,024 rows in one launch, and one row more: tokens with up to all of the rows."""
    enc_case(gpu, oracle, B, T, C, V, gen.tokens_zipf(gen.rng(B + T), B * T, V), B * T + C, reps=2)


@pytest.mark.parametrize("rows,C", [(1024, 768), (1024, 772), (1000, 1100), (1024, 1600), (1024, 1601), (601, 2650),
                                    (512, 3201)])
@pytest.mark.parametrize("V", [27, 5000])
def test_few_rows_of_many_channels(gpu, oracle, rows, C, V):
    """One, two and three slices of 64 channels per wavefront, the last group of them not full, and
    one row slice more than the one launch takes."""
    enc_case(gpu, oracle, 1, rows, C, V, gen.tokens_zipf(gen.rng(C), rows, V), rows + C, modes=("blocked",))


@pytest.mark.parametrize("rows", [8191, 8192, 8193, 20500])
def test_one_frequent_token(gpu, oracle, rows):
    inp = np.zeros(rows, np.int32)
    inp[::1000] = 1 + np.arange(inp[::1000].size)
    enc_case(gpu, oracle, 1, rows, 36, 30, inp, rows, modes=("blocked",))


def test_offsets_beyond_32_bits(gpu):
    """More than 2^30 gradient elements in a chunk: the channels at both ends and in the middle."""
    T, C, V = 65536, 16448, 3
    g = torch.Generator("cuda").manual_seed(1)
    dout = torch.randn(T * C, device="cuda", generator=g)
    inp = gen.tokens_zipf(gen.rng(5), T, V)
    dwte, dwpe = torch.zeros(V * C, device="cuda"), torch.zeros(T * C, device="cuda")
    gpu.encoder_backward(dwte, dwpe, dout, dev(inp), 1, T, C)
    cols = torch.tensor([0, 31, 32, 8000, C - 2, C - 1], device="cuda")
    d = host(dout.view(T, C)[:, cols].contiguous())
    want, pe = np.zeros((V, 6), np.float32), np.zeros((T, 6), np.float32)
    blocked_encoder_backward(want, pe, d, inp, 1, T, 6)
    assert np.array_equal(host(dwte.view(V, C)[:, cols].contiguous()), want)
    assert torch.equal(dwpe.view(torch.int32), dout.view(torch.int32))
