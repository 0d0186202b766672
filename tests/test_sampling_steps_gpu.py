"""Sampling from wide vocabularies: the pairs that a chunk of a row gives to the row's list, the
list's selection at its limits, and stream numbers that go with the launch."""
from array import array

import numpy as np
import pytest
import torch

import plain_qwen3 as plain

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rows_of(V, k):
    """Rows where a chunk's choice can go wrong."""
    g = torch.Generator().manual_seed(V + k)
    inf = float("-inf")
    x = torch.randn(9, V, generator=g) * 2.5
    x[1] = torch.linspace(-4, 9, V)                          # all of the top k in the last chunk
    x[2] = torch.where(torch.arange(V) % 512 == 3, x[2] + 20.0, x[2])   # one thread of a chunk holds them
    x[3, 5:] = inf                                           # fewer finite logits than k
    x[4] = inf                                               # none
    x[5] = 20.0 + torch.round(x[5]) / 8                      # hundreds of ties of every value
    x[6, ::7] = float("nan")
    x[7] = 1.0                                               # all equal
    x[8, :] = inf
    x[8, V - k:] = torch.arange(k, dtype=torch.float32) / k  # exactly k, at the row's end
    return x


@pytest.mark.parametrize("V", [16385, 20480, 32000, 151936])
@pytest.mark.parametrize("k", [2, 20, 69, 70, 71, 128, 129, 257])
def test_many_blocks_a_row_choose_as_the_plain_sampler(V, k):
    from edge_infer_amd.csrc import lib
    logits = rows_of(V, k)
    dev, n = logits.to(DEV), logits.shape[0]
    streams, counters = array("i", range(n)), array("i", [3 * r for r in range(n)])
    on_gpu = [torch.tensor(list(a), dtype=torch.int32, device=DEV) for a in (streams, counters)]
    scratch = torch.zeros(lib.sample_scratch_size(n, V), dtype=torch.int32, device=DEV)
    for top_p in (1.0, 0.8):
        prob = torch.empty(n, device=DEV)
        given = torch.empty(n, dtype=torch.int32, pin_memory=True)
        lib.sample(dev, 0.7, top_p, k, 5, streams, counters, given, prob, scratch)
        torch.cuda.synchronize()
        arrays, one_block = (torch.empty(n, dtype=torch.int32, device=DEV) for _ in range(2))
        one_prob = torch.empty(n, device=DEV)
        lib.sample(dev, 0.7, top_p, k, 5, *on_gpu, arrays, None, scratch)
        lib.sample(dev, 0.7, top_p, k, 5, *on_gpu, one_block, one_prob)
        expected = [plain.sample(logits[r].numpy(), 0.7, top_p, k, plain.uniform(5, r, 3 * r))
                    for r in range(n)]
        assert given.tolist() == expected and arrays.tolist() == expected
        assert one_block.tolist() == expected and torch.equal(prob, one_prob)


def test_sampler_takes_any_whole_numbers_and_many_rows():
    from edge_infer_amd.sampling import Sampler, SamplingParams
    logits = torch.randn(65, 32000, generator=torch.Generator().manual_seed(1))
    dev, sampler = logits.to(DEV), Sampler(DEV)
    params = SamplingParams(temperature=0.9, top_p=0.9, top_k=30, seed=9)
    streams, counters = list(range(65)), [7] * 65
    expected = [plain.sample(row.numpy(), 0.9, 0.9, 30, plain.uniform(9, r, 7))
                for r, row in enumerate(logits)]
    assert sampler(dev, params, streams, counters) == expected
    assert sampler(dev[:64], params, np.arange(64), tuple(counters[:64])) == expected[:64]
    assert sampler.sample_device(dev[:3], params, streams[:3], counters[:3]).tolist() == expected[:3]
    for wrong in ([0, 2 ** 31], ["a", 1]):
        with pytest.raises((RuntimeError, TypeError, ValueError, OverflowError)):
            sampler(dev[:2], params, wrong, [0, 0])
