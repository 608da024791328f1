"""The knapsack over rows shared by workgroups of one, two and four sets of threads, bit for bit against the oracle: row
lengths where the split, the scores held per thread or the number of sets change, more than five options (one
candidate a step instead of two), the widest widths (whose sums share an integer), budgets that no multiplier reaches."""
import numpy as np
import pytest
import torch

from oracle import select_oracle as S
from rdkv_amd import knapsack_solver as ks
from tests.gpu_util import require_gpu, t2n, to_dev

pytestmark = pytest.mark.gpu

EPS = {0: 1.0, 1: 0.5, 2: 0.25, 3: 0.08, 4: 0.011, 6: 0.002, 8: 0.000057, 16: 0.0, 200: 1e-7, 255: 0.0}


def _check(s, budget, options, group, max_iters=64):
    opt = torch.tensor([float(o) for o in options])
    got, counts = ks.knapsack_allocate(to_dev(s), to_dev(budget), EPS, max_iters, 0.01, opt, with_counts=True,
                                       group_rows=group)
    exp = np.concatenate([S.knapsack_bit_allocation_batched(s[g:g + group], budget[g:g + group], epsilon=EPS,
                                                            max_iters=max_iters, bit_options=options)
                          for g in range(0, len(s), group)])
    np.testing.assert_array_equal(t2n(got).astype(np.int64), exp)
    np.testing.assert_array_equal(t2n(counts), np.stack([(exp == w).sum(axis=1) for w in options], axis=1))


# four sets / two / one; 2, 4 and 8 scores a thread; a chunk beyond what is held; rows too short to share
@pytest.mark.parametrize("B,T", [(8, 1023), (8, 1024), (1, 1025), (8, 2047), (3, 3000), (64, 2048), (256, 1024), (8, 16385),
                                 (8, 31337), (9, 40000), (2, 65537), (1, 131073), (40, 8193)])
def test_rows_shared_by_sets(B, T):
    require_gpu()
    rng = np.random.default_rng(B + T)
    s = np.exp(rng.standard_normal((B, T)) * 1.5 + 2.0).astype(np.float32)
    _check(s, rng.uniform(0.5, 9.0, B).astype(np.float32), (0, 2, 4, 8, 16), B)


@pytest.mark.parametrize("T", [1024, 6000, 20000])
def test_options_and_budgets(T):
    require_gpu()
    rng = np.random.default_rng(T)
    s = np.exp(rng.standard_normal((4, T)) * 1.5 + 2.0).astype(np.float32)
    budget = rng.uniform(0.5, 9.0, 4).astype(np.float32)
    _check(s, budget, (0, 1, 2, 3, 4, 6, 8, 16), 4)
    _check(s, budget * 10, (0, 200, 255), 2)
    _check(s, budget, (0, 2, 4, 8), 4, max_iters=5)
    _check(s, np.array([1.0, 6.0, 1.0, 3.0], np.float32), (2, 4, 8), 2)      # (none below 2: every doubling)
    _check(np.full((2, T), 3.0, np.float32), np.array([4.0, 300.0], np.float32), (0, 4, 255), 2)


@pytest.mark.parametrize("B,T", [(8, 31744), (8, 16384), (2, 131072), (64, 2048), (8, 4096)])
def test_four_launches_side_by_side(B, T):
    """Calls on streams of their own, whose workgroups wait for each other, find room together: the results of the calls
    alone, none with the width of a wait that was given up."""
    require_gpu()
    g = torch.Generator(device="cuda:0").manual_seed(T)
    scores = [(torch.randn(B, T, generator=g, device="cuda:0") * 1.5 + 2).exp() for _ in range(4)]
    want = [ks.knapsack_allocate(s, 2.0, ks.DEFAULT_EPSILON_V, with_counts=True) for s in scores]
    streams = [torch.cuda.Stream() for _ in scores]
    for stream, s in zip(streams, scores):
        with torch.cuda.stream(stream):
            ks.knapsack_allocate(s, 2.0, ks.DEFAULT_EPSILON_V)            # (the stream's scratch)
    torch.cuda.synchronize()
    got = []
    for _ in range(20):
        for stream, s in zip(streams, scores):
            with torch.cuda.stream(stream):
                got.append(ks.knapsack_allocate(s, 2.0, ks.DEFAULT_EPSILON_V, with_counts=True))
    torch.cuda.synchronize()
    for i, (widths, counts) in enumerate(got):
        assert torch.equal(widths, want[i % 4][0]) and torch.equal(counts, want[i % 4][1])
