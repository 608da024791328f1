"""The knapsack over short rows (a wavefront per row, a workgroup per group) and over rows of 4096 ..
8191 scores (eight workgroups each), bit for bit against the oracle: row lengths around the lanes and
registers a row is held in, groups up to and past the sixteen of a workgroup, option sets that reach
the unrolled count and pass it, budgets no multiplier reaches, constant rows."""
import numpy as np
import pytest
import torch

from oracle import select_oracle as S
from rdkv_amd import knapsack_solver as ks
from tests.gpu_util import require_gpu, t2n, to_dev

pytestmark = pytest.mark.gpu

EPS = {0: 1.0, 1: 0.5, 2: 0.25, 3: 0.08, 4: 0.011, 6: 0.002, 8: 0.000057, 16: 0.0}


def _check(s, budget, options, group, max_iters=64):
    opt = None if options is None else torch.tensor([float(o) for o in options])
    got, counts = ks.knapsack_allocate(to_dev(s), to_dev(budget), EPS, max_iters, 0.01, opt, with_counts=True,
                                       group_rows=group)
    exp = np.concatenate([S.knapsack_bit_allocation_batched(s[g:g + group], budget[g:g + group], epsilon=EPS,
                                                            max_iters=max_iters, bit_options=options)
                          for g in range(0, len(s), group)])
    np.testing.assert_array_equal(t2n(got).astype(np.int64), exp)
    widths = [0, 2, 4, 8, 16] if options is None else list(options)
    np.testing.assert_array_equal(t2n(counts), np.stack([(exp == w).sum(axis=1) for w in widths], axis=1))


@pytest.mark.parametrize("T", [1, 2, 63, 64, 65, 127, 128, 129, 200, 256, 257])
@pytest.mark.parametrize("group,groups", [(1, 3), (3, 2), (8, 4), (16, 1), (17, 1)])
def test_short_rows(T, group, groups):
    require_gpu()
    rng = np.random.default_rng(100 * T + group)
    s = np.exp(rng.standard_normal((group * groups, T)) * 1.5 + 2.0).astype(np.float32)
    s[0] = 3.0
    budget = rng.uniform(0.5, 9.0, len(s)).astype(np.float32)
    _check(s, budget, None, group)
    _check(s, budget, (0, 2, 4, 8), group)
    _check(s, budget, (0, 1, 2, 3, 4, 6, 8, 16), group)
    _check(s, budget, (0, 2, 4, 8), group, max_iters=3)


def test_short_rows_with_budgets_no_multiplier_reaches():
    """Every row doubles to the end, where the rows of a group end their rounds together."""
    require_gpu()
    rng = np.random.default_rng(4)
    s = (np.exp(rng.standard_normal((16, 96)) * 2.0) * np.logspace(0, 6, 16)[:, None]).astype(np.float32)
    s[5] = 0.0
    budget = np.full(16, 1.0, np.float32)
    budget[::3] = 6.0
    for group in (2, 8, 16):
        _check(s, budget, (2, 4, 8), group)


@pytest.mark.parametrize("B,T", [(1, 4096), (3, 4097), (8, 6001), (64, 8191), (65, 4100), (2, 4095)])
def test_rows_shared_by_eight_workgroups(B, T):
    require_gpu()
    rng = np.random.default_rng(B + T)
    s = np.exp(rng.standard_normal((B, T)) * 1.5 + 2.0).astype(np.float32)
    _check(s, rng.uniform(0.5, 9.0, B).astype(np.float32), None, B)
