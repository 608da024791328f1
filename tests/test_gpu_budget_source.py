"""The knapsack's budget formed inside its launches - one value, or what a V allocation's counts leave the K side -
against the same budgets as a tensor: every form of the solver, heads that keep all, few or no tokens."""
import pytest
import torch

from rdkv_amd import _lib, knapsack_solver as ks, obkv_fast
from tests.gpu_util import DEV, require_gpu

pytestmark = pytest.mark.gpu
SHAPES = [(8, 128), (3, 256), (1, 1), (8, 257), (300, 500), (8, 4096), (8, 9000), (2, 20001)]   # group, two-launch, shared rows


def _scores(B, T):
    g = torch.Generator().manual_seed(B + T)
    return torch.exp(torch.randn(B, T, generator=g) * 1.5).to(DEV)


@pytest.mark.parametrize("B,T", SHAPES)
@pytest.mark.parametrize("value", [0.0, 1.7, 3.3333333, 40.0])
def test_one_value_for_every_row(B, T, value):
    require_gpu()
    s = _scores(B, T)
    exp, n_exp = ks.knapsack_allocate(s, torch.full((B,), value, device=DEV), ks.DEFAULT_EPSILON_V, with_counts=True)
    got, n_got = ks.knapsack_allocate(s, value, ks.DEFAULT_EPSILON_V, with_counts=True)
    assert torch.equal(got, exp) and torch.equal(n_got, n_exp)


@pytest.mark.parametrize("B,T", SHAPES)
@pytest.mark.parametrize("zero_col", [0, 2, -1])
def test_budget_from_counts(B, T, zero_col):
    require_gpu()
    tokens, D, bits = 5000, 128, 5000 * 128 * 1.3
    g = torch.Generator().manual_seed(T)
    counts = torch.randint(0, tokens + 1, (B, 4), generator=g, dtype=torch.int32)
    counts[0] = tokens                                   # nothing kept: a budget for one token
    counts[-1] = 0
    counts = counts.to(DEV)
    tensor = torch.empty(B, device=DEV)
    _lib.check(_lib.load().rdkv_k_budget_per_head(counts.data_ptr(), 4, zero_col, B, tokens, D, bits, tensor.data_ptr(),
                                                  _lib.stream_of(tensor.device)))
    kept = (tokens - counts[:, zero_col] if zero_col >= 0 else torch.full((B,), tokens, device=DEV)).clamp(min=1)
    assert torch.equal(tensor, bits / (D * kept.float()))
    s = _scores(B, T)
    exp = ks.knapsack_allocate(s, tensor, ks.DEFAULT_EPSILON_K, group_rows=B)
    got = ks.knapsack_allocate(s, ks.KeptBudget(counts, zero_col, tokens, D, bits), ks.DEFAULT_EPSILON_K, group_rows=B)
    assert torch.equal(got, exp)


def test_a_heads_allocation_takes_every_kind_of_budget():
    """One value, a tensor, or what ``_k_budget_per_head`` makes of a V allocation's counts."""
    require_gpu()
    s = _scores(8, 128)
    counts = torch.tensor([[h * 100, 0, 0, 0, 900 - h * 100] for h in range(8)], dtype=torch.int32, device=DEV)
    budget = obkv_fast._k_budget_per_head(counts, None, 900, 128, 900 * 128 * 1.5)
    tensor = 900 * 128 * 1.5 / (128 * (900 - counts[:, 0]).float())
    kw = dict(epsilon=ks.DEFAULT_EPSILON_K, bit_options=torch.tensor([0.0, 2.0, 4.0, 8.0]))
    exp = obkv_fast._allocate_k_bits_per_head(s, tensor, **kw)
    got = obkv_fast._allocate_k_bits_per_head(s, budget, **kw)
    assert got.dtype == exp.dtype == torch.int64 and torch.equal(got, exp)
    narrow = obkv_fast._allocate_k_bits_per_head(s, budget, out_dtype=torch.uint8, **kw)
    assert narrow.dtype == torch.uint8 and torch.equal(narrow.long(), exp)
    assert torch.equal(obkv_fast._allocate_k_bits_per_head(s, 1.5, **kw),
                       obkv_fast._allocate_k_bits_per_head(s, torch.full((8,), 1.5, device=DEV), **kw))


def test_counts_that_do_not_fit_are_refused():
    require_gpu()
    s = _scores(4, 128)
    good = torch.zeros(4, 5, dtype=torch.int32, device=DEV)
    for bad in (good[:3], good.long(), good.t().contiguous().t(), good.cpu()):
        with pytest.raises((AssertionError, RuntimeError)):
            ks.knapsack_allocate(s, ks.KeptBudget(bad, 0, 100, 128, 1e4), ks.DEFAULT_EPSILON_K)
    with pytest.raises((AssertionError, RuntimeError)):
        ks.knapsack_allocate(s, ks.KeptBudget(good, 5, 100, 128, 1e4), ks.DEFAULT_EPSILON_K)
