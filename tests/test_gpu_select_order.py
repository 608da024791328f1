"""The K allocation and the token order of a layer in one launch (rdkv_select_layer_start) against the calls one by one: the
same widths, order, ranks, class sizes, host words and int16 copies, at lengths around the 1024 tokens of a workgroup, the
sixteen bytes of a load and the split of the rows, with widths that no class has."""
import ctypes

import pytest
import torch

from rdkv_amd import _lib, knapsack_solver as ks, obkv_fast
from tests.gpu_util import DEV, require_gpu

pytestmark = pytest.mark.gpu

EPS = {0: 1.0, 1: 0.7, 2: 0.3, 3: 0.1, 4: 0.0138, 6: 0.002, 8: 0.000048, 16: 0.0, 255: 0.0}


def _floats(v):
    return (ctypes.c_float * len(v))(*v)


@pytest.mark.parametrize("H,T,D", [(1, 1, 4), (3, 15, 128), (8, 16, 128), (2, 17, 64), (16, 1023, 128), (8, 1024, 128), (8, 1025, 256),
                                   (4, 2047, 129), (8, 4099, 128), (5, 31337, 128), (2, 65535, 128), (1, 65536, 8)])
@pytest.mark.parametrize("v_options,k_options", [((0, 2, 4, 8, 16), (0, 2, 4, 8)), ((0, 4), (2, 4, 8, 16)), ((0, 3, 8, 255), (0, 1, 2, 3, 4, 6, 8, 16)),
                                                 ((6, 2, 16), (0, 6))])
def test_one_call_against_the_calls_one_by_one(H, T, D, v_options, k_options):
    require_gpu()
    lib, dev = _lib.load(), torch.device(DEV)
    g = torch.Generator(device=DEV).manual_seed(H + T)
    scores = (torch.randn(H, T + 3, generator=g, device=DEV) * 1.5 + 2).exp()[:, 1:T + 1]
    channels = torch.randn(H, D + 1, generator=g, device=DEV).exp()[:, :D]
    v_budget, k_kept, zero = 2.0, 0.5 * 2 * max(T // 4, 1) * D * 16, v_options.index(0) if 0 in v_options else -1
    stream = _lib.stream_of(dev)
    for pool in ((7, 1, 1), (5, 0, 0), (1, 1, 1)):
        rows = obkv_fast.apply_score_pooling(scores, "avg" if pool[1] else "max", pool[0], "reflect" if pool[2] else "zero") if pool[0] > 1 else scores
        opt = lambda o: torch.tensor([float(x) for x in o])
        v_exp, counts_exp = ks.knapsack_allocate(rows, v_budget, EPS, bit_options=opt(v_options), with_counts=True)
        k_exp = ks.knapsack_allocate(channels, ks.KeptBudget(counts_exp, zero, T, D, k_kept), EPS, bit_options=opt(k_options))
        order_e, rank_e = (torch.empty(H, T, dtype=torch.int32, device=DEV) for _ in range(2))
        plan_e = torch.empty(lib.rdkv_pack_layer_plan_ints(H, T), dtype=torch.int32, device=DEV)
        mm_e = torch.empty(H * 2 * D, device=DEV)
        words = _lib.host_words(dev, 12 * H)
        _lib.check(lib.rdkv_pack_layer_plan_start(v_exp.data_ptr(), 1, T, k_exp.data_ptr(), 1, D, H, T, D, order_e.data_ptr(), T, rank_e.data_ptr(),
                                                  T, plan_e.data_ptr(), mm_e.data_ptr(), 2 * D, words.take(12 * H), words.tag, stream))
        numbers = words.read(dev)
        T16 = -(-T // 16) * 16
        for fill in (0, 255):                                    # (whatever lies behind a row's end)
            v = torch.full((H, T16), fill, dtype=torch.uint8, device=DEV)
            pooled, counts = torch.empty(H, T, device=DEV), torch.empty(H, len(v_options), dtype=torch.int32, device=DEV)
            k = torch.empty(H, D, dtype=torch.uint8, device=DEV)
            order, rank, plan, mm = torch.full_like(order_e, -1), torch.full_like(rank_e, -1), torch.empty_like(plan_e), torch.empty_like(mm_e)
            v16, k16 = torch.empty(H, T, dtype=torch.int16, device=DEV), torch.empty(H, D, dtype=torch.int16, device=DEV)
            ws = _lib.workspace(dev, lib.rdkv_knapsack_workspace_bytes(H))
            ws.fill_(165)                                        # (what another call left there)
            words = _lib.host_words(dev, 12 * H)
            _lib.check(lib.rdkv_select_layer_start(
                scores.data_ptr(), scores.stride(0), H, T, *pool, pooled.data_ptr(), v_budget, _floats(v_options), _floats([EPS[o] for o in v_options]),
                len(v_options), zero, v.data_ptr(), T16, counts.data_ptr(), channels.data_ptr(), channels.stride(0), D, k_kept, _floats(k_options),
                _floats([EPS[o] for o in k_options]), len(k_options), k.data_ptr(), 64, 0.01, order.data_ptr(), rank.data_ptr(), plan.data_ptr(),
                mm.data_ptr(), 2 * D, v16.data_ptr(), k16.data_ptr(), words.take(12 * H), words.tag, ws.data_ptr(), ws.numel(), stream))
            assert words.read(dev) == numbers
            for got, exp in ((v[:, :T], v_exp), (k, k_exp), (counts, counts_exp), (order, order_e), (rank, rank_e), (plan[:12 * H], plan_e[:12 * H]),
                             (mm.view(torch.int32), mm_e.view(torch.int32)), (v16, v_exp.to(torch.int16)), (k16, k_exp.to(torch.int16))):
                assert torch.equal(got, exp)


def test_refusals():
    require_gpu()
    lib = _lib.load()
    x = torch.zeros(64, device=DEV)
    one = _floats([0.0])

    def call(H=1, T=8, D=4, stride=16, v=x, bits=one, n=1):
        return lib.rdkv_select_layer_start(x.data_ptr(), 8, H, T, 1, 1, 1, None, 1.0, bits, one, n, 0, v.data_ptr(), stride, x.data_ptr(), x.data_ptr(), 4, D,
                                           1.0, one, one, 1, x.data_ptr(), 64, 0.01, x.data_ptr(), x.data_ptr(), x.data_ptr(), None, 0, None, None,
                                           x.data_ptr(), 1, x.data_ptr(), 0, None)

    assert call() == _lib.RDKV_EWORKSPACE
    assert call(H=17) == call(T=65537) == call(D=257) == _lib.RDKV_EUNSUPPORTED
    assert call(stride=8) == call(stride=17) == call(v=x[1:]) == _lib.RDKV_EINVAL
