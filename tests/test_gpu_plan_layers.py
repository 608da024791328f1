"""The token and channel plan of several layers against a stable sort: token counts around the wavefront's 256 and the
workgroup's 4096 tokens, every integer type, more layers than a launch takes; and the K min / max over its order."""
import ctypes

import pytest
import torch

from rdkv_amd import _lib
from tests.gpu_util import DEV, require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,L,dtype", [(1, 1, 1, torch.uint8), (64, 2, 3, torch.int64), (255, 3, 1, torch.int16),
                                         (257, 1, 9, torch.int32), (4095, 2, 2, torch.uint8), (4096, 5, 1, torch.int64),
                                         (4097, 2, 8, torch.int64), (12289, 2, 17, torch.int16), (270000, 1, 1, torch.uint8)])
def test_plan_against_a_stable_sort(T, H, L, dtype):
    require_gpu()
    g = torch.Generator(device=DEV).manual_seed(T)
    token, channel = torch.tensor([2, 4, 8, 16, 0, 3], device=DEV), torch.tensor([2, 4, 8, 16, 0], device=DEV)
    cls = torch.randint(0, 6 if T == 257 else 5, (L, H, T), device=DEV, generator=g)
    vb = [token[cls[l]].to(dtype) for l in range(L)]
    kb = [channel[torch.randint(0, 5, (H, 128), device=DEV, generator=g)].to(dtype) for _ in range(L)]
    N = L * H
    K = [torch.randn(H, T, 128, device=DEV, dtype=torch.float16, generator=g) for _ in range(L)]
    lib = _lib.load()
    order = torch.full((N, T), -7, dtype=torch.int32, device=DEV)
    plan = torch.full((lib.rdkv_pack_layer_plan_ints(N, T),), -7, dtype=torch.int32, device=DEV)
    k8 = torch.empty(N, 128, dtype=torch.uint8, device=DEV)
    mm = torch.empty(N, 3, 2, 128, dtype=torch.float32, device=DEV)
    words = _lib.host_words(plan.device, 12 * N)
    at = lambda ts: (ctypes.c_void_p * L)(*[t.data_ptr() for t in ts])
    es, stream = vb[0].element_size(), _lib.stream_of(plan.device)
    _lib.check(lib.rdkv_plan_layers(at(vb), es, at(kb), es, L, H, T, 128, order.data_ptr(), plan.data_ptr(), mm.data_ptr(), 768,
                                    k8.data_ptr(), words.take(12 * N), words.tag, stream))
    strides = (ctypes.c_int64 * (2 * L))(*[s for k in K for s in (k.stride(0), k.stride(1))])
    _lib.check(lib.rdkv_pack_layers_k_minmax(at(K), strides, L, H, T, 128, order.data_ptr(), T, plan.data_ptr(), mm.data_ptr(),
                                             768 * H, stream))
    numbers = torch.tensor(words.read(plan.device)).view(N, 12)
    flat = cls.view(N, T)
    assert torch.equal(order, flat.argsort(dim=1, stable=True).int())
    counts = torch.stack([(flat == k).sum(1) for k in range(6)], 1)
    widths = torch.cat([k.long() for k in kb])
    channels = torch.stack([(widths == 2).sum(1), (widths == 4).sum(1), (widths >= 8).sum(1)], 1)
    assert torch.equal(plan[:4 * N].view(N, 4).long(), counts[:, :4])
    assert torch.equal(numbers[:, :6], counts.cpu()) and torch.equal(numbers[:, 6:9], channels.cpu())
    assert not numbers[:, 9:].any() and torch.equal(k8.long(), widths)
    # the order-preserving integers of the extremes of the kept rows
    bits = mm.view(L, H * 768)[:, :H * 256].reshape(N, 2, 128).view(torch.int32)      # (a layer's heads 256 apart)
    value = torch.where(bits < 0, bits ^ -2147483648, ~bits).view(torch.float32)
    for n in range(N):
        kept = K[n // H][n % H][flat[n] < 4].float()
        if len(kept):
            assert torch.equal(value[n, 0], kept.amin(0)) and torch.equal(value[n, 1], kept.amax(0))

    # one layer by the entry that also ranks the quantized tokens
    one, rank, plan_1 = torch.empty_like(order[:H]), torch.empty_like(order[:H]), torch.empty_like(plan)
    _lib.check(lib.rdkv_pack_layer_plan(vb[0].data_ptr(), es, T, kb[0].data_ptr(), es, 128, H, T, 128, one.data_ptr(), T,
                                        rank.data_ptr(), T, plan_1.data_ptr(), stream))
    quantized = (cls[0] < 3).int()
    assert torch.equal(one, order[:H]) and torch.equal(rank, (quantized.cumsum(1) - quantized).int())
