"""The work items' scale fields as the device fills them, against the host's routine: scales at every power where the shift
changes, zero, subnormals, infinity and NaN, and what the host receives, bit for bit."""
import numpy as np
import pytest
import torch

from rdkv_amd import _lib, stream_cache
from tests.gpu_util import DEV, require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads", [1, 3, 8])
@pytest.mark.parametrize("n_work", [0, 1, 300])
def test_scale_fields(heads, n_work):
    require_gpu()
    lib, dev = _lib.load(), torch.device(DEV)
    v = [0.0, 1e-40, 1.0, np.inf, np.nan, 65504.0, 3e38] + [x for e in range(7, 42) for x in (2.0 ** e, np.nextafter(np.float32(2.0 ** e), np.float32(0)))]
    v = np.resize(np.asarray(v, dtype=np.float32), -(-len(v) // heads) * heads)
    units, layers = len(v), len(v) // heads
    k = np.arange(units, dtype=np.float32) / 7
    scales = torch.from_numpy(np.stack([k.reshape(layers, heads), v.reshape(layers, heads)], axis=1).copy()).to(DEV)
    work = np.zeros(n_work, dtype=stream_cache.WORK_DTYPE)
    work["unit"] = np.arange(n_work) * 5 % units
    work["tile_begin"] = np.arange(n_work)
    head = np.arange(256, dtype=np.uint8)                # another table ahead of the items
    host = torch.zeros(256 + 128 * n_work, dtype=torch.uint8, pin_memory=True)
    host.numpy()[:256] = head
    host.numpy()[256:] = work.view(np.uint8).reshape(-1)
    on_dev = torch.full((256 + 128 * n_work + 16,), 7, dtype=torch.uint8, device=DEV)
    words = _lib.host_words(dev, 2 * units)
    call = lambda n, h, u: lib.rdkv_stream_tables_device(host.data_ptr(), on_dev.data_ptr(), 256 + 128 * n_work, 256, n,
                                                         scales.data_ptr(), h, u, words.ptr, words.tag, _lib.stream_of(dev))
    words.take(2 * units)
    _lib.check(call(n_work, heads, units))
    got = np.asarray(words.read(dev), dtype=np.int32)
    both = np.stack([k, v], axis=1)
    assert (got == both.reshape(-1).view(np.int32)).all()
    if n_work:
        _lib.check(lib.rdkv_stream_work_scales(work.ctypes.data, n_work, both.ctypes.data, units))
    assert on_dev.cpu().numpy().tobytes() == head.tobytes() + work.tobytes() + bytes([7] * 16)
    assert call(n_work + 1, heads, units) == _lib.RDKV_EINVAL
    assert call(n_work, heads, units + (1 if heads > 1 else -units)) == _lib.RDKV_EINVAL
