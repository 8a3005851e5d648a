"""The host object's two ways (csrc/feature_batch.c): pinned rows, 32
environments at a time, up to 256, and copies above.  At the edges of a piece
and of the staging, on one handle used for larger and smaller calls in turn,
the features are those of the device entry, bit for bit, and nothing past
`count` rows is written."""
from __future__ import annotations

import numpy as np
import pytest

from turbinator_c_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("max_batch", [1, 40, 300])
def test_host_object_equals_device_entry(torch_cuda, hip, max_batch):
    torch = torch_cuda
    b = synth.make_batch(max_batch, seed=9, variant=synth.SPECIAL, threads=16)
    dev = [torch.from_numpy(x).cuda() for x in (b.obs, b.mission, b.cameras)]
    out = torch.empty((max_batch, 142), device="cuda")
    s = torch.cuda.current_stream()
    assert hip.extract_features_device(*dev, out, max_batch, s) == 1
    torch.cuda.synchronize()
    want = out.cpu().numpy().view(np.uint32)
    with hip.FeatureBatch.create(0, max_batch) as handle:
        for count in (300, 257, 256, 255, 65, 64, 33, 32, 31, 1, 40, 256):
            if count > max_batch:
                continue
            print(f"[gpu-case] host object {count} of {max_batch}", flush=True)
            # other rows first in the arrays, so that a stale row would show
            first = (max_batch - count) // 2
            rows = slice(first, first + count)
            got = np.full((count + 1, 142), 7.0, np.float32)
            assert handle.extract_host(np.ascontiguousarray(b.obs[rows]),
                                       np.ascontiguousarray(b.mission[rows]),
                                       np.ascontiguousarray(b.cameras[rows]), count, got) == 1
            assert (got[count] == 7.0).all()
            assert np.array_equal(got[:count].view(np.uint32), want[rows]), count


def test_small_handles_take_no_device_memory(torch_cuda, hip):
    """A handle whose every batch goes through its pinned rows has no device
    buffers: eight of them would take 69 MB."""
    torch = torch_cuda
    b = synth.make_batch(256, seed=10, threads=16)
    got = np.empty((256, 142), np.float32)
    with hip.FeatureBatch.create(0, 256) as handle:  # the runtime's own first allocations
        assert handle.extract_host(b.obs, b.mission, b.cameras, 256, got) == 1
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    handles = [hip.FeatureBatch.create(0, 256) for _ in range(8)]
    try:
        taken = free - torch.cuda.mem_get_info()[0]
        print(f"[gpu-case] eight handles of 256: {taken} bytes of device memory", flush=True)
        assert taken < 16 << 20, taken
    finally:
        for handle in handles:
            handle.destroy()
