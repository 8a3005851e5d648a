"""The compact actor's workgroup shapes (csrc/sac_actor.hip): a row's outputs
do not depend on the batch it is acted on in.  Every batch size around a
shape's bounds (and around a group's and a workgroup's rows) against the rows
of a larger batch in another shape, bit for bit, with infinite and NaN
features and the last rows of a batch among them; hidden widths with 1, 4, 5,
8, 9 and 16 tiles, odd ones included."""
from __future__ import annotations

import numpy as np
import pytest

from turbinator_c_amd import actor

pytestmark = pytest.mark.gpu

SIZES = (1, 15, 16, 17, 33, 63, 4095, 4096, 4097, 8191, 8192, 8193, 16384, 16385)


@pytest.mark.parametrize("hidden", [16, 61, 65, 128, 130, 256])
def test_rows_do_not_depend_on_the_batch(torch_cuda, hidden):
    torch = torch_cuda
    print(f"[gpu-case] actor shapes, hidden {hidden}", flush=True)
    rng = np.random.default_rng(hidden)
    n = 20000
    feats = rng.uniform(-1, 1, (n, 142)).astype(np.float32)
    feats[rng.integers(0, n, 200), rng.integers(0, 142, 200)] = np.inf
    feats[rng.integers(0, n, 100), rng.integers(0, 142, 100)] = np.nan
    for k in SIZES:
        feats[k - 1, 5] = -np.inf
    dev = []
    for (o, i), b in actor.layer_shapes(hidden):
        dev += [torch.from_numpy((rng.standard_normal((o, i)) * 0.1).astype(np.float32)).cuda(),
                torch.from_numpy(rng.standard_normal(b).astype(np.float32)).cuda()]
    s = torch.cuda.current_stream()
    packed = torch.empty(actor.packed_bytes(hidden), dtype=torch.uint8, device="cuda")
    assert actor.pack_device(*dev, hidden, packed, s) == 1
    f = torch.from_numpy(feats).cuda()
    z = torch.from_numpy(rng.standard_normal((n, 15)).astype(np.float32)).cuda()

    def act(k, normals):
        out = [torch.full((k + 1, w), 7.0, device="cuda") for w in (15, 1, 30)]
        assert actor.act_device(packed, hidden, f, normals, *out, k, s) == 1
        torch.cuda.synchronize()
        out = [o.cpu().numpy().view(np.uint32) for o in out]
        for o in out:  # nothing past the batch
            assert (o[k:].reshape(-1) == np.float32(7.0).view(np.uint32)).all(), (hidden, k)
        return [o.reshape(-1)[:k * w].reshape(k, w) for o, w in zip(out, (15, 1, 30))]

    for normals in (z, None):
        want = act(n, normals)
        for k in SIZES:
            for got, full, name in zip(act(k, normals), want, ("actions", "log_prob", "raw")):
                bad = np.flatnonzero((got != full[:k]).any(axis=1))
                assert not bad.size, (hidden, k, name, bad[:5])
