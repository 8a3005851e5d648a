"""The feature kernel's forms by batch and by camera (csrc/features.hip): the
limits on workgroups in flight change at 4,096 and 6,144 environments, and a
call without cameras has instantiations of its own, one for each width of
LiDAR load, plain and with diagnostics.  A row's features are the same bits in
every form; without cameras the last sixteen are zero."""
from __future__ import annotations

import numpy as np
import pytest

from turbinator_c_amd import synth

pytestmark = pytest.mark.gpu


def _bits(t):
    return t.cpu().numpy().view(np.uint32)


@pytest.mark.parametrize("layout", ["batch", "records"])
def test_rows_do_not_depend_on_the_batch(torch_cuda, hip, layout):
    torch, n = torch_cuda, 6145
    b = synth.make_batch(512, seed=21, variant=synth.SPECIAL, threads=16)
    tile = np.arange(n) % 512
    obs, mission, cameras = (torch.from_numpy(x[tile]).cuda() for x in (b.obs, b.mission, b.cameras))
    strides = (16592, 40, 16384)
    if layout == "records":
        rec = torch.zeros((n, 33040), dtype=torch.uint8, device="cuda")
        for view, at in ((obs, 0), (mission, 16592), (cameras, 16640)):
            flat = view.contiguous().view(torch.uint8).reshape(n, -1)
            rec[:, at:at + flat.shape[1]] = flat
        obs, mission, cameras = rec, rec[:, 16592:], rec[:, 16640:]
        strides = (33040,) * 3
    s = torch.cuda.current_stream()
    want = None
    for k in (n, 6144, 6143, 4096, 4095, 1):
        for cams in (cameras, None):
            print(f"[gpu-case] {layout} {k} cameras {cams is not None}", flush=True)
            out = torch.full((n, 142), 7.0, device="cuda")
            assert hip.extract_features_strided_device(
                obs, strides[0], mission, strides[1], cams, strides[2], out, k, s) == 1
            got = _bits(out)
            if want is None:
                want = got
            assert np.array_equal(got[:k, :126], want[:k, :126])
            assert np.array_equal(got[:k, 126:], want[:k, 126:] if cams is not None
                                  else np.zeros((k, 16), np.uint32))
            assert (out[k:] == 7.0).all()


@pytest.mark.parametrize("pad", [0, 2, 1])  # 16-, 8- and 4-byte LiDAR loads
def test_without_cameras_in_every_form(torch_cuda, hip, pad):
    torch, n = torch_cuda, 300
    b = synth.make_batch(n, seed=22, variant=synth.SPECIAL, threads=16)
    rows = torch.zeros((n, 4148 + 4), device="cuda")
    obs = rows.view(-1)[pad:pad + n * (4148 + pad)].view(n, 4148 + pad)
    obs[:, :4148] = torch.from_numpy(b.obs).cuda()
    mission, cameras = (torch.from_numpy(x).cuda() for x in (b.mission, b.cameras))
    stride = (4148 + pad) * 4
    s = torch.cuda.current_stream()
    index = torch.arange(n, device="cuda", dtype=torch.int32).flip(0).contiguous()
    index[7] = n  # reads nothing, NaN row

    def strided(cams):
        out = torch.full((n, 142), 7.0, device="cuda")
        assert hip.extract_features_strided_device(obs, stride, mission, 40, cams, 16384, out, n, s) == 1
        return out

    def indexed(cams):
        out = torch.full((n, 142), 7.0, device="cuda")
        assert hip.extract_features_indexed_device(obs, stride, mission, 40, cams, 16384, n, index,
                                                   out, n, s) == 1
        return out

    print(f"[gpu-case] without cameras, obs stride {stride}", flush=True)
    full = _bits(strided(cameras))
    blind = _bits(strided(None))
    assert np.array_equal(blind[:, :126], full[:, :126]) and not blind[:, 126:].any()
    picked = indexed(None)
    assert torch.isnan(picked[7]).all()
    keep = np.arange(n) != 7
    assert np.array_equal(_bits(picked)[keep], blind[::-1][keep])
    if pad == 0:
        out = torch.full((n, 142), 7.0, device="cuda")
        diag = torch.zeros((2, n, 432), dtype=torch.uint8, device="cuda")
        assert hip.extract_features_diagnostics_device(obs, mission, cameras, out, diag[0], n, s) == 1
        assert hip.extract_features_diagnostics_device(obs, mission, None, out, diag[1], n, s) == 1
        assert np.array_equal(_bits(out), blind)
        seen, unseen = diag.cpu().numpy()
        # 64 sector minima and 64 position / count words, then the cameras' bytes
        assert np.array_equal(seen[:, :384], unseen[:, :384]) and not unseen[:, 384:].any()
