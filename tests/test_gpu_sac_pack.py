"""The packed actor buffer, byte for byte against its layout restated in numpy:
per layer the row-scaled weights' fp16 pieces in matrix-operand order, biases
and unscale exponents per tile, then the fp32 copy of the first layer; zeros
in every padding row, column and gap (hip_features.h, csrc/sac_actor.hip).
Hidden widths at both ends, at tile and chunk edges and odd; rows of zeros,
of subnormals and with a spread far past fp16's range."""
from __future__ import annotations

import numpy as np
import pytest

from turbinator_c_amd import actor

pytestmark = pytest.mark.gpu


def restated(weights, hidden):
    tiles = -(-hidden // 16)
    chunks = -(-tiles // 2)
    shapes = [(142, hidden, 5, tiles), (hidden, hidden, chunks, tiles), (hidden, 30, chunks, 2)]
    out = bytearray()

    def align():
        out.extend(bytes(-len(out) % 256))

    for layer, (k, n, kc, nt) in enumerate(shapes):
        w, b = weights[2 * layer], weights[2 * layer + 1]
        order = [(p // 2 if p % 2 == 0 else 15 + p // 2) if layer == 2 else p for p in range(n)]
        rows = np.zeros((16 * nt, 32 * max(kc, -(-k // 32))), np.float32)
        rows[:n, :k] = w[order]
        bias = np.zeros(16 * nt, np.float32)
        bias[:n] = b[order]
        scale = np.zeros(16 * nt, np.int32)
        bits = np.abs(rows[:n]).max(axis=1).view(np.uint32)
        scale[:n] = 141 - (bits >> 23).astype(np.int32)
        x = np.ldexp(rows, scale[:, None])
        hi = x.astype(np.float16)
        lo = (x - hi.astype(np.float32)).astype(np.float16)
        lane, s = np.arange(64)[:, None], np.arange(8)[None, :]
        for tile in range(nt):
            for c in range(kc):
                if layer == 0:
                    col = 32 * c + 8 * (lane >> 4) + s
                else:
                    col = 16 * (2 * c + (s >> 2)) + 4 * (lane >> 4) + (s & 3)
                for piece in (hi, lo):
                    out += piece[16 * tile + (lane & 15), col].tobytes()
        align()
        for tile in range(nt):
            t = slice(16 * tile, 16 * tile + 16)
            undo = -scale[t] - (0 if layer == 0 else 14)
            undo[np.arange(16 * tile, 16 * tile + 16) >= n] = 0
            out += bias[t].tobytes() + undo.astype(np.int32).tobytes()
        align()
    out += weights[0].tobytes()
    align()
    return np.frombuffer(bytes(out), np.uint8)


@pytest.mark.parametrize("hidden", [16, 17, 37, 128, 200, 255, 256])
def test_packed_bytes(torch_cuda, hidden):
    torch = torch_cuda
    print(f"[gpu-case] pack hidden {hidden}", flush=True)
    rng = np.random.default_rng(hidden)
    weights = []
    for (n, k), b in actor.layer_shapes(hidden):
        w = rng.standard_normal((n, k)).astype(np.float32)
        w[1] *= np.float32(2.0) ** rng.integers(-60, 20, k).astype(np.float32)
        w[2] = 0.0
        w[3] *= np.float32(1e-41)
        w[4] *= np.float32(1e30)
        weights += [w, rng.standard_normal(b).astype(np.float32)]
    dev = [torch.from_numpy(w).cuda() for w in weights]
    # guard words after the buffer: the kernel writes exactly packed_bytes
    total = actor.packed_bytes(hidden)
    packed = torch.full((total + 256,), 0xa5, dtype=torch.uint8, device="cuda")
    assert actor.pack_device(*dev, hidden, packed, torch.cuda.current_stream()) == 1
    torch.cuda.synchronize()
    got = packed.cpu().numpy()
    assert (got[total:] == 0xa5).all()
    want = restated(weights, hidden)
    assert want.size == total
    bad = np.flatnonzero(got[:total] != want)
    assert not bad.size, (hidden, bad.size, bad[:8], got[bad[:8]], want[bad[:8]])
