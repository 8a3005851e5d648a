"""The onboard and actor-input entries' workgroup shapes (csrc/onboard.hip): a
row's outputs do not depend on the batch it comes in.  Every batch size around
a shape's bounds (the least share of 8, one workgroup per CU and two, one, two
and four groups of 16, whole rounds and their rest, the two-stream form)
against the rows of a batch in another shape, bit for bit, and each shape on
the generator's non-finite and signed-zero rows."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from tests.test_gpu_onboard import compare, in_window, run_onboard
from turbinator_c_amd import synth

pytestmark = pytest.mark.gpu

SIZES = (1, 7, 8, 9, 15, 16, 17, 31, 33, 1000, 2048, 2049, 4095, 4097, 5000, 8191, 8192, 8193,
         9000, 16383, 16384, 16385, 20011, 32767, 32768, 32769, 33025, 40960, 40961, 49153, 65537)


@pytest.fixture(scope="module")
def tiled(torch_cuda):
    """4,096 distinct environments (ordinary and special), tiled on the device."""
    torch = torch_cuda
    parts = [synth.make_batch(2048, seed=71, threads=16),
             synth.make_batch(1024, seed=72, variant=synth.SPECIAL, threads=16),
             synth.make_batch(1024, seed=73, variant=synth.EDGE_QUARTERS, threads=16)]
    obs = in_window(np.concatenate([p.obs for p in parts]))
    mission = np.concatenate([p.mission for p in parts])
    order = np.random.default_rng(7).permutation(4096)
    rows = torch.arange(65600, device="cuda") % 4096
    return (torch.from_numpy(obs[order]).cuda()[rows].contiguous(),
            torch.from_numpy(mission[order]).cuda()[rows].contiguous())


@pytest.mark.parametrize("diag", [False, True])
def test_onboard_rows_do_not_depend_on_the_batch(torch_cuda, hip, tiled, diag):
    torch = torch_cuda
    obs, mission = tiled
    s = torch.cuda.current_stream()

    def run(n):
        out = [torch.full((n + 1, w), 7.0, device="cuda") for w in (24, 15, 5)]
        assert hip.onboard_tactical_prior_device(obs, mission, out[0], out[1],
                                                 out[2] if diag else None, n, s) == 1
        torch.cuda.synchronize()
        return out

    want = run(4096)
    for n in SIZES:
        print(f"[gpu-case] onboard {n} diag {diag}", flush=True)
        for got, full, k in zip(run(n), want, (0, 1, 2)):
            if k == 2 and not diag:
                continue
            assert bool((got[n] == 7.0).all()), n  # nothing past the batch
            rows = torch.arange(n, device="cuda") % 4096
            same = got[:n].view(torch.int32) == full[rows].view(torch.int32)
            assert bool(same.all()), (n, k, torch.nonzero(~same)[:5].tolist())


@pytest.mark.parametrize("small,large,most", [(8, 64, 1.3), (8192, 9000, 1.43),
                                              (32768, 34000, 1.39)])
def test_scans_are_shared_out(torch_cuda, hip, small, large, most):
    """Where every environment is scanned through clutter, a batch a little
    above a shape's bound must not take much longer than one at it: its
    workgroups are spread over the CUs.  With 16, 32 and 64 environments in
    every workgroup the larger batches took 1.46, 1.67 and 1.53 times the
    smaller ones' time, in shares 1.14, 1.19 and 1.25; the bounds lie halfway.
    Medians of alternating runs of one device, so that clocks cancel."""
    torch = torch_cuda
    print(f"[gpu-case] onboard times {small} / {large}", flush=True)
    b = synth.make_batch(4096, seed=79, threads=16)
    mission = b.mission.copy()
    mission[:, 4], mission[:, 5] = 1.0, 0.0  # slalom
    rows = torch.arange(large, device="cuda") % 4096
    obs = torch.from_numpy(in_window(b.obs)).cuda()[rows].contiguous()
    d_mission = torch.from_numpy(mission).cuda()[rows].contiguous()
    out = [torch.empty((large, w), device="cuda") for w in (24, 15, 5)]
    s = torch.cuda.current_stream()
    times = {small: [], large: []}
    for _ in range(15):
        for n in times:
            first, last = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            first.record(s)
            for _ in range(100):
                assert hip.onboard_tactical_prior_device(obs, d_mission, *out, n, s) == 1
            last.record(s)
            last.synchronize()
            times[n].append(first.elapsed_time(last) * 10.0)
    at = {n: float(np.median(t)) for n, t in times.items()}
    print(f"[gpu-case] us {at}", flush=True)
    assert at[large] < most * at[small], at


@pytest.mark.parametrize("n", [9000, 17000, 33000])
def test_one_wild_arm_input(torch_cuda, hip, n):
    """Ordinary environments with one arm input that is NaN, infinite or large:
    a quad's lanes each read one arm, a lane of the largest batches all four,
    and both must take the environment for the same kind of input."""
    torch = torch_cuda
    print(f"[gpu-case] onboard one wild arm input {n}", flush=True)
    b = synth.make_batch(4096, seed=77, threads=16)
    obs, e = in_window(b.obs), np.arange(4096)
    wild = np.array([np.nan, np.inf, -np.inf, 1.2e4, -3.0e5], np.float32)
    obs[e, 16 + e % 16] = wild[e // 16 % 5]
    d_obs, d_mission = torch.from_numpy(obs).cuda(), torch.from_numpy(b.mission).cuda()
    rows = torch.arange(n, device="cuda") % 4096

    def run(o, m):
        out = [torch.full((o.shape[0], w), 7.0, device="cuda") for w in (24, 15)]
        s = torch.cuda.current_stream()
        assert hip.onboard_tactical_prior_device(o, m, *out, None, o.shape[0], s) == 1
        assert hip.synchronize(s) == 1
        return out

    small = run(d_obs, d_mission)
    large = run(d_obs[rows].contiguous(), d_mission[rows].contiguous())
    for k in range(2):
        same = large[k].view(torch.int32) == small[k][rows].view(torch.int32)
        assert bool(same.all()), (n, k, int((~same).any(1).sum()), torch.nonzero(~same)[:5].tolist())
    compare(run_onboard(torch, hip, obs, b.mission), oracle.onboard(obs, b.mission), "wild arm")


@pytest.mark.parametrize("n", [1, 47, 1024, 10000, 17000])
def test_special_rows_in_every_shape(torch_cuda, hip, n):
    b = synth.make_batch(n, seed=500 + n, variant=synth.SPECIAL, threads=16)
    # 3e38 overflows inside the reference's formulas, where the last bit of an
    # angle decides an infinity's sign
    obs, mission = in_window(b.obs), b.mission.copy()
    obs[np.abs(obs) == np.float32(3e38)] = np.float32(7.5)
    mission[np.abs(mission) == np.float32(3e38)] = np.float32(0.25)
    print(f"[gpu-case] onboard special {n}", flush=True)
    compare(run_onboard(torch_cuda, hip, obs, mission), oracle.onboard(obs, mission),
            f"special {n}")


@pytest.mark.parametrize("n", [1, 16, 17, 512, 513, 2500, 3071, 3072, 3073])
def test_actor_rows_do_not_depend_on_the_batch(torch_cuda, hip, tiled, n):
    torch = torch_cuda
    obs, mission = tiled
    print(f"[gpu-case] actor inputs {n}", flush=True)
    g = torch.Generator("cuda").manual_seed(5)
    cameras = torch.randint(0, 256, (4096, 16384), dtype=torch.uint8, device="cuda", generator=g)
    s = torch.cuda.current_stream()
    widths = {"proprio": 91, "mission_vec": 49, "tactical": 24, "prior": 15, "lidar": 12288,
              "luma": 16384}

    def run(k, lidar=True, luma=True):
        out = {w: torch.full((k + 1, v), 7.0, device="cuda") for w, v in widths.items()}
        assert hip.actor_inputs_device(
            obs, mission, cameras, out["proprio"], out["mission_vec"], out["tactical"],
            out["prior"], out["lidar"] if lidar else None, out["luma"] if luma else None, k,
            s) == 1
        torch.cuda.synchronize()
        return out

    want = run(4000)
    for planes in ((True, True), (True, False), (False, True), (False, False)):
        got = run(n, *planes)
        for w in widths:
            if (w == "lidar" and not planes[0]) or (w == "luma" and not planes[1]):
                assert bool((got[w] == 7.0).all())
                continue
            assert bool((got[w][n] == 7.0).all()), (w, planes)
            same = got[w][:n].view(torch.int32) == want[w][:n].view(torch.int32)
            assert bool(same.all()), (w, planes, torch.nonzero(~same)[:5].tolist())
