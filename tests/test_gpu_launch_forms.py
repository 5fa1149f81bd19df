"""Forms a step's passes take by size, against the forms they replace.

The wave runs as blocks of the force launch in small scenes and as a launch of
its own otherwise; a profiled step always launches it by itself.  Both must
give the same state to the bit.  Small scans take one launch, larger ones and
scans in place two or more."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _same(a, b, what):
    for k in a:
        assert np.array_equal(a[k].view(np.uint32), b[k].view(np.uint32)), (what, k)


@pytest.mark.parametrize("n,W,H,band", [
    (1, 3, 2, 1.0), (300, 32, 32, 1.0), (4096, 33, 31, 1.0), (4096, 128, 100, 1.0),
    (4096, 131, 64, 1.0), (20_011, 250, 97, 0.0), (20_011, 16, 16, 1.0),
    (65_536, 512, 512, 1.0), (65_536, 361, 362, 1.0), (65_537, 512, 512, 1.0)])
def test_wave_in_the_force_launch(gpu, cwa, n, W, H, band):
    from coupledwateranimation_amd import configs

    print(f"fused wave n={n} {W}x{H} band={band}", flush=True)
    spec = configs.dam_break_diff(max(n, 64), 64, 5)
    p = spec.params.copy()
    p.couple_band *= band
    pos = spec.pos[:n].copy()
    rng = np.random.default_rng(n)
    vel = np.zeros_like(pos)
    vel[:, :3] = rng.normal(0.0, 0.3, (n, 3))
    h = rng.normal(0.0, 0.02, (2, H, W)).astype(np.float32)
    states = []
    for profiled in (False, True):
        with cwa.Scene(p, pos, vel, None, (W, H), h[0], h[1]) as s:
            (s.step_profiled if profiled else s.step)(spec.dt, 5)
            states.append(s.readback())
            states[-1]["colflux"] = s.grid_host()["colflux"]
    _same(*states, (n, W, H, band))


@pytest.mark.parametrize("n", [1, 8191, 8192, 8193, 65_535, 65_536, 65_537])
@pytest.mark.parametrize("form", ["apart", "misaligned", "in place"])
def test_scan_in_one_launch(gpu, cwa, n, form):
    import torch
    from coupledwateranimation_amd import _lib

    print(f"scan n={n} {form}", flush=True)
    x = np.random.default_rng(n).integers(0, 40, n).astype(np.int32)
    buf = torch.zeros(n + 8, dtype=torch.int32, device=gpu)
    src = buf[1:n + 1] if form == "misaligned" else buf[:n]
    src.copy_(torch.from_numpy(x))
    out = buf if form == "in place" else torch.full((n + 1,), -1, dtype=torch.int32, device=gpu)
    _lib.check(cwa.lib().cwa_scan_exclusive_i32(src.data_ptr(), out.data_ptr(), n, None))
    assert np.array_equal(out[:n + 1].cpu().numpy(), np.concatenate([[0], np.cumsum(x)]))
    if form != "in place":
        assert np.array_equal(src.cpu().numpy(), x)


def _scene_state(cwa, spec, pos, vel, force, limit, steps):
    from coupledwateranimation_amd.scene import set_lane_split_limit

    old = set_lane_split_limit(limit)
    try:
        with cwa.Scene(spec.params, pos, vel, force, spec.wave_size, spec.height0,
                       spec.height1) as s:
            s.step(spec.dt, steps)
            return s.readback(), s.grid_host()
    finally:
        set_lane_split_limit(old)


@pytest.mark.parametrize("n,shape", [(1, "block"), (15, "block"), (16, "block"), (17, "block"),
                                     (63, "block"), (65, "block"), (4097, "block"),
                                     (2000, "dense"), (32_768, "block"), (32_769, "block")])
def test_force_with_four_lanes(gpu, cwa, n, shape):
    """Four lanes per particle against one: the same terms in another order.
    With up to 64 neighbours a sum of 64 terms, each order within
    64 * 2^-24 of the terms' total; twice that, for terms that add up to no
    more than four times the largest force."""
    from coupledwateranimation_amd import configs

    print(f"force lanes n={n} {shape}", flush=True)
    spec = configs.dam_break_diff(max(n, 64), 96, 7)
    rng = np.random.default_rng(n)
    pos = spec.pos[:n].copy()
    if shape == "dense":  # every column longer than 64 candidates: the re-search
        pos[:, :3] = 0.4 + rng.uniform(0.0, 2.0 * spec.params.h, (n, 3))
    vel, force = np.zeros_like(pos), np.zeros_like(pos)
    vel[:, :3] = rng.normal(0.0, 0.3, (n, 3))
    force[:, :3] = rng.normal(0.0, 5.0, (n, 3))
    (a, _), (b, _) = [_scene_state(cwa, spec, pos, vel, force, k, 1) for k in (-1, 0)]
    terms = 64 if shape == "block" else n
    tol = 4 * 2 * terms * 2.0 ** -24
    for k in ("force", "vel", "pos"):
        assert np.abs(a[k] - b[k]).max() <= tol * np.abs(b[k]).max(), k
    # the next grid, from the keys and run lists the pass leaves
    _, g = _scene_state(cwa, spec, pos, vel, force, -1, 3)
    assert np.array_equal(g["list"], np.argsort(g["key"], kind="stable"))
    assert np.array_equal(g["count"], np.bincount(g["key"], minlength=g["count"].size))
