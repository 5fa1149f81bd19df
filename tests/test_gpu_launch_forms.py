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
