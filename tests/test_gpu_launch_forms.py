"""Forms a step's passes take by size, against the forms they replace.

The wave runs as blocks of the force launch in small scenes and as a launch of
its own otherwise; a profiled step always launches it by itself.  Both must
give the same state to the bit."""
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
