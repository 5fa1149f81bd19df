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


@pytest.mark.parametrize("sx,sz", [(1, 1), (-1, 1), (1, -1), (-1, -1)])
@pytest.mark.parametrize("n,W,H", [(4096, 128, 100), (4096, 131, 64), (50_000, 256, 256)])
def test_wave_tiles_mirrored_and_replayed(gpu, cwa, n, W, H, sx, sz):
    """A heightfield mirrored along an axis, stepped eagerly, from graphs and with
    the wave in a launch of its own."""
    from coupledwateranimation_amd import configs

    print(f"wave tiles n={n} {W}x{H} {sx} {sz}", flush=True)
    spec = configs.dam_break_diff(n, 64, 5)
    p = spec.params.copy()
    for a, sign in ((0, sx), (1, sz)):
        if sign < 0:
            p.wave_origin[a] += 1.0 / p.wave_uv_scale[a]
            p.wave_uv_scale[a] *= -1.0
    h = np.random.default_rng(n).normal(0.0, 0.02, (2, H, W)).astype(np.float32)
    states = []
    for form in ("step", "graph", "profiled"):
        with cwa.Scene(p, spec.pos, spec.vel, None, (W, H), h[0], h[1]) as s:
            if form == "profiled":
                s.step_profiled(spec.dt, 15)
            else:
                s.step(spec.dt, 15, graph=form == "graph")
            states.append(s.readback())
    _same(states[0], states[2], "eager")
    _same(states[1], states[2], "graph")


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


@pytest.mark.parametrize("which", ["pos", "vel"])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_force_of_a_particle_that_left_the_numbers(gpu, cwa, which, value):
    """A particle without neighbours adds nothing, whatever its own record holds and
    however many neighbours the particle has that shares its loads: one lane per
    particle gives the finite numbers that four lanes give."""
    from coupledwateranimation_amd import configs

    print(f"force {which} {value}", flush=True)
    spec = configs.dam_break_diff(2048, 96, 7)
    n = 2000
    rng = np.random.default_rng(3)
    pos, vel = spec.pos[:n].copy(), np.zeros((n, 4), np.float32)
    vel[:, :3] = rng.normal(0.0, 0.3, (n, 3))
    odd = rng.permutation(n)[:40]
    if which == "vel":  # apart from the others, each alone
        pos[odd, :3] = 0.35 + 0.6 * rng.random((40, 3))
        pos[odd, 1] = 0.02 * np.arange(40) + 0.1
    (pos if which == "pos" else vel)[odd, rng.integers(0, 3, 40)] = value
    (a, _), (b, _) = [_scene_state(cwa, spec, pos, vel, None, k, 1) for k in (-1, 0)]
    for k in ("force", "vel", "pos"):
        assert np.array_equal(np.isfinite(a[k]), np.isfinite(b[k])), k
        both = np.isfinite(a[k])
        err = np.abs(a[k][both] - b[k][both]).max()
        assert err <= 512 * 2.0 ** -24 * np.abs(b[k][both]).max(), k


@pytest.mark.parametrize("shape", ["1", "20", "21", "32", "33", "64", "65", "300", "columns",
                                   "lattice", "far"])
def test_density_by_packed_points(gpu, cwa, oracle, shape):
    """The one-lane pass finds every neighbour, whatever the length of a column
    (chunks of 32 candidates, 20 tested at once), the number of a particle's
    words (more than eight, more than are recorded) and its distance to the
    grid.  Its sum differs from the four-lane pass's in order only: within
    2 * terms * 2^-24 of it, all terms being positive."""
    from coupledwateranimation_amd import configs
    from coupledwateranimation_amd.scene import set_lane_split_limit

    print(f"packed density {shape}", flush=True)
    spec = configs.dam_break_diff(4096, 96, 7)
    h = spec.params.h
    cell, lo = spec.params.cell_size, np.array(list(spec.params.grid_min))
    rng = np.random.default_rng(len(shape))
    if shape.isdigit():      # one column of so many candidates
        pos = lo + cell * (3 + 0.9 * rng.random((int(shape), 3)))
    elif shape == "columns":  # 3 x 3 columns of several chunks each
        pos = lo + cell * (2 + 3 * rng.random((700, 3)))
    elif shape == "lattice":
        pos = spec.pos[:4001, :3].astype(np.float64)
    else:                    # beyond the range of the packed coordinates, and at the grid
        pos = np.concatenate([spec.pos[:500, :3], spec.pos[:500, :3] + 20_000 * h])
    n = len(pos)
    p4 = np.zeros((n, 4), np.float32)
    p4[:, :3] = pos
    zero = np.zeros((96, 96), np.float32)
    got = []
    old = set_lane_split_limit(0)
    try:
        for limit in (0, 1 << 20):
            set_lane_split_limit(limit)
            with cwa.Scene(spec.params, p4, np.zeros_like(p4), None, (96, 96), zero, zero) as s:
                s.step(spec.dt, 1)
                got.append((s.neighbour_counts(), s.readback()))
    finally:
        set_lane_split_limit(old)
    counts = oracle.neighbor_counts(spec.params, p4, all_pairs=True)
    assert np.array_equal(got[0][0], counts) and np.array_equal(got[1][0], counts)
    assert counts.max() > 1 or n == 1
    a, b = got[0][1]["rho"], got[1][1]["rho"]
    assert np.abs(a - b).max() <= 2 * counts.max() * 2.0 ** -24 * np.abs(b).max()


@pytest.mark.parametrize("n,W,H", [(1, 3, 5), (2, 4, 4), (3, 7, 3), (255, 33, 31), (1025, 16, 64),
                                   (4099, 65, 63)])
def test_tape_copies_whole_states(gpu, cwa, n, W, H):
    """Checkpoints and the final state come back as they were, whatever remains
    past the last 16 bytes of an array: a backward pass (which replays the steps
    from the checkpoints) leaves the forward's final state, and a plain run gives
    that state too."""
    from coupledwateranimation_amd import configs
    from coupledwateranimation_amd.gradient import Tape

    print(f"tape copies n={n} {W}x{H}", flush=True)
    spec = configs.dam_break_diff(max(n, 64), 64, 5)
    rng = np.random.default_rng(n)
    vel = np.zeros((n, 4), np.float32)
    vel[:, :3] = rng.normal(0.0, 0.3, (n, 3))
    h = rng.normal(0.0, 0.02, (2, H, W)).astype(np.float32)
    make = lambda: cwa.Scene(spec.params, spec.pos[:n].copy(), vel, None, (W, H),  # noqa: E731
                             h[0], h[1])
    with make() as plain:
        plain.step(spec.dt, 7)
        ref = plain.readback()
    with make() as s:
        tape = Tape(s, 7, 3)
        tape.forward(spec.dt)
        _same(s.readback(), ref, "forward")
        grads = [tape.backward(dheight0=np.ones((H, W), np.float32)) for _ in range(2)]
        _same(s.readback(), ref, "backward")
        tape.close()
    assert grads[0][0] == grads[1][0]
    assert np.array_equal(grads[0][2], grads[1][2])


@pytest.mark.parametrize("counts", [(1,), (2, 3, 5), (15, 16, 17, 1), (63, 64, 65, 257), (4097, 700),
                                    (20_000,)])
def test_batched_pairs_with_four_lanes(gpu, cwa, counts):
    """Batches of up to 80 000 particles sum a particle's candidates with four
    lanes, larger ones with one: the same scenes, alone and with others that make
    the batch large, to the bit."""
    from coupledwateranimation_amd import batch2d

    print(f"batched lanes {counts}", flush=True)
    others = (30_000, 30_000, 30_000)
    n, nw = sum(counts), 40 * len(counts)
    got = []
    for sizes in (counts, counts + others):
        spec = batch2d.dam_break_batch(sizes, [40] * len(sizes), seed=3)
        rng = np.random.default_rng(n)
        spec.xv[:n, 2:] = rng.normal(0.0, 0.5, (n, 2))
        spec.xv[:n:7, 0] = spec.xv[0, 0]  # some on a line, two points on each other
        if n > 1:
            spec.xv[1, :2] = spec.xv[0, :2]
        spec.enabled = np.ones(spec.n_total, np.int32)
        spec.enabled[:n:5] = 0
        b = spec.make()
        b.step(spec.dt, 3)
        r = b.readback()
        b.close()
        got.append({k: np.ascontiguousarray(r[k][:n]) for k in ("xv", "rp", "enabled")} |
                   {k: np.ascontiguousarray(r[k][:nw]) for k in ("h0", "h1")})
    for k in got[0]:
        assert np.array_equal(got[0][k].view(np.uint32), got[1][k].view(np.uint32)), k


@pytest.mark.parametrize("counts", [(1,), (5, 63, 65), (1000, 2049, 17), (30_000, 30_001, 30_003)])
@pytest.mark.parametrize("substeps", [1, 2])
def test_batched_keys_from_the_step_before(gpu, cwa, counts, substeps):
    """A call of several steps hashes each step's keys in the force pass before;
    calls of one step hash them afresh.  Same grid and state to the bit, eager and
    from graphs, also when the caller moves particles between calls."""
    import torch
    from coupledwateranimation_amd import batch2d

    print(f"batched keys {counts} x{substeps}", flush=True)
    spec = batch2d.dam_break_batch(counts, [33] * len(counts), seed=4)
    spec.params.sph_substeps = substeps
    rng = np.random.default_rng(sum(counts))
    spec.xv[:, 2:] = rng.normal(0.0, 3.0, (spec.n_total, 2))  # cells change
    got = []
    for calls, graph in (([1] * 23, False), ([23], False), ([3, 1, 8, 9, 2], True),
                         ([6, 17], True), ([23], True)):
        b = spec.make()
        done = 0
        for c in calls:
            b.step(spec.dt, c, graph=graph)
            done += c
        state = b.readback() | {f"slot_{k}": np.asarray(v) for k, v in b.slots().items()}
        # the caller puts the particles elsewhere: the next call starts from there
        class View:
            __cuda_array_interface__ = {"data": (int(b.views().xv), False),
                                        "shape": (spec.n_total, 4), "typestr": "<f4",
                                        "version": 2}
        torch.as_tensor(View(), device=gpu)[:, :2] *= 0.5
        torch.cuda.synchronize()
        b.step(spec.dt, 2, graph=graph)
        state |= {f"moved_{k}": v for k, v in b.readback().items()}
        b.close()
        got.append(state)
    for other in got[1:]:
        for k, v in got[0].items():
            assert np.array_equal(v, other[k], equal_nan=v.dtype.kind == "f"), k


@pytest.mark.parametrize("h", [0.02, 0.01, 0.004])
@pytest.mark.parametrize("counts", [(1,), (5, 63, 64, 65), (700,)])
def test_batched_keys_in_sparse_grids(gpu, cwa, counts, h):
    """The same with 14 to 250 000 cells a particle: run lists cleared cell by cell
    or, with more than 1 024, particle by particle."""
    from coupledwateranimation_amd import batch2d

    print(f"batched sparse {counts} h={h}", flush=True)
    spec = batch2d.dam_break_batch(counts, [33] * len(counts), seed=4, dt=1e-4,
                                   params=batch2d.unit_square_params(h=h))
    rng = np.random.default_rng(sum(counts))
    spec.xv[:, 2:] = rng.normal(0.0, 20.0, (spec.n_total, 2))
    got = []
    for calls, graph in (([1] * 9, False), ([9], False), ([9], True)):
        b = spec.make()
        for c in calls:
            b.step(spec.dt, c, graph=graph)
        got.append(b.readback())
        b.close()
    for other in got[1:]:
        for k, v in got[0].items():
            assert np.array_equal(v, other[k], equal_nan=v.dtype.kind == "f"), k


@pytest.mark.parametrize("n", [262_144, 262_145, 270_011])
@pytest.mark.parametrize("coarse", [1, 2])
def test_runs_listed_beside_the_scan(gpu, cwa, n, coarse):
    """Builds of more than 2^18 particles list their runs in the scan's launch of
    tile sums, or by themselves where the scan takes one launch (65 536 cells or
    fewer): the list is the stable order of the keys on each."""
    from coupledwateranimation_amd import configs

    print(f"runs beside the scan n={n} coarse={coarse}", flush=True)
    spec = configs.dam_break_large(3, n=n, wave=64)
    p = spec.params.copy()
    p.cell_size *= coarse
    for a in range(3):
        p.grid_dims[a] = max(1, -(-p.grid_dims[a] // coarse))
    rng = np.random.default_rng(n)
    vel = np.zeros_like(spec.pos)
    vel[:, :3] = rng.normal(0.0, 1.0, (n, 3))
    with cwa.Scene(p, spec.pos, vel, None, spec.wave_size, spec.height0, spec.height1) as s:
        s.step(spec.dt, 3)
        g = s.grid_host()
    assert np.array_equal(g["list"], np.argsort(g["key"], kind="stable"))
    assert np.array_equal(g["count"], np.bincount(g["key"], minlength=g["count"].size))
    assert np.array_equal(g["offset"], np.concatenate([[0], np.cumsum(g["count"])]))


@pytest.mark.parametrize("n", [262_144, 262_145, 786_432, 786_433, 1_000_003])
@pytest.mark.parametrize("order", ["random", "nearly", "one cell"])
@pytest.mark.parametrize("static", [False, True])
def test_grid_builds_in_any_order(gpu, cwa, n, order, static):
    """Builds of up to 2^18 points list their runs where the keys are counted, up to
    3 * 2^18 in a pass of their own, larger ones place them in the cells' segments:
    the stable order of the keys on each."""
    import ctypes as C

    import torch
    from coupledwateranimation_amd import _lib

    print(f"grid build n={n} {order} static={static}", flush=True)
    cells = 20
    rng = np.random.default_rng(n)
    pos = np.ones((n, 4), np.float32)
    pos[:, :3] = rng.random((n, 3)) * (0.9 / cells if order == "one cell" else 1.0)
    if order == "nearly":
        c = np.minimum((pos[:, :3] * cells).astype(np.int64), cells - 1)
        near = (c[:, 2] * cells + c[:, 0]) * cells + c[:, 1] + rng.integers(-2, 3, n)
        pos = pos[np.argsort(near, kind="stable")]
    d = torch.tensor(pos, device=gpu)
    key, cnt, off, lst = [torch.full((k,), -1, dtype=torch.int32, device=gpu)
                          for k in (n, cells ** 3, cells ** 3 + 1, n)]
    fn = cwa.lib().cwa_grid_build_static if static else cwa.lib().cwa_grid_build
    _lib.check(fn(d.data_ptr(), n, (C.c_float * 3)(0, 0, 0), 1.0 / cells,
                  (C.c_int32 * 3)(cells, cells, cells), key.data_ptr(), cnt.data_ptr(),
                  off.data_ptr(), lst.data_ptr(), None))
    torch.cuda.synchronize()
    k = key.cpu().numpy()
    count = np.bincount(k, minlength=cells ** 3)
    assert np.array_equal(lst.cpu().numpy(), np.argsort(k, kind="stable"))
    assert np.array_equal(cnt.cpu().numpy(), count)
    assert np.array_equal(off.cpu().numpy(), np.concatenate([[0], np.cumsum(count)]))


@pytest.mark.parametrize("n,listed", [(350_000, True), (370_000, False)])
def test_box_grids_of_many_pairs(gpu, cwa, oracle, n, listed):
    """The same with boxes over about six cells each: fewer and more pairs than
    2^21, against the oracle."""
    import ctypes as C

    import torch
    from coupledwateranimation_amd import _lib

    cells = 20
    rng = np.random.default_rng(n)
    x, h = np.ones((n, 4), np.float32), np.full((n, 4), 0.02, np.float32)
    x[:, :3] = 0.1 + 0.8 * rng.random((n, 3))
    ref = oracle.grid_build_boxes(x, h, (0.0,) * 3, (1.0 / cells,) * 3, (cells,) * 3)
    print(f"box grid n={n} pairs={ref['total']}", flush=True)
    assert (ref["total"] <= 1 << 21) == listed
    cap, total = ref["total"], C.c_int64()
    dx, dh = torch.tensor(x, device=gpu), torch.tensor(h, device=gpu)
    got = {k: torch.full((m,), -1, dtype=torch.int32, device=gpu)
           for k, m in (("count", cells ** 3), ("offset", cells ** 3 + 1), ("list", cap))}
    _lib.check(cwa.lib().cwa_grid_build_boxes(
        dx.data_ptr(), dh.data_ptr(), n, (C.c_float * 3)(0, 0, 0),
        (C.c_float * 3)(*[1.0 / cells] * 3), (C.c_int32 * 3)(cells, cells, cells),
        *[got[k].data_ptr() for k in ("count", "offset", "list")], cap, C.byref(total), None))
    assert total.value == cap
    for k, v in got.items():
        assert np.array_equal(v.cpu().numpy(), ref[k]), k
