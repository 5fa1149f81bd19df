"""The packed points of the one-lane density pass never rule out a neighbour.

A host restatement of pack_point and pack_test (cwa_device.hpp) over pairs at
up to the support radius, at offsets up to the range in which a point's
candidates are tested at all, with coordinates on both sides of the 256-unit
wrap.  Constants are read from the header."""
import re
from pathlib import Path

import numpy as np
import pytest

SRC = (Path(__file__).resolve().parent.parent / "coupledwateranimation_amd" / "csrc" /
       "cwa_device.hpp").read_text()


def _const(name):
    return float(re.search(rf"constexpr \w+ {name} = ([0-9.]+)f?;", SRC).group(1))


UNITS, LT, RANGE = (_const(k) for k in ("kPackUnits", "kPackLt", "kPackRange"))


def _pack(p, gmin, scale):
    f = np.floor(((p - gmin).astype(np.float32) * scale).astype(np.float32))
    b = f.astype(np.int64) & 255
    return (b[:, 0] | b[:, 1] << 8 | b[:, 2] << 16).astype(np.uint32)


def _dist2(a, b):
    d = (b - a).astype(np.uint32)  # wraps, as the kernel's subtraction
    byte = np.stack([(d >> s) & 255 for s in (0, 8, 16, 24)], 1).astype(np.int64)
    byte -= 256 * (byte > 127)
    return (byte * byte).sum(1)


@pytest.mark.parametrize("h", [0.0232, 1.0, 3.7e-3])
@pytest.mark.parametrize("offset", [0.0, 1.7, 300.0, 12_000.0])
def test_no_neighbour_is_ruled_out(h, offset):
    rng = np.random.default_rng(int(offset) + int(1000 * h))
    n = 400_000
    scale = np.float32(UNITS) / np.float32(h)
    gmin = np.array([-0.3, 0.11, 0.0], np.float32)
    a = (gmin + np.float32(h) * (offset + rng.uniform(-3, 3, (n, 3)))).astype(np.float32)
    way = rng.normal(size=(n, 3))
    way[: n // 4] = np.sign(way[: n // 4]) * (rng.random((n // 4, 3)) < 0.5)  # axes, diagonals
    way /= np.maximum(np.linalg.norm(way, axis=1, keepdims=True), 1e-9)
    r = np.where(rng.random(n) < 0.7, 1.0, rng.random(n))
    b = (a + (h * r)[:, None] * way).astype(np.float32)
    near = ((a.astype(np.float64) - b) ** 2).sum(1) < np.float64(h) ** 2
    inside = (np.abs((a - gmin) * scale) < RANGE).all(1)
    assert inside.all() and near.sum() > n // 4
    d2 = _dist2(_pack(a, gmin, scale), _pack(b, gmin, scale))
    assert d2[near].max() < LT
    # and most of what is far is ruled out: beyond 1.1 h, short of the wrap
    far = np.minimum(1.1 + 0.4 * rng.random(n), 1.5)
    c = (a + (h * far)[:, None] * way).astype(np.float32)
    moved = np.abs(way).max(1) > 0
    assert (_dist2(_pack(a, gmin, scale), _pack(c, gmin, scale))[moved] >= LT).mean() > 0.9


def test_bound():
    err = np.sqrt(1.25 ** 2 + 2 * 2.25 ** 2 + 1.0)
    assert (UNITS + err) ** 2 < LT < (UNITS + err + 0.2) ** 2
    assert UNITS + 2.25 < 127                 # a neighbour's bytes do not wrap
    assert RANGE * 4 * 2.0 ** -24 <= 0.25     # rounding of both scaled coordinates
