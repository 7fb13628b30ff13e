"""The Morton grid's range (physkit_amd/csrc/pk_trim.hpp, the header compiled for the host): the
sample is not the same body of every world of a batch, whatever the worlds' size; a few bodies
far away do not widen the range, and nothing else loses its cells: not a scene whose bodies
mostly share a coordinate, nor the bodies above a flat layer, nor that layer's own order."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EXE = os.path.join(ROOT, "tests", "cpp", "_build", "trim_check")


@pytest.fixture(scope="module")
def ask():
    os.makedirs(os.path.dirname(EXE), exist_ok=True)
    subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "-O2", "-std=c++20", "-ffp-contract=off",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    "-I", os.path.join(ROOT, "physkit_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "trim_check.hip"), "-o", EXE], check=True, capture_output=True)

    def run(text):
        return np.array(subprocess.run([EXE], input=text, capture_output=True, text=True, check=True).stdout.split(), float)

    return run


@pytest.mark.parametrize("worlds", [1024, 2048, 4096, 1000, 1])
@pytest.mark.parametrize("size", [2, 16, 64, 256, 1025])
def test_sample_spreads_over_the_worlds_bodies(ask, worlds, size):
    n = worlds * size
    if n <= 1024:
        pytest.skip("every body of such a scene is taken")
    s = ask(f"S {n}").astype(np.int64)
    assert len(s) == 1024 and s[0] >= 0 and s[-1] < n and (np.diff(s) > 0).all()
    # each body of a world is met about 1024 / size times, and no more often than 6 sigma of chance
    mean = 1024.0 / min(size, 1024)
    assert np.bincount(s % size).max() <= mean + 6.0 * np.sqrt(mean) + 1.0


def _range(ask, pos):
    out = ask(f"R {len(pos)} " + " ".join(repr(float(x)) for x in pos.T.ravel()))
    return out.reshape(3, 2)


def _outside(pos, r):
    return ((pos < r[:, 0]) | (pos > r[:, 1])).sum(0)


@pytest.mark.parametrize("n", [40, 200, 1024, 5000])
def test_few_outliers_are_cut(ask, n):
    rng = np.random.default_rng(n)
    pos = rng.uniform(0.0, 10.0, (n, 3))
    bulk = pos.copy()
    out = [7] if n < 1024 else [7, n // 3]
    pos[out, 1] = -1e6
    r = _range(ask, pos)
    if n >= 64:
        assert r[1, 0] > -50.0
        assert _outside(bulk, r).max() == 0
    else:
        assert r[1, 0] == -1e6  # too few to tell: the exact bounds


@pytest.mark.parametrize("frac", [0.0, 0.004, 0.03, 0.2])
def test_no_more_than_a_few_lose_their_cells(ask, frac):
    """A flat layer with a share of the bodies far above it, in equal worlds with their ground
    as body 0: at most one in 128 ends outside, and the layer's axis is not cut finer than
    the layer is wide."""
    rng = np.random.default_rng(3)
    worlds, size = 1024, 16
    pos = rng.uniform(-20.0, 20.0, (worlds * size, 3))
    pos[:, 1] = 0.5 + 1e-6 * rng.normal(size=len(pos))
    up = rng.random(len(pos)) < frac
    pos[up, 1] = rng.uniform(50.0, 400.0, int(up.sum()))
    pos[::size] = [0.0, -0.5, 0.0]
    r = _range(ask, pos)
    assert _outside(pos, r).max() <= len(pos) / 128
    wide = np.minimum(pos.max(0) - pos.min(0), 40.0)
    assert (r[:, 1] - r[:, 0] >= 0.99 * wide).all()


def test_one_place_keeps_the_exact_bounds(ask):
    pos = np.zeros((2000, 3))
    pos[1999] = [3.0, -4.0, 5.0]
    np.testing.assert_array_equal(_range(ask, pos), [[0.0, 3.0], [-4.0, 0.0], [0.0, 5.0]])
