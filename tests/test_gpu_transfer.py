"""Body state between the caller's arrays and the device, where its route changes: up to 256
KiB the kernels use pinned memory directly, up to 16 MiB it goes through device memory in one
piece, above in 16 MiB halves. Downloads
return the uploaded state bit for bit, any subset of the arrays, and set_state reaches the
named bodies alone."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# 153 bytes a body downloaded, 108 uploaded: around 256 KiB, one half and several halves
SIZES = [1, 63, 1712, 1713, 1714, 2428, 109600, 109700, 230000]


def _scene(pk, n):
    rng = np.random.default_rng(n)
    q = rng.normal(size=(n, 4))
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    return {"shape_offsets": np.array([0, 8], np.uint32), "verts": pk.mesh.box((0.5, 0.4, 0.3)).vertices,
            "is_static": (rng.random(n) < 0.1).astype(np.uint8), "shape": np.zeros(n, np.uint32),
            "pos": rng.normal(size=(n, 3)) * 50, "vel": rng.normal(size=(n, 3)), "angvel": rng.normal(size=(n, 3)),
            "quat": q, "mass": np.ones(n), "inertia": np.tile(np.eye(3).reshape(9), (n, 1)),
            "restitution": np.full(n, 0.5), "friction": np.full(n, 0.5)}


@pytest.mark.parametrize("n", SIZES)
def test_download_and_set_state(pk, n):
    s = _scene(pk, n)
    g = pk.GpuWorld()
    g.load_scene(s)
    b = g.bodies()
    for f in ("pos", "vel", "angvel", "quat"):
        np.testing.assert_array_equal(b[f], s[f])
    assert not b["moved"].any()
    assert np.isfinite(b["fat"]).all() and (b["fat"][:, :3] < s["pos"]).all() and (b["fat"][:, 3:] > s["pos"]).all()
    # a subset of the arrays
    pos, moved = np.full((n, 3), -1.0), np.full(n, 9, np.uint8)
    st = pk.pkg_body_state(pos=pos.ctypes.data_as(pk.D), moved=moved.ctypes.data_as(pk.U8))
    assert g.L.pkg_download_bodies(g.h, C.byref(st)) == 0
    np.testing.assert_array_equal(pos, s["pos"])
    assert not moved.any()
    # some bodies get new velocities and orientations, the others keep theirs
    rng = np.random.default_rng(n + 1)
    ids = rng.permutation(n)[:max(1, n - n // 7)].astype(np.uint32)
    vel, quat = rng.normal(size=(len(ids), 3)), s["quat"][ids[::-1]]
    g.set_state(ids, vel=vel, quat=quat)
    want_v, want_q = s["vel"].copy(), s["quat"].copy()
    want_v[ids], want_q[ids] = vel, quat
    b = g.bodies()
    np.testing.assert_array_equal(b["vel"], want_v)
    np.testing.assert_array_equal(b["quat"], want_q)
    for f in ("pos", "angvel"):
        np.testing.assert_array_equal(b[f], s[f])
    g.set_state(np.arange(n, dtype=np.uint32), **{f: s[f] for f in ("pos", "vel", "angvel", "quat")})
    b = g.bodies()
    for f in ("pos", "vel", "angvel", "quat"):
        np.testing.assert_array_equal(b[f], s[f])
    g.close()


def test_transfer_memory_follows_the_call(pk):
    """What a context keeps for its transfers is at most four times a call's bytes, in pinned and in
    device memory, not the largest call's: 8 contexts of 1,800 bodies (269 KiB down) hold at
    most 8 MiB of device memory for them (and one granule of 2 MiB each)."""
    from test_zz_no_alloc import Hip
    hip = Hip().L

    def free():
        assert hip.hipDeviceSynchronize() == 0
        f, t = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    worlds = []
    for k in range(8):
        worlds.append(pk.GpuWorld())
        worlds[-1].load_scene(_scene(pk, 1800))
    before = free()
    got = [g.bodies()["pos"] for g in worlds]
    used = before - free()
    print(f"[transfer] {used / 2**20:.1f} MiB of device memory for 8 contexts' transfers", flush=True)
    assert used <= (8 + 16) << 20
    want = _scene(pk, 1800)["pos"]
    for g, p in zip(worlds, got):
        np.testing.assert_array_equal(p, want)
        g.close()


def test_growing_and_shrinking_calls(pk):
    """One context whose calls go up and down over every size of the kept memory."""
    n = 230000
    s = _scene(pk, n)
    g = pk.GpuWorld()
    g.load_scene(s)
    rng = np.random.default_rng(6)
    want = s["vel"].copy()
    for count in (1, 9362, 9363, 3000, 20000, 599186, 180000, 64, 230000):
        ids = rng.permutation(n)[:min(count, n)].astype(np.uint32)
        v = rng.normal(size=(len(ids), 3))
        g.set_state(ids, vel=v)
        want[ids] = v
        got = np.full((n, 3), -1.0)
        st = pk.pkg_body_state(vel=got.ctypes.data_as(pk.D))
        assert g.L.pkg_download_bodies(g.h, C.byref(st)) == 0
        np.testing.assert_array_equal(got, want)
    g.close()
