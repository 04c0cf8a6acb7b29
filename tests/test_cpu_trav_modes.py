"""The step traversal's forms for one instance and for identity transforms
against its general form, on the host: the same hits (bit for bit), occlusion and
fetch counts, for rays with zero, negative-zero and axis-parallel
components, masked instances, empty BLASes and rotated single instances."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import raygen
from cpu_harness import build as hbuild
from cpu_harness import harness
from solhip import scenes
from solhip.records import HIT, RAY

GENERAL, SINGLE, IDENTITY = 0, 1, 2


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    here = os.path.dirname(hbuild.__file__)
    out = str(tmp_path_factory.mktemp("modes") / "libmodes.so")
    subprocess.run(["/opt/rocm/bin/hipcc", "--cuda-host-only", "-O2", "-fPIC", "-shared", "-std=c++17",
                    "-ffp-contract=off", "-o", out, os.path.join(here, "modes_cpu.hip")], check=True)
    L = C.CDLL(out)
    vp = C.c_void_p
    L.hc_scene_create.restype = vp
    L.hc_scene_create.argtypes = [vp, vp, C.c_uint32, vp, vp, vp, C.c_uint32, C.POINTER(C.c_int)]
    L.hc_scene_destroy.argtypes = [vp]
    L.hc_set_build_flags.argtypes = [C.c_uint32]
    L.hc_trace_mode.argtypes = [vp, vp, C.c_uint32, C.c_uint32, C.c_uint32, vp, vp]
    saved, harness._lib = harness._lib, L
    yield L
    harness._lib = saved


def _trace(lib, hs, rays, mode, any_hit):
    rays = np.ascontiguousarray(rays, RAY)
    hits = np.zeros(len(rays), HIT)
    counts = np.zeros(4, np.uint64)
    lib.hc_trace_mode(hs.h, rays.ctypes.data, len(rays), int(any_hit), mode, hits.ctypes.data, counts.ctypes.data)
    return hits.tobytes(), counts.tolist()


def _rays(sd, extent):
    r = np.concatenate([raygen.random_rays(1500, (0, 0, 0), extent, seed=1), raygen.axis_rays(600),
                        raygen.aimed_rays(sd, 600, seed=2),
                        raygen.random_rays(300, (0, 0, 0), extent, seed=3, tmin=0.3, tmax=0.9)])
    # signed zeros in origins and directions
    rng = np.random.default_rng(4)
    z = r[:800].copy()
    for f in ("o", "d"):
        v = z[f]
        pick = rng.random(v.shape) < 0.4
        v[pick] = np.where(rng.random(pick.sum()) < 0.5, 0.0, -0.0)
        z[f] = v
    z["d"][(z["d"] == 0).all(axis=1)] = (1.0, -0.0, 0.0)
    return np.concatenate([r, z])


def _rotated(sd, seed):
    rng = np.random.default_rng(seed)
    m = np.eye(4)
    m[:3, :3] = scenes.random_rotation(rng) * rng.uniform(0.3, 2.0, size=3)
    m[:3, 3] = rng.uniform(-0.5, 0.5, size=3)
    return scenes.with_transforms(sd, [m] * len(sd.instance_descs))


def _masked(sd):
    sd.instance_descs["id_mask"][::2] &= 0x00FFFFFF
    return sd


SINGLES = {
    "soup": lambda: scenes.random_soup(800, seed=5),
    "terrain": lambda: scenes.heightfield(32),
    "rotated": lambda: _rotated(scenes.random_soup(500, seed=6), 7),
    "triangle": scenes.single_triangle,
    "masked": lambda: _masked(scenes.random_soup(50, seed=8)),
}


@pytest.mark.parametrize("any_hit", [False, True])
@pytest.mark.parametrize("flags", [0, 1], ids=["morton", "sah"])
@pytest.mark.parametrize("name", sorted(SINGLES))
def test_single_instance_form(lib, name, flags, any_hit):
    sd = SINGLES[name]()
    hs = harness.HostScene(sd, flags)
    rays = _rays(sd, 2.0)
    assert _trace(lib, hs, rays, SINGLE, any_hit) == _trace(lib, hs, rays, GENERAL, any_hit)


def _overlapping(n):
    """n copies of two meshes, all at the identity"""
    a, b = scenes.random_soup(300, seed=9).blas[0], scenes.heightfield(16).blas[0]
    cam = scenes.Camera((0.0, 0.0, 4.0), (0.0, 0.0, 0.0))
    return scenes.assemble("over", [a, b], [k % 2 for k in range(n)], [np.eye(4)] * n, [0] * n,
                           [scenes.material((1, 1, 1))], cam, 2.0)


IDENTITIES = {
    "cornell": scenes.cornell_box,
    "overlapping": lambda: _overlapping(9),
    "masked": lambda: _masked(_overlapping(6)),
    "one": lambda: scenes.random_soup(200, seed=10),
    "empty": scenes.empty_scene,
}


@pytest.mark.parametrize("any_hit", [False, True])
@pytest.mark.parametrize("flags", [0, 1], ids=["morton", "sah"])
@pytest.mark.parametrize("name", sorted(IDENTITIES))
def test_identity_form(lib, name, flags, any_hit):
    sd = IDENTITIES[name]()
    hs = harness.HostScene(sd, flags)
    rays = _rays(sd, 2.0) if name != "empty" else raygen.random_rays(50, (0, 0, 0), 1.0)
    assert _trace(lib, hs, rays, IDENTITY, any_hit) == _trace(lib, hs, rays, GENERAL, any_hit)
