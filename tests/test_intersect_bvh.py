"""Triangle test, BVH build and traversal on the CPU: the oracle's
Moller-Trumbore against FP64 and known answers, BVH traversal (the
oracle's own median BVH and the product's binned-SAH BVH) against brute
force, any-hit against closest hit, and the host BVH's invariants."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from globillum_amd import scenes
from globillum_amd.context import build_bvh2

FMAX = np.finfo(np.float32).max


def test_intersect_known_answer(oracle):
    hit, t, u, v = oracle.intersect_tri((-1, -1, 0), (1, -1, 0), (0, 1, 0), (0, 0, -2), (0, 0, 1))
    assert hit and t == 2.0
    # P = (1-u-v) a + u b + v c = (0, 0, 0)  ->  u = 1/4, v = 1/2
    assert u == pytest.approx(0.25) and v == pytest.approx(0.5)
    # behind the origin, parallel, outside the edge
    assert not oracle.intersect_tri((-1, -1, 0), (1, -1, 0), (0, 1, 0), (0, 0, 2), (0, 0, 1))[0]
    assert not oracle.intersect_tri((-1, -1, 0), (1, -1, 0), (0, 1, 0), (0, 0, -1), (1, 0, 0))[0]
    assert not oracle.intersect_tri((-1, -1, 0), (1, -1, 0), (0, 1, 0), (5, 0, -1), (0, 0, 1))[0]


def test_intersect_fp32_vs_fp64(oracle):
    rng = np.random.default_rng(0)
    agree = 0
    n = 3000
    for _ in range(n):
        a, b, c = rng.normal(size=(3, 3))
        o = rng.normal(size=3) * 3
        u, v = rng.uniform(0, 1, 2)
        if u + v > 1:
            u, v = 1 - u, 1 - v
        target = a + u * (b - a) + v * (c - a)
        d = target - o
        d /= np.linalg.norm(d)
        a, b, c, o, d = (x.astype(np.float32).astype(np.float64) for x in (a, b, c, o, d))
        nrm = np.cross(b - a, c - a)
        cos = abs(np.dot(d, nrm)) / np.linalg.norm(nrm)
        h32, t32, u32, v32 = oracle.intersect_tri(a, b, c, o, d)
        h64, t64, u64, v64 = oracle.intersect_tri(a, b, c, o, d, f64=True)
        if h32 and h64:
            agree += 1
            # FP32 error grows as 1/cos at grazing incidence
            assert abs(t32 - t64) <= 2e-6 * (abs(t64) + 1.0) / max(cos, 1e-3)
            # hit point reconstructs from the barycentrics
            P = (1 - u64 - v64) * a + u64 * b + v64 * c
            assert np.allclose(P, o + t64 * d, atol=1e-9)
        elif h32 != h64:
            # only at the triangle border
            assert min(u64, v64, 1 - u64 - v64) > -1e-5
    assert agree > 0.98 * n


def _random_rays(rng, n, lo, hi):
    o = rng.uniform(lo, hi, (n, 3)).astype(np.float32)
    d = rng.normal(size=(n, 3)).astype(np.float32)
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return o, d


@pytest.fixture(scope="module")
def c1():
    return scenes.cornell_boxes()


@pytest.fixture(scope="module")
def terrain_small():
    return scenes.terrain_spheres(cells=(48, 48), n_spheres=60, w=64, h=36, spp=2)


def test_bvh_traversal_equals_brute_force(oracle, c1, terrain_small):
    rng = np.random.default_rng(3)
    for sc, lo, hi in ((c1, -0.2, 1.2), (terrain_small, -5.0, 105.0)):
        own = oracle.OracleScene(sc.tris)
        sah = oracle.OracleScene(sc.tris, bvh2=build_bvh2(sc.tris))
        o, d = _random_rays(rng, 60000, lo, hi)
        if sc is terrain_small:
            o[:, 1] = rng.uniform(0, 15, len(o))
        tmax = np.where(rng.random(len(o)) < 0.3, rng.uniform(0, 20, len(o)), FMAX).astype(np.float32)
        ref = own.brute_closest(o, d, tmax)
        assert (own.trace_closest(o, d, tmax) == ref).all()
        assert (sah.trace_closest(o, d, tmax) == ref).all()
        assert 0.05 < (ref["ref"] != 0xFFFFFFFF).mean() < 1.0


def test_random_soup_traversal(oracle):
    rng = np.random.default_rng(5)
    from globillum_amd._lib import TRI
    tris = np.zeros(3000, TRI)
    c = rng.uniform(0, 10, (3000, 1, 3))
    v = (c + rng.normal(size=(3000, 3, 3)) * 0.5).astype(np.float32)
    tris["a"], tris["b"], tris["c"] = v[:, 0], v[:, 1], v[:, 2]
    own = oracle.OracleScene(tris)
    sah = oracle.OracleScene(tris, bvh2=build_bvh2(tris, max_leaf=8))
    o, d = _random_rays(rng, 20000, -1, 11)
    tmax = np.full(len(o), FMAX, np.float32)
    ref = own.brute_closest(o, d, tmax)
    assert (own.trace_closest(o, d, tmax) == ref).all()
    assert (sah.trace_closest(o, d, tmax) == ref).all()


def test_closest_hit_ties_break_to_lower_id(oracle):
    # two coincident triangles: equal t, the lower id wins in every traversal
    from globillum_amd._lib import TRI
    tris = np.zeros(4, TRI)
    quad = np.array([[0, 0, 0], [1, 0, 0], [1, 1, 0], [0, 1, 0]], np.float32)
    for i, (a, b, c) in enumerate([(0, 1, 2), (0, 2, 3), (0, 1, 2), (0, 2, 3)]):
        tris[i]["a"], tris[i]["b"], tris[i]["c"] = quad[a], quad[b], quad[c]
    tris = tris[[2, 0, 3, 1]]  # ids: duplicates at (0,1) and (2,3)
    own = oracle.OracleScene(tris, max_leaf=1)
    o = np.array([[0.7, 0.2, -1], [0.2, 0.7, -1]], np.float32)
    d = np.array([[0, 0, 1], [0, 0, 1]], np.float32)
    h = own.trace_closest(o, d, np.full(2, FMAX, np.float32))
    assert h["ref"].tolist() == [0, 2]
    assert (h == own.brute_closest(o, d, np.full(2, FMAX, np.float32))).all()


def test_any_hit_matches_closest(oracle, terrain_small):
    rng = np.random.default_rng(9)
    sc = oracle.OracleScene(terrain_small.tris, bvh2=build_bvh2(terrain_small.tris))
    o, d = _random_rays(rng, 30000, 0, 100)
    o[:, 1] = rng.uniform(0, 15, len(o))
    tmax = rng.uniform(0, 40, len(o)).astype(np.float32)
    h = sc.trace_closest(o, d, np.full(len(o), FMAX, np.float32))
    any_ = sc.trace_any(o, d, tmax)
    assert np.array_equal(any_.astype(bool), (h["ref"] != 0xFFFFFFFF) & (h["t"] <= tmax))


def test_host_bvh_invariants(terrain_small):
    tris = terrain_small.tris
    nodes, idx = build_bvh2(tris, max_leaf=4)
    assert sorted(idx.tolist()) == list(range(len(tris)))
    ib = nodes.view(np.int32).reshape(-1, 8)
    box = nodes.reshape(-1, 8)[:, 2:8]
    V = np.stack([tris["a"], tris["b"], tris["c"]], 1)
    seen = 0
    for i in range(len(ib)):
        x, y = ib[i, 0], ib[i, 1]
        lo, hi = box[i, :3], box[i, 3:]
        if x & 1:
            for ch in (x >> 1, y):
                assert np.all(box[ch, :3] >= lo) and np.all(box[ch, 3:] <= hi)
        else:
            cnt = x >> 1
            assert 1 <= cnt <= 15
            seen += cnt
            pts = V[idx[y:y + cnt]].reshape(-1, 3)
            assert np.all(pts >= lo) and np.all(pts <= hi)
    assert seen == len(tris)


def test_host_bvh_empty_and_errors():
    import ctypes as C
    from globillum_amd import _lib
    lib = _lib.load()
    h = C.c_void_p()
    assert lib.gi_bvh_build(None, 5, 4, C.byref(h)) == 1
    from globillum_amd._lib import TRI
    one = np.zeros(1, TRI)
    one["b"] = (1, 0, 0)
    one["c"] = (0, 1, 0)
    nodes, idx = build_bvh2(one)
    assert len(nodes) == 8 and idx.tolist() == [0]


def test_empty_slots_are_never_hit(tmp_path):
    """The kernels' slab test, compiled for the host from the same header
    (tests/csrc/slab_check.cpp): empty child slots miss for all eight sign
    combinations and for limits up to infinity and NaN; boxes at finite
    distances within the limit hit."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    exe = str(tmp_path / "slab_check")
    r = subprocess.run([shutil.which("g++") or "g++", "-O2", "-std=c++17", "-ffp-contract=off", "-o", exe,
                        os.path.join(root, "tests", "csrc", "slab_check.cpp")], capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and " 0 bad" in r.stdout, r.stdout
