"""What the library asks of the HIP allocator, and what it does when it is
refused: each case runs in a process of its own, behind tests/csrc/
hip_alloc_stub.cpp, which passes the calls on and refuses sizes above a
limit on request."""
import os
import shutil
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import ctypes as C, sys
stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
class S:
    def __getattr__(self, k): return C.c_uint64.in_dll(stub, "stub_" + k).value
    def __setattr__(self, k, v): C.c_uint64.in_dll(stub, "stub_" + k).value = v
S = S()
flags_all = lambda: C.c_uint32.in_dll(stub, "stub_pinned_flags_all").value
import numpy as np
from globillum_amd import scenes
from globillum_amd._lib import GiError
from globillum_amd.context import Context
import pyoracle as oracle
from test_gpu_trace import _assert_hits_equal
FMAX = np.finfo(np.float32).max
def rays(n, seed=1):
    rng = np.random.default_rng(seed)
    return (rng.uniform(-0.9, 0.9, (n, 3)).astype(np.float32), rng.normal(size=(n, 3)).astype(np.float32),
            np.full(n, FMAX, np.float32))
def same_image(ctx, sc):
    ref, _ = oracle.OracleScene(sc.tris, sc.mats, sc.lights).render(sc.views, sc.opts)
    assert (ctx.render().image(0).reshape(-1, 3) == ref).all()
def same_hits(ctx, sc, n, seed=1):
    o, d, t = rays(n, seed)
    osc = oracle.OracleScene(sc.tris)
    ref = osc.trace_closest(o, d, t)
    _assert_hits_equal(ctx.trace_closest(o, d, t), ref, osc, o, d, t)
    assert ((ctx.trace_any(o, d, t) != 0) == (ref["ref"] != 0xFFFFFFFF)).all()
"""


@pytest.fixture(scope="module")
def child(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("stub") / "alloc_stub.so")
    cxx = shutil.which("g++") or "g++"
    r = subprocess.run([cxx, "-O1", "-std=c++17", "-shared", "-fPIC", "-o", so,
                        os.path.join(ROOT, "tests", "csrc", "hip_alloc_stub.cpp"), "-ldl"],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr

    def run(body):
        env = dict(os.environ, PYTHONPATH=os.pathsep.join([ROOT, os.path.join(ROOT, "oracle"), os.path.join(ROOT, "tests")]))
        r = subprocess.run([sys.executable, "-c", PRELUDE + body, so], capture_output=True, text=True, timeout=100,
                           env=env, cwd=ROOT)
        assert r.returncode == 0, r.stdout + r.stderr

    return run


def test_pinned_memory_is_coherent(child):
    """Kernels write results straight into the pinned blocks and the host
    reads them after an event: that needs coherent memory, which the calls
    ask for by flag (hipHostMallocCoherent) and leave to no default."""
    child("""
sc = scenes.cornell_boxes(w=64, h=48, spp=2, depth=3)
with Context(0).upload(sc) as ctx:
    same_hits(ctx, sc, 1000)
    same_image(ctx, sc)
assert S.pinned > 0 and flags_all() & 0x40000000, (S.pinned, hex(flags_all()))
""")


def test_refused_pinned_memory(child):
    """Without pinned memory, or without room for the largest pinned call's
    ray buffers, images and host-array traces go by copies: the same results
    and no error, also from the calls after the refusal."""
    child("""
sc = scenes.cornell_boxes(w=300, h=301, spp=1, depth=3)
with Context(0).upload(sc) as ctx:
    S.max_pinned = 0
    for n in (1, 1000, 16384, 20000):
        same_hits(ctx, sc, n, n)
    same_image(ctx, sc)
    same_image(ctx, sc)
    assert S.refused > 0 and S.pinned == 0
    S.max_pinned = 2 ** 64 - 1
    same_image(ctx, sc)
    same_hits(ctx, sc, 1000)
    assert S.pinned > 0
with Context(0).upload(sc) as ctx:
    n = S.refused
    S.max_device = 100000
    same_hits(ctx, sc, 1000)
    assert S.refused > n
    S.max_device = 2 ** 64 - 1
    same_hits(ctx, sc, 1000, 2)
    same_image(ctx, sc)
""")


def test_calls_after_a_refused_upload(child):
    """A texture upload that the device has no memory for fails with that
    error, once: the calls after it, uploads among them, work as before."""
    child("""
sc = scenes.cornell_boxes(w=40, h=30, spp=1, depth=2)
with Context(0).upload(sc) as ctx:
    same_hits(ctx, sc, 100)
    for again in (lambda: same_hits(ctx, sc, 100), lambda: ctx.upload(sc, builder="sah"), lambda: same_image(ctx, sc)):
        S.max_device = 1 << 20
        try:
            ctx.upload_texture(np.zeros((1024, 1024, 4), np.uint8))
            assert False, "granted"
        except GiError as e:
            assert "memory" in str(e), e
        S.max_device = 2 ** 64 - 1
        again()
""")


def test_renders_after_a_refused_workspace(child):
    """A render whose path buffers are refused fails; a smaller one behind it
    does not run on what the refused growth left (the buffers it had are
    freed by then)."""
    child("""
sc = scenes.cornell_boxes(w=40, h=30, spp=2, depth=2)
big = scenes.cornell_boxes(w=256, h=256, spp=16, depth=2)
with Context(0).upload(sc) as ctx:
    same_image(ctx, sc)
    S.max_device = 4 << 20
    try:
        ctx.render(big.views, big.opts)
        assert False, "granted"
    except GiError as e:
        assert "memory" in str(e), e
    ref, _ = oracle.OracleScene(sc.tris, sc.mats, sc.lights).render(sc.views, sc.opts)
    assert (ctx.render(sc.views, sc.opts).image(0).reshape(-1, 3) == ref).all()
    S.max_device = 2 ** 64 - 1
    ref, _ = oracle.OracleScene(big.tris, big.mats, big.lights).render(big.views, big.opts)
    assert (ctx.render(big.views, big.opts).image(0).reshape(-1, 3) == ref).all()
""")
