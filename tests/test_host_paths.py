"""libsbgpu.so's host paths over a stand-in for the HIP runtime
(tests/fake_hip.cpp) in which kernels do nothing and streams count their work:
what a call leaves queued when it fails, and in which order it waits and
copies.  Runs without a GPU, each test in a process of its own."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import ctypes, sys
sys.path.insert(0, {root!r})
fake = ctypes.CDLL({fake!r}, mode=ctypes.RTLD_GLOBAL)
fake.fake_watch.argtypes = [ctypes.c_void_p]
fake.fake_watched.restype = ctypes.c_char_p
import numpy as np
from solidboolean_amd import native as N
STREAM, AUX = 0, 1  # the context's streams, in the order it makes them
ctx = N.Context(0)
def locked(a):
    out = N.host_array(a.nbytes).view(a.dtype).reshape(a.shape)
    out[...] = a
    return out
def soup(nt):
    return ctx.mesh(np.random.default_rng(nt).random((30, 3)), np.arange(3 * nt).reshape(nt, 3) % 30)
"""


@pytest.fixture(scope="session")
def fake_hip(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("fake_hip") / "libfakehip.so")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-o", out,
                           os.path.join(ROOT, "tests", "fake_hip.cpp")])
    return out


def run(fake_hip, body):
    done = subprocess.run([sys.executable, "-c", PRELUDE.format(root=ROOT, fake=fake_hip) + body], text=True,
                          capture_output=True, timeout=120)
    assert done.returncode == 0, done.stdout + done.stderr
    return done.stdout


CALLS = {
    "components": ("k_cc_labels", 0, "soup(200).components(locked(np.zeros(200, np.uint8)))"),
    "half_edges": ("k_he_query", 0,
                   "ctx.half_edges(locked(np.arange(300, dtype=np.uint32).reshape(-1, 3)), np.arange(9, dtype=np.uint64))"),
    "tri_tri_batch": ("k_tritri_raw", 0, "ctx.tri_tri_batch(locked(np.ones((500, 9))), np.ones((500, 9)))"),
    "classify_points": ("k_vote", 0, "M.classify_points(locked(np.ones((70000, 3))))"),
    "adjoint": ("k_volume", 0, "ctx.adjoint(locked(np.ones((30, 3))), np.zeros((4, 5)), np.zeros((6, 3)))"),
    "pair": ("k_vote", 0, "A.classify_pair(B, P, out=(locked(np.zeros(900, np.uint8)), locked(np.zeros(700, np.uint8))))"),
    "split pair": ("k_vote", 1, "A.classify_pair(B, P, out=(locked(np.zeros(400000, np.uint8)),"
                                " locked(np.zeros(300000, np.uint8))))"),
}


def test_pair_lists_share_page_locked_memory(fake_hip):
    """Lists kept alive together, and made after others were dropped, take their
    hit counts' page-locked words from blocks of the context's."""
    run(fake_hip, """
A, B = soup(50), soup(60)
def lists(n):
    out = [A.find_pairs(B) for _ in range(n)]
    for p in out:
        p.tri_tri(A, B, N.FP64, stats=False)
    return out
lists(1)
before = fake.fake_host_allocs()
keep = lists(1000)
assert fake.fake_host_allocs() == before
for p in keep[:600]:
    p.close()
keep += lists(600)
assert fake.fake_host_allocs() == before
keep += lists(1000)
assert fake.fake_host_allocs() == before + 1
""")


def test_classification_survives_a_failed_allocation(fake_hip):
    """No C++ exception leaves the classification entry points when the heap is
    exhausted: once its buffers stand, a call allocates nothing and succeeds."""
    run(fake_hip, """
A, B = soup(50), soup(60)
P = A.find_pairs(B)
P.tri_tri(A, B, N.FP64, stats=False)
def calls(out=None):
    out = A.classify_pair(B, P, out=out)
    A.classify_triangles(B, P, 0)
    B.classify_triangles(A, P, 1)
    return out
out = calls()
fake.fake_fail_new(1)
calls(out)
fake.fake_fail_new(0)
""")


@pytest.mark.parametrize("name", CALLS)
def test_failed_call_leaves_nothing_queued(fake_hip, name):
    """A launch that fails after the call's arrays were queued to the GPU, or after
    a side's votes were queued to page-locked arrays: the call raises, and no
    copy or kernel that could still touch the caller's memory is left behind."""
    kernel, skip, call = CALLS[name]
    a, b = (400000, 300000) if name == "split pair" else (900, 700)
    run(fake_hip, f"""
M = soup(40)
A, B = soup({a}), soup({b})
P = A.find_pairs(B)
P.tri_tri(A, B, N.FP64, stats=False)
fake.fake_drain()
fake.fake_fail_kernel({kernel.encode()!r}, {skip})
try:
    {call}
except N.SbgError as e:
    print("raised", e)
else:
    raise SystemExit("the call did not fail")
assert not fake.fake_pending(STREAM), "work left on the context stream"
assert not fake.fake_pending(AUX), "work left on the second stream"
""")
