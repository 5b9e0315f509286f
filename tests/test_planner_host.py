"""The planner on the host: plans are made and run against a stand-in for the HIP runtime
(hip_host_stub.c, preloaded into a child process), which allocates from the heap and records the
shape of every launch instead of running it."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

CHILD = """
import ctypes, importlib.util
spec = importlib.util.spec_from_file_location("_lib", {lib!r})
L = importlib.util.module_from_spec(spec)
spec.loader.exec_module(L)
lib = L.lib()
stub = ctypes.CDLL(None)
stub.stub_most_groups.restype = stub.stub_most_threads.restype = stub.stub_launches.restype = ctypes.c_ulonglong

def plan(dtype, *ext, axes=L.AXES_INNERMOST):
    h = ctypes.c_void_p()
    return lib.afft_plan_create(ctypes.byref(h), dtype, len(ext), L.extents_arg(ext), axes, 0), h

def largest_prime(n):
    p, most = 2, 1
    while p * p <= n:
        while n % p == 0:
            most, n = p, n // p
        p += 1
    return max(most, n) if n > 1 else most
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("stub") / "libhip_host_stub.so")
    r = subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-w", "-I/opt/rocm/include",
                        os.path.join(HERE, "hip_host_stub.c"), "-o", out], capture_output=True, text=True)
    if r.returncode:
        pytest.skip("no C compiler or HIP headers: " + r.stderr[-300:])
    return out


def run_child(stub, code):
    head = CHILD.format(lib=os.path.join(ROOT, "accelerate-fft_amd", "afft", "_lib.py"))
    r = subprocess.run([sys.executable, "-c", head + code], env=dict(os.environ, LD_PRELOAD=stub),
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]


def test_every_long_smooth_length_has_a_plan(stub):
    """Lengths beyond one workgroup with prime factors up to 13: two factors with kernels of their
    own (the most balanced ones may have none: Complex Double 2 * 13^6 = 2197 * 4394 has no tile of
    4394), or chirp-z where there are no such factors (Complex Double 11^7)."""
    run_child(stub, """
lo, hi = 1 << 22, 1 << 25
lengths = {1}
for p in (2, 3, 5, 7, 11, 13):
    lengths |= {a * p ** k for a in lengths for k in range(1, 26) if a * p ** k <= hi}
bad = []
for n in sorted(lengths):
    if n < lo or largest_prime(n) < 7:
        continue
    for dtype in (L.C64, L.C128):
        st, h = plan(dtype, n)
        if st:
            bad.append((dtype, n, st))
        else:
            lib.afft_plan_destroy(h)
assert not bad, (len(bad), bad[:10])
""")


def test_the_identity_copies_whole_tiles(stub):
    """A transform over extents of 1 is a copy: at least 256 elements to a workgroup, and a grid of
    fewer than 2^32 threads for arrays of 2^32 elements too."""
    run_child(stub, """
for dtype in (L.C64, L.C128):
    for shape, axes in (((1000, 1), L.AXES_INNERMOST), (((1 << 24) + 3, 1), L.AXES_INNERMOST),
                        (((1 << 32) + 3, 1), L.AXES_INNERMOST), ((1, 1), L.AXES_ALL)):
        st, h = plan(dtype, *shape, axes=axes)
        assert st == 0
        stub.stub_reset()
        assert lib.afft_exec(h, -1, 256, 512, 1.0, None) == 0  # (no kernel reads these addresses)
        groups, threads = stub.stub_most_groups(), stub.stub_most_threads()
        assert 1 <= groups <= max(1024, shape[0] // 256 + 1), (dtype, shape, groups)
        assert threads < 1 << 32
        lib.afft_plan_destroy(h)
""")


def test_spectral_images_of_4_gib_stay_fused(stub):
    """The fused spectral convolution runs the row transforms twice and one launch over the columns,
    also for images of 4 GiB and more whose column tiles read whole lines (the unfused one transforms the
    columns on their own)."""
    run_child(stub, """
for dtype, h, w in ((L.C64, 32, 1 << 20), (L.C64, 32, 1 << 24), (L.C64, 512, 1 << 21), (L.C128, 16, 1 << 24)):
    st, h1 = plan(dtype, h, w)
    assert st == 0
    stub.stub_reset()
    assert lib.afft_exec(h1, -1, 256, 256, 1.0, None) == 0
    rows = stub.stub_launches()
    assert lib.afft_spectral_conv_fwd(dtype, 1, h, w, 256, 512, 768, None) == 0  # (makes the tables)
    stub.stub_reset()
    assert lib.afft_spectral_conv_fwd(dtype, 1, h, w, 256, 512, 768, None) == 0
    assert stub.stub_launches() == 2 * rows + 1, (dtype, h, w, rows, stub.stub_launches())
""")
