"""The depth bound that lets the overdraw raster drop triangles (tri_bound.h),
against a walk of random triangles in the reference's own f32 arithmetic
(tests/native/tri_bound.cpp, built here by g++)."""
import ctypes as C
import os
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ is missing")


class Count(C.Structure):
    _fields_ = [("tris", C.c_long), ("bounded", C.c_long), ("samples", C.c_long), ("below", C.c_long),
                ("worst", C.c_double)]


@pytest.fixture(scope="module")
def sweep(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("tri_bound") / "libtri_bound.so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-fno-fast-math", "-shared", "-fPIC",
                    "-I" + os.path.join(REPO, "swraster-viewer_amd", "csrc"),
                    os.path.join(REPO, "tests", "native", "tri_bound.cpp"), "-o", out], check=True)
    fn = C.CDLL(out).tri_bound_sweep
    fn.argtypes = [C.c_uint64] + 4 * [C.c_int] + 2 * [C.c_double] + [C.POINTER(Count)]

    def run(*args):
        n = Count()
        fn(*args, C.byref(n))
        return n
    return run


# slivers whose edge values round by more than their area, at 4K and at the
# largest frame; frames whose i32 edge constants wrap; triangles of ordinary
# shape, which must keep their bound.  bounded: the least share with a bound.
@pytest.mark.parametrize("W,H,kind,size,ratio,count,bounded", [
    (3840, 2160, 0, 2500, 4.0, 15000, 0.0), (3840, 2160, 0, 300, 1.5, 20000, 0.5), (1280, 720, 0, 900, 15.0, 20000, 0.0),
    (32000, 32000, 0, 600, 8.0, 2000, 0.0), (5120, 2880, 1, 1200, 4.0, 150, 0.0), (7680, 4320, 1, 1500, 4.0, 150, 0.0),
    (3840, 2160, 2, 40, 1.3, 4000, 0.99), (1920, 1080, 2, 200, 4.0, 1000, 0.95)])
def test_no_covered_sample_below_the_bound(sweep, W, H, kind, size, ratio, count, bounded):
    n = sweep(W + kind, count, W, H, kind, size, ratio)
    print(n.tris, n.bounded, n.samples, n.below, n.worst)
    assert n.samples > 0
    assert n.below == 0, f"{n.below} of {n.samples} samples below, by up to {n.worst:.1e} of the depth"
    assert n.bounded >= bounded * n.tris
