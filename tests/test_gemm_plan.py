"""The complex GEMM's plan on the host: how long a chain of additions it allows."""
import ctypes as ct
import pathlib
import shutil
import subprocess

import pytest

NATIVE = pathlib.Path(__file__).parent / "native"


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.fail("no g++ to build the host program")
    path = tmp_path_factory.mktemp("plan") / "libgemm_plan_check.so"
    subprocess.run([cxx, "-O2", "-std=c++17", "-fPIC", "-shared", "-o", str(path), str(NATIVE / "gemm_plan_check.cpp")],
                   check=True)
    lib = ct.CDLL(str(path))

    def call(fp64, m, n, k):
        out = (ct.c_int * 3)()
        lib.gemm_plan_of(int(fp64), m, n, k, out)
        return tuple(out)

    return call


def _longest_chain(fp64, m, n, k):
    """K of a split with 32 x 32 tiles split, doubling, to 2048 (FP32: 1024) workgroups,
    256 of K and more a split, 64 splits at most, in whole slabs of 16."""
    tiles = -(-m // 32) * -(-n // 32)
    splits = 1
    while tiles * splits < (2048 if fp64 else 1024) and k // (2 * splits) >= 256 and splits < 64:
        splits *= 2
    return -(-(-(-k // splits)) // 16) * 16


# projections (projectors x columns x plane waves), Galerkin and Gram blocks, back
# projections and rotations of the smallest to the largest cells, ragged ones among them
BANDS = [1, 2, 4, 20, 37, 80, 96, 160, 240, 333, 480, 1500]
WAVES = [813, 1153, 1647, 4573, 6589, 9141, 17000, 23847]


@pytest.mark.parametrize("fp64", [True, False])
def test_chains_of_a_split(plan, fp64):
    shapes = [(p, c, n) for p in (64, 128, 256, 416, 512) for c in BANDS for n in WAVES]
    shapes += [(r, c, n) for r in BANDS for c in BANDS for n in WAVES]
    shapes += [(n, c, p) for p in (64, 512, 900) for c in BANDS for n in WAVES]
    for m, n, k in shapes:
        _, splits, kps = plan(fp64, m, n, k)
        assert kps <= _longest_chain(fp64, m, n, k), (m, n, k)
        assert kps % 16 == 0 and splits * kps >= k, (m, n, k)
        # the workspace is sized for FP64
        assert splits <= plan(True, m, n, k)[1], (m, n, k)
