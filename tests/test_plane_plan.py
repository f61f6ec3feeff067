"""The plane kernel's workgroup on the host: no other one leaves more waves on a CU."""
import ctypes as ct
import pathlib
import shutil
import subprocess

import pytest

NATIVE = pathlib.Path(__file__).parent / "native"
LDS = 160 * 1024
SIMDS = 4


@pytest.fixture(scope="module")
def waves_of(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.fail("no g++ to build the host program")
    path = tmp_path_factory.mktemp("plan") / "libplane_plan_check.so"
    subprocess.run([cxx, "-O2", "-std=c++17", "-fPIC", "-shared", "-o", str(path),
                    str(NATIVE / "plane_plan_check.cpp")], check=True)
    lib = ct.CDLL(str(path))
    return lambda *a: lib.plane_group_waves_of(*(ct.c_long(v) for v in a[:3]), *a[3:])


def _resident(waves, fixed, per_wave, per_simd):
    """Waves on a CU: workgroups that its LDS holds, and whose waves, spread over the
    SIMDs, its registers hold."""
    return waves * min(LDS // (fixed + waves * per_wave), per_simd // (waves // SIMDS))


# lines of 2 to 128 complex values, from the half of them to all; 2 waves a SIMD (wide and
# full FP64 kernels) to 4 (FP32)
@pytest.mark.parametrize("element", [8, 16])
@pytest.mark.parametrize("per_simd", [2, 3, 4])
def test_most_waves_on_a_cu(waves_of, element, per_simd):
    for n in [2, 7, 16, 30, 35, 40, 45, 48, 49, 54, 56, 60, 63, 64, 70, 72, 80, 96, 100, 128]:
        for rows in {n // 2 + 1, n}:
            fixed, per_wave = (rows + 2) * (n | 1) * element, n * 6 * element
            fits = [w for w in (4, 8) if fixed + w * per_wave <= LDS]
            got = waves_of(fixed, per_wave, LDS, SIMDS * per_simd, 8)
            if not fits:
                assert got == 0, (n, rows)
                continue
            best = max(_resident(w, fixed, per_wave, per_simd) for w in fits)
            assert got == min(w for w in fits if _resident(w, fixed, per_wave, per_simd) == best), (n, rows)
            assert waves_of(fixed, per_wave, LDS, SIMDS * per_simd, 4) in (0, 4)


def test_planes_of_48_in_double_precision(waves_of):
    # 31 of 48 lines, 8 lines a wave, registers for three waves a SIMD: three workgroups
    # of four waves, or one of eight
    assert waves_of(33 * 49 * 16, 48 * 8 * 16, LDS, 12, 8) == 4
