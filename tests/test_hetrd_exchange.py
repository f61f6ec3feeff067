"""The exchange of the one-launch tridiagonalisation, walked on the host over the
kernel's own rules (tests/native/hetrd_exchange_check.cpp): no workgroup reads words
that another may already have refilled, however late it is."""
import ctypes as ct
import pathlib
import shutil
import subprocess

import pytest

NATIVE = pathlib.Path(__file__).parent / "native"


@pytest.fixture(scope="module")
def exchange(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.fail("no g++ to build the host model")
    path = tmp_path_factory.mktemp("exchange") / "libhetrd_exchange_check.so"
    subprocess.run([cxx, "-O2", "-std=c++17", "-fPIC", "-shared", "-o", str(path),
                    str(NATIVE / "hetrd_exchange_check.cpp")], check=True)
    return ct.CDLL(str(path))


def test_every_reader_publishes_the_next_step(exchange):
    # the launch rule: rows a workgroup rpw, ceil(n / rpw) workgroups, at most one a CU
    for n in list(range(2, 90)) + [100, 144, 145, 160, 240, 380, 480, 512, 513, 640, 1025]:
        for rpw in {1, 2, 3, (n + 71) // 72, (n + 255) // 256, n}:
            assert exchange.hetrd_unguarded_readers(n, -(-n // rpw)) == 0, (n, rpw)


@pytest.mark.parametrize("n", [2, 3, 4, 5, 9, 16, 31])
def test_a_late_workgroup_finds_its_values(exchange, n):
    for groups in range(1, n + 1):
        for late in range(groups):
            assert exchange.hetrd_with_late_group(n, groups, late) == 0, (groups, late)
