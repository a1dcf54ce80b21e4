"""csrc/resident_choice.h, built with the host compiler: which calls of many queries over few keys go to the kernel that keeps a
head's K and V in LDS, at shapes that were measured on both kernels."""
import ctypes
import os
import subprocess

import pytest

from conftest import PKG


@pytest.fixture(scope="module")
def choice(tmp_path_factory):
    d = tmp_path_factory.mktemp("resident")
    (d / "t.cpp").write_text('#include "%s"\nextern "C" int64_t choice(int64_t B, int64_t Hq, int64_t Hkv, int64_t nq, int64_t nk) { return resident_choice(B, Hq, Hkv, nq, nk); }\n'
                             'extern "C" int64_t shares(int64_t units, int64_t tasks, int64_t nb) { return resident_shares(units, tasks, nb); }\n' % os.path.join(PKG, "csrc", "resident_choice.h"))
    subprocess.run([os.environ.get("CXX", "g++"), "-O2", "-shared", "-fPIC", "-o", str(d / "t.so"), str(d / "t.cpp")], check=True)
    lib = ctypes.CDLL(str(d / "t.so"))
    lib.choice.argtypes, lib.choice.restype = [ctypes.c_int64] * 5, ctypes.c_int64
    lib.shares.argtypes, lib.shares.restype = [ctypes.c_int64] * 3, ctypes.c_int64
    lib.choice.shares = lib.shares
    return lib.choice


# (B, Hq, Hkv, nq, nk), microseconds streamed and resident
@pytest.mark.parametrize("shape,streamed,resident", [
    ((64, 16, 16, 128, 333), 46.5, 67.8),           # few queries a head: half of the waves without a block
    ((32, 32, 16, 96, 62), 20.4, 23.9), ((16, 12, 12, 713, 21), 22.7, 26.5), ((8, 64, 16, 2986, 32), 158.4, 179.4),
    ((2, 32, 32, 21267, 21), 141.0, 161.9), ((1, 32, 4, 2071, 36), 14.6, 16.1), ((1, 1, 1, 32768, 25), 8.0, 9.3), ((32, 16, 16, 2252, 8), 121.5, 140.6),
    ((2, 16, 16, 4096, 333), 37.3, 35.0), ((1, 24, 24, 32000, 333), 163.7, 143.3), ((1, 16, 16, 16000, 352), 57.1, 52.2), ((2, 8, 8, 10000, 256), 34.5, 33.0),
    ((2, 8, 8, 32768, 174), 91.7, 76.2), ((32, 4, 4, 4041, 140), 89.4, 73.9), ((1, 24, 24, 30000, 77), 98.1, 93.4)])
def test_the_faster_of_the_two_kernels(choice, shape, streamed, resident):
    assert (choice(*shape) > 0) == (resident < streamed)


def test_workgroups_fit_a_launch(choice):
    """Up to the streaming kernel's 2^24 blocks of 32 queries: 512 threads a workgroup, fewer than 2^32 in all, and no more than
    have a block of queries for a wave."""
    seen = 0
    for B, H, Hkv, nq in ((1 << 20, 15, 15, 1), (1 << 16, 255, 255, 30), (1 << 14, 512, 512, 64), (1 << 10, 64, 8, 8000), (64, 40, 40, 200000), (1, 8, 1, 1 << 25), (1, 1, 1, 1 << 28)):
        for nk in (1, 96, 448):
            shares, tasks = choice(B, H, Hkv, nq, nk), H // Hkv * ((nq + 31) // 32)
            seen += shares > 0
            assert 0 <= shares <= (tasks + 7) // 8 and B * Hkv * shares * 512 < 1 << 32
    assert seen > 3


def test_the_numbers_passed_over_are_no_better(choice):
    for units in (1, 3, 16, 32, 100, 255, 256, 257, 5000):
        for tasks in (1, 7, 8, 9, 64, 100, 128, 500, 1000, 2047, 2048, 2049, 8000, 100000):
            for nb in (1, 3, 11):
                clocks = lambda x: -(-units * x // 256) * (13000 + 250 * nb + -(-tasks // (8 * x)) * (6800 + 1000 * nb))
                assert choice.shares(units, tasks, nb) == min(range(1, min(256, -(-tasks // 8)) + 1), key=clocks)
