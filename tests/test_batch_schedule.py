"""How a batch is launched (rocrand_amd/csrc/rr_batch_schedule.hpp, compiled here with g++
behind tests/batch_schedule_shim.cpp): one launch only for several groups of bounded output
and tiles, and never many small tiles for a group that fills the chip with fewer."""
import ctypes
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "rocrand_amd", "csrc")
MIB = 1 << 20


@pytest.fixture(scope="module")
def schedule(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    so = str(tmp_path_factory.mktemp("schedule") / "libschedule.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I", CSRC,
                    os.path.join(HERE, "batch_schedule_shim.cpp"), "-o", so], check=True)
    f = ctypes.CDLL(so).batch_schedule_of
    f.argtypes = [ctypes.c_size_t] * 3 + [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p]

    def call(groups, nbytes, inter_tiles, philox_vecs=()):
        arr, tile = (ctypes.c_size_t * max(1, len(philox_vecs)))(*philox_vecs), ctypes.c_uint(0)
        return bool(f(groups, nbytes, inter_tiles, arr, len(philox_vecs), ctypes.byref(tile))), tile.value

    return call


def test_long_mrg32k3a_streams_take_their_groups_kernels(schedule):
    """512 tiles a stream, whatever its length: 16 streams have few tiles for any output."""
    assert not schedule(3, 16 << 30, 16 * 512)[0]
    assert not schedule(3, 4 << 30, 4 * 512)[0]
    assert schedule(3, 256 * MIB, 16 * 512)[0]


def test_long_philox_streams_take_their_groups_kernels(schedule):
    assert not schedule(3, 1024 * MIB, 0, [4 * MIB] * 16)[0]
    assert not schedule(3, 512 * MIB + 4, 0, [2 * MIB] * 16)[0]
    assert schedule(3, 512 * MIB, 0, [2 * MIB - 1] * 16)[0]


def test_one_group_takes_its_own_kernel(schedule):
    for vecs in (1, 1000, 262144):
        assert not schedule(1, 16 * vecs * 4, 0, [vecs] * 4)[0]
    assert not schedule(1, MIB, 64)[0]


def test_many_tiles_take_their_groups_kernels(schedule):
    assert schedule(6, 32 * MIB, 4096, [1000] * 4096)[0]
    assert not schedule(6, 32 * MIB, 4097, [1000] * 4096)[0]
    assert not schedule(2, MIB, 8193)[0]


@pytest.mark.parametrize("groups,inter,vecs,most", [
    (2, 0, [4096] * 256, 4096), (2, 2500, [4300] * 128, 4096), (1, 0, [32768] * 4, 256), (1, 0, [262144] * 4, 300)])
def test_tiles_are_fine_but_few(schedule, groups, inter, vecs, most):
    tile = schedule(groups, 16 * sum(vecs), inter, vecs)[1]
    assert tile in (256, 512, 1024, 2048, 4096)
    count = lambda t: inter + sum(v // t + 1 for v in vecs)  # noqa: E731
    assert count(tile) <= most or tile == 4096
    assert tile == 256 or count(tile // 2) > (4096 if groups > 1 else 256)
