"""The descriptor blocks of the one-shot batched call (rocrand_amd/csrc/rr_staging.hpp, compiled
here with g++ behind tests/staging_shim.cpp, a stand-in for the HIP runtime): what happens to
blocks whose streams are destroyed or captured, and to errors that the caller has not read."""
import ctypes
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "rocrand_amd", "csrc")
ROCM = "/opt/rocm/include"
DONE, NOT_READY, GONE, OTHER = 0, 600, 900, 101
KIB64 = 64 << 10


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.isdir(ROCM):
        pytest.skip("g++ or the HIP headers not available")
    so = str(tmp_path_factory.mktemp("staging") / "libstaging.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I", CSRC, "-I", ROCM,
                    "-Wl,-Bsymbolic", os.path.join(HERE, "staging_shim.cpp"), "-o", so], check=True)
    L = ctypes.CDLL(so)
    L.staging_new.restype = ctypes.c_void_p
    L.staging_use.restype = ctypes.c_void_p
    L.staging_use.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int, ctypes.c_int]
    L.staging_collect.argtypes = [ctypes.c_void_p]
    return L


class Pool:
    def __init__(self, L):
        self.L, self.p = L, L.staging_new()

    def use(self, query=DONE, nbytes=1000, captured=False):
        return self.L.staging_use(self.p, nbytes, captured, query)

    def collect(self):
        self.L.staging_collect(self.p)

    def set(self, last=0, sync=0):
        self.L.staging_set(last, sync)

    def counts(self):
        c = (ctypes.c_int * 4)()
        self.L.staging_counts(c)
        return dict(zip(("mallocs", "syncs", "queries", "last"), c))


def test_a_finished_block_is_used_again(lib):
    p = Pool(lib)
    a = p.use()
    assert p.use(nbytes=KIB64) == a and p.use(nbytes=KIB64 + 1) != a
    assert p.use(NOT_READY) == a and p.use() != a  # still in use: another block
    c = p.counts()
    assert c["syncs"] == 0 and c["last"] == 0


@pytest.mark.parametrize("query", [DONE, NOT_READY, GONE])
def test_an_unread_error_stays_for_the_caller(lib, query):
    p = Pool(lib)
    p.use(query)
    p.set(last=OTHER)
    p.use()
    p.collect()
    assert p.counts()["last"] == OTHER


@pytest.mark.parametrize("query", [NOT_READY, GONE])
def test_a_querys_own_error_is_not_left_behind(lib, query):
    p = Pool(lib)
    p.use(query)
    p.collect()
    assert p.counts()["last"] == 0


def test_a_block_whose_stream_is_gone_comes_back_after_a_wait_for_the_device(lib):
    p = Pool(lib)
    a = p.use(GONE)
    b = p.use(GONE)  # the first one's failure shows here: one wait, no allocation
    assert b == a and p.counts() == {"mallocs": 1, "syncs": 1, "queries": 1, "last": 0}
    for _ in range(10):
        assert p.use(GONE) == a
    assert p.counts()["mallocs"] == 1
    # while another block is free nothing waits
    big = p.use(nbytes=1 << 20)
    syncs = p.counts()["syncs"]
    assert p.use(GONE, nbytes=1 << 20) == big and p.counts()["syncs"] == syncs


def test_a_failed_wait_leaves_the_block_out_of_use(lib):
    p = Pool(lib)
    a = p.use(GONE)
    p.set(sync=OTHER)
    b = p.use(NOT_READY)
    assert b != a and p.counts()["last"] == 0
    p.set()
    assert p.use() == a


def test_a_captured_call_asks_nothing_and_keeps_its_block(lib):
    p = Pool(lib)
    a = p.use(GONE)
    b = p.use(captured=True)
    assert b != a
    assert p.counts() == {"mallocs": 2, "syncs": 0, "queries": 0, "last": 0}
    assert b not in {p.use(NOT_READY) for _ in range(4)}
    c = p.use(DONE)
    p.collect()
    assert p.use(captured=True) == c  # a free block, without an allocation
