"""The LinearBackend's way of results to the caller's memory (tritify_amd/csrc/kt_fetch.h) on a runtime that runs its
copies as late as it may: sizes around the blocks, and every call of it failing at every time. Where no pinned memory or
event is to be had the results come all the same, and nothing of a call is pending when it returns."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ALLOC, EVENT, COPY, RECORD = 1, 2, 3, 4


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fetch") / "fetch_host.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-shared", "-fPIC", "-I", os.path.join(ROOT, "tritify_amd", "csrc"),
                    os.path.join(ROOT, "tests", "fetch_host.cpp"), "-o", so], check=True)
    L = C.CDLL(so)
    L.fetch_case.restype, L.fetch_case.argtypes = C.c_int, [C.c_size_t, C.c_int, C.c_int]
    L.fetch_block.restype = C.c_size_t
    return L


def sizes(host):
    b = host.fetch_block()
    return [8, b - 8, b, b + 8, 2 * b, 2 * b + 8, 5 * b - 8]


def test_bytes(host):
    for n in sizes(host):
        assert host.fetch_case(n, 0, 0) == 3, n


@pytest.mark.parametrize("kind", [ALLOC, EVENT])
@pytest.mark.parametrize("at", [0, 1])
def test_without_pinned_memory(host, kind, at):
    for n in sizes(host):
        assert host.fetch_case(n, kind, at) == 3, n


@pytest.mark.parametrize("kind,error", [(COPY, 4), (RECORD, 5)])
@pytest.mark.parametrize("at", range(6))
def test_failed_copies_leave_nothing_pending(host, kind, error, at):
    for n in sizes(host):
        r = host.fetch_case(n, kind, at)
        assert r & 0xF0 == 0, n
        assert r >> 8 in (0, error) and (r == 3) == (r >> 8 == 0), n
