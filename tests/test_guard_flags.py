"""Flags of the tests whether a clip or a projection may fire (csrc/guard_flags.h): one that no kernel reached reads "may fire",
and threads that ask for their first one at the same time share one allocation."""
import ctypes
import os
import subprocess

import pytest

from nl_hecate_amd import ffi

SOURCE = r"""
#include "guard_flags.h"
#include <atomic>
#include <cstdlib>
#include <set>
#include <thread>
#include <vector>
using namespace nlh;

extern "C" int may_fire(int fired, int reached) {
    GuardFlags<4> flags;
    GuardFlag *f = flags.lowered([](size_t n) { return std::malloc(n); });
    if (reached) f->reached = 1;
    if (fired) f->fired = 1;
    return !guard_clear(f);
}
// allocations and different places of `threads` first calls at once
extern "C" int first_calls(int threads, int *places) {
    GuardFlags<64> flags;
    std::atomic<int> allocations{0}, ready{0};
    std::vector<GuardFlag *> got(threads);
    std::vector<std::thread> all;
    for (int i = 0; i < threads; i++)
        all.emplace_back([&, i] {
            ready++;
            while (ready < threads) {}
            got[i] = flags.lowered([&](size_t n) { allocations++; return std::malloc(n); });
        });
    for (auto &t : all) t.join();
    *places = (int)std::set<GuardFlag *>(got.begin(), got.end()).size();
    return allocations;
}
extern "C" int without_memory() {
    GuardFlags<4> flags;
    return flags.lowered([](size_t) -> void * { return nullptr; }) == nullptr && flags.lowered([](size_t n) { return std::malloc(n); }) != nullptr;
}
"""


@pytest.fixture(scope="module")
def flags(tmp_path_factory):
    at = tmp_path_factory.mktemp("flags")
    (at / "flags.cpp").write_text(SOURCE)
    csrc = os.path.join(os.path.dirname(os.path.abspath(ffi.__file__)), "csrc")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-pthread", "-I", csrc, "-o", str(at / "flags.so"),
                           str(at / "flags.cpp")])
    return ctypes.CDLL(str(at / "flags.so"))


def test_only_a_kernel_that_ran_can_clear(flags):
    assert [flags.may_fire(f, r) for f, r in ((0, 0), (1, 0), (1, 1), (0, 1))] == [1, 1, 1, 0]


def test_first_calls_of_several_threads(flags):
    for _ in range(50):
        places = ctypes.c_int()
        assert flags.first_calls(4, ctypes.byref(places)) == 1 and places.value == 4
    assert flags.without_memory() == 1
