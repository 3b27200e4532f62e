"""The host's side of the beam loop's progress checks (csrc/beam_report.h) without a GPU: a stand-in for the stream, in a
program of its own."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "beam_report.h"
#include <stdio.h>
#include <stdlib.h>
#include <time.h>
#include <thread>
#include <chrono>

struct Fake {
    int *drains;      // how often the stream was waited for
    bool drainable;
    int running;      // what state() says
    static void *pinned(size_t n) { return aligned_alloc(64, n); }
    int state() const { return running; }
    bool drain() const { ++*drains; return drainable; }
};
using Slot = ReportSlot<Fake>;
#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)

int main() {
    int drains = 0;
    // a call that ends with launches on their way waits for them before its slot goes to the next call
    BeamReport *first;
    { Slot s(Fake{&drains, true, 1}); first = s.get(); CHECK(first); s.launching(); }
    CHECK(drains == 1);
    // one that has waited does not wait again, and one that launched nothing neither
    { Slot s(Fake{&drains, true, 1}); CHECK(s.get() == first); s.launching(); s.drained(); }
    { Slot s(Fake{&drains, true, 1}); CHECK(s.get() == first); }
    CHECK(drains == 1);
    // a slot whose stream cannot be waited for is not lent out again
    { Slot s(Fake{&drains, false, 1}); CHECK(s.get() == first); s.launching(); }
    CHECK(drains == 2);
    { Slot s(Fake{&drains, true, 1}); CHECK(s.get() != first); s.get()->check = 5; }
    // a borrowed slot holds no check of the call before
    { Slot s(Fake{&drains, true, 1}); CHECK(s.get()->check == 0); }
    // 64 calls at once: the others have no slot
    {
        Slot *all[64];
        int with = 0;
        for (auto &p : all) { p = new Slot(Fake{&drains, true, 1}); with += p->get() != nullptr; }
        CHECK(with == 63);
        for (auto p : all) delete p;
    }
    // the wait ends with the report, with a stream that has ended without one, and with a stream's error
    {
        Slot s(Fake{&drains, true, 1});
        BeamReport *r = s.get();
        std::thread gpu([r] { std::this_thread::sleep_for(std::chrono::milliseconds(200)); __atomic_store_n(&r->check, 10, __ATOMIC_RELEASE); });
        CHECK(s.wait(10) == 0);
        gpu.join();
        timespec t; clock_gettime(CLOCK_PROCESS_CPUTIME_ID, &t);
        printf("cpu_ms %ld\n", t.tv_sec * 1000 + t.tv_nsec / 1000000);
    }
    { Slot s(Fake{&drains, true, 0}); CHECK(s.wait(10) == -1); }
    { Slot s(Fake{&drains, true, -702}); CHECK(s.wait(10) == -702); }
    return 0;
}
"""


@pytest.fixture(scope="module")
def output(tmp_path_factory):
    d = tmp_path_factory.mktemp("report_slot")
    (d / "t.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-pthread", "-I", os.path.join(ROOT, "vectorlink-gpu_amd", "csrc"),
                    str(d / "t.cpp"), "-o", str(d / "t")], check=True)
    r = subprocess.run([str(d / "t")], capture_output=True, text=True, timeout=60)
    return r


def test_slots_and_waits(output):
    assert output.returncode == 0, output.stdout


def test_a_long_wait_leaves_the_core_to_others(output):
    """The stand-in GPU reports after 200 ms: a wait that only looks takes 200 ms of a core.  One that sleeps takes the 2 ms
    until it does, and a look of some us every 20 us and more (the rest: starting the program, allocating)."""
    assert output.returncode == 0, output.stdout
    cpu_ms = int(output.stdout.split("cpu_ms")[1].split()[0])
    assert cpu_ms < 60, cpu_ms
