"""The mixed flash's buffers (csrc/mixed_data.h) when device memory runs out.

They are made on the first mixed call.  An allocation that fails ends that
call with an error and leaves the handle usable, so whichever one fails, the
next call has to make exactly those that are missing: a kernel launched with
a null list writes through it.  On the CPU, with an allocator that fails at
each allocation in turn."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "spuma-multiphysics_amd", "csrc")
SOURCE = """#include "mixed_data.h"
#include <cstdio>
#include <cstdlib>
#include <new>
#include <type_traits>
using namespace ramd;
int main() {
    const struct { int ns; bool prune, pure; } models[] = {{1, false, true}, {1, true, false}, {1, false, false}, {2, false, false}, {2, true, false}};
    for (const auto& m : models)
        for (int fail = 0;; ++fail) {
            MixedScratch s;
            int calls = 0, made = 0;
            const auto alloc = [&](auto*& p, size_t n) {
                if (p) return;
                if (calls++ == fail) throw std::bad_alloc();
                p = static_cast<std::remove_reference_t<decltype(p)>>(std::malloc(n * sizeof(*p)));
                ++made;
            };
            bool failed = false;
            try { s.need(m.ns, m.prune, m.pure, 5, alloc); } catch (const std::bad_alloc&) { failed = true; }
            const int before = made;
            s.need(m.ns, m.prune, m.pure, 5, alloc);
            const int buffers = 3 + (m.prune ? 0 : 2) + (m.pure ? 4 : 0);
            const bool searched = s.search.records && s.search.restarts && s.search.restartCount == s.counts + kRestartCount &&
                                  s.search.slowCount == s.counts + kSlowCount;
            const bool directed = s.saturation && s.searchList && s.search.again && s.search.single &&
                                  s.search.againCount == s.counts + kAgainCount && s.search.singleCount == s.counts + kSingleCount;
            if (!(s.sets && s.queue && s.counts && (m.prune || searched) && (!m.pure || directed) && made == buffers &&
                  (!failed || before == fail) && failed == (fail < buffers)))
                return std::printf("model %d %d %d, allocation %d\\n", m.ns, m.prune, m.pure, fail), 1;
            if (!failed) break;
        }
    std::puts("ok");
}
"""


def test_a_failed_allocation_leaves_the_rest_to_the_next_call(tmp_path):
    (tmp_path / "scratch.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, "-o", str(tmp_path / "scratch"),
                    str(tmp_path / "scratch.cpp")], check=True)
    run = subprocess.run([str(tmp_path / "scratch")], capture_output=True, text=True)
    assert run.stdout == "ok\n", run.stdout
