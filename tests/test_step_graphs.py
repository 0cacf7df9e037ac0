"""Which captured graphs run() launches (csrc/step_graphs.hpp), compiled for the
host: a capture of several steps that fails leaves run() its one-step graph."""
import subprocess

from cmag_amd import build as B

SOURCE = r"""
#include <cstdio>
#include <vector>

#include "step_graphs.hpp"

// a graph is a pointer to its steps; captures of more than `limit` fail
struct Host {
    unsigned limit;
    std::vector<unsigned> captured, failed;
    cmag::StepGraphs<unsigned*> g;
    int prepare(unsigned steps) {
        return g.prepare(steps,
                         [&](unsigned k, unsigned** out) {
                             (k > limit ? failed : captured).push_back(k);
                             if (k > limit) return -2;
                             *out = new unsigned(k);
                             return 0;
                         },
                         [](unsigned* q) { delete q; });
    }
    unsigned launched(unsigned steps, unsigned& launches) {
        unsigned done = 0;
        for (unsigned k = 0; k < steps; ++launches) {
            unsigned n = 0;
            const unsigned* q = g.next(steps - k, n);
            if (!q || *q != n) return 0;
            k += n;
            done += n;
        }
        return done;
    }
};

int main() {
    const unsigned runs[] = {5, 5, 5, 40, 40, 40, 3, 3, 1, 1, 40, 40};
    for (unsigned limit : {16u, 15u, 4u, 1u}) {
        Host h{limit};
        for (unsigned steps : runs) {
            unsigned launches = 0;
            const int rc = h.prepare(steps);
            const unsigned done = rc == 0 ? h.launched(steps, launches) : 0;
            std::printf("limit %u run %u rc %d steps %u launches %u\n", limit, steps, rc, done, launches);
        }
        std::printf("limit %u captured", limit);
        for (unsigned k : h.captured) std::printf(" %u", k);
        std::printf(" failed");
        for (unsigned k : h.failed) std::printf(" %u", k);
        std::printf("\n");
    }
    Host none{0};
    std::printf("none rc %d\n", none.prepare(3));
    return 0;
}
"""


def test_a_failed_capture_leaves_the_single_steps(tmp_path):
    src, exe = tmp_path / "host.cpp", tmp_path / "host"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{B.CSRC}", str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.splitlines()
    rows = [dict(zip(x.split()[::2], map(int, x.split()[1::2]))) for x in out if " rc " in x and x.startswith("limit")]
    assert len(rows) == 48
    for r in rows:
        assert r["rc"] == 0 and r["steps"] == r["run"], r
    first = {r["limit"]: r["launches"] for r in rows if r["run"] == 40}  # the last run of 40
    assert first == {16: 2 + 8, 15: 40 // 5, 4: 13 + 1, 1: 40}
    # a count that failed is not tried again by the next equal run
    assert "limit 16 captured 1 5 16 failed" in out
    assert "limit 15 captured 1 5 failed 16" in out
    assert "limit 4 captured 1 3 failed 5 16" in out
    assert "limit 1 captured 1 failed 5 16 3" in out
    # without the one-step graph there is nothing to launch: the error
    assert out[-1] == "none rc -2"
