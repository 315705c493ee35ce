"""A run's start clears the status and sets its host error word in one
wavefront (status_begin, shared with the kernels): no lane's result depends on
the order in which the lanes' stores land."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r'''
#include <cstdio>
#include <cstring>
#include <algorithm>
#include <numeric>
#include <random>
#include <vector>
#include "ft_types.h"
using namespace ft;
int main() {
    std::vector<uint32_t> lane(256);
    std::iota(lane.begin(), lane.end(), 0u);
    std::mt19937 g(1);
    uint32_t word = 0;
    for (int k = 0; k < 200; ++k) {  // first to last, last to first, then any order
        if (k == 1) std::reverse(lane.begin(), lane.end());
        if (k > 1) std::shuffle(lane.begin(), lane.end(), g);
        struct { DevStatus st; uint32_t after[4]; } s;
        memset(&s, 0xA5, sizeof s);
        for (uint32_t i : lane) status_begin(&s.st, i, &word);
        if (s.st.host_err != &word) return printf("order %d: host_err is %p\n", k, (void *)s.st.host_err), 1;
        s.st.host_err = nullptr;
        DevStatus zero;
        memset(&zero, 0, sizeof zero);
        if (memcmp(&s.st, &zero, sizeof zero)) return printf("order %d: a word was left\n", k), 1;
        for (uint32_t a : s.after) if (a != 0xA5A5A5A5u) return printf("order %d: past the end\n", k), 1;
    }
    return 0;
}
'''


def test_status_begin_in_any_lane_order(tmp_path):
    src, exe = tmp_path / "s.cpp", tmp_path / "s"
    src.write_text(SRC)
    subprocess.run(["g++", "-O1", "-std=c++17", f"-I{os.path.join(ROOT, 'footile_amd', 'csrc')}", "-o", str(exe),
                    str(src)], check=True)
    r = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert r.returncode == 0, r.stdout


def test_every_kernel_starts_its_status_so():
    """No kernel zeroes the status's words or stores host_err by itself but
    the one that keeps a failed run's status."""
    for name in ("ft_pipeline.hip", "ft_diff.hip"):
        with open(os.path.join(ROOT, "footile_amd", "csrc", name)) as f:
            text = f.read()
        assert "reinterpret_cast<uint32_t *>(st)[" not in text, name
        assert text.count("st->host_err =") == (1 if name == "ft_pipeline.hip" else 0), name
