"""CPU check of the key-split prefill plan (csrc/prefill_split.hpp, compiled with the host
compiler): over random chunks, windows and head shapes
  - the workgroups (pf_split_item over pf_split_grid) are each (KV head, piece, block) once;
  - the pieces of ct tiles cover every block's tiles, and every block's tiles cover
    exactly the keys its rows see;
  - the partials fit what the workspace reserves (pf_split_ws_bytes), and the workgroups
    with tiles fit the resident ones.
"""
from __future__ import annotations

import pathlib
import shutil
import subprocess

import pytest

CSRC = pathlib.Path(__file__).resolve().parent.parent / "gguf-runner_amd" / "csrc"

MAIN = r"""
#include "prefill_split.hpp"
#include <cstdio>
#include <random>
#include <set>
#include <tuple>
using namespace gr;
#define CHECK(x) do { if (!(x)) { printf("failed: %s (m %d heads %d/%d p0 %d w %d image %d bm %d bn %d)\n", #x, m, kv * mul, kv, p0, w, img, bm, bn); return 1; } } while (0)
int main() {
    std::mt19937 r(7);
    auto pick = [&](int lo, int hi) { return lo + (int)(r() % (unsigned)(hi - lo + 1)); };
    int planned = 0;
    for (int it = 0; it < 4000; it++) {
        const int kv = pick(1, 17), mul = pick(1, 17), m = pick(0, 3) ? pick(1, 700) : pick(1, 5000);
        const int p0 = pick(0, 2) ? pick(0, 9000) : 0, w = pick(0, 1) ? 0 : pick(1, 2000), img = pick(0, 4) == 0;
        const int bm = pick(0, 1) ? 128 : 64, bn = 32 << pick(0, 2), slots = 256 * pick(1, 2), d = 64 << pick(0, 2);
        const PrefillSplit s = pf_split_plan(m, kv * mul, kv, p0, w, img, bm, bn, slots, pick(1, 4));
        if (s.n_splits == 0) continue;
        planned++;
        CHECK(s.ct > 0 && s.n_splits > 1 && s.n_qb == (m * mul + bm - 1) / bm);
        CHECK(pf_split_part_bytes(s, kv, d) <= pf_split_ws_bytes(slots, bm, d));
        int64_t tiles = 0, wgs = 0;
        for (int qb = 0; qb < s.n_qb; qb++) {
            const int t = pf_split_tiles(qb, bm, bn, m, mul, p0, w, img);
            int lo = 1 << 30, hi = 0;  // keys of the block's rows
            for (int row = qb * bm; row < (qb + 1) * bm && row < m * mul; row++) {
                const int pos = p0 + row / mul;
                int a = w ? (pos + 1 > w ? pos + 1 - w : 0) : 0;
                int b = pos + 1;
                if (img) a = a < p0 ? a : p0, b = p0 + m;
                lo = a < lo ? a : lo, hi = b > hi ? b : hi;
            }
            CHECK(t == (hi + bn - 1) / bn - lo / bn);
            CHECK((t + s.ct - 1) / s.ct <= s.n_splits);
            tiles += t, wgs += (t + s.ct - 1) / s.ct;
        }
        CHECK(tiles * kv == s.tiles && wgs * kv == s.wgs && s.wgs <= slots);
        std::set<std::tuple<int, int, int>> seen;
        const int grid = pf_split_grid(kv, s.n_qb, s.n_splits);
        int n = 0;
        for (int b = 0; b < grid; b++) {
            const PfSplitItem i = pf_split_item(b, kv, s.n_qb, s.n_splits);
            if (i.qb >= s.n_qb) continue;
            n++;
            CHECK(i.g >= 0 && i.g < kv && i.piece >= 0 && i.piece < s.n_splits && i.qb >= 0);
            seen.insert({i.g, i.piece, i.qb});
        }
        CHECK(n == kv * s.n_qb * s.n_splits && (int)seen.size() == n);
    }
    printf("planned %d\n", planned);
    return planned > 1000 ? 0 : 1;
}
"""


def test_split_plan_covers_every_key_once(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("no host C++ compiler")
    src = tmp_path / "plan.cpp"
    src.write_text(MAIN)
    exe = tmp_path / "plan"
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{CSRC}",
                    str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
