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


CHOOSE = r"""
#include "prefill_split.hpp"
#include <algorithm>
#include <chrono>
#include <cstdio>
#include <random>
using namespace gr;
// the first piece length that fits, by trying each
static PrefillSplit each(int m, int h, int kv, int p0, int w, int img, int bm, int bn, int slots, int min_ct) {
    PrefillSplit s;
    const int mul = h / kv, n_qb = (int)(((int64_t)m * mul + bm - 1) / bm);
    int longest = 0;
    int64_t total = 0;
    for (int qb = 0; qb < n_qb; qb++) {
        const int t = pf_split_tiles(qb, bm, bn, m, mul, p0, w, img);
        longest = std::max(longest, t), total += t;
    }
    for (int ct = std::max<int64_t>(min_ct, (total * kv + slots - 1) / slots); ct < longest; ct++) {
        int64_t wgs = 0;
        for (int qb = 0; qb < n_qb; qb++) wgs += (pf_split_tiles(qb, bm, bn, m, mul, p0, w, img) + ct - 1) / ct;
        const int n = (longest + ct - 1) / ct;
        if (wgs * kv > slots || (int64_t)n_qb * kv * n > kPfSplitSlots * (int64_t)slots) continue;
        s.ct = ct, s.n_splits = n, s.tiles = total * kv, s.wgs = (int)(wgs * kv);
        break;
    }
    return s;
}
int main() {
    std::mt19937 r(11);
    auto pick = [&](int lo, int hi) { return lo + (int)(r() % (unsigned)(hi - lo + 1)); };
    int taken = 0, left = 0;
    for (int it = 0; it < 6000; it++) {
        const int kv = pick(1, 9), h = kv * pick(1, 9), m = pick(0, 3) ? pick(1, 700) : pick(1, 5000);
        const int p0 = pick(0, 2) ? pick(0, 9000) : 0, w = pick(0, 1) ? 0 : pick(1, 3000), img = pick(0, 4) == 0;
        const int bm = pick(0, 1) ? 128 : 64, bn = 32 << pick(0, 2), slots = 256 * pick(1, 2), min_ct = pick(1, 4);
        const float whole = 1 + pick(0, 300), per_wg = 0.01f * pick(0, 3);
        const PrefillSplit a = each(m, h, kv, p0, w, img, bm, bn, slots, min_ct);
        const PrefillSplit b = pf_split_plan(m, h, kv, p0, w, img, bm, bn, slots, min_ct);
        if (a.ct != b.ct || a.n_splits != b.n_splits || a.tiles != b.tiles || a.wgs != b.wgs) return printf("plan\n"), 1;
        const float cost = 1.1f * std::max((float)a.tiles / 256, (float)a.ct) + 1.0f + per_wg * a.wgs;
        const PrefillSplit c = pf_split_choose(m, h, kv, p0, w, img, bm, bn, slots, min_ct, whole, 256, per_wg);
        const bool want = a.n_splits > 0 && cost < whole;
        if (want != (c.n_splits > 0) || (want && c.ct != a.ct)) return printf("choice\n"), 1;
        (want ? taken : left)++;
    }
    // host time of a call's plan: chunks that the launch rule hands to it, `whole` as a split
    // that just loses would have it
    double worst = 0;
    const int shapes[][5] = {{4096, 14, 2, 0, 128}, {8192, 8, 1, 0, 64}, {8192, 8, 4, 0, 32}, {65000, 1, 1, 0, 64},
                             {1500, 32, 8, 0, 64}, {64, 32, 8, 100000, 64}, {16000, 4, 1, 8000, 128}, {4096, 14, 2, 8000, 128}, {2000, 14, 2, 3000, 128}};
    for (auto& s : shapes) {
        const float whole = (s[0] + 2 * s[3]) / (float)s[4] + 2;
        double best = 1e9;
        for (int i = 0; i < 30; i++) {
            const auto t = std::chrono::steady_clock::now();
            volatile int n = pf_split_choose(s[0], s[1], s[2], s[3], 0, 0, 128, s[4], 512, 1, whole, 256, 0.03f).n_splits;
            (void)n;
            best = std::min(best, std::chrono::duration<double>(std::chrono::steady_clock::now() - t).count() * 1e6);
        }
        printf("%d tokens, %d / %d heads after %d: %.1f us\n", s[0], s[1], s[2], s[3], best);
        worst = std::max(worst, best);
    }
    printf("taken %d left %d worst %.1f us\n", taken, left, worst);
    return taken > 500 && left > 500 && worst < 20 ? 0 : 1;
}
"""


def test_split_choice_is_the_first_fit_and_cheap(tmp_path):
    """The bisected plan is the first piece length that fits; the choice against an unsplit launch
    is the cost rule's; and it costs a call a few microseconds at most (trying every piece
    length took 20 to 200)."""
    if not shutil.which("g++"):
        pytest.skip("no host C++ compiler")
    src = tmp_path / "choose.cpp"
    src.write_text(CHOOSE)
    exe = tmp_path / "choose"
    subprocess.run(["g++", "-std=c++17", "-O2", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{CSRC}",
                    str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout


# 16-bit launches timed both ways: (tokens, heads, KV heads, head_dim, tokens before, split).
SHORT = [(16, 14, 2, 64, 250, 0), (40, 14, 2, 64, 400, 0), (88, 14, 2, 64, 504, 0), (40, 32, 8, 64, 250, 0),
         (150, 14, 2, 64, 0, 0), (88, 32, 8, 128, 250, 0), (88, 32, 4, 128, 250, 0), (40, 8, 4, 256, 130, 0),
         (88, 16, 2, 256, 130, 0), (256, 14, 2, 64, 0, 1), (150, 14, 2, 64, 130, 1), (40, 14, 2, 64, 1000, 1),
         (203, 14, 2, 64, 3001, 1), (2, 32, 8, 128, 400, 1), (88, 32, 8, 128, 700, 1), (150, 32, 8, 128, 0, 1),
         (64, 32, 8, 128, 4000, 1), (512, 8, 4, 256, 8000, 1), (40, 8, 4, 256, 400, 1), (4096, 14, 2, 64, 0, 0)]


def test_split_of_16bit_launches_pays_for_its_combine(tmp_path):
    """Short chunks over short caches, whose combine launch costs more than the cut saves (11.3
    us whole, 14.9 cut: 16 tokens after 250, 14 / 2 heads of 64), stay whole; longer ones are cut."""
    if not shutil.which("g++"):
        pytest.skip("no host C++ compiler")
    src = tmp_path / "short.cpp"
    calls = "".join(f"    bad += check({m}, {h}, {g}, {d}, {p0}, {want});\n" for m, h, g, d, p0, want in SHORT)
    src.write_text('#include "prefill_split.hpp"\n#include <cstdio>\n'
                   "static int check(int m, int h, int g, int d, int p0, int want) {\n"
                   "    const bool split = gr::pf_split_16bit_plan(m, h, g, d, p0, 0, 0).n_splits > 0;\n"
                   "    if (split != (want != 0)) printf(\"%d tokens, %d / %d heads of %d after %d: split %d\\n\", m, h, g, d, p0, split);\n"
                   "    return split != (want != 0);\n}\n"
                   "int main() {\n    int bad = 0;\n" + calls + "    return bad;\n}\n")
    exe = tmp_path / "short"
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{CSRC}",
                    str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
