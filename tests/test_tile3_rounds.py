"""CPU check of the fused 3-D step's schedule (csrc/tile3_rounds.hpp): for every
sweep of every tile up to 15 cells a side, each line is taken once, the waves
that add at the same time touch no cell of each other, and no tile whose lines
allow one phase is given two."""
import os
import subprocess
import tempfile

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "amrclaw_amd",
                    "csrc")
PROG = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "tile3_rounds.hpp"
using namespace amrgpu;

static int tr, tq, tp, lpw, n, nlines, rounds;
// the cells (fast, slow) within one line of those of wave w in round r
static std::vector<char> reach(int w, int r) {
    const int m = (tq > tp ? tq : tp) + 2;
    std::vector<char> c((size_t)(n + 2) * (m + 2), 0);
    for (int k = 0; k < lpw; k++) {
        const int line = (w * rounds + r) * lpw + k;
        if (line >= nlines) break;
        const int slow = line / n, fast = line % n;
        for (int a = 0; a < 3; a++)
            for (int b = 0; b < 3; b++) c[(size_t)(slow + a) * (n + 2) + fast + b] = 1;
    }
    return c;
}
static bool meet(const std::vector<char>& a, const std::vector<char>& b) {
    for (size_t k = 0; k < a.size(); k++)
        if (a[k] && b[k]) return true;
    return false;
}

int main() {
    int one = 0, two = 0, pairs = 0;
    for (tr = 1; tr <= 15; tr++)
        for (tq = 1; tq <= 15; tq++)
            for (tp = 1; tp <= 15; tp++) {
                const Tile3Rounds s = tile3_rounds(tr, tq, tp);
                lpw = 64 / (tr + 1);
                n = (tq < tp ? tq : tp) + 2;
                nlines = (tq + 2) * (tp + 2);
                rounds = s.rounds;
                std::vector<int> seen(nlines, 0);
                for (int w = 0; w < s.waves; w++)
                    for (int r = 0; r < rounds; r++)
                        for (int k = 0; k < lpw; k++) {
                            const int line = (w * rounds + r) * lpw + k;
                            if (line < nlines) seen[line]++;
                        }
                for (int v : seen)
                    if (v != 1) return std::printf("line %d %d %d\n", tr, tq, tp), 1;
                bool apart = true;   // of any two waves
                for (int r = 0; r < rounds; r++)
                    for (int v = 0; v < s.waves; v++)
                        for (int w = v + 1; w < s.waves; w++) {
                            const bool m = meet(reach(v, r), reach(w, r));
                            if (m && (s.phases == 1 || (w - v) % 2 == 0))
                                return std::printf("cells %d %d %d\n", tr, tq, tp), 1;
                            apart = apart && !m;
                        }
                // by the distance rule, which the cells may beat by chance
                const bool room = s.waves == 4 && (rounds - 1) * lpw + 1 >= 2 * n + 3;
                if (room != (s.phases == 1)) return std::printf("phases %d %d %d\n", tr, tq, tp), 1;
                if (room && !apart) return std::printf("rule %d %d %d\n", tr, tq, tp), 1;
                (s.waves == 2 ? pairs : s.phases == 1 ? one : two)++;
            }
    std::printf("%d %d %d\n", one, two, pairs);
    return 0;
}
"""


def test_schedule_of_every_tile():
    with tempfile.TemporaryDirectory() as d:
        src, exe = os.path.join(d, "t.cpp"), os.path.join(d, "t")
        open(src, "w").write(PROG)
        subprocess.run(["g++", "-std=c++17", "-O2", "-I" + CSRC, src, "-o", exe], check=True)
        r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    one, two, pairs = (int(v) for v in r.stdout.split())
    assert one + two + pairs == 15 ** 3 and min(one, two, pairs) > 0
