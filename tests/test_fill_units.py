"""CPU check of the fill programs' units (csrc/fill_plan.cpp): what one launch
runs side by side.  On random hierarchies, no two operations of different stages
that lie in different units touch a cell of each other, every operation is in one
unit, and a unit's operations stand by stage."""
import os
import subprocess
import tempfile

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "amrclaw_amd",
                    "csrc")
PROG = r"""
#include <algorithm>
#include <cstdio>
#include <random>
#include <set>
#include "fill_plan.hpp"
using namespace amrgpu;

// cells as (buffer, cell) numbers
using Cells = std::vector<int64_t>;
struct Touch { Cells w, r; };

static void rect(Cells& c, const FillPlan& P, int b, int i0, int j0, int ni, int nj) {
    for (int j = j0; j < j0 + nj; j++)
        for (int i = i0; i < i0 + ni; i++) c.push_back(((int64_t)b << 32) + (int64_t)j * P.bufs[b].nrow + i);
}

static Touch touch(const FillPlan& P, const HierGeom& H, const FillOp& op) {
    Touch t;
    const FillBuf& d = P.bufs[op.dst];
    if (op.type == FOP_COPY) {
        rect(t.w, P, op.dst, op.di0, op.dj0, op.ni, op.nj);
        for (int b = 0; b < (int)P.bufs.size(); b++)
            if (P.bufs[b].kind == 0 && P.bufs[b].level == op.src_level && P.bufs[b].patch == op.src)
                rect(t.r, P, b, op.si0, op.sj0, op.ni, op.nj);
    } else if (op.type == FOP_INTERP || op.type == FOP_FILVAL) {
        const bool fv = op.type == FOP_FILVAL;
        const int ni = fv ? (op.ni - 2) * op.ratx : op.ni, nj = fv ? (op.nj - 2) * op.raty : op.nj;
        for (int j = 0; j < nj; j++)
            for (int i = 0; i < ni; i++)
                if (!P.masks[op.mask_off + (size_t)j * ni + i])
                    rect(t.w, P, op.dst, (fv ? NGHOST : op.di0) + i, (fv ? NGHOST : op.dj0) + j, 1, 1);
        rect(t.r, P, op.src, 0, 0, P.bufs[op.src].nrow, P.bufs[op.src].ncol);
    } else if (op.type == FOP_COPYBACK) {
        rect(t.w, P, op.dst, op.di0, op.dj0, op.ni, op.nj);
        rect(t.r, P, op.src, 0, 0, op.ni, op.nj);
    } else if (op.type == FOP_COARSEN) {
        rect(t.w, P, op.dst, 0, 0, op.ni, op.nj);
        rect(t.r, P, op.src, 0, 0, 2 * op.ni, 2 * op.nj);
    } else if (op.type == FOP_RING) {
        rect(t.r, P, op.src, 0, 0, op.ni, op.nj);
    } else {   // boundary conditions, side by side as fill.hip runs them
        const int n = d.nrow, m = d.ncol;
        auto x = [&](int i, int from) { rect(t.w, P, op.dst, i, 0, 1, m); rect(t.r, P, op.dst, from, 0, 1, m); };
        auto y = [&](int j, int from) { rect(t.w, P, op.dst, 0, j, n, 1); rect(t.r, P, op.dst, 0, from, n, 1); };
        const int *b = op.bc, *mb = H.mthbc;
        for (int i = 0; i < b[0]; i++) x(i, mb[0] == 3 ? 2 * b[0] - 1 - i : b[0]);
        for (int i = b[1] - 1; b[1] > 0 && i < n; i++) x(i, mb[1] == 3 ? 2 * b[1] - 3 - i : b[1] - 2);
        for (int j = 0; j < b[2]; j++) y(j, mb[2] == 3 ? 2 * b[2] - 1 - j : b[2]);
        for (int j = b[3] - 1; b[3] > 0 && j < m; j++) y(j, mb[3] == 3 ? 2 * b[3] - 3 - j : b[3] - 2);
    }
    std::sort(t.w.begin(), t.w.end());
    std::sort(t.r.begin(), t.r.end());
    return t;
}

static bool meet(const Cells& a, const Cells& b) {
    for (size_t i = 0, j = 0; i < a.size() && j < b.size();)
        if (a[i] == b[j]) return true;
        else if (a[i] < b[j]) i++;
        else j++;
    return false;
}

static int side_by_side = 0;
static bool check(const FillPlan& P, const HierGeom& H, const char* what) {
    const int n = (int)P.ops.size();
    std::vector<int> unit(n, -1);
    int at = 0;
    for (int u = 0; u < (int)P.units.size(); u++) {
        if (P.units[u].item0 != at || P.units[u].n < 1) return std::printf("%s: units\n", what), false;
        for (int k = 0; k < P.units[u].n; k++, at++) {
            const int o = P.order[at];
            // what an operation other than a copy reads is FP64 scratch or arena
            if (P.ops[o].type != FOP_COPY && P.ops[o].type != FOP_BC && P.bufs[P.ops[o].src].kind == 0)
                return std::printf("%s: operation %d (type %d) reads a level\n", what, o, P.ops[o].type), false;
            if (unit[o] >= 0) return std::printf("%s: twice\n", what), false;
            unit[o] = u;
            if (k > 0 && P.ops[P.order[at - 1]].stage > P.ops[o].stage)
                return std::printf("%s: stages\n", what), false;
        }
    }
    if (at != n) return std::printf("%s: missing\n", what), false;
    std::vector<Touch> t;
    for (const FillOp& op : P.ops) t.push_back(touch(P, H, op));
    for (int a = 0; a < n; a++)
        for (int b = 0; b < n; b++) {
            if (P.ops[a].stage >= P.ops[b].stage || unit[a] == unit[b]) continue;
            if (meet(t[a].w, t[b].w) || meet(t[a].w, t[b].r) || meet(t[a].r, t[b].w))
                return std::printf("%s: operations %d (type %d) and %d (type %d)\n", what, a, P.ops[a].type, b,
                                   P.ops[b].type), false;
            side_by_side++;
        }
    return true;
}

static void geom(HierGeom& H, int N) {
    H.nlev = 2;
    for (int l : {1, 2, (int)FILL_OLDSLOT}) {
        auto& L = H.lev[l];
        L.iregsz = L.jregsz = l == 1 ? N : 2 * N;
        L.ratx = L.raty = 2;
        L.hx = L.hy = (l == 1 ? 1.0 : 0.5) / N;
    }
}

int main() {
    std::mt19937 r(5);
    std::string e;
    FillPlan P;
    int plans = 0;
    for (int t = 0; t < 80; t++) {
        const int N = 24;
        HierGeom H;
        geom(H, N);
        const int s1 = std::vector<int>{6, 8, 12, 24, 3}[r() % 5];
        for (int j = 0; j < N; j += s1)
            for (int i = 0; i < N; i += s1) H.lev[1].boxes.push_back({i, i + s1 - 1, j, j + s1 - 1});
        auto fine = [&](int w, int d) {
            std::vector<std::array<int, 4>> v;
            for (int j = d; j + w <= 2 * N; j += w)
                for (int i = d; i + w <= 2 * N; i += w)
                    if (r() % 4) v.push_back({i, i + w - 1, j, j + w - 1});
            return v;
        };
        H.lev[2].boxes = fine(4 + 2 * (r() % 6), 2 * (r() % 3));
        H.lev[FILL_OLDSLOT].boxes = fine(4 + 2 * (r() % 6), 2 * (r() % 3));
        H.xperdom = r() % 2;
        H.yperdom = r() % 2;
        for (int k = 0; k < 4; k++) H.mthbc[k] = (k < 2 ? H.xperdom : H.yperdom) ? 2 : (r() % 2 ? 1 : 3);
        RichPlan R;
        for (int l : {1, 2})
            if (plan_fill_level(H, l, 2, P, e) && ++plans && !check(P, H, "fill")) return 1;
        if (plan_filval(H, 2, 2, P, e) && ++plans && !check(P, H, "filval")) return 1;
        if (plan_saveqc(H, 2, 2, P, e) && ++plans && !check(P, H, "saveqc")) return 1;
        if (plan_richardson(H, 1, 2, R, e) && ++plans && !check(R.fill, H, "richardson")) return 1;
    }
    // four grids with two outer sides each: the boundary conditions wait for
    // the copies along those sides, not for the one into the inner corner
    HierGeom H;
    geom(H, 32);
    for (int j = 0; j < 32; j += 16)
        for (int i = 0; i < 32; i += 16) H.lev[1].boxes.push_back({i, i + 15, j, j + 15});
    for (int k = 0; k < 4; k++) H.mthbc[k] = k % 2 ? 1 : 3;
    if (!plan_fill_level(H, 1, 2, P, e) || !check(P, H, "corners")) return 1;
    std::printf("%d %d %zu %zu\n", plans, side_by_side, P.ops.size(), P.units.size());
    return 0;
}
"""


def test_units_are_independent():
    with tempfile.TemporaryDirectory() as d:
        src, exe = os.path.join(d, "t.cpp"), os.path.join(d, "t")
        open(src, "w").write(PROG)
        subprocess.run(["g++", "-std=c++17", "-O2", "-I" + CSRC, src,
                        os.path.join(CSRC, "fill_plan.cpp"), "-o", exe], check=True)
        r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    plans, pairs, ops, units = (int(v) for v in r.stdout.split())
    assert plans > 200 and pairs > 10000
    assert (ops, units) == (16, 8)
