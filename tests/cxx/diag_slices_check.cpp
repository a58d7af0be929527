// Host-side check of build_diag_slices (csrc/tile_plans.cpp), no GPU: for each
// matrix below the planner's answer, its diagonals and its slices' offsets
// equal those found row by row.  Built once plainly and once with the host
// code under AddressSanitizer by tests/test_diag_slices.py.
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <set>
#include <vector>

#include "matrix.hpp"
#include "native.hpp"

using namespace dspmm;

struct Rows {
    std::vector<std::vector<int>> r;
};

static uint64_t g_s = 1;
static int rnd(int n) {
    g_s = g_s * 6364136223846793005ull + 1442695040888963407ull;
    return (int)((g_s >> 33) % (uint64_t)n);
}

static Rows band(int nr, int n, int step) {
    Rows a;
    a.r.resize((size_t)nr);
    for (int i = 0; i < nr; i++)
        for (int k = 0; k < n; k++) a.r[(size_t)i].push_back(i + k * step);
    return a;
}

static Rows stencil(int n) {
    Rows a;
    for (int i = 0; i < n * n * n; i++) {
        a.r.emplace_back();
        for (int x = -1; x <= 1; x++)
            for (int y = -1; y <= 1; y++)
                for (int z = -1; z <= 1; z++) {
                    const int p = i / (n * n) + x, q = i / n % n + y, s = i % n + z;
                    if (p >= 0 && p < n && q >= 0 && q < n && s >= 0 && s < n)
                        a.r.back().push_back((p * n + q) * n + s);
                }
    }
    return a;
}

// Every row on its own choice of `n` of `many` diagonals; `order` shuffles rows.
static Rows picked(int nr, int n, int many, bool order) {
    Rows a = band(nr, 0, 1);
    for (int i = 0; i < nr; i++) {
        std::set<int> d;
        while ((int)d.size() < n) d.insert(rnd(many));
        for (int k : d) a.r[(size_t)i].push_back(i + 7 * k);
        if (order)
            for (int k = n - 1; k > 0; k--) std::swap(a.r[(size_t)i][(size_t)k], a.r[(size_t)i][(size_t)rnd(k + 1)]);
    }
    return a;
}

static bool check(const char *name, const Rows &a, int want) {
    std::vector<int> rp{0}, ci, diags, off;
    std::set<int> all;
    size_t longest = 0;
    int64_t groups = 0;
    std::vector<int> exp_off{0};
    const int nr = (int)a.r.size();
    for (int i = 0; i < nr; i += kDiagRows) {
        size_t most = 0;
        for (int j = i; j < std::min(nr, i + kDiagRows); j++) most = std::max(most, a.r[(size_t)j].size());
        groups += (int64_t)(most + 3) / 4;
        longest = std::max(longest, most);
        exp_off.push_back((int)groups);
    }
    for (int i = 0; i < nr; i++) {
        for (int c : a.r[(size_t)i]) {
            ci.push_back(c);
            all.insert(c - i);
        }
        rp.push_back((int)ci.size());
    }
    const bool expect = !ci.empty() && longest <= (size_t)kDiagRowMax && (int)all.size() <= kDiagMax &&
                        (double)groups * 4 * kDiagRows <= kDiagPad * (double)ci.size() + 4 * kDiagRows;
    const bool got = build_diag_slices(rp, ci, nr, diags, off);
    bool ok = got == expect && (int)expect == want;
    if (got && ok) ok = off == exp_off && diags == std::vector<int>(all.begin(), all.end());
    printf("%s: %s%s\n", name, got ? "fits" : "does not fit", ok ? "" : got == expect ? "  (not what the case is for)" : "  WRONG");
    return ok;
}

int main() {
    int good = 0, n = 0;
    auto t = [&](const char *name, const Rows &a, int want) {
        n++;
        good += check(name, a, want);
    };
    t("no rows", Rows{}, 0);
    t("empty rows", band(200, 0, 1), 0);
    for (int nr : {63, 64, 1000}) t("band", band(nr, 8, 3), 1);
    for (int nr : {1, 65}) t("a band's slice of one row", band(nr, 8, 3), 0);
    t("rows of the most nonzeros", band(300, kDiagRowMax, 2), 1);
    t("one nonzero more", band(300, kDiagRowMax + 1, 2), 0);
    Rows one = band(300, 8, 2);
    for (int k = 8; k <= kDiagRowMax; k++) one.r[299].push_back(299 + 2 * k);
    t("one long row at the end", one, 0);
    t("stencil", stencil(12), 1);
    t("all diagonals used", picked(6000, 20, kDiagMax, false), 1);
    t("in any order", picked(6000, 20, kDiagMax, true), 1);
    t("one diagonal more", picked(6000, 20, kDiagMax + 1, false), 0);
    Rows last = band(5000, 16, 2);             // the distance too many in the last row alone
    for (int k = 0; k < kDiagMax - 16; k++) last.r[(size_t)k] = {k, k + 40 + 2 * k};
    t("the most diagonals, few rows each", last, 1);
    last.r[4999].back() = 4999 + 31;
    t("and one in the last row", last, 0);
    Rows pad = band(640, 0, 1);                // one row of a slice, the others empty
    for (int i = 0; i < 640; i += 64)
        for (int k = 0; k < 30; k++) pad.r[(size_t)i].push_back(i + k);
    t("mostly padding", pad, 0);
    Rows twice = band(500, 8, 1);
    for (auto &r : twice.r) r[3] = r[2];
    t("a column twice", twice, 1);
    Rows far = band(130, 2, 1);
    for (auto &r : far.r) r = {0, INT_MAX - 1};
    t("distances over the whole range", far, 0);
    Rows near = band(100, 2, 1);
    for (auto &r : near.r) r = {0, INT_MAX - 1, 5, 6};
    t("columns that all rows have", near, 1);
    printf("%d of %d checks ok\n", good, n);
    return good == n ? 0 : 1;
}
