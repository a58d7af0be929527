// selector.cpp -- the learned default configuration of dspmm_spmm_ex.
//
// A nearest-neighbour rule over a corpus measured on MI355X (the table in
// selector_table.inc is generated by selector.py from the autotuner's full
// timing tables): the query matrix's features -- log2 rows, log2 mean row
// length, coefficient of variation of the row length, log2(max / mean row
// length) and the column reuse of 16-row windows -- are compared, in
// standardised units, with the corpus entries at the nearest measured dense
// width; the kSelK nearest vote with their per-configuration
// log(time / best time), and the configuration with the smallest total
// wins.  Used for row-major FP32 operands when no tuned configuration is
// cached; everything else keeps the static heuristic.
#include <algorithm>
#include <cmath>
#include <map>
#include <tuple>
#include <vector>

#include "matrix.hpp"

namespace dspmm {
namespace {
#include "selector_table.inc"
}  // namespace

bool learned_select(dspmm_matrix_s *A, int nv, dspmm_config *out) {
    if (kSelEntries == 0 || A->nr == 0 || A->nnz == 0 || nv < 1) return false;
    const double mean = std::max(A->mean, 1e-3);
    const double q[5] = {std::log2((double)std::max(1, A->nr)), std::log2(mean), A->cv,
                         std::log2(std::max((double)A->max_len, 1.0) / mean), column_reuse(A)};
    // nearest measured dense width (in log2)
    int best_nv = -1;
    double best_gap = 1e30;
    for (int i = 0; i < kSelEntries; i++) {
        const double gap = std::fabs(std::log2((double)kSelTable[i].nv) - std::log2((double)nv));
        if (gap < best_gap) {
            best_gap = gap;
            best_nv = kSelTable[i].nv;
        }
    }
    std::vector<std::pair<double, int>> dist;
    for (int i = 0; i < kSelEntries; i++) {
        if (kSelTable[i].nv != best_nv) continue;
        double d = 0;
        for (int k = 0; k < 5; k++) {
            const double z = (q[k] - kSelTable[i].f[k]) / kSelScale[k];
            d += z * z;
        }
        dist.emplace_back(d, i);
    }
    if (dist.empty()) return false;
    std::sort(dist.begin(), dist.end());
    const int k = std::min<int>(kSelK, (int)dist.size());
    using Key = std::tuple<int, int, int, int, int, int>;
    std::map<Key, double> score;
    for (int j = 0; j < k; j++)
        for (int c = 0; c < kSelTop; c++) {
            const SelEntry &e = kSelTable[dist[(size_t)j].second];
            if (e.logratio[c] >= 99.f) continue;
            score[Key(e.cfg[c][0], e.cfg[c][1], e.cfg[c][2], e.cfg[c][3], e.cfg[c][4], e.cfg[c][5])] = 0;
        }
    for (auto &kv : score)
        for (int j = 0; j < k; j++) {
            const SelEntry &e = kSelTable[dist[(size_t)j].second];
            double lr = 2.0;                 // missing from a top list: counts as e^2 slower
            for (int c = 0; c < kSelTop; c++)
                if (e.logratio[c] < 99.f &&
                    Key(e.cfg[c][0], e.cfg[c][1], e.cfg[c][2], e.cfg[c][3], e.cfg[c][4], e.cfg[c][5]) == kv.first)
                    lr = e.logratio[c];
            kv.second += lr;
        }
    if (score.empty()) return false;
    const auto win = std::min_element(score.begin(), score.end(),
                                      [](const auto &a, const auto &b) { return a.second < b.second; });
    dspmm_config c{};
    std::tie(c.variant, c.vec, c.lanes, c.tile_nnz, c.unroll, c.row_stride) = win->first;
    if ((c.variant == DSPMM_VARIANT_SPMV_TILED) != (nv == 1)) return false;
    // lanes that covered the measured width in one slab cover this one too
    if (c.lanes > 0 && c.vec > 0 && c.lanes * c.vec >= best_nv) c.lanes = 0;
    *out = c;
    return true;
}

}  // namespace dspmm
