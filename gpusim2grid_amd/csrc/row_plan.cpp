#include "row_plan.hpp"

#include <algorithm>
#include <numeric>

namespace g2g {

RowPlan build_row_plan(const NrPlan& P)
{
    RowPlan R;
    const int n = P.n;
    R.n = n;
    // the buses with unknowns in the plan's elimination order (a bus's
    // unknowns are eliminated together)
    std::vector<int> bus_of_unknown(static_cast<size_t>(P.d), -1);
    for (int i = 0; i < n; ++i) {
        if (P.col_th[i] >= 0) bus_of_unknown[P.col_th[i]] = i;
        if (P.row_q[i] >= 0) bus_of_unknown[P.row_q[i]] = i;
    }
    std::vector<int> order, pos(static_cast<size_t>(n), -1);
    for (int k = 0; k < P.d; ++k) {
        const int b = bus_of_unknown[P.lu.perm[k]];
        if (b < 0) return R;
        if (pos[b] < 0) {
            pos[b] = static_cast<int>(order.size());
            order.push_back(b);
        }
    }
    const int nb = static_cast<int>(order.size());
    // symbolic elimination of the bus graph: children before parents.  A bus's
    // column: its later neighbours and its children's columns, sorted.
    std::vector<std::vector<int>> st(static_cast<size_t>(nb));
    std::vector<int> lev(static_cast<size_t>(nb), 0), mark(static_cast<size_t>(nb), -1), head(static_cast<size_t>(nb), -1),
        next(static_cast<size_t>(nb), -1);
    // (Ybus may hold an entry without its transpose: both ends see it)
    std::vector<int> tp(static_cast<size_t>(nb) + 1, 0), ti;
    for (int pass = 0; pass < 2; ++pass) {
        if (pass) {
            for (int k = 0; k < nb; ++k) tp[k + 1] += tp[k];
            ti.resize(static_cast<size_t>(tp[nb]));
        }
        for (int i = 0; i < n; ++i) {
            if (pos[i] < 0) continue;
            for (int q = P.Yp[i]; q < P.Yp[i + 1]; ++q) {
                const int x = pos[i], y = pos[P.Yi[q]];
                if (y < 0 || x == y) continue;
                if (pass) ti[tp[std::min(x, y)]++] = std::max(x, y);
                else ++tp[std::min(x, y) + 1];
            }
        }
    }
    for (int k = 0; k < nb; ++k) {
        auto& s = st[k];
        mark[k] = k;
        auto add = [&](int j) {
            if (mark[j] != k) {
                mark[j] = k;
                s.push_back(j);
            }
        };
        for (int q = k ? tp[k - 1] : 0; q < tp[k]; ++q) add(ti[q]);
        for (int c = head[k]; c >= 0; c = next[c])
            for (int j : st[c])
                if (j != k) add(j);
        std::sort(s.begin(), s.end());
        if (s.empty()) continue;
        const int p = s.front();
        next[k] = head[p];
        head[p] = k;
        lev[p] = std::max(lev[p], lev[k] + 1);
    }
    // renumber by level: a bus's neighbours in its column are its ancestors,
    // which lie on higher levels
    std::vector<int> by(static_cast<size_t>(nb));
    std::iota(by.begin(), by.end(), 0);
    std::stable_sort(by.begin(), by.end(), [&](int a, int b) { return lev[a] < lev[b]; });
    std::vector<int> num(static_cast<size_t>(nb));
    for (int k = 0; k < nb; ++k) num[by[k]] = k;
    R.nb = nb;
    R.bus_of.resize(static_cast<size_t>(n));
    std::vector<int> num_of_bus(static_cast<size_t>(n), -1);
    for (int k = 0; k < nb; ++k) {
        R.bus_of[k] = order[by[k]];
        num_of_bus[R.bus_of[k]] = k;
    }
    for (int i = 0, at = nb; i < n; ++i)
        if (num_of_bus[i] < 0) {
            R.bus_of[at] = i;
            num_of_bus[i] = at++;
        }
    std::vector<std::vector<int>> col(static_cast<size_t>(nb));
    std::vector<int> level(static_cast<size_t>(nb)), diag(static_cast<size_t>(nb)), bus_of_diag;
    R.n_lev = 0;
    for (int k = 0; k < nb; ++k) {
        auto& c = col[k];
        c = std::move(st[by[k]]);
        for (int& j : c) j = num[j];
        std::sort(c.begin(), c.end());
        if (static_cast<int>(c.size()) > kRowMaxC) return R;
        level[k] = lev[by[k]];
        R.n_lev = std::max(R.n_lev, level[k] + 1);
        diag[k] = R.n_blk;
        R.n_blk += 1 + 2 * static_cast<int>(c.size());
        bus_of_diag.resize(static_cast<size_t>(R.n_blk), -1);
        bus_of_diag[diag[k]] = k;
    }
    if (nb == 0 || nb >= (1 << 23) || R.n_blk >= (1 << 28) || R.n_lev > kRowMaxLev) return R;
    // block (i, j): its diagonal, or in the record of the one eliminated first
    auto block = [&](int i, int j) {
        if (i == j) return diag[i];
        const int k = std::min(i, j), o = std::max(i, j);
        const auto& c = col[k];
        const auto it = std::lower_bound(c.begin(), c.end(), o);
        if (it == c.end() || *it != o) return -1;
        const int a = static_cast<int>(it - c.begin());
        return diag[k] + (i > j ? 1 : 2) + 2 * a;  // L(i, k), U(k, j)
    };
    R.lev_ptr.assign(static_cast<size_t>(R.n_lev) + 1, 0);
    for (int k = 0; k < nb; ++k) ++R.lev_ptr[level[k] + 1];
    for (int l = 0; l < R.n_lev; ++l) R.lev_ptr[l + 1] += R.lev_ptr[l];
    for (int l = 0; l < R.n_lev; ++l) R.lev_blk.push_back(diag[R.lev_ptr[l]]);
    R.lev_blk.push_back(R.n_blk);
    // records: a level's terms gathered by target, in pivot order
    struct Term { int d, w, run; };
    struct Run { int tgt, cnt, at; };
    std::vector<Term> t;
    std::vector<Run> runs;
    std::vector<int> run_of(static_cast<size_t>(R.n_blk) + nb, -1), run_lev(static_cast<size_t>(R.n_blk) + nb, -1), ord_run,
        place;
    R.rec.reserve(16 * static_cast<size_t>(nb));
    R.rec2.reserve(8 * static_cast<size_t>(nb));
    R.rec_ptr.push_back(0);
    for (int l = 0; l < R.n_lev; ++l) {
        t.clear();
        runs.clear();
        auto put = [&](int tgt, int id, int d, int w) {
            if (run_lev[id] != l) {
                run_lev[id] = l;
                run_of[id] = static_cast<int>(runs.size());
                runs.push_back({tgt, 0, 0});
            }
            ++runs[run_of[id]].cnt;
            t.push_back({d, w, run_of[id]});
        };
        for (int k = R.lev_ptr[l]; k < R.lev_ptr[l + 1]; ++k) {
            const auto& c = col[k];
            for (size_t a = 0; a < c.size(); ++a) {
                const int dl = 1 + 2 * static_cast<int>(a);
                for (size_t b = 0; b < c.size(); ++b) {
                    const int tgt = block(c[a], c[b]);
                    if (tgt < 0) return R;
                    put(tgt, tgt, diag[k], dl | ((2 + 2 * static_cast<int>(b)) << 8));
                }
                put(kRowRhs | c[a], R.n_blk + c[a], diag[k], dl | (k << 8));
            }
        }
        // blocks before right-hand sides, long records first: a wavefront's
        // lanes run about as many terms
        ord_run.resize(runs.size());
        std::iota(ord_run.begin(), ord_run.end(), 0);
        std::stable_sort(ord_run.begin(), ord_run.end(), [&](int x, int y) {
            const bool rx = runs[x].tgt & kRowRhs, ry = runs[y].tgt & kRowRhs;
            if (rx != ry) return ry;
            return runs[x].cnt > runs[y].cnt;
        });
        place.resize(t.size());
        int at = 0;
        for (int r : ord_run) {
            runs[r].at = at;
            at += runs[r].cnt;
        }
        {
            std::vector<int> fill_at(runs.size(), 0);
            for (size_t q = 0; q < t.size(); ++q) place[runs[t[q].run].at + fill_at[t[q].run]++] = static_cast<int>(q);
        }
        int n_invert = 0;
        for (int r : ord_run) {
            int tgt = runs[r].tgt;
            const int cnt = runs[r].cnt, *q = place.data() + runs[r].at;
            if (cnt > kRowMaxTerms) return R;
            // the diagonal block of a bus of the next level
            if (!(tgt & kRowRhs) && bus_of_diag[tgt] >= 0 && level[bus_of_diag[tgt]] == l + 1) {
                ++n_invert;
                tgt |= kRowInvert;
            }
            const int first = static_cast<int>(R.term.size() / 2);
            if (first >= (1 << 24)) return R;
            const Term &t1 = t[q[0]], &t2 = t[q[cnt > 1 ? 1 : 0]];
            R.rec.insert(R.rec.end(), {tgt, first | (cnt << 24), t1.d, t1.w});
            R.rec2.insert(R.rec2.end(), {t2.d, t2.w});
            for (int e = 2; e < cnt; ++e) R.term.insert(R.term.end(), {t[q[e]].d, t[q[e]].w});
        }
        R.rec_ptr.push_back(static_cast<int>(R.rec.size() / 4));
        // every bus above level 0 has a child on the level below it
        if (l + 1 < R.n_lev && n_invert != R.lev_ptr[l + 2] - R.lev_ptr[l + 1]) return R;
    }
    for (int k = 0; k < nb; ++k) {
        const int first = static_cast<int>(R.back_col.size());
        if (first >= (1 << 24)) return R;
        const auto& c = col[k];
        R.back.insert(R.back.end(), {diag[k], first | (static_cast<int>(c.size()) << 24), c.size() > 0 ? c[0] : k,
                                     c.size() > 1 ? c[1] : k});
        if (c.size() > 2) R.back_col.insert(R.back_col.end(), c.begin() + 2, c.end());
    }
    R.solo_f = R.solo_b = R.n_lev;
    while (R.solo_f > 0 && R.rec_ptr[R.solo_f] - R.rec_ptr[R.solo_f - 1] <= kLanes) --R.solo_f;
    while (R.solo_b > 0 && R.lev_ptr[R.solo_b] - R.lev_ptr[R.solo_b - 1] <= kLanes) --R.solo_b;
    // mismatch slices
    std::vector<char> present(static_cast<size_t>(R.n_blk), 0);
    auto pq = [&](int b) { return P.row_q[b] >= 0; };
    std::vector<int> deg(static_cast<size_t>(nb)), ord(static_cast<size_t>(nb));
    for (int k = 0; k < nb; ++k) {
        const int b = R.bus_of[k];
        deg[k] = 0;
        for (int q = P.Yp[b]; q < P.Yp[b + 1]; ++q) deg[k] += P.Yi[q] != b;
        present[diag[k]] = 1;
    }
    std::iota(ord.begin(), ord.end(), 0);
    std::stable_sort(ord.begin(), ord.end(), [&](int a, int b) { return deg[a] > deg[b]; });
    R.n_slice = (nb + kLanes - 1) / kLanes;
    R.slice_ptr.push_back(0);
    R.slice_bus.reserve(4 * static_cast<size_t>(R.n_slice) * kLanes);
    R.diag_y.reserve(2 * static_cast<size_t>(R.n_slice) * kLanes);
    R.ent.reserve(4 * (static_cast<size_t>(P.nY) + kLanes * static_cast<size_t>(kLanes)));
    R.ent_y.reserve(2 * (static_cast<size_t>(P.nY) + kLanes * static_cast<size_t>(kLanes)));
    for (int s = 0; s < R.n_slice; ++s) {
        const int width = deg[ord[s * kLanes]];
        const size_t e0 = R.ent.size() / 4;
        R.ent.resize((e0 + static_cast<size_t>(width) * kLanes) * 4);
        R.ent_y.resize((e0 + static_cast<size_t>(width) * kLanes) * 2, 0.0);
        for (int ln = 0; ln < kLanes; ++ln) {
            const int at = s * kLanes + ln;
            int q_used = 0;
            if (at < nb) {
                const int k = ord[at], b = R.bus_of[k];
                int yd = -1;
                for (int q = P.Yp[b]; q < P.Yp[b + 1]; ++q) {
                    const int j = P.Yi[q];
                    if (j == b) {
                        yd = q;
                        continue;
                    }
                    const int kj = num_of_bus[j];
                    int code = -1;
                    if (kj < nb) {
                        const int bl = block(k, kj);
                        if (bl < 0) return R;
                        present[bl] = 1;
                        code = bl << 2 | (pq(j) ? 2 : 0) | (pq(b) ? 1 : 0);
                    }
                    const size_t e = e0 + static_cast<size_t>(q_used) * kLanes + ln;
                    const int w[4] = {kj, code, q, 0};
                    std::copy(w, w + 4, R.ent.begin() + 4 * e);
                    R.ent_y[2 * e] = P.Yx[2 * q];
                    R.ent_y[2 * e + 1] = P.Yx[2 * q + 1];
                    ++q_used;
                }
                if (yd < 0) return R;
                R.slice_bus.insert(R.slice_bus.end(), {k, static_cast<int>(static_cast<unsigned>(diag[k]) |
                                                                          (pq(b) ? 0x80000000u : 0u)), yd, b});
                R.diag_y.insert(R.diag_y.end(), {P.Yx[2 * yd], P.Yx[2 * yd + 1]});
            } else {
                R.slice_bus.insert(R.slice_bus.end(), {-1, 0, -1, 0});
                R.diag_y.insert(R.diag_y.end(), {0.0, 0.0});
            }
            for (int q = q_used; q < width; ++q) {  // padding: adds 0 x V of bus 0, no block
                const size_t e = e0 + static_cast<size_t>(q) * kLanes + ln;
                const int w[4] = {0, -1, -1, 0};
                std::copy(w, w + 4, R.ent.begin() + 4 * e);
            }
        }
        R.slice_ptr.push_back(static_cast<int>((R.ent.size() / 4) / kLanes));
    }
    for (int q = 0; q < R.n_blk; ++q)
        if (!present[q]) R.fill.push_back(q);
    R.n_fill = static_cast<int>(R.fill.size());
    R.ok = true;
    return R;
}

}  // namespace g2g
