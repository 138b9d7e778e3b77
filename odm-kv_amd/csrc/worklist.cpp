// The decode work list, cut on the host: every (segment, level) run of tiles into items of about equal cost
// (include/odmkv.h: odmkv_worklist_cut).  Host arithmetic only.
//
// The list is cut again for every store a prompt fills and after every flush and rewind, between kernels that wait for
// it; in Python (numpy and heapq) a 32k-token layer took 0.5 to 1 ms, here 5 to 15 us.
#include "common.h"

#include <math.h>
#include <string.h>
#include <algorithm>
#include <exception>
#include <functional>
#include <queue>
#include <vector>

namespace {

// what one compute unit was measured to need per 64-token tile of each level (nanoseconds; 2, 3, 4, 8 bits, exact rows)
// and per work item (microseconds: start, table, query rotation, combining the wavefronts)
const int64_t kTileCost[5] = {300, 420, 450, 890, 1310};
const int64_t kTileBytes[5] = {TILE * 16 * 2 + 2 * TILE * 4, TILE * 16 * 3 + 2 * TILE * 4, TILE * 16 * 4 + 2 * TILE * 4,
                               TILE * 16 * 8 + 2 * TILE * 4, 2 * TILE * HD * 2};
const double kItemFixedUs = 4.0;        // what the cuts without chains are compared with (its choices were measured shape by shape)
// Chains (a workgroup that walks several quantised levels of a pair) by a rule, not by the cost model, which is off by a
// third either way on lists of several rounds: they are taken when the quantised runs number at least 1.5 per compute unit
// and 2.5 per pair, cut so that the workgroups number 1.5 per compute unit or, with more pairs than that, one per pair
// beside the exact items.  Measured whole calls: 64 sequences x 2048 tokens x 8 kv-heads, four levels each: 90 -> 67 us;
// 16 x 8192 tokens with four levels: 44 -> 36 us; 16 x 8192 tokens with two levels: no gain at any cut, not taken by the
// rule.  The link and rotation costs below only rank the workgroups for the dispatch order.
const double kChainLinkUs = 1.8;
const double kChainRotateUs = 1.0;
const double kChainRunsPerCu = 1.5;
const double kChainRunsPerPair = 2.5;
const double kPairChainRunsPerPlace = 1.5;   // two workgroups per compute unit: chains where the runs number this many per place

struct Item { int64_t s, li, t0, nt, cnt, seg0; int follow, cont; };
struct Run { int64_t s, li, nt, t0, cnt; };

struct Cutter {
    int nseg, n_cu;
    std::vector<Run> runs;              // segment by segment, levels ascending
    std::vector<int> q;                 // the quantised ones
    std::vector<double> q_end, q_start, seg_cost, seg_start;
    std::vector<char> q_first;          // a segment's first quantised run
    int64_t total, total_bytes, min_cost;

    static int64_t step_of(int64_t per_item, int li) {
        const double r = rint((double)per_item / (double)kTileCost[li]);
        return r > 1.0 ? (r < 1073741824.0 ? (int64_t)r : 1073741824) : 1;      // (no run has 2^30 tiles)
    }
    int64_t n_pieces(int64_t per_item) const {
        int64_t step[5], n = 0;
        for (int li = 0; li < 5; ++li) step[li] = step_of(per_item, li);
        for (const Run& r : runs) n += (uint32_t)(r.nt + step[r.li] - 1) / (uint32_t)step[r.li];
        return n;
    }
    // the coarsest cut with at most `target` items (a run's last piece may be short): the first of a ladder of costs, each
    // a 64th above the last, whose pieces do not exceed it.  Pieces fall along the ladder, so the rung is found by bisection.
    template <class Count> int64_t first_rung(int64_t target, Count count) const {
        std::vector<int64_t> rung(1, std::max(total / std::max<int64_t>(target, 1), min_cost));
        while (rung.back() < total) rung.push_back(rung.back() + std::max<int64_t>(rung.back() / 64, 1));
        size_t lo = 0, hi = 1;                     // (usually a few rungs up: doubling steps, then halving ones)
        while (hi < rung.size() - 1 && count(rung[hi]) > target) { lo = hi; hi = std::min(2 * hi + 1, rung.size() - 1); }
        if (count(rung[lo]) <= target) return rung[lo];
        while (hi > lo + 1) {
            const size_t mid = (lo + hi) / 2;
            if (count(rung[mid]) > target) lo = mid;
            else hi = mid;
        }
        return rung[std::min(hi, rung.size() - 1)];
    }
    int64_t fit(int64_t target) const {
        return first_rung(target, [this](int64_t per) { return n_pieces(per); });
    }
    static void pieces_of(const Run& r, int64_t step, std::vector<Item>& out) {
        for (int64_t a = 0; a < r.nt; a += step) {
            const int64_t n = std::min(step, r.nt - a);
            out.push_back({r.s, r.li, r.t0 + a, n, std::min(r.cnt - a * TILE, n * TILE), r.t0, 0, 0});
        }
    }
    std::vector<Item> cut(int64_t per_item) const {
        std::vector<Item> out;
        out.reserve(n_pieces(per_item));
        for (const Run& r : runs) pieces_of(r, step_of(per_item, (int)r.li), out);
        return out;
    }
    // -- chains: the quantised levels of a segment as ONE run of work, cut into pieces of equal cost; a piece that crosses a
    // level boundary becomes consecutive items of one workgroup (one query rotation, one result)
    int64_t chain_pieces(int s, int64_t per_item) const { return (int64_t)ceil(seg_cost[s] / (double)std::max<int64_t>(per_item, 1)); }
    int64_t n_chained(int64_t per_item) const {
        int64_t n = 0;
        for (int s = 0; s < nseg; ++s) n += chain_pieces(s, per_item);
        const int64_t step = step_of(per_item, 4);
        for (const Run& r : runs)
            if (r.li == 4) n += (uint32_t)(r.nt + step - 1) / (uint32_t)step;
        return n;
    }
    int64_t fit_chained(int64_t target) const {
        return first_rung(target, [this](int64_t per) { return n_chained(per); });
    }
    std::vector<Item> cut_chained(int64_t per_item) const {
        struct Start { int run; int64_t off; bool head; };
        std::vector<Start> st;
        const int nq = (int)q.size();
        for (int i = 0; i < nq; ++i) st.push_back({i, 0, q_first[i] != 0});      // every run's first tile,
        for (int s = 0; s < nseg; ++s) {                                         // and the boundaries inside runs
            const int64_t k = chain_pieces(s, per_item);
            for (int64_t j = 1; j < k; ++j) {
                const double x = seg_start[s] + (double)j * seg_cost[s] / (double)k;   // on the line of all runs' cost
                int r = (int)(std::upper_bound(q_end.begin(), q_end.end(), x) - q_end.begin());
                r = std::min(r, nq - 1);
                const Run& run = runs[q[r]];
                int64_t off = (int64_t)rint((x - q_start[r]) / (double)kTileCost[run.li]);
                off = std::min(std::max<int64_t>(off, 0), run.nt);
                if (off == run.nt) { r = std::min(r + 1, nq - 1); off = 0; }     // a boundary on a run's end belongs to the next run
                st.push_back({r, off, true});
            }
        }
        // duplicates: the one that starts a chain first
        std::stable_sort(st.begin(), st.end(), [](const Start& a, const Start& b) {
            if (a.run != b.run) return a.run < b.run;
            if (a.off != b.off) return a.off < b.off;
            return a.head && !b.head;
        });
        st.erase(std::unique(st.begin(), st.end(), [](const Start& a, const Start& b) { return a.run == b.run && a.off == b.off; }), st.end());
        std::vector<Item> out;
        int head = -1;
        for (size_t i = 0; i < st.size(); ++i) {
            const Run& r = runs[q[st[i].run]];
            const bool last = i + 1 == st.size() || st[i + 1].run != st[i].run;
            const int64_t n = (last ? r.nt : st[i + 1].off) - st[i].off;
            if (st[i].head) head = (int)i;
            else if (head >= 0) out[head].follow += 1;
            out.push_back({r.s, r.li, r.t0 + st[i].off, n, std::min(r.cnt - st[i].off * TILE, n * TILE), r.t0, 0, st[i].head ? 0 : 1});
        }
        const int64_t step = step_of(per_item, 4);
        for (const Run& r : runs)
            if (r.li == 4) pieces_of(r, step, out);
        std::stable_sort(out.begin(), out.end(), [](const Item& a, const Item& b) {
            if (a.s != b.s) return a.s < b.s;
            if (a.li != b.li) return a.li < b.li;
            return a.t0 < b.t0;
        });
        return out;
    }
    // microseconds of one workgroup, roughly: per workgroup (a continued item adds to the one before it)
    static std::vector<double> cost(const std::vector<Item>& items) {
        std::vector<double> own, extra;
        for (const Item& it : items) {
            const double c = (double)it.nt * (double)kTileCost[it.li] * 1e-3;
            if (!it.cont) { own.push_back(0.0); extra.push_back((double)it.follow); }
            if (!own.empty()) own.back() += c;
        }
        for (size_t i = 0; i < own.size(); ++i)
            own[i] = kItemFixedUs + own[i] + kChainLinkUs * extra[i] + (extra[i] > 0 ? kChainRotateUs : 0.0);
        return own;
    }
    // the time a longest-first assignment to the compute units would take; infinity where the sum alone says that it takes
    // longer than `bound`
    double makespan(const std::vector<Item>& items, double bound) const {
        std::vector<double> c = cost(items);
        if (c.empty()) return 0.0;
        double sum = 0.0;
        for (double v : c) sum += v;
        if (sum > (bound + 1e-6) * n_cu) return INFINITY;
        std::sort(c.begin(), c.end(), std::greater<double>());
        if ((int)c.size() <= n_cu) return c[0];
        std::priority_queue<double, std::vector<double>, std::greater<double>> free_at(std::greater<double>(),
                                                                                      std::vector<double>(c.begin(), c.begin() + n_cu));
        double top = c[0];
        for (size_t i = (size_t)n_cu; i < c.size(); ++i) {
            const double t = free_at.top() + c[i];
            free_at.pop();
            free_at.push(t);
            top = std::max(top, t);
        }
        return top;
    }
};

}  // namespace

static int worklist_cut(const int64_t* counts, const int64_t* seg_tile, int nseg, int n_cu, int64_t target_items,
                        int64_t min_item_bytes, int chains, int pairs, int waves, odmkv_worklist_choice_t* choice,
                        int32_t* table, uint64_t capacity, odmkv_worklist_shape_t* shape) {
    ODMKV_CHECK_ARG(counts && seg_tile && choice && shape && (table || !capacity), "odmkv_worklist_cut: null pointer");
    ODMKV_CHECK_ARG(nseg > 0 && n_cu > 0 && min_item_bytes >= 0, "odmkv_worklist_cut: bad sizes (segments %d, compute units %d)", nseg, n_cu);
    Cutter k;
    k.nseg = nseg; k.n_cu = n_cu; k.total = 0; k.total_bytes = 0;
    k.min_cost = min_item_bytes * kTileCost[0] / kTileBytes[0];          // the same floor, as a cost
    int64_t q_bytes[4] = {0, 0, 0, 0};
    // the runs of tiles, segment by segment (the merge finds a segment's items next to each other)
    int n_exact = 0, n_pairs = 0;
    k.seg_cost.assign(nseg, 0.0); k.seg_start.assign(nseg, 0.0);
    double line = 0.0;
    for (int s = 0; s < nseg; ++s) {
        k.seg_start[s] = line;
        bool first = true;
        for (int li = 0; li < 5; ++li) {
            const int64_t c = counts[(size_t)li * nseg + s], t0 = seg_tile[(size_t)li * (nseg + 1) + s];
            // exact segments grow between rebuilds: their whole capacity
            const int64_t nt = li == 4 ? seg_tile[(size_t)li * (nseg + 1) + s + 1] - t0 : (c + TILE - 1) / TILE;
            if (nt <= 0) continue;
            ODMKV_CHECK_ARG(nt < (1 << 30), "odmkv_worklist_cut: %lld tiles of level %d in segment %d", (long long)nt, li, s);
            k.total += nt * kTileCost[li]; k.total_bytes += nt * kTileBytes[li];
            k.runs.push_back({s, li, nt, t0, c});
            if (li == 4) { n_exact += 1; continue; }
            q_bytes[li] += nt * kTileBytes[li];
            const double cst = (double)(nt * kTileCost[li]);
            k.q.push_back((int)k.runs.size() - 1);
            k.q_start.push_back(line);
            line += cst;
            k.q_end.push_back(line);
            k.seg_cost[s] += cst;
            k.q_first.push_back(first);
            n_pairs += first;
            first = false;
        }
    }
    const bool may_chain = !k.q.empty() && (int)k.q.size() > n_pairs && chains != 0;
    bool paired = pairs == 1;
    std::vector<Item> items;
    if (target_items > 0) {
        items = may_chain && chains == 1 ? k.cut_chained(k.fit_chained(target_items)) : k.cut(k.fit(target_items));
    } else if (choice->valid && fabs((double)(k.total_bytes - choice->total_bytes)) <= 0.05 * (double)choice->total_bytes) {
        // the comparison is repeated only when the store has grown by more than 5 % since the last one (a decode-time
        // flush adds a fraction of a percent): until then its winner is cut again
        const int64_t target = (int64_t)(n_cu * choice->multiple);
        items = choice->chained && may_chain ? k.cut_chained(k.fit_chained(target)) : k.cut(k.fit(target));
        paired = choice->paired != 0;
    } else {
        // With a target the cut is the coarsest one that does not exceed it.  Without one, a few cuts are compared by the
        // time a longest-first assignment of their items to the compute units would take, and the best is kept.
        bool have = false, best_chained = false;
        double best_t = 0.0, best_mult = 1.0;
        if (chains != 1 || !may_chain) {
            const double mults[5] = {1.0, 1.5, 2.0, 3.0, 4.0};
            for (double m : mults) {
                std::vector<Item> cand = k.cut(k.fit((int64_t)(n_cu * m)));
                const double t = k.makespan(cand, have ? best_t : INFINITY);
                if (!have || t < best_t - 1e-9) { have = true; best_t = t; best_mult = m; items.swap(cand); }
            }
        }
        const double nq = (double)k.q.size();
        if (pairs != 0 && (paired || (have && (int)items.size() > n_cu))) {
            // More items than compute units: the workgroups would run in rounds, each paying its start (work item,
            // rotation, table, first bytes: about 4 us) and its end (combine) with the compute unit to itself.
            // Two eight-wavefront workgroups per compute unit overlap one's start and end with the other's
            // stream (measured: a 16 x 8192-token batch 28.1 -> 25.9 us, 64 x 2048 tokens 52 -> 40 us; lists of
            // one item per compute unit lose 5-10 %, and keep the wide workgroups).  Cut for one round of the
            // 2 x n_cu places; where the runs alone are many more than that, chain a pair's levels instead.
            paired = true;
            if (may_chain && (chains == 1 || nq + n_exact > kPairChainRunsPerPlace * 2 * n_cu)) {
                best_mult = std::max(2.0, (double)(n_pairs + n_exact) / n_cu);
                items = k.cut_chained(k.fit_chained((int64_t)(n_cu * best_mult)));
                best_chained = true;
            } else {
                best_mult = 2.0;
                items = k.cut(k.fit(2 * (int64_t)n_cu));
            }
        } else if (may_chain && (chains == 1 || (nq >= kChainRunsPerCu * n_cu && nq >= kChainRunsPerPair * n_pairs))) {
            best_mult = std::max(1.5, (double)(n_pairs + n_exact) / n_cu);
            items = k.cut_chained(k.fit_chained((int64_t)(n_cu * best_mult)));
            best_chained = true;
        }
        choice->valid = 1; choice->multiple = best_mult; choice->total_bytes = k.total_bytes;
        choice->chained = best_chained; choice->paired = paired;
    }
    const int n = (int)items.size();
    int n_heads = 0;
    for (const Item& it : items) n_heads += !it.cont;
    const bool chained = n > 0 && n_heads != n;
    paired = paired && n > 0;
    const bool ordered = n > n_cu || chained || paired;
    const uint64_t at_range = (uint64_t)n * 8, at_order = at_range + (((uint64_t)nseg + 1 + 3) & ~3ull);
    shape->need = at_order + (ordered ? n_heads : 0);
    shape->range_at = at_range; shape->order_at = at_order;
    shape->n_items = n; shape->ordered = ordered;
    shape->n_workgroups = chained ? n_heads : 0;
    shape->two_per_cu = paired;
    // Wavefronts per item: eight for short items (less set-up, a lighter combine), twelve for long ones.
    // Items of 6 to 15 tiles that are mostly 3 bits and wider: twelve as well, 2-3 % ahead of eight (measured on a 28-head, 3-bit
    // store of 32k tokens: their loops wait on memory, and a third wavefront a SIMD pays).  Short items whose quantised tokens are
    // nearly all of 2 bits: twelve too, us a layer with eight / twelve: 600 tokens 10.83 / 10.64, 8192 11.60 / 11.35, 28 heads over 4
    // 11.77 / 11.59; with a quarter of 3 bits among them (8192 tokens at 2.25 bits) 12.02 / 12.24, at 3 bits 12.07 / 12.37.
    double q_tiles = 0.0;
    int64_t q_groups = 0;
    {
        double own = 0.0;                                               // quantised tiles per workgroup (chained), or per item
        for (int i = 0; i < n; ++i) {
            if (!items[i].cont) { if (own > 0) { q_tiles += own; q_groups += 1; } own = 0.0; }
            if (items[i].li < 4) own += (double)items[i].nt;
        }
        if (own > 0) { q_tiles += own; q_groups += 1; }
    }
    const double mean = q_groups ? q_tiles / (double)q_groups : 0.0;
    const int64_t q_all = q_bytes[0] + q_bytes[1] + q_bytes[2] + q_bytes[3];
    const double q_floor = (double)std::max<int64_t>(q_all, 1);
    const bool medium = mean >= 6 && (double)(q_all - q_bytes[0]) >= 0.5 * q_floor;
    const bool narrow = (double)q_bytes[0] >= 0.9 * q_floor;
    const int automatic = q_groups && (mean >= 16 || medium || narrow) ? 12 : 8;
    shape->wavefronts = paired ? 8 : waves > 0 ? waves : automatic;
    if (capacity < shape->need) {
        odmkv_set_error("odmkv_worklist_cut: the table needs %llu integers, %llu given", (unsigned long long)shape->need, (unsigned long long)capacity);
        return ODMKV_ENOSPACE;
    }
    memset(table, 0, shape->need * sizeof(int32_t));
    int32_t* range = table + at_range;
    for (int i = 0; i < n; ++i) {
        const Item& it = items[i];
        const int32_t row[8] = {(int32_t)it.s, (int32_t)it.li, (int32_t)it.t0, (int32_t)it.nt, (int32_t)it.cnt, (int32_t)it.seg0, it.follow, it.cont};
        memcpy(table + (size_t)i * 8, row, sizeof row);
        range[it.s + 1] += 1;
    }
    for (int s = 0; s < nseg; ++s) range[s + 1] += range[s];
    if (ordered) {
        // the workgroups' first items, longest workgroup first
        const std::vector<double> c = Cutter::cost(items);
        std::vector<int> head, by(n_heads);
        for (int i = 0; i < n; ++i) if (!items[i].cont) head.push_back(i);
        for (int i = 0; i < n_heads; ++i) by[i] = i;
        std::stable_sort(by.begin(), by.end(), [&](int a, int b) { return c[a] > c[b]; });
        // two per compute unit: the first n_cu workgroups land one per compute unit, the next n_cu beside them in the same
        // order of compute units; taken shortest first, the shortest joins the longest (a 16 x 8192-token batch
        // 26.0 -> 25.5 us; long and short alternating: 32 us)
        if (paired && n_heads > n_cu) std::reverse(by.begin() + n_cu, by.begin() + std::min(n_heads, 2 * n_cu));
        for (int i = 0; i < n_heads; ++i) table[at_order + i] = head[by[i]];
    }
    return 0;
}

extern "C" int odmkv_worklist_cut(const int64_t* counts, const int64_t* seg_tile, int nseg, int n_cu, int64_t target_items,
                                  int64_t min_item_bytes, int chains, int pairs, int waves, odmkv_worklist_choice_t* choice,
                                  int32_t* table, uint64_t capacity, odmkv_worklist_shape_t* shape) {
    try {                                                     // (callers are C: nothing is thrown through them)
        return worklist_cut(counts, seg_tile, nseg, n_cu, target_items, min_item_bytes, chains, pairs, waves, choice, table, capacity, shape);
    } catch (const std::exception& e) {
        odmkv_set_error("odmkv_worklist_cut: %s", e.what());
        return ODMKV_ENOMEM;
    }
}
