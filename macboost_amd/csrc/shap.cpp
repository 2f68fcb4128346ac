// shap.cpp — host side of TreeSHAP: the contribution-table plan (groups of
// paths, their outcome bits and columns) and the choice between it and the
// path-per-lane kernels, for the booster and the kernel seam.
#include <algorithm>
#include <cstring>

#include "core.hpp"

namespace mb {

namespace {

// Doubles of a set's tables before its last tree: trees are split into sets so
// that a set's columns stay in the 256 MB last-level cache and scratch stays bounded
// (the last tree adds 1,024 groups of 12 columns of 2^12 doubles at most: with it
// below 0.7 GB).
constexpr size_t SET_DOUBLES = (size_t)1 << 25;
// Bytes of a slab's outcomes and of its runs.
constexpr size_t SLAB_BYTES = (size_t)128 << 20;
// Bytes of the sums that several sets share: more rows go in passes, each making
// the sets' tables again (a pass is 671k rows of 100 columns).
constexpr size_t SUM_BYTES = (size_t)512 << 20;
// Workgroups that share the batches of a row block.  A share's end cuts a feature's
// sum, so their number goes by the plan alone: a row's result does not depend on the
// other rows of its call.  Each costs a store of its rows' sums, fewer leave the
// chip idle for few rows.  100 trees of depth 6, 1k, 20k and 200k rows of 100 columns:
// 0.31, 0.37 and 1.30 ms with 32 shares, 0.28, 0.34 and 1.24 with 64, 0.28, 0.33 and
// 1.26 with 96, 0.28, 0.35 and 1.29 with 128 (0.26, 0.33 and 1.33 when each call took
// what filled the chip).  50 trees of depth 9, 20k rows: 4.21 ms with 64, 3.83 with
// 128, 3.70 with 256, 3.74 with 512 (3.81); many batches a share repay the stores.
int plan_shares(int32_t batches) {
    return std::max(1, std::min(std::clamp(batches / 16, 96, 256), batches));
}

// One tree's groups, appended to a set.
class TreeGroups {
public:
    TreeGroups(ShapPlan &plan, ShapSetPlan &sp, const TreeView &tr, size_t tree,
               int nodes_per_tree, int32_t cols)
        : plan_(plan), sp_(sp), tr_(tr), node0_((int64_t)tree * nodes_per_tree), cols_(cols) {}

    // Appends the tree; the doubles its columns take.
    size_t add() {
        std::vector<uint8_t> &h = plan_.height;
        h.assign((size_t)tr_.nodes, 0);
        for (int n = (tr_.nodes - 1) / 2 - 1; n >= 0; --n)    // slots with both children
            if (tr_.feature[n] >= 0)
                h[(size_t)n] = (uint8_t)(1 + std::max(h[(size_t)(2 * n + 1)], h[(size_t)(2 * n + 2)]));
        if (h[0] > 0) walk(0);                         // a lone leaf: bias only
        return doubles_;
    }

private:
    bool split(int n) const { return plan_.height[(size_t)n] > 0; }

    double share(int n, bool left) const {
        const double cp = (double)tr_.cover[n];
        return cp > 0 ? (double)tr_.cover[2 * n + (left ? 1 : 2)] / cp : 0.0;
    }

    mbk::ShapTest test(int n, bool left, int bit) const {
        if (tr_.feature[n] >= cols_) invalid("a tree splits on a feature past the data's columns");
        return {tr_.feature[n], tr_.threshold[n],
                (uint32_t)tr_.flags[n] | (left ? 0x100u : 0u) | ((uint32_t)bit << 16),
                (int32_t)(node0_ + n)};
    }

    // Appends a group's test.  Where missing values go left at a NaN threshold they are
    // all that does, which is no single compare with it: a row goes right there if it
    // is at or below +inf, left if it is not above -inf and not -inf.  (As a case of its
    // own in the kernel: outcomes of 20k rows x 50 trees of depth 8 394 -> 435 us.)
    void push(mbk::ShapTest t) {
        const uint32_t side = mbk::FLAG_DEFAULT_LEFT | 0x100u;
        if (!std::isnan(t.threshold) || (t.flags & mbk::FLAG_CATEGORICAL) ||
            !(t.flags & mbk::FLAG_DEFAULT_LEFT)) {
            sp_.tests.push_back(t);
        } else if (t.flags & 0x100u) {
            t.threshold = -INFINITY;
            sp_.tests.push_back(t);                    // NaN or -inf
            t.flags &= ~side;
            sp_.tests.push_back(t);                    // not -inf
        } else {
            t.threshold = INFINITY;
            t.flags ^= side;
            sp_.tests.push_back(t);                    // not NaN
        }
    }

    // Repeated features of the ancestors share one bit, whose unfollowed share
    // is the product of theirs, root first.
    void walk(int n) {
        if (plan_.height[(size_t)n] <= 2) { group(n); return; }
        if (depth_ >= 12) internal("TreeSHAP supports paths of at most 12 splits");
        const int32_t f = tr_.feature[n];
        int b = 0;
        while (b < anc_ && anc_feature_[b] != f) ++b;
        const bool fresh = b == anc_;
        const double before = fresh ? 1.0 : anc_zero_[b];
        anc_feature_[b] = f;
        anc_ += fresh;
        for (int left = 1; left >= 0; --left) {
            path_[depth_++] = test(n, left != 0, b);
            anc_zero_[b] = before * share(n, left != 0);
            walk(2 * n + (left ? 1 : 2));
            --depth_;
        }
        anc_zero_[b] = before;
        anc_ -= fresh;
    }

    // The group of root g: the ancestors' bits, then one per split inside.
    void group(int g) {
        mbk::ShapGroup G{};
        G.test_start = (int32_t)sp_.tests.size();
        G.val_start = (int32_t)sp_.vals.size();
        G.col_start = (int32_t)sp_.col_feature.size();
        G.anc = anc_;
        G.bits = anc_;
        for (int k = 0; k < depth_; ++k) push(path_[k]);
        sp_.vals.insert(sp_.vals.end(), anc_zero_, anc_zero_ + anc_);
        sp_.col_feature.insert(sp_.col_feature.end(), anc_feature_, anc_feature_ + anc_);
        int feature[SHAP_FEATURES];
        std::copy(anc_feature_, anc_feature_ + anc_, feature);
        int nf = anc_, extra = 0;
        const int at[3] = {g, 2 * g + 1, 2 * g + 2};
        for (int k = 0; k < 3; ++k) {
            if ((k > 0 && !split(g)) || !split(at[k])) continue;
            push(test(at[k], true, G.bits));
            const int32_t f = tr_.feature[at[k]];
            int c = 0;
            while (c < nf && feature[c] != f) ++c;
            if (c == nf) {
                feature[nf++] = f;
                sp_.col_feature.push_back(f);
            }
            G.inside[k] = (uint32_t)c | ((uint32_t)G.bits << 8) | 0x10000u;
            ++G.bits;
            extra = k == 0 ? 1 : 2;
            sp_.vals.push_back(share(at[k], true));
            sp_.vals.push_back(share(at[k], false));
        }
        // the leaves: g itself, or the children's positions 0 .. 3 (a child that
        // is a leaf at its left position)
        const int n0 = (int)sp_.vals.size();
        for (int q = 0; q < 4; ++q) {
            int n = g;
            bool path = q == 0;
            if (split(g)) {
                const int c = at[1 + (q >> 1)];
                path = split(c) || !(q & 1);
                n = split(c) ? 2 * c + 1 + (q & 1) : c;
            }
            path = path && tr_.feature[n] < 0;          // a split without children: no path
            if (path) G.leaves |= 1u << q;
            sp_.vals.push_back(path ? (double)tr_.leaf[n] : 0.0);
        }
        G.leaf_start = n0;
        G.num_cols = nf;
        G.num_tests = (int32_t)sp_.tests.size() - G.test_start;
        while (sp_.tests.size() % 4) sp_.tests.push_back(sp_.tests.back());   // whole quads
        sp_.groups.push_back(G);
        if (depth_ + extra > 12) internal("TreeSHAP supports paths of at most 12 splits");
        if (G.bits > mbk::SHAP_MAX_BITS) plan_.fits = false;
        sp_.set.max_bits = std::max(sp_.set.max_bits, G.bits);
        sp_.set.max_slots = std::max(sp_.set.max_slots, anc_ + extra);
        doubles_ += (size_t)nf << G.bits;
        const int64_t leaves = __builtin_popcount(G.leaves);
        plan_.paths += leaves;
        plan_.evals += leaves << G.bits;
    }

    static constexpr int SHAP_FEATURES = 16;
    ShapPlan &plan_;
    ShapSetPlan &sp_;
    const TreeView &tr_;
    int64_t node0_;
    int32_t cols_;
    size_t doubles_ = 0;
    mbk::ShapTest path_[12];
    int32_t anc_feature_[12];
    double anc_zero_[12];
    int depth_ = 0, anc_ = 0;
};

// The set's columns in feature order, cut into LDS batches, and the runs of the
// workgroups that share them.
void order_columns(ShapSetPlan &sp, int32_t cols) {
    constexpr uint32_t BATCH = 4096;                   // doubles (SHAP_LDS_DOUBLES)
    const size_t n = sp.col_feature.size();
    std::vector<uint32_t> &at = sp.at, &order = sp.order;
    at.assign((size_t)cols + 1, 0u);
    order.resize(2 * n);
    sp.col_off.resize(n);
    sp.items.resize(n);
    sp.batches.clear();
    for (int32_t f : sp.col_feature) at[(size_t)f + 1]++;
    for (int32_t f = 0; f < cols; ++f) at[(size_t)f + 1] += at[(size_t)f];
    for (size_t g = 0; g < sp.groups.size(); ++g)
        for (int32_t c = 0; c < sp.groups[g].num_cols; ++c) {
            const size_t q = (size_t)(sp.groups[g].col_start + c);
            const uint32_t k = at[(size_t)sp.col_feature[q]]++;
            order[2 * k] = (uint32_t)q;
            order[2 * k + 1] = (uint32_t)g;
        }
    uint32_t off = 0;
    for (size_t k = 0; k < n; ++k) {
        const uint32_t g = order[2 * k + 1], len = 1u << sp.groups[g].bits;
        if (sp.batches.empty() || sp.batches.back().table_len + len > BATCH)
            sp.batches.push_back({(uint32_t)k, 0, off, 0});
        mbk::ShapBatch &b = sp.batches.back();
        sp.items[k] = {g, b.table_len};
        sp.col_off[order[2 * k]] = off;
        b.num_items += 1;
        b.table_len += len;
        off += len;
    }
    sp.set.table_len = off;
    sp.set.num_groups = (int32_t)sp.groups.size();
    sp.set.num_batches = (int32_t)sp.batches.size();
    sp.set.shares = plan_shares(sp.set.num_batches);
    // a run ends with its feature or with its workgroup's share of the batches
    sp.run_first.assign((size_t)cols + 1, 0u);
    sp.run_item.assign(1, 0u);
    uint32_t run = 0;
    size_t k = 0;
    for (int64_t q = 0; q < sp.set.shares; ++q) {
        const int64_t b1 = (int64_t)sp.set.num_batches * (q + 1) / sp.set.shares;
        if (b1 == 0) continue;
        const mbk::ShapBatch &b = sp.batches[(size_t)(b1 - 1)];
        for (const size_t end = (size_t)b.item_start + (size_t)b.num_items; k < end; ++k) {
            const int32_t f = sp.col_feature[order[2 * k]];
            if (k + 1 < end && sp.col_feature[order[2 * k + 2]] == f) continue;
            sp.items[k].offset_run |= ++run << 12;
            sp.run_first[(size_t)f + 1] = run;
            sp.run_item.push_back((uint32_t)k + 1);
        }
    }
    for (int32_t f = 0; f < cols; ++f)
        sp.run_first[(size_t)f + 1] = std::max(sp.run_first[(size_t)f + 1], sp.run_first[(size_t)f]);
    sp.set.num_runs = (int32_t)run;
}

void make_plan(ShapPlan &plan, const std::vector<TreeView> &trees, size_t first, size_t step,
               int nodes_per_tree, int32_t cols) {
    plan.num_sets = 0;
    plan.paths = plan.evals = 0;
    plan.fits = true;
    size_t doubles = SET_DOUBLES;
    for (size_t t = first; t < trees.size() && plan.fits; t += step) {
        if (!(trees[t].cover && trees[t].cover[0] > 0)) continue;
        if (doubles >= SET_DOUBLES) {                  // the set before is full
            if (plan.num_sets == plan.sets.size()) plan.sets.emplace_back();
            plan.sets[plan.num_sets++].clear();
            doubles = 0;
        }
        TreeGroups tg(plan, plan.sets[plan.num_sets - 1], trees[t], t, nodes_per_tree, cols);
        doubles += tg.add();
    }
    for (size_t k = 0; k < plan.num_sets && plan.fits; ++k) {
        order_columns(plan.sets[k], cols);
        plan.fits = plan.sets[k].set.num_runs < 1 << 20;   // an item's bits for its run
    }
    plan.made = true;
}

template <typename T>
size_t append(std::vector<char> &blob, const std::vector<T> &v) {
    blob.resize((blob.size() + 15) / 16 * 16);
    const size_t off = blob.size();
    const char *p = reinterpret_cast<const char *>(v.data());
    blob.insert(blob.end(), p, p + v.size() * sizeof(T));
    return off;
}

// Grown to n elements; sizes of pooled buffers are rounded up (to an eighth of
// their power of two) so that calls of similar sizes share blocks.
template <typename T>
T *reserve(DevBuf<T> &b, size_t n) {
    if (b.n >= n) return b.ptr;
    if (b.pooled) {
        size_t unit = 1;
        while (unit * 8 < n) unit *= 2;
        n = (n + unit - 1) / unit * unit;
    }
    b.alloc(n);
    return b.ptr;
}

// Whether the call's rows are few enough for launch_shap_rows, which costs a path
// evaluation per path and row where tables cost `evals` of them and two launches more.
// Host rows of 20 columns, tables / few rows, us a call:
//   1 tree of depth 6     1 row 80 / 54, 4,000 100 / 78, 16,000 192 / 198
//   20 of depth 6         1 row 113 / 76, 500 101 / 94, 1,000 104 / 119
//   100 of depth 9        1 row 1,967 / 636, 500 1,961 / 2,029
//   10 of depth 11        1 row 2,666 / 372, 1,000 2,660 / 1,800, 2,000 2,679 / 3,102
//   100 stumps            1 row 93 / 64, 5,000 118 / 97, 8,000 131 / 124
//   100 of depth 3        1 row 140 / 74, 4,000 151 / 143, 8,000 174 / 220
//   1,000 of depth 4      64 rows 338 / 311, 500 331 / 426
// (short paths are the cheaper ones).  With tables for any rows, calls of few rows and few
// trees took up to 1.7 times as long as by path.
bool few_rows(const ShapPlan &plan, int64_t rows) {
    int32_t slots = 0;                                 // features of the longest path
    for (size_t k = 0; k < plan.num_sets; ++k) {
        if (plan.sets[k].set.num_runs > mbk::SHAP_FEW_RUNS) return false;
        slots = std::max(slots, plan.sets[k].set.max_slots);
    }
    const int64_t launches = slots <= 4 ? 1600000 : 700000;   // in path evaluations
    return rows <= 8192 && rows * plan.paths <= launches + plan.evals / 2;
}

// Every column's place in the feature order, made by the plan's first call of few rows.
const std::vector<uint32_t> &column_places(ShapSetPlan &sp) {
    const size_t n = sp.col_feature.size();
    if (sp.col_at.size() != n) {
        sp.col_at.resize(n);
        for (size_t k = 0; k < n; ++k) sp.col_at[sp.order[2 * k]] = (uint32_t)k;
    }
    return sp.col_at;
}

// TreeSHAP of few rows, in slabs of rows whose entries and sums stay bounded.
void run_rows(hipStream_t s, const ShapCall &c, ShapPlan &plan, ShapScratch &sc) {
    std::vector<char> &blob = sc.blob;
    blob.clear();
    struct Offsets { size_t tests, groups, vals, run_first, col_at, run_item; };
    std::vector<Offsets> offs;
    size_t columns = 1;
    for (size_t k = 0; k < plan.num_sets; ++k) {
        ShapSetPlan &sp = plan.sets[k];
        offs.push_back({append(blob, sp.tests), append(blob, sp.groups), append(blob, sp.vals),
                        append(blob, sp.run_first), append(blob, column_places(sp)),
                        append(blob, sp.run_item)});
        columns = std::max(columns, sp.col_at.size());
    }
    const bool several = plan.num_sets > 1;
    int64_t slab = (int64_t)(SLAB_BYTES / 8 / columns);
    if (several) slab = std::min(slab, (int64_t)(SUM_BYTES / 8 / (size_t)c.cols));
    slab = std::min(c.rows, std::max<int64_t>(1, slab));
    char *d = reserve(sc.arrays, blob.size());
    reserve(sc.runs, columns * (size_t)slab);
    if (several) reserve(sc.sums, (size_t)slab * (size_t)c.cols);
    MB_HIP(hipMemcpyAsync(d, blob.data(), blob.size(), hipMemcpyHostToDevice, s));
    for (int64_t r0 = 0; r0 < c.rows; r0 += slab)
        for (size_t k = 0; k < plan.num_sets; ++k) {
            const Offsets &o = offs[k];
            mbk::ShapSetDev dev{};
            dev.tests = reinterpret_cast<mbk::ShapTest *>(d + o.tests);
            dev.groups = reinterpret_cast<mbk::ShapGroup *>(d + o.groups);
            dev.vals = reinterpret_cast<double *>(d + o.vals);
            dev.run_first = reinterpret_cast<uint32_t *>(d + o.run_first);
            dev.col_at = reinterpret_cast<uint32_t *>(d + o.col_at);
            dev.run_item = reinterpret_cast<uint32_t *>(d + o.run_item);
            mbk::ShapRows w{};
            w.x = c.x;
            w.rows = c.rows;
            w.row0 = r0;
            w.num_rows = std::min(slab, c.rows - r0);
            w.cols = c.cols;
            w.data_bins = c.data_bins;
            w.masks = c.masks;
            w.entries = sc.runs.ptr;
            w.total = several ? sc.sums.ptr : nullptr;
            w.first = k == 0;
            w.last = k + 1 == plan.num_sets;
            w.bias = c.bias;
            w.out = c.out;
            MB_HIP(mbk::launch_shap_rows(s, plan.sets[k].set, dev, w));
        }
}

// TreeSHAP by path per lane (k_treeshap_rows / k_treeshap).
void run_paths(hipStream_t s, const std::vector<TreeView> &trees, size_t first, size_t step,
               int nodes_per_tree, const ShapCall &c, ShapScratch &sc) {
    const ShapTables st = shap_tables(trees, first, step, nodes_per_tree);
    const StreamIdle idle{s};                          // before the arrays go
    // Each array goes from where it was made: put together on the host first, those of
    // 10 trees of depth 12 made a call of 1 to 200 rows 22 ms instead of 15.4.
    size_t bytes = 0;
    auto place = [&](const auto &v) {
        const size_t at = (bytes + 15) / 16 * 16;
        bytes = at + v.size() * sizeof(v[0]);
        return at;
    };
    const size_t op = place(st.paths), oe = place(st.elems), ou = place(st.uniq);
    char *d = reserve(sc.arrays, bytes);
    auto copy = [&](size_t at, const auto &v) {
        MB_HIP(hipMemcpyAsync(d + at, v.data(), v.size() * sizeof(v[0]), hipMemcpyHostToDevice, s));
    };
    copy(op, st.paths);
    copy(oe, st.elems);
    copy(ou, st.uniq);
    double *phi = nullptr;
    if (mbk::treeshap_needs_scratch(c.cols))
        phi = reserve(sc.sums, (size_t)((c.rows + 63) / 64) * 64 * (size_t)c.cols);
    MB_HIP(mbk::launch_treeshap(s, c.x, c.rows, c.cols, c.data_bins, c.masks,
                                reinterpret_cast<mbk::ShapPath *>(d + op), (int)st.paths.size(),
                                st.max_elems, reinterpret_cast<mbk::ShapElem *>(d + oe),
                                reinterpret_cast<mbk::ShapUniq *>(d + ou), c.bias, c.out, phi));
}

}  // namespace

bool treeshap(hipStream_t s, const std::vector<TreeView> &trees, size_t first, size_t step,
              int nodes_per_tree, const ShapCall &c, ShapPlan &plan, ShapScratch &sc) {
    if (!plan.made) make_plan(plan, trees, first, step, nodes_per_tree, c.cols);
    if (plan.fits && plan.paths == 0) return false;
    // A row's last bits depend on the order of its sums, which the path kernels do not
    // share: the rows of the call do not enter that choice (they do between tables and
    // few rows, whose sums are the same).
    if (!plan.fits) {
        run_paths(s, trees, first, step, nodes_per_tree, c, sc);
        MB_HIP(hipStreamSynchronize(s));
        return true;
    }
    if (few_rows(plan, c.rows)) {
        run_rows(s, c, plan, sc);
        MB_HIP(hipStreamSynchronize(s));               // the arrays leave with this call
        return true;
    }
    // Slab: rows whose outcomes (and runs) take SLAB_BYTES at most.
    constexpr int64_t BLOCK = mbk::SHAP_BLOCK_ROWS;
    const int64_t blocks_all = (c.rows + BLOCK - 1) / BLOCK;
    size_t row_bytes = 1;
    for (size_t k = 0; k < plan.num_sets; ++k) {
        const ShapSetPlan &sp = plan.sets[k];
        row_bytes = std::max({row_bytes, sp.groups.size() * (sp.set.max_bits > 8 ? 2 : 1),
                              (size_t)sp.set.num_runs * 8});
    }
    const bool several = plan.num_sets > 1;
    const int64_t sum_rows = (int64_t)(SUM_BYTES / 8 / (size_t)c.cols);
    int64_t blocks = (int64_t)(SLAB_BYTES / row_bytes / BLOCK);
    if (several) blocks = std::min(blocks, sum_rows / BLOCK);
    blocks = std::min(blocks_all, std::max<int64_t>(1, blocks));
    const int64_t slab = blocks * BLOCK;
    std::vector<char> &blob = sc.blob;
    blob.clear();
    struct Offsets { size_t tests, groups, vals, col_off, items, batches, run_first; };
    std::vector<Offsets> offs;
    size_t table = 2, pattern_bytes = 16, runs = 1;
    for (size_t k = 0; k < plan.num_sets; ++k) {
        const ShapSetPlan &sp = plan.sets[k];
        offs.push_back({append(blob, sp.tests), append(blob, sp.groups), append(blob, sp.vals),
                        append(blob, sp.col_off), append(blob, sp.items),
                        append(blob, sp.batches), append(blob, sp.run_first)});
        table = std::max(table, sp.set.table_len);
        pattern_bytes = std::max(pattern_bytes, sp.groups.size() * (size_t)slab *
                                                    (sp.set.max_bits > 8 ? 2 : 1));
        runs = std::max(runs, (size_t)sp.set.num_runs * (size_t)slab);
    }
    char *d = reserve(sc.arrays, blob.size());
    reserve(sc.table, table);
    reserve(sc.patterns, pattern_bytes);
    reserve(sc.runs, runs);
    // rows of a pass over the sets, whole slabs
    int64_t pass = c.rows;
    if (several) {
        pass = std::min(c.rows, std::max(slab, sum_rows / slab * slab));
        reserve(sc.sums, (size_t)pass * (size_t)c.cols);
    }
    MB_HIP(hipMemcpyAsync(d, blob.data(), blob.size(), hipMemcpyHostToDevice, s));
    for (int64_t p0 = 0; p0 < c.rows; p0 += pass) {
        const int64_t p1 = std::min(c.rows, p0 + pass);
        for (size_t k = 0; k < plan.num_sets; ++k) {
            const ShapSetPlan &sp = plan.sets[k];
            const Offsets &o = offs[k];
            const mbk::ShapSetDev dev{reinterpret_cast<mbk::ShapTest *>(d + o.tests),
                                      reinterpret_cast<mbk::ShapGroup *>(d + o.groups),
                                      reinterpret_cast<double *>(d + o.vals),
                                      reinterpret_cast<uint32_t *>(d + o.col_off),
                                      reinterpret_cast<mbk::ShapItem *>(d + o.items),
                                      reinterpret_cast<mbk::ShapBatch *>(d + o.batches),
                                      reinterpret_cast<uint32_t *>(d + o.run_first),
                                      nullptr, nullptr};
            MB_HIP(mbk::launch_shap_tables(s, sp.set, dev, sc.table.ptr));
            for (int64_t r0 = p0; r0 < p1; r0 += slab) {
                mbk::ShapSlab w{};
                w.x = c.x;
                w.rows = c.rows;
                w.row0 = r0;
                w.slab_rows = std::min(slab, (p1 - r0 + BLOCK - 1) / BLOCK * BLOCK);
                w.cols = c.cols;
                w.data_bins = c.data_bins;
                w.masks = c.masks;
                w.table = sc.table.ptr;
                w.patterns = sc.patterns.ptr;
                w.runs = sc.runs.ptr;
                w.total = several ? sc.sums.ptr : nullptr;
                w.total_row0 = p0;
                w.total_rows = pass;
                w.first = k == 0;
                w.last = k + 1 == plan.num_sets;
                w.bias = c.bias;
                w.out = c.out;
                MB_HIP(mbk::launch_shap_slab(s, sp.set, dev, w));
            }
        }
    }
    MB_HIP(hipStreamSynchronize(s));                   // the arrays leave with this call
    return true;
}

}  // namespace mb
