// kernels_infer.hip — gfx950 inference kernels: batch forest prediction on raw
// features (predict_forest, Shaders.swift:1541-1584), the binned single-tree
// walk used for per-iteration validation (predict_tree_binned, :1763-1781) and
// exact TreeSHAP (gpu_treeshap, :1656-1734).
//
// TreeSHAP here computes path contributions once per split outcome into tables
// and looks every row's up (few rows: by the row's own outcomes, no tables), all in
// double precision with a fixed summation order and a single rounding to f32 at the
// end.  Trees too deep for tables (more
// than 12 outcome bits) give each row a wavefront and each root-to-leaf path a
// lane, with the row's phi in LDS.
#include <algorithm>

#include "grad.h"
#include "mbk.h"

#include <math.h>

namespace mbk {

__device__ __forceinline__ bool raw_goes_left(float v, uint32_t flags, float thr,
                                              const uint32_t *mask_node, int32_t data_bins) {
    if (flags & FLAG_CATEGORICAL) {
        uint32_t cat = (uint32_t)data_bins;            // unseen -> missing
        if (isfinite(v)) {
            const float r = rintf(v);
            if (r >= 0.0f && (int64_t)r < data_bins) cat = (uint32_t)r;
        }
        return mask_node ? ((mask_node[cat >> 5] >> (cat & 31u)) & 1u) != 0 : false;
    }
    if (isnan(v)) return (flags & FLAG_DEFAULT_LEFT) != 0;
    return v <= thr;
}

// Compute units of the current device (cached per device id).
static int device_cus() {
    static int cache[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (cache[dev] == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            n <= 0)
            n = 256;
        cache[dev] = n;
    }
    return cache[dev];
}

// Batch prediction: a workgroup takes 64 rows, a row per lane.  Each of its 16
// wavefronts walks them down every 16th tree of a chunk, two trees at a time, and
// leaves their values in LDS, where the first wavefront adds them in tree order
// (f32, as one thread walking them in turn would: bit for bit).  The first `stage`
// heap slots of a chunk's trees are staged in LDS as one 8-byte word each
// (threshold or leaf value; feature and flags, negative at a leaf), and so are the
// rows' values of the features a listed forest uses ([slot][64]: lanes reading different
// features of their own rows hit different banks), so a step of the walk is two LDS
// reads.  One thread per row took a chain of three dependent global loads per step,
// each lane's on a line of its own: 100 trees of depth 6 over 100 features took 230 us
// for 1 to 20k rows (20 and 28 us now) and 795 us for 500k (309 us).  Bound by the
// instructions and LDS latency of a step.  A forest whose nodes fit next to a tile's
// features (160 KB) is staged once per workgroup; else LDS is held to 80 KB where the
// features allow it, for two workgroups (32 wavefronts) per CU.
constexpr int PRED_THREADS = 1024;
constexpr int PRED_WAVES = PRED_THREADS / 64;

// Features of the nodes a row can reach: heap slots under a leaf may hold anything,
// and the walk reads every listed feature's column.  Workgroups mark the features of
// FOREST_NODES nodes or more each in mark (PRED_MARK_WORDS, zero between launches: a bit
// per feature, a past-the-map flag, the workgroups done); the last to finish lists them.
// Bound by the loads on the way up to the root.  One workgroup for the whole forest
// held a call up by some 1.2 us per 1,024 nodes: 4,096 rows of 100 trees of depth 12 took
// 1,058 us, now 131, 1,000 of depth 9 1,515, now 431.  Up to FOREST_ALONE nodes it is
// still the faster (40 of depth 6: 22 us, 28 with two workgroups).
constexpr int64_t FOREST_NODES = 4096, FOREST_ALONE = 16384;
constexpr int MARK_PAST = PRED_MAP / 32, MARK_DONE = MARK_PAST + 1;
static_assert(PRED_MARK_WORDS == MARK_DONE + 1, "mark's layout");

__global__ __launch_bounds__(1024) void k_forest_features(const int32_t *__restrict__ feature,
                                                          int64_t nodes, uint32_t nodes_per_tree,
                                                          uint32_t *mark,
                                                          uint32_t *__restrict__ info) {
    __shared__ uint32_t used[PRED_MAP];
    __shared__ uint32_t tot[16];
    __shared__ uint32_t past, last;
    if (threadIdx.x == 0) past = 0;
    for (int k = threadIdx.x; k < PRED_MAP; k += 1024) used[k] = 0;
    __syncthreads();
    for (int64_t k = (int64_t)blockIdx.x * 1024 + threadIdx.x; k < nodes;
         k += (int64_t)gridDim.x * 1024) {
        const int32_t f = feature[k];
        if (f < 0) continue;
        const uint32_t n = (uint32_t)(k % nodes_per_tree);
        const int32_t *heap = feature + (k - n);
        int32_t above = 0;                             // negative: a leaf on the way
        for (uint32_t a = n; a > 0;) {
            a = (a - 1) >> 1;
            above |= heap[a];
        }
        if (above < 0) continue;
        if (f >= PRED_MAP) past = 1;
        else used[f] = 1;
    }
    __syncthreads();
    if (gridDim.x > 1) {
        if (threadIdx.x < PRED_MAP / 32) {
            uint32_t bits = 0;
            for (int k = 0; k < 32; ++k) bits |= used[threadIdx.x * 32 + k] << k;
            if (bits) atomicOr(&mark[threadIdx.x], bits);
        }
        if (threadIdx.x == 0 && past) atomicOr(&mark[MARK_PAST], 1u);
        __threadfence();
        __syncthreads();
        if (threadIdx.x == 0) last = atomicAdd(&mark[MARK_DONE], 1u) == gridDim.x - 1;
        __syncthreads();
        if (!last) return;
        __threadfence();
        if (threadIdx.x < PRED_MAP / 32) {
            const uint32_t bits = atomicExch(&mark[threadIdx.x], 0u);
            for (int k = 0; k < 32; ++k) used[threadIdx.x * 32 + k] = (bits >> k) & 1u;
        }
        if (threadIdx.x == 0) {
            past = atomicExch(&mark[MARK_PAST], 0u);
            atomicExch(&mark[MARK_DONE], 0u);
        }
        __syncthreads();
    }
    uint32_t u[4], mine = 0;                           // features 4 t .. 4 t + 3
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        u[q] = used[4 * threadIdx.x + q];
        mine += u[q];
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t incl = mine;
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t p = (uint32_t)__shfl_up((int)incl, o, 64);
        if (lane >= o) incl += p;
    }
    if (lane == 63) tot[wave] = incl;
    __syncthreads();
    uint32_t slot = incl - mine, total = 0;
    for (int w = 0; w < 16; ++w) {
        if (w < wave) slot += tot[w];
        total += tot[w];
    }
    if (threadIdx.x == 0) info[0] = past || total > (uint32_t)PRED_SLOTS ? 0xFFFFFFFFu : total;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        info[1 + PRED_SLOTS + 4 * threadIdx.x + q] = slot;
        if (u[q]) {
            if (slot < (uint32_t)PRED_SLOTS) info[1 + slot] = 4 * threadIdx.x + q;
            ++slot;
        }
    }
}

// Heap slot g of the forest as a walk reads it, the feature given by its slot
// when the rows' features are in LDS.
__device__ __forceinline__ PredNode pred_node(const ForestDev &f, int64_t g, bool in_lds,
                                              const uint32_t *info) {
    const int32_t feat = f.feature[g];
    if (feat < 0) return PredNode{f.leaf[g], -1};
    // (a slot under a leaf may hold a feature past the map)
    const int32_t slot = in_lds ? (int32_t)info[1 + PRED_SLOTS + min(feat, PRED_MAP - 1)] : feat;
    const int32_t flags = f.flags[g] & 3;
    // a categorical split without masks sends every row right
    if ((flags & FLAG_CATEGORICAL) && !f.mask) return PredNode{NAN, slot << 2};
    return PredNode{f.threshold[g], slot << 2 | flags};
}

__global__ __launch_bounds__(256) void k_forest_pack(ForestDev f, int64_t nodes,
                                                     const uint32_t *__restrict__ info,
                                                     int32_t max_slots,
                                                     PredNode *__restrict__ packed) {
    const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (g < nodes) packed[g] = pred_node(f, g, info && info[0] <= (uint32_t)max_slots, info);
}

hipError_t launch_forest_pack(hipStream_t s, const ForestDev &f, int32_t max_slots,
                              uint32_t *mark, uint32_t *info, PredNode *packed) {
    const int64_t nodes = (int64_t)f.num_trees * f.nodes_per_tree;
    const int64_t blocks = nodes <= FOREST_ALONE ? 1
                           : std::min<int64_t>((nodes + FOREST_NODES - 1) / FOREST_NODES, device_cus());
    if (info)
        hipLaunchKernelGGL(k_forest_features, dim3((unsigned)blocks), dim3(1024), 0, s, f.feature,
                           nodes, (uint32_t)f.nodes_per_tree, mark, info);
    if (packed && nodes > 0)
        hipLaunchKernelGGL(k_forest_pack, dim3((unsigned)((nodes + 255) / 256)), dim3(256), 0, s, f,
                           nodes, info, std::min(max_slots, PRED_SLOTS), packed);
    return hipGetLastError();
}

// CAT: the forest has category masks; DEEP: heaps of more than `stage` slots;
// X_LDS: the rows' features are in LDS.
template <bool CAT, bool DEEP, bool X_LDS>
__device__ __forceinline__ void predict_rows(PredNode *pred_lds, const ForestDev &f,
                                             const float *__restrict__ x, int64_t rows,
                                             int32_t data_bins, float base,
                                             float *__restrict__ out,
                                             const uint32_t *__restrict__ info,
                                             const PredNode *__restrict__ packed, int32_t chunk,
                                             int32_t stage, int32_t steps) {
    const int32_t npt = f.nodes_per_tree;
    PredNode *s_node = pred_lds;                                          // [chunk][stage]
    float *s_leaf = reinterpret_cast<float *>(s_node + (size_t)chunk * stage);   // [chunk][64]
    float *s_x = s_leaf + chunk * 64;                                     // [slots][64]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int32_t mine = f.tree_first < f.num_trees
                             ? (f.num_trees - f.tree_first + f.tree_step - 1) / f.tree_step : 0;
    for (int64_t row0 = (int64_t)blockIdx.x * 64; row0 < rows; row0 += (int64_t)gridDim.x * 64) {
        const int64_t past = rows - 1 - row0;              // rows past the end: the last row
        const uint32_t r = (int64_t)lane <= past ? (uint32_t)lane : (uint32_t)past;
        const float *xb = x + row0;
        if (X_LDS)
            for (uint32_t c = wave; c < info[0]; c += PRED_WAVES)
                s_x[c * 64 + lane] = xb[(int64_t)info[1 + c] * rows + r];
        float acc = base;                                  // seeded with the base, trees in order
        for (int32_t t0 = 0; t0 < mine; t0 += chunk) {
            const int32_t nt = min(chunk, mine - t0);
            auto heap = [&](int32_t t) {                   // chunk tree t's first node
                return (int64_t)(f.tree_first + (int64_t)(t0 + t) * f.tree_step) * npt;
            };
            auto load = [&](int64_t g) { return packed ? packed[g] : pred_node(f, g, X_LDS, info); };
            // a forest of one chunk stays for every tile of rows
            for (int32_t t = mine <= chunk && row0 >= (int64_t)gridDim.x * 64 ? nt : wave; t < nt;
                 t += PRED_WAVES) {
                const int64_t h = heap(t);
                for (int32_t n = lane; n < stage; n += 64) s_node[t * stage + n] = load(h + n);
            }
            __syncthreads();
            for (int32_t t = wave; t < nt; t += 2 * PRED_WAVES) {
                const int32_t t2 = t + PRED_WAVES < nt ? t + PRED_WAVES : t;
                const int32_t first[2] = {t * stage, t2 * stage};
                const int64_t h[2] = {heap(t), heap(t2)};
                int32_t n[2] = {0, 0};
                PredNode nd[2] = {s_node[first[0]], s_node[first[1]]};
                for (int32_t d = 0; d < steps; ++d) {
                    if (__ballot((nd[0].meta & nd[1].meta) >= 0) == 0) break;   // leaves everywhere
                    float v[2];
    #pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const int32_t slot = max(nd[j].meta, 0) >> 2;
                        v[j] = X_LDS ? s_x[slot * 64 + lane] : xb[(int64_t)slot * rows + r];
                    }
    #pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const uint32_t meta = (uint32_t)nd[j].meta;
                        const bool split = nd[j].meta >= 0;
                        bool left = (v[j] <= nd[j].value) | (isnan(v[j]) & ((meta & FLAG_DEFAULT_LEFT) != 0));
                        if (CAT && split && (meta & FLAG_CATEGORICAL))
                            left = raw_goes_left(v[j], FLAG_CATEGORICAL, 0.0f,
                                                 f.mask + (h[j] + n[j]) * 8, data_bins);
                        // a leaf stays where it is
                        n[j] = split ? 2 * n[j] + 2 - (int32_t)left : n[j];
                        if (!DEEP || n[j] < stage) nd[j] = s_node[first[j] + n[j]];
                        else if (split) nd[j] = load(h[j] + n[j]);
                    }
                }
                s_leaf[t * 64 + lane] = nd[0].value;
                s_leaf[t2 * 64 + lane] = nd[1].value;
            }
            __syncthreads();
            if (wave == 0) {
                int32_t t = 0;
                for (; t + 8 <= nt; t += 8) {
                    float v[8];
    #pragma unroll
                    for (int j = 0; j < 8; ++j) v[j] = s_leaf[(t + j) * 64 + lane];
    #pragma unroll
                    for (int j = 0; j < 8; ++j) acc += v[j];
                }
                for (; t < nt; ++t) acc += s_leaf[t * 64 + lane];
            }
        }
        if (wave == 0 && (int64_t)lane <= past) out[(row0 + lane) * f.out_stride] = acc;
    }
}

template <bool CAT, bool DEEP>
__global__ __launch_bounds__(PRED_THREADS) void k_predict_forest(
    ForestDev f, const float *__restrict__ x, int64_t rows, int32_t data_bins, float base,
    float *__restrict__ out, const uint32_t *__restrict__ info,
    const PredNode *__restrict__ packed, int32_t max_slots, int32_t chunk, int32_t stage,
    int32_t steps) {
    extern __shared__ PredNode pred_lds[];
    if (info && info[0] <= (uint32_t)max_slots)
        predict_rows<CAT, DEEP, true>(pred_lds, f, x, rows, data_bins, base, out, info, packed,
                                      chunk, stage, steps);
    else
        predict_rows<CAT, DEEP, false>(pred_lds, f, x, rows, data_bins, base, out, info, packed,
                                       chunk, stage, steps);
}

// The same walk by a thread per row, for few trees: no tile to stage and no barrier, a
// chain of dependent loads per tree that other rows' wavefronts hide.
template <bool PACKED>
__global__ __launch_bounds__(256) void k_predict_few(ForestDev f, const float *__restrict__ x,
                                                     int64_t rows, int32_t data_bins, float base,
                                                     float *__restrict__ out,
                                                     const uint32_t *__restrict__ info,
                                                     const PredNode *__restrict__ packed,
                                                     int32_t max_slots, int32_t steps) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= rows) return;
    const bool by_slot = PACKED && info && info[0] <= (uint32_t)max_slots;
    float acc = base;                                  // seeded with the base, trees in order
    for (int32_t t = f.tree_first; t < f.num_trees; t += f.tree_step) {
        const int64_t h = (int64_t)t * f.nodes_per_tree;
        int64_t g = h;
        PredNode nd{};
        auto load = [&] {
            if (PACKED) nd = packed[g];
            else nd.meta = f.feature[g];
        };
        load();
        for (int32_t d = 0; d < steps && nd.meta >= 0; ++d) {
            int64_t feat = PACKED ? nd.meta >> 2 : nd.meta;
            if (by_slot) feat = info[1 + feat];
            const uint32_t flags = PACKED ? (uint32_t)nd.meta & 3u : f.flags[g];
            const float thr = PACKED ? nd.value : f.threshold[g];
            const bool left = raw_goes_left(x[feat * rows + i], flags, thr,
                                            f.mask ? f.mask + g * 8 : nullptr, data_bins);
            g += g - h + (left ? 1 : 2);
            load();
        }
        acc += PACKED ? nd.value : nd.meta < 0 ? f.leaf[g] : f.threshold[g];
    }
    out[i * f.out_stride] = acc;
}

// Trees the walk takes, splits on the longest path of the heap, and heap slots of a
// tree that a tile stages: whole trees up to depth 7, the first seven levels of deeper
// ones (a chunk has to hold a tree for every wavefront).
static int32_t walked_trees(const ForestDev &f) {
    return std::max(1, (f.num_trees - f.tree_first + f.tree_step - 1) / f.tree_step);
}
static int32_t heap_steps(int32_t npt) {
    int32_t steps = 0;
    while (steps < 30 && (2 << steps) <= npt) ++steps;
    return steps;
}
static int32_t staged_slots(int32_t npt) { return npt <= 255 ? npt : 127; }
static int64_t staged_bytes(int32_t npt) {             // and a tree's values of a tile
    return staged_slots(npt) * (int64_t)sizeof(PredNode) + 64 * 4;
}

PredictRoute predict_route(const ForestDev &f, int64_t rows) {
    const int32_t npt = std::max(1, f.nodes_per_tree), trees = walked_trees(f);
    PredictRoute r{};
    // With fewer trees than a tile has wavefronts its time no longer falls with them (2M
    // rows of 100 columns, 1 / 10 / 15 / 20 trees of depth 6: 468 / 579 / 604 / 582 us), a
    // thread per row's does: 36 / 421 / 574 / 761.  But a row's trees x (splits + leaf) are
    // one chain of loads, which only many rows hide: 100k rows 8 / 51 us for 1 / 10 trees, in
    // tiles 20 / 33; 500k rows 13 / 94 and 96 / 122.  Even near 60 chain^2 rows: 5 trees
    // 50k, 8 200k, 12 400k, 12 stumps 50k, 36 stumps 250k (36 x 4 never).  Past depth 6 a
    // tile reads the deepest nodes from memory too: 6 trees of depth 9 even near 80k, 10
    // 400k, 3 of depth 12 20k.  One tree, or chains of 12, take no longer than a tile's
    // barriers at any rows: 1 row, 1 tree of depth 6 / 9 / 11 4.6 / 4.7 / 5.1 us, in tiles
    // 5.5 / 6.5 / 7.8; 3 of depth 3 4.6 and 5.2, of depth 4 5.3 and 5.3.
    const int64_t chain = (int64_t)trees * (1 + std::min(6, heap_steps(npt)));
    r.few = trees == 1 || chain <= 12 ||
            ((trees < PRED_WAVES || chain <= 80) && rows >= 60 * chain * chain);
    // Packed nodes are one load each.  They pay for their launch (3 us) where every tile
    // of rows reads them again: trees deeper than a tile stages, or more of them than it
    // stages at once.  100 trees of depth 9, 20k / 500k rows: 62 / 796 us, packed 56 /
    // 647; 300 of depth 6 79 / 1,216, packed 75 / 1,034; 100 of depth 6, staged once, 29 /
    // 313, packed 32 / 308.  Below 16k rows nothing gains.
    const bool once = npt == staged_slots(npt) && trees * staged_bytes(npt) <= LDS_BYTES;
    r.pack = !r.few && !once && rows >= 16384;
    // Features in LDS cost their columns' loads and save a load a step, which many trees
    // repay, and rows enough the listing: 100 columns, 100 / 300 / 1,000 trees of depth 6,
    // 500k rows 308 / 1,034 / 3,346 us without, 482 / 990 / 2,890 with them, 50k rows 53 /
    // 144 / 465 and 82 / 151 / 419.
    r.list = !r.few && trees >= 256 && rows * trees >= (int64_t)1 << 24;
    return r;
}

hipError_t launch_predict_forest(hipStream_t s, const ForestDev &f, const float *x, int64_t rows,
                                 int32_t data_bins, float base, float *out, const uint32_t *info,
                                 const PredNode *packed, int32_t max_slots) {
    if (rows <= 0) return hipSuccess;
    const int32_t slots = info ? std::max(0, std::min(max_slots, PRED_SLOTS)) : 0;
    const int32_t mine = walked_trees(f), npt = std::max(1, f.nodes_per_tree);
    const int32_t stage = staged_slots(npt), steps = heap_steps(npt);
    if (predict_route(f, rows).few) {
        auto *few = packed ? &k_predict_few<true> : &k_predict_few<false>;
        hipLaunchKernelGGL(few, dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, s, f, x, rows,
                           data_bins, base, out, info, packed, slots, steps);
        return hipGetLastError();
    }
    const int32_t x_bytes = slots * 64 * 4, tree_bytes = (int32_t)staged_bytes(npt);
    const bool whole = x_bytes + (int64_t)mine * tree_bytes <= LDS_BYTES;
    const int32_t budget = (x_bytes <= (40 << 10) ? 80 : 160) << 10;
    int32_t chunk = (budget - x_bytes) / tree_bytes;
    if (chunk > PRED_WAVES) chunk -= chunk % PRED_WAVES;   // whole rounds of the wavefronts
    chunk = whole ? mine : std::max(1, std::min(chunk, mine));
    const size_t lds = (size_t)chunk * tree_bytes + (size_t)x_bytes;
    const int64_t tiles = (rows + 63) / 64, resident = lds <= (80 << 10) ? 2 : 1;
    const int64_t grid = whole ? std::min(tiles, resident * device_cus()) : tiles;
    const bool deep = npt > stage;
    auto *kern = f.mask ? (deep ? &k_predict_forest<true, true> : &k_predict_forest<true, false>)
                        : (deep ? &k_predict_forest<false, true> : &k_predict_forest<false, false>);
    const hipError_t e = allow_all_lds(reinterpret_cast<const void *>(kern));
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(PRED_THREADS), lds, s, f, x,
                       rows, data_bins, base, out, info, packed, slots, chunk, stage, steps);
    return hipGetLastError();
}

// The walk over the training rows, up to eight rows per thread walked level by
// level together, that also counts the rows reaching each node of the deepest
// level (counters in LDS, one global add per non-empty node per block).  The
// split records (feature, bin | flags << 8) and leaf values are staged in LDS,
// so each level costs one global gather per row: the row's bin byte.
// With GRAD the walk also starts the next tree's gradient pass on the updated
// predictions: per-block maxima of |g| and h into gpart (as k_grad_max's
// partials) and, with g_out / h_out, every row's g and h.
// Rows per thread R and threads per block T go by the rows (walk_rows): R
// independent rows hide the levels' gathers where there are rows enough to fill
// the chip, but a few blocks of 8,192 rows each leave it idle (20k rows, depth 6:
// three blocks, 24.3 us; 79 blocks of 256 single rows, 6.8 us; 1M rows 35.3 -> 22.0
// us with 2 rows per thread, 2M 30.5 -> 26.4 with 4; 200k without gradients 27.9 ->
// 6.8 with 1).
constexpr int WALK_MAX_BLOCKS = 512;                   // two 1,024-thread blocks per CU

struct WalkGrad {
    GradParams gp;
    const float *labels;
    const float *weights;
    uint32_t *gpart;
    float *g_out, *h_out;
};

template <bool GRAD, int WALK_THREADS, int WALK_ROWS>
__global__ __launch_bounds__(WALK_THREADS, 8) void k_walk_count(const uint8_t *__restrict__ bins_fm,
                                                             int64_t rows, int32_t nb,
                                                             int32_t max_depth, TreeOut tree,
                                                             float *__restrict__ preds,
                                                             uint32_t *__restrict__ count,
                                                             const uint8_t *__restrict__ kept,
                                                             WalkGrad wg) {
    extern __shared__ uint32_t wc_lds[];
    const uint32_t deep = 1u << max_depth, deep_start = deep - 1;
    const uint32_t internal = deep - 1, total = 2 * deep - 1;
    uint32_t *s_cnt = wc_lds;                        // [deep]
    int32_t *s_feat = reinterpret_cast<int32_t *>(wc_lds + deep);    // [internal]
    uint32_t *s_bf = wc_lds + deep + internal;       // [internal] bin | flags << 8
    float *s_leaf = reinterpret_cast<float *>(wc_lds + deep + 2 * internal);   // [total]
    for (uint32_t k = threadIdx.x; k < deep; k += blockDim.x) s_cnt[k] = 0;
    for (uint32_t k = threadIdx.x; k < internal; k += blockDim.x) {
        const NodeSplit s = tree.split[k];
        s_feat[k] = s.feature;
        s_bf[k] = (s.bin & 0xFFu) | ((s.flags & 0xFFu) << 8);
    }
    for (uint32_t k = threadIdx.x; k < total; k += blockDim.x) s_leaf[k] = tree.leaf[k];
    __syncthreads();
    constexpr int64_t CHUNK = (int64_t)WALK_THREADS * WALK_ROWS;
    uint32_t mg = 0, mh = 0;
    for (int64_t c0 = (int64_t)blockIdx.x * CHUNK; c0 < rows; c0 += (int64_t)gridDim.x * CHUNK) {
        const int64_t base = c0 + threadIdx.x;
        uint32_t n[WALK_ROWS];
#pragma unroll
        for (int k = 0; k < WALK_ROWS; ++k) n[k] = 0;
        // which rows count, loaded up front with the first level's bins
        uint32_t counts = count ? (1u << WALK_ROWS) - 1u : 0u;
        if (count && kept) {
#pragma unroll
            for (int k = 0; k < WALK_ROWS; ++k) {
                const int64_t i = base + (int64_t)k * WALK_THREADS;
                if (i < rows && !kept[i]) counts &= ~(1u << k);
            }
        }
        // few rows per thread: their predictions and labels load before the walk
        constexpr bool EARLY = WALK_ROWS <= 2;
        float early_p[WALK_ROWS], early_y[WALK_ROWS];
        if (EARLY && preds) {
#pragma unroll
            for (int k = 0; k < WALK_ROWS; ++k) {
                const int64_t i = base + (int64_t)k * WALK_THREADS;
                early_p[k] = i < rows ? preds[i] : 0.0f;
                early_y[k] = GRAD && i < rows ? wg.labels[i] : 0.0f;
            }
        }
        for (int32_t d = 0; d < max_depth; ++d) {
            uint32_t b[WALK_ROWS];
#pragma unroll
            for (int k = 0; k < WALK_ROWS; ++k) {
                const int64_t i = base + (int64_t)k * WALK_THREADS;
                const int32_t f = n[k] < internal ? s_feat[n[k]] : -1;
                b[k] = (i < rows && f >= 0) ? bins_fm[(int64_t)f * rows + i] : 0xFFFFFFFFu;
            }
#pragma unroll
            for (int k = 0; k < WALK_ROWS; ++k) {
                if (b[k] == 0xFFFFFFFFu) continue;   // past the end, or at a leaf
                const uint32_t bf = s_bf[n[k]], bin = bf & 0xFFu, flags = bf >> 8;
                bool left;
                if (flags & FLAG_CATEGORICAL)
                    left = ((tree.mask[n[k] * 8 + (b[k] >> 5)] >> (b[k] & 31u)) & 1u) != 0;
                else if (b[k] == (uint32_t)(nb - 1)) left = (flags & FLAG_DEFAULT_LEFT) != 0;
                else left = b[k] <= bin;
                n[k] = 2 * n[k] + 1 + (left ? 0 : 1);
            }
        }
#pragma unroll
        for (int k = 0; k < WALK_ROWS; ++k) {
            const int64_t i = base + (int64_t)k * WALK_THREADS;
            if (i >= rows) continue;
            if (preds) {                             // null: counts only
                const float np = (EARLY ? early_p[k] : preds[i]) + s_leaf[n[k]];
                preds[i] = np;
                if (GRAD) {
                    float g, h;
                    const float w = wg.gp.has_weights ? wg.weights[i] : 1.0f;
                    row_grad(wg.gp, np, EARLY ? early_y[k] : wg.labels[i], w, g, h);
                    mg = max(mg, __float_as_uint(fabsf(g)));
                    mh = max(mh, __float_as_uint(h));
                    if (wg.g_out) { wg.g_out[i] = g; wg.h_out[i] = h; }
                }
            }
            if (((counts >> k) & 1u) && n[k] >= deep_start) atomicAdd(&s_cnt[n[k] - deep_start], 1u);
        }
    }
    if (GRAD) {
        __shared__ uint32_t red[2][WALK_THREADS / 64];
        for (int o = 32; o > 0; o >>= 1) {
            mg = max(mg, (uint32_t)__shfl_xor((int)mg, o, 64));
            mh = max(mh, (uint32_t)__shfl_xor((int)mh, o, 64));
        }
        if ((threadIdx.x & 63) == 0) { red[0][threadIdx.x >> 6] = mg; red[1][threadIdx.x >> 6] = mh; }
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t a = red[0][0], b = red[1][0];
            for (int k = 1; k < WALK_THREADS / 64; ++k) { a = max(a, red[0][k]); b = max(b, red[1][k]); }
            wg.gpart[2 * blockIdx.x] = a;
            wg.gpart[2 * blockIdx.x + 1] = b;
        }
    }
    if (!count) return;                              // null: predictions only
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < deep; k += blockDim.x)
        if (s_cnt[k]) atomicAdd(&count[deep_start + k], s_cnt[k]);
}

// Launches the walk with the rows per thread that fill 512 blocks (or, below
// 131,072 rows, with single rows in 256-thread blocks); returns the grid.
template <bool GRAD>
static hipError_t walk_rows(hipStream_t s, const uint8_t *bins_fm, int64_t rows, int32_t num_bins,
                            int32_t max_depth, const TreeOut &tree, float *preds, uint32_t *count,
                            const uint8_t *kept, const WalkGrad &wg, int *blocks) {
    const size_t deep = (size_t)1 << max_depth;
    const size_t lds = (deep + 2 * (deep - 1) + (2 * deep - 1)) * sizeof(uint32_t);
    int64_t grid = 0;
#define MBK_WALK(T, R)                                                                           \
    {                                                                                            \
        grid = std::min<int64_t>((rows + (T) * (R) - 1) / ((T) * (R)), WALK_MAX_BLOCKS);         \
        auto *kern = &k_walk_count<GRAD, T, R>;                                                  \
        hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(T), lds, s, bins_fm, rows, num_bins, \
                           max_depth, tree, preds, count, kept, wg);                             \
    }
    if (rows <= 256 * WALK_MAX_BLOCKS) MBK_WALK(256, 1)
    else if (rows <= 1024 * WALK_MAX_BLOCKS) MBK_WALK(1024, 1)
    else if (rows <= 2048 * WALK_MAX_BLOCKS) MBK_WALK(1024, 2)
    else if (rows <= 4096 * WALK_MAX_BLOCKS) MBK_WALK(1024, 4)
    else MBK_WALK(1024, 8)
#undef MBK_WALK
    *blocks = (int)grid;
    return hipGetLastError();
}

hipError_t launch_walk_count(hipStream_t s, const uint8_t *bins_fm, int64_t rows,
                             int32_t num_bins, int32_t max_depth, const TreeOut tree,
                             float *preds, uint32_t *count, const uint8_t *kept) {
    if (rows <= 0) return hipSuccess;
    int blocks = 0;
    return walk_rows<false>(s, bins_fm, rows, num_bins, max_depth, tree, preds, count, kept,
                            WalkGrad{}, &blocks);
}

hipError_t launch_walk_count_grad(hipStream_t s, const uint8_t *bins_fm, int64_t rows,
                                  int32_t num_bins, int32_t max_depth, const TreeOut tree,
                                  float *preds, uint32_t *count, const uint8_t *kept,
                                  const GradParams &gp, const float *labels,
                                  const float *weights, uint32_t *gpart, float *g_out,
                                  float *h_out, int *partials) {
    *partials = 0;
    if (rows <= 0 || !preds) return hipErrorInvalidValue;
    if (gp.objective == 7) return hipErrorInvalidValue;   // one output per row only
    return walk_rows<true>(s, bins_fm, rows, num_bins, max_depth, tree, preds, count, kept,
                           WalkGrad{gp, labels, weights, gpart, g_out, h_out}, partials);
}

// Binned single-tree prediction (predict_tree_binned, Shaders.swift:1763-1781):
// the same walk with the tree staged in LDS, without counts.
hipError_t launch_predict_binned(hipStream_t s, const uint8_t *bins_fm, int64_t rows,
                                 int32_t num_bins, int32_t max_depth, const TreeOut tree,
                                 float *preds) {
    return launch_walk_count(s, bins_fm, rows, num_bins, max_depth, tree, preds, nullptr, nullptr);
}

// ---------------------------------------------------------------------------
// validation metric (evalMetricRaw, Booster.swift:1855-1918): each block's double
// sum of the rows' terms; the host adds the blocks in order, so the value does not
// depend on timing.  Reading the predictions back and summing them on one host
// thread left the GPU idle for 0.2 ms after every tree of a 200k-row validation
// set; this takes 4.7 us and no wait.
// ---------------------------------------------------------------------------

constexpr int METRIC_THREADS = 256;
constexpr int METRIC_BLOCKS = 256;                     // at most, a row per thread below

__device__ __forceinline__ double metric_term(int metric, double p, double y, double param) {
    switch (metric) {
    case METRIC_RMSE: return (p - y) * (p - y);
    case METRIC_MAE: return fabs(p - y);
    case METRIC_PINBALL: {
        const double d = y - p;
        return d >= 0 ? param * d : (param - 1) * d;
    }
    case METRIC_LOGLOSS: {
        const double q = 1 / (1 + exp(-p));
        const double a = q < 1e-12 ? 1e-12 : q, b = 1 - q < 1e-12 ? 1e-12 : 1 - q;   // NaN stays
        return -(y * log(a) + (1 - y) * log(b));
    }
    case METRIC_POISSON: {
        const double mu = exp(p);
        return 2 * ((y > 0 ? y * log(y / mu) : 0) - (y - mu));
    }
    default: {                                         // Tweedie, param = rho
        const double mu = exp(p);
        const double a = y > 0 ? pow(y, 2 - param) / ((1 - param) * (2 - param)) : 0;
        return 2 * (a - y * pow(mu, 1 - param) / (1 - param) + pow(mu, 2 - param) / (2 - param));
    }
    }
}

__global__ __launch_bounds__(METRIC_THREADS) void k_metric(int metric, double param, int32_t K,
                                                           const float *__restrict__ preds,
                                                           const float *__restrict__ labels,
                                                           int64_t rows,
                                                           double *__restrict__ partial) {
    __shared__ double red[METRIC_THREADS / 64];
    double sum = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * METRIC_THREADS + threadIdx.x; i < rows;
         i += (int64_t)gridDim.x * METRIC_THREADS) {
        if (metric == METRIC_MULTI_LOGLOSS) {          // class k's scores at preds[k * rows]
            double m = -INFINITY, e = 0.0;
            for (int k = 0; k < K; ++k) m = fmax(m, (double)preds[(int64_t)k * rows + i]);
            for (int k = 0; k < K; ++k) e += exp((double)preds[(int64_t)k * rows + i] - m);
            sum -= (double)preds[(int64_t)(int)labels[i] * rows + i] - m - log(e);
        } else {
            sum += metric_term(metric, (double)preds[i], (double)labels[i], param);
        }
    }
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < METRIC_THREADS / 64; ++k) sum += red[k];
        partial[blockIdx.x] = sum;
    }
}

int metric_blocks(int64_t rows) {
    return (int)std::max<int64_t>(
        1, std::min<int64_t>((rows + METRIC_THREADS - 1) / METRIC_THREADS, METRIC_BLOCKS));
}

hipError_t launch_metric(hipStream_t s, int metric, double param, int32_t num_classes,
                         const float *preds, const float *labels, int64_t rows,
                         double *partial) {
    if (rows <= 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_metric, dim3((unsigned)metric_blocks(rows)), dim3(METRIC_THREADS), 0, s,
                       metric, param, num_classes, preds, labels, rows, partial);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// TreeSHAP
// ---------------------------------------------------------------------------

constexpr int SHAP_MAX_U = 12;                         // maxDepth <= 12

// Lane-per-row TreeSHAP for wide data (more columns than k_treeshap_rows
// keeps in LDS): every lane walks all paths for its row, phi in a global
// [blocks][cols][64] fp64 scratch.
__global__ __launch_bounds__(64) void k_treeshap(const float *__restrict__ x, int64_t rows,
                                                 int32_t cols, int32_t data_bins,
                                                 const uint32_t *__restrict__ masks,
                                                 const ShapPath *__restrict__ paths,
                                                 int32_t num_paths,
                                                 const ShapElem *__restrict__ elems,
                                                 const ShapUniq *__restrict__ uniq, float bias,
                                                 float *__restrict__ out,
                                                 double *__restrict__ phi_global) {
    const int lane = threadIdx.x;
    const int64_t i = (int64_t)blockIdx.x * 64 + lane;
    const bool valid = i < rows;
    const int64_t irow = valid ? i : 0;
    double *phi = phi_global + (int64_t)blockIdx.x * 64 * cols;   // this block's [cols][64]
    for (int f = 0; f < cols; ++f) phi[f * 64 + lane] = 0.0;
    for (int32_t p = 0; p < num_paths; ++p) {
        const ShapPath P = paths[p];
        double one[SHAP_MAX_U], zero[SHAP_MAX_U];
        int feat[SHAP_MAX_U];
#pragma unroll
        for (int u = 0; u < SHAP_MAX_U; ++u) {
            one[u] = 1.0;
            zero[u] = 1.0;
            feat[u] = 0;
            if (u < P.num_uniq) {
                const ShapUniq q = uniq[P.uniq_start + u];
                zero[u] = q.zero;
                feat[u] = q.feature;
            }
        }
        for (int e = 0; e < P.num_elem; ++e) {
            const ShapElem el = elems[P.elem_start + e];
            const float v = x[(int64_t)el.feature * rows + irow];
            const bool left = raw_goes_left(v, el.flags, el.threshold,
                                            masks ? masks + (int64_t)el.node * 8 : nullptr,
                                            data_bins);
            const double o = (left == ((el.flags & 0x100u) != 0)) ? 1.0 : 0.0;
#pragma unroll
            for (int u = 0; u < SHAP_MAX_U; ++u)
                if (u == el.uniq) one[u] *= o;
        }
        const int U = P.num_uniq;
        // EXTEND with the dummy element at index 0 (SHAP.swift:266-279)
        double pw[SHAP_MAX_U + 1];
        pw[0] = 1.0;
#pragma unroll
        for (int j = 1; j <= SHAP_MAX_U; ++j) {
            pw[j] = 0.0;
            if (j <= U) {
                const double o = one[j - 1], z = zero[j - 1];
#pragma unroll
                for (int q = j - 1; q >= 0; --q) {
                    pw[q + 1] += o * pw[q] * (double)(q + 1) / (double)(j + 1);
                    pw[q] = z * pw[q] * (double)(j - q) / (double)(j + 1);
                }
            }
        }
        // unwound sums per unique feature (SHAP.swift:307-325)
#pragma unroll
        for (int u = 0; u < SHAP_MAX_U; ++u) {
            if (u < U) {
                const double o = one[u], z = zero[u];
                double total = 0.0;
                if (o != 0.0) {
                    double next = 0.0;
#pragma unroll
                    for (int q = SHAP_MAX_U; q >= 0; --q)
                        if (q == U) next = pw[q];
#pragma unroll
                    for (int q = SHAP_MAX_U - 1; q >= 0; --q) {
                        if (q < U) {
                            const double tmp = next / ((double)(q + 1) * o);
                            total += tmp;
                            next = pw[q] - tmp * z * (double)(U - q);
                        }
                    }
                } else if (z != 0.0) {
#pragma unroll
                    for (int q = SHAP_MAX_U - 1; q >= 0; --q)
                        if (q < U) total += pw[q] / (z * (double)(U - q));
                }
                const double contrib = total * (double)(U + 1) * (o - z) * P.leaf;
                phi[feat[u] * 64 + lane] += contrib;
            }
        }
    }
    if (!valid) return;
    float *orow = out + i * (int64_t)(cols + 1);
    for (int f = 0; f < cols; ++f) orow[f] = (float)phi[f * 64 + lane];
    orow[cols] = bias;
}

// The contributions of one root-to-leaf path with U unique features: zero[u] is
// feature u's unfollowed share (1 for u >= U), bit u of ones says that the row
// follows every split of feature u on the path.  emit(u, contribution), u = 0 ..
// U - 1.
template <int MAXU, typename Emit>
__device__ __forceinline__ void path_contributions(int U, const double (&zero)[MAXU],
                                                   uint32_t ones, double leaf, Emit emit) {
    double one[MAXU];
#pragma unroll
    for (int u = 0; u < MAXU; ++u) one[u] = ((ones >> u) & 1u) ? 1.0 : 0.0;
    // EXTEND with the dummy element at index 0 (SHAP.swift:266-279).  The
    // weights (q+1)/(j+1) and (j-q)/(j+1) are compile-time constants here,
    // one multiply each instead of a multiply and a divide (a rounding
    // apart from the divided form).
    double pw[MAXU + 1];
    pw[0] = 1.0;
#pragma unroll
    for (int j = 1; j <= MAXU; ++j) {
        pw[j] = 0.0;
        if (j <= U) {
            const double o = one[j - 1], z = zero[j - 1];
#pragma unroll
            for (int q = j - 1; q >= 0; --q) {
                const double up = (double)(q + 1) / (double)(j + 1);
                const double down = (double)(j - q) / (double)(j + 1);
                pw[q + 1] += o * pw[q] * up;
                pw[q] = z * pw[q] * down;
            }
        }
    }
    // 1 / (U - q) for q < U: U divisions per path, shared by every
    // unique feature's unwinding
    double inv_uq[MAXU];
#pragma unroll
    for (int q = 0; q < MAXU; ++q) inv_uq[q] = q < U ? 1.0 / (double)(U - q) : 0.0;
    // unwound sums per unique feature (SHAP.swift:307-325).  one[u] is 0
    // or 1, so the o != 0 form divides by the constant q + 1 (a multiply
    // by its reciprocal here) and the o == 0 form by z (U - q) (one 1/z
    // per feature).  Both forms share one loop: a wavefront's lanes take
    // both.
#pragma unroll
    for (int u = 0; u < MAXU; ++u) {
        if (u < U) {
            const double o = one[u], z = zero[u];
            const bool on = o != 0.0, live = on || z != 0.0;
            const double inv_z = (!on && z != 0.0) ? 1.0 / z : 0.0;
            double total = 0.0;
            double next = 0.0;
#pragma unroll
            for (int q = MAXU; q >= 0; --q)
                if (q == U) next = pw[q];
#pragma unroll
            for (int q = MAXU - 1; q >= 0; --q) {
                if (q < U) {
                    const double rq = 1.0 / (double)(q + 1);
                    const double tmp = on ? next * rq
                                          : (live ? pw[q] * inv_z * inv_uq[q] : 0.0);
                    total += tmp;
                    if (on) next = pw[q] - tmp * z * (double)(U - q);
                }
            }
            emit(u, total * (double)(U + 1) * (o - z) * leaf);
        }
    }
}

// Path-parallel TreeSHAP: one wavefront per row (grid-stride), one lane per
// root-to-leaf path, 64 paths per pass.  The row's feature values and its phi
// sit in LDS; each lane runs the same fp64 EXTEND/UNWIND as k_treeshap for its
// path and adds its unique features' contributions to phi with ds_add_f64.
// One wavefront owns a row's phi, so the order of the adds is fixed (pass
// order, then the LDS unit's lane order) and the output is deterministic.
template <int MAXU>
__global__ __launch_bounds__(64) void k_treeshap_rows(const float *__restrict__ x, int64_t rows,
                                                      int32_t cols, int32_t data_bins,
                                                      const uint32_t *__restrict__ masks,
                                                      const ShapPath *__restrict__ paths,
                                                      int32_t num_paths,
                                                      const ShapElem *__restrict__ elems,
                                                      const ShapUniq *__restrict__ uniq,
                                                      float bias, float *__restrict__ out) {
    extern __shared__ double row_lds[];                // phi [cols], then x [cols] as f32
    double *phi = row_lds;
    float *xr = reinterpret_cast<float *>(row_lds + cols);
    const int lane = threadIdx.x;
    for (int64_t i = blockIdx.x; i < rows; i += gridDim.x) {
        for (int f = lane; f < cols; f += 64) {
            xr[f] = x[(int64_t)f * rows + i];
            phi[f] = 0.0;
        }
        __syncthreads();
        for (int32_t c = 0; c < num_paths; c += 64) {
            const int32_t p = c + lane;
            if (p >= num_paths) continue;
            const ShapPath P = paths[p];
            const int U = P.num_uniq;
            // one[u] is a product of 0/1 indicators: held as bit u of `ones`
            double zero[MAXU];
            int feat[MAXU];
#pragma unroll
            for (int u = 0; u < MAXU; ++u) {
                zero[u] = 1.0;
                feat[u] = 0;
                if (u < U) {
                    const ShapUniq q = uniq[P.uniq_start + u];
                    zero[u] = q.zero;
                    feat[u] = q.feature;
                }
            }
            uint32_t ones = (1u << MAXU) - 1u;
#pragma unroll
            for (int e = 0; e < MAXU; ++e) {
                if (e >= P.num_elem) break;
                const ShapElem el = elems[P.elem_start + e];
                const bool left = raw_goes_left(xr[el.feature], el.flags, el.threshold,
                                                masks ? masks + (int64_t)el.node * 8 : nullptr,
                                                data_bins);
                if (left != ((el.flags & 0x100u) != 0)) ones &= ~(1u << el.uniq);
            }
            path_contributions<MAXU>(U, zero, ones, P.leaf, [&](int u, double v) {
                atomicAdd(&phi[feat[u]], v);
            });
        }
        __syncthreads();
        float *orow = out + i * (int64_t)(cols + 1);
        for (int f = lane; f < cols; f += 64) orow[f] = (float)phi[f];
        if (lane == 0) orow[cols] = bias;
        __syncthreads();                               // before the next row reuses the LDS
    }
}

// ---- TreeSHAP from contribution tables -------------------------------------
//
// A path's contributions depend on the row only through which of its splits the
// row follows, so they are computed once per outcome instead of once per row.
// Paths are grouped by the lowest ancestors whose subtree holds at most two
// levels of splits (four leaves): a group's outcome is one bit per feature
// among its root's ancestors and one per split inside (7 bits at depth 6), and
// its leaves' contributions to a feature are summed into one column of 2^bits
// doubles.  Four launches:
//   k_shap_tables    the columns (EXTEND/UNWIND once per group and outcome)
//   k_shap_patterns  every row's outcome per group
//   k_shap_sum       per row and feature the sum of its columns' entries
//   k_shap_finish    the runs of k_shap_sum added up, in f32, row-major
// Two levels per group: one level (leaf pairs) needs 192 lookups per row and
// depth-6 tree, two 112, three 80 out of tables 6 times the size that no longer
// stream through LDS.  200k rows x 100 trees of depth 6: 36.4 ms with a path
// evaluation per row, now 1.1 ms (outcomes 0.62, sums 0.35, finish 0.11, tables 0.03).

constexpr int SHAP_LDS_DOUBLES = 4096;                 // one batch of columns
constexpr int SHAP_THREADS = SHAP_BLOCK_ROWS / 4;      // four rows per thread

// The contributions of a group's leaf position q to the group's columns, for an
// outcome: emit(column, contribution), each column at most once.
template <int MAXU, typename Emit>
__device__ __forceinline__ void leaf_contributions(const ShapGroup &g,
                                                   const double *__restrict__ vals, int q,
                                                   uint32_t pattern, Emit emit) {
    const double *anc = vals + g.val_start, *share = anc + g.anc;
    double zero[MAXU];
    int col[MAXU];
    uint32_t ones = pattern & ((1u << g.anc) - 1u);
#pragma unroll
    for (int u = 0; u < MAXU; ++u) {
        zero[u] = u < g.anc ? anc[u] : 1.0;
        col[u] = u;
    }
    int slots = g.anc;
    // the splits inside on this leaf's path: the root, then a child
    const double *sh = share;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const uint32_t in = g.inside[k];
        if (in == 0) continue;
        const double left = sh[0], right = sh[1];
        sh += 2;
        if (k > 0 && (q >> 1) != k - 1) continue;
        const bool go_left = k == 0 ? q < 2 : (q & 1) == 0;
        const bool follows = (((pattern >> ((in >> 8) & 0xFFu)) & 1u) != 0) == go_left;
        const int c = (int)(in & 0xFFu);
        int at = slots;
#pragma unroll
        for (int u = 0; u < MAXU; ++u)
            if (u < slots && col[u] == c) at = u;
#pragma unroll
        for (int u = 0; u < MAXU; ++u) {
            if (u == at) {
                zero[u] *= go_left ? left : right;
                col[u] = c;
            }
        }
        if (at == slots) {
            ones |= 1u << at;
            ++slots;
        }
        if (!follows) ones &= ~(1u << at);
    }
    path_contributions<MAXU>(slots, zero, ones, vals[g.leaf_start + q], [&](int u, double v) {
        emit(col[u], v);
    });
}

// One workgroup of one wavefront per (group, 64 outcomes): a lane per outcome
// walks the group's leaves; sums per column in LDS (a lane's own slots), then
// stored coalesced.  Bound by fp64 arithmetic, but 128 outcomes per group
// stand for any number of rows (100 trees of depth 6: 0.8M path evaluations
// against 1280M for 200k rows).
template <int MAXU>
__global__ __launch_bounds__(64) void k_shap_tables(const ShapGroup *__restrict__ groups,
                                                    const double *__restrict__ vals,
                                                    const uint32_t *__restrict__ col_off,
                                                    double *__restrict__ table) {
    __shared__ double acc[SHAP_MAX_COLS][64];
    const ShapGroup g = groups[blockIdx.x];
    const uint32_t first = blockIdx.y * 64u;
    if (first >= (1u << g.bits)) return;
    const int lane = threadIdx.x;
    const uint32_t pattern = first + (uint32_t)lane;
    for (int c = 0; c < g.num_cols; ++c) acc[c][lane] = 0.0;
    for (int q = 0; q < 4; ++q)
        if ((g.leaves >> q) & 1u)
            leaf_contributions<MAXU>(g, vals, q, pattern, [&](int c, double v) { acc[c][lane] += v; });
    if (pattern < (1u << g.bits))
        for (int c = 0; c < g.num_cols; ++c)
            table[(size_t)col_off[g.col_start + c] + pattern] = acc[c][lane];
}

template <typename PT> struct ShapPack;                // four rows' outcomes
template <> struct ShapPack<uint8_t> {
    uint32_t w;
    __device__ __forceinline__ void set(const uint32_t (&p)[4]) {
        w = p[0] | (p[1] << 8) | (p[2] << 16) | (p[3] << 24);
    }
    __device__ __forceinline__ uint32_t get(int k) const { return (w >> (8 * k)) & 0xFFu; }
};
template <> struct ShapPack<uint16_t> {
    uint32_t w[2];
    __device__ __forceinline__ void set(const uint32_t (&p)[4]) {
        w[0] = p[0] | (p[1] << 16);
        w[1] = p[2] | (p[3] << 16);
    }
    __device__ __forceinline__ uint32_t get(int k) const {
        return (w[k >> 1] >> (16 * (k & 1))) & 0xFFFFu;
    }
};

// Outcomes of SHAP_BLOCK_ROWS rows x per_block groups per workgroup; a lane holds rows
// lane, lane + 64, + 128, + 192 of its wavefront's 256, so the feature loads are
// coalesced (the split is the same for every lane: its column is a scalar
// address) and its four outcomes are one packed store.  Bound by the
// instructions per row and split: with the split's flags scalar, a numeric one is
// a single compare (v > thr where missing goes left, v <= thr where not; NaN
// fails both) and the bit's conditional set (200k rows x 1,600 groups: 755 us,
// 1,640 us with the general form for every split, 615 us once small launches
// were spread over more workgroups).
template <typename PT>
__global__ __launch_bounds__(SHAP_THREADS) void k_shap_patterns(
    const float *__restrict__ x, int64_t rows, int64_t row0, int32_t data_bins,
    const uint32_t *__restrict__ masks, const ShapGroup *__restrict__ groups, int32_t num_groups,
    const ShapTest *__restrict__ tests, int32_t per_block,
    ShapPack<PT> *__restrict__ out, size_t pitch) {
    const int64_t base = row0 + (int64_t)blockIdx.x * SHAP_BLOCK_ROWS;
    const int64_t past = rows - 1 - base;              // rows past the end: the last row
    uint32_t r[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t i = (threadIdx.x >> 6) * 256 + (threadIdx.x & 63) + 64 * k;
        r[k] = (int64_t)i <= past ? i : (uint32_t)past;
    }
    const float *xb = x + base;
    const int g0 = blockIdx.y * per_block, g1 = min(num_groups, g0 + per_block);
    for (int gi = g0; gi < g1; ++gi) {
        const ShapGroup g = groups[gi];
        uint32_t fail[4] = {0, 0, 0, 0};
        // four tests at a time: one 64-B scalar load, 16 feature loads in flight
        for (int t = 0; t < g.num_tests; t += 4) {
            ShapTest T[4];
            float v[4][4];
#pragma unroll
            for (int j = 0; j < 4; ++j) T[j] = tests[g.test_start + t + j];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float *col = xb + (int64_t)T[j].feature * rows;
#pragma unroll
                for (int k = 0; k < 4; ++k) v[j][k] = col[r[k]];
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t flags = T[j].flags, bit = 1u << (flags >> 16);
                const bool when_left = (flags & 0x100u) != 0;
                if (flags & FLAG_CATEGORICAL) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const bool left = raw_goes_left(
                            v[j][k], flags & 0xFFu, T[j].threshold,
                            masks ? masks + (int64_t)T[j].node * 8 : nullptr, data_bins);
                        if (left != when_left) fail[k] |= bit;
                    }
                } else if (flags & FLAG_DEFAULT_LEFT) {
                    const uint32_t above = when_left ? bit : 0u, rest = bit ^ above;
#pragma unroll
                    for (int k = 0; k < 4; ++k) fail[k] |= v[j][k] > T[j].threshold ? above : rest;
                } else {
                    const uint32_t rest = when_left ? bit : 0u, within = bit ^ rest;
#pragma unroll
                    for (int k = 0; k < 4; ++k) fail[k] |= v[j][k] <= T[j].threshold ? within : rest;
                }
            }
        }
        uint32_t pat[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) pat[k] = ~fail[k] & ((1u << g.bits) - 1u);
        ShapPack<PT> w;
        w.set(pat);
        out[(size_t)gi * pitch + (size_t)blockIdx.x * SHAP_THREADS + threadIdx.x] = w;
    }
}

// One workgroup per (SHAP_BLOCK_ROWS rows, share of the batches).  Items (one column of
// one group) are ordered by feature; a batch's columns are contiguous and go
// through LDS, where 64 lanes look up their outcomes.  A lane's four rows sum in
// registers until the feature ends or the share does (a run), then the run's
// sums are stored: no atomics, so the order is fixed.  Bound by the random
// 8-byte LDS reads (depth 6: 2.2G of them for 200k rows x 100 trees in 349 us; 459 with
// fewer shares) and, for long columns, by their loads: 20k rows x 50 trees of depth 8
// took 405 us with 1,024 rows per workgroup and 231 to 249 us with 2,048.
template <typename PT>
__global__ __launch_bounds__(SHAP_THREADS) void k_shap_sum(const ShapItem *__restrict__ items,
                                                  const ShapBatch *__restrict__ batches,
                                                  int32_t num_batches,
                                                  const double *__restrict__ table,
                                                  const ShapPack<PT> *__restrict__ patterns,
                                                  size_t pitch, double *__restrict__ runs,
                                                  size_t run_pitch) {
    __shared__ double2 cols2[SHAP_LDS_DOUBLES / 2];
    double *cols = reinterpret_cast<double *>(cols2);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int b0 = (int)((int64_t)num_batches * blockIdx.y / gridDim.y);
    const int b1 = (int)((int64_t)num_batches * (blockIdx.y + 1) / gridDim.y);
    const ShapPack<PT> *pat = patterns + (size_t)blockIdx.x * SHAP_THREADS + threadIdx.x;
    double *dst = runs + (size_t)blockIdx.x * SHAP_BLOCK_ROWS + wave * 256 + lane;
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    for (int b = b0; b < b1; ++b) {
        const ShapBatch B = batches[b];
        __syncthreads();                               // the last batch's lookups are done
        const double2 *src = reinterpret_cast<const double2 *>(table + B.table_off);
        for (uint32_t k = threadIdx.x; k < B.table_len / 2; k += SHAP_THREADS) cols2[k] = src[k];
        __syncthreads();
        const ShapItem *it = items + B.item_start;
        for (int i = 0; i < B.num_items; i += 4) {
            ShapPack<PT> w[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (i + j < B.num_items) w[j] = pat[(size_t)it[i + j].group * pitch];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (i + j >= B.num_items) break;
                const uint32_t off = it[i + j].offset_run & 0xFFFu, run = it[i + j].offset_run >> 12;
#pragma unroll
                for (int k = 0; k < 4; ++k) acc[k] += cols[off + w[j].get(k)];
                if (run != 0) {
                    double *d = dst + (size_t)(run - 1) * run_pitch;
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        d[64 * k] = acc[k];
                        acc[k] = 0.0;
                    }
                }
            }
        }
    }
}

// Adds up each feature's runs (and, with several table sets, the sums of the
// earlier ones: total, [cols][total_rows] f64), 64 rows x 64 features per workgroup
// through an LDS transpose; the last set writes f32 rows and the bias.
__global__ __launch_bounds__(256) void k_shap_finish(const double *__restrict__ runs,
                                                     size_t run_pitch,
                                                     const uint32_t *__restrict__ run_first,
                                                     int64_t row0, int64_t rows, int32_t cols,
                                                     double *__restrict__ total,
                                                     int64_t total_row0, int64_t total_rows,
                                                     int first, int last, float bias,
                                                     float *__restrict__ out) {
    __shared__ float tile[64][65];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t r0 = row0 + (int64_t)blockIdx.x * 64;
    const int f0 = blockIdx.y * 64;
    const int nf = min(64, cols - f0);
    const int64_t row = r0 + lane;
    for (int f = wave; f < nf; f += 4) {
        double v = 0.0;
        double *sum = total + (size_t)(f0 + f) * (size_t)total_rows + (size_t)(row - total_row0);
        if (!first && row < rows) v = *sum;
        for (uint32_t k = run_first[f0 + f]; k < run_first[f0 + f + 1]; ++k)
            v += runs[(size_t)k * run_pitch + (size_t)(row - row0)];
        if (!last) {
            if (row < rows) *sum = v;
        } else {
            tile[lane][f] = (float)v;
        }
    }
    if (!last) return;
    __syncthreads();
    const int64_t nr = rows - r0 < 64 ? rows - r0 : 64;
    for (int q = wave; q < nr; q += 4) {
        float *o = out + (r0 + q) * (int64_t)(cols + 1);
        if (lane < nf) o[f0 + lane] = tile[q][lane];
        if (lane == 0 && f0 + 64 >= cols) o[cols] = bias;
    }
}

// Few rows: the same sums, to the last bit, without tables.  100 trees of depth 6, one row
// 210 us a call with tables, 126 so.  Two launches:
//   k_shap_entries    every row's entries of the columns, by its own outcome per group
//   k_shap_entry_sums per row the runs of k_shap_sum, then their sums as k_shap_finish's
// A row costs a path evaluation per leaf where the tables cost 2^bits of them for all
// rows, so it takes over while rows are fewer than a share of that (few_rows in shap.cpp).

// One workgroup per (group, 64 rows), a row per lane: wavefront w checks every fourth
// quad of the group's tests, then takes leaf position w; the leaves' contributions
// to a column are added in their order (a leaf without the column adds 0, which
// changes no sum).  Bound by the latency of one fp64 path evaluation.
template <int MAXU>
__global__ __launch_bounds__(256) void k_shap_entries(ShapRows a, ShapSetDev d, int32_t max_cols) {
    extern __shared__ double s_part[];                 // [4][max_cols][64]
    __shared__ uint32_t s_fail[4][64];
    const ShapGroup g = d.groups[blockIdx.x];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double *part = s_part + lane;
    auto slot = [&](int leaf, int c) { return (leaf * max_cols + c) * 64; };
    const int64_t local = (int64_t)blockIdx.y * 64 + lane;
    const int64_t r = a.row0 + (local < a.num_rows ? local : a.num_rows - 1);
    uint32_t fail = 0;
    for (int t = wave * 4; t < g.num_tests; t += 16) {  // padded to whole quads
        ShapTest T[4];
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) T[j] = d.tests[g.test_start + t + j];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = a.x[(int64_t)T[j].feature * a.rows + r];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t flags = T[j].flags;
            const bool left = raw_goes_left(v[j], flags & 0xFFu, T[j].threshold,
                                            a.masks ? a.masks + (int64_t)T[j].node * 8 : nullptr,
                                            a.data_bins);
            if (left != ((flags & 0x100u) != 0)) fail |= 1u << (flags >> 16);
        }
    }
    s_fail[wave][lane] = fail;
    for (int c = 0; c < g.num_cols; ++c) part[slot(wave, c)] = 0.0;
    __syncthreads();
    const uint32_t pattern = ~(s_fail[0][lane] | s_fail[1][lane] | s_fail[2][lane] | s_fail[3][lane]) &
                             ((1u << g.bits) - 1u);
    const int q = __builtin_amdgcn_readfirstlane(wave);
    if ((g.leaves >> q) & 1u)
        leaf_contributions<MAXU>(g, d.vals, q, pattern,
                                 [&](int c, double v) { part[slot(q, c)] = v; });
    __syncthreads();
    if (local >= a.num_rows) return;
    for (int c = wave; c < g.num_cols; c += 4) {
        double sum = 0.0;
#pragma unroll
        for (int k = 0; k < 4; ++k) sum += part[slot(k, c)];
        a.entries[(size_t)d.col_at[g.col_start + c] * (size_t)a.num_rows + (size_t)local] = sum;
    }
}

// One workgroup per a.tile rows (a power of two): a thread per run and row, then per
// feature and row.  Bound by the longest run's chain of adds.
constexpr int SHAP_SUM_THREADS = 256;
__global__ __launch_bounds__(SHAP_SUM_THREADS) void k_shap_entry_sums(ShapRows a, ShapSetDev d,
                                                                      int32_t num_runs) {
    extern __shared__ double s_run[];                  // [num_runs][tile]
    const int64_t first = (int64_t)blockIdx.x * a.tile;
    const uint32_t n = (uint32_t)num_runs * (uint32_t)a.tile;
    for (uint32_t k = threadIdx.x; k < n; k += SHAP_SUM_THREADS) {
        const uint32_t run = k / (uint32_t)a.tile;
        const int64_t local = first + (k & (uint32_t)(a.tile - 1));
        const double *src = a.entries + (size_t)(local < a.num_rows ? local : a.num_rows - 1);
        const uint32_t i1 = d.run_item[run + 1];
        uint32_t i = d.run_item[run];
        double sum = 0.0;
        for (; i + 8 <= i1; i += 8) {
            double v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = src[(size_t)(i + j) * (size_t)a.num_rows];
#pragma unroll
            for (int j = 0; j < 8; ++j) sum += v[j];
        }
        for (; i < i1; ++i) sum += src[(size_t)i * (size_t)a.num_rows];
        s_run[k] = sum;
    }
    __syncthreads();
    const int32_t live = (int32_t)(a.num_rows - first < a.tile ? a.num_rows - first : a.tile);
    for (int32_t k = threadIdx.x; k < live * a.cols; k += SHAP_SUM_THREADS) {
        const int32_t t = k / a.cols, f = k - t * a.cols;
        double *total = a.total + (size_t)f * (size_t)a.num_rows + (size_t)(first + t);
        double v = 0.0;
        if (!a.first) v = *total;
        for (uint32_t run = d.run_first[f]; run < d.run_first[f + 1]; ++run)
            v += s_run[run * (uint32_t)a.tile + (uint32_t)t];
        if (!a.last) {
            *total = v;
            continue;
        }
        float *o = a.out + (a.row0 + first + t) * (int64_t)(a.cols + 1);
        o[f] = (float)v;
        if (f == 0) o[a.cols] = a.bias;
    }
}

hipError_t launch_shap_rows(hipStream_t s, const ShapSet &set, const ShapSetDev &d,
                            const ShapRows &w) {
    if (w.num_rows <= 0 || w.num_rows > (int64_t)65535 * 64 || set.num_runs > SHAP_FEW_RUNS ||
        set.max_bits > SHAP_MAX_BITS || (!(w.first && w.last) && !w.total))
        return hipErrorInvalidValue;
    ShapRows a = w;
    a.tile = 1;
    while (a.tile < 8 && a.tile < w.num_rows && 2 * a.tile * set.num_runs <= SHAP_FEW_RUNS) a.tile *= 2;
    const dim3 grid((unsigned)set.num_groups, (unsigned)((w.num_rows + 63) / 64));
    // a group's features: its longest path's and one more split inside
    const int32_t max_cols = std::min(set.max_slots + 1, SHAP_MAX_COLS);
#define MBK_SHAP_ENTRIES(U)                                                                    \
    hipLaunchKernelGGL(k_shap_entries<U>, grid, dim3(256),                                     \
                       (size_t)max_cols * 4 * 64 * sizeof(double), s, a, d, max_cols)
    if (set.num_groups > 0) {
        if (set.max_slots <= 4) MBK_SHAP_ENTRIES(4);
        else if (set.max_slots <= 6) MBK_SHAP_ENTRIES(6);
        else if (set.max_slots <= 8) MBK_SHAP_ENTRIES(8);
        else MBK_SHAP_ENTRIES(SHAP_MAX_U);
    }
#undef MBK_SHAP_ENTRIES
    hipLaunchKernelGGL(k_shap_entry_sums, dim3((unsigned)((w.num_rows + a.tile - 1) / a.tile)),
                       dim3(SHAP_SUM_THREADS), (size_t)set.num_runs * (size_t)a.tile * sizeof(double),
                       s, a, d, set.num_runs);
    return hipGetLastError();
}

hipError_t launch_shap_tables(hipStream_t s, const ShapSet &set, const ShapSetDev &d,
                              double *table) {
    if (set.num_groups == 0) return hipSuccess;
    const dim3 grid((unsigned)set.num_groups, (unsigned)((((size_t)1 << set.max_bits) + 63) / 64));
#define MBK_SHAP_TABLES(U)                                                                      \
    hipLaunchKernelGGL(k_shap_tables<U>, grid, dim3(64), 0, s, d.groups, d.vals, d.col_off, table)
    if (set.max_slots <= 4) MBK_SHAP_TABLES(4);
    else if (set.max_slots <= 6) MBK_SHAP_TABLES(6);
    else if (set.max_slots <= 8) MBK_SHAP_TABLES(8);
    else MBK_SHAP_TABLES(SHAP_MAX_U);
#undef MBK_SHAP_TABLES
    return hipGetLastError();
}

template <typename PT>
static hipError_t shap_slab(hipStream_t s, const ShapSet &set, const ShapSetDev &d,
                            const ShapSlab &w) {
    const unsigned blocks = (unsigned)(w.slab_rows / SHAP_BLOCK_ROWS);
    const size_t pitch = (size_t)w.slab_rows / 4;
    ShapPack<PT> *pat = reinterpret_cast<ShapPack<PT> *>(w.patterns);
    if (set.num_groups > 0) {
        // a group is a chain of scalar and feature loads: at least 2,048
        // workgroups (eight per CU) hide it, at most 64 groups each
        const int64_t per = std::max<int64_t>(1, (int64_t)set.num_groups * blocks / 2048);
        const int32_t per_block = (int32_t)std::min<int64_t>(per, 64);
        hipLaunchKernelGGL(k_shap_patterns<PT>,
                           dim3(blocks, (unsigned)((set.num_groups + per_block - 1) / per_block)),
                           dim3(SHAP_THREADS), 0, s, w.x, w.rows, w.row0, w.data_bins, w.masks, d.groups,
                           set.num_groups, d.tests, per_block, pat, pitch);
        hipLaunchKernelGGL(k_shap_sum<PT>, dim3(blocks, (unsigned)set.shares),
                           dim3(SHAP_THREADS), 0, s,
                           d.items, d.batches, set.num_batches, w.table, pat, pitch, w.runs,
                           (size_t)w.slab_rows);
    }
    const int64_t live = std::min<int64_t>(w.slab_rows, w.rows - w.row0);
    hipLaunchKernelGGL(k_shap_finish, dim3((unsigned)((live + 63) / 64), (unsigned)((w.cols + 63) / 64)),
                       dim3(256), 0, s, w.runs, (size_t)w.slab_rows, d.run_first, w.row0, w.rows,
                       w.cols, w.total, w.total_row0, w.total_rows, w.first, w.last, w.bias, w.out);
    return hipGetLastError();
}

hipError_t launch_shap_slab(hipStream_t s, const ShapSet &set, const ShapSetDev &d,
                            const ShapSlab &w) {
    if (w.rows <= 0 || w.slab_rows <= 0 || w.slab_rows % SHAP_BLOCK_ROWS != 0 ||
        set.max_bits > SHAP_MAX_BITS || set.shares < 1 || set.shares > 65535 ||
        (!(w.first && w.last) && !w.total))
        return hipErrorInvalidValue;
    return set.max_bits > 8 ? shap_slab<uint16_t>(s, set, d, w) : shap_slab<uint8_t>(s, set, d, w);
}

// Columns up to which k_treeshap_rows runs (12 B of LDS per column).
constexpr int SHAP_ROW_MAX_COLS = 4096;

bool treeshap_needs_scratch(int cols) { return cols > SHAP_ROW_MAX_COLS; }

hipError_t launch_treeshap(hipStream_t s, const float *x, int64_t rows, int32_t cols,
                           int32_t data_bins, const uint32_t *masks, const ShapPath *paths,
                           int32_t num_paths, int32_t max_elems, const ShapElem *elems,
                           const ShapUniq *uniq, float bias, float *out, double *phi_global) {
    if (rows <= 0) return hipSuccess;
    if (max_elems < 1 || max_elems > SHAP_MAX_U) return hipErrorInvalidValue;
    if (!treeshap_needs_scratch(cols)) {
        // the per-lane path arrays sized to the longest path: fewer registers,
        // more wavefronts per SIMD
        const unsigned blocks = (unsigned)std::min<int64_t>(rows, (int64_t)1 << 22);
        const size_t lds = (size_t)cols * (sizeof(double) + sizeof(float));
#define MBK_SHAP_ROWS(U)                                                                        \
        hipLaunchKernelGGL(k_treeshap_rows<U>, dim3(blocks), dim3(64), lds, s, x, rows, cols,   \
                           data_bins, masks, paths, num_paths, elems, uniq, bias, out)
        if (max_elems <= 4) MBK_SHAP_ROWS(4);
        else if (max_elems <= 6) MBK_SHAP_ROWS(6);
        else if (max_elems <= 8) MBK_SHAP_ROWS(8);
        else MBK_SHAP_ROWS(SHAP_MAX_U);
#undef MBK_SHAP_ROWS
        return hipGetLastError();
    }
    if (!phi_global) return hipErrorInvalidValue;      // wide data: phi in the caller's scratch
    const unsigned blocks = (unsigned)((rows + 63) / 64);
    hipLaunchKernelGGL(k_treeshap, dim3(blocks), dim3(64), 0, s, x, rows, cols, data_bins, masks,
                       paths, num_paths, elems, uniq, bias, out, phi_global);
    return hipGetLastError();
}


}  // namespace mbk
