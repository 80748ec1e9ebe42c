// orb_batched.hip -- the batched (device-driven) ORB build.
//
// The plain form asks the host after every bisection pass.  Here the whole
// build runs on the device with no host round trip:
//
//  * the cell heap lives in HBM; the level schedule (which heap ids a level
//    bisects) depends only on d, so the host computes it once;
//  * every cell of a level is bisected in the same launches.  One streaming
//    pass over a cell's keys bins each key against the 255 candidate cuts of
//    the next 8 bisection steps (the midpoints the serial loop could visit,
//    computed with the same float arithmetic).  The candidates are sorted, so
//    prefix sums of the 256-bin histogram give count(x < c) (or <= c) at
//    every candidate, and a replay kernel walks the reference's termination
//    rule over them: 8 passes of src/orbit.cpp:149-231 per HBM read, bit-exact
//    by construction.  Four rounds cover the 32-pass cap;
//  * a cell of at most 8832 keys (7680 with ids, 5120 with weights) is
//    handed to a subtree kernel: one 1024-thread block loads its x, y, z
//    into LDS once, runs every remaining level of the cell's subtree there
//    (the same 8-pass histogram rounds and replay, exact Hoare by ballot
//    scans) and writes x, y, z back once;
//  * the partition of the remaining (large) cells uses the same exact Hoare
//    kernels as the plain form;
//  * which kernels a level launches follows from the cell sizes the host
//    expects (level_kernels): one block a cell with the keys in registers
//    (k_b_cell), few chunks (k_m_*, k_mw_*), a cut predicted from a sample
//    (k_p_*), the chunk kernels of every size otherwise.
#include "orb_device.hpp"

namespace orb {

constexpr int kRounds = (ORB_MAX_PASSES + kHistK - 1) / kHistK;  // 4
// Leaves under a subtree root (the subtree kernel's key capacity is SubCap).
constexpr int kSmallLeaves = 64;
constexpr int kReduceRows = 64;                // chunk histograms per reduce block

struct BatchedState {
    int32_t d = 0, levels_mode = -1;
    int64_t cap = 0;
    int32_t D = 0;
    bool complete = true;              // every level lists all its splittable cells
    std::vector<int32_t> level_n;      // [D+1] cells per level (index l)
    std::vector<uint8_t> level_cover;  // [D+1] the level's cells hold every particle
    std::vector<int64_t> level_off;    // [D+1] offset into level_ids
    std::vector<int32_t> level_min_leaf;  // [D+1] fewest leaves under a cell of the level
    DevBuf<LevelEntry> level_ids;      // all levels' cells, concatenated
    DevBuf<orb_cell> heap;             // [cap]
    DevBuf<uint8_t> exists;            // [cap]
    DevBuf<uint8_t> sub;               // [cap] cell handled inside a subtree kernel
    DevBuf<uint16_t> chunk_hist;       // [max_chunks][256]
    DevBuf<uint32_t> cell_hist;        // cell_hist_words
    DevBuf<uint64_t> chunk_hist_w;     // weighted builds: [max_chunks][256] weight sums
    DevBuf<uint64_t> cell_hist_w;      // weighted builds: [max_level_cells][256]
    bool hist_w_clean = false;         // cell_hist_w all zero (as cell_hist)
    bool sample_clean = false;         // sample_hist all zero (as cell_hist)
    DevBuf<uint64_t> trace;            // [cap][32]
    DevBuf<int32_t> level_passes;      // [64]
    PinBuf<int32_t> hpasses;           // [64]
    // captured build: valid while its signature (graph_signature) holds
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    std::vector<uint64_t> gsig;
    // cell_hist rows are added to by k_b_hist_reduce and consumed and
    // re-zeroed by k_b_replay in the same round, so the buffer is all zero
    // between builds; it is cleared after allocation and after a failure
    bool hist_clean = false;
};

// The previous level's due row swaps as a kernel argument (nCells = 0:
// none).
struct PendingFinalDev {
    const LevelEntry *entries;
    int32_t nCells;
    const SplitRec *splits;
    float *x, *y, *z;
    uint32_t *pid, *w;
};

// ---------------------------------------------------------------------------
// schedule (host): ids per level, data-independent
// ---------------------------------------------------------------------------
int schedule_levels(int32_t d, int32_t levels_mode, int64_t cap,
                    std::vector<std::vector<int32_t>> &levels, bool *complete,
                    std::vector<int32_t> *min_leaf)
{
    // existence and nLeafCells follow from d alone (left = ceil(n/2),
    // right = n - left), so the schedule needs no particle data
    const int32_t D = n_levels(d);
    std::vector<uint8_t> ex((size_t)cap, 0);
    std::vector<orb_cell> hp((size_t)cap);
    std::memset(hp.data(), 0, sizeof(orb_cell) * hp.size());
    hp[0].nLeafCells = d;
    ex[0] = 1;
    std::vector<int32_t> ids;
    levels.assign((size_t)D + 1, {});
    if (min_leaf) min_leaf->assign((size_t)D + 2, 0);
    *complete = true;
    for (int32_t l = 1; l <= D; ++l) {
        int32_t bad = -1;
        if (!level_cells(d, levels_mode, l, ex, hp, ids, &bad)) return ORB_ERR_UB;
        if (levels_mode == ORB_LEVELS_REFERENCE && l >= D) break;
        // the subtree kernel needs every cell of depth l-1 with >= 2 leaves
        int64_t a = (int64_t(1) << (l - 1)) - 1, e = (int64_t(1) << l) - 2;
        int32_t expect = 0;
        for (int64_t id = a; id <= e; ++id)
            if (ex[(size_t)id] && hp[(size_t)id].nLeafCells >= 2) expect++;
        if (expect != (int32_t)ids.size()) *complete = false;
        for (int32_t id : ids) {
            int32_t nl = hp[(size_t)id].nLeafCells;
            if (min_leaf && ((*min_leaf)[(size_t)l] == 0 || nl < (*min_leaf)[(size_t)l]))
                (*min_leaf)[(size_t)l] = nl;
            int32_t left = (nl + 1) / 2;
            int32_t lid = left_child_id(id), rid = right_child_id(id);
            if (rid >= cap) return ORB_ERR_ARG;
            hp[(size_t)lid].nLeafCells = left;
            hp[(size_t)rid].nLeafCells = nl - left;
            ex[(size_t)lid] = ex[(size_t)rid] = 1;
        }
        levels[(size_t)l] = ids;
    }
    return ORB_OK;
}

static int make_schedule(Ctx &c, BatchedState &b, int32_t levels_mode, bool *complete)
{
    b.d = c.d;
    b.levels_mode = levels_mode;
    b.cap = c.cap;
    b.D = n_levels(c.d);
    std::vector<std::vector<int32_t>> levels;
    ORB_TRY(schedule_levels(c.d, levels_mode, c.cap, levels, complete, &b.level_min_leaf));
    const int32_t lmax = levels_mode == ORB_LEVELS_REFERENCE ? b.D - 1 : b.D;
    std::vector<LevelEntry> all;
    b.level_n.assign((size_t)b.D + 2, 0);
    b.level_off.assign((size_t)b.D + 2, 0);
    b.level_cover.assign((size_t)b.D + 2, 0);
    for (int32_t l = 1; l < (int32_t)levels.size(); ++l) {
        b.level_off[(size_t)l] = (int64_t)all.size();
        b.level_n[(size_t)l] = (int32_t)levels[(size_t)l].size();
        // every particle sits in a cell of depth l-1 while each earlier level
        // split all cells of its depth
        const int32_t expect = l == 1 ? 1 : 2 * b.level_n[(size_t)l - 1];
        b.level_cover[(size_t)l] = (l == 1 || b.level_cover[(size_t)l - 1]) &&
                                   b.level_n[(size_t)l] == expect;
        for (int32_t id : levels[(size_t)l])
            all.push_back(LevelEntry{id, 0, (int32_t)c.cap, l, 0, lmax, *complete ? 1 : 0, 0});
    }
    ORB_TRY(b.level_ids.alloc(all.size() + 1));
    if (!all.empty())
        ORB_HIP(hipMemcpy(b.level_ids.p, all.data(), sizeof(LevelEntry) * all.size(),
                          hipMemcpyHostToDevice));
    return ORB_OK;
}

// ---------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------
// Fresh build state: root cell, empty heap and flags, range(0) = [0, n),
// cleared status and pass counters (no memset or host copy: graph-safe).
__global__ void k_b_init(orb_cell *heap, uint8_t *exists, uint8_t *sub, int64_t cap,
                         orb_cell root, uint64_t *trace, int64_t trace_n, int32_t *level_passes,
                         uint32_t *ranges, uint32_t n, int32_t *status)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t k = i; k < cap; k += stride) {
        ranges[2 * k] = 0u;
        ranges[2 * k + 1] = k == 0 ? n : 0u;
        store_root_or_zero(&heap[k], root, k == 0);
        exists[k] = k == 0 ? 1 : 0;
        sub[k] = 0;
    }
    for (int64_t k = i; k < trace_n; k += stride) trace[k] = ~0ull;
    if (i < 64) level_passes[i] = 0;
    if (i < 2) status[i] = 0;
}

// End of a build: its status pair and pass counters into pinned memory (two
// copy commands less).
__global__ void k_b_done(const int32_t *status, const int32_t *level_passes, int32_t *hstatus,
                         int32_t *hpasses)
{
    const int t = threadIdx.x;
    hpasses[t] = level_passes[t];
    if (t < 2) hstatus[t] = status[t];
}

// Which kernels a level's launches hold, for its cell records: cells of at
// most sub_max keys (and kSmallLeaves leaves) go to the subtree kernel, cells
// of at most cell_max keys to k_b_cell (0: not launched), cells of at most
// chunk_max keys to the chunk kernels.  A level whose kernels do not take
// every size, or after which the build ends (both chosen from the sizes the
// host expects), leaves a larger cell alone and counts it in the build's pass
// counter 0; the host then runs the levels again with the chunk path (again =
// 1), which skips the cells that are split already.
struct LevelMode {
    uint32_t sub_max, cell_max, chunk_max;
    int32_t again;
};
constexpr int kFlagBlock = 3;  // CellRec.flags: the cell goes to k_b_cell

// Level record of entry i from the device heap (cells inside a finished
// subtree, and cells that a left-alone ancestor has not made yet, are
// skipped); returns its chunk count.
__device__ inline uint32_t level_rec(const LevelEntry *entries, int32_t i, const orb_cell *heap,
                                     const uint8_t *exists, const uint32_t *ranges,
                                     const uint8_t *sub, const LevelMode mode, CellRec *recs,
                                     int32_t *level_passes)
{
    const LevelEntry en = entries[i];
    const int32_t id = en.id;
    const int64_t g = (int64_t)en.hb + id;
    const orb_cell cl = heap[g];
    CellRec r;
    r.begin = ranges[2 * g];
    r.end = ranges[2 * g + 1];
    if (r.end < r.begin) r.end = r.begin;
    r.cut = cell_get_cut(cl);
    r.axis = cl.cutAxis;
    r.found = 0;
    r.nLeaf = cl.nLeafCells;
    r.margin_l = cl.cutMarginLeft;
    r.margin_r = cl.cutMarginRight;
    r.id = id;
    r.passes = 0;
    r.hb = en.hb;
    r.capr = en.capr;
    r.lp = en.lp;
    r.st = en.st;
    r.lmax = en.lmax;
    const uint32_t n = r.end - r.begin;
    const int64_t gl = (int64_t)en.hb + left_child_id(id);
    if (sub[g] || !exists[g] || (mode.again && exists[gl])) {
        r.flags = 1;
    } else if (mode.sub_max && en.sub_ok && n <= mode.sub_max && cl.nLeafCells <= kSmallLeaves) {
        r.flags = 2;
    } else if (mode.cell_max && n <= mode.cell_max && !en.last) {
        r.flags = kFlagBlock;
    } else if (n <= mode.chunk_max && !en.last) {
        r.flags = 0;
    } else {
        r.flags = 1;
        atomicAdd(&level_passes[en.lp & ~63], 1);
    }
    recs[i] = r;
    return r.flags ? 0u : (n + (uint32_t)kChunk - 1u) / (uint32_t)kChunk;
}

// The previous level's last Hoare row swaps, from blocks [fb0, gridDim.x) of
// a level's first launch: cell c's rows from its range in the map and its
// split (the cell records are being rewritten by the other blocks).
__device__ inline void level_finals(uint32_t fb0, const PendingFinalDev &fin,
                                    const uint32_t *ranges)
{
    const int32_t c = (int32_t)((blockIdx.x - fb0) * blockDim.x + threadIdx.x);
    if (c >= fin.nCells) return;
    const LevelEntry en = fin.entries[c];
    const int64_t g = (int64_t)en.hb + en.id;
    hoare_final_rows(ranges[2 * g], ranges[2 * g + 1], fin.splits[c], fin.x, fin.y, fin.z, fin.pid,
                     fin.w);
}

__global__ void k_b_recs(const LevelEntry *entries, int32_t nCells, const orb_cell *heap,
                         const uint8_t *exists, const uint32_t *ranges, const uint8_t *sub,
                         LevelMode mode, CellRec *recs, uint32_t *nchunks, int32_t *level_passes,
                         uint32_t rec_blocks, PendingFinalDev fin)
{
    if (blockIdx.x >= rec_blocks) {  // uniform
        level_finals(rec_blocks, fin, ranges);
        return;
    }
    int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i > nCells) return;
    nchunks[i] = i == nCells ? 0u
                             : level_rec(entries, i, heap, exists, ranges, sub, mode, recs, level_passes);
}

// A level of fewer than kRecsScan cells in one block of kRecsScan threads,
// a cell per thread: the cell records and the exclusive scan of their chunk
// counts into first[] (first[nCells] = the level's chunks), in place of a
// record launch and a scan launch.  kFill (levels of few chunks): the block
// also fills the chunk records and clears the cells' key counters.
template <bool kFill>
__global__ __launch_bounds__(kRecsScan) void k_b_recs_scan(
    const LevelEntry *__restrict__ entries, int32_t nCells, const orb_cell *__restrict__ heap,
    const uint8_t *__restrict__ exists, const uint32_t *__restrict__ ranges,
    const uint8_t *__restrict__ sub, LevelMode mode, CellRec *recs,
    uint32_t *__restrict__ first, int32_t *__restrict__ level_passes, uint4 *chunk_desc,
    uint32_t max_chunks, unsigned long long *sel_lists, PendingFinalDev fin)
{
    if (blockIdx.x > 0) {  // uniform: the previous level's row swaps
        level_finals(1u, fin, ranges);
        return;
    }
    constexpr int kW = kRecsScan / 64;
    __shared__ uint32_t wsum[kW];
    __shared__ uint32_t s_first[kFill ? kRecsScan : 1], s_begin[kFill ? kRecsScan : 1];
    __shared__ uint32_t s_end[kFill ? kRecsScan : 1];
    __shared__ int32_t s_axis[kFill ? kRecsScan : 1];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const uint32_t v =
        t < nCells ? level_rec(entries, t, heap, exists, ranges, sub, mode, recs, level_passes) : 0u;
    const uint32_t inc = wave_inclusive_scan(v);
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    uint32_t pre = 0;
    for (int i = 0; i < w; ++i) pre += wsum[i];
    if (t <= nCells) first[t] = pre + inc - v;  // t = nCells: the level's chunk count
    if constexpr (kFill) {
        if (t <= nCells) s_first[t] = pre + inc - v;
        if (t < nCells) {
            const CellRec &r = recs[t];  // this thread's own
            s_begin[t] = r.begin;
            s_end[t] = r.end;
            s_axis[t] = r.axis >= 0 && r.axis <= 2 ? r.axis : (int32_t)kChunkIdle;
            if (v) sel_lists[pre + inc - v] = 0ull;
        }
        __syncthreads();
        uint32_t total = s_first[nCells];
        if (total > max_chunks) total = max_chunks;
        for (uint32_t q = (uint32_t)t; q < total; q += kRecsScan) {
            // every chunk of the table is searched (other cells have none)
            const uint32_t cell = chunk_to_cell(s_first, nCells, q);
            const uint32_t cb = s_begin[cell] + (q - s_first[cell]) * (uint32_t)kChunk, ce = s_end[cell];
            chunk_desc[q] = make_uint4(cb, ce - cb < (uint32_t)kChunk ? ce : cb + (uint32_t)kChunk,
                                       cell, (uint32_t)s_axis[cell]);
        }
    }
}

// in-order index t in [1, 255] of the depth-8 candidate tree on [lo, hi]
__device__ inline float candidate(int t, float lo, float hi)
{
    int node = kBins / 2, step = kBins / 4;
    while (node != t) {
        float m = cell_cut(lo, hi);
        if (t < node) {
            hi = m;
            node -= step;
        } else {
            lo = m;
            node += step;
        }
        step >>= 1;
    }
    return cell_cut(lo, hi);
}

// Exact bin of key v in [lo, hi] among the 255 candidate cuts of the next 8
// bisection steps, without a table: the walk down the candidate tree
// computes each midpoint with the cut arithmetic (cell.h:74-76) and counts
// the candidates at or below v (LE = 0) or below v (LE = 1).  The
// candidates are sorted, so a node that qualifies takes its whole left
// subtree with it.
template <int LE>
__device__ inline int bin_walk(float v, float lo, float hi)
{
    int e = 0;
#pragma unroll
    for (int d = 0; d < kHistK; ++d) {
        const float m = cell_cut(lo, hi);
        const bool right = LE ? (m < v) : (m <= v);
        if (right) {
            e += 1 << (kHistK - 1 - d);
            lo = m;
        } else {
            hi = m;
        }
    }
    return e;
}

// Bin of key v among the sorted candidates cand[1..255] (cand[0] = -inf,
// cand[256] = +inf): the number of candidates <= v (LE = 0) or < v (LE = 1).
// The candidates sit close to lo + j*(hi-lo)/256, so the arithmetic estimate
// is checked against its two neighbours (one pair of LDS reads); an estimate
// that misses (rounding at a bin edge, or a window a few ulps wide) takes the
// eight steps of the exact walk.  (Stepping along the table instead took up to
// 255 reads a key where candidates are equal, which is where keys tie: 2^26
// keys on 256 values, <=, root level 7.26 ms, now 1.21.)
template <int LE>
__device__ inline int bin_of(const float *cand, float v, float lo, float hi, float scale, int &tie)
{
    const float ef = fminf(fmaxf((v - lo) * scale, 0.0f), (float)(kBins - 1));
    int e = (int)ef;
    const float c0 = cand[e], c1 = cand[e + 1];
    const bool ok = LE ? (c0 < v && v <= c1) : (c0 <= v && v < c1);
    if (__builtin_expect(!ok, 0)) e = bin_walk<LE>(v, lo, hi);
    // the candidate v equals, if any: cand[e] (<) or cand[e + 1] (<=)
    tie = LE ? (cand[e + 1] == v ? e + 1 : 0) : (cand[e] == v ? e : 0);
    return e;
}

// How far (in bins) the estimate (v - lo) * scale must stay from both edges
// of its bin for that bin to be exact without the table.  With
// M = max(|lo|, |hi|): a candidate is at most 8 float midpoints deep, each
// midpoint of values in [lo, hi] off the exact one by at most 2^-24 M (the
// sum's rounding) plus 2^-150 (a halving into the subnormals), so candidate
// j sits within 2^-21 M + 2^-147 of lo + j (hi - lo) / 256, i.e. within
// (2^-21 M + 2^-147) * scale (1 + 3 * 2^-24) bins of j.  The estimate itself
// carries four roundings (v - lo, hi - lo, 256 / width, the product), at
// most 2^-14 bins anywhere in [0, 256].  The returned bound doubles both
// terms; M >= 2^126 (sums that could overflow) returns 1: never trusted.
__device__ inline float bin_tolerance(float lo, float hi, float scale)
{
    const float m = fmaxf(fabsf(lo), fabsf(hi));
    return m < 0x1p126f ? 0x1p-13f + (m + 0x1p-120f) * (0x1p-20f * scale) : 1.0f;
}

// Bin e of key v in [lo, hi] when the estimate lies more than tol from both
// edges of [e, e + 1) (lim = 0.5 - tol: the fraction's distance from 0.5 is
// below lim): candidate e is then strictly below v and candidate e + 1
// strictly above, so e is the bin for both comparisons and v ties no
// candidate.  False when the table has to decide (NaN estimates included).
// An estimate at or past 256 needs no test of its own: v <= hi keeps it
// within 2^-14 of 256, too close to that edge to pass.
__device__ inline bool bin_estimate(float v, float lo, float scale, float lim, int &e)
{
    const float ef = (v - lo) * scale;
    e = (int)ef;
    return fabsf(__builtin_amdgcn_fractf(ef) - 0.5f) < lim;
}

// The candidate table of a cell into LDS, with the -inf / +inf sentinels
// at 0 and kBins: each thread loads its entry (cand_entry, issued before the
// chunk's keys so that waiting for it does not wait for them), then stores it.
__device__ inline float cand_entry(const float *cell_cand, uint32_t cell)
{
    const int t = threadIdx.x;
    return t ? cell_cand[(size_t)cell * kBins + t] : -INFINITY;
}
__device__ inline void store_cands(float *cand, float entry)
{
    const int t = threadIdx.x;
    cand[t] = entry;
    if (t == 0) cand[kBins] = INFINITY;
}

// The keys of a chunk (record dd) that wave w reads, 16 loads of 64
// consecutive keys, through a range-checked descriptor: loads past the
// chunk's end return 0.  A chunk that is not live (past the level's count,
// or of a cell that is not searched) gets an empty range: its loads return
// 0 and touch no memory.
template <int kPerWave>
__device__ inline void issue_chunk_loads(const float *x, const float *y, const float *z, bool live,
                                         uint4 dd, uint32_t sb, int lane, float (&vv)[kPerWave])
{
    const uint32_t ax = uniform(dd.w), b = uniform(dd.x), e = uniform(dd.y);
    const float *kp = axis_ptr(x, y, z, live ? (int)ax : 0) + (live ? b : 0u);
    const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(kp), 0, live ? (int)((e - b) * 4u) : 0, 0x00020000);
    // the whole offset in the per-lane operand: the range check covers it,
    // not the scalar offset
#pragma unroll
    for (int j = 0; j < kPerWave; ++j)
        vv[j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
            kr, (int)((sb + (uint32_t)lane) * 4u + 256u * (uint32_t)j), 0, 0));
}

// The first round's candidate table of every searched cell of the level
// (the 255 cuts of the next 8 bisection steps from the cell's margins): once
// per cell here instead of once per chunk in the round.  A wave per cell
// (for_cell_groups), four entries per lane.
// The launch also fills the level's chunk table (k_fill_chunks' work): the
// first `fill_blocks` blocks take the chunks, the others the cells.
__global__ __launch_bounds__(kBlock) void k_b_tables(const uint32_t *__restrict__ first,
                                                     int32_t nCells,
                                                     const CellRec *__restrict__ recs,
                                                     uint32_t *__restrict__ chunk_cell,
                                                     uint4 *__restrict__ chunk_desc,
                                                     uint32_t max_chunks,
                                                     float *__restrict__ cell_cand, int32_t group,
                                                     uint32_t fill_blocks)
{
    if (blockIdx.x < fill_blocks) {  // uniform
        uint32_t total = first[nCells];
        if (total > max_chunks) total = max_chunks;
        for (uint32_t q = blockIdx.x * blockDim.x + threadIdx.x; q < total;
             q += fill_blocks * blockDim.x)
            fill_chunk(q, first, nCells, recs, chunk_cell, chunk_desc);
        return;
    }
    const int lane = threadIdx.x & 63;
    // a cell whose chunks are read: searched, not found, not in a subtree
    auto active = [&](int32_t c) {
        const CellRec &r = recs[c];
        return !r.found && !r.flags && r.axis >= 0 && r.axis <= 2;
    };
    for_cell_groups(nCells, group, blockIdx.x - fill_blocks, gridDim.x - fill_blocks, active,
                    [&](int32_t c) {
        const float l = recs[c].margin_l, h = recs[c].margin_r;
        float4 v;
        v.x = lane ? candidate(4 * lane, l, h) : 0.0f;  // entry 0 is never read
        v.y = candidate(4 * lane + 1, l, h);
        v.z = candidate(4 * lane + 2, l, h);
        v.w = candidate(4 * lane + 3, l, h);
        reinterpret_cast<float4 *>(cell_cand + (size_t)c * kBins)[lane] = v;
    });
}

// First histogram round: one block per chunk bins every key of the chunk
// over the cell's 255 candidate cuts and writes the chunk's 256-bin row and,
// for the stable partition's stopper counts, its tie row.  Wave w takes the quarter [1024w, 1024w + 1024) of the
// chunk, 64 consecutive keys per load.  A key's bin is the estimate
// (v - lo) * 256 / (hi - lo) clamped to [-0.5, 255.5] whenever that estimate
// lies more than the tolerance from a bin edge (a clamped estimate lies a
// half bin outside the margins, past every candidate on its side: bin 0 or
// 255); otherwise the candidate table decides.  One chunk in flight per
// block: eight blocks per CU (64 VGPRs) hide the loads better than a block
// that keeps its next chunk's keys in registers.
template <int LE>
__global__ __launch_bounds__(kBlock) void k_b_hist(
    const CellRec *__restrict__ recs, int32_t nCells, const uint32_t *__restrict__ first,
    const uint4 *__restrict__ chunk_desc, uint32_t max_chunks, const float *__restrict__ x,
    const float *__restrict__ y, const float *__restrict__ z, const float *__restrict__ cell_cand,
    uint16_t *__restrict__ chunk_hist, uint16_t *__restrict__ chunk_tie, int rev)
{
    constexpr int kW = kBlock / 64;
    constexpr int kPerWave = kMaskWords / kW;  // 16 loads of 64 keys
    __shared__ float cand[kBins + 1];
    __shared__ uint32_t hist[kW][kBins];
    __shared__ uint32_t ties[kBins];  // keys equal to candidate j (rare)
    const int t = threadIdx.x, lane = t & 63, w = (int)uniform((uint32_t)t >> 6);
    const uint32_t sb = (uint32_t)(w * kPerWave * 64);  // chunk position of the quarter
    const uint32_t total = first[nCells];
    for (uint32_t q0 = blockIdx.x;; q0 += gridDim.x) {
        const uint32_t q = rev && q0 < total ? total - 1u - q0 : q0;  // from the last (rev)
        const uint4 d = chunk_record(chunk_desc, q, max_chunks);
        const uint32_t b = uniform(d.x), e = uniform(d.y), cell = uniform(d.z);
        const uint32_t axis = uniform(d.w);
        keep_values(b, e, cell, axis);  // the whole record, in flight with total
        if (q >= total) break;
        if (axis > 2u) continue;  // uniform: the cell is not searched
        const float ce = cand_entry(cell_cand, cell);  // issued before the keys
        float v[kPerWave];
        issue_chunk_loads(x, y, z, true, d, sb, lane, v);
        const float lo = uniform(recs[cell].margin_l), hi = uniform(recs[cell].margin_r);
        store_cands(cand, ce);
#pragma unroll
        for (int u = 0; u < kW; ++u) hist[u][t] = 0u;
        ties[t] = 0u;
        __syncthreads();
        const float width = hi - lo;
        const float scale = width > 0.0f ? (float)kBins / width : 0.0f;
        // clamping is exact while the estimate stays within a quarter bin of
        // the truth; past that every key goes to the table
        const float lim = 0.5f - bin_tolerance(lo, hi, scale);
        const float limx = lim > 0.25f ? lim : -1.0f;
        const uint32_t len = e - b;
        uint32_t *h = hist[w];
        auto scan = [&](auto full) __attribute__((always_inline)) {
            static_for<0, kPerWave>([&](auto jc) __attribute__((always_inline)) {
                constexpr int j = decltype(jc)::value;
                const uint32_t p0 = sb + 64u * (uint32_t)j;  // chunk position of lane 0
                const bool ok = decltype(full)::value || p0 + (uint32_t)lane < len;
                const float vj = v[j];
                const float ef = __builtin_amdgcn_fmed3f((vj - lo) * scale, -0.5f, 255.5f);
                int bin = (int)ef;
                const bool slow = !(fabsf(__builtin_amdgcn_fractf(ef) - 0.5f) < limx);
                if (__ballot(ok && slow)) {  // wave-uniform; rare: near a bin edge
                    if (ok && slow) {
                        int tj;
                        bin = bin_of<LE>(cand, vj, lo, hi, scale, tj);
                        if (chunk_tie && tj) atomicAdd(&ties[tj], 1u);
                    }
                }
                if (ok) atomicAdd(&h[bin], 1u);
            });
        };
        if (len == (uint32_t)kChunk) scan(std::true_type{});  // uniform
        else scan(std::false_type{});
        __syncthreads();
        const uint32_t sum = hist[0][t] + hist[1][t] + hist[2][t] + hist[3][t];  // <= 4096
        chunk_hist[(size_t)q * kBins + t] = (uint16_t)sum;
        if (chunk_tie) chunk_tie[(size_t)q * kBins + t] = (uint16_t)ties[t];
        __syncthreads();  // the next chunk rewrites cand, hist and ties
    }
}

// Second histogram round.  Wave w takes the quarter [1024w, 1024w + 1024)
// of the chunk, 16 keys per lane (64 consecutive keys per load).  Keys below
// lo and above hi are counted in registers, the few in the window [lo, hi]
// are binned, and each wave packs its window keys, in position order, into
// its quarter's slots of `pack` (comp[8q + w] = how many; comp[8q + 4] = the
// chunk's keys below lo).  Later windows lie inside this one, so later
// rounds need only these keys.  The wave also leaves two of the chunk's
// bitmasks for the Hoare partition (bit j of word k = chunk position
// 64k + j): keys above hi (masks[q][0]) and keys in the window (masks[q][1]).
// The cell's final cut lies in [lo, hi], so these decide every stopper bit
// but those of the packed keys.
// Eight waves per SIMD (the compiler would keep the load offsets in scalar
// registers and stop at seven).
template <int LE>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_b_hist_window(
    const CellRec *__restrict__ recs, int32_t nCells, const uint32_t *__restrict__ first,
    const uint4 *__restrict__ chunk_desc, uint32_t max_chunks, const float *__restrict__ x,
    const float *__restrict__ y, const float *__restrict__ z, const float *__restrict__ cell_cand,
    uint16_t *__restrict__ chunk_hist, float *__restrict__ pack, uint32_t *__restrict__ comp,
    uint64_t *__restrict__ masks, int rev)
{
    constexpr int kW = kBlock / 64;
    constexpr int kPerWave = kMaskWords / kW;  // 16 loads of 64 keys
    __shared__ float cand[kBins + 1];
    __shared__ uint32_t hist[kBins];  // window keys are few: one histogram
    __shared__ uint32_t sm[4];
    __shared__ float wkeys[kW][kChunk / kW];  // each wave's window keys, packed
    __shared__ uint64_t words[kW][2][kPerWave];  // each wave's mask words, staged
    const int t = threadIdx.x, lane = t & 63, w = (int)uniform((uint32_t)t >> 6);
    const uint64_t lanes_below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    const uint32_t total = first[nCells];
    for (uint32_t q0 = blockIdx.x;; q0 += gridDim.x) {
        const uint32_t q = rev && q0 < total ? total - 1u - q0 : q0;  // from the last (rev)
        const uint4 d = chunk_record(chunk_desc, q, max_chunks);
        const uint32_t b = uniform(d.x), e = uniform(d.y), cell = uniform(d.z);
        const uint32_t axis = uniform(d.w);
        keep_values(b, e, cell, axis);  // the whole record, in flight with total
        if (q >= total) break;
        if (axis > 2u) continue;  // uniform: the cell is not searched
        if (recs[cell].found) continue;  // uniform: the first round found the cut
        // the chunk's keys through a range-checked descriptor: loads past the
        // chunk's end return 0 and are masked out below, with no branches
        const float *kp = axis_ptr(x, y, z, (int)axis) + b;
        const float ce = cand_entry(cell_cand, cell);
        const __amdgpu_buffer_rsrc_t kr =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(kp), 0, (int)((e - b) * 4u), 0x00020000);
        const uint32_t sb = (uint32_t)(w * kPerWave * 64);  // chunk position of the quarter
        float v[kPerWave];
        // the whole offset in the per-lane operand: the range check covers
        // it, not the scalar offset
#pragma unroll
        for (int j = 0; j < kPerWave; ++j)
            v[j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                kr, (int)((sb + (uint32_t)lane) * 4u + 256u * (uint32_t)j), 0, 0));
        const float lo = uniform(recs[cell].margin_l), hi = uniform(recs[cell].margin_r);
        store_cands(cand, ce);
        hist[t] = 0u;
        __syncthreads();
        const float width = hi - lo;
        const float scale = width > 0.0f ? (float)kBins / width : 0.0f;
        const uint32_t len = e - b;
        uint32_t below = 0, packed = 0;  // wave-uniform
        float *dst = pack + b + sb;
        float *wk = wkeys[w];
        auto scan = [&](auto full) __attribute__((always_inline)) {
            static_for<0, kPerWave>([&](auto jc) __attribute__((always_inline)) {
                constexpr int j = decltype(jc)::value;
                uint64_t valid = ~0ull;
                if constexpr (!decltype(full)::value) {
                    const uint32_t p0 = sb + 64u * (uint32_t)j;  // chunk position of lane 0
                    valid = p0 >= len ? 0ull
                                      : (len - p0 >= 64u ? ~0ull : (1ull << (len - p0)) - 1ull);
                }
                const float vj = v[j];
                const uint64_t mB = __ballot(vj < lo) & valid;
                const uint64_t mG = __ballot(vj > hi) & valid;
                const uint64_t mW = valid & ~mB & ~mG;
                below += (uint32_t)__popcll(mB);
                // staged by one lane: a cross-lane write into a register would
                // be lost if the compiler moved that register under a partial
                // exec mask (the binning below is divergent)
                if (lane == 0) {
                    words[w][0][j] = mG;
                    words[w][1][j] = mW;
                }
                if (mW) {  // wave-uniform: most loads have no key in the window
                    if ((mW >> lane) & 1ull) {
                        const uint32_t slot = packed + (uint32_t)__popcll(mW & lanes_below);
                        dst[slot] = vj;
                        wk[slot] = vj;
                    }
                    packed += (uint32_t)__popcll(mW);
                }
            });
        };
        if (len == (uint32_t)kChunk) scan(std::true_type{});  // uniform
        else scan(std::false_type{});
        // the quarter's keys that are neither below nor in the window
        const uint32_t mine = len > sb ? (len - sb < 1024u ? len - sb : 1024u) : 0u;
        const uint32_t above = mine - below - packed;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        __builtin_amdgcn_wave_barrier();
        const uint64_t mineG = lane < kPerWave ? words[w][0][lane] : 0ull;
        const uint64_t mineW = lane < kPerWave ? words[w][1][lane] : 0ull;
        for (uint32_t k = (uint32_t)lane; k < packed; k += 64) {
            const float vk = wk[k];
            int tj;  // ties: the stopper counts of cells past this round use the packed keys
            atomicAdd(&hist[bin_of<LE>(cand, vk, lo, hi, scale, tj)], 1u);
        }
        uint64_t *mq = masks + (size_t)q * (2 * kMaskWords) + w * kPerWave;
        if (lane < kPerWave) {
            mq[lane] = mineG;
            mq[kMaskWords + lane] = mineW;
        }
        if (lane == 0) {
            comp[8 * (size_t)q + w] = packed;
            sm[w] = below | (above << 16);  // each <= 1024
        }
        __syncthreads();
        const uint32_t ba = sm[0] + sm[1] + sm[2] + sm[3];
        if (t == 0) comp[8 * (size_t)q + 4] = ba & 0xffffu;
        uint32_t sum = hist[t];
        if (t == 0) sum += ba & 0xffffu;
        if (t == kBins - 1) sum += ba >> 16;
        chunk_hist[(size_t)q * kBins + t] = (uint16_t)sum;
        __syncthreads();  // the next chunk rewrites cand, hist and sm
    }
}

// Sums chunk histograms into cell histograms: block g takes chunks
// [g*64, g*64+64), thread t owns bin t; all 64 row loads are in flight at
// once, and one atomic per (block, cell, bin) flushes a run.
__global__ __launch_bounds__(kBlock) void k_b_hist_reduce(const CellRec *recs, int32_t nCells,
                                                          const uint32_t *first,
                                                          const uint32_t *chunk_cell,
                                                          const uint16_t *chunk_hist,
                                                          uint32_t *cell_hist)
{
    __shared__ int32_t scell[kReduceRows];  // cell of each row, -1 if not live
    const uint32_t total = first[nCells];
    for (uint32_t q0 = blockIdx.x * (uint32_t)kReduceRows; q0 < total;
         q0 += gridDim.x * (uint32_t)kReduceRows) {
    const uint32_t nrows = total - q0 < (uint32_t)kReduceRows ? total - q0 : (uint32_t)kReduceRows;
    const int t = threadIdx.x;
    if (t < kReduceRows) {
        int32_t cl = -1;
        if ((uint32_t)t < nrows) {
            uint32_t cell = chunk_cell[q0 + t];
            const CellRec &r = recs[cell];
            if (!(r.found || r.flags)) cl = (int32_t)cell;
        }
        scell[t] = cl;
    }
    __syncthreads();
    int32_t cur = -1;
    uint32_t acc = 0;
    uint32_t v[kReduceRows];  // every row's load in flight at once
#pragma unroll
    for (int u = 0; u < kReduceRows; ++u)
        v[u] = ((uint32_t)u < nrows && scell[u] >= 0) ? chunk_hist[(size_t)(q0 + u) * kBins + t] : 0u;
#pragma unroll
    for (int u = 0; u < kReduceRows; ++u) {
        const int32_t cl = (uint32_t)u < nrows ? scell[u] : cur;
        if (cl != cur) {
            if (cur >= 0 && acc) atomicAdd(&cell_hist[(size_t)cur * kBins + t], acc);
            cur = cl;
            acc = 0;
        }
        acc += v[u];
    }
    if (cur >= 0 && acc) atomicAdd(&cell_hist[(size_t)cur * kBins + t], acc);
    __syncthreads();  // scell is rewritten for the next tile
    }
}

__device__ inline void record_level_passes(int32_t *level_passes, int32_t l, int32_t passes)
{
    // a plain read filters almost every atomic once the level maximum is in
    if (passes > *((volatile int32_t *)&level_passes[l])) atomicMax(&level_passes[l], passes);
}

// A level's pass count is the most passes any of its cells took, so a cell
// records its count once, when it finishes.  The cells a wave (or block)
// finishes share one running maximum, recorded per run of cells with the
// same counter (one build's level) and at the end: thousands of cells of a
// level finishing in one round would otherwise queue thousands of atomics
// on one word.
struct PassMax {
    int32_t lp = -1, mx = 0;
    __device__ void add(int32_t *level_passes, int32_t l, int32_t p)
    {
        if (l != lp) {
            flush(level_passes);
            lp = l;
            mx = p;
        } else if (p > mx) {
            mx = p;
        }
    }
    __device__ void flush(int32_t *level_passes)
    {
        if (lp >= 0) record_level_passes(level_passes, lp, mx);
        lp = -1;
    }
};

// End of a 4-wave block whose lanes 0 each hold a PassMax: the waves' last
// runs are combined in LDS and recorded by one thread (one atomic per block
// where its waves share a counter).  Every thread of the block calls it.
__device__ inline void flush_block(PassMax &pm, int32_t *level_passes)
{
    __shared__ int32_t s_lp[kBlock / 64], s_mx[kBlock / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) {
        s_lp[w] = pm.lp;
        s_mx[w] = pm.mx;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        PassMax b;
        for (int i = 0; i < kBlock / 64; ++i)
            if (s_lp[i] >= 0) b.add(level_passes, s_lp[i], s_mx[i]);
        b.flush(level_passes);
    }
}

// One histogram round of the bisection controller (orbit.cpp:149-231),
// replayed by a whole wave.  P[j] (j in [1, 255]) is the count below
// candidate cut j of the round that starts from margins [lo, hi].  Counts
// grow with j and so does the controller's difference, so the passes it
// makes are the binary-search path towards b, the first node whose
// difference is > 0 (go left at a node >= b, right otherwise); the round
// stops at the first node of that path within +-2 of the target.  b comes
// from one ballot count, the path from b alone, so the 8 counts are read in
// parallel instead of one dependent read per pass.
struct RoundOut {
    float L, R;
    int32_t passes;
    bool found;
    int32_t node;  // the candidate the round stopped at (when found)
};

// The controller's difference for a left count (uint32) or a left weight
// (uint64, weighted builds): weights grow with the candidate as counts do.
__device__ inline int64_t round_diff(uint32_t left, float target)
{
    return difference_from_target(left, target);
}
__device__ inline int64_t round_diff(uint64_t left, float target)
{
    return difference_from_target_w(left, target);
}

// The path of one round from b, the first candidate whose difference is
// > 0 (nle + 1), with count_at(j) = P[j] for the path's candidates.
template <class T, class CountAt>
__device__ inline RoundOut replay_path(uint32_t nle, CountAt count_at, float lo, float hi,
                                       float target, int32_t passes0, int lane,
                                       uint64_t *trace_row)
{
    const int b = 1 + (int)nle;
    const int steps = kHistK < ORB_MAX_PASSES - passes0 ? kHistK : ORB_MAX_PASSES - passes0;
    int nodes[kHistK];
    {
        int node = kBins / 2, step = kBins / 4;
#pragma unroll
        for (int d = 0; d < kHistK; ++d) {
            nodes[d] = node;
            node = node >= b ? node - step : node + step;
            step >>= 1;
        }
    }
    T cnt[kHistK];
#pragma unroll
    for (int d = 0; d < kHistK; ++d) cnt[d] = count_at(nodes[d]);
    int s = steps;
#pragma unroll
    for (int d = kHistK - 1; d >= 0; --d) {
        const int64_t df = round_diff(cnt[d], target);
        if (d < steps && df < 3 && df > -3) s = d;
    }
    const bool found = s < steps;
    const int moves = found ? s : steps;
    float L = lo, R = hi;
#pragma unroll
    for (int d = 0; d < kHistK; ++d) {
        if (d < moves) {
            const float cut = cell_cut(L, R);
            if (nodes[d] >= b) R = cut;
            else L = cut;
        }
    }
    const int used = found ? s + 1 : steps;
    if (trace_row && lane < used) {
        T v = 0;
#pragma unroll
        for (int d = 0; d < kHistK; ++d)
            if (d == lane) v = cnt[d];
        trace_row[passes0 + lane] = v;
    }
    int32_t stop = 0;
#pragma unroll
    for (int d = 0; d < kHistK; ++d)
        if (d == s) stop = nodes[d];
    return RoundOut{L, R, passes0 + used, found, found ? stop : 0};
}

template <class T>
__device__ inline RoundOut replay_round(const T *P, float lo, float hi, float target,
                                        int32_t passes0, int lane, uint64_t *trace_row)
{
    uint32_t nle = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int j = 4 * lane + 1 + q;
        const bool le0 = j < kBins && round_diff(P[j], target) <= 0;
        nle += (uint32_t)__popcll(__ballot(le0));
    }
    return replay_path<T>(nle, [&](int j) { return P[j]; }, lo, hi, target, passes0, lane,
                          trace_row);
}

// replay_round with the round's prefix sums in registers, not in LDS: lane l
// holds P[4l + 1 + q] in pv[q].  The path's counts are read across lanes
// (uniform indices), so no store, fence or load stands between the scan and
// the replay.
template <class T>
__device__ inline RoundOut replay_round_lanes(const T (&pv)[4], float lo, float hi, float target,
                                              int32_t passes0, int lane, uint64_t *trace_row)
{
    uint32_t nle = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int j = 4 * lane + 1 + q;
        const bool le0 = j < kBins && round_diff(pv[q], target) <= 0;
        nle += (uint32_t)__popcll(__ballot(le0));
    }
    auto count_at = [&](int j) {  // j in [1, 255], the same in every lane
        const int q = (j - 1) & 3;
        const T v = q == 0 ? pv[0] : (q == 1 ? pv[1] : (q == 2 ? pv[2] : pv[3]));
        return lane_value(v, (j - 1) >> 2);
    };
    return replay_path<T>(nle, count_at, lo, hi, target, passes0, lane, trace_row);
}

// The record's found field after a round that found its cut at candidate
// ro.node of [lo, hi]: 1 + node when that candidate differs from its
// neighbours (the stopper counts can then come from the round's histograms;
// equal candidates -- a window a few ulps wide -- would split the keys equal
// to the cut over several tie bins), else 1 (found, the keys are read); 0
// when not found.
__device__ inline int32_t found_encoding(const RoundOut &ro, float lo, float hi)
{
    if (!ro.found) return 0;
    const int j = ro.node;
    const float cj = candidate(j, lo, hi);
    const float cp = j > 1 ? candidate(j - 1, lo, hi) : -INFINITY;
    const float cn = j < kBins - 1 ? candidate(j + 1, lo, hi) : INFINITY;
    return (cj == cp || cj == cn) ? 1 : 1 + j;
}

// Lane 0 of the replaying wave: the round's margins into the cell's record
// and heap cell; a finished cell (cut found, or the pass cap with the last
// midpoint) records its passes (into pm when given) and is split at once
// (orbit.cpp:235-250).
__device__ inline void finish_round(CellRec r, int32_t c, const RoundOut &ro, int32_t found_enc,
                                    CellRec *recs, orb_cell *heap, int32_t *level_passes,
                                    uint8_t *exists, int32_t *status, PassMax *pm = nullptr)
{
    const float L = ro.L, R = ro.R;
    const int32_t passes = ro.passes;
    const bool found = ro.found;
    r.margin_l = L;
    r.margin_r = R;
    r.cut = cell_cut(L, R);
    r.passes = passes;
    r.found = found_enc;  // the stopper counts read this round's histograms
    recs[c] = r;
    orb_cell &hc = heap[(int64_t)r.hb + r.id];
    hc.cutMarginLeft = L;
    hc.cutMarginRight = R;
    hc.foundCut = found;
    if (!found && passes < ORB_MAX_PASSES) return;  // a later round records it
    if (pm) pm->add(level_passes, r.lp, passes);
    else record_level_passes(level_passes, r.lp, passes);
    const orb_cell p = hc;
    orb_cell lc, rc;
    uint32_t *wl = reinterpret_cast<uint32_t *>(&lc);
    uint32_t *wr = reinterpret_cast<uint32_t *>(&rc);
#pragma unroll
    for (int j = 0; j < (int)(sizeof(orb_cell) / 4); ++j) wl[j] = wr[j] = 0u;
    const int64_t hb = r.hb;
    if (right_child_id(r.id) >= r.capr || !cell_split(p, lc, rc)) {
        report_error(status + r.st, r.lp & 63, kErrSplit, r.id);
        return;
    }
    heap[hb + lc.id] = lc;
    heap[hb + rc.id] = rc;
    exists[hb + lc.id] = 1;
    exists[hb + rc.id] = 1;
}


// A predicted window of a cell (large levels, k_p_choose): [lo, hi], its keys
// in bins 1 to 253 (bin 0: below, 255: above), and the keys [klo, khi] of the bins
// that can hold the cut (k_p_narrow).  The bins come from the sample's 1024 linear
// ones over the cell's margins, of which the window takes [bl, bu): each is cut
// into as many as its share of the window's sample (kSampleBins bytes a cell,
// the window bins before each), so that keys in a few tight clumps are told
// apart as well as even ones (two clumps of 0.01, 2^26 keys to 256: 10.1 ms with
// bins of one width, which a clump falls into one of, now 4.6).
constexpr int kSampleBins = 1024;
constexpr int kWindowBins = kBins - 3;
struct Window {
    float lo, hi, klo, khi;
    float base, scale;  // sample bin of v: (v - base) * scale
    uint32_t bl, bu;
};

// Sample bins per unit of a cell's margins (0, one bin, where that is not finite).
__device__ inline float sample_scale(float width)
{
    return width > 0x1p-100f ? (float)kSampleBins / width : 0.0f;
}

// The bin of a key in the window (tab: the window bins before each sample bin):
// grows with the key (a difference, a product by a positive number and their
// fraction keep order in float32), so keys of smaller bins are smaller.
__device__ inline uint32_t window_bin(float v, const Window &wd, const uint8_t *tab)
{
    const float t = __builtin_amdgcn_fmed3f((v - wd.base) * wd.scale, (float)wd.bl, (float)wd.bu);
    const uint32_t s = (uint32_t)t < wd.bu ? (uint32_t)t : wd.bu - 1u;
    const uint32_t b = tab[s], n = (s + 1u < (uint32_t)kSampleBins ? tab[s + 1u] : (uint32_t)kWindowBins) - b;
    const uint32_t part = (uint32_t)((t - (float)s) * (float)n);
    return 1u + b + (part < n ? part : n ? n - 1u : 0u);
}

// The passes of a predicted cell that its window decides: a candidate left of
// klo (right of khi) has a difference of -3 or less (3 or more).  Stops at
// the first candidate inside, or at the pass cap.
__device__ inline void window_passes(const Window &wd, float &L, float &R, int32_t &passes)
{
    while (passes < ORB_MAX_PASSES) {
        const float c = cell_cut(L, R);
        if (c < wd.klo) L = c;
        else if (c > wd.khi) R = c;
        else break;
        ++passes;
    }
}

// Whether the final cut lets the window's masks stand (a search that ends at
// the pass cap may end outside); else the cell is left alone and counted.
__device__ inline bool window_holds(const Window &wd, float L, float R)
{
    const float c = cell_cut(L, R);
    return !(c < wd.lo) && !(c > wd.hi);
}

// Rounds 3 and 4 gather a searching cell's keys into up to 64 lists (see
// k_b_select): list r covers a contiguous range of the cell's chunks.
constexpr int kSelLists = 64;
struct SelLists {
    uint32_t f, S, R;  // first chunk, chunks per list, lists
    __device__ SelLists(uint32_t first_chunk, uint32_t nch)
    {
        f = first_chunk;
        S = (nch + kSelLists - 1u) / kSelLists;
        R = S ? (nch + S - 1u) / S : 0u;
    }
    __device__ uint32_t list_of_chunk(uint32_t q) const { return (q - f) / S; }
    __device__ uint32_t start_chunk(uint32_t r) const { return f + r * S; }
};

// One wave per cell: prefix sums of the cell histogram in registers, then
// the wave replays up to 8 passes of the bisection controller.
__global__ __launch_bounds__(kBlock) void k_b_replay(CellRec *recs, int32_t nCells,
                                                     uint32_t *cell_hist, orb_cell *heap,
                                                     uint64_t *trace, int32_t *level_passes,
                                                     uint8_t *exists, int32_t *status,
                                                     float *next_cand, const uint32_t *first,
                                                     unsigned long long *sel_clear, int32_t group)
{
    const int lane = threadIdx.x & 63;
    auto active = [&](int32_t c) { return !recs[c].found && !recs[c].flags; };
    PassMax pm;  // lane 0
    for_cell_groups(nCells, group, active, [&](int32_t c) {
    const CellRec r = recs[c];
    uint4 *row = reinterpret_cast<uint4 *>(cell_hist + (size_t)c * kBins);
    const uint4 h4 = row[lane];
    row[lane] = make_uint4(0u, 0u, 0u, 0u);  // the next round starts from zero
    const uint32_t s0 = h4.x, s1 = s0 + h4.y, s2 = s1 + h4.z, s3 = s2 + h4.w;
    const uint32_t base = wave_inclusive_scan(s3) - s3;
    // P[4 lane + 1 + q] (P[j] = keys in bins below j)
    const uint32_t pv[4] = {base + s0, base + s1, base + s2, base + s3};
    const uint32_t n = r.end - r.begin;
    const float target = difference_target(n, r.nLeaf);
    const RoundOut ro = replay_round_lanes(pv, r.margin_l, r.margin_r, target, r.passes, lane,
                                           trace ? trace + ((size_t)r.hb + r.id) * ORB_MAX_PASSES
                                                 : nullptr);
    if (next_cand && !ro.found) {  // the next round's candidate table (uniform)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int j = 4 * lane + i;
            next_cand[(size_t)c * kBins + j] = j ? candidate(j, ro.L, ro.R) : 0.0f;
        }
    }
    if (sel_clear) {  // rounds 3 and 4 gather from zero
        const uint32_t f = first[c];
        const SelLists sl(f, first[c + 1] - f);
        if ((uint32_t)lane < sl.R) sel_clear[sl.start_chunk((uint32_t)lane)] = 0ull;
    }
    if (lane != 0) return;
    finish_round(r, c, ro, found_encoding(ro, r.margin_l, r.margin_r), recs, heap, level_passes,
                 exists, status, &pm);
    });
    flush_block(pm, level_passes);
}

// Rounds 3 and 4 read only the keys that the window round packed and that
// lie inside the margins after round 2 (every later candidate lies inside
// them).  k_b_select gathers them, per searching cell, into up to 64 lists
// in `sel`, each over a contiguous range of the cell's chunks: the list fills
// positions from its range's first particle on, which it cannot outgrow, and
// its counter (kept at the range's first chunk) takes the atomics of a 64th of
// the chunks even in a cell of the whole level.

// A wave takes a chunk: it reads the quarters' packed keys laid end to end,
// four loads per lane in flight, counts those inside the cell's margins and
// those below (with the keys below the window round's margins, which that
// round counted per chunk), reserves slots in its list with one 64-bit atomic
// (keys | below << 32) and writes the keys there.  Up to 256 keys stay in
// registers in between.  Grouped or clustered keys leave a good part of the chunk
// in the window, a serial chain for a wave of more chunks: with four a wave
// 2^26 keys in runs of 512 took 47 us a level, with one 20; 2^27 even keys 20 and 15.
// PRED: the window's keys in [klo, khi]; the keys left of them are counted
// already (k_p_narrow).
template <bool PRED>
__global__ __launch_bounds__(kBlock) void k_b_select(const CellRec *__restrict__ recs,
                                                     int32_t nCells,
                                                     const uint32_t *__restrict__ first,
                                                     const uint4 *__restrict__ chunk_desc,
                                                     uint32_t max_chunks,
                                                     const float *__restrict__ ckeys,
                                                     const uint32_t *__restrict__ comp,
                                                     float *__restrict__ sel,
                                                     unsigned long long *__restrict__ sel_lists,
                                                     const Window *__restrict__ windows)
{
    constexpr uint32_t kW = kBlock / 64;
    constexpr int kSelBatch = 4;
    constexpr uint32_t kStep = 64u * kSelBatch;
    const int lane = threadIdx.x & 63;
    const uint32_t total = first[nCells];
    for (uint32_t q = uniform(blockIdx.x * kW + (threadIdx.x >> 6)); q < total; q += gridDim.x * kW) {
        const uint4 d = chunk_record(chunk_desc, q, max_chunks);
        const uint32_t counts = lane < 5 ? comp[8 * (size_t)q + lane] : 0u;
        const uint32_t b = uniform(d.x), e = uniform(d.y), cell = uniform(d.z);
        if (uniform(d.w) > 2u) continue;  // uniform, as below
        const CellRec &r = recs[cell];
        if (uniform((uint32_t)(r.found | r.flags))) continue;
        const float lo = uniform(PRED ? windows[cell].klo : r.margin_l);
        const float hi = uniform(PRED ? windows[cell].khi : r.margin_r);
        // key t of the chunk lies at t + at[j] of the last quarter j with ex[j] <= t
        uint32_t ex[kW + 1] = {0u}, at[kW];
#pragma unroll
        for (int j = 0; j < (int)kW; ++j) {
            uint32_t off, cnt;
            wave_share(b, e, j, off, cnt);
            at[j] = b + off - ex[j];
            ex[j + 1] = ex[j] + lane_value(counts, j);
        }
        const uint32_t T = ex[kW];
        float v[kSelBatch];
        auto load_batch = [&](uint32_t t0) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < kSelBatch; ++u) {
                const uint32_t t = t0 + 64u * (uint32_t)u + (uint32_t)lane;
                uint32_t a = at[0];
#pragma unroll
                for (int j = 1; j < (int)kW; ++j) a = t >= ex[j] ? at[j] : a;
                v[u] = t < T ? ckeys[t + a] : 0.0f;
            }
        };
        auto kept = [&](uint32_t t0, int u) __attribute__((always_inline)) {
            return __ballot(t0 + 64u * (uint32_t)u + (uint32_t)lane < T && !(v[u] < lo) && !(v[u] > hi));
        };
        uint32_t ns = 0, nb = PRED ? 0u : lane_value(counts, (int)kW);
        for (uint32_t t0 = 0; t0 < T; t0 += kStep) {
            load_batch(t0);
#pragma unroll
            for (int u = 0; u < kSelBatch; ++u) {
                ns += (uint32_t)__popcll(kept(t0, u));
                if (!PRED)
                    nb += (uint32_t)__popcll(
                        __ballot(t0 + 64u * (uint32_t)u + (uint32_t)lane < T && v[u] < lo));
            }
        }
        if (!(ns | nb)) continue;
        const uint32_t f = first[cell];
        const SelLists sl(f, first[cell + 1] - f);
        const uint32_t qs = sl.start_chunk(sl.list_of_chunk(q));
        uint32_t slot = 0;
        if (lane == 0)
            slot = (uint32_t)atomicAdd(&sel_lists[qs], (unsigned long long)ns | ((unsigned long long)nb << 32));
        slot = lane_value(slot, 0) + r.begin + (qs - f) * (uint32_t)kChunk;
        if (!ns) continue;
        for (uint32_t t0 = 0; t0 < T; t0 += kStep) {
            if (T > kStep) load_batch(t0);  // uniform: one batch is still in registers
#pragma unroll
            for (int u = 0; u < kSelBatch; ++u) {
                const uint64_t m = kept(t0, u);
                if (m >> lane & 1ull)
                    sel[slot + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                         __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u))] = v[u];
                slot += (uint32_t)__popcll(m);
            }
        }
    }
}

// A predicted cell that its window does not carry: nothing of it is written,
// the host's second run of the levels builds it.
__device__ inline void leave_alone(const CellRec &r, int32_t c, CellRec *recs, int32_t *level_passes)
{
    recs[c].flags = 1;
    atomicAdd(&level_passes[r.lp & ~63], 1);
}

// Rounds 3 and 4 of each searching cell from its gathered keys, a wave per
// cell: lane r reads list r's count (its counts below add up to the cell's
// count below the margins), the keys of all lists are read laid end to end
// and binned against the round's candidates in LDS (keys below the margins
// add to bin 0, as in the chunk rounds; keys above them are never read by
// the replay), and the round is replayed.  A cell that neither found its
// cut nor reached the pass cap runs round 4 over the same keys with the
// narrowed margins (the keys that now fall below them join the count
// below).  The record, heap cell and split are written as after any round.
// PRED (large levels): the rounds start from the cell's own margins; the
// passes that the window decides come first.
constexpr int kFinBatch = 8;  // gathered keys per lane in flight
template <int LE, bool PRED>
__global__ __launch_bounds__(kBlock) void k_b_finish(CellRec *recs, int32_t nCells,
                                                     const uint32_t *__restrict__ first,
                                                     const float *__restrict__ sel,
                                                     const unsigned long long *__restrict__ sel_lists,
                                                     orb_cell *heap, uint64_t *trace,
                                                     int32_t *level_passes, uint8_t *exists,
                                                     int32_t *status, int32_t group,
                                                     const Window *__restrict__ windows)
{
    __shared__ float cand[4][kBins + 1];
    __shared__ uint32_t P[4][kBins + 1];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    float *cw = cand[w];
    uint32_t *pw = P[w];
    auto active = [&](int32_t c) { return !recs[c].found && !recs[c].flags; };
    PassMax pm;  // lane 0
    for_cell_groups(nCells, group, active, [&](int32_t c) {
    CellRec r = recs[c];
    const uint32_t f = first[c], nch = first[c + 1] - f;
    const SelLists sl(f, nch);
    // list `lane`: its keys from position kpos on (at most the positions of
    // its chunk range, whatever the counter holds)
    uint32_t mr = 0, kpos = 0;
    uint32_t below = 0;
    if ((uint32_t)lane < sl.R) {
        const uint32_t qs = sl.start_chunk((uint32_t)lane);
        const uint32_t qn = (uint32_t)lane + 1u < sl.R ? sl.start_chunk((uint32_t)lane + 1u) : f + nch;
        const unsigned long long e = sel_lists[qs];
        kpos = r.begin + (qs - f) * (uint32_t)kChunk;
        const uint32_t span = (qn < f + nch ? r.begin + (qn - f) * (uint32_t)kChunk : r.end) - kpos;
        mr = (uint32_t)e < span ? (uint32_t)e : span;
        below = (uint32_t)(e >> 32);
    }
    below = wave_sum(below);
    const uint32_t lincl = wave_inclusive_scan(mr), lex = lincl - mr;
    const uint32_t m = (uint32_t)__shfl((int)lincl, 63, 64);
    const float target = difference_target(r.end - r.begin, r.nLeaf);
    uint64_t *trow = trace ? trace + ((size_t)r.hb + r.id) * ORB_MAX_PASSES : nullptr;
    Window wd{};
    if constexpr (PRED) {
        wd = windows[c];
        window_passes(wd, r.margin_l, r.margin_r, r.passes);
    }
    while (true) {
        const float lo = r.margin_l, hi = r.margin_r;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        __builtin_amdgcn_wave_barrier();  // the wave's last replay has read the tables
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int j = 4 * lane + i;
            cw[j] = j == 0 ? -INFINITY : candidate(j, lo, hi);
            pw[j] = 0u;
        }
        if (lane == 0) cw[kBins] = INFINITY;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        __builtin_amdgcn_wave_barrier();
        const float width = hi - lo;
        const float scale = width > 0.0f ? (float)kBins / width : 0.0f;
        uint32_t bl = 0;
        for (uint32_t k0 = 0; k0 < m; k0 += 64u * kFinBatch) {
            float v[kFinBatch];  // all of a batch's loads in flight
#pragma unroll
            for (int u = 0; u < kFinBatch; ++u) {
                // key k of the cell: list j = the last with lex_j <= k
                const uint32_t k = k0 + 64u * (uint32_t)u + (uint32_t)lane;
                int j = 0;
#pragma unroll
                for (int st = 32; st > 0; st >>= 1)
                    if ((uint32_t)__shfl((int)lex, j + st, 64) <= k) j += st;
                const uint32_t at =
                    (uint32_t)__shfl((int)kpos, j, 64) + (k - (uint32_t)__shfl((int)lex, j, 64));
                v[u] = k < m ? sel[at] : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < kFinBatch; ++u) {
                if (k0 + 64u * (uint32_t)u + (uint32_t)lane >= m) continue;
                if (v[u] < lo) ++bl;
                else if (!(v[u] > hi)) {
                    int tj;
                    atomicAdd(&pw[bin_of<LE>(cw, v[u], lo, hi, scale, tj)], 1u);
                }
            }
        }
        const uint32_t left = below + wave_sum(bl);  // every round reads every listed key
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        __builtin_amdgcn_wave_barrier();
        // P[j] = the keys below the margins + bins < j
        const uint32_t s0 = pw[4 * lane], s1 = s0 + pw[4 * lane + 1];
        const uint32_t s2 = s1 + pw[4 * lane + 2], s3 = s2 + pw[4 * lane + 3];
        const uint32_t base = left + wave_inclusive_scan(s3) - s3;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        __builtin_amdgcn_wave_barrier();
        pw[4 * lane + 1] = base + s0;
        pw[4 * lane + 2] = base + s1;
        pw[4 * lane + 3] = base + s2;
        pw[4 * lane + 4] = base + s3;
        if (lane == 0) pw[0] = 0u;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        __builtin_amdgcn_wave_barrier();
        const RoundOut ro = replay_round(pw, lo, hi, target, r.passes, lane, trow);
        if (ro.found || ro.passes >= ORB_MAX_PASSES) {  // uniform
            if (PRED && !window_holds(wd, ro.L, ro.R)) {
                if (lane == 0) leave_alone(r, c, recs, level_passes);
                break;
            }
            if (lane == 0)
                finish_round(r, c, ro, found_encoding(ro, lo, hi), recs, heap, level_passes,
                             exists, status, &pm);
            break;
        }
        r.margin_l = ro.L;
        r.margin_r = ro.R;
        r.passes = ro.passes;
    }
    });
    flush_block(pm, level_passes);
}

// Counts the bins of a wave's keys (those of lanes with `in`): one addition
// where they share a bin, as keys that tie at a cut do (64 lanes adding to one
// LDS word wait for each other).
__device__ inline void count_bin(uint32_t *hist, int bin, bool in)
{
    const uint64_t m = __ballot(in);
    if (!m) return;  // uniform
    const int src = __builtin_ctzll(m);
    const int b0 = (int)lane_value((uint32_t)bin, src);
    if (__ballot(in && bin == b0) == m) {
        if ((int)(threadIdx.x & 63) == src) atomicAdd(&hist[b0], (uint32_t)__popcll(m));
    } else if (in) {
        atomicAdd(&hist[bin], 1u);
    }
}

// The same two rounds with a block per cell, for levels of few cells (whose
// cells hold the most gathered keys): the waves bin their shares of the
// keys into one LDS histogram, wave 0 prefix-sums and replays, and the
// round's outcome reaches the other waves through LDS.
constexpr int kFinBlockCells = 1024;  // levels up to this many cells
// (Sixteen waves, and one addition where a wave's keys share a bin: where many
// keys tie at the cut, a cell of 2^26 keys on 512 coordinate values lists
// 131072 of them. Four waves took 962 us a level there over two rounds, these
// 322 over the predicted window's three or four; 18 us at 2^27 even keys.)
constexpr int kFinBlock = 1024;
template <int LE, bool PRED>
__global__ __launch_bounds__(kFinBlock) void k_b_finish_block(CellRec *recs, int32_t nCells,
                                                           const uint32_t *__restrict__ first,
                                                           const float *__restrict__ sel,
                                                           const unsigned long long *__restrict__ sel_lists,
                                                           orb_cell *heap, uint64_t *trace,
                                                           int32_t *level_passes, uint8_t *exists,
                                                           int32_t *status,
                                                           const Window *__restrict__ windows)
{
    constexpr int kW = kFinBlock / 64;
    __shared__ float cand[kBins + 1];
    __shared__ uint32_t hist[kBins], P[kBins + 1];
    __shared__ uint32_t sm[kW];
    __shared__ float s_lr[2];
    __shared__ int32_t s_pf[2];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    PassMax pm;  // thread 0
    for (int32_t c = blockIdx.x; c < nCells; c += gridDim.x) {
        CellRec r = recs[c];
        if (r.found || r.flags) continue;  // uniform
        const uint32_t f = first[c], nch = first[c + 1] - f;
        const SelLists sl(f, nch);
        // every wave holds the list table (list `lane`: count, first position)
        uint32_t mr = 0, kpos = 0, bw = 0;
        if ((uint32_t)lane < sl.R) {
            const uint32_t qs = sl.start_chunk((uint32_t)lane);
            const uint32_t qn =
                (uint32_t)lane + 1u < sl.R ? sl.start_chunk((uint32_t)lane + 1u) : f + nch;
            const unsigned long long e = sel_lists[qs];
            kpos = r.begin + (qs - f) * (uint32_t)kChunk;
            const uint32_t span =
                (qn < f + nch ? r.begin + (qn - f) * (uint32_t)kChunk : r.end) - kpos;
            mr = (uint32_t)e < span ? (uint32_t)e : span;
            bw = (uint32_t)(e >> 32);
        }
        const uint32_t below = wave_sum(bw);
        const uint32_t lincl = wave_inclusive_scan(mr), lex = lincl - mr;
        const uint32_t m = (uint32_t)__shfl((int)lincl, 63, 64);
        const float target = difference_target(r.end - r.begin, r.nLeaf);
        uint64_t *trow = trace ? trace + ((size_t)r.hb + r.id) * ORB_MAX_PASSES : nullptr;
        // a batch of the listed keys, all of its loads in flight; a cell of one
        // batch keeps it in registers for every round
        constexpr uint32_t kStep = (uint32_t)kFinBlock * kFinBatch;
        float v[kFinBatch];
        auto load_batch = [&](uint32_t k0) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < kFinBatch; ++u) {
                // key k of the cell: list j = the last with lex_j <= k
                const uint32_t k = k0 + (uint32_t)(kFinBlock * u + t);
                int j = 0;
#pragma unroll
                for (int st = 32; st > 0; st >>= 1)
                    if ((uint32_t)__shfl((int)lex, j + st, 64) <= k) j += st;
                const uint32_t at = (uint32_t)__shfl((int)kpos, j, 64) +
                                    (k - (uint32_t)__shfl((int)lex, j, 64));
                v[u] = k < m ? sel[at] : 0.0f;
            }
        };
        if (m <= kStep) load_batch(0u);
        Window wd{};
        if constexpr (PRED) {
            wd = windows[c];
            window_passes(wd, r.margin_l, r.margin_r, r.passes);
        }
        while (true) {
            const float lo = r.margin_l, hi = r.margin_r;
            __syncthreads();  // the last round (or cell) has read the tables
            if (t < kBins) {
                cand[t] = t ? candidate(t, lo, hi) : -INFINITY;
                hist[t] = 0u;
            }
            if (t == 0) cand[kBins] = INFINITY;
            __syncthreads();
            const float width = hi - lo;
            const float scale = width > 0.0f ? (float)kBins / width : 0.0f;
            uint32_t bl = 0;
            for (uint32_t k0 = 0; k0 < m; k0 += kStep) {
                if (m > kStep) load_batch(k0);  // uniform
#pragma unroll
                for (int u = 0; u < kFinBatch; ++u) {
                    const bool on = k0 + (uint32_t)(kFinBlock * u + t) < m;
                    const bool lt = on && v[u] < lo, in = on && !(v[u] < lo) && !(v[u] > hi);
                    bl += lt ? 1u : 0u;
                    int tj, bin = 0;
                    if (in) bin = bin_of<LE>(cand, v[u], lo, hi, scale, tj);
                    count_bin(hist, bin, in);
                }
            }
            bl = wave_sum(bl);
            if (lane == 0) sm[w] = bl;
            __syncthreads();  // the binning is complete
            if (w == 0) {
                // every round reads every listed key
                const uint32_t left = below + wave_sum(lane < kW ? sm[lane] : 0u);
                // P[j] = the keys below the margins + bins < j
                const uint32_t s0 = hist[4 * lane], s1 = s0 + hist[4 * lane + 1];
                const uint32_t s2 = s1 + hist[4 * lane + 2], s3 = s2 + hist[4 * lane + 3];
                const uint32_t base = left + wave_inclusive_scan(s3) - s3;
                P[4 * lane + 1] = base + s0;
                P[4 * lane + 2] = base + s1;
                P[4 * lane + 3] = base + s2;
                P[4 * lane + 4] = base + s3;
                if (lane == 0) P[0] = 0u;
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
                __builtin_amdgcn_wave_barrier();
                const RoundOut ro = replay_round(P, lo, hi, target, r.passes, lane, trow);
                if (lane == 0) {
                    s_lr[0] = ro.L;
                    s_lr[1] = ro.R;
                    s_pf[0] = ro.passes;
                    s_pf[1] = (ro.found ? 1 : 0) | (ro.node << 1);
                }
            }
            __syncthreads();
            RoundOut ro;
            ro.L = s_lr[0];
            ro.R = s_lr[1];
            ro.passes = s_pf[0];
            ro.found = (s_pf[1] & 1) != 0;
            ro.node = s_pf[1] >> 1;
            if (ro.found || ro.passes >= ORB_MAX_PASSES) {  // uniform
                if (PRED && !window_holds(wd, ro.L, ro.R)) {
                    if (t == 0) leave_alone(r, c, recs, level_passes);
                    break;
                }
                if (t == 0)
                    finish_round(r, c, ro, found_encoding(ro, lo, hi), recs, heap, level_passes,
                                 exists, status, &pm);
                break;
            }
            r.margin_l = ro.L;
            r.margin_r = ro.R;
            r.passes = ro.passes;
        }
    }
    if (t == 0) pm.flush(level_passes);
}

// ---------------------------------------------------------------------------
// large levels: the cut's window from a sample, one pass over the keys
// ---------------------------------------------------------------------------
// The rounds above read every key twice: once to find the window that holds
// the cut, once to count and pack the keys of that window.  Any window will
// do that the cut lies in, so here a sample of the keys (about 16384 a cell or
// more) picks it, 6 standard deviations wide each way, and the one full pass
// counts exactly:
//   k_p_sample  16-key segments spread evenly over each chunk into the cell's
//               1024 linear bins, and how far keys of one segment and of
//               adjacent ones agree
//   k_p_choose  per cell: the window.  Neighbours in memory may be neighbours in
//               space (particles grouped by object or by hash cell): a segment
//               is then worth as little as one draw, and the deviation grows
//               with it (sample_spread)
//   k_p_window  as k_b_hist_window: keys below and above the window counted,
//               its keys packed per chunk quarter and counted in the window's bins
//   (k_b_hist_reduce)
//   k_p_narrow  per cell: the bins that can hold the cut
// k_b_select gathers the keys of those bins and k_b_finish runs the
// controller's rounds on them from the cell's own margins.  Exact: counts
// grow with the candidate, so a candidate left of the kept bins has at most
// the keys left of them, whose difference is -3 or less, and the controller
// goes right there whatever the candidate's own count is; likewise on the
// other side.  A cell whose counts contradict its window (the sample missed) is
// left alone, counted, and built by the levels' second run.  Builds with a
// trace need every pass's count and keep the two full rounds.
// Measured at 2^27 keys, a level's search (keys read to cut found): 227 us,
// of it the window pass 147 (3.7 TB/s of keys), the sample 25, the gather 15 and
// the finish 18, from 296 with two full rounds.  Below kPredKeys a cell's sample would have
// to be a good part of its keys.
constexpr int kSegment = 16;         // keys of a segment (64 B, a DPP row of lanes)
constexpr int kSampleRow = kSampleBins + 128;  // the bins, pairs in a segment, pairs across two
constexpr int kSampleLines = 64;     // lines (of four segments) a block
constexpr int64_t kPredKeys = 65536;  // smallest expected cell of such a level
constexpr int64_t kPredLevelKeys = int64_t(1) << 24;  // and keys of the build

// Segment i of the 4 ls of chunk q starts here, then at the next multiple of 16
// in memory (the start moves with the chunk, so that no period of the input
// meets every segment).
__device__ inline uint32_t sample_segment(uint32_t q, uint32_t i, uint32_t ls)
{
    const uint32_t span = (uint32_t)kChunk / (4u * ls);  // a power of two, at least 64
    return i * span + ((q * 0x9e3779b1u) >> 20 & (span - 1u) & ~(uint32_t)(kSegment - 1));
}

__global__ __launch_bounds__(kBlock) void k_p_sample(
    const CellRec *__restrict__ recs, int32_t nCells, const uint32_t *__restrict__ first,
    const uint4 *__restrict__ chunk_desc, uint32_t max_chunks, const float *__restrict__ x,
    const float *__restrict__ y, const float *__restrict__ z, uint32_t ls, uint32_t *sample_hist)
{
    constexpr int kW = kBlock / 64;
    constexpr int kPer = kSampleLines / kW;  // 16 lines a wave, all in flight
    __shared__ uint32_t hist[kSampleRow];
    const int t = threadIdx.x, lane = t & 63, w = (int)uniform((uint32_t)t >> 6);
    const uint32_t total = first[nCells];
    const uint32_t per_block = (uint32_t)kSampleLines / ls;  // chunks a block
    for (uint32_t q0 = blockIdx.x * per_block; q0 < total; q0 += gridDim.x * per_block) {
        const uint32_t cell0 = uniform(chunk_record(chunk_desc, q0, max_chunks).z);
        for (int k = t; k < kSampleRow; k += kBlock) hist[k] = 0u;
        float v[kPer];
        uint32_t cell[kPer];
        bool ok[kPer];
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const uint32_t line = (uint32_t)(w * kPer + j);
            const uint32_t q = q0 + line / ls;
            const uint4 d = chunk_record(chunk_desc, q, max_chunks);
            const uint32_t b = uniform(d.x), e = uniform(d.y), axis = uniform(d.w);
            const uint32_t off = sample_segment(q, 4u * (line % ls) + (uint32_t)(lane / kSegment), ls);
            const uint32_t p = ((b + off + (uint32_t)(kSegment - 1)) & ~(uint32_t)(kSegment - 1)) +
                               (uint32_t)(lane % kSegment);
            cell[j] = uniform(d.z);
            ok[j] = q < total && axis <= 2u && p < e;
            v[j] = ok[j] ? axis_ptr(x, y, z, (int)axis)[p] : 0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const uint64_t on = __ballot(ok[j]);
            if (!on) continue;  // uniform
            const float lo = uniform(recs[cell[j]].margin_l), hi = uniform(recs[cell[j]].margin_r);
            const int bin = (int)__builtin_amdgcn_fmed3f((v[j] - lo) * sample_scale(hi - lo), 0.0f,
                                                         (float)(kSampleBins - 1));
            // the block's last chunks may be another cell's (uniform)
            const bool mine = cell[j] == cell0;
            auto count = [&](int at) __attribute__((always_inline)) {
                if (mine) atomicAdd(&hist[at], 1u);
                else atomicAdd(&sample_hist[(size_t)cell[j] * kSampleRow + at], 1u);
            };
            if (ok[j]) count(bin);
            // every fourth line, if whole, in pairs by the 16-bin group of the larger
            // key: within a segment (lanes i and 7 - i of every eight, 1 to 7 keys
            // apart) and with the next segment
            if (j % 4 == 0 && on == ~0ull) {
                const int near = (int)dpp_move<0x141, 0xf>((uint32_t)bin), far = __shfl_xor(bin, kSegment, 64);
                if (!(lane & 4)) count(kSampleBins + ((bin > near ? bin : near) >> 4));
                if (!(lane & kSegment)) count(kSampleBins + 64 + ((bin > far ? bin : far) >> 4));
            }
        }
        __syncthreads();
        for (int k = t; k < kSampleRow; k += kBlock)
            if (hist[k]) atomicAdd(&sample_hist[(size_t)cell0 * kSampleRow + k], hist[k]);
        __syncthreads();
    }
}

// The variance of the sample's count below the quantile `mid`, relative to that
// of independent draws: 1 for keys in no order, up to 16 where each segment lies
// on one side.  Lane l brings the sample's keys up to the end of its 16-bin group
// (inc, of s) and the pairs, within a segment and across two, whose larger key
// lies in it.  With F the share of keys below a bound, A and B the shares of
// pairs with both below it, within and across, a segment's count varies about
// its surroundings' by 16 (F - B) + 16 * 15 (A - B): keys that agree over many
// segments (long runs) are met by each of them and vary less.  A - B counts less
// two of its standard deviations (even keys stay at 1).  Taken at the bounds of
// the quantile's group; where neither splits the keys it is unknown: 16.
__device__ inline float sample_spread(uint32_t inc, float s, float mid, uint32_t in, uint32_t across)
{
    const int lane = threadIdx.x & 63;
    const uint32_t pi = wave_inclusive_scan(in), pa = wave_inclusive_scan(across);
    const float np = (float)lane_value(pi, 63);  // as many across
    const float F = s > 0.0f ? (float)inc / s : 0.0f;
    const float A = np > 0.0f ? (float)pi / np : 0.0f, B = np > 0.0f ? (float)pa / np : 0.0f;
    const float even = F * (1.0f - F);
    const bool known = even > 0.05f && np > 0.0f;
    const float noise = 2.0f * sqrtf((A * (1.0f - A) + B * (1.0f - B)) / np);
    const float v = known ? (F - B + (float)(kSegment - 1) * fmaxf(A - B - noise, 0.0f)) / even : 0.0f;
    // the quantile's group, and the bounds at its two ends
    const int g = __popcll(__ballot((float)inc <= mid));
    const bool use = known && (lane == g || lane + 1 == g);
    if (!__ballot(use)) return (float)kSegment;  // uniform
    const uint32_t m = wave_max(use ? __float_as_uint(fmaxf(v, 0.0f)) : 0u);  // (bits keep the order)
    return fminf(fmaxf(__uint_as_float(m), 1.0f), (float)kSegment);
}

// A wave per cell: the window from the sample, and the row cleared.
__global__ __launch_bounds__(kBlock) void k_p_choose(const CellRec *__restrict__ recs, int32_t nCells,
                                                     uint32_t *sample_hist, Window *__restrict__ windows,
                                                     uint32_t *__restrict__ window_bins)
{
    constexpr int kPer = kSampleBins / 64;  // 16 bins a lane
    const int lane = threadIdx.x & 63;
    const int32_t c = (int32_t)((blockIdx.x * kBlock + threadIdx.x) >> 6);
    if (c >= nCells || recs[c].flags) return;  // uniform
    uint4 *row = reinterpret_cast<uint4 *>(sample_hist + (size_t)c * kSampleRow) + lane * (kPer / 4);
    uint32_t *pairs = sample_hist + (size_t)c * kSampleRow + kSampleBins + lane;
    const uint32_t in = pairs[0], across = pairs[64];
    pairs[0] = 0u;
    pairs[64] = 0u;
    uint32_t h[kPer];
#pragma unroll
    for (int u = 0; u < kPer / 4; ++u) {
        const uint4 a = row[u];
        h[4 * u] = a.x;
        h[4 * u + 1] = a.y;
        h[4 * u + 2] = a.z;
        h[4 * u + 3] = a.w;
    }
#pragma unroll
    for (int u = 0; u < kPer / 4; ++u) row[u] = make_uint4(0u, 0u, 0u, 0u);
    uint32_t mine = 0;
#pragma unroll
    for (int u = 0; u < kPer; ++u) mine += h[u];
    const uint32_t inc = wave_inclusive_scan(mine);
    const float s = (float)lane_value(inc, 63);
    const int32_t nl = recs[c].nLeaf;
    const float ratio = (float)((nl + 1) / 2) / (float)nl;
    const float mid = s * ratio;
    const float dev =
        6.0f * sqrtf(s * ratio * (1.0f - ratio) * sample_spread(inc, s, mid, in, across)) + 8.0f;
    uint32_t below = 0, reach = 0, cum = inc - mine;  // whole bins under each bound
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        cum += h[u];
        below += (float)cum < mid - dev ? 1u : 0u;
        reach += (float)cum < mid + dev ? 1u : 0u;
    }
    const uint32_t bl = wave_sum(below), bu0 = wave_sum(reach) + 1u;
    const uint32_t bu = bu0 < (uint32_t)kSampleBins ? bu0 : (uint32_t)kSampleBins;
    // the window's share of the sample before each of its bins, as window bins
    // (no sample in it: by position)
    uint32_t ca = 0, cb = 0;  // the sample before bl and before bu
    cum = inc - mine;
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        const uint32_t bin = (uint32_t)(lane * kPer + u);
        ca = bin == bl ? cum : ca;
        cb = bin == bu ? cum : cb;
        cum += h[u];
    }
    ca = lane_value(ca, (int)(bl / kPer));
    cb = bu < (uint32_t)kSampleBins ? lane_value(cb, (int)(bu / kPer)) : lane_value(inc, 63);
    const float per = (float)kWindowBins / (float)(cb > ca ? cb - ca : bu - bl);
    uint32_t packed[kPer / 4] = {};
    cum = inc - mine;
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        const uint32_t bin = (uint32_t)(lane * kPer + u);
        const uint32_t at = cb > ca ? cum - ca : bin - bl;
        const uint32_t b = bin < bl ? 0u : bin >= bu ? (uint32_t)kWindowBins : (uint32_t)((float)at * per);
        packed[u / 4] |= (b < (uint32_t)kWindowBins ? b : (uint32_t)kWindowBins) << (8 * (u % 4));
        cum += h[u];
    }
    reinterpret_cast<uint4 *>(window_bins + (size_t)c * (kSampleBins / 4))[lane] =
        make_uint4(packed[0], packed[1], packed[2], packed[3]);
    if (lane == 0) {
        const float lo = recs[c].margin_l, hi = recs[c].margin_r, step = (hi - lo) / (float)kSampleBins;
        const float wl = bl == 0u ? lo : fminf(fmaxf(lo + (float)bl * step, lo), hi);
        const float wr = bu >= (uint32_t)kSampleBins ? hi : fminf(fmaxf(lo + (float)bu * step, wl), hi);
        windows[c] = Window{wl, wr, wl, wr, lo, sample_scale(hi - lo), bl, bu};
    }
}

// Window pass (see k_b_hist_window for its packing and masks).
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_p_window(
    const Window *__restrict__ windows, const uint32_t *__restrict__ window_bins, int32_t nCells,
    const uint32_t *__restrict__ first, const uint4 *__restrict__ chunk_desc, uint32_t max_chunks,
    const float *__restrict__ x,
    const float *__restrict__ y, const float *__restrict__ z, uint16_t *__restrict__ chunk_hist,
    float *__restrict__ pack, uint32_t *__restrict__ comp, uint64_t *__restrict__ masks, int rev)
{
    constexpr int kW = kBlock / 64;
    constexpr int kPerWave = kMaskWords / kW;  // 16 loads of 64 keys
    __shared__ uint32_t hist[kBins];
    __shared__ uint32_t tab[kSampleBins / 4];
    static_assert(kSampleBins / 4 == kBlock, "a word of the table per thread");
    __shared__ uint32_t sm[4];
    __shared__ float wkeys[kW][kChunk / kW];     // each wave's window keys, packed
    __shared__ uint64_t words[kW][2][kPerWave];  // each wave's mask words, staged
    const int t = threadIdx.x, lane = t & 63, w = (int)uniform((uint32_t)t >> 6);
    const uint64_t lanes_below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    const uint32_t total = first[nCells];
    for (uint32_t q0 = blockIdx.x;; q0 += gridDim.x) {
        const uint32_t q = rev && q0 < total ? total - 1u - q0 : q0;  // from the last (rev)
        const uint4 d = chunk_record(chunk_desc, q, max_chunks);
        const uint32_t b = uniform(d.x), e = uniform(d.y), cell = uniform(d.z);
        const uint32_t axis = uniform(d.w);
        keep_values(b, e, cell, axis);  // the whole record, in flight with total
        if (q >= total) break;
        if (axis > 2u) continue;  // uniform: the cell is not searched
        const uint32_t sb = (uint32_t)(w * kPerWave * 64);  // chunk position of the quarter
        const uint32_t tw = window_bins[(size_t)cell * kBlock + (uint32_t)t];  // issued before the keys
        float v[kPerWave];
        issue_chunk_loads(x, y, z, true, d, sb, lane, v);
        Window wd;
        wd.lo = uniform(windows[cell].lo);
        wd.hi = uniform(windows[cell].hi);
        wd.base = uniform(windows[cell].base);
        wd.scale = uniform(windows[cell].scale);
        wd.bl = uniform(windows[cell].bl);
        wd.bu = uniform(windows[cell].bu);
        const float lo = wd.lo, hi = wd.hi;
        tab[t] = tw;
        hist[t] = 0u;
        __syncthreads();
        const uint32_t len = e - b;
        uint32_t below = 0, packed = 0;  // wave-uniform
        float *dst = pack + b + sb;
        float *wk = wkeys[w];
        auto scan = [&](auto full) __attribute__((always_inline)) {
            static_for<0, kPerWave>([&](auto jc) __attribute__((always_inline)) {
                constexpr int j = decltype(jc)::value;
                uint64_t valid = ~0ull;
                if constexpr (!decltype(full)::value) {
                    const uint32_t p0 = sb + 64u * (uint32_t)j;  // chunk position of lane 0
                    valid = p0 >= len ? 0ull
                                      : (len - p0 >= 64u ? ~0ull : (1ull << (len - p0)) - 1ull);
                }
                const float vj = v[j];
                const uint64_t mB = __ballot(vj < lo) & valid;
                const uint64_t mG = __ballot(vj > hi) & valid;
                const uint64_t mW = valid & ~mB & ~mG;
                below += (uint32_t)__popcll(mB);
                if (lane == 0) {  // staged by one lane, as in k_b_hist_window
                    words[w][0][j] = mG;
                    words[w][1][j] = mW;
                }
                if (mW) {  // wave-uniform
                    if ((mW >> lane) & 1ull) {
                        const uint32_t slot = packed + (uint32_t)__popcll(mW & lanes_below);
                        dst[slot] = vj;
                        wk[slot] = vj;
                    }
                    packed += (uint32_t)__popcll(mW);
                }
            });
        };
        if (len == (uint32_t)kChunk) scan(std::true_type{});  // uniform
        else scan(std::false_type{});
        const uint32_t mine = len > sb ? (len - sb < 1024u ? len - sb : 1024u) : 0u;
        const uint32_t above = mine - below - packed;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        __builtin_amdgcn_wave_barrier();
        const uint64_t mineG = lane < kPerWave ? words[w][0][lane] : 0ull;
        const uint64_t mineW = lane < kPerWave ? words[w][1][lane] : 0ull;
        for (uint32_t k = (uint32_t)lane; k < packed; k += 64)
            atomicAdd(&hist[window_bin(wk[k], wd, reinterpret_cast<const uint8_t *>(tab))], 1u);
        uint64_t *mq = masks + (size_t)q * (2 * kMaskWords) + w * kPerWave;
        if (lane < kPerWave) {
            mq[lane] = mineG;
            mq[kMaskWords + lane] = mineW;
        }
        if (lane == 0) {
            comp[8 * (size_t)q + w] = packed;
            sm[w] = below | (above << 16);  // each <= 1024
        }
        __syncthreads();
        const uint32_t ba = sm[0] + sm[1] + sm[2] + sm[3];
        if (t == 0) comp[8 * (size_t)q + 4] = ba & 0xffffu;
        uint32_t sum = hist[t];
        if (t == 0) sum += ba & 0xffffu;
        if (t == kBins - 1) sum += ba >> 16;
        chunk_hist[(size_t)q * kBins + t] = (uint16_t)sum;
        __syncthreads();  // the next chunk rewrites hist and sm
    }
}

// A float32 as an unsigned number of the same order, and back.
__device__ inline uint32_t ordered(float v)
{
    const uint32_t u = __float_as_uint(v);
    return u & 0x80000000u ? ~u : u | 0x80000000u;
}
__device__ inline float from_ordered(uint32_t u)
{
    return __uint_as_float(u & 0x80000000u ? u & 0x7fffffffu : ~u);
}

// A wave per cell: from the counts of the window's bins (bin 0: keys below the
// window, 255: above), the bins [b1, b2] that can hold the cut, the floats
// [klo, khi] that lie in them, and the cell's lists with the keys left of them.  A cell whose counts contradict the window
// is left alone (see above).
__global__ __launch_bounds__(kBlock) void k_p_narrow(CellRec *recs, int32_t nCells, uint32_t *cell_hist,
                                                     Window *__restrict__ windows,
                                                     const uint32_t *__restrict__ window_bins,
                                                     const uint32_t *__restrict__ first,
                                                     unsigned long long *__restrict__ sel_lists,
                                                     int32_t *level_passes)
{
    __shared__ uint4 tables[kBlock / 64][kSampleBins / 16];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int32_t c = (int32_t)((blockIdx.x * kBlock + threadIdx.x) >> 6);
    if (c >= nCells || recs[c].flags) return;  // uniform
    uint4 *row = reinterpret_cast<uint4 *>(cell_hist + (size_t)c * kBins);
    const uint4 h4 = row[lane];
    tables[w][lane] = reinterpret_cast<const uint4 *>(window_bins + (size_t)c * (kSampleBins / 4))[lane];
    row[lane] = make_uint4(0u, 0u, 0u, 0u);  // the next level adds to zero
    const uint32_t s0 = h4.x, s1 = s0 + h4.y, s2 = s1 + h4.z, s3 = s2 + h4.w;
    const uint32_t base = wave_inclusive_scan(s3) - s3;
    // P[4 lane + 1 + q] (P[j] = keys in bins below j)
    const uint32_t pv[4] = {base + s0, base + s1, base + s2, base + s3};
    const float target = difference_target(uniform(recs[c].end) - uniform(recs[c].begin),
                                           (int32_t)uniform((uint32_t)recs[c].nLeaf));
    uint32_t left = 0, right = 0;  // j in [1, 255] with difference <= -3, resp. < 3
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const bool in = 4 * lane + 1 + q < kBins;
        const int32_t df = difference_from_target(pv[q], target);
        left += (uint32_t)__popcll(__ballot(in && df <= -3));
        right += (uint32_t)__popcll(__ballot(in && df < 3));
    }
    // the last j with difference <= -3 is `left` (differences grow with j),
    // the first with difference >= 3 is right + 1
    const Window wd = windows[c];
    const bool low_ok = left >= 1u || wd.lo == recs[c].margin_l;    // P[1]: the keys below the window
    const bool high_ok = right < 255u || wd.hi == recs[c].margin_r;  // P[255]: all but those above
    const uint32_t b1 = left >= 1u ? left : 1u, b2 = right < 255u ? right : 254u;
    const uint32_t cnt = lane_value(b1 & 3u ? ((b1 & 3u) == 1u ? pv[0] : (b1 & 3u) == 2u ? pv[1] : pv[2]) : pv[3],
                                    (int)((b1 - 1u) >> 2));  // P[b1]
    if (!low_ok || !high_ok || b1 > 254u || b2 < 1u) {
        if (lane == 0) {
            recs[c].flags = 1;
            atomicAdd(&level_passes[recs[c].lp & ~63], 1);
        }
        return;
    }
    const uint32_t f = first[c];
    const SelLists sl(f, first[c + 1] - f);
    if ((uint32_t)lane < sl.R)
        sel_lists[sl.start_chunk((uint32_t)lane)] = lane == 0 ? (unsigned long long)cnt << 32 : 0ull;
    // both bins hold keys (their counts decide), so each end lies in the window;
    // a 64-way search over the floats between, the table in LDS
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    __builtin_amdgcn_wave_barrier();
    const uint8_t *tab = reinterpret_cast<const uint8_t *>(tables[w]);
    const uint32_t olo = ordered(wd.lo), ohi = ordered(wd.hi) + 1u;
    float klo = wd.lo, khi = wd.hi;
    if (window_bin(wd.lo, wd, tab) < b1)  // uniform
        klo = from_ordered(1u + wave_last_true(olo, ohi, [&](uint32_t k) {
            return window_bin(from_ordered(k), wd, tab) < b1;
        }));
    if (window_bin(wd.hi, wd, tab) > b2)
        khi = from_ordered(wave_last_true(olo, ohi, [&](uint32_t k) {
            return window_bin(from_ordered(k), wd, tab) <= b2;
        }));
    if (lane == 0) {
        windows[c].klo = klo;
        windows[c].khi = khi;
    }
}

// ---------------------------------------------------------------------------
// weighted rounds (workload weights w(p_i), documentation/notes.tex:259-271,
// 326-336): the bins hold weight sums (64-bit) instead of counts, and the
// controller compares the weight left of each candidate with the cell's
// weight times the left share.  Every round bins every key of a searching
// cell (no window packing), so a row's total is the chunk's weight and a
// cell histogram's total the cell's weight.
// ---------------------------------------------------------------------------
// The weights of a chunk (record dd) as issue_chunk_loads reads its keys: past
// the chunk's end 0.
template <int kPerWave>
__device__ inline void issue_weight_loads(const uint32_t *wgt, uint4 dd, uint32_t sb, int lane,
                                          uint32_t (&wv)[kPerWave])
{
    const uint32_t b = uniform(dd.x), e = uniform(dd.y);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint32_t *>(wgt) + b, 0, (int)((e - b) * 4u), 0x00020000);
#pragma unroll
    for (int j = 0; j < kPerWave; ++j)
        wv[j] = __builtin_amdgcn_raw_buffer_load_b32(
            wr, (int)((sb + (uint32_t)lane) * 4u + 256u * (uint32_t)j), 0, 0);
}

// A wave's keys and weights into the block's row of weight sums: keys outside
// the margins add up in registers (as atomics they would share two words) and
// keys of weight 0, those past the chunk's end among them, add nothing.
template <int LE, int kPerWave>
__device__ inline void bin_weights(const float (&v)[kPerWave], const uint32_t (&wv)[kPerWave], float lo,
                                   float hi, unsigned long long *hist, int lane)
{
    const float width = hi - lo;
    const float scale = width > 0.0f ? (float)kBins / width : 0.0f;
    const float lim = 0.5f - bin_tolerance(lo, hi, scale);
    uint64_t below = 0ull, above = 0ull;
    static_for<0, kPerWave>([&](auto jc) __attribute__((always_inline)) {
        constexpr int j = decltype(jc)::value;
        const float vj = v[j];
        const bool lt = vj < lo, gt = vj > hi;
        below += lt ? wv[j] : 0u;
        above += gt ? wv[j] : 0u;
        if (!lt && !gt && wv[j]) {
            int bin;
            if (!bin_estimate(vj, lo, scale, lim, bin)) bin = bin_walk<LE>(vj, lo, hi);
            atomicAdd(&hist[bin], (unsigned long long)wv[j]);
        }
    });
    below = wave_sum(below);
    above = wave_sum(above);
    if (lane == 0) {
        if (below) atomicAdd(&hist[0], (unsigned long long)below);
        if (above) atomicAdd(&hist[kBins - 1], (unsigned long long)above);
    }
}

template <int LE>
__global__ __launch_bounds__(kBlock) void k_bw_hist(
    const CellRec *__restrict__ recs, int32_t nCells, const uint32_t *__restrict__ first,
    const uint4 *__restrict__ chunk_desc, uint32_t max_chunks, const float *__restrict__ x,
    const float *__restrict__ y, const float *__restrict__ z, const uint32_t *__restrict__ wgt,
    uint64_t *__restrict__ chunk_hist_w)
{
    __shared__ unsigned long long hist[kBins];
    constexpr int kPerWave = kMaskWords / (kBlock / 64);  // 16 loads of 64 keys and weights
    const int t = threadIdx.x, lane = t & 63, w = (int)uniform((uint32_t)t >> 6);
    const uint32_t sb = (uint32_t)(w * kPerWave * 64);
    const uint32_t total = first[nCells];
    for (uint32_t q = blockIdx.x;; q += gridDim.x) {
        const uint4 d = chunk_record(chunk_desc, q, max_chunks);
        const uint32_t b = uniform(d.x), e = uniform(d.y), cell = uniform(d.z);
        const uint32_t axis = uniform(d.w);
        keep_values(b, e, cell, axis);
        if (q >= total) break;
        if (axis > 2u) continue;  // uniform: the cell is not searched
        const CellRec &r = recs[cell];
        if (r.found) continue;    // uniform: an earlier round found the cut
        float v[kPerWave];
        issue_chunk_loads(x, y, z, true, d, sb, lane, v);
        uint32_t wv[kPerWave];
        issue_weight_loads(wgt, d, sb, lane, wv);
        const float lo = uniform(r.margin_l), hi = uniform(r.margin_r);
        hist[t] = 0ull;
        __syncthreads();
        bin_weights<LE>(v, wv, lo, hi, hist, lane);
        __syncthreads();
        chunk_hist_w[(size_t)q * kBins + t] = hist[t];
        __syncthreads();  // the next chunk rewrites hist
    }
}

// Chunk rows into cell rows (64-bit): block g takes chunks [64g, 64g + 64),
// thread t bin t, one atomic per (block, cell, bin).
__global__ __launch_bounds__(kBlock) void k_bw_reduce(const CellRec *recs, int32_t nCells,
                                                      const uint32_t *first,
                                                      const uint32_t *chunk_cell,
                                                      const uint64_t *chunk_hist_w,
                                                      uint64_t *cell_hist_w)
{
    __shared__ int32_t scell[kReduceRows];
    const uint32_t total = first[nCells];
    const int t = threadIdx.x;
    for (uint32_t q0 = blockIdx.x * (uint32_t)kReduceRows; q0 < total;
         q0 += gridDim.x * (uint32_t)kReduceRows) {
        const uint32_t nrows =
            total - q0 < (uint32_t)kReduceRows ? total - q0 : (uint32_t)kReduceRows;
        if (t < kReduceRows) {
            int32_t cl = -1;
            if ((uint32_t)t < nrows) {
                const uint32_t cell = chunk_cell[q0 + t];
                const CellRec &r = recs[cell];
                if (!(r.found || r.flags) && r.axis >= 0 && r.axis <= 2) cl = (int32_t)cell;
            }
            scell[t] = cl;
        }
        __syncthreads();
        int32_t cur = -1;
        unsigned long long acc = 0;
        for (uint32_t u0 = 0; u0 < nrows; u0 += 16u) {
            // 16 rows' loads in flight: 22 -> 11.5 us a launch at 2^24 keys
            // against one row after another
            uint64_t v[16];
#pragma unroll
            for (uint32_t u = 0; u < 16u; ++u)
                v[u] = u0 + u < nrows && scell[u0 + u] >= 0
                           ? chunk_hist_w[(size_t)(q0 + u0 + u) * kBins + t] : 0ull;
#pragma unroll
            for (uint32_t u = 0; u < 16u; ++u) {
                const int32_t cl = u0 + u < nrows ? scell[u0 + u] : cur;
                if (cl != cur) {
                    if (cur >= 0 && acc)
                        atomicAdd(reinterpret_cast<unsigned long long *>(cell_hist_w) +
                                      (size_t)cur * kBins + t,
                                  acc);
                    cur = cl;
                    acc = 0;
                }
                acc += v[u];
            }
        }
        if (cur >= 0 && acc)
            atomicAdd(reinterpret_cast<unsigned long long *>(cell_hist_w) + (size_t)cur * kBins + t,
                      acc);
        __syncthreads();  // scell is rewritten for the next tile
    }
}

// One wave per cell: prefix sums of the cell's weight histogram in registers,
// the cell's weight (the row's total), then up to 8 passes of the controller.
__global__ __launch_bounds__(kBlock) void k_bw_replay(CellRec *recs, int32_t nCells,
                                                      uint64_t *cell_hist_w, orb_cell *heap,
                                                      uint64_t *trace, int32_t *level_passes,
                                                      uint8_t *exists, int32_t *status)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int32_t c = blockIdx.x * 4 + w;
    if (c >= nCells) return;  // uniform per wave
    CellRec r = recs[c];
    if (r.found || r.flags || r.axis < 0 || r.axis > 2) return;
    uint64_t *row = cell_hist_w + (size_t)c * kBins;
    uint64_t h[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        h[i] = row[4 * lane + i];
        row[4 * lane + i] = 0ull;  // the next round starts from zero
    }
    const uint64_t s0 = h[0], s1 = s0 + h[1], s2 = s1 + h[2], s3 = s2 + h[3];
    const uint64_t base = wave_inclusive_scan(s3) - s3;
    // P[4 lane + 1 + q] (P[j] = weight in bins below j)
    const uint64_t pv[4] = {base + s0, base + s1, base + s2, base + s3};
    const uint64_t weight = lane_value(pv[3], 63);  // every key of the cell was binned
    const float target = difference_target_w(weight, r.nLeaf);
    const RoundOut ro = replay_round_lanes(pv, r.margin_l, r.margin_r, target, r.passes, lane,
                                           trace ? trace + ((size_t)r.hb + r.id) * ORB_MAX_PASSES
                                                 : nullptr);
    if (lane != 0) return;
    // found: the partition reads the keys (no stopper counts from the bins)
    finish_round(r, c, ro, ro.found ? 1 : 0, recs, heap, level_passes, exists, status);
}

// ---------------------------------------------------------------------------
// LDS-resident subtree kernel
// ---------------------------------------------------------------------------
struct SubCell {
    orb_cell cell;
    uint32_t lb, le;   // local range in the block's LDS arrays
    int32_t valid;
    int32_t pad;
};

// Word j of a cell record held the same in every lane (0 past its end), so
// that lane j can write it.
constexpr int kCellWords = (int)(sizeof(orb_cell) / 4);
__device__ inline uint32_t cell_word(const orb_cell &c, int j)
{
    const uint32_t *p = reinterpret_cast<const uint32_t *>(&c);
    uint32_t v = 0u;
#pragma unroll
    for (int q = 0; q < kCellWords; ++q) v = j == q ? p[q] : v;
    return v;
}

// An LDS address as the buffer-to-LDS loads take it (the LDS address space).
typedef __attribute__((address_space(3))) void LdsVoid;
__device__ inline LdsVoid *lds_ptr(void *p)
{
    return (LdsVoid *)p;
}

__device__ inline void lds_wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    __builtin_amdgcn_wave_barrier();
}

// Keys of [pb, pe) in LDS below the cut (lt) or at most the cut (le), summed
// over the wave: one ballot + popcount per 64 keys, four LDS reads in flight.
__device__ inline uint32_t wave_count_below(const float *key, uint32_t pb, uint32_t pe, float cut,
                                            int le_cmp, int lane)
{
    uint32_t cnt = 0;
    for (uint32_t base = pb; base < pe; base += 256u) {
        float v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const uint32_t p = base + (uint32_t)(64 * u + lane);
            v[u] = p < pe ? key[p] : INFINITY;  // never below a finite cut
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const bool below = le_cmp ? (v[u] <= cut) : (v[u] < cut);
            cnt += (uint32_t)__popcll(__ballot(below));
        }
    }
    return cnt;
}

// The weight of the keys of [pb, pe) below the cut (weighted build), summed
// over the wave in 64 bits.
__device__ inline uint64_t wave_weight_below(const float *key, const uint32_t *wgt, uint32_t pb,
                                             uint32_t pe, float cut, int le_cmp, int lane)
{
    uint64_t s = 0;
    for (uint32_t p = pb + (uint32_t)lane; p < pe; p += 64u) {
        const float v = key[p];
        const bool below = le_cmp ? (v <= cut) : (v < cut);
        s += below ? (uint64_t)wgt[p] : 0ull;
    }
    return wave_sum(s);
}

// The total weight of [pb, pe), summed over the wave.
__device__ inline uint64_t wave_weight_total(const uint32_t *wgt, uint32_t pb, uint32_t pe, int lane)
{
    uint64_t s = 0;
    for (uint32_t p = pb + (uint32_t)lane; p < pe; p += 64u) s += wgt[p];
    return wave_sum(s);
}

// The left count (unweighted) or left weight (weighted) of [pb, pe).
template <bool W>
__device__ inline uint64_t wave_left(const float *key, const uint32_t *wgt, uint32_t pb, uint32_t pe,
                                     float cut, int le_cmp, int lane)
{
    if constexpr (W) return wave_weight_below(key, wgt, pb, pe, cut, le_cmp, lane);
    else return wave_count_below(key, pb, pe, cut, le_cmp, lane);
}

// The termination rule's difference for a left count or weight.
template <bool W>
__device__ inline int64_t left_difference(uint64_t left, float target)
{
    if constexpr (W) return difference_from_target_w(left, target);
    else return difference_from_target((uint32_t)left, target);
}

// The LDS capacity of the subtree kernel (keys of one subtree root) per
// payload: x, y, z (12 B), the two 16-bit stopper lists (4 B), with ids a
// 16-bit local index (2 B), with weights the weight (4 B) and 64-bit
// histogram slots; 155-163 KB of gfx950's 160 KiB LDS in each variant.  A
// level's cells sit within a few keys of n / 2^(l-1), so the plain
// capacity stays a little above 8192 for a level of 8192-key cells to
// qualify whole.
// A block of 512 threads holds half as much (plain particles only): two share
// a CU, so that one's barriers, replays and children lie under the other's
// binning; levels of many cells take it.
template <bool IDS, bool W, int kThreads = 1024>
struct SubCap {
    static constexpr int value = W ? 5120 : (IDS ? 7680 : 8832);
};
template <>
struct SubCap<false, false, 512> {
    static constexpr int value = 4224;
};

static int32_t subtree_capacity(const Ctx &c)
{
    if (c.weighted) return SubCap<true, true>::value;
    return c.track_ids ? SubCap<true, false>::value : SubCap<false, false>::value;
}

// Every remaining level of the subtree under a small cell, in LDS: the cell's
// x, y, z (and ids' local index, weights) are loaded once, every remaining
// level is built there, and x, y, z are written back once.
//
// A depth's cells are taken up to 16 at a time (a slot each; 8 in a block of
// 512 threads); a slot has 16 / (cells) waves when the depth has fewer cells.  The bisection
// controller (orbit.cpp:149-231) runs in rounds of 8 passes, as the chunk
// path's histogram rounds do: the slot's waves bin the cell's keys over the
// 255 candidate cuts of its margins into a 256-bin LDS histogram (two 16-bit
// bins per word; 64-bit bins of weight sums with W), and the slot's first
// wave prefix-sums it in place and replays up to 8 passes (replay_round),
// exact by construction.  The Hoare partition (partition.cpp:28-60) is the
// stopper closed form: stopper lists by ballot scans, the crossing K by a
// 64-way search, K swaps, the final swap.  Every barrier is reached by all
// waves the same number of times.
// IDS: particle ids move with the particles; a 16-bit local index rides along
// in LDS and the ids are permuted once at the write-back.  W: workload
// weights ride along in LDS and the histograms sum weights.
template <bool IDS, bool W, int kSubBlock>
__global__ __launch_bounds__(kSubBlock) void k_b_subtree(const CellRec *recs, int32_t nCells,
                                                         orb_cell *heap, uint8_t *exists,
                                                         uint8_t *sub, uint32_t *ranges, float *x,
                                                         float *y, float *z, int le_cmp,
                                                         uint64_t *trace, int32_t *level_passes,
                                                         int32_t *status, uint32_t *pid,
                                                         uint32_t *wgt, int32_t group)
{
    constexpr int kCap = SubCap<IDS, W, kSubBlock>::value;
    constexpr int kSubWaves = kSubBlock / 64;  // histogram slots
    using HistWord = typename std::conditional<W, unsigned long long, uint32_t>::type;
    constexpr int kHistWords = W ? kBins : kBins / 2;  // W: a bin per word; else two
    __shared__ float sx[kCap], sy[kCap], sz[kCap];
    __shared__ uint32_t sw[W ? kCap : 1];
    // the two stopper lists (16-bit), reused as the cell's 32-bit ids at the end
    __shared__ uint32_t spos_raw[kCap];
    __shared__ uint16_t sidx[IDS ? kCap : 1];
    uint16_t *const slpos = reinterpret_cast<uint16_t *>(spos_raw);
    uint16_t *const srpos = slpos + kCap;
    // during a histogram round the stopper lists are free: each wave queues
    // its slow keys there (and with W their weights in the second half)
    constexpr int kQueue = ((W ? kCap / 2 : kCap) / kSubWaves) & ~63;
    static_assert(kQueue >= 64 && kSubWaves * kQueue <= (W ? kCap / 2 : kCap), "queue fits");
    __shared__ HistWord shist[kSubWaves][kHistWords];
    __shared__ SubCell scells[2][kSmallLeaves];  // a depth's cells and the next's
    __shared__ float sL[kSubWaves], sR[kSubWaves];
    __shared__ int32_t sPasses[kSubWaves], sFound[kSubWaves];
    __shared__ uint64_t sWt[kSubWaves];
    __shared__ uint32_t sTL[kSubWaves], sTR[kSubWaves], sK[kSubWaves], sI[kSubWaves];
    __shared__ int32_t s_ncur, s_nvalid, s_err;
    // the block's pass maxima per level of the build slot in s_lp0, flushed
    // with one atomicMax per level when the slot changes and at the end
    __shared__ int32_t s_lpmax[64];
    __shared__ int32_t s_lp0;
    __shared__ uint64_t s_gmask;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const uint64_t lanes_below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    if (t < 64) s_lpmax[t] = 0;
    if (t == 0) s_lp0 = -1;
    // every wave histogram starts clear and is left clear by the round that
    // used it
    for (int i = t; i < kSubWaves * kHistWords; i += kSubBlock) (&shist[0][0])[i] = 0;
    __syncthreads();
    // groups of `group` consecutive cells (a power of two <= 64): wave 0 reads
    // the group's flags in one load and the block takes the subtree roots
    // among them, so a level with few roots (or none) costs a few loads per
    // block, not one per cell
    for (int32_t g0 = blockIdx.x * group; g0 < nCells; g0 += gridDim.x * group) {
    if (w == 0) {
        const int32_t cc = g0 + lane;
        const bool root = lane < group && cc < nCells && recs[cc].flags == 2;
        const uint64_t m = __ballot(root);
        if (lane == 0) s_gmask = m;
    }
    __syncthreads();
    uint64_t gm = s_gmask;  // uniform
    __syncthreads();        // read before wave 0 rewrites it
    while (gm) {
    const int32_t c = g0 + __builtin_ctzll(gm);
    gm &= gm - 1ull;
    const CellRec rr = recs[c];
    if ((rr.lp - (rr.lp & 63)) != s_lp0) {
        if (t < 64 && s_lp0 >= 0 && s_lpmax[t] > 0) atomicMax(&level_passes[s_lp0 + t], s_lpmax[t]);
        __syncthreads();
        if (t < 64) s_lpmax[t] = 0;
        if (t == 0) s_lp0 = rr.lp - (rr.lp & 63);
        __syncthreads();
    }
    const uint32_t begin = rr.begin, n = rr.end - rr.begin;
    const int64_t hb = rr.hb;
    const int32_t level = rr.lp & 63, lmax = rr.lmax;
    int32_t *st = status + rr.st;
    if (n > (uint32_t)kCap) {
        // the level records hand over at most kCap keys; refuse anything else
        if (t == 0) report_error(st, level, kErrSplit, rr.id);
        continue;
    }
    // the root cell's 13 words, one per lane of wave 0 (no struct copy)
    uint32_t root_w = 0u;
    if (t < kCellWords) root_w = reinterpret_cast<const uint32_t *>(heap + hb + rr.id)[t];
    {
        // the cell's arrays straight from memory into LDS, through no
        // registers: wave w takes the 64-key pieces that start at
        // 64 w + 1024 u below n, one buffer load to LDS per piece and array,
        // all in flight together.  The range check is the cell's byte count:
        // keys past n land as 0 in slots below kCap (a piece starts below
        // n <= kCap, and kCap is a multiple of 64).
        static_assert(kCap % 64 == 0, "whole 64-key pieces");
        const int nb = (int)(n * 4u);
        const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(x + begin, 0, nb, 0x00020000);
        const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc(y + begin, 0, nb, 0x00020000);
        const __amdgpu_buffer_rsrc_t rz = __builtin_amdgcn_make_buffer_rsrc(z + begin, 0, nb, 0x00020000);
        for (uint32_t k0 = 64u * (uint32_t)w; k0 < n; k0 += (uint32_t)kSubBlock) {
            const int vo = (int)(4u * (k0 + (uint32_t)lane));
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, lds_ptr(sx + k0), 4, vo, 0, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ry, lds_ptr(sy + k0), 4, vo, 0, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rz, lds_ptr(sz + k0), 4, vo, 0, 0, 0);
            if constexpr (W) {
                const __amdgpu_buffer_rsrc_t rw =
                    __builtin_amdgcn_make_buffer_rsrc(wgt + begin, 0, nb, 0x00020000);
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, lds_ptr(sw + k0), 4, vo, 0, 0, 0);
            }
        }
        if (IDS)
            for (uint32_t k = (uint32_t)t; k < n; k += (uint32_t)kSubBlock) sidx[k] = (uint16_t)k;
        // the loads have written LDS before the barrier below lets any wave read it
        __builtin_amdgcn_s_waitcnt(0);
    }
    int cb = 0;  // scells[cb]: this depth's cells
    if (t < kCellWords) reinterpret_cast<uint32_t *>(&scells[0][0].cell)[t] = root_w;
    if (t == 0) {
        scells[0][0].lb = 0;
        scells[0][0].le = n;
        scells[0][0].valid = 1;
        s_ncur = 1;
        s_nvalid = 1;
        s_err = 0;
    }
    __syncthreads();
    for (int32_t l = level; l <= lmax; ++l) {
        const int32_t ncur = s_ncur;
        if (ncur == 0 || s_nvalid == 0 || s_err) break;
        if (2 * ncur > kSmallLeaves) {
            // cannot happen while the root has <= kSmallLeaves leaves; refuse
            // rather than leave the subtree half built
            if (t == 0) report_error(st, l, kErrSplit, rr.id);
            break;
        }
        const int nslots = ncur >= kSubWaves ? kSubWaves : ncur;   // ncur is a power of two
        const int g = kSubWaves / nslots;                           // waves per cell
        const int nbatch = ncur >= kSubWaves ? ncur / kSubWaves : 1;
        const int slot = w / g, part = w % g, w0 = slot * g;
        for (int bt = 0; bt < nbatch; ++bt) {
            const int32_t k = bt * nslots + slot;
            const SubCell sc = scells[cb][k];
            const bool valid = sc.valid != 0;
            orb_cell cl = sc.cell;
            const uint32_t lb = sc.lb, le = sc.le, m = le - lb;
            const float *key = cl.cutAxis == 0 ? sx : (cl.cutAxis == 1 ? sy : sz);
            if (part == 0 && lane == 0) {
                scells[cb ^ 1][2 * k].valid = 0;
                scells[cb ^ 1][2 * k + 1].valid = 0;
            }
            // this wave's part of the cell
            const uint32_t seg = ((m + (uint32_t)g - 1u) / (uint32_t)g + 63u) & ~63u;
            uint32_t pb = lb + (uint32_t)part * seg, pe = pb + seg;
            if (pb > le) pb = le;
            if (pe > le) pe = le;
            float target;
            if constexpr (W) {
                // the cell's weight (count.cpp:14-17 with weights): the g waves
                // of the cell add their parts through LDS
                const uint64_t pw = valid ? wave_weight_total(sw, pb, pe, lane) : 0ull;
                if (lane == 0) sWt[w] = pw;
                __syncthreads();
                const uint64_t tot = wave_sum(lane < g ? (uint64_t)sWt[w0 + lane] : 0ull);
                target = difference_target_w(tot, cl.nLeafCells);
            } else {
                target = difference_target(m, cl.nLeafCells);
            }
            uint64_t *trow = trace ? trace + ((size_t)hb + cl.id) * ORB_MAX_PASSES : nullptr;
            float L = cl.cutMarginLeft, R = cl.cutMarginRight;
            int32_t passes = 0;
            bool found = false;
            // the slot's g waves bin their parts into the slot's one histogram
            // (its first wave's); that wave replays from it and clears it.  Two
            // barriers per round; amask (the same in every wave) holds the
            // batch's slots still searching.
            HistWord *const myhist = shist[w0];
            uint32_t amask = (uint32_t)__ballot(lane < nslots && scells[cb][bt * nslots + lane].valid);
            while (amask) {
                const bool act = ((amask >> slot) & 1u) != 0u;
                if (act) {
                    const float width = R - L;
                    const float scale = width > 0.0f ? (float)kBins / width : 0.0f;
                    const float lim = 0.5f - bin_tolerance(L, R, scale);
                    // keys outside [L, R] (most of them after the first
                    // round) are counted in registers and added to bins 0 and
                    // 255 once per wave: as atomics they would all hit the
                    // same two LDS words
                    uint32_t nbelow = 0, nabove = 0;     // wave-uniform counts
                    uint64_t wbelow = 0ull, wabove = 0ull;  // W: this lane's weights
                    // keys too close to a bin edge for the estimate (about 1%
                    // in a first round) queue in the wave's part of the free
                    // stopper-list space and are walked 64 at a time, not one
                    // divergent walk per load that holds one
                    float *const qk = reinterpret_cast<float *>(spos_raw) + w * kQueue;
                    uint32_t *const qw = spos_raw + (W ? kCap / 2 : 0) + w * kQueue;  // W: weights
                    uint32_t qn = 0;  // wave-uniform
                    auto drain = [&]() {
                        lds_wave_sync();  // the queue's stores before its loads
                        for (uint32_t k = (uint32_t)lane; k < qn; k += 64u) {
                            const float vv = qk[k];
                            const int b = le_cmp ? bin_walk<1>(vv, L, R) : bin_walk<0>(vv, L, R);
                            if constexpr (W) atomicAdd(&myhist[b], (unsigned long long)qw[k]);
                            else atomicAdd(&myhist[b >> 1], (b & 1) ? 0x10000u : 1u);
                        }
                        lds_wave_sync();  // its loads before the next stores
                        qn = 0;
                    };
                    // 256 keys per call (64 per load); a full group (every
                    // group but the part's last) needs no bounds checks
                    auto group = [&](uint32_t base, auto full) __attribute__((always_inline)) {
                        constexpr bool kFull = decltype(full)::value;
                        float v[4];
                        uint32_t wv[W ? 4 : 1];
                        bool in[4];
#pragma unroll
                        for (int u = 0; u < 4; ++u) {  // four LDS reads in flight
                            const uint32_t p = base + (uint32_t)(64 * u + lane);
                            in[u] = kFull || p < pe;
                            v[u] = in[u] ? key[p] : 0.0f;
                            if constexpr (W) wv[u] = in[u] ? sw[p] : 0u;
                        }
                        // the four bins first, without branches, then the
                        // queueing of slow keys, then the atomics of the other
                        // keys in the window: no key waits for the previous
                        // key's atomic
                        int bin[4];
                        bool slow[4], fast[4];
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const float vv = v[u];
                            const bool below = vv < L, above = vv > R;  // past every candidate
                            // bin_estimate's test; the clamp only keeps the
                            // conversion of keys outside [L, R] in range
                            const float ef = (vv - L) * scale;
                            bin[u] = (int)fminf(fmaxf(ef, 0.0f), 256.0f);
                            const bool est = fabsf(__builtin_amdgcn_fractf(ef) - 0.5f) < lim;
                            const bool inwin = in[u] && !below && !above;
                            slow[u] = inwin && !est;
                            fast[u] = inwin && est;
                            if constexpr (W) {
                                wbelow += in[u] && below ? (uint64_t)wv[u] : 0ull;
                                wabove += in[u] && above ? (uint64_t)wv[u] : 0ull;
                            } else {
                                nbelow += (uint32_t)__popcll(__ballot(in[u] && below));
                                nabove += (uint32_t)__popcll(__ballot(in[u] && above));
                            }
                        }
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const uint64_t sm = __ballot(slow[u]);
                            if (sm) {  // wave-uniform
                                if (qn + 64u > (uint32_t)kQueue) drain();
                                if (slow[u]) {
                                    const uint32_t at = qn + (uint32_t)__popcll(sm & lanes_below);
                                    qk[at] = v[u];
                                    if constexpr (W) qw[at] = wv[u];
                                }
                                qn += (uint32_t)__popcll(sm);
                            }
                        }
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            if (!fast[u]) continue;
                            if constexpr (W) {
                                atomicAdd(&myhist[bin[u]], (unsigned long long)wv[u]);
                            } else {
                                // bin b: half b & 1 of word b >> 1
                                atomicAdd(&myhist[bin[u] >> 1], 1u << ((bin[u] & 1) << 4));
                            }
                        }
                    };
                    uint32_t base = pb;
                    for (; base + 256u <= pe; base += 256u) group(base, std::true_type{});
                    if (base < pe) group(base, std::false_type{});
                    if (qn) drain();
                    if constexpr (W) {
                        const uint64_t sb = wave_sum(wbelow), sa = wave_sum(wabove);
                        if (lane == 0) {
                            if (sb) atomicAdd(&myhist[0], (unsigned long long)sb);
                            if (sa) atomicAdd(&myhist[kBins - 1], (unsigned long long)sa);
                        }
                    } else if (lane == 0) {
                        // bin 0: the low half of word 0; bin 255: the high half of the last word
                        if (nbelow) atomicAdd(&myhist[0], nbelow);
                        if (nabove) atomicAdd(&myhist[kHistWords - 1], nabove << 16);
                    }
                }
                __syncthreads();  // every histogram of the round is complete
                if (act && part == 0) {
                    // the slot's histogram read and cleared, its prefix sums
                    // in registers, then up to 8 passes of the controller on them
                    RoundOut ro;
                    if constexpr (W) {
                        uint64_t h[4];
#pragma unroll
                        for (int i = 0; i < 4; ++i) h[i] = myhist[4 * lane + i];
#pragma unroll
                        for (int i = 0; i < 4; ++i) myhist[4 * lane + i] = 0ull;  // this lane's bins
                        const uint64_t s0 = h[0], s1 = s0 + h[1], s2 = s1 + h[2], s3 = s2 + h[3];
                        const uint64_t base = wave_inclusive_scan(s3) - s3;
                        // P[4 lane + 1 + q] (P[j] = weight in bins below j)
                        const uint64_t pv[4] = {base + s0, base + s1, base + s2, base + s3};
                        ro = replay_round_lanes(pv, L, R, target, passes, lane, trow);
                    } else {
                        // two 16-bit bins per word: counts <= kCap
                        const uint2 hw = reinterpret_cast<const uint2 *>(myhist)[lane];
                        reinterpret_cast<uint2 *>(myhist)[lane] = make_uint2(0u, 0u);  // this lane's bins
                        const uint32_t w01 = hw.x, w23 = hw.y;
                        const uint32_t s0 = w01 & 0xffffu, s1 = s0 + (w01 >> 16);
                        const uint32_t s2 = s1 + (w23 & 0xffffu), s3 = s2 + (w23 >> 16);
                        const uint32_t base = wave_inclusive_scan(s3) - s3;  // <= kCap
                        // P[4 lane + 1 + q] (P[j] = keys in bins below j)
                        const uint32_t pv[4] = {base + s0, base + s1, base + s2, base + s3};
                        ro = replay_round_lanes(pv, L, R, target, passes, lane, trow);
                    }
                    if (lane == 0) {
                        sL[slot] = ro.L;
                        sR[slot] = ro.R;
                        sPasses[slot] = ro.passes;
                        sFound[slot] = ro.found ? 1 : 0;
                    }
                }
                __syncthreads();  // the slots' new margins out, every histogram clear
                {
                    // slots still searching: one read per lane, not one per slot
                    const bool on = ((amask >> lane) & 1u) != 0u && lane < kSubWaves;
                    const bool more = on && !sFound[lane] && sPasses[lane] < ORB_MAX_PASSES;
                    amask = (uint32_t)__ballot(more);
                }
                if (act) {
                    L = sL[slot];
                    R = sR[slot];
                    passes = sPasses[slot];
                    found = sFound[slot] != 0;
                }
            }
            // ---- partition: stopper lists (each wave one contiguous part)
            const float cut = cell_cut(L, R);
            uint32_t tl = 0, tr = 0;
            // 256 keys per call; a full group (every group but the part's
            // last) needs no bounds checks
            auto count_group = [&](uint32_t base, auto full) __attribute__((always_inline)) {
                constexpr bool kFull = decltype(full)::value;
                float v[4];
                bool in[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const uint32_t p = base + (uint32_t)(64 * u + lane);
                    in[u] = kFull || p < pe;
                    v[u] = in[u] ? key[p] : 0.0f;
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    tl += (uint32_t)__popcll(__ballot(in[u] && v[u] >= cut));
                    tr += (uint32_t)__popcll(__ballot(in[u] && v[u] <= cut));
                }
            };
            if (valid) {
                uint32_t base = pb;
                for (; base + 256u <= pe; base += 256u) count_group(base, std::true_type{});
                if (base < pe) count_group(base, std::false_type{});
            }
            if (lane == 0) {
                sTL[w] = tl;
                sTR[w] = tr;
            }
            __syncthreads();
            // the slot's waves' stopper counts: totals and this wave's offsets,
            // by a scan across lanes (lane q holds wave w0 + q)
            uint32_t oL, oR, TL, TR;
            {
                const uint32_t a = lane < g ? sTL[w0 + lane] : 0u;
                const uint32_t b2 = lane < g ? sTR[w0 + lane] : 0u;
                const uint32_t ia = wave_inclusive_scan(a), ib = wave_inclusive_scan(b2);
                TL = (uint32_t)__shfl((int)ia, 63);
                TR = (uint32_t)__shfl((int)ib, 63);
                oL = (uint32_t)__shfl((int)(ia - a), part);
                oR = (uint32_t)__shfl((int)(ib - b2), part);
            }
            uint16_t *const Lp = slpos + lb;
            uint16_t *const Rp = srpos + lb;
            auto list_group = [&](uint32_t base, auto full) __attribute__((always_inline)) {
                constexpr bool kFull = decltype(full)::value;
                float v[4];
                bool in[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const uint32_t p = base + (uint32_t)(64 * u + lane);
                    in[u] = kFull || p < pe;
                    v[u] = in[u] ? key[p] : 0.0f;
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const uint32_t p = base + (uint32_t)(64 * u + lane);
                    const bool isL = in[u] && v[u] >= cut, isR = in[u] && v[u] <= cut;
                    const uint64_t mL = __ballot(isL), mR = __ballot(isR);
                    if (isL) Lp[oL + __popcll(mL & lanes_below)] = (uint16_t)(p - lb);
                    if (isR) Rp[oR + __popcll(mR & lanes_below)] = (uint16_t)(p - lb);
                    oL += (uint32_t)__popcll(mL);
                    oR += (uint32_t)__popcll(mR);
                }
            };
            if (valid) {
                uint32_t base = pb;
                for (; base + 256u <= pe; base += 256u) list_group(base, std::true_type{});
                if (base < pe) list_group(base, std::false_type{});
            }
            __syncthreads();
            const bool bad = valid && (m == 0 || TL == 0);
            if (valid && !bad && part == 0) {
                // K = #{t : L[t] < R[TR-1-t]} (true then false in t)
                uint32_t lo = 0, hi = TL < TR ? TL : TR;
                while (hi - lo > 64u) {
                    const uint32_t span = hi - lo;
                    const uint32_t tp = lo + (uint32_t)(((lane + 1) * span) / 65u);
                    const uint64_t mk = __ballot(Lp[tp] < Rp[TR - 1 - tp]);
                    if (mk == 0ull) {
                        hi = lo + span / 65u;
                    } else {
                        const int j = 63 - __clzll((long long)mk);
                        const uint32_t tj = lo + (uint32_t)(((j + 1) * span) / 65u);
                        const uint32_t tn = j < 63 ? lo + (uint32_t)(((j + 2) * span) / 65u) : hi;
                        lo = tj + 1;
                        hi = tn;
                    }
                }
                {
                    const uint32_t tp = lo + (uint32_t)lane;
                    lo += (uint32_t)__popcll(__ballot(tp < hi && Lp[tp] < Rp[TR - 1 - tp]));
                }
                const uint32_t K = lo;
                uint32_t i;
                if (K == 0) {
                    i = Lp[0];
                } else {
                    i = Rp[TR - K];
                    if (K < TL && Lp[K] < i) i = Lp[K];
                }
                if (lane == 0) {
                    sK[slot] = K;
                    sI[slot] = i;
                }
            }
            __syncthreads();
            if (valid && !bad) {
                const uint32_t K = sK[slot];
                for (uint32_t tt = (uint32_t)(part * 64 + lane); tt < K; tt += (uint32_t)(g * 64)) {
                    const uint32_t a = lb + Lp[tt], b2 = lb + Rp[TR - 1 - tt];
                    const float ax = sx[a], ay = sy[a], az = sz[a];
                    sx[a] = sx[b2];
                    sy[a] = sy[b2];
                    sz[a] = sz[b2];
                    sx[b2] = ax;
                    sy[b2] = ay;
                    sz[b2] = az;
                    if constexpr (W) {
                        const uint32_t wa = sw[a];
                        sw[a] = sw[b2];
                        sw[b2] = wa;
                    }
                    if (IDS) {
                        const uint16_t ia = sidx[a];
                        sidx[a] = sidx[b2];
                        sidx[b2] = ia;
                    }
                }
            }
            __syncthreads();
            if (valid && part == 0) {
                // the slot's first wave, all lanes with the same values: the
                // cell and its children are written a word per lane
                cl.cutMarginLeft = L;
                cl.cutMarginRight = R;
                cl.foundCut = found;
                const uint32_t cw = cell_word(cl, lane);
                if (lane < kCellWords) reinterpret_cast<uint32_t *>(heap + hb + cl.id)[lane] = cw;
                if (lane == 0) atomicMax(&s_lpmax[l], passes);  // LDS: the slots' waves finish together

                orb_cell lc, rc;
                uint32_t *wl = reinterpret_cast<uint32_t *>(&lc);
                uint32_t *wr = reinterpret_cast<uint32_t *>(&rc);
#pragma unroll
                for (int j = 0; j < kCellWords; ++j) wl[j] = wr[j] = 0u;
                const uint32_t i = sI[slot];
                // the reference splits a level's cells before it partitions any
                const bool split_ok = right_child_id(cl.id) < rr.capr && cell_split(cl, lc, rc);
                if (!split_ok || bad) {
                    if (lane == 0) {
                        s_err = 1;
                        report_error(st, l, split_ok ? kErrPartition : kErrSplit, cl.id);
                    }
                } else {
                    if (lb + i != le - 1 && lane < 5) {
                        // Hoare's last step, an array per lane
                        const uint32_t a = lb + i, b2 = le - 1;
                        if (lane < 3) {
                            float *arr = lane == 0 ? sx : (lane == 1 ? sy : sz);
                            const float va = arr[a];
                            arr[a] = arr[b2];
                            arr[b2] = va;
                        } else if (lane == 3) {
                            if constexpr (W) {
                                const uint32_t wa = sw[a];
                                sw[a] = sw[b2];
                                sw[b2] = wa;
                            }
                        } else if (IDS) {
                            const uint16_t ia = sidx[a];
                            sidx[a] = sidx[b2];
                            sidx[b2] = ia;
                        }
                    }
                    const int64_t gl = hb + lc.id, gr = hb + rc.id;
                    // lanes [0, 13): the left child's words, [32, 45): the right's
                    const int half = lane >> 5, wj = lane & 31;
                    const uint32_t kw = cell_word(half ? rc : lc, wj);
                    SubCell *nx = scells[cb ^ 1];
                    if (wj < kCellWords) {
                        reinterpret_cast<uint32_t *>(heap + (half ? gr : gl))[wj] = kw;
                        reinterpret_cast<uint32_t *>(&nx[2 * k + half].cell)[wj] = kw;
                    }
                    if (lane == 0) {
                        exists[gl] = 1;
                        exists[gr] = 1;
                        sub[gl] = 1;
                        sub[gr] = 1;
                        ranges[2 * gl] = begin + lb;
                        ranges[2 * gl + 1] = begin + lb + i;
                        ranges[2 * gr] = begin + lb + i;
                        ranges[2 * gr + 1] = begin + le;
                        nx[2 * k].lb = lb;
                        nx[2 * k].le = lb + i;
                        nx[2 * k].valid = lc.nLeafCells >= 2;
                        nx[2 * k + 1].lb = lb + i;
                        nx[2 * k + 1].le = le;
                        nx[2 * k + 1].valid = rc.nLeafCells >= 2;
                    }
                }
            }
            __syncthreads();  // the next batch reuses the position lists and the slots
        }
        const int32_t nn = 2 * ncur;  // <= kSmallLeaves = 64 (checked above)
        if (w == 0) {
            const uint64_t vm = __ballot(lane < nn && scells[cb ^ 1][lane].valid);
            if (lane == 0) {
                s_ncur = nn;
                s_nvalid = (int32_t)__popcll(vm);
            }
        }
        cb ^= 1;
        __syncthreads();
    }
    for (uint32_t k = (uint32_t)t; k < n; k += kSubBlock) {
        x[begin + k] = sx[k];
        y[begin + k] = sy[k];
        z[begin + k] = sz[k];
        if constexpr (W) wgt[begin + k] = sw[k];
    }
    if (IDS) {
        // the stopper lists are free: stage the cell's ids, then permute them
        for (uint32_t k = (uint32_t)t; k < n; k += kSubBlock) spos_raw[k] = pid[begin + k];
        __syncthreads();
        for (uint32_t k = (uint32_t)t; k < n; k += kSubBlock) pid[begin + k] = spos_raw[sidx[k]];
    }
    __syncthreads();  // the next cell reuses the LDS arrays
    }
    }
    if (t < 64 && s_lp0 >= 0 && s_lpmax[t] > 0) atomicMax(&level_passes[s_lp0 + t], s_lpmax[t]);
}

// ---------------------------------------------------------------------------
// one level of a mid-sized cell by one block
// ---------------------------------------------------------------------------
// A cell too large for the subtree kernel but of at most kRows * kThreads keys
// takes its whole level in one block: the cut-axis keys are read
// once into registers (kRows per lane: wave w holds the contiguous part
// [w * 64 * rows, (w + 1) * 64 * rows), 64 consecutive keys a row), every
// histogram round, the stopper masks and the pair lists come from there, and
// x, y, z (and the payload) are swapped in place.  The chunk path reads the
// keys twice and takes 16 dependent launches a level; what bounds this kernel
// is the swap's memory traffic on levels that fill the chip (12 B read and
// written per key, 4 B more for the keys) and its own serial phases on levels
// of few cells.  Measured: a level of 4096 cells of 16384 keys 451 us (chunk
// path 530), one of 8192 of 8192 keys 433 us, one of two 32768-key cells 45 us, of four 16384-key cells 34 us
// (chunk path 85).
//
// rows is a multiple of 4, so a wave's part is whole 256-key groups; keys
// past the cell's end are +INF in their lane (never below a cut, never an
// R-stopper) and are masked out of the L-stopper words.
//
// Latency decides on levels of few cells: 1024 threads a cell.  Levels that
// fill the chip take 512-thread blocks of twice the rows, two to a CU (256
// threads, four to a CU, where the cells allow), so that one block's barriers
// and replays lie under the others' traffic.
constexpr int kCellRowsMax = 40;
constexpr uint32_t kCellTiny = 10u * 1024u, kCellSmall = 20u * 1024u, kCellLarge = 40u * 1024u;  // capacities
constexpr int32_t kCellManyCells = 256;  // more than a cell per CU
static_assert(kCellRowsMax <= 64 && kCellLarge <= 65536u, "a mask word per lane, 16-bit positions");

template <int kThreads, int kRows, int kArrays>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_b_cell(CellRec *recs, int32_t nCells, orb_cell *heap,
                                                       uint8_t *exists, uint32_t *ranges, float *x,
                                                       float *y, float *z, uint32_t *pid,
                                                       uint32_t *wgt, int le_cmp, uint64_t *trace,
                                                       int32_t *level_passes, int32_t *status)
{
    static_assert(kRows % 4 == 0 && kRows <= kCellRowsMax, "whole groups, a mask word per lane");
    constexpr int kWaves = kThreads / 64;
    constexpr uint32_t kCap = (uint32_t)kRows * kThreads;
    constexpr int kBatch = 4;  // pairs per thread in flight
    // a swapped pair's two positions differ and no position is in two pairs:
    // at most n / 2 pairs
    __shared__ uint16_t slist[2][kCap / 2];
    __shared__ uint32_t hist[kBins];
    __shared__ uint32_t s_cnt[2][kWaves];
    __shared__ float s_lr[2];
    __shared__ int32_t s_pf[2];
    __shared__ uint32_t s_K, s_i;
    const int t = threadIdx.x, lane = t & 63, w = (int)uniform((uint32_t)t >> 6);
    for (int32_t c = blockIdx.x; c < nCells; c += gridDim.x) {
        if (uniform((uint32_t)recs[c].flags) != (uint32_t)kFlagBlock) continue;
        const CellRec &rec = recs[c];  // this block alone writes it, at the search's end
        const uint32_t begin = uniform(rec.begin), n = uniform(rec.end) - begin;
        const int axis = (int)uniform((uint32_t)rec.axis);
        const int32_t id = (int32_t)uniform((uint32_t)rec.id), hb = (int32_t)uniform((uint32_t)rec.hb);
        if (n > kCap || axis < 0 || axis > 2) {
            // the level records hand over neither; refuse anything else
            if (t == 0) report_error(status + rec.st, rec.lp & 63, kErrSplit, id);
            continue;
        }
        const uint32_t rows = 4u * ((n + 4u * kThreads - 1u) / (4u * kThreads));
        const uint32_t wb = 64u * rows * (uint32_t)w;
        const uint32_t len = wb < n ? (n - wb < 64u * rows ? n - wb : 64u * rows) : 0u;
        const float *const key = axis_ptr(x, y, z, axis) + begin;
        float v[kRows];
        // f(row) over the rows in use, unrolled (v stays in registers), a
        // uniform branch per four rows
        auto each_row = [&](auto f) __attribute__((always_inline)) {
            // a value of its own: otherwise the compiler keeps every group's
            // comparison in scalar registers from one sweep to the next
            uint32_t used = rows;
            asm volatile("" : "+s"(used));
            static_for<0, kRows / 4>([&](auto gc) __attribute__((always_inline)) {
                constexpr int g = decltype(gc)::value;
                if (4u * (uint32_t)g < used)
                    static_for<4 * g, 4 * g + 4>(
                        [&](auto jc) __attribute__((always_inline)) { f(jc); });
                __builtin_amdgcn_sched_barrier(0);
            });
        };
        {
            const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<float *>(key), 0, (int)(n * 4u), 0x00020000);
            each_row([&](auto jc) __attribute__((always_inline)) {
                constexpr int j = decltype(jc)::value;
                v[j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                    kr, (int)((wb + 64u * (uint32_t)j + (uint32_t)lane) * 4u), 0, 0));
            });
        }
        for (int q = t; q < kBins; q += kThreads) hist[q] = 0u;
        if (len < 64u * rows) {  // wave-uniform: the cell's end lies in (or before) this part
            each_row([&](auto jc) __attribute__((always_inline)) {
                constexpr int j = decltype(jc)::value;
                if (64u * (uint32_t)j + (uint32_t)lane >= len) v[j] = INFINITY;
            });
        }
        __syncthreads();
        // ---- the bisection controller in rounds of 8 passes (orbit.cpp:149-231)
        const float target = difference_target(n, (int32_t)uniform((uint32_t)rec.nLeaf));
        uint64_t *trow = trace ? trace + ((size_t)hb + id) * ORB_MAX_PASSES : nullptr;
        float lo = uniform(rec.margin_l), hi = uniform(rec.margin_r);
        int32_t passes = 0;
        bool found = false;
        while (true) {
            const float width = hi - lo;
            const float scale = width > 0.0f ? (float)kBins / width : 0.0f;
            const float lim = 0.5f - bin_tolerance(lo, hi, scale);
            uint32_t below = 0;  // wave-uniform; keys above the margins are in no prefix sum
            uint64_t slow = 0ull;  // this lane's rows too close to a bin edge for the estimate
            each_row([&](auto jc) __attribute__((always_inline)) {
                constexpr int j = decltype(jc)::value;
                const bool lt = v[j] < lo, in = !lt && !(v[j] > hi);
                below += (uint32_t)__popcll(__ballot(lt));
                const float ef = (v[j] - lo) * scale;
                const int bin = (int)__builtin_amdgcn_fmed3f(ef, 0.0f, 255.5f);
                const bool est = fabsf(__builtin_amdgcn_fractf(ef) - 0.5f) < lim;
                if (in && est) atomicAdd(&hist[bin], 1u);
                slow |= in && !est ? 1ull << j : 0ull;
            });
            while (__ballot(slow != 0ull)) {
                // exact bins of the slow keys (about 1 in 2000 of a first
                // round; every one where coordinates sit on a grid), read
                // again: four rows a step, their loads in flight together
                float sv[4];
                bool on[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    on[u] = slow != 0ull;
                    const uint32_t row = on[u] ? (uint32_t)__builtin_ctzll(slow) : 0u;
                    slow &= slow - 1ull;  // 0 stays 0
                    sv[u] = on[u] ? key[wb + 64u * row + (uint32_t)lane] : 0.0f;
                }
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (on[u])
                        atomicAdd(&hist[le_cmp ? bin_walk<1>(sv[u], lo, hi) : bin_walk<0>(sv[u], lo, hi)],
                                  1u);
            }
            if (lane == 0 && below) atomicAdd(&hist[0], below);
            __syncthreads();
            if (w == 0) {
                const uint4 h4 = reinterpret_cast<const uint4 *>(hist)[lane];
                reinterpret_cast<uint4 *>(hist)[lane] = make_uint4(0u, 0u, 0u, 0u);
                const uint32_t s0 = h4.x, s1 = s0 + h4.y, s2 = s1 + h4.z, s3 = s2 + h4.w;
                const uint32_t base = wave_inclusive_scan(s3) - s3;
                // P[4 lane + 1 + q] (P[j] = keys in bins below j)
                const uint32_t pv[4] = {base + s0, base + s1, base + s2, base + s3};
                const RoundOut ro = replay_round_lanes(pv, lo, hi, target, passes, lane, trow);
                if (lane == 0) {
                    s_lr[0] = ro.L;
                    s_lr[1] = ro.R;
                    s_pf[0] = ro.passes;
                    s_pf[1] = ro.found ? 1 : 0;
                }
            }
            __syncthreads();
            lo = uniform(s_lr[0]);
            hi = uniform(s_lr[1]);
            passes = (int32_t)uniform((uint32_t)s_pf[0]);
            found = uniform((uint32_t)s_pf[1]) != 0u;
            if (found || passes >= ORB_MAX_PASSES) break;
        }
        // ---- Hoare (partition.cpp:28-60): stopper words, a word per lane
        const float cut = cell_cut(lo, hi);
        uint64_t mineL = 0ull, mineR = 0ull;
        each_row([&](auto jc) __attribute__((always_inline)) {
            constexpr int j = decltype(jc)::value;
            constexpr uint32_t p0 = 64u * (uint32_t)j;
            const uint64_t valid =
                p0 >= len ? 0ull : (len - p0 >= 64u ? ~0ull : (1ull << (len - p0)) - 1ull);
            const uint64_t mL = __ballot(!(v[j] < cut)) & valid;
            const uint64_t mR = __ballot(!(v[j] > cut)) & valid;
            mineL = lane == j ? mL : mineL;
            mineR = lane == j ? mR : mineR;
        });
        const uint32_t cL = (uint32_t)__popcll(mineL), cR = (uint32_t)__popcll(mineR);
        const uint32_t iL = wave_inclusive_scan(cL), iR = wave_inclusive_scan(cR);
        if (lane == 63) {
            s_cnt[0][w] = iL;
            s_cnt[1][w] = iR;
        }
        __syncthreads();
        // the waves' stopper counts, wave q in lane q, and their prefix sums
        const uint32_t wL = lane < kWaves ? s_cnt[0][lane] : 0u;
        const uint32_t wR = lane < kWaves ? s_cnt[1][lane] : 0u;
        const uint32_t pL = wave_inclusive_scan(wL) - wL, pR = wave_inclusive_scan(wR) - wR;
        const uint32_t TL = lane_value(pL + wL, 63), TR = lane_value(pR + wR, 63);
        const bool bad = n == 0u || TL == 0u;  // the reference's loop leaves the cell
        // With A(p) the L-stoppers before position p and B(p) the R-stoppers
        // at or after it (A grows, B shrinks), K = max over p of
        // min(A(p), B(p)) and i = the last p with A(p) <= K <= B(p).  Both lie
        // in one word: the last whose start has A <= B, resp. A <= K <= B.
        const uint32_t aL = lane_value(pL, w), aR = lane_value(pR, w);
        const uint32_t xA = aL + iL - cL, xB = TR - (aR + iR - cR);  // A and B at this lane's word
        if (t == (kWaves > 1 ? 64 : 0))  // the cell's margins, its passes, its children
            finish_round(rec, c, RoundOut{lo, hi, passes, found, 0}, found ? 1 : 0, recs, heap,
                         level_passes, exists, status);
        // A and B at bit `lane` of word q of this wave, and just after it
        auto at_bit = [&](int q, uint32_t &a0, uint32_t &b0, uint32_t &a1, uint32_t &b1) {
            const uint64_t mL = lane_value(mineL, q), mR = lane_value(mineR, q);
            a0 = lane_value(xA, q) + __builtin_amdgcn_mbcnt_hi(
                     (uint32_t)(mL >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mL, 0u));
            b0 = lane_value(xB, q) - __builtin_amdgcn_mbcnt_hi(
                     (uint32_t)(mR >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mR, 0u));
            a1 = a0 + (uint32_t)((mL >> lane) & 1ull);
            b1 = b0 - (uint32_t)((mR >> lane) & 1ull);
        };
        if (!bad) {
            const uint64_t mk = __ballot(lane < kWaves && pL + pR <= TR);
            if (w == 63 - __clzll((long long)mk)) {  // A <= B at the start of this wave's part
                const uint64_t mw = __ballot((uint32_t)lane < rows && xA <= xB);
                uint32_t a0, b0, a1, b1;
                at_bit(63 - __clzll((long long)mw), a0, b0, a1, b1);
                // the maximum over the word's positions, and the word's end
                const uint32_t k0 = a0 < b0 ? a0 : b0, k1 = a1 < b1 ? a1 : b1;
                const uint32_t best = wave_max(k0 > k1 ? k0 : k1);
                if (lane == 0) s_K = best;
            }
        }
        __syncthreads();
        const int64_t lid = left_child_id(id), rid = right_child_id(id);
        if (bad || rid >= (int32_t)uniform((uint32_t)rec.capr)) {
            if (t == 0) report_error(status + rec.st, rec.lp & 63, kErrPartition, id);
            continue;  // uniform
        }
        const uint32_t K = uniform(s_K);
        {
            const uint64_t mk = __ballot(lane < kWaves && pL <= K && K + pR <= TR);
            if (w == 63 - __clzll((long long)mk)) {
                const uint64_t mw = __ballot((uint32_t)lane < rows && xA <= K && K <= xB);
                const int q = 63 - __clzll((long long)mw);
                uint32_t a0, b0, a1, b1;
                at_bit(q, a0, b0, a1, b1);
                const uint64_t mb = __ballot(a0 <= K && K <= b0);
                if (lane == 0) s_i = wb + 64u * (uint32_t)q + 63u - (uint32_t)__clzll((long long)mb);
            }
        }
        {
            // the pairs' positions: L_t at t, R_t at t
            const uint32_t xL = iL - cL, xR = iR - cR;
            each_row([&](auto jc) __attribute__((always_inline)) {
                constexpr int j = decltype(jc)::value;
                const uint32_t pos = wb + 64u * (uint32_t)j + (uint32_t)lane;
                const uint64_t mL = lane_value(mineL, j), mR = lane_value(mineR, j);
                const uint32_t oL = aL + lane_value(xL, j), oR = aR + lane_value(xR, j);
                if (oL < K && mL) {  // uniform
                    const uint32_t idx = oL + __builtin_amdgcn_mbcnt_hi(
                        (uint32_t)(mL >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mL, 0u));
                    if (((mL >> lane) & 1ull) && idx < K) slist[0][idx] = (uint16_t)pos;
                }
                if (oR + (uint32_t)__popcll(mR) + K > TR && mR) {  // uniform
                    const uint32_t idx = oR + __builtin_amdgcn_mbcnt_hi(
                        (uint32_t)(mR >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mR, 0u));
                    if (((mR >> lane) & 1ull) && idx + K >= TR) slist[1][TR - 1u - idx] = (uint16_t)pos;
                }
            });
        }
        __syncthreads();
        const uint32_t i = uniform(s_i);
        const CellArrays<true> ca(x, y, z, pid, wgt, begin);
        const int na = ca.count;  // uniform, at most kArrays
        for (uint32_t j0 = (uint32_t)t; j0 < K + (uint32_t)t; j0 += kThreads * kBatch) {
            uint32_t pa[kBatch], pb[kBatch];
            uint32_t va[kArrays][kBatch] = {}, vb[kArrays][kBatch] = {};
#pragma unroll
            for (int u = 0; u < kBatch; ++u) {
                const uint32_t jj = j0 + (uint32_t)(u * kThreads);
                pa[u] = jj < K ? 4u * slist[0][jj] : 0u;
                pb[u] = jj < K ? 4u * slist[1][jj] : 0u;
            }
#pragma unroll
            for (int arr = 0; arr < kArrays; ++arr) {
                if (arr >= na) break;
#pragma unroll
                for (int u = 0; u < kBatch; ++u) {
                    if (j0 + (uint32_t)(u * kThreads) < K) {
                        va[arr][u] = ca.load(arr, pa[u]);
                        vb[arr][u] = ca.load(arr, pb[u]);
                    }
                }
            }
#pragma unroll
            for (int arr = 0; arr < kArrays; ++arr) {
                if (arr >= na) break;
#pragma unroll
                for (int u = 0; u < kBatch; ++u) {
                    if (j0 + (uint32_t)(u * kThreads) < K) {
                        ca.store(arr, pa[u], vb[arr][u]);
                        ca.store(arr, pb[u], va[arr][u]);
                    }
                }
            }
        }
        __syncthreads();  // every pair is in place before the last row swap
        if (t < na && i != n - 1u) {
            // Hoare's last step (partition.cpp:61-62), an array per lane
            const uint32_t a = ca.load(t, 4u * i), b = ca.load(t, 4u * (n - 1u));
            ca.store(t, 4u * i, b);
            ca.store(t, 4u * (n - 1u), a);
        }
        if (t == 0) {
            const int64_t gl = hb + lid, gr = hb + rid;
            ranges[2 * gl] = begin;
            ranges[2 * gl + 1] = begin + i;
            ranges[2 * gr] = begin + i;
            ranges[2 * gr + 1] = begin + n;
        }
        // (the next cell's first barrier stands before it rewrites any LDS
        // that a wave still reads here)
    }
}

// ---------------------------------------------------------------------------
// levels of few chunks whose cells are too large for k_b_cell
// ---------------------------------------------------------------------------
// A level of at most kMidLevelChunks chunks, its cells at most kMidChunks
// chunks each, is bound by its launches, not by memory: the chunk path takes
// 16 of them, 4-7 us each however little they do.  Here it takes six:
//   k_b_recs_scan<true>  cell records, chunk table, the cells' key counters
//   k_m_hist             round 1 per chunk, added to the cell's row (atomics:
//                        few blocks share a row)
//   k_m_window           every block replays round 1 from its cell's row (a
//                        1 KB read in place of two launches), then takes the
//                        window pass and adds round 2's counts to the cell's second row
//   k_m_narrow           round 2 likewise; masks, packed keys and the cell's list
//                        narrowed to its margins
//   k_m_tail             a block per cell: the later rounds over the listed keys,
//                        the stopper masks, K, i and the swap plan
//   k_hoare_swap
// The same rounds, masks and plan as the chunk path's.  The five top levels of
// 2^20 keys (1 to 16 cells): 52 us of kernels a level, from 89.  The line at 512
// chunks a cell: the tables of one tail block (of 256: 3000001 keys to 500 leaves
// 588 -> 607 us, 2^24 stable ones to 256 1350 -> 1370; of 1024, before k_m_narrow,
// 638 -> 655).  The level's size matters little: against a line at 2048 chunks,
// whole builds of 12M keys take 1347 -> 1165 us, 2^24 stable ones 1458 -> 1350,
// 5e7 even ones, with predicted windows, 4317 -> 4310 and 5e7 tied ones 3121 ->
// 3167.  Past 16384 the one block that fills the chunk table takes longer than the
// launches saved: with the line at 65536, 2^27 even keys 10033 -> 10236 us.
constexpr int kMidChunks = 512;         // per cell: k_m_tail's tables
constexpr int64_t kMidLevelChunks = 16384;

// A cell's search between the launches of such a level: state[0 .. nCells) after
// one round, state[nCells ..) after the next (weighted levels take them in turn).
struct RoundState {
    float L, R;
    int32_t passes, found;
};
__device__ inline RoundState load_state(const RoundState *p)
{
    const RoundState s = *p;
    return RoundState{uniform(s.L), uniform(s.R), (int32_t)uniform((uint32_t)s.passes),
                      (int32_t)uniform((uint32_t)s.found)};
}

// The next round of a cell from its row of counts, by a whole wave.
__device__ inline RoundState replay_row(const uint32_t *row, const CellRec &r, const RoundState &s, int lane,
                                        uint64_t *trace_row)
{
    const uint4 h4 = reinterpret_cast<const uint4 *>(row)[lane];
    const uint32_t s0 = h4.x, s1 = s0 + h4.y, s2 = s1 + h4.z, s3 = s2 + h4.w;
    const uint32_t base = wave_inclusive_scan(s3) - s3;
    // P[4 lane + 1 + q] (P[j] = keys in bins below j)
    const uint32_t pv[4] = {base + s0, base + s1, base + s2, base + s3};
    const float target = difference_target(uniform(r.end) - uniform(r.begin),
                                           (int32_t)uniform((uint32_t)r.nLeaf));
    const RoundOut ro = replay_round_lanes(pv, s.L, s.R, target, s.passes, lane, trace_row);
    return RoundState{uniform(ro.L), uniform(ro.R), ro.passes, ro.found ? 1 : 0};
}

// Where a cell's passes are traced, for the one wave that traces them.
__device__ inline uint64_t *trace_of(uint64_t *trace, const CellRec &r, bool mine)
{
    return trace && mine ? trace + ((size_t)r.hb + r.id) * ORB_MAX_PASSES : nullptr;
}

// Round 1: as k_b_hist, without a candidate table (the exact bin of a key
// near a bin edge comes from the walk) and with the chunk's row added to the
// cell's.
template <int LE>
__global__ __launch_bounds__(kBlock) void k_m_hist(const CellRec *__restrict__ recs, int32_t nCells,
                                                   const uint32_t *__restrict__ first,
                                                   const uint4 *__restrict__ chunk_desc,
                                                   uint32_t max_chunks, const float *__restrict__ x,
                                                   const float *__restrict__ y,
                                                   const float *__restrict__ z,
                                                   uint32_t *__restrict__ cell_hist)
{
    constexpr int kW = kBlock / 64;
    constexpr int kPerWave = kMaskWords / kW;  // 16 loads of 64 keys
    __shared__ uint32_t hist[kW][kBins];
    const int t = threadIdx.x, lane = t & 63, w = (int)uniform((uint32_t)t >> 6);
    const uint32_t sb = (uint32_t)(w * kPerWave * 64);
    const uint32_t total = first[nCells];
    for (uint32_t q = blockIdx.x;; q += gridDim.x) {
        const uint4 d = chunk_record(chunk_desc, q, max_chunks);
        const uint32_t b = uniform(d.x), e = uniform(d.y), cell = uniform(d.z);
        const uint32_t axis = uniform(d.w);
        keep_values(b, e, cell, axis);
        if (q >= total) break;
        if (axis > 2u) continue;  // uniform: the cell is not searched
        float v[kPerWave];
        issue_chunk_loads(x, y, z, true, d, sb, lane, v);
        const float lo = uniform(recs[cell].margin_l), hi = uniform(recs[cell].margin_r);
#pragma unroll
        for (int u = 0; u < kW; ++u) hist[u][t] = 0u;
        __syncthreads();
        const float width = hi - lo;
        const float scale = width > 0.0f ? (float)kBins / width : 0.0f;
        const float lim = 0.5f - bin_tolerance(lo, hi, scale);
        const float limx = lim > 0.25f ? lim : -1.0f;  // as k_b_hist
        const uint32_t len = e - b;
        static_for<0, kPerWave>([&](auto jc) __attribute__((always_inline)) {
            constexpr int j = decltype(jc)::value;
            const bool ok = sb + 64u * (uint32_t)j + (uint32_t)lane < len;
            const float ef = __builtin_amdgcn_fmed3f((v[j] - lo) * scale, -0.5f, 255.5f);
            int bin = (int)ef;
            const bool slow = ok && !(fabsf(__builtin_amdgcn_fractf(ef) - 0.5f) < limx);
            if (__ballot(slow)) {  // wave-uniform; rare
                if (slow) bin = bin_walk<LE>(v[j], lo, hi);
            }
            if (ok) atomicAdd(&hist[w][bin], 1u);
        });
        __syncthreads();
        const uint32_t sum = hist[0][t] + hist[1][t] + hist[2][t] + hist[3][t];
        if (sum) atomicAdd(&cell_hist[(size_t)cell * kBins + t], sum);
        __syncthreads();  // the next chunk rewrites hist
    }
}

// Window pass: as k_b_hist_window, from round 1's outcome: the keys inside the
// margins go to the chunk quarter's slots of `pack` (in position order) and are
// counted for round 2, with the keys below, in the cell's second row.  A cell
// whose cut round 1 found has that cut as its window.
template <int LE>
__global__ __launch_bounds__(kBlock) void k_m_window(
    const CellRec *__restrict__ recs, int32_t nCells, const uint32_t *__restrict__ first,
    const uint4 *__restrict__ chunk_desc, uint32_t max_chunks, const float *__restrict__ x,
    const float *__restrict__ y, const float *__restrict__ z, uint32_t *cell_hist,
    RoundState *__restrict__ state, uint64_t *trace, float *__restrict__ pack,
    uint64_t *__restrict__ masks)
{
    constexpr int kW = kBlock / 64;
    constexpr int kPerWave = kMaskWords / kW;
    __shared__ float wkeys[kW][kChunk / kW];  // each wave's window keys, packed
    __shared__ uint32_t hist[kBins];
    __shared__ uint64_t words[kW][2][kPerWave];
    const int t = threadIdx.x, lane = t & 63, w = (int)uniform((uint32_t)t >> 6);
    const uint64_t lanes_below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    const uint32_t sb = (uint32_t)(w * kPerWave * 64);
    const uint32_t total = first[nCells];
    for (uint32_t q = blockIdx.x;; q += gridDim.x) {
        const uint4 d = chunk_record(chunk_desc, q, max_chunks);
        const uint32_t b = uniform(d.x), e = uniform(d.y), cell = uniform(d.z);
        const uint32_t axis = uniform(d.w);
        keep_values(b, e, cell, axis);
        if (q >= total) break;
        if (axis > 2u) continue;  // uniform: the cell is not searched
        float v[kPerWave];
        issue_chunk_loads(x, y, z, true, d, sb, lane, v);
        const CellRec &r = recs[cell];
        hist[t] = 0u;
        const bool lead = q == uniform(first[cell]);  // the cell's first chunk keeps its state
        const RoundState ro = replay_row(cell_hist + (size_t)cell * kBins, r,
                                         RoundState{uniform(r.margin_l), uniform(r.margin_r), 0, 0}, lane,
                                         trace_of(trace, r, lead && w == 0));
        if (lead && t == 0) state[cell] = ro;
        const float cut = cell_cut(ro.L, ro.R);
        const float lo = ro.found ? cut : ro.L, hi = ro.found ? cut : ro.R;
        __syncthreads();  // the row is clear
        const uint32_t len = e - b;
        uint32_t below = 0, packed = 0;  // wave-uniform
        float *dst = pack + b + sb;
        float *wk = wkeys[w];
        static_for<0, kPerWave>([&](auto jc) __attribute__((always_inline)) {
            constexpr int j = decltype(jc)::value;
            const uint32_t p0 = sb + 64u * (uint32_t)j;  // chunk position of lane 0
            const uint64_t valid =
                p0 >= len ? 0ull : (len - p0 >= 64u ? ~0ull : (1ull << (len - p0)) - 1ull);
            const uint64_t mB = __ballot(v[j] < lo) & valid;
            const uint64_t mG = __ballot(v[j] > hi) & valid;
            const uint64_t mW = valid & ~mB & ~mG;
            below += (uint32_t)__popcll(mB);
            if (lane == 0) {  // staged by one lane, as in k_b_hist_window
                words[w][0][j] = mG;
                words[w][1][j] = mW;
            }
            if (mW) {  // wave-uniform: most loads have no key in the window
                if ((mW >> lane) & 1ull) {
                    const uint32_t slot = packed + (uint32_t)__popcll(mW & lanes_below);
                    dst[slot] = v[j];
                    wk[slot] = v[j];
                }
                packed += (uint32_t)__popcll(mW);
            }
        });
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        __builtin_amdgcn_wave_barrier();
        if (!ro.found) {  // uniform: round 2's row
            const float width = hi - lo;
            const float scale = width > 0.0f ? (float)kBins / width : 0.0f;
            const float lim = 0.5f - bin_tolerance(lo, hi, scale);
            for (uint32_t k = (uint32_t)lane; k < packed; k += 64u) {
                int bin;
                if (!bin_estimate(wk[k], lo, scale, lim, bin)) bin = bin_walk<LE>(wk[k], lo, hi);
                atomicAdd(&hist[bin], 1u);
            }
            if (lane == 0 && below) atomicAdd(&hist[0], below);
        }
        uint64_t *mq = masks + (size_t)q * (2 * kMaskWords) + w * kPerWave;
        if (lane < kPerWave) {
            mq[lane] = words[w][0][lane];
            mq[kMaskWords + lane] = words[w][1][lane];
        }
        __syncthreads();
        if (hist[t]) atomicAdd(&cell_hist[((size_t)nCells + cell) * kBins + (size_t)t], hist[t]);
        __syncthreads();  // the next chunk rewrites the tables
    }
}

// Narrows each chunk from round 1's margins to round 2's (1/65536 of the cell's):
// the packed keys outside them settle their mask bits, those inside are packed
// again and go to the cell's list in `sel` (in any order, for the later rounds),
// whose counter (keys | keys below << 32) takes their number.  One tail block a
// cell then has few keys left, also where the keys lie in a clump that
// one bin of round 1 holds: without this pass 2^23 keys to 64 leaves, x in a clump
// of 0.01, took 2577 us, now 960; even keys pay a launch and save a round of the tail.
// A wave a chunk (a block a chunk replayed the rows in four waves and met at
// barriers: 21 us at 4096 chunks).
__global__ __launch_bounds__(kBlock) void k_m_narrow(
    const CellRec *__restrict__ recs, int32_t nCells, const uint32_t *__restrict__ first,
    const uint4 *__restrict__ chunk_desc, uint32_t max_chunks, const uint32_t *__restrict__ cell_hist,
    RoundState *state, uint64_t *trace, float *pack, uint64_t *masks, float *__restrict__ sel,
    unsigned long long *__restrict__ sel_lists)
{
    constexpr int kW = kBlock / 64;
    constexpr int kQuarter = kMaskWords / kW;  // words per packing quarter
    constexpr int kBatch = 4;                  // words in flight
    const int lane = threadIdx.x & 63, w = (int)uniform((uint32_t)threadIdx.x >> 6);
    const uint32_t total = first[nCells];
    for (uint32_t q = blockIdx.x * (uint32_t)kW + (uint32_t)w;; q += gridDim.x * (uint32_t)kW) {
        const uint4 d = chunk_record(chunk_desc, q, max_chunks);
        const uint32_t b = uniform(d.x), e = uniform(d.y), cell = uniform(d.z);
        const uint32_t axis = uniform(d.w);
        keep_values(b, e, cell, axis);
        if (q >= total) break;
        if (axis > 2u) continue;  // uniform: the cell is not searched
        uint64_t *mq = masks + (size_t)q * (2 * kMaskWords);
        uint64_t G = mq[lane];
        const uint64_t W = mq[kMaskWords + lane];
        const CellRec &r = recs[cell];
        const uint32_t begin = uniform(r.begin), f = uniform(first[cell]);
        const uint32_t cw = (uint32_t)__popcll(W), in = wave_inclusive_scan(cw);
        // before this word in its quarter
        const int quarter = lane & ~(kQuarter - 1);
        const uint32_t ex = in - cw - (uint32_t)__shfl((int)(in - cw), quarter, 64);
        float *const keys = pack + b + 64u * (uint32_t)quarter;
        // a word of few keys by its own lane, their loads in flight with the row;
        // of more by the wave, a key a lane
        const bool few = cw <= (uint32_t)kBatch;
        float own[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) own[u] = few && (uint32_t)u < cw ? keys[ex + (uint32_t)u] : 0.0f;
        const bool lead = q == f;
        RoundState ro = load_state(state + cell);
        if (!ro.found)  // uniform
            ro = replay_row(cell_hist + ((size_t)nCells + cell) * kBins, r, ro, lane, trace_of(trace, r, lead));
        if (lead && lane == 0) state[(size_t)nCells + cell] = ro;
        const float cut = cell_cut(ro.L, ro.R);
        const float lo = ro.found ? cut : ro.L, hi = ro.found ? cut : ro.R;
        uint64_t kept = 0ull;
        {
            uint64_t wd = few ? W : 0ull;
#pragma unroll
            for (int u = 0; u < kBatch; ++u) {
                const uint64_t bit = wd & (0ull - wd);  // 0: no key left
                wd ^= bit;
                const bool lt = own[u] < lo, gt = own[u] > hi;
                G |= gt ? bit : 0ull;
                kept |= lt || gt ? 0ull : bit;
            }
        }
        // word `at` (-1: none) and its keys, a lane each; sub: the keys wanted of them
        auto load_word = [&](int at, uint64_t sub) {
            const uint64_t m = at >= 0 ? lane_value(W, at) : 0ull;
            const uint32_t k = (at >= 0 ? lane_value(ex, at) : 0u) +
                               (uint32_t)__builtin_amdgcn_mbcnt_hi(
                                   (uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
            return (m & sub) >> lane & 1ull ? pack[b + 64u * (uint32_t)(at & ~(kQuarter - 1)) + k] : 0.0f;
        };
        for (uint64_t todo = __ballot(!few); todo;) {  // uniform
            float v[kBatch];
            int at[kBatch];
#pragma unroll
            for (int u = 0; u < kBatch; ++u) {
                at[u] = todo ? __builtin_ctzll(todo) : -1;
                todo &= todo - 1ull;  // 0 stays 0
                v[u] = load_word(at[u], ~0ull);
            }
#pragma unroll
            for (int u = 0; u < kBatch; ++u) {
                const uint64_t mB = __ballot(v[u] < lo), mG = __ballot(v[u] > hi);
                if (lane == at[u]) {
                    G |= W & mG;
                    kept = W & ~mB & ~mG;
                }
            }
        }
        const uint32_t below = e - b - wave_sum((uint32_t)__popcll(G)) - wave_sum((uint32_t)__popcll(kept));
        const uint64_t words = __ballot(kept != 0ull);
        if (words) {  // uniform; rare with even keys
            const uint32_t ck = (uint32_t)__popcll(kept), ink = wave_inclusive_scan(ck);
            const uint32_t exk = ink - ck, exq = exk - (uint32_t)__shfl((int)exk, quarter, 64);
            // (where round 1 or 2 found the cut no later round reads the list)
            uint32_t slot = 0;
            if (!ro.found && lane == 0)
                slot = (uint32_t)atomicAdd(&sel_lists[f], (unsigned long long)lane_value(ink, 63));
            slot = begin + uniform(slot);
            for (uint64_t todo = words; todo;) {  // uniform
                float v[kBatch];
                int at[kBatch];
                uint64_t m[kBatch];
#pragma unroll
                for (int u = 0; u < kBatch; ++u) {
                    at[u] = todo ? __builtin_ctzll(todo) : -1;
                    todo &= todo - 1ull;
                    m[u] = at[u] >= 0 ? lane_value(kept, at[u]) : 0ull;
                    v[u] = load_word(at[u], m[u]);
                }
#pragma unroll
                for (int u = 0; u < kBatch; ++u) {
                    if (at[u] < 0) break;  // uniform
                    const uint32_t k = (uint32_t)__builtin_amdgcn_mbcnt_hi(
                        (uint32_t)(m[u] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m[u], 0u));
                    const uint32_t to = 64u * (uint32_t)(at[u] & ~(kQuarter - 1)) + lane_value(exq, at[u]) + k;
                    const uint32_t list = slot + lane_value(exk, at[u]) + k;
                    if ((m[u] >> lane) & 1ull) {
                        pack[b + to] = v[u];  // (up to the keys read so far: later words' lie behind)
                        // the cell's list: from its first particle on (at most the cell's keys)
                        if (!ro.found) sel[list] = v[u];
                    }
                }
            }
        }
        mq[lane] = G;
        mq[kMaskWords + lane] = kept;
        if (lane == 0 && below) atomicAdd(&sel_lists[f], (unsigned long long)below << 32);
    }
}

// ---------------------------------------------------------------------------
// weighted levels of few chunks
// ---------------------------------------------------------------------------
// The weighted rounds bin every key of a searching cell in each of the four
// rounds (a weight histogram needs every key).  On a level of few chunks
// every block replays the round before from its cell's row of weight sums,
// starting from the margins the block of the cell's first chunk left in the
// round before that (state[round parity]), then bins its chunk and adds its
// row to the cell's row of this round: one launch a round where the chunk path
// takes three.  k_mw_masks replays the last round and writes the stopper
// masks, k_m_tail<true> takes the split and the plan.

// The state after `round` rounds: the state before it and its row.  Every wave
// that calls it gets it; trace_row (the round's left weights) where wanted.
__device__ inline RoundState weighted_state(const CellRec &r, uint32_t cell, int32_t nCells, int round,
                                            const RoundState *state, const uint64_t *rows, int lane,
                                            uint64_t *trace_row)
{
    RoundState s{uniform(r.margin_l), uniform(r.margin_r), 0, 0};
    if (round == 0) return s;
    if (round > 1) {
        s = load_state(state + (size_t)((round - 1) & 1) * (size_t)nCells + cell);
        if (s.found) return s;
    }
    const uint64_t *row = rows + ((size_t)(round - 1) * (size_t)nCells + cell) * kBins;
    const ulonglong2 a = reinterpret_cast<const ulonglong2 *>(row)[2 * lane];
    const ulonglong2 b2 = reinterpret_cast<const ulonglong2 *>(row)[2 * lane + 1];
    const uint64_t s0 = a.x, s1 = s0 + a.y, s2 = s1 + b2.x, s3 = s2 + b2.y;
    const uint64_t base = wave_inclusive_scan(s3) - s3;
    const uint64_t pv[4] = {base + s0, base + s1, base + s2, base + s3};
    const uint64_t weight = lane_value(pv[3], 63);  // every key of the cell was binned
    const float target = difference_target_w(weight, (int32_t)uniform((uint32_t)r.nLeaf));
    const RoundOut ro = replay_round_lanes(pv, s.L, s.R, target, s.passes, lane, trace_row);
    return RoundState{uniform(ro.L), uniform(ro.R), ro.passes, ro.found ? 1 : 0};
}

template <int LE>
__global__ __launch_bounds__(kBlock) void k_mw_hist(
    const CellRec *__restrict__ recs, int32_t nCells, const uint32_t *__restrict__ first,
    const uint4 *__restrict__ chunk_desc, uint32_t max_chunks, const float *__restrict__ x,
    const float *__restrict__ y, const float *__restrict__ z, const uint32_t *__restrict__ wgt,
    int round, RoundState *state, uint64_t *rows, uint64_t *trace)
{
    constexpr int kW = kBlock / 64;
    constexpr int kPerWave = kMaskWords / kW;  // 16 loads of 64 keys and weights
    __shared__ unsigned long long hist[kBins];
    const int t = threadIdx.x, lane = t & 63, w = (int)uniform((uint32_t)t >> 6);
    const uint32_t sb = (uint32_t)(w * kPerWave * 64);
    const uint32_t total = first[nCells];
    for (uint32_t q = blockIdx.x;; q += gridDim.x) {
        const uint4 d = chunk_record(chunk_desc, q, max_chunks);
        const uint32_t b = uniform(d.x), e = uniform(d.y), cell = uniform(d.z);
        const uint32_t axis = uniform(d.w);
        keep_values(b, e, cell, axis);
        if (q >= total) break;
        if (axis > 2u) continue;  // uniform: the cell is not searched
        float v[kPerWave];
        issue_chunk_loads(x, y, z, true, d, sb, lane, v);
        uint32_t wv[kPerWave];
        issue_weight_loads(wgt, d, sb, lane, wv);
        const CellRec &r = recs[cell];
        const bool lead = q == uniform(first[cell]);  // the cell's first chunk keeps its state
        uint64_t *trow = trace && lead && w == 0
                             ? trace + ((size_t)r.hb + r.id) * ORB_MAX_PASSES : nullptr;
        const RoundState s = weighted_state(r, cell, nCells, round, state, rows, lane, trow);
        if (lead && t == 0) state[(size_t)(round & 1) * (size_t)nCells + cell] = s;
        if (s.found) continue;  // uniform
        hist[t] = 0ull;
        __syncthreads();
        bin_weights<LE>(v, wv, s.L, s.R, hist, lane);
        __syncthreads();
        if (hist[t])
            atomicAdd(reinterpret_cast<unsigned long long *>(rows) +
                          ((size_t)round * (size_t)nCells + cell) * kBins + t, hist[t]);
        __syncthreads();  // the next chunk rewrites hist
    }
}

// The stopper masks of each chunk at its cell's cut (the state after the last
// round, which the block of the cell's first chunk leaves for k_m_tail).
__global__ __launch_bounds__(kBlock) void k_mw_masks(
    const CellRec *__restrict__ recs, int32_t nCells, const uint32_t *__restrict__ first,
    const uint4 *__restrict__ chunk_desc, uint32_t max_chunks, const float *__restrict__ x,
    const float *__restrict__ y, const float *__restrict__ z, RoundState *state,
    const uint64_t *__restrict__ rows, uint64_t *__restrict__ masks, uint64_t *trace)
{
    constexpr int kW = kBlock / 64;
    constexpr int kPerWave = kMaskWords / kW;
    const int t = threadIdx.x, lane = t & 63, w = (int)uniform((uint32_t)t >> 6);
    const uint32_t sb = (uint32_t)(w * kPerWave * 64);
    const uint32_t total = first[nCells];
    for (uint32_t q = blockIdx.x;; q += gridDim.x) {
        const uint4 d = chunk_record(chunk_desc, q, max_chunks);
        const uint32_t b = uniform(d.x), e = uniform(d.y), cell = uniform(d.z);
        const uint32_t axis = uniform(d.w);
        keep_values(b, e, cell, axis);
        if (q >= total) break;
        if (axis > 2u) continue;
        float v[kPerWave];
        issue_chunk_loads(x, y, z, true, d, sb, lane, v);
        const CellRec &r = recs[cell];
        const bool lead = q == uniform(first[cell]);
        uint64_t *trow = trace && lead && w == 0
                             ? trace + ((size_t)r.hb + r.id) * ORB_MAX_PASSES : nullptr;
        const RoundState s = weighted_state(r, cell, nCells, kRounds, state, rows, lane, trow);
        if (lead && t == 0) state[(size_t)(kRounds & 1) * (size_t)nCells + cell] = s;
        const float cut = cell_cut(s.L, s.R);
        const uint32_t len = e - b;
        uint64_t mineL = 0ull, mineR = 0ull;
        static_for<0, kPerWave>([&](auto jc) __attribute__((always_inline)) {
            constexpr int j = decltype(jc)::value;
            const bool in = sb + 64u * (uint32_t)j + (uint32_t)lane < len;
            const uint64_t mL = __ballot(in && !(v[j] < cut));
            const uint64_t mR = __ballot(in && !(v[j] > cut));
            mineL = lane == j ? mL : mineL;
            mineR = lane == j ? mR : mineR;
        });
        uint64_t *mq = masks + (size_t)q * (2 * kMaskWords) + w * kPerWave;
        if (lane < kPerWave) {
            mq[lane] = mineL;
            mq[kMaskWords + lane] = mineR;
        }
    }
}

// The rest of a cell's search and its split, a block per cell: after rounds 1 and
// 2 (state) the later rounds over the listed keys (those inside the margins),
// the cell's record and children, the stopper masks of its chunks from the
// narrowed words and packed keys, the chunks' stopper offsets, K and i
// as in k_b_cell (the crossing chunk, its word, its bit), the children's
// ranges, and each chunk's swap unit as k_hoare_plan makes it.  WEIGHTED: the
// search and the masks are done (state, k_mw_masks); the chunks' counts come
// from the masks.  STABLE: the chunks' offsets of the keys going left (<= cut:
// the R-stoppers) and right, for k_stable_scatter, in place of K, i and the plan.
// A cell of a stable level is never left alone (where the level's scatter fills
// the other buffer, all of its cells have to), so its chunks go through the
// tables kMidChunks at a time.  o=2 builds, host time: 2^16 to 64 leaves 403 ->
// 234 us, 2^20 to 1024 804 -> 500 us, 500003 with ids and weights 741 -> 422 us.
constexpr int kTailBlock = 1024;
template <bool WEIGHTED, bool STABLE>
__global__ __launch_bounds__(kTailBlock) void k_m_tail(
    CellRec *recs, int32_t nCells, const uint32_t *__restrict__ first, uint32_t *cell_hist,
    const float *__restrict__ sel, const unsigned long long *__restrict__ sel_lists,
    const float *__restrict__ pack, const RoundState *__restrict__ state, uint64_t *rows, uint64_t *masks, uint64_t *chunk_pre, SplitRec *splits,
    SwapPlan *plan, uint32_t *ranges, orb_cell *heap, uint8_t *exists, int le_cmp, uint64_t *trace,
    int32_t *level_passes, int32_t *status)
{
    constexpr int kW = kTailBlock / 64;
    __shared__ uint32_t hist[kBins];
    __shared__ uint32_t preL[kMidChunks + 1], preR[kMidChunks + 1];
    __shared__ uint64_t s_sum[kW];
    __shared__ uint32_t s_cnt[kW];
    __shared__ float s_lr[2];
    __shared__ int32_t s_pf[2];
    __shared__ uint32_t s_K, s_i, s_ks;
    const int t = threadIdx.x, lane = t & 63, w = (int)uniform((uint32_t)t >> 6);
    for (int32_t c = blockIdx.x; c < nCells; c += gridDim.x) {
        const CellRec &rec = recs[c];  // this block alone writes it
        if (uniform((uint32_t)rec.flags) != 0u) {
            if (t == 0) splits[c] = SplitRec{0u, 0u, 0u, 0u};
            continue;  // uniform
        }
        const uint32_t begin = uniform(rec.begin), n = uniform(rec.end) - begin;
        const int32_t id = (int32_t)uniform((uint32_t)rec.id), hb = (int32_t)uniform((uint32_t)rec.hb);
        const uint32_t f = uniform(first[c]), nch = uniform(first[c + 1]) - f;
        // the cell's rows: the next level adds to zero
        auto clear_rows = [&] {
            if constexpr (WEIGHTED) {
                for (int q = t; q < kRounds * kBins; q += kTailBlock)
                    rows[((size_t)(q / kBins) * (size_t)nCells + c) * kBins + q % kBins] = 0ull;
            } else if (t < 2 * kBins) {
                cell_hist[((size_t)(t / kBins) * (size_t)nCells + c) * kBins + t % kBins] = 0u;
            }
        };
        // a cell that the swap leaves alone: no split, no unit in its chunks
        auto idle = [&](int kind) {
            if (t == 0) {
                report_error(status + rec.st, rec.lp & 63, kind, id);
                splits[c] = SplitRec{0u, 0u, 0u, 0u};
            }
            for (uint32_t k = (uint32_t)t; k < nch; k += kTailBlock)
                reinterpret_cast<uint4 *>(plan + f + k)[0] = make_uint4(~0u, 0u, 0u, 0u);
        };
        if (!STABLE && nch > (uint32_t)kMidChunks) {
            // the level records hand over at most kMidChunks; refuse anything else
            clear_rows();
            idle(kErrSplit);
            continue;  // uniform
        }
        float lo = uniform(rec.margin_l), hi = uniform(rec.margin_r);
        int32_t passes = 0;
        bool found = false;
        if constexpr (WEIGHTED) {
            if (nch) {
                const RoundState s = state[(size_t)(kRounds & 1) * (size_t)nCells + c];
                lo = uniform(s.L);
                hi = uniform(s.R);
                passes = (int32_t)uniform((uint32_t)s.passes);
                found = uniform((uint32_t)s.found) != 0u;
            } else {
                // no chunk carried the rounds of an empty cell: its first pass
                // finds 0 of 0
                passes = 1;
                found = true;
                if (trace && t == 0) trace[((size_t)hb + id) * ORB_MAX_PASSES] = 0ull;
            }
            clear_rows();
        } else {
            uint64_t *trow = trace ? trace + ((size_t)hb + id) * ORB_MAX_PASSES : nullptr;
            // (no chunk carries the rounds of an empty cell: rows of zeros)
            RoundState r2{lo, hi, 0, 0};
            if (nch) r2 = load_state(state + (size_t)nCells + c);
            else r2 = replay_row(cell_hist + (size_t)c * kBins, rec, r2, lane, w == 0 ? trow : nullptr);
            lo = r2.L;
            hi = r2.R;
            passes = r2.passes;
            found = r2.found != 0;
            const unsigned long long list = n ? sel_lists[f] : 0ull;
            const uint32_t m = uniform((uint32_t)list) < n ? uniform((uint32_t)list) : n;
            const uint32_t nbelow = uniform((uint32_t)(list >> 32));
            const float target = difference_target(n, (int32_t)uniform((uint32_t)rec.nLeaf));
            if (t < kBins) hist[t] = 0u;
            __syncthreads();
            clear_rows();
            while (!found && passes < ORB_MAX_PASSES) {
                const float width = hi - lo;
                const float scale = width > 0.0f ? (float)kBins / width : 0.0f;
                const float lim = 0.5f - bin_tolerance(lo, hi, scale);
                uint32_t below = 0;  // wave-uniform
                for (uint32_t k0 = 0; k0 < m; k0 += 4u * kTailBlock) {
                    float v[4];
                    bool in[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const uint32_t k = k0 + (uint32_t)(u * kTailBlock + t);
                        in[u] = k < m;
                        v[u] = in[u] ? sel[begin + k] : 0.0f;
                    }
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const bool lt = in[u] && v[u] < lo, on = in[u] && !(v[u] < lo) && !(v[u] > hi);
                        below += (uint32_t)__popcll(__ballot(lt));
                        int bin = 0;
                        if (on && !bin_estimate(v[u], lo, scale, lim, bin))
                            bin = le_cmp ? bin_walk<1>(v[u], lo, hi) : bin_walk<0>(v[u], lo, hi);
                        count_bin(hist, bin, on);
                    }
                }
                if (lane == 0 && below) atomicAdd(&hist[0], below);
                if (t == 0 && nbelow) atomicAdd(&hist[0], nbelow);  // the keys below the list's
                __syncthreads();
                if (w == 0) {
                    const uint4 h4 = reinterpret_cast<const uint4 *>(hist)[lane];
                    reinterpret_cast<uint4 *>(hist)[lane] = make_uint4(0u, 0u, 0u, 0u);
                    const uint32_t s0 = h4.x, s1 = s0 + h4.y, s2 = s1 + h4.z, s3 = s2 + h4.w;
                    const uint32_t base = wave_inclusive_scan(s3) - s3;
                    const uint32_t pv[4] = {base + s0, base + s1, base + s2, base + s3};
                    const RoundOut ro = replay_round_lanes(pv, lo, hi, target, passes, lane, trow);
                    if (lane == 0) {
                        s_lr[0] = ro.L;
                        s_lr[1] = ro.R;
                        s_pf[0] = ro.passes;
                        s_pf[1] = ro.found ? 1 : 0;
                    }
                }
                __syncthreads();
                lo = uniform(s_lr[0]);
                hi = uniform(s_lr[1]);
                passes = (int32_t)uniform((uint32_t)s_pf[0]);
                found = uniform((uint32_t)s_pf[1]) != 0u;
            }
        }
        const float cut = cell_cut(lo, hi);
        // ---- the chunks' masks and stopper offsets, kMidChunks at a time (a
        // cell of the stable partition may hold more: its level's other buffer
        // takes over, so none of its cells can be left alone)
        uint64_t off = 0ull, all = 0ull;  // this thread's chunk; the chunks so far
        for (uint32_t tile = 0; tile == 0u || tile < nch; tile += (uint32_t)kMidChunks) {
            const uint32_t nt = nch - tile < (uint32_t)kMidChunks ? nch - tile : (uint32_t)kMidChunks;
            if constexpr (WEIGHTED) {
                for (uint32_t k = (uint32_t)w; k < nt; k += kW) {
                    const uint64_t *mq = masks + (size_t)(f + tile + k) * (2 * kMaskWords);
                    const uint32_t nl = wave_sum((uint32_t)__popcll(mq[lane]));
                    const uint32_t nr = wave_sum((uint32_t)__popcll(mq[kMaskWords + lane]));
                    if (lane == 0) {
                        preL[k] = nl;
                        preR[k] = nr;
                    }
                }
            } else {
                // ---- stopper masks: a wave per kPer chunks, a word per lane
                constexpr int kPer = 4;
                for (uint32_t k0 = (uint32_t)(w * kPer); k0 < nt; k0 += (uint32_t)(kW * kPer)) {
                    uint64_t G[kPer], W[kPer];
                    float v0[kPer];
                    const float *pk[kPer];
#pragma unroll
                    for (int u = 0; u < kPer; ++u) {
                        const uint32_t k = tile + (k0 + (uint32_t)u < nt ? k0 + (uint32_t)u : nt - 1u);
                        const uint64_t *mq = masks + (size_t)(f + k) * (2 * kMaskWords);
                        G[u] = mq[lane];
                        W[u] = mq[kMaskWords + lane];
                    }
#pragma unroll
                    for (int u = 0; u < kPer; ++u) {
                        const uint32_t k = tile + (k0 + (uint32_t)u < nt ? k0 + (uint32_t)u : nt - 1u);
                        const uint32_t cw = (uint32_t)__popcll(W[u]);
                        const uint32_t ex = wave_inclusive_scan(cw) - cw;
                        const int q0 = lane & ~15;  // first word of this lane's quarter
                        const uint32_t rank = ex - (uint32_t)__shfl((int)ex, q0, 64);
                        pk[u] = pack + begin + k * (uint32_t)kChunk + 64u * (uint32_t)q0 + rank;
                        v0[u] = W[u] ? *pk[u] : 0.0f;
                    }
#pragma unroll
                    for (int u = 0; u < kPer; ++u) {
                        const uint32_t k = tile + k0 + (uint32_t)u;
                        if (k0 + (uint32_t)u >= nt) break;  // uniform
                        const uint32_t p0 = k * (uint32_t)kChunk + 64u * (uint32_t)lane;
                        const uint64_t valid =
                            p0 >= n ? 0ull : (n - p0 >= 64u ? ~0ull : (1ull << (n - p0)) - 1ull);
                        uint64_t L = G[u], R = valid & ~G[u] & ~W[u], wd = W[u];
                        float vk = v0[u];
                        const float *at = pk[u];
                        while (wd) {
                            const uint32_t bit = (uint32_t)__builtin_ctzll(wd);
                            wd &= wd - 1ull;
                            L |= (!(vk < cut) ? 1ull : 0ull) << bit;
                            R |= (!(vk > cut) ? 1ull : 0ull) << bit;
                            if (wd) vk = *++at;
                        }
                        uint64_t *mq = masks + (size_t)(f + k) * (2 * kMaskWords);
                        mq[lane] = L;
                        mq[kMaskWords + lane] = R;
                        const uint32_t nl = wave_sum((uint32_t)__popcll(L));
                        const uint32_t nr = wave_sum((uint32_t)__popcll(R));
                        if (lane == 0) {
                            preL[k - tile] = nl;
                            preR[k - tile] = nr;
                        }
                    }
                }
            }
            __syncthreads();
            uint64_t mine = (uint32_t)t < nt ? (uint64_t)preL[t] | ((uint64_t)preR[t] << 32) : 0ull;
            if constexpr (STABLE) {
                // keys going left, and the chunk's others
                const uint32_t b0 = (tile + (uint32_t)t) * (uint32_t)kChunk;
                const uint32_t len = n - b0 < (uint32_t)kChunk ? n - b0 : (uint32_t)kChunk;
                const uint32_t nle = hi32(mine);
                mine = (uint32_t)t < nt ? (uint64_t)nle | ((uint64_t)(len - nle) << 32) : 0ull;
            }
            const uint64_t inc = wave_inclusive_scan(mine);
            if (lane == 63) s_sum[w] = inc;
            __syncthreads();
            const uint64_t ws = lane < kW ? s_sum[lane] : 0ull;
            const uint64_t wp = wave_inclusive_scan(ws);
            off = all + inc - mine + lane_value(wp, w) - lane_value(ws, w);
            all += lane_value(wp, 63);
            if ((uint32_t)t <= nt && t <= kMidChunks) {
                preL[t] = lo32(off);
                preR[t] = hi32(off);
                chunk_pre[f + (uint32_t)c + tile + (uint32_t)t] = off;
            }
            if constexpr (STABLE) __syncthreads();  // the next tile rewrites the tables
        }
        const uint32_t TL = lo32(all), TR = hi32(all);
        if (t == 64)  // the cell's margins, its passes, its children
            finish_round(rec, c, RoundOut{lo, hi, passes, found, 0}, found ? 1 : 0, recs, heap,
                         level_passes, exists, status);
        const int64_t lid = left_child_id(id), rid = right_child_id(id);
        if constexpr (STABLE) {
            // as k_stable_ranges: an empty side is no error
            if (t == 0) {
                if (rid >= (int64_t)rec.capr) {
                    report_error(status + rec.st, rec.lp & 63, kErrPartition, id);
                } else {
                    splits[c] = SplitRec{TL, TR, 0u, TL};
                    const int64_t gl = hb + lid, gr = hb + rid;
                    ranges[2 * gl] = begin;
                    ranges[2 * gl + 1] = begin + TL;
                    ranges[2 * gr] = begin + TL;
                    ranges[2 * gr + 1] = begin + n;
                }
            }
            // k_stable_scatter reads the cut and the axis of the record
            __syncthreads();  // the next cell rewrites the tables
            continue;
        }
        if (n == 0u || TL == 0u || rid >= (int64_t)(int32_t)uniform((uint32_t)rec.capr)) {
            // empty cell or no key >= cut: the reference's loop leaves the cell
            idle(kErrPartition);
            __syncthreads();  // the next cell rewrites the tables
            continue;  // uniform
        }
        // ---- K and i (see k_b_cell); A and B at this thread's chunk
        const uint32_t cA = lo32(off), cB = TR - hi32(off);
        auto last_chunk = [&](bool pred) {  // the last chunk where pred holds (true, then false)
            const uint64_t mb = __ballot((uint32_t)t < nch && pred);
            if (lane == 0) s_cnt[w] = (uint32_t)__popcll(mb);
            __syncthreads();
            if (t == 0) {
                uint32_t k = 0;
                for (int u = 0; u < kW; ++u) k += s_cnt[u];
                s_ks = k - 1u;  // it holds at chunk 0
            }
            __syncthreads();
        };
        // A and B at bit `lane` of the word of chunk k that pred(A, B) picks
        // (the last whose start it holds at), and just after it
        auto at_bit = [&](uint32_t k, auto pred, uint32_t &q, uint32_t &a0, uint32_t &b0,
                          uint32_t &a1, uint32_t &b1) {
            const uint64_t *mq = masks + (size_t)(f + k) * (2 * kMaskWords);
            const uint64_t L = mq[lane], R = mq[kMaskWords + lane];
            const uint32_t cL = (uint32_t)__popcll(L), cR = (uint32_t)__popcll(R);
            const uint32_t xA = preL[k] + wave_inclusive_scan(cL) - cL;
            const uint32_t xB = TR - (preR[k] + wave_inclusive_scan(cR) - cR);
            q = 63u - (uint32_t)__clzll((long long)__ballot(pred(xA, xB)));
            const uint64_t mL = lane_value(L, (int)q), mR = lane_value(R, (int)q);
            a0 = lane_value(xA, (int)q) + (uint32_t)__builtin_amdgcn_mbcnt_hi(
                     (uint32_t)(mL >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mL, 0u));
            b0 = lane_value(xB, (int)q) - (uint32_t)__builtin_amdgcn_mbcnt_hi(
                     (uint32_t)(mR >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mR, 0u));
            a1 = a0 + (uint32_t)((mL >> lane) & 1ull);
            b1 = b0 - (uint32_t)((mR >> lane) & 1ull);
        };
        last_chunk(cA <= cB);
        if (w == 0) {
            uint32_t q, a0, b0, a1, b1;
            at_bit(s_ks, [](uint32_t a, uint32_t b) { return a <= b; }, q, a0, b0, a1, b1);
            const uint32_t k0 = a0 < b0 ? a0 : b0, k1 = a1 < b1 ? a1 : b1;
            const uint32_t best = wave_max(k0 > k1 ? k0 : k1);
            if (lane == 0) s_K = best;
        }
        __syncthreads();
        const uint32_t K = uniform(s_K);
        last_chunk(cA <= K && K <= cB);
        if (w == 0) {
            const uint32_t k = s_ks;
            uint32_t q, a0, b0, a1, b1;
            at_bit(k, [&](uint32_t a, uint32_t b) { return a <= K && K <= b; }, q, a0, b0, a1, b1);
            const uint64_t mb = __ballot(a0 <= K && K <= b0);
            if (lane == 0)
                s_i = k * (uint32_t)kChunk + 64u * q + 63u - (uint32_t)__clzll((long long)mb);
        }
        __syncthreads();
        const uint32_t i = uniform(s_i);
        // ---- the swap plan, a chunk per thread (k_hoare_plan)
        if ((uint32_t)t < nch) {
            const uint32_t kc = (uint32_t)t;
            const int owner = 2ull * i >= (uint64_t)n ? 0 : 1;
            const uint32_t t0 = owner ? TR - preR[kc + 1] : preL[kc];
            uint32_t t1 = owner ? TR - preR[kc] : preL[kc + 1];
            if (t1 > K) t1 = K;
            uint4 p0 = make_uint4(~0u, 0u, 0u, 0u), p1 = make_uint4(0u, 0u, 0u, 0u);
            if (t0 < t1) {
                // the first partner chunk: the last k with at(partner, k) <= ap0
                const uint32_t *pre = owner ? preL : preR;
                const uint32_t ap0 = owner ? t0 : TR - t1;
                uint32_t a = 0, b = nch - 1u;
                while (a < b) {
                    const uint32_t mid = (a + b + 1u) >> 1;
                    if (pre[mid] <= ap0) a = mid;
                    else b = mid - 1u;
                }
                p0 = make_uint4(t0 | ((uint32_t)owner << 31), t1, TR, begin);
                p1 = make_uint4(f, nch, a, f + (uint32_t)c);
            }
            uint4 *dst = reinterpret_cast<uint4 *>(plan + f + kc);
            dst[0] = p0;
            dst[1] = p1;
        }
        if (t == 0) {
            splits[c] = SplitRec{TL, TR, K, i};
            const int64_t gl = hb + lid, gr = hb + rid;
            ranges[2 * gl] = begin;
            ranges[2 * gl + 1] = begin + i;
            ranges[2 * gr] = begin + i;
            ranges[2 * gr + 1] = begin + n;
        }
        __syncthreads();  // the next cell rewrites the tables
    }
}

// ---------------------------------------------------------------------------
// orchestration
// ---------------------------------------------------------------------------
// The most cells of a predicted level: at least kPredKeys keys each (less what a
// level's sizes vary by).
static size_t predicted_cells(const Ctx &c)
{
    return (size_t)(c.n / (kPredKeys / 2)) + 2;
}

// Words of the cells' rows of counts: a row a cell (the chunk path), or two on
// levels of few chunks (fewer than kRecsScan cells).
size_t cell_hist_words(const Ctx &c)
{
    const size_t m = (size_t)c.max_level_cells;
    return std::max(m, 2 * std::min(m, (size_t)kRecsScan)) * kBins;
}

// Rows of weight sums: one a cell (the chunk path), or one a cell and round
// for levels of few chunks (fewer than kRecsScan cells).
static size_t hist_w_rows(const Ctx &c)
{
    const size_t m = (size_t)c.max_level_cells;
    return std::max(m, (size_t)kRounds * std::min(m, (size_t)kRecsScan));
}

static int ensure_state(Ctx &c, int32_t levels_mode, bool *complete)
{
    if (!c.batched) c.batched = new (std::nothrow) BatchedState;
    if (!c.batched) return ORB_ERR_NOMEM;
    BatchedState &b = *c.batched;
    if (b.levels_mode != levels_mode || b.d != c.d) ORB_TRY(make_schedule(c, b, levels_mode, complete));
    else *complete = b.complete;
    b.complete = *complete;
    ORB_TRY(b.heap.alloc((size_t)c.cap));
    ORB_TRY(b.exists.alloc((size_t)c.cap));
    ORB_TRY(b.sub.alloc((size_t)c.cap));
    ORB_TRY(b.chunk_hist.alloc(kHistRegions * (size_t)(c.max_chunks + 1) * kBins));
    // a fresh (or grown, hence reallocated) buffer is cleared before use
    if (b.cell_hist.n < cell_hist_words(c)) b.hist_clean = false;
    ORB_TRY(b.cell_hist.alloc(cell_hist_words(c)));
    ORB_TRY(b.level_passes.alloc(64));
    ORB_TRY(b.hpasses.alloc(64));
    if (c.trace) ORB_TRY(b.trace.alloc((size_t)c.cap * ORB_MAX_PASSES));
    if (c.weighted) {
        ORB_TRY(b.chunk_hist_w.alloc((size_t)(c.max_chunks + 1) * kBins));
        const size_t rows = hist_w_rows(c);
        if (b.cell_hist_w.n < rows * kBins) b.hist_w_clean = false;
        ORB_TRY(b.cell_hist_w.alloc(rows * kBins));
    }
    if (!c.weighted) ORB_TRY(c.sel.alloc((size_t)c.stride));  // rounds 3 and 4
    if (!c.weighted && c.n >= kPredLevelKeys) {
        const size_t cells = predicted_cells(c);
        if (c.sample_hist.n < cells * kSampleRow) b.sample_clean = false;
        ORB_TRY(c.sample_hist.alloc(cells * kSampleRow));
        ORB_TRY(c.windows.alloc(cells * (sizeof(Window) + kSampleBins) / 4));
    }
    // every buffer the launches touch exists before a capture starts
    ORB_TRY(preallocate_scratch(c));
    return ORB_OK;
}

int32_t subtree_max_keys(const Ctx &c)
{
    const int32_t cap = subtree_capacity(c);
    return c.sub_max_keys < 0 ? cap : (c.sub_max_keys > cap ? cap : c.sub_max_keys);
}

// The subtree kernel's limit on a level of `cells` cells.  A level that gives
// every CU several takes the half-sized blocks: at 2^26 keys the five levels
// from 8192-key cells down took 2.37 ms in whole blocks, 1.69 ms and 0.43 ms
// with the first of them in k_b_cell.  With fewer cells latency decides, and the whole
// block's levels are the shorter.
constexpr int32_t kSubManyCells = 1024;
static int32_t subtree_limit(const Ctx &c, int32_t cells)
{
    const int32_t whole = subtree_max_keys(c);
    return cells > kSubManyCells && !c.track_ids && !c.weighted
               ? std::min(whole, SubCap<false, false, 512>::value) : whole;
}

static void drop_graph(BatchedState &b)
{
    if (b.exec) (void)hipGraphExecDestroy(b.exec);
    if (b.graph) (void)hipGraphDestroy(b.graph);
    b.exec = nullptr;
    b.graph = nullptr;
    b.gsig.clear();
}

// What a captured build holds fixed: the settings that choose its launches,
// the launch shapes, and the address of every device buffer it touches (a
// buffer freed and allocated again -- orb_enable_ids off and on, a level
// table grown by a service call with more cells -- has a new address, and a
// replay through the old one would write freed memory).
static std::vector<uint64_t> graph_signature(const Ctx &c, const BatchedState &b,
                                             int32_t levels_mode)
{
    std::vector<uint64_t> s = {(uint64_t)levels_mode, (uint64_t)c.cmp, (uint64_t)c.part,
                               (uint64_t)c.trace, (uint64_t)c.track_ids, (uint64_t)c.weighted,
                               (uint64_t)c.n,
                               (uint64_t)c.d, (uint64_t)c.max_chunks,
                               (uint64_t)c.max_level_cells, (uint64_t)(int64_t)c.sub_max_keys};
    const void *bufs[] = {c.pos.p, c.tmp.p, c.pid.p, c.pid_tmp.p, c.ranges.p, c.recs.p,
                          c.cell_nchunks.p, c.cell_first.p, c.chunk_cell.p, c.chunk_desc.p,
                          c.chunk_ltle.p, c.chunk_cnt.p, c.chunk_pre.p, c.scan_partials.p,
                          c.packed.p, c.masks.p, c.cell_cand.p, c.splits.p, c.chunk_comp.p,
                          c.sel.p, c.sel_lists.p, c.swap_plan.p, c.status.p, c.stamps.p, b.level_ids.p, b.heap.p, b.exists.p,
                          b.sub.p, b.chunk_hist.p, b.cell_hist.p, b.trace.p, b.level_passes.p,
                          c.wt.p, c.wt_tmp.p, b.chunk_hist_w.p, b.cell_hist_w.p, c.sample_hist.p, c.windows.p, c.hstatus.p, b.hpasses.p};
    for (const void *p : bufs) s.push_back((uint64_t)(uintptr_t)p);
    s.push_back((uint64_t)c.tune_chunk_blocks.size());
    for (int32_t v : c.tune_chunk_blocks) s.push_back((uint64_t)(int64_t)v);
    s.push_back((uint64_t)c.tune_sub_blocks.size());
    for (int32_t v : c.tune_sub_blocks) s.push_back((uint64_t)(int64_t)v);
    return s;
}

int enqueue_level(Ctx &c, const LevelEntry *entries, int32_t nCells, orb_cell *heap,
                  uint8_t *exists, uint8_t *sub, uint16_t *chunk_hist, uint32_t *cell_hist,
                  uint64_t *trace, int32_t *level_passes, int32_t *status, bool any_subtree,
                  bool full_cover, int32_t level, uint64_t *chunk_hist_w, uint64_t *cell_hist_w,
                  const PendingFinal *fin_in, bool defer_final, const LevelKernels &kernels)
{
    if (c.weighted && (!chunk_hist_w || !cell_hist_w)) return ORB_ERR_STATE;
    if (!c.weighted && (c.sel.n < (size_t)c.stride || c.sel_lists.n < (size_t)c.max_chunks + 1))
        return ORB_ERR_STATE;  // rounds 3 and 4 gather into these
    const int32_t sub_max = kernels.sub_max ? std::min((int32_t)kernels.sub_max, subtree_max_keys(c))
                                            : subtree_max_keys(c);
    const bool use_subtree = any_subtree && c.part == ORB_PART_HOARE && sub_max > 0;
    if (kernels.cell_max && (c.part != ORB_PART_HOARE || c.weighted)) return ORB_ERR_STATE;
    const bool mid = kernels.chunks == kChunksMid;
    if (mid && nCells >= kRecsScan) return ORB_ERR_STATE;  // one block fills its tables
    const LevelMode mode{use_subtree ? (uint32_t)sub_max : 0u, kernels.cell_max,
                         kernels.chunks == kChunksAll || (mid && c.part == ORB_PART_STABLE_LE) ? ~0u
                         : mid ? (uint32_t)(kMidChunks * kChunk) : 0u,
                         kernels.again ? 1 : 0};
    const int32_t cgroup = cell_group(nCells);
    // Chunk order: the first round walks the level's chunks from the last, so
    // it starts with the chunks the previous level's swap wrote last (still in
    // the memory-side cache), and the window round walks them from the first,
    // starting with the chunks the first round read last.  (Measured at C2:
    // -0.26 ms per build against both forward; reversing the swap on
    // alternate levels as well gained less.)
    const int rev = 1;
    const int le = c.cmp == ORB_CMP_LE ? 1 : 0;
    c.cur_level = level;  // chunk_grid() and the subtree grid read the level's shapes
    struct LevelScope {
        Ctx &c;
        ~LevelScope() { c.cur_level = -1; }
    } scope{c};
    // the level's first launch also runs the previous level's last row swaps
    // (extra blocks: the records it rewrites are not what they read)
    PendingFinalDev fin{nullptr, 0, c.splits.p, c.x(), c.y(), c.z(), c.ids(), c.weights()};
    if (fin_in && fin_in->nCells > 0) {
        fin.entries = fin_in->entries;
        fin.nCells = fin_in->nCells;
    }
    if (nCells < kRecsScan) {
        const unsigned gf = (unsigned)((fin.nCells + kRecsScan - 1) / kRecsScan);
        hipLaunchKernelGGL(mid ? k_b_recs_scan<true> : k_b_recs_scan<false>, dim3(1 + gf),
                           dim3(kRecsScan), 0, c.stream, entries, nCells, heap, exists, c.ranges.p, sub,
                           mode, c.recs.p, c.cell_first.p, level_passes, c.chunk_desc.p,
                           (uint32_t)c.max_chunks,
                           reinterpret_cast<unsigned long long *>(c.sel_lists.p), fin);
        ORB_HIP(hipGetLastError());
    } else {
        unsigned g1 = (unsigned)((nCells + 1 + kBlock - 1) / kBlock);
        const unsigned gf = (unsigned)((fin.nCells + kBlock - 1) / kBlock);
        hipLaunchKernelGGL(k_b_recs, dim3(g1 + gf), dim3(kBlock), 0, c.stream, entries, nCells, heap,
                           exists, c.ranges.p, sub, mode, c.recs.p, c.cell_nchunks.p, level_passes,
                           g1, fin);
        ORB_HIP(hipGetLastError());
        if (kernels.chunks == kChunksAll)
            ORB_TRY(scan_exclusive_u32(c, c.cell_nchunks.p, c.cell_first.p, (size_t)nCells + 1));
    }
    if (kernels.chunks == kChunksAll) {
        // the chunk table, and the first round's candidate tables (not used
        // by weighted builds)
        const int tb = timing_mark(c);
        const unsigned fill_blocks =
            (unsigned)std::min<int64_t>(16384, std::max<int64_t>(1, (c.max_chunks + kBlock - 1) / kBlock));
        const unsigned cand_blocks = c.weighted || kernels.predict ? 0u : cell_group_blocks(nCells, cgroup);
        hipLaunchKernelGGL(k_b_tables, dim3(fill_blocks + cand_blocks), dim3(kBlock), 0, c.stream,
                           c.cell_first.p, nCells, c.recs.p, c.chunk_cell.p, c.chunk_desc.p,
                           (uint32_t)c.max_chunks, c.cell_cand.p, cgroup, fill_blocks);
        ORB_HIP(hipGetLastError());
        ORB_TRY(timing_pair(c, tb, kTimeCount));
    }
    // tie rows: only the stable partition's stopper counts read them
    uint16_t *chunk_tie =
        c.part == ORB_PART_STABLE_LE ? chunk_hist + (size_t)(c.max_chunks + 1) * kBins : nullptr;
    uint16_t *later_hist = chunk_hist + 2 * (size_t)(c.max_chunks + 1) * kBins;
    if (use_subtree) {
        // one block fits a CU (LDS): four blocks per CU by default, each
        // taking groups of consecutive cells; a group holds about
        // nCells / 1024 cells (1 to 64), so a level of subtree roots spreads
        // over every CU and a level with none is read in few loads
        int32_t sb = 1024;
        if (level >= 0 && level < (int32_t)c.tune_sub_blocks.size() &&
            c.tune_sub_blocks[(size_t)level] > 0)
            sb = c.tune_sub_blocks[(size_t)level];
        int32_t group = 1;
        while (group < 64 && (int64_t)group * 2 * 1024 <= (int64_t)nCells) group *= 2;
        const int32_t ngroups = (nCells + group - 1) / group;
        const unsigned gs = (unsigned)(ngroups < sb ? ngroups : sb);
        const bool half = !c.track_ids && !c.weighted && sub_max <= SubCap<false, false, 512>::value;
        auto subtree =
            half ? k_b_subtree<false, false, 512>
            : c.track_ids ? (c.weighted ? k_b_subtree<true, true, 1024> : k_b_subtree<true, false, 1024>)
                          : (c.weighted ? k_b_subtree<false, true, 1024> : k_b_subtree<false, false, 1024>);
        hipLaunchKernelGGL(subtree, dim3(gs), dim3(half ? 512 : 1024), 0, c.stream, c.recs.p, nCells, heap,
                           exists, sub, c.ranges.p, c.x(), c.y(), c.z(), le, trace, level_passes,
                           status, c.ids(), c.weights(), group);
        ORB_HIP(hipGetLastError());
    }
    if (kernels.cell_max) {
        const bool payload = c.ids() != nullptr;
        const bool large = kernels.cell_max > kCellSmall, many = nCells > kCellManyCells;
        const bool tiny = kernels.cell_max <= kCellTiny;
        auto cell = large  ? (payload ? k_b_cell<1024, 40, 4> : k_b_cell<1024, 40, 3>)
                    : many ? (tiny ? (payload ? k_b_cell<256, 40, 4> : k_b_cell<256, 40, 3>)
                                   : (payload ? k_b_cell<512, 40, 4> : k_b_cell<512, 40, 3>))
                           : (payload ? k_b_cell<1024, 20, 4> : k_b_cell<1024, 20, 3>);
        hipLaunchKernelGGL(cell, dim3((unsigned)std::min<int32_t>(nCells, 65536)),
                           dim3(!large && many ? (tiny ? 256 : 512) : 1024), 0, c.stream, c.recs.p, nCells, heap,
                           exists, c.ranges.p, c.x(), c.y(), c.z(), c.ids(), c.weights(), le, trace,
                           level_passes, status);
        ORB_HIP(hipGetLastError());
    }
    if (kernels.chunks == kChunksNone) return ORB_OK;
    const unsigned gq = chunk_grid(c);
    if (mid) {
        int tb = timing_mark(c);
        unsigned long long *lists = reinterpret_cast<unsigned long long *>(c.sel_lists.p);
        static_assert(sizeof(RoundState) == sizeof(SplitRec), "they follow the splits");
        RoundState *state = reinterpret_cast<RoundState *>(c.splits.p + c.max_level_cells);
        const uint32_t mc = (uint32_t)c.max_chunks;
        if (c.weighted) {
            for (int r = 0; r < kRounds; ++r)
                hipLaunchKernelGGL(le ? k_mw_hist<1> : k_mw_hist<0>, dim3(gq), dim3(kBlock), 0, c.stream,
                                   c.recs.p, nCells, c.cell_first.p, c.chunk_desc.p, mc, c.x(), c.y(),
                                   c.z(), c.weights(), r, state, cell_hist_w, trace);
        } else {
            hipLaunchKernelGGL(le ? k_m_hist<1> : k_m_hist<0>, dim3(gq), dim3(kBlock), 0, c.stream,
                               c.recs.p, nCells, c.cell_first.p, c.chunk_desc.p, mc, c.x(), c.y(), c.z(),
                               cell_hist);
            hipLaunchKernelGGL(le ? k_m_window<1> : k_m_window<0>, dim3(gq), dim3(kBlock), 0, c.stream,
                               c.recs.p, nCells, c.cell_first.p, c.chunk_desc.p, mc, c.x(), c.y(), c.z(),
                               cell_hist, state, trace, c.packed.p, c.masks.p);
            hipLaunchKernelGGL(k_m_narrow, dim3((gq + 3) / 4), dim3(kBlock), 0, c.stream, c.recs.p, nCells,
                               c.cell_first.p, c.chunk_desc.p, mc, cell_hist, state, trace, c.packed.p,
                               c.masks.p, c.sel.p, lists);
        }
        ORB_HIP(hipGetLastError());
        ORB_TRY(timing_pair(c, tb, kTimeCount));
        const int tp = timing_mark(c);
        if (c.weighted)
            hipLaunchKernelGGL(k_mw_masks, dim3(gq), dim3(kBlock), 0, c.stream, c.recs.p, nCells,
                               c.cell_first.p, c.chunk_desc.p, mc, c.x(), c.y(), c.z(), state, cell_hist_w,
                               c.masks.p, trace);
        const bool stable = c.part == ORB_PART_STABLE_LE;
        hipLaunchKernelGGL(c.weighted ? (stable ? k_m_tail<true, true> : k_m_tail<true, false>)
                                      : (stable ? k_m_tail<false, true> : k_m_tail<false, false>),
                           dim3((unsigned)std::max<int32_t>(nCells, 1)), dim3(kTailBlock), 0, c.stream,
                           c.recs.p, nCells, c.cell_first.p, cell_hist, c.sel.p, lists, c.packed.p, state,
                           cell_hist_w, c.masks.p, c.chunk_pre.p, c.splits.p,
                           reinterpret_cast<SwapPlan *>(c.swap_plan.p), c.ranges.p, heap, exists, le,
                           trace, level_passes, status);
        ORB_HIP(hipGetLastError());
        if (stable) {
            ORB_TRY(launch_stable_scatter(c, nCells, full_cover, true));
            return timing_pair(c, tp, kTimePartition);
        }
        ORB_TRY(launch_hoare_swap(c, nCells, 0));
        ORB_TRY(timing_pair(c, tp, kTimePartition));
        return defer_final ? ORB_OK : launch_hoare_final(c, nCells);
    }
    const unsigned gr = (unsigned)((gq + kReduceRows - 1) / kReduceRows);  // a block per 64-row tile
    const unsigned gw = (unsigned)((nCells + 3) / 4);
    if (c.weighted) {
        // weight-sum rounds over every key, then the partition from the keys
        for (int r = 0; r < kRounds; ++r) {
            const int tb = timing_mark(c);
            if (le)
                hipLaunchKernelGGL(k_bw_hist<1>, dim3(gq), dim3(kBlock), 0, c.stream, c.recs.p,
                                   nCells, c.cell_first.p, c.chunk_desc.p, (uint32_t)c.max_chunks,
                                   c.x(), c.y(), c.z(), c.weights(), chunk_hist_w);
            else
                hipLaunchKernelGGL(k_bw_hist<0>, dim3(gq), dim3(kBlock), 0, c.stream, c.recs.p,
                                   nCells, c.cell_first.p, c.chunk_desc.p, (uint32_t)c.max_chunks,
                                   c.x(), c.y(), c.z(), c.weights(), chunk_hist_w);
            ORB_HIP(hipGetLastError());
            ORB_TRY(timing_pair(c, tb, kTimeCount));
            hipLaunchKernelGGL(k_bw_reduce, dim3(gr), dim3(kBlock), 0, c.stream, c.recs.p, nCells,
                               c.cell_first.p, c.chunk_cell.p, chunk_hist_w, cell_hist_w);
            hipLaunchKernelGGL(k_bw_replay, dim3(gw), dim3(kBlock), 0, c.stream, c.recs.p, nCells,
                               cell_hist_w, heap, trace, level_passes, exists, status);
            ORB_HIP(hipGetLastError());
        }
        const int tp = timing_mark(c);
        if (c.part == ORB_PART_HOARE) {
            ORB_TRY(launch_hoare(c, nCells, status, nullptr, 0, defer_final));
        } else {
            ORB_TRY(invalidate_stamps(c, nCells));  // the stopper counts read the keys
            ORB_TRY(launch_stable_le(c, nCells, status, full_cover, nullptr));
        }
        ORB_TRY(timing_pair(c, tp, kTimePartition));
        return ORB_OK;
    }
    if (kernels.predict) {
        const int tb = timing_mark(c);
        Window *windows = reinterpret_cast<Window *>(c.windows.p);
        uint32_t *window_bins = c.windows.p + predicted_cells(c) * (sizeof(Window) / 4);
        const uint32_t mc = (uint32_t)c.max_chunks;
        const uint32_t ls = kernels.predict, per_block = (uint32_t)kSampleLines / ls;
        hipLaunchKernelGGL(k_p_sample, dim3((gq + per_block - 1) / per_block), dim3(kBlock), 0, c.stream,
                           c.recs.p, nCells, c.cell_first.p, c.chunk_desc.p, mc, c.x(), c.y(), c.z(), ls,
                           c.sample_hist.p);
        hipLaunchKernelGGL(k_p_choose, dim3(gw), dim3(kBlock), 0, c.stream, c.recs.p, nCells,
                           c.sample_hist.p, windows, window_bins);
        hipLaunchKernelGGL(k_p_window, dim3(gq), dim3(kBlock), 0, c.stream, windows, window_bins, nCells,
                           c.cell_first.p, c.chunk_desc.p, mc, c.x(), c.y(), c.z(), later_hist, c.packed.p,
                           c.chunk_comp.p, c.masks.p, rev);
        ORB_HIP(hipGetLastError());
        ORB_TRY(timing_pair(c, tb, kTimeCount));
        hipLaunchKernelGGL(k_b_hist_reduce, dim3(gr), dim3(kBlock), 0, c.stream, c.recs.p, nCells,
                           c.cell_first.p, c.chunk_cell.p, later_hist, cell_hist);
        hipLaunchKernelGGL(k_p_narrow, dim3(gw), dim3(kBlock), 0, c.stream, c.recs.p, nCells, cell_hist,
                           windows, window_bins, c.cell_first.p,
                           reinterpret_cast<unsigned long long *>(c.sel_lists.p), level_passes);
        ORB_HIP(hipGetLastError());
    }
    for (int r = 0; r < 2 && !kernels.predict; ++r) {
        const int tb = timing_mark(c);
        // rounds 1 and 2 over every key of the searching cells; the second
        // also packs the keys inside its margins, per chunk quarter
#define ORB_HIST(L)                                                                              \
    hipLaunchKernelGGL((k_b_hist<L>), dim3(gq), dim3(kBlock), 0, c.stream, c.recs.p, nCells,     \
                       c.cell_first.p, c.chunk_desc.p, (uint32_t)c.max_chunks, c.x(), c.y(), c.z(), \
                       c.cell_cand.p, chunk_hist, chunk_tie, rev)
#define ORB_HIST_WINDOW(L)                                                                       \
    hipLaunchKernelGGL((k_b_hist_window<L>), dim3(gq), dim3(kBlock), 0, c.stream, c.recs.p,      \
                       nCells, c.cell_first.p, c.chunk_desc.p, (uint32_t)c.max_chunks, c.x(), c.y(), \
                       c.z(), c.cell_cand.p, later_hist, c.packed.p, c.chunk_comp.p, c.masks.p, !rev)
        if (le) {
            if (r == 0) ORB_HIST(1);
            else ORB_HIST_WINDOW(1);
        } else {
            if (r == 0) ORB_HIST(0);
            else ORB_HIST_WINDOW(0);
        }
#undef ORB_HIST
#undef ORB_HIST_WINDOW
        ORB_HIP(hipGetLastError());
        ORB_TRY(timing_pair(c, tb, kTimeCount));
        hipLaunchKernelGGL(k_b_hist_reduce, dim3(gr), dim3(kBlock), 0, c.stream, c.recs.p, nCells,
                           c.cell_first.p, c.chunk_cell.p, r == 0 ? chunk_hist : later_hist,
                           cell_hist);
        hipLaunchKernelGGL(k_b_replay, dim3(cell_group_blocks(nCells, cgroup)), dim3(kBlock), 0,
                           c.stream, c.recs.p, nCells, cell_hist, heap, trace, level_passes, exists,
                           status, r == 0 ? c.cell_cand.p : nullptr, c.cell_first.p,
                           r == 1 ? reinterpret_cast<unsigned long long *>(c.sel_lists.p) : nullptr,
                           cgroup);
        ORB_HIP(hipGetLastError());
    }
    {
        // rounds 3 and 4 from the packed keys inside the margins, gathered
        // per cell once
        const int tb = timing_mark(c);
        const unsigned gs = (gq + kBlock / 64 - 1) / (kBlock / 64);
        unsigned long long *lists = reinterpret_cast<unsigned long long *>(c.sel_lists.p);
        const bool pred = kernels.predict != 0;
        const Window *windows = reinterpret_cast<const Window *>(c.windows.p);
        hipLaunchKernelGGL(pred ? k_b_select<true> : k_b_select<false>, dim3(gs), dim3(kBlock), 0, c.stream,
                           c.recs.p, nCells, c.cell_first.p, c.chunk_desc.p, (uint32_t)c.max_chunks,
                           c.packed.p, c.chunk_comp.p, c.sel.p, lists, windows);
        ORB_HIP(hipGetLastError());
        if (nCells <= kFinBlockCells) {  // a block per cell
            auto finish = pred ? (le ? k_b_finish_block<1, true> : k_b_finish_block<0, true>)
                               : (le ? k_b_finish_block<1, false> : k_b_finish_block<0, false>);
            hipLaunchKernelGGL(finish, dim3((unsigned)std::max<int32_t>(nCells, 1)), dim3(kFinBlock), 0,
                               c.stream, c.recs.p, nCells, c.cell_first.p, c.sel.p, lists, heap,
                               trace, level_passes, exists, status, windows);
        } else {
            auto finish = pred ? (le ? k_b_finish<1, true> : k_b_finish<0, true>)
                               : (le ? k_b_finish<1, false> : k_b_finish<0, false>);
            hipLaunchKernelGGL(finish, dim3(cell_group_blocks(nCells, cgroup)), dim3(kBlock), 0,
                               c.stream, c.recs.p, nCells, c.cell_first.p, c.sel.p, lists, heap,
                               trace, level_passes, exists, status, cgroup, windows);
        }
        ORB_HIP(hipGetLastError());
        ORB_TRY(timing_pair(c, tb, kTimeCount));
    }
    const int tp = timing_mark(c);
    HistCounts hc;
    hc.hist = chunk_hist;
    hc.tie = chunk_tie;
    hc.le = le;
    hc.pack = c.packed.p;
    hc.comp = c.chunk_comp.p;
    hc.windows_all = kernels.predict ? 1 : 0;
    if (c.part == ORB_PART_HOARE) ORB_TRY(launch_hoare(c, nCells, status, &hc, 0, defer_final));
    else ORB_TRY(launch_stable_le(c, nCells, status, full_cover, &hc));
    ORB_TRY(timing_pair(c, tp, kTimePartition));
    return ORB_OK;
}

// Adds a build's level; returns whether the build is expected to end there
// (every cell of it finishes in the subtree kernel).
bool LevelShape::add(const Ctx &c, int64_t n, int32_t d, int32_t level, bool complete, bool alone)
{
    int64_t l = 0, h = 0;
    const int32_t m = orb_level_shape(n, d, level, &l, &h);
    if (m <= 0) {  // unknown
        known = false;
        return false;
    }
    // counts within the termination rule's +-2 a split of the exact shares,
    // four a level allowed for
    h += 4 * (int64_t)level;
    l -= 4 * (int64_t)level;
    sub_max = subtree_limit(c, alone ? m : 0);
    fewest = cells ? std::min(fewest, l) : l;
    const int64_t max_leaf = ((int64_t)d + (int64_t(1) << (level - 1)) - 1) >> (level - 1);
    const bool subtree = complete && c.part == ORB_PART_HOARE && !c.weighted && sub_max > 0 &&
                         h <= sub_max && max_leaf <= kSmallLeaves;
    // sizes below the root follow the weights: twice the even share allowed for
    if (c.weighted && level > 1) h *= 2;
    if (!subtree) {
        lo = cells_above ? std::min(lo, l) : l;
        hi = std::max(hi, h);
        cells_above += m;
    }
    cells += m;
    keys += n;
    return subtree;
}

// The kernels of a level of that shape.  k_b_cell takes cells that fit its
// registers in two launches where the chunk path needs sixteen and reads the
// keys once, not twice; a level whose every cell fits it or the subtree kernel
// goes without the chunk kernels.  The lines: a block a cell holds 40960
// keys; a level of few chunks a cell (kMidChunks, kMidLevelChunks) is
// bound by its launches.
LevelKernels level_kernels(const Ctx &c, const LevelShape &s)
{
    LevelKernels k;
    if (!s.known) return k;
    k.sub_max = (uint32_t)s.sub_max;
    if (s.cells_above == 0) {  // subtree cells only
        k.chunks = kChunksNone;
        return k;
    }
    const bool few = s.keys / kChunk + s.cells <= kMidLevelChunks && s.cells < kRecsScan;
    if (!c.weighted && c.part == ORB_PART_HOARE) {
        if (s.lo <= (int64_t)kCellLarge)
            k.cell_max = s.hi <= (int64_t)kCellTiny    ? kCellTiny
                         : s.hi <= (int64_t)kCellSmall ? kCellSmall : kCellLarge;
        if (s.hi <= (int64_t)kCellLarge) {
            k.chunks = kChunksNone;
            return k;
        }
    }
    if (few && s.hi <= (int64_t)kMidChunks * kChunk) k.chunks = kChunksMid;
    return k;
}

// All launches of one batched build, in stream order; no allocation, no
// host synchronisation, no memset: the sequence can be captured.  again: the
// levels once more over a build whose launches left cells alone (LevelMode),
// with every kernel and without the fresh start.
static int enqueue_build(Ctx &c, int32_t levels_mode, bool again)
{
    BatchedState &b = *c.batched;
    uint64_t *trace = c.trace ? b.trace.p : nullptr;
    const int64_t trace_n = c.trace ? c.cap * ORB_MAX_PASSES : 0;
    const orb_cell root = cell_root(c.d);
    if (again) {
        ORB_TRY(launch_zero_u32(c.stream, reinterpret_cast<uint32_t *>(b.level_passes.p), 1));
    } else {
        hipLaunchKernelGGL(k_b_init, dim3(1024), dim3(kBlock), 0, c.stream, b.heap.p, b.exists.p,
                           b.sub.p, (int64_t)c.cap, root, trace, trace_n, b.level_passes.p,
                           c.ranges.p, (uint32_t)c.n, c.status.p);
        ORB_HIP(hipGetLastError());
    }
    const int32_t lmax = levels_mode == ORB_LEVELS_REFERENCE ? b.D - 1 : b.D;
    // the cell sizes each level expects: cells split by count, so they follow
    // from n and d (orb_level_shape, within the termination rule's +-2 a
    // split).  They give the chunk kernels' grids and the level's kernels;
    // where every cell of a level is expected to finish in the subtree
    // kernel, the build ends there.  Weighted builds split by weight: their
    // sizes only choose between the two forms of the chunk path.
    c.level_chunk_hint.assign((size_t)lmax + 2, -1);
    std::vector<LevelKernels> kernels((size_t)lmax + 2);
    std::vector<uint8_t> no_sub((size_t)lmax + 2, 0);  // no cell expected small enough
    int32_t last = lmax;
    if (!again) {
        for (int32_t l = 1; l <= lmax; ++l) {
            LevelShape shape;
            const bool ends = shape.add(c, c.n, c.d, l, b.complete, true);
            if (!shape.known) break;
            if (!c.weighted) c.level_chunk_hint[(size_t)l] = c.n / kChunk + shape.cells + 1;
            kernels[(size_t)l] = level_kernels(c, shape);
            if (!c.weighted) no_sub[(size_t)l] = shape.fewest > shape.sub_max;
            if (!c.weighted && !c.trace && c.part == ORB_PART_HOARE && c.n >= kPredLevelKeys &&
                kernels[(size_t)l].chunks == kChunksAll && shape.fewest >= kPredKeys) {
                // sample lines a chunk: at least 256 lines (16384 keys) a cell
                int32_t ls = 1;
                while (ls < 16 && ls * (shape.fewest / kChunk) < 256) ls *= 2;
                kernels[(size_t)l].predict = ls;
            }
            if (ends) {
                last = l;
                break;
            }
        }
    }
    // a level's last Hoare row swaps run in the next level's first launch;
    // the last level's at the end
    PendingFinal fin;
    for (int32_t l = 1; l <= last; ++l) {
        const int32_t nCells = b.level_n[(size_t)l];
        if (nCells == 0) continue;
        const int tlevel = timing_mark(c);
        // the subtree kernel runs where a cell may be small enough for it:
        // cells split by count, so one with nLeaf leaves holds about
        // n * nLeaf / d keys; where even the smallest expected cell is above
        // the limit (sizes by weight: several times above it), the launch is
        // left out -- only a speed choice, every cell is built either way
        const int64_t few = c.n * (int64_t)b.level_min_leaf[(size_t)l] / (c.d > 0 ? c.d : 1);
        const bool may_sub = !no_sub[(size_t)l] && few <= 4 * (int64_t)subtree_max_keys(c);
        const LevelEntry *entries = b.level_ids.p + b.level_off[(size_t)l];
        LevelKernels k = kernels[(size_t)l];
        k.again = again;
        ORB_TRY(enqueue_level(c, entries, nCells, b.heap.p, b.exists.p, b.sub.p, b.chunk_hist.p,
                              b.cell_hist.p, trace, b.level_passes.p, c.status.p,
                              b.complete && may_sub, b.level_cover[(size_t)l] != 0, l,
                              b.chunk_hist_w.p, b.cell_hist_w.p, &fin, true, k));
        fin.entries = entries;
        fin.nCells = c.part == ORB_PART_HOARE && k.chunks != kChunksNone ? nCells : 0;
        ORB_TRY(timing_pair(c, tlevel, kTimeLevel + l));
    }
    for (int32_t l = last + 1; l <= lmax; ++l)  // nothing left: their time is the marks'
        if (b.level_n[(size_t)l]) ORB_TRY(timing_pair(c, timing_mark(c), kTimeLevel + l));
    if (fin.nCells > 0) ORB_TRY(launch_hoare_final(c, fin.nCells));
    hipLaunchKernelGGL(k_b_done, dim3(1), dim3(64), 0, c.stream, c.status.p, b.level_passes.p,
                       c.hstatus.p, b.hpasses.p);
    ORB_HIP(hipGetLastError());
    return particles_home(c);  // in-stream: the capture ends where it began
}

int build_batched(Ctx &c, int32_t levels_mode, orb_build_info *info)
{
    bool complete = true;
    ORB_TRY(ensure_state(c, levels_mode, &complete));
    BatchedState &b = *c.batched;
    timing_reset(c);
    c.table_ids.clear();
    c.ranges_on_host = false;

    if (!b.hist_clean) {
        ORB_TRY(launch_zero_u32(c.stream, b.cell_hist.p, cell_hist_words(c)));
        b.hist_clean = true;
    }
    if (c.sample_hist.p && !b.sample_clean) {
        ORB_TRY(launch_zero_u32(c.stream, c.sample_hist.p, c.sample_hist.n));
        b.sample_clean = true;
    }
    if (c.weighted && !b.hist_w_clean) {
        ORB_TRY(launch_zero_u64(c.stream, b.cell_hist_w.p, hist_w_rows(c) * kBins));
        b.hist_w_clean = true;
    }
    c.trace_weighted = c.weighted;
    ORB_TRY(particles_home(c));
    const bool graph = c.use_graph && !c.timing;
    if (graph) {
        std::vector<uint64_t> sig = graph_signature(c, b, levels_mode);
        if (!b.exec || sig != b.gsig) {
            drop_graph(b);
            ORB_HIP(hipStreamBeginCapture(c.stream, hipStreamCaptureModeThreadLocal));
            int rc = enqueue_build(c, levels_mode, false);
            hipGraph_t g = nullptr;
            hipError_t e = hipStreamEndCapture(c.stream, &g);
            if (rc < 0) {
                if (g) (void)hipGraphDestroy(g);
                return rc;
            }
            ORB_HIP(e);
            b.graph = g;
            ORB_HIP(hipGraphInstantiate(&b.exec, b.graph, nullptr, nullptr, 0));
            b.gsig = std::move(sig);
        }
        ORB_HIP(hipGraphLaunch(b.exec, c.stream));
    } else {
        ORB_TRY(enqueue_build(c, levels_mode, false));
    }
    c.table_ids.clear();

    // status and pass counts are in the pinned words once the stream is done
    // (k_b_done); the tree stays in HBM until a getter asks for it
    // (batched_pull_results)
    ORB_HIP(hipStreamSynchronize(c.stream));
    if (b.hpasses.p[0] > 0) {
        // cells larger than their level's kernels expected (keys that tie at
        // a cut do not split evenly) were left alone: the rest of the build
        ORB_TRY(enqueue_build(c, levels_mode, true));
        ORB_HIP(hipStreamSynchronize(c.stream));
    }
    c.results_on_device = true;
    ORB_TRY(timing_collect(c));
    const int32_t lmax = levels_mode == ORB_LEVELS_REFERENCE ? b.D - 1 : b.D;
    for (int32_t l = 1; l <= lmax; ++l) {
        info->nlevels = l;
        if (b.level_n[(size_t)l] == 0) continue;
        info->level_passes[l - 1] = b.hpasses.p[l];
        info->total_passes += b.hpasses.p[l];
    }
    if (status_error(c.hstatus.p, &info->error_cell)) {
        b.hist_clean = false;  // an aborted subtree may leave rows behind
        b.hist_w_clean = false;
        b.sample_clean = false;
        return ORB_ERR_UB;
    }
    return ORB_OK;
}

int batched_pull_results(Ctx &c)
{
    if (!c.batched || !c.results_on_device) return ORB_OK;
    BatchedState &b = *c.batched;
    c.heap.resize((size_t)c.cap);
    c.exists.resize((size_t)c.cap);
    const bool small = c.cap <= kHostTreeCells;
    orb_cell *heap = small ? reinterpret_cast<orb_cell *>(c.hranges.p + 2 * c.cap) : c.heap.data();
    uint8_t *exists = small ? reinterpret_cast<uint8_t *>(heap + c.cap) : c.exists.data();
    if (small && !c.ranges_on_host)
        ORB_HIP(hipMemcpyAsync(c.hranges.p, c.ranges.p, 2 * sizeof(uint32_t) * (size_t)c.cap,
                               hipMemcpyDeviceToHost, c.stream));
    ORB_HIP(hipMemcpyAsync(heap, b.heap.p, sizeof(orb_cell) * (size_t)c.cap,
                           hipMemcpyDeviceToHost, c.stream));
    ORB_HIP(hipMemcpyAsync(exists, b.exists.p, (size_t)c.cap, hipMemcpyDeviceToHost, c.stream));
    if (c.trace && b.trace.p) {
        c.trace_counts.resize((size_t)c.cap * ORB_MAX_PASSES);
        ORB_HIP(hipMemcpyAsync(c.trace_counts.data(), b.trace.p,
                               sizeof(uint64_t) * c.trace_counts.size(), hipMemcpyDeviceToHost,
                               c.stream));
    }
    ORB_HIP(hipStreamSynchronize(c.stream));
    if (small) {
        std::memcpy(c.heap.data(), heap, sizeof(orb_cell) * (size_t)c.cap);
        std::memcpy(c.exists.data(), exists, (size_t)c.cap);
        c.ranges_on_host = true;
    }
    c.results_on_device = false;
    return ORB_OK;
}

void batched_drop_graph(Ctx &c)
{
    if (c.batched) drop_graph(*c.batched);
}

void batched_release(Ctx &c)
{
    if (!c.batched) return;
    BatchedState &b = *c.batched;
    drop_graph(b);
    b.level_ids.release();
    b.heap.release();
    b.exists.release();
    b.sub.release();
    b.chunk_hist.release();
    b.cell_hist.release();
    b.chunk_hist_w.release();
    b.cell_hist_w.release();
    b.trace.release();
    b.level_passes.release();
    b.hpasses.release();
    delete c.batched;
    c.batched = nullptr;
}

}  // namespace orb
