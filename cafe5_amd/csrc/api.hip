// api.hip -- host side of libcafe_gpu.so: context, planning and the C ABI of
// include/cafe_gpu.h.
#include <math.h>
#include <stdarg.h>
#include <ctype.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <functional>
#include <map>
#include <mutex>
#include <new>
#include <numeric>
#include <set>
#include <string>
#include <vector>

#include "cafe_gpu.h"
#include "engine.h"

namespace cafe {
hipError_t launch_build(int algo, const double* d_lam, const double* d_t, const double* d_lg, int n,
                        int first_slot, int N, int Np, long long slot_elems, double* mt64, float* mt32,
                        float* lf32, hipStream_t stream, const unsigned char* copies, int top, int* band);
hipError_t launch_fill_zero(void* p, long long bytes, hipStream_t stream);
hipError_t launch_matrix_rows(const double* M, int N, int Np, double* out, hipStream_t stream);
size_t recon_table_doubles(int n_prog, int Lp);
hipError_t launch_block_max(const ReconNode* nodes, int n_prog, const double* mt64, int Np, long long slot_elems,
                            int Lp, double* tab, hipStream_t st);
hipError_t launch_reconstruct(const ReconNode* nodes, int n_prog, const ReconKid* kids, const double* mt64, int N,
                              int Np, long long slot_elems, const double* tab, const int* counts_T, int F,
                              const int2* fams, int nf, const double* prior, int B, int Rr, double* L_all, int Lp,
                              int n_nodes, int* states, int* err, hipStream_t st);
hipError_t launch_fold(const double* mt64, const float* lf32, double* out64, float* out32, const double* err64,
                       const float* err32, int n_dev, int n_rows, int N, int Np, long long slot_elems,
                       int first_slot, int n, hipStream_t stream);
hipError_t f64_dispatch(const MfmaShape& s, int grid, const PruneParams& p, hipStream_t st, int* per_cu);
int f64_level_stride(int nt);
hipError_t launch_f64_levels(int nt, int max_tiles, const int* op_steps, const int* level_ops, int n_levels,
                             const PruneParams& p, hipStream_t st);
hipError_t launch_prune_mfma(const MfmaShape& s, int grid, const PruneParams& p, hipStream_t st);
hipError_t mfma_occupancy(const MfmaShape& s, int* per_cu);
hipError_t f16_dispatch(const MfmaShape& s, int grid, const PruneParams& p, hipStream_t st, int* per_cu);
hipError_t launch_split_f16(const float* mt32, _Float16* hi, _Float16* lo, int Np, long long slot_elems, int n_slots,
                            hipStream_t st);
int lane_rows_for(int rows);
int lane_max_slots(int lane_rows);
hipError_t lane_dispatch(int lr, int ns, int grid, size_t shm, const PruneParams& p, hipStream_t st, int* per_cu);
hipError_t launch_pack(const SegDesc* segs, int n_segs, const BucketDev* buckets, const int* perm,
                       const int* flags, int F, int mask, int* fam_list, TileDesc* out_tiles,
                       const int* class_off, int* class_count, int* fam_count, int tile, hipStream_t st);
hipError_t launch_finalize(int model, int T, int K, int F, const double* val, const int* flag,
                           const double* cat_probs, double* lnl, double* cat, double* post, int* fail,
                           double* total, hipStream_t st);
}  // namespace cafe

using namespace cafe;

// side streams per context: the size classes of one pruning pass (as many as
// the runtime's default hardware queues per process)
constexpr int kSideStreams = 4;

// Fixed device scratch of the entry points that allocate nothing
// (cafe_gpu_reconstruct_noalloc): a reconstruction's program, family list,
// state rows, error flag, block maxima and per-family L rows.  Every device
// the library runs on holds its own copy for the life of the process.  In host
// code `scratch` names a host-side stand-in, never the device memory: its
// device address comes from hipGetSymbolAddress, once per device (see
// fixed_scratch_of), and only that address is handed to kernels and copies.
constexpr size_t kFixedScratchBytes = (size_t)32 << 20;
static __device__ __align__(256) unsigned char scratch[kFixedScratchBytes];

namespace {

thread_local std::string g_last_error;

int fail(int code, const char* fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_last_error = buf;
    return code;
}

#define HIP_OR_FAIL(expr)                                                                          \
    do {                                                                                           \
        hipError_t _e = (expr);                                                                    \
        if (_e != hipSuccess)                                                                      \
            return fail(_e == hipErrorOutOfMemory ? CAFE_GPU_ENOMEM : CAFE_GPU_EDEVICE, "%s: %s", \
                        #expr, hipGetErrorString(_e));                                             \
    } while (0)

int round_up(int x, int m) { return (x + m - 1) / m * m; }
size_t align256(size_t x) { return (x + 255) / 256 * 256; }

// Grow-only device buffer.
struct DevBuf {
    void* p = nullptr;
    size_t bytes = 0;
    hipError_t ensure(size_t need)
    {
        if (need <= bytes) return hipSuccess;
        if (p) (void)hipFree(p);
        p = nullptr;
        bytes = 0;
        hipError_t e = hipMalloc(&p, need);
        if (e == hipSuccess) bytes = need;
        return e;
    }
    void release()
    {
        if (p) (void)hipFree(p);
        p = nullptr;
        bytes = 0;
    }
    template <typename T> T* as() const { return (T*)p; }
};

// Grow-only pinned host memory.
struct PinnedBuf {
    char* p = nullptr;
    size_t bytes = 0;
    hipError_t ensure(size_t need)
    {
        if (need <= bytes) return hipSuccess;
        if (p) (void)hipHostFree(p);
        p = nullptr;
        bytes = 0;
        hipError_t e = hipHostMalloc((void**)&p, need);
        if (e == hipSuccess) bytes = need;
        return e;
    }
    void release()
    {
        if (p) (void)hipHostFree(p);
        p = nullptr;
        bytes = 0;
    }
};

struct BucketHost {
    int B, R, count, fam_begin, max_count;
    bool operator==(const BucketHost& o) const
    {
        return B == o.B && R == o.R && count == o.count && fam_begin == o.fam_begin && max_count == o.max_count;
    }
};

// A table of an evaluation's input block.
struct DevView {
    void* p = nullptr;
    template <typename T> T* as() const { return (T*)p; }
};

// Device buffers of one evaluation (eager calls or a plan).
struct EvalBufs {
    DevBuf fb_tiles, fb_count, val, flag, lnl, cat, post, fail, total, scratch, root, fam_list, cols_x, cols_meta;
    // the inputs: put() together on the host, then one block (commit_inputs)
    DevBuf inputs;
    DevView node_slot, prior64, catp, buckets, tiles, ntiles, segs, class_off, units;
    std::vector<char> block;
    std::vector<std::pair<DevView*, size_t>> views;
    std::vector<BucketDev> bucket_h;   // the bucket table (plan_prune adds the programs and units)
    void put(DevView& v, const void* src, size_t bytes)
    {
        const size_t at = align256(block.size());
        block.resize(at + bytes);
        if (bytes) memcpy(block.data() + at, src, bytes);
        views.push_back({&v, at});
    }
    void release_all()
    {
        DevBuf* all[] = {&fb_tiles, &fb_count, &val, &flag, &lnl, &cat, &post, &fail, &total, &scratch, &root,
                         &fam_list, &cols_x, &cols_meta, &inputs};
        for (DevBuf* b : all) b->release();
    }
};

// A program over pattern columns: its steps and columns in Patterns' buffers.
struct PatternProg {
    int step0 = 0, n_steps = 0, col0 = 0, n_cols = 0, n_pat = 0;
    int n_slots = 0, n_slots_reuse = 0, n_slots_hot = 0;   // of its three step lists
};
struct PatternUnit {
    PatternProg prog;
    int bucket;
    int n;         // patterns
    int xs;        // entries per column
    int list0;     // their representatives' place in `reps`
    int level;     // 1 + the largest level of a unit it reads (0: none)
};
// The subtree patterns of the families under the tree (UnitDev), made by the
// first evaluation that can use them and kept until another tree or other
// families are set.
struct Patterns {
    bool made = false;
    std::vector<PatternUnit> units;     // per bucket contiguous
    std::vector<PatternProg> main;      // per bucket
    std::vector<int> first_unit;        // per bucket (and the end)
    DevBuf ext;                         // count table with the units' pattern rows after the leaves'
    DevBuf steps, steps_reuse, steps_hot;   // programs (outputs in their children's slots; and hot)
    DevBuf cols, reps;
    void clear()
    {
        made = false;
        units.clear();
        main.clear();
        first_unit.clear();
    }
    void release_all()
    {
        for (DevBuf* b : {&ext, &steps, &steps_reuse, &steps_hot, &cols, &reps}) b->release();
    }
};

}  // namespace

struct cafe_gpu_ctx {
    int device = 0;
    int n_cu = 256;
    hipStream_t stream = nullptr;
    // size classes of one pruning phase run concurrently on these (default
    // priority), forked from and joined back to `stream` with join_ev
    std::vector<hipStream_t> side;
    std::vector<hipEvent_t> join_ev;
    hipEvent_t ev[6] = {};
    double timings[4] = {0, 0, 0, 0};
    bool build_timed = false;   // ev[4], ev[5] bracket a build that timings[0] does not hold yet
    PinnedBuf stage_in;         // uploads; stage_ev: the last one has left it
    hipEvent_t stage_ev = nullptr;
    PinnedBuf stage_out;        // downloads
    DevBuf lg;

    // matrix pool
    int N = 0, Np = 0, capacity = 0;
    long long slot_elems = 0;
    DevBuf mt64, mt32, lf32, keys, get_rows;
    DevBuf band32;         // per slot and 16-row tile of mt32: its nonzero k-tiles (band_entry)
    DevBuf mt16h, mt16l;   // split-FP16 halves of mt32 (BATCHED16; made by its evaluations)
    std::vector<char> built;   // per slot: 0 no, 1 every copy, 2 FP64 and the FP32 copies a plan read

    // tree program
    int n_nodes = 0, tree_leaves = 0, n_slots = 0, max_children = 2;
    std::vector<int> parent_h, leaf_col_h;   // the tree as set
    DevBuf d_recon;                          // reconstruction: program, families, prior, states, flags
    DevBuf d_recon_scratch;                  // reconstruction: per-family L rows
    char* fixed_scratch = nullptr;           // this device's copy of `scratch` (device address)
    std::vector<OpDev> ops;
    DevBuf d_steps;
    int n_steps = 0;
    DevBuf d_steps_lane;     // the same steps with output-reusing slots (split-FP16 kernel)
    int n_slots_lane = 0;
    DevBuf d_steps_hot;      // and with the vector the next op reads kept in registers (per-lane kernel)
    int n_slots_hot = 0;
    // and sorted by level (children's ops first), interior steps naming their
    // child's op: the recompute of short lists
    DevBuf d_steps_level, d_op_steps;
    std::vector<int> level_ops;   // first op of every level, and the end

    // families
    int F = 0, n_leaves = 0;
    std::vector<int> perm;
    std::vector<int> fam_max;   // per family of the caller: its largest count
    std::vector<BucketHost> buckets;
    DevBuf d_counts, d_perm;
    std::vector<int> counts_T;   // as uploaded: [leaf][F], bucket-sorted
    Patterns pat;

    // error model, and the pools with it folded into every matrix (leaf
    // branches read those)
    int n_dev = 0, err_rows = 0;
    DevBuf d_err64, d_err32, mt64e, mt32e;

    // buffers of eager evaluations (plans own their own)
    EvalBufs eager;
    long long pool_gen = 0;   // bumped by matrix_reset; plans check it
    // measured launch shapes: (path, tiles per vector, leaves) -> shape
    struct TuneEntry {
        int path, nt, leaves, kernel, ntw, w, lds, grid_mult;
        // the plan's size classes it was measured in (bit nt - 1 per class of
        // nt tiles); 0: any plan
        unsigned long long plan_classes;
    };
    std::vector<TuneEntry> tuning;
    // bumped by set_tree, set_families and by set_error_model when it adds or
    // removes the model or changes its shape (buffers a plan's graph points
    // into); plans check it.  Same-shape error-model rows are updated in place.
    long long input_gen = 0;
};

namespace {

int check_ctx(cafe_gpu_ctx* ctx)
{
    if (!ctx) return fail(CAFE_GPU_EINVAL, "null context");
    if (hipSetDevice(ctx->device) != hipSuccess) return fail(CAFE_GPU_EDEVICE, "hipSetDevice failed");
    return CAFE_GPU_OK;
}

// Host transfers go through pinned memory on the context's stream: a copy from
// or to pageable memory is staged by the runtime in small pieces, waits for the
// device each time (10 us and more per table; 85 us per MB), and is not ordered
// with the stream.

// Enqueues a copy of `bytes` at src to the device; src is free on return.
int upload(cafe_gpu_ctx* ctx, void* dst, const void* src, size_t bytes)
{
    if (!bytes) return CAFE_GPU_OK;
    HIP_OR_FAIL(hipEventSynchronize(ctx->stage_ev));   // (an event never recorded is complete)
    HIP_OR_FAIL(ctx->stage_in.ensure(std::max<size_t>(bytes, 64 * 1024)));
    memcpy(ctx->stage_in.p, src, bytes);
    HIP_OR_FAIL(hipMemcpyAsync(dst, ctx->stage_in.p, bytes, hipMemcpyHostToDevice, ctx->stream));
    HIP_OR_FAIL(hipEventRecord(ctx->stage_ev, ctx->stream));
    return CAFE_GPU_OK;
}

// The evaluation's input tables as one block.
int commit_inputs(cafe_gpu_ctx* ctx, EvalBufs& b)
{
    HIP_OR_FAIL(b.inputs.ensure(std::max<size_t>(b.block.size(), 256)));
    if (int rc = upload(ctx, b.inputs.p, b.block.data(), b.block.size())) return rc;
    for (auto& v : b.views) v.first->p = (char*)b.inputs.p + v.second;
    return CAFE_GPU_OK;
}

// Device to host, after the stream's work so far; returns with the data.  Copies
// from kDirectCopy on go to their place at once (the runtime pins it; through
// here 3 MB of root vectors took 640 us, this way 360), smaller ones through
// the staging buffer (200 KB: 775 us a step against 865).
struct Fetch {
    void* dst;
    const void* src;
    size_t bytes;
};
constexpr size_t kDirectCopy = (size_t)256 << 10;
constexpr size_t kStageOut = 2 * kDirectCopy;   // (what does not fit goes to its place too)

int fetch(cafe_gpu_ctx* ctx, const std::vector<Fetch>& list)
{
    size_t used = 0;
    for (const Fetch& f : list) {
        const bool staged = f.bytes < kDirectCopy && used + f.bytes <= kStageOut;
        HIP_OR_FAIL(hipMemcpyAsync(staged ? ctx->stage_out.p + used : f.dst, f.src, f.bytes, hipMemcpyDeviceToHost,
                                   ctx->stream));
        if (staged) used += align256(f.bytes);
    }
    HIP_OR_FAIL(hipStreamSynchronize(ctx->stream));
    used = 0;
    for (const Fetch& f : list) {
        if (!(f.bytes < kDirectCopy && used + f.bytes <= kStageOut)) continue;
        memcpy(f.dst, ctx->stage_out.p + used, f.bytes);
        used += align256(f.bytes);
    }
    return CAFE_GPU_OK;
}

// Device address of this device's `scratch` array, resolved once per device
// with that device current (cafe_gpu_create makes it current first).
int fixed_scratch_of(int device, char** out)
{
    static std::mutex mu;
    static std::map<int, char*> addr;
    std::lock_guard<std::mutex> lock(mu);
    auto it = addr.find(device);
    if (it == addr.end()) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(CAFE_GPU_EDEVICE, "hipGetSymbolAddress(scratch) failed on device %d: %s", device,
                        hipGetErrorString(e));
        it = addr.emplace(device, (char*)p).first;
    }
    *out = it->second;
    return CAFE_GPU_OK;
}

// Pools with the error model folded in: sized with the matrix pool (outside
// any graph capture).
int ensure_fold_pools(cafe_gpu_ctx* ctx)
{
    if (!ctx->n_dev || !ctx->capacity) return CAFE_GPU_OK;
    HIP_OR_FAIL(ctx->mt64e.ensure(sizeof(double) * ctx->slot_elems * ctx->capacity));
    HIP_OR_FAIL(ctx->mt32e.ensure(sizeof(float) * ctx->slot_elems * ctx->capacity));
    return CAFE_GPU_OK;
}

// Enqueues the error-model fold of slots first .. first+n-1 (nothing without
// an error model) into the FP64 pool (fp64) and the FP32 one (fp32).
int enqueue_fold(cafe_gpu_ctx* ctx, int first, int n, hipStream_t st, bool fp64 = true, bool fp32 = true)
{
    if (!ctx->n_dev || n <= 0) return CAFE_GPU_OK;
    HIP_OR_FAIL(launch_fold(ctx->mt64.as<double>(), ctx->lf32.as<float>(), fp64 ? ctx->mt64e.as<double>() : nullptr,
                            fp32 ? ctx->mt32e.as<float>() : nullptr, ctx->d_err64.as<double>(),
                            ctx->d_err32.as<float>(), ctx->n_dev, ctx->err_rows, ctx->N, ctx->Np, ctx->slot_elems,
                            first, n, st));
    return CAFE_GPU_OK;
}

// Sethi-Ullman order: evaluate the interior child that needs the most live
// partial vectors first, so at most ~log2(n) + 2 vectors are live at once.
struct Planner {
    const std::vector<std::vector<int>>& kids;
    const std::vector<int>& leaf_col;
    std::vector<int> need, slot_of;
    std::vector<char> used;
    std::vector<OpDev> ops;
    std::vector<ChildDev> out_kids;
    int max_slot = -1;
    // reuse: a node's output may take one of its children's slots (a kernel
    // whose lanes read every child before writing the output, in order)
    bool reuse = false;
    // hot (with reuse): the last interior child a node's op reads is the op
    // just before it, so its vector is read from the kernel's hot registers
    // (in_slot kHotSlot) and takes no slot; so is every output that the next
    // op reads (out_slot kHotSlot), and the root's
    bool hot = false;

    Planner(const std::vector<std::vector<int>>& k, const std::vector<int>& lc, bool r = false, bool h = false)
        : kids(k), leaf_col(lc), need(k.size(), -1), slot_of(k.size(), -1), reuse(r || h), hot(h) {}

    std::vector<int> interior_order(int u)
    {
        std::vector<int> in;
        for (int c : kids[u])
            if (leaf_col[c] < 0) in.push_back(c);
        std::stable_sort(in.begin(), in.end(), [&](int a, int b) { return need[a] > need[b]; });
        return in;
    }

    int compute_need(int u)
    {
        if (leaf_col[u] >= 0) return need[u] = 0;
        for (int c : kids[u]) compute_need(c);
        auto in = interior_order(u);
        int n = (int)in.size() + 1;   // children held + a fresh output slot
        for (size_t i = 0; i < in.size(); ++i) n = std::max(n, (int)i + need[in[i]]);
        return need[u] = n;
    }

    int alloc()
    {
        for (size_t i = 0; i < used.size(); ++i)
            if (!used[i]) {
                used[i] = 1;
                max_slot = std::max(max_slot, (int)i);
                return (int)i;
            }
        used.push_back(1);
        max_slot = std::max(max_slot, (int)used.size() - 1);
        return (int)used.size() - 1;
    }

    void emit(int u, bool store = true)
    {
        auto in = interior_order(u);
        for (size_t i = 0; i < in.size(); ++i) emit(in[i], !hot || i + 1 < in.size());
        if (reuse)
            for (int c : in)
                if (slot_of[c] != kHotSlot) used[slot_of[c]] = 0;
        const int out = hot && !store ? kHotSlot : alloc();
        OpDev op;
        op.node = u;
        op.out_slot = out;
        op.n_child = (int)kids[u].size();
        op.child_begin = (int)out_kids.size();
        for (int c : kids[u]) {   // product in descendant order
            ChildDev ch;
            ch.node = c;
            ch.leaf_col = leaf_col[c];
            ch.in_slot = leaf_col[c] >= 0 ? -1 : slot_of[c];
            ch.pad = 0;
            out_kids.push_back(ch);
        }
        ops.push_back(op);
        if (!reuse)
            for (int c : in) used[slot_of[c]] = 0;
        slot_of[u] = out;
    }
};

// Children of every node, in increasing index, and the root.
std::vector<std::vector<int>> children_of(const std::vector<int>& parent, int& root)
{
    std::vector<std::vector<int>> kids(parent.size());
    root = -1;
    for (int i = 0; i < (int)parent.size(); ++i) {
        if (parent[i] < 0) root = i;
        else kids[parent[i]].push_back(i);
    }
    return kids;
}

// A flat list of child steps from a planner's ops.
std::vector<StepDev> flatten_steps(const std::vector<OpDev>& ops, const std::vector<ChildDev>& kids)
{
    std::vector<StepDev> steps;
    for (size_t o = 0; o < ops.size(); ++o) {
        const OpDev& op = ops[o];
        for (int k = 0; k < op.n_child; ++k) {
            const ChildDev& ch = kids[op.child_begin + k];
            int ctl = op.out_slot;
            if (k == 0) ctl |= kStepFirst;
            if (k == op.n_child - 1) ctl |= kStepLast;
            if (o + 1 == ops.size()) ctl |= kStepRoot;
            steps.push_back(StepDev{ch.node, ch.leaf_col, ch.in_slot, ctl});
        }
    }
    return steps;
}

// Buckets of fewer families are not searched for patterns: at one point a few
// tiles wait for one chain of steps, which more launches only lengthen.  (Grids
// of many points would gain little by a lower limit, families of one small bucket
// having few patterns in common: 483 families at each of 64 points kept 74 to
// 100% of their contractions at a limit of 16.)
constexpr int kPatternFamilies = 512;
// A node is a candidate while its patterns are at most half of the families:
// one step of 50,000 gamma families 1.49 ms, against 1.52 at a quarter and 1.62
// at an eighth (16,000 at B = 500: 19.4, 20.5, 21.8); past a half the columns
// written and read cost what the shared work saves.
constexpr int kPatternShare = 2;
// A unit's descendant becomes a unit of its own where that divides its work by
// three or more; otherwise it is computed along, one launch less (1.51, 1.52
// and 1.70 ms dividing by 2, by 6 and never; 5,000 families 0.75, 0.78, 0.76).
constexpr int kPatternNest = 3;

// 16-row tiles of a bucket's vectors and root rows (sizes 0..R).
int tiles_of(const BucketHost& bk)
{
    return std::max(round_up(bk.B + 1, kTile), round_up(bk.R + 1, kTile)) / kTile;
}

// Entries of a pattern column of a bucket: whole row tiles, and the rows the
// per-lane kernel writes and gathers.  That kernel's instance covers every
// bucket of the size class (33 rows for bounds 20 and 28 side by side, where
// the first alone takes 21), so the class's largest vector decides.
int column_entries(const std::vector<BucketHost>& buckets, int bi)
{
    const BucketHost& bk = buckets[bi];
    int rows = 0;   // of the class
    for (const BucketHost& o : buckets)
        if (tiles_of(o) == tiles_of(bk)) rows = std::max(rows, std::max(o.B, o.R) + 1);
    return round_up(std::max({bk.B + 1, bk.R + 1, lane_rows_for(rows)}), kTile);
}

// Pattern ids of the pairs (a[f], b[f]), a < na and b < nb, numbered in order
// of appearance; 0 where there are more than `limit`.
int pair_patterns(const std::vector<int>& a, int na, const std::vector<int>& b, int nb, int limit, std::vector<int>& id,
                  std::vector<int>& table)
{
    const int F = (int)a.size();
    id.resize(F);
    const long long space = (long long)na * nb;
    int n = 0;
    if (space <= 1 << 20) {
        table.assign(space, -1);
        for (int f = 0; f < F; ++f) {
            int& t = table[(size_t)a[f] * nb + b[f]];
            if (t < 0) {
                if (n == limit) return 0;
                t = n++;
            }
            id[f] = t;
        }
        return n;
    }
    // open addressing: slots of (key, id)
    size_t size = 1024;
    while (size < 4 * (size_t)limit) size <<= 1;
    std::vector<std::pair<long long, int>> slots(size, {-1, 0});
    for (int f = 0; f < F; ++f) {
        const long long key = (long long)a[f] * nb + b[f];
        size_t h = (size_t)((unsigned long long)key * 0x9E3779B97F4A7C15ull >> 20) & (size - 1);
        while (slots[h].first >= 0 && slots[h].first != key) h = (h + 1) & (size - 1);
        if (slots[h].first < 0) {
            if (n == limit) return 0;
            slots[h] = {key, n++};
        }
        id[f] = slots[h].second;
    }
    return n;
}

// Finds the units of every bucket, their programs and those of the buckets,
// and uploads them.  A pass over every node's ids on the host: 0.8 ms for 10,000
// families of 34 taxa, 3.9 for 50,000, 87 for 200,000 of 100 taxa (several times
// that on a slower host) -- what two evaluations and more gain by it -- so it is
// left to the first evaluation that can share (root vectors and reconstructions
// do not), and its result is kept while the same tree and counts are set again,
// as a model that sets both for every score does.
int find_patterns(cafe_gpu_ctx* ctx)
{
    Patterns& P = ctx->pat;
    const int F = ctx->F, nl = ctx->n_leaves, n = ctx->n_nodes;
    const auto& leaf = ctx->leaf_col_h;
    int root;
    const auto kids = children_of(ctx->parent_h, root);
    std::vector<int> order;   // children first
    {
        std::vector<std::pair<int, int>> stack{{root, 0}};
        while (!stack.empty()) {
            auto& top = stack.back();
            const int u = top.first;
            if (top.second < (int)kids[u].size()) {
                stack.push_back({kids[u][top.second++], 0});
                continue;
            }
            stack.pop_back();
            if (leaf[u] < 0) order.push_back(u);
        }
    }
    std::vector<int> row(n, -1);   // a unit node's row of the extended count table
    int n_rows = nl;
    std::vector<int> rows;   // [n_rows - nl][F]
    std::vector<StepDev> steps[3];   // in order, with reuse, hot
    std::vector<ColDev> cols;
    std::vector<int> reps, table;
    P.main.resize(ctx->buckets.size());
    for (int bi = 0; bi < (int)ctx->buckets.size(); ++bi) {
        const BucketHost& bk = ctx->buckets[bi];
        const int xs = column_entries(ctx->buckets, bi);
        P.first_unit.push_back((int)P.units.size());
        std::vector<std::vector<int>> ids(n);
        std::vector<int> count(n, 0);   // patterns of a node (0: not a candidate)
        if (bk.count >= kPatternFamilies) {
            const int limit = bk.count / kPatternShare;
            for (int u = 0; u < n; ++u)
                if (leaf[u] >= 0) {
                    const int* c = ctx->counts_T.data() + (size_t)leaf[u] * F + bk.fam_begin;
                    ids[u].assign(c, c + bk.count);
                    count[u] = bk.max_count + 1;
                }
            for (int u : order) {
                if (u == root) continue;
                bool all = true;
                for (int c : kids[u]) all = all && count[c] > 0;
                if (!all) continue;
                std::vector<int> cur = ids[kids[u][0]], next;
                int m = count[kids[u][0]];
                for (size_t k = 1; k < kids[u].size() && m > 0; ++k) {
                    m = pair_patterns(cur, m, ids[kids[u][k]], count[kids[u][k]], limit, next, table);
                    cur.swap(next);
                }
                if (kids[u].size() == 1 && leaf[kids[u][0]] >= 0) {   // (a leaf's counts are not numbered by appearance)
                    const std::vector<int> one(bk.count, 0);
                    m = pair_patterns(cur, m, one, 1, limit, next, table);
                    cur.swap(next);
                }
                if (m == 0 || (long long)m * xs >= 1 << 28) continue;
                ids[u].swap(cur);
                count[u] = m;
            }
        }
        // units, top down: candidates under a node that is none, and those
        // under a unit that divide its patterns
        std::vector<char> unit(n, 0);
        std::vector<int> inside(n, 0);   // patterns of the unit that computes a node (0: none)
        for (auto it = order.rbegin(); it != order.rend(); ++it)
            for (int c : kids[*it]) {
                if (leaf[c] >= 0 || count[c] == 0) continue;
                unit[c] = inside[*it] == 0 || (long long)count[c] * kPatternNest <= inside[*it];
                inside[c] = unit[c] ? count[c] : inside[*it];
            }
        std::vector<int> unit_of(n, -1), level(n, 0), code(n, -1);
        auto program = [&](int top, bool is_unit) {
            // the tree below top, its leaves and units in columns
            std::vector<int> walk{top}, pats, leaves;
            int lev = 0;
            while (!walk.empty()) {
                const int u = walk.back();
                walk.pop_back();
                for (int c : kids[u]) {
                    if (leaf[c] >= 0) {
                        leaves.push_back(c);
                    } else if (unit[c]) {
                        pats.push_back(c);
                        lev = std::max(lev, level[c] + 1);
                    } else {
                        walk.push_back(c);
                    }
                }
            }
            PatternProg pr;
            pr.col0 = (int)cols.size();
            pr.n_pat = (int)pats.size();
            for (int c : pats) {
                code[c] = (int)cols.size() - pr.col0;
                cols.push_back(ColDev{row[c], xs});
            }
            for (int c : leaves) {
                code[c] = (int)cols.size() - pr.col0;
                cols.push_back(ColDev{leaf[c], 0});
            }
            pr.n_cols = (int)cols.size() - pr.col0;
            pr.step0 = (int)steps[0].size();
            int* n_slots[3] = {&pr.n_slots, &pr.n_slots_reuse, &pr.n_slots_hot};
            for (int v = 0; v < 3; ++v) {
                Planner pl(kids, code, v > 0, v == 2);
                pl.compute_need(top);
                pl.emit(top, v < 2);
                *n_slots[v] = std::max(1, pl.max_slot + 1);
                std::vector<StepDev> st = flatten_steps(pl.ops, pl.out_kids);
                for (StepDev& s : st) {
                    if (is_unit) s.ctl &= ~kStepRoot;
                    if (s.leaf_col >= 0 && s.leaf_col < pr.n_pat) {
                        s.ctl |= kStepPattern;
                        s.in_slot = unit_of[s.node];
                    }
                }
                if (is_unit)   // the branch's contraction, written as columns
                    st.push_back(StepDev{top, -1, pl.slot_of[top],
                                         kStepFirst | kStepLast | kStepOut |
                                             (ctx->parent_h[top] == root ? kStepRoot : 0)});
                pr.n_steps = (int)st.size();
                steps[v].insert(steps[v].end(), st.begin(), st.end());
            }
            for (int c : pats) code[c] = -1;
            for (int c : leaves) code[c] = -1;
            if (is_unit) level[top] = lev;
            return pr;
        };
        for (int u : order) {
            if (!unit[u]) continue;
            if (row[u] < 0) {
                row[u] = n_rows++;
                rows.resize((size_t)(n_rows - nl) * F, 0);
            }
            std::copy(ids[u].begin(), ids[u].end(), rows.begin() + (size_t)(row[u] - nl) * F + bk.fam_begin);
            PatternUnit un;
            unit_of[u] = (int)P.units.size();
            un.prog = program(u, true);
            un.bucket = bi;
            un.n = count[u];
            un.xs = xs;
            un.list0 = (int)reps.size();
            un.level = level[u];
            reps.resize(reps.size() + un.n, -1);
            for (int f = 0; f < bk.count; ++f) {
                int& r = reps[un.list0 + ids[u][f]];
                if (r < 0) r = bk.fam_begin + f;
            }
            P.units.push_back(un);
        }
        P.main[bi] = program(root, false);
    }
    P.first_unit.push_back((int)P.units.size());
    if (!P.units.empty()) {
        HIP_OR_FAIL(P.ext.ensure(sizeof(int) * (size_t)n_rows * F));
        HIP_OR_FAIL(hipMemcpy(P.ext.p, ctx->d_counts.p, sizeof(int) * (size_t)nl * F, hipMemcpyDeviceToDevice));
        HIP_OR_FAIL(hipMemcpy(P.ext.as<int>() + (size_t)nl * F, rows.data(), sizeof(int) * rows.size(), hipMemcpyHostToDevice));
        auto put = [&](DevBuf& b, const void* v, size_t bytes) -> int {
            HIP_OR_FAIL(b.ensure(bytes));
            HIP_OR_FAIL(hipMemcpy(b.p, v, bytes, hipMemcpyHostToDevice));
            return CAFE_GPU_OK;
        };
        if (int rc = put(P.steps, steps[0].data(), sizeof(StepDev) * steps[0].size())) return rc;
        if (int rc = put(P.steps_reuse, steps[1].data(), sizeof(StepDev) * steps[1].size())) return rc;
        if (int rc = put(P.steps_hot, steps[2].data(), sizeof(StepDev) * steps[2].size())) return rc;
        if (int rc = put(P.cols, cols.data(), sizeof(ColDev) * cols.size())) return rc;
        if (int rc = put(P.reps, reps.data(), sizeof(int) * reps.size())) return rc;
    }
    return CAFE_GPU_OK;
}

// The same for a caller that needs none: without memory for them every bucket
// keeps its whole program.
void make_patterns(cafe_gpu_ctx* ctx)
{
    Patterns& P = ctx->pat;
    if (P.made) return;
    P.clear();
    int rc;
    try {
        rc = find_patterns(ctx);
    } catch (const std::bad_alloc&) {
        rc = CAFE_GPU_ENOMEM;
    }
    if (rc != CAFE_GPU_OK) {
        (void)hipGetLastError();
        P.clear();
        P.release_all();
    }
    P.made = true;
}

}  // namespace

// ===========================================================================
// C ABI
// ===========================================================================
extern "C" {

const char* cafe_gpu_last_error(void) { return g_last_error.c_str(); }

int cafe_gpu_create(int device, cafe_gpu_ctx** out)
{
    if (!out) return fail(CAFE_GPU_EINVAL, "null output pointer");
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0)
        return fail(CAFE_GPU_EDEVICE, "no HIP device available");
    if (device < 0 || device >= n) return fail(CAFE_GPU_EINVAL, "device %d out of range", device);
    HIP_OR_FAIL(hipSetDevice(device));
    auto* ctx = new cafe_gpu_ctx();
    ctx->device = device;
    int cu = 0;
    if (hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && cu > 0)
        ctx->n_cu = cu;
    if (hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking) != hipSuccess) {
        delete ctx;
        return fail(CAFE_GPU_EDEVICE, "hipStreamCreate failed");
    }
    for (auto& e : ctx->ev) (void)hipEventCreate(&e);
    (void)hipEventCreateWithFlags(&ctx->stage_ev, hipEventDisableTiming);
    ctx->side.assign(kSideStreams, nullptr);
    for (auto& st : ctx->side)
        if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess) {
            cafe_gpu_destroy(ctx);
            return fail(CAFE_GPU_EDEVICE, "hipStreamCreate failed");
        }
    if (int rc = fixed_scratch_of(device, &ctx->fixed_scratch)) {
        const std::string msg = cafe_gpu_last_error();
        cafe_gpu_destroy(ctx);
        return fail(rc, "%s", msg.c_str());
    }
    ctx->join_ev.assign(2 * (kSideStreams + 1), nullptr);
    for (auto& e : ctx->join_ev) (void)hipEventCreateWithFlags(&e, hipEventDisableTiming);
    // log-gamma of integers from the host libm: the reference's
    // lgamma cache (probability.cpp:69-75)
    std::vector<double> lg(kLgammaN);
    for (int i = 0; i < kLgammaN; ++i) lg[i] = lgamma((double)i);
    if (ctx->lg.ensure(sizeof(double) * kLgammaN) != hipSuccess ||
        hipMemcpy(ctx->lg.p, lg.data(), sizeof(double) * kLgammaN, hipMemcpyHostToDevice) != hipSuccess) {
        cafe_gpu_destroy(ctx);
        return fail(CAFE_GPU_ENOMEM, "log-gamma table upload failed");
    }
    // (here, so that the calls that allocate nothing find it)
    if (ctx->stage_out.ensure(kStageOut) != hipSuccess) {
        cafe_gpu_destroy(ctx);
        return fail(CAFE_GPU_ENOMEM, "pinned staging buffer");
    }
    *out = ctx;
    return CAFE_GPU_OK;
}

int cafe_gpu_destroy(cafe_gpu_ctx* ctx)
{
    if (!ctx) return CAFE_GPU_OK;
    (void)hipSetDevice(ctx->device);
    if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
    DevBuf* bufs[] = {&ctx->lg, &ctx->mt64, &ctx->mt32, &ctx->lf32, &ctx->keys, &ctx->get_rows,
                      &ctx->d_steps, &ctx->d_steps_lane, &ctx->d_steps_hot, &ctx->d_steps_level, &ctx->d_op_steps, &ctx->d_counts, &ctx->d_perm, &ctx->d_err64,
                      &ctx->d_err32, &ctx->mt64e, &ctx->mt32e, &ctx->mt16h, &ctx->mt16l, &ctx->band32, &ctx->d_recon,
                      &ctx->d_recon_scratch};
    for (DevBuf* b : bufs) b->release();
    ctx->eager.release_all();
    ctx->pat.release_all();
    for (auto& e : ctx->ev)
        if (e) (void)hipEventDestroy(e);
    for (auto& e : ctx->join_ev)
        if (e) (void)hipEventDestroy(e);
    if (ctx->stage_ev) (void)hipEventDestroy(ctx->stage_ev);
    ctx->stage_in.release();
    ctx->stage_out.release();
    for (auto& st : ctx->side)
        if (st) {
            (void)hipStreamSynchronize(st);
            (void)hipStreamDestroy(st);
        }
    if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
    delete ctx;
    return CAFE_GPU_OK;
}

int cafe_gpu_matrix_reset(cafe_gpu_ctx* ctx, int N, int capacity)
{
    if (int rc = check_ctx(ctx)) return rc;
    if (N < 2 || N * 2 + 2 > kLgammaN) return fail(CAFE_GPU_EINVAL, "matrix size %d out of range", N);
    if (capacity < 1) return fail(CAFE_GPU_EINVAL, "capacity must be positive");
    const int Np = round_up(N + kTile, 32);   // >= round_up(N, 16) + 16, whole 32-wide transpose tiles
    const long long slot_elems = (long long)Np * Np;
    const size_t n64 = sizeof(double) * slot_elems * capacity;
    const size_t n32 = sizeof(float) * slot_elems * capacity;
    // every plan made over the old pool is stale from here on, and until the
    // new pool is complete the context has none
    HIP_OR_FAIL(hipStreamSynchronize(ctx->stream));
    ctx->pool_gen++;
    ctx->N = ctx->Np = ctx->capacity = 0;
    ctx->slot_elems = 0;
    ctx->built.clear();
    HIP_OR_FAIL(ctx->mt64.ensure(n64));
    HIP_OR_FAIL(ctx->mt32.ensure(n32));
    HIP_OR_FAIL(ctx->lf32.ensure(n32));
    const size_t nband = sizeof(int) * (size_t)(Np / kTile) * capacity;
    HIP_OR_FAIL(ctx->band32.ensure(nband));
    if (ctx->n_dev) {
        HIP_OR_FAIL(ctx->mt64e.ensure(n64));
        HIP_OR_FAIL(ctx->mt32e.ensure(n32));
    }
    // padding rows/columns must read as zero
    HIP_OR_FAIL(launch_fill_zero(ctx->mt64.p, (long long)n64, ctx->stream));
    HIP_OR_FAIL(launch_fill_zero(ctx->mt32.p, (long long)n32, ctx->stream));
    HIP_OR_FAIL(launch_fill_zero(ctx->lf32.p, (long long)n32, ctx->stream));
    HIP_OR_FAIL(launch_fill_zero(ctx->band32.p, (long long)nband, ctx->stream));
    ctx->N = N;
    ctx->Np = Np;
    ctx->slot_elems = slot_elems;
    ctx->capacity = capacity;
    if (int rc = enqueue_fold(ctx, 0, capacity, ctx->stream)) return rc;
    HIP_OR_FAIL(hipStreamSynchronize(ctx->stream));
    ctx->built.assign(capacity, 0);
    return CAFE_GPU_OK;
}

int cafe_gpu_matrix_build(cafe_gpu_ctx* ctx, int n, const double* lambda_q, const double* t_q,
                          int first_slot, int algo)
{
    if (int rc = check_ctx(ctx)) return rc;
    if (ctx->N == 0) return fail(CAFE_GPU_ESTATE, "matrix_reset has not been called");
    if (n < 0 || first_slot < 0 || first_slot + n > ctx->capacity)
        return fail(CAFE_GPU_EINVAL, "slots %d..%d exceed capacity %d", first_slot, first_slot + n,
                    ctx->capacity);
    if (algo != CAFE_GPU_BUILD_CLOSED_FORM && algo != CAFE_GPU_BUILD_RECURRENCE)
        return fail(CAFE_GPU_EINVAL, "unknown build algorithm %d", algo);
    if (n == 0) return CAFE_GPU_OK;
    if (!lambda_q || !t_q) return fail(CAFE_GPU_EINVAL, "null key arrays");
    for (int i = 0; i < n; ++i)
        if (!(lambda_q[i] >= 0) || !(t_q[i] >= 0) || !std::isfinite(lambda_q[i]) || !std::isfinite(t_q[i]))
            return fail(CAFE_GPU_EINVAL, "key %d has an invalid lambda or branch length", i);
    HIP_OR_FAIL(ctx->keys.ensure(sizeof(double) * 2 * n));
    double* d_lam = ctx->keys.as<double>();
    double* d_t = d_lam + n;
    std::vector<double> both(lambda_q, lambda_q + n);
    both.insert(both.end(), t_q, t_q + n);
    if (int rc = upload(ctx, d_lam, both.data(), sizeof(double) * 2 * n)) return rc;
    HIP_OR_FAIL(hipEventRecord(ctx->ev[4], ctx->stream));
    HIP_OR_FAIL(launch_build(algo, d_lam, d_t, ctx->lg.as<double>(), n,
                             first_slot, ctx->N, ctx->Np, ctx->slot_elems, ctx->mt64.as<double>(),
                             ctx->mt32.as<float>(), ctx->lf32.as<float>(), ctx->stream, nullptr, 0,
                             ctx->band32.as<int>()));
    if (int rc = enqueue_fold(ctx, first_slot, n, ctx->stream)) return rc;
    HIP_OR_FAIL(hipEventRecord(ctx->ev[5], ctx->stream));
    ctx->build_timed = true;   // (everything that reads the matrices runs on the stream)
    for (int i = 0; i < n; ++i) ctx->built[first_slot + i] = 1;
    return CAFE_GPU_OK;
}

int cafe_gpu_matrix_get(cafe_gpu_ctx* ctx, int slot, double* out)
{
    if (int rc = check_ctx(ctx)) return rc;
    if (!out) return fail(CAFE_GPU_EINVAL, "null output");
    if (slot < 0 || slot >= ctx->capacity || !ctx->built[slot])
        return fail(CAFE_GPU_ENOTFOUND, "matrix slot %d is not built", slot);
    // up to 512 KB turned on the host (twelve calls at 166 sizes 830 us, 970 through
    // the kernel and the larger copy); at 401 sizes the kernel: 1,150 against 1,980
    const size_t slot_bytes = sizeof(double) * (size_t)ctx->N * ctx->Np;
    if (slot_bytes <= kStageOut) {
        HIP_OR_FAIL(hipMemcpyAsync(ctx->stage_out.p, ctx->mt64.as<double>() + (long long)slot * ctx->slot_elems, slot_bytes,
                                   hipMemcpyDeviceToHost, ctx->stream));
        HIP_OR_FAIL(hipStreamSynchronize(ctx->stream));
        const double* cm = (const double*)ctx->stage_out.p;
        for (int s = 0; s < ctx->N; ++s)
            for (int c = 0; c < ctx->N; ++c) out[(size_t)s * ctx->N + c] = cm[(size_t)c * ctx->Np + s];
        return CAFE_GPU_OK;
    }
    const size_t bytes = sizeof(double) * (size_t)ctx->N * ctx->N;
    HIP_OR_FAIL(ctx->get_rows.ensure(bytes));
    HIP_OR_FAIL(launch_matrix_rows(ctx->mt64.as<double>() + (long long)slot * ctx->slot_elems, ctx->N, ctx->Np,
                                   ctx->get_rows.as<double>(), ctx->stream));
    return fetch(ctx, {{out, ctx->get_rows.p, bytes}});
}

int cafe_gpu_set_tree(cafe_gpu_ctx* ctx, int n_nodes, const int* parent, const int* leaf_col)
{
    if (int rc = check_ctx(ctx)) return rc;
    if (n_nodes < 2 || !parent || !leaf_col) return fail(CAFE_GPU_EINVAL, "tree needs >= 2 nodes");
    std::vector<std::vector<int>> kids(n_nodes);
    std::vector<int> lc(leaf_col, leaf_col + n_nodes);
    int root = -1, n_leaves = 0;
    for (int i = 0; i < n_nodes; ++i) {
        if (parent[i] < 0) {
            if (root >= 0) return fail(CAFE_GPU_EINVAL, "tree has more than one root");
            root = i;
        } else if (parent[i] >= n_nodes || parent[i] == i) {
            return fail(CAFE_GPU_EINVAL, "node %d has an invalid parent", i);
        } else {
            kids[parent[i]].push_back(i);
        }
        if (lc[i] >= 0) ++n_leaves;
    }
    if (root < 0) return fail(CAFE_GPU_EINVAL, "tree has no root");
    for (int i = 0; i < n_nodes; ++i) {
        if (lc[i] >= 0 && !kids[i].empty()) return fail(CAFE_GPU_EINVAL, "leaf %d has children", i);
        if (lc[i] < 0 && kids[i].empty()) return fail(CAFE_GPU_EINVAL, "interior node %d has no children", i);
        if (lc[i] >= n_leaves) return fail(CAFE_GPU_EINVAL, "leaf column %d out of range", lc[i]);
        int d = 0;
        for (int p = i; p != root; p = parent[p])
            if (++d > n_nodes) return fail(CAFE_GPU_EINVAL, "tree has a cycle");
    }
    if (lc[root] >= 0) return fail(CAFE_GPU_EINVAL, "root cannot be a leaf");
    std::vector<char> seen(n_leaves, 0);
    for (int i = 0; i < n_nodes; ++i)
        if (lc[i] >= 0) {
            if (seen[lc[i]]) return fail(CAFE_GPU_EINVAL, "leaf column %d used twice", lc[i]);
            seen[lc[i]] = 1;
        }
    Planner pl(kids, lc);
    pl.compute_need(root);
    pl.used.clear();
    pl.emit(root);
    // the per-lane kernel's program: the same order, the vector each op reads
    // from the op just before it in registers, the others in output-reusing
    // slots
    Planner ph(kids, lc, true, true);
    ph.compute_need(root);
    ph.used.clear();
    ph.emit(root, false);
    if (pl.max_slot + 1 > kMaxSlots)
        return fail(CAFE_GPU_EINVAL, "tree needs %d live partial vectors (max %d)", pl.max_slot + 1, kMaxSlots);
    HIP_OR_FAIL(hipStreamSynchronize(ctx->stream));   // nothing reads what is replaced here
    ctx->input_gen++;
    if (n_nodes != ctx->n_nodes || !std::equal(parent, parent + n_nodes, ctx->parent_h.begin()) || lc != ctx->leaf_col_h)
        ctx->pat.clear();
    ctx->n_nodes = n_nodes;
    ctx->tree_leaves = n_leaves;
    ctx->parent_h.assign(parent, parent + n_nodes);
    ctx->leaf_col_h.assign(leaf_col, leaf_col + n_nodes);
    ctx->max_children = 1;
    for (auto& k : kids) ctx->max_children = std::max(ctx->max_children, (int)k.size());
    ctx->n_slots = pl.max_slot + 1;
    ctx->ops = pl.ops;
    // the program as a flat list of child steps
    const std::vector<StepDev> steps = flatten_steps(pl.ops, pl.out_kids);
    ctx->n_steps = (int)steps.size();
    HIP_OR_FAIL(ctx->d_steps.ensure(sizeof(StepDev) * steps.size()));
    HIP_OR_FAIL(hipMemcpy(ctx->d_steps.p, steps.data(), sizeof(StepDev) * steps.size(), hipMemcpyHostToDevice));
    // the lane kernel's program: the same order, outputs reusing child slots
    Planner pr(kids, lc, true);
    pr.compute_need(root);
    pr.used.clear();
    pr.emit(root);
    const std::vector<StepDev> lsteps = flatten_steps(pr.ops, pr.out_kids);
    ctx->n_slots_lane = pr.max_slot + 1;
    HIP_OR_FAIL(ctx->d_steps_lane.ensure(sizeof(StepDev) * lsteps.size()));
    HIP_OR_FAIL(hipMemcpy(ctx->d_steps_lane.p, lsteps.data(), sizeof(StepDev) * lsteps.size(),
                          hipMemcpyHostToDevice));
    const std::vector<StepDev> hsteps = flatten_steps(ph.ops, ph.out_kids);
    ctx->n_slots_hot = std::max(1, ph.max_slot + 1);
    HIP_OR_FAIL(ctx->d_steps_hot.ensure(sizeof(StepDev) * hsteps.size()));
    HIP_OR_FAIL(hipMemcpy(ctx->d_steps_hot.p, hsteps.data(), sizeof(StepDev) * hsteps.size(),
                          hipMemcpyHostToDevice));
    // level by level: an op's level is one past its interior children's
    std::vector<int> level(n_nodes, 0), by_level(pl.ops.size()), op_of(n_nodes, -1);
    for (const OpDev& op : pl.ops)   // (children before parents)
        for (int c : kids[op.node])
            if (lc[c] < 0) level[op.node] = std::max(level[op.node], level[c] + 1);
    std::iota(by_level.begin(), by_level.end(), 0);
    std::stable_sort(by_level.begin(), by_level.end(),
                     [&](int a, int b) { return level[pl.ops[a].node] < level[pl.ops[b].node]; });
    std::vector<StepDev> vsteps;
    std::vector<int> op_steps;
    ctx->level_ops.clear();
    for (int i = 0; i < (int)by_level.size(); ++i) {
        const OpDev& op = pl.ops[by_level[i]];
        if (i == 0 || level[op.node] != level[pl.ops[by_level[i - 1]].node]) ctx->level_ops.push_back(i);
        op_of[op.node] = i;
        op_steps.push_back((int)vsteps.size());
        for (int k = 0; k < op.n_child; ++k) {
            const int c = pl.out_kids[op.child_begin + k].node;
            vsteps.push_back(StepDev{c, lc[c], lc[c] >= 0 ? -1 : op_of[c],
                                     (k == 0 ? kStepFirst : 0) | (k + 1 == op.n_child ? kStepLast : 0) |
                                         (op.node == root ? kStepRoot : 0)});
        }
    }
    ctx->level_ops.push_back((int)by_level.size());
    HIP_OR_FAIL(ctx->d_steps_level.ensure(sizeof(StepDev) * vsteps.size()));
    HIP_OR_FAIL(hipMemcpy(ctx->d_steps_level.p, vsteps.data(), sizeof(StepDev) * vsteps.size(), hipMemcpyHostToDevice));
    HIP_OR_FAIL(ctx->d_op_steps.ensure(sizeof(int) * op_steps.size()));
    HIP_OR_FAIL(hipMemcpy(ctx->d_op_steps.p, op_steps.data(), sizeof(int) * op_steps.size(), hipMemcpyHostToDevice));
    return CAFE_GPU_OK;
}

int cafe_gpu_set_families(cafe_gpu_ctx* ctx, int F, int n_leaves, const int* counts, const int* bound_B,
                          const int* bound_R, int B, int R)
{
    if (int rc = check_ctx(ctx)) return rc;
    if (F < 1 || n_leaves < 1 || !counts) return fail(CAFE_GPU_EINVAL, "need at least one family and leaf");
    std::vector<int> fb(F), fr(F), top(F, 0);
    for (int f = 0; f < F; ++f) {
        fb[f] = bound_B ? bound_B[f] : B;
        fr[f] = bound_R ? bound_R[f] : R;
        if (fb[f] < 1 || fr[f] < 1) return fail(CAFE_GPU_EINVAL, "family %d has a non-positive bound", f);
        for (int i = 0; i < n_leaves; ++i) {
            const int c = counts[(size_t)f * n_leaves + i];
            if (c < 0 || c > fb[f])
                return fail(CAFE_GPU_EINVAL, "family %d leaf %d count %d outside 0..%d", f, i, c, fb[f]);
            top[f] = std::max(top[f], c);
        }
    }
    std::vector<int> order(F);
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
        return fb[a] != fb[b] ? fb[a] < fb[b] : fr[a] < fr[b];
    });
    std::vector<BucketHost> buckets;
    for (int k = 0; k < F; ++k) {
        const int f = order[k];
        if (buckets.empty() || buckets.back().B != fb[f] || buckets.back().R != fr[f])
            buckets.push_back(BucketHost{fb[f], fr[f], 0, k, 0});
        auto& b = buckets.back();
        b.count++;
        b.max_count = std::max(b.max_count, top[f]);
    }
    HIP_OR_FAIL(hipStreamSynchronize(ctx->stream));
    ctx->input_gen++;
    std::vector<int> cT((size_t)n_leaves * F);
    for (int k = 0; k < F; ++k)
        for (int i = 0; i < n_leaves; ++i) cT[(size_t)i * F + k] = counts[(size_t)order[k] * n_leaves + i];
    // (the patterns are of the sorted counts and the sizes; the caller's order may change)
    if (cT != ctx->counts_T || buckets != ctx->buckets) ctx->pat.clear();
    HIP_OR_FAIL(ctx->d_counts.ensure(sizeof(int) * cT.size()));
    HIP_OR_FAIL(ctx->d_perm.ensure(sizeof(int) * F));
    HIP_OR_FAIL(hipMemcpy(ctx->d_counts.p, cT.data(), sizeof(int) * cT.size(), hipMemcpyHostToDevice));
    HIP_OR_FAIL(hipMemcpy(ctx->d_perm.p, order.data(), sizeof(int) * F, hipMemcpyHostToDevice));
    ctx->perm = order;
    ctx->fam_max = top;
    ctx->F = F;
    ctx->n_leaves = n_leaves;
    ctx->buckets.swap(buckets);
    ctx->counts_T.swap(cT);
    return CAFE_GPU_OK;
}

int cafe_gpu_bucket_count(cafe_gpu_ctx* ctx, int* n)
{
    if (!ctx || !n) return fail(CAFE_GPU_EINVAL, "null argument");
    *n = (int)ctx->buckets.size();
    return CAFE_GPU_OK;
}

int cafe_gpu_bucket_info(cafe_gpu_ctx* ctx, int i, int* B, int* R, int* count)
{
    if (!ctx) return fail(CAFE_GPU_EINVAL, "null context");
    if (i < 0 || i >= (int)ctx->buckets.size()) return fail(CAFE_GPU_EINVAL, "bucket %d out of range", i);
    if (B) *B = ctx->buckets[i].B;
    if (R) *R = ctx->buckets[i].R;
    if (count) *count = ctx->buckets[i].count;
    return CAFE_GPU_OK;
}

int cafe_gpu_set_error_model(cafe_gpu_ctx* ctx, int n_dev, int n_rows, const double* rows)
{
    if (int rc = check_ctx(ctx)) return rc;
    if (!rows) {
        if (ctx->n_dev) ctx->input_gen++;
        ctx->n_dev = 0;
        ctx->err_rows = 0;
        return CAFE_GPU_OK;
    }
    if (n_dev < 1 || n_dev % 2 == 0 || n_rows < 1)
        return fail(CAFE_GPU_EINVAL, "error model needs an odd number of deviations and >= 1 row");
    if (n_dev != ctx->n_dev || n_rows != ctx->err_rows) ctx->input_gen++;   // same shape: in place
    HIP_OR_FAIL(hipStreamSynchronize(ctx->stream));
    const size_t n = (size_t)n_dev * n_rows;
    std::vector<float> r32(rows, rows + n);
    HIP_OR_FAIL(ctx->d_err64.ensure(sizeof(double) * n));
    HIP_OR_FAIL(ctx->d_err32.ensure(sizeof(float) * n));
    HIP_OR_FAIL(hipMemcpy(ctx->d_err64.p, rows, sizeof(double) * n, hipMemcpyHostToDevice));
    HIP_OR_FAIL(hipMemcpy(ctx->d_err32.p, r32.data(), sizeof(float) * n, hipMemcpyHostToDevice));
    ctx->n_dev = n_dev;
    ctx->err_rows = n_rows;
    // fold into every slot of an existing pool (later builds fold their own slots)
    if (int rc = ensure_fold_pools(ctx)) return rc;
    if (int rc = enqueue_fold(ctx, 0, ctx->capacity, ctx->stream)) return rc;
    HIP_OR_FAIL(hipStreamSynchronize(ctx->stream));
    return CAFE_GPU_OK;
}

}  // extern "C"


namespace {

// Kernel size class: buckets whose vectors have the same number of 16-row
// tiles.
struct KernelClass {
    int key;             // of its buckets (plan_prune)
    int nt;              // 16-row tiles of the class's largest vector
    int slot_tiles;      // 16-row tiles of its largest stored (non-root) vector
    MfmaShape s32, s64;  // launch shapes of the FP32 and FP64 MFMA kernels
    MfmaShape s16;       // launch shape of the split-FP16 kernel (BATCHED16)
    MfmaShape r64;       // FP64 recompute of the FP32 pass (a few tiles: latency)
    int lane_rows = 0;   // > 0: the FP32 main pass runs k_prune_lane with this many rows (64-family tiles)
    bool f64 = false;    // the main pass is k_prune_f64's (final values)
    long long fams = 0;  // its family-likelihoods
    bool plain = false;  // PLAIN64, or vectors over 64 tiles (1,024 rows): f64 on every path
    int lane_slots = 0;  // its slot instance
    int lane_per_cu = 0; // its workgroups resident per CU
    int lane_grid_mult = 0;   // workgroups per resident slot (0: default)
    int fb = 1;          // matrix-core main pass: blocks of 16 families per tile
    bool tuned = false;  // its shape came from the context's tuning table
    int r16 = 0;         // 16-family tiles its families fill (the recompute lists' capacity)
    int r_begin = 0;     // offset of its FP64 recompute list
    int begin, end;      // its main tiles
    int seg_begin = 0, seg_end = 0;   // its (bucket, point) segments
    // byte offsets of its global scratch in the main pass and the FP64
    // recompute: disjoint, since one class's recompute can run beside another
    // class's main pass
    size_t off_main = 0, off_r64 = 0, off_level = 0;
    int level_tiles = 0;   // most tiles its recompute takes level by level (0: none)
    int stream = 0;      // side stream of its launches
    // subtree patterns: its buckets run their programs over units' columns,
    // made level by level before the main pass (tiles, their count's place)
    bool pat = false;
    int max_pat = 0, n_cols = 0;            // most pattern and leaf columns of a program
    int n_slots = 0, n_slots_lane = 0, n_slots_hot = 0;   // most partial vectors of a program (in order, reuse, hot)
    struct Level {
        int begin, n, count_at;
    };
    std::vector<Level> levels;
};

// Host-side description of one pruning sequence over a tile list.
struct PrunePlan {
    int path = 0, model = 0;
    std::vector<KernelClass> classes;
    std::vector<int> class_counts;   // main tiles per class (+ padding)
    std::vector<int> main_order;     // main-pass launch order (longest first)
    int light_stream = 0;            // the side stream expected to finish its main-pass work first
    bool has_f64 = false;            // a class's main pass reads the FP64 pool
    int n_split = 0;                 // BATCHED16: pool slots converted to FP16 halves before pruning
    int n_tiles = 0, n_segs = 0, maxLR = 0;
    int r16_total = 0;               // capacity of the FP64 recompute lists (16-family tiles)
    int waves_per_cu = 16;           // persistent grid: resident waves per CU
    int n_cu = 256;
    PruneParams base{};
    // fb_count layout: [0, n) FP64 recompute tiles per class, [n] families
    // recomputed in FP64, [n + 1] those with FP64 values near the subnormal range
    int fam_count_off() const { return (int)classes.size(); }
    // a lane-kernel launch: as an MFMA launch with partials in LDS
    int grid_lane(int per_cu, int max_tiles, int mult = 0) const
    {
        const long long want = (long long)n_cu * std::max(1, per_cu) * (mult > 0 ? mult : 16);
        const int g = (int)std::max(1LL, std::min(want, (long long)max_tiles));
        return g >= 8 ? g / 8 * 8 : g;
    }
    // an MFMA launch: a multiple of the workgroups of its shape that are
    // resident at once.  Each workgroup takes an equal static share of the
    // tiles, so with many more workgroups than slots the dispatcher evens
    // out the per-CU load as slots free up (16x: the small-vector classes run
    // ~25% faster than with exactly one resident round).  Kernels with
    // partials in global scratch, which grows with the grid, take 2x.
    int grid(const MfmaShape& s, int max_tiles) const
    {
        const int per_cu = s.per_cu > 0 ? s.per_cu : std::max(1, waves_per_cu / std::max(1, s.w));
        const long long want = (long long)n_cu * per_cu * (s.grid_mult > 0 ? s.grid_mult : (s.lds ? 16 : 2));
        const int g = (int)std::max(1LL, std::min(want, (long long)max_tiles));
        return g >= 8 ? g / 8 * 8 : g;
    }
};

// MFMA launch shape for vectors of nt 16-row tiles: W waves per workgroup
// split the output tiles, NTW per wave, so that W NTW >= nt (one pass; the
// scaled FP32 kernel needs the whole vector in one pass).  Small vectors run
// one wave per family tile (throughput), large ones several (latency).
MfmaShape mfma_shape(int nt)
{
    MfmaShape s{1, 1, false, 0};
    if (nt <= 4) s = {std::max(1, nt), 1, false, 0};
    else if (nt <= 8) s = {(nt + 1) / 2, 2, false, 0};
    else if (nt <= 16) s = {(nt + 3) / 4, 4, false, 0};
    else if (nt <= 32) s = {(nt + 7) / 8, 8, false, 0};
    else s = {(nt + 15) / 16, 16, false, 0};   // up to 64 tiles
    return s;
}

// FP32 launch shape of a plan with few families, whose time is the chain of
// steps of the tiles each CU holds: one row tile per wave, as many waves as the
// vector has tiles.  A score of 8,000 families of 34 taxa at B = 100 379 -> 312
// us, 5,000 at 150 417 -> 381, 2,000 at 200 429 -> 366, 1,000 of 60 taxa at 120 983
// -> 561.  More families fill the chip and the wider shapes' fewer loads win; the
// line, 32 families per CU, lies between the sizes where that happens (one step
// over shared subtrees, this shape against the 32-family tiles taken from there
// on): 34 taxa at B = 100 8,191 families 161 us against 204, 12,000 202 against 221,
// 32,000 296 against 290; at 150 5,000 families 254 against 335, 8,000 291 against
// 310 (275 on 16-family tiles), 12,000 341 against 323; 60 taxa at 120 8,000 246
// against 292, 16,000 295 against 324; 200,000 gamma families 1.25 ms against 0.94.
MfmaShape mfma_shape_few(int nt) { return {1, nt <= 4 ? 4 : nt <= 8 ? 8 : 16, false, 0}; }

// FP32 launch shape with 32-family tiles (two blocks of 16 per MFMA operand)
// for vectors of up to 32 tiles (kMaxTilesFb2): two output tiles per wave
// over 4, 8 or 16 waves (the products and factors of both blocks are held per
// output tile, so more tiles per wave would spill).
constexpr int kMaxTilesFb2 = 32;
MfmaShape mfma_shape_fb2(int nt)
{
    MfmaShape s{2, nt <= 8 ? 4 : nt <= 16 ? 8 : 16, false, 0};
    s.fb = 2;
    if (s.w == 16) s.grid_mult = 1;   // one resident round (global partials grow with the grid)
    return s;
}

// Built-in family-block choice of the FP32 kernel: 32-family tiles for the
// 17-32-tile vectors (one output tile of sixteen waves per 16 families would
// otherwise stream each matrix operand for one MFMA: 1.5x slower at B = 500)
// and for the only matrix-core class of a plan when it fills the device
// with at least one 32-family tile per CU (measured 1.1-1.4x faster: B = 100,
// 150; with 2,000 families, 9% slower); 16-family tiles for smaller vectors
// when several matrix-core classes run concurrently, where the shorter tile
// lists leave fewer waves resident beside the other classes and the step
// gains nothing.
int builtin_fb32(int path, int nt, bool only_mfma_class, long long fam_points, int n_cu)
{
    if (path != CAFE_GPU_PATH_BATCHED32 || nt > kMaxTilesFb2) return 1;
    return nt > 16 || (only_mfma_class && fam_points >= 32LL * n_cu) ? 2 : 1;
}

// Partials of the FP64 kernel: 2 KB per stored tile and family block.
size_t f64_frag_bytes(const MfmaShape& s, int n_slots, int nt) { return (size_t)n_slots * nt * s.fb * 64 * 32; }

size_t f64_shm(const MfmaShape& s, int n_slots, int nt, int n_leaves)
{
    return (size_t)f64_meta_bytes(s.w, s.fb, n_leaves, s.staged) + (s.lds ? f64_frag_bytes(s, n_slots, nt) : 0);
}

// FP64 shape (k_prune_f64) for vectors of nt tiles and a list of `tiles`
// 16-family tiles.  One wave per row tile and 16 families per workgroup, with
// the partials in LDS, wherever they fit a CU (150 KB): against global partials
// 3.51 to 4.93 ms per step (160,000 family-likelihoods, 101 rows, 34 taxa) and
// 9.8 to 13.0 (80,000, 201 rows, 60 taxa).  Two differences, where the list
// fills the chip:
//  - up to 5 tiles per vector 32 families, as one wave's matrix loads are then
//    most of its step: 3.08 -> 2.56 ms (320,000, 61 rows);
//  - vectors past LDS stream matrices and partials from L2: 2 x 2 blocks per
//    wave use every load twice, 8.2 -> 6.0 ms (24,000, 401 rows).
// Short lists of such vectors (the recompute) are one tile's chain of steps:
// two row tiles in each of 16 waves take all 32 tiles of 501 rows in one pass
// (search at B = 500: 45.0 -> 43.6 ms).
MfmaShape f64_shape(int nt, long long tiles, int n_slots, int n_leaves, int n_cu)
{
    MfmaShape s{1, 1, true, 0};
    s.staged = n_leaves <= 512;   // their counts take 32 KB; more stay in memory
    s.w = std::min(16, nt);
    s.lds = s.staged && f64_shm(s, n_slots, nt, n_leaves) <= 150 * 1024;
    if (s.lds && nt <= 5 && tiles >= 16LL * n_cu) {
        MfmaShape two = s;
        two.fb = 2;
        if (f64_shm(two, n_slots, nt, n_leaves) <= 75 * 1024) s = two;
    } else if (!s.lds && s.staged) {
        s.ntw = 2;
        s.fb = tiles >= 4LL * n_cu ? 2 : 1;
        s.w = std::min(s.fb == 2 ? 8 : 16, (nt + 1) / 2);
    }
    s.shm = f64_shm(s, n_slots, nt, n_leaves);
    return s;
}

int f64_occupancy(MfmaShape& s)
{
    const PruneParams none{};
    HIP_OR_FAIL(f64_dispatch(s, 0, none, nullptr, &s.per_cu));
    return CAFE_GPU_OK;
}

size_t f64_scratch_bytes(const MfmaShape& s, int n_slots, int nt, int grid)
{
    return s.lds ? 0 : (size_t)grid * f64_frag_bytes(s, n_slots, nt);
}

// Dynamic LDS of an MFMA launch without its partials: the bookkeeping and the
// tile's leaf counts.
size_t mfma_meta_only(const MfmaShape& s, int n_slots, int n_leaves, int n_pat)
{
    return (size_t)mfma_meta_bytes(n_slots, s.w, s.fb) + (size_t)mfma_count_bytes(n_leaves, s.fb) +
           (size_t)mfma_pat_bytes(n_pat, s.fb);
}

// Partial vectors go to LDS when the workgroup's share stays small enough for
// several workgroups per CU; the rest use the global scratch.
void place_partials(MfmaShape& s, int n_slots, int slot_tiles, int n_leaves, int n_pat)
{
    const size_t meta = mfma_meta_only(s, n_slots, n_leaves, n_pat);
    const size_t frag = (size_t)n_slots * slot_tiles * s.fb * 64 * 4 * 4;
    if (s.fb > 1)   // two workgroups per CU, or one of 8 waves
        s.lds = s.w <= 8 && meta + frag + 4096 <= (s.w >= 8 ? 144 : 76) * 1024;
    else
        s.lds = (s.w <= 4 && meta + frag + 4096 <= 64 * 1024 && (meta + frag) / s.w <= 20 * 1024) ||
                (s.w > 4 && s.ntw == 1 && meta + frag + 4096 <= 76 * 1024);   // (latency shapes)
    s.shm = meta + (s.lds ? frag : 0);
}

// The split-FP16 kernel takes vectors of up to 32 tiles (eight waves of four
// tiles without spilling registers); BATCHED16 runs larger ones on the FP32
// matrix-core kernel.
constexpr int kF16MaxTiles = 32;
constexpr int kMfmaMaxTiles = 64;     // the matrix-core shapes' largest vectors (1,024 rows)
constexpr int kMaxRows = 2048;        // the largest vectors of any path

// The split-FP16 kernel's partials: per 32-row block and lane three 16-byte
// B operands (hi, lo, bound).
size_t f16_frag_bytes(int n_slots, int slot_tiles) { return (size_t)3 * n_slots * ((slot_tiles + 1) / 2) * 64 * 16; }

size_t f16_meta_only(const MfmaShape& s, int n_slots, int n_leaves, int n_pat)
{
    return (size_t)f16_meta_bytes(n_slots, s.w) + (size_t)mfma_count_bytes(n_leaves) + (size_t)f16_pat_bytes(n_pat);
}

void place_partials16(MfmaShape& s, int n_slots, int slot_tiles, int n_leaves, int n_pat)
{
    const size_t meta = f16_meta_only(s, n_slots, n_leaves, n_pat);
    const size_t frag = f16_frag_bytes(n_slots, slot_tiles);
    // two workgroups per CU (its registers allow two waves per SIMD)
    s.lds = s.w <= 4 && meta + frag + 4096 <= 76 * 1024;
    s.shm = meta + (s.lds ? frag : 0);
}

size_t f16_scratch_bytes(const MfmaShape& s, int n_slots, int slot_tiles, int grid)
{
    return s.lds ? 0 : (size_t)grid * f16_frag_bytes(n_slots, slot_tiles);
}

// A class runs over subtree patterns from this many family-likelihoods on: each
// level of units is a launch more (2,000 families of 12 taxa at B = 100, three
// levels: 305 -> 285 us a step).
constexpr long long kPatternWork = 1024;
// Recompute lists of vectors past LDS run level by level up to this many tiles
// (256 families), with their vectors in at most kLevelBytes: shorter vectors'
// chains are short (0.1 ms at 101 rows, 0.4 at 201) beside a launch per level.
constexpr int kLevelTiles = 16;
constexpr size_t kLevelBytes = (size_t)256 << 20;
// Columns of one evaluation, at most.
constexpr size_t kPatternBytes = (size_t)8 << 30;

// Dynamic LDS of a lane-kernel launch: the tile's leaf counts.
size_t lane_shm(int n_leaves) { return (size_t)n_leaves * 64 * sizeof(int); }

// Global scratch of an MFMA launch (partials not in LDS), bytes.
size_t mfma_scratch_bytes(const MfmaShape& s, int n_slots, int slot_tiles, int grid)
{
    if (s.lds) return 0;
    return (size_t)grid * n_slots * slot_tiles * s.fb * 64 * 4 * 4;
}

// The tuning entry for a class of a plan whose size classes are plan_classes
// (bit nt - 1 per class of nt tiles), if the context holds one: an entry
// measured in a plan of the same classes, else one for any plan.
const cafe_gpu_ctx::TuneEntry* find_tuning(const cafe_gpu_ctx* ctx, int path, int nt,
                                           unsigned long long plan_classes)
{
    const cafe_gpu_ctx::TuneEntry* any = nullptr;
    for (const auto& e : ctx->tuning) {
        if (e.path != path || e.nt != nt || e.leaves != ctx->n_leaves) continue;
        if (e.plan_classes == plan_classes) return &e;
        if (e.plan_classes == 0 && !any) any = &e;
    }
    return any;
}

// The matrix-core shape a tuning entry names for a class of nt tiles whose
// stored vectors have slot_tiles tiles, when that kernel instance exists,
// covers the class (tiles per wave x waves >= nt) and fits a CU (occupancy
// query; LDS partials only where they fit).
bool tuned_mfma_shape(cafe_gpu_ctx* ctx, int path, const cafe_gpu_ctx::TuneEntry& e, const KernelClass& kc, int nt,
                      int slot_tiles, MfmaShape& s)
{
    if ((e.kernel != 0 && e.kernel != 2) || path == CAFE_GPU_PATH_PLAIN64 || e.ntw < 1 || e.w < 1 || e.ntw * e.w < nt)
        return false;
    const bool f16 = path == CAFE_GPU_PATH_BATCHED16 && e.kernel == 0;
    if (f16 && nt > kF16MaxTiles) return false;
    const bool fp64 = path == CAFE_GPU_PATH_BATCHED64;
    // 32-family tiles: the FP64 kernel, and the FP32 kernel's main pass
    // (BATCHED32, or BATCHED16 classes past the split-FP16 kernel's sizes)
    if (e.kernel == 2 && !fp64 && (nt > kMaxTilesFb2 || (path == CAFE_GPU_PATH_BATCHED16 && nt <= kF16MaxTiles)))
        return false;
    s = MfmaShape{e.ntw, e.w, e.lds != 0, 0, 0};
    s.fb = e.kernel == 2 ? 2 : 1;
    hipError_t q = hipSuccess;
    const PruneParams none{};
    if (fp64) {
        s.shm = f64_shm(s, kc.n_slots, nt, kc.n_cols);
        if (s.shm > 150 * 1024 || ctx->n_leaves > 512) return false;   // LDS partials that do not fit
        q = f64_dispatch(s, 0, none, nullptr, &s.per_cu);
    } else {
        if (f16) place_partials16(s, kc.n_slots_lane, slot_tiles, kc.n_cols, kc.max_pat);
        else place_partials(s, kc.n_slots, slot_tiles, kc.n_cols, kc.max_pat);
        if (e.lds && !s.lds) return false;   // LDS partials that do not fit
        if (!e.lds && s.lds) {               // global scratch asked for
            s.lds = false;
            s.shm = f16 ? f16_meta_only(s, kc.n_slots_lane, kc.n_cols, kc.max_pat)
                        : mfma_meta_only(s, kc.n_slots, kc.n_cols, kc.max_pat);
        }
        q = f16 ? f16_dispatch(s, 0, none, nullptr, &s.per_cu) : mfma_occupancy(s, &s.per_cu);
    }
    if (q != hipSuccess || s.per_cu < 1) {
        (void)hipGetLastError();
        return false;   // no such instance, or it does not fit a CU
    }
    s.grid_mult = std::max(0, e.grid_mult);
    return true;
}

// Replaces a class's built-in launch shape by its tuning entry where the entry
// is usable (the kernel itself -- per lane or matrix cores -- was chosen when
// the class's tiles were made); otherwise the class keeps its shape.
int apply_tuning(cafe_gpu_ctx* ctx, int path, KernelClass& kc, unsigned long long plan_classes)
{
    const cafe_gpu_ctx::TuneEntry* e = find_tuning(ctx, path, kc.nt, plan_classes);
    if (!e || path == CAFE_GPU_PATH_PLAIN64) return CAFE_GPU_OK;
    if (kc.lane_rows > 0) {
        if (e->kernel == 1) {
            kc.lane_grid_mult = std::max(0, e->grid_mult);
            kc.tuned = true;
        }
        return CAFE_GPU_OK;
    }
    MfmaShape s;
    if (!tuned_mfma_shape(ctx, path, *e, kc, kc.nt, kc.slot_tiles, s)) return CAFE_GPU_OK;
    if (s.fb != kc.fb) return CAFE_GPU_OK;   // the tiles were cut for another width
    if (path == CAFE_GPU_PATH_BATCHED16 && e->kernel == 0) kc.s16 = s;
    else if (path == CAFE_GPU_PATH_BATCHED64) kc.s64 = s;
    else kc.s32 = s;
    kc.tuned = true;
    return CAFE_GPU_OK;
}

// Validates a descriptor and puts node slots, priors and category probabilities
// into b's input block (plan_prune completes and uploads it); sizes the
// per-point outputs.
int upload_eval_inputs(cafe_gpu_ctx* ctx, EvalBufs& b, const cafe_gpu_eval_desc* d, int& P)
{
    if (!d) return fail(CAFE_GPU_EINVAL, "null descriptor");
    if (ctx->n_nodes == 0) return fail(CAFE_GPU_ESTATE, "set_tree has not been called");
    if (ctx->F == 0) return fail(CAFE_GPU_ESTATE, "set_families has not been called");
    if (ctx->N == 0) return fail(CAFE_GPU_ESTATE, "matrix_reset has not been called");
    if (ctx->n_leaves != ctx->tree_leaves)
        return fail(CAFE_GPU_EINVAL, "families have %d leaves, tree has %d", ctx->n_leaves, ctx->tree_leaves);
    if (d->model != CAFE_GPU_MODEL_BASE && d->model != CAFE_GPU_MODEL_GAMMA)
        return fail(CAFE_GPU_EINVAL, "unknown model %d", d->model);
    if (d->path < CAFE_GPU_PATH_PLAIN64 || d->path > CAFE_GPU_PATH_BATCHED16)
        return fail(CAFE_GPU_EINVAL, "unknown path %d", d->path);
    const int K = d->n_cat;
    if (d->n_trials < 1 || K < 1 || (d->model == CAFE_GPU_MODEL_BASE && K != 1))
        return fail(CAFE_GPU_EINVAL, "bad trial/category counts");
    if (!d->node_slot || !d->prior) return fail(CAFE_GPU_EINVAL, "null node_slot or prior");
    if (d->model == CAFE_GPU_MODEL_GAMMA && !d->cat_probs) return fail(CAFE_GPU_EINVAL, "gamma needs cat_probs");
    const int h = ctx->n_dev ? (ctx->n_dev - 1) / 2 : 0;
    int maxR = 0;
    for (auto& bk : ctx->buckets) {
        if (std::max(bk.B, bk.R) + 1 > ctx->N)
            return fail(CAFE_GPU_EINVAL, "bucket B=%d R=%d needs matrices of size %d (pool has %d)", bk.B, bk.R,
                        std::max(bk.B, bk.R) + 1, ctx->N);
        if (ctx->n_dev && (bk.B >= ctx->err_rows || bk.max_count + h > bk.B))
            return fail(CAFE_GPU_EINVAL, "error model does not cover bucket B=%d (max count %d)", bk.B,
                        bk.max_count);
        maxR = std::max(maxR, bk.R);
    }
    if (d->prior_stride < maxR) return fail(CAFE_GPU_EINVAL, "prior_stride %d < max R %d", d->prior_stride, maxR);
    P = d->n_trials * K;
    const long long ns = (long long)P * ctx->n_nodes;
    std::vector<int> slot(d->node_slot, d->node_slot + ns);
    const int root = ctx->ops.back().node;
    for (long long i = 0; i < ns; ++i) {
        const int node = (int)(i % ctx->n_nodes);
        if (node == root) {
            slot[i] = 0;
            continue;
        }
        if (slot[i] < 0 || slot[i] >= ctx->capacity || !ctx->built[slot[i]])
            return fail(CAFE_GPU_ENOTFOUND, "node %d of point %lld uses matrix slot %d, which is not built", node,
                        i / ctx->n_nodes, slot[i]);
        if (ctx->built[slot[i]] == 2 && (d->path == CAFE_GPU_PATH_BATCHED32 || d->path == CAFE_GPU_PATH_BATCHED16))
            return fail(CAFE_GPU_ENOTFOUND,
                        "matrix slot %d holds the FP64 matrix and only the FP32 copies a plan read; build it with "
                        "cafe_gpu_matrix_build for this path", slot[i]);
    }
    const int nb = (int)ctx->buckets.size();
    std::vector<double> pr64((size_t)nb * d->prior_stride, 0.0);
    std::vector<BucketDev>& bd = b.bucket_h;
    bd.assign(nb, BucketDev{});
    for (int i = 0; i < nb; ++i) {
        const auto& bh = ctx->buckets[i];
        for (int j = 0; j < bh.R; ++j) pr64[(size_t)i * d->prior_stride + j] = d->prior[(size_t)i * d->prior_stride + j];
        bd[i].B = bh.B;
        bd[i].R = bh.R;
        bd[i].L = bh.B + 1;
        bd[i].Lp = round_up(bh.B + 1, kTile);
        bd[i].Rp = round_up(bh.R + 1, kTile);
        bd[i].fam_begin = bh.fam_begin;
        bd[i].count = bh.count;
        bd[i].prior_off = i * d->prior_stride;
        bd[i].out = -1;
    }
    std::vector<double> cp(K, 1.0);
    if (d->cat_probs) cp.assign(d->cat_probs, d->cat_probs + K);
    b.block.clear();
    b.views.clear();
    b.put(b.node_slot, slot.data(), sizeof(int) * ns);
    b.put(b.prior64, pr64.data(), sizeof(double) * pr64.size());
    b.put(b.catp, cp.data(), sizeof(double) * K);
    const size_t PF = (size_t)P * ctx->F;
    HIP_OR_FAIL(b.val.ensure(sizeof(double) * PF));
    HIP_OR_FAIL(b.flag.ensure(sizeof(int) * PF));
    const size_t TF = (size_t)d->n_trials * ctx->F;
    HIP_OR_FAIL(b.lnl.ensure(sizeof(double) * TF));
    HIP_OR_FAIL(b.cat.ensure(sizeof(double) * TF * K));
    HIP_OR_FAIL(b.post.ensure(sizeof(double) * TF * K));
    HIP_OR_FAIL(b.fail.ensure(sizeof(int) * TF));
    HIP_OR_FAIL(b.total.ensure(sizeof(double) * d->n_trials));
    return CAFE_GPU_OK;
}

// Builds and uploads the tile list for `n_points` parameter points (heaviest
// classes and buckets first, grouped by kernel size class) and sizes the
// scratch.  `whole` are the keys of the classes that do not run over subtree
// patterns although they could.
int plan_over(cafe_gpu_ctx* ctx, EvalBufs& b, int path, int model, int n_points, const int* point_ids,
              double* root_out, int root_stride, PrunePlan& pp, const std::set<int>& whole)
{
    pp = PrunePlan();
    pp.path = path;
    pp.model = model;
    pp.n_cu = ctx->n_cu;
    int maxLR = 0;
    for (auto& bk : ctx->buckets)
        maxLR = std::max(maxLR, std::max(round_up(bk.B + 1, kTile), round_up(bk.R + 1, kTile)));
    pp.maxLR = maxLR;
    std::vector<std::pair<int, int>> bucket_class;   // (class key, bucket)
    for (int bi = 0; bi < (int)ctx->buckets.size(); ++bi) {
        const BucketHost& bk = ctx->buckets[bi];
        // vectors (sizes 0..B) and root rows (sizes 0..R) up to 2,048 rows:
        // the FP32 and FP16 shapes take up to 64 tiles of 16, larger vectors
        // run on the FP64 kernel in every path
        if (std::max(bk.B + 1, bk.R + 1) > kMaxRows)
            return fail(CAFE_GPU_EINVAL, "bucket B=%d R=%d exceeds the sizes this path supports", bk.B, bk.R);
        // PLAIN64: one class per power of two of 4-tile blocks (the FP64
        // kernel takes vectors of any length)
        int key = tiles_of(bk);
        if (path == CAFE_GPU_PATH_PLAIN64) {
            int pow2 = 4;
            while (pow2 < key) pow2 <<= 1;
            key = pow2;
        }
        bucket_class.push_back({key, bi});
    }
    // heavy classes (and, within a class, larger buckets) first
    std::stable_sort(bucket_class.begin(), bucket_class.end(), [&](const std::pair<int, int>& x,
                                                                   const std::pair<int, int>& y) {
        if (x.first != y.first) return x.first > y.first;
        return ctx->buckets[x.second].B > ctx->buckets[y.second].B;
    });
    // size classes the one-family-per-lane FP32 kernel takes: all vectors and
    // root rows within one of its row counts, and the tree's slots within its
    // instances
    std::map<int, int> key_rows;
    for (auto& bc : bucket_class) {
        const BucketHost& bk = ctx->buckets[bc.second];
        key_rows[bc.first] = std::max(key_rows[bc.first], std::max(bk.B + 1, bk.R + 1));
    }
    auto lane_rows_of = [&](int key) {
        if (path != CAFE_GPU_PATH_BATCHED32 && path != CAFE_GPU_PATH_BATCHED16) return 0;
        const int lr = lane_rows_for(key_rows[key]);
        return lr > 0 && ctx->n_slots_hot + 1 <= lane_max_slots(lr) ? lr : 0;
    };
    // size classes the matrix cores take (those the per-lane kernel does not),
    // and the family-likelihoods of each class
    int n_mfma_keys = 0;
    for (const auto& kr : key_rows)
        if (lane_rows_of(kr.first) == 0) ++n_mfma_keys;
    long long mfma_fams = 0;     // of all of them
    std::map<int, long long> key_fams;
    std::map<int, int> key_nt;   // and the tiles of its largest vector
    for (auto& bc : bucket_class) {
        key_fams[bc.first] += (long long)ctx->buckets[bc.second].count * n_points;
        key_nt[bc.first] = std::max(key_nt[bc.first], tiles_of(ctx->buckets[bc.second]));
    }
    for (const auto& kf : key_fams)
        if (lane_rows_of(kf.first) == 0) mfma_fams += kf.second;
    // the plan's size classes, for the tuning entries measured in a plan
    unsigned long long plan_classes = 0;
    for (const auto& kr : key_rows)
        if (kr.first >= 1 && kr.first <= 64) plan_classes |= 1ull << (kr.first - 1);
    // the classes that run over subtree patterns: those with units, enough
    // family-likelihoods, on a kernel that reads columns, with their columns
    // within the memory set aside
    auto can_share = [&](int key) {
        const bool f64 = path == CAFE_GPU_PATH_PLAIN64 || path == CAFE_GPU_PATH_BATCHED64 || key > kMfmaMaxTiles;
        return !root_out && !(f64 && ctx->n_leaves > 512) && !whole.count(key);   // (past 512 the counts are not staged)
    };
    std::map<int, long long> key_work;   // of the buckets that are searched
    for (auto& bc : bucket_class)
        if (ctx->buckets[bc.second].count >= kPatternFamilies)
            key_work[bc.first] += (long long)ctx->buckets[bc.second].count * n_points;
    for (const auto& kw : key_work)
        if (can_share(kw.first) && kw.second >= kPatternWork) make_patterns(ctx);
    const Patterns& pat = ctx->pat;
    const int nb = (int)ctx->buckets.size();
    int max_point = 0;
    for (int i = 0; i < n_points; ++i) max_point = std::max(max_point, point_ids[i] + 1);
    std::map<int, bool> key_pat;
    size_t pat_bytes = 0;
    if (!pat.units.empty())
        for (const auto& kr : key_rows) {
            const int key = kr.first;
            if (!can_share(key)) continue;
            long long fams = 0;
            size_t bytes = 0;
            for (auto& bc : bucket_class) {
                if (bc.first != key || pat.first_unit[bc.second] == pat.first_unit[bc.second + 1]) continue;
                fams += (long long)ctx->buckets[bc.second].count * n_points;
                for (int u = pat.first_unit[bc.second]; u < pat.first_unit[bc.second + 1]; ++u)
                    bytes += 8 * (size_t)pat.units[u].n * max_point * pat.units[u].xs;
            }
            if (fams < kPatternWork || pat_bytes + bytes > kPatternBytes) continue;
            key_pat[key] = true;
            pat_bytes += bytes;
        }
    std::vector<TileDesc> tiles;
    std::vector<SegDesc> segs;
    int prev_key = -1;
    for (auto& bc : bucket_class) {
        const BucketHost& bk = ctx->buckets[bc.second];
        if (pp.classes.empty() || bc.first != prev_key) {
            KernelClass kc{};
            kc.key = bc.first;
            kc.begin = kc.end = (int)tiles.size();
            kc.fams = key_fams[bc.first];
            kc.seg_begin = kc.seg_end = (int)segs.size();
            kc.pat = key_pat.count(bc.first) > 0;
            kc.n_cols = kc.pat ? 0 : ctx->n_leaves;
            kc.n_slots = kc.pat ? 0 : ctx->n_slots;
            kc.n_slots_lane = kc.pat ? 0 : ctx->n_slots_lane;
            kc.n_slots_hot = kc.pat ? 0 : ctx->n_slots_hot;
            if (kc.pat) {
                auto add = [&](const PatternProg& pr) {
                    kc.max_pat = std::max(kc.max_pat, pr.n_pat);
                    kc.n_cols = std::max(kc.n_cols, pr.n_cols);
                    kc.n_slots = std::max(kc.n_slots, pr.n_slots);
                    kc.n_slots_lane = std::max(kc.n_slots_lane, pr.n_slots_reuse);
                    kc.n_slots_hot = std::max(kc.n_slots_hot, pr.n_slots_hot);
                };
                for (auto& o : bucket_class) {
                    if (o.first != bc.first) continue;
                    add(pat.main[o.second]);
                    for (int u = pat.first_unit[o.second]; u < pat.first_unit[o.second + 1]; ++u) add(pat.units[u].prog);
                }
            }
            // the kernel is chosen here: its tiles carry 64 families (per
            // lane) or 16 (matrix cores)
            kc.plain = path == CAFE_GPU_PATH_PLAIN64 || bc.first > kMfmaMaxTiles;
            kc.f64 = kc.plain || path == CAFE_GPU_PATH_BATCHED64;
            kc.lane_rows = kc.plain ? 0 : lane_rows_of(bc.first);
            if (kc.f64)
                kc.fb = f64_shape(key_nt[bc.first], kc.fams / kTile, kc.n_slots, kc.n_cols, ctx->n_cu).fb;
            kc.fb = kc.lane_rows > 0 ? 1
                  : kc.f64           ? kc.fb
                                     : builtin_fb32(path, bc.first, n_mfma_keys == 1, key_fams[bc.first], ctx->n_cu);
            if (const cafe_gpu_ctx::TuneEntry* te = kc.plain ? nullptr : find_tuning(ctx, path, bc.first, plan_classes)) {
                MfmaShape probe;
                if (tuned_mfma_shape(ctx, path, *te, kc, bc.first, bc.first, probe)) {
                    kc.lane_rows = 0;
                    kc.fb = probe.fb;
                }
            }
            if (kc.lane_rows > 0) {
                kc.lane_slots = kc.n_slots_hot + 1;   // the stored slots and the hot array
                const PruneParams none{};
                HIP_OR_FAIL(lane_dispatch(kc.lane_rows, kc.lane_slots, 0, lane_shm(kc.n_cols), none, nullptr,
                                          &kc.lane_per_cu));
                if (kc.lane_per_cu == 0) kc.lane_rows = 0;   // no instance fits: matrix-core kernel
            }
            pp.classes.push_back(kc);
            prev_key = bc.first;
        }
        KernelClass& kc = pp.classes.back();
        const int ci = (int)pp.classes.size() - 1;
        kc.nt = std::max(kc.nt, tiles_of(bk));
        kc.slot_tiles = std::max(kc.slot_tiles, round_up(bk.B + 1, kTile) / kTile);
        const int tw = kc.lane_rows > 0 ? 64 : kTile * kc.fb;   // families per tile
        for (int pi = 0; pi < n_points; ++pi) {
            for (int f0 = 0; f0 < bk.count; f0 += tw)
                tiles.push_back(TileDesc{bc.second, point_ids[pi], f0, std::min(tw, bk.count - f0)});
            for (int f0 = 0; f0 < bk.count; f0 += kSegChunk)
                segs.push_back(SegDesc{bc.second, point_ids[pi], ci, f0});
        }
        kc.r16 += n_points * ((bk.count + kTile - 1) / kTile);
        kc.end = (int)tiles.size();
        kc.seg_end = (int)segs.size();
    }
    const int n_cls = (int)pp.classes.size();
    // a shape over patterns that does not fit is no error: its class leaves them below
    auto fit = [](const KernelClass& kc, hipError_t e, MfmaShape& sh) {
        if (e == hipSuccess || !kc.pat) return e;
        (void)hipGetLastError();
        sh.per_cu = 0;
        return hipSuccess;
    };
    for (auto& kc : pp.classes) {
        if (kc.f64) {
            pp.has_f64 = true;
            kc.s64 = f64_shape(kc.nt, kc.fams / kTile, kc.n_slots, kc.n_cols, ctx->n_cu);
            if (int rc = f64_occupancy(kc.s64)) return rc;
            continue;
        }
        kc.s32 = kc.fb == 2 ? mfma_shape_fb2(kc.nt)
               : kc.nt >= 2 && kc.nt <= 16 && mfma_fams < 32LL * ctx->n_cu ? mfma_shape_few(kc.nt)
                                                                         : mfma_shape(kc.nt);
        kc.r64 = f64_shape(kc.nt, 1, ctx->n_slots, ctx->n_leaves, ctx->n_cu);
        place_partials(kc.s32, kc.n_slots, kc.slot_tiles, kc.n_cols, kc.max_pat);
        HIP_OR_FAIL(fit(kc, mfma_occupancy(kc.s32, &kc.s32.per_cu), kc.s32));
        if (int rc = f64_occupancy(kc.r64)) return rc;
        if (path == CAFE_GPU_PATH_BATCHED16 && kc.nt <= kF16MaxTiles) {
            // the program whose outputs reuse a child's slot (the store's
            // maxima exchange orders all reads before the writes)
            kc.s16 = mfma_shape(kc.nt);
            place_partials16(kc.s16, kc.n_slots_lane, kc.slot_tiles, kc.n_cols, kc.max_pat);
            const PruneParams none{};
            HIP_OR_FAIL(fit(kc, f16_dispatch(kc.s16, 0, none, nullptr, &kc.s16.per_cu), kc.s16));
            if (kc.s16.per_cu == 0 && kc.s16.lds) {   // LDS does not fit: global scratch
                kc.s16.lds = false;
                kc.s16.shm = f16_meta_only(kc.s16, kc.n_slots_lane, kc.n_cols, kc.max_pat);
                HIP_OR_FAIL(fit(kc, f16_dispatch(kc.s16, 0, none, nullptr, &kc.s16.per_cu), kc.s16));
            }
        }
    }
    // Measured shapes from the context's tuning table replace the built-in
    // ones where they exist and fit the class.
    for (auto& kc : pp.classes)
        if (!kc.plain)
            if (int rc = apply_tuning(ctx, path, kc, plan_classes)) return rc;
    // A pattern column takes two to four times a leaf's LDS (exponent and bound
    // beside the offset): a tree of many two-leaf clades can be too wide for a
    // CU that way (from about 640 taxa with 32-family tiles) and still fit with
    // its leaves.
    for (auto& kc : pp.classes) {
        if (!kc.pat || kc.lane_rows > 0) continue;
        const bool f16 = !kc.f64 && path == CAFE_GPU_PATH_BATCHED16 && kc.nt <= kF16MaxTiles;
        if ((kc.f64 ? kc.s64 : f16 ? kc.s16 : kc.s32).per_cu > 0) continue;
        std::set<int> out = whole;
        out.insert(kc.key);
        return plan_over(ctx, b, path, model, n_points, point_ids, root_out, root_stride, pp, out);
    }
    // Main-pass classes to side streams, longest first onto the least loaded
    // stream.  Estimated cost: contraction work (tiles x nt^2, plus a per-tile
    // overhead) and a floor for the serial chain of one large tile; a
    // per-lane class counts a quarter (it runs unpadded at the full vector
    // rate beside the matrix-core classes).  On the uneven-size workload that
    // was 3.46 ms per step against 3.48 at the full count and 3.52 at half
    // while every class ran whole programs; over shared subtrees, which
    // shorten the per-lane classes most, it is 2.75 against 2.66 and 2.69.
    {
        std::vector<double> cost(n_cls);
        std::vector<int> order(n_cls);
        for (int ci = 0; ci < n_cls; ++ci) {
            const KernelClass& kc = pp.classes[ci];
            const double tiles = kc.r16;   // in 16-family tiles
            cost[ci] = (tiles * (kc.nt * kc.nt + 8.0) + 2500.0 * kc.nt * kc.nt) * (kc.lane_rows > 0 ? 0.25 : 1.0);
            order[ci] = ci;
        }
        std::stable_sort(order.begin(), order.end(), [&](int a, int b2) { return cost[a] > cost[b2]; });
        std::vector<double> load(kSideStreams, 0.0);
        for (int ci : order) {
            const int k = (int)(std::min_element(load.begin(), load.end()) - load.begin());
            pp.classes[ci].stream = k;
            load[k] += cost[ci];
        }
        pp.main_order = order;
        // the stream that frees up first: that of the per-lane classes (at
        // full VALU rate they end well before their estimate), else the one
        // with the least estimated work
        pp.light_stream = (int)(std::min_element(load.begin(), load.begin() + std::max(1, std::min(kSideStreams, n_cls))) -
                                load.begin());
        for (int ci : order)
            if (pp.classes[ci].lane_rows > 0) {
                pp.light_stream = pp.classes[ci].stream;
                break;
            }
    }
    pp.n_tiles = (int)tiles.size();
    pp.class_counts.assign(n_cls + 4, 0);
    for (int i = 0; i < n_cls; ++i) pp.class_counts[i] = pp.classes[i].end - pp.classes[i].begin;
    // the units: bucket-table entries after the buckets', columns, and per
    // class and level their tiles (lists of representatives)
    std::vector<BucketDev>& bd = b.bucket_h;
    std::vector<UnitDev> units(pat.units.size(), UnitDev{});
    long long n64 = 0, n32 = 0, n_meta = 0;
    if (pat_bytes > 0) {
        auto set_prog = [](BucketDev& d, const PatternProg& pr) {
            d.step0 = pr.step0;
            d.n_steps = pr.n_steps;
            d.col0 = pr.col0;
            d.n_cols = pr.n_cols;
            d.n_pat = pr.n_pat;
        };
        bd.resize(nb);
        for (int i = 0; i < nb; ++i) set_prog(bd[i], pat.main[i]);
        for (int u = 0; u < (int)pat.units.size(); ++u) {
            BucketDev d = bd[pat.units[u].bucket];
            set_prog(d, pat.units[u].prog);
            d.out = u;
            d.list0 = pat.units[u].list0;
            d.fam_begin = 0;
            d.count = pat.units[u].n;
            bd.push_back(d);
        }
        for (auto& kc : pp.classes) {
            if (!kc.pat) continue;
            const int tw = kc.lane_rows > 0 ? 64 : kTile * kc.fb;
            std::vector<std::vector<TileDesc>> level;
            for (auto& bc : bucket_class) {
                if (bc.first != kc.key) continue;
                for (int u = pat.first_unit[bc.second]; u < pat.first_unit[bc.second + 1]; ++u) {
                    const PatternUnit& pu = pat.units[u];
                    UnitDev& ud = units[u];
                    ud.n = pu.n;
                    ud.xs = pu.xs;
                    long long& top = kc.f64 ? n64 : n32;
                    ud.x0 = top;
                    top += (long long)pu.n * max_point * ud.xs;
                    ud.m0 = n_meta;
                    n_meta += (long long)pu.n * max_point;
                    if ((int)level.size() <= pu.level) level.resize(pu.level + 1);
                    for (int pi = 0; pi < n_points; ++pi)
                        for (int i0 = 0; i0 < pu.n; i0 += tw)
                            level[pu.level].push_back(TileDesc{nb + u, point_ids[pi], pu.list0 + i0, -std::min(tw, pu.n - i0)});
                }
            }
            for (auto& l : level) {
                kc.levels.push_back(KernelClass::Level{(int)tiles.size(), (int)l.size(), (int)pp.class_counts.size()});
                pp.class_counts.push_back((int)l.size());
                tiles.insert(tiles.end(), l.begin(), l.end());
            }
        }
    }
    // [0, n_cls] offsets of the 16-family recompute lists (room for all of a
    // class's families in 16-family tiles)
    std::vector<int> class_off(n_cls + 1, 0);
    for (int i = 0; i < n_cls; ++i) {
        pp.classes[i].r_begin = class_off[i];
        class_off[i + 1] = class_off[i] + pp.classes[i].r16;
    }
    pp.r16_total = class_off[n_cls];
    pp.n_segs = (int)segs.size();

    HIP_OR_FAIL(b.fb_tiles.ensure(sizeof(TileDesc) * (size_t)std::max(1, pp.r16_total)));
    HIP_OR_FAIL(b.fb_count.ensure(sizeof(int) * (n_cls + 2)));
    HIP_OR_FAIL(b.fam_list.ensure(sizeof(int) * (size_t)max_point * (size_t)ctx->F));
    b.put(b.tiles, tiles.data(), sizeof(TileDesc) * tiles.size());
    b.put(b.ntiles, pp.class_counts.data(), sizeof(int) * pp.class_counts.size());
    b.put(b.segs, segs.data(), sizeof(SegDesc) * pp.n_segs);
    b.put(b.class_off, class_off.data(), sizeof(int) * (n_cls + 1));
    b.put(b.buckets, bd.data(), sizeof(BucketDev) * bd.size());
    if (pat_bytes > 0) {
        b.put(b.units, units.data(), sizeof(UnitDev) * units.size());
        HIP_OR_FAIL(b.cols_x.ensure(sizeof(double) * n64 + sizeof(float) * n32 * (path == CAFE_GPU_PATH_BATCHED16 ? 2 : 1)));
        HIP_OR_FAIL(b.cols_meta.ensure((sizeof(double) + sizeof(int)) * n_meta));
    }
    if (int rc = commit_inputs(ctx, b)) return rc;

    // Global scratch: per class and pass (classes of one pass run
    // concurrently, passes one after another).
    size_t main_sz = 0, r64_sz = 0;
    for (int ci = 0; ci < n_cls; ++ci) {
        KernelClass& kc = pp.classes[ci];
        int n = pp.class_counts[ci];
        for (const auto& l : kc.levels) n = std::max(n, l.n);
        size_t mb = 0;
        if (kc.f64) mb = f64_scratch_bytes(kc.s64, kc.n_slots, kc.nt, pp.grid(kc.s64, n));
        else if (kc.lane_rows > 0) mb = 0;
        else if (path == CAFE_GPU_PATH_BATCHED16 && kc.nt <= kF16MaxTiles) mb = f16_scratch_bytes(kc.s16, kc.n_slots_lane, kc.slot_tiles, pp.grid(kc.s16, n));
        else mb = mfma_scratch_bytes(kc.s32, kc.n_slots, kc.slot_tiles, pp.grid(kc.s32, n));
        kc.off_main = main_sz;
        main_sz += align256(mb);
        if (!kc.f64) {
            kc.off_r64 = r64_sz;
            r64_sz += align256(f64_scratch_bytes(kc.r64, ctx->n_slots, kc.nt, pp.grid(kc.r64, kc.r16)));
            if (!kc.r64.lds) {
                const size_t tile = sizeof(double) * kTile * ctx->ops.size() * f64_level_stride(kc.nt);
                kc.level_tiles = (int)std::min<size_t>(std::min(kLevelTiles, kc.r16), kLevelBytes / tile);
                kc.off_level = r64_sz;
                r64_sz += align256(tile * kc.level_tiles);
            }
        }
    }
    for (auto& kc : pp.classes) {
        kc.off_r64 += main_sz;
        kc.off_level += main_sz;
    }
    HIP_OR_FAIL(b.scratch.ensure(std::max<size_t>(main_sz + r64_sz, 256)));

    PruneParams& p = pp.base;
    p.buckets = b.buckets.as<BucketDev>();
    p.steps = ctx->d_steps.as<StepDev>();
    p.n_steps = ctx->n_steps;
    p.n_leaves = ctx->n_leaves;
    p.n_nodes = ctx->n_nodes;
    p.node_slot = b.node_slot.as<int>();
    p.counts_T = ctx->d_counts.as<int>();
    p.F = ctx->F;
    p.perm = ctx->d_perm.as<int>();
    p.mt64 = ctx->mt64.as<double>();
    p.mt32 = ctx->mt32.as<float>();
    p.band = ctx->band32.as<int>();
    p.band_stride = ctx->Np / kTile;
    p.slot_elems = ctx->slot_elems;
    p.Np = ctx->Np;
    p.leaf64 = ctx->n_dev ? ctx->mt64e.as<double>() : ctx->mt64.as<double>();
    p.leaf32 = ctx->n_dev ? ctx->mt32e.as<float>() : ctx->lf32.as<float>();
    p.cm32 = ctx->lf32.as<float>();
    p.n_dev = ctx->n_dev;
    p.prior64 = b.prior64.as<double>();
    p.model = model;
    p.out_val = b.val.as<double>();
    p.out_flag = b.flag.as<int>();
    p.root_out = root_out;
    p.root_stride = root_stride;
    p.fam_list = b.fam_list.as<int>();
    p.vec_exp = 120 / std::max(1, ctx->max_children) - kMatExp;
    // split FP16: a factor is below 2^(kMatExp16 + a) and a node's product of
    // max_children factors stays inside FP32; vectors stay inside FP16
    p.vec_exp16 = std::min(15, 126 / std::max(1, ctx->max_children) - kMatExp16);
    if (path == CAFE_GPU_PATH_BATCHED16) {
        const size_t n16 = sizeof(_Float16) * (size_t)ctx->slot_elems * ctx->capacity;
        HIP_OR_FAIL(ctx->mt16h.ensure(n16));
        HIP_OR_FAIL(ctx->mt16l.ensure(n16));
        pp.n_split = ctx->capacity;
    }
    p.mt16h = ctx->mt16h.as<_Float16>();
    p.mt16l = ctx->mt16l.as<_Float16>();
    p.scratch = b.scratch.p;
    p.n_slots = ctx->n_slots;
    p.zero = 0;
    p.units = nullptr;   // (set for the launches of the classes that use them)
    p.max_pat = 0;
    if (pat_bytes > 0) {
        p.cols = pat.cols.as<ColDev>();
        p.x64 = b.cols_x.as<double>();
        p.x32 = (float*)(p.x64 + n64);
        p.xe32 = p.x32 + n32;
        p.xm_c = b.cols_meta.as<double>();
        p.xm_e = (int*)(p.xm_c + n_meta);
    }
    return CAFE_GPU_OK;
}

// The columns are what an evaluation can do without: where the device has no
// room for them (or for the rest beside them), every class runs its whole
// program.
int plan_prune(cafe_gpu_ctx* ctx, EvalBufs& b, int path, int model, int n_points, const int* point_ids,
               double* root_out, int root_stride, PrunePlan& pp)
{
    const size_t block = b.block.size(), views = b.views.size();
    std::set<int> whole;
    for (;;) {
        const int rc = plan_over(ctx, b, path, model, n_points, point_ids, root_out, root_stride, pp, whole);
        const size_t n = whole.size();
        for (const auto& kc : pp.classes)
            if (kc.pat) whole.insert(kc.key);
        if (rc != CAFE_GPU_ENOMEM || whole.size() == n) return rc;
        (void)hipGetLastError();
        b.cols_x.release();
        b.cols_meta.release();
        b.block.resize(block);   // (the tables put before)
        b.views.resize(views);
        b.bucket_h.resize(ctx->buckets.size());
    }
}

// Enqueues the pruning sequence: the main path per size class, then
// (device-side lists, no host round trip) the FP64 recompute of the families
// a reduced path's bound did not certify.  late_build (when set) enqueues the
// FP64 pool, which only the recompute stages read: it runs on the side stream
// expected to finish its main-pass work first, after that work.
int enqueue_prune(cafe_gpu_ctx* ctx, EvalBufs& b, const PrunePlan& pp, hipStream_t st, hipEvent_t ev_main,
                  hipEvent_t ev_fb, bool concurrent, const std::vector<hipEvent_t>* cls_ev = nullptr,
                  const std::function<int(hipStream_t)>* late_build = nullptr)
{
    const int n_cls = (int)pp.classes.size();
    int* d_cnt = b.ntiles.as<int>();
    int* fbc = b.fb_count.as<int>();
    char* scratch = (char*)pp.base.scratch;
    HIP_OR_FAIL(launch_fill_zero(b.fb_count.p, sizeof(int) * (n_cls + 2), st));
    // BATCHED16 reads the FP16 halves of the FP32 matrices
    if (pp.path == CAFE_GPU_PATH_BATCHED16)
        HIP_OR_FAIL(launch_split_f16(ctx->mt32.as<float>(), ctx->mt16h.as<_Float16>(), ctx->mt16l.as<_Float16>(),
                                     ctx->Np, ctx->slot_elems, pp.n_split, st));

    // Two stages per size class: the main pass, then (reduced paths) the FP64
    // recompute of the families the bound did not certify, which packs its
    // class's flagged families into a list sized on the device and prunes it.
    TileDesc* fb64 = b.fb_tiles.as<TileDesc>();
    const int* coff = b.class_off.as<int>();
    const int fam_off = pp.fam_count_off();
    const SegDesc* segs = b.segs.as<SegDesc>();
    auto stage_main = [&](int ci, hipStream_t s) -> int {
        const KernelClass& kc = pp.classes[ci];
        const int n = pp.class_counts[ci];
        PruneParams q = pp.base;
        q.tiles = b.tiles.as<TileDesc>() + kc.begin;
        q.n_tiles_dev = d_cnt + ci;
        q.slot_tiles = kc.slot_tiles;
        q.scratch = scratch + kc.off_main;
        q.n_slots = kc.n_slots;
        const bool lane = kc.lane_rows > 0;   // BATCHED32 / BATCHED16: small vectors, one family per lane
        if (lane) {
            q.steps = ctx->d_steps_hot.as<StepDev>();
            q.n_slots = kc.n_slots_hot;
        }
        const bool f16 = !kc.f64 && !lane && pp.path == CAFE_GPU_PATH_BATCHED16 && kc.nt <= kF16MaxTiles;
        if (f16) {
            q.steps = ctx->d_steps_lane.as<StepDev>();
            q.n_slots = kc.n_slots_lane;
        }
        if (kc.f64) q.slot_tiles = kc.nt;
        auto launch = [&](const PruneParams& a, int tiles) -> int {
            if (kc.f64) HIP_OR_FAIL(f64_dispatch(kc.s64, pp.grid(kc.s64, tiles), a, s, nullptr));
            else if (lane)
                HIP_OR_FAIL(lane_dispatch(kc.lane_rows, kc.lane_slots,
                                          pp.grid_lane(kc.lane_per_cu, tiles, kc.lane_grid_mult), lane_shm(kc.n_cols), a,
                                          s, nullptr));
            else if (f16) HIP_OR_FAIL(f16_dispatch(kc.s16, pp.grid(kc.s16, tiles), a, s, nullptr));
            else HIP_OR_FAIL(launch_prune_mfma(kc.s32, pp.grid(kc.s32, tiles), a, s));
            return CAFE_GPU_OK;
        };
        if (kc.pat) {
            q.units = b.units.as<UnitDev>();
            q.max_pat = kc.max_pat;
            q.n_leaves = kc.n_cols;
            q.steps = (lane ? ctx->pat.steps_hot : f16 ? ctx->pat.steps_reuse : ctx->pat.steps).as<StepDev>();
            q.counts_T = ctx->pat.ext.as<int>();
            for (const auto& l : kc.levels) {
                PruneParams a = q;
                a.tiles = b.tiles.as<TileDesc>() + l.begin;
                a.n_tiles_dev = d_cnt + l.count_at;
                a.fam_list = ctx->pat.reps.as<int>();
                if (int rc = launch(a, l.n)) return rc;
            }
        }
        // (final FP64 values: nothing to recompute)
        if (kc.f64 && !kc.plain) q.near_floor = fbc + fam_off + 1;
        return launch(q, n);
    };
    auto stage_r64 = [&](int ci, hipStream_t s) -> int {
        const KernelClass& kc = pp.classes[ci];
        if (kc.f64) return CAFE_GPU_OK;
        HIP_OR_FAIL(launch_pack(segs + kc.seg_begin, kc.seg_end - kc.seg_begin, b.buckets.as<BucketDev>(),
                                pp.base.perm, b.flag.as<int>(), pp.base.F, kFlagRecompute64, b.fam_list.as<int>(),
                                fb64, coff, fbc, fbc + fam_off, kTile, s));
        PruneParams q = pp.base;
        q.tiles = fb64 + kc.r_begin;
        q.n_tiles_dev = fbc + ci;
        q.slot_tiles = kc.nt;
        q.scratch = scratch + kc.off_r64;
        q.near_floor = fbc + fam_off + 1;
        // short lists level by level (which of the two works is decided on the device)
        if (kc.level_tiles > 0) {
            PruneParams a = q;
            a.steps = ctx->d_steps_level.as<StepDev>();
            a.scratch = scratch + kc.off_level;
            HIP_OR_FAIL(launch_f64_levels(kc.nt, kc.level_tiles, ctx->d_op_steps.as<int>(), ctx->level_ops.data(),
                                          (int)ctx->level_ops.size() - 1, a, s));
            q.skip_tiles = kc.level_tiles;
        }
        HIP_OR_FAIL(f64_dispatch(kc.r64, pp.grid(kc.r64, kc.r16), q, s, nullptr));
        return CAFE_GPU_OK;
    };

    // Stage by stage over the classes: every main pass, then every FP64
    // recompute.
    // When concurrent, the classes of one stage run on the side streams (the
    // main passes on their longest-first assignment, the recomputes round
    // robin in that order: measured 1.5% faster per step than placing the
    // recomputes by their vectors' length) and st waits for all of them
    // before the next stage: a recompute is a latency-bound chain on a few
    // tiles, and beside a main pass it would slow that pass down.
    // (a single class still takes two streams when the FP64 pool is to be built
    // beside its main pass: 2,000 families 221 -> 193 us a step)
    const int S = concurrent ? std::min((int)ctx->side.size(), std::max(n_cls, late_build ? 2 : 0)) : 0;
    const int light = n_cls == 1 ? S - 1 : pp.light_stream;
    if (late_build && S <= 1)
        if (int rc = (*late_build)(st)) return rc;
    using Launch = std::function<int(int, hipStream_t)>;
    auto stage = [&](int idx, const Launch& launch) -> int {
        if (S <= 1) {
            for (int ci = 0; ci < n_cls; ++ci) {
                if (cls_ev && idx == 0) HIP_OR_FAIL(hipEventRecord((*cls_ev)[ci], st));
                if (int rc = launch(ci, st)) return rc;
            }
            if (cls_ev && idx == 0) HIP_OR_FAIL(hipEventRecord((*cls_ev)[n_cls], st));
            return CAFE_GPU_OK;
        }
        hipEvent_t* ev = ctx->join_ev.data() + idx * (kSideStreams + 1);
        HIP_OR_FAIL(hipEventRecord(ev[0], st));
        for (int k = 0; k < S; ++k) HIP_OR_FAIL(hipStreamWaitEvent(ctx->side[k], ev[0], 0));
        for (int i = 0; i < n_cls; ++i) {
            const int ci = pp.main_order[i];
            const int k = idx == 0 ? pp.classes[ci].stream % S : i % S;
            if (int rc = launch(ci, ctx->side[k])) return rc;
        }
        if (idx == 0 && late_build)
            if (int rc = (*late_build)(ctx->side[light % S])) return rc;
        for (int k = 0; k < S; ++k) {
            HIP_OR_FAIL(hipEventRecord(ev[1 + k], ctx->side[k]));
            HIP_OR_FAIL(hipStreamWaitEvent(st, ev[1 + k], 0));
        }
        return CAFE_GPU_OK;
    };
    if (int rc = stage(0, stage_main)) return rc;
    if (ev_main) HIP_OR_FAIL(hipEventRecord(ev_main, st));
    if (pp.path == CAFE_GPU_PATH_BATCHED32 || pp.path == CAFE_GPU_PATH_BATCHED16)
        if (int rc = stage(1, stage_r64)) return rc;
    if (ev_fb) HIP_OR_FAIL(hipEventRecord(ev_fb, st));
    return CAFE_GPU_OK;
}

int enqueue_finalize(cafe_gpu_ctx* ctx, EvalBufs& b, int model, int T, int K, hipStream_t st)
{
    HIP_OR_FAIL(launch_finalize(model, T, K, ctx->F, b.val.as<double>(), b.flag.as<int>(), b.catp.as<double>(),
                                b.lnl.as<double>(), b.cat.as<double>(), b.post.as<double>(), b.fail.as<int>(),
                                b.total.as<double>(), st));
    return CAFE_GPU_OK;
}

int copy_results(cafe_gpu_ctx* ctx, EvalBufs& b, const PrunePlan& pp, int model, int T, int K, double* lnl,
                 double* cat, double* post, double* total, long long* n_fallback)
{
    const size_t TF = (size_t)T * ctx->F;
    int h[2] = {0, 0};
    std::vector<Fetch> list;
    if (total) list.push_back({total, b.total.p, sizeof(double) * T});
    if (n_fallback) list.push_back({h, b.fb_count.as<int>() + pp.fam_count_off(), sizeof(int) * 2});
    if (lnl) list.push_back({lnl, b.lnl.p, sizeof(double) * TF});
    if (cat && model == CAFE_GPU_MODEL_GAMMA) list.push_back({cat, b.cat.p, sizeof(double) * TF * K});
    if (post && model == CAFE_GPU_MODEL_GAMMA) list.push_back({post, b.post.p, sizeof(double) * TF * K});
    if (int rc = fetch(ctx, list)) return rc;
    if (n_fallback) *n_fallback = (long long)h[0] + (long long)h[1];
    return CAFE_GPU_OK;
}

double elapsed_ms(hipEvent_t a, hipEvent_t b)
{
    float ms = 0;
    if (hipEventElapsedTime(&ms, a, b) != hipSuccess) return 0.0;
    return ms;
}

// Pupko reconstruction of families f0 .. f0+nf-1 (cafe_gpu_reconstruct).  The
// device working memory -- program, child lists, prior, the resident families'
// list and state rows, the error flag, the table of block maxima and then per
// family of a launch the L rows -- comes from the context's grow-only buffers
// when `fixed` is null, else from the fixed region [fixed, fixed +
// fixed_bytes), in which case nothing is allocated: launches are sized to fit
// the region and a family that does not fit on its own is rejected.
int reconstruct_impl(cafe_gpu_ctx* ctx, const int* node_slot, const double* prior, int B, int R, int f0, int nf,
                     int* states, char* fixed, size_t fixed_bytes)
{
    if (int rc = check_ctx(ctx)) return rc;
    if (!node_slot || !prior || !states) return fail(CAFE_GPU_EINVAL, "null argument");
    if (ctx->n_nodes == 0 || ctx->F == 0) return fail(CAFE_GPU_ESTATE, "tree and families must be set first");
    if (ctx->N == 0) return fail(CAFE_GPU_ESTATE, "matrix_reset has not been called");
    if (B < 0 || R < 0 || B + 1 > ctx->N) return fail(CAFE_GPU_EINVAL, "bounds B=%d R=%d do not fit matrices of %d", B, R, ctx->N);
    if (f0 < 0 || nf < 0 || f0 + nf > ctx->F) return fail(CAFE_GPU_EINVAL, "family range out of range");
    if (ctx->n_leaves != ctx->tree_leaves)
        return fail(CAFE_GPU_EINVAL, "families have %d leaves, tree has %d", ctx->n_leaves, ctx->tree_leaves);
    if (nf == 0) return CAFE_GPU_OK;
    const int n = ctx->n_nodes;
    const int Rr = std::min(B, R) + 1;   // gene_family_reconstructor.cpp:149-151
    const int Lp = B + 1;
    auto up = [](size_t b) { return (b + 255) / 256 * 256; };
    if (fixed) {
        // the documented limit: a family's rows at 12 bytes per node and size,
        // its list entry and states, and 28 bytes of program per node (what is
        // laid out below stays under it)
        const size_t per = sizeof(int) + sizeof(int) * (size_t)n +
                           (size_t)Lp * ((size_t)n * (sizeof(double) + sizeof(int)) + sizeof(double));
        const size_t head = up((size_t)20 * n) + up(sizeof(int) * std::max(1, n - 1)) + up(sizeof(int) * n) +
                            up(sizeof(double) * Rr) + 4 * 256;
        if (fixed_bytes <= head || (fixed_bytes - head) / per < 1)
            return fail(CAFE_GPU_EINVAL,
                        "one family of %d nodes with vectors of %d sizes needs %zu bytes of scratch; the fixed "
                        "scratch holds %zu",
                        n, Lp, head + per, fixed_bytes);
    }
    // the interior nodes, children first (depth first, children in increasing
    // index)
    std::vector<std::vector<int>> kids(n);
    int root = -1;
    for (int i = 0; i < n; ++i) {
        if (ctx->parent_h[i] < 0) root = i;
        else kids[ctx->parent_h[i]].push_back(i);
    }
    std::vector<ReconNode> prog;
    std::vector<ReconKid> kid_list;
    std::vector<int> place(n, -1);
    std::vector<std::pair<int, int>> stack{{root, 0}};
    while (!stack.empty()) {
        auto& top = stack.back();
        const int u = top.first;
        if (top.second < (int)kids[u].size()) {
            stack.push_back({kids[u][top.second++], 0});
            continue;
        }
        stack.pop_back();
        int slot = -1;
        if (u != root) {
            slot = node_slot[u];
            if (slot < 0 || slot >= ctx->capacity)
                return fail(CAFE_GPU_EINVAL, "node %d: matrix slot %d outside the pool", u, slot);
            if (!ctx->built[slot])   // matrix_cache::get_matrix throws on a miss (matrix_cache.cpp:88-104)
                return fail(CAFE_GPU_ENOTFOUND, "node %d uses matrix slot %d, which is not built", u, slot);
        }
        if (ctx->leaf_col_h[u] >= 0) continue;
        place[u] = (int)prog.size();
        prog.push_back(ReconNode{u, (int)kid_list.size(), (int)kids[u].size(), slot});
        for (int c : kids[u]) {
            const int col = ctx->leaf_col_h[c];
            kid_list.push_back(ReconKid{col, node_slot[c], col >= 0 ? c : place[c], 0});
        }
    }
    if (kid_list.size() + 1 != (size_t)n)
        return fail(CAFE_GPU_EINVAL, "reconstruction program does not cover the tree (internal)");
    const int n_prog = (int)prog.size();
    // count-row (sorted) index of each caller family
    std::vector<int> sorted_of(ctx->F);
    for (int s = 0; s < ctx->F; ++s) sorted_of[ctx->perm[s]] = s;
    // Device layout: program | kids | prior | flag | table | families | states,
    // then the L rows.  `chunk` families run per launch (their L rows within 2
    // GB), `held` have their list entries and states on the device at once
    // (all of them, or the fixed region's launch).
    const size_t o_kids = up(sizeof(ReconNode) * n_prog);
    const size_t o_pri = o_kids + up(sizeof(ReconKid) * kid_list.size());
    const size_t o_err = o_pri + up(sizeof(double) * Rr);
    const size_t o_tab = o_err + 256;
    const size_t row_bytes = sizeof(double) * (size_t)(n_prog - 1) * (Lp + (Lp & 1));
    const size_t list_bytes = sizeof(int2) + sizeof(int) * (size_t)n;
    size_t tab_bytes = up(sizeof(double) * recon_table_doubles(n_prog, Lp));
    size_t held = (size_t)nf, chunk;
    if (fixed) {
        // the table where it leaves the families half of the region (without
        // it no block is skipped)
        if (o_tab + tab_bytes > fixed_bytes / 2) tab_bytes = 0;
        const size_t head = o_tab + tab_bytes + 2 * 256;
        size_t fit = fixed_bytes > head ? (fixed_bytes - head) / (row_bytes + list_bytes) : 0;
        if (fit >= (size_t)kRecFew) fit = fit / kRecFT * kRecFT;
        if (fit < 1) return fail(CAFE_GPU_EINVAL, "fixed scratch layout overflows (internal)");
        held = chunk = std::min(held, fit);
        if (chunk % kRecFT && chunk >= (size_t)kRecFew) held = chunk = chunk / kRecFT * kRecFT;
    } else {
        chunk = std::max<size_t>(64, ((size_t)2 << 30) / std::max<size_t>(row_bytes, 1) / kRecFT * kRecFT);
        chunk = std::min(chunk, (held + kRecFT - 1) / kRecFT * kRecFT);
    }
    const size_t o_fam = o_tab + tab_bytes;
    const size_t o_st = o_fam + up(sizeof(int2) * held);
    const size_t o_rows = o_st + up(sizeof(int) * held * n);
    char* base;
    double* rows;
    if (fixed) {
        base = fixed;
        rows = (double*)(fixed + o_rows);
        if (o_rows + chunk * row_bytes > fixed_bytes)
            return fail(CAFE_GPU_EINVAL, "fixed scratch layout overflows (internal)");
    } else {
        HIP_OR_FAIL(ctx->d_recon.ensure(o_rows));
        HIP_OR_FAIL(ctx->d_recon_scratch.ensure(std::max<size_t>(chunk * row_bytes, 256)));
        base = (char*)ctx->d_recon.p;
        rows = ctx->d_recon_scratch.as<double>();
    }
    const ReconNode* d_prog = (const ReconNode*)base;
    double* tab = tab_bytes ? (double*)(base + o_tab) : nullptr;
    hipStream_t st = ctx->stream;
    HIP_OR_FAIL(hipMemcpyAsync(base, prog.data(), sizeof(ReconNode) * prog.size(), hipMemcpyHostToDevice, st));
    HIP_OR_FAIL(hipMemcpyAsync(base + o_kids, kid_list.data(), sizeof(ReconKid) * kid_list.size(), hipMemcpyHostToDevice, st));
    HIP_OR_FAIL(hipMemcpyAsync(base + o_pri, prior, sizeof(double) * Rr, hipMemcpyHostToDevice, st));
    HIP_OR_FAIL(launch_fill_zero(base + o_err, sizeof(int), st));
    if (tab)
        HIP_OR_FAIL(launch_block_max(d_prog, n_prog, ctx->mt64.as<double>(), ctx->Np, ctx->slot_elems, Lp, tab, st));
    // large families first: their products fall off later, so they take several
    // times longer, and four of a size share a wave's matrix blocks
    int flag = 0;
    std::vector<int2> fams(held);
    std::vector<int> at(ctx->N + 1);
    for (size_t h0 = 0; h0 < (size_t)nf; h0 += held) {
        const size_t nh = std::min(held, (size_t)nf - h0);
        auto key = [&](size_t k) { return ctx->N - 1 - std::min(ctx->fam_max[f0 + h0 + k], ctx->N - 1); };
        std::fill(at.begin(), at.end(), 0);
        for (size_t k = 0; k < nh; ++k) ++at[key(k) + 1];
        for (int i = 0; i < ctx->N; ++i) at[i + 1] += at[i];
        for (size_t k = 0; k < nh; ++k) fams[at[key(k)]++] = int2{sorted_of[f0 + h0 + k], (int)k};
        HIP_OR_FAIL(hipMemcpyAsync(base + o_fam, fams.data(), sizeof(int2) * nh, hipMemcpyHostToDevice, st));
        for (size_t c0 = 0; c0 < nh; c0 += chunk)
            HIP_OR_FAIL(launch_reconstruct(d_prog, n_prog, (const ReconKid*)(base + o_kids), ctx->mt64.as<double>(),
                                           ctx->N, ctx->Np, ctx->slot_elems, tab, ctx->d_counts.as<int>(), ctx->F,
                                           (const int2*)(base + o_fam) + c0, (int)std::min(chunk, nh - c0),
                                           (const double*)(base + o_pri), B, Rr, rows, Lp, n,
                                           (int*)(base + o_st), (int*)(base + o_err), st));
        // (fams and the state rows are used again)
        if (int rc = fetch(ctx, {{states + h0 * n, base + o_st, sizeof(int) * nh * n}, {&flag, base + o_err, sizeof(int)}}))
            return rc;
    }
    if (flag) return fail(CAFE_GPU_EINVAL, "a leaf count is outside the matrices (N = %d)", ctx->N);
    return CAFE_GPU_OK;
}

}  // namespace

// One device-resident evaluation (see cafe_gpu_plan_* in cafe_gpu.h).
struct cafe_gpu_plan {
    cafe_gpu_ctx* ctx = nullptr;
    EvalBufs bufs;
    PrunePlan pp;
    int model = 0, path = 0, T = 0, K = 0, n_keys = 0, algo = 0;
    DevBuf d_keys;           // lambdas, then branch lengths
    double* lam() const { return d_keys.as<double>(); }
    double* t() const { return d_keys.as<double>() + n_keys; }
    DevBuf d_copies;         // per key: the FP32 copies the plan's kernels read (kCopy* bits)
    int copy_top = 0;        // kCopyColTop: rows and columns of the per-lane classes
    long long pool_gen = 0, input_gen = 0;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    bool graph_ok = false;
    hipEvent_t ev[5] = {};
    std::vector<hipEvent_t> cls_ev;   // around each main-pass class launch (profile runs)
    std::vector<double> cls_ms;       // their times in the last profile run
};

namespace {

// build -> prune -> recompute -> finalize; events bracket the phases when
// `timed` (ev[0] start, ev[1] after build, ev[2] after the main prune,
// ev[3] after the recompute passes, ev[4] after finalize)
int plan_enqueue(cafe_gpu_plan* pl, bool timed)
{
    cafe_gpu_ctx* ctx = pl->ctx;
    hipStream_t st = ctx->stream;
    // BATCHED32 reads the FP64 pool only in its recompute stages: concurrent
    // runs with the recurrence build make the FP32 pools first and the FP64
    // one beside the main pass
    const bool split = !timed && pl->algo != 0 && !pl->pp.has_f64 &&
                       (pl->pp.path == CAFE_GPU_PATH_BATCHED32 || pl->pp.path == CAFE_GPU_PATH_BATCHED16);
    if (timed) HIP_OR_FAIL(hipEventRecord(pl->ev[0], st));
    HIP_OR_FAIL(launch_build(pl->algo, pl->lam(), pl->t(), ctx->lg.as<double>(), pl->n_keys,
                             0, ctx->N, ctx->Np, ctx->slot_elems, split ? nullptr : ctx->mt64.as<double>(),
                             ctx->mt32.as<float>(), ctx->lf32.as<float>(), st, pl->d_copies.as<unsigned char>(),
                             pl->copy_top, ctx->band32.as<int>()));
    // the folded FP32 leaf pool is read by the reduced paths only
    const bool reduced = pl->pp.path == CAFE_GPU_PATH_BATCHED32 || pl->pp.path == CAFE_GPU_PATH_BATCHED16;
    if (int rc = enqueue_fold(ctx, 0, pl->n_keys, st, !split, reduced)) return rc;
    if (timed) HIP_OR_FAIL(hipEventRecord(pl->ev[1], st));
    const std::function<int(hipStream_t)> build64 = [&](hipStream_t s) -> int {
        HIP_OR_FAIL(launch_build(pl->algo, pl->lam(), pl->t(), ctx->lg.as<double>(),
                                 pl->n_keys, 0, ctx->N, ctx->Np, ctx->slot_elems, ctx->mt64.as<double>(), nullptr,
                                 nullptr, s, nullptr, 0, nullptr));
        return enqueue_fold(ctx, 0, pl->n_keys, s, true, false);
    };
    // profile runs issue the size classes one after another (standalone kernel
    // times); executions and the captured graph run them concurrently
    if (int rc = enqueue_prune(ctx, pl->bufs, pl->pp, st, timed ? pl->ev[2] : nullptr, timed ? pl->ev[3] : nullptr,
                               !timed, timed ? &pl->cls_ev : nullptr, split ? &build64 : nullptr))
        return rc;
    if (int rc = enqueue_finalize(ctx, pl->bufs, pl->model, pl->T, pl->K, st)) return rc;
    if (timed) HIP_OR_FAIL(hipEventRecord(pl->ev[4], st));
    return CAFE_GPU_OK;
}

// Captures plan_enqueue into a graph; returns false (stream left clean) if the
// runtime refuses any step of the capture.
bool plan_capture(cafe_gpu_plan* pl, bool timed)
{
    hipStream_t st = pl->ctx->stream;
    if (hipStreamBeginCapture(st, hipStreamCaptureModeRelaxed) != hipSuccess) return false;
    const int rc = plan_enqueue(pl, timed);
    hipGraph_t g = nullptr;
    const hipError_t e = hipStreamEndCapture(st, &g);
    if (rc != CAFE_GPU_OK || e != hipSuccess || !g) {
        if (g) (void)hipGraphDestroy(g);
        (void)hipGetLastError();
        return false;
    }
    hipGraphExec_t ex = nullptr;
    if (hipGraphInstantiate(&ex, g, nullptr, nullptr, 0) != hipSuccess) {
        (void)hipGraphDestroy(g);
        (void)hipGetLastError();
        return false;
    }
    pl->graph = g;
    pl->exec = ex;
    return true;
}

// A plan's graph and launch parameters point into the context's pool and
// input buffers and were sized for its tree, families and error model.
int plan_current(cafe_gpu_plan* pl)
{
    if (pl->pool_gen != pl->ctx->pool_gen)
        return fail(CAFE_GPU_ESTATE, "matrix pool was reset after the plan was made");
    if (pl->input_gen != pl->ctx->input_gen)
        return fail(CAFE_GPU_ESTATE, "tree, families or error-model shape changed after the plan was made");
    return CAFE_GPU_OK;
}

// Slots 0 .. n_keys-1 hold the plan's matrices once an execution is enqueued:
// the FP64 pool and the FP32 copies the plan reads.
void plan_mark_built(cafe_gpu_plan* pl)
{
    for (int i = 0; i < pl->n_keys; ++i) pl->ctx->built[i] = 2;
}

// The FP32 copies each key's users read in this plan: a leaf branch's
// matrix gives leaf columns (c-major); an interior branch's matrix is an
// MFMA A operand (row-major; also what the split-FP16 halves come from) or,
// in the per-lane classes, columns of the top-left lane_rows x lane_rows
// block (c-major).  FP64 paths read no FP32 copy.
void plan_copies(const cafe_gpu_ctx* ctx, const cafe_gpu_eval_desc* d, const PrunePlan& pp, int P, int n_keys,
                 std::vector<unsigned char>& copies, int& top)
{
    copies.assign(n_keys, 0);
    top = 0;
    if (pp.path != CAFE_GPU_PATH_BATCHED32 && pp.path != CAFE_GPU_PATH_BATCHED16) return;
    bool mfma = false;
    for (const auto& kc : pp.classes) {
        if (kc.lane_rows > 0) top = std::max(top, kc.lane_rows);
        else mfma = true;
    }
    const unsigned char interior = (mfma ? kCopyRow : 0) | (top > 0 ? kCopyColTop : 0);
    const int root = ctx->ops.back().node;
    for (long long i = 0; i < (long long)P * ctx->n_nodes; ++i) {
        const int node = (int)(i % ctx->n_nodes);
        if (node == root) continue;
        const int s = d->node_slot[i];
        if (s >= 0 && s < n_keys) copies[s] |= ctx->leaf_col_h[node] >= 0 ? kCopyCol : interior;
    }
}

}  // namespace

extern "C" {

int cafe_gpu_eval(cafe_gpu_ctx* ctx, const cafe_gpu_eval_desc* d, double* lnl, double* cat, double* post,
                  double* total, long long* n_fallback)
{
    if (int rc = check_ctx(ctx)) return rc;
    EvalBufs& b = ctx->eager;
    int P = 0;
    if (int rc = upload_eval_inputs(ctx, b, d, P)) return rc;
    std::vector<int> pts(P);
    std::iota(pts.begin(), pts.end(), 0);
    PrunePlan pp;
    if (int rc = plan_prune(ctx, b, d->path, d->model, P, pts.data(), nullptr, 0, pp)) return rc;
    HIP_OR_FAIL(hipEventRecord(ctx->ev[0], ctx->stream));
    if (int rc = enqueue_prune(ctx, b, pp, ctx->stream, ctx->ev[1], ctx->ev[2], true)) return rc;
    if (int rc = enqueue_finalize(ctx, b, d->model, d->n_trials, d->n_cat, ctx->stream)) return rc;
    HIP_OR_FAIL(hipEventRecord(ctx->ev[3], ctx->stream));
    if (int rc = copy_results(ctx, b, pp, d->model, d->n_trials, d->n_cat, lnl, cat, post, total, n_fallback))
        return rc;
    ctx->timings[1] = elapsed_ms(ctx->ev[0], ctx->ev[1]);
    ctx->timings[2] = elapsed_ms(ctx->ev[1], ctx->ev[2]);
    ctx->timings[3] = elapsed_ms(ctx->ev[2], ctx->ev[3]);
    return CAFE_GPU_OK;
}

int cafe_gpu_root_vectors(cafe_gpu_ctx* ctx, const cafe_gpu_eval_desc* d, int trial, int cat_k, int f0, int nf,
                          double* out)
{
    if (int rc = check_ctx(ctx)) return rc;
    EvalBufs& b = ctx->eager;
    int P = 0;
    if (int rc = upload_eval_inputs(ctx, b, d, P)) return rc;
    if (trial < 0 || trial >= d->n_trials || cat_k < 0 || cat_k >= d->n_cat)
        return fail(CAFE_GPU_EINVAL, "trial/category out of range");
    if (f0 < 0 || nf < 0 || f0 + nf > ctx->F || !out) return fail(CAFE_GPU_EINVAL, "family range out of range");
    int maxR = 0;
    for (auto& bk : ctx->buckets) maxR = std::max(maxR, bk.R);
    HIP_OR_FAIL(b.root.ensure(sizeof(double) * (size_t)ctx->F * maxR));
    const int point = trial * d->n_cat + cat_k;
    PrunePlan pp;
    if (int rc = plan_prune(ctx, b, d->path, d->model, 1, &point, b.root.as<double>(), maxR, pp)) return rc;
    if (int rc = enqueue_prune(ctx, b, pp, ctx->stream, nullptr, nullptr, true)) return rc;
    bool same = true;   // one R: the rows as they are
    for (auto& bk : ctx->buckets) same = same && bk.R == maxR;
    if (same)
        return fetch(ctx, {{out, b.root.as<double>() + (size_t)f0 * maxR, sizeof(double) * (size_t)nf * maxR}});
    std::vector<double> h((size_t)nf * maxR);
    if (int rc = fetch(ctx, {{h.data(), b.root.as<double>() + (size_t)f0 * maxR, sizeof(double) * h.size()}})) return rc;
    std::vector<int> famR(ctx->F);
    for (auto& bk : ctx->buckets)
        for (int k = 0; k < bk.count; ++k) famR[ctx->perm[bk.fam_begin + k]] = bk.R;
    size_t o = 0;
    for (int f = f0; f < f0 + nf; ++f)
        for (int j = 0; j < famR[f]; ++j) out[o++] = h[(size_t)(f - f0) * maxR + j];
    return CAFE_GPU_OK;
}

int cafe_gpu_reconstruct(cafe_gpu_ctx* ctx, const int* node_slot, const double* prior, int B, int R, int f0, int nf,
                         int* states)
{
    return reconstruct_impl(ctx, node_slot, prior, B, R, f0, nf, states, nullptr, 0);
}

int cafe_gpu_reconstruct_noalloc(cafe_gpu_ctx* ctx, const int* node_slot, const double* prior, int B, int R,
                                 int f0, int nf, int* states)
{
    if (int rc = check_ctx(ctx)) return rc;
    if (!ctx->fixed_scratch) return fail(CAFE_GPU_ESTATE, "fixed scratch not resolved for device %d", ctx->device);
    return reconstruct_impl(ctx, node_slot, prior, B, R, f0, nf, states, ctx->fixed_scratch, kFixedScratchBytes);
}

int cafe_gpu_tuning_set(cafe_gpu_ctx* ctx, int path, int tiles, int leaves, int kernel, int ntw, int w, int lds,
                        int grid_mult)
{
    if (!ctx) return fail(CAFE_GPU_EINVAL, "null context");
    if (path < CAFE_GPU_PATH_PLAIN64 || path > CAFE_GPU_PATH_BATCHED16 || tiles < 1 || leaves < 1 || kernel < 0 ||
        kernel > 2 || ntw < 0 || w < 0 || grid_mult < 0)
        return fail(CAFE_GPU_EINVAL, "invalid tuning entry");
    // the new entry applies to any plan: it replaces every entry of the class
    ctx->tuning.erase(std::remove_if(ctx->tuning.begin(), ctx->tuning.end(),
                                     [&](const cafe_gpu_ctx::TuneEntry& e) {
                                         return e.path == path && e.nt == tiles && e.leaves == leaves;
                                     }),
                      ctx->tuning.end());
    ctx->tuning.push_back(cafe_gpu_ctx::TuneEntry{path, tiles, leaves, kernel, ntw, w, lds ? 1 : 0, grid_mult, 0});
    return CAFE_GPU_OK;
}

int cafe_gpu_tuning_clear(cafe_gpu_ctx* ctx)
{
    if (!ctx) return fail(CAFE_GPU_EINVAL, "null context");
    ctx->tuning.clear();
    return CAFE_GPU_OK;
}

int cafe_gpu_tuning_load(cafe_gpu_ctx* ctx, const char* path, int* n_loaded)
{
    if (!ctx || !path) return fail(CAFE_GPU_EINVAL, "null argument");
    FILE* fh = fopen(path, "r");
    if (!fh) return fail(CAFE_GPU_EINVAL, "cannot open tuning file %s", path);
    std::vector<cafe_gpu_ctx::TuneEntry> entries;
    char line[512];
    int lineno = 0;
    while (fgets(line, sizeof(line), fh)) {
        ++lineno;
        char* hash = strchr(line, '#');
        if (hash) *hash = 0;
        cafe_gpu_ctx::TuneEntry e{};
        const int n = sscanf(line, "%d %d %d %d %d %d %d %d", &e.path, &e.nt, &e.leaves, &e.kernel, &e.ntw, &e.w,
                             &e.lds, &e.grid_mult);
        if (n <= 0) continue;   // blank or comment
        bool ok = n == 8 && e.path >= CAFE_GPU_PATH_PLAIN64 && e.path <= CAFE_GPU_PATH_BATCHED16 && e.nt >= 1 &&
                  e.leaves >= 1 && e.kernel >= 0 && e.kernel <= 2 && e.ntw >= 0 && e.w >= 0 && e.grid_mult >= 0;
        // optional "plan=n1,n2,...": the tiles per vector of every size class
        // of the plan the entry was measured in (the entry's own among them)
        if (ok) {
            if (const char* pc = strstr(line, "plan=")) {
                pc += 5;
                for (;;) {
                    char* end = nullptr;
                    const long v = strtol(pc, &end, 10);
                    if (end == pc || v < 1 || v > 64) {
                        ok = false;
                        break;
                    }
                    e.plan_classes |= 1ull << (v - 1);
                    pc = end;
                    if (*pc != ',') break;
                    ++pc;
                }
                ok = ok && (*pc == 0 || isspace((unsigned char)*pc)) && (e.plan_classes >> (e.nt - 1) & 1);
            }
        }
        if (!ok) {
            fclose(fh);
            return fail(CAFE_GPU_EINVAL, "%s:%d: malformed tuning entry", path, lineno);
        }
        e.lds = e.lds ? 1 : 0;
        entries.push_back(e);
    }
    fclose(fh);
    ctx->tuning = entries;
    if (n_loaded) *n_loaded = (int)entries.size();
    return CAFE_GPU_OK;
}

int cafe_gpu_last_timings(cafe_gpu_ctx* ctx, double* ms4)
{
    if (!ctx || !ms4) return fail(CAFE_GPU_EINVAL, "null argument");
    if (ctx->build_timed) {
        float ms = 0;
        if (hipEventSynchronize(ctx->ev[5]) == hipSuccess && hipEventElapsedTime(&ms, ctx->ev[4], ctx->ev[5]) == hipSuccess)
            ctx->timings[0] = ms;
        ctx->build_timed = false;
    }
    for (int i = 0; i < 4; ++i) ms4[i] = ctx->timings[i];
    return CAFE_GPU_OK;
}

int cafe_gpu_plan_create(cafe_gpu_ctx* ctx, const cafe_gpu_eval_desc* d, int n_keys, const double* lambda_q,
                         const double* t_q, int algo, int use_graph, cafe_gpu_plan** out)
{
    if (int rc = check_ctx(ctx)) return rc;
    if (!out) return fail(CAFE_GPU_EINVAL, "null output pointer");
    if (ctx->N == 0) return fail(CAFE_GPU_ESTATE, "matrix_reset has not been called");
    if (n_keys < 1 || n_keys > ctx->capacity)
        return fail(CAFE_GPU_EINVAL, "%d keys do not fit the pool capacity %d", n_keys, ctx->capacity);
    if (algo != CAFE_GPU_BUILD_CLOSED_FORM && algo != CAFE_GPU_BUILD_RECURRENCE)
        return fail(CAFE_GPU_EINVAL, "unknown build algorithm %d", algo);
    if (!lambda_q || !t_q) return fail(CAFE_GPU_EINVAL, "null key arrays");
    auto* pl = new cafe_gpu_plan();
    pl->ctx = ctx;
    // the plan builds its keys into slots 0 .. n_keys-1 at every execution:
    // they count as built while its inputs are validated, and are marked
    // built in the context only once an execution has been enqueued
    const std::vector<char> built_before = ctx->built;
    for (int i = 0; i < n_keys; ++i) ctx->built[i] = 1;
    int P = 0;
    int rc = upload_eval_inputs(ctx, pl->bufs, d, P);
    ctx->built = built_before;
    std::vector<int> pts(P);
    std::iota(pts.begin(), pts.end(), 0);
    if (rc == CAFE_GPU_OK) rc = plan_prune(ctx, pl->bufs, d->path, d->model, P, pts.data(), nullptr, 0, pl->pp);
    if (rc == CAFE_GPU_OK && pl->d_keys.ensure(sizeof(double) * 2 * n_keys) != hipSuccess)
        rc = fail(CAFE_GPU_ENOMEM, "key upload buffers");
    if (rc != CAFE_GPU_OK) {
        pl->bufs.release_all();
        delete pl;
        return rc;
    }
    pl->model = d->model;
    pl->path = d->path;
    pl->T = d->n_trials;
    pl->K = d->n_cat;
    pl->n_keys = n_keys;
    pl->algo = algo;
    pl->pool_gen = ctx->pool_gen;
    pl->input_gen = ctx->input_gen;
    for (auto& e : pl->ev) (void)hipEventCreate(&e);
    pl->cls_ev.assign(pl->pp.classes.size() + 1, nullptr);
    for (auto& e : pl->cls_ev) (void)hipEventCreate(&e);
    {
        std::vector<unsigned char> copies;
        plan_copies(ctx, d, pl->pp, pl->T * pl->K, n_keys, copies, pl->copy_top);
        if (pl->d_copies.ensure(copies.size()) != hipSuccess ||
            hipMemcpy(pl->d_copies.p, copies.data(), copies.size(), hipMemcpyHostToDevice) != hipSuccess) {
            cafe_gpu_plan_destroy(pl);
            return fail(CAFE_GPU_ENOMEM, "plan copy table");
        }
    }
    *out = pl;
    if ((rc = cafe_gpu_plan_set_keys(pl, lambda_q, t_q)) != CAFE_GPU_OK) {
        cafe_gpu_plan_destroy(pl);
        *out = nullptr;
        return rc;
    }
    if (use_graph) pl->graph_ok = plan_capture(pl, false);   // eager launches if the runtime refuses
    return CAFE_GPU_OK;
}

int cafe_gpu_plan_set_keys(cafe_gpu_plan* pl, const double* lambda_q, const double* t_q)
{
    if (!pl || !lambda_q || !t_q) return fail(CAFE_GPU_EINVAL, "null argument");
    for (int i = 0; i < pl->n_keys; ++i)
        if (!(lambda_q[i] >= 0) || !(t_q[i] >= 0) || !std::isfinite(lambda_q[i]) || !std::isfinite(t_q[i]))
            return fail(CAFE_GPU_EINVAL, "key %d has an invalid lambda or branch length", i);
    HIP_OR_FAIL(hipSetDevice(pl->ctx->device));
    // (the executions before read theirs: the copy is behind them on the stream)
    std::vector<double> both(lambda_q, lambda_q + pl->n_keys);
    both.insert(both.end(), t_q, t_q + pl->n_keys);
    return upload(pl->ctx, pl->lam(), both.data(), sizeof(double) * both.size());
}

int cafe_gpu_plan_execute(cafe_gpu_plan* pl)
{
    if (!pl) return fail(CAFE_GPU_EINVAL, "null plan");
    if (int rc = plan_current(pl)) return rc;
    cafe_gpu_ctx* ctx = pl->ctx;
    if (pl->graph_ok) HIP_OR_FAIL(hipGraphLaunch(pl->exec, ctx->stream));
    else if (int rc = plan_enqueue(pl, false)) return rc;
    plan_mark_built(pl);
    return CAFE_GPU_OK;
}

int cafe_gpu_plan_synchronize(cafe_gpu_plan* pl)
{
    if (!pl) return fail(CAFE_GPU_EINVAL, "null plan");
    HIP_OR_FAIL(hipStreamSynchronize(pl->ctx->stream));
    return CAFE_GPU_OK;
}

int cafe_gpu_plan_results(cafe_gpu_plan* pl, double* lnl, double* cat, double* post, double* total,
                          long long* n_fallback)
{
    if (!pl) return fail(CAFE_GPU_EINVAL, "null plan");
    if (int rc = plan_current(pl)) return rc;
    return copy_results(pl->ctx, pl->bufs, pl->pp, pl->model, pl->T, pl->K, lnl, cat, post, total, n_fallback);
}

int cafe_gpu_plan_profile(cafe_gpu_plan* pl, double* ms4, int* graph_ok)
{
    if (!pl || !ms4) return fail(CAFE_GPU_EINVAL, "null argument");
    if (int rc = plan_current(pl)) return rc;
    cafe_gpu_ctx* ctx = pl->ctx;
    HIP_OR_FAIL(hipSetDevice(ctx->device));
    if (int rc = plan_enqueue(pl, true)) return rc;
    plan_mark_built(pl);
    HIP_OR_FAIL(hipStreamSynchronize(ctx->stream));
    if (graph_ok) *graph_ok = pl->graph_ok ? 1 : 0;
    ms4[0] = elapsed_ms(pl->ev[0], pl->ev[1]);
    ms4[1] = elapsed_ms(pl->ev[1], pl->ev[2]);
    ms4[2] = elapsed_ms(pl->ev[2], pl->ev[3]);
    ms4[3] = elapsed_ms(pl->ev[3], pl->ev[4]);
    pl->cls_ms.assign(pl->pp.classes.size(), 0.0);
    for (size_t i = 0; i < pl->pp.classes.size(); ++i) pl->cls_ms[i] = elapsed_ms(pl->cls_ev[i], pl->cls_ev[i + 1]);
    return CAFE_GPU_OK;
}

int cafe_gpu_plan_class_times(cafe_gpu_plan* pl, int cap, int* n_classes, int* class_nt, long long* class_tiles,
                              double* ms, int* launch)
{
    if (!pl || !n_classes) return fail(CAFE_GPU_EINVAL, "null argument");
    const int n = (int)pl->pp.classes.size();
    *n_classes = n;
    if (pl->cls_ms.size() != (size_t)n) return fail(CAFE_GPU_ESTATE, "cafe_gpu_plan_profile has not been run");
    for (int i = 0; i < n && i < cap; ++i) {
        if (class_nt) class_nt[i] = pl->pp.classes[i].nt;
        if (class_tiles) class_tiles[i] = pl->pp.class_counts[i];
        if (ms) ms[i] = pl->cls_ms[i];
        if (launch) {
            const KernelClass& kc = pl->pp.classes[i];
            const int n = pl->pp.class_counts[i];
            int* l = launch + 6 * i;
            if (kc.f64) {
                l[0] = kc.plain ? 2 : 0;
                l[1] = kc.s64.ntw;
                l[2] = kc.s64.w;
                l[3] = kc.s64.lds ? 1 : 0;
                l[4] = pl->pp.grid(kc.s64, n);
                l[5] = kTile * kc.s64.fb;
            } else if ((pl->path == CAFE_GPU_PATH_BATCHED32 || pl->path == CAFE_GPU_PATH_BATCHED16) &&
                       kc.lane_rows > 0) {
                l[0] = 1;
                l[1] = kc.lane_rows;
                l[2] = 1;
                l[3] = 0;
                l[4] = pl->pp.grid_lane(kc.lane_per_cu, n, kc.lane_grid_mult);
                l[5] = 64;
            } else {
                const bool f16 = pl->path == CAFE_GPU_PATH_BATCHED16 && kc.nt <= kF16MaxTiles;
                const MfmaShape& sh = f16 ? kc.s16 : kc.s32;
                l[0] = f16 ? 3 : 0;
                l[1] = sh.ntw;
                l[2] = sh.w;
                l[3] = sh.lds ? 1 : 0;
                l[4] = pl->pp.grid(sh, n);
                l[5] = kTile * sh.fb;
            }
        }
    }
    return CAFE_GPU_OK;
}

int cafe_gpu_plan_recompute_counts(cafe_gpu_plan* pl, long long* fp64, long long* plain)
{
    if (!pl) return fail(CAFE_GPU_EINVAL, "null plan");
    int h[2] = {0, 0};
    HIP_OR_FAIL(hipSetDevice(pl->ctx->device));
    HIP_OR_FAIL(hipMemcpyAsync(h, pl->bufs.fb_count.as<int>() + pl->pp.fam_count_off(), sizeof(int) * 2,
                               hipMemcpyDeviceToHost, pl->ctx->stream));
    HIP_OR_FAIL(hipStreamSynchronize(pl->ctx->stream));
    if (fp64) *fp64 = h[0];
    if (plain) *plain = h[1];
    return CAFE_GPU_OK;
}

int cafe_gpu_plan_destroy(cafe_gpu_plan* pl)
{
    if (!pl) return CAFE_GPU_OK;
    (void)hipSetDevice(pl->ctx->device);
    (void)hipStreamSynchronize(pl->ctx->stream);
    if (pl->exec) (void)hipGraphExecDestroy(pl->exec);
    if (pl->graph) (void)hipGraphDestroy(pl->graph);
    for (auto& e : pl->ev)
        if (e) (void)hipEventDestroy(e);
    for (auto& e : pl->cls_ev)
        if (e) (void)hipEventDestroy(e);
    pl->bufs.release_all();
    pl->d_keys.release();
    pl->d_copies.release();
    delete pl;
    return CAFE_GPU_OK;
}

}  // extern "C"
