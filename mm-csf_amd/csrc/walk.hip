// Entry points of the chunked root walk (the kernel is in walk_kernel.hpp,
// instantiated per operation in walk_mttkrp.hip, walk_loss.hip,
// walk_lossgrad.hip, walk_wgrad.hip and walk_ttm.hip).
#include <algorithm>
#include <mutex>

#include "walk.hpp"

namespace mmcsf {

namespace {

WalkArgs args_of(const Csf &c, const Factors &F) {
    const int N = c.ndims;
    WalkArgs a{};
    for (int l = 0; l < N - 1; ++l) {
        a.ptr[l] = c.ptr[l].p;
        a.idx[l] = c.idx[l].p;
        a.cnt[l] = (uint32_t)c.cnt[l];
    }
    a.cnt[N - 1] = (uint32_t)c.nnz;
    a.slc = c.fbrSlc.p;
    a.leaf = c.leaf.p;
    a.val = c.vals.p;
    a.fbit = c.fbit.p;
    a.sbit = c.sbit.p;
    a.frank = c.frank.p;
    a.jrank = c.jrank.p;
    a.cost = c.chunkCost.p;
    a.pos = c.pos.p;
    const uint64_t es = F.dtype == MMCSF_F32 ? 4 : 2;
    for (int l = 0; l < N; ++l) {
        a.U[l] = F.U[c.order[l]];
        a.tabBytes[l] = (uint32_t)(c.rows[l] * (uint64_t)F.R * es);
    }
    a.nnz = (uint32_t)c.nnz;
    a.R = F.R;
    a.cols = F.R;
    a.alpha = 1.f;
    return a;
}

// Columns that one float32 MTTKRP pass takes.  A pass holds a group's rows,
// partial sums and loads in flight in registers.  Past two column blocks (64
// columns) it runs at two waves per SIMD, and past four (128) it spills: passes
// over 64 columns, which read the tree again, take over where nothing speaks
// against them:
//   - Rows that are no multiple of 128 bytes are read line by line in one pass,
//     but a line that two passes share is read by both.  That shows where the
//     lines come from past the L2s: uniform 3-D tables, 4M nonzeros, R = 72,
//     passes / one pass 0.75-0.84 at 1 MB of tables, 0.88-0.96 at 4 MB, 0.9-1.05
//     at 9, 1.06-1.15 at 18, 1.15-1.22 at 35 (R = 144: 0.72-0.84 at 18 MB,
//     1.13-1.17 at 30M nonzeros and 230 MB).  Tables past 8 MB therefore need
//     whole lines, R % 32 == 0 (30M nonzeros, 410 MB: R = 96 0.94-0.98, 160 0.90-0.96).
//   - Each pass is a launch and its latencies.  At R = 72 and 96 the passes gain
//     from about 1.5M nonzeros on (3-D, one mode: 200000 nonzeros 1.16 times the
//     time, 800000 1.07-1.13, 1.6M 0.99-1.03, 2M 0.93-1.02); up to R = 160, where
//     one pass spills, they cost nothing at 200000 (0.92-1.01), at 192 1.09-1.13.
//   - From 97 to 128 columns one pass has no half-used block to lose: two take
//     0.84-1.17 of its time near, 0.95-1.24 far.
//   - Past 192 columns, over near tables, four passes take 0.75 to 1.23 of one's
//     time from mode to mode; far ones of whole lines 0.70-1.01.
// 32-column passes of 4-D walks at R = 64 gain where modes are uniform (0.72-1.02)
// and lose where all but one are skewed (1.04-1.16): one pass.  Bfloat16 rows
// are half as wide and stay in one pass (R = 128: 2.38 / 2.45 ms, 2M nonzeros
// R = 256 284 / 410 us).
int pass_columns(int N, const WalkArgs &a, const Factors &F) {
    const int R = F.R;
    if (F.dtype != MMCSF_F32 || R <= 64) return R;
    uint64_t bytes = 0;
    for (int l = 1; l < N; ++l) bytes += a.tabBytes[l];
    const bool near = bytes < (8ull << 20), lines = R % 32 == 0;
    const bool many = a.nnz >= 3u << 19;
    if (R <= 96) return many && (near || lines) ? 64 : R;
    if (R <= 128) return R;
    if (R <= 192) return (near || lines) && (many || R <= 160) ? 64 : R;
    return many && !near && lines ? 64 : R;
}

// the pass that starts at column `at`: `width` columns, fewer at the end, but
// never fewer than four left over (a lane's load)
int pass_width(int R, int at, int width) {
    const int left = R - at;
    if (left <= width) return left;
    return left - width < 4 ? width - 4 : width;
}

// moves a walk to the columns from `at` on
void take_columns(int N, WalkArgs &a, const Factors &F, int at, int cols) {
    const uint32_t skip = (uint32_t)at * (F.dtype == MMCSF_F32 ? 4u : 2u);
    for (int l = 0; l < N; ++l) {
        if (a.U[l]) a.U[l] = static_cast<const char *>(a.U[l]) + skip;
        a.tabBytes[l] -= std::min(a.tabBytes[l], skip);
    }
    a.out += at;
    a.cols = cols;
}

// launches an MTTKRP walk once per pass over columns
template <typename L>
void walk_columns(int N, const WalkArgs &a, const Factors &F, L launch) {
    const int width = pass_columns(N, a, F);
    for (int at = 0; at < F.R;) {
        WalkArgs p = a;
        const int cols = pass_width(F.R, at, width);
        take_columns(N, p, F, at, cols);
        launch(p);
        at += cols;
    }
}

__global__ void k_zero_f64(double *p) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *p = 0.0;
}

__global__ void k_half(double *p) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *p *= 0.5;
}

}  // namespace

// the walk addresses factor rows by 32-bit byte offsets and masks the rows it
// does not need with out-of-range buffer offsets: every table of the tree's
// levels must stay below 4 GiB - 4 KiB (counted at 4 bytes per element)
static bool tables_fit(const Csf &c, int R) {
    for (int l = 0; l < c.ndims; ++l)
        if (c.rows[l] * (uint64_t)R * 4u > 0xFFFFF000ull) return false;
    return true;
}

// row loads of the walk are VEC elements wide (16 bytes, or 8 bytes for
// bfloat16 rows with R % 8 != 0); rows of `out` are written as float4.  At
// ranks that four does not divide both are 16-byte accesses at 4-byte
// boundaries.
void check_walk_align(const Csf &c, const Factors &F, int skipLevel, const float *out) {
    const bool ragged = F.R % 4 != 0;
    const uintptr_t need = ragged ? 4 : (F.dtype == MMCSF_BF16 && F.R % 8 != 0) ? 8 : 16;
    for (int l = 0; l < c.ndims; ++l) {
        if (l == skipLevel) continue;
        const void *p = F.U[c.order[l]];
        MMCSF_REQUIRE(p != nullptr, MMCSF_ERR_ARG, "missing factor matrix");
        MMCSF_REQUIRE(reinterpret_cast<uintptr_t>(p) % need == 0, MMCSF_ERR_ARG,
                      "factor pointer is not aligned to " + std::to_string(need) + " bytes");
    }
    MMCSF_REQUIRE(!out || reinterpret_cast<uintptr_t>(out) % (ragged ? 4 : 16) == 0, MMCSF_ERR_ARG,
                  ragged ? "output pointer is not aligned to 4 bytes" : "output pointer is not aligned to 16 bytes");
}

bool walk_aligned(const Csf &c, const Factors &F, int skipLevel, const float *out) {
    const uintptr_t need = F.R % 4 != 0 ? 4 : (F.dtype == MMCSF_BF16 && F.R % 8 != 0) ? 8 : 16;
    for (int l = 0; l < c.ndims; ++l)
        if (l != skipLevel && reinterpret_cast<uintptr_t>(F.U[c.order[l]]) % need != 0) return false;
    return reinterpret_cast<uintptr_t>(out) % (F.R % 4 != 0 ? 4 : 16) == 0;
}

// What a walk can run: every multiple of four, and any float32 rank from 4 on.
static bool walk_fits(const Csf &c, int R, int dtype) {
    return R >= 4 && R <= 256 && (R % 4 == 0 || dtype == MMCSF_F32) && tables_fit(c, R) &&
           (c.nnz == 0 || (c.fbit.p && c.frank.p && c.chunkCost.p && (c.ndims == 3 || (c.sbit.p && c.jrank.p))));
}

// Short tensors at wide ranks that four does not divide: the walk takes them in
// one spilling pass or a launch per pass, the per-group kernels, one column a
// lane, in one launch.  Group kernel / walk, root mode: 50000 nonzeros R = 129 18 /
// 24 us, COO 15 / 23; 200000 R = 255 41 / 50, COO 35 / 54; 700000 R = 161 90 / 70
// (3-D, tables of 4 MB), 85 / 98 (4-D), 193 / 219 (COO, 200 MB); 1.4M 163 / 116,
// 164 / 162, 328 / 357; up to R = 127 the walk from 50000 nonzeros on (17 / 17).
static bool group_kernel_shorter(uint64_t nnz, int R) { return R > 128 && R % 4 != 0 && nnz < 1u << 20; }

// Below a rank of 4 the row is narrower than one lane's load and the per-group
// kernel serves it.  At R = 10 (HB-CSF, 3.3M nonzeros, 123457 x 70001 x 9973) the
// per-group kernel, one column a lane in groups of 64, takes 324 us; the whole
// call 334 -> 53 us.
bool walk_supports(const Csf &c, int R, int dtype) {
    return walk_fits(c, R, dtype) && !group_kernel_shorter(c.nnz, R);
}

void mttkrp_root(const Csf &c, const Factors &F, float *out, hipStream_t s, bool accumulate) {
    if (c.nnz == 0) return;
    MMCSF_REQUIRE(walk_supports(c, F.R, F.dtype), MMCSF_ERR_UNSUPPORTED,
                  "root walk needs R >= 4, start bitmasks and factor tables below 4 GiB");
    check_walk_align(c, F, 0, out);
    WalkArgs a = args_of(c, F);
    a.out = out;
    a.accum = accumulate ? 1 : 0;
    walk_columns(c.ndims, a, F, [&](const WalkArgs &p) { walk_launch<kMttkrp>(c.ndims, F, p, s); });
}

// The COO type's root-mode MTTKRP as a walk: the coordinates are read once per
// chunk, 64 of a level to a load, where the per-group kernel reads each
// nonzero's with a load of its own for every group.  Serves what walk_supports
// serves and factors at the walk's alignment; the per-group kernel takes the
// rest.  2000 x 2000 x 2000, 1M nonzeros, R = 32: 54 -> 19 us the call.
bool coo_walk_supports(const Format &f, const Factors &F) {
    if (F.R < 4 || F.R > 256 || (F.R % 4 != 0 && F.dtype != MMCSF_F32)) return false;
    if (!f.cooCost.p || group_kernel_shorter(f.nnz, F.R)) return false;
    const uintptr_t need = F.R % 4 != 0 ? 4 : (F.dtype == MMCSF_BF16 && F.R % 8 != 0) ? 8 : 16;
    for (int l = 1; l < f.ndims; ++l) {
        if (f.dims[f.cooOrder[l]] * (uint64_t)F.R * 4u > 0xFFFFF000ull) return false;
        if (reinterpret_cast<uintptr_t>(F.U[f.cooOrder[l]]) % need != 0) return false;
    }
    return true;
}

void mttkrp_coo_walk(const Format &f, const Factors &F, float *out, hipStream_t s) {
    const int N = f.ndims;
    WalkArgs a{};
    for (int l = 0; l < N - 1; ++l) a.idx[l] = f.cooKeys[l].p;
    a.leaf = f.cooKeys[N - 1].p;
    a.val = f.cooVals.p;
    a.cost = f.cooCost.p;
    const uint64_t es = F.dtype == MMCSF_F32 ? 4 : 2;
    for (int l = 0; l < N; ++l) {
        a.U[l] = F.U[f.cooOrder[l]];
        a.tabBytes[l] = (uint32_t)(f.dims[f.cooOrder[l]] * (uint64_t)F.R * es);
        a.cnt[l] = (uint32_t)f.nnz;
    }
    a.nnz = (uint32_t)f.nnz;
    a.R = F.R;
    a.cols = F.R;
    a.alpha = 1.f;
    a.out = out;
    walk_columns(N, a, F, [&](const WalkArgs &p) { walk_launch<kMttkrp, kCoo>(N, F, p, s); });
}

// The modes below the root of a tree that serves every mode.  A tree holds an
// output row's nonzeros in many places; scattering each partial row there is
// bound by the additions (float atomics that meet in the L2, or in LDS on the
// hottest rows: one row of a Zipf(1.2) mode takes ~18 % of them).  A level map
// lists the nonzeros by output row, so the same walk as from a root sums every
// row in registers; it finds a nonzero's fiber by the rank of its start bit and
// reads coordinates and value where the tree holds them (a few 4-byte reads of
// their own line each; the price of 4 bytes per nonzero and level instead of a
// tree per mode).  One tree, 20M nonzeros, 500000 x 200000 x 50000, R = 32, the
// two modes below the root: 7.19 -> 2.59 ms.  Those reads bound it: each lane's
// is a line of its own past the L2, ~8.6 CU clocks apiece.
bool map_walk_supports(const Csf &c, const Factors &F, int outLevel, const float *out) {
    return walk_fits(c, F.R, F.dtype) && walk_aligned(c, F, outLevel, out);
}

void mttkrp_map_walk(const Csf &c, int outLevel, const Factors &F, float *out, hipStream_t s, bool accumulate) {
    WalkArgs a = args_of(c, F);
    a.ord = c.map[outLevel].ord.p;
    a.cost = c.map[outLevel].cost.p;
    a.outLevel = outLevel;
    // the other levels, in tree order, as the walk's levels 1..N-1
    const uint64_t es = F.dtype == MMCSF_F32 ? 4 : 2;
    for (int l = 0, to = 1; l < c.ndims; ++l) {
        if (l == outLevel) continue;
        a.U[to] = F.U[c.order[l]];
        a.tabBytes[to] = (uint32_t)(c.rows[l] * (uint64_t)F.R * es);
        ++to;
    }
    a.out = out;
    a.accum = accumulate ? 1 : 0;
    walk_columns(c.ndims, a, F, [&](const WalkArgs &p) { walk_launch<kMttkrp, kMap>(c.ndims, F, p, s); });
}

// The root walks of several trees in one launch, into zeroed outputs.  A walk of
// few chunks per wave is a chain of ~8 memory latencies and a launch; the modes'
// chains then run side by side (300 x 200 x 100, 20000 nonzeros, R = 32: six
// launches for the outputs and the walks, 34 us a call, are two, 20 us).
// unlike: trees whose nonzeros cost differently (HB-CSF's parts).  The blocks are
// then shared by the rows above the leaf that a walk reads and the slices that it
// writes, each as 8 nonzeros, instead of by chunks (as 2 nonzeros: 2 to 5 % slower
// over the sizes and laws that go together; as none: up to 1.7 times the time).
bool mttkrp_roots(const Csf *const *trees, int walks, const Factors &F, float *const *outs, hipStream_t s,
                  bool unlike) {
    WalkSet set{};
    uint64_t weight[kMaxDims];
    for (int m = 0; m < walks; ++m) {
        const Csf &c = *trees[m];
        for (int l = 1; l < c.ndims; ++l)
            if (!F.U[c.order[l]]) return false;
        if (c.nnz == 0 || !walk_supports(c, F.R, F.dtype) || !walk_aligned(c, F, 0, outs[m])) return false;
        set.walk[m] = args_of(c, F);
        set.walk[m].out = outs[m];
        weight[m] = unlike ? c.nnz + 8 * (c.cnt[c.ndims - 2] + c.cnt[0]) : (c.nnz + 63) / 64;
    }
    const int N = trees[0]->ndims, R = F.R;
    // passes over columns as for one walk; the first decides for all of them
    const int width = pass_columns(N, set.walk[0], F);
    for (int at = 0; at < R;) {
        WalkSet p = set;
        const int cols = pass_width(R, at, width);
        for (int m = 0; m < walks; ++m) take_columns(N, p.walk[m], F, at, cols);
        if (!walk_launch_set<kMttkrp>(N, F, p, walks, weight, at > 0, s)) return false;
        at += cols;
    }
    return true;
}

bool cp_supports(int R) { return R >= 1 && R <= 128 && R % 4 == 0; }

void cp_forward(const Csf &c, const Factors &F, float *resid, double *loss, hipStream_t s) {
    MMCSF_REQUIRE(tables_fit(c, F.R), MMCSF_ERR_UNSUPPORTED, "CP completion needs factor tables below 4 GiB");
    hipLaunchKernelGGL(k_zero_f64, dim3(1), dim3(64), 0, s, loss);
    MMCSF_HIP(hipGetLastError());
    if (c.nnz > 0) {
        WalkArgs a = args_of(c, F);
        a.resid = resid;
        a.sumsq = loss;
        walk_launch<kLossResid>(c.ndims, F, a, s);
    }
    hipLaunchKernelGGL(k_half, dim3(1), dim3(64), 0, s, loss);
    MMCSF_HIP(hipGetLastError());
}

void cp_gradient(const Csf &c, const Factors &F, const float *weights, float alpha, float *grad, double *loss,
                 hipStream_t s) {
    if (c.nnz == 0) return;
    MMCSF_REQUIRE(tables_fit(c, F.R), MMCSF_ERR_UNSUPPORTED, "CP completion needs factor tables below 4 GiB");
    WalkArgs a = args_of(c, F);
    a.out = grad;
    a.alpha = alpha;
    if (weights) {
        a.wts = weights;
        walk_launch<kWeightGrad>(c.ndims, F, a, s);
    } else {
        a.sumsq = loss;
        walk_launch<kLossGrad>(c.ndims, F, a, s);
    }
}

void ttm_fibers(const Csf &c, const Factors &F, float *Y, hipStream_t s) {
    if (c.nnz == 0) return;
    MMCSF_REQUIRE(F.R % 4 == 0 && walk_supports(c, F.R, F.dtype), MMCSF_ERR_UNSUPPORTED, "TTM needs R % 4 == 0, R <= 256 and factor tables below 4 GiB");
    const int leaf = c.ndims - 1;
    const uintptr_t need = (F.dtype == MMCSF_BF16 && F.R % 8 != 0) ? 8 : 16;
    MMCSF_REQUIRE(F.U[c.order[leaf]] && reinterpret_cast<uintptr_t>(F.U[c.order[leaf]]) % need == 0, MMCSF_ERR_ARG,
                  "factor pointer is not aligned to " + std::to_string(need) + " bytes");
    WalkArgs a = args_of(c, F);
    a.out = Y;
    // Y past the 256 MB memory-side cache cannot be read back from it, and its
    // lines only push the factor rows out: written around the caches (20M
    // nonzeros, 10M fibers, R = 32, 1.28 GB of rows: 486 -> 459 us).  Smaller
    // outputs stay where their reader finds them.
    if (c.cnt[c.ndims - 2] * (uint64_t)F.R * 4u > (256ull << 20)) walk_launch<kTtmStream>(c.ndims, F, a, s);
    else walk_launch<kTtm>(c.ndims, F, a, s);
}

void preload_kernels(unsigned what) {
    static std::mutex lock;
    static unsigned done[64];
    int dev = 0;
    MMCSF_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= 64) return;
    std::lock_guard<std::mutex> g(lock);
    const unsigned load = what & ~done[dev];
    if (!done[dev]) preload_group_kernels();
    if (load & kPreTree) walk_preload<kMttkrp>();
    if (load & kPreSet) walk_preload_set<kMttkrp>();
    if (load & kPreCoo) walk_preload<kMttkrp, kCoo>();
    if (load & kPreMap) walk_preload<kMttkrp, kMap>();
    if (load & kPreCp) {
        walk_preload<kLossResid>();
        walk_preload<kLossGrad>();
        walk_preload<kWeightGrad>();
    }
    done[dev] |= load;
}

void cp_half(double *loss, hipStream_t s) {
    hipLaunchKernelGGL(k_half, dim3(1), dim3(64), 0, s, loss);
    MMCSF_HIP(hipGetLastError());
}

}  // namespace mmcsf
