// GPU format builder: sort / scan / segment passes that produce the
// reference's COO, B-CSF, HB-CSF and MM-CSF arrays bit for bit.
//
// Reference flows restated here (util.h):
//   order_tensormode        255-311
//   sort_COOtensor / sort_MI_CSF   412-527 (full-key sort: one legal order)
//   create_HCSR / create_TiledHCSR 760-850 / 1320-1436
//   create_fbrLikeSlcInds   1770-1783
//   make_TiledBin           1887-1952
//   create_HYB / _4D, make_HybBin  852-1142, 1786-1885
#include <cstdio>
#include <cstdlib>
#include <cmath>
#include <cstring>
#include <rocprim/rocprim.hpp>

#include <algorithm>
#include <numeric>

#include "mmcsf_internal.hpp"
#include "mttkrp_kernels.hpp"

namespace mmcsf {

namespace {

constexpr unsigned kBS = 256;

inline unsigned nblk(uint64_t n) { return (unsigned)std::max<uint64_t>(1, (n + kBS - 1) / kBS); }

int bitwidth(uint64_t v) {  // bits needed for values 0..v
    int b = 1;
    while (b < 64 && (v >> b)) ++b;
    return b;
}

struct Temp {
    DevArray<uint8_t> buf;
    void *get(size_t bytes) {
        if (buf.n < bytes) buf.tmp(std::max<size_t>(bytes, 256));
        return buf.p;
    }
};

// out[i] = sum_{j<i} in[j]; returns the total.
uint64_t exclusive_sum(const uint32_t *in, uint32_t *out, uint64_t n, hipStream_t s, Temp &tmp) {
    if (n == 0) return 0;
    size_t bytes = 0;
    MMCSF_HIP(rocprim::exclusive_scan(nullptr, bytes, in, out, 0u, (size_t)n, rocprim::plus<uint32_t>(), s));
    MMCSF_HIP(rocprim::exclusive_scan(tmp.get(bytes), bytes, in, out, 0u, (size_t)n,
                                      rocprim::plus<uint32_t>(), s));
    // both addends of the total in one synchronisation
    uint32_t last[2] = {0, 0};
    MMCSF_HIP(hipMemcpyAsync(&last[0], in + n - 1, 4, hipMemcpyDeviceToHost, s));
    MMCSF_HIP(hipMemcpyAsync(&last[1], out + n - 1, 4, hipMemcpyDeviceToHost, s));
    MMCSF_HIP(hipStreamSynchronize(s));
    return (uint64_t)last[0] + last[1];
}

void inclusive_max(const uint32_t *in, uint32_t *out, uint64_t n, hipStream_t s, Temp &tmp) {
    if (n == 0) return;
    size_t bytes = 0;
    MMCSF_HIP(rocprim::inclusive_scan(nullptr, bytes, in, out, (size_t)n, rocprim::maximum<uint32_t>(), s));
    MMCSF_HIP(rocprim::inclusive_scan(tmp.get(bytes), bytes, in, out, (size_t)n,
                                      rocprim::maximum<uint32_t>(), s));
}

// ---------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------
__global__ void k_iota(uint32_t *p, uint64_t n) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i < n) p[i] = (uint32_t)i;
}

struct PackSpec {
    const uint32_t *src[kMaxDims];
    int shift[kMaxDims];
    int nlev;
};

// key[i] = packed coordinates of element i, perm[i] = i (perm may be null)
__global__ void k_pack_first(PackSpec ps, uint64_t *__restrict__ key, uint32_t *__restrict__ perm, uint64_t n) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint64_t k = 0;
    for (int l = 0; l < ps.nlev; ++l) k |= (uint64_t)ps.src[l][i] << ps.shift[l];
    key[i] = k;
    if (perm) perm[i] = (uint32_t)i;
}

// The inverse of the packing: the coordinates of a sorted key, one stream in
// and one out per level.  Gathering them through the permutation instead costs
// a random 4-byte read per nonzero and level (20M nonzeros: 0.385 ms a level;
// three levels here: 0.071 ms).
struct UnpackSpec {
    uint32_t *dst[kMaxDims];
    int shift[kMaxDims];
    uint32_t mask[kMaxDims];
    int nlev;
};
__global__ void k_unpack(UnpackSpec us, const uint64_t *__restrict__ key, uint64_t n) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint64_t k = key[i];
    for (int l = 0; l < us.nlev; ++l) us.dst[l][i] = (uint32_t)(k >> us.shift[l]) & us.mask[l];
}

// key[p] = packed coordinates of element perm[p]
__global__ void k_pack(PackSpec ps, const uint32_t *__restrict__ perm, uint64_t *__restrict__ key,
                       uint64_t n) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t e = perm[i];
    uint64_t k = 0;
    for (int l = 0; l < ps.nlev; ++l) k |= (uint64_t)ps.src[l][e] << ps.shift[l];
    key[i] = k;
}

__global__ void k_gather_u32(const uint32_t *__restrict__ src, const uint32_t *__restrict__ perm,
                             uint32_t *__restrict__ dst, uint64_t n) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[perm[i]];
}

__global__ void k_gather_f32(const float *__restrict__ src, const uint32_t *__restrict__ perm,
                             float *__restrict__ dst, uint64_t n) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[perm[i]];
}

struct Keys {
    const uint32_t *k[kMaxDims];
};

// d[p] = first level whose coordinate differs from position p-1 (0 at p=0,
// N when the whole coordinate repeats); runPos[p] = p at a leaf-fiber key
// change (d <= N-2), else 0 -- the max-scan input for the -f chunk rule.
__global__ void k_first_diff(Keys K, int N, uint8_t *__restrict__ d, uint32_t *__restrict__ runPos,
                             uint64_t n) {
    uint64_t p = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (p >= n) return;
    int fd = 0;
    if (p > 0) {
        fd = N;
        for (int l = N - 1; l >= 0; --l)
            if (K.k[l][p] != K.k[l][p - 1]) fd = l;
    }
    d[p] = (uint8_t)fd;
    runPos[p] = (fd <= N - 2) ? (uint32_t)p : 0u;
}

// Leaf-fiber start flag: a key change at a fiber level, or the run of equal
// fiber keys reaching a multiple of the -f threshold (util.h:1364-1382).
__global__ void k_leaf_flag(const uint8_t *__restrict__ d, const uint32_t *__restrict__ runStart,
                            int N, uint64_t fthr, uint32_t *__restrict__ flag, uint64_t n) {
    uint64_t p = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (p >= n) return;
    bool f = d[p] <= N - 2;
    if (!f && runStart) f = ((p - runStart[p]) % fthr) == 0;
    flag[p] = f ? 1u : 0u;
}

// Scatter of the leaf-fiber level: pointer, index, first-diff level and
// start position of every leaf fiber.
__global__ void k_scatter_leaf(const uint32_t *__restrict__ flag, const uint32_t *__restrict__ fid,
                               const uint8_t *__restrict__ d, const uint32_t *__restrict__ key2,
                               uint32_t *__restrict__ ptr, uint32_t *__restrict__ idx,
                               uint8_t *__restrict__ dF, uint64_t n) {
    uint64_t p = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (p >= n || !flag[p]) return;
    uint32_t f = fid[p];
    ptr[f] = (uint32_t)p;
    idx[f] = key2[p];
    dF[f] = d[p];
}

// flag[f] = (dF[f] <= lev) for leaf fibers
__global__ void k_level_flag(const uint8_t *__restrict__ dF, int lev, uint32_t *__restrict__ flag,
                             uint64_t nf) {
    uint64_t f = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (f < nf) flag[f] = dF[f] <= lev ? 1u : 0u;
}

// 4-D fbrS split (util.h:1388-1404).  One thread walks one run of equal
// (k0,k1) keys over its leaf fibers.  A new fbrS starts at leaf fiber q when
// the current fbrS (started at nonzero s) already counts more than
// fsthr nonzeros by the reference's counter, which reads q - s for the very
// first fbrS of the tensor and q - s + 1 after every reset.
__global__ void k_fbrs_split(const uint32_t *__restrict__ runs, uint64_t nruns, uint64_t nf,
                             const uint32_t *__restrict__ leafPtr, uint64_t fsthr,
                             uint32_t *__restrict__ jflag) {
    uint64_t r = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (r >= nruns) return;
    uint32_t f0 = runs[r];
    uint32_t f1 = (r + 1 < nruns) ? runs[r + 1] : (uint32_t)nf;
    uint64_t s = leafPtr[f0];
    jflag[f0] = 1u;
    for (uint32_t f = f0 + 1; f < f1; ++f) {
        uint64_t q = leafPtr[f];
        uint64_t count = (q - s) + (s > 0 ? 1u : 0u);
        if (count > fsthr) {
            jflag[f] = 1u;
            s = q;
        } else {
            jflag[f] = 0u;
        }
    }
}

// Compaction of flagged leaf fibers into an upper level:
//   ptr[ord] = value_of(f) (index into the level below), idx[ord] = key[pos(f)]
__global__ void k_scatter_upper(const uint32_t *__restrict__ flag, const uint32_t *__restrict__ ord,
                                const uint32_t *__restrict__ below, const uint32_t *__restrict__ leafPtr,
                                const uint32_t *__restrict__ key, uint32_t *__restrict__ ptr,
                                uint32_t *__restrict__ idx, const uint32_t *__restrict__ key0,
                                uint32_t *__restrict__ slc, uint64_t nf) {
    uint64_t f = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (f >= nf || !flag[f]) return;
    uint32_t o = ord[f];
    ptr[o] = below ? below[f] : (uint32_t)f;
    uint32_t pos = leafPtr[f];
    idx[o] = key[pos];
    if (slc) slc[o] = key0[pos];
}

__global__ void k_set(uint32_t *p, uint64_t i, uint32_t v) { p[i] = v; }

__global__ void k_zero_words(uint32_t *p, uint64_t n) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

// per 64-nonzero chunk: the number of slices starting in it
__global__ void k_chunk_starts(int N, const uint32_t *__restrict__ p0, const uint32_t *__restrict__ p1,
                               const uint32_t *__restrict__ p2, uint64_t nS, uint32_t *cnt) {
    uint64_t s = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (s >= nS) return;
    uint32_t x = p1[p0[s]];
    if (N == 4) x = p2[x];
    atomicAdd(cnt + (x >> 6), 1u);
}

// traversal cost of a chunk: 64 units (its leaf rows), wf per leaf fiber
// starting in it (the fiber-level rows, read once per fiber segment) and ws
// per slice start (row writes and the join of the group runs)
__global__ void k_chunk_cost(const uint32_t *__restrict__ cnt, const uint32_t *__restrict__ fbit, uint64_t n,
                             bool plain, uint32_t wf, uint32_t ws, uint32_t *cost) {
    uint64_t c = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (c < n) {
        const uint32_t fs = (uint32_t)(__popc(fbit[2 * c]) + __popc(fbit[2 * c + 1]));
        cost[c] = plain ? 1u : 64u + wf * fs + ws * cnt[c];
    }
}

// bit ptr[i] of `bits` for every entry i < n (first child of every entry; ptr
// ascending).  A block's kMarkEntries entries fall on few consecutive words
// (a leaf fiber holds a handful of nonzeros): it sets them in an LDS window and
// adds each word that it touched to memory once.  One global atomic per entry
// instead waits on the entries that share its word (10.3M fibers of 20M
// nonzeros: 0.445 ms, here 0.028).  Entries past the window go to memory.
constexpr uint32_t kMarkEntries = 2048, kMarkWords = 2048;
__global__ __launch_bounds__(kBS) void k_mark_starts(const uint32_t *__restrict__ ptr, uint64_t n, uint32_t *bits) {
    __shared__ uint32_t win[kMarkWords];
    const uint64_t i0 = blockIdx.x * (uint64_t)kMarkEntries;
    const uint64_t i1 = min(n, i0 + kMarkEntries);
    for (uint32_t w = threadIdx.x; w < kMarkWords; w += kBS) win[w] = 0u;
    __syncthreads();
    const uint32_t w0 = ptr[i0] >> 5, used = min((ptr[i1 - 1] >> 5) - w0 + 1, kMarkWords);
    for (uint64_t i = i0 + threadIdx.x; i < i1; i += kBS) {
        const uint32_t p = ptr[i], w = (p >> 5) - w0;
        if (w < kMarkWords) atomicOr(&win[w], 1u << (p & 31));
        else atomicOr(bits + (p >> 5), 1u << (p & 31));
    }
    __syncthreads();
    for (uint32_t w = threadIdx.x; w < used; w += kBS)
        if (win[w]) atomicOr(bits + w0 + w, win[w]);
}

// ---------------------------------------------------------------------------
// bins
// ---------------------------------------------------------------------------
struct BinBounds {
    int64_t LB[kNumBins], UB[kNumBins];
};

BinBounds bin_bounds(uint64_t totNnz) {
    // make_TiledBin / make_HybBin bin table (util.h:1796-1812, 1897-1916)
    const int64_t TB = 512;
    BinBounds b;
    int64_t lb[kNumBins] = {0, 2, 4, 8, 16, 1024, 4 * TB, 8 * TB, 16 * TB, 32 * TB};
    int64_t ub[kNumBins] = {3, 5, 9, 17, 1025, 4 * TB + 1, 8 * TB + 1, 16 * TB + 1, 32 * TB + 1,
                            (int64_t)totNnz + 1};
    for (int i = 0; i < kNumBins; ++i) { b.LB[i] = lb[i]; b.UB[i] = ub[i]; }
    b.UB[0] = 1025;  // bins 0..4 merged
    return b;
}

// weight of slice s: (level-1 entries if withFibers) + nonzeros
__global__ void k_slice_bin(int N, const uint32_t *__restrict__ p0, const uint32_t *__restrict__ p1,
                            const uint32_t *__restrict__ p2, bool withFibers, BinBounds bb,
                            int8_t *__restrict__ bin, uint64_t nslc) {
    uint64_t s = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (s >= nslc) return;
    uint32_t a = p0[s], b = p0[s + 1];
    uint64_t nz;
    if (N == 3) nz = (uint64_t)p1[b] - p1[a];
    else nz = (uint64_t)p2[p1[b]] - p2[p1[a]];
    // the reference accumulates the weight in an int (util.h:1921)
    int w = (int)((withFibers ? (uint64_t)(b - a) : 0) + nz);
    int sel = -1;
    for (int k = 0; k < kNumBins; ++k)
        if ((int64_t)w > bb.LB[k] && (int64_t)w < bb.UB[k]) { sel = k; break; }
    bin[s] = (int8_t)sel;
}

__global__ void k_csl_bin(const uint32_t *__restrict__ ptr, BinBounds bb, int8_t *__restrict__ bin,
                          uint64_t n) {
    uint64_t s = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (s >= n) return;
    int w = (int)(ptr[s + 1] - ptr[s]);
    int sel = -1;
    for (int k = 0; k < kNumBins; ++k)
        if ((int64_t)w > bb.LB[k] && (int64_t)w < bb.UB[k]) { sel = k; break; }
    bin[s] = (int8_t)sel;
}

__global__ void k_eq_flag(const int8_t *__restrict__ v, int8_t want, uint32_t *__restrict__ flag,
                          uint64_t n) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i < n) flag[i] = v[i] == want ? 1u : 0u;
}

__global__ void k_compact_idx(const uint32_t *__restrict__ flag, const uint32_t *__restrict__ pos,
                              uint32_t *__restrict__ out, uint64_t n) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i < n && flag[i]) out[pos[i]] = (uint32_t)i;
}

// stable per-bin lists of slice ordinals (slcMapperBin push order)
void bin_lists(const int8_t *bin, uint64_t n, DevArray<uint32_t> &list, uint64_t *counts,
               uint64_t &dropped, hipStream_t s, Temp &tmp) {
    TmpArray<uint32_t> flag(n), pos(n);
    uint64_t tot = 0, cnt[kNumBins];
    std::vector<DevArray<uint32_t>> parts(kNumBins);
    for (int b = 0; b < kNumBins; ++b) {
        hipLaunchKernelGGL(k_eq_flag, dim3(nblk(n)), dim3(kBS), 0, s, bin, (int8_t)b, flag.p, n);
        cnt[b] = exclusive_sum(flag.p, pos.p, n, s, tmp);
        parts[b].tmp(cnt[b]);
        if (cnt[b])
            hipLaunchKernelGGL(k_compact_idx, dim3(nblk(n)), dim3(kBS), 0, s, flag.p, pos.p,
                               parts[b].p, n);
        tot += cnt[b];
    }
    list.alloc(tot);
    uint64_t off = 0;
    for (int b = 0; b < kNumBins; ++b) {
        counts[b] = cnt[b];
        if (cnt[b])
            MMCSF_HIP(hipMemcpyAsync(list.p + off, parts[b].p, cnt[b] * 4, hipMemcpyDeviceToDevice, s));
        off += cnt[b];
    }
    MMCSF_HIP(hipStreamSynchronize(s));
    dropped = n - tot;
}

// seg[i] = segment containing item i for a pointer array ptr[0..nseg]
__global__ void k_mark_seg(const uint32_t *__restrict__ ptr, uint32_t *__restrict__ mark, uint64_t nseg) {
    uint64_t s = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (s >= 1 && s < nseg) atomicAdd(&mark[ptr[s]], 1u);  // segments are never empty
}

void segment_ids(const uint32_t *ptr, uint64_t nseg, uint64_t nitems, DevArray<uint32_t> &seg,
                 hipStream_t s, Temp &tmp) {
    seg.tmp(nitems);
    if (nitems == 0) return;
    TmpArray<uint32_t> mark(nitems);
    MMCSF_HIP(hipMemsetAsync(mark.p, 0, nitems * 4, s));
    hipLaunchKernelGGL(k_mark_seg, dim3(nblk(nseg)), dim3(kBS), 0, s, ptr, mark.p, nseg);
    size_t bytes = 0;
    MMCSF_HIP(rocprim::inclusive_scan(nullptr, bytes, mark.p, seg.p, (size_t)nitems,
                                      rocprim::plus<uint32_t>(), s));
    MMCSF_HIP(rocprim::inclusive_scan(tmp.get(bytes), bytes, mark.p, seg.p, (size_t)nitems,
                                      rocprim::plus<uint32_t>(), s));
}

}  // namespace

// ---------------------------------------------------------------------------
// order_tensormode, util.h:255-311
// ---------------------------------------------------------------------------
void order_tensormode(int ndims, const uint64_t *dims, int mode, bool nat, int *order) {
    int natMode[kMaxDims], len[kMaxDims];
    bool taken[kMaxDims];
    for (int m = 0; m < ndims; ++m) {
        natMode[m] = (m + mode) % ndims;
        len[m] = (int)dims[natMode[m]];
        taken[m] = false;
    }
    if (nat) {
        for (int i = 0; i < ndims; ++i) order[i] = natMode[i];
        return;
    }
    // ascending lengths of positions 1..N-1; position 0 stays `mode`
    for (int i = 1; i < ndims; i++)
        for (int j = i + 1; j < ndims; j++)
            if (len[i] > len[j]) std::swap(len[i], len[j]);
    order[0] = mode;
    taken[mode] = true;
    for (int i = 1; i < ndims; i++)
        for (int j = 0; j < ndims; j++)
            if ((uint64_t)(int64_t)len[i] == dims[j] && !taken[j]) {
                order[i] = j;
                taken[j] = true;
                break;
            }
}

// ---------------------------------------------------------------------------
// full-key LSD radix sort of the nonzeros
// ---------------------------------------------------------------------------
void sort_coo(const Tensor &t, const int *order, DevArray<uint32_t> *keys, DevArray<float> &vals,
              hipStream_t s, DevArray<uint32_t> *pos, bool keepKeys) {
    const int N = t.ndims;
    const uint64_t n = t.nnz;
    if (n == 0) {
        for (int l = 0; l < N; ++l) keys[l].alloc(0);
        vals.alloc(0);
        if (pos) pos->alloc(0);
        return;
    }
    Temp tmp;
    int bits[kMaxDims];
    for (int l = 0; l < N; ++l) bits[l] = bitwidth(t.dims[order[l]] ? t.dims[order[l]] - 1 : 0);
    // group levels into <=64-bit passes, least significant group first
    std::vector<std::pair<int, int>> groups;  // [lo, hi) level ranges
    int hi = N;
    while (hi > 0) {
        int lo = hi, tot = 0;
        while (lo > 0 && tot + bits[lo - 1] <= 64) { tot += bits[lo - 1]; --lo; }
        if (lo == hi) fail(MMCSF_ERR_UNSUPPORTED, "coordinate wider than 64 bits");
        groups.push_back({lo, hi});
        hi = lo;
    }
    for (int l = 0; l < N; ++l) {
        if (keepKeys || l == N - 1) keys[l].alloc(n);
        else keys[l].tmp(n);
    }
    vals.alloc(n);
    // The sorts carry the permutation, two buffers in turn; the last result is
    // the caller's when it asks for the positions.  One sort without them
    // carries the values themselves.
    const bool carryVals = groups.size() == 1 && !pos;
    DevArray<uint32_t> permA, permB;
    if (!carryVals) {
        if (pos) permA.alloc(n);
        else permA.tmp(n);
        permB.tmp(n);
    }
    DevArray<uint32_t> *cur = groups.size() % 2 ? &permB : &permA, *next = groups.size() % 2 ? &permA : &permB;
    TmpArray<uint64_t> k1(n), k2(n);
    bool first = true;
    for (auto [lo, hi2] : groups) {
        PackSpec ps{};
        int shift = 0;
        ps.nlev = hi2 - lo;
        for (int l = hi2 - 1; l >= lo; --l) {
            ps.src[l - lo] = t.inds[order[l]].p;
            ps.shift[l - lo] = shift;
            shift += bits[l];
        }
        if (first) hipLaunchKernelGGL(k_pack_first, dim3(nblk(n)), dim3(kBS), 0, s, ps, k1.p, cur->p, n);
        else hipLaunchKernelGGL(k_pack, dim3(nblk(n)), dim3(kBS), 0, s, ps, cur->p, k1.p, n);
        first = false;
        size_t bytes = 0;
        if (carryVals) {
            MMCSF_HIP(rocprim::radix_sort_pairs(nullptr, bytes, k1.p, k2.p, t.vals.p, vals.p, (size_t)n, 0u,
                                                (unsigned)shift, s));
            MMCSF_HIP(rocprim::radix_sort_pairs(tmp.get(bytes), bytes, k1.p, k2.p, t.vals.p, vals.p, (size_t)n, 0u,
                                                (unsigned)shift, s));
        } else {
            MMCSF_HIP(rocprim::radix_sort_pairs(nullptr, bytes, k1.p, k2.p, cur->p, next->p, (size_t)n, 0u,
                                                (unsigned)shift, s));
            MMCSF_HIP(rocprim::radix_sort_pairs(tmp.get(bytes), bytes, k1.p, k2.p, cur->p, next->p,
                                                (size_t)n, 0u, (unsigned)shift, s));
            std::swap(cur, next);
        }
        if (lo == 0) {  // the last sort: its keys hold the levels up to hi2
            UnpackSpec us{};
            us.nlev = hi2;
            for (int l = 0; l < hi2; ++l) {
                us.dst[l] = keys[l].p;
                us.shift[l] = ps.shift[l];
                us.mask[l] = (uint32_t)((1ull << bits[l]) - 1);
            }
            hipLaunchKernelGGL(k_unpack, dim3(nblk(n)), dim3(kBS), 0, s, us, k2.p, n);
            for (int l = hi2; l < N; ++l)
                hipLaunchKernelGGL(k_gather_u32, dim3(nblk(n)), dim3(kBS), 0, s, t.inds[order[l]].p, cur->p,
                                   keys[l].p, n);
        }
    }
    if (!carryVals)
        hipLaunchKernelGGL(k_gather_f32, dim3(nblk(n)), dim3(kBS), 0, s, t.vals.p, cur->p, vals.p, n);
    MMCSF_HIP(hipGetLastError());
    MMCSF_HIP(hipStreamSynchronize(s));
    if (pos) *pos = std::move(permA);
}

// ---------------------------------------------------------------------------
// CSF scan (create_TiledHCSR semantics)
// ---------------------------------------------------------------------------
void build_csf(int N, const uint64_t *dims, uint64_t n, const int *order, DevArray<uint32_t> *keys,
               DevArray<float> &&vals, uint64_t fthr, uint64_t fsthr, Csf &c, hipStream_t s) {
    Temp tmp;
    c.ndims = N;
    for (int l = 0; l < N; ++l) {
        c.order[l] = order[l];
        c.rows[l] = dims[order[l]];
    }
    c.nnz = n;
    if (n == 0) {
        for (int l = 0; l < N - 1; ++l) {
            c.cnt[l] = 0;
            c.ptr[l].alloc(1);
            hipLaunchKernelGGL(k_set, dim3(1), dim3(1), 0, s, c.ptr[l].p, 0, 0u);
        }
        c.cnt[N - 1] = 0;
        MMCSF_HIP(hipStreamSynchronize(s));
        return;
    }
    if (fthr < 1) fthr = 1;  // -f 0 behaves like -f 1 (util.h:1364: fiberNnz starts at 1)
    Keys K{};
    for (int l = 0; l < N; ++l) K.k[l] = keys[l].p;
    TmpArray<uint8_t> d(n);
    TmpArray<uint32_t> a(n), b(n);  // a: run positions -> run starts; b: flags
    hipLaunchKernelGGL(k_first_diff, dim3(nblk(n)), dim3(kBS), 0, s, K, N, d.p, a.p, n);
    const uint32_t *runStart = nullptr;
    DevArray<uint32_t> rs;
    if (fthr < n) {
        rs.tmp(n);
        inclusive_max(a.p, rs.p, n, s, tmp);
        runStart = rs.p;
    }
    hipLaunchKernelGGL(k_leaf_flag, dim3(nblk(n)), dim3(kBS), 0, s, d.p, runStart, N, fthr, b.p, n);
    rs.release();
    // leaf-fiber ordinals
    uint64_t nLeaf = exclusive_sum(b.p, a.p, n, s, tmp);
    const int LL = N - 2;  // leaf-fiber level
    c.ptr[LL].alloc(nLeaf + 1);
    c.idx[LL].alloc(nLeaf);
    TmpArray<uint8_t> dF(nLeaf);
    hipLaunchKernelGGL(k_scatter_leaf, dim3(nblk(n)), dim3(kBS), 0, s, b.p, a.p, d.p, keys[LL].p,
                       c.ptr[LL].p, c.idx[LL].p, dF.p, n);
    hipLaunchKernelGGL(k_set, dim3(1), dim3(1), 0, s, c.ptr[LL].p, nLeaf, (uint32_t)n);
    c.cnt[LL] = nLeaf;
    d.release();
    a.release();
    b.release();

    TmpArray<uint32_t> flag(nLeaf), ord(nLeaf);
    if (N == 3) {
        // slices over leaf fibers
        hipLaunchKernelGGL(k_level_flag, dim3(nblk(nLeaf)), dim3(kBS), 0, s, dF.p, 0, flag.p, nLeaf);
        uint64_t nS = exclusive_sum(flag.p, ord.p, nLeaf, s, tmp);
        c.ptr[0].alloc(nS + 1);
        c.idx[0].alloc(nS);
        hipLaunchKernelGGL(k_scatter_upper, dim3(nblk(nLeaf)), dim3(kBS), 0, s, flag.p, ord.p,
                           (const uint32_t *)nullptr, c.ptr[LL].p, keys[0].p, c.ptr[0].p, c.idx[0].p,
                           (const uint32_t *)nullptr, (uint32_t *)nullptr, nLeaf);
        hipLaunchKernelGGL(k_set, dim3(1), dim3(1), 0, s, c.ptr[0].p, nS, (uint32_t)nLeaf);
        c.cnt[0] = nS;
        // fbrLikeSlcInds: slice coordinate of every fiber = key0 at its start
        c.fbrSlc.alloc(nLeaf);
        hipLaunchKernelGGL(k_gather_u32, dim3(nblk(nLeaf)), dim3(kBS), 0, s, keys[0].p, c.ptr[LL].p,
                           c.fbrSlc.p, nLeaf);
    } else {
        // level 1 (fbrS): key change at level <= 1, plus the 128-nnz split
        TmpArray<uint32_t> jflag(nLeaf);
        hipLaunchKernelGGL(k_level_flag, dim3(nblk(nLeaf)), dim3(kBS), 0, s, dF.p, 1, flag.p, nLeaf);
        if (fsthr < n) {
            uint64_t nRuns = exclusive_sum(flag.p, ord.p, nLeaf, s, tmp);
            TmpArray<uint32_t> runs(nRuns);
            hipLaunchKernelGGL(k_compact_idx, dim3(nblk(nLeaf)), dim3(kBS), 0, s, flag.p, ord.p, runs.p,
                               nLeaf);
            hipLaunchKernelGGL(k_fbrs_split, dim3(nblk(nRuns)), dim3(kBS), 0, s, runs.p, nRuns, nLeaf,
                               c.ptr[LL].p, fsthr, jflag.p);
        } else {
            MMCSF_HIP(hipMemcpyAsync(jflag.p, flag.p, nLeaf * 4, hipMemcpyDeviceToDevice, s));
        }
        uint64_t nJ = exclusive_sum(jflag.p, ord.p, nLeaf, s, tmp);
        c.ptr[1].alloc(nJ + 1);
        c.idx[1].alloc(nJ);
        c.fbrSlc.alloc(nJ);
        hipLaunchKernelGGL(k_scatter_upper, dim3(nblk(nLeaf)), dim3(kBS), 0, s, jflag.p, ord.p,
                           (const uint32_t *)nullptr, c.ptr[LL].p, keys[1].p, c.ptr[1].p, c.idx[1].p,
                           keys[0].p, c.fbrSlc.p, nLeaf);
        hipLaunchKernelGGL(k_set, dim3(1), dim3(1), 0, s, c.ptr[1].p, nJ, (uint32_t)nLeaf);
        c.cnt[1] = nJ;
        // level 0 (slices): ptr0 = fbrS ordinal of the slice's first leaf fiber
        TmpArray<uint32_t> sord(nLeaf);
        hipLaunchKernelGGL(k_level_flag, dim3(nblk(nLeaf)), dim3(kBS), 0, s, dF.p, 0, flag.p, nLeaf);
        uint64_t nS = exclusive_sum(flag.p, sord.p, nLeaf, s, tmp);
        c.ptr[0].alloc(nS + 1);
        c.idx[0].alloc(nS);
        hipLaunchKernelGGL(k_scatter_upper, dim3(nblk(nLeaf)), dim3(kBS), 0, s, flag.p, sord.p, ord.p,
                           c.ptr[LL].p, keys[0].p, c.ptr[0].p, c.idx[0].p, (const uint32_t *)nullptr,
                           (uint32_t *)nullptr, nLeaf);
        hipLaunchKernelGGL(k_set, dim3(1), dim3(1), 0, s, c.ptr[0].p, nS, (uint32_t)nJ);
        c.cnt[0] = nS;
    }
    c.cnt[N - 1] = n;
    c.leaf = std::move(keys[N - 1]);
    c.vals = std::move(vals);
    for (int l = 0; l < N - 1; ++l) keys[l].release();
    MMCSF_HIP(hipStreamSynchronize(s));
    build_walk_bits(c, s);
}

__global__ void k_word_pop(const uint32_t *__restrict__ bits, uint64_t words, uint32_t *__restrict__ cnt) {
    uint64_t w = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (w < words) cnt[w] = (uint32_t)(__popc(bits[2 * w]) + __popc(bits[2 * w + 1]));
}

bool build_walk_ranks(Csf &c, hipStream_t s, bool check) {
    const int N = c.ndims;
    const uint64_t n = c.nnz, nL = c.cnt[N - 2];
    if (n == 0) return true;
    Temp tmp;
    auto ranks = [&](const DevArray<uint32_t> &bits, uint64_t items, uint64_t starts, DevArray<uint32_t> &rank) {
        const uint64_t words = (items + 63) / 64;
        rank.alloc(words);
        TmpArray<uint32_t> cnt(words);
        hipLaunchKernelGGL(k_word_pop, dim3(nblk(words)), dim3(kBS), 0, s, bits.p, words, cnt.p);
        if (check) return exclusive_sum(cnt.p, rank.p, words, s, tmp) == starts;
        size_t bytes = 0;
        MMCSF_HIP(rocprim::exclusive_scan(nullptr, bytes, cnt.p, rank.p, 0u, (size_t)words,
                                          rocprim::plus<uint32_t>(), s));
        MMCSF_HIP(rocprim::exclusive_scan(tmp.get(bytes), bytes, cnt.p, rank.p, 0u, (size_t)words,
                                          rocprim::plus<uint32_t>(), s));
        return true;
    };
    bool ok = ranks(c.fbit, n, nL, c.frank);
    if (N == 4) ok = ranks(c.sbit, nL, c.cnt[1], c.jrank) && ok;
    return ok;
}

// ---------------------------------------------------------------------------
// start bitmasks for the chunked root traversal: bit x of fbit = nonzero x
// starts a leaf fiber; 4-D: bit f of sbit = leaf fiber f starts a level-1
// entry.  Word arrays carry two spare words so 64-entry windows never read
// past the end.
// ---------------------------------------------------------------------------
void build_walk_bits(Csf &c, hipStream_t s) {
    const int N = c.ndims;
    const uint64_t n = c.nnz, nL = c.cnt[N - 2];
    auto mark = [&](DevArray<uint32_t> &bits, uint64_t items, const uint32_t *ptr, uint64_t nptr) {
        const uint64_t words = items / 32 + 3;
        bits.alloc(words);
        hipLaunchKernelGGL(k_zero_words, dim3(nblk(words)), dim3(kBS), 0, s, bits.p, words);
        if (nptr)
            hipLaunchKernelGGL(k_mark_starts, dim3((unsigned)((nptr + kMarkEntries - 1) / kMarkEntries)), dim3(kBS), 0, s,
                               ptr, nptr, bits.p);
    };
    mark(c.fbit, n, c.ptr[N - 2].p, nL);
    if (N == 4) mark(c.sbit, nL, c.ptr[1].p, c.cnt[1]);
    (void)build_walk_ranks(c, s);
    // cost prefix over chunks: waves split the traversal by cost, not by
    // nonzeros (chunks where many slices start take longer)
    const uint64_t chunks = (n + 63) / 64;
    c.chunkCost.alloc(chunks + 1);
    if (chunks) {
        Temp tmp;
        TmpArray<uint32_t> cnt(chunks), cost(chunks);
        hipLaunchKernelGGL(k_zero_words, dim3(nblk(chunks)), dim3(kBS), 0, s, cnt.p, chunks);
        if (c.cnt[0])
            hipLaunchKernelGGL(k_chunk_starts, dim3(nblk(c.cnt[0])), dim3(kBS), 0, s, N, c.ptr[0].p, c.ptr[1].p,
                               N == 4 ? c.ptr[2].p : (const uint32_t *)nullptr, c.cnt[0], cnt.p);
        // the weighted total (at most chunks * 64 (1 + wf) + ws * slices, every
        // slice starting in one chunk) must fit the 32-bit prefix; else split
        // by chunks
        const uint32_t wf = 1, ws = 24;
        const bool plain = chunks * 64ull * (1 + wf) + ws * (uint64_t)c.cnt[0] >= 0xF0000000ull;
        hipLaunchKernelGGL(k_chunk_cost, dim3(nblk(chunks)), dim3(kBS), 0, s, cnt.p, c.fbit.p, chunks, plain, wf, ws,
                           cost.p);
        uint64_t total = exclusive_sum(cost.p, c.chunkCost.p, chunks, s, tmp);
        hipLaunchKernelGGL(k_set, dim3(1), dim3(1), 0, s, c.chunkCost.p, chunks, (uint32_t)total);
    } else {
        hipLaunchKernelGGL(k_set, dim3(1), dim3(1), 0, s, c.chunkCost.p, 0, 0u);
    }
    MMCSF_HIP(hipGetLastError());
    MMCSF_HIP(hipStreamSynchronize(s));
}

// rows of sorted nonzeros starting in each 64-nonzero chunk, as the chunk's cost
// (64, and ws per start: row writes and the join of the group runs)
__global__ void k_row_cost(const uint32_t *__restrict__ key, uint64_t n, bool plain, uint32_t ws,
                           uint32_t *__restrict__ cost) {
    const uint64_t x = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    const bool starts = x < n && (x == 0 || key[x] != key[x - 1]);
    const uint64_t m = __ballot(starts);
    if (x < n && (threadIdx.x & 63) == 0) cost[x >> 6] = plain ? 1u : 64u + ws * (uint32_t)__popcll(m);
}

void build_row_cost(const uint32_t *key, uint64_t n, uint64_t rows, DevArray<uint32_t> &prefix, hipStream_t s) {
    const uint64_t chunks = (n + 63) / 64;
    prefix.alloc(chunks + 1);
    Temp tmp;
    TmpArray<uint32_t> cost(chunks + 1);
    const uint32_t ws = 24;  // as for the trees
    const bool plain = chunks * 64 + ws * std::min(n, rows) >= 0xF0000000ull;
    // the entry past the chunks costs nothing: the scan over it leaves the total
    // there, and the host need not read it
    hipLaunchKernelGGL(k_set, dim3(1), dim3(1), 0, s, cost.p, chunks, 0u);
    if (n) hipLaunchKernelGGL(k_row_cost, dim3(nblk(n)), dim3(kBS), 0, s, key, n, plain, ws, cost.p);
    size_t bytes = 0;
    MMCSF_HIP(rocprim::exclusive_scan(nullptr, bytes, cost.p, prefix.p, 0u, (size_t)(chunks + 1),
                                      rocprim::plus<uint32_t>(), s));
    MMCSF_HIP(rocprim::exclusive_scan(tmp.get(bytes), bytes, cost.p, prefix.p, 0u, (size_t)(chunks + 1),
                                      rocprim::plus<uint32_t>(), s));
    MMCSF_HIP(hipGetLastError());
    MMCSF_HIP(hipStreamSynchronize(s));
}

// ---------------------------------------------------------------------------
// make_TiledBin (util.h:1887-1952)
// ---------------------------------------------------------------------------
void build_bins_tiled(Csf &c, hipStream_t s) {
    Temp tmp;
    uint64_t nS = c.cnt[0];
    TmpArray<int8_t> bin(nS);
    if (nS)
        hipLaunchKernelGGL(k_slice_bin, dim3(nblk(nS)), dim3(kBS), 0, s, c.ndims, c.ptr[0].p, c.ptr[1].p,
                           c.ndims == 4 ? c.ptr[2].p : (const uint32_t *)nullptr, true, bin_bounds(c.nnz),
                           bin.p, nS);
    bin_lists(bin.p, nS, c.binList, c.binCount, c.dropped, s, tmp);
    c.hasBins = true;
}

// ---------------------------------------------------------------------------
// create_HYB / create_HYB_4D + make_HybBin
// ---------------------------------------------------------------------------
namespace {

enum : uint8_t { kCOO = 0, kCSL = 1, kCSF = 2 };

// per slice: class, nnz, non-CSF nnz (for the shift), COO/CSL/CSF flags
__global__ void k_hyb_class(int N, const uint32_t *__restrict__ p0, const uint32_t *__restrict__ p1,
                            const uint32_t *__restrict__ p2, uint8_t *__restrict__ cls,
                            uint32_t *__restrict__ fCoo, uint32_t *__restrict__ fCsl,
                            uint32_t *__restrict__ fCsf, uint32_t *__restrict__ nzCsl,
                            uint32_t *__restrict__ nzSub, uint64_t nslc) {
    uint64_t s = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (s >= nslc) return;
    uint32_t a = p0[s], b = p0[s + 1];
    uint64_t nLeafF, nz;
    if (N == 3) {
        nLeafF = b - a;
        nz = (uint64_t)p1[b] - p1[a];
    } else {
        nLeafF = (uint64_t)p1[b] - p1[a];
        nz = (uint64_t)p2[p1[b]] - p2[p1[a]];
    }
    uint8_t k;
    if (nz == 1) k = kCOO;                        // util.h:883 / 1026
    else if (N == 3 && nz == nLeafF) k = kCSL;    // every fiber of length 1 (util.h:885)
    else k = kCSF;
    cls[s] = k;
    fCoo[s] = k == kCOO;
    fCsl[s] = k == kCSL;
    fCsf[s] = k == kCSF;
    nzCsl[s] = k == kCSL ? (uint32_t)nz : 0u;
    // fibers (= nonzeros) consumed by COO / CSL slices (util.h:957, 1104)
    nzSub[s] = k == kCSF ? 0u : (uint32_t)nz;
}

struct HybOut {
    uint32_t *cooInd[kMaxDims];
    float *cooVal;
    uint32_t *cslPtr, *cslIdx, *cslInd1, *cslInd2;
    float *cslVal;
    uint32_t *hPtr[kMaxDims - 1], *hIdx[kMaxDims - 1];
    uint32_t *hLeaf;
    float *hVal;
};

struct CsfIn {
    const uint32_t *ptr[kMaxDims - 1], *idx[kMaxDims - 1];
    const uint32_t *leaf;
    const float *vals;
};

// slice-level outputs: COO entries, CSL slice pointers, CSF slice pointers
__global__ void k_hyb_slices(int N, CsfIn in, const uint8_t *__restrict__ cls,
                             const uint32_t *__restrict__ oCoo, const uint32_t *__restrict__ oCsl,
                             const uint32_t *__restrict__ oCsf, const uint32_t *__restrict__ cslOff,
                             const uint32_t *__restrict__ sub, HybOut o, uint64_t nslc) {
    uint64_t s = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (s >= nslc) return;
    uint32_t a = in.ptr[0][s];
    uint8_t k = cls[s];
    if (k == kCOO) {
        uint32_t c = oCoo[s];
        uint32_t leafF = (N == 3) ? a : in.ptr[1][a];
        uint32_t x = in.ptr[N - 2][leafF];
        o.cooInd[0][c] = in.idx[0][s];
        o.cooInd[1][c] = in.idx[1][a];
        if (N == 4) o.cooInd[2][c] = in.idx[2][leafF];
        o.cooInd[N - 1][c] = in.leaf[x];
        o.cooVal[c] = in.vals[x];
    } else if (k == kCSL) {
        uint32_t c = oCsl[s];
        o.cslPtr[c] = cslOff[s];
        o.cslIdx[c] = in.idx[0][s];
    } else {
        uint32_t c = oCsf[s];
        o.hPtr[0][c] = a - sub[s];
        o.hIdx[0][c] = in.idx[0][s];
    }
}

// level-1 entries (3-D: fibers; 4-D: fbrS) of CSL / CSF slices
__global__ void k_hyb_lvl1(int N, CsfIn in, const uint32_t *__restrict__ slcOf,
                           const uint8_t *__restrict__ cls, const uint32_t *__restrict__ cslOff,
                           const uint32_t *__restrict__ sub, HybOut o, uint64_t n1) {
    uint64_t j = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (j >= n1) return;
    uint32_t s = slcOf[j];
    uint8_t k = cls[s];
    if (k == kCSL) {  // 3-D only: one nonzero per fiber
        uint32_t pos = cslOff[s] + (uint32_t)(j - in.ptr[0][s]);
        uint32_t x = in.ptr[1][j];
        o.cslInd1[pos] = in.idx[1][j];
        o.cslInd2[pos] = in.leaf[x];
        o.cslVal[pos] = in.vals[x];
    } else if (k == kCSF) {
        uint32_t nj = (uint32_t)j - sub[s];
        o.hPtr[1][nj] = in.ptr[1][j] - sub[s];
        o.hIdx[1][nj] = in.idx[1][j];
    }
}

// 4-D leaf fibers of CSF slices
__global__ void k_hyb_lvl2(CsfIn in, const uint32_t *__restrict__ slcOf2,
                           const uint8_t *__restrict__ cls, const uint32_t *__restrict__ sub, HybOut o,
                           uint64_t n2) {
    uint64_t f = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (f >= n2) return;
    uint32_t s = slcOf2[f];
    if (cls[s] != kCSF) return;
    uint32_t nf = (uint32_t)f - sub[s];
    o.hPtr[2][nf] = in.ptr[2][f] - sub[s];
    o.hIdx[2][nf] = in.idx[2][f];
}

__global__ void k_hyb_nnz(CsfIn in, const uint32_t *__restrict__ slcOfNnz, const uint8_t *__restrict__ cls,
                          const uint32_t *__restrict__ sub, HybOut o, uint64_t n) {
    uint64_t x = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (x >= n) return;
    uint32_t s = slcOfNnz[x];
    if (cls[s] != kCSF) return;
    uint32_t nx = (uint32_t)x - sub[s];
    o.hLeaf[nx] = in.leaf[x];
    o.hVal[nx] = in.vals[x];
}

// compose two segment maps: out[i] = outer[inner[i]]
__global__ void k_compose(const uint32_t *__restrict__ inner, const uint32_t *__restrict__ outer,
                          uint32_t *__restrict__ out, uint64_t n) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i < n) out[i] = outer[inner[i]];
}

}  // namespace

// level-1 entry x of the CSL walk tree (one per nonzero) takes its slice's
// coordinate
__global__ void k_csl_slice_of(const uint32_t *__restrict__ ptr, const uint32_t *__restrict__ idx, uint64_t nS,
                               uint32_t *slc) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i >= nS) return;
    for (uint32_t x = ptr[i]; x < ptr[i + 1]; ++x) slc[x] = idx[i];
}

// The CSL part (slices whose leaf fibers all hold one nonzero) is a CSF tree
// with one level-1 entry per nonzero: ptr[0] = cslPtr, idx[0] = cslIdx,
// ptr[1] = 0, 1, ..., idx[1] = cslInd1, leaf = cslInd2.  Walked by the chunked
// root walk like the CSF part; the CSL arrays themselves stay as built.
void build_csl_walk(Hyb &h, hipStream_t s) {
    Csf &t = h.cslWalk;
    t = Csf{};
    if (h.ndims != 3 || h.cslNnz == 0) return;
    const uint64_t n = h.cslNnz, nS = h.nCsl;
    t.ndims = 3;
    for (int l = 0; l < 3; ++l) {
        t.order[l] = h.order[l];
        t.rows[l] = h.csf.rows[l];
    }
    t.nnz = n;
    t.cnt[0] = nS;
    t.cnt[1] = n;
    t.cnt[2] = n;
    auto copy = [&](DevArray<uint32_t> &dst, const uint32_t *src, uint64_t count) {
        dst.alloc(count);
        MMCSF_HIP(hipMemcpyAsync(dst.p, src, count * 4, hipMemcpyDeviceToDevice, s));
    };
    copy(t.ptr[0], h.cslPtr.p, nS + 1);
    copy(t.idx[0], h.cslIdx.p, nS);
    t.ptr[1].alloc(n + 1);
    hipLaunchKernelGGL(k_iota, dim3(nblk(n + 1)), dim3(kBS), 0, s, t.ptr[1].p, n + 1);
    copy(t.idx[1], h.cslInd1.p, n);
    copy(t.leaf, h.cslInd2.p, n);
    t.vals.alloc(n);
    MMCSF_HIP(hipMemcpyAsync(t.vals.p, h.cslVal.p, n * 4, hipMemcpyDeviceToDevice, s));
    t.fbrSlc.alloc(n);
    hipLaunchKernelGGL(k_csl_slice_of, dim3(nblk(nS)), dim3(kBS), 0, s, h.cslPtr.p, h.cslIdx.p, nS, t.fbrSlc.p);
    MMCSF_HIP(hipGetLastError());
    MMCSF_HIP(hipStreamSynchronize(s));
    build_walk_bits(t, s);
}

void build_hyb(int N, const uint64_t *dims, Csf &&src, Hyb &h, hipStream_t s) {
    (void)dims;
    Temp tmp;
    h.ndims = N;
    for (int l = 0; l < N; ++l) h.order[l] = src.order[l];
    const uint64_t n = src.nnz;
    const uint64_t nS = src.cnt[0];
    const uint64_t n1 = src.cnt[1];
    const uint64_t nL = src.cnt[N - 2];
    TmpArray<uint8_t> cls(nS);
    TmpArray<uint32_t> fCoo(nS), fCsl(nS), fCsf(nS), nzCsl(nS), nzSub(nS);
    TmpArray<uint32_t> oCoo(nS), oCsl(nS), oCsf(nS), cslOff(nS), sub(nS);
    if (nS)
        hipLaunchKernelGGL(k_hyb_class, dim3(nblk(nS)), dim3(kBS), 0, s, N, src.ptr[0].p, src.ptr[1].p,
                           N == 4 ? src.ptr[2].p : (const uint32_t *)nullptr, cls.p, fCoo.p, fCsl.p,
                           fCsf.p, nzCsl.p, nzSub.p, nS);
    uint64_t nCoo = exclusive_sum(fCoo.p, oCoo.p, nS, s, tmp);
    uint64_t nCsl = exclusive_sum(fCsl.p, oCsl.p, nS, s, tmp);
    uint64_t nCsf = exclusive_sum(fCsf.p, oCsf.p, nS, s, tmp);
    uint64_t cslNnz = exclusive_sum(nzCsl.p, cslOff.p, nS, s, tmp);
    uint64_t subTot = exclusive_sum(nzSub.p, sub.p, nS, s, tmp);
    h.cooNnz = nCoo;
    h.cslNnz = cslNnz;
    h.nCsl = nCsl;
    for (int l = 0; l < N; ++l) h.cooInd[l].alloc(nCoo);
    h.cooVal.alloc(nCoo);
    h.cslPtr.alloc(nCsl + 1);
    h.cslIdx.alloc(nCsl);
    h.cslInd1.alloc(cslNnz);
    h.cslInd2.alloc(cslNnz);
    h.cslVal.alloc(cslNnz);
    // CSF part sizes: every non-CSF slice consumes exactly one entry per level
    // for COO (4-D) and one fiber per nonzero for CSL (3-D)
    Csf &c = h.csf;
    c.ndims = N;
    for (int l = 0; l < N; ++l) {
        c.order[l] = src.order[l];
        c.rows[l] = src.rows[l];
    }
    c.nnz = n - subTot;
    c.cnt[0] = nCsf;
    if (N == 3) {
        c.cnt[1] = nL - subTot;
    } else {
        c.cnt[1] = n1 - subTot;  // a 4-D non-CSF slice is a COO slice: one fbrS
        c.cnt[2] = nL - subTot;
    }
    c.cnt[N - 1] = c.nnz;
    for (int l = 0; l < N - 1; ++l) {
        c.ptr[l].alloc(c.cnt[l] + 1);
        c.idx[l].alloc(c.cnt[l]);
    }
    c.leaf.alloc(c.nnz);
    c.vals.alloc(c.nnz);

    HybOut o{};
    for (int l = 0; l < N; ++l) o.cooInd[l] = h.cooInd[l].p;
    o.cooVal = h.cooVal.p;
    o.cslPtr = h.cslPtr.p;
    o.cslIdx = h.cslIdx.p;
    o.cslInd1 = h.cslInd1.p;
    o.cslInd2 = h.cslInd2.p;
    o.cslVal = h.cslVal.p;
    for (int l = 0; l < N - 1; ++l) { o.hPtr[l] = c.ptr[l].p; o.hIdx[l] = c.idx[l].p; }
    o.hLeaf = c.leaf.p;
    o.hVal = c.vals.p;
    CsfIn in{};
    for (int l = 0; l < N - 1; ++l) { in.ptr[l] = src.ptr[l].p; in.idx[l] = src.idx[l].p; }
    in.leaf = src.leaf.p;
    in.vals = src.vals.p;

    if (nS)
        hipLaunchKernelGGL(k_hyb_slices, dim3(nblk(nS)), dim3(kBS), 0, s, N, in, cls.p, oCoo.p, oCsl.p,
                           oCsf.p, cslOff.p, sub.p, o, nS);
    // level-1 entries
    DevArray<uint32_t> slcOf1;
    segment_ids(src.ptr[0].p, nS, n1, slcOf1, s, tmp);
    if (n1)
        hipLaunchKernelGGL(k_hyb_lvl1, dim3(nblk(n1)), dim3(kBS), 0, s, N, in, slcOf1.p, cls.p, cslOff.p,
                           sub.p, o, n1);
    DevArray<uint32_t> slcOfLeafF;
    if (N == 4) {
        DevArray<uint32_t> jOf2;
        segment_ids(src.ptr[1].p, n1, nL, jOf2, s, tmp);
        slcOfLeafF.tmp(nL);
        if (nL)
            hipLaunchKernelGGL(k_compose, dim3(nblk(nL)), dim3(kBS), 0, s, jOf2.p, slcOf1.p, slcOfLeafF.p,
                               nL);
        if (nL)
            hipLaunchKernelGGL(k_hyb_lvl2, dim3(nblk(nL)), dim3(kBS), 0, s, in, slcOfLeafF.p, cls.p, sub.p,
                               o, nL);
    } else {
        slcOfLeafF = std::move(slcOf1);
    }
    // nonzeros
    {
        DevArray<uint32_t> fOfNnz;
        TmpArray<uint32_t> slcOfNnz(n);
        segment_ids(src.ptr[N - 2].p, nL, n, fOfNnz, s, tmp);
        if (n)
            hipLaunchKernelGGL(k_compose, dim3(nblk(n)), dim3(kBS), 0, s, fOfNnz.p, slcOfLeafF.p,
                               slcOfNnz.p, n);
        if (n)
            hipLaunchKernelGGL(k_hyb_nnz, dim3(nblk(n)), dim3(kBS), 0, s, in, slcOfNnz.p, cls.p, sub.p, o,
                               n);
    }
    // closing entries (util.h:976-978, 1125-1127)
    hipLaunchKernelGGL(k_set, dim3(1), dim3(1), 0, s, c.ptr[N - 2].p, c.cnt[N - 2], (uint32_t)c.nnz);
    for (int l = N - 3; l >= 0; --l)
        hipLaunchKernelGGL(k_set, dim3(1), dim3(1), 0, s, c.ptr[l].p, c.cnt[l], (uint32_t)c.cnt[l + 1]);
    hipLaunchKernelGGL(k_set, dim3(1), dim3(1), 0, s, h.cslPtr.p, nCsl, (uint32_t)cslNnz);
    // fbrLikeSlcInds of the CSF part (used by the kernels)
    {
        DevArray<uint32_t> so;
        segment_ids(c.ptr[0].p, c.cnt[0], c.cnt[1], so, s, tmp);
        c.fbrSlc.alloc(c.cnt[1]);
        if (c.cnt[1])
            hipLaunchKernelGGL(k_compose, dim3(nblk(c.cnt[1])), dim3(kBS), 0, s, so.p, c.idx[0].p,
                               c.fbrSlc.p, c.cnt[1]);
    }
    // bins: CSF slices by nnz (make_HybBin), CSL slices by nnz
    {
        TmpArray<int8_t> bin(c.cnt[0]);
        if (c.cnt[0])
            hipLaunchKernelGGL(k_slice_bin, dim3(nblk(c.cnt[0])), dim3(kBS), 0, s, N, c.ptr[0].p,
                               c.ptr[1].p, N == 4 ? c.ptr[2].p : (const uint32_t *)nullptr, false,
                               bin_bounds(n), bin.p, c.cnt[0]);
        bin_lists(bin.p, c.cnt[0], c.binList, c.binCount, c.dropped, s, tmp);
        c.hasBins = true;
        TmpArray<int8_t> cb(nCsl);
        if (nCsl)
            hipLaunchKernelGGL(k_csl_bin, dim3(nblk(nCsl)), dim3(kBS), 0, s, h.cslPtr.p, bin_bounds(n), cb.p,
                               nCsl);
        uint64_t cdrop = 0;
        bin_lists(cb.p, nCsl, h.cslBinList, h.cslBinCount, cdrop, s, tmp);
    }
    MMCSF_HIP(hipStreamSynchronize(s));
    build_walk_bits(c, s);
    // the source CSF is consumed
    Csf dead = std::move(src);
    (void)dead;
}


// ---------------------------------------------------------------------------
// Level maps: the nonzeros of a tree in the order of one level's coordinates.
// ---------------------------------------------------------------------------
namespace {

// coordinate of level `lvl` (an index level) of every stored nonzero
__global__ void k_level_coord(int N, int lvl, uint32_t fibers, const uint32_t *__restrict__ fbit,
                              const uint32_t *__restrict__ frank,
                              const uint32_t *__restrict__ sbit, const uint32_t *__restrict__ jrank,
                              const uint32_t *__restrict__ idx, uint32_t entries, uint64_t n,
                              uint32_t *__restrict__ key, uint32_t *__restrict__ pos) {
    uint64_t x = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (x >= n) return;
    pos[x] = (uint32_t)x;
    if (!idx) return;
    // (a loaded file's bits are not to be trusted with an index)
    uint32_t e = min(dev::rank_of(fbit, frank, (uint32_t)x), fibers - 1);
    if (N == 4 && lvl == 1) e = dev::rank_of(sbit, jrank, e);
    key[x] = idx[min(e, entries - 1)];
}

}  // namespace

void build_level_maps(Csf &c, hipStream_t s) {
    const int N = c.ndims;
    const uint64_t n = c.nnz, nL = c.cnt[N - 2];
    if (n == 0) return;
    Temp tmp;
    TmpArray<uint32_t> pos(n), key(n), sorted(n);
    for (int l = 1; l < N; ++l) {
        const bool leaf = l == N - 1;
        hipLaunchKernelGGL(k_level_coord, dim3(nblk(n)), dim3(kBS), 0, s, N, l, (uint32_t)nL, c.fbit.p, c.frank.p,
                           c.sbit.p, c.jrank.p, leaf ? (const uint32_t *)nullptr : c.idx[l].p,
                           leaf ? 1u : (uint32_t)c.cnt[l], n, key.p, pos.p);
        c.map[l].ord.alloc(n);
        const uint32_t *k = leaf ? c.leaf.p : key.p;
        const unsigned bits = (unsigned)bitwidth(c.rows[l] ? c.rows[l] - 1 : 0);
        size_t bytes = 0;
        MMCSF_HIP(rocprim::radix_sort_pairs(nullptr, bytes, k, sorted.p, pos.p, c.map[l].ord.p, (size_t)n, 0u, bits, s));
        MMCSF_HIP(rocprim::radix_sort_pairs(tmp.get(bytes), bytes, k, sorted.p, pos.p, c.map[l].ord.p, (size_t)n, 0u,
                                            bits, s));
        build_row_cost(sorted.p, n, c.rows[l], c.map[l].cost, s);
    }
}

namespace {

// Row counts of one mode.  What bounds a plain histogram is the hot rows: on a
// Zipf(1.2) mode the top row takes ~18 % of the increments, and global atomics
// on one address run one after another (20M nonzeros: 37 ms).  Every block
// therefore counts in an LDS table of kHistSlots (row, count) pairs, hashed by
// row and claimed first come, first served (a hot row comes within the first
// elements), and adds each pair to the global counts once; rows that find
// their slot taken are cold and go to the global counts directly.
// 20M nonzeros in 500000 rows, Zipf(1.2): 37.5 ms with plain atomics, 0.34 here.
constexpr int kHistThreads = 1024;
constexpr uint32_t kHistBits = 13, kHistSlots = 1u << kHistBits;
constexpr uint32_t kNoRow = 0xffffffffu;  // coordinates are below 2^31
__global__ __launch_bounds__(kHistThreads) void k_hist_cached(const uint32_t *__restrict__ idx, uint64_t n,
                                                              uint32_t *__restrict__ cnt) {
    __shared__ uint32_t row[kHistSlots], num[kHistSlots];
    for (uint32_t i = threadIdx.x; i < kHistSlots; i += kHistThreads) {
        row[i] = kNoRow;
        num[i] = 0;
    }
    __syncthreads();
    for (uint64_t i = blockIdx.x * (uint64_t)kHistThreads + threadIdx.x; i < n; i += (uint64_t)gridDim.x * kHistThreads) {
        const uint32_t v = idx[i];
        const uint32_t slot = (v * 2654435761u) >> (32 - kHistBits);
        uint32_t owner = row[slot];
        if (owner == kNoRow) {
            owner = atomicCAS(&row[slot], kNoRow, v);
            if (owner == kNoRow) owner = v;
        }
        if (owner == v) atomicAdd(&num[slot], 1u);
        else atomicAdd(&cnt[v], 1u);
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < kHistSlots; i += kHistThreads)
        if (num[i]) atomicAdd(&cnt[row[i]], num[i]);
}

// out = the number of leading entries (counts in descending order, prefix =
// their inclusive sums) it takes to reach `want`
__global__ void k_reach(const uint64_t *__restrict__ prefix, uint64_t rows, double want, uint32_t *out) {
    const uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i >= rows) return;
    const double before = i ? (double)prefix[i - 1] : 0.0;
    if (before < want && (i + 1 == rows || (double)prefix[i] >= want)) *out = (uint32_t)(i + 1);
}

// The distinct pairs of two modes' coordinates among the nonzeros, for the mode
// pairs (0,1), (0,2), (1,2), estimated from the pairs whose hash starts with
// `shift` zero bits: a pair is in the sample or not with all its nonzeros, so
// the sample's distinct pairs times 2^shift is the estimate.  `shift` leaves
// 2^(kPairBits - 1) to 2^kPairBits nonzeros in the sample, so its pairs are that
// times the pairs per nonzero, and the estimate's standard deviation is one over
// their square root: 0.5 % where nearly every nonzero is a pair of its own, 1 % at
// 0.19 pairs per nonzero.  (The multipliers that mix the two coordinates are odd
// and arbitrary: the fraction bits of the square roots of 2, 3, 5 and 7.)  One
// pass over the index arrays, four nonzeros per lane and load.  Sampled pairs wait in an LDS
// queue per wave (coordinates are below 2^31: the mode pair fits above the key)
// and go 64 at a time into an open-addressing table of mask + 1 slots (key + 1;
// 0 is free), at least twice the sample; a pair that finds no slot within
// kPairProbes counts as new.  Without the queue nearly every hash of a wave
// waited for some lane's trip to the table, past the L2: 20M nonzeros took
// 350 us, with it 160 us (three hashes per nonzero); a tree built to be compared
// and dropped takes 4.5 ms.
constexpr int kPairBits = 16, kPairProbes = 64;
constexpr int kPairQueue = 2 * 3 * 256;  // a wave's step adds 3 x 256 at most
__global__ __launch_bounds__(kBS) void k_pair_count(const uint32_t *__restrict__ i0, const uint32_t *__restrict__ i1,
                                                    const uint32_t *__restrict__ i2, uint64_t dim1, uint64_t dim2,
                                                    uint64_t n, int shift, unsigned long long *table, uint32_t mask,
                                                    uint32_t *found) {
    __shared__ uint64_t queues[kBS / 64][kPairQueue];
    const int lane = threadIdx.x & 63;
    volatile uint64_t *const queue = queues[threadIdx.x / 64];
    int held = 0;  // the same in every lane
    uint32_t fresh[3] = {0, 0, 0};
    auto drain = [&] {
        __builtin_amdgcn_wave_barrier();
        for (int e = lane; e < held; e += 64) {
            const uint64_t key = queue[e];
            uint64_t h = key * 0x9e3779b97f4a7c15ull;
            h ^= h >> 32;
            uint32_t at = (uint32_t)h & mask;
            bool isNew = true;
            for (int probe = 0; probe < kPairProbes; ++probe, at = (at + 1) & mask) {
                unsigned long long have = __hip_atomic_load(table + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (have == 0) {
                    have = atomicCAS(table + at, 0ull, (unsigned long long)key + 1);
                    if (have == 0) break;
                }
                if (have == key + 1) {
                    isNew = false;
                    break;
                }
            }
            const int pair = (int)(key >> 62);
            fresh[0] += isNew && pair == 0;
            fresh[1] += isNew && pair == 1;
            fresh[2] += isNew && pair == 2;
        }
        __builtin_amdgcn_wave_barrier();
        held = 0;
    };
    auto offer = [&](bool in, uint32_t a, uint32_t b, uint64_t width, uint64_t pair) {
        uint32_t h = a * 0x6a09e667u + b * 0xbb67ae85u;
        h ^= h >> 15;
        h *= 0x3c6ef373u;
        h ^= h >> 13;
        h *= 0xa54ff53bu;
        h ^= h >> 16;
        in = in && (shift == 0 || h >> (32 - shift) == 0);
        const uint64_t who = __ballot(in);
        if (in) queue[held + __popcll(who & ((1ull << lane) - 1))] = (a * width + b) | pair << 62;
        held += __popcll(who);
    };
    auto count = [&](bool in, uint32_t a, uint32_t b, uint32_t c) {
        offer(in, a, b, dim1, 0);
        offer(in, a, c, dim2, 1);
        offer(in, b, c, dim2, 2);
    };
    const uint64_t t = blockIdx.x * (uint64_t)kBS + threadIdx.x, threads = (uint64_t)gridDim.x * kBS;
    const uint64_t n4 = n / 4, steps = (n4 + threads - 1) / threads;
    for (uint64_t k = 0; k < steps; ++k) {
        const uint64_t i = k * threads + t;
        const bool in = i < n4;
        uint4 a = make_uint4(0, 0, 0, 0), b = a, c = a;
        if (in) {
            a = reinterpret_cast<const uint4 *>(i0)[i];
            b = reinterpret_cast<const uint4 *>(i1)[i];
            c = reinterpret_cast<const uint4 *>(i2)[i];
        }
        count(in, a.x, b.x, c.x);
        count(in, a.y, b.y, c.y);
        count(in, a.z, b.z, c.z);
        count(in, a.w, b.w, c.w);
        if (held > kPairQueue / 2) drain();
    }
    if (blockIdx.x == 0) {  // the last n % 4 nonzeros
        const uint64_t i = n4 * 4 + threadIdx.x;
        const bool in = i < n;
        count(in, in ? i0[i] : 0, in ? i1[i] : 0, in ? i2[i] : 0);
    }
    drain();
    for (int p = 0; p < 3; ++p) {
        for (int off = 32; off; off >>= 1) fresh[p] += __shfl_down(fresh[p], off, 64);
        if (lane == 0 && fresh[p]) atomicAdd(found + p, fresh[p]);
    }
}

}  // namespace

// Per mode m, the rows that hold `frac` of the nonzeros, most used rows first:
// the working set of gathers from that mode's factor table (small for skewed
// modes, most of the rows for uniform ones).  Counted, ordered and summed on
// the GPU; the host reads the results of all modes at once.
void hot_footprints(const Tensor &t, double frac, uint64_t *hot, hipStream_t s) {
    const uint64_t n = t.nnz;
    for (int m = 0; m < t.ndims; ++m) hot[m] = 0;
    if (n == 0) return;
    uint64_t most = 0;
    for (int m = 0; m < t.ndims; ++m) most = std::max(most, t.dims[m]);
    Temp tmp;
    TmpArray<uint32_t> cnt(most), sorted(most), found(kMaxDims);
    TmpArray<uint64_t> prefix(most);
    hipLaunchKernelGGL(k_zero_words, dim3(1), dim3(kBS), 0, s, found.p, (uint64_t)kMaxDims);
    const unsigned blocks = (unsigned)std::min<uint64_t>(2ull * device_cu_count(), (n + kHistThreads - 1) / kHistThreads);
    for (int m = 0; m < t.ndims; ++m) {
        const uint64_t rows = t.dims[m];
        if (rows == 0) continue;
        hipLaunchKernelGGL(k_zero_words, dim3(nblk(rows)), dim3(kBS), 0, s, cnt.p, rows);
        hipLaunchKernelGGL(k_hist_cached, dim3(blocks), dim3(kHistThreads), 0, s, t.inds[m].p, n, cnt.p);
        MMCSF_HIP(hipGetLastError());
        const unsigned bits = (unsigned)bitwidth(n);
        size_t bytes = 0;
        MMCSF_HIP(rocprim::radix_sort_keys_desc(nullptr, bytes, cnt.p, sorted.p, (size_t)rows, 0u, bits, s));
        MMCSF_HIP(rocprim::radix_sort_keys_desc(tmp.get(bytes), bytes, cnt.p, sorted.p, (size_t)rows, 0u, bits, s));
        MMCSF_HIP(rocprim::inclusive_scan(nullptr, bytes, sorted.p, prefix.p, (size_t)rows, rocprim::plus<uint64_t>(), s));
        MMCSF_HIP(rocprim::inclusive_scan(tmp.get(bytes), bytes, sorted.p, prefix.p, (size_t)rows,
                                          rocprim::plus<uint64_t>(), s));
        hipLaunchKernelGGL(k_reach, dim3(nblk(rows)), dim3(kBS), 0, s, prefix.p, rows, frac * (double)n, found.p + m);
        MMCSF_HIP(hipGetLastError());
    }
    uint32_t h[kMaxDims];
    MMCSF_HIP(hipMemcpyAsync(h, found.p, sizeof(h), hipMemcpyDeviceToHost, s));
    MMCSF_HIP(hipStreamSynchronize(s));
    for (int m = 0; m < t.ndims; ++m) hot[m] = h[m];
}

// pairs[m] = the distinct coordinate pairs of the two modes other than m of a
// 3-D tensor (an estimate past 2^kPairBits nonzeros): the level-1 entries of the
// trees that have the one at the root and the other below, before the -f split
// cuts long fibers
void pair_counts(const Tensor &t, double *pairs, hipStream_t s) {
    const uint64_t n = t.nnz;
    pairs[0] = pairs[1] = pairs[2] = 0.0;
    if (n == 0) return;
    int shift = 0;
    while ((n >> shift) > (1ull << kPairBits)) ++shift;
    uint32_t slots = 1024;
    while (slots < 6 * (n >> shift)) slots *= 2;
    TmpArray<unsigned long long> table(slots);
    TmpArray<uint32_t> found(3);
    hipLaunchKernelGGL(k_zero_words, dim3(nblk(2ull * slots)), dim3(kBS), 0, s, reinterpret_cast<uint32_t *>(table.p),
                       2ull * slots);
    hipLaunchKernelGGL(k_zero_words, dim3(1), dim3(kBS), 0, s, found.p, (uint64_t)3);
    const unsigned blocks = (unsigned)std::min<uint64_t>(3ull * device_cu_count(), (n + 4 * kBS - 1) / (4 * kBS));
    hipLaunchKernelGGL(k_pair_count, dim3(blocks), dim3(kBS), 0, s, t.inds[0].p, t.inds[1].p, t.inds[2].p, t.dims[1],
                       t.dims[2], n, shift, table.p, slots - 1, found.p);
    MMCSF_HIP(hipGetLastError());
    uint32_t h[3];
    MMCSF_HIP(hipMemcpyAsync(h, found.p, sizeof(h), hipMemcpyDeviceToHost, s));
    MMCSF_HIP(hipStreamSynchronize(s));
    for (int p = 0; p < 3; ++p) pairs[2 - p] = std::ldexp((double)h[p], shift);
}


// ---------------------------------------------------------------------------
// MM-CSF mixed-mode partition support (mm_partition_reuseBased,
// util.h:2167-2512): the level-1 entry of every nonzero in a mode's CSF and
// the nonzeros under each entry (nnzPerFiber)
// ---------------------------------------------------------------------------
// first nonzero of level-1 entry j (j = cnt1: nnz), and a mark at it
__global__ void k_l1_start(int N, const uint32_t *__restrict__ p1, const uint32_t *__restrict__ p2, uint64_t cnt1,
                           uint64_t nnz, uint32_t *start, uint32_t *mark) {
    uint64_t j = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (j > cnt1) return;
    if (j == cnt1) {
        start[j] = (uint32_t)nnz;
        return;
    }
    const uint32_t x = N == 3 ? p1[j] : p2[p1[j]];
    start[j] = x;
    mark[x] = 1u;
}

__global__ void k_l1_count(const uint32_t *__restrict__ start, uint64_t cnt1, uint32_t *cnt) {
    uint64_t j = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (j < cnt1) cnt[j] = start[j + 1] - start[j];
}

// entry of sorted nonzero k = (marks before k) + mark[k] - 1, written at its
// tensor position; nonzeros of the last slice (from lastStart on) outside
// its first entry e0 resolve to e0 - 1 (kNoEntry when e0 = 0)
__global__ void k_l1_ids(const uint32_t *__restrict__ excl, const uint32_t *__restrict__ mark,
                         const uint32_t *__restrict__ pos, uint64_t nnz, uint32_t lastStart, uint32_t e0,
                         uint32_t *idT) {
    uint64_t k = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (k >= nnz) return;
    uint32_t id = excl[k] + mark[k] - 1u;
    if (k >= lastStart && id != e0) id = e0 == 0 ? 0xFFFFFFFFu : e0 - 1u;
    idT[pos[k]] = id;
}

void level1_ids(const Csf &c, const uint32_t *pos, DevArray<uint32_t> &idT, DevArray<uint32_t> &cnt, hipStream_t s) {
    const int N = c.ndims;
    const uint64_t n = c.nnz, c1 = c.cnt[1];
    idT.alloc(n);
    cnt.alloc(c1 + 1);
    if (n == 0) return;
    Temp tmp;
    TmpArray<uint32_t> start(c1 + 1), mark(n), excl(n);
    hipLaunchKernelGGL(k_zero_words, dim3(nblk(n)), dim3(kBS), 0, s, mark.p, n);
    hipLaunchKernelGGL(k_l1_start, dim3(nblk(c1 + 1)), dim3(kBS), 0, s, N, c.ptr[1].p,
                       N == 4 ? c.ptr[2].p : (const uint32_t *)nullptr, c1, n, start.p, mark.p);
    hipLaunchKernelGGL(k_zero_words, dim3(1), dim3(kBS), 0, s, cnt.p + c1, (uint64_t)1);
    hipLaunchKernelGGL(k_l1_count, dim3(nblk(c1)), dim3(kBS), 0, s, start.p, c1, cnt.p);
    exclusive_sum(mark.p, excl.p, n, s, tmp);
    // the last slice's first level-1 entry and its first nonzero
    uint32_t e0 = 0, lastStart = 0;
    MMCSF_HIP(hipMemcpyAsync(&e0, c.ptr[0].p + (c.cnt[0] - 1), 4, hipMemcpyDeviceToHost, s));
    MMCSF_HIP(hipStreamSynchronize(s));
    MMCSF_HIP(hipMemcpyAsync(&lastStart, start.p + e0, 4, hipMemcpyDeviceToHost, s));
    MMCSF_HIP(hipStreamSynchronize(s));
    hipLaunchKernelGGL(k_l1_ids, dim3(nblk(n)), dim3(kBS), 0, s, excl.p, mark.p, pos, n, lastStart, e0, idT.p);
    MMCSF_HIP(hipGetLastError());
    MMCSF_HIP(hipStreamSynchronize(s));
}

__global__ void k_gather_sel_u32(const uint32_t *__restrict__ src, const uint32_t *__restrict__ sel, uint64_t n,
                                 uint32_t *dst) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[sel[i]];
}
__global__ void k_gather_sel_f32(const float *__restrict__ src, const uint32_t *__restrict__ sel, uint64_t n,
                                 float *dst) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[sel[i]];
}

// the nonzeros at tensor positions sel[0..n) as a tensor of their own
void gather_tensor(const Tensor &t, const uint32_t *sel, uint64_t n, Tensor &out, hipStream_t s) {
    out.ndims = t.ndims;
    out.nnz = n;
    for (int m = 0; m < t.ndims; ++m) {
        out.dims[m] = t.dims[m];
        out.inds[m].alloc(n);
        if (n) hipLaunchKernelGGL(k_gather_sel_u32, dim3(nblk(n)), dim3(kBS), 0, s, t.inds[m].p, sel, n, out.inds[m].p);
    }
    out.vals.alloc(n);
    if (n) hipLaunchKernelGGL(k_gather_sel_f32, dim3(nblk(n)), dim3(kBS), 0, s, t.vals.p, sel, n, out.vals.p);
    MMCSF_HIP(hipGetLastError());
}

}  // namespace mmcsf
