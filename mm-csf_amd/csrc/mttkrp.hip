// MTTKRP kernels and launchers (gfx950).
//
// Reference kernels these replace (mttkrp_gpu.cu):
//   MM-CSF root / fbrS / fiber / leaf output: mttkrp_MIHCSR_kernel_slc_atomic_fbrLvlPar[_4D]
//     (716, 774), ..._fbrS_atomic_fbrLvlPar_4D (1134), ..._fbr_atomic_fbrLvlPar[_4D]
//     (1060, 1095), ..._all_atomic_fbrLvlPar[_4D] (1438, 1475); chosen by the output
//     mode's level in modeOrder as in MTTKRP_MIHCSR_GPU (3610-3719).
//   B-CSF: mttkrp_HCSR_kernel_smllBin / _hvyBin [_4D] (539-713): root output.
//   HB-CSF: mttkrp_HYB_COO_kernel[_4D] (196, 255), mttkrp_CSL_kernel_bin / _hvyBin
//     (346, 427) and the B-CSF kernels on the CSF part.
//   COO: mttkrp_COO_kernel_loop[_4D] (102, 161).
// The reference kernels accumulate every r of a lane into one scalar and are
// only correct for R <= 32 (e.g. mttkrp_gpu.cu:487-494); these keep one
// accumulator per column and are correct for any R up to 256.
#include <algorithm>

#include "mmcsf_internal.hpp"
#include "mttkrp_kernels.hpp"

namespace mmcsf {

namespace {

using dev::Row;
using dev::upper_index;

constexpr int kBlock = 256;

// --------------------------------------------------------------------------
// Root-mode CSF walker for what the chunked walk does not serve (R < 4, tables
// of 4 GiB and more).  Persistent: every group of G lanes owns one contiguous,
// equal share of the nonzeros.
// --------------------------------------------------------------------------
template <int N, int G, int NV, int VEC, int B, typename T>
__global__ __launch_bounds__(kBlock) void k_csf(CsfArgs a) {
    using RowT = Row<G, NV, VEC>;
    constexpr int LF = N - 2;  // leaf-fiber level
    const int R = a.R;
    const int lane = threadIdx.x % G;
    const uint64_t ngroups = (uint64_t)gridDim.x * blockDim.x / G;
    const uint64_t grp = (blockIdx.x * (uint64_t)blockDim.x + threadIdx.x) / G;
    const uint32_t x0 = (uint32_t)(grp * a.nnz / ngroups);
    const uint32_t x1 = (uint32_t)((grp + 1) * a.nnz / ngroups);
    if (x0 >= x1) return;
    const T *U1 = static_cast<const T *>(a.U[1]);
    const T *U2 = static_cast<const T *>(a.U[2]);
    const T *UL = static_cast<const T *>(a.U[N - 1]);
    const uint32_t *__restrict__ ptrL = a.ptr[LF];

    uint32_t f = upper_index(ptrL, a.cnt[LF], x0);
    uint32_t fend = ptrL[f + 1];
    uint32_t j = f, jend = 0;
    if constexpr (N == 4) {
        j = upper_index(a.ptr[1], a.cnt[1], f);
        jend = a.ptr[1][j + 1];
    }
    uint32_t slc = a.slc[j];

    RowT aF, aJ, aS, t;
    aF.zero();
    aJ.zero();
    aS.zero();
    auto end_fiber = [&]() {
        if constexpr (N == 3) {
            t.load(U1, a.idx[1][f], R, lane);
            aS.fma_had(aF, t);
        } else {
            t.load(U2, a.idx[2][f], R, lane);
            aJ.fma_had(aF, t);
        }
        aF.zero();
    };
    auto end_j = [&]() {
        if constexpr (N == 4) {
            t.load(U1, a.idx[1][j], R, lane);
            aS.fma_had(aJ, t);
            aJ.zero();
        }
    };
    auto next_slice = [&](uint32_t ns) {
        if (ns == slc) return;
        aS.atomic_add(a.out, slc, R, lane);
        aS.zero();
        slc = ns;
    };
    for (uint32_t xb = x0; xb < x1; xb += B) {
        // every index of the batch before the first row: a row's load waits for its
        // index, and one wait then serves the batch
        uint32_t li[B];
        float vv[B];
        RowT rows[B];
#pragma unroll
        for (int k = 0; k < B; ++k) {
            const uint32_t x = xb + k;
            li[k] = 0;
            vv[k] = 0.f;
            if (x < x1) {
                li[k] = a.leaf[x];
                vv[k] = a.val[x];
            }
        }
#pragma unroll
        for (int k = 0; k < B; ++k)
            if (xb + k < x1) rows[k].load(UL, li[k], R, lane);
#pragma unroll
        for (int k = 0; k < B; ++k) {
            const uint32_t x = xb + k;
            if (x >= x1) break;
            if (x == fend) {
                end_fiber();
                ++f;
                fend = ptrL[f + 1];
                if constexpr (N == 4) {
                    if (f == jend) {
                        end_j();
                        ++j;
                        jend = a.ptr[1][j + 1];
                        next_slice(a.slc[j]);
                    }
                } else {
                    next_slice(a.slc[f]);
                }
            }
            aF.fma(vv[k], rows[k]);
        }
    }
    end_fiber();
    end_j();
    aS.atomic_add(a.out, slc, R, lane);
}

// --------------------------------------------------------------------------
// Level-map MTTKRP for what the mapped walk does not serve (R > 3: tables of 4 GiB
// and more, bfloat16 rows at 8-byte boundaries): every group sums a
// contiguous run of the nonzeros in the order of the output level.
// --------------------------------------------------------------------------
struct MapArgs {
    const uint32_t *ord, *fbit, *frank, *sbit, *jrank;
    const uint32_t *slc, *idx1, *idx2, *leaf;
    const float *val;
    const void *U[4];  // per level; U[outLevel] is not read
    float *out;
    uint32_t nnz, perGroup;
    int R, outLevel;
};

template <int N, int G, int NV, int VEC, int B, typename T>
__global__ __launch_bounds__(kBlock) void k_map(MapArgs a) {
    using RowT = Row<G, NV, VEC>;
    const int lane = threadIdx.x % G;
    const uint64_t grp = (blockIdx.x * (uint64_t)blockDim.x + threadIdx.x) / G;
    const uint64_t x0 = grp * (uint64_t)a.perGroup;
    if (x0 >= a.nnz) return;
    const uint32_t x1 = (uint32_t)min((uint64_t)a.nnz, x0 + a.perGroup);
    uint32_t cur = 0xffffffffu;
    RowT acc;
    acc.zero();
    for (uint32_t q = (uint32_t)x0; q < x1; ++q) {
        const uint32_t x = a.ord[q];
        const uint32_t f = dev::rank_of(a.fbit, a.frank, x);
        const uint32_t j = N == 4 ? dev::rank_of(a.sbit, a.jrank, f) : f;
        const uint32_t c[4] = {a.slc[j], a.idx1[j], N == 4 ? a.idx2[f] : a.leaf[x], N == 4 ? a.leaf[x] : 0u};
        uint32_t row = 0;
        RowT p, t;
        bool first = true;
#pragma unroll
        for (int l = 0; l < N; ++l) {
            if (l == a.outLevel) {
                row = c[l];
                continue;
            }
            t.load(static_cast<const T *>(a.U[l]), c[l], a.R, lane);
            if (first) p = t;
            else p.mul(t);
            first = false;
        }
        if (row != cur) {
            if (cur != 0xffffffffu) acc.atomic_add(a.out, cur, a.R, lane);
            acc.zero();
            cur = row;
        }
        acc.fma(a.val[x], p);
    }
    acc.atomic_add(a.out, cur, a.R, lane);
}

// --------------------------------------------------------------------------
// Modes below the root at R <= 3, which no walk serves, in stored order: every
// nonzero's row is added to its output row, a lane per nonzero.  Neighbours with
// one output row (the nonzeros of a fiber) are summed by shuffles first; rows that
// come early in a block (the hot ones do) are held in LDS, in float64, in sets of
// four by their low bits, and added to memory once; the others pass through a
// stage of the wave, from which consecutive lanes add to consecutive columns of a
// row.  (With one place by the low bits, a hot row that finds it taken collects
// every nonzero of the block as a float32 addition: relative error 8e-6 instead
// of 1.6e-7.)  Bound by the structure's reads and the latency of the rows.  R = 1,
// group kernel over level maps / here: the two modes below the root of
// 300 x 200 x 1000, 4M nonzeros, 772 and 624 / 28 and 31 us; every mode of
// 20000 x 5000 x 800 x 300, 4M, 3.52 / 0.58 ms.
// (At R = 4 to 16 it would take 0.25 to 0.9 of the mapped walk's time where modes
// are skewed, but a hot row's total then collects a float32 addition from every
// block: relative error 3.4e-7 where the walk's is 1.2e-7.)
// --------------------------------------------------------------------------
struct ScatterArgs {
    const uint32_t *fbit, *frank, *sbit, *jrank;
    const uint32_t *slc, *idx1, *idx2, *leaf;
    const float *val;
    const float *U[4];  // per level; U[outLevel] is not read
    float *out;
    uint32_t nnz;
    int outLevel;
};

constexpr int kScatterBlock = 1024;

template <int N, int R>
__global__ __launch_bounds__(kScatterBlock) void k_scatter(ScatterArgs a) {
    constexpr int kStage = 16, kStride = R | 1;
    constexpr uint32_t kSlots = R == 1 ? 4096 : 2048, kNone = 0xffffffffu;  // coordinates are below 2^31
    __shared__ __align__(16) uint32_t held[kSlots];
    __shared__ double acc[R][kSlots];
    __shared__ volatile float stage[kScatterBlock / 64][kStage * kStride];
    __shared__ volatile uint32_t stageRow[kScatterBlock / 64][kStage];
    for (uint32_t i = threadIdx.x; i < kSlots; i += blockDim.x) {
        held[i] = kNone;
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r][i] = 0.0;
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint64_t chunks = ((uint64_t)a.nnz + 63) / 64, waves = (uint64_t)gridDim.x * (blockDim.x >> 6);
    const uint64_t wv = blockIdx.x * (uint64_t)(blockDim.x >> 6) + w;
    const uint32_t cb = (uint32_t)(wv * chunks / waves), ce = (uint32_t)((wv + 1) * chunks / waves);
    for (uint32_t c = cb; c < ce; ++c) {
        const bool in = (uint64_t)c * 64 + lane < a.nnz;
        const uint32_t x = in ? c * 64u + (uint32_t)lane : a.nnz - 1u;
        const uint32_t f = dev::rank_of(a.fbit, a.frank, x);
        const uint32_t j = N == 4 ? dev::rank_of(a.sbit, a.jrank, f) : f;
        const uint32_t at[4] = {a.slc[j], a.idx1[j], N == 4 ? a.idx2[f] : a.leaf[x], N == 4 ? a.leaf[x] : 0u};
        uint32_t row = 0;
#pragma unroll
        for (int l = 0; l < N; ++l)
            if (l == a.outLevel) row = at[l];
        float p[R];
        const float v = a.val[x];
#pragma unroll
        for (int r = 0; r < R; ++r) p[r] = v;
#pragma unroll
        for (int l = 0; l < N; ++l)
            if (l != a.outLevel) {
                const float *u = a.U[l] + (size_t)at[l] * R;
#pragma unroll
                for (int r = 0; r < R; ++r) p[r] *= u[r];
            }
        // (lanes past the tensor hold its last row: nothing, also where a factor
        // is not finite)
#pragma unroll
        for (int r = 0; r < R; ++r) p[r] = in ? p[r] : 0.f;
        // neighbours with one output row: their sum to the first of them
        const uint32_t before = __shfl_up(row, 1, 64);
        const bool first = lane == 0 || row != before;
        const uint64_t heads = __ballot(first);
        if (heads != ~0ull) {
            const int run = __popcll(heads & (~0ull >> (63 - lane)));
            for (int off = 1; off < 64; off <<= 1) {
                const bool same = __shfl_down(run, off, 64) == run && lane + off < 64;
                if (__ballot(same) == 0) break;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const float o = __shfl_down(p[r], off, 64);
                    if (same) p[r] += o;
                }
            }
        }
        // the row's place among the four of its set, or a free one
        uint32_t slot = row % (kSlots / 4) * 4;
        bool mineHeld = false;
        if (first && in) {
            const uint4 q = *reinterpret_cast<const uint4 *>(held + slot);
            const uint32_t owner[4] = {q.x, q.y, q.z, q.w};
            int way = owner[0] == row ? 0 : owner[1] == row ? 1 : owner[2] == row ? 2 : owner[3] == row ? 3 : 4;
            for (int t = 0; way == 4 && t < 4; ++t) {
                if (owner[t] != kNone) continue;
                const uint32_t was = atomicCAS(&held[slot + t], kNone, row);
                if (was == kNone || was == row) way = t;
            }
            mineHeld = way < 4;
            slot += (uint32_t)way & 3u;
        }
        if (mineHeld) {
#pragma unroll
            for (int r = 0; r < R; ++r) unsafeAtomicAdd(&acc[r][slot], (double)p[r]);
        }
        // the other rows through the wave's stage, so that one request adds to all
        // columns of a row
        uint64_t cold = __ballot(first && in && !mineHeld);
        while (cold) {
            const int mine = __popcll(cold & ((1ull << lane) - 1)), n = min(__popcll(cold), kStage);
            const bool put = ((cold >> lane) & 1) && mine < kStage;
            __builtin_amdgcn_wave_barrier();
            if (put) {
                stageRow[w][mine] = row;
#pragma unroll
                for (int r = 0; r < R; ++r) stage[w][mine * kStride + r] = p[r];
            }
            __builtin_amdgcn_wave_barrier();
            for (int i = lane; i < n * R; i += 64)
                unsafeAtomicAdd(a.out + (size_t)stageRow[w][i / R] * R + i % R, (float)stage[w][i / R * kStride + i % R]);
            __builtin_amdgcn_wave_barrier();
            cold &= ~__ballot(put);
        }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < kSlots; i += blockDim.x) {
        const uint32_t row = held[i];
        if (row == kNone) continue;
#pragma unroll
        for (int r = 0; r < R; ++r) unsafeAtomicAdd(a.out + (size_t)row * R + r, (float)acc[r][i]);
    }
}

// --------------------------------------------------------------------------
// COO (sorted by modeOrder): keys[0] is the output coordinate
// --------------------------------------------------------------------------
struct CooArgs {
    const uint32_t *key[4];
    const float *val;
    const void *U[4];  // per level
    float *out;
    uint32_t nnz;
    uint32_t perGroup;
    int R;
    int store;         // 1: every output row occurs once (HB-CSF COO part): plain stores
};

template <int N, int G, int NV, int VEC, int B, typename T>
__global__ __launch_bounds__(kBlock) void k_coo(CooArgs a) {
    using RowT = Row<G, NV, VEC>;
    const int lane = threadIdx.x % G;
    const uint64_t grp = (blockIdx.x * (uint64_t)blockDim.x + threadIdx.x) / G;
    const uint64_t x0l = grp * (uint64_t)a.perGroup;
    if (x0l >= a.nnz) return;
    const uint32_t x0 = (uint32_t)x0l;
    const uint32_t x1 = (uint32_t)min((uint64_t)a.nnz, x0l + a.perGroup);
    const int R = a.R;
    uint32_t cur = a.key[0][x0];
    RowT acc;
    acc.zero();
    for (uint32_t xb = x0; xb < x1; xb += B) {
        uint32_t k0[B];
        float vv[B];
        RowT r1[B], r2[B], r3[B];
#pragma unroll
        for (int k = 0; k < B; ++k) {
            uint32_t x = xb + k;
            if (x < x1) {
                k0[k] = a.key[0][x];
                vv[k] = a.val[x];
                r1[k].load(static_cast<const T *>(a.U[1]), a.key[1][x], R, lane);
                r2[k].load(static_cast<const T *>(a.U[2]), a.key[2][x], R, lane);
                if constexpr (N == 4) r3[k].load(static_cast<const T *>(a.U[3]), a.key[3][x], R, lane);
            }
        }
#pragma unroll
        for (int k = 0; k < B; ++k) {
            if (xb + k >= x1) break;
            if (k0[k] != cur) {
                if (a.store) acc.store(a.out, cur, R, lane);
                else acc.atomic_add(a.out, cur, R, lane);
                acc.zero();
                cur = k0[k];
            }
            RowT p;
            p.had(r1[k], r2[k]);
            if constexpr (N == 4) p.mul(r3[k]);
            acc.fma(vv[k], p);
        }
    }
    if (a.store) acc.store(a.out, cur, R, lane);
    else acc.atomic_add(a.out, cur, R, lane);
}

// --------------------------------------------------------------------------
// HB-CSF CSL part: slices whose fibers all hold one nonzero
// --------------------------------------------------------------------------
struct CslArgs {
    const uint32_t *ptr, *idx, *ind1, *ind2;
    const float *val;
    const void *U1, *U2;
    float *out;
    uint32_t nnz, nslc, perGroup;
    int R;
};

template <int G, int NV, int VEC, int B, typename T>
__global__ __launch_bounds__(kBlock) void k_csl(CslArgs a) {
    using RowT = Row<G, NV, VEC>;
    const int lane = threadIdx.x % G;
    const uint64_t grp = (blockIdx.x * (uint64_t)blockDim.x + threadIdx.x) / G;
    const uint64_t x0l = grp * (uint64_t)a.perGroup;
    if (x0l >= a.nnz) return;
    const uint32_t x0 = (uint32_t)x0l;
    const uint32_t x1 = (uint32_t)min((uint64_t)a.nnz, x0l + a.perGroup);
    const int R = a.R;
    uint32_t s = upper_index(a.ptr, a.nslc, x0);
    uint32_t send = a.ptr[s + 1];
    RowT acc;
    acc.zero();
    for (uint32_t xb = x0; xb < x1; xb += B) {
        float vv[B];
        RowT r1[B], r2[B];
#pragma unroll
        for (int k = 0; k < B; ++k) {
            uint32_t x = xb + k;
            if (x < x1) {
                vv[k] = a.val[x];
                r1[k].load(static_cast<const T *>(a.U1), a.ind1[x], R, lane);
                r2[k].load(static_cast<const T *>(a.U2), a.ind2[x], R, lane);
            }
        }
#pragma unroll
        for (int k = 0; k < B; ++k) {
            uint32_t x = xb + k;
            if (x >= x1) break;
            if (x == send) {
                acc.atomic_add(a.out, a.idx[s], R, lane);
                acc.zero();
                ++s;
                send = a.ptr[s + 1];
            }
            RowT p;
            p.had(r1[k], r2[k]);
            acc.fma(vv[k], p);
        }
    }
    acc.atomic_add(a.out, a.idx[s], R, lane);
}

__global__ void k_zero(float *p, uint64_t n) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = 0.f;
}

struct ZeroArgs {
    float *p[kMaxDims + 1];
    uint64_t n[kMaxDims + 1];
};

// array blockIdx.y, 16 bytes a lane between its unaligned ends
__global__ void k_zero_all(ZeroArgs z) {
    float *p = z.p[blockIdx.y];
    const uint64_t n = z.n[blockIdx.y];
    const uint64_t head = min(n, (uint64_t)((16 - (reinterpret_cast<uintptr_t>(p) & 15)) & 15) / 4);
    const uint64_t quads = (n - head) / 4;
    const uint64_t t = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x, stride = (uint64_t)gridDim.x * blockDim.x;
    float4 *q = reinterpret_cast<float4 *>(p + head);
    for (uint64_t i = t; i < quads; i += stride) q[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (t < head) p[t] = 0.f;
    if (t < n - head - 4 * quads) p[head + 4 * quads + t] = 0.f;
}

// --------------------------------------------------------------------------
// dispatch over the row geometry
// --------------------------------------------------------------------------
struct Geo {
    int G, NV, VEC;
};

Geo pick_geometry(int R, int dtype) {
    if (R < 1 || R > 256) fail(MMCSF_ERR_UNSUPPORTED, "R must be in 1..256");
    if (R % 4 == 0) {
        int r4 = R / 4, g = 1;
        while (g < r4 && g < 16) g *= 2;
        return Geo{g, (r4 + g - 1) / g, 4};
    }
    if (dtype == MMCSF_BF16) fail(MMCSF_ERR_UNSUPPORTED, "bfloat16 factors need R % 4 == 0");
    return Geo{64, (R + 63) / 64, 1};
}

uint32_t per_group_for(uint64_t nnz, int G) {
    uint64_t target = (uint64_t)device_cu_count() * (2048 / G) * 2;
    uint64_t pg = (nnz + target - 1) / std::max<uint64_t>(target, 1);
    return (uint32_t)std::max<uint64_t>(pg, 16);
}

template <template <int, int, int, int, typename> class K, typename Args, typename T>
void run_geo(const Geo &g, Args &a, uint64_t groups, hipStream_t s) {
    uint64_t threads = groups * (uint64_t)g.G;
    dim3 grid((unsigned)std::max<uint64_t>(1, (threads + kBlock - 1) / kBlock)), block(kBlock);
#define MMCSF_GEO(GG, NN, VV)                                                                  \
    if (g.G == GG && g.NV == NN && g.VEC == VV) {                                              \
        constexpr int Bk = (NN >= 3) ? 2 : (NN == 2 ? 4 : 8);                                  \
        K<GG, NN, VV, Bk, T>::launch(grid, block, s, a);                                       \
        MMCSF_HIP(hipGetLastError());                                                          \
        return;                                                                                \
    }
    MMCSF_GEO(1, 1, 4)
    MMCSF_GEO(2, 1, 4)
    MMCSF_GEO(4, 1, 4)
    MMCSF_GEO(8, 1, 4)
    MMCSF_GEO(16, 1, 4)
    MMCSF_GEO(16, 2, 4)
    MMCSF_GEO(16, 3, 4)
    MMCSF_GEO(16, 4, 4)
    if constexpr (std::is_same<T, float>::value) {
        MMCSF_GEO(64, 1, 1)
        MMCSF_GEO(64, 2, 1)
        MMCSF_GEO(64, 3, 1)
        MMCSF_GEO(64, 4, 1)
    }
#undef MMCSF_GEO
    fail(MMCSF_ERR_UNSUPPORTED, "no kernel for this rank");
}

// kernel selectors with a uniform template signature
template <int N>
struct CooSel {
    template <int G, int NV, int VEC, int B, typename T>
    struct K {
        static void launch(dim3 g, dim3 b, hipStream_t s, const CooArgs &a) {
            k_coo<N, G, NV, VEC, B, T><<<g, b, 0, s>>>(a);
        }
    };
};
template <int G, int NV, int VEC, int B, typename T>
struct CslK {
    static void launch(dim3 g, dim3 b, hipStream_t s, const CslArgs &a) {
        k_csl<G, NV, VEC, B, T><<<g, b, 0, s>>>(a);
    }
};

template <int N>
struct CsfLaunch {
    template <int G, int NV, int VEC, int B, typename T>
    struct K {
        static void launch(dim3, dim3, hipStream_t s, const CsfArgs &a) {
            auto fn = k_csf<N, G, NV, VEC, B, T>;
            int perCU = 0;
            MMCSF_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU, fn, kBlock, 0));
            fn<<<dim3((unsigned)(device_cu_count() * std::max(perCU, 1))), dim3(kBlock), 0, s>>>(a);
        }
    };
};

template <int N>
struct MapLaunch {
    template <int G, int NV, int VEC, int B, typename T>
    struct K {
        static void launch(dim3 g, dim3 b, hipStream_t s, const MapArgs &a) {
            k_map<N, G, NV, VEC, B, T><<<g, b, 0, s>>>(a);
        }
    };
};

template <int N>
void launch_csf_t(const Geo &g, CsfArgs &a, int dtype, hipStream_t s) {
    if (dtype == MMCSF_F32)
        run_geo<CsfLaunch<N>::template K, CsfArgs, float>(g, a, 1, s);
    else
        run_geo<CsfLaunch<N>::template K, CsfArgs, uint16_t>(g, a, 1, s);
}

template <int N>
void launch_map_t(const Geo &g, MapArgs &a, int dtype, hipStream_t s) {
    const uint64_t groups = (a.nnz + a.perGroup - 1) / a.perGroup;
    if (dtype == MMCSF_F32)
        run_geo<MapLaunch<N>::template K, MapArgs, float>(g, a, groups, s);
    else
        run_geo<MapLaunch<N>::template K, MapArgs, uint16_t>(g, a, groups, s);
}

template <int N, int R>
void launch_scatter(const ScatterArgs &a, hipStream_t s) {
    auto fn = k_scatter<N, R>;
    int perCU = 0;
    MMCSF_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU, fn, kScatterBlock, 0));
    // every wave a chunk at least
    const uint64_t chunks = ((uint64_t)a.nnz + 63) / 64;
    const uint64_t blocks = std::min<uint64_t>((uint64_t)device_cu_count() * std::max(perCU, 1),
                                               (chunks + kScatterBlock / 64 - 1) / (kScatterBlock / 64));
    fn<<<dim3((unsigned)blocks), dim3(kScatterBlock), 0, s>>>(a);
    MMCSF_HIP(hipGetLastError());
}

template <int N>
void run_scatter(const ScatterArgs &a, int R, hipStream_t s) {
    if (R == 1) launch_scatter<N, 1>(a, s);
    else if (R == 2) launch_scatter<N, 2>(a, s);
    else launch_scatter<N, 3>(a, s);
}

void check_align(const void *p, int dtype, const Geo &g) {
    size_t need = g.VEC == 4 ? (dtype == MMCSF_F32 ? 16 : 8) : (dtype == MMCSF_F32 ? 4 : 2);
    if (reinterpret_cast<uintptr_t>(p) % need)
        fail(MMCSF_ERR_ARG, "factor / output pointer is not aligned to " + std::to_string(need) + " bytes");
}

}  // namespace

void preload_group_kernels() {
    // one kernel of this translation unit: its code object loads with it
    hipFuncAttributes attr;
    MMCSF_HIP(hipFuncGetAttributes(&attr, reinterpret_cast<const void *>(k_zero)));
}

int device_cu_count() {
    static int cus = 0;
    if (!cus) {
        int dev = 0;
        MMCSF_HIP(hipGetDevice(&dev));
        MMCSF_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        if (cus <= 0) cus = 256;
    }
    return cus;
}

void fill_zero(float *p, uint64_t n, hipStream_t s) {
    if (!n) return;
    uint64_t blocks = std::min<uint64_t>((n + 255) / 256, 65536);
    hipLaunchKernelGGL(k_zero, dim3((unsigned)blocks), dim3(256), 0, s, p, n);
    MMCSF_HIP(hipGetLastError());
}

static void launch_csf(const Csf &c, const Geo &g, const Factors &F, float *out, hipStream_t s) {
    CsfArgs a{};
    for (int l = 0; l < c.ndims - 1; ++l) {
        a.ptr[l] = c.ptr[l].p;
        a.idx[l] = c.idx[l].p;
        a.cnt[l] = (uint32_t)c.cnt[l];
    }
    a.cnt[c.ndims - 1] = (uint32_t)c.nnz;
    a.slc = c.fbrSlc.p;
    a.leaf = c.leaf.p;
    a.val = c.vals.p;
    for (int l = 0; l < c.ndims; ++l) a.U[l] = F.U[c.order[l]];
    a.out = out;
    a.nnz = (uint32_t)c.nnz;
    a.R = F.R;
    if (c.ndims == 3) launch_csf_t<3>(g, a, F.dtype, s);
    else launch_csf_t<4>(g, a, F.dtype, s);
}

void fill_zero_all(float *const *p, const uint64_t *n, int arrays, hipStream_t s) {
    ZeroArgs z{};
    uint64_t most = 0;
    for (int i = 0; i < arrays; ++i) {
        z.p[i] = p[i];
        z.n[i] = n[i];
        most = std::max(most, n[i]);
    }
    if (!most) return;
    const uint64_t blocks = std::min<uint64_t>((most / 4 + 255) / 256 + 1, 8192);
    hipLaunchKernelGGL(k_zero_all, dim3((unsigned)blocks, (unsigned)arrays), dim3(256), 0, s, z);
    MMCSF_HIP(hipGetLastError());
}

void mttkrp_csf(const Csf &c, const uint64_t *dims, int outLevel, const Factors &F, float *out,
                hipStream_t s, hipEvent_t evStart, hipEvent_t evEnd, bool accumulate, bool zeroed, bool anyAlign) {
    const int N = c.ndims;
    if (!accumulate && !zeroed) fill_zero(out, dims[c.order[outLevel]] * (uint64_t)F.R, s);
    if (evStart) MMCSF_HIP(hipEventRecord(evStart, s));
    struct EndMark {
        hipEvent_t e;
        hipStream_t s;
        ~EndMark() {
            if (e) (void)hipEventRecord(e, s);
        }
    } endMark{evEnd, s};
    if (c.nnz == 0) return;
    Geo g = pick_geometry(F.R, F.dtype);
    check_align(out, MMCSF_F32, g);
    for (int l = 0; l < N; ++l)
        if (l != outLevel) {
            MMCSF_REQUIRE(F.U[c.order[l]] != nullptr, MMCSF_ERR_ARG, "missing factor matrix");
            check_align(F.U[c.order[l]], F.dtype, g);
        }
    if (outLevel > 0) {
        const LevelMap &map = c.map[outLevel];
        MMCSF_REQUIRE(map.ord.p != nullptr, MMCSF_ERR_ARG, "this format serves its root mode only");
        // (every size measured, 150000 to 20M nonzeros, 1.4 to 20 times the group kernel)
        if (F.R <= 3) {
            ScatterArgs a{};
            a.fbit = c.fbit.p;
            a.frank = c.frank.p;
            a.sbit = c.sbit.p;
            a.jrank = c.jrank.p;
            a.slc = c.fbrSlc.p;
            a.idx1 = c.idx[1].p;
            a.idx2 = c.idx[2].p;
            a.leaf = c.leaf.p;
            a.val = c.vals.p;
            for (int l = 0; l < N; ++l) a.U[l] = static_cast<const float *>(F.U[c.order[l]]);
            a.out = out;
            a.nnz = (uint32_t)c.nnz;
            a.outLevel = outLevel;
            if (N == 3) run_scatter<3>(a, F.R, s);
            else run_scatter<4>(a, F.R, s);
            return;
        }
        if (map_walk_supports(c, F, outLevel, out)) {
            mttkrp_map_walk(c, outLevel, F, out, s, accumulate);
            return;
        }
        MapArgs a{};
        a.ord = map.ord.p;
        a.fbit = c.fbit.p;
        a.frank = c.frank.p;
        a.sbit = c.sbit.p;
        a.jrank = c.jrank.p;
        a.slc = c.fbrSlc.p;
        a.idx1 = c.idx[1].p;
        a.idx2 = c.idx[2].p;
        a.leaf = c.leaf.p;
        a.val = c.vals.p;
        for (int l = 0; l < N; ++l) a.U[l] = F.U[c.order[l]];
        a.out = out;
        a.nnz = (uint32_t)c.nnz;
        a.perGroup = per_group_for(c.nnz, g.G);
        a.R = F.R;
        a.outLevel = outLevel;
        if (N == 3) launch_map_t<3>(g, a, F.dtype, s);
        else launch_map_t<4>(g, a, F.dtype, s);
        return;
    }
    if (walk_supports(c, F.R, F.dtype) && (!anyAlign || walk_aligned(c, F, 0, out))) {
        mttkrp_root(c, F, out, s, accumulate);  // checks the alignment its row loads need
        return;
    }
    launch_csf(c, g, F, out, s);
}

void mttkrp_mode(const Format &f, int mode, const Factors &F, float *out, hipStream_t s, hipEvent_t evStart,
                 hipEvent_t evEnd, bool zeroed) {
    if (f.mixed) {
        // every partition adds its nonzeros' contributions, with the kernel of
        // the level the mode takes in its tree (mttkrp_gpu.cu:3610-3719)
        if (!zeroed) fill_zero(out, f.dims[mode] * (uint64_t)F.R, s);
        if (evStart) MMCSF_HIP(hipEventRecord(evStart, s));
        for (int p = 0; p < f.ndims; ++p) {
            if (!f.partNnz[p]) continue;
            int lvl = 0;
            for (int l = 0; l < f.ndims; ++l)
                if (f.part[p].order[l] == mode) lvl = l;
            mttkrp_csf(f.part[p], f.dims, lvl, F, out, s, nullptr, nullptr, true);
        }
        if (evEnd) MMCSF_HIP(hipEventRecord(evEnd, s));
        return;
    }
    if (f.hasTree[mode]) {
        // MM-CSF refuses bfloat16 rows at 8-byte boundaries where 16 are needed;
        // the one-tree types (whose caches may hold root trees, though none is
        // built) take them in every mode but their root
        mttkrp_csf(f.tree[mode], f.dims, 0, F, out, s, evStart, evEnd, false, zeroed, f.type != MMCSF_TYPE_MMCSF);
        return;
    }
    int lvl = 0;
    for (int l = 0; l < f.ndims; ++l)
        if (f.csf.order[l] == mode) lvl = l;
    mttkrp_csf(f.csf, f.dims, lvl, F, out, s, evStart, evEnd, false, zeroed);
}

void mttkrp_coo(const Format &f, const Factors &F, float *out, hipStream_t s) {
    const int N = f.ndims;
    fill_zero(out, f.dims[f.cooOrder[0]] * (uint64_t)F.R, s);
    if (f.nnz == 0) return;
    Geo g = pick_geometry(F.R, F.dtype);
    check_align(out, MMCSF_F32, g);
    CooArgs a{};
    for (int l = 0; l < N; ++l) {
        a.key[l] = f.cooKeys[l].p;
        a.U[l] = F.U[f.cooOrder[l]];
        if (l) {
            MMCSF_REQUIRE(a.U[l] != nullptr, MMCSF_ERR_ARG, "missing factor matrix");
            check_align(a.U[l], F.dtype, g);
        }
    }
    if (coo_walk_supports(f, F)) {
        mttkrp_coo_walk(f, F, out, s);
        return;
    }
    a.val = f.cooVals.p;
    a.out = out;
    a.nnz = (uint32_t)f.nnz;
    a.R = F.R;
    a.store = 0;
    a.perGroup = per_group_for(f.nnz, g.G);
    uint64_t groups = (a.nnz + a.perGroup - 1) / a.perGroup;
    if (N == 3) {
        if (F.dtype == MMCSF_F32) run_geo<CooSel<3>::template K, CooArgs, float>(g, a, groups, s);
        else run_geo<CooSel<3>::template K, CooArgs, uint16_t>(g, a, groups, s);
    } else {
        if (F.dtype == MMCSF_F32) run_geo<CooSel<4>::template K, CooArgs, float>(g, a, groups, s);
        else run_geo<CooSel<4>::template K, CooArgs, uint16_t>(g, a, groups, s);
    }
}

void mttkrp_hyb(const Hyb &h, const uint64_t *dims, const Factors &F, float *out, hipStream_t s) {
    const int N = h.ndims;
    Geo g = pick_geometry(F.R, F.dtype);
    check_align(out, MMCSF_F32, g);
    for (int l = 1; l < N; ++l) {
        MMCSF_REQUIRE(F.U[h.order[l]] != nullptr, MMCSF_ERR_ARG, "missing factor matrix");
        check_align(F.U[h.order[l]], F.dtype, g);
    }
    // the CSF part's walk loads wider rows than the COO / CSL kernels: refuse
    // its misaligned factors before any part is launched
    if (h.csf.nnz && walk_supports(h.csf, F.R, F.dtype)) check_walk_align(h.csf, F, 0, out);
    if (h.cslWalk.nnz && walk_supports(h.cslWalk, F.R, F.dtype)) check_walk_align(h.cslWalk, F, 0, out);
    fill_zero(out, dims[h.order[0]] * (uint64_t)F.R, s);
    // COO part: slices with one nonzero; each output row is written once
    if (h.cooNnz) {
        CooArgs a{};
        for (int l = 0; l < N; ++l) {
            a.key[l] = h.cooInd[l].p;
            a.U[l] = F.U[h.order[l]];
        }
        a.val = h.cooVal.p;
        a.out = out;
        a.nnz = (uint32_t)h.cooNnz;
        a.R = F.R;
        a.store = 1;
        a.perGroup = per_group_for(h.cooNnz, g.G);
        uint64_t groups = (a.nnz + a.perGroup - 1) / a.perGroup;
        if (N == 3) {
            if (F.dtype == MMCSF_F32) run_geo<CooSel<3>::template K, CooArgs, float>(g, a, groups, s);
            else run_geo<CooSel<3>::template K, CooArgs, uint16_t>(g, a, groups, s);
        } else {
            if (F.dtype == MMCSF_F32) run_geo<CooSel<4>::template K, CooArgs, float>(g, a, groups, s);
            else run_geo<CooSel<4>::template K, CooArgs, uint16_t>(g, a, groups, s);
        }
    }
    // The walked parts, which share no slice, in one launch where the walks are
    // short: up to 2^19 nonzeros, and up to 2^22 where the CSF part is at least half
    // the CSL part (a sweep of random sizes and laws, R = 10 to 64, in turn / together:
    // 1.1-1.2 below 2^21, 1.09-1.15 from there to 2^22, 1.05 past it with 0.83 at worst;
    // larger CSL parts 1.11 below 2^19, 1.06 past it with 0.82 at worst).  A part of at
    // most 256 nonzeros is a latency, whatever the other's size (1.03-1.2).  The parts'
    // nonzeros cost differently; with the blocks shared by nonzeros one part's waited
    // for the other's (5M nonzeros, R = 40: 170 us in turn, 257 together).
    const uint64_t csf = h.csf.nnz, csl = h.cslWalk.nnz;
    if (csf && csl &&
        (csf + csl <= 1u << 19 || (csl <= 2 * csf && csf + csl <= 1u << 22) || std::min(csf, csl) <= 256)) {
        const Csf *trees[2] = {&h.csf, &h.cslWalk};
        float *const outs[2] = {out, out};
        if (mttkrp_roots(trees, 2, F, outs, s, true)) return;
    }
    // CSL part (3-D): walked as a tree of one-nonzero fibers; the CSL kernel
    // where the walk cannot run (R < 4, tables above 4 GiB)
    if (h.cslNnz && h.cslWalk.nnz && walk_supports(h.cslWalk, F.R, F.dtype)) {
        mttkrp_root(h.cslWalk, F, out, s);
    } else if (h.cslNnz) {
        CslArgs a{};
        a.ptr = h.cslPtr.p;
        a.idx = h.cslIdx.p;
        a.ind1 = h.cslInd1.p;
        a.ind2 = h.cslInd2.p;
        a.val = h.cslVal.p;
        a.U1 = F.U[h.order[1]];
        a.U2 = F.U[h.order[2]];
        a.out = out;
        a.nnz = (uint32_t)h.cslNnz;
        a.nslc = (uint32_t)h.nCsl;
        a.R = F.R;
        a.perGroup = per_group_for(h.cslNnz, g.G);
        uint64_t groups = (a.nnz + a.perGroup - 1) / a.perGroup;
        if (F.dtype == MMCSF_F32) run_geo<CslK, CslArgs, float>(g, a, groups, s);
        else run_geo<CslK, CslArgs, uint16_t>(g, a, groups, s);
    }
    // CSF part: root-mode walker (accumulates on top of the other parts' rows,
    // which are disjoint from its slices)
    if (h.csf.nnz) {
        if (walk_supports(h.csf, F.R, F.dtype)) mttkrp_root(h.csf, F, out, s);
        else launch_csf(h.csf, g, F, out, s);
    }
}

}  // namespace mmcsf
