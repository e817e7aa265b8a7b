// sf_searcher.hip -- uniform-grid neighbour searcher for gfx950.
//
// Replaces CudaGNBaseSearcher::BuildGNSearcher / CudaGNSearcher::SortData
// (cuda_neighbor_searcher.cu:36-116): FP32 cell hash, a stable LSD radix sort
// of 32-bit cell keys (wave64 ballot matching for in-wave ranks, LDS digit
// counters per wave, a scanned per-block digit histogram), cellStart from the
// sorted keys, and one gather of the persistent particle state.
#include "sf_internal.h"

namespace sf {

// ---------------------------------------------------------------------------
// hash: keys[i] = cell of pm[i]  (Pos2GridHash, helper_thrust.cuh:65-89)
template <bool kBatch>
__global__ __launch_bounds__(kBlock) void k_hash(SFConst k, const float4* __restrict__ pm,
                                                 const uint16_t* __restrict__ scene, uint32_t* __restrict__ keys,
                                                 uint8_t* __restrict__ wflag, int n) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const float4 p = pm[i];
    int cx, cy, cz;
    cell_of(k, p.x, p.y, p.z, cx, cy, cz);
    uint32_t key = cell_key(k, cx, cy, cz);
    if constexpr (kBatch) key += (uint32_t)scene[i] * k.C;
    keys[i] = key;
    if (wflag) wflag[i] = p.w > 0.f ? 1 : 0;  // the caller may have changed labels too
}
void launch_hash(const SFConst& k, const float4* pm, const uint16_t* scene, uint32_t* keys, uint8_t* wflag, int n,
                 hipStream_t s) {
    if (n <= 0) return;
    if (scene)
        k_hash<true><<<(n + kBlock - 1) / kBlock, kBlock, 0, s>>>(k, pm, scene, keys, wflag, n);
    else
        k_hash<false><<<(n + kBlock - 1) / kBlock, kBlock, 0, s>>>(k, pm, nullptr, keys, wflag, n);
}
void launch_hash_boundary(const SFConst& k, const float4* bp, uint32_t* keys, int nb, hipStream_t s) {
    launch_hash(k, bp, nullptr, keys, nullptr, nb, s);
}

// ---------------------------------------------------------------------------
// radix sort
RadixPlan make_radix_plan(uint32_t num_cells) {
    RadixPlan p;
    int K = 0;
    if (num_cells > 1) {
        uint32_t m = num_cells - 1;
        while (m) {
            ++K;
            m >>= 1;
        }
    }
    if (K < 1) K = 1;
    p.passes = (K + 7) / 8;
    int sh = 0;
    for (int i = 0; i < p.passes; ++i) {
        int rem_passes = p.passes - i, rem_bits = K - sh;
        int b = (rem_bits + rem_passes - 1) / rem_passes;
        p.shift[i] = sh;
        p.bits[i] = b;
        sh += b;
    }
    return p;
}

// lanes of the wave whose digit equals this lane's digit (among valid lanes)
SF_DEV uint64_t match_digit(uint32_t d, int bits, bool valid) {
    uint64_t m = __ballot(valid);
    for (int b = 0; b < bits; ++b) {
        const bool bit = (d >> b) & 1u;
        const uint64_t bb = __ballot(bit);
        m &= bit ? bb : ~bb;
    }
    return m;
}

// per-block digit counts -> hist[d * nblocks + block]
__global__ __launch_bounds__(kRsThreads) void k_rs_upsweep(const uint32_t* __restrict__ keys, int n, int shift,
                                                           int bits, uint32_t* __restrict__ hist) {
    __shared__ uint32_t cnt[256];
    const int t = threadIdx.x;
    cnt[t] = 0;
    __syncthreads();
    const uint32_t mask = (1u << bits) - 1u;
    const int base = blockIdx.x * kRsTile;
    const uint64_t lt = __lanemask_lt();
#pragma unroll 4
    for (int r = 0; r < kRsItems; ++r) {
        const int idx = base + r * kRsThreads + t;
        const bool valid = idx < n;
        const uint32_t d = valid ? (keys[idx] >> shift) & mask : 0u;
        const uint64_t peers = match_digit(d, bits, valid);
        if (valid && (peers & lt) == 0) atomicAdd(&cnt[d], (uint32_t)__popcll(peers));
    }
    __syncthreads();
    if (t <= (int)mask) hist[(size_t)t * gridDim.x + blockIdx.x] = cnt[t];
}

// exclusive scan of hist[0, total) in place by one workgroup of 1024
// threads; *total_out (if given) receives the sum
template <class U>
SF_DEV void scan_range(U* __restrict__ hist, int total, U* __restrict__ total_out) {
    __shared__ U wsum[16];
    __shared__ U carry_s;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    if (t == 0) carry_s = 0;
    __syncthreads();
    for (int base = 0; base < total; base += 1024 * 4) {
        U v[4];
        U s = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int idx = base + t * 4 + q;
            v[q] = idx < total ? hist[idx] : (U)0;
            s += v[q];
        }
        // inclusive wave scan of s
        U x = s;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            U y = __shfl_up(x, o, 64);
            if (lane >= o) x += y;
        }
        if (lane == 63) wsum[w] = x;
        __syncthreads();
        if (w == 0) {
            U ws = lane < 16 ? wsum[lane] : (U)0;
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) {
                U y = __shfl_up(ws, o, 64);
                if (lane >= o) ws += y;
            }
            if (lane < 16) wsum[lane] = ws;  // inclusive over waves
        }
        __syncthreads();
        const U carry = carry_s;
        U run = carry + (w > 0 ? wsum[w - 1] : (U)0) + x - s;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int idx = base + t * 4 + q;
            if (idx < total) hist[idx] = run;
            run += v[q];
        }
        __syncthreads();
        if (t == 1023) carry_s = carry + wsum[15];
        __syncthreads();
    }
    if (total_out && t == 0) *total_out = carry_s;
    __syncthreads();
}
template <class U>
__global__ __launch_bounds__(1024) void k_rs_scan(U* __restrict__ hist, int total, U* __restrict__ total_out) {
    scan_range<U>(hist, total, total_out);
}

// stable scatter: each wave ranks a contiguous chunk of 64*kRsItems keys
__global__ __launch_bounds__(kRsThreads) void k_rs_downsweep(const uint32_t* __restrict__ kin,
                                                             const uint32_t* __restrict__ vin, uint32_t* __restrict__ kout,
                                                             uint32_t* __restrict__ vout, int n, int shift, int bits,
                                                             const uint32_t* __restrict__ hist) {
    __shared__ uint32_t wcnt[4][256];
    const int t = threadIdx.x, w = t >> 6, lane = t & 63;
    for (int q = 0; q < 4; ++q) wcnt[q][t] = 0;
    __syncthreads();
    const uint32_t mask = (1u << bits) - 1u;
    const uint64_t lt = __lanemask_lt();
    const int base = blockIdx.x * kRsTile + w * (64 * kRsItems);
    uint32_t key[kRsItems], val[kRsItems], rank[kRsItems];
    volatile uint32_t* wc = wcnt[w];
#pragma unroll
    for (int r = 0; r < kRsItems; ++r) {
        const int idx = base + r * 64 + lane;
        const bool valid = idx < n;
        key[r] = valid ? kin[idx] : 0xffffffffu;
        val[r] = valid ? (vin ? vin[idx] : (uint32_t)idx) : 0u;
        const uint32_t d = valid ? (key[r] >> shift) & mask : 0u;
        const uint64_t peers = match_digit(d, bits, valid);
        const uint32_t before = (uint32_t)__popcll(peers & lt);
        const uint32_t c = wc[d];
        rank[r] = c + before;
        if (valid && before == 0) wc[d] = c + (uint32_t)__popcll(peers);
    }
    __syncthreads();
    {
        const uint32_t c0 = wcnt[0][t], c1 = wcnt[1][t], c2 = wcnt[2][t];
        const uint32_t g = t <= (int)mask ? hist[(size_t)t * gridDim.x + blockIdx.x] : 0u;
        __syncthreads();
        wcnt[0][t] = g;
        wcnt[1][t] = g + c0;
        wcnt[2][t] = g + c0 + c1;
        wcnt[3][t] = g + c0 + c1 + c2;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kRsItems; ++r) {
        const int idx = base + r * 64 + lane;
        if (idx < n) {
            const uint32_t d = (key[r] >> shift) & mask;
            const uint32_t pos = wcnt[w][d] + rank[r];
            if (pos < (uint32_t)n) {  // always true for a consistent histogram; keeps a bug in bounds
                kout[pos] = key[r];
                vout[pos] = val[r];
            }
        }
    }
}

int radix_sort(const uint32_t* keys, int n, const RadixPlan& plan, const SortBuffers& b, const uint32_t** sorted_keys,
               const uint32_t** perm, hipStream_t s) {
    *sorted_keys = b.kA;
    *perm = b.vA;
    if (n <= 0) return SF_OK;
    const int nblocks = (n + kRsTile - 1) / kRsTile;
    const uint32_t* kin = keys;
    const uint32_t* vin = nullptr;  // identity on the first pass
    uint32_t* ko = b.kA;
    uint32_t* vo = b.vA;
    for (int p = 0; p < plan.passes; ++p) {
        k_rs_upsweep<<<nblocks, kRsThreads, 0, s>>>(kin, n, plan.shift[p], plan.bits[p], b.hist);
        const int total = nblocks << plan.bits[p];
        k_rs_scan<uint32_t><<<1, 1024, 0, s>>>(b.hist, total, nullptr);
        k_rs_downsweep<<<nblocks, kRsThreads, 0, s>>>(kin, vin, ko, vo, n, plan.shift[p], plan.bits[p], b.hist);
        *sorted_keys = ko;
        *perm = vo;
        kin = ko;
        vin = vo;
        ko = (ko == b.kA) ? b.kB : b.kA;
        vo = (vo == b.vA) ? b.vB : b.vA;
    }
    SF_HIP(hipGetLastError());
    return SF_OK;
}

// ---------------------------------------------------------------------------
// cellStart[c] = number of particles with key < c, c in [0, C]
// (CountingInCell_CUDA + exclusive_scan, cuda_neighbor_searcher.cu:45-47),
// after a radix sort (the incremental sort's placement writes its own)
__global__ __launch_bounds__(kBlock) void k_cell_start(const uint32_t* __restrict__ sk, int n, uint32_t C,
                                                       const uint32_t* __restrict__ wpre, uint32_t* __restrict__ cs,
                                                       uint2* __restrict__ ct, PhasePos pp, IncClear z) {
    const uint32_t c = blockIdx.x * kBlock + threadIdx.x;
    // pph[t] = pm[plist[t]]: coalesced stores, loads that walk each phase's
    // slots in increasing order
    if (pp.pph && c < (uint32_t)n) pp.pph[c] = ldo(pp.pm, ldo(pp.plist, c));
    if (c < z.parts) z.part[c] = 0ull;
    if (c > C) return;
    if (z.in_count) {
        z.in_count[c] = 0ull;
        z.head[c] = 0u;
    }
    uint32_t lo = 0, hi = (uint32_t)n;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (sk[mid] < c) lo = mid + 1;
        else hi = mid;
    }
    cs[c] = lo;
    if (ct) ct[c] = make_uint2(lo, wpre ? wpre[lo] : 0u);
}
void launch_cell_start(const uint32_t* sorted_keys, int n, uint32_t C, const uint32_t* wpre, uint32_t* cell_start,
                       uint2* ct, PhasePos pp, IncClear z, hipStream_t s) {
    uint32_t total = C + 1;
    if (pp.pph && (uint32_t)n > total) total = (uint32_t)n;
    if (z.parts > total) total = z.parts;
    k_cell_start<<<(total + kBlock - 1) / kBlock, kBlock, 0, s>>>(sorted_keys, n, C, wpre, cell_start, ct, pp, z);
}

// ---------------------------------------------------------------------------
// reorder of the persistent state (the zipped payload of sort_by_key,
// cuda_neighbor_searcher.cu:90-111)
// Each block gathers one water-prefix tile (kWpTile slots) and stores the
// tile's water count in wpart[block] for the prefix that follows.
constexpr int kWpItems = 8;
constexpr int kWpTile = kBlock * kWpItems;
static_assert(kWpTile == kMoveTile, "the tiles whoever counts the moves sums over");
__global__ __launch_bounds__(kBlock) void k_gather(GatherArgs a, int n, uint32_t* __restrict__ wpart) {
    __shared__ uint32_t ws[kBlock / 64];
    const int t = threadIdx.x;
    uint32_t c = 0;
#pragma unroll
    for (int q = 0; q < kWpItems; ++q) {
        const int i = blockIdx.x * kWpTile + q * kBlock + t;
        if (i >= n) break;
        uint32_t p = a.perm[i];
        if (p >= (uint32_t)n) p = (uint32_t)i;  // a permutation of [0, n) never takes this branch
        const float4 pm = a.pm_in[p];
        a.pm_out[i] = pm;
        a.vr_out[i] = a.vr_in[p];
        a.cs_out[i] = a.cs_in[p];
        if (a.multi) {
            a.cda_out[i] = a.cda_in[p];
            a.amc_out[i] = a.amc_in[p];
        }
        const uint32_t water = pm.w > 0.f ? 1u : 0u;
        a.wflag[i] = (uint8_t)water;
        c += water;
    }
    for (int o = 32; o > 0; o >>= 1) c += __shfl_down(c, o, 64);
    if ((t & 63) == 0) ws[t >> 6] = c;
    __syncthreads();
    if (t == 0) {
        uint32_t sum = 0;
        for (int q = 0; q < kBlock / 64; ++q) sum += ws[q];
        wpart[blockIdx.x] = sum;
    }
}

__global__ __launch_bounds__(kBlock) void k_boundary_gather(const uint32_t* __restrict__ perm,
                                                            const float4* __restrict__ in, float4* __restrict__ out,
                                                            int nb) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= nb) return;
    uint32_t p = perm[i];
    if (p >= (uint32_t)nb) p = (uint32_t)i;
    out[i] = in[p];
}
void launch_boundary_gather(const uint32_t* perm, const float4* bp_in, float4* bp_out, int nb, hipStream_t s) {
    if (nb <= 0) return;
    k_boundary_gather<<<(nb + kBlock - 1) / kBlock, kBlock, 0, s>>>(perm, bp_in, bp_out, nb);
}

// ComputeBoundaryVolume_CUDA (cuda_sph_system_gpu.cuh:18-66): bpv.w enters as
// +-1 (label sign) and leaves as +-V_b.
__global__ __launch_bounds__(kBlock) void k_boundary_volume(SFConst k, float4* __restrict__ bpv,
                                                            const uint32_t* __restrict__ bcs, int nb) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= nb) return;
    const float4 pi = bpv[i];
    int cx, cy, cz;
    cell_of(k, pi.x, pi.y, pi.z, cx, cy, cz);
    float sum = 0.f;
    for_columns(k, cx, cy, cz, [&](uint32_t c0, uint32_t c1) {
        const uint32_t e = bcs[c1];
        for (uint32_t j = bcs[c0]; j < e; ++j) {
            if ((int)j == i) continue;
            const float4 pj = bpv[j];
            const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
            sum += poly6_r2(k, dx * dx + dy * dy + dz * dz);
        }
    });
    const float v = 1.f / fmaxf(sum, kEps);
    // every thread reads only .xyz of other slots, so writing .w is race-free
    bpv[i].w = pi.w < 0.f ? -v : v;
}
void launch_boundary_volume(const SFConst& k, float4* bpv, const uint32_t* bcs, int nb, hipStream_t s) {
    if (nb <= 0) return;
    k_boundary_volume<<<(nb + kBlock - 1) / kBlock, kBlock, 0, s>>>(k, bpv, bcs, nb);
}

// Cells whose 27-cell neighbourhood holds boundary particles: the passes'
// boundary loops skip the others, and walk only the columns that hold any
// (a face cell has 3 of 9; the boundary never moves, so the list is made once
// per upload).  near[c] = 1 if any, + 2 if any of label 1, + 16 x the number
// of such columns.
// Label 1 first, if there is any: each such particle marks the cells around
// its own (all that mark a byte write the same).
__global__ __launch_bounds__(kBlock) void k_boundary_mark(SFConst k, const float4* __restrict__ bpv, int nb,
                                                          uint8_t* __restrict__ near) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= nb) return;
    const float4 b = bpv[i];
    if (b.w >= 0.f) return;
    int cx, cy, cz;
    cell_of(k, b.x, b.y, b.z, cx, cy, cz);
    for_columns(k, cx, cy, cz, [&](uint32_t c0, uint32_t c1) {
        for (uint32_t c = c0; c < c1; ++c) near[c] = 2;
    });
}
// near, and row[c] = where cell c's non-empty column ranges start among those
// of all cells, whose number is left in *total (the blocks' rows lie in the
// order the atomics leave).  Each boundary particle is in one column range of
// at most 27 cells, so at most 27 x 2^27 ranges: the sums fit 32 bits.
__global__ __launch_bounds__(kBlock) void k_boundary_near(SFConst k, const uint32_t* __restrict__ bcs,
                                                          uint8_t* __restrict__ near, uint32_t* __restrict__ row,
                                                          uint32_t* __restrict__ total) {
    __shared__ uint32_t sums[kBlock / 64], base;
    const uint32_t c = blockIdx.x * kBlock + threadIdx.x;
    const int lane = (int)(threadIdx.x & 63u), w = (int)(threadIdx.x >> 6);
    uint32_t cols = 0;
    if (c < k.C) {
        const int cz = (int)(c % (uint32_t)k.gz), cy = (int)((c / (uint32_t)k.gz) % (uint32_t)k.gy);
        const int cx = (int)(c / ((uint32_t)k.gz * (uint32_t)k.gy));
        for_columns(k, cx, cy, cz, [&](uint32_t c0, uint32_t c1) { cols += bcs[c1] > bcs[c0] ? 1u : 0u; });
        near[c] = (uint8_t)((cols ? 1u : 0u) | (near[c] & 2u) | (cols << 4));
    }
    uint32_t x = cols;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) sums[w] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t all = 0;
        for (int q = 0; q < kBlock / 64; ++q) all += sums[q];
        base = all ? atomicAdd(total, all) : 0u;
    }
    __syncthreads();
    if (c >= k.C) return;
    uint32_t at = base + x - cols;
    for (int q = 0; q < w; ++q) at += sums[q];
    row[c] = at;
}
// The rows themselves, in for_columns order.
__global__ __launch_bounds__(kBlock) void k_boundary_rows(SFConst k, const uint32_t* __restrict__ bcs,
                                                          const uint8_t* __restrict__ near,
                                                          const uint32_t* __restrict__ row, uint2* __restrict__ ranges) {
    const uint32_t c = blockIdx.x * kBlock + threadIdx.x;
    if (c >= k.C || !near[c]) return;
    const int cz = (int)(c % (uint32_t)k.gz), cy = (int)((c / (uint32_t)k.gz) % (uint32_t)k.gy);
    const int cx = (int)(c / ((uint32_t)k.gz * (uint32_t)k.gy));
    uint2* out = ranges + row[c];
    for_columns(k, cx, cy, cz, [&](uint32_t c0, uint32_t c1) {
        const uint32_t s = bcs[c0], e = bcs[c1];
        if (e > s) *out++ = make_uint2(s, e);
    });
}
void launch_boundary_near(const SFConst& k, const float4* bpv, int nb, const uint32_t* bcs, uint8_t* near,
                          uint32_t* row, uint32_t* total, hipStream_t s) {
    if (k.C == 0) return;
    if (k.blabel1 && nb > 0) k_boundary_mark<<<(nb + kBlock - 1) / kBlock, kBlock, 0, s>>>(k, bpv, nb, near);
    k_boundary_near<<<(k.C + kBlock - 1) / kBlock, kBlock, 0, s>>>(k, bcs, near, row, total);
}
void launch_boundary_rows(const SFConst& k, const uint32_t* bcs, const uint8_t* near, const uint32_t* row,
                          uint2* ranges, hipStream_t s) {
    if (k.C == 0) return;
    k_boundary_rows<<<(k.C + kBlock - 1) / kBlock, kBlock, 0, s>>>(k, bcs, near, row, ranges);
}

// ---------------------------------------------------------------------------
// wpre[i] = number of water particles among sorted slots [0, i), i in [0, n]:
// lets a neighbour loop see how many water / sand particles a contiguous
// cell range holds (wpre[e] - wpre[s]) and skip ranges without the phase it
// needs.  Two kernels around a tiny scan of per-block counts.
int wprefix_blocks(int n) { return (n + kWpTile - 1) / kWpTile; }

// tile's slot prefixes from its scanned partial (thread t owns kWpItems
// consecutive slots); slot n (one past the end) receives the total.
// emit(i, prefix, value) is called for every slot i < n.
// Up to kDirectTiles tiles, each prefix block sums the tile counts it needs
// itself instead of waiting for a one-block scan launch: the sum of cnt[q]
// over q in [lo, b) (before) and over [lo, hi) (all), by the whole block.
constexpr int kDirectTiles = 4096;
int g_direct_tiles = kDirectTiles;  // sf_set_prefix_scan_threshold
template <class U>
SF_DEV void block_sums(const U* __restrict__ cnt, uint32_t lo, uint32_t b, uint32_t hi, U& before, U& all) {
    __shared__ U red[2][kBlock / 64];
    U a = 0, p = 0;
    uint32_t q = lo + threadIdx.x;
    for (; q + 7u * kBlock < hi; q += 8u * kBlock) {  // eight loads in flight
        U c[8];
#pragma unroll
        for (uint32_t m = 0; m < 8u; ++m) c[m] = cnt[q + m * kBlock];
#pragma unroll
        for (uint32_t m = 0; m < 8u; ++m) {
            a += c[m];
            p += q + m * kBlock < b ? c[m] : (U)0;
        }
    }
    for (; q < hi; q += kBlock) {
        const U c = cnt[q];
        a += c;
        p += q < b ? c : (U)0;
    }
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_down(a, o, 64);
        p += __shfl_down(p, o, 64);
    }
    if ((threadIdx.x & 63u) == 0) {
        red[0][threadIdx.x >> 6] = a;
        red[1][threadIdx.x >> 6] = p;
    }
    __syncthreads();
    all = 0;
    before = 0;
    for (int w = 0; w < kBlock / 64; ++w) {
        all += red[0][w];
        before += red[1][w];
    }
}

template <class U, class V, class Emit>
SF_DEV void tile_prefix(V v, int n, int tile, U part, U* __restrict__ out, Emit&& emit) {
    __shared__ U wsum[kBlock / 64];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int base = tile * kWpTile + t * kWpItems;
    U f[kWpItems];
    U s = 0;
    if (base + kWpItems <= n) {
        v.load8(base, f);  // whole run in range: vector loads
    } else {
#pragma unroll
        for (int q = 0; q < kWpItems; ++q) f[q] = base + q < n ? v(base + q) : (U)0;
    }
#pragma unroll
    for (int q = 0; q < kWpItems; ++q) s += f[q];
    U x = s;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        U y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    U run = part + x - s;
    for (int q = 0; q < w; ++q) run += wsum[q];
#pragma unroll
    for (int q = 0; q < kWpItems; ++q) {
        const int i = base + q;
        if (i <= n) out[i] = run;
        if (i < n) emit(i, run, f[q]);
        run += f[q];
    }
}
struct NoEmit {
    template <class U>
    SF_DEV void operator()(int, U, U) const {}
};

// Per-slot values of the prefixes; load8(i, f) reads slots i .. i + 7 (i a
// multiple of 8, all below n) with vector loads.
// A count of particles and, in the upper half, of the water among them
// (counts stay below 2^27).
SF_DEV uint64_t counted(bool one, bool water) { return one ? (water ? 0x100000001ull : 1ull) : 0ull; }
struct ArrayVal {
    const uint64_t* a;
    SF_DEV uint64_t operator()(int i) const { return a[i]; }
    SF_DEV void load8(int i, uint64_t* f) const {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const ulonglong2 v = *reinterpret_cast<const ulonglong2*>(a + i + 2 * q);
            f[2 * q] = v.x;
            f[2 * q + 1] = v.y;
        }
    }
};
struct FlagVal {
    const uint8_t* f;
    SF_DEV uint32_t operator()(int i) const { return f[i]; }
    SF_DEV void load8(int i, uint32_t* o) const {
        const uint2 w = *reinterpret_cast<const uint2*>(f + i);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            o[q] = (w.x >> (8 * q)) & 0xffu;
            o[4 + q] = (w.y >> (8 * q)) & 0xffu;
        }
    }
};

// Exclusive prefixes of the incremental sort: the blocks' totals over
// [0, n1) into out1[0, n1] (blocks [0, nb1); there is one total per kBlock
// slots, so each block sums all of those before its own itself), and the
// newcomer counts over [0, n2) into out2[0, n2], whose sums per tile of
// kWpTile cells are in part.
// scanned = 0: part holds the raw tile sums, and each block sums those
// before it within its own prefix (the block holding slot n thereby ends on
// the total, as the scan would give it).
__global__ __launch_bounds__(kBlock) void k_inc_prefix(const uint64_t* __restrict__ totals, int n1, int nb1,
                                                       uint64_t* __restrict__ out1,
                                                       const uint64_t* __restrict__ in_count, int n2,
                                                       uint64_t* __restrict__ out2, const uint64_t* __restrict__ part,
                                                       int scanned) {
    const int b = (int)blockIdx.x - nb1;  // tile of the counts
    uint64_t before = 0, all;
    if (b < 0) {
        const uint32_t first = blockIdx.x * (uint32_t)kWpTile;
        block_sums(totals, 0u, first, first, before, all);
        tile_prefix(ArrayVal{totals}, n1, (int)blockIdx.x, before, out1, NoEmit{});
        return;
    }
    if (scanned) before = part[b];
    else block_sums(part, 0u, (uint32_t)b, gridDim.x - (uint32_t)nb1, before, all);
    tile_prefix(ArrayVal{in_count}, n2, b, before, out2, NoEmit{});
}
// Water prefix of the gathered slots (k_gather left the tile counts in
// wpart) and the slots grouped by phase (water first, each group in slot
// order) so that a pass over one phase can give every XCD an equal
// contiguous share of it.
// With scanned = 0, wpart holds the raw per-tile counts and each block sums
// the counts before its tile, and all of them, itself (a few thousand tiles
// at most), instead of waiting for a one-block scan launch.
__global__ __launch_bounds__(kBlock) void k_wprefix_plist(const uint8_t* __restrict__ wflag, int n,
                                                          const uint32_t* __restrict__ wpart, int scanned,
                                                          uint32_t* __restrict__ wpre, uint32_t* __restrict__ plist) {
    uint32_t nwater, part;
    if (scanned) {
        nwater = wpart[gridDim.x];
        part = wpart[blockIdx.x];
    } else {
        block_sums(wpart, 0u, blockIdx.x, gridDim.x, part, nwater);
    }
    tile_prefix<uint32_t>(FlagVal{wflag}, n, (int)blockIdx.x, part, wpre, [&](int i, uint32_t pre, uint32_t water) {
        plist[water ? pre : nwater + (uint32_t)i - pre] = (uint32_t)i;
    });
}
int set_direct_tiles(int tiles) {
    const int prev = g_direct_tiles;
    g_direct_tiles = tiles < 0 ? kDirectTiles : tiles;
    return prev;
}
void launch_gather_wprefix(const GatherArgs& a, int n, uint32_t* wpart, uint32_t* wpre, uint32_t* plist,
                           hipStream_t s) {
    const int nb = wprefix_blocks(n + 1);
    k_gather<<<nb, kBlock, 0, s>>>(a, n, wpart);
    const int scanned = nb > g_direct_tiles ? 1 : 0;
    if (scanned) k_rs_scan<uint32_t><<<1, 1024, 0, s>>>(wpart, nb, wpart + nb);
    k_wprefix_plist<<<nb, kBlock, 0, s>>>(a.wflag, n, wpart, scanned, wpre, plist);
}

// ---------------------------------------------------------------------------
// Incremental stable sort and reorder.  The particles are in the previous
// step's sorted order and most keep their cell, so the stable sort by the new
// keys is rebuilt without radix passes: within each new cell the particles
// are ordered by current index, so a particle's output slot is
//   newStart(c) + #(stayers of c before it) + #(newcomers of c before it),
// where stayers of c are the particles of c's old block whose key is still c
// (a prefix over "key unchanged" flags counts them) and newcomers are the
// few particles whose key changed to c (chained per cell, in the order the
// atomics leave; a newcomer's rank is the count of smaller indices in its
// cell's chain, which that order does not change).
// newStart(c) = stayers in cells < c + newcomers in cells < c.
// The result is the stable sort's, element for element.
//
// A chain is dependent loads, walked by every particle of its cell: some 0.27
// us per newcomer of the fullest cell.  With every particle of 500k + 500k
// moving by about a cell the build takes 149 us (163 with contiguous lists,
// filled by a launch of their own); only where hundreds enter one cell at
// once does the chain lose to them (500 of 101k: 193 against 111 us, the
// solve of such a pile 300; 3000: 820 against 370, solve 1160).
//
// Every count carries the water's share in its upper half, so the same sums
// give the number of water particles before a slot, that is the particle's
// index within its phase, and the placement reorders everything at once:
// permutation, keys, the persistent state, the phase list, the positions in
// phase order and the cell table.  With the tile sums of both prefixes taken
// by whoever wrote the keys, two launches follow the advect; they were seven
// (two prefix passes, newcomer lists, permutation, gather, water prefix,
// cell table), each at least 2-4 us however small the scene, and they moved
// the permutation, the flags and the positions once more each.
__global__ __launch_bounds__(kBlock) void k_inc_flag(const uint32_t* __restrict__ key, const uint32_t* __restrict__ old,
                                                     const uint8_t* __restrict__ wflag, int n, Newcomers nc) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    const bool valid = i < n;
    count_moves(valid ? key[i] : 0u, valid ? old[i] : 0u, valid && wflag[i] != 0, i, n, nc);
}
// The slots before j whose key did not change (count_moves: the block's own
// before it, and the blocks' totals before its block).
SF_DEV uint64_t stay_before(const PlaceArgs& a, uint32_t j) {
    const uint32_t l = j % (uint32_t)kBlock ? a.local[j] : 0u;
    return a.stay_base[j / (uint32_t)kBlock] + (((uint64_t)(l >> 16) << 32) | (l & 0xffffu));
}
__global__ __launch_bounds__(kBlock) void k_inc_place(PlaceArgs a, int n, uint32_t C, int place_blocks) {
    if ((int)blockIdx.x >= place_blocks) {
        // the new cell table, and the next sort's counters
        const uint32_t c = (blockIdx.x - (uint32_t)place_blocks) * kBlock + threadIdx.x;
        if (c < a.parts) a.part[c] = 0ull;
        if (c > C) return;
        const uint64_t before = stay_before(a, a.ct_old[c].x) + a.in_start[c];
        const uint2 e = make_uint2((uint32_t)before, (uint32_t)(before >> 32));
        a.cell[c] = e.x;
        a.ct[c] = e;
        a.in_count[c] = 0ull;
        a.head_next[c] = 0u;
        if (c == C) *a.nwater = e.y;
        return;
    }
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const uint32_t c = a.key[i], o = a.old_key[i];
    const float4 pm = a.g.pm_in[i], vr = a.g.vr_in[i], cs = a.g.cs_in[i];
    const uint32_t oa = a.ct_old[c].x, ob = a.ct_old[c + 1].x;
    const uint64_t s = a.in_start[c], e = a.in_start[c + 1];
    const uint64_t nwater = stay_before(a, (uint32_t)n) + a.in_start[C];  // all water, in the upper half
    const uint64_t sa = stay_before(a, oa);
    const uint32_t u = (uint32_t)i;
    uint64_t rank = 0;  // of the cell: stayers before, then newcomers before
    if (c == o || (u >= oa && u < ob)) rank = stay_before(a, u) - sa;
    else if (u >= ob) rank = stay_before(a, ob) - sa;
    // the cell's chain is as long as its newcomer count; the count ends the walk
    uint32_t left = (uint32_t)e - (uint32_t)s;
    for (uint32_t q = left ? a.head[c] : 0u; q != 0u; q = a.next[(q & kChainIndex) - 1u]) {
        if ((q & kChainIndex) - 1u < u) rank += counted(true, (q & ~kChainIndex) != 0u);
        if (--left == 0u) break;
    }
    const uint64_t at = sa + s + rank;
    const uint32_t pos = (uint32_t)at, wbefore = (uint32_t)(at >> 32);
    if (pos >= (uint32_t)n) return;  // never for consistent counts; keeps a bug in bounds
    const bool water = pm.w > 0.f;
    const uint32_t t = water ? wbefore : (uint32_t)(nwater >> 32) + pos - wbefore;
    a.perm[pos] = u;
    a.sorted_keys[pos] = c;
    a.g.pm_out[pos] = pm;
    a.g.vr_out[pos] = vr;
    a.g.cs_out[pos] = cs;
    if (a.g.multi) {
        a.g.cda_out[pos] = a.g.cda_in[i];
        a.g.amc_out[pos] = a.g.amc_in[i];
    }
    a.g.wflag[pos] = water ? 1 : 0;
    if (t < (uint32_t)n) {
        a.plist[t] = pos;
        a.pph[t] = pm;
    }
}

uint32_t inc_parts(uint32_t C) { return (uint32_t)wprefix_blocks((int)C + 1); }
void launch_incremental_sort(const PlaceArgs& a, const Newcomers& nc, int n, uint32_t C, bool flags_done,
                             hipStream_t s) {
    if (n <= 0) return;
    const int gn = (n + kBlock - 1) / kBlock;
    // in_count, the chains and part are zero here: every build clears them
    if (!flags_done) k_inc_flag<<<gn, kBlock, 0, s>>>(a.key, a.old_key, a.g.wflag, n, nc);
    const int nb1 = wprefix_blocks(gn + 1), nb2 = (int)a.parts;
    const int scanned = nb2 > g_direct_tiles ? 1 : 0;
    if (scanned) k_rs_scan<uint64_t><<<1, 1024, 0, s>>>(a.part, nb2, nullptr);
    k_inc_prefix<<<nb1 + nb2, kBlock, 0, s>>>(nc.totals, gn, nb1, a.stay_base, a.in_count, (int)C, a.in_start, a.part,
                                              scanned);
    k_inc_place<<<gn + (int)((C + 1 + kBlock - 1) / kBlock), kBlock, 0, s>>>(a, n, C, gn);
}

// in-range neighbour counts: r^2 = dx*dx + dy*dy + dz*dz in FP32, left to
// right without contraction, compared with h^2
__global__ __launch_bounds__(kBlock) void k_nbr_count(SFConst k, const float4* __restrict__ pm,
                                                      const uint16_t* __restrict__ scene,
                                                      const uint32_t* __restrict__ cs, uint32_t* __restrict__ cnt,
                                                      uint32_t* __restrict__ cand, int n) {
#pragma clang fp contract(off)
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const float4 pi = pm[i];
    const uint32_t cb = scene ? (uint32_t)scene[i] * k.C : 0u;
    int cx, cy, cz;
    cell_of(k, pi.x, pi.y, pi.z, cx, cy, cz);
    uint32_t c = 0, cc = 0;
    for_columns(k, cx, cy, cz, [&](uint32_t c0, uint32_t c1) {
        const uint32_t s0 = cs[cb + c0], e = cs[cb + c1];
        cc += e - s0;
        for (uint32_t j = s0; j < e; ++j) {
#pragma clang fp contract(off)
            // written out here (not via helpers) so the pragma governs every
            // operation and nothing is fused into an FMA
            const float4 pj = pm[j];
            const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
            const float xx = dx * dx, yy = dy * dy, zz = dz * dz;
            const float r2 = (xx + yy) + zz;
            c += r2 < k.h2 ? 1u : 0u;
        }
    });
    cnt[i] = c;
    cand[i] = cc;
}
void launch_nbr_count(const SFConst& k, const float4* pm, const uint16_t* scene, const uint32_t* cs, uint32_t* cnt,
                      uint32_t* cand, int n, hipStream_t s) {
    if (n <= 0) return;
    k_nbr_count<<<(n + kBlock - 1) / kBlock, kBlock, 0, s>>>(k, pm, scene, cs, cnt, cand, n);
}

}  // namespace sf
