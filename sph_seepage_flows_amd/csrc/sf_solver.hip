// sf_solver.hip -- the per-step solver passes of the coupled SPH-DEM seepage
// step on gfx950 (one thread per particle over the cell-sorted arrays; each
// thread walks its 27-cell neighbourhood as 9 contiguous z-ranges).
//
// Pass structure (dependencies of cuda_wcsph_sf_solver.cpp:44-177):
//   P1 density + EOS            <- ComputeSFDensity_CUDA, ComputeSFPressure(ByTait)_CUDA
//   P2 avg flow / voidage / sat <- ComputeSFAvgFlow_CUDA
//   P3 sand voidage | water adhesion
//                               <- ComputeSFSandVoidage_CUDA, Compute(Multi)SFWaterAdhesionForces_CUDA
//   P4 sand momentum + colour   <- Compute(Multi)SFSandLinearMomentum_CUDA, ComputeSFWetSandColor_CUDA
//   P5 water momentum           <- ComputeSFWaterLinearMomentum_CUDA
//   CFL (optional), advect      <- ComputeSubTimeStepsByCFL, CudaSFParticles::Advect,
//                                  SFWaterBoundaryConstrain_CUDA
// ExtraForces (acc = g) is folded into P4/P5, which write the final acc.
#include <type_traits>

#include "sf_internal.h"
#include "sf_nlist.h"

namespace sf {

// Tait EOS B((rho/rho0)^7 - 1) (cuda_wcsph_sf_solver_gpu.cuh:34) evaluated as
// B * u * (1 + x + ... + x^6) with u = (rho - rho0) / rho0, x = rho / rho0,
// which avoids the cancellation of x^7 - 1 near rest density.
SF_DEV float eos(const SFConst& k, float rho) {
    float p;
    if (k.tait) {
        const float x = rho / k.rho0;
        const float u = (rho - k.rho0) / k.rho0;
        const float s = 1.f + x * (1.f + x * (1.f + x * (1.f + x * (1.f + x * (1.f + x)))));
        p = k.stiff * u * s;
    } else {
        p = k.stiff * (rho - k.rho0);  // ComputeSFPressure_CUDA (cuda_sph_sf_solver_gpu.cuh:497)
    }
    if (p < 0.f) p *= k.neg_scale;
    return p;
}

// The water count: a wave that knows it from its arguments, and its own
// position (and in P4 velocity and saturation) from the phase order, starts
// its walk two dependent loads earlier and reads contiguously: P4 257 -> 230
// us and P1 189 -> 183 at 4M.  P5 keeps the slot's record, which it needs
// anyway (with the position from the phase order 124 -> 127 us at 1M).
SF_DEV uint32_t water_count(const Fields& f) { return f.nw >= 0 ? (uint32_t)f.nw : *f.nwater; }
// Position and mass of the particle of phase index t in slot i.
SF_DEV float4 own_pos(const Fields& f, uint32_t t, int i) {
    return f.nw >= 0 ? ldo(f.pph, t) : ldo(f.pm, (uint32_t)i);
}

// The same as its neighbours see it: pph[t], which is also pi while nothing was
// written since the build.
SF_DEV float4 built_pos(const Fields& f, uint32_t t, const float4& pi) { return f.fresh ? pi : ldo(f.pph, t); }

// First cell key of slot i's scene (batched handles), 0 otherwise.
template <bool B>
SF_DEV uint32_t scene_base(const SFConst& k, const Fields& f, int i) {
    if constexpr (B) return (uint32_t)ldo(f.scene, (uint32_t)i) * k.C;
    else return 0u;
}

// Every S-th slot j of [s, e) whose test(j, pm[j]) holds goes to the list,
// in slot order.  Four candidates per round: four independent loads in
// flight per lane (the loop is otherwise bound by one dependent global load
// per candidate) from one base address with immediate offsets, and one
// list-full check per round (a list at CAP or more is flushed first; a round
// then leaves at most CAP + 3 entries, which the list has room for).
// The pairs reach apply in the same order whenever the flushes fall.
template <uint32_t S, int NB, int CAP, class Test, class Fetch, class Apply>
SF_DEV void filter_push(NList<NB, CAP>& L, const float4* __restrict__ pm, uint32_t s, uint32_t e, Test&& test,
                        Fetch&& fetch, Apply&& apply) {
    static_assert(CAP >= 4, "a round pushes up to four candidates");
    uint32_t j = s;
    for (; j + 3u * S < e; j += 4u * S) {
        // slot offsets stay below 2^31 bytes, so base + 16 q S does not wrap
        const float4* q = reinterpret_cast<const float4*>(reinterpret_cast<const char*>(pm) + j * 16u);
        const float4 a = q[0], b = q[S], c = q[2u * S], d = q[3u * S];
        const bool ka = test(j, a), kb = test(j + S, b), kc = test(j + 2u * S, c), kd = test(j + 3u * S, d);
        if (__ballot(L.cnt >= CAP)) nl_flush2(L, fetch, apply);
        L.slot[L.cnt * NB] = j;
        L.cnt += ka ? 1 : 0;
        L.slot[L.cnt * NB] = j + S;
        L.cnt += kb ? 1 : 0;
        L.slot[L.cnt * NB] = j + 2u * S;
        L.cnt += kc ? 1 : 0;
        L.slot[L.cnt * NB] = j + 3u * S;
        L.cnt += kd ? 1 : 0;
    }
    for (; j < e; j += S) {
        const float4 a = ldo(pm, j);
        nl_push2(L, test(j, a), j, fetch, apply);
    }
}

// Phase-index range of one phase in the cells [c0, c1) of a column: a slot
// range [s, e) holds the water candidates pph[wpre[s], wpre[e]) and the sand
// candidates pph[nw + s - wpre[s], nw + e - wpre[e]), each in slot order (the
// cell table holds both ends).
SF_DEV uint2 phase_range(const uint2* __restrict__ ct, uint32_t c0, uint32_t c1, bool water, uint32_t nw) {
    const uint2 a = ldo(ct, c0), b = ldo(ct, c1);
    return water ? make_uint2(a.y, b.y) : make_uint2(nw + (a.x - a.y), nw + (b.x - b.y));
}

SF_DEV float sq3(float d) { return d * d * d; }

// ---------------------------------------------------------------------------
// Wave-staged neighbour columns.  The 64 lanes of a wave hold consecutive
// slots of the cell-sorted order, so they sit in a few consecutive cells of
// one grid column (x, y), rarely two or three, and their 27-cell
// neighbourhoods overlap almost entirely: lane by lane, the eight or so lanes
// of one cell would load exactly the same candidates.  Here the lanes that
// share a column (a "segment") take, for each of the 9 neighbour columns, the
// union of their z-ranges -- one contiguous slot range, from the first lane's
// range start to the last lane's range end -- load it once with coalesced
// loads into the wave's LDS stage, and each lane then walks its own window
// of the union from LDS.  Each wave owns its stage; the lanes of one wave
// order their LDS accesses with wave-scope fences only.
constexpr int kStage = 128;  // candidates staged per chunk and wave

SF_DEV void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
template <class T>
SF_DEV T lane_value(T v, int lane) {
    return __builtin_amdgcn_readlane(v, lane);
}

// For the lanes with `active` set: fn(j, staged_j) over every slot j of the
// lane's 9 column ranges (cells z-1..z+1), column by column.  prep(pm[j]) is what gets staged (once per wave, not per
// lane).  need(nw, ns), given the water / sand counts of a column's union
// range, may skip the whole column.  Must be called by all lanes of the wave
// (uniform control flow).
// With L > 1 lanes per particle (adjacent lanes, same cell), lane sub of a
// particle takes the slots j = first + sub + L m of each of its ranges
// [first, last), in increasing j, however the ranges fall into stage chunks
// (the same split as a per-lane walk of the ranges).
// With Water set, the walk covers only the water candidates: phase indices
// [wpre[s], wpre[e]) of each column range, staged from pph.  range(a, b) sees
// each of the lane's own 9 cell-table pairs (range start, range end).
template <int L = 1, bool Water = false, class Prep, class Need, class Fn, class Range>
SF_DEV void staged_walk(const SFConst& k, const Fields& f, float4* __restrict__ stage, bool active, uint32_t cb,
                        int cx, int cy, int cz, Prep&& prep, Need&& need, Fn&& fn, Range&& range) {
    static_assert((L & (L - 1)) == 0, "lanes per particle: a power of two");
    const int lane = (int)(threadIdx.x & 63u);
    const uint32_t sub = (uint32_t)lane & (uint32_t)(L - 1);
    const uint32_t col = cb + (uint32_t)((cx * k.gy + cy) * k.gz);
    const int zlo = cz > 0 ? cz - 1 : 0;
    const int zhi = cz + 1 < k.gz ? cz + 1 : k.gz - 1;
    uint64_t todo = __ballot(active);
    while (todo) {
        const int lead = __builtin_ctzll(todo);
        const uint32_t lcol = lane_value(col, lead);
        const bool mine = active && col == lcol;
        const uint64_t seg = __ballot(mine);
        todo &= ~seg;
        const int last = 63 - __builtin_clzll(seg);
        const int sx = lane_value(cx, lead), sy = lane_value(cy, lead);
        const uint32_t scb = lane_value(cb, lead);
        for (int dx = -1; dx <= 1; ++dx) {
            const int x = sx + dx;
            if (x < 0 || x >= k.gx) continue;
            for (int dy = -1; dy <= 1; ++dy) {
                const int y = sy + dy;
                if (y < 0 || y >= k.gy) continue;
                const uint32_t base = scb + (uint32_t)((x * k.gy + y) * k.gz);
                uint2 a = make_uint2(0u, 0u), b = make_uint2(0u, 0u);
                if (mine) {
                    a = ldo(f.ct + base, (uint32_t)zlo);
                    b = ldo(f.ct + base, (uint32_t)zhi + 1u);
                    range(a, b);
                }
                const uint32_t ax = Water ? a.y : a.x, bx = Water ? b.y : b.x;
                const uint32_t us = lane_value(ax, lead), ue = lane_value(bx, last);
                if (us >= ue) continue;
                const uint32_t nw = lane_value(b.y, last) - lane_value(a.y, lead);
                if (!need(nw, (lane_value(b.x, last) - lane_value(a.x, lead)) - nw)) continue;
                const float4* __restrict__ src = Water ? f.pph : f.pm;
                for (uint32_t u = us; u < ue; u += (uint32_t)kStage) {
                    const uint32_t m = ue - u < (uint32_t)kStage ? ue - u : (uint32_t)kStage;
                    for (uint32_t q = (uint32_t)lane; q < m; q += 64u) stage[q] = prep(ldo(src, u + q));
                    wave_sync();
                    const uint32_t wlo = ax > u ? ax : u, whi = bx < u + m ? bx : u + m;
                    constexpr uint32_t S = (uint32_t)L;
                    uint32_t j = wlo + ((ax + sub - wlo) & (S - 1u));  // j = ax + sub (mod L)
                    for (; j + 3u * S < whi; j += 4u * S) {
                        const float4 q0 = stage[j - u], q1 = stage[j + S - u], q2 = stage[j + 2u * S - u],
                                     q3 = stage[j + 3u * S - u];
                        fn(j, q0);
                        fn(j + S, q1);
                        fn(j + 2u * S, q2);
                        fn(j + 3u * S, q3);
                    }
                    for (; j < whi; j += S) fn(j, stage[j - u]);
                    wave_sync();
                }
            }
        }
    }
}

// The filtered walk of the passes: every candidate j of the particle's 9
// column ranges with test(src[j]) goes to the lane's list, lane sub (of S per
// particle) taking j = s + sub + S m of each range [s, e) in increasing j,
// exactly as filter_push over the ranges.  range(b, c0, c1) gives an active
// lane's [s, e) in src for the cells [b + c0, b + c1) of a column.  The filter is
// bound by the texture address unit, which costs the same per wave load
// instruction whatever it carries, so where the wave's ranges overlap it
// loads them once: when every particle of the wave sits in one grid column,
// its lanes in cell order (most waves of an ordered region), the lanes walk
// the same 9 columns, and a column whose union range (first lane's start to
// last lane's end) fits KS candidates is staged in LDS with coalesced loads
// (one per lane up to 64) and filtered from there.  Other columns, and waves
// spread over several columns, filter from memory per lane.  Either way a
// lane's list gets the same entries in the same order, so which way a column
// goes does not change the sums.  Must be called by all lanes of the wave.
// P2, P3 and P4's water walk stage the other phase's candidates (P2 216 ->
// 200 us, P3 216 -> 203, P4 176 -> 155 at 500k + 500k interpenetrating, all
// with 256-thread workgroups and before P3 and P4 read P2's saved neighbours;
// where little is listed, the stage's LDS leaves fewer of the waves that find
// nothing resident: 2 x 4 us of 1.12 ms at 4M).
constexpr uint32_t kStageList = 64;  // longest union range staged per wave: P2, P3, P4's water
// P5's candidates are both phases': 16 water particles span 2-3 cells, so the
// union is 4-5 cells of 8 water particles, or of 16 particles where the
// phases interpenetrate (64-80).  96 instead of 64, with 256-thread workgroups:
// P5 255 -> 227 us at 500k + 500k interpenetrating, 137 -> 138 us where they
// are apart.
constexpr uint32_t kStageWm = 96;
#define SF_STAGE(name, KS)                              \
    __shared__ float4 name##_lds[(NB / 64) * (KS)];     \
    float4* name = name##_lds + (threadIdx.x >> 6) * (KS)
template <uint32_t S, uint32_t KS, int NB, int CAP, class Range, class Test, class Fetch, class Apply>
SF_DEV void column_filter(const SFConst& k, const float4* __restrict__ src, float4* __restrict__ stage, bool active,
                          uint32_t cb, int cx, int cy, int cz, NList<NB, CAP>& L, Range&& range, Test&& test,
                          Fetch&& fetch, Apply&& apply) {
    static_assert(CAP >= 4, "a round pushes up to four candidates");
    static_assert(KS <= 128, "at most two staged candidates per lane");
    const int lane = (int)(threadIdx.x & 63u);
    const uint32_t sub = (uint32_t)lane % S;
    const uint64_t act = __ballot(active);
    if (!act) return;
    const int lead = __builtin_ctzll(act), last = 63 - __builtin_clzll(act);
    const uint32_t col = cb + (uint32_t)((cx * k.gy + cy) * k.gz);
    const uint32_t zlo = (uint32_t)(cz > 0 ? cz - 1 : 0), zhi = (uint32_t)(cz + 1 < k.gz ? cz + 1 : k.gz - 1);
    const bool one = !__ballot(active && (col != lane_value(col, lead) || cz < lane_value(cz, lead) ||
                                          cz > lane_value(cz, last)));  // wave-uniform
    if (!one) {
        if (!active) return;
        for (int dx = -1; dx <= 1; ++dx) {
            const int x = cx + dx;
            if (x < 0 || x >= k.gx) continue;
            for (int dy = -1; dy <= 1; ++dy) {
                const int y = cy + dy;
                if (y < 0 || y >= k.gy) continue;
                const uint2 r = range(0u, cb + (uint32_t)((x * k.gy + y) * k.gz) + zlo,
                                      cb + (uint32_t)((x * k.gy + y) * k.gz) + zhi + 1u);
                filter_push<S>(L, src, r.x + sub, r.y, test, fetch, apply);
            }
        }
        return;
    }
    // one column: its coordinates, the bounds checks and the columns' first
    // cells are the wave's (scalar registers and arithmetic)
    const int sx = lane_value(cx, lead), sy = lane_value(cy, lead);
    const uint32_t scb = lane_value(cb, lead);
    for (int dx = -1; dx <= 1; ++dx) {
        const int x = sx + dx;
        if (x < 0 || x >= k.gx) continue;
        for (int dy = -1; dy <= 1; ++dy) {
            const int y = sy + dy;
            if (y < 0 || y >= k.gy) continue;
            uint2 r = make_uint2(0u, 0u);
            if (active) r = range(scb + (uint32_t)((x * k.gy + y) * k.gz), zlo, zhi + 1u);
            const uint32_t us = lane_value(r.x, lead), ue = lane_value(r.y, last);
            if (us >= ue) continue;
            if (ue - us <= KS) {
                for (uint32_t q = (uint32_t)lane; q < ue - us; q += 64u) stage[q] = ldo(src + us, q);
                wave_sync();
                uint32_t j = r.x + sub;
                for (; j + 3u * S < r.y; j += 4u * S) {
                    const float4 a = stage[j - us], b = stage[j + S - us], c = stage[j + 2u * S - us],
                                 d = stage[j + 3u * S - us];
                    const bool ka = test(j, a), kb = test(j + S, b), kc = test(j + 2u * S, c), kd = test(j + 3u * S, d);
                    if (__ballot(L.cnt >= CAP)) nl_flush2(L, fetch, apply);
                    L.slot[L.cnt * NB] = j;
                    L.cnt += ka ? 1 : 0;
                    L.slot[L.cnt * NB] = j + S;
                    L.cnt += kb ? 1 : 0;
                    L.slot[L.cnt * NB] = j + 2u * S;
                    L.cnt += kc ? 1 : 0;
                    L.slot[L.cnt * NB] = j + 3u * S;
                    L.cnt += kd ? 1 : 0;
                }
                for (; j < r.y; j += S) nl_push2(L, test(j, stage[j - us]), j, fetch, apply);
                wave_sync();
            } else if (active) {
                filter_push<S>(L, src, r.x + sub, r.y, test, fetch, apply);
            }
        }
    }
}

// Lanes per particle of the interface passes (P2, P3), whose work sits at the
// water-sand interface (PassCfg::lanes): several lanes per particle let the
// few thousand waves of a small handle hide load latency.
template <class L>
void with_lanes(int lanes, L&& l) {
    switch (lanes) {
    case 4: l(std::integral_constant<int, 4>{}); break;
    case 2: l(std::integral_constant<int, 2>{}); break;
    default: l(std::integral_constant<int, 1>{}); break;
    }
}
// Sums x over the LP lanes of a particle (adjacent lanes, fixed butterfly).
template <int LP>
SF_DEV float lane_sum(float x) {
#pragma unroll
    for (int o = 1; o < LP; o <<= 1) x += __shfl_xor(x, o);
    return x;
}

// Host-side launch dispatch over (batched?, workgroup size, list capacity);
// the choices are kNbChoices x kCapChoices.
template <int V>
using IC = std::integral_constant<int, V>;
template <class L>
void dispatch(const Fields& f, PassCfg c, L&& l) {
    auto with_cap = [&](auto B, auto NB) {
        if (c.cap == 8) l(B, NB, IC<8>{});
        else l(B, NB, IC<16>{});
    };
    auto with_nb = [&](auto B) {
        if (c.nb == 64) with_cap(B, IC<64>{});
        else if (c.nb == 128) with_cap(B, IC<128>{});
        else with_cap(B, IC<256>{});
    };
    if (f.scene) with_nb(std::true_type{});
    else with_nb(std::false_type{});
}

// ---------------------------------------------------------------------------
// Interface lists.  The avg-flow and voidage/adhesion passes (P2, P3) need
// each particle's neighbours of the other phase only.  Most particles have
// none in their 9 column ranges (the cell table gives each range's water and
// sand counts).  For those the empty sums' results are written directly
// (write_no_interface); the rest are listed, water and sand apart
// (list_interface), and P2 and P3 run over the lists.  In a step the density
// pass does both, since it already loads every water particle's 9 cell-table
// pairs; k_interface does the same for a lone avg-flow run.  The counters
// start at zero: the water momentum pass (after P2 and P3 have read them)
// clears them for the next step, and a lone density or avg-flow run clears
// them first (launch_zero_counts).  The list order the atomics leave does
// not matter: each listed particle's sums are its own lanes' work in
// candidate order.

// What P2 then P3 leave for particle i with empty sums; rpi = (rho, p).
// Later passes read the sand's voidage / saturation (drag, capillary bridges)
// and the water's records; the rest is output only and written here when the
// fields are read directly (full_empty) or taped (den4), else on request.
SF_DEV void write_empty_outputs(const Fields& f, int i, bool sand) {
    f.flow[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    f.adh[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (!sand) {
        f.es[i] = make_float2(1.f, 0.f);
        f.xf[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
}
// Water particle i's (rho~, p / rho~^2) from (rho, p) and its voidage eps:
// the neighbour records (Fields::rec0) with pi = (position, mass), t its phase
// index, and wt where taped.
SF_DEV void write_water_terms(const Fields& f, int i, uint32_t t, const float4& pi, float2 rpi, float eps) {
    const float rt = rpi.x / fmaxf(kEps, eps);
    const float pt = rpi.y / fmaxf(kEps, rt * rt);
    if (f.den4) f.wt[i] = make_float2(rt, pt);
    if (!f.fresh) f.recm[t] = pi.w;
    f.rec0[t] = make_float4(pi.x, pi.y, pi.z, rt);
    const float4 v = ldo(f.vr, (uint32_t)i);
    f.rec1[t] = make_float4(v.x, v.y, v.z, pt);
}
SF_DEV void write_no_interface(const Fields& f, int i, uint32_t t, bool sand, float2 rpi, const float4& pi) {
    if (sand) {
        f.es[i] = make_float2(0.f, 0.f);
    } else {
        write_water_terms(f, i, t, pi, rpi, 1.f);
    }
    if (f.full_empty || f.den4) write_empty_outputs(f, i, sand);
    if (f.den4) {
        reinterpret_cast<float*>(f.den4)[4 * i] = 0.f;
        reinterpret_cast<float*>(f.den4)[4 * i + 1] = 0.f;
    }
}
// Appends phase index t of every listed lane to its phase's list (water at
// ilist[0, nw), sand at ilist[nw, n)): one atomic per block and phase, each
// listed lane taking its rank among the block's.  Atomics on one word pass one
// after another, about 9 ns each: one per wave (23.4k for 500k + 500k
// interpenetrating particles, both counters on one cache line) held the
// density pass of that scene to 288 us, one per block on lines of their own
// leaves it at 76 us (step 1.26 -> 1.05 ms).  A list never grows past its phase's size (that would
// take a missed clear of the counters).  Must be called by all threads of the
// block; `sand` is the same for all lanes of a wave.
template <int NB>
SF_DEV void list_interface(const Fields& f, bool listed, bool sand, uint32_t t, uint32_t nw, uint32_t n) {
    constexpr int W = NB / 64;
    __shared__ uint32_t cnt[2][W], base[2];  // listed lanes of each wave, by phase; the block's first entries
    const int lane = (int)(threadIdx.x & 63u), w = (int)(threadIdx.x >> 6);
    const uint64_t m = __ballot(listed);
    if (lane < 2) cnt[lane][w] = (lane == 1) == sand ? (uint32_t)__popcll(m) : 0u;
    __syncthreads();
    if (threadIdx.x < 2) {
        uint32_t c = 0;
        for (int q = 0; q < W; ++q) c += cnt[threadIdx.x][q];
        base[threadIdx.x] = c ? atomicAdd(f.icount + threadIdx.x * kCountStride, c) : 0u;
    }
    __syncthreads();
    if (!listed) return;
    const int ph = sand ? 1 : 0;
    uint32_t q = base[ph] + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
    for (int v = 0; v < w; ++v) q += cnt[ph][v];
    if (q < (sand ? n - nw : nw)) f.ilist[(sand ? nw : 0u) + q] = t;
}

// ---------------------------------------------------------------------------
// P1: water density (self counted twice, :466 + loop) and pressure; sand gets
// rho_sand and p = 0.  Only water candidates are walked (sand adds nothing);
// branch-free: max(h^2 - r^2, 0) vanishes outside the support.  The kDenL
// lanes of a particle split both the candidates and the boundary particles.
// The boundary particles of the 27 cells around a cell for lane sub of L
// lanes per particle: fn(b) for j = s + sub + L m of each column's range
// [s, e), columns in for_columns order and j increasing (the order of a plain
// walk of the 9 columns; near = bnear[cell] counts those that hold any).
// Three columns' ranges, then the lane's first three candidates of each, are
// loaded together: a face cell's 3 columns take two round trips (P5 124 -> 117
// us at 1M against all nine columns' ranges and first candidates; P1 60 -> 57,
// one column's range ahead).
template <int L, class Fn>
SF_DEV void boundary_walk(const Fields& f, uint32_t near, uint32_t cell, uint32_t sub, Fn&& fn) {
    const uint32_t n = near >> 4;
    const uint2* __restrict__ ranges = f.brange + ldo(f.brow, cell);  // above 2^29 of them too
    for (uint32_t q = 0; q < n; q += 3u) {
        uint2 r[3];
        float4 b[3][3];
#pragma unroll
        for (uint32_t m = 0; m < 3u; ++m) {
            r[m] = q + m < n ? ldo(ranges, q + m) : make_uint2(0u, 0u);
            r[m].x += sub;
        }
#pragma unroll
        for (int m = 0; m < 3; ++m)
#pragma unroll
            for (uint32_t t = 0; t < 3u; ++t)
                b[m][t] = r[m].x + t * (uint32_t)L < r[m].y ? ldo(f.bpv, r[m].x + t * (uint32_t)L)
                                                            : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int m = 0; m < 3; ++m) {
#pragma unroll
            for (uint32_t t = 0; t < 3u; ++t)
                if (r[m].x + t * (uint32_t)L < r[m].y) fn(b[m][t]);
            for (uint32_t j = r[m].x + 3u * (uint32_t)L; j < r[m].y; j += (uint32_t)L) fn(ldo(f.bpv, j));
        }
    }
}

constexpr int kDenL = 2;  // lanes per water particle in the density pass
template <bool B, int NB>
__global__ __launch_bounds__(NB) void k_density(SFConst k, Fields f, int n) {
    __shared__ float4 stage_lds[(NB / 64) * kStage];
    float4* stage = stage_lds + (threadIdx.x >> 6) * kStage;
    constexpr uint32_t PB = NB / kDenL;  // water particles per block
    const uint32_t nw = water_count(f), ns = (uint32_t)n - nw;
    const PhaseBlock pb = phase_block((nw + PB - 1) / PB, (ns + NB - 1) / NB);
    if (pb.phase < 0) return;
    if (pb.phase == 1) {  // sand: rho_sand, p = 0; listed if a column range holds water
        const uint32_t t = pb.blk * NB + threadIdx.x;
        const bool valid = t < ns;
        int i = 0;
        uint32_t other = 0;
        if (valid) {
            i = (int)ldo(f.plist, nw + t);
            // every grain has rho_sand and p = 0; the passes use the constant,
            // so the field is written here only when it is read directly or
            // taped, else on request (launch_fill_empty)
            if (f.full_empty || f.den4) f.rp[i] = make_float2(k.rho_s, 0.f);
            const float4 p = ldo(f.pph, nw + t);
            if (!f.fresh) f.rec0[nw + t] = ldo(f.pm, (uint32_t)i);
            const uint32_t cb = scene_base<B>(k, f, i);
            int cx, cy, cz;
            cell_of(k, p.x, p.y, p.z, cx, cy, cz);
            for_columns(k, cx, cy, cz, [&](uint32_t c0, uint32_t c1) {
                other += ldo(f.ct, cb + c1).y - ldo(f.ct, cb + c0).y;
            });
        }
        const bool listed = valid && other != 0u;
        list_interface<NB>(f, listed, true, nw + t, nw, (uint32_t)n);
        if (valid) f.iface[t] = listed ? 1 : 0;
        if (valid) {  // every grain's velocity and saturation by phase index (P2 sets the listed ones' .w)
            const float4 v = ldo(f.vr, (uint32_t)i);
            f.vq[nw + t] = make_float4(v.x, v.y, v.z, 0.f);
        }
        if (valid && !listed) write_no_interface(f, i, nw + t, true, make_float2(k.rho_s, 0.f), make_float4(0.f, 0.f, 0.f, 0.f));
        return;
    }
    const uint32_t t = pb.blk * PB + threadIdx.x / kDenL;
    const bool lead = (threadIdx.x % kDenL) == 0;
    const bool water = t < nw;
    const int i = water ? (int)ldo(f.plist, t) : 0;
    const float4 pi = water ? own_pos(f, t, i) : make_float4(0.f, 0.f, 0.f, -1.f);
    const uint32_t cb = water ? scene_base<B>(k, f, i) : 0u;
    int cx, cy, cz;
    cell_of(k, pi.x, pi.y, pi.z, cx, cy, cz);
    float sf = 0.f, sb = 0.f;
    uint32_t other = 0;  // sand in the particle's 9 column ranges
    auto add = [&](uint32_t, const float4& pj) {
        const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
        // h^2 - r^2 as one fused chain (three FMAs, one rounding each)
        const float d = fmaxf(fmaf(-dz, dz, fmaf(-dy, dy, fmaf(-dx, dx, k.h2))), 0.f);
        sf += pj.w * sq3(d);
    };
    auto count = [&](uint2 a, uint2 b) { other += (b.x - a.x) - (b.y - a.y); };
    // A wave whose particles all sit in one grid column stages the water
    // candidates of its 9 columns once; a wave over several columns would
    // stage once per column it holds, one after another, so its lanes walk
    // their own ranges instead.  Both give each lane the same candidates in
    // the same order (staged_walk), hence the same sums.
    const uint64_t act = __ballot(water);
    const uint32_t col = cb + (uint32_t)((cx * k.gy + cy) * k.gz);
    const bool one = !__ballot(water && col != lane_value(col, act ? __builtin_ctzll(act) : 0));
    if (one) {
        staged_walk<kDenL, true>(
            k, f, stage, water, cb, cx, cy, cz, [](float4 p) { return p; }, [](uint32_t, uint32_t) { return true; },
            add, count);
    } else if (water) {
        const uint32_t sub = threadIdx.x % kDenL;
        for_columns(k, cx, cy, cz, [&](uint32_t c0, uint32_t c1) {
            const uint2 a = ldo(f.ct, cb + c0), b = ldo(f.ct, cb + c1);
            count(a, b);
            uint32_t j = a.y + sub;
            for (; j + 3u * kDenL < b.y; j += 4u * kDenL) {
                const float4 q0 = ldo(f.pph, j), q1 = ldo(f.pph, j + kDenL), q2 = ldo(f.pph, j + 2u * kDenL),
                             q3 = ldo(f.pph, j + 3u * kDenL);
                add(j, q0);
                add(j + kDenL, q1);
                add(j + 2u * kDenL, q2);
                add(j + 3u * kDenL, q3);
            }
            for (; j < b.y; j += kDenL) add(j, ldo(f.pph, j));
        });
    }
    const uint32_t cell = cell_key(k, cx, cy, cz);
    const uint32_t near = water ? ldo(f.bnear, cell) : 0u;
    if (near) {  // boundary particles within the 27 cells
        const uint32_t sub = threadIdx.x % kDenL;
        auto badd = [&](const float4& b) {
            const float dx = pi.x - b.x, dy = pi.y - b.y, dz = pi.z - b.z;
            const float d = fmaxf(k.h2 - (dx * dx + dy * dy + dz * dz), 0.f);
            sb += fabsf(b.w) * sq3(d);
        };
        // the columns that hold any, one after another (this pass keeps its
        // registers low), the next one's range and four candidates' loads in
        // flight at a time, summed in increasing j
        const uint32_t n = near >> 4;
        const uint2* __restrict__ ranges = f.brange + ldo(f.brow, cell);
        uint2 next = ldo(ranges, 0u);
        for (uint32_t q = 0; q < n; ++q) {
            const uint2 r = next;
            next = ldo(ranges, q + 1u < n ? q + 1u : q);
            uint32_t j = r.x + sub;
            for (; j + 3u * kDenL < r.y; j += 4u * kDenL) {
                const float4 b0 = ldo(f.bpv, j), b1 = ldo(f.bpv, j + kDenL), b2 = ldo(f.bpv, j + 2u * kDenL),
                             b3 = ldo(f.bpv, j + 3u * kDenL);
                badd(b0);
                badd(b1);
                badd(b2);
                badd(b3);
            }
            for (; j < r.y; j += kDenL) badd(ldo(f.bpv, j));
        }
    }
#pragma unroll
    for (int o = 1; o < kDenL; o <<= 1) {
        sf += __shfl_xor(sf, o);
        sb += __shfl_xor(sb, o);
    }
    const bool listed = water && lead && other != 0u;
    list_interface<NB>(f, listed, false, t, nw, (uint32_t)n);
    if (!water || !lead) return;
    f.wl[t] = listed ? 1 : 0;
    const float rho = pi.w * k.w0 + k.w_coef * (sf + k.rho0 * sb);
    const float2 rpi = make_float2(rho, eos(k, rho));
    f.rp[i] = rpi;
    if (!listed) {
        write_no_interface(f, i, t, false, rpi, pi);
    } else {
        const float4 v = ldo(f.vr, (uint32_t)i);
        f.vq[t] = make_float4(v.x, v.y, v.z, built_pos(f, t, pi).w * frcp(rho));
    }
}
void launch_density(const SFConst& k, const Fields& f, int n, PassCfg c, hipStream_t s) {
    if (n <= 0) return;
    dispatch(f, c, [&](auto B, auto NB, auto) {
        k_density<decltype(B)::value, decltype(NB)::value><<<phase_grid(n * kDenL, NB), (int)NB, 0, s>>>(k, f, n);
    });
}

// ---------------------------------------------------------------------------
// k_interface: the interface lists and the empty sums' results, as the
// density pass leaves them, for a lone avg-flow run.
__global__ void k_zero_counts(uint32_t* __restrict__ c) {
    if (threadIdx.x < 2) c[threadIdx.x * kCountStride] = 0u;
}
template <bool B>
__global__ __launch_bounds__(kBlock) void k_interface(SFConst k, Fields f, int n) {
    const uint32_t nw = water_count(f), ns = (uint32_t)n - nw;
    const PhaseBlock pb = phase_block((nw + kBlock - 1) / kBlock, (ns + kBlock - 1) / kBlock);
    if (pb.phase < 0) return;
    const bool sand_i = pb.phase == 1;
    const uint32_t u = pb.blk * kBlock + threadIdx.x;  // index within the phase
    const uint32_t t = (sand_i ? nw : 0u) + u;
    const bool valid = u < (sand_i ? ns : nw);
    int i = 0;
    uint32_t other = 0;
    float4 pi = make_float4(0.f, 0.f, 0.f, 0.f);
    if (valid) {
        i = (int)ldo(f.plist, t);
        pi = ldo(f.pph, t);
        if (!f.fresh && sand_i) f.rec0[t] = ldo(f.pm, (uint32_t)i);
        const uint32_t cb = scene_base<B>(k, f, i);
        int cx, cy, cz;
        cell_of(k, pi.x, pi.y, pi.z, cx, cy, cz);
        for_columns(k, cx, cy, cz, [&](uint32_t c0, uint32_t c1) {
            const uint2 a = ldo(f.ct, cb + c0), b = ldo(f.ct, cb + c1);
            const uint32_t w = b.y - a.y;
            other += sand_i ? w : (b.x - a.x) - w;
        });
    }
    const bool listed = valid && other != 0u;
    list_interface<kBlock>(f, listed, sand_i, t, nw, (uint32_t)n);
    if (valid && !sand_i) f.wl[u] = listed ? 1 : 0;
    if (valid && sand_i) f.iface[u] = listed ? 1 : 0;
    if (valid && !listed) write_no_interface(f, i, t, sand_i, ldo(f.rp, (uint32_t)i), pi);
}
__global__ __launch_bounds__(kBlock) void k_fill_empty(SFConst k, Fields f, int n) {
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= (uint32_t)n) return;
    const uint32_t nw = water_count(f);
    const bool sand = t >= nw;
    const int i = (int)ldo(f.plist, t);
    if (sand) f.rp[i] = make_float2(k.rho_s, 0.f);
    if (sand ? ldo(f.iface, t - nw) : ldo(f.wl, t)) return;
    write_empty_outputs(f, i, sand);
}
void launch_fill_empty(const SFConst& k, const Fields& f, int n, hipStream_t s) {
    if (n > 0) k_fill_empty<<<(n + kBlock - 1) / kBlock, kBlock, 0, s>>>(k, f, n);
}
void launch_zero_counts(const Fields& f, hipStream_t s) { k_zero_counts<<<1, 64, 0, s>>>(f.icount); }
void launch_interface(const SFConst& k, const Fields& f, int n, hipStream_t s) {
    if (f.scene) k_interface<true><<<phase_grid(n, kBlock), kBlock, 0, s>>>(k, f, n);
    else k_interface<false><<<phase_grid(n, kBlock), kBlock, 0, s>>>(k, f, n);
}

template <int NB, int LP>
struct PhaseSlot {
    int i;         // the particle's slot
    uint32_t t;    // its phase index (plist[t] = i)
    uint32_t q;    // its place in its phase's list
    uint32_t sub;  // its lane among LP
    bool sand;
};
// The listed particle of this thread (false: none; slot and phase index 0
// then, the phase still the block's).
template <int NB, int LP>
SF_DEV bool phase_slot(const Fields& f, uint32_t nw, uint32_t cw, uint32_t cs, PhaseBlock pb, PhaseSlot<NB, LP>& ps) {
    constexpr uint32_t PB = NB / LP;  // particles per block
    ps.i = 0;
    ps.t = 0;
    ps.q = 0;
    ps.sand = pb.phase == 1;
    const uint32_t q = pb.blk * PB + threadIdx.x / LP;
    ps.sub = threadIdx.x % LP;
    if (q >= (ps.sand ? cs : cw)) return false;
    ps.q = q;
    ps.t = ldo(f.ilist, (ps.sand ? nw : 0u) + q);
    ps.i = (int)ldo(f.plist, ps.t);
    return true;
}
// body(phase_block) for the blocks of listed particles this block takes.  How
// much is listed is known on the device only, and a block for every particle
// that could be listed launches mostly waves that find nothing to do where
// the interface is thin (250k of them at 4M: 2 x 31 us).  The grid stops at
// kListBlocks, a multiple of 8 so that a block stays on its XCD's share, and
// each block takes every kListBlocks-th block of the mapping.
constexpr int kListBlocks = 16384;
inline int list_grid(int n, int lanes, int nb) {
    const int all = phase_grid(n * lanes, nb);
    return all < kListBlocks ? all : kListBlocks;
}
template <int NB, int LP, class Body>
SF_DEV void for_listed(const Fields& f, Body&& body) {
    constexpr uint32_t PB = NB / LP;  // particles per block
    const uint32_t cw = f.icount[0], cs = f.icount[kCountStride];
    const uint32_t na = (cw + PB - 1) / PB, nb = (cs + PB - 1) / PB;
    uint32_t b = blockIdx.x;
    PhaseBlock pb = phase_block(na, nb, b);
    if (pb.phase < 0) return;  // before the loop: nothing it hoists is waited for
    do {
        body(cw, cs, pb);
        b += gridDim.x;
        pb = phase_block(na, nb, b);
    } while (pb.phase >= 0);  // past the share's end, so are all later ones
}

// Squared length and kernel weight of a pair within h, their roundings the
// same wherever they are inlined: near the edge h^2 - r^2 keeps few digits, and
// P3's quotients (its own sums over P2's) are only as good as the two agree.
SF_DEV float pair_r2(v3 d) { return fmaf(d.z, d.z, fmaf(d.x, d.x, d.y * d.y)); }
SF_DEV float edge_weight(const SFConst& k, const float4& pi, const float4& pj) {
    return k.w_coef * sq3(k.h2 - pair_r2(mk3(pi.x - pj.x, pi.y - pj.y, pi.z - pj.z)));
}

// ---------------------------------------------------------------------------
// Saved neighbours (Fields::nl).  P2, P3 and P4's water walk need the same
// pairs, a particle and the other phase's within h, of which a walk of the 27
// cells keeps one candidate in six: the walk's filter was most of each pass.
// P2 saves what it keeps (a coalesced 4-byte store per pair) and the others
// read that.  500k + 500k interpenetrating: P3 203 -> 143 us, P4 150 -> 132, P5
// (with its walk over the water alone) 221 -> 161, for 200 -> 235 in P2: step
// 916 -> 851.  An entry costs its store and loads (4 bytes a row, rows of a
// wave as long as its fullest lane); what is left is the pairs' gathers.
// First saved lane of the particle at place q of its phase's list.
SF_DEV uint32_t saved_lane(uint32_t lanes, bool sand, uint32_t nw, uint32_t q) {
    return (sand ? (nw * lanes + 63u) & ~63u : 0u) + q * lanes;
}
// Entry 0 of saved lane G, of `rows` entries 64 apart.
SF_DEV uint32_t* saved_row(const Fields& f, uint32_t G, uint32_t rows) {
    return f.nl + ((size_t)(G >> 6) * rows * 64u + (G & 63u));
}
// apply over the saved neighbours of the particle whose lanes start at G0,
// lane sub of S taking its share: whole lanes of the writer's where there are
// as many or more, every (S / lanes)-th entry of one where there are fewer.
// The indices go through the lane's LDS list, eight loads in flight.
template <uint32_t S, int NB, int CAP, class Fetch, class Apply>
SF_DEV void saved_pairs(const Fields& f, uint32_t lanes, uint32_t G0, uint32_t sub, NList<NB, CAP>& L, Fetch&& fetch,
                        Apply&& apply) {
    static_assert(CAP >= 8, "a round takes eight entries");
    const uint32_t step = S > lanes ? S / lanes : 1u, rows = (uint32_t)kSaved / lanes;
    for (uint32_t l = sub & (lanes - 1u); l < lanes; l += S) {
        const uint32_t G = G0 + l, cnt = ldo(f.nlc, G);
        const uint32_t* __restrict__ e = saved_row(f, G, rows);
        for (uint32_t r = S > lanes ? sub / lanes : 0u; r < cnt;) {
            L.cnt = 0;
            do {
                uint32_t v[8];
#pragma unroll
                for (uint32_t c = 0; c < 8u; ++c) v[c] = e[(r + c * step < cnt ? r + c * step : r) * 64u];
#pragma unroll
                for (uint32_t c = 0; c < 8u; ++c) {
                    L.slot[(L.cnt + (int)c) * NB] = v[c];
                }
                const uint32_t left = (cnt - r + step - 1u) / step;
                L.cnt += left < 8u ? (int)left : 8;
                r += 8u * step;
            } while (r < cnt && L.cnt + 8 <= CAP);
            nl_flush2(L, fetch, apply);
        }
    }
}

// ---------------------------------------------------------------------------
// P2 (ComputeSFAvgFlow_CUDA): water i -> voidage 1 - sum_sand V W and the
// average sand velocity; sand i -> average water velocity and saturation.
// (Sand voidage from this pass is overwritten by P3 before anything reads it,
// so a sand particle only needs its water neighbours, a water particle only
// its sand neighbours.)
// Water particles also store (rho / max(eps, voidage), p / max(eps, that^2)), the
// per-particle factors the water momentum pass needs from every neighbour.
// Candidates are filtered four at a time into the lane's list; the flush
// fetches each kept neighbour's fields (by phase index u: every neighbour
// within h is listed, see Fields::vq) ahead of its use.
template <bool B, int NB, int CAP, int LP>
SF_DEV void avg_flow(const SFConst& k, const Fields& f, NList<NB, CAP>& L, float4* __restrict__ stage, uint32_t nw,
                     uint32_t cw, uint32_t cs, PhaseBlock pb) {
    PhaseSlot<NB, LP> ps;
    const bool active = phase_slot(f, nw, cw, cs, pb, ps);
    if (!__ballot(active)) return;  // the other lanes of a wave help to stage its candidates
    const int i = ps.i;
    const uint32_t sub = ps.sub;
    const bool sand_i = ps.sand;
    const float4 pi = own_pos(f, ps.t, i);
    const uint32_t cb = scene_base<B>(k, f, i);
    int cx, cy, cz;
    cell_of(k, pi.x, pi.y, pi.z, cx, cy, cz);
    float vsum = 0.f;
    v3 av = mk3(0.f, 0.f, 0.f);
    const float inv_rho_s = k.rho_s != 0.f ? 1.f / k.rho_s : 0.f;
    auto in_range = [&](uint32_t, const float4& pj) {
        const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
        const float r2 = dx * dx + dy * dy + dz * dz;
        return r2 < k.h2;
    };
    struct Nbr {
        float4 pj, vj;
    };
    // neighbours within h are listed: their fields by phase index (a water
    // neighbour's volume beside its velocity: two 16-byte loads a pair)
    auto fetch = [&](uint32_t u) { return Nbr{ldo(f.pph, u), ldo(f.vq, u)}; };
    const uint32_t G = saved_lane(LP, sand_i, nw, ps.q) + sub;
    constexpr uint32_t rows = (uint32_t)kSaved / LP;
    uint32_t* __restrict__ saved = saved_row(f, G, rows);
    uint32_t kept = 0;
    auto pair = [&](uint32_t u, const Nbr& q) {
        if (kept < rows) saved[kept * 64u] = u;
        ++kept;
        const float4 pj = q.pj;
        const float w = edge_weight(k, pi, pj);
        const float vw = (sand_i ? q.vj.w : -pj.w * inv_rho_s) * w;
        av += xyz(q.vj) * vw;
        vsum += vw;
    };
    column_filter<LP, kStageList>(
        k, f.pph, stage, active, cb, cx, cy, cz, L,
        [&](uint32_t b, uint32_t c0, uint32_t c1) { return phase_range(f.ct + b, c0, c1, sand_i, nw); }, in_range, fetch, pair);
    nl_flush2(L, fetch, pair);
    if (!active) return;
    uint32_t most = kept;
#pragma unroll
    for (int o = 1; o < LP; o <<= 1) {
        const uint32_t other = __shfl_xor(most, o);
        most = most > other ? most : other;
    }
    f.nlc[G] = (uint8_t)(most > rows ? kSavedOver : kept);
    vsum = lane_sum<LP>(vsum);
    av = mk3(lane_sum<LP>(av.x), lane_sum<LP>(av.y), lane_sum<LP>(av.z));
    if (sub != 0) return;
    f.nlq[ps.t] = ps.q;
    const v3 fl = vsum != 0.f ? av * (1.f / vsum) : mk3(0.f, 0.f, 0.f);
    f.flow[i] = f4(fl, 0.f);
    if (f.den4) reinterpret_cast<float*>(f.den4)[4 * i] = vsum;
    const float eps_i = sand_i ? 1.f : 1.f - vsum;
    f.es[i] = make_float2(eps_i, sand_i ? vsum : 0.f);
    const float4 pj = built_pos(f, ps.t, pi);
    float x;  // what P3's neighbours need besides the position
    if (sand_i) {
        x = -pj.w * bezier(k.gadh, vsum);
        reinterpret_cast<float*>(f.vq)[4 * ps.t + 3] = vsum;  // saturation, for P4
    } else {
        const float2 rpi = ldo(f.rp, (uint32_t)i);
        write_water_terms(f, i, ps.t, pi, rpi, eps_i);
        x = pj.w * frcp(rpi.x) * eps_i;
        f.vws[ps.t] = vsum;
    }
    f.wq[ps.t] = make_float4(pj.x, pj.y, pj.z, x);
}
template <bool B, int NB, int CAP, int LP>
__global__ __launch_bounds__(NB) void k_avg_flow(SFConst k, Fields f, int n) {
    SF_NLIST(L);
    SF_STAGE(stage, kStageList);
    const uint32_t nw = water_count(f);
    for_listed<NB, LP>(f, [&](uint32_t cw, uint32_t cs, PhaseBlock pb) {
        avg_flow<B, NB, CAP, LP>(k, f, L, stage, nw, cw, cs, pb);
    });
}
void launch_avg_flow(const SFConst& k, const Fields& f, int n, PassCfg c, hipStream_t s) {
    if (n <= 0) return;
    dispatch(f, c, [&](auto B, auto NB, auto CAP) {
        with_lanes(c.lanes, [&](auto LP) {
            k_avg_flow<decltype(B)::value, decltype(NB)::value, decltype(CAP)::value, decltype(LP)::value>
                <<<list_grid(n, LP, NB), (int)NB, 0, s>>>(k, f, n);
        });
    });
}

// ---------------------------------------------------------------------------
// P3: sand i -> voidage from water neighbours; water i -> adhesion force.
// Over the neighbours P2 saved, each lane its own; the walk of P2 where they
// were too many.
// A pair is bound by its gathers, so P2 leaves one 16-byte record per neighbour
// (Fields::wq), with the adhesion curve taken once a grain and not once a pair,
// and the sums of weights that P2 has already made (P3 143 -> 122 us, and P2,
// which reads the volume instead of dividing, 235 -> 207 at 500k + 500k
// interpenetrating).
template <bool B, int NB, int CAP, int LP>
SF_DEV void voidage_adhesion(const SFConst& k, const Fields& f, NList<NB, CAP>& L, float4* __restrict__ stage,
                             uint32_t nw, uint32_t cw, uint32_t cs, PhaseBlock pb) {
    PhaseSlot<NB, LP> ps;
    const bool active = phase_slot(f, nw, cw, cs, pb, ps);
    if (!__ballot(active)) return;
    const int i = ps.i;
    const uint32_t sub = ps.sub;
    const float4 pi = own_pos(f, ps.t, i);
    const uint32_t cb = scene_base<B>(k, f, i);
    int cx, cy, cz;
    cell_of(k, pi.x, pi.y, pi.z, cx, cy, cz);
    auto in_range = [&](uint32_t, const float4& pj) {
        const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
        const float r2 = dx * dx + dy * dy + dz * dz;
        return r2 < k.h2;
    };
    const uint32_t G = saved_lane(LP, ps.sand, nw, ps.q);
    const bool over = active && ldo(f.nlc, G + sub) == kSavedOver;  // of all the particle's lanes
    const bool read = active && !over;
    // neighbours within h are listed: P2 left all that a pair needs of them
    auto fetch = [&](uint32_t u) { return ldo(f.wq, u); };
    if (ps.sand) {
        float num = 0.f;
        auto pair = [&](uint32_t, const float4& pj) {
            num += pj.w * edge_weight(k, pi, pj);
        };
        if (read) saved_pairs<LP>(f, LP, G, sub, L, fetch, pair);
        column_filter<LP, kStageList>(
            k, f.pph, stage, over, cb, cx, cy, cz, L,
            [&](uint32_t b, uint32_t c0, uint32_t c1) { return phase_range(f.ct + b, c0, c1, true, nw); }, in_range, fetch, pair);
        nl_flush2(L, fetch, pair);
        if (!active) return;
        num = lane_sum<LP>(num);
        if (sub != 0) return;
        const float den = ldo(f.vq, ps.t).w;  // the sum of the weights: the saturation
        f.es[i].x = den != 0.f ? num / den : 0.f;
        f.adh[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (f.den4) reinterpret_cast<float*>(f.den4)[4 * i + 1] = den;
        return;
    }
    const float mi = pi.w;
    v3 F = mk3(0.f, 0.f, 0.f);
    auto pair = [&](uint32_t, const float4& pj) {
        const v3 dp = mk3(pi.x - pj.x, pi.y - pj.y, pi.z - pj.z);
        const float l = fsqrt(pair_r2(dp));
        const float A = adhesion_A(k, l);
        if (A != 0.f) F += dp * (pj.w * mi * A * frcp(fmaxf(kEps, l)));
    };
    if (read) saved_pairs<LP>(f, LP, G, sub, L, fetch, pair);
    column_filter<LP, kStageList>(
        k, f.pph, stage, over, cb, cx, cy, cz, L,
        [&](uint32_t b, uint32_t c0, uint32_t c1) { return phase_range(f.ct + b, c0, c1, false, nw); }, in_range, fetch, pair);
    nl_flush2(L, fetch, pair);
    if (!active) return;
    F = mk3(lane_sum<LP>(F.x), lane_sum<LP>(F.y), lane_sum<LP>(F.z));
    if (sub != 0) return;
    f.adh[i] = f4(F, 0.f);
    const float vs = ldo((const float*)f.vws, ps.t);  // P2's sum of the grains' V W
    const float4 avg = vs != 0.f ? f4(F * (1.f / vs), 0.f) : make_float4(0.f, 0.f, 0.f, 0.f);
    f.xf[i] = avg;
    // what a grain's buoyancy sums need of this particle (sand momentum
    // pass): m / rho~ and m p / max(eps, rho_sand rho~), both zero unless the
    // voidage lies in (0, 1]
    const float2 rpi = ldo(f.rp, (uint32_t)i);
    const float eps = f.es[i].x;
    float a = 0.f, g = 0.f;
    if (eps > 0.f && eps <= 1.f) {
        const float dj = rpi.x * frcp(fmaxf(kEps, eps));
        a = mi * frcp(dj);
        g = mi * rpi.y * frcp(fmaxf(kEps, k.rho_s * dj));
    }
    f.xq[ps.t] = make_float4(avg.x, avg.y, avg.z, g);
    f.wbq[ps.t] = make_float4(pi.x, pi.y, pi.z, a);
    if (f.den4) reinterpret_cast<float*>(f.den4)[4 * i + 1] = vs;
}
template <bool B, int NB, int CAP, int LP>
__global__ __launch_bounds__(NB) void k_voidage_adhesion(SFConst k, Fields f, int n) {
    SF_NLIST(L);
    SF_STAGE(stage, kStageList);
    const uint32_t nw = water_count(f);
    for_listed<NB, LP>(f, [&](uint32_t cw, uint32_t cs, PhaseBlock pb) {
        voidage_adhesion<B, NB, CAP, LP>(k, f, L, stage, nw, cw, cs, pb);
    });
}
void launch_voidage_adhesion(const SFConst& k, const Fields& f, int n, PassCfg c, hipStream_t s) {
    if (n <= 0) return;
    dispatch(f, c, [&](auto B, auto NB, auto CAP) {
        with_lanes(c.lanes, [&](auto LP) {
            k_voidage_adhesion<decltype(B)::value, decltype(NB)::value, decltype(CAP)::value, decltype(LP)::value>
                <<<list_grid(n, LP, NB), (int)NB, 0, s>>>(k, f, n);
        });
    });
}

// ---------------------------------------------------------------------------
// P4: sand linear momentum (DEM + capillary + buoyancy + adhesion + boundary
// DEM + walls + drag), acc = g + 2 (f + df) / m, then the wet-sand colour.
//
// Sand-sand forces vanish beyond r_c = 2R + s_rupture (DEM needs overlap,
// the bridge H < s_rupture), and r_c < h / 2, so along each axis a grain only
// reaches its own cell and the one neighbour on its nearer side: the contact
// search walks 2 x 2 x 2 cells instead of 27 (same non-zero terms).

constexpr int kSmL = 2;  // lanes per sand particle (as in the water momentum pass)
template <bool B, int NB, int CAP>
__global__ __launch_bounds__(NB) void k_sand_momentum(SFConst k, Fields f, int n) {
    SF_NLIST(L);
    SF_STAGE(stage, kStageList);
    constexpr uint32_t PB = NB / kSmL;  // sand particles per block
    const uint32_t nw = water_count(f), ns = (uint32_t)n - nw;
    const PhaseBlock pb = phase_block(0u, (ns + PB - 1) / PB);
    const uint32_t t = pb.blk * PB + threadIdx.x / kSmL;
    const uint32_t sub = threadIdx.x % kSmL;  // this lane's share of the particle's candidates
    if (pb.phase < 0) return;  // the whole block
    // lanes past the last grain help to stage their wave's water candidates
    const int i = t < ns ? (int)ldo(f.plist, nw + t) : 0;
    const uint32_t self = t < ns ? nw + t : 0u;  // this particle's phase index
    const float4 pi = own_pos(f, self, i);
    const bool active = t < ns && pi.w < 0.f;
    if (!__ballot(active)) return;
    const uint32_t cb = scene_base<B>(k, f, i);
    if constexpr (B) {  // the scene's friction, capillary curve and drag coefficient
        const SceneConst sc = f.sct[ldo(f.scene, (uint32_t)i)];
        k.tan2 = sc.tan2;
        k.tanphi = sc.tanphi;
        k.cd = sc.cd;
        k.gcap = sc.gcap;
    }
    const float mi = -pi.w;
    const v3 xi = xyz(pi);
    const float4 vsi = ldo(f.vq, self);  // velocity, saturation
    const v3 vi = xyz(vsi);
    const float rho_i = k.rho_s;  // the density pass's value for every grain
    const float2 esi = ldo(f.es, (uint32_t)i);
    const float sat_i = vsi.w;
    const float twoR = 2.f * k.R;
    const float cap_r = twoR + k.cap_srup;
    const float cap_r2 = cap_r * cap_r;
    const float vol_i = mi / fmaxf(kEps, rho_i);
    int cx, cy, cz;
    cell_of(k, pi.x, pi.y, pi.z, cx, cy, cz);
    v3 fsum = mk3(0.f, 0.f, 0.f);
    float vw = 0.f;

    // sand-sand: DEM contact or liquid bridge
    struct SandNbr {
        float4 pj, vj;  // vj.w: saturation
    };
    // candidates are phase indices u (pph[u] = pm[plist[u]], vq[u] = the
    // velocity and saturation of slot plist[u])
    auto fetch_sand = [&](uint32_t u) { return SandNbr{ldo(f.pph, u), ldo(f.vq, u)}; };
    auto contact = [&](uint32_t, const SandNbr& q) {
        const float4 pj = q.pj;
        const v3 dji = mk3(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z);
        const float dist = fsqrt(dot(dji, dji));
        if (dist < twoR) {
            fsum += dem_contact(dji, dist, xyz(q.vj) - vi, twoR, k.kn, k.ks, k.tan2);
        } else {
            const float H = dist - twoR;
            if (H > 0.f && H < k.cap_srup) fsum += capillary(k, dji, dist, H, (sat_i + q.vj.w) * 0.5f);
        }
    };
    if (active) {
        const float rcm = cap_r + 1e-3f * k.h;  // conservative against FP32 cell edges
        int xa, xb, ya, yb, za, zb;
        near_span(pi.x, k.lox, k.h, cx, k.gx, rcm, xa, xb);
        near_span(pi.y, k.loy, k.h, cy, k.gy, rcm, ya, yb);
        near_span(pi.z, k.loz, k.h, cz, k.gz, rcm, za, zb);
        for (int x = xa; x <= xb; ++x)
            for (int y = ya; y <= yb; ++y) {
                const uint32_t base = cb + (uint32_t)((x * k.gy + y) * k.gz);
                const uint2 a = ldo(f.ct, base + (uint32_t)za), b = ldo(f.ct, base + (uint32_t)zb + 1u);
                // the sand candidates of the range, as phase indices
                filter_push<kSmL>(L, f.pph, nw + (a.x - a.y) + sub, nw + (b.x - b.y), [&](uint32_t u, const float4& pj) {
                    const float dx = pj.x - pi.x, dy = pj.y - pi.y, dz = pj.z - pi.z;
                    const float r2 = dx * dx + dy * dy + dz * dz;
                    return u != self && r2 < cap_r2;
                }, fetch_sand, contact);
            }
        nl_flush2(L, fetch_sand, contact);
    }
    // water neighbours: buoyancy (ComputeSFSandBuoyancyForces) + adhesion
    // (ComputeSFSandAdhesionTerm)
    struct WaterNbr {
        float4 pa;  // position, m_j / rho~_j
        float4 xg;  // avgAdhesion, m_j p_j / max(eps, rho_sand rho~_j)
    };
    // a water neighbour within h has this grain in its columns, so it is
    // listed and the voidage/adhesion pass wrote its record at its phase
    // index u (the two factors zero where rho~_j is undefined: voidage
    // outside (0, 1])
    auto fetch_water = [&](uint32_t u) { return WaterNbr{ldo(f.wbq, u), ldo(f.xq, u)}; };
    auto water = [&](uint32_t, const WaterNbr& q) {
        const float4 pj = q.pa;
        const v3 dji = mk3(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z);
        const float r2 = dot(dji, dji);
        const float w = k.w_coef * sq3(k.h2 - r2);
        vw += pj.w * w;
        const float gs = spiky_s(k, fsqrt(r2));
        // gradW(x_i - x_j) = gs * (x_i - x_j) = -gs * dji
        fsum += dji * (mi * q.xg.w * gs);
        fsum += xyz(q.xg) * (w * vol_i);
    };
    // a grain with no water in its 9 column ranges (the density pass flagged
    // the others) has nothing to walk
    const bool wet = active && ldo(f.iface, t);
    bool over = false;
    if (wet) {  // P2 saved its neighbours
        const uint32_t G = saved_lane((uint32_t)f.nl_lanes, true, nw, ldo(f.nlq, self));
        over = ldo(f.nlc, G) == kSavedOver;
        if (!over) saved_pairs<kSmL>(f, (uint32_t)f.nl_lanes, G, sub, L, fetch_water, water);
    }
    column_filter<kSmL, kStageList>(
        k, f.pph, stage, over, cb, cx, cy, cz, L,
        [&](uint32_t b, uint32_t c0, uint32_t c1) { return phase_range(f.ct + b, c0, c1, true, nw); },
        [&](uint32_t, const float4& pj) {
            const float dx = pj.x - pi.x, dy = pj.y - pi.y, dz = pj.z - pi.z;
            const float r2 = dx * dx + dy * dy + dz * dz;
            return r2 < k.h2;
        },
        fetch_water, water);
    nl_flush2(L, fetch_water, water);
    if (!active) return;
    if (k.blabel1) {  // ComputeSFUniRadiusDemBoundaryForces: label 1 only
        const uint32_t cell = cell_key(k, cx, cy, cz), near = ldo(f.bnear, cell);
        if (near & 2u)
            boundary_walk<kSmL>(f, near, cell, sub, [&](const float4& b) {
                if (b.w < 0.f) fsum += dem_force(xi - xyz(b), -vi, twoR, k.kn, k.ks, k.tan2);
            });
    }
#pragma unroll
    for (int o = 1; o < kSmL; o <<= 1) {
        fsum.x += __shfl_xor(fsum.x, o);
        fsum.y += __shfl_xor(fsum.y, o);
        fsum.z += __shfl_xor(fsum.z, o);
        vw += __shfl_xor(vw, o);
    }
    if (sub != 0) return;
    fsum += world_walls(k, xi, vi);
    v3 df = mk3(0.f, 0.f, 0.f);
    const float eps_i = esi.x;
    if (eps_i < 1.f && eps_i > 0.f) {
        const float cd = k.multi ? ldo(f.cda, (uint32_t)i).x : k.cd;
        const float ome = 1.f - eps_i;
        const float dc = cd * (eps_i * eps_i * eps_i) / (ome * ome);
        if (dc != 0.f) {
            const v3 fl = xyz(ldo(f.flow, (uint32_t)i));
            df = (fl - vi) * (k.grav_abs * k.rho0 * (eps_i * eps_i) / dc * mi / rho_i);
        }
    }
    const float4 drag = vw != 0.f ? f4(df * (1.f / vw), 0.f) : make_float4(0.f, 0.f, 0.f, 0.f);
    f.xf[i] = drag;
    f.rec1[self] = drag;
    if (f.den4) reinterpret_cast<float*>(f.den4)[4 * i + 2] = vw;
    const v3 a = mk3(k.gvx, k.gvy, k.gvz) + (fsum + df) * (2.f / mi);
    f.acc[i] = f4(a, 0.f);
    // ComputeSFWetSandColor_CUDA (:952-977)
    float4 c = ldo((const float4*)f.cs, (uint32_t)i);
    if (c.w < sat_i) {
        c.x = k.dryr + (k.wetr - k.dryr) * sat_i;
        c.y = k.dryg + (k.wetg - k.dryg) * sat_i;
        c.z = k.dryb + (k.wetb - k.dryb) * sat_i;
        c.w = sat_i;
        f.cs[i] = c;
    }
}
// one wave per workgroup: no wave's LDS and slot wait for the slowest of four
// (15.1 -> 13.6 us at 24k, 71 -> 69 at 1M apart, 158 -> 150 interpenetrating,
// 255 -> 255 at 4M)
int sand_momentum_nb(int) { return 64; }
void launch_sand_momentum(const SFConst& k, const Fields& f, int n, PassCfg c, hipStream_t s) {
    if (n <= 0) return;
    if (!c.chosen) c.nb = sand_momentum_nb(n);
    dispatch(f, c, [&](auto B, auto NB, auto CAP) {
        k_sand_momentum<decltype(B)::value, decltype(NB)::value, decltype(CAP)::value>
            <<<phase_grid(n * kSmL, NB), (int)NB, 0, s>>>(k, f, n);
    });
}

// ---------------------------------------------------------------------------
// P5: water linear momentum (pressure + artificial viscosity + seepage +
// boundary pressure/viscosity), acc = g + a - F_adh / m.  kWmL adjacent lanes
// share a particle: each filters every kWmL-th candidate of the ranges into
// its own list (column_filter, which stages the candidates in LDS where the
// wave's ranges overlap), and the partial sums are combined with shuffles.
constexpr int kWmL = 4;
// A neighbour's data in the water momentum pass, by phase index u:
// r0 = (position, w) with w > 0 for water, w = -mass for a grain (load_sand).
// WmRecords reads the two records (Fields::rec0; every water particle has mass
// f.mw), WmMasses the mass besides; both walk the water alone and take the
// grains that P2 saved, so an interpenetrating cell's grains are not filtered
// again (P5 221 -> 161 us at 500k + 500k interpenetrating, 4M dam 323 -> 300).
// WmMoved is for positions a caller may have written since the build (two
// calls, a handed-out buffer): the records hold everything as it is now, and
// both phases are walked, what P2 saved having been kept by the build's
// positions; the grains only where P1 counted any in the 27 cells (1M apart
// 128 us, 170 with every particle walking both phases and one body for either
// kind, 133 with one walk over both by slot).  All
// three give a particle the same terms, water before grains; the same bits
// where as many lanes saved the grains as share the particle (four).
struct WmRecords {
    static constexpr bool fresh = true;
    float4 r0, r1;
    SF_DEV static WmRecords load(const Fields& f, uint32_t u) { return {ldo(f.rec0, u), ldo(f.rec1, u)}; }
    SF_DEV static WmRecords load_sand(const Fields& f, uint32_t u) { return {ldo(f.pph, u), ldo(f.rec1, u)}; }
    SF_DEV float water_mass(const Fields& f) const { return f.mw; }
    SF_DEV float2 wt() const { return make_float2(r0.w, r1.w); }
    SF_DEV v3 vel() const { return xyz(r1); }
    SF_DEV v3 drag() const { return xyz(r1); }
    SF_DEV bool is_water() const { return r0.w >= 0.f; }
};
struct WmMasses : WmRecords {
    float m;
    SF_DEV static WmMasses load(const Fields& f, uint32_t u) {
        return {WmRecords::load(f, u), ldo(reinterpret_cast<const float*>(f.pph), 4u * u + 3u)};
    }
    SF_DEV static WmMasses load_sand(const Fields& f, uint32_t u) { return {WmRecords::load_sand(f, u), 0.f}; }
    SF_DEV float water_mass(const Fields&) const { return m; }
};
struct WmMoved : WmRecords {
    static constexpr bool fresh = false;
    float m;
    SF_DEV static WmMoved load(const Fields& f, uint32_t u) { return {WmRecords::load(f, u), ldo((const float*)f.recm, u)}; }
    SF_DEV static WmMoved load_sand(const Fields& f, uint32_t u) { return {WmRecords::load(f, u), 0.f}; }
    SF_DEV float water_mass(const Fields&) const { return m; }
    SF_DEV bool is_water() const { return m >= 0.f; }
};
template <bool B, class Nbr, int NB, int CAP>
__global__ __launch_bounds__(NB) void k_water_momentum(SFConst k, Fields f, int n) {
    SF_NLIST(L);
    SF_STAGE(stage, kStageWm);
    // P2 and P3 have read the interface lists: the next density pass lists
    // into counters that start at zero
    if (blockIdx.x == 0 && threadIdx.x < 2) f.icount[threadIdx.x * kCountStride] = 0u;
    constexpr uint32_t PB = NB / kWmL;  // water particles per block
    const uint32_t nw = water_count(f);
    const PhaseBlock pb = phase_block((nw + PB - 1) / PB, 0u);
    if (pb.phase < 0) return;  // the whole block
    const uint32_t t = pb.blk * PB + threadIdx.x / kWmL;
    const uint32_t sub = threadIdx.x % kWmL;  // this lane's share of the particle's candidates
    // lanes past the last particle take part in the staged walk without a range
    const int i = t < nw ? (int)ldo(f.plist, t) : 0;
    const Nbr self = Nbr::load(f, t < nw ? t : 0u);
    const float4 pi = self.r0;
    const bool active = t < nw && self.is_water();
    const uint32_t cb = scene_base<B>(k, f, i);
    const float mi = self.water_mass(f);
    const v3 vi = self.vel();
    const float2 wti = self.wt();  // (rho~_i, p_i / rho~_i^2)
    const float p_i = ldo(f.rp, (uint32_t)i).y;
    const float rt_i = wti.x;
    const float inv_rt_i = frcp(rt_i);
    const float bpress = -k.rho0 * (p_i / fmaxf(kEps, k.rho0 * k.rho0));
    const float bvisc = -k.bnu / (2.f * k.rho0);
    int cx, cy, cz;
    cell_of(k, pi.x, pi.y, pi.z, cx, cy, cz);
    v3 a = mk3(0.f, 0.f, 0.f);
    auto fetch = [&](uint32_t u) { return Nbr::load(f, u); };
    auto fetch_sand = [&](uint32_t u) { return Nbr::load_sand(f, u); };
    // the products in one order of roundings wherever the body is inlined
    auto dot_yxz = [](v3 u, v3 w) { return fmaf(u.z, w.z, fmaf(u.x, w.x, u.y * w.y)); };
    auto spiky = [&](float r2, float rs) {  // spiky gradient / r
        const float r = r2 * rs;
        const float hr = k.h - r;
        return r >= kEps ? k.g_coef * hr * hr * rs : 0.f;
    };
    // water j: ComputeSFWaterPressureTerm + ArtificialViscosity
    auto water = [&](uint32_t, const Nbr& q) {
        const float4 pj = q.r0;
        const v3 d = mk3(pi.x - pj.x, pi.y - pj.y, pi.z - pj.z);
        const float r2 = dot_yxz(d, d);
        const float gs = spiky(r2, frsq(r2));
        const float2 wtj = q.wt();
        const float mj = q.water_mass(f);
        float s = -mj * (wti.y + wtj.y);
        const v3 dv = vi - q.vel();
        const float dd = dot_yxz(dv, d);
        const float pij = -k.nu * frcp(rt_i + wtj.x) * (dd * frcp(r2 + kEps));
        s += dd < 0.f ? -mj * pij : 0.f;
        a += d * (s * gs);
    };
    // sand j: ComputeSFWaterSeepageTerm
    auto sand = [&](uint32_t, const Nbr& q) {
        const float4 pj = q.r0;
        const v3 d = mk3(pi.x - pj.x, pi.y - pj.y, pi.z - pj.z);
        const float r2 = dot_yxz(d, d);
        const float gs = spiky(r2, frsq(r2));
        const float mj = -pj.w;
        const float rho_j = k.rho_s;  // the density pass gives every grain rho_sand
        const float w = k.w_coef * sq3(k.h2 - r2);
        a += d * (-mj * p_i * frcp(fmaxf(kEps, rt_i * rho_j)) * gs);
        a += q.drag() * (-w * inv_rt_i);
    };
    // the particle's own slot passes too: d = 0 makes its term exactly zero
    // (the spiky factor is 0 below r = eps), and acc adds g afterwards
    auto in_range = [&](uint32_t, const float4& pj) {
        const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
        const float r2 = dx * dx + dy * dy + dz * dz;
        return r2 < k.h2;
    };
    auto water_range = [&](uint32_t b, uint32_t c0, uint32_t c1) { return phase_range(f.ct + b, c0, c1, true, nw); };
    auto sand_range = [&](uint32_t b, uint32_t c0, uint32_t c1) { return phase_range(f.ct + b, c0, c1, false, nw); };
    if constexpr (Nbr::fresh) {
        column_filter<kWmL, kStageWm>(k, f.rec0, stage, active, cb, cx, cy, cz, L, water_range, in_range, fetch, water);
        nl_flush2(L, fetch, water);
        bool over = false;
        if (active && ldo(f.wl, t)) {  // listed: grains in its 27 cells
            const uint32_t G = saved_lane((uint32_t)f.nl_lanes, false, nw, ldo(f.nlq, t));
            over = ldo(f.nlc, G) == kSavedOver;
            if (!over) saved_pairs<kWmL>(f, (uint32_t)f.nl_lanes, G, sub, L, fetch_sand, sand);
        }
        column_filter<kWmL, kStageWm>(k, f.pph, stage, over, cb, cx, cy, cz, L, sand_range, in_range, fetch_sand, sand);
        nl_flush2(L, fetch_sand, sand);
    } else {
        // the caller may have changed labels too: a neighbour counts as what it is now
        auto was_water = [&](uint32_t u, Nbr q) {
            if (q.is_water()) {
                water(u, q);
            } else {
                q.r0.w = q.m;
                q.r1 = ldo((const float4*)f.xf, ldo(f.plist, u));
                sand(u, q);
            }
        };
        auto was_sand = [&](uint32_t u, Nbr q) {
            if (q.r0.w <= 0.f) {
                sand(u, q);
            } else {  // no pass gave it a density
                q.m = q.r0.w;
                q.r0.w = 0.f;
                q.r1 = ldo(f.vr, ldo(f.plist, u));
                q.r1.w = 0.f;
                water(u, q);
            }
        };
        column_filter<kWmL, kStageWm>(k, f.rec0, stage, active, cb, cx, cy, cz, L, water_range, in_range, fetch, was_water);
        nl_flush2(L, fetch, was_water);
        const bool listed = active && ldo(f.wl, t);
        column_filter<kWmL, kStageWm>(k, f.rec0, stage, listed, cb, cx, cy, cz, L, sand_range, in_range, fetch_sand,
                                      was_sand);
        nl_flush2(L, fetch_sand, was_sand);
    }
    if (!active) return;
    const uint32_t cell = cell_key(k, cx, cy, cz);
    if (const uint32_t near = ldo(f.bnear, cell)) {  // boundary particles within the 27 cells
        boundary_walk<kWmL>(f, near, cell, sub, [&](const float4& b) {
            const v3 d = mk3(pi.x - b.x, pi.y - b.y, pi.z - b.z);
            const float r2 = dot(d, d);
            if (r2 >= k.h2) return;
            const float rs = frsq(r2);
            const float r = r2 * rs;
            const float hr = k.h - r;
            const float gs = r >= kEps ? k.g_coef * hr * hr * rs : 0.f;
            const float vb = fabsf(b.w);
            float s = vb * bpress;  // ComputeBoundaryPressure (densityi = rho0, :944)
            const float dd = dot(vi, d);
            if (dd < 0.f) s += -vb * k.rho0 * (bvisc * (dd * frcp(r2 + kEps)));  // ComputeBoundaryViscosity
            a += d * (s * gs);
        });
    }
#pragma unroll
    for (int o = 1; o < kWmL; o <<= 1) {
        a.x += __shfl_xor(a.x, o);
        a.y += __shfl_xor(a.y, o);
        a.z += __shfl_xor(a.z, o);
    }
    if (sub != 0) return;
    // adhesion: P3 wrote it for the listed water; the rest has none
    const v3 ad = ldo(f.wl, t) ? xyz(ldo(f.adh, (uint32_t)i)) : mk3(0.f, 0.f, 0.f);
    const v3 acc = mk3(k.gvx, k.gvy, k.gvz) + a - ad * (1.f / mi);
    f.acc[i] = f4(acc, 0.f);
}
// one wave per workgroup, as in the sand momentum pass, up to kWmOneWave
// particles (24.7 -> 20.4 us at 24k, 134.5 -> 128 at 1M, 169 -> 168 at
// 2M); above, neighbouring waves on one CU share more of its L1 than they
// wait for each other (4M: 335 us with 256 threads, 354 with 64)
int water_momentum_nb(int n) {
    constexpr int kWmOneWave = 2 << 20;
    return n <= kWmOneWave ? 64 : 256;
}
void launch_water_momentum(const SFConst& k, const Fields& f, int n, PassCfg c, hipStream_t s) {
    if (n <= 0) return;
    if (!c.chosen) c.nb = water_momentum_nb(n);
    dispatch(f, c, [&](auto B, auto NB, auto CAP) {
        constexpr bool b = decltype(B)::value;
        constexpr int nb = decltype(NB)::value, cap = decltype(CAP)::value;
        if (f.rec) k_water_momentum<b, WmRecords, nb, cap><<<phase_grid(n * kWmL, NB), nb, 0, s>>>(k, f, n);
        else if (f.fresh) k_water_momentum<b, WmMasses, nb, cap><<<phase_grid(n * kWmL, NB), nb, 0, s>>>(k, f, n);
        else k_water_momentum<b, WmMoved, nb, cap><<<phase_grid(n * kWmL, NB), nb, 0, s>>>(k, f, n);
    });
}

// ---------------------------------------------------------------------------
// CFL sub-step count (ComputeSubTimeStepsByCFL, cuda_wcsph_sf_solver.cu:35-58),
// computed on the device so the step needs no host round trip.
constexpr int kCflBlocks = 1024;
int cfl_partials(int) { return kCflBlocks; }

__global__ __launch_bounds__(kBlock) void k_cfl_partial(const float4* __restrict__ acc, int n, float* __restrict__ part) {
#pragma clang fp contract(off)
    __shared__ float sm[kBlock / 64];
    float m = 0.f;
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        const float4 a = acc[i];
        const float xx = a.x * a.x, yy = a.y * a.y, zz = a.z * a.z;
        m = fmaxf(m, (xx + yy) + zz);
    }
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_down(m, o, 64));
    if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        float r = sm[0];
        for (int q = 1; q < kBlock / 64; ++q) r = fmaxf(r, sm[q]);
        part[blockIdx.x] = r;
    }
}
__global__ __launch_bounds__(kBlock) void k_cfl_final(const float* __restrict__ part, int np, CflOut* out, float h,
                                                      float render_interval, float m, float c, float scale,
                                                      float params_dt, FrameDev* frame) {
#pragma clang fp contract(off)
    __shared__ float sm[kBlock / 64];
    float r = 0.f;
    for (int q = threadIdx.x; q < np; q += kBlock) r = fmaxf(r, part[q]);
    for (int o = 32; o > 0; o >>= 1) r = fmaxf(r, __shfl_down(r, o, 64));
    if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = r;
    __syncthreads();
    if (threadIdx.x == 0) {
        float mr = sm[0];
        for (int q = 1; q < kBlock / 64; ++q) mr = fmaxf(mr, sm[q]);
        const float amax = sqrtf(mr);
        const float fmax_ = amax * m;
        const float dts = 0.4f * h / c;
        const float dtf = 0.25f * sqrtf(h * m / fmax_);
        const float inner = dtf < dts ? dtf : dts;
        const float lim = scale * inner;
        const float dt = params_dt < lim ? params_dt : lim;
        FrameDev fr;
        if (frame) fr = *frame;
        const float ri = (frame && (fr.flags & kFrameAdaptive)) ? fr.remaining : render_interval;
        const float q = ri / dt;
        uint32_t k = q >= 4294967295.f ? 0xffffffffu : (q >= 1.f ? (uint32_t)q : 1u);
        CflOut o;
        o.dt = dt;
        o.nsub = k;
        o.amax = amax;
        o.ri = ri;
        *out = o;
        if (frame) {
            // the host loop's updates, in its float arithmetic (main.cpp:246,
            // cuda_sf_system.cu:95)
            const float step = ri / (float)k;
            if (fr.flags & kFrameElapsed) fr.elapsed = fr.elapsed + step;
            if (fr.flags & kFrameAdaptive) fr.remaining = ri - step;
            fr.count += 1;
            *frame = fr;
        }
    }
}
void launch_cfl(const SFConst& k, const float4* acc, int n, float* partials, CflOut* out, float render_interval,
                float sph_mass, float speed_of_sound, float scale, float params_dt, FrameDev* frame, hipStream_t s) {
    int nb = (n + kBlock - 1) / kBlock;
    if (nb > kCflBlocks) nb = kCflBlocks;
    if (nb < 1) nb = 1;
    k_cfl_partial<<<nb, kBlock, 0, s>>>(acc, n, partials);
    k_cfl_final<<<1, kBlock, 0, s>>>(partials, nb, out, k.h, render_interval, sph_mass, speed_of_sound, scale,
                                      params_dt, frame);
}

// ---------------------------------------------------------------------------
// advect: sand damping (AccDampingForSand), symplectic Euler, then the water
// box clamp and label-1 boundary push (SFWaterBoundaryConstrain_CUDA).
SF_DEV float sgnf(float v) { return (float)((0.f < v) - (v < 0.f)); }
__global__ __launch_bounds__(kBlock) void k_advect(SFConst k, AdvectArgs a, int n) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    uint32_t key = 0, old = 0;
    bool is_water = false;
    if (i < n) {
        const float dt = a.dt_dev ? a.dt_dev->ri / (float)a.dt_dev->nsub : a.dt;
        const float4 p = a.pm_in[i];
        const float4 v = a.vr_in[i];
        float4 ac = a.acc[i];
        if (p.w < 0.f) {
            const float qx = ac.x * (v.x + 0.5f * dt * ac.x);
            const float qy = ac.y * (v.y + 0.5f * dt * ac.y);
            const float qz = ac.z * (v.z + 0.5f * dt * ac.z);
            ac.x *= 1.f - k.damping * sgnf(qx);
            ac.y *= 1.f - k.damping * sgnf(qy);
            ac.z *= 1.f - k.damping * sgnf(qz);
            a.acc[i] = ac;  // the reference stores the damped acceleration
        }
        v3 nv = mk3(v.x + dt * ac.x, v.y + dt * ac.y, v.z + dt * ac.z);
        v3 np = mk3(p.x + dt * nv.x, p.y + dt * nv.y, p.z + dt * nv.z);
        if (p.w > 0.f) {
            const v3 pre = np;
            const float r2 = 2.f * k.rw;
            if (np.x > k.hix - r2) { np.x = k.hix - r2; nv.x = fminf(nv.x, 0.f); }
            if (np.x < k.lox + r2) { np.x = k.lox + r2; nv.x = fmaxf(nv.x, 0.f); }
            if (np.y > k.hiy - r2) { np.y = k.hiy - r2; nv.y = fminf(nv.y, 0.f); }
            if (np.y < k.loy + r2) { np.y = k.loy + r2; nv.y = fmaxf(nv.y, 0.f); }
            if (np.z > k.hiz - r2) { np.z = k.hiz - r2; nv.z = fminf(nv.z, 0.f); }
            if (np.z < k.loz + r2) { np.z = k.loz + r2; nv.z = fmaxf(nv.z, 0.f); }
            if (k.blabel1) {
                int cx, cy, cz;
                cell_of(k, pre.x, pre.y, pre.z, cx, cy, cz);
                // only where a label-1 particle is near: four candidates' loads
                // in flight, in increasing j
                const bool collider = a.bnear[cell_key(k, cx, cy, cz)] & 2u;
                if (collider) for_columns(k, cx, cy, cz, [&](uint32_t c0, uint32_t c1) {
                    const uint32_t be = a.bcell[c1];
                    for (uint32_t j0 = a.bcell[c0]; j0 < be; j0 += 4u) {
                        float4 q[4];
#pragma unroll
                        for (uint32_t m = 0; m < 4u; ++m) q[m] = a.bpv[j0 + m < be ? j0 + m : j0];
#pragma unroll
                        for (uint32_t m = 0; m < 4u; ++m) {
                            const float4 b = q[m];
                            if (j0 + m >= be || b.w >= 0.f) continue;
                            const v3 dp = pre - xyz(b);
                            const float dl = sqrtf(dot(dp, dp));
                            const float ov = dl - r2;
                            if (ov < 0.f) {
                                nv = nv * 0.f;
                                np += dp * (1.f / dl) * (-ov);
                            }
                        }
                    }
                });
            }
        }
        a.pm_out[i] = f4(np, p.w);
        a.vr_out[i] = f4(nv, v.w);
        if (a.keys_out) {  // the next build's hash (k_hash)
            int cx, cy, cz;
            cell_of(k, np.x, np.y, np.z, cx, cy, cz);
            key = cell_key(k, cx, cy, cz);
            if (a.scene) key += (uint32_t)a.scene[i] * k.C;
            a.keys_out[i] = key;
            old = a.old_keys[i];
            is_water = p.w > 0.f;
        }
    }
    if (a.keys_out) count_moves(key, old, is_water, i, n, a.nc);  // and its change flags (k_inc_flag)
}
void launch_advect(const SFConst& k, const AdvectArgs& a, int n, hipStream_t s) {
    if (n <= 0) return;
    k_advect<<<(n + kBlock - 1) / kBlock, kBlock, 0, s>>>(k, a, n);
}

}  // namespace sf
