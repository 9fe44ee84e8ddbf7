// jl_energy.hip - uint8 "energy" BFS fields for the MAGAT builder on gfx950.
//
// A field is one row search (jl_bfs.h) capped at 255 levels, as
// generate_energy_map_kernel's is (energy_map.cu:174), by one wavefront where
// the map fits one, else by a workgroup; 255 - d leaves as 16-byte row
// segments, its eight bits from the search's level planes by one 8x8 bit
// transpose per 8 cells.  Jobs are dealt out in short runs to wavefronts (or
// workgroups) all over the chip, and a run's jobs that need a field are
// balloted.  The reference launches one 128-thread block per
// row whether or not its row needs a refresh (energy_map.cu:262-271) and
// finds the changed rows with a host-synchronised cumsum
// (grid_world_simulator.cpp:707-753); here the incremental derived state is
// one launch on small maps (the scan, the packed rows and the fields of
// changed goals: goal_changed_refresh_kernel).
//
// Bound by VALU issue when every field is new.  16,000 fields of i.i.d.
// 128 x 128 maps: 6.46 -> 0.19 ms (before: one wavefront per 64 jobs, one
// after the other, with an LDS write per cell and level; now 6,497 VALU
// instructions each, issue 1.0 of the time); 131,072 of 64 x 64, a third of
// the cells obstacles: 2.06 -> 0.25 ms.
#include <type_traits>

#include "jl_bfs.h"
#include "jl_common.h"

namespace jl {
namespace {

constexpr int kEnergyHigh = 4;     // register planes of level bits 4..7: all of a level below 256
constexpr int kEnergyBatches = 16;  // 16 levels each
constexpr int kEnergyWaves = 4;    // wavefronts of a workgroup whose wavefronts search on their own

template <int H, int R, bool kSplit>
constexpr int energy_waves() {
    return kSplit ? SearchShape<H, R>::kMaxWaves : kEnergyWaves;
}

template <int H, int R, bool kSplit, int kWaves = energy_waves<H, R, kSplit>()>
using EnergyLds = SearchLds<H, R, kSplit, false, kWaves>;

// Planes of the highest level bits in LDS (flipped once in 64 and 128 levels),
// where the registers have no room for them, of maps of at most kRows rows:
// one wavefront's [plane][word][row].
template <int N, int kRows>
struct LdsPlanes {
    uint32_t* words;
    __device__ __forceinline__ uint32_t* word(int p, int i) const {
        return words + (p * N + i) * kRows + (threadIdx.x & (kRows - 1));
    }
    __device__ __forceinline__ uint32_t value(int p, int i) const { return *word(p, i); }
    __device__ __forceinline__ void flip(int p, bool first, const uint32_t (&a)[N]) const {
        if ((threadIdx.x & (kWave - 1)) < kRows) {
#pragma unroll
            for (int i = 0; i < N; ++i) *word(p, i) = first ? a[i] : *word(p, i) ^ a[i];
        }
    }
};
struct NoPlanes : NoTallPlanes {
    __device__ __forceinline__ uint32_t value(int, int) const { return 0; }
};

// One field by the calling wavefront (kSplit: the workgroup, each wavefront on
// its rows); every lane calls it with uniform arguments, the goal on the map.
template <int H, int R, bool kSplit, int kHigh = kEnergyHigh, typename Lds, typename Tall = NoPlanes>
__device__ __forceinline__ void energy_field(const uint32_t* __restrict__ env_bits, int W, int gx, int gy,
                                             uint8_t* __restrict__ out, int wave, int waves, Lds& s,
                                             const Tall& tall = {}) {
    static_assert(kHigh == kEnergyHigh || (kHigh == kEnergyHigh - 2 && !std::is_same_v<Tall, NoPlanes>), "every level bit");
    using S = SearchShape<H, R>;
    constexpr int HW = S::HW, N = S::N;
    // (taken afresh for every field: the addresses that follow from it would
    // otherwise be held across the search)
    int lane = threadIdx.x & (kWave - 1);
    asm volatile("" : "+v"(lane));
    const int x0 = (kSplit ? wave * S::kStep : 0) + lane * R;
    SearchPlanes<H, R, kHigh> P;
    load_search_rows<H, R>(env_bits, W, x0, P.avail);
    search_rows<H, R, kSplit, kHigh, kEnergyBatches, false>(P, gx, gy, x0, lane, wave, waves, s, tall);
    uint32_t vis[N];
    load_search_rows<H, R>(env_bits, W, x0, vis);
    const bool own = own_lane<H, R, kSplit>(lane, wave, waves);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int x = x0 + i / HW, k = i % HW;
        // reached cells, the goal's own included where it is an obstacle
        const uint32_t v = (vis[i] & ~P.avail[i]) | (x == gx && k == (gy >> 5) ? 1u << (gy & 31) : 0u);
        // bits of 255 - d: each level bit inverted, none of an unreached cell
        const uint32_t e0 = v & (((x + gx + gy) & 1) ? 0xAAAAAAAAu : 0x55555555u);
        asm volatile("" ::: "memory");  // one word after the other (registers)
        uint32_t p6, p7;  // level bits 6 and 7
        if constexpr (kHigh == kEnergyHigh) {
            p6 = P.high[2][i];
            p7 = P.high[3][i];
        } else {
            p6 = P.tall > 0 ? tall.value(0, i) : 0u;
            p7 = P.tall > 1 ? tall.value(1, i) : 0u;
        }
        if (own && x < W) {
            uint4* row = reinterpret_cast<uint4*>(out + (size_t)x * H + k * 32);
#pragma unroll 1
            for (uint32_t h = 0; h < 2; ++h) {
                uint64_t b[2];
#pragma unroll
                for (uint32_t q = 0; q < 2; ++q) {
                    const uint32_t lo = gather_bytes(e0, v & ~P.low[0][i], v & ~P.low[1][i], v & ~P.low[2][i], 2 * h + q);
                    const uint32_t hi = gather_bytes(v & ~P.high[0][i], v & ~P.high[1][i], v & ~p6, v & ~p7, 2 * h + q);
                    b[q] = transpose8x8((uint64_t)hi << 32 | lo);
                }
                row[h] = make_uint4((uint32_t)b[0], (uint32_t)(b[0] >> 32), (uint32_t)b[1], (uint32_t)(b[1] >> 32));
            }
        }
    }
    if (kSplit) lds_barrier();  // the exchange is rewritten by the next field
}

// This wavefront's (kSplit: this workgroup's) run of `per` jobs of `count`.
template <bool kSplit>
__device__ __forceinline__ int run_begin(int per, int wave) {
    return (kSplit ? (int)blockIdx.x : (int)blockIdx.x * kEnergyWaves + wave) * per;
}

// Jobs are state rows (launch_energy_map_kernel semantics).
template <int H, int R, bool kSplit>
__global__ __launch_bounds__((kWave * energy_waves<H, R, kSplit>())) void energy_rows_kernel(
    const uint32_t* __restrict__ grid_bits, uint8_t* __restrict__ energy, const uint16_t* __restrict__ states,
    int length, int E, int A, int W, int incremental_only, int per, int waves) {
    __shared__ EnergyLds<H, R, kSplit> s_search;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const size_t cells = (size_t)W * H;
    const int begin = run_begin<kSplit>(per, wave);
    const int end = begin + per < length ? begin + per : length;
    for (int c0 = begin; c0 < end; c0 += kWave) {
        const int b = c0 + lane;
        bool run = false;
        uint32_t env = 0, agent = 0, gx = 0, gy = 0;
        if (b < end) {
            const uint4 r = *reinterpret_cast<const uint4*>(states + (size_t)b * 8);
            env = r.x & 0xFFFFu;
            agent = r.x >> 16;
            gx = r.z & 0xFFFFu;
            gy = r.z >> 16;
            const uint32_t reset = r.w >> 16;
            run = !(incremental_only && reset == 0) && env < (uint32_t)E && agent < (uint32_t)A &&
                  gx < (uint32_t)W && gy < (uint32_t)H;
        }
        for (uint64_t todo = __ballot(run); todo; todo &= todo - 1) {
            const int src = __builtin_ctzll(todo);
            const int e = __builtin_amdgcn_readlane((int)env, src), a = __builtin_amdgcn_readlane((int)agent, src);
            const int x = __builtin_amdgcn_readlane((int)gx, src), y = __builtin_amdgcn_readlane((int)gy, src);
            energy_field<H, R, kSplit>(grid_bits + (size_t)e * (cells / 32), W, x, y,
                                       energy + ((size_t)e * A + a) * cells, wave, waves, s_search);
        }
    }
}

// Jobs are simulator agents whose goal_changed flag is set (or all).
template <int H, int R, bool kSplit>
__global__ __launch_bounds__((kWave * energy_waves<H, R, kSplit>())) void energy_flagged_kernel(
    jl_sim_t s, uint8_t* __restrict__ energy, int all_agents, const int64_t* __restrict__ prefix,
    uint16_t* __restrict__ changed, int per, int waves) {
    __shared__ EnergyLds<H, R, kSplit> s_search;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const int A = s.n_agents, W = s.map_w;
    const int N = s.n_envs * A;
    // the scan's total: no goal changed, no field and no row to write
    if (!all_agents && prefix && prefix[N - 1] == 0) return;
    const size_t cells = (size_t)W * H;
    const int begin = run_begin<kSplit>(per, wave);
    const int end = begin + per < N ? begin + per : N;
    for (int c0 = begin; c0 < end; c0 += kWave) {
        const int g = c0 + lane;
        bool run = false;
        uint32_t gx = 0, gy = 0;
        if (g < end) {
            gx = s.goal_x[g];
            gy = s.goal_y[g];
            const bool flagged = s.goal_changed[g] != 0;
            run = (all_agents || flagged) && gx < (uint32_t)W && gy < (uint32_t)H;
            if (!all_agents && flagged && prefix && changed && (!kSplit || wave == 0)) {
                const int64_t slot = prefix[g] - 1;
                const uint32_t e = (uint32_t)(g / A), a = (uint32_t)(g - (int)e * A);
                uint4 v;
                v.x = (e & 0xFFFFu) | (a << 16);
                v.y = (uint32_t)s.cur_x[g] | ((uint32_t)s.cur_y[g] << 16);
                v.z = gx | (gy << 16);
                v.w = (uint32_t)s.actions[g] | (1u << 16);
                *reinterpret_cast<uint4*>(changed + slot * 8) = v;
            }
        }
        for (uint64_t todo = __ballot(run); todo; todo &= todo - 1) {
            const int src = __builtin_ctzll(todo);
            const int x = __builtin_amdgcn_readlane((int)gx, src), y = __builtin_amdgcn_readlane((int)gy, src);
            const int gi = c0 + src;
            const int e = gi / A;
            energy_field<H, R, kSplit>(s.grid_bits + (size_t)e * (cells / 32), W, x, y, energy + (size_t)gi * cells,
                                       wave, waves, s_search);
        }
    }
}

// Incremental derived state in one launch: goal_changed_scan_kernel and
// energy_flagged_kernel together, for at most kRefreshGroups * 1,024 agents
// on maps of at most 4,096 cells and 64 rows.  Workgroup w owns agents
// [w * 1024, (w + 1) * 1024): it sums the values before its range and all of
// them (16-byte words from the L2), scans its range and writes the prefixes;
// each changed agent writes its state row at prefix - 1 (and zero rows over
// the gap that a value above 1 leaves below it), and the rows of the range
// at or past the total are cleared, so every row is written once without
// ordering between workgroups (grid_world_simulator.cpp:709-733,
// pack_changed_agent_state_kernel, 128_agents_map_step.cu:469-511).  Then
// each wavefront runs the energy BFS of its changed agents
// (energy_map.cu:80-272).
constexpr int kRefreshThreads = 1024;
constexpr int kRefreshWaves = kRefreshThreads / kWave;
constexpr int kRefreshGroups = 128;

template <int H>
__global__ __launch_bounds__(kRefreshThreads) void goal_changed_refresh_kernel(jl_sim_t s, uint8_t* __restrict__ energy,
                                                                            int64_t* __restrict__ prefix,
                                                                            int64_t* __restrict__ count,
                                                                            uint16_t* __restrict__ changed) {
    __shared__ EnergyLds<H, 1, false, kRefreshWaves> s_search;
    __shared__ int64_t s_before[kRefreshWaves];
    __shared__ int64_t s_all[kRefreshWaves];
    __shared__ uint32_t s_scan[kRefreshWaves];
    __shared__ uint32_t s_goal[kRefreshThreads];  // (held in LDS: the search leaves no registers for it)
    // 16 wavefronts have 128 registers each, which do not hold a search of
    // rows of eight words: it keeps two level planes in LDS (10,000 agents on 16
    // x 256 maps, no goal changed: 5.0 us; as two launches, 8.0)
    constexpr int kWords = SearchShape<H, 1>::N, kMaxRows = kMarkedCells / H;
    constexpr bool kLdsPlanes = kWords >= 8;
    __shared__ uint32_t s_planes[kLdsPlanes ? kRefreshWaves : 1][kLdsPlanes ? 2 * kWords * kMaxRows : 1];
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);  // uniform per wavefront
    const int A = s.n_agents, W = s.map_w;
    const int N = s.n_envs * A;
    const int c0 = blockIdx.x * kRefreshThreads;
    const int g = c0 + tid;
    const uint8_t* f = s.goal_changed;
    const uint32_t v = g < N ? f[g] : 0u;
    uint32_t gx = 0, gy = 0;
    if (g < N) {
        gx = s.goal_x[g];
        gy = s.goal_y[g];
    }
    // the values before the range and all of them (c0 is a multiple of 16)
    uint64_t before = 0, all = 0;
    const bool vec = (reinterpret_cast<uintptr_t>(f) & 15u) == 0;
    const int words = vec ? N / 16 : 0;
#pragma unroll 8
    for (int k = tid; k < words; k += kRefreshThreads) {
        const uint4 w = reinterpret_cast<const uint4*>(f)[k];
        const uint32_t t = byte_sum(w.x) + byte_sum(w.y) + byte_sum(w.z) + byte_sum(w.w);
        all += t;
        before += k * 16 < c0 ? t : 0u;
    }
    for (int k = words * 16 + tid; k < N; k += kRefreshThreads) {
        all += f[k];
        before += k < c0 ? f[k] : 0u;
    }
    for (int off = kWave / 2; off > 0; off >>= 1) {
        before += __shfl_xor(before, off, kWave);
        all += __shfl_xor(all, off, kWave);
    }
    // this thread's value scanned across the workgroup (a wavefront's sum is
    // at most 64 * 255)
    uint32_t incl = v;
    for (int off = 1; off < kWave; off <<= 1) {
        const uint32_t t = __shfl_up(incl, off, kWave);
        if (lane >= off) incl += t;
    }
    s_goal[tid] = gx | (gy << 16);
    if (lane == 0) {
        s_before[wave] = (int64_t)before;
        s_all[wave] = (int64_t)all;
    }
    if (lane == kWave - 1) s_scan[wave] = incl;
    __syncthreads();
    int64_t run = incl, total = 0;
#pragma unroll
    for (int k = 0; k < kRefreshWaves; ++k) {
        run += s_before[k] + (k < wave ? s_scan[k] : 0u);
        total += s_all[k];
    }
    if (g < N) {
        prefix[g] = run;
        if (g == N - 1) count[0] = run;
    }
    if (changed && g < N) {
        const uint4 zero = make_uint4(0, 0, 0, 0);
        uint4* rows = reinterpret_cast<uint4*>(changed);
        if (g >= total) rows[g] = zero;
        if (v) {
            for (int64_t r = run - v; r < run - 1; ++r) rows[r] = zero;
            const uint32_t e = (uint32_t)(g / A), a = (uint32_t)(g - (int)e * A);
            uint4 row;
            row.x = (e & 0xFFFFu) | (a << 16);
            row.y = (uint32_t)s.cur_x[g] | ((uint32_t)s.cur_y[g] << 16);
            row.z = gx | (gy << 16);
            row.w = (uint32_t)s.actions[g] | (1u << 16);
            rows[run - 1] = row;
        }
    }
    // the energy fields of this wavefront's changed agents
    const int cells = W * H;
    for (uint64_t todo = __ballot(v != 0 && gx < (uint32_t)W && gy < (uint32_t)H); todo; todo &= todo - 1) {
        const int src = __builtin_ctzll(todo);
        const uint32_t goal = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_goal[wave * kWave + src]);
        const int x = (int)(goal & 0xFFFFu), y = (int)(goal >> 16);
        const int gi = c0 + wave * kWave + src;
        const int e = gi / A;
        const uint32_t* bits = s.grid_bits + (size_t)e * (cells / 32);
        uint8_t* out = energy + (size_t)gi * cells;
        if constexpr (kLdsPlanes) {
            energy_field<H, 1, false, kEnergyHigh - 2>(bits, W, x, y, out, wave, kRefreshWaves, s_search,
                                                       LdsPlanes<kWords, kMaxRows>{s_planes[wave]});
        } else {
            energy_field<H, 1, false>(bits, W, x, y, out, wave, kRefreshWaves, s_search);
        }
    }
}

// Workgroups and jobs per run.  A launch that makes every job's field is dealt
// out in runs of about a quarter of what a resident wavefront (kSplit:
// workgroup) does in all, so that the hardware evens out their lengths; one
// that looks for the few changed goals, in one run per resident wavefront.
struct EnergyGrid {
    int groups, per, waves;
};
template <int H, int R, bool kSplit>
EnergyGrid energy_grid(int jobs, int W, bool every) {
    EnergyGrid g;
    g.waves = kSplit ? split_waves<H, R>(W) : kEnergyWaves;
    const int runs_per_group = kSplit ? 1 : kEnergyWaves;
    constexpr int kPerCu = SearchShape<H, R>::N < 8 ? 16 : 12;  // resident wavefronts
    int runs = device_cus() * (kPerCu / g.waves) * runs_per_group * (every ? 4 : 1);
    if (runs > jobs) runs = jobs;
    g.per = (jobs + runs - 1) / runs;
    runs = (jobs + g.per - 1) / g.per;
    g.groups = (runs + runs_per_group - 1) / runs_per_group;
    return g;
}

// f.template operator()<R, kSplit>() with the lane layout of a W x H map: a
// wavefront on its own where its lanes' registers hold the rows (at most 8
// words each, 130 registers), else the map split over a workgroup.  A first MAGAT
// stage of 64 envs of 128 agents, us, with this line at 4, 8 and 16 words (250
// registers, none spilled): 128 x 96 179, 118, 118; 256 x 64 183, 124, 124; 100 x
// 160 195, 194, 186; 160 x 128 205, 249, 231; 128 x 192 326, 326, 195; 256 x 96
// 351, 380, 247; 256 x 128 351, 379, 243; 128 x 256 437, 437, 252.  So 8 against
// 4 holds where a wavefront then is alone, and 16 would gain on the larger maps.
template <int H, typename F>
int with_energy_layout(int W, F f) {
    constexpr int kAlone = SearchShape<H, 4>::N <= 8 ? 4 : (SearchShape<H, 2>::N <= 8 ? 2 : 1);
    if (W <= kWave) return f.template operator()<1, false>();
    if constexpr (kAlone >= 2) {
        if (W <= 2 * kWave) return f.template operator()<2, false>();
        if constexpr (kAlone == 4) return f.template operator()<4, false>();
        else return f.template operator()<2, true>();
    } else {
        return f.template operator()<1, true>();
    }
}

template <int H>
struct LaunchRows {
    const uint32_t* grid_bits;
    uint8_t* energy;
    const uint16_t* states;
    int length, n_envs, n_agents, map_w, incremental_only;
    hipStream_t stream;
    template <int R, bool kSplit>
    int operator()() const {
        const EnergyGrid g = energy_grid<H, R, kSplit>(length, map_w, !incremental_only);
        hipLaunchKernelGGL((energy_rows_kernel<H, R, kSplit>), dim3(g.groups), dim3(kWave * g.waves), 0, stream,
                           grid_bits, energy, states, length, n_envs, n_agents, map_w, incremental_only, g.per, g.waves);
        return launch_status();
    }
};

template <int H>
struct LaunchFlagged {
    const jl_sim_t* s;
    uint8_t* energy;
    int all_agents;
    const int64_t* prefix;
    uint16_t* changed;
    hipStream_t stream;
    template <int R, bool kSplit>
    int operator()() const {
        const EnergyGrid g = energy_grid<H, R, kSplit>(s->n_envs * s->n_agents, s->map_w, all_agents != 0);
        hipLaunchKernelGGL((energy_flagged_kernel<H, R, kSplit>), dim3(g.groups), dim3(kWave * g.waves), 0, stream, *s,
                           energy, all_agents, prefix, changed, g.per, g.waves);
        return launch_status();
    }
};

}  // namespace
}  // namespace jl

using namespace jl;

extern "C" int jl_energy_maps(const uint32_t* grid_bits, uint8_t* energy, const uint16_t* states,
                              int32_t length, int32_t n_envs, int32_t n_agents, int32_t map_w,
                              int32_t map_h, int32_t incremental_only, jl_stream_t stream) {
    if (!grid_bits || !energy || n_envs <= 0 || n_agents <= 0 || length < 0) return JL_ERR_ARG;
    if (length == 0) return JL_OK;
    if (!states) return JL_ERR_ARG;
    if (!profile_ok(map_w, map_h)) return JL_ERR_PROFILE;
    JL_DISPATCH_H(map_h, {
        return with_energy_layout<H>(map_w, LaunchRows<H>{grid_bits, energy, states, length, n_envs, n_agents, map_w,
                                                          incremental_only, (hipStream_t)stream});
    });
    return JL_ERR_PROFILE;
}

extern "C" int jl_energy_maps_flagged(const jl_sim_t* s, uint8_t* energy, int32_t all_agents,
                                      const int64_t* changed_prefix, uint16_t* changed_states,
                                      jl_stream_t stream) {
    if (!s || !energy || !s->grid_bits || !s->goal_x || !s->goal_y || !s->goal_changed)
        return JL_ERR_ARG;
    if (s->n_envs <= 0 || s->n_agents <= 0) return JL_ERR_ARG;
    if (!profile_ok(s->map_w, s->map_h)) return JL_ERR_PROFILE;
    JL_DISPATCH_H(s->map_h, {
        return with_energy_layout<H>(s->map_w, LaunchFlagged<H>{s, energy, all_agents, changed_prefix, changed_states,
                                                               (hipStream_t)stream});
    });
    return JL_ERR_PROFILE;
}

extern "C" int jl_goal_changed_refresh(const jl_sim_t* s, uint8_t* energy, int64_t* prefix, int64_t* count,
                                       uint16_t* changed_states, jl_stream_t stream) {
    if (!s || !energy || !prefix || !count || !s->grid_bits || !s->goal_x || !s->goal_y ||
        !s->goal_changed)
        return JL_ERR_ARG;
    if (s->n_envs <= 0 || s->n_agents <= 0) return JL_ERR_ARG;
    if (!profile_ok(s->map_w, s->map_h)) return JL_ERR_PROFILE;
    if (changed_states && (!s->cur_x || !s->cur_y || !s->actions)) return JL_ERR_ARG;
    const int64_t N = (int64_t)s->n_envs * s->n_agents;
    const int cells = s->map_w * s->map_h;
    if (N <= (int64_t)kRefreshThreads * kRefreshGroups && s->map_w <= kWave && cells <= 4096) {
        const unsigned grid = (unsigned)((N + kRefreshThreads - 1) / kRefreshThreads);
        JL_DISPATCH_H(s->map_h, {
            hipLaunchKernelGGL(goal_changed_refresh_kernel<H>, dim3(grid), dim3(kRefreshThreads), 0,
                               (hipStream_t)stream, *s, energy, prefix, count, changed_states);
        });
        return launch_status();
    }
    const int rc = jl_goal_changed_scan(s, prefix, count, changed_states, stream);
    if (rc) return rc;
    return jl_energy_maps_flagged(s, energy, 0, prefix, changed_states, stream);
}
