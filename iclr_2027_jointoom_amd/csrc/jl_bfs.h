// jl_bfs.h - wavefront-level bit-parallel BFS over one map.
//
// A map row is held as bit masks over its columns.  A level expands the
// frontier with shifts inside the row (y +- 1, carrying across words) and
// with the frontier rows above and below (x +- 1: another register or a DPP
// whole-wavefront shift by one lane), masks with the free cells not reached
// yet, and stops when no lane found a new cell.  Every access but the final
// stores is a register op, so a level costs a few VALU instructions per word
// instead of one thread per frontier node with two workgroup barriers
// (energy_map.cu:174-245, mapf_gpt_cuda.cu:255-318).  BFS distances are
// unique, so the field equals the reference's level-synchronous queue BFS.
//
// wave_bfs, wave_bfs_batched, wave_bfs_levels: rows of 64-bit words, row x =
// lane + 64 r.  search_rows: maps of any size, R consecutive rows per lane.
#pragma once

#include "jl_common.h"

namespace jl {

// Value of lane - 1 (lane 0 reads 0) and of lane + 1 (lane 63 reads 0): DPP
// wave_shr:1 / wave_shl:1 on both halves, no LDS round trip; bound_ctrl
// writes the 0 of the lane without a source.  Every lane of the wavefront
// must be active.
__device__ __forceinline__ uint64_t from_lane_below(uint64_t v) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, 0x138, 0xF, 0xF, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), 0x138, 0xF, 0xF, true);
    return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ uint64_t from_lane_above(uint64_t v) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, 0x130, 0xF, 0xF, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), 0x130, 0xF, 0xF, true);
    return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ uint32_t word_from_below(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x138, 0xF, 0xF, true);
}

__device__ __forceinline__ uint32_t word_from_above(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x130, 0xF, 0xF, true);
}

// One level of a row held in 64 bits: the new frontier (the cells of `avail`
// that neighbour the frontier: `up` / `down` its rows of the lanes below
// and above, `left` / `right` its own row shifted by one column) is returned
// and removed from `avail`.  Per 32-bit half: a = up | right and
// b = down | left (a DPP lane move folded into each OR), then gfx950's
// three-input bit operation twice, (a | b) & avail (truth table 0xA8 with
// a, b, avail as its first, second and third input) and avail & ~(a | b)
// (0x02): four VALU instructions per half instead of the six of an OR3, an
// AND and an XOR after the two ORs.
__device__ __forceinline__ uint64_t level_step(uint64_t up, uint64_t down, uint64_t left, uint64_t right,
                                               uint64_t& avail) {
    const uint32_t a_lo = (uint32_t)up | (uint32_t)right, a_hi = (uint32_t)(up >> 32) | (uint32_t)(right >> 32);
    const uint32_t b_lo = (uint32_t)down | (uint32_t)left, b_hi = (uint32_t)(down >> 32) | (uint32_t)(left >> 32);
    const uint32_t v_lo = (uint32_t)avail, v_hi = (uint32_t)(avail >> 32);
    // (the builtin returns a signed int: each half is taken as uint32_t
    // before it is widened, so no sign bit reaches the high half)
    const uint32_t n_lo = (uint32_t)__builtin_amdgcn_bitop3_b32(a_lo, b_lo, v_lo, 0xA8);
    const uint32_t n_hi = (uint32_t)__builtin_amdgcn_bitop3_b32(a_hi, b_hi, v_hi, 0xA8);
    const uint32_t r_lo = (uint32_t)__builtin_amdgcn_bitop3_b32(a_lo, b_lo, v_lo, 0x02);
    const uint32_t r_hi = (uint32_t)__builtin_amdgcn_bitop3_b32(a_hi, b_hi, v_hi, 0x02);
    avail = ((uint64_t)r_hi << 32) | r_lo;
    return ((uint64_t)n_hi << 32) | n_lo;
}

// Value of a fixed lane, wavefront-uniform.
__device__ __forceinline__ uint64_t lane_value(uint64_t v, int lane) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), lane);
    return ((uint64_t)hi << 32) | lo;
}

template <int H>
struct RowWords {
    static constexpr int HW = (H + 63) / 64;
    static constexpr uint64_t kLastMask = (H % 64 == 0) ? ~0ull : ((1ull << (H % 64)) - 1ull);
};

// Free-cell masks of the rows owned by this lane (0 for rows >= W).
template <int H, int R>
__device__ __forceinline__ void load_free_rows(const uint32_t* __restrict__ env_bits, int W,
                                               uint64_t (&fr)[R][RowWords<H>::HW]) {
    constexpr int HW = RowWords<H>::HW;
    const int lane = threadIdx.x & (kWave - 1);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int x = lane + kWave * r;
#pragma unroll
        for (int k = 0; k < HW; ++k) {
            uint64_t v = 0;
            if (x < W) {
                const uint32_t* row = env_bits + (size_t)x * (H / 32);
                if (H == 32) {
                    v = (uint64_t)(~row[0]) & 0xFFFFFFFFull;
                } else {
                    // a row of H % 64 == 32 columns ends in half a word: its
                    // upper half is not read (it would be the next row's)
                    const uint64_t lo = row[2 * k];
                    const uint64_t hi = 2 * k + 1 < H / 32 ? row[2 * k + 1] : 0xFFFFFFFFu;
                    v = ~(lo | (hi << 32));
                }
                if (k == HW - 1) v &= RowWords<H>::kLastMask;
            }
            fr[r][k] = v;
        }
    }
}

// Runs the BFS from the free cell (gx, gy) and writes dist[x*H+y] = level for
// every reached cell except the start.  dist must already hold the
// "unreached" value and the start cell its 0.
template <int H, int R>
__device__ void wave_bfs(const uint64_t (&fr)[R][RowWords<H>::HW], int gx, int gy, uint16_t* dist) {
    constexpr int HW = RowWords<H>::HW;
    const int lane = threadIdx.x & (kWave - 1);
    uint64_t front[R][HW];
    uint64_t avail[R][HW];  // free cells not reached yet
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
        for (int k = 0; k < HW; ++k) {
            front[r][k] = 0;
            avail[r][k] = fr[r][k];
        }
    }
    {
        const int owner_lane = gx & (kWave - 1);
        const int owner_r = gx / kWave;
        const uint64_t bit = 1ull << (gy & 63);
#pragma unroll
        for (int r = 0; r < R; ++r) {
#pragma unroll
            for (int k = 0; k < HW; ++k) {
                if (lane == owner_lane && r == owner_r && k == (gy >> 6)) {
                    front[r][k] = bit;
                    avail[r][k] &= ~bit;
                }
            }
        }
    }
    for (int level = 1;; ++level) {
        uint64_t nf[R][HW];
        bool any_new = false;
#pragma unroll
        for (int r = 0; r < R; ++r) {
#pragma unroll
            for (int k = 0; k < HW; ++k) {
                // vertical neighbours: row x-1 and x+1 of the same column word
                uint64_t up = from_lane_below(front[r][k]);
                uint64_t down = from_lane_above(front[r][k]);
                if (r > 0) {
                    const uint64_t wrap = lane_value(front[r - 1][k], kWave - 1);
                    if (lane == 0) up = wrap;
                }
                if (r + 1 < R) {
                    const uint64_t wrap = lane_value(front[r + 1][k], 0);
                    if (lane == kWave - 1) down = wrap;
                }
                // horizontal neighbours inside the row (y+1: <<1, y-1: >>1)
                uint64_t left = front[r][k] << 1;
                uint64_t right = front[r][k] >> 1;
                if (k > 0) left |= front[r][k - 1] >> 63;
                if (k + 1 < HW) right |= front[r][k + 1] << 63;
                const uint64_t n = level_step(up, down, left, right, avail[r][k]);
                nf[r][k] = n;
                any_new |= (n != 0);
            }
        }
        if (!__any(any_new)) break;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int x = lane + kWave * r;
#pragma unroll
            for (int k = 0; k < HW; ++k) {
                front[r][k] = nf[r][k];
                uint64_t m = nf[r][k];
                // two new cells per pass, the lowest and the highest (the same
                // cell twice when one is left)
                uint16_t* row_dist = dist + x * H + k * 64;
                while (m) {
                    const int lo = __ffsll((unsigned long long)m) - 1;
                    const int hi = 63 - __clzll((long long)m);
                    row_dist[lo] = (uint16_t)level;
                    row_dist[hi] = (uint16_t)level;
                    m &= ~((1ull << lo) | (1ull << hi));
                }
            }
        }
    }
}

// wave_bfs for one row per lane (R = 1), in batches of 16 levels: the levels
// of a batch are unrolled into straight-line code (expansion, then the new cells ORed
// into the batch mask and into the planes of the level's 4 low bits, chosen
// at compile time), and only after the batch are its cells' distances
// L0 + (plane bits) written, one pass over the batch mask.  The search stops
// after the first batch whose last level reached no cell (levels past the
// last reach nothing, so the field is wave_bfs's).  The single wavefront's
// search is a chain of dependent instructions; the batch keeps the writes
// off that chain and lets the plane and mask updates fill its gaps.
template <int H>
__device__ void wave_bfs_batched(const uint64_t (&fr)[RowWords<H>::HW], int gx, int gy, uint16_t* dist) {
    constexpr int HW = RowWords<H>::HW;
    constexpr int kBatch = 16;
    const int lane = threadIdx.x & (kWave - 1);
    uint64_t front[HW], avail[HW];  // avail: free cells not reached yet
#pragma unroll
    for (int k = 0; k < HW; ++k) {
        front[k] = 0;
        avail[k] = fr[k];
        if (lane == gx && k == (gy >> 6)) {
            front[k] = 1ull << (gy & 63);
            avail[k] &= ~front[k];
        }
    }
    uint16_t* row_dist = dist + lane * H;
    for (int L0 = 1;; L0 += kBatch) {
        uint64_t bm[HW], p0[HW], p1[HW], p2[HW], p3[HW];
#pragma unroll
        for (int k = 0; k < HW; ++k) bm[k] = p0[k] = p1[k] = p2[k] = p3[k] = 0;
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            uint64_t nf[HW];
#pragma unroll
            for (int k = 0; k < HW; ++k) {
                const uint64_t up = from_lane_below(front[k]);
                const uint64_t down = from_lane_above(front[k]);
                uint64_t left = front[k] << 1;
                uint64_t right = front[k] >> 1;
                if (k > 0) left |= front[k - 1] >> 63;
                if (k + 1 < HW) right |= front[k + 1] << 63;
                nf[k] = level_step(up, down, left, right, avail[k]);
            }
#pragma unroll
            for (int k = 0; k < HW; ++k) {
                front[k] = nf[k];
                bm[k] |= nf[k];
                if (j & 1) p0[k] |= nf[k];
                if (j & 2) p1[k] |= nf[k];
                if (j & 4) p2[k] |= nf[k];
                if (j & 8) p3[k] |= nf[k];
            }
        }
#pragma unroll
        for (int k = 0; k < HW; ++k) {
            uint64_t m = bm[k];
            while (m) {
                const int c = __ffsll((unsigned long long)m) - 1;
                const uint32_t j = (uint32_t)((p0[k] >> c) & 1u) | (uint32_t)((p1[k] >> c) & 1u) << 1 |
                                   (uint32_t)((p2[k] >> c) & 1u) << 2 | (uint32_t)((p3[k] >> c) & 1u) << 3;
                row_dist[k * 64 + c] = (uint16_t)(L0 + (int)j);
                m &= m - 1;
            }
        }
        bool more = false;
#pragma unroll
        for (int k = 0; k < HW; ++k) more |= front[k] != 0;
        if (!__any(more)) break;
    }
}

// Level bits of a search on a map of at most 4,096 cells (levels stay below
// 4,096): bit 0 is the cell's colour, bits 1-3 are planes in registers, the
// eight high ones planes in LDS.
constexpr int kFieldPlanes = 12;
constexpr int kHighPlanes = kFieldPlanes - 4;
// LDS of one wavefront's high planes: [plane][lane] 64-bit words.
constexpr int kHighPlaneBytes = kHighPlanes * kWave * 8;

// The even columns (y = 2 i) and the odd columns (y = 2 i + 1) of one map row
// of at most 64 columns, bit i.
struct ColumnPair {
    uint32_t even, odd;
};

// A row's words (H / 32 of them) unshuffled: three delta swaps gather the
// even and the odd bits of each 16, byte permutes do the rest.
template <int H>
__device__ __forceinline__ ColumnPair split_columns(uint64_t row) {
    static_assert(H == 32 || H == 64, "one or two words per row");
    uint32_t w[2] = {(uint32_t)row, (uint32_t)(row >> 32)};
#pragma unroll
    for (int k = 0; k < H / 32; ++k) {
        uint32_t t = (w[k] ^ (w[k] >> 1)) & 0x22222222u;
        w[k] ^= t ^ (t << 1);
        t = (w[k] ^ (w[k] >> 2)) & 0x0C0C0C0Cu;
        w[k] ^= t ^ (t << 2);
        t = (w[k] ^ (w[k] >> 4)) & 0x00F000F0u;
        w[k] ^= t ^ (t << 4);
    }
    if (H == 32) w[1] = 0;
    return {__builtin_amdgcn_perm(w[1], w[0], 0x06040200u), __builtin_amdgcn_perm(w[1], w[0], 0x07050301u)};
}

// The cells of one colour of the checkerboard that are in r's cells of the
// other colour or next to them, for wave_bfs_levels: index i of the other
// colour is a neighbour in this row and in the rows of both adjacent lanes,
// and so is this row's index i - 1 or i + 1, which `turn` rotates into place
// and `keep` clears of the bit that came round.
__device__ __forceinline__ uint32_t next_colour(uint32_t r, uint32_t turn, uint32_t keep) {
    const uint32_t beside = __builtin_amdgcn_alignbit(r, r, turn);
    uint32_t t = (uint32_t)__builtin_amdgcn_bitop3_b32(beside, keep, r, 0xEA);  // (beside & keep) | r
    t |= word_from_below(r);
    return t | word_from_above(r);
}

// a ^ b ^ c, one instruction.
__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c) {
    return (uint32_t)__builtin_amdgcn_bitop3_b32(a, b, c, 0x96);
}

// wave_bfs_batched without a distance array: the level of every reached cell
// of this lane's row is left bit-sliced, bits 1-3 in lowp[0..2] and bits 4-11
// in s_high[b - 4][lane] (this wavefront's kHighPlaneBytes of LDS), the
// reached cells in vis (the start included, at level 0; it must be a free
// cell); the planes of cells not reached hold anything.  One wavefront, one
// map row per lane, rows of at most 64 columns.
//
// A grid is bipartite: the cells at even levels are those of the start's
// colour of the checkerboard, and a level only reaches cells of the other
// colour than the one before.  A row's cells of the start's colour (`own`)
// and the others (`off`) are a 32-bit word each, and a level is one step from
// one word to the other, five VALU instructions: the words hold everything
// reached so far, since a reached cell but the start has a reached neighbour
// one level below it, so no frontier and no set of cells still free is kept.
// (Both colours in one 64-bit word, twice the words at every level, and a
// frontier beside the cells still free: ten instructions.)  Bit 0 of a level
// is its cell's colour.  With m the level's number >> 1, a cell reached at m
// lies outside the words of steps 0 .. m - 1, so bit 0 of m is the parity of
// the number of steps, bit 1 of the number of odd steps, bit 2 of every
// fourth's, at which the cell is outside its word: two steps at a time are
// one three-input exclusive OR (the complements cancel).  Batch b runs levels
// 16 b + 1 .. 16 b + 16 unrolled and flips, at the cells outside, the planes
// of the batch number's changed bits, two on average, by LDS atomics.  The
// search stops after the first batch whose last level reached nothing.
//
// An even column's off-colour neighbours in its row have its own index and
// the index below, an odd column's its own and the index above.  s_high's
// words hold own in their lower half and off in their upper half.
template <int H>
__device__ void wave_bfs_levels(ColumnPair free, int gx, int gy, ColumnPair& vis, ColumnPair (&lowp)[3],
                                uint64_t* s_high) {
    const int lane = threadIdx.x & (kWave - 1);
    const bool own_odd = (lane + gx + gy) & 1;  // own: this row's odd columns
    const uint32_t free_own = own_odd ? free.odd : free.even, free_off = own_odd ? free.even : free.odd;
    const uint32_t start = lane == gx ? 1u << (gy >> 1) : 0u;
    const uint32_t to_off = own_odd ? 31u : 1u, to_own = 32u - to_off;  // right by 1 or left by 1
    const uint32_t keep_off = own_odd ? ~1u : ~0u >> 1, keep_own = own_odd ? ~0u >> 1 : ~1u;
    uint32_t own = start, off = 0, last;
    uint32_t po[3] = {0, 0, 0}, pf[3] = {0, 0, 0};
#pragma unroll
    for (int p = 0; p < kHighPlanes; ++p) s_high[p * kWave + lane] = 0;
    for (int b = 0;; ++b) {
        uint32_t so[3] = {0, 0, 0}, sf[3] = {0, 0, 0};  // the words at the first of two flips
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            off = next_colour(own, to_off, keep_off) & free_off;
#pragma unroll
            for (int p = 0; p < 3; ++p) {
                const int every = 1 << p;
                if (k % (2 * every) == every - 1) {
                    so[p] = own;
                    sf[p] = off;
                }
                if (k % (2 * every) == 2 * every - 1) {
                    po[p] = xor3(po[p], so[p], own);
                    pf[p] = xor3(pf[p], sf[p], off);
                }
            }
            if (k == 7) {
                const int hb = __builtin_amdgcn_readfirstlane(b), change = hb ^ (hb + 1);
                const uint64_t outside = ~((uint64_t)off << 32 | own);
                for (int p = 0; p < kHighPlanes && (change >> p); ++p)
                    atomicXor(reinterpret_cast<unsigned long long*>(s_high + p * kWave + lane), outside);
            }
            last = own;
            own = (uint32_t)__builtin_amdgcn_bitop3_b32(next_colour(off, to_own, keep_own), free_own, start, 0xEA);
        }
        if (!__any(own != last)) break;
    }
    vis.even = own_odd ? off : own;
    vis.odd = own_odd ? own : off;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
        lowp[p].even = own_odd ? pf[p] : po[p];
        lowp[p].odd = own_odd ? po[p] : pf[p];
    }
}

// 8x8 bit-matrix transpose: bit c of byte b moves to bit b of byte c.
__device__ __forceinline__ uint64_t transpose8x8(uint64_t x) {
    uint64_t t = (x ^ (x >> 7)) & 0x00AA00AA00AA00AAull;
    x = x ^ t ^ (t << 7);
    t = (x ^ (x >> 14)) & 0x0000CCCC0000CCCCull;
    x = x ^ t ^ (t << 14);
    t = (x ^ (x >> 28)) & 0x00000000F0F0F0F0ull;
    x = x ^ t ^ (t << 28);
    return x;
}

// Bytes q of four words, in a word.
__device__ __forceinline__ uint32_t gather_bytes(uint32_t a, uint32_t b, uint32_t c, uint32_t d, uint32_t q) {
    const uint32_t sel = 0x0C0C0400u + q * 0x0101u;
    return __builtin_amdgcn_perm(b, a, sel) | __builtin_amdgcn_perm(d, c, sel) << 16;
}

// ---------------------------------------------------------------------------
// Row search: one field on a map whose rows do not fit one 64-bit word per
// lane.  A lane holds R consecutive map rows (x = row0 + R * lane + r), so a
// row's x +- 1 neighbours are another register of the lane or, at the ends of
// its block, one DPP lane move: no word of the search leaves the registers.
//
// The two colours of the checkerboard are searched in turn, as in
// wave_bfs_levels: words of everything reached so far of the goal's colour
// (`own`) and of the other (`off`), and a level is one step from one to the
// other.  A row is folded in the middle: index y < H / 2 stands for the
// columns y and H - 1 - y, which are of different colours, so an `own` word
// holds one of the two at each index and the `off` word the other.  Whatever
// the row's parity, the neighbours of index y are the indices y - 1 and y + 1
// of the row itself and y of the rows beside it, and at the last index also
// itself (the two middle columns).  A level costs five VALU instructions per
// folded word (two funnel shifts, two ORs, one three-input bit operation),
// half a row's words (rounded up) instead of all of them with six.
//
// Levels are held bit-sliced: bit 0 is the cell's colour; a cell's other bits
// follow the search until the cell is reached, which freezes them: whenever
// a level's number changes a bit, that bit's plane is flipped at every cell
// not reached (bit 1 after every step of a colour, bit 2 after every second,
// ...; two flips of bit 1 at a time).  Bits 1-3 and kHigh more are planes in
// registers; the planes of higher bits, flipped rarely (bit k once in 2^k
// levels), lie in LDS (the first kTall of a split search) and in the memory of
// the field being searched, which the caller writes last (TallPlanes).  The search's result is unfolded.
//
// Split (kSplit): maps of more rows than one wavefront's 64 R are split over
// the wavefronts of a workgroup.  Neighbouring wavefronts overlap: each also
// searches the kGhost lanes of rows beyond its own on either side, which stay
// right in its own rows for kGhost * R = 8 levels; after every 8 levels the
// owners' rows replace the overlap through LDS.  One barrier in 8 levels,
// against one per level with the boundary rows alone (256 x 256: five
// wavefronts instead of four, but 8 times fewer barriers and LDS round trips).
// A wavefront in none of whose rows, overlap included, the first of those 8
// levels reaches a cell leaves the others out.
// ---------------------------------------------------------------------------
constexpr int kSplitLevels = 8;  // levels between two exchanges of a split search

template <int H, int R>
struct SearchShape {
    static constexpr int HW = H / 32;              // words per row
    static constexpr int N = R * HW;               // words per lane
    static constexpr int M = (HW + 1) / 2;         // words per folded row and colour
    static constexpr int K = R * M;                // words per lane and colour
    static constexpr int kGhost = kSplitLevels / R;  // overlapping lanes on each side of a split
    static constexpr int kStep = (kWave - 2 * kGhost) * R;  // rows from one wavefront of a split to the next
    static constexpr int kMaxWaves = (256 - kWave * R + kStep - 1) / kStep + 1;
    static_assert(kSplitLevels % R == 0 && H % 32 == 0, "row search shape");
};

// Wavefronts of a split search of W rows (tile rows past W included).
template <int H, int R>
__host__ __device__ constexpr int split_waves(int W) {
    const int rows = (W + 7) / 8 * 8;
    return rows <= kWave * R ? 1
                             : (rows - kWave * R + SearchShape<H, R>::kStep - 1) / SearchShape<H, R>::kStep + 1;
}

// LDS of one wavefront of a search.
template <int H, int R, bool kSplit, bool kCount>
struct SearchWaveLds {
    using S = SearchShape<H, R>;
    static constexpr int kTall = kSplit && kCount ? 2 : 0;                  // level planes held here
    uint2 edge[kSplit ? 2 : 1][2][kSplit ? S::N : 1][kSplit ? S::kGhost : 1];  // a split's overlapping rows
    uint2 before[kCount ? S::K * kWave : 1];                                // cells reached before a batch
    uint32_t tall[kTall ? kTall : 1][kTall ? S::N : 1][kTall ? kWave : 1];
};

// LDS of the searches of a workgroup of at most kWaves wavefronts: a launch of
// `waves` allocates bytes(waves).
template <int H, int R, bool kSplit, bool kCount, int kWaves>
struct SearchLds {
    using Wave = SearchWaveLds<H, R, kSplit, kCount>;
    uint32_t flag[2][kWaves];  // count << 1 | cells left to expand
    uint32_t count[16];
    uint32_t cell[8];
    alignas(16) Wave wave[kWaves];
    static constexpr size_t bytes(int waves) {
        return (sizeof(SearchLds) - (kWaves - waves) * sizeof(Wave) + 15) / 16 * 16;
    }
};

// One wavefront's part of a search's result.
template <int H, int R, int kHigh>
struct SearchPlanes {
    static constexpr int N = SearchShape<H, R>::N;
    uint32_t avail[N];           // free cells not reached
    uint32_t low[3][N];          // level bits 1..3
    uint32_t high[kHigh][N];     // level bits 4 .. 3 + kHigh
    int tall;                    // planes of the bits above in use (TallPlanes)
    int batches;                 // of 16 levels searched: every level is at most 16 * batches
};

// One lane's words.
template <int H, int R>
using LaneWords = uint32_t[SearchShape<H, R>::N];

// One lane's words of one colour.
template <int H, int R>
using ColourWords = uint32_t[SearchShape<H, R>::K];

// Index bits of row r that stand for the columns of the lower half in the own
// words (even0: this lane's row 0 has even columns of the goal's colour).
__device__ __forceinline__ uint32_t own_lower(bool even0, int r) {
    return even0 == (r % 2 == 0) ? 0x55555555u : 0xAAAAAAAAu;
}

template <int H, int R>
__device__ __forceinline__ void fold_rows(const LaneWords<H, R>& w, bool even0, ColourWords<H, R>& own,
                                          ColourWords<H, R>& off) {
    using S = SearchShape<H, R>;
#pragma unroll
    for (int i = 0; i < S::K; ++i) {
        const int r = i / S::M, k = i % S::M;
        const uint32_t m = own_lower(even0, r), half = S::HW % 2 != 0 && k == S::M - 1 ? 0xFFFFu : ~0u;
        const uint32_t lower = w[r * S::HW + k], upper = __builtin_bitreverse32(w[r * S::HW + S::HW - 1 - k]);
        own[i] = ((lower & m) | (upper & ~m)) & half;
        off[i] = ((upper & m) | (lower & ~m)) & half;
    }
}

template <int H, int R>
__device__ __forceinline__ void unfold_rows(const ColourWords<H, R>& own, const ColourWords<H, R>& off, bool even0,
                                            LaneWords<H, R>& w) {
    using S = SearchShape<H, R>;
#pragma unroll
    for (int i = 0; i < S::K; ++i) {
        const int r = i / S::M, k = i % S::M;
        const uint32_t m = own_lower(even0, r);
        const uint32_t lower = (own[i] & m) | (off[i] & ~m), upper = (off[i] & m) | (own[i] & ~m);
        if (S::HW % 2 != 0 && k == S::M - 1) {
            w[r * S::HW + k] = (lower & 0xFFFFu) | __builtin_bitreverse32(upper & 0xFFFFu);
        } else {
            w[r * S::HW + k] = lower;
            w[r * S::HW + S::HW - 1 - k] = __builtin_bitreverse32(upper);
        }
    }
}

// One level: `to` becomes the free cells of its colour beside those of `from`.
// kPair: p is flipped at the cells outside `to` as they were and as they are;
// kNews: returns whether `to` changed.
template <int H, int R, bool kPair, bool kNews>
__device__ __forceinline__ uint32_t expand_rows(const ColourWords<H, R>& from, const ColourWords<H, R>& fr,
                                                ColourWords<H, R>& to, ColourWords<H, R>& p) {
    using S = SearchShape<H, R>;
    constexpr int M = S::M, K = S::K;
    uint32_t news = 0;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        const int r = i / M, k = i % M;
        const uint32_t up = r > 0 ? from[r > 0 ? i - M : 0] : word_from_below(from[(R - 1) * M + k]);
        const uint32_t down = r + 1 < R ? from[r + 1 < R ? i + M : 0] : word_from_above(from[k]);
        const uint32_t before = k > 0 ? __builtin_amdgcn_alignbit(from[i], from[k > 0 ? i - 1 : 0], 31) : from[i] << 1;
        uint32_t after;  // the last index is its own neighbour
        if (k + 1 < M) after = __builtin_amdgcn_alignbit(from[k + 1 < M ? i + 1 : 0], from[i], 1);
        else if (S::HW % 2 == 0) after = (uint32_t)((int32_t)from[i] >> 1);
        else after = (from[i] >> 1) | (from[i] & 0x8000u);
        const uint32_t a = up | after, b = down | before;
        const uint32_t n = (uint32_t)__builtin_amdgcn_bitop3_b32(a, b, fr[i], 0xA8);  // (a | b) & fr
        if (kPair) p[i] = xor3(p[i], to[i], n);
        if (kNews) news |= to[i] ^ n;
        to[i] = n;
    }
    // levels are not interleaved: a level's words are independent enough, and
    // two levels' worth of them would not fit the registers
    __builtin_amdgcn_sched_barrier(0);
    return news;
}

// p ^= ~a for every word.
template <int N>
__device__ __forceinline__ void flip_outside(uint32_t (&p)[N], const uint32_t (&a)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) p[i] = ~(p[i] ^ a[i]);
}

// Sum over the wavefront's lanes, wavefront-uniform (DPP steps that leave it in lane 63).
__device__ __forceinline__ int wave_sum(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, false);   // quad_perm [1,0,3,2]
    v += __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, false);   // quad_perm [2,3,0,1]
    v += __builtin_amdgcn_update_dpp(0, v, 0x141, 0xF, 0xF, false);  // row_half_mirror
    v += __builtin_amdgcn_update_dpp(0, v, 0x140, 0xF, 0xF, false);  // row_mirror
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);  // row_bcast15 into rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);  // row_bcast31 into rows 2 and 3
    return __builtin_amdgcn_readlane(v, kWave - 1);
}

// Free-cell words of a lane's rows, from map row x0 on (0 for rows past W).
template <int H, int R>
__device__ __forceinline__ void load_search_rows(const uint32_t* __restrict__ env_bits, int W, int x0,
                                                 LaneWords<H, R>& fr) {
    constexpr int HW = SearchShape<H, R>::HW;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int x = x0 + r;
        const uint32_t* row = env_bits + (size_t)(x < W ? x : 0) * HW;
#pragma unroll
        for (int k = 0; k < HW; ++k) {
            const uint32_t w = row[k];
            fr[r * HW + k] = x < W ? ~w : 0u;
        }
    }
}

// Lanes of this wavefront whose rows are its own (the others overlap a
// neighbour's, whose copy counts).
template <int H, int R, bool kSplit>
__device__ __forceinline__ bool own_lane(int lane, int wave, int waves) {
    if (!kSplit) return true;
    constexpr int G = SearchShape<H, R>::kGhost;
    return (lane >= G || wave == 0) && (lane < kWave - G || wave + 1 == waves);
}

// No planes past the register ones (searches capped below 2^(4 + kHigh) levels).
struct NoTallPlanes {
    template <int N>
    __device__ __forceinline__ void flip(int, bool, const uint32_t (&)[N]) const {}
};

// The search from (gx, gy) (inside the map; reached whether free or not) over
// the free rows in P.avail.  kCap: levels from 16 * kCap on stay unreached
// (0: no cap).  Returns, when kCount, the sum over levels of max(0, cells -
// kLimit).  Every lane of the wavefront (kSplit: of the workgroup)
// calls it with the same goal, and with the first of its map rows in x0.
template <int H, int R, bool kSplit, int kHigh, int kCap, bool kCount, int kLimit = kMaxFrontier, typename Lds,
          typename Tall>
__device__ __forceinline__ int search_rows(SearchPlanes<H, R, kHigh>& P, int gx, int gy, int x0, int lane, int wave, int waves,
                                           Lds& s, const Tall& tall) {
    using S = SearchShape<H, R>;
    constexpr int HW = S::HW, N = S::N, M = S::M, K = S::K, G = S::kGhost;
    const bool mine = own_lane<H, R, kSplit>(lane, wave, waves);
    const bool even0 = ((x0 + gx + gy) & 1) == 0;
    // the cells reached before a batch, read back only where its levels are
    // counted (volatile: kept in LDS, not forwarded through registers)
    const auto before_words = [&]() {
        int l = lane;
        // the address taken afresh, or held across the search: a split of
        // seven words per lane (224 columns) has no register left to hold it;
        // elsewhere holding it is 1 % of a stage of new fields faster
        if constexpr (kSplit && N == 7) asm("" : "+v"(l));
        return reinterpret_cast<volatile uint32_t*>(s.wave[wave].before + l);
    };
    uint32_t own[K], off[K], fr_own[K], fr_off[K];
    uint32_t low_own[3][K], low_off[3][K], high_own[kHigh][K], high_off[kHigh][K];
    P.tall = 0;
    {
        uint32_t w[N];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            w[i] = (x0 + i / HW == gx && i % HW == (gy >> 5)) ? 1u << (gy & 31) : 0u;
            P.avail[i] |= w[i];
        }
        fold_rows<H, R>(P.avail, even0, fr_own, fr_off);
        fold_rows<H, R>(w, even0, own, off);  // (the goal is in own)
    }
#pragma unroll
    for (int i = 0; i < K; ++i) {
        off[i] = 0;
        low_own[0][i] = low_own[1][i] = low_own[2][i] = low_off[0][i] = low_off[1][i] = low_off[2][i] = 0;
#pragma unroll
        for (int p = 0; p < kHigh; ++p) high_own[p][i] = high_off[p][i] = 0;
    }
    auto reached_cells = [&]() -> int {
        int c = 0;
#pragma unroll
        for (int i = 0; i < K; ++i) c += __popc(own[i]) + __popc(off[i]);
        return c;
    };
    int slot = 0, cells = kCount ? reached_cells() : 0;
    bool big = false;  // kCount: 8 levels of the batch reached more than kLimit cells
    // After kSplitLevels levels: whether any cell is left to expand (news:
    // this lane's last level reached one); sets big.  kSplit: the overlap is
    // taken from its owners.
    auto meet = [&](uint32_t news) -> bool {
        const bool left = news != 0;
        int reached = 0;
        if (kCount) {
            const int now = reached_cells();
            reached = now > cells ? now - cells : 0;  // (a goal alone is lost)
            cells = now;
        }
        if constexpr (!kSplit) {
            // more than kLimit cells need a lane with more than its share
            if (kCount && __any(reached > kLimit / kWave)) big |= wave_sum(reached) > kLimit;
            return __any(left) != 0;
        } else {
            const bool lo = lane >= G && lane < 2 * G, hi = lane >= kWave - 2 * G && lane < kWave - G;
            if (lo || hi) {
                uint2* out = &s.wave[wave].edge[slot][hi ? 1 : 0][0][hi ? lane - (kWave - 2 * G) : lane - G];
#pragma unroll
                for (int i = 0; i < K; ++i) out[i * G] = make_uint2(own[i], off[i]);
            }
            const bool more = __any(left && mine) != 0;
            const int sum = kCount ? wave_sum(mine ? reached : 0) : 0;
            if (lane == 0) s.flag[slot][wave] = (uint32_t)sum << 1 | (more ? 1u : 0u);
            lds_barrier();
            const uint32_t all = s.flag[slot][lane < waves ? lane : 0];
            const bool from_lo = lane < G && wave > 0, from_hi = lane >= kWave - G && wave + 1 < waves;
            if (from_lo || from_hi) {
                const uint2* in = from_lo ? &s.wave[wave - 1].edge[slot][1][0][lane]
                                          : &s.wave[wave + 1].edge[slot][0][0][lane - (kWave - G)];
#pragma unroll
                for (int i = 0; i < K; ++i) {
                    const uint2 v = in[i * G];
                    own[i] = v.x;
                    off[i] = v.y;
                }
            }
            slot ^= 1;
            // (the wavefronts' counts are added up only where one of them
            // has more than its share)
            if (kCount && __any((int)(all >> 1) * waves > kLimit))
                big |= wave_sum(lane < waves ? (int)(all >> 1) : 0) > kLimit;
            return __any(all & 1u) != 0;
        }
    };
    // levels 1 .. 7 of eight, their flips included; the eighth and the flips
    // before it follow.  False: none of them, nor the eighth, reaches a cell
    // here (split searches), and none was searched: their flips of bits 1 and
    // 2 cancel
    auto seven = [&]() -> bool {
        if (kSplit) {
            const uint32_t news = expand_rows<H, R, false, true>(own, fr_off, off, low_off[0]);
            if (!__any(news != 0)) return false;
        } else {
            expand_rows<H, R, false, false>(own, fr_off, off, low_off[0]);
        }
        expand_rows<H, R, true, false>(off, fr_own, own, low_own[0]);   // 2: bit 1 at steps 0 and 1
        expand_rows<H, R, true, false>(own, fr_off, off, low_off[0]);   // 3
        flip_outside(low_own[1], own);
        flip_outside(low_off[1], off);
        expand_rows<H, R, false, false>(off, fr_own, own, low_own[0]);  // 4
        expand_rows<H, R, false, false>(own, fr_off, off, low_off[0]);  // 5
        expand_rows<H, R, true, false>(off, fr_own, own, low_own[0]);   // 6: steps 2 and 3
        expand_rows<H, R, true, false>(own, fr_off, off, low_off[0]);   // 7
        flip_outside(low_own[1], own);
        flip_outside(low_off[1], off);
        return true;
    };
    int overflow = 0;
    for (int b = 0;; ++b) {
        // levels 16 b + 1 .. 16 b + 16
        if (kCount) {
            big = false;
            volatile uint32_t* before = before_words();
#pragma unroll
            for (int i = 0; i < K; ++i) {
                before[2 * i * kWave] = own[i];
                before[2 * i * kWave + 1] = off[i];
            }
        }
        uint32_t news = 0;
        bool act = seven();
        flip_outside(low_own[2], own);
        flip_outside(low_off[2], off);
        if (act) news = expand_rows<H, R, false, true>(off, fr_own, own, low_own[0]);
        bool more = meet(news);
        if (more) {
            act = seven();
            if (kCap && b + 1 == kCap) break;  // level 16 * kCap stays out
            // the level's number reaches 16 (b + 1)
            flip_outside(low_own[2], own);
            flip_outside(low_off[2], off);
            const int hb = __builtin_amdgcn_readfirstlane(b), change = hb ^ (hb + 1);
#pragma unroll
            for (int p = 0; p < kHigh; ++p) {
                if (p == 0 || ((change >> p) & 1)) {
                    flip_outside(high_own[p], own);
                    flip_outside(high_off[p], off);
                }
            }
            if (change >> kHigh) {
                uint32_t outside[N];
                unfold_rows<H, R>(own, off, even0, outside);
#pragma unroll
                for (int i = 0; i < N; ++i) outside[i] = ~outside[i];
                for (int p = 0; change >> (kHigh + p); ++p) {
                    tall.flip(p, p == P.tall, outside);
                    if (p == P.tall) P.tall = p + 1;
                }
            }
            news = 0;
            if (act) news = expand_rows<H, R, false, true>(off, fr_own, own, low_own[0]);
            more = meet(news);
        }
        if (kCount && big) {
            // count the cells of each of the batch's levels, told apart by
            // their four low bits
            if (kSplit) {
                lds_barrier();
                if (threadIdx.x < 16) s.count[threadIdx.x] = 0;
                lds_barrier();
            }
            volatile uint32_t* before = before_words();
            for (int v = 0; v < 16; ++v) {
                int c = 0;
#pragma unroll
                for (int i = 0; i < K; ++i) {
                    uint32_t m = (v & 1) ? off[i] & ~before[2 * i * kWave + 1] : own[i] & ~before[2 * i * kWave];
#pragma unroll
                    for (int p = 0; p < 3; ++p) {
                        const uint32_t bit = (v & 1) ? low_off[p][i] : low_own[p][i];
                        m &= ((v >> (p + 1)) & 1) ? bit : ~bit;
                    }
                    c += __popc(m);
                }
                c = wave_sum(mine ? c : 0);
                if (kSplit) {
                    if (lane == 0) atomicAdd(&s.count[v], (uint32_t)c);
                } else if (c > kLimit) {
                    overflow += c - kLimit;
                }
            }
            if (kSplit) {
                lds_barrier();
                for (int v = 0; v < 16; ++v) {
                    const int c = __builtin_amdgcn_readfirstlane((int)s.count[v]);
                    if (c > kLimit) overflow += c - kLimit;
                }
                lds_barrier();
            }
        }
        P.batches = b + 1;
        if (!more) break;
    }
    // the goal, which a search without a second cell has lost, is at level 0
#pragma unroll
    for (int p = 0; p < 3; ++p) unfold_rows<H, R>(low_own[p], low_off[p], even0, P.low[p]);
#pragma unroll
    for (int p = 0; p < kHigh; ++p) unfold_rows<H, R>(high_own[p], high_off[p], even0, P.high[p]);
    uint32_t reached[N];
    unfold_rows<H, R>(own, off, even0, reached);
    unfold_rows<H, R>(fr_own, fr_off, even0, P.avail);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const uint32_t goal = (x0 + i / HW == gx && i % HW == (gy >> 5)) ? 1u << (gy & 31) : 0u;
        P.avail[i] &= ~(reached[i] | goal);
#pragma unroll
        for (int p = 0; p < 3; ++p) P.low[p][i] &= ~goal;
#pragma unroll
        for (int p = 0; p < kHigh; ++p) P.high[p][i] &= ~goal;
    }
    return overflow;
}

// (a, b) of the rows beside this wavefront's own in a split, from their
// owners into the overlapping lanes (the owners' first and last rows are what
// a wavefront's rows border on).  Called by the whole workgroup after a
// search; the caller lets every wavefront past it before the next search.
template <int H, int R, typename Lds>
__device__ __forceinline__ void meet_rows(LaneWords<H, R>& a, LaneWords<H, R>& b, int lane, int wave, int waves, Lds& s) {
    constexpr int N = SearchShape<H, R>::N, G = SearchShape<H, R>::kGhost;
    lds_barrier();  // the search's last exchange has been read
    const bool lo = lane >= G && lane < 2 * G, hi = lane >= kWave - 2 * G && lane < kWave - G;
    if (lo || hi) {
        uint2* out = &s.wave[wave].edge[0][hi ? 1 : 0][0][hi ? lane - (kWave - 2 * G) : lane - G];
#pragma unroll
        for (int i = 0; i < N; ++i) out[i * G] = make_uint2(a[i], b[i]);
    }
    lds_barrier();
    const bool from_lo = lane < G && wave > 0, from_hi = lane >= kWave - G && wave + 1 < waves;
    if (from_lo || from_hi) {
        const uint2* in = from_lo ? &s.wave[wave - 1].edge[0][1][0][lane]
                                  : &s.wave[wave + 1].edge[0][0][0][lane - (kWave - G)];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const uint2 v = in[i * G];
            a[i] = v.x;
            b[i] = v.y;
        }
    }
}

}  // namespace jl
