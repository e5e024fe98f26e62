// incsort.hip -- the per-step cell sort, updated instead of redone.
//
// Between two steps few particles change cell (0.05% of the 8.4M-particle
// slab per step, about 1% of a batch of small scenes).  The sorted
// order of step n+1 -- the stable sort of the new keys, i.e. ascending
// (key, slot) -- is the sorted order of step n with the moved particles
// taken out and put back at their new places:
//   * the transfer kernel copies step n's sorted keys and slots (the
//     snapshot) as it reads them;
//   * G2P appends each particle whose new key differs from its old one to a
//     list (new key, slot, old sorted position; kMoveLists sub-lists);
//   * k_inc_route marks every entry's old position as gone and puts the entry
//     into the bucket of the snapshot tile its place lies in (a binary search
//     over the tiles' first entries);
//   * k_inc_merge, one workgroup per tile, finds the places in the tile,
//     ranks the insertions that share one, and writes every unmoved entry at
//     i - (removed before i) + (inserted at or before i) and every inserted
//     entry at its place - (removed before it) + (inserted before it).
// The result is bit-identical to a stable radix sort of the new keys.  The
// device-side plan words pick this path or the full radix sort each step
// (the other path's launches return at once): the full sort runs when the
// list overflowed, a tile drew more entries than its bucket holds, or the
// snapshot is not the previous step's (first step, state written, a
// single scene's store reordered, a batch's layout changed).  The step's item
// count resets the words and the tile counts afterwards (launch_items with
// plan).  Launch order within a step: launch_inc_prepare, the radix sort
// (which reads the decision), launch_inc_merge.
//
// What bounds it: the merge's 16 bytes per particle; the routing is a chain
// of dependent loads per entry, hidden behind the other entries.  Before,
// every entry's place was searched in the whole snapshot, and the removals
// and insertions were bucketed by counts, a scan in one workgroup and a second
// pass (searches twice as long and two launches more).  Measured, the four
// kernels before and the two now, us: 2.1M slab 38 -> 20, 8.4M slab 85 -> 47
// (64 beside the grid's clear), uneven batch of 11.0M 190 -> 86 (114 beside the
// clear), served batch of 2.6M 114 -> 49 (beside it).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "blockscan.h"
#include "gridclear.h"
#include "launch.h"

namespace mpm {

constexpr int kIncWG = 256;

// (key, slot) order of two sort entries.
__device__ __forceinline__ bool entry_less(uint32_t ka, uint32_t sa, uint32_t kb, uint32_t sb) {
    return ka < kb || (ka == kb && sa < sb);
}

__global__ void k_inc_set(uint32_t* plan, uint32_t snap_ok) {
    if (threadIdx.x < kMoveLists) plan[kPlanLists + threadIdx.x * kMoveCountStride] = 0u;
    if (threadIdx.x != 0) return;
    plan[kPlanSnapOk] = snap_ok;
    plan[kPlanOverflow] = 0u;
}

// The entries of the sub-lists: blockIdx.x % kMoveLists picks the sub-list,
// the other blocks of the grid with that remainder stride over its filled
// part (a sub-list's count is at most its capacity unless it overflowed,
// and then no update runs).  j: the entry's index in the list arrays.
#define FOR_LIST_ENTRIES(plan, j)                                                                             \
    const uint32_t r_ = blockIdx.x % (uint32_t)kMoveLists;                                                    \
    const uint32_t c_ = (plan)[kPlanLists + r_ * kMoveCountStride];                                           \
    const uint32_t base_ = r_ * (plan)[kPlanCap];                                                             \
    const uint32_t step_ = (gridDim.x / (uint32_t)kMoveLists) * kIncWG;                                       \
    for (uint32_t q_ = (blockIdx.x / (uint32_t)kMoveLists) * kIncWG + threadIdx.x, j = base_ + q_; q_ < c_; \
         q_ += step_, j = base_ + q_)

// Each list entry's old position marked, and the entry put into its tile's
// bucket (its counter in a line of its own: atomics on one line wait for each
// other).  The tiles' net change is counted apart, and only for the entries
// that leave their tile, which about three in four do not: counted for all of
// them in one word with the bucket's, a batch of 11.0M particles took 52 us
// here, 31 now, the grid clear beside it.
__global__ void __launch_bounds__(kIncWG) k_inc_route(uint32_t* __restrict__ plan, MoveList L,
                                                      const uint32_t* __restrict__ snap_k,
                                                      const uint32_t* __restrict__ snap_p, uint32_t tiles) {
    if (!plan_incremental(plan)) return;
    FOR_LIST_ENTRIES(plan, j) {
        const uint32_t k = L.key[j], s = L.slot[j], pos = L.pos[j];
        atomicOr(&L.gone[pos >> 5], 1u << (pos & 31u));
        uint32_t lo = 0, hi = tiles;  // the last tile whose first entry is not above (k, s)
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            const size_t i = (size_t)mid * kIncTile;
            if (entry_less(k, s, snap_k[i], snap_p[i])) hi = mid;
            else lo = mid;
        }
        const uint32_t from = pos / (uint32_t)kIncTile;
        if (from != lo) {
            atomicAdd(&L.tnet[from], ~0u);
            atomicAdd(&L.tnet[lo], 1u);
        }
        uint2* const bucket = L.ins + (size_t)lo * kIncBucket;
        const uint32_t q = atomicAdd(&bucket->x, 1u);
        if (q < (uint32_t)kIncStage) bucket[kIncBucket - kIncStage + q] = uint2{k, s};
        else plan[kPlanOverflow] = 1u;
    }
}

// The net change of the tiles before each tile, by one workgroup: for more
// than kSumTiles tiles (below, the merge's workgroups add up the tiles before
// them themselves: one launch less, at most 16 loads a thread).
constexpr uint32_t kSumTiles = 8192;
__global__ void __launch_bounds__(kScanWG) k_inc_offsets(const uint32_t* __restrict__ plan, MoveList L,
                                                         uint32_t tiles) {
    if (!plan_incremental(plan)) return;
    __shared__ uint32_t ws[kScanWG / 64];
    uint32_t before = 0;
    for (uint32_t t0 = 0; t0 < tiles; t0 += kScanTile) {
        uint32_t v[kScanIPT], sum = 0;
#pragma unroll
        for (int r = 0; r < kScanIPT; ++r) {
            const uint32_t t = t0 + threadIdx.x * kScanIPT + r;
            v[r] = t < tiles ? L.tnet[t] : 0u;
            sum += v[r];
        }
        uint32_t tot;
        uint32_t run = before + block_exclusive_scan(sum, ws, tot);
#pragma unroll
        for (int r = 0; r < kScanIPT; ++r) {
            const uint32_t t = t0 + threadIdx.x * kScanIPT + r;
            if (t < tiles) L.tbase[t] = run;
            run += v[r];
        }
        before += tot;
    }
}

constexpr int kTileIPT = 4;  // entries per thread of the tiles below

// Number of tile entries below (key, slot).
__device__ __forceinline__ uint32_t place_in_tile(const uint32_t* sk, const uint32_t* sp, uint32_t cnt, uint32_t k,
                                                  uint32_t s) {
    uint32_t lo = 0, hi = cnt;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (entry_less(sk[mid], sp[mid], k, s)) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// Number of entries of a[0..n) (ascending) that are < v.
__device__ __forceinline__ uint32_t count_below(const uint32_t* a, uint32_t n, uint32_t v) {
    uint32_t lo = 0, hi = n;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (a[mid] < v) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// One snapshot tile per workgroup, its entries in registers (and in LDS for
// the search of the places); it also clears the tile's marks and bucket
// for the next step (on a step that the update does not run too: after an overflow some
// are left).  The few insertions are ranked by counting, so that an entry
// finds its shift by one popcount and a search among the places.  tbase:
// where k_inc_offsets has run, else null.
__global__ void __launch_bounds__(kIncTile / kTileIPT) k_inc_merge(const uint32_t* __restrict__ plan, MoveList L,
                                                                   const uint32_t* __restrict__ snap_k,
                                                                   const uint32_t* __restrict__ snap_p, uint32_t n,
                                                                   const uint32_t* __restrict__ tbase,
                                                                   uint32_t* __restrict__ out_k,
                                                                   uint32_t* __restrict__ out_p) {
    constexpr int WG = kIncTile / kTileIPT, WORDS = kIncTile / 32;
    static_assert(WORDS == 64, "the marks of a tile are scanned by one wave");
    __shared__ uint32_t sk[kIncTile], sp[kIncTile];
    __shared__ uint32_t gone[WORDS + 1], gone_before[WORDS + 1];  // one more: the end of a full tile
    __shared__ uint32_t mk[kIncStage], ms[kIncStage], sorted[kIncStage];  // insertions; their places, ascending
    __shared__ uint32_t ws[WG / 64];
    const uint32_t t = blockIdx.x, tid = threadIdx.x;
    const uint32_t i0 = t * kIncTile, cnt = n - i0 < kIncTile ? n - i0 : kIncTile;
    uint32_t* const marks = L.gone + (size_t)t * WORDS;
    uint2* const bucket = L.ins + (size_t)t * kIncBucket;
    if (!plan_incremental(plan)) {
        if (tid < WORDS) marks[tid] = 0u;
        if (tid == 0) bucket->x = 0u;
        return;
    }
    const uint32_t drawn = bucket->x;  // at most kIncStage (else overflow)
    const uint32_t nm = drawn < (uint32_t)kIncStage ? drawn : (uint32_t)kIncStage;
    uint32_t key[kTileIPT], slot[kTileIPT];
#pragma unroll
    for (int r = 0; r < kTileIPT; ++r) {
        const uint32_t i = tid + r * WG, ic = i < cnt ? i : 0u;
        key[r] = snap_k[i0 + ic];
        slot[r] = snap_p[i0 + ic];
    }
    for (uint32_t q = tid; q < nm; q += WG) {
        const uint2 e = bucket[kIncBucket - kIncStage + q];
        mk[q] = e.x;
        ms[q] = e.y;
    }
    if (tid < WORDS) {  // one wave
        const uint32_t w = marks[tid];
        marks[tid] = 0u;
        uint32_t incl = (uint32_t)__popc(w);
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t up = __shfl_up(incl, off, 64);
            if ((int)tid >= off) incl += up;
        }
        gone[tid] = w;
        gone_before[tid] = incl - (uint32_t)__popc(w);
        if (tid == WORDS - 1) {
            gone[WORDS] = 0u;
            gone_before[WORDS] = incl;
        }
    }
    if (nm) {
#pragma unroll
        for (int r = 0; r < kTileIPT; ++r) {
            sk[tid + r * WG] = key[r];
            sp[tid + r * WG] = slot[r];
        }
    }
    uint32_t shift = 0;
    if (tbase) {
        shift = tbase[t];
        __syncthreads();
    } else {
        // eight loads in flight at a time: the sum is a latency, not work
        uint32_t part = 0;
        for (uint32_t q = tid; q < t; q += 8 * WG) {
            uint32_t c[8];
#pragma unroll
            for (uint32_t u = 0; u < 8; ++u) c[u] = L.tnet[q + u * WG < t ? q + u * WG : t];
#pragma unroll
            for (uint32_t u = 0; u < 8; ++u)
                if (q + u * WG < t) part += c[u];
        }
        block_exclusive_scan<WG>(part, ws, shift);
    }
    if (tid == 0) bucket->x = 0u;  // every thread has read it
    const uint32_t base = i0 + shift;
    auto removed = [&](uint32_t i) -> uint32_t {  // before position i of the tile
        return gone_before[i >> 5] + (uint32_t)__popc(gone[i >> 5] & ((1u << (i & 31u)) - 1u));
    };
    for (uint32_t q = tid; q < nm; q += WG) {
        const uint32_t k = mk[q], s = ms[q];
        const uint32_t l = place_in_tile(sk, sp, cnt, k, s);
        uint32_t rank = 0;  // (key, slot) order is also the order of the places
        for (uint32_t x = 0; x < nm; ++x) rank += entry_less(mk[x], ms[x], k, s) ? 1u : 0u;
        sorted[rank] = l;
        const uint32_t dst = base + l - removed(l) + rank;
        if (dst < n) {  // always, for a list that matches the snapshot
            out_k[dst] = k;
            out_p[dst] = s;
        }
    }
    if (nm) __syncthreads();  // uniform
#pragma unroll
    for (int r = 0; r < kTileIPT; ++r) {
        const uint32_t i = tid + r * WG;
        if (i >= cnt || ((gone[i >> 5] >> (i & 31u)) & 1u)) continue;
        const uint32_t dst = base + i - removed(i) + count_below(sorted, nm, i + 1u);  // places <= i
        if (dst < n) {
            out_k[dst] = key[r];
            out_p[dst] = slot[r];
        }
    }
}

// ------------------------------------------------------------ small scenes
// The same update in one launch.  A small scene's step is a chain of short
// launches, so here every workgroup reads the whole move list (a few percent
// of the particles) and keeps what falls into its tile, instead of passes
// that bucket the list first: the removals and insertions before the tile
// give its offset, a scan over the tile's positions the place of every entry
// in it.  Up to kMatch insertions are ranked in LDS by counting; more (a layer
// of a lattice that crosses cells in one step, a scene that loses its numbers
// in one) are sorted in memory by the tile's workgroup.  The list holds every
// particle, so there is no overflow and no full sort to launch beside it.
// What bounds it: the list, read by every workgroup (12 bytes an entry, from
// L2), and the ranking of a tile's insertions; the host takes the radix sort
// instead where that is the shorter (see run_sort_small).  Measured at 16,384 particles: six radix launches of 41 us
// and their gaps and a grid clear of 5 us before, one of 8.6 us for both now.
// A tile of the last order in LDS, the positions taken out of it and what is
// put into it.
constexpr int kMatch = 512;  // insertions kept in LDS
struct TileLds {
    static constexpr int TILE = kUpdateTile;
    uint32_t sk[TILE], sp[TILE];
    uint32_t ins[TILE + 1];     // insertions at each place of the tile (TILE: after its last entry)
    uint32_t before[TILE + 1];  // removals (low 12 bits) and insertions before each place
    uint32_t gone[TILE / 32];   // removed positions
    union {
        struct {
            uint32_t mk[kMatch], ms[kMatch], place[kMatch];  // insertions and their places
        };
        struct {
            uint32_t run[TILE / kTileIPT / 64][256], at[256];  // of sort_insertions
        };
    };
    uint32_t nmatch, diff[2], ws[TILE / kTileIPT / 64];
    // where the unmoved entry at place l goes in the new order, less the
    // insertions at l; base: where the tile begins
    __device__ __forceinline__ uint32_t bucket(uint32_t base, uint32_t l) const {
        return base + l - (before[l] & 4095u) + (before[l] >> 12);
    }
};

// Counts the nm insertions in T.mk/T.ms into T.ins and scans the places.  Call
// it after a barrier; ends with T complete for every thread.
__device__ __forceinline__ void scan_places(TileLds& T, uint32_t cnt, uint32_t nm) {
    constexpr int TILE = TileLds::TILE, IPT = kTileIPT, WG = TILE / IPT;
    static_assert(TILE <= 2048, "removals of a tile take 12 bits of `before`");
    const uint32_t tid = threadIdx.x;
    for (uint32_t q = tid; q < nm; q += WG) {
        T.place[q] = place_in_tile(T.sk, T.sp, cnt, T.mk[q], T.ms[q]);
        atomicAdd(&T.ins[T.place[q]], 1u);
    }
    __syncthreads();
    // thread tid scans places IPT * tid ..
    uint32_t d[IPT], c[IPT];
    uint32_t ds = 0, is = 0, dsum, isum;
#pragma unroll
    for (int r = 0; r < IPT; ++r) {
        const uint32_t i = tid * IPT + r;
        d[r] = ds;
        c[r] = is;
        ds += (T.gone[i >> 5] >> (i & 31u)) & 1u;
        is += T.ins[i];
    }
    const uint32_t dpre = block_exclusive_scan<WG>(ds, T.ws, dsum);
    const uint32_t ipre = block_exclusive_scan<WG>(is, T.ws, isum);
#pragma unroll
    for (int r = 0; r < IPT; ++r) T.before[tid * IPT + r] = (dpre + d[r]) | ((ipre + c[r]) << 12);
    if (tid == 0) T.before[TILE] = dsum | (isum << 12);
    __syncthreads();
}
// The tile's unmoved entries; base: where the tile begins in the new order.
__device__ __forceinline__ void put_unmoved(const TileLds& T, uint32_t cnt, uint32_t n, uint32_t base,
                                            uint32_t* __restrict__ out_k, uint32_t* __restrict__ out_p) {
#pragma unroll
    for (int r = 0; r < kTileIPT; ++r) {
        const uint32_t i = threadIdx.x + r * (TileLds::TILE / kTileIPT);
        if (i >= cnt || ((T.gone[i >> 5] >> (i & 31u)) & 1u)) continue;
        const uint32_t dst = T.bucket(base, i) + T.ins[i];
        if (dst < n) {  // always, for a list that matches the snapshot
            out_k[dst] = T.sk[i];
            out_p[dst] = T.sp[i];
        }
    }
}
// The nm insertions themselves, ranked among those at the same place.
__device__ __forceinline__ void put_inserted(const TileLds& T, uint32_t nm, uint32_t n, uint32_t base,
                                             uint32_t* __restrict__ out_k, uint32_t* __restrict__ out_p) {
    for (uint32_t q = threadIdx.x; q < nm; q += TileLds::TILE / kTileIPT) {
        const uint32_t k = T.mk[q], s = T.ms[q], l = T.place[q];
        uint32_t rank = 0;
        if (T.ins[l] > 1u)
            for (uint32_t x = 0; x < nm; ++x) rank += T.place[x] == l && entry_less(T.mk[x], T.ms[x], k, s) ? 1u : 0u;
        const uint32_t dst = T.bucket(base, l) + rank;
        if (dst < n) {
            out_k[dst] = k;
            out_p[dst] = s;
        }
    }
}

// The m entries at (ak, ap) sorted by (key, slot) by one workgroup: a stable
// pass per byte that is not the same in all of them, ping-pong with (bk, bp).
// Returns whether the result is in (ak, ap).  Ends with a barrier.
// Ranked by counting instead, every entry against all others at its place,
// the time grew with the square (10,000 entries 58 ms, 40,000 0.93 s; now the
// step that has them takes 0.22 and 0.68 ms): a layer of 4,096 particles made
// its step of 60 us one of 14 ms.
__device__ bool sort_insertions(TileLds& T, uint32_t* ak, uint32_t* ap, uint32_t* bk, uint32_t* bp, uint32_t m) {
    constexpr uint32_t IPT = kTileIPT, WAVES = TileLds::TILE / kTileIPT / 64, CHUNK = TileLds::TILE;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    if (tid < 2u) T.diff[tid] = 0u;
    __syncthreads();
    const uint32_t k0 = ak[0], s0 = ap[0];
    uint32_t dk = 0, ds = 0;
    for (uint32_t q = tid; q < m; q += WAVES * 64u) {
        dk |= ak[q] ^ k0;
        ds |= ap[q] ^ s0;
    }
    if (dk) atomicOr(&T.diff[0], dk);
    if (ds) atomicOr(&T.diff[1], ds);
    __syncthreads();
    dk = T.diff[0];
    ds = T.diff[1];
    bool in_a = true;
    for (int byte = 0; byte < 8; ++byte) {  // of the slot, then of the key
        const int shift = 8 * (byte & 3);
        if ((((byte < 4 ? ds : dk) >> shift) & 255u) == 0u) continue;  // uniform
        const uint32_t *ik = in_a ? ak : bk, *ip = in_a ? ap : bp;
        uint32_t *ok = in_a ? bk : ak, *op = in_a ? bp : ap;
        const uint32_t* const word = byte < 4 ? ip : ik;
        // at: where each digit's next entry goes
        static_assert(WAVES * 64u == 256u, "a thread per digit");
        T.at[tid] = 0u;
        __syncthreads();
        for (uint32_t q = tid; q < m; q += 256u) atomicAdd(&T.at[(word[q] >> shift) & 255u], 1u);
        __syncthreads();
        uint32_t all;
        const uint32_t first = block_exclusive_scan<256>(T.at[tid], T.ws, all);
        T.at[tid] = first;
        // a wave takes 4 x 64 consecutive entries of a chunk; run: its count
        // of each digit so far, then where its first of the digit goes
        for (uint32_t c0 = 0; c0 < m; c0 += CHUNK) {
#pragma unroll
            for (uint32_t w = 0; w < WAVES; ++w) T.run[w][tid] = 0u;
            __syncthreads();
            uint32_t k[IPT], s[IPT], d[IPT], rank[IPT];
#pragma unroll
            for (uint32_t r = 0; r < IPT; ++r) {
                const uint32_t q = c0 + (wave * IPT + r) * 64u + lane, qc = q < m ? q : m - 1u;
                k[r] = ik[qc];
                s[r] = ip[qc];
            }
#pragma unroll
            for (uint32_t r = 0; r < IPT; ++r) {
                const bool valid = c0 + (wave * IPT + r) * 64u + lane < m;
                d[r] = ((byte < 4 ? s[r] : k[r]) >> shift) & 255u;
                uint64_t same = __ballot(valid);
#pragma unroll
                for (int b = 0; b < 8; ++b) {
                    const uint64_t set = __ballot((d[r] >> b) & 1u);
                    same &= (d[r] >> b) & 1u ? set : ~set;
                }
                const uint32_t before = (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
                rank[r] = before + (valid ? T.run[wave][d[r]] : 0u);
                asm volatile("" ::: "memory");  // a wave's LDS accesses are in order
                if (valid && before == 0u) T.run[wave][d[r]] += (uint32_t)__popcll(same);
                asm volatile("" ::: "memory");
            }
            __syncthreads();
            uint32_t to = T.at[tid];
#pragma unroll
            for (uint32_t w = 0; w < WAVES; ++w) {
                const uint32_t c = T.run[w][tid];
                T.run[w][tid] = to;
                to += c;
            }
            T.at[tid] = to;
            __syncthreads();
#pragma unroll
            for (uint32_t r = 0; r < IPT; ++r) {
                if (c0 + (wave * IPT + r) * 64u + lane >= m) continue;
                const uint32_t dst = T.run[wave][d[r]] + rank[r];
                ok[dst] = k[r];
                op[dst] = s[r];
            }
            __syncthreads();
        }
        in_a = !in_a;
    }
    return in_a;
}

// Clear of the touched blocks of a grid, one group of blocks per wave.
__device__ __forceinline__ void clear_blocks(const GridClear& C, int64_t wave) {
    const int lane = threadIdx.x & 63;
    const int64_t b0 = wave * kClearGroup;
    const uint32_t todo = (uint32_t)__ballot(lane < kClearGroup && b0 + lane < C.nsb && C.touched[b0 + lane] != 0u);
    if (!todo) return;
    const unsigned long long cnt =
        clear_group(C.grid, C.plane, C.touched, b0, todo, C.nfields, lane, C.active != nullptr);
    if (C.active && cnt && lane == 0) atomicAdd(C.active, cnt);
}

__global__ void __launch_bounds__(kIncWG) k_sort_update(const uint32_t* __restrict__ plan, MoveList L,
                                                        const uint32_t* __restrict__ snap_k,
                                                        const uint32_t* __restrict__ snap_p, uint32_t n,
                                                        uint32_t tiles, uint32_t* out_k, uint32_t* out_p,
                                                        uint32_t* tmp_k,
                                                        uint32_t* tmp_p, GridClear C) {
    if (blockIdx.x >= tiles) {
        clear_blocks(C, (int64_t)(blockIdx.x - tiles) * (kIncWG / 64) + (threadIdx.x >> 6));
        return;
    }
    constexpr int TILE = kUpdateTile, IPT = kTileIPT;
    static_assert(TILE == kIncWG * IPT);
    __shared__ TileLds T;
    uint32_t (&sk)[TILE] = T.sk, (&sp)[TILE] = T.sp, (&ins)[TILE + 1] = T.ins;
    const uint32_t t = blockIdx.x, tid = threadIdx.x;
    const uint32_t i0 = t * TILE, cnt = n - i0 < TILE ? n - i0 : TILE;
    const bool last = t + 1 == tiles;
#pragma unroll
    for (int r = 0; r < IPT; ++r) {
        const uint32_t i = tid + r * kIncWG;
        if (i < cnt) {
            sk[i] = snap_k[i0 + i];
            sp[i] = snap_p[i0 + i];
        }
        ins[i] = 0u;
    }
    if (tid < TILE / 32) T.gone[tid] = 0u;
    if (tid == 0) {
        ins[TILE] = 0u;
        T.nmatch = 0u;
    }
    const uint32_t nk = last ? 0u : snap_k[i0 + TILE], np = last ? 0u : snap_p[i0 + TILE];
    __syncthreads();
    const uint32_t fk = sk[0], fp = sp[0];
    // whether (k, s) goes into this tile: -1 an earlier one, 0 this, 1 a later one
    auto side = [&](uint32_t k, uint32_t s) -> int {
        if (t > 0 && entry_less(k, s, fk, fp)) return -1;
        return !last && !entry_less(k, s, nk, np) ? 1 : 0;
    };
    // every list entry, once over the workgroup: a wave takes four sub-lists
    // side by side (their loads in flight together), then all take what did
    // not fit into them
    const uint32_t cap = small_list_cap(n);
    constexpr uint32_t WAVES = kIncWG / 64, OWN = kSmallLists / WAVES;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63u;
    const uint32_t spilled = plan[kPlanLists + kSmallLists * kMoveCountStride];
    uint32_t own[OWN], longest = 0;
#pragma unroll
    for (uint32_t u = 0; u < OWN; ++u) {
        const uint32_t c = plan[kPlanLists + (wave + u * WAVES) * kMoveCountStride];
        own[u] = c < cap ? c : cap;
        longest = own[u] > longest ? own[u] : longest;
    }
    auto for_list = [&](auto&& fn) {
        for (uint32_t q = lane; q < longest; q += 64u) {
            uint32_t k[OWN], s[OWN], pos[OWN];
#pragma unroll
            for (uint32_t u = 0; u < OWN; ++u) {
                const uint32_t j = (wave + u * WAVES) * cap + q;
                if (q < own[u]) {
                    k[u] = L.key[j];
                    s[u] = L.slot[j];
                    pos[u] = L.pos[j];
                }
            }
#pragma unroll
            for (uint32_t u = 0; u < OWN; ++u)
                if (q < own[u]) fn(k[u], s[u], pos[u]);
        }
        for (uint32_t q = tid; q < spilled; q += kIncWG) {
            const uint32_t j = kSmallLists * cap + q;
            fn(L.key[j], L.slot[j], L.pos[j]);
        }
    };
    uint32_t db = 0, ib = 0;
    for_list([&](uint32_t k, uint32_t s, uint32_t pos) {
        if (pos < i0) ++db;
        else if (pos - i0 < cnt) atomicOr(&T.gone[(pos - i0) >> 5], 1u << ((pos - i0) & 31u));
        const int w = side(k, s);
        if (w < 0) ++ib;
        if (w == 0) {
            const uint32_t q = atomicAdd(&T.nmatch, 1u);
            if (q < kMatch) {
                T.mk[q] = k;
                T.ms[q] = s;
            } else {
                atomicAdd(&ins[place_in_tile(sk, sp, cnt, k, s)], 1u);
            }
        }
    });
    __syncthreads();
    const uint32_t nm = T.nmatch;
    uint32_t dtot, itot;
    block_exclusive_scan(db, T.ws, dtot);
    block_exclusive_scan(ib, T.ws, itot);
    const uint32_t base = i0 - dtot + itot;
    scan_places(T, cnt, nm < kMatch ? nm : kMatch);
    if (nm <= (uint32_t)kMatch) {  // uniform
        put_unmoved(T, cnt, n, base, out_k, out_p);
        put_inserted(T, nm, n, base, out_k, out_p);
        return;
    }
    // more: gathered in arbitrary order and sorted in the tile's part of the
    // new order, in scratch and in the output (nothing else is there yet).
    // The places ascend with the entries, so entry q goes to its place less
    // the removals before it plus q.
    if (base > n || nm > n - base) return;  // never, for a list that matches the snapshot
    if (tid == 0) T.nmatch = 0u;
    __syncthreads();
    for_list([&](uint32_t k, uint32_t s, uint32_t) {
        if (side(k, s) != 0) return;
        const uint32_t q = base + atomicAdd(&T.nmatch, 1u);
        tmp_k[q] = k;
        tmp_p[q] = s;
    });
    __syncthreads();
    const bool in_tmp = sort_insertions(T, tmp_k + base, tmp_p + base, out_k + base, out_p + base, nm);
    if (!in_tmp) {
        for (uint32_t q = tid; q < nm; q += kIncWG) {
            tmp_k[base + q] = out_k[base + q];
            tmp_p[base + q] = out_p[base + q];
        }
        __syncthreads();
    }
    put_unmoved(T, cnt, n, base, out_k, out_p);
    for (uint32_t q = tid; q < nm; q += kIncWG) {
        const uint32_t k = tmp_k[base + q], s = tmp_p[base + q], l = place_in_tile(sk, sp, cnt, k, s);
        const uint32_t dst = base + l - (T.before[l] & 4095u) + q;
        if (dst < n) {
            out_k[dst] = k;
            out_p[dst] = s;
        }
    }
}

__global__ void k_update_init(uint32_t* plan, MoveList* dev, MoveList L) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < (uint32_t)kPlanWords) plan[i] = 0u;
    if (i == 0u) *dev = L;
}
void launch_update_init(uint32_t* plan, MoveList* dev, const MoveList& L, hipStream_t st) {
    hipLaunchKernelGGL(k_update_init, dim3((kPlanWords + 255) / 256), dim3(256), 0, st, plan, dev, L);
}

void launch_sort_update(const uint32_t* plan, const MoveList& L, const uint32_t* snap_k, const uint32_t* snap_p,
                        int64_t n, uint32_t* out_k, uint32_t* out_p, uint32_t* tmp_k, uint32_t* tmp_p,
                        const GridClear& clear, hipStream_t st) {
    const uint32_t tiles = (uint32_t)((n + kUpdateTile - 1) / kUpdateTile);
    const int64_t waves = (clear.nsb + kClearGroup - 1) / kClearGroup;
    const uint32_t extra = (uint32_t)((waves + kIncWG / 64 - 1) / (kIncWG / 64));
    hipLaunchKernelGGL(k_sort_update, dim3(tiles + extra), dim3(kIncWG), 0, st, plan, L, snap_k, snap_p, (uint32_t)n,
                       tiles, out_k, out_p, tmp_k, tmp_p, clear);
}

uint32_t inc_tiles(int64_t n) { return (uint32_t)((n + kIncTile - 1) / kIncTile); }

void launch_inc_set(uint32_t* plan, uint32_t snap_ok, hipStream_t st) {
    hipLaunchKernelGGL(k_inc_set, dim3(1), dim3(64), 0, st, plan, snap_ok);
}

void launch_inc_prepare(uint32_t* plan, const MoveList& L, const uint32_t* snap_k, const uint32_t* snap_p, int64_t n,
                        hipStream_t st) {
    if (n <= 0) return;
    // 16 workgroups per sub-list
    hipLaunchKernelGGL(k_inc_route, dim3(16 * kMoveLists), dim3(kIncWG), 0, st, plan, L, snap_k, snap_p,
                       inc_tiles(n));
}

void launch_inc_merge(const uint32_t* plan, const MoveList& L, const uint32_t* snap_k, const uint32_t* snap_p,
                      int64_t n, uint32_t* out_k, uint32_t* out_p, hipStream_t st) {
    if (n <= 0) return;
    const uint32_t tiles = inc_tiles(n);
    const bool scanned = tiles > kSumTiles;
    if (scanned) hipLaunchKernelGGL(k_inc_offsets, dim3(1), dim3(kScanWG), 0, st, plan, L, tiles);
    hipLaunchKernelGGL(k_inc_merge, dim3(tiles), dim3(kIncTile / kTileIPT), 0, st, plan, L, snap_k, snap_p,
                       (uint32_t)n, scanned ? (const uint32_t*)L.tbase : nullptr, out_k, out_p);
}

}  // namespace mpm
