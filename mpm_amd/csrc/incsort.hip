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
//   * here every list entry finds its place among the snapshot (lb: the
//     number of snapshot entries before it in (key, slot) order) by a binary
//     search, and the removed positions and insertion places are bucketed
//     by snapshot tile (counts, one scan, then an append per entry);
//   * one pass over the snapshot tiles finishes the job: each workgroup
//     ranks its tile's few removals and insertions in LDS and writes every
//     unmoved entry at i - (removed before i) + (inserted at or before i)
//     and every inserted entry at lb - (removed before lb) + (inserted
//     before it).
// The result is bit-identical to a stable radix sort of the new keys.  The
// device-side plan words pick this path or the full radix sort each step
// (the other path's launches return at once): the full sort runs when the
// list overflowed, a tile drew more entries than its merge stages, or the
// snapshot is not the previous step's (first step, state written, a
// single scene's store reordered, a batch's layout changed).  The step's item count resets the words afterwards
// (launch_items with plan).  Launch order within a step: launch_inc_prepare,
// the radix sort (which reads the decision), launch_inc_merge.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "blockscan.h"
#include "launch.h"

namespace mpm {

constexpr int kIncWG = 256;

// (key, slot) order of two sort entries.
__device__ __forceinline__ bool entry_less(uint32_t ka, uint32_t sa, uint32_t kb, uint32_t sb) {
    return ka < kb || (ka == kb && sa < sb);
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

// Each list entry's place among the snapshot, by binary search (a chain
// of dependent loads, the entries all in flight at once; in a batch within
// the entry's member), and the tile counts of its old position and of its
// place (zero on entry: the merge clears them after use).
__global__ void __launch_bounds__(kIncWG) k_inc_locate(const uint32_t* __restrict__ plan, MoveList L,
                                                       const uint32_t* __restrict__ snap_k,
                                                       const uint32_t* __restrict__ snap_p, int64_t n,
                                                       uint32_t tiles) {
    if (!plan_incremental(plan)) return;
    FOR_LIST_ENTRIES(plan, j) {
        const uint32_t k = L.key[j], s = L.slot[j];
        uint32_t lo = 0, hi = (uint32_t)n;  // the place lies in [lo, hi]
        if (L.nranges) {  // a batch: within its member's range (a short search in a cached table first)
            uint32_t a = 0, b = L.nranges;
            while (b - a > 1) {
                const uint32_t mid = (a + b) >> 1;
                if (L.range_start[mid] <= s) a = mid;
                else b = mid;
            }
            lo = L.range_start[a];
            hi = L.range_start[a + 1];
        }
        while (lo < hi) {
            const uint32_t mid = lo + ((hi - lo) >> 1);
            if (entry_less(snap_k[mid], snap_p[mid], k, s)) lo = mid + 1;
            else hi = mid;
        }
        L.lb[j] = lo;
        atomicAdd(&L.tcount[L.pos[j] / (uint32_t)kIncTile], 1u);
        atomicAdd(&L.tcount[tiles + 1u + lo / (uint32_t)kIncTile], 1u);
    }
}

// Bucket offsets: exclusive scans of the two count arrays (tiles + 1
// entries each) into the bucket cursors, by one workgroup per array (each
// thread a run of consecutive counts); a tile with more entries than the
// merge stages sends this step to the full sort.
__global__ void __launch_bounds__(kScanWG) k_inc_offsets(uint32_t* __restrict__ plan, MoveList L, uint32_t tiles) {
    if (!plan_incremental(plan)) return;
    __shared__ uint32_t ws[kScanWG / 64];
    const uint32_t m = tiles + 1u;
    const uint32_t* const cnt = L.tcount + (size_t)blockIdx.x * m;
    uint32_t* const cur = L.tnext + (size_t)blockIdx.x * m;
    const uint32_t per = (m + kScanWG - 1) / kScanWG;
    const uint32_t t0 = threadIdx.x * per < m ? threadIdx.x * per : m;
    const uint32_t t1 = t0 + per < m ? t0 + per : m;
    uint32_t sum = 0;
    bool over = false;
    for (uint32_t t = t0; t < t1; ++t) {
        const uint32_t v = cnt[t];
        over = over || v > (uint32_t)kIncStage;
        sum += v;
    }
    uint32_t tot;
    uint32_t run = block_exclusive_scan(sum, ws, tot);
    for (uint32_t t = t0; t < t1; ++t) {
        cur[t] = run;
        run += cnt[t];
    }
    if (over) plan[kPlanOverflow] = 1u;
}

// Each entry's old position and entry index appended to the buckets of
// their tiles (the order inside a bucket is arbitrary: the merge ranks it).
__global__ void __launch_bounds__(kIncWG) k_inc_bucket(const uint32_t* __restrict__ plan, MoveList L,
                                                       uint32_t tiles) {
    if (!plan_incremental(plan)) return;
    FOR_LIST_ENTRIES(plan, j) {
        const uint32_t pos = L.pos[j], lb = L.lb[j];
        L.del_b[atomicAdd(&L.tnext[pos / (uint32_t)kIncTile], 1u)] = pos;
        L.ins_b[atomicAdd(&L.tnext[tiles + 1u + lb / (uint32_t)kIncTile], 1u)] = j;
    }
}

// One snapshot tile [i0, i1) per workgroup (the last one, past n when n is
// a multiple of the tile, takes the insertions at n); it also zeroes the
// tile's counts, also on a step the update does not run (after an overflow
// the counts are left over).  After the bucketing
// the cursors sit at the end of each bucket, so a bucket starts at
// cursor - count.  Removed positions are distinct and list entries have
// distinct (key, slot), so ranking by counting gives each its own place.
__global__ void __launch_bounds__(kIncWG) k_inc_merge(const uint32_t* __restrict__ plan, MoveList L,
                                                      const uint32_t* __restrict__ snap_k,
                                                      const uint32_t* __restrict__ snap_p, int64_t n, uint32_t tiles,
                                                      uint32_t* __restrict__ out_k, uint32_t* __restrict__ out_p) {
    const uint32_t t = blockIdx.x;
    if (!plan_incremental(plan)) {  // an overflow after the counting: clear them for the next step
        if (threadIdx.x == 0) {
            L.tcount[t] = 0u;
            L.tcount[tiles + 1u + t] = 0u;
        }
        return;
    }
    __shared__ uint32_t dr[kIncStage], sdel[kIncStage];              // removed positions: as bucketed, ascending
    __shared__ uint32_t ir[kIncStage], ik[kIncStage], is[kIncStage];  // insertions: place, key, slot
    __shared__ uint32_t slb[kIncStage];                                // insertion places, ascending
    const int64_t i0 = (int64_t)t * kIncTile;
    const int64_t i1 = i0 + kIncTile < n ? i0 + kIncTile : n;
    const uint32_t dc = L.tcount[t], rc = L.tcount[tiles + 1u + t];  // <= kIncStage (else overflow)
    const uint32_t d0 = L.tnext[t] - dc, r0 = L.tnext[tiles + 1u + t] - rc;
    for (uint32_t q = threadIdx.x; q < dc; q += kIncWG) dr[q] = L.del_b[d0 + q];
    for (uint32_t q = threadIdx.x; q < rc; q += kIncWG) {
        const uint32_t j = L.ins_b[r0 + q];
        ir[q] = L.lb[j];
        ik[q] = L.key[j];
        is[q] = L.slot[j];
    }
    __syncthreads();  // every thread has read the counts
    if (threadIdx.x == 0) {  // zero for the next step's counting
        L.tcount[t] = 0u;
        L.tcount[tiles + 1u + t] = 0u;
    }
    for (uint32_t q = threadIdx.x; q < dc; q += kIncWG) {
        const uint32_t v = dr[q];
        uint32_t r = 0;
        for (uint32_t x = 0; x < dc; ++x) r += dr[x] < v ? 1u : 0u;
        sdel[r] = v;
    }
    __syncthreads();
    for (uint32_t q = threadIdx.x; q < rc; q += kIncWG) {
        const uint32_t k = ik[q], s = is[q], lb = ir[q];
        uint32_t r = 0;  // (key, slot) order is also the order of the places
        for (uint32_t x = 0; x < rc; ++x) r += entry_less(ik[x], is[x], k, s) ? 1u : 0u;
        slb[r] = lb;
        const uint32_t dst = lb - (d0 + count_below(sdel, dc, lb)) + r0 + r;
        if ((int64_t)dst < n) {  // always, for a list that matches the snapshot
            out_k[dst] = k;
            out_p[dst] = s;
        }
    }
    __syncthreads();
    // consecutive lanes take consecutive entries: loads and (shifted) stores stay contiguous
    for (int64_t i = i0 + threadIdx.x; i < i1; i += kIncWG) {
        const uint32_t iu = (uint32_t)i;
        const uint32_t dl = count_below(sdel, dc, iu);
        if (dl < dc && sdel[dl] == iu) continue;  // moved
        const uint32_t dst = iu - (d0 + dl) + r0 + count_below(slb, rc, iu + 1u);  // places <= i
        if ((int64_t)dst < n) {
            out_k[dst] = snap_k[i];
            out_p[dst] = snap_p[i];
        }
    }
}

// ------------------------------------------------------------ small scenes
// The same update in one launch.  A small scene's step is a chain of short
// launches, so here every workgroup reads the whole move list (a few percent
// of the particles) and keeps what falls into its tile, instead of passes
// that bucket the list first: the removals and insertions before the tile
// give its offset, a scan over the tile's positions the place of every entry
// in it.  Insertions at one place are put into scratch in arbitrary order,
// then ranked among themselves.  The list holds every particle, so there is
// no overflow and no full sort to launch beside it.
// What bounds it: the list's entries times the tiles (12 bytes each, from
// L2); the host takes the radix sort instead where that is the larger (see
// run_sort_small).  Measured at 16,384 particles: six radix launches of 41 us
// and their gaps and a grid clear of 5 us before, one of 8.6 us for both now.
constexpr int kMatch = 512;  // of a tile's insertions, those kept in LDS

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

// Clear of the touched blocks of a grid, 8 consecutive blocks per wave.
__device__ __forceinline__ void clear_blocks(const GridClear& C, int64_t wave) {
    const int lane = threadIdx.x & 63;
    const int64_t b0 = wave * 8;
    uint64_t todo = __ballot(lane < 8 && b0 + lane < C.nsb && C.touched[b0 + lane] != 0u);
    unsigned long long cnt = 0;
    while (todo) {
        const int64_t b = b0 + __builtin_ctzll(todo);
        todo &= todo - 1;
        const int64_t ni = b * 64 + lane;
        cnt += (unsigned long long)__popcll(__ballot(C.grid[ni] > 0.0f));
        for (int f = 0; f < C.nfields; ++f) C.grid[(int64_t)f * C.plane + ni] = 0.0f;
        if (lane == 0) C.touched[b] = 0u;
    }
    if (C.active && cnt && lane == 0) atomicAdd(C.active, cnt);
}

__global__ void __launch_bounds__(kIncWG) k_sort_update(const uint32_t* __restrict__ plan, MoveList L,
                                                        const uint32_t* __restrict__ snap_k,
                                                        const uint32_t* __restrict__ snap_p, uint32_t n,
                                                        uint32_t tiles, uint32_t* __restrict__ out_k,
                                                        uint32_t* __restrict__ out_p, uint32_t* tmp_k,
                                                        uint32_t* tmp_p, GridClear C) {
    if (blockIdx.x >= tiles) {
        clear_blocks(C, (int64_t)(blockIdx.x - tiles) * (kIncWG / 64) + (threadIdx.x >> 6));
        return;
    }
    constexpr int TILE = kUpdateTile, IPT = TILE / kIncWG;
    __shared__ uint32_t sk[TILE], sp[TILE];
    __shared__ uint32_t ins[TILE + 1];        // insertions at each place of the tile (TILE: after its last entry)
    __shared__ uint32_t before[TILE + 1];     // removals (low 11 bits) and insertions before each place
    __shared__ uint32_t gone[TILE / 32];      // removed positions
    __shared__ uint32_t mk[kMatch], ms[kMatch], place[kMatch];  // the tile's insertions and their places
    __shared__ uint32_t nmatch, ws[kIncWG / 64];
    static_assert(TILE <= 1024, "removals of a tile take 11 bits of `before`");
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
    if (tid < TILE / 32) gone[tid] = 0u;
    if (tid == 0) {
        ins[TILE] = 0u;
        nmatch = 0u;
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
        else if (pos - i0 < cnt) atomicOr(&gone[(pos - i0) >> 5], 1u << ((pos - i0) & 31u));
        const int w = side(k, s);
        if (w < 0) ++ib;
        if (w == 0) {
            const uint32_t q = atomicAdd(&nmatch, 1u);
            if (q < kMatch) {
                mk[q] = k;
                ms[q] = s;
            } else {
                atomicAdd(&ins[place_in_tile(sk, sp, cnt, k, s)], 1u);
            }
        }
    });
    __syncthreads();
    const uint32_t nm = nmatch;
    for (uint32_t q = tid; q < (nm < kMatch ? nm : kMatch); q += kIncWG) {
        place[q] = place_in_tile(sk, sp, cnt, mk[q], ms[q]);
        atomicAdd(&ins[place[q]], 1u);
    }
    __syncthreads();
    uint32_t dtot, itot, dsum, isum;
    block_exclusive_scan(db, ws, dtot);
    block_exclusive_scan(ib, ws, itot);
    // thread tid scans places IPT * tid ..
    uint32_t d[IPT], c[IPT];
    uint32_t ds = 0, is = 0;
#pragma unroll
    for (int r = 0; r < IPT; ++r) {
        const uint32_t i = tid * IPT + r;
        d[r] = ds;
        c[r] = is;
        ds += (gone[i >> 5] >> (i & 31u)) & 1u;
        is += ins[i];
    }
    const uint32_t dpre = block_exclusive_scan(ds, ws, dsum);
    const uint32_t ipre = block_exclusive_scan(is, ws, isum);
#pragma unroll
    for (int r = 0; r < IPT; ++r) before[tid * IPT + r] = (dpre + d[r]) | ((ipre + c[r]) << 11);
    if (tid == 0) before[TILE] = dsum | (isum << 11);
    __syncthreads();
    const uint32_t base = i0 - dtot + itot;
    // first place in the new order of what is inserted at place l
    auto bucket = [&](uint32_t l) -> uint32_t { return base + l - (before[l] & 2047u) + (before[l] >> 11); };
#pragma unroll
    for (int r = 0; r < IPT; ++r) {
        const uint32_t i = tid + r * kIncWG;
        if (i >= cnt || ((gone[i >> 5] >> (i & 31u)) & 1u)) continue;
        const uint32_t dst = bucket(i) + ins[i];
        if (dst < n) {  // always, for a list that matches the snapshot
            out_k[dst] = sk[i];
            out_p[dst] = sp[i];
        }
    }
    if (nm == 0u) return;  // uniform
    __syncthreads();       // sk is free: from here on the bucket cursors
    uint32_t* const cur = sk;
#pragma unroll
    for (int r = 0; r < IPT; ++r) cur[tid + r * kIncWG] = 0u;
    // the places were found with sk; entries beyond kMatch need it again, so
    // their place is found in the snapshot in memory
    __shared__ uint32_t cur_last;
    if (tid == 0) cur_last = 0u;
    __syncthreads();
    auto for_matches = [&](auto&& fn) {
        if (nm <= kMatch) {
            for (uint32_t q = tid; q < nm; q += kIncWG) fn(mk[q], ms[q], place[q]);
        } else {
            for_list([&](uint32_t k, uint32_t s, uint32_t) {
                if (side(k, s) == 0) fn(k, s, place_in_tile(snap_k + i0, snap_p + i0, cnt, k, s));
            });
        }
    };
    for_matches([&](uint32_t k, uint32_t s, uint32_t l) {
        const uint32_t u = atomicAdd(l < TILE ? &cur[l] : &cur_last, 1u);
        const uint32_t dst = bucket(l) + u;
        if (dst >= n) return;
        uint32_t* const ok = ins[l] == 1u ? out_k : tmp_k;
        uint32_t* const op = ins[l] == 1u ? out_p : tmp_p;
        ok[dst] = k;
        op[dst] = s;
    });
    __syncthreads();
    for_matches([&](uint32_t k, uint32_t s, uint32_t l) {
        const uint32_t c0 = ins[l], b0 = bucket(l);
        if (c0 == 1u || b0 + c0 > n) return;
        uint32_t rank = 0;
        for (uint32_t u = 0; u < c0; ++u) rank += entry_less(tmp_k[b0 + u], tmp_p[b0 + u], k, s) ? 1u : 0u;
        out_k[b0 + rank] = k;
        out_p[b0 + rank] = s;
    });
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
    const int64_t waves = (clear.nsb + 7) / 8;
    const uint32_t extra = (uint32_t)((waves + kIncWG / 64 - 1) / (kIncWG / 64));
    hipLaunchKernelGGL(k_sort_update, dim3(tiles + extra), dim3(kIncWG), 0, st, plan, L, snap_k, snap_p, (uint32_t)n,
                       tiles, out_k, out_p, tmp_k, tmp_p, clear);
}

uint32_t inc_tiles(int64_t n) { return (uint32_t)(n / kIncTile + 1); }

void launch_inc_set(uint32_t* plan, uint32_t snap_ok, hipStream_t st) {
    hipLaunchKernelGGL(k_inc_set, dim3(1), dim3(64), 0, st, plan, snap_ok);
}

void launch_inc_prepare(uint32_t* plan, const MoveList& L, const uint32_t* snap_k, const uint32_t* snap_p, int64_t n,
                        hipStream_t st) {
    const uint32_t tiles = inc_tiles(n);
    // 16 workgroups per sub-list
    hipLaunchKernelGGL(k_inc_locate, dim3(16 * kMoveLists), dim3(kIncWG), 0, st, plan, L, snap_k, snap_p, n, tiles);
    hipLaunchKernelGGL(k_inc_offsets, dim3(2), dim3(kScanWG), 0, st, plan, L, tiles);
}

void launch_inc_merge(const uint32_t* plan, const MoveList& L, const uint32_t* snap_k, const uint32_t* snap_p,
                      int64_t n, uint32_t* out_k, uint32_t* out_p, hipStream_t st) {
    const uint32_t tiles = inc_tiles(n);
    hipLaunchKernelGGL(k_inc_bucket, dim3(16 * kMoveLists), dim3(kIncWG), 0, st, plan, L, tiles);
    hipLaunchKernelGGL(k_inc_merge, dim3(tiles), dim3(kIncWG), 0, st, plan, L, snap_k, snap_p, n, tiles, out_k,
                       out_p);
}

}  // namespace mpm
