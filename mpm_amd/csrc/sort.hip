// sort.hip -- stable LSD radix sort of (key, value) uint32 pairs and a
// device-wide exclusive scan, written for wave64 (gfx950).
//
// One pass over a digit (6 to 9 bits, planned by radix_passes) is three
// launches:
//   hist    : per-tile digit histogram, stored digit-major (digit * tiles + tile)
//   scan    : exclusive scan of that table -> global base of (digit, tile)
//   scatter : per-tile stable ranking (64-key chunks ranked with 8 ballots,
//             chunk prefix sums in LDS), staged in LDS in digit order, then
//             written out so that runs of one digit are contiguous stores.
// Stability follows from ranking by (tile, chunk, lane) = input order.
// A sort that mostly does not run (the plan words chose the incremental
// update) is one launch instead, which does all passes when it has to
// (k_radix_all).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "blockscan.h"
#include "launch.h"

namespace mpm {

constexpr int kMaxRadixBits = 9;
constexpr int kMaxRadix = 1 << kMaxRadixBits;
constexpr int kSortWG = 256;
constexpr int kSortIPT = 8;
constexpr int kSortTile = kSortWG * kSortIPT;  // 2048 keys per tile
constexpr int kSortChunks = kSortTile / 64;    // 32 chunks of 64 keys
constexpr int kChunksPerWave = kSortChunks / (kSortWG / 64);

template <int BITS>
__device__ __forceinline__ uint64_t digit_match(uint32_t digit, uint64_t active) {
    uint64_t m = active;
#pragma unroll
    for (int b = 0; b < BITS; ++b) {
        bool bit = (digit >> b) & 1u;
        uint64_t bb = __ballot(bit);
        m &= bit ? bb : ~bb;
    }
    return m;
}

// One tile's digit histogram.
template <int BITS>
__device__ __forceinline__ void hist_tile(const uint32_t* keys, int64_t n, int shift, uint32_t mask, uint32_t* hist,
                                          int64_t tiles, int64_t tile) {
    constexpr int kRadix = 1 << BITS;
    __shared__ uint32_t h[kRadix];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    for (int i = tid; i < kRadix; i += kSortWG) h[i] = 0;
    __syncthreads();
    const int64_t base = tile * kSortTile;
    // all of the wave's key loads are issued before the first is used
    uint32_t kk[kChunksPerWave];
#pragma unroll
    for (int c = 0; c < kChunksPerWave; ++c) {
        const int64_t idx = base + (int64_t)(wave * kChunksPerWave + c) * 64 + lane;
        kk[c] = idx < n ? keys[idx] : 0u;
    }
#pragma unroll
    for (int c = 0; c < kChunksPerWave; ++c) {
        const int64_t idx = base + (int64_t)(wave * kChunksPerWave + c) * 64 + lane;
        const bool valid = idx < n;
        const uint64_t active = __ballot(valid);
        if (active == 0) continue;  // wave-uniform: the tail of the last tile
        const uint32_t digit = (kk[c] >> shift) & mask;
        const uint64_t m = digit_match<BITS>(digit, active);
        const int leader = __ffsll((unsigned long long)m) - 1;
        if (valid && lane == leader) atomicAdd(&h[digit], (uint32_t)__popcll(m));
    }
    __syncthreads();
    for (int d = tid; d < kRadix; d += kSortWG) hist[(int64_t)d * tiles + tile] = h[d];
}
template <int BITS>
__global__ void __launch_bounds__(kSortWG) k_radix_hist(const uint32_t* __restrict__ keys, int64_t n, int shift,
                                                        uint32_t mask, uint32_t* __restrict__ hist, int64_t tiles,
                                                        const uint32_t* __restrict__ plan) {
    if (plan && plan_incremental(plan)) return;
    hist_tile<BITS>(keys, n, shift, mask, hist, tiles, blockIdx.x);
}

// Where a tile's digits begin in the output: in the scanned digit table, or
// summed up from the raw one (few tiles), or the digit's row of the table
// scanned by itself, with the rows' totals apart.
enum DigitBase { kScanned, kRaw, kRows };

// One tile of a pass, put in its place.
template <int BITS, DigitBase BASE>
__device__ __forceinline__ void scatter_tile(const uint32_t* keys_in, const uint32_t* vals_in, uint32_t* keys_out,
                                             uint32_t* vals_out, int64_t n, int shift, uint32_t mask,
                                             const uint32_t* hist_scan, const uint32_t* row_total, int64_t tiles,
                                             int64_t tile) {
    constexpr int kRadix = 1 << BITS;
    // digits per thread: 2 (9 bits), 1 (8 bits), or 1 for the first kRadix
    // threads and none for the rest (narrower digits)
    constexpr int DPT = kRadix >= kSortWG ? kRadix / kSortWG : 1;
    static_assert(kRadix < kSortWG || DPT * kSortWG == kRadix, "radix must be a multiple of the workgroup size");
    const bool owns = kRadix >= kSortWG || (int)threadIdx.x < kRadix;
    __shared__ uint16_t chunk_off[kSortChunks][kRadix];  // 16 KB (8 bits) or 32 KB (9 bits)
    __shared__ uint32_t digit_base[kRadix];
    __shared__ uint32_t global_base[kRadix];
    __shared__ uint32_t stage_k[kSortTile];
    __shared__ uint32_t stage_v[kSortTile];
    __shared__ uint32_t wave_sums[kSortWG / 64];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int64_t base = tile * kSortTile;
    const int tile_count = (int)((n - base) < kSortTile ? (n - base) : kSortTile);

    uint32_t* co32 = reinterpret_cast<uint32_t*>(&chunk_off[0][0]);
    for (int i = tid; i < kSortChunks * kRadix / 2; i += kSortWG) co32[i] = 0u;  // kRadix >= 2
    __syncthreads();

    uint32_t my_key[kChunksPerWave], my_val[kChunksPerWave], my_digit[kChunksPerWave], my_rank[kChunksPerWave];
#pragma unroll
    for (int c = 0; c < kChunksPerWave; ++c) {
        int chunk = wave * kChunksPerWave + c;
        int64_t idx = base + (int64_t)chunk * 64 + lane;
        bool valid = idx < n;
        uint32_t k = valid ? keys_in[idx] : 0u;
        uint32_t v = valid ? vals_in[idx] : 0u;
        uint32_t digit = (k >> shift) & mask;
        uint64_t active = __ballot(valid);
        uint64_t m = digit_match<BITS>(digit, active);
        uint64_t lt = (lane == 0) ? 0ull : ((~0ull) >> (64 - lane));
        my_rank[c] = (uint32_t)__popcll(m & lt);
        int leader = __ffsll((unsigned long long)m) - 1;
        if (valid && lane == leader) chunk_off[chunk][digit] = (uint16_t)__popcll(m);
        my_key[c] = k;
        my_val[c] = v;
        my_digit[c] = valid ? digit : 0xFFFFFFFFu;
    }
    __syncthreads();

    // Per digit: exclusive prefix over chunks (thread t owns digits
    // t*DPT .. t*DPT+DPT-1, so digit order follows thread order).
    uint32_t dtot[DPT];
    uint32_t total = 0;
#pragma unroll
    for (int j = 0; j < DPT; ++j) {
        dtot[j] = 0;
        if (!owns) continue;
        const int d = tid * DPT + j;
        uint32_t acc = 0;
        for (int c = 0; c < kSortChunks; ++c) {
            uint32_t cnt = chunk_off[c][d];
            chunk_off[c][d] = (uint16_t)acc;
            acc += cnt;
        }
        dtot[j] = acc;
        total += acc;
        if (BASE != kRaw) global_base[d] = hist_scan[(int64_t)d * tiles + tile];
    }
    if (BASE == kRows) {
        static_assert(BASE != kRows || kRadix == kSortWG, "one thread per digit");
        uint32_t all;
        global_base[tid] += block_exclusive_scan(row_total[tid], wave_sums, all);
    }
    if (BASE == kRaw) {
        // few tiles: the digit table is not scanned beforehand; each
        // workgroup forms its bases from the raw counts, as the sum over
        // smaller digits of their totals plus this digit's earlier tiles
        uint32_t gtot[DPT];
        uint32_t gsum = 0;
#pragma unroll
        for (int j = 0; j < DPT; ++j) {
            gtot[j] = 0;
            if (!owns) continue;
            const int d = tid * DPT + j;
            uint32_t before = 0, all = 0;
            for (int64_t t = 0; t < tiles; ++t) {
                const uint32_t c = hist_scan[(int64_t)d * tiles + t];
                before += t < tile ? c : 0u;
                all += c;
            }
            global_base[d] = before;
            gtot[j] = all;
            gsum += all;
        }
        uint32_t gall;
        uint32_t run = block_exclusive_scan(gsum, wave_sums, gall);
        if (owns) {
#pragma unroll
            for (int j = 0; j < DPT; ++j) {
                global_base[tid * DPT + j] += run;
                run += gtot[j];
            }
        }
    }
    // Block exclusive scan of the per-thread digit totals.
    uint32_t incl = total;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        uint32_t up = __shfl_up(incl, off, 64);
        if (lane >= off) incl += up;
    }
    if (lane == 63) wave_sums[wave] = incl;
    __syncthreads();
    uint32_t wave_prefix = 0;
    for (int w = 0; w < wave; ++w) wave_prefix += wave_sums[w];
    if (owns) {
        uint32_t run = wave_prefix + incl - total;
#pragma unroll
        for (int j = 0; j < DPT; ++j) {
            digit_base[tid * DPT + j] = run;
            run += dtot[j];
        }
    }
    __syncthreads();

#pragma unroll
    for (int c = 0; c < kChunksPerWave; ++c) {
        if (my_digit[c] == 0xFFFFFFFFu) continue;
        int chunk = wave * kChunksPerWave + c;
        uint32_t d = my_digit[c];
        uint32_t pos = digit_base[d] + chunk_off[chunk][d] + my_rank[c];
        stage_k[pos] = my_key[c];
        stage_v[pos] = my_val[c];
    }
    __syncthreads();

    for (int i = tid; i < tile_count; i += kSortWG) {
        uint32_t k = stage_k[i];
        uint32_t d = (k >> shift) & mask;
        int64_t out = (int64_t)global_base[d] + (i - (int64_t)digit_base[d]);
        keys_out[out] = k;
        vals_out[out] = stage_v[i];
    }
}
template <int BITS, bool RAW>
__global__ void __launch_bounds__(kSortWG) k_radix_scatter(const uint32_t* __restrict__ keys_in,
                                                           const uint32_t* __restrict__ vals_in,
                                                           uint32_t* __restrict__ keys_out,
                                                           uint32_t* __restrict__ vals_out, int64_t n, int shift,
                                                           uint32_t mask, const uint32_t* __restrict__ hist_scan,
                                                           int64_t tiles, const uint32_t* __restrict__ plan) {
    if (plan && plan_incremental(plan)) return;
    scatter_tile<BITS, RAW ? kRaw : kScanned>(keys_in, vals_in, keys_out, vals_out, n, shift, mask, hist_scan,
                                              nullptr, tiles, blockIdx.x);
}

// All passes of a sort in one launch, for steps whose sort mostly does not
// run: then it costs one launch that returns at once (5 us) instead of 12 to
// 16 (54 to 74 us of the 2.1M slab's 541 us step).  Run, it is the slower one:
// its 9 to 12 phases wait at counters in memory, and the caches' contents are
// dropped between them.  A workgroup per compute unit: fewer poll the counters
// (1.1M keys: 250 us, with four 450).
// The work is numbered in the order in which it may run -- per pass every
// tile's histogram, every digit's row of the table scanned, every tile's
// scatter -- and workgroups draw the numbers one by one.  A piece waits until
// all pieces of the phase before it are done; these have smaller numbers, so
// workgroups that run hold them and every wait ends, whatever the number of
// workgroups that the device runs at a time.  Data of one phase reaches
// the next through the fences on both sides of the counters; the pointers
// alias and are not restrict.  The item count of the step clears the counters.
constexpr int kAllBits = 8, kAllGrid = 256;
struct RadixAll {
    const uint32_t *kin, *vin;
    uint32_t *ka, *va, *kb, *vb, *hist, *plan;
    int64_t n, tiles;
    uint32_t per;      // tiles of a piece
    int passes, bits;  // the key's bits, split evenly
};
__global__ void __launch_bounds__(kSortWG) k_radix_all(RadixAll A) {
    if (plan_incremental(A.plan)) return;
    constexpr uint32_t ROWS = 1u << kAllBits;
    __shared__ uint32_t drawn, ws[kSortWG / 64];
    const uint32_t T = (uint32_t)A.tiles, P = (T + A.per - 1u) / A.per;
    const uint32_t per_pass = 2u * P + ROWS, total = per_pass * (uint32_t)A.passes;
    uint32_t* const row_total = A.hist + A.tiles * ROWS;
    for (;;) {
        // the whole workgroup between the two single-thread parts (without it
        // the compiler joins them across the turns, and the first wave's other
        // lanes run ahead of its first)
        __syncthreads();
        if (threadIdx.x == 0) {
            const uint32_t g = atomicAdd(&A.plan[kPlanTicket], 1u);
            const uint32_t q = g % per_pass, part = q < P ? 0u : (q < P + ROWS ? 1u : 2u);
            const uint32_t phase = 3u * (g / per_pass) + part;
            if (g < total && phase > 0u) {
                const uint32_t need = part == 2u ? ROWS : P;  // pieces of the phase before
                while (__hip_atomic_load(&A.plan[kPlanDone + phase - 1u], __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT) < need)
                    __builtin_amdgcn_s_sleep(32);
            }
            drawn = g;
        }
        __syncthreads();
        const uint32_t g = drawn;
        if (g >= total) return;  // uniform
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");  // drops what the caches hold of other dies' data
        const uint32_t pass = g / per_pass, q = g % per_pass;
        const uint32_t part = q < P ? 0u : (q < P + ROWS ? 1u : 2u), phase = 3u * pass + part;
        int shift = 0, width = 0;
        for (uint32_t p = 0; p <= pass; ++p) {
            shift += width;
            width = (A.bits - shift + A.passes - (int)p - 1) / (A.passes - (int)p);
        }
        const uint32_t mask = (1u << width) - 1u;
        const uint32_t* const ki = pass == 0u ? A.kin : (pass & 1u ? A.ka : A.kb);
        const uint32_t* const vi = pass == 0u ? A.vin : (pass & 1u ? A.va : A.vb);
        const uint32_t piece = part == 2u ? q - P - ROWS : q;
        const uint32_t t1 = (piece + 1u) * A.per < T ? (piece + 1u) * A.per : T;
        if (part == 0u) {
            for (uint32_t t = piece * A.per; t < t1; ++t) {
                hist_tile<kAllBits>(ki, A.n, shift, mask, A.hist, A.tiles, t);
                __syncthreads();
            }
        } else if (part == 1u) {
            uint32_t* const row = A.hist + (int64_t)(q - P) * A.tiles;
            uint32_t before = 0;
            for (uint32_t t0 = 0; t0 < T; t0 += kSortWG) {
                const uint32_t t = t0 + threadIdx.x, c = t < T ? row[t] : 0u;
                uint32_t tot;
                const uint32_t pre = block_exclusive_scan(c, ws, tot);
                if (t < T) row[t] = before + pre;
                before += tot;
            }
            if (threadIdx.x == 0) row_total[q - P] = before;
        } else {
            for (uint32_t t = piece * A.per; t < t1; ++t) {
                scatter_tile<kAllBits, kRows>(ki, vi, pass & 1u ? A.kb : A.ka, pass & 1u ? A.vb : A.va, A.n, shift,
                                              mask, A.hist, row_total, A.tiles, t);
                __syncthreads();
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every wave's stores have left it
        __syncthreads();
        if (threadIdx.x == 0) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            atomicAdd(&A.plan[kPlanDone + phase], 1u);
        }
    }
}

// ------------------------------------------------------------------ scan
// (kScanWG, kScanIPT, block_exclusive_scan: blockscan.h)

__global__ void __launch_bounds__(kScanWG) k_scan_reduce(const uint32_t* __restrict__ in, int64_t n,
                                                         uint32_t* __restrict__ partial,
                                                         const uint32_t* __restrict__ plan) {
    if (plan && plan_incremental(plan)) return;
    __shared__ uint32_t ws[kScanWG / 64];
    const int64_t tile = blockIdx.x, base = tile * kScanTile;
    uint32_t s = 0;
#pragma unroll
    for (int i = 0; i < kScanIPT; ++i) {
        int64_t idx = base + (int64_t)threadIdx.x * kScanIPT + i;
        s += idx < n ? in[idx] : 0u;
    }
    uint32_t tot;
    block_exclusive_scan(s, ws, tot);
    if (threadIdx.x == 0) partial[tile] = tot;
}

// Exclusive scan of each tile, offset by the tile prefix: partial_scan[b]
// (already scanned), or with RAW the sum of the unscanned tile totals
// partial[0..b), which the workgroup adds up itself (few tiles: this saves
// the launches of scanning them).  in and out may alias.  If total !=
// null, the last thread of the last tile writes the grand total.
template <bool RAW>
__global__ void __launch_bounds__(kScanWG) k_scan_down(const uint32_t* in, int64_t n, const uint32_t* partial_scan,
                                                       uint32_t* out, uint32_t* total, const uint32_t* plan) {
    if (plan && plan_incremental(plan)) return;
    __shared__ uint32_t ws[kScanWG / 64];
    const int64_t tile = blockIdx.x;
    uint32_t tile_prefix = 0;
    if (partial_scan) {
        if (RAW) {
            uint32_t part = 0;
            for (int64_t t = threadIdx.x; t < tile; t += kScanWG) part += partial_scan[t];
            block_exclusive_scan(part, ws, tile_prefix);
        } else {
            tile_prefix = partial_scan[tile];
        }
    }
    int64_t base = tile * kScanTile;
    uint32_t v[kScanIPT];
    uint32_t s = 0;
#pragma unroll
    for (int i = 0; i < kScanIPT; ++i) {
        int64_t idx = base + (int64_t)threadIdx.x * kScanIPT + i;
        v[i] = idx < n ? in[idx] : 0u;
        s += v[i];
    }
    uint32_t tot;
    uint32_t pre = block_exclusive_scan(s, ws, tot);
    uint32_t off = tile_prefix + pre;
#pragma unroll
    for (int i = 0; i < kScanIPT; ++i) {
        int64_t idx = base + (int64_t)threadIdx.x * kScanIPT + i;
        if (idx < n) out[idx] = off;
        off += v[i];
    }
    if (total && blockIdx.x == gridDim.x - 1 && threadIdx.x == kScanWG - 1) *total = off;
}

int64_t scan_temp_words(int64_t n) {
    int64_t words = 0;
    while (n > kScanTile) {
        int64_t tiles = (n + kScanTile - 1) / kScanTile;
        words += tiles;
        n = tiles;
    }
    return words + 64;
}

// Exclusive scan in place over n words; temp holds scan_temp_words(n).
// total (device, may be null) receives the sum.
void exclusive_scan(uint32_t* data, int64_t n, uint32_t* temp, uint32_t* total, hipStream_t st,
                    const uint32_t* plan) {
    if (n <= 0) return;
    if (n <= kScanTile) {
        hipLaunchKernelGGL(k_scan_down<false>, dim3(1), dim3(kScanWG), 0, st, data, n, (const uint32_t*)nullptr, data,
                           total, plan);
        return;
    }
    int64_t tiles = (n + kScanTile - 1) / kScanTile;
    uint32_t* partial = temp;
    const unsigned grid = (unsigned)tiles;
    hipLaunchKernelGGL(k_scan_reduce, dim3(grid), dim3(kScanWG), 0, st, data, n, partial, plan);
    if (tiles <= 2048) {  // each tile sums at most 2047 tile totals itself
        hipLaunchKernelGGL(k_scan_down<true>, dim3(grid), dim3(kScanWG), 0, st, data, n, (const uint32_t*)partial,
                           data, total, plan);
        return;
    }
    exclusive_scan(partial, tiles, temp + tiles, nullptr, st, plan);
    hipLaunchKernelGGL(k_scan_down<false>, dim3(grid), dim3(kScanWG), 0, st, data, n, (const uint32_t*)partial, data,
                       total, plan);
}

int64_t radix_tiles(int64_t n) { return (n + kSortTile - 1) / kSortTile; }
// Sorts of at most this many tiles skip the separate digit-table scan.
constexpr int64_t kRawTiles = 32;
int64_t radix_hist_words(int64_t n) { return radix_tiles(n) * kMaxRadix; }

// Digit widths.  Large sorts (>= 2^20 keys) use digits of at most 7 bits:
// the scatter of a 2048-key tile then writes runs of >= 16 keys per digit,
// and on the 8.4M-particle slab (25-bit keys) 4 passes of 7/6/6/6 bits take
// 0.31 ms against 0.37 ms for 3 passes of 9/8/8 and 0.35 ms for 5 passes of
// 5-6 bits.  Small sorts are launch-bound and use as few passes as 8- or
// 9-bit digits allow.  Bits are split as evenly as possible, widest first.
int radix_passes(int key_bits, int64_t n) {
    if (n >= (int64_t(1) << 20)) return (key_bits + 6) / 7;
    const int p8 = (key_bits + 7) / 8, p9 = (key_bits + 8) / 9;
    return p9 < p8 ? p9 : p8;
}
static int digit_bits(int key_bits, int64_t n, int pass) {
    const int passes = radix_passes(key_bits, n);
    int done = 0;
    for (int p = 0; p < pass; ++p) done += (key_bits - done + (passes - p) - 1) / (passes - p);
    return (key_bits - done + (passes - pass) - 1) / (passes - pass);
}

// Sorts (kin,vin) (read only) into (ka,va)/(kb,vb) ping-pong buffers;
// returns 0 if the result is in (ka,va), 1 if in (kb,vb).
int radix_sort_pairs(const uint32_t* kin, const uint32_t* vin, uint32_t* ka, uint32_t* va, uint32_t* kb, uint32_t* vb,
                     int64_t n, int key_bits, uint32_t* hist, uint32_t* scan_temp, hipStream_t st,
                     const ProfileHook& prof, uint32_t* plan, bool one_launch) {
    if (n <= 0) return 0;
    int64_t tiles = radix_tiles(n);
    if (one_launch && plan) {
        static_assert(kPlanDone + 3 * 4 <= kPlanLists, "three counters per pass, at most four passes");
        const uint32_t per = (uint32_t)((tiles + kAllGrid - 1) / kAllGrid);
        const RadixAll A{kin, vin, ka, va, kb, vb, hist, plan, n, tiles, per, (key_bits + kAllBits - 1) / kAllBits,
                         key_bits};
        prof.begin("sort_scatter");
        hipLaunchKernelGGL(k_radix_all, dim3((unsigned)(tiles < kAllGrid ? tiles : kAllGrid)), dim3(kSortWG), 0, st, A);
        prof.end("sort_scatter");
        return (A.passes & 1) ? 0 : 1;
    }
    const int passes = radix_passes(key_bits, n);
    const unsigned grid = (unsigned)tiles;
    const uint32_t *ki = kin, *vi = vin;
    uint32_t *ko = ka, *vo = va;
    int shift = 0;
    for (int p = 0; p < passes; ++p) {
        const int bits = digit_bits(key_bits, n, p);
        const uint32_t mask = (1u << bits) - 1u;
        // digit widths of the plan: 9 or 8 bits, or 6-7 under a narrower plan
        const int dw = bits > 8 ? 9 : (bits > 7 ? 8 : (bits > 6 ? 7 : 6));
        const int radix = 1 << dw;
        prof.begin("sort_hist");
#define MPM_HIST(B) hipLaunchKernelGGL(k_radix_hist<B>, dim3(grid), dim3(kSortWG), 0, st, ki, n, shift, mask, hist, \
                                       tiles, plan)
        if (dw == 9) MPM_HIST(9);
        else if (dw == 8) MPM_HIST(8);
        else if (dw == 7) MPM_HIST(7);
        else MPM_HIST(6);
#undef MPM_HIST
        prof.end("sort_hist");
        // up to kRawTiles tiles the scatter reads the raw digit table itself
        // (one launch fewer per pass for small sorts)
        const bool raw = tiles <= kRawTiles;
        prof.begin("sort_scan");
        if (!raw) exclusive_scan(hist, tiles * radix, scan_temp, nullptr, st, plan);
        prof.end("sort_scan");
        prof.begin("sort_scatter");
#define MPM_SCATTER(B, R) hipLaunchKernelGGL((k_radix_scatter<B, R>), dim3(grid), dim3(kSortWG), 0, st, ki, vi, ko, \
                                             vo, n, shift, mask, hist, tiles, plan)
        if (raw) {
            if (dw == 9) MPM_SCATTER(9, true);
            else if (dw == 8) MPM_SCATTER(8, true);
            else if (dw == 7) MPM_SCATTER(7, true);
            else MPM_SCATTER(6, true);
        } else {
            if (dw == 9) MPM_SCATTER(9, false);
            else if (dw == 8) MPM_SCATTER(8, false);
            else if (dw == 7) MPM_SCATTER(7, false);
            else MPM_SCATTER(6, false);
        }
#undef MPM_SCATTER
        prof.end("sort_scatter");
        shift += bits;
        ki = ko;
        vi = vo;
        ko = (ko == ka) ? kb : ka;
        vo = (vo == va) ? vb : va;
    }
    return (passes & 1) ? 0 : 1;
}

}  // namespace mpm
