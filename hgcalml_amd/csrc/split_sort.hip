// Stable sort of integer keys from a known range -- a counting sort in two
// levels, written for the index tables of this library (HBM-bound integer work):
// the inverse neighbour index (keys: the target of every slot of the neighbour
// table), the hits in bin order (keys: flat bin index) and the condensates'
// selection order (keys: pieces of the beta ordering).
//
//   level 1  keys are cut into tiles of 2^lo_bits consecutive values. Every
//            workgroup counts the items of its stretch of the input per tile (LDS
//            atomics), a scan over (tile, workgroup) turns the counts into
//            positions, and the workgroups move their items, as (key, value)
//            records, into tile order -- a batch of 12,288 items of the stretch at
//            a time is put into tile order in LDS first and leaves from there, so that
//            the records of a tile are written next to each other. (One 8-byte
//            write per record straight from the walk: 138 us for 9.75 M items in
//            1172 tiles.) A wave walks its part of the batch in order and ranks the
//            64 items of a step among the equal digits of that step with one ballot
//            per bit, so the move is stable.
//   level 2  one workgroup per tile sorts the tile's records by key in the same
//            way (count per wave, scan over the tile's keys, ordered walk) into a
//            stage in LDS, from where the tile's values leave in whole lines,
//            together with the first position of every key. Tiles of up to
//            20,480 items are held in registers between the count and the walk, larger
//            ones are read twice.
// 9.75 M items, 150,000 keys (the inverse index of a kNN table): 205 -> 119 us; 64 M items, a million
// keys: 1.32 -> 0.84 ms (kNN table), 0.92 -> 0.80 (banded). Bound by vector issue and LDS latency of
// the walks (16 waves per CU); the memory traffic alone would take 60 us and 0.4 ms.
//
// Items whose key lies outside [0, n_keys) carry the key n_keys and end up last.
#include "hgc_common.hpp"

#include <algorithm>
#include <cstring>

#include <rocprim/rocprim.hpp>

namespace hgc {
namespace {

constexpr int kMaxTiles = 8192;
constexpr int kMinLoBits = 5;
constexpr int kMaxLoBits = 10;
constexpr int kTileItems = 16384;   // items per tile aimed at: what level 2 holds in registers, with a margin
constexpr int kMinItemsPerGroup = 4096;
constexpr int kMaxGroups = 256;     // one workgroup of level 1 fills a CU's LDS
constexpr int kCountThreads = 1024;
constexpr int kMoveWaves = 16;
constexpr int kMoveThreads = kMoveWaves * kWave;
constexpr int kMoveSteps = 12;      // steps of 64 items a wave of level 1 takes per batch
constexpr int kBatch = kMoveThreads * kMoveSteps;
// Up to this many tiles a batch is put into tile order in one pass over a counter per wave and tile (52 us for
// 9.75 M items in 586 tiles, the two passes of the wide kernel 71); beyond, clearing and scanning those
// counters outweighs a batch (64 M items in 3907 tiles, half the waves for want of LDS: 690 us against 410).
constexpr int kFewTiles = 1536;
constexpr int kWantedTiles = 512;   // small key ranges are cut finer, so that level 2 has workgroups to spread

struct Plan {
    int lo_bits, n_tiles, n_groups, per_group;
    bool ok;
};

Plan make_plan(long long total, int n_keys, int per_key) {
    Plan p{};
    p.lo_bits = kMinLoBits;
    while (p.lo_bits < kMaxLoBits && ((long long)std::max(per_key, 1) << (p.lo_bits + 1)) <= kTileItems &&
           (n_keys >> (p.lo_bits + 1)) >= kWantedTiles)
        ++p.lo_bits;
    while (p.lo_bits < kMaxLoBits && (n_keys >> p.lo_bits) + 1 > kMaxTiles) ++p.lo_bits;
    p.n_tiles = (n_keys >> p.lo_bits) + 1;  // keys run from 0 to n_keys inclusive
    p.ok = p.n_tiles <= kMaxTiles && total < (1ll << 31);
    const long long per_group = std::max<long long>(kMinItemsPerGroup, (total + kMaxGroups - 1) / kMaxGroups);
    p.per_group = (int)((per_group + kWave - 1) / kWave * kWave);
    p.n_groups = (int)std::max<long long>(1, (total + p.per_group - 1) / p.per_group);
    return p;
}

__device__ __forceinline__ uint32_t clamp_key(int k, uint32_t n_keys) { return (uint32_t)k < n_keys ? (uint32_t)k : n_keys; }

// The lanes among `active` whose `digit` agrees with this lane's in its low `bits` bits. Written on the
// halves with the bit as a sign mask: four vector instructions a bit (one v_bitop3 per half),
// where the 64-bit select form took ten and half of the sort's time.
__device__ __forceinline__ uint64_t same_digit_lanes(uint32_t digit, int bits, uint64_t active) {
    uint32_t lo = (uint32_t)active, hi = (uint32_t)(active >> 32);
    for (int b = 0; b < bits; ++b) {
        const uint32_t mask = (uint32_t)__builtin_amdgcn_sbfe((int)digit, b, 1);  // 0 or all ones
        const uint64_t with = __ballot(mask != 0u);
        lo &= ~((uint32_t)with ^ mask);
        hi &= ~((uint32_t)(with >> 32) ^ mask);
    }
    return ((uint64_t)hi << 32) | lo;
}

// LDS accesses of one wave execute in program order; this only keeps the compiler from
// moving them across the point where lanes hand a counter to each other. (A memory fence
// would also wait for the global stores in flight and serialise the walk.)
__device__ __forceinline__ void lds_order_point() { __builtin_amdgcn_wave_barrier(); }

// A barrier that orders the workgroup's LDS traffic only: __syncthreads() would also wait for the
// global stores in flight, which nobody in the workgroup reads back.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

__device__ __forceinline__ int lanes_below(uint64_t mask) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// ---- level 1 ---------------------------------------------------------------

constexpr int kAhead = 8;  // steps of 64 items whose loads are issued together (memory-level parallelism)

// Positions are counted from where a workgroup's stretch (or its tile, level 2) begins: a walk looks up to a batch
// beyond the end of its stretch, which as a position among all items, of which there may be 2^31 - 1, would not
// fit into an int.
struct Stretch {
    int first, count;
};
__device__ __forceinline__ Stretch stretch_of(int group, int per_group, int total) {
    const long long first = min((long long)group * per_group, (long long)total);
    return {(int)first, (int)min((long long)per_group, total - first)};
}

// keys[first], keys[first + STRIDE], ...
template <int STRIDE, int N>
__device__ __forceinline__ void load_items(const int *__restrict__ keys, int first, int last, int (&key)[N]) {
    // loads past the end re-read the last item: no branch, all of them in flight together
#pragma unroll
    for (int a = 0; a < N; ++a) key[a] = keys[min(first + a * STRIDE, last)];
}

// counts[tile * n_groups + group]: items of the group's stretch that fall into the tile
__global__ __launch_bounds__(kCountThreads) void tile_count_kernel(const int *__restrict__ keys, int total,
                                                                   uint32_t n_keys, int lo_bits, int n_tiles,
                                                                   int n_groups, int per_group,
                                                                   int *__restrict__ counts) {
    extern __shared__ int s_count[];  // [n_tiles]
    for (int t = threadIdx.x; t < n_tiles; t += blockDim.x) s_count[t] = 0;
    __syncthreads();
    const Stretch own = stretch_of(blockIdx.x, per_group, total);
    for (int e0 = (int)threadIdx.x; e0 - (int)threadIdx.x < own.count; e0 += kCountThreads * kAhead) {
        int raw[kAhead];
        load_items<kCountThreads>(keys + own.first, e0, own.count - 1, raw);
#pragma unroll
        for (int a = 0; a < kAhead; ++a)
            if (e0 + a * kCountThreads < own.count) atomicAdd(&s_count[clamp_key(raw[a], n_keys) >> lo_bits], 1);
    }
    __syncthreads();
    for (int t = threadIdx.x; t < n_tiles; t += blockDim.x) counts[(size_t)t * n_groups + blockIdx.x] = s_count[t];
    if (blockIdx.x == 0 && threadIdx.x == 0) counts[(size_t)n_tiles * n_groups] = 0;  // the scan's last element
}

// exclusive sum over the workgroup's threads (all of them call it)
__device__ __forceinline__ int block_exclusive_sum(int x, int *wave_sums) {
    const int wave = threadIdx.x >> 6, lane = lane_id();
    const int incl = wave_inclusive_sum(x);
    if (lane == kWave - 1) wave_sums[wave] = incl;
    lds_barrier();
    const int upto = wave_inclusive_sum(lane < kMoveWaves ? wave_sums[lane] : 0);
    return incl - x + (wave == 0 ? 0 : readlane_i32(upto, wave - 1));
}

// records[position] = (key, value), grouped by tile, in input order inside a tile: up to kFewTiles tiles,
// a counter per wave and tile
__global__ __launch_bounds__(kMoveThreads) void tile_move_kernel(const int *__restrict__ keys, int total,
                                                                 uint32_t n_keys, int lo_bits, int tile_bits,
                                                                 int n_tiles, int n_groups, int per_group,
                                                                 const int *__restrict__ starts,
                                                                 uint2 *__restrict__ records) {
    __shared__ uint2 s_stage[kBatch];  // tile order
    __shared__ int s_wave_sums[kMoveWaves];
    extern __shared__ int s_next[];                                            // [n_tiles] next record of the tile
    int *const s_local = s_next + n_tiles;                                     // [n_tiles + 1] its first place in the batch
    const int row = (n_tiles + 1) & ~1;
    uint16_t *const s_count = reinterpret_cast<uint16_t *>(s_local + n_tiles + 1);  // [kMoveWaves][row]
    const int wave = threadIdx.x >> 6, lane = lane_id();
    uint16_t *const mine = s_count + wave * row;
    for (int t = threadIdx.x; t < n_tiles; t += kMoveThreads) s_next[t] = starts[(size_t)t * n_groups + blockIdx.x];
    const Stretch own = stretch_of(blockIdx.x, per_group, total);
    const int tiles_per_thread = (n_tiles + kMoveThreads - 1) / kMoveThreads;

    for (int b0 = 0; b0 < own.count; b0 += kBatch) {
        const int in_batch = min(kBatch, own.count - b0);
        const int per_wave = ((in_batch + kMoveWaves - 1) / kMoveWaves + kWave - 1) / kWave * kWave;
        const int w0 = min(wave * per_wave, in_batch), w1 = min(w0 + per_wave, in_batch);
        int key[kMoveSteps];
        for (int i = threadIdx.x; i < kMoveWaves * row / 2; i += kMoveThreads) reinterpret_cast<uint32_t *>(s_count)[i] = 0;
        load_items<kWave>(keys + own.first, b0 + w0 + lane, own.count - 1, key);
        lds_barrier();
#pragma unroll
        for (int a = 0; a < kMoveSteps; ++a) {
            key[a] = (int)clamp_key(key[a], n_keys);
            if (w0 + a * kWave + lane < w1) {
                const uint32_t tile = (uint32_t)key[a] >> lo_bits;
                atomicAdd(reinterpret_cast<uint32_t *>(mine) + (tile >> 1), 1u << (16 * (tile & 1)));
            }
        }
        lds_barrier();
        // counts -> first places: exclusive scan over (tile, wave)
        int sum = 0;
        for (int i = 0; i < tiles_per_thread; ++i) {
            const int t = (int)threadIdx.x * tiles_per_thread + i;
            if (t < n_tiles)
#pragma unroll
                for (int w = 0; w < kMoveWaves; ++w) sum += s_count[w * row + t];
        }
        int at = block_exclusive_sum(sum, s_wave_sums);
        for (int i = 0; i < tiles_per_thread; ++i) {
            const int t = (int)threadIdx.x * tiles_per_thread + i;
            if (t < n_tiles) {
                s_local[t] = at;
#pragma unroll
                for (int w = 0; w < kMoveWaves; ++w) {
                    const int c = s_count[w * row + t];
                    s_count[w * row + t] = (uint16_t)at;
                    at += c;
                }
            }
        }
        if (threadIdx.x == 0) s_local[n_tiles] = in_batch;
        lds_barrier();
#pragma unroll
        for (int a = 0; a < kMoveSteps; ++a) {
            if (w0 + a * kWave >= w1) break;  // wave-uniform
            const bool valid = w0 + a * kWave + lane < w1;
            const uint32_t tile = valid ? (uint32_t)key[a] >> lo_bits : 0u;
            const uint64_t peers = same_digit_lanes(tile, tile_bits, __ballot(valid));
            const int rank = lanes_below(peers);
            int place = 0;
            if (valid) place = mine[tile];
            lds_order_point();
            if (valid && rank == 0) mine[tile] = (uint16_t)(place + (int)__popcll(peers));
            lds_order_point();
            if (valid) s_stage[place + rank] = make_uint2((uint32_t)key[a], (uint32_t)own.first + (uint32_t)(b0 + w0 + a * kWave + lane));
        }
        lds_barrier();
        for (int i = threadIdx.x; i < in_batch; i += kMoveThreads) {
            const uint2 rec = s_stage[i];
            const uint32_t tile = rec.x >> lo_bits;
            records[(size_t)(s_next[tile] + (i - s_local[tile]))] = rec;
        }
        lds_barrier();
        for (int t = threadIdx.x; t < n_tiles; t += kMoveThreads) s_next[t] += s_local[t + 1] - s_local[t];
    }
}

// One stable pass over a batch in LDS: the items (wave w holds positions w0 + a * 64 + lane of the
// batch in step a, those below w1) go to `stage` in the order of their BITS digit bits at `shift`. counters:
// [2^BITS][kMoveWaves] 16-bit. A wave walks its steps in order and counts its items per digit on
// the way, which gives every item its place among the wave's equals; an exclusive scan over
// (digit, wave) gives the first place of those. Ends with the batch in `stage`, all waves in step.
template <int BITS>
__device__ __forceinline__ void batch_pass(int (&key)[kMoveSteps], int (&val)[kMoveSteps], int w0, int w1, int shift, uint16_t *counters,
                                           int *wave_sums, uint2 *stage) {
    const int wave = threadIdx.x >> 6, lane = lane_id();
    uint32_t *const pairs = reinterpret_cast<uint32_t *>(counters);  // of two waves
    constexpr int n_pairs = (kMoveWaves / 2) << BITS;                // at most one per thread
    if ((int)threadIdx.x < n_pairs) pairs[threadIdx.x] = 0;
    lds_barrier();
    int place[kMoveSteps];
    const uint32_t mask = (1u << BITS) - 1u;
#pragma unroll
    for (int a = 0; a < kMoveSteps; ++a) {
        if (w0 + a * kWave >= w1) break;  // wave-uniform
        const bool valid = w0 + a * kWave + lane < w1;
        const uint32_t digit = ((uint32_t)key[a] >> shift) & mask;
        const uint64_t peers = same_digit_lanes(digit, BITS, __ballot(valid));
        const int rank = lanes_below(peers);
        uint16_t *const mine = counters + digit * kMoveWaves + wave;
        int before = 0;
        if (valid) before = *mine;
        lds_order_point();
        if (valid && rank == 0) *mine = (uint16_t)(before + (int)__popcll(peers));
        lds_order_point();
        place[a] = before + rank;
    }
    lds_barrier();
    const uint32_t pair = (int)threadIdx.x < n_pairs ? pairs[threadIdx.x] : 0u;
    const int first = block_exclusive_sum((int)(pair & 0xffffu) + (int)(pair >> 16), wave_sums);
    if ((int)threadIdx.x < n_pairs) pairs[threadIdx.x] = (uint32_t)first | ((uint32_t)(first + (int)(pair & 0xffffu)) << 16);
    lds_barrier();
#pragma unroll
    for (int a = 0; a < kMoveSteps; ++a) {
        if (w0 + a * kWave >= w1) break;  // wave-uniform
        if (w0 + a * kWave + lane < w1) {
            const uint32_t digit = ((uint32_t)key[a] >> shift) & mask;
            stage[counters[digit * kMoveWaves + wave] + place[a]] = make_uint2((uint32_t)key[a], (uint32_t)val[a]);
        }
    }
    lds_barrier();
}

// records[position] = (key, value), grouped by tile, in input order inside a tile: any number of tiles
template <int BITS>
__global__ __launch_bounds__(kMoveThreads) void tile_move_wide_kernel(const int *__restrict__ keys, int total,
                                                                 uint32_t n_keys, int lo_bits, int n_tiles, int n_groups,
                                                                 int per_group, const int *__restrict__ starts,
                                                                 uint2 *__restrict__ records) {
    __shared__ uint2 s_stage[kBatch];
    __shared__ __attribute__((aligned(4))) uint16_t s_counters[kMoveWaves << BITS];
    __shared__ int s_wave_sums[kMoveWaves];
    extern __shared__ int s_next[];  // [n_tiles] next record of the tile, behind it:
    uint16_t *const s_local = reinterpret_cast<uint16_t *>(s_next + n_tiles);  // its first place in the batch (where it has items)
    const int wave = threadIdx.x >> 6, lane = lane_id();
    for (int t = threadIdx.x; t < n_tiles; t += kMoveThreads) s_next[t] = starts[(size_t)t * n_groups + blockIdx.x];
    const Stretch own = stretch_of(blockIdx.x, per_group, total);

    for (int b0 = 0; b0 < own.count; b0 += kBatch) {
        const int in_batch = min(kBatch, own.count - b0);
        const int per_wave = ((in_batch + kMoveWaves - 1) / kMoveWaves + kWave - 1) / kWave * kWave;
        const int w0 = min(wave * per_wave, in_batch), w1 = min(w0 + per_wave, in_batch);
        int key[kMoveSteps], val[kMoveSteps];
        load_items<kWave>(keys + own.first, b0 + w0 + lane, own.count - 1, key);
#pragma unroll
        for (int a = 0; a < kMoveSteps; ++a) {
            key[a] = (int)clamp_key(key[a], n_keys);
            val[a] = (int)((uint32_t)own.first + (uint32_t)(b0 + w0 + a * kWave + lane));
        }
        batch_pass<BITS>(key, val, w0, w1, lo_bits, s_counters, s_wave_sums, s_stage);
#pragma unroll
        for (int a = 0; a < kMoveSteps; ++a)
            if (w0 + a * kWave + lane < w1) {
                const uint2 rec = s_stage[w0 + a * kWave + lane];
                key[a] = (int)rec.x;
                val[a] = (int)rec.y;
            }
        batch_pass<BITS>(key, val, w0, w1, lo_bits + BITS, s_counters, s_wave_sums, s_stage);
        // where the tiles of this batch begin in it; only the tiles that have items are touched
        for (int i = threadIdx.x; i < in_batch; i += kMoveThreads) {
            const uint32_t tile = s_stage[i].x >> lo_bits;
            if (i == 0 || s_stage[i - 1].x >> lo_bits != tile) s_local[tile] = (uint16_t)i;
        }
        lds_barrier();
        int next[kMoveSteps];
#pragma unroll
        for (int a = 0; a < kMoveSteps; ++a) {
            const int i = a * kMoveThreads + (int)threadIdx.x;
            if (i < in_batch) {
                const uint2 rec = s_stage[i];
                const uint32_t tile = rec.x >> lo_bits;
                const int at = s_next[tile] + (i - (int)s_local[tile]);
                records[at] = rec;
                // the last item of a tile carries its position on to the next batch
                next[a] = i + 1 == in_batch || s_stage[i + 1].x >> lo_bits != tile ? at + 1 : -1;
                key[a] = (int)tile;
            }
        }
        lds_barrier();
#pragma unroll
        for (int a = 0; a < kMoveSteps; ++a)
            if (a * kMoveThreads + (int)threadIdx.x < in_batch && next[a] >= 0) s_next[key[a]] = next[a];
    }
}

int launch_split(const Plan &plan, const int *keys, int total, uint32_t n_keys, int *counts,
                 int *starts, void *temp, size_t temp_bytes, uint2 *records, hipStream_t s) {
    tile_count_kernel<<<plan.n_groups, kCountThreads, plan.n_tiles * sizeof(int), s>>>(
        keys, total, n_keys, plan.lo_bits, plan.n_tiles, plan.n_groups, plan.per_group, counts);
    int rc = check_launch("tile_count");
    if (rc) return rc;
    const size_t cells = (size_t)plan.n_tiles * plan.n_groups + 1;
    HGC_HIP(rocprim::exclusive_scan(temp, temp_bytes, counts, starts, 0, cells, rocprim::plus<int>(), s));
    if (plan.n_tiles <= kFewTiles) {
        int tile_bits = 1;
        while ((1 << tile_bits) < plan.n_tiles) ++tile_bits;
        const size_t lds = (2 * (size_t)plan.n_tiles + 1) * sizeof(int) +
                           (size_t)kMoveWaves * ((plan.n_tiles + 1) & ~1) * sizeof(uint16_t);
        tile_move_kernel<<<plan.n_groups, kMoveThreads, lds, s>>>(keys, total, n_keys, plan.lo_bits, tile_bits,
                                                                           plan.n_tiles, plan.n_groups, plan.per_group,
                                                                           starts, records);
        return check_launch("tile_move");
    }
    const size_t lds = plan.n_tiles * (sizeof(int) + sizeof(uint16_t));
    if (plan.n_tiles <= 1 << 12)
        tile_move_wide_kernel<6><<<plan.n_groups, kMoveThreads, lds, s>>>(
            keys, total, n_keys, plan.lo_bits, plan.n_tiles, plan.n_groups, plan.per_group, starts, records);
    else
        tile_move_wide_kernel<7><<<plan.n_groups, kMoveThreads, lds, s>>>(
            keys, total, n_keys, plan.lo_bits, plan.n_tiles, plan.n_groups, plan.per_group, starts, records);
    return check_launch("tile_move_wide");
}

// ---- level 2 ---------------------------------------------------------------

constexpr int kSortWaves = 16;  // counters (4 bytes per wave and key) and stage: 148 KB of LDS at the most
constexpr int kSortSteps = 20;  // steps of 64 records a wave holds in registers between the count and the walk
constexpr int kHeldItems = kSortWaves * kWave * kSortSteps;

// What the stage holds: twice as many items as a tile aims at where the counters leave the room
constexpr int stage_items(int lo_bits) { return lo_bits <= 8 ? 32768 : kHeldItems; }

// One workgroup per tile. The tile's values leave through a stage in LDS, so that global memory
// sees whole lines instead of one 4-byte write per slot. A tile with more items than the registers
// hold (few keys, or a few that most items share) reads its records twice, kAhead steps at a time, one with
// more than the stage holds writes its values one by one. (Step by step every wave waits for one load after
// the other: 5 M items of 300 keys 540 us, now 402; the index of 6.4 M slots that name 2000 of 100,000
// vertices 569, now 427.)
template <int LO_BITS>
__global__ __launch_bounds__(kSortWaves *kWave) void tile_sort_kernel(const uint2 *__restrict__ records,
                                                                      const int *__restrict__ starts, int n_groups,
                                                                      uint32_t n_keys, int *__restrict__ offsets,
                                                                      int *__restrict__ order) {
    constexpr int T = 1 << LO_BITS;
    __shared__ int s_cursor[kSortWaves][T];
    __shared__ int s_total[T];
    constexpr int kStage = stage_items(LO_BITS);
    __shared__ int s_stage[kStage];
    const int wave = threadIdx.x >> 6, lane = lane_id();
    const int tile = blockIdx.x;
    const int begin_tile = starts[(size_t)tile * n_groups], in_tile = starts[(size_t)(tile + 1) * n_groups] - begin_tile;
    const bool held = in_tile <= kHeldItems, staged = in_tile <= kStage;
    order += begin_tile;
    for (int t = threadIdx.x; t < T * kSortWaves; t += blockDim.x) (&s_cursor[0][0])[t] = 0;
    const int per_wave = (max(in_tile - 1, 0) / (kSortWaves * kWave) + 1) * kWave;
    const Stretch own = stretch_of(wave, per_wave, in_tile);
    records += (size_t)begin_tile + own.first;
    uint2 rec[kSortSteps];
    if (held) {
#pragma unroll
        for (int a = 0; a < kSortSteps; ++a)
            if (a * kWave < own.count) rec[a] = records[min(a * kWave + lane, own.count - 1)];  // wave-uniform
    }
    lds_barrier();
    if (held) {
#pragma unroll
        for (int a = 0; a < kSortSteps; ++a)
            if (a * kWave + lane < own.count) atomicAdd(&s_cursor[wave][rec[a].x & (T - 1)], 1);
    } else {
        for (int e0 = lane; e0 - lane < own.count; e0 += kWave * kAhead) {
            uint32_t key[kAhead];
#pragma unroll
            for (int a = 0; a < kAhead; ++a) key[a] = records[min(e0 + a * kWave, own.count - 1)].x;
#pragma unroll
            for (int a = 0; a < kAhead; ++a)
                if (e0 + a * kWave < own.count) atomicAdd(&s_cursor[wave][key[a] & (T - 1)], 1);
        }
    }
    lds_barrier();
    // per key: the waves' counts become their first positions inside the key's run
    for (int t = threadIdx.x; t < T; t += blockDim.x) {
        int at = 0;
#pragma unroll
        for (int w = 0; w < kSortWaves; ++w) {
            const int c = s_cursor[w][t];
            s_cursor[w][t] = at;
            at += c;
        }
        s_total[t] = at;
    }
    lds_barrier();
    if (wave == 0) {  // exclusive scan of the run lengths over the tile's keys
        int carry = 0;
        for (int t0 = 0; t0 < T; t0 += kWave) {
            // a tile of fewer keys than the wave has lanes (T = 32): the lanes beyond it stay out of the table
            const bool in_table = t0 + lane < T;
            const int len = in_table ? s_total[t0 + lane] : 0;
            const int incl = wave_inclusive_sum(len);
            if (in_table) s_total[t0 + lane] = carry + incl - len;
            carry += readlane_i32(incl, kWave - 1);
        }
    }
    lds_barrier();
    const uint32_t first_target = (uint32_t)tile << LO_BITS;
    for (int t = threadIdx.x; t < T; t += blockDim.x) {
        const int at = s_total[t];  // relative to the tile's first item
        // entry n_keys: where the items without a valid key begin
        if (offsets && first_target + t <= n_keys) offsets[first_target + t] = begin_tile + at;
#pragma unroll
        for (int w = 0; w < kSortWaves; ++w) s_cursor[w][t] += at;
    }
    lds_barrier();
    // the place of this lane's record of a step, relative to the tile's first
    auto place_of = [&](uint32_t key, bool valid) {
        const uint32_t t = key & (T - 1);
        const uint64_t peers = same_digit_lanes(t, LO_BITS, __ballot(valid));
        const int rank = lanes_below(peers);
        int at = 0;
        if (valid) at = s_cursor[wave][t];
        lds_order_point();
        if (valid && rank == 0) s_cursor[wave][t] = at + (int)__popcll(peers);
        lds_order_point();
        return at + rank;
    };
    if (held) {
#pragma unroll
        for (int a = 0; a < kSortSteps; ++a) {
            if (a * kWave >= own.count) break;  // wave-uniform
            const bool valid = a * kWave + lane < own.count;
            const int place = place_of(rec[a].x, valid);
            if (valid) s_stage[place] = (int)rec[a].y;
        }
    } else {
        for (int c0 = 0; c0 < own.count; c0 += kWave * kAhead) {  // wave-uniform
            uint2 r[kAhead];
#pragma unroll
            for (int a = 0; a < kAhead; ++a) r[a] = records[min(c0 + a * kWave + lane, own.count - 1)];
#pragma unroll
            for (int a = 0; a < kAhead; ++a) {
                if (c0 + a * kWave >= own.count) break;  // wave-uniform
                const bool valid = c0 + a * kWave + lane < own.count;
                const int place = place_of(r[a].x, valid);
                if (valid && staged) s_stage[place] = (int)r[a].y;
                if (valid && !staged) order[place] = (int)r[a].y;
            }
        }
        if (!staged) return;
    }
    lds_barrier();
    for (int i = threadIdx.x; i < in_tile; i += blockDim.x) order[i] = s_stage[i];
}


size_t scan_bytes(size_t n) {
    size_t temp = 0;
    (void)rocprim::exclusive_scan(nullptr, temp, (const int *)nullptr, (int *)nullptr, 0, n, rocprim::plus<int>(),
                                  (hipStream_t) nullptr);
    return align_up(temp);
}

}  // namespace

bool stable_key_sort_supported(long long total, int n_keys, int per_key_hint) {
    return n_keys >= 1 && make_plan(std::max<long long>(total, 1), n_keys, per_key_hint).ok;
}

size_t stable_key_sort_workspace_bytes(long long total, int n_keys, int per_key_hint) {
    total = std::max<long long>(total, 1);
    const Plan p = make_plan(total, std::max(n_keys, 1), per_key_hint);
    const size_t cells = (size_t)p.n_tiles * p.n_groups + 1;
    return align_up((size_t)total * sizeof(uint2)) + 2 * align_up(cells * sizeof(int)) + scan_bytes(cells);
}

int stable_key_sort(const int *d_keys, long long total, int n_keys, int per_key_hint,
                    int *d_offsets, int *d_order, void *workspace, size_t workspace_bytes, hipStream_t s) {
    if (total <= 0) return d_offsets ? launch_fill_i32(d_offsets, 0, (long long)n_keys + 1, s) : HGC_OK;
    const Plan plan = make_plan(total, n_keys, per_key_hint);
    if (!plan.ok) return fail(HGC_ERR_UNSUPPORTED, "key range too wide for the two-level sort");
    if (!workspace || !aligned256(workspace) ||
        workspace_bytes < stable_key_sort_workspace_bytes(total, n_keys, per_key_hint))
        return fail(HGC_ERR_WORKSPACE, "sort workspace missing, misaligned or too small");
    Carver carve(workspace);
    const size_t cells = (size_t)plan.n_tiles * plan.n_groups + 1;
    uint2 *records = carve.take<uint2>(total);
    int *counts = carve.take<int>(cells);
    int *starts = carve.take<int>(cells);
    void *temp = carve.base + carve.used;
    size_t temp_bytes = workspace_bytes - carve.used;
    const int rc = launch_split(plan, d_keys, (int)total, (uint32_t)n_keys, counts, starts, temp, temp_bytes, records, s);
    if (rc) return rc;
#define HGC_TILE_SORT(B)                                                                                          \
    case B:                                                                                                       \
        tile_sort_kernel<B><<<plan.n_tiles, kSortWaves * kWave, 0, s>>>(records, starts, plan.n_groups,       \
                                                                           (uint32_t)n_keys, d_offsets, d_order); \
        break
    switch (plan.lo_bits) {
        HGC_TILE_SORT(5);
        HGC_TILE_SORT(6);
        HGC_TILE_SORT(7);
        HGC_TILE_SORT(8);
        HGC_TILE_SORT(9);
        HGC_TILE_SORT(10);
    }
#undef HGC_TILE_SORT
    return check_launch("tile_sort");
}

}  // namespace hgc
