// Exact binned k-nearest-neighbour search, one wave64 per query point.
//
// Reference behaviour restated here:
//   modules/compiled/binned_select_knn_kernel.cc:19-196 (search, defaults, stop rule)
//   modules/compiled/binstepper.h:11-97                 (shell of bins at distance d)
//   modules/binned_select_knn_op.py:92-95               (un-sort, fused when a sorting is given)
//   modules/compiled/select_knn_kernel.cc:158,244-245   (radius rule)
//
// Two searches, chosen by collects(): collect_nearest (every coordinate binned, up to 129 neighbours), described where
// it stands, and walk_shells for the rest. walk_shells' design (gfx950, wave64):
//   * Points arrive grouped by bin, so the bins of one row of the grid (last
//     binned dimension running) are one contiguous range of points. A shell of
//     half-width d is cut into such ranges ("segments"); the 64 lanes look up 64
//     segments at once (cutting each against the current K-th distance) and
//     prefix-sum their lengths. Every non-empty segment marks the position of
//     its first candidate in a strip of LDS; the wave then walks the
//     concatenated candidate list 64 points per step, fully coalesced, and finds
//     the segment of a position as the prefix maximum of the marks.
//   * Each lane evaluates one candidate: serial fp32 sum of squared coordinate
//     differences in coordinate order (no FMA contraction), packed with the
//     candidate's index into a 64-bit key (distance bits high, index low), so a
//     single unsigned compare orders by (distance, index).
//   * The K-1 best keys live in registers, sorted across the lanes (rank r in
//     lane r%64, register r/64). A ballot finds the candidates that beat the
//     current K-th key; each is inserted with one DPP wave shift and two
//     compares, and the new K-th key is read back with a readlane. When 20 or
//     more of a step's 64 candidates enter (the first steps of every query), the
//     step is sorted across the lanes by a bitonic network and merged into the
//     list in one go instead.
//   * The shell loop stops exactly as the reference does: list full and
//     ((bw*d)*bw)*d > K-th distance, or no bin of the shell inside the grid.
//   * Only the rows of a shell that lie inside the grid and within reach of the
//     search get a slot: one per row on a face of the shell (its run), one or
//     two per inner row (its end caps).
//   * Optionally (callers that group the points by half-bin cells) the queries of
//     crowded bins walk a nested grid of half the bin width: walk_shells<FINE>.
//   * The kernel is bound by vector ALU issue; LDS holds only the marks. No
//     atomics, no barriers; every wave is its own workgroup and exits on its own.
#include "hgc_common.hpp"

namespace hgc {
namespace {

constexpr int kMaxBinDims = 5;
constexpr uint64_t kEmptyKey = ~0ull;

struct KnnParams {
    const float *coord;
    const int *bin_idx;
    const int *direction;
    const int *dim_bin_idx;
    const int *bin_boundaries;
    const int *cell_boundaries;  // NESTED kernels: one entry per half-bin cell
    const int *n_bins;
    const float *bin_width;
    const int *sorting;  // may be null
    const float *shift;  // may be null: what the binning subtracted from the binned coordinates
    int *out_idx;
    float *out_dist;
    int *status;      // may be null: device status word for data errors
    float radius_sq;  // < 0: no radius
    int n_vert, K, n_coords, n_bin_dim, n_bboundaries, tf_compat, use_direction;
    int rank_base;       // WINDOW kernels: the neighbour ranks below this one are in the output already
    // fine_bits = n_bin_dim: bin_idx is that of the spatial grouping, bin_idx[q] = bin << fine_bits |
    // half-bin bits, and the points of a bin are grouped by these cells. NESTED kernels: a query
    // whose bin holds more than fine_min_population points walks the nested grid of half the bin
    // width over cell_boundaries.
    int fine_bits, fine_min_population;
};

// The kernel's arguments, read again where they are needed: at eight waves a SIMD a wave has 78 scalar registers, and what
// the compiler keeps in them from the first instruction on (it knows that arguments do not change) it moves to lanes of a
// vector register and back, four at a time, by vector instructions, of which the search is made. (With these, the grid's
// numbers by scalar loads, the first cube's prefix sum used again and no last merge for up to 32 keys: 474 -> 436 vector
// instructions per query of the batch of 16 events, 1156 -> 1097 us; 100,000 2-D Gaussian points, K = 10 124 -> 117; 150,000 4-D
// points, K = 64 1074 -> 1039, 362 -> 356. One of the others taken out again, the batch, three runs each, 1109 to 1119 us with all of
// them: scalar loads 1119 to 1124, prefix sum 1122 to 1133, last merge 1129 to 1137; 1174 without any. Seven waves with more
// registers: 1200. Half-widths 1 and 2 of the first cube looked up together: 1115.)
typedef const __attribute__((address_space(4))) KnnParams *KernelArgs;
__device__ __forceinline__ KernelArgs kernel_args() {
    KernelArgs a = (KernelArgs)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(a));
    return a;
}

// a value of its own, not one of four that were loaded together and stay together
__device__ __forceinline__ int alone(int v) {
    asm("" : "+s"(v));
    return v;
}

// a data error of this lane, into the status word (if there is one)
__device__ __forceinline__ void report(int flag) {
    int *const status = kernel_args()->status;
    if (status) atomicOr(status, flag);
}

template <int C>
__device__ __forceinline__ float dist_sq(const float (&q)[C > 0 ? C : 1], const float *__restrict__ coord, int j,
                                         int n_coords, const float *__restrict__ qrow) {
    float acc = 0.f;
    if constexpr (C > 0) {
        // uniform base + 32-bit byte offset: the load takes its base from scalar registers
        uint32_t offset = (uint32_t)j * (uint32_t)(C * sizeof(float));
        if constexpr (C == 3) {  // 12 j by a shift and a shift-add: a 32-bit multiplication takes four issue slots
            uint32_t j4 = (uint32_t)j << 2;
            asm("" : "+v"(j4));
            offset = (j4 << 1) + j4;
        }
        const float *r = reinterpret_cast<const float *>(reinterpret_cast<const char *>(coord) + offset);
        float x[C];
        if constexpr (C == 4 || C == 8) {  // rows are 16-byte aligned (checked on the host)
#pragma unroll
            for (int c = 0; c < C; c += 4) {
                const float4 v = *reinterpret_cast<const float4 *>(r + c);
                x[c] = v.x; x[c + 1] = v.y; x[c + 2] = v.z; x[c + 3] = v.w;
            }
        } else if constexpr (C == 6) {     // 8-byte aligned
#pragma unroll
            for (int c = 0; c < C; c += 2) {
                const float2 v = *reinterpret_cast<const float2 *>(r + c);
                x[c] = v.x; x[c + 1] = v.y;
            }
        } else if constexpr (C == 2) {
            const float2 v = *reinterpret_cast<const float2 *>(r);
            x[0] = v.x; x[1] = v.y;
        } else {
#pragma unroll
            for (int c = 0; c < C; ++c) x[c] = r[c];
        }
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const float d = q[c] - x[c];
            acc = c == 0 ? d * d : acc + d * d;  // 0 + a square is the square
        }
    } else {
        const float *r = coord + (size_t)j * n_coords;
        for (int c = 0; c < n_coords; ++c) {
            const float d = qrow[c] - r[c];
            acc = acc + d * d;
        }
    }
    return acc;
}

// A value that is the same in every lane, told to the compiler: what is computed from it
// then sits in scalar registers. (Loads through pointers the compiler cannot prove read-only
// are vector loads even at a wave-uniform address.) Not everything gains by it: a vector
// instruction takes one scalar operand only, so values that meet in one instruction, like
// the two edge distances of a dimension, are better left in vector registers.
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ float uniform(float v) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

extern "C" __device__ int __llvm_amdgcn_writelane(int, int, int) __asm("llvm.amdgcn.writelane");

// `into` with lane `lane` (wave-uniform) replaced by the wave-uniform `value`
__device__ __forceinline__ uint64_t writelane_u64(uint64_t value, int lane, uint64_t into) {
    const uint32_t lo = (uint32_t)__llvm_amdgcn_writelane((int)(uint32_t)value, lane, (int)(uint32_t)into);
    const uint32_t hi = (uint32_t)__llvm_amdgcn_writelane((int)(uint32_t)(value >> 32), lane, (int)(uint32_t)(into >> 32));
    return ((uint64_t)hi << 32) | lo;
}

// lane i receives v from lane i-1; lane 0 (and lanes whose source is masked off) read 0
__device__ __forceinline__ uint64_t wave_shift_up1_zero(uint64_t v) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)v, 0x138, 0xf, 0xf, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(v >> 32), 0x138, 0xf, 0xf, true);
    return ((uint64_t)hi << 32) | lo;
}

// Sorted insert of the wave-uniform key c into the ascending list held across
// the lanes (and register levels); the largest key falls off the end. Lanes
// holding a larger key take their left neighbour's key (DPP wave shift under the
// execution mask of exactly those lanes), then c is written into the first of
// them. A key that is larger than everything in the list changes nothing.
template <int S>
__device__ __forceinline__ void sorted_insert(uint64_t (&key)[S], uint64_t c) {
    if constexpr (S == 1) {
        const uint64_t old = key[0];
        const bool larger = old > c;
        const uint64_t run = __builtin_amdgcn_ballot_w64(larger);  // contiguous upper lanes, the list is sorted
        if (run) {
            if (larger) key[0] = wave_shift_up1_zero(old);
            key[0] = writelane_u64(c, __ffsll((long long)run) - 1, key[0]);
        }
    } else {
        uint64_t carry = 0;   // what enters lane 0 of the next register level
        bool placed = false;  // wave-uniform
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const uint64_t old = key[s];
            const uint64_t last = readlane_u64(old, kWave - 1);
            const bool larger = placed || old > c;
            const uint64_t run = __builtin_amdgcn_ballot_w64(larger);
            if (run) {
                if (larger) key[s] = wave_shift_up1_u64(old, carry);
                if (!placed) {
                    key[s] = writelane_u64(c, __ffsll((long long)run) - 1, key[s]);
                    placed = true;
                }
            }
            carry = last;
        }
    }
}

// value of lane `src` (taken modulo 64); one LDS crossbar pass, no bounds logic
__device__ __forceinline__ int from_lane_i32(int v, int src) { return __builtin_amdgcn_ds_bpermute(src << 2, v); }

__device__ __forceinline__ uint64_t from_lane_u64(uint64_t v, int src) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute(src << 2, (int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_ds_bpermute(src << 2, (int)(uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
}

// ---- bulk insert: sort a batch of 64 keys across the lanes and merge it into the list ----
//
// A compare-exchange step of the bitonic network between lanes i and i^J. Which
// of the two lanes keeps the smaller key is a compile-time lane pattern, so it
// sits in scalar registers as a constant and the swap decision is one 64-bit
// compare plus a scalar xor; keys are unique apart from the empty key, for which
// a swap changes nothing.
constexpr uint64_t keeps_min_mask(int k, int j) {
    uint64_t m = 0;
    for (int i = 0; i < 64; ++i)
        if (((i & j) == 0) == ((i & k) == 0)) m |= 1ull << i;
    return m;
}

template <int K, int J>
__device__ __forceinline__ uint64_t compare_exchange(uint64_t key) {
    constexpr uint64_t kMin = keeps_min_mask(K, J);
    const uint64_t other = from_lane_u64(key, lane_id() ^ J);
    const uint64_t lt = __builtin_amdgcn_ballot_w64(other < key);
    // the lane that keeps the smaller key swaps when the other one is smaller, its partner when not
    const bool swap = __builtin_amdgcn_inverse_ballot_w64(lt ^ ~kMin);
    return swap ? other : key;
}

template <int K>
__device__ __forceinline__ uint64_t bitonic_merge_steps(uint64_t key) {
    if constexpr (K >= 64) key = compare_exchange<K, 32>(key);
    if constexpr (K >= 32) key = compare_exchange<K, 16>(key);
    if constexpr (K >= 16) key = compare_exchange<K, 8>(key);
    if constexpr (K >= 8) key = compare_exchange<K, 4>(key);
    if constexpr (K >= 4) key = compare_exchange<K, 2>(key);
    return compare_exchange<K, 1>(key);
}

// ascending sort of one key per lane; the lanes from `n` on hold the empty key, and up to 32 keys need no last merge
__device__ __forceinline__ uint64_t wave_sort_u64(uint64_t key, int n = kWave) {
    key = bitonic_merge_steps<2>(key);
    key = bitonic_merge_steps<4>(key);
    key = bitonic_merge_steps<8>(key);
    key = bitonic_merge_steps<16>(key);
    key = bitonic_merge_steps<32>(key);
    return n <= kWave / 2 ? key : bitonic_merge_steps<64>(key);
}

// the 64 smallest of an ascending list and an ascending batch, ascending:
// min(list[i], batch[63-i]) is a bitonic sequence, six more steps sort it
__device__ __forceinline__ uint64_t merge_lowest_64(uint64_t list, uint64_t batch) {
    const uint64_t rev = from_lane_u64(batch, (kWave - 1) - lane_id());
    return bitonic_merge_steps<128>(rev < list ? rev : list);
}

// Merges an ascending batch of 64 keys into the list of S ascending runs of 64
// (run s holds ranks 64 s .. 64 s + 63): run by run, min(run[i], carry[63-i])
// and max(run[i], carry[63-i]) are bitonic sequences that hold the 64 smallest
// and the 64 largest of the two; six steps sort each, the smaller half stays,
// the larger one is carried to the next run. What falls off the last run is dropped.
template <int S>
__device__ __forceinline__ void merge_batch(uint64_t (&key)[S], uint64_t batch) {
#pragma unroll
    for (int s = 0; s < S; ++s) {
        if (s + 1 == S) {
            key[s] = merge_lowest_64(key[s], batch);
        } else {
            const uint64_t rev = from_lane_u64(batch, (kWave - 1) - lane_id());
            const bool take = rev < key[s];
            const uint64_t low = take ? rev : key[s], high = take ? key[s] : rev;
            key[s] = bitonic_merge_steps<128>(low);
            batch = bitonic_merge_steps<128>(high);
        }
    }
}

// below this many entering candidates in a step of 64 the one-by-one insert is cheaper
// (150,000 points, walks by shells of both kinds, ms a call at 12 / 16 / 20 / 24 / 32: K = 200 4-D clusters 1.42 / 1.37 /
// 1.34 / 1.35 / 1.42, 4-D Gaussian 2.15 / 2.04 / 2.01 / 2.03 / 2.18, 3-D uniform 1.26 / 1.15 / 1.09 / 1.09 / 1.18; K = 64 5-D
// clusters 0.65 / 0.64 / 0.64 / 0.64 / 0.66, 6-D clusters 1.00 / 1.00 / 1.01 / 1.03 / 1.06)
constexpr int kBulkInsertMin = 20;
// lists of more runs than this would insert one by one (a merge costs 12 more steps per run)
constexpr int kBulkInsertMaxRuns = 8;

// NEAR_FIRST (the kernels of the nested grid that walk shells, i.e. 3-D and 4-D points with 130 to 513 neighbours):
// segments of a batch whose bins are at least sqrt(kNearFirst) * d bin widths away (shell d) are walked after the nearer
// ones (150,000 points, K = 200, ms a call without, and at 0.3 / 0.45 / 0.6 / 0.75: 4-D Gaussian 2.69, 1.95 / 2.01 / 2.11 /
// 2.22; 4-D clusters 1.49, 1.35 / 1.32 / 1.31 / 1.33; 4-D uniform 1.79, 1.72 / 1.63 / 1.54 / 1.50; 3-D clusters 1.18, 1.10 /
// 1.05 / 1.02 / 1.03; 3-D Gaussian 1.74, 1.31 / 1.36 / 1.42 / 1.49)
constexpr float kNearFirst = 0.45f;

// Candidates of one batch of segments that are walked per refill of a wave's
// strip of segment marks (one byte of LDS each); a multiple of 512.
constexpr int kMarkCap = 2048;

// How far a place in a grid, in bins, and the bins that points were given may be off: three roundings of the place for the
// query and two for a point, each 2^-24 of the number of bins, twice that for the hardware's reciprocal. A thousandth
// of a bin, which the bounds below allow anyway, covers grids of up to kNarrowGrid bins per dimension; beyond that
// edges count `edge` of a bin less and widths are taken `scale` of themselves (a neighbour beyond the next bin is at
// least half a bin away; where the places are good to less than a quarter of a bin nothing is pruned).
constexpr int kNarrowGrid = 1 << 10;
struct GridSlack {
    float edge, scale;
};
__device__ __forceinline__ GridSlack grid_slack(int most_bins) {
    if (most_bins <= kNarrowGrid) return {1e-3f, 1.f};
    const float off = (float)most_bins * 0x1p-21f;
    return {fmaxf(1e-3f, off), off < 0.25f ? 1.f - 2.f * off : 0.f};
}

// q = x / w, r = x % w for 0 <= x < 2^22 and w < 2^13, without an integer divide: with inv_w
// within an ulp of 1 / w (the hardware's approximate reciprocal will do) the float quotient is
// off by at most one, the remainder says which way
__device__ __forceinline__ void divmod_small(int x, int w, float inv_w, int &q, int &r) {
    q = (int)((float)x * inv_w);
    r = x - q * w;
    const int fix = (r >= w ? 1 : 0) - (r < 0 ? 1 : 0);
    q += fix;
    r -= fix * w;
}

// The walk over the shells of bins around query q (one wave), which leaves the Kn smallest keys
// in `key`. FINE: the walk runs on the nested grid of half the bin width (see KnnParams::fine_bits).
// Its cells are numbered 2 k + h per dimension (bin k, half h); the points of a bin come grouped
// by half-bin cell with the LAST dimension's half as the lowest bit, so a run of cells along the
// last dimension is contiguous inside a bin and falls into one piece per bin it touches: a row of
// the shell at distance d takes up to d + 1 segments instead of one. Any grid gives the same
// result, the K smallest keys: the choice is one of cost only.
//
// A walk on the nested grid gives up (returns false, the list is to be discarded) when it has not
// ended after shell kFineMaxShell: its shells have 2^(B-1) times the rows of the bins' shells
// and more segments per row, which pays only while few of them are needed. All coordinates
// being binned, that is the rule where the bin's neighbourhood is about as crowded as the bin.
constexpr int kFineMaxShell = 3;

template <int C, int NB, int S, bool MAPPED, bool WINDOW, bool FINE, bool NEAR_FIRST, bool CALLERS>
__device__ __forceinline__ bool walk_shells(const KnnParams &p, const int q, const int lane, uint8_t *const marks,
                                            const int Kn, const uint64_t floor_key, uint64_t (&key)[S]) {
    constexpr int kDims = NB > 0 ? NB : kMaxBinDims;  // array extents
    {
        // query coordinates (wave-uniform)
        float qc[C > 0 ? C : 1];
        const float *qrow = p.coord + (size_t)q * p.n_coords;
        if constexpr (C > 0) {
#pragma unroll
            for (int c = 0; c < C; ++c) qc[c] = qrow[c];
        }

        const int B = NB > 0 ? NB : p.n_bin_dim;
        const int own_cell = uniform(p.bin_idx[q]);   // with fine_bits: bin and half-bin bits
        const int own_bin = own_cell >> p.fine_bits;
        int nb[kDims], qb[kDims];
        int cells_per_event = 1, in_event = 0;
        int outside = 0;  // negative: the row lies outside the grid
        int reach_max = 0;  // beyond this shell distance no bin is inside the grid
#pragma unroll
        for (int i = 0; i < kDims; ++i) {
            nb[i] = 1;
            qb[i] = 0;
            if (i < B) {
                nb[i] = uniform(p.n_bins[i]);
                qb[i] = uniform(p.dim_bin_idx[(size_t)q * (B + 1) + 1 + i]);
                cells_per_event *= nb[i];
                in_event = in_event * nb[i] + qb[i];
                if (CALLERS) outside |= qb[i] | (nb[i] - 1 - qb[i]);
                if (FINE) {
                    nb[i] *= 2;
                    qb[i] = 2 * qb[i] + ((own_cell >> (B - 1 - i)) & 1);
                }
                reach_max = max(reach_max, max(qb[i], nb[i] - 1 - qb[i]));
            }
        }
        const int event_base = own_bin - own_bin % max(cells_per_event, 1);
        // A row outside the grid, or of another bin than the own one, does not say where the query is: then the whole grid
        // of the event is walked from the nearest bin inside, and (with bins of no width) nothing is pruned.
        const bool placed = !CALLERS || (outside >= 0 && own_bin - event_base == in_event);
        if (!placed) {
            reach_max = 0;
#pragma unroll
            for (int i = 0; i < kDims; ++i)
                if (i < B) {
                    qb[i] = max(min(qb[i], nb[i] - 1), 0);
                    reach_max = max(reach_max, max(qb[i], nb[i] - 1 - qb[i]));
                }
        }
        const int nb_last = nb[B - 1], qb_last = qb[B - 1];
        const int bins_last = FINE ? nb_last >> 1 : nb_last;  // bins (not cells) along the last dimension
        const float bw = !placed ? 0.f : FINE ? 0.5f * p.bin_width[0] : p.bin_width[0];
        GridSlack slack{1e-3f, 1.f};
        if constexpr (CALLERS) {  // (the package's own grids are narrow)
            int most_bins = 0;
#pragma unroll
            for (int i = 0; i < kDims; ++i) most_bins = max(most_bins, nb[i]);
            slack = grid_slack(most_bins);
        }
        const float inv_bw = 1.f / bw;
        const float gap_bw = bw * slack.scale;           // for lower bounds of distances
        const float bins_per_unit = 1.001f / gap_bw;  // generous by 0.1 %, for the pruning bound only

        // Position of the query inside its own bin, in bin widths: to_lower[i] is a
        // lower bound of its distance to the bin's lower edge, to_upper[i] to the
        // upper edge (both 0 when the binning shift is unknown). They tighten the
        // lower bound of the distance to neighbouring bins used for pruning.
        float to_lower[kDims], to_upper[kDims];
#pragma unroll
        for (int i = 0; i < kDims; ++i) {
            to_lower[i] = 0.f;
            to_upper[i] = 0.f;
            if (i < B && p.shift) {
                const float frac = (qrow[i] - p.shift[i]) * inv_bw - (float)qb[i];
                if (frac >= 0.f && frac <= 1.f) {
                    to_lower[i] = fmaxf(frac - slack.edge, 0.f);
                    to_upper[i] = fmaxf(1.f - frac - slack.edge, 0.f);
                }
            }
        }
        const float tl_last = to_lower[B - 1], tu_last = to_upper[B - 1];

        const bool has_radius = p.radius_sq >= 0.f;
        const int kth_lane = (Kn - 1) & (kWave - 1);
        const int kth_level = (Kn - 1) >> 6;
        // The K-th key is re-read once per step of 64 candidates, not per insert.
        uint64_t thr = kEmptyKey;  // current K-th key: candidates at or above it cannot enter
        // first key beyond the radius: d² <= r² <=> key < (bits(r²) + 1) << 32 for the non-negative r²
        const uint64_t radius_limit = has_radius ? (uint64_t)(__float_as_uint(p.radius_sq) + 1u) << 32 : kEmptyKey;
        uint64_t cut = radius_limit;  // min(thr, radius_limit): what a candidate's key has to stay below

        // Row and slot numbers of a shell are divided as floats (divmod_small), which is exact below
        // 2^22 for divisors below 2^13: no shell has more rows than the grid, times the pieces of
        // a row on the nested grid.
        {
            long long grid_rows = FINE ? nb_last / 2 + 2 : 2;
            bool rows_fit = true, is_grid = event_base >= 0 && nb_last > 0;  // false: a bin, or numbers of bins, that no grid has
            for (int i = 0; i < B - 1; ++i) {
                grid_rows = min(grid_rows * nb[i], 1ll << 40);
                rows_fit = rows_fit && (i == 0 || nb[i] < (1 << 13));  // the leading digit is what the divisions leave
                is_grid = is_grid && nb[i] > 0;
            }
            // (flat bins are 32 bits)
            if (CALLERS && grid_rows < (1ll << 22)) is_grid = is_grid && 2ll * event_base + grid_rows * nb_last <= 1ll << 32;
            if (!rows_fit || grid_rows >= (1ll << 22) || !is_grid) {
                if (FINE) return false;  // the grid of bins may do
                if (p.status && lane == 0) atomicOr(p.status, is_grid ? HGC_FLAG_SHELL_TOO_WIDE : HGC_FLAG_BIN_BEYOND_TABLE);
                return true;  // the list stays empty
            }
        }
        // the first shell whose slots need more than one batch of 64 (walked whole: (2d+1)^(B-1)
        // rows and (2d-1)^(B-1) inner rows; on the nested grid d + 1 pieces per row)
        const int first_cut_shell = FINE ? 2 : (B == 2 ? 17 : B == 3 ? 3 : B == 4 ? 2 : 1);

        // Shell 0 (the query's own bin) never ends the search. When it cannot fill
        // the list either (so that it cannot prune shell 1), it is walked together
        // with shell 1: every row of that shell then takes its whole run of the last
        // dimension, and the run of the centre row contains the own bin.
        bool with_own_bin = false;
        if (reach_max > 0 && own_bin >= 0 && own_bin < p.n_bboundaries - 1) {
            if (FINE)
                with_own_bin = p.cell_boundaries[own_cell + 1] - p.cell_boundaries[own_cell] <= Kn;
            else
                with_own_bin = p.bin_boundaries[own_bin + 1] -
                                   p.bin_boundaries[own_bin] <= Kn;
        }
        for (int d = uniform(with_own_bin ? 1 : 0); d <= reach_max; ++d) {
            if (FINE && d > kFineMaxShell) return false;
            // The shell is walked as rows of bins (cells) along the last dimension. Only rows inside
            // the grid and within reach of the search are numbered: per leading dimension the
            // offsets -below[i] .. -below[i] + width[i] - 1, where an offset o is within reach when
            // (|o| - 1 + distance to the facing edge of the own bin) bin widths do not exceed the
            // K-th distance (the radius) as it is when the shell begins, generously rounded.
            // (A shell whose slots fit one batch anyway is cut to the grid only.)
            const bool cut_to_reach = d >= first_cut_shell;
            float reach_bins = 3.0e9f;
            if (cut_to_reach) {
                float reach2_shell = thr == kEmptyKey ? 3.0e38f : __uint_as_float((uint32_t)(thr >> 32));
                if (has_radius) reach2_shell = fminf(reach2_shell, p.radius_sq);
                if (reach2_shell < 1.0e37f) reach_bins = __builtin_amdgcn_sqrtf(reach2_shell) * bins_per_unit + 1.001f;
            }
            int below[kDims], width[kDims], below_in[kDims], width_in[kDims];
            float inv_width[kDims], inv_width_in[kDims];
            int n_rows = 1;
            int n_inner = 1;  // rows with every leading offset inside +-(d - 1): they contribute end caps only
#pragma unroll
            for (int i = 0; i < kDims - 1; ++i) {
                below[i] = below_in[i] = 0;
                width[i] = width_in[i] = 1;
                inv_width[i] = inv_width_in[i] = 1.f;
                if (i < B - 1) {
                    int lo_i = min(d, qb[i]), hi_i = min(d, nb[i] - 1 - qb[i]);
                    if (cut_to_reach) {
                        lo_i = min(lo_i, uniform((int)fminf(reach_bins - to_lower[i], 1.0e9f)));
                        hi_i = min(hi_i, uniform((int)fminf(reach_bins - to_upper[i], 1.0e9f)));
                    }
                    below[i] = lo_i;
                    width[i] = lo_i + hi_i + 1;
                    below_in[i] = min(lo_i, max(d - 1, 0));
                    width_in[i] = below_in[i] + min(hi_i, max(d - 1, 0)) + 1;
                    if (i > 0) {  // the leading digit of a row number is what the divisions leave
                        inv_width[i] = __builtin_amdgcn_rcpf((float)width[i]);
                        inv_width_in[i] = __builtin_amdgcn_rcpf((float)width_in[i]);
                    }
                    n_rows *= width[i];  // at most the rows of the grid: see rows_fit
                    n_inner *= width_in[i];
                }
            }
            // the last dimension: are the end caps (offsets -d and +d) inside the grid and within reach?
            int lo_last = min(d, qb_last), hi_last = min(d, nb_last - 1 - qb_last);
            if (cut_to_reach) {
                lo_last = min(lo_last, uniform((int)fminf(reach_bins - tl_last, 1.0e9f)));
                hi_last = min(hi_last, uniform((int)fminf(reach_bins - tu_last, 1.0e9f)));
            }
            const bool low_caps = lo_last == d, high_caps = hi_last == d;
            // Segments per row on the nested grid: a run falls into one piece per bin it touches
            // (an inner row uses two of them for its end caps).
            const int P = FINE ? max(2, ((qb_last + hi_last) >> 1) - ((qb_last - lo_last) >> 1) + 1) : 1;
            const float inv_P = __builtin_amdgcn_rcpf((float)P);
            const float near2 = kNearFirst * (bw * (float)d) * (bw * (float)d);
            // Slots of the shell. Grid of bins: one per row (the run of a row on a face of the
            // shell, one end cap of an inner row) and, when both end caps are in reach, one more per
            // inner row. When the own bin is walked with shell 1 every row is a run. Nested grid:
            // P per row.
            const bool runs_only = d == 0 || (d == 1 && with_own_bin);
            const int n_slots = d == 0 ? 1 : FINE ? n_rows * P : (!runs_only && low_caps && high_caps) ? n_rows + n_inner : n_rows;

            // batches of 64 slots; NEAR_FIRST: from the middle of the numbering outwards, so that the rows
            // with small leading offsets, the nearer ones, come first (1 to 2 % of the kernel time)
            const int n_batches = (n_slots + kWave - 1) / kWave;
            for (int slot_lin = 0, turn = 0; slot_lin < n_slots; slot_lin += kWave, ++turn) {
                int slot0 = slot_lin;
                if constexpr (NEAR_FIRST) {
                    const int mid = (n_batches - 1) >> 1;
                    slot0 = kWave * ((turn & 1) ? mid + ((turn + 1) >> 1) : mid - (turn >> 1));
                }
                // ---- each lane resolves one segment of the shell ----
                int seg_start = 0, seg_len = 0;
                [[maybe_unused]] bool far_segment = false;  // NEAR_FIRST: walked after the near ones of its batch
                const int slot = slot0 + lane;
                // Nothing farther than `reach2` can still enter the list (K-th distance
                // once the list is full, the radius cut otherwise). A bin at offset o
                // from the query's bin is at least (|o|-1) bin widths, plus the
                // distance to the facing edge of the own bin, away in that dimension.
                float reach2 = thr == kEmptyKey ? 3.0e38f : __uint_as_float((uint32_t)(thr >> 32));
                if (has_radius) reach2 = fminf(reach2, p.radius_sq);
                if (slot < n_slots) {
                    int row, piece;
                    bool inner = false;  // numbered among the inner rows
                    if (FINE) {
                        divmod_small(slot, P, inv_P, row, piece);
                    } else {
                        inner = slot >= n_rows;
                        row = inner ? slot - n_rows : slot;
                        piece = (inner || !low_caps) ? 1 : 0;  // the end cap an inner row takes in this slot
                    }
                    const bool second = piece == 1;
                    bool on_face = runs_only;
                    int cell = 0, halves = 0;
                    float gap2 = 0.f;  // squared lower bound of the distance to this row of bins
                    int off[kDims];
#pragma unroll
                    for (int i = kDims - 2; i >= 0; --i) {
                        off[i] = 0;
                        if (i < B - 1) {
                            // digits of the row number: offsets of the leading dimensions
                            const int below_i = inner ? below_in[i] : below[i];
                            if (i > 0) {
                                int digit;
                                divmod_small(row, inner ? width_in[i] : width[i], inner ? inv_width_in[i] : inv_width[i],
                                             row, digit);
                                off[i] = digit - below_i;
                            } else {
                                off[i] = row - below_i;  // what is left is the leading digit
                            }
                        }
                    }
#pragma unroll
                    for (int i = 0; i < kDims - 1; ++i) {
                        if (i < B - 1) {
                            const int o = off[i];
                            const int k = qb[i] + o;  // inside the grid: the numbered rows all are
                            on_face = on_face || o == d || o == -d;
                            if (FINE) {
                                cell = cell * (nb[i] >> 1) + (k >> 1);
                                halves = (halves << 1) | (k & 1);
                            } else {
                                cell = cell * nb[i] + k;
                            }
                            const float edge = o > 0 ? to_upper[i] : to_lower[i];
                            const float g = o == 0 ? 0.f : ((float)(abs(o) - 1) + edge) * gap_bw;
                            gap2 += g * g;
                        }
                    }
                    // a whole run of the last dimension (rows on a face of the shell), or one of the
                    // two end caps
                    const float cap_gap = ((float)(d - 1) + (second ? tu_last : tl_last)) * gap_bw;
                    const float cap2 = gap2 + cap_gap * cap_gap;
                    // bins of a run that are provably too far are cut off (bound
                    // generous by 0.1 % and a thousandth of a bin)
                    const float rest = fmaxf(reach2 - 0.999f * gap2, 0.f);
                    const float span = rest < 1.0e37f ? __builtin_amdgcn_sqrtf(rest) * bins_per_unit + 1.001f : 3.0e9f;
                    const int run_lo = max(qb_last - d, qb_last - (int)fminf(span - tl_last, 1.0e9f));
                    const int run_hi = min(qb_last + d, qb_last + (int)fminf(span - tu_last, 1.0e9f));
                    const int cap = second ? qb_last + d : qb_last - d;
                    int lo = on_face ? run_lo : cap;
                    int hi = on_face ? run_hi : cap;
                    bool too_far = on_face ? 0.999f * gap2 > reach2 : (piece > 1 || 0.999f * cap2 > reach2);
                    if constexpr (NEAR_FIRST) far_segment = (on_face ? gap2 : cap2) > near2;
                    lo = max(lo, 0);
                    hi = min(hi, nb_last - 1);
                    if (FINE) {
                        if (on_face) {
                            // piece number `piece` of the run: the part inside one bin, counted from the
                            // first bin any run of this shell can touch (not from this row's own first
                            // bin: the run shrinks with the K-th distance while the row's slots may lie
                            // in two batches)
                            const int bin = ((qb_last - lo_last) >> 1) + piece;
                            lo = max(lo, 2 * bin);
                            hi = min(hi, 2 * bin + 1);
                        }
                    }
                    if (!too_far && lo <= hi) {
                        if (FINE) {
                            const int bin = event_base + cell * bins_last + (lo >> 1);
                            if (bin + 1 < p.n_bboundaries) {
                                const int first = (((bin << (B - 1)) | halves) << 1) | (lo & 1);
                                const int last = ((((bin << (B - 1)) | halves) << 1) | (hi & 1)) + 1;
                                seg_start = p.cell_boundaries[first];
                                seg_len = p.cell_boundaries[last] - seg_start;
                            } else if (p.status) {
                                atomicOr(p.status, HGC_FLAG_BIN_BEYOND_TABLE);
                            }
                        } else {
                            const int first = event_base + cell * nb_last + lo;
                            const int last = event_base + cell * nb_last + hi + 1;
                            // bins beyond the table are skipped, as by the reference, which prints "idx out of range"
                            if constexpr (CALLERS) {
                                const int there = min(last, p.n_bboundaries - 1);
                                if (first < there) {
                                    seg_start = p.bin_boundaries[first];
                                    seg_len = p.bin_boundaries[there] - seg_start;
                                }
                                if (p.status && there < last) atomicOr(p.status, HGC_FLAG_BIN_BEYOND_TABLE);
                            } else if (last < p.n_bboundaries) {
                                seg_start = p.bin_boundaries[first];
                                seg_len = p.bin_boundaries[last] - seg_start;
                            } else if (p.status) {
                                atomicOr(p.status, HGC_FLAG_BIN_BEYOND_TABLE);
                            }
                        }
                    }
                }
                // The segments whose lower bound of the distance is within near2 come first in the
                // candidate list, the others behind them (marks 65..128, so that the prefix maximum
                // keeps the two apart): fewer candidates enter the list only to be pushed out again.
                int seg_off, total;
                uint8_t mark;
                if constexpr (NEAR_FIRST) {
                    const int end_near = wave_inclusive_sum(far_segment ? 0 : seg_len);
                    const int end_far = wave_inclusive_sum(far_segment ? seg_len : 0);
                    const int total_near = readlane_i32(end_near, kWave - 1);
                    seg_off = (far_segment ? total_near + end_far : end_near) - seg_len;
                    total = total_near + readlane_i32(end_far, kWave - 1);
                    mark = (uint8_t)(lane + (far_segment ? kWave + 1 : 1));
                } else {
                    const int seg_end_off = wave_inclusive_sum(seg_len);
                    seg_off = seg_end_off - seg_len;
                    total = readlane_i32(seg_end_off, kWave - 1);
                    mark = (uint8_t)(lane + 1);
                }
                // candidate position -> point index for the owning segment; kept one lane up,
                // so that the mark (lane number + 1) is the lane to read it from
                // (DPP wave_ror:1; lane 63's value goes to lane 0, which is where mark 64 reads)
                const int seg_delta = __builtin_amdgcn_update_dpp(0, seg_start - seg_off, 0x13c, 0xf, 0xf, false);

                // ---- walk the concatenated candidates, 64 per step ----
                // Every non-empty segment marks its first position of the list with its
                // lane number + 1 (+ 64 for the far ones) in this wave's strip of LDS; the owner of a
                // position is then the prefix maximum of the marks (offsets rise with the lane).
                uint32_t owner_carry = 0;
                for (int c0 = 0; c0 < total; c0 += kMarkCap) {
                    const int chunk = min(kMarkCap, total - c0);
                    for (int base = 0; base < chunk; base += kWave * 8)
                        *reinterpret_cast<uint64_t *>(marks + base + lane * 8) = 0;
                    wave_lds_fence();
                    const int rel = seg_off - c0;
                    if (seg_len > 0 && rel >= 0 && rel < chunk) marks[rel] = mark;
                    wave_lds_fence();
                    for (int t = 0; t < chunk; t += kWave) {
                        const int c = c0 + t + lane;
                        uint32_t owner = wave_inclusive_max(marks[t + lane]);
                        owner = max(owner, owner_carry);
                        owner_carry = (uint32_t)readlane_i32((int)owner, kWave - 1);
                        const int j = c + from_lane_i32(seg_delta, (int)owner);
                        // lane masks are combined as integers on the scalar side
                        const bool in_list = c < total;
                        uint64_t valid = __builtin_amdgcn_ballot_w64(in_list) & __builtin_amdgcn_ballot_w64(j != q);
                        const int jj = in_list ? j : q;
                        const uint32_t id = MAPPED ? *reinterpret_cast<const uint32_t *>(
                                                         reinterpret_cast<const char *>(p.sorting) + ((uint32_t)jj << 2))
                                                   : (uint32_t)jj;
                        const float dsq = dist_sq<C>(qc, p.coord, jj, p.n_coords, qrow);
                        if (p.use_direction) {
                            const int dj = p.direction[jj];
                            valid &= ~__builtin_amdgcn_ballot_w64(dj == 1 || dj == 2);  // may not be a neighbour
                        }
                        const uint64_t ck = ((uint64_t)__float_as_uint(dsq) << 32) | id;
                        if (WINDOW) valid &= __builtin_amdgcn_ballot_w64(ck > floor_key);
                        // below the K-th key and (keys compare like distances) within the radius
                        uint64_t beats = valid & __builtin_amdgcn_ballot_w64(ck < cut);
                        if (beats) {
                            if (S <= kBulkInsertMaxRuns && (int)__popcll(beats) >= kBulkInsertMin) {
                                const bool enters = __builtin_amdgcn_inverse_ballot_w64(beats);
                                const uint64_t batch = wave_sort_u64(enters ? ck : kEmptyKey);
                                // an empty list (its smallest key is the empty key) is replaced
                                if (readlane_u64(key[0], 0) == kEmptyKey) key[0] = batch;
                                else merge_batch<S>(key, batch);
                                beats = 0;
                            }
                            while (beats) {
                                const int src = __ffsll((long long)beats) - 1;
                                beats &= beats - 1;
                                const uint64_t cand = readlane_u64(ck, src);
                                // a candidate that an earlier insert of this step has pushed beyond the
                                // K-th rank lands in a spare rank behind it or, in a list without one,
                                // is larger than every key and changes nothing
                                sorted_insert<S>(key, cand);
                            }
#pragma unroll
                            for (int s = 0; s < S; ++s)
                                if (s == kth_level) thr = readlane_u64(key[s], kth_lane);
                            // the low word of radius_limit is 0: the high words decide
                            cut = (uint32_t)(thr >> 32) < (uint32_t)(radius_limit >> 32) ? thr : radius_limit;
                        }
                    }
                }
            }

            // stop rule (fp32, evaluated left to right); on the nested grid, which the reference does
            // not have, with a margin for points that rounding has put into the neighbouring cell
            float reach = bw * (float)d;
            reach = reach * bw;
            reach = reach * (float)d;
            if (FINE) reach *= 0.998f;
            uint64_t kth = kEmptyKey;
#pragma unroll
            for (int s = 0; s < S; ++s)
                if (s == kth_level) kth = readlane_u64(key[s], kth_lane);
            if (kth != kEmptyKey && reach > __uint_as_float((uint32_t)(kth >> 32))) break;
            if (has_radius && reach > p.radius_sq) break;
        }
    }
    return true;
}

// ---- the search of up to 129 neighbours: collect, cut, sort once ----
//
// Bound by the issue of vector instructions (80 % busy), as walk_shells is, and most of those went into resolving the
// segments of one small shell after another, steps with a few candidates, and sorted inserts of keys that leave the
// list again. Here a query collects candidates, unsorted, in LDS:
//   * first the cube of bins around it that holds enough points (the boundary table says how many, before any
//     distance), or the next larger ones until Kn candidates are collected;
//   * then the Kn-th distance is bounded by bisection (counts are ballots) and what lies beyond is dropped;
//   * then one pass over the rows of bins outside the cube that the bound reaches;
//   * then the keys that are left are sorted, once.
// Vector instructions per query: 16 events of 1.14 M 3-D points, K = 32, radius 0.1 about 700 -> 474, 150,000 4-D
// points, K = 64 1476 -> 1074 (now 436 and 1039, see kernel_args). The whole search, by shells -> collected: these two 1399 -> 1173 us and 429 -> 372 us;
// 240,000 3-D points, K = 41 367 -> 307; 4-D Gaussian, K = 65 467 -> 410; 4-D uniform, K = 64 361 -> 305; 2-D
// clusters, K = 32 186 -> 130; 3-D clusters, K = 96 489 -> 319. Tried and taken back: first regions that leave out the
// corners of the cube (fewer candidates, but a second pass for every query: 4 to 13 % slower), up to three pieces of a
// row per lane on the nested grid (level in 4-D, 3-D 7 % slower), two queries per wave one after the other (level).
constexpr int kBufferKeys = 256;  // collected keys per query, in LDS
// The first cube holds more than Kn + Kn / 2 points. 16 events of 3-D points, K = 32, radius 0.1: 1188 / 1186 / 1182 /
// 1173 / 1163 us for 1 / 1.125 / 1.25 / 1.5 / 2 Kn; 4-D Gaussian, K = 32: 408 us up to 1.5, 437 at 2; others level.
constexpr int kFirstCubeShift = 1;
constexpr int kFineMaxCube = 3;  // on the nested grid a query gives up beyond this half-width

// keys 0 .. n of `buffer` cut down to between Kn and `most` of the smallest (Kn <= most <= n): returns how many are
// left; the key (cut, cut_id) becomes one that the Kn-th smallest does not exceed. Distances first, and where more
// than `most` keys share the Kn-th distance the indices decide. REPEATED: a key may be there several times.
template <bool REPEATED>
__device__ __forceinline__ int cut_to_smallest(uint64_t *const buffer, const int lane, const int n, const int Kn,
                                               const int most, uint32_t &cut, uint32_t &cut_id) {
    constexpr int kRegs = kBufferKeys / kWave;
    uint64_t k[kRegs];
    uint32_t largest = 0;
#pragma unroll
    for (int u = 0; u < kRegs; ++u) {
        k[u] = kEmptyKey;
        if (u * kWave < n) {
            const bool there = u * kWave + lane < n;
            if (there) k[u] = buffer[u * kWave + lane];
            largest = max(largest, there ? (uint32_t)(k[u] >> 32) : 0u);
        }
    }
    uint32_t hi = (uint32_t)readlane_i32((int)wave_inclusive_max(largest), kWave - 1);
    // (empty lanes count when hi is the pattern of all ones; no square has it)
    auto count = [&](uint32_t limit) {
        int c = 0;
#pragma unroll
        for (int u = 0; u < kRegs; ++u)
            if (u * kWave < n) c += (int)__popcll(__builtin_amdgcn_ballot_w64((uint32_t)(k[u] >> 32) <= limit));
        return c;
    };
    int left = n;
    uint32_t tie_limit = 0xffffffffu;  // keys at distance `hi` stay up to this index
    if (n > most) {
        uint32_t lo = 0, step = 2u << 23;  // count(lo) < Kn, or lo = 0
        for (;;) {
            lo = hi > step ? hi - step : 0;
            if (lo == 0) break;
            const int c = count(lo);
            if (c < Kn) break;
            hi = lo;
            left = c;
            step = min(2 * step, 1u << 30);
            if (left <= most) break;
        }
        while (left > most && hi - lo > 1) {
            const uint32_t mid = lo + ((hi - lo) >> 1);
            const int c = count(mid);
            if (c >= Kn) {
                hi = mid;
                left = c;
            } else {
                lo = mid;
            }
        }
        if (left > most && lo == 0) {
            const int c = count(0);
            if (c >= Kn) {
                hi = 0;
                left = c;
            }
        }
        if (left > most) {  // more than `most` - Kn keys share the Kn-th distance
            uint32_t tie_lo = 0;  // fewer than Kn keys with this limit, or 0 (Kn at most)
            uint32_t last_id = 0;  // of the keys within `hi`: halving from 2^32 down to it is most of the steps otherwise
#pragma unroll
            for (int u = 0; u < kRegs; ++u) last_id = max(last_id, (uint32_t)(k[u] >> 32) <= hi ? (uint32_t)k[u] : 0u);
            tie_limit = (uint32_t)readlane_i32((int)wave_inclusive_max(last_id), kWave - 1);
            while (left > most && tie_limit - tie_lo > 1) {
                const uint32_t mid = tie_lo + ((tie_limit - tie_lo) >> 1);
                const uint64_t limit = (uint64_t)hi << 32 | mid;
                int c = 0;
#pragma unroll
                for (int u = 0; u < kRegs; ++u) c += (int)__popcll(__builtin_amdgcn_ballot_w64(k[u] <= limit));
                if (c >= Kn) {
                    tie_limit = mid;
                    left = c;
                } else {
                    tie_lo = mid;
                }
            }
            // one too many with the limit 1: points 0 and 1 share the Kn-th distance, and point 0 completes the list
            if (!REPEATED && left > most) tie_limit = 0;
            if (REPEATED && left > most) {  // that, or a key many times over, of which as many stay as fit
                auto count_up_to = [&](uint64_t limit) {
                    int c = 0;
#pragma unroll
                    for (int u = 0; u < kRegs; ++u) c += (int)__popcll(__builtin_amdgcn_ballot_w64(k[u] <= limit));
                    return c;
                };
                const uint64_t first_id = (uint64_t)hi << 32;
                if (tie_limit == 1 && count_up_to(first_id) >= Kn) tie_limit = 0;
                const uint64_t limit = first_id | tie_limit;
                int spare = most - (limit > 0 ? count_up_to(limit - 1) : 0);
#pragma unroll
                for (int u = 0; u < kRegs; ++u) {
                    const uint64_t same = __builtin_amdgcn_ballot_w64(k[u] == limit);
                    const int before = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(same >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)same, 0));
                    if (k[u] == limit && before >= spare) k[u] = kEmptyKey;
                    spare = max(0, spare - (int)__popcll(same));
                }
            }
        }
        const uint64_t limit = (uint64_t)hi << 32 | tie_limit;
        int at = 0;
        wave_lds_fence();
#pragma unroll
        for (int u = 0; u < kRegs; ++u) {
            if (u * kWave < n) {
                const uint64_t m = __builtin_amdgcn_ballot_w64(k[u] <= limit && u * kWave + lane < n);
                const int before = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
                if (__builtin_amdgcn_inverse_ballot_w64(m)) buffer[at + before] = k[u];
                at += (int)__popcll(m);
            }
        }
        wave_lds_fence();
        left = at;
    }
    cut = min(cut, hi);
    cut_id = tie_limit;
    return left;
}

// table[i] with the table in scalar registers and a 32-bit byte offset (the package's own tables, below 2^30 entries)
__device__ __forceinline__ int table_entry(const int *__restrict__ table, int i) {
    return *reinterpret_cast<const int *>(reinterpret_cast<const char *>(table) + ((uint32_t)i << 2));
}

// Taken where every coordinate is binned and up to 129 neighbours are asked for. With more coordinates the Kn-th
// distance is many bins wide, and the walk by shells, which tightens it as it goes, looks at fewer candidates (80,000
// points in 5-D, 4 of them binned, K = 32: 423 us by shells, 635 us collected).
constexpr bool collects(int C, int NB, int S, bool window) { return C == NB && NB >= 2 && NB <= 4 && S <= 2 && !window; }

// a bound of the squared distances with this pattern or a smaller one; at least the smallest normal number, since the
// hardware's square root takes smaller ones as zero
__device__ __forceinline__ float bound_of(uint32_t pattern) { return __uint_as_float(max(pattern, 0x00800000u)); }

// The Kn smallest keys of query q, ascending, in `key` (ranks beyond the points there are: the empty key). FINE as in
// walk_shells. False: nothing is decided (the grid of bins, or walk_shells, has to do it). CALLERS as in knn_wave_kernel.
template <int C, int NB, int S, bool MAPPED, bool FINE, bool CALLERS>
__device__ __forceinline__ bool collect_nearest(const KnnParams &p, const int q, const int lane, uint8_t *const marks,
                                                uint64_t *const buffer, const int Kn, uint64_t (&key)[S]) {
    static_assert(C > 0 && NB >= 2 && NB <= 4 && S <= 2 && (!FINE || NB >= 3));
    constexpr int B = NB;
    const int n_bboundaries = alone(p.n_bboundaries);
    const bool use_direction = alone(p.use_direction) != 0;
    float qc[C];
    const float *qrow = p.coord + (size_t)q * C;
#pragma unroll
    for (int c = 0; c < C; ++c) qc[c] = qrow[c];

    // Dimension i of the query's place in the grid is worked out in lane i (one vector instruction for all of them)
    // and read from there.
    const int own_cell = uniform(p.bin_idx[q]);
    const int own_bin = own_cell >> p.fine_bits;
    const int dim = min(lane, B - 1);
    int nb_v = p.n_bins[dim], qb_v = p.dim_bin_idx[(size_t)q * (B + 1) + 1 + dim];
    int in_event = 0, cells_per_event = 1;  // number of the own bin inside its event
    [[maybe_unused]] int nb_s[B], qb_s[B];  // the same by scalar loads
#pragma unroll
    for (int i = 0; i < B; ++i) {
        nb_s[i] = p.n_bins[i], qb_s[i] = p.dim_bin_idx[(size_t)q * (B + 1) + 1 + i];
        in_event = in_event * nb_s[i] + qb_s[i];
        cells_per_event *= nb_s[i];
    }
    int event_base = own_bin - in_event;
    bool placed = true;
    if constexpr (CALLERS) {
        // The bin says which event it is. A row outside the grid, or of another bin than the own one, does not say where
        // the query is: then the whole grid of the event is walked from the nearest bin inside, and nothing is pruned.
        event_base = own_bin - own_bin % max(cells_per_event, 1);
        placed = own_bin - event_base == in_event && !__builtin_amdgcn_ballot_w64((uint32_t)qb_v >= (uint32_t)nb_v);
        if (!placed) qb_v = max(min(qb_v, nb_v - 1), 0);
    }
    if (FINE) {
        nb_v *= 2;
        qb_v = 2 * qb_v + ((own_cell >> (B - 1 - dim)) & 1);
    }
    const int top_v = nb_v - 1 - qb_v;  // bins above the own one
    int nb[B], qb[B];
    long long grid_rows = 1;
    bool rows_fit = true;
#pragma unroll
    for (int i = 0; i < B; ++i) {
        nb[i] = FINE ? 2 * nb_s[i] : nb_s[i];
        qb[i] = CALLERS ? readlane_i32(qb_v, i) : FINE ? 2 * qb_s[i] + ((own_cell >> (B - 1 - i)) & 1) : qb_s[i];
        if (i < B - 1) {
            grid_rows *= nb[i];
            rows_fit = rows_fit && (i == 0 || nb[i] < (1 << 13)) && (!CALLERS || nb[i] > 0);
        }
    }
    const int nb_last = nb[B - 1], qb_last = qb[B - 1];
    const int bins_last = FINE ? nb_last >> 1 : nb_last;
    grid_rows *= FINE ? bins_last + 1 : 2;  // slots of a pass
    bool no_grid = event_base < 0;  // a bin, or numbers of bins, that no grid has
    if (CALLERS && grid_rows < (1ll << 22))  // (grid_rows is twice the rows here; flat bins are 32 bits)
        no_grid = no_grid || grid_rows <= 0 || nb_last < 1 || event_base >= n_bboundaries - 1 || 2ll * event_base + grid_rows * nb_last > 1ll << 32;
    if (!rows_fit || grid_rows >= (1ll << 22) || no_grid) {  // see divmod_small
        if (FINE) return false;  // the grid of bins may do
        if (lane == 0) report(no_grid ? HGC_FLAG_BIN_BEYOND_TABLE : HGC_FLAG_SHELL_TOO_WIDE);
        return true;  // the list stays empty
    }
    const float bw = !placed ? 0.f : FINE ? 0.5f * p.bin_width[0] : p.bin_width[0];
    // Coordinates without bounds leave widths without a meaning: then nothing is pruned, the whole grid is walked.
    bool prunes = bw > 1e-30f && bw < 1e18f;  // (the square stays finite)
    const float inv_bw = __builtin_amdgcn_rcpf(bw);  // within an ulp
    float bins_per_unit = 1.001f * inv_bw, gap_scale = 0.999f * (bw * bw);  // bounds are generous by 0.1 %
    GridSlack slack{1e-3f, 1.f};
    if constexpr (CALLERS) {  // (the package's own grids are narrow)
        int most_bins = nb_last;
#pragma unroll
        for (int i = 0; i < B - 1; ++i) most_bins = max(most_bins, nb[i]);
        slack = grid_slack(most_bins);
        prunes = prunes && slack.scale > 0.f;
        bins_per_unit /= slack.scale;
        gap_scale *= slack.scale * slack.scale;
    }
    if (!prunes) bins_per_unit = 3.0e38f, gap_scale = 0.f;

    // number of the first bin of a row of the grid, from the number of the row
    auto row_base = [&](int row) {
        return event_base + (CALLERS ? row * bins_last : (int)__umul24(row, bins_last));
    };
    // a caller's table: the points of bins first .. last - 1 of a row, without the bins beyond the table, which are skipped
    // as by the reference, which prints "idx out of range"
    int seg_start = 0, seg_len = 0;
    [[maybe_unused]] auto callers_run = [&](int first, int last) {
        const int there = min(last, n_bboundaries - 1);
        if (first < there) {
            seg_start = p.bin_boundaries[first];
            seg_len = p.bin_boundaries[there] - seg_start;
        }
        if (there < last) report(HGC_FLAG_BIN_BEYOND_TABLE);
    };

    // lower bounds of the distance to the edges of the own bin, in bin widths, as in walk_shells
    float tl_v = 0.f, tu_v = 0.f;
    if (p.shift) {
        const float frac = (qrow[dim] - p.shift[dim]) * inv_bw - (float)qb_v;
        if (frac >= 0.f && frac <= 1.f) {
            tl_v = fmaxf(frac - slack.edge, 0.f);
            tu_v = fmaxf(1.f - frac - slack.edge, 0.f);
        }
    }
    float from_lower[B], from_upper[B];  // 1 - these bounds
#pragma unroll
    for (int i = 0; i < B - 1; ++i) {
        from_lower[i] = __int_as_float(readlane_i32(__float_as_int(1.f - tl_v), i));
        from_upper[i] = __int_as_float(readlane_i32(__float_as_int(1.f - tu_v), i));
    }
    const float tl_last = __int_as_float(readlane_i32(__float_as_int(tl_v), B - 1));
    const float tu_last = __int_as_float(readlane_i32(__float_as_int(tu_v), B - 1));

    const bool has_radius = p.radius_sq >= 0.f;
    // candidates beyond this distance pattern are not collected: the radius, then the bound of the Kn-th distance
    uint32_t cut = has_radius ? __float_as_uint(p.radius_sq) : 0xffffffffu;
    uint32_t cut_id = 0xffffffffu;  // and at this distance those beyond this index
    const int kept = Kn + (Kn >> 2) + 4;  // a cut leaves up to so many keys

    // The first cube: the smallest one that holds more than `enough` points, of half-width 0 .. kCubes (no wider than
    // the radius asks for). One lane per row of bins (on the nested grid per row and bin that the row's three cells
    // touch, always two).
    const int enough = Kn + (Kn >> kFirstCubeShift);
    int first_end = 0;  // prefix sum of the rows' lengths
    int d_out, d_radius = 1 << 30;  // the cube of half-width d_radius holds everything within the radius
    if (has_radius && prunes)
        d_radius = max(1, uniform((int)fminf(__builtin_ceilf(__builtin_amdgcn_sqrtf(bound_of(__float_as_uint(p.radius_sq))) * bins_per_unit), 1.0e9f)));
    {
        int off[B], ring = 0;
        bool in_grid = true;
        if constexpr (FINE) {
            int row = lane >> 1;
            in_grid = row < (B == 3 ? 9 : 27);
#pragma unroll
            for (int i = B - 2; i >= 0; --i) {
                off[i] = (i > 0 ? row % 3 : row) - 1;
                row /= 3;
            }
        } else if constexpr (B == 4) {
            off[0] = (lane >> 4) - 1, off[1] = ((lane >> 2) & 3) - 1, off[2] = (lane & 3) - 1;
        } else if constexpr (B == 3) {
            off[0] = (lane >> 3) - 3, off[1] = (lane & 7) - 3;
        } else {
            off[0] = lane - 3;
        }
        int cell = 0, halves = 0;
#pragma unroll
        for (int i = 0; i < B - 1; ++i) {
            const int k = qb[i] + off[i];
            in_grid = in_grid && (uint32_t)k < (uint32_t)nb[i];
            ring = max(ring, abs(off[i]));
            if (FINE) {
                cell = (int)__umul24(cell, nb[i] >> 1) + (k >> 1);
                halves = (halves << 1) | (k & 1);
            } else {
                cell = (int)__umul24(cell, nb[i]) + k;
            }
        }
        // What the radius leaves of a row: with bins wider than the radius the cube is mostly beyond it (60,000 4-D Gaussian
        // points, radius 0.1, K = 40: 139 -> 80 us a call; 16 events of 1.14 M points, radius 0.1: 1183 -> 1171).
        int lo_most = 1 << 30, hi_most = 1 << 30;
        if (has_radius && prunes) {
            float gap2 = 0.f;
#pragma unroll
            for (int i = 0; i < B - 1; ++i) {
                const float of = (float)off[i];
                const float g = fmaxf(fmaxf(of - from_upper[i], -of - from_lower[i]), 0.f);
                gap2 = __builtin_fmaf(g, g, gap2);
            }
            const float rest = bound_of(cut) - gap2 * gap_scale;
            const float span = __builtin_amdgcn_sqrtf(fmaxf(rest, 0.f)) * bins_per_unit + 1.001f;
            in_grid = in_grid && rest >= 0.f;
            lo_most = (int)fminf(span - tl_last, 1.0e9f);
            hi_most = (int)fminf(span - tu_last, 1.0e9f);
        }
        if constexpr (FINE) {
            const int own = uniform(p.cell_boundaries[own_cell + 1]) - uniform(p.cell_boundaries[own_cell]);
            d_out = own > enough ? 0 : 1;
            const int bin_last = ((qb_last - 1) >> 1) + (lane & 1);
            const int lo = max(max(qb_last - min(d_out, lo_most), 0), 2 * bin_last);
            const int hi = min(min(qb_last + min(d_out, hi_most), nb_last - 1), 2 * bin_last + 1);
            const int bin = row_base(cell) + bin_last;
            if (in_grid && ring <= d_out && lo <= hi && bin + 1 < n_bboundaries) {
                const int base = ((bin << (B - 1)) | halves) << 1;
                seg_start = table_entry(p.cell_boundaries, base | (lo & 1));
                seg_len = table_entry(p.cell_boundaries, (base | (hi & 1)) + 1) - seg_start;
            }
            if (in_grid && ring <= d_out && lo <= hi && bin + 1 >= n_bboundaries) report(HGC_FLAG_BIN_BEYOND_TABLE);
        } else {
            constexpr int kCubes = B == 4 ? 1 : 3;
            // lanes without a row look at the own one
            const int row = in_grid ? row_base(cell) : own_bin - qb_last;
            auto look = [&](int d) {  // the part of the row inside the cube of half-width d
                const int from = max(qb_last - min(d, lo_most), 0), to = min(qb_last + min(d, hi_most), nb_last - 1) + 1;
                seg_start = seg_len = 0;
                if constexpr (CALLERS) {
                    if (in_grid && ring <= d && from < to) callers_run(row + from, row + to);
                } else {
                    const bool wanted = in_grid && ring <= d && row < n_bboundaries - to;
                    if (wanted) {
                        seg_start = table_entry(p.bin_boundaries, row + from);
                        seg_len = table_entry(p.bin_boundaries, row + to) - seg_start;
                    }
                    if (in_grid && ring <= d && !wanted) report(HGC_FLAG_BIN_BEYOND_TABLE);
                }
                first_end = wave_inclusive_sum(seg_len);
                return readlane_i32(first_end, kWave - 1);
            };
            d_out = 1;
            const int held = look(1);
            if (kCubes > 1 && held <= enough && d_radius > 1) {
                d_out = 2;
                if (look(2) <= enough && d_radius > 2) {
                    d_out = 3;
                    look(3);
                }
            } else if (held > 4 * enough && placed && own_bin + 1 < n_bboundaries &&
                       uniform(p.bin_boundaries[own_bin + 1]) - uniform(p.bin_boundaries[own_bin]) > enough) {
                d_out = 0;  // crowded: the own bin does
                look(0);
            }
            d_out = uniform(d_out);
        }
        if (FINE) first_end = wave_inclusive_sum(seg_len);
    }

    int n_kept = 0;  // keys in the buffer
    // Where keys have been cut at one distance, every step with a candidate compares indices too: the buffer counts as full.
    // Without it all candidates at the Kn-th distance enter and the buffer is cut every few steps: 4000 points in one place,
    // 3-D, K = 65 240 us, with it 102 (by shells 118); 20,000 on a lattice of 5^4 sites, K = 129 357 -> 238 (235). Compared in
    // every step the indices cost searches without equal distances 0.5 to 2 %.
    int room = kBufferKeys;
    int d_in = -1;   // the cube of this half-width has been walked (-1: none)
    for (;;) {
        const bool bounded = prunes && cut < 0x7f000000u;
        // Everything within the bound; where the list is not full and a radius reaches far, larger cubes come first (with
        // radius 3 in the unit square, 60,000 points, K = 40 one pass over everything takes 1045 us, this 97).
        const bool last_pass = bounded && d_in >= 0 && (n_kept >= Kn || d_radius <= 2 * d_in + 2);
        int below[B], width[B], below_in[B], width_in[B];
        float inv_width[B], inv_width_in[B];
        int n_rows = 1, n_inner = 1, lo_last = 0, hi_last = 0, first_bin = 0, P = 1, n_slots = 1;
        bool low_caps = false, high_caps = false;
        float inv_P = 1.f;
        if (d_in >= 0) {
            float reach_bins = 3.0e9f;
            if (bounded) reach_bins = __builtin_amdgcn_sqrtf(bound_of(cut)) * bins_per_unit + 1.001f;
            if (FINE && (last_pass ? reach_bins > (float)(kFineMaxCube + 2) : d_out > kFineMaxCube)) return false;
            const int d_most = last_pass ? 1 << 30 : d_out;
            const int lo_v = min(min(d_most, qb_v), (int)fminf(reach_bins - tl_v, 1.0e9f));
            const int hi_v = min(min(d_most, top_v), (int)fminf(reach_bins - tu_v, 1.0e9f));
            bool beyond = false;  // anything outside the cube walked before
#pragma unroll
            for (int i = 0; i < B - 1; ++i) {
                const int lo_i = readlane_i32(lo_v, i), hi_i = readlane_i32(hi_v, i);
                below[i] = lo_i;
                width[i] = lo_i + hi_i + 1;
                below_in[i] = min(lo_i, d_in);
                width_in[i] = below_in[i] + min(hi_i, d_in) + 1;
                inv_width[i] = inv_width_in[i] = 1.f;
                if (i > 0) {
                    inv_width[i] = __builtin_amdgcn_rcpf((float)width[i]);
                    inv_width_in[i] = __builtin_amdgcn_rcpf((float)width_in[i]);
                }
                n_rows *= width[i];
                n_inner *= width_in[i];
                beyond = beyond || lo_i > d_in || hi_i > d_in;
            }
            lo_last = readlane_i32(lo_v, B - 1);
            hi_last = readlane_i32(hi_v, B - 1);
            low_caps = lo_last > d_in;
            high_caps = hi_last > d_in;
            if (!beyond && !low_caps && !high_caps) break;
            if (FINE) {
                first_bin = (qb_last - lo_last) >> 1;
                P = ((qb_last + hi_last) >> 1) - first_bin + 1;
                inv_P = __builtin_amdgcn_rcpf((float)P);
            }
            // one slot per row and, where both end caps of the rows that cross the walked cube matter, one more for those
            n_slots = FINE ? n_rows * P : low_caps && high_caps ? n_rows + n_inner : n_rows;
        }

        for (int slot0 = 0; slot0 < n_slots; slot0 += kWave) {
            const float reach2 = prunes && cut < 0x7f000000u ? bound_of(cut) : 3.0e38f;
            const int slot = slot0 + lane;
            if (d_in >= 0) seg_start = seg_len = 0;
            if (d_in >= 0 && slot < n_slots) {
                int row, piece = 0;
                bool inner = false;
                if (FINE) {
                    divmod_small(slot, P, inv_P, row, piece);
                } else {
                    inner = slot >= n_rows;
                    row = inner ? slot - n_rows : slot;
                }
                int off[B];
#pragma unroll
                for (int i = B - 2; i >= 0; --i) {
                    const int below_i = inner ? below_in[i] : below[i];
                    if (i > 0) {
                        int digit;
                        divmod_small(row, inner ? width_in[i] : width[i], inner ? inv_width_in[i] : inv_width[i], row, digit);
                        off[i] = digit - below_i;
                    } else {
                        off[i] = row - below_i;
                    }
                }
                bool on_face = false;
                int cell = 0, halves = 0;
                float gap2 = 0.f;  // squared lower bound of the distance to this row, in bin widths
#pragma unroll
                for (int i = 0; i < B - 1; ++i) {
                    const int o = off[i], k = qb[i] + o;
                    on_face = on_face || abs(o) > d_in;
                    if (FINE) {
                        cell = (int)__umul24(cell, nb[i] >> 1) + (k >> 1);
                        halves = (halves << 1) | (k & 1);
                    } else {
                        cell = (int)__umul24(cell, nb[i]) + k;
                    }
                    const float of = (float)o;
                    const float g = fmaxf(fmaxf(of - from_upper[i], -of - from_lower[i]), 0.f);
                    gap2 = __builtin_fmaf(g, g, gap2);
                }
                gap2 *= gap_scale;
                // bins of the row within reach (bound generous by 0.1 % and a thousandth of a bin)
                const float rest = reach2 - gap2;
                const float span = __builtin_amdgcn_sqrtf(fmaxf(rest, 0.f)) * bins_per_unit + 1.001f;
                int lo = -min(lo_last, (int)fminf(span - tl_last, 1.0e9f));
                int hi = min(hi_last, (int)fminf(span - tu_last, 1.0e9f));
                if (FINE) {
                    // the part inside one bin, less the cells walked before
                    const int bin = first_bin + piece;
                    lo = max(lo, 2 * bin - qb_last);
                    hi = min(hi, 2 * bin + 1 - qb_last);
                    if (!on_face) {
                        if (lo < -d_in) hi = min(hi, -d_in - 1);
                        else lo = max(lo, d_in + 1);
                    }
                } else if (!on_face) {
                    if (low_caps && !inner) hi = min(hi, -d_in - 1);
                    else lo = max(lo, d_in + 1);
                }
                if (rest >= 0.f && lo <= hi) {
                    if (FINE) {
                        const int bin = row_base(cell) + ((qb_last + lo) >> 1);
                        if (bin + 1 < n_bboundaries) {
                            const int base = ((bin << (B - 1)) | halves) << 1;
                            seg_start = table_entry(p.cell_boundaries, base | ((qb_last + lo) & 1));
                            seg_len = table_entry(p.cell_boundaries, (base | ((qb_last + hi) & 1)) + 1) - seg_start;
                        } else {
                            report(HGC_FLAG_BIN_BEYOND_TABLE);
                        }
                    } else {
                        const int first = row_base(cell) + qb_last + lo;
                        const int last = first + (hi - lo) + 1;
                        if constexpr (CALLERS) {
                            callers_run(first, last);
                        } else if (last < n_bboundaries) {
                            seg_start = table_entry(p.bin_boundaries, first);
                            seg_len = table_entry(p.bin_boundaries, last) - seg_start;
                        } else {
                            report(HGC_FLAG_BIN_BEYOND_TABLE);
                        }
                    }
                }
            }
            const int seg_end = d_in >= 0 ? wave_inclusive_sum(seg_len) : first_end;
            const int seg_off = seg_end - seg_len;
            const int total = readlane_i32(seg_end, kWave - 1);
            // kept one lane up, so that the mark (lane number + 1) is the lane to read it from: see walk_shells
            const int seg_delta = __builtin_amdgcn_update_dpp(0, seg_start - seg_off, 0x13c, 0xf, 0xf, false);
            uint32_t owner_carry = 0;
            for (int c0 = 0; c0 < total; c0 += kMarkCap) {
                const int chunk = min(kMarkCap, total - c0);
                for (int base = 0; base < chunk; base += kWave * 8)
                    *reinterpret_cast<uint64_t *>(marks + base + lane * 8) = 0;
                wave_lds_fence();
                const int rel = seg_off - c0;
                if (seg_len > 0 && rel >= 0 && rel < chunk) marks[rel] = (uint8_t)(lane + 1);
                wave_lds_fence();
                for (int t = 0; t < chunk; t += kWave) {
                    const int c = c0 + t + lane;
                    uint32_t owner = wave_inclusive_max(marks[t + lane]);
                    owner = max(owner, owner_carry);
                    owner_carry = (uint32_t)readlane_i32((int)owner, kWave - 1);
                    const int j = c + from_lane_i32(seg_delta, (int)owner);
                    const bool in_list = c < total;
                    uint64_t valid = __builtin_amdgcn_ballot_w64(in_list) & __builtin_amdgcn_ballot_w64(j != q);
                    const int jj = in_list ? j : q;
                    const uint32_t id = MAPPED ? *reinterpret_cast<const uint32_t *>(
                                                     reinterpret_cast<const char *>(p.sorting) + ((uint32_t)jj << 2))
                                               : (uint32_t)jj;
                    const float dsq = dist_sq<C>(qc, p.coord, jj, C, qrow);
                    if (use_direction) {
                        const int dj = kernel_args()->direction[jj];
                        valid &= ~__builtin_amdgcn_ballot_w64(dj == 1 || dj == 2);  // may not be a neighbour
                    }
                    uint64_t enters = valid & __builtin_amdgcn_ballot_w64(__float_as_uint(dsq) <= cut);
                    if (enters) {
                        if (__builtin_expect(n_kept + (int)__popcll(enters) > room, 0)) {
                            const uint64_t ck = (uint64_t)__float_as_uint(dsq) << 32 | id;
                            enters &= __builtin_amdgcn_ballot_w64(ck <= ((uint64_t)cut << 32 | cut_id));
                            if (n_kept + (int)__popcll(enters) > kBufferKeys) {
                                wave_lds_fence();
                                n_kept = cut_to_smallest<CALLERS>(buffer, lane, n_kept, Kn, kept, cut, cut_id);
                                enters &= __builtin_amdgcn_ballot_w64(ck <= ((uint64_t)cut << 32 | cut_id));
                                room = cut_id == 0xffffffffu ? kBufferKeys : 0;
                            }
                        }
                        const int at = n_kept + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(enters >> 32),
                                                                               __builtin_amdgcn_mbcnt_lo((uint32_t)enters, 0));
                        if (__builtin_amdgcn_inverse_ballot_w64(enters)) buffer[at] = (uint64_t)__float_as_uint(dsq) << 32 | id;
                        n_kept += (int)__popcll(enters);
                    }
                }
            }
        }
        // done: everything within the bound, the radius or the grid has been seen
        if (last_pass || d_out >= d_radius || !__builtin_amdgcn_ballot_w64(max(qb_v, top_v) > d_out)) break;
        d_in = d_out;
        if (n_kept >= Kn) {
            wave_lds_fence();
            n_kept = cut_to_smallest<CALLERS>(buffer, lane, n_kept, Kn, kept, cut, cut_id);
        }
        d_out = d_out < 4 ? d_out + 1 : d_out + (d_out >> 1);
    }

    wave_lds_fence();
    if (n_kept > S * kWave) n_kept = cut_to_smallest<CALLERS>(buffer, lane, n_kept, Kn, S * kWave, cut, cut_id);
    key[0] = wave_sort_u64(lane < n_kept ? buffer[lane] : kEmptyKey, n_kept);
    if constexpr (S == 2) {
        key[1] = kEmptyKey;
        if (n_kept > kWave) merge_batch<S>(key, wave_sort_u64(kWave + lane < n_kept ? buffer[kWave + lane] : kEmptyKey));
    }
    return true;
}

// C: coordinates per point, NB: binned dimensions (0 for either: taken from the
// arguments), S: registers of the sorted list per lane, MAPPED: results in the
// index space and at the positions of `sorting`.
// WINDOW: more neighbours are asked for than the registers hold (64 S). The search then runs
// once per window of 64 S ranks: launch t finds the 64 S smallest keys ABOVE the last key of
// launch t-1 (read back from the output row) and writes them behind it. Every launch walks
// the shells from the query's bin again and stops by the same rule on its own list, so each
// window is exact; slow (the walk is repeated) but without a bound on K.
// NESTED: the search runs over a nested grid (see KnnParams::fine_bits): a query whose bin holds more
// than fine_min_population points walks the nested grid (and the grid of bins after all when that
// walk gives up), the others the grid of bins.
template <int C, int NB, int S, bool MAPPED, bool WINDOW, bool NESTED, bool CALLERS>
__device__ __forceinline__ void search_query(const KnnParams &p, const int q, const int lane, uint8_t *const marks,
                                             uint64_t *const buffer) {
    constexpr bool kCollects = collects(C, NB, S, WINDOW);
    bool crowded = false;
    if constexpr (NESTED) {
        const int own_bin = uniform(p.bin_idx[q]) >> p.fine_bits;
        if (own_bin + 1 < p.n_bboundaries)
            crowded = p.bin_boundaries[own_bin + 1] -
                          p.bin_boundaries[own_bin] > p.fine_min_population;
    }

    const int K = p.K;
    const int rank_base = WINDOW ? p.rank_base : 0;
    const int Kn = WINDOW ? min(K - 1 - rank_base, S * kWave) : K - 1;  // neighbours (besides the point itself) to find
    const int self_id = MAPPED ? p.sorting[q] : q;
    const size_t out_row = (size_t)self_id * K;
    const int pad_idx = p.tf_compat ? self_id : -1;

    bool searching = Kn > 0;
    uint64_t floor_key = 0;  // WINDOW: only keys above this one are candidates
    if (WINDOW && rank_base > 0) {
        const int last_idx = p.out_idx[out_row + rank_base];
        const float last_dist = p.out_dist[out_row + rank_base];
        if (last_idx == pad_idx) searching = false;  // the windows before found fewer points than they had room for
        floor_key = ((uint64_t)__float_as_uint(last_dist) << 32) | (uint32_t)last_idx;
    }
    if (p.use_direction) {
        const int dq = p.direction[q];
        if (dq == 0 || dq == 2) searching = false;  // may not have neighbours
    }

    uint64_t key[S];
#pragma unroll
    for (int s = 0; s < S; ++s) key[s] = kEmptyKey;

    if (searching) {
        if constexpr (kCollects) {
            if constexpr (NESTED) {
                if (!crowded || !collect_nearest<C, NB, S, MAPPED, true, CALLERS>(p, q, lane, marks, buffer, Kn, key))
                    collect_nearest<C, NB, S, MAPPED, false, CALLERS>(p, q, lane, marks, buffer, Kn, key);
            } else {
                collect_nearest<C, NB, S, MAPPED, false, CALLERS>(p, q, lane, marks, buffer, Kn, key);
            }
        } else {
            bool found = false;
            if constexpr (NESTED) {
                found = crowded && walk_shells<C, NB, S, MAPPED, WINDOW, true, NESTED, CALLERS>(p, q, lane, marks, Kn, floor_key, key);
                if (!found) {
#pragma unroll
                    for (int s = 0; s < S; ++s) key[s] = kEmptyKey;
                }
            }
            if (!found) walk_shells<C, NB, S, MAPPED, WINDOW, false, NESTED, CALLERS>(p, q, lane, marks, Kn, floor_key, key);
        }
    }

    // ---- write the row: slot 0 = self, then ascending (distance, index) ----
    const KernelArgs args = kernel_args();
    const int id = kCollects && MAPPED ? args->sorting[q] : self_id, pad = args->tf_compat ? id : -1;
    const size_t row = (size_t)id * args->K;
    int *const out_idx = args->out_idx;
    float *const out_dist = args->out_dist;
    if (lane == 0 && rank_base == 0) {
        out_idx[row] = id;
        out_dist[row] = 0.f;
    }
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int rank = s * kWave + lane;
        if (rank < Kn) {
            const bool filled = key[s] != kEmptyKey;
            out_idx[row + 1 + rank_base + rank] = filled ? (int)(uint32_t)key[s] : pad;
            out_dist[row + 1 + rank_base + rank] = filled ? __uint_as_float((uint32_t)(key[s] >> 32)) : 0.f;
        }
    }
}

// CALLERS: bin rows and boundary table were handed over by a caller, may contradict each other and be of any size, the
// grid may be of any width, and `sorting` may repeat itself. Without, they are those of the package's own binning, which need
// no such checks (1.14 M 3-D points in 16 events on 43 bins, K = 32: 1150 us with them, 1040 without, 1185 by shells; 4-D, K = 200
// by shells 1525 and 1440; with checks for every call the searches on the package's own grid were 1 to 4 % slower).
template <int C, int NB, int S, bool MAPPED, bool CALLERS, bool WINDOW = false, bool NESTED = false>
__global__ __launch_bounds__(kWave)
__attribute__((amdgpu_waves_per_eu(S <= 2 ? 8 : 1, 8)))
void knn_wave_kernel(const KnnParams p) {
    __shared__ __attribute__((aligned(8))) uint8_t marks[kMarkCap];
    __shared__ uint64_t buffer[collects(C, NB, S, WINDOW) ? kBufferKeys : 1];
    // queries come in bin order and differ a lot in cost from region to region:
    // chunks of 512 of them are dealt to the XCDs in turn
    const int q = xcd_chunked_block<512>(blockIdx.x, gridDim.x);
    search_query<C, NB, S, MAPPED, WINDOW, NESTED, CALLERS>(p, q, lane_id(), marks, buffer);
}

template <int C, int NB, bool MAPPED, bool CALLERS>
int launch_levels(const KnnParams &p, hipStream_t s) {
    const int levels = std::max(1, ceil_div(p.K - 1, kWave));
    const dim3 grid(p.n_vert), block(kWave);
    if (levels > kBulkInsertMaxRuns) {  // more neighbours than the registers hold: one launch per window of ranks
        KnnParams window = p;
        for (window.rank_base = 0; window.rank_base < p.K - 1; window.rank_base += kBulkInsertMaxRuns * kWave) {
            knn_wave_kernel<C, NB, kBulkInsertMaxRuns, MAPPED, CALLERS, true><<<grid, block, 0, s>>>(window);
            const int rc = check_launch("knn_wave_kernel (window of ranks)");
            if (rc) return rc;
        }
        return HGC_OK;
    }
    if constexpr (MAPPED && !CALLERS && C == NB && NB >= 3 && NB <= 4) {  // all coordinates binned: a crowded bin has its neighbours close by
        if (p.fine_bits > 0 && p.cell_boundaries) {
            switch (levels) {
                case 1: knn_wave_kernel<C, NB, 1, MAPPED, CALLERS, false, true><<<grid, block, 0, s>>>(p); break;
                case 2: knn_wave_kernel<C, NB, 2, MAPPED, CALLERS, false, true><<<grid, block, 0, s>>>(p); break;
                case 3:
                case 4: knn_wave_kernel<C, NB, 4, MAPPED, CALLERS, false, true><<<grid, block, 0, s>>>(p); break;
                default: knn_wave_kernel<C, NB, 8, MAPPED, CALLERS, false, true><<<grid, block, 0, s>>>(p); break;
            }
            return check_launch("knn_wave_kernel (nested grid)");
        }
    }
    switch (levels) {
        case 1: knn_wave_kernel<C, NB, 1, MAPPED, CALLERS><<<grid, block, 0, s>>>(p); break;
        case 2: knn_wave_kernel<C, NB, 2, MAPPED, CALLERS><<<grid, block, 0, s>>>(p); break;
        case 3:
        case 4: knn_wave_kernel<C, NB, 4, MAPPED, CALLERS><<<grid, block, 0, s>>>(p); break;
        default: knn_wave_kernel<C, NB, 8, MAPPED, CALLERS><<<grid, block, 0, s>>>(p); break;
    }
    return check_launch("knn_wave_kernel");
}

// The usual shapes (up to 8 coordinates; binned dimensions = min(3, coordinates), the reference
// wrapper's default, or min(4, coordinates), the pipeline's own grid) get kernels with both
// numbers fixed at compile time, anything else the one that reads them.
template <bool MAPPED, bool CALLERS>
int launch_coords(const KnnParams &p, hipStream_t s) {
    if (p.n_coords == 2 && p.n_bin_dim == 2) return launch_levels<2, 2, MAPPED, CALLERS>(p, s);
    if (p.n_coords == 3 && p.n_bin_dim == 3) return launch_levels<3, 3, MAPPED, CALLERS>(p, s);
    if (p.n_coords == 4 && p.n_bin_dim == 3) return launch_levels<4, 3, MAPPED, CALLERS>(p, s);
    if (p.n_coords == 4 && p.n_bin_dim == 4) return launch_levels<4, 4, MAPPED, CALLERS>(p, s);
    if (p.n_coords == 5 && p.n_bin_dim == 4) return launch_levels<5, 4, MAPPED, CALLERS>(p, s);
    if (p.n_coords == 6 && p.n_bin_dim == 4) return launch_levels<6, 4, MAPPED, CALLERS>(p, s);
    if (p.n_coords == 7 && p.n_bin_dim == 4) return launch_levels<7, 4, MAPPED, CALLERS>(p, s);
    if (p.n_coords == 8 && p.n_bin_dim == 4) return launch_levels<8, 4, MAPPED, CALLERS>(p, s);
    if (p.n_coords == 5 && p.n_bin_dim == 3) return launch_levels<5, 3, MAPPED, CALLERS>(p, s);
    if (p.n_coords == 6 && p.n_bin_dim == 3) return launch_levels<6, 3, MAPPED, CALLERS>(p, s);
    if (p.n_coords == 7 && p.n_bin_dim == 3) return launch_levels<7, 3, MAPPED, CALLERS>(p, s);
    if (p.n_coords == 8 && p.n_bin_dim == 3) return launch_levels<8, 3, MAPPED, CALLERS>(p, s);
    return launch_levels<0, 0, MAPPED, CALLERS>(p, s);
}

}  // namespace

int binned_select_knn_strided(const float *d_coord, const int *d_bin_idx, const int *d_direction,
                              const int *d_dim_bin_idx, const int *d_bin_boundaries,
                              const int *d_n_bins, const float *d_bin_width, const int *d_sorting,
                              const float *d_shift, float max_radius, int *d_indices, float *d_dist, int n_vert,
                              int n_neigh, int n_coords, int n_bin_dim, int n_bboundaries, int tf_compat,
                              int use_direction, int bins_bound, bool callers_table,
                              const int *d_cell_boundaries, int fine_bits, int fine_min_population, hipStream_t s) {
    // same conditions as the reference op (binned_select_knn_kernel.cc:336-352)
    HGC_REQUIRE(n_bin_dim > 1, "BinnedSelectKnnOp expects at least 2 binning dimensions.");
    HGC_REQUIRE(n_bin_dim < 6, "BinnedSelectKnnOp expects maximum 5 binning dimensions.");
    HGC_REQUIRE(n_coords > 1, "BinnedSelectKnnOp expects at least 2 dimensions.");
    HGC_REQUIRE(n_coords >= n_bin_dim, "fewer coordinates than binning dimensions");
    HGC_REQUIRE(n_vert >= 0, "negative number of points");
    HGC_REQUIRE(n_neigh >= 1, "n_neighbours must be positive");
    HGC_REQUIRE((long long)n_vert * n_neigh < (1ll << 31), "n_vert * n_neighbours overflows int32");
    // candidate rows are addressed by 32-bit byte offsets
    HGC_REQUIRE((unsigned long long)n_vert * (unsigned long long)n_coords * sizeof(float) < (1ull << 32),
                "coordinate matrix must stay below 4 GiB");
    HGC_REQUIRE(n_bboundaries >= 2, "bin boundary table too short");
    HGC_REQUIRE(fine_bits == 0 || (fine_bits == n_bin_dim && fine_bits <= 4),
                "a nested grid has one bit per binned dimension, four at most");
    if (n_vert == 0) return HGC_OK;
    HGC_REQUIRE(d_coord && d_bin_idx && d_dim_bin_idx && d_bin_boundaries && d_n_bins && d_bin_width &&
                    d_indices && d_dist,
                "null pointer");
    HGC_REQUIRE(!use_direction || d_direction,
                "BinnedSelectKnnOp needs a direction tensor (0,1,2,other) with length nvert if use_direction=True.");
    HGC_REQUIRE((n_coords != 4 && n_coords != 2 && n_coords != 6 && n_coords != 8) ||
                    (reinterpret_cast<uintptr_t>(d_coord) & 15u) == 0,
                "coordinate matrix must be 16-byte aligned");

    KnnParams p;
    p.coord = d_coord;
    p.bin_idx = d_bin_idx;
    p.direction = d_direction;
    p.dim_bin_idx = d_dim_bin_idx;
    p.bin_boundaries = d_bin_boundaries;
    p.n_bins = d_n_bins;
    p.bin_width = d_bin_width;
    p.sorting = d_sorting;
    p.shift = d_shift;
    p.out_idx = d_indices;
    p.out_dist = d_dist;
    p.status = status_word();
    p.radius_sq = max_radius > 0.f ? max_radius * max_radius : -1.f;
    p.n_vert = n_vert;
    p.K = n_neigh;
    p.n_coords = n_coords;
    p.n_bin_dim = n_bin_dim;
    p.n_bboundaries = n_bboundaries;
    p.tf_compat = tf_compat;
    p.use_direction = use_direction;
    p.rank_base = 0;
    p.cell_boundaries = d_cell_boundaries;
    p.fine_bits = fine_bits;
    p.fine_min_population = fine_min_population;
    // the package's own tables are read with 32-bit byte offsets, and their bins per dimension are few
    callers_table = callers_table || n_bboundaries >= 1 << 30 || bins_bound > kNarrowGrid;
    if (!d_sorting) return launch_coords<false, true>(p, s);  // (the package's own points come with a sorting)
    return callers_table ? launch_coords<true, true>(p, s) : launch_coords<true, false>(p, s);
}

}  // namespace hgc

using namespace hgc;

extern "C" {

int hgc_binned_select_knn_fused(const float *d_coord, const int *d_bin_idx, const int *d_direction,
                                const int *d_dim_bin_idx, const int *d_bin_boundaries,
                                const int *d_n_bins, const float *d_bin_width, const int *d_sorting,
                                const float *d_shift, float max_radius, int *d_indices, float *d_dist, int n_vert, int n_neigh,
                                int n_coords, int n_bin_dim, int n_bboundaries, int tf_compat,
                                int use_direction, hgc_stream_t stream) {
    return binned_select_knn_strided(d_coord, d_bin_idx, d_direction, d_dim_bin_idx, d_bin_boundaries, d_n_bins,
                                     d_bin_width, d_sorting, d_shift, max_radius, d_indices, d_dist, n_vert, n_neigh,
                                     n_coords, n_bin_dim, n_bboundaries, tf_compat, use_direction, 0, true,
                                     nullptr, 0, 0, as_stream(stream));
}

int hgc_binned_select_knn(const float *d_coord, const int *d_bin_idx, const int *d_direction,
                          const int *d_dim_bin_idx, const int *d_bin_boundaries, const int *d_n_bins,
                          const float *d_bin_width, int *d_indices, float *d_dist, int n_vert, int n_neigh,
                          int n_coords, int n_bin_dim, int n_bboundaries, int tf_compat, int use_direction,
                          hgc_stream_t stream) {
    return hgc_binned_select_knn_fused(d_coord, d_bin_idx, d_direction, d_dim_bin_idx, d_bin_boundaries,
                                       d_n_bins, d_bin_width, nullptr, nullptr, -1.f, d_indices, d_dist, n_vert,
                                       n_neigh, n_coords, n_bin_dim, n_bboundaries, tf_compat, use_direction,
                                       stream);
}

}  // extern "C"
