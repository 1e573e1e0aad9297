// Gradient of the GravNet neighbour accumulation for rows of 16 to 128 features: both outputs from one
// gather over the inverse neighbour index, 16 lanes per target vertex.
//
// Reference behaviour restated here:
//   modules/compiled/accumulate_knn_grad_kernel.cc:36-97   (feature gradient)
//   modules/compiled/accumulate_knn_grad_kernel.cc:99-165  (weight gradient)
//
// For an entry (v, n) of target m's inverse list (idx[v, n] == m) the feature gradient of m adds
// (g[v,f]/K)*w[v,n] + max part, in ascending (v, n) order (the reference CPU kernel's order: the
// result is bit-identical to it), and the weight gradient of slot (v, n) is the dot product of
// g[v, :] with feat[m, :], which the group holds in registers.
//
// Layout as in the forward (accumulate_rows.hpp): a group of 16 lanes owns a target and up to 64 of its
// features, lane l VEC consecutive ones; four groups per wave. The group's lanes fetch the list
// entries, weights and row offsets of 16 entries at once and hand them on as DPP operands. What a
// gathered row costs is then one 16-byte load per lane for the mean half, one dword for the
// arg-max slots and a masked 16-byte load for the few features whose maximum sits at this entry,
// for four targets together. One wave per target with one dword per lane ran its three loads
// per entry at the L1's narrow-load rate (95 % busy, vector issue 62 %):
// Gaussian points in bin order, 150,000 vertices, 4-D, K = 64, F = 64 535 -> 294 us; 240,000, 3-D, K = 40,
// F = 32 571 -> 293 us; a million, K = 64, F = 128 5.75 -> 4.45 ms. What bounds it now: the L1's address and return path
// (77 and 90 % busy at 150,000 vertices), vector issue at 66 %, and at a million vertices the
// L2 misses (37 % of the return path's time).
// Where this split loses: tables without locality (60,000 vertices, K = 24, targets drawn at random, F = 100 and 128 212 ->
// 232 us, F = 64 136 -> 144), and a few targets that the whole table names, where a list's entries are one serial
// chain, longer per entry with four targets a wave (50 targets, F = 64 3.96 -> 5.32 ms). The host does not know a
// table's lists, and tables of a neighbour search have neither.
//
// GravNet accumulates over a table without its self column and needs the inverse index of the whole table for the
// distances: `skip` lets the gather run on that one and pass over the entries of column 0 (one in K + 1), instead of
// deriving a second index (a training step at 150,000 vertices, K = 64: 2.17 -> 2.11 ms; 240,000, K = 40: 2.27 -> 2.17).
//
// The loads of an entry depend on one another (slots, then the max half they gate), so two entries at a
// time move through a pipeline: slots two steps ahead, rows one step ahead, arithmetic.
// The dot products of four entries are reduced across the 16 lanes by a transposing exchange (three
// instructions per value with DPP).
#include <algorithm>

#include "accumulate_rows.hpp"

namespace hgc {

// accumulate_grad_records.hip
int launch_weight_grad_to_table(const int *inv_off, const int *inv_slots, const float *gw_list, float *gw, int n_vert,
                                long long total, const int *wanted, hipStream_t s);

namespace {

using namespace acc;

// How the mean part (g / divisor) * w is formed with the bits of the two operations:
//   kPow2    divisor a power of two: g * (w / divisor), exact apart from subnormal quotients
//   kScaled  g has been divided beforehand: rows of F quotients, so that with a max half its rows are twice as long
//   kDivide  an IEEE divide per element and entry
enum Scale { kPow2, kScaled, kDivide };

struct GradRows {
    const float *g, *g_max;       // mean and max half of the upstream gradient, rows of `pitch` floats (g_max: 2F)
    const float *w, *feat;
    const unsigned char *maxslot;
    const int *inv_off, *inv_slots, *order;
    float *gw, *gfeat;
    // Weight gradients in the order of the inverse index, moved to their slots by a pass of its own, where *scattered is
    // set (see list_order_may_pay; both null: never)
    float *gw_list;
    const int *scattered;
    unsigned long long g_bytes, g_max_bytes, slot_bytes;  // sizes seen by the hardware's range check
    int n_vert, K, F, blocks, pitch;
    int skip;  // 1: the inverse index is that of a table with one more column in front (K + 1), which is left out
    FastDiv div_k;  // by K + skip
    float divisor;
    uint32_t slot_shift;  // maxslot has been moved down by this many bytes onto a multiple of 4
    bool negate;  // gw receives -(gradient * w): the chain rule through w = exp(-d)
};

// Does byte E of `packed` equal `key`? The compiler makes one SDWA compare of it, and keeps the wait states between
// a compare and a vector use of its mask.
template <int E>
__device__ __forceinline__ uint64_t byte_is(uint32_t packed, uint32_t key) {
    return __builtin_amdgcn_ballot_w64(((packed >> (8 * E)) & 255u) == key);
}

// Arg-max slots of VEC features, packed in one word. ALIGNED: they start on a multiple of VEC (1, 2 or 4)
// and come in one load of that width; otherwise out of the eight bytes around them, which start on a
// multiple of 4 and end with the table's last word (last_pair: where the last eight bytes begin).
template <int VEC, bool ALIGNED>
struct SlotBytes {
    uint32_t v[ALIGNED ? 1 : 3];
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rsrc, uint32_t offset, uint32_t last_pair) {
        if constexpr (ALIGNED) {
            if constexpr (VEC == 4) v[0] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)offset, 0, 0);
            else if constexpr (VEC == 2) v[0] = __builtin_amdgcn_raw_buffer_load_b16(rsrc, (int)offset, 0, 0);
            else v[0] = __builtin_amdgcn_raw_buffer_load_b8(rsrc, (int)offset, 0, 0);
        } else {
            // (the offset of an entry beyond the list is moved into the table here: its row still reads zeros)
            const uint32_t at = min(offset & ~3u, last_pair);
            const auto two = __builtin_amdgcn_raw_buffer_load_b64(rsrc, (int)at, 0, 0);
            v[0] = two[0];
            v[1] = two[1];
            v[2] = (offset - at) * 8u;
        }
    }
    __device__ __forceinline__ uint32_t packed() const {
        if constexpr (ALIGNED) return v[0];
        else return (uint32_t)((((uint64_t)v[1] << 32) | v[0]) >> (v[2] & 63u));
    }
};

// Behind a matrix of half of kMaxRowBytes, and twice of it behind one of kMaxRowBytes
constexpr uint32_t kNoHalfRow = 0x7fffe000u;
static_assert(kNoHalfRow >= kMaxRowBytes / 2 && 2ull * kNoHalfRow >= kMaxRowBytes && 2ull * kNoHalfRow + 8 * kRowLanes * 4 < 1ull << 32);

// what the group's lanes hold of 16 entries
struct Entries {
    uint32_t row;    // byte offset of the (mean half's) gradient row, behind the matrices beyond the list
    uint32_t slots;  // byte offset of the arg-max slots
    uint32_t key;    // slot of the entry
    int slot;        // its flat number v K + slot, -1 beyond the list
    float w, w_mean; // weight, and what the mean half is multiplied by
};

// Two entries on their way through the pipeline: arg-max slots (requested two steps ahead), gradient
// rows (requested one step ahead, the max half by the slots), arithmetic. own[e]: the lanes whose element e
// is theirs. (150,000 vertices, own features of 0 in the place of the others and now: K = 40, F = 22 178 and
// 177 us, F = 50 229 and 231; K = 16, F = 127 208 and 212.)
// TWICE: the max half lies in rows twice as long as those of the mean half.
template <int VEC, bool MAX, bool ALIGNED, Tail TAIL, bool TWICE>
struct Step {
    SlotBytes<VEC, ALIGNED> sb[2];
    float gm[2][VEC], gx[2][VEC];
    uint64_t hit[2][VEC];

    template <int E>
    __device__ __forceinline__ void request_slots(__amdgpu_buffer_rsrc_t MS, const Entries &en, uint32_t lane_col, uint32_t last_pair) {
        if constexpr (MAX) {
            sb[0].load(MS, group_bcast<entry_lane(E)>(en.slots) + lane_col, last_pair);
            sb[1].load(MS, group_bcast<entry_lane(E + 1)>(en.slots) + lane_col, last_pair);
        }
    }
    template <int U>
    __device__ __forceinline__ void request_row(__amdgpu_buffer_rsrc_t G, __amdgpu_buffer_rsrc_t GX, uint32_t row, uint32_t lane_bytes,
                                                uint32_t key) {
        const uint32_t at = row + lane_bytes;
        load_cols<VEC>(G, at, gm[U]);
        if constexpr (MAX) {
            const uint32_t slots = sb[U].packed();
            hit[U][0] = byte_is<0>(slots, key);
            uint64_t any = hit[U][0];
            if constexpr (VEC > 1) any |= hit[U][1] = byte_is<1>(slots, key);
            if constexpr (VEC > 2) any |= hit[U][2] = byte_is<2>(slots, key);
            if constexpr (VEC > 3) any |= hit[U][3] = byte_is<3>(slots, key);
            // about F/K features of a row have their maximum at one entry: the other lanes aim out of range
            const uint32_t at_max = TWICE ? (row << 1) + lane_bytes : at;
            load_cols<VEC>(GX, __builtin_amdgcn_inverse_ballot_w64(any) ? at_max : kNoRow, gx[U]);
        }
    }
    template <int E>
    __device__ __forceinline__ void request_rows(__amdgpu_buffer_rsrc_t G, __amdgpu_buffer_rsrc_t GX, const Entries &en,
                                                 uint32_t lane_bytes) {
        request_row<0>(G, GX, group_bcast<entry_lane(E)>(en.row), lane_bytes, group_bcast<entry_lane(E)>(en.key));
        request_row<1>(G, GX, group_bcast<entry_lane(E + 1)>(en.row), lane_bytes, group_bcast<entry_lane(E + 1)>(en.key));
    }
    // An entry beyond its list reads zeros and has weight 0: it adds 0 to a sum that started at +0.
    template <int U, Scale SCALE, bool WGRAD>
    __device__ __forceinline__ void add(float w, float w_mean, const float (&xo)[VEC], const float (&xk)[VEC],
                                        const uint64_t (&own)[VEC], float divisor, float (&acc)[VEC], float &val) const {
        float dot = 0.f;
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            const float g = TAIL != kElements || __builtin_amdgcn_inverse_ballot_w64(own[e]) ? gm[U][e] : 0.f;
            const float part = SCALE == kDivide ? (g / divisor) * w : g * w_mean;
            if (WGRAD) dot = __builtin_fmaf(g, xk[e], dot);
            if constexpr (MAX) {
                const uint64_t here = TAIL == kElements ? hit[U][e] & own[e] : hit[U][e];
                const float gsel = VEC == 1 ? gx[U][e] : __builtin_amdgcn_inverse_ballot_w64(here) ? gx[U][e] : 0.f;
                if (WGRAD) dot = __builtin_fmaf(gsel, xo[e], dot);
                const float part_max = gsel * w;
                const float sum = part + part_max;
                acc[e] = acc[e] + sum;
            } else {
                acc[e] = acc[e] + part;  // the reference's "+ 0" cannot change the sum
            }
        }
        val = TAIL != kLanes || __builtin_amdgcn_inverse_ballot_w64(own[0]) ? dot : 0.f;
    }
};

template <int VEC, bool MAX, Scale SCALE, bool ALIGNED, Tail TAIL, bool WGRAD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5, 8))) void accumulate_grad_rows_kernel(const GradRows p) {
    const int lane = lane_id(), l = lane & (kRowLanes - 1);
    if (WGRAD) {
        // weight gradient of padded slots: they sort behind the last target's entries
        const int first = p.inv_off[p.n_vert], total = p.n_vert * (p.K + p.skip);
        for (long long i = first + (long long)blockIdx.x * blockDim.x + threadIdx.x; i < total;
             i += (long long)gridDim.x * blockDim.x) {
            const int slot = p.inv_slots[i], v = fast_div(slot, p.div_k);
            if (slot - v * (p.K + p.skip) >= p.skip) p.gw[slot - (v + 1) * p.skip] = 0.f;
        }
    }
    // The groups of a workgroup trade their targets so that those of a wave have lists of similar length: a
    // wave runs for as long as its longest one (kNN tables, mean 64 of standard deviation 23: 79 entries of
    // time per list as they come, 74 sorted; a group pair that shares a target stays together).
    __shared__ int s_vertex[16], s_block[16], s_begin[16], s_count[16], s_from[16];
    const int group = threadIdx.x / kRowLanes;
    {
        const GroupTask first = group_task(p.order, p.n_vert, p.blocks);
        if (l == 0) {
            const int begin = first.vertex >= 0 ? p.inv_off[first.vertex] : 0;
            s_vertex[group] = first.vertex;
            s_block[group] = first.block;
            s_begin[group] = begin;
            s_count[group] = first.vertex >= 0 ? p.inv_off[first.vertex + 1] - begin : 0;
        }
        __syncthreads();
        const int own = s_count[group], other = s_count[l];
        const uint64_t below = __builtin_amdgcn_ballot_w64(other < own || (other == own && l < group));
        if (l == 0) s_from[__popcll((below >> (lane & 48)) & 0xffffull)] = group;
        __syncthreads();
    }
    const int from = s_from[group];
    const GroupTask task = {s_vertex[from], s_block[from]};
    const bool live = task.vertex >= 0;
    const int m = live ? task.vertex : 0;
    const int begin = s_begin[from], count = s_count[from];
    // of the wave's longest list
    const int longest = max(max(readlane_i32(count, 0), readlane_i32(count, 16)),
                            max(readlane_i32(count, 32), readlane_i32(count, 48)));

    const __amdgpu_buffer_rsrc_t G = make_rows(p.g, p.g_bytes);
    const __amdgpu_buffer_rsrc_t GX = make_rows(p.g_max, MAX ? p.g_max_bytes : 0);
    const __amdgpu_buffer_rsrc_t MS = make_rows(p.maxslot, MAX ? p.slot_bytes : 0);
    const float inv_divisor = 1.f / p.divisor;
    const bool in_list_order = WGRAD && p.scattered && *p.scattered;

    // A lane at the end of a row that is no multiple of VEC, and the lanes behind it, take the last VEC
    // columns (never columns of the next row); what they share with another lane counts there (see TAIL).
    const int fb = task.block * (kRowLanes * VEC) + l * VEC;
    const int f = min(fb, p.F - VEC);
    const uint32_t lane_bytes = (uint32_t)f * 4u, lane_col = (uint32_t)f + p.slot_shift;
    const uint32_t last_pair = (uint32_t)p.slot_bytes - 8u;
    float xo[VEC], xk[VEC], acc[VEC];
    uint64_t own[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
        own[e] = __builtin_amdgcn_ballot_w64(f + e >= fb);
        xo[e] = WGRAD && live && f + e >= fb ? p.feat[(size_t)m * p.F + f + e] : 0.f;
        xk[e] = SCALE == kScaled ? xo[e] : (float)((double)xo[e] * (1.0 / (double)p.divisor));
        acc[e] = 0.f;
    }

    constexpr bool kTwice = MAX && SCALE == kScaled;
    constexpr uint32_t no_row = kTwice ? kNoHalfRow : kNoRow;
    const int *list = p.inv_slots + begin + entry_lane(l);
    const int mine = count - entry_lane(l);  // this lane has an entry of chunk c0 if c0 < mine
    auto entries_of = [&](int slot, int c0) {
        Entries en;
        const int v = fast_div(slot, p.div_k), n = slot - v * (p.K + p.skip) - p.skip;
        const bool here = c0 < mine && n >= 0;  // column 0 of an index of the whole table is nobody's
        en.key = (uint32_t)n;
        en.slot = here ? slot - (v + 1) * p.skip : -1;
        en.row = here ? (uint32_t)v * (uint32_t)(p.pitch * 4) : no_row;
        en.slots = here ? (uint32_t)v * (uint32_t)p.F : kNoRow;
        return en;
    };
    auto weight_of = [&](const Entries &e) { return e.slot >= 0 ? p.w[e.slot] : 0.f; };
    auto set_weight = [&](Entries &e, float w) {
        e.w = w;
        e.w_mean = SCALE == kPow2 ? w * inv_divisor : w;
    };

    // slots of the list two chunks ahead, weights and offsets one chunk ahead
    const int slot = 0 < mine ? list[0] : 0;
    int slot_next = kRowLanes < mine ? list[kRowLanes] : 0;
    Entries en = entries_of(slot, 0);
    set_weight(en, weight_of(en));
    // Entries that name the target itself: the first one (lowest slot) carries the max part. Later ones (padding by
    // repeated self references) have a slot that no maximum names; the weight gradient counts the maxima of the
    // first one for them too, on the same gradient row: theirs is the dot product of the first.
    constexpr uint32_t kNoSlot = 0x1ff;
    struct Selves {
        uint64_t first, repeats;  // lanes whose entry is one
    };
    bool self_seen = false;
    auto mark_selves = [&](Entries &e, int c0) {
        Selves s{0, 0};
        if (MAX) {
            const bool self = c0 < mine && e.row == (uint32_t)m * (uint32_t)(p.pitch * 4);
            if (__builtin_amdgcn_ballot_w64(self)) {
                const int lowest = group_min(self ? (int)e.key : 1 << 30);
                const bool first = self && !self_seen && (int)e.key == lowest;
                s.first = __builtin_amdgcn_ballot_w64(first);
                s.repeats = __builtin_amdgcn_ballot_w64(self && !first);
                if (self && !first) e.key = kNoSlot;
                self_seen = self_seen || lowest < (1 << 30);
            }
        }
        return s;
    };
    Selves selves = mark_selves(en, 0);
    float self_dot = 0.f;

    Step<VEC, MAX, ALIGNED, TAIL, kTwice> st[2];
    st[0].template request_slots<0>(MS, en, lane_col, last_pair);
    st[1].template request_slots<2>(MS, en, lane_col, last_pair);
    st[0].template request_rows<0>(G, GX, en, lane_bytes);
    for (int c0 = 0; c0 < longest; c0 += kRowLanes) {
        const int slot_after = c0 + 2 * kRowLanes < mine ? list[c0 + 2 * kRowLanes] : 0;
        Entries next = entries_of(slot_next, c0 + kRowLanes);
        const float w_next = weight_of(next);
        set_weight(next, 0.f);
        const Selves next_selves = mark_selves(next, c0 + kRowLanes);
        float r[4] = {0.f, 0.f, 0.f, 0.f}, val[4];
        // step I: rows of step I + 1 and slots of step I + 2 are requested, then step I is added up
#define HGC_STEP(I)                                                                                                           \
    {                                                                                                                         \
        constexpr int kRows = (I) * 2 + 2, kSlots = (I) * 2 + 4;                                                              \
        st[((I) + 1) & 1].template request_rows<(kRows & 15)>(G, GX, kRows < 16 ? en : next, lane_bytes);                     \
        st[(I) & 1].template request_slots<(kSlots & 15)>(MS, kSlots < 16 ? en : next, lane_col, last_pair);                             \
        __builtin_amdgcn_sched_barrier(0);                                                                                    \
        constexpr int kA = entry_lane((I) * 2), kB = entry_lane((I) * 2 + 1);                                                 \
        const float wa = group_bcast<kA>(en.w), wb = group_bcast<kB>(en.w);                                                   \
        st[(I) & 1].template add<0, SCALE, WGRAD>(wa, SCALE == kPow2 ? group_bcast<kA>(en.w_mean) : wa, xo, xk, own, p.divisor,  \
                                                  acc, val[((I) & 1) * 2]);                                                   \
        st[(I) & 1].template add<1, SCALE, WGRAD>(wb, SCALE == kPow2 ? group_bcast<kB>(en.w_mean) : wb, xo, xk, own, p.divisor,  \
                                                  acc, val[((I) & 1) * 2 + 1]);                                               \
        if (WGRAD && ((I) & 1)) r[(I) >> 1] = group_sum_4(val, lane);                                                         \
        __builtin_amdgcn_sched_barrier(0);                                                                                    \
    }
        HGC_STEP(0)
        HGC_STEP(1)
        HGC_STEP(2)
        HGC_STEP(3)
        if (c0 + 8 < longest) {
            HGC_STEP(4)
            HGC_STEP(5)
            set_weight(next, w_next);
            HGC_STEP(6)
            HGC_STEP(7)
        }
#undef HGC_STEP
        if (WGRAD) {
            float sum = (l & 2) ? ((l & 1) ? r[3] : r[2]) : ((l & 1) ? r[1] : r[0]);
            if (p.blocks == 2) sum = sum + __shfl_xor(sum, kRowLanes, kWave);  // the other half of the row
            if (MAX && selves.first) {
                const uint32_t in_group = (uint32_t)(selves.first >> (lane & 48)) & 0xffffu;
                const float dot = __shfl(sum, (lane & 48) + __builtin_ctz(in_group | 0x10000u), kWave);
                self_dot = in_group ? dot : self_dot;
            }
            if (MAX && selves.repeats) sum = __builtin_amdgcn_inverse_ballot_w64(selves.repeats) ? self_dot : sum;
            if (en.slot >= 0 && task.block == 0) {
                const float value = p.negate ? -(sum * en.w) : sum;
                if (in_list_order) __builtin_nontemporal_store(value, p.gw_list + begin + c0 + entry_lane(l));
                else p.gw[en.slot] = value;
            }
        }
        slot_next = slot_after;
        en = next;
        selves = next_selves;
    }
    if (!live || fb >= p.F) return;
    float *const out = p.gfeat + (size_t)m * p.F + f;
    if (TAIL == kElements && f < fb) {
#pragma unroll
        for (int e = 1; e < VEC; ++e)
            if (f + e >= fb) __builtin_nontemporal_store(acc[e], out + e);
    } else {
        store_cols<VEC>(out, acc);
    }
}

template <int VEC, bool MAX, Scale SCALE, bool WGRAD>
void launch_packed(const GradRows &p, hipStream_t s) {
    const dim3 grid(ceil_div((long long)p.n_vert * p.blocks, 256 / kRowLanes)), block(256);
#define HGC_ROWS(ALIGNED, TAIL) accumulate_grad_rows_kernel<VEC, MAX, SCALE, ALIGNED, TAIL, WGRAD><<<grid, block, 0, s>>>(p)
    const Tail tail = row_tail(p.F, VEC, p.blocks);
    if constexpr (VEC == 1) {  // rows of 16 features
        HGC_ROWS(MAX, kFull);
    } else if constexpr (MAX && VEC != 3) {
        if (p.slot_shift != 0 || tail == kElements) HGC_ROWS(false, kElements);  // (right for full lanes too)
        else if (tail == kFull) HGC_ROWS(true, kFull);
        else HGC_ROWS(true, kLanes);
    } else {
        if (tail == kFull) HGC_ROWS(false, kFull);
        else if (tail == kLanes) HGC_ROWS(false, kLanes);
        else HGC_ROWS(false, kElements);
    }
#undef HGC_ROWS
}

template <int VEC>
int launch_rows(const GradRows &p, bool mean_and_max, bool want_w, Scale scale, hipStream_t s) {
#define HGC_SCALES(MAX, WG)                                                        \
    do {                                                                           \
        if (scale == kPow2) launch_packed<VEC, MAX, kPow2, WG>(p, s);              \
        else if (scale == kScaled) launch_packed<VEC, MAX, kScaled, WG>(p, s);     \
        else launch_packed<VEC, MAX, kDivide, WG>(p, s);                           \
    } while (0)
    if (!want_w) HGC_SCALES(false, false);
    else if (mean_and_max) HGC_SCALES(true, true);
    else HGC_SCALES(false, true);
#undef HGC_SCALES
    return check_launch("accumulate_grad_rows_kernel");
}

// the mean half of the gradient (rows of `pitch` floats) divided by the divisor, rows of F
__global__ __launch_bounds__(256) void divide_mean_half_kernel(const float *__restrict__ g, float *__restrict__ out,
                                                               long long total, int F, int pitch, float divisor) {
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= total) return;
    const long long v = t / F;
    out[t] = g[(size_t)v * pitch + (size_t)(t - v * F)] / divisor;
}

}  // namespace

bool accumulate_grad_rows_covers(int n_feat, int n_neigh, bool mean_and_max, bool slots, unsigned long long g_bytes) {
    return n_feat >= kRowLanes && n_feat <= 8 * kRowLanes && (!mean_and_max || (slots && n_neigh <= 254)) &&
           g_bytes <= kMaxRowBytes;
}

// The weight gradients of the targets in flight are 4-byte writes into the rows of everything that names them. Where those
// rows, with the gradient rows and slots that are gathered, are more than an XCD's L2 holds, lines leave it before they are
// whole and are written several times (fabric traffic five times the compulsory one at a million vertices, F = 128, window
// +-2000). In the order of the lists the values leave in whole lines, and a pass moves them to their slots. Whether that pays
// depends on how far apart the vertices of a list are; us of the gradient, slot by slot / in list order:
//   up to 2.6 MB of rows  slower: a million, K = 64, F = 128, banded +-1000 3773 / 3912, +-300 3546 / 3761
//   3.8 to 10 MB          faster: the same, +-1500 4318 / 3910, +-2000 4602 / 3985, +-3000 5127 / 4612, +-4000 6105 / 5966; K = 24,
//                         F = 64, +-4000 1680 / 1412, +-8000 2067 / 1996; 300,000, K = 64, F = 128, +-2000 1417 / 1216; 410,000,
//                         K = 40, F = 100, +-4000 1613 / 1492; a search's table, hits ordered by a coordinate, K = 40, F = 128
//                         1280 / 1273, a million, K = 64 4387 / 4100
//   16 to 50 MB           slower: a million, K = 64, F = 128, +-6000 7358 / 7577, +-16000 8400 / 9018; K = 24, F = 64, +-16000
//                         2420 / 2582; 300,000, K = 64, F = 128, +-16000 2560 / 2805; search tables, hits in no order, 16 events of
//                         410,000, K = 40, F = 128 2350 / 2426, 32 events of a million, K = 64 8249 / 8439 (but with K = 24 near
//                         50 MB F = 64, +-32000 2828 / 2767, a search's table of 700,000, F = 128 3006 / 2939)
//   beyond, where all     slower: 300,000, K = 64, F = 128, +-32000 2869 / 3032; targets drawn at random, 300,000, K = 64, F = 64
//   rows are up to 540    1808 / 1946, F = 128 2589 / 2812, 500,000, F = 64 2954 / 3318; a search's table of one event of 300,000,
//   MB, twice the         K = 64, F = 128 2592 / 2824; level: random, 410,000, K = 40, F = 128 2725 / 2726, 800,000, K = 24, F = 64
//   Infinity Cache        2352 / 2318
//   beyond 79 MB, where   faster: a million, K = 64, F = 128, +-32000 13385 / 11575, random 12771 / 11156; K = 24, F = 64, +-64000
//   they are 670 MB and   3826 / 3384, random 3242 / 2950; random, 500,000, K = 64, F = 128 5263 / 4785, 700,000, K = 24, F = 128
//   more                  3783 / 3482
// So the host asks for the size (100,000, +-2000 359 / 353, 20,000 87 / 93; asking and moving nothing costs 10 to 20 us) and leaves
// tables with a processing order as they are (300,000 vertices, K = 40, F = 128 907 / 1091), and the device looks at the span. (A
// mean alone gathers half as much.)
constexpr int kSpanSamples = 1024;
constexpr float kSpanNear = 3 << 20, kSpanFar = 12 << 20, kSpanWhole = 64 << 20;  // bytes; an XCD's L2 has 4 MB
constexpr long long kRowsWhole = 600ll << 20;

static bool list_order_may_pay(int n_vert, int n_feat, int n_neigh, bool mean_and_max) {
    return mean_and_max && (long long)n_vert * n_neigh >= 16000000 && n_neigh >= 24 && n_feat >= 64;
}

// *scattered = whether list order pays by the span of the rows between the first and the last vertex that name a target, on average
__global__ __launch_bounds__(kSpanSamples) void list_span_kernel(const int *__restrict__ inv_off, const int *__restrict__ inv_slots,
                                                                 int n_vert, int K, int row_bytes, int *__restrict__ scattered) {
    __shared__ float s_span[kSpanSamples / kWave];
    const int m = (int)((long long)threadIdx.x * n_vert / kSpanSamples);
    const int begin = inv_off[m], end = inv_off[m + 1];
    float span = begin < end ? (float)(inv_slots[end - 1] / K - inv_slots[begin] / K) : 0.f;
    for (int off = kWave / 2; off > 0; off >>= 1) span += __shfl_xor(span, off);
    if (lane_id() == 0) s_span[threadIdx.x / kWave] = span;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < kSpanSamples / kWave; ++i) span += s_span[i];
        const float bytes = span * (1.f / kSpanSamples) * (float)row_bytes;
        *scattered = (bytes > kSpanNear && bytes <= kSpanFar) || (bytes > kSpanWhole && (long long)n_vert * row_bytes >= kRowsWhole);
    }
}

static bool scratch_covers(int n_vert, int n_feat, int n_neigh, bool mean_and_max) {
    const unsigned long long n = (unsigned long long)std::max(n_vert, 0) * std::max(n_feat, 0) * sizeof(float);
    return accumulate_grad_rows_covers(n_feat, n_neigh, mean_and_max, true, n * (mean_and_max ? 2 : 1));
}

size_t accumulate_grad_rows_quotient_bytes(int n_vert, int n_feat, int n_neigh, bool mean_and_max, float divisor) {
    if (!scratch_covers(n_vert, n_feat, n_neigh, mean_and_max)) return 0;
    if (divisor == (float)(int)divisor && is_pow2((int)divisor)) return 0;
    return align_up((size_t)std::max(n_vert, 0) * n_feat * sizeof(float));
}

size_t accumulate_grad_rows_scratch_bytes(int n_vert, int n_feat, int n_neigh, bool mean_and_max, float divisor) {
    const size_t quotients = accumulate_grad_rows_quotient_bytes(n_vert, n_feat, n_neigh, mean_and_max, divisor);
    if (!scratch_covers(n_vert, n_feat, n_neigh, mean_and_max) || !list_order_may_pay(n_vert, n_feat, n_neigh, mean_and_max)) return quotients;
    return quotients + align_up((size_t)n_vert * n_neigh * sizeof(float)) + align_up(sizeof(int));
}

// Returns 1 where the shape is not covered. gw == nullptr: feature gradient only (mean only). scratch (may be null)
// holds, where there is room for them,
//   the quotients g / divisor where the divisor is no power of two (accumulate_grad_rows_quotient_bytes): N F divides in a
//   pass of their own instead of N K F inside the gather (150,000 vertices, K = 40, F = 64: 287 -> 262 us);
//   behind them the weight gradients in list order and whether they leave so (accumulate_grad_rows_scratch_bytes, see
//   list_order_may_pay), for an index without `skip`, no processing order and inv_slots on a 16-byte boundary.
int launch_accumulate_grad_rows(const float *g, const float *w, const float *feat, const unsigned char *maxslot,
                                const int *inv_off, const int *inv_slots, float *gw, float *gfeat, int n_vert, int K, int F,
                                int g_cols, bool mean_and_max, const int *order, float divisor, bool negate, int skip,
                                void *scratch, size_t scratch_bytes, hipStream_t s) {
    const bool want_w = gw != nullptr;
    const unsigned long long g_bytes = (unsigned long long)n_vert * g_cols * 4ull;
    if (!accumulate_grad_rows_covers(F, K, mean_and_max, maxslot != nullptr, g_bytes) || (mean_and_max && !want_w)) return 1;
    GradRows p;
    Scale scale = kDivide;
    p.g = g;
    const size_t quotient_bytes = accumulate_grad_rows_quotient_bytes(n_vert, F, K, mean_and_max, divisor);
    const bool room = scratch && scratch_bytes >= accumulate_grad_rows_scratch_bytes(n_vert, F, K, mean_and_max, divisor);
    p.gw_list = nullptr;
    p.scattered = nullptr;
    // (the list is read four entries at a time)
    if (room && want_w && skip == 0 && !order && list_order_may_pay(n_vert, F, K, mean_and_max) && (reinterpret_cast<uintptr_t>(inv_slots) & 15u) == 0) {
        char *const behind = static_cast<char *>(scratch) + quotient_bytes;
        int *const scattered = reinterpret_cast<int *>(behind + align_up((size_t)n_vert * K * sizeof(float)));
        p.gw_list = reinterpret_cast<float *>(behind);
        p.scattered = scattered;
        const int row_bytes = 4 * g_cols + 4 * K + F;
        list_span_kernel<<<1, kSpanSamples, 0, s>>>(inv_off, inv_slots, n_vert, K, row_bytes, scattered);
        if (const int rc = check_launch("list_span_kernel")) return rc;
    }
    if (divisor == (float)(int)divisor && is_pow2((int)divisor)) {
        scale = kPow2;
    } else if (scratch && scratch_bytes >= quotient_bytes) {
        scale = kScaled;
        const long long total = (long long)n_vert * F;
        divide_mean_half_kernel<<<ceil_div(total, 256), 256, 0, s>>>(g, static_cast<float *>(scratch), total, F, g_cols, divisor);
        const int rc = check_launch("divide_mean_half_kernel");
        if (rc) return rc;
        p.g = static_cast<const float *>(scratch);
    }
    p.g_max = mean_and_max ? g + F : nullptr;
    p.w = w;
    p.feat = feat;
    p.inv_off = inv_off;
    p.inv_slots = inv_slots;
    p.order = order;
    p.gw = gw;
    p.gfeat = gfeat;
    p.g_bytes = scale == kScaled ? (unsigned long long)n_vert * F * 4ull : g_bytes;
    p.g_max_bytes = g_bytes - (unsigned long long)F * 4ull;
    p.slot_shift = (uint32_t)(reinterpret_cast<uintptr_t>(maxslot) & 3u);
    p.maxslot = maxslot - p.slot_shift;
    p.slot_bytes = ((unsigned long long)n_vert * F + p.slot_shift + 3ull) / 4 * 4;  // whole words
    p.n_vert = n_vert;
    p.K = K;
    p.F = F;
    p.pitch = scale == kScaled ? F : g_cols;
    p.skip = skip;
    p.div_k = make_fast_div(K + skip);
    p.divisor = divisor;
    p.negate = negate;
    int vec, rc;
    row_shape(F, vec, p.blocks);
    switch (vec) {
        case 1: rc = launch_rows<1>(p, mean_and_max, want_w, scale, s); break;
        case 2: rc = launch_rows<2>(p, mean_and_max, want_w, scale, s); break;
        case 3: rc = launch_rows<3>(p, mean_and_max, want_w, scale, s); break;
        default: rc = launch_rows<4>(p, mean_and_max, want_w, scale, s); break;
    }
    if (rc || !p.gw_list) return rc;
    return launch_weight_grad_to_table(inv_off, inv_slots, p.gw_list, gw, n_vert, (long long)n_vert * K, p.scattered, s);
}

}  // namespace hgc
