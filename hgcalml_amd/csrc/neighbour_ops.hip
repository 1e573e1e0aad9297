// Ops next to the accumulate path that run over the same neighbour table:
//   * squared distances to listed neighbours (LocalDistance),
//   * push_knn forward and gradient.
//
// Reference behaviour restated here:
//   modules/compiled/push_knn_kernel.cc:40-62
//   modules/compiled/push_knn_grad_kernel.cc:23-71
//   modules/compiled/local_distance_kernel.cc:18-70
//
// The reference's device kernels scatter with atomicAdd; here every scatter is
// an ordered gather through the inverse neighbour index (ascending (vertex,
// slot) per target), so results do not depend on scheduling.
#include "accumulate_rows.hpp"

#include <algorithm>

namespace hgc {

// accumulate.hip
int accumulate_forward(const float *d_distances, const float *d_feat, const int *d_idxs, float *d_out_feat,
                       int *d_out_maxidxs, unsigned char *d_out_maxslots, int n_vert, int n_neigh, int n_feat,
                       int n_out_feat, int mean_and_max, float divisor, const int *d_order, float *d_out_weights,
                       hgc_stream_t stream);
int accumulate_gradient(const float *d_grad_from_out_features, const float *d_distances, const float *d_feat,
                        const int *d_max_feat_indices, const unsigned char *d_max_slots, const int *d_neigh_indices,
                        const int *d_inv_offsets, const int *d_inv_slots, float *d_out_grad_distances,
                        float *d_out_grad_features, int n_vert, int n_neigh, int n_feat, int n_grad_from_out_feat,
                        int mean_and_max, float divisor, const int *d_order, void *records, size_t records_bytes,
                        bool negate, void *scratch, size_t scratch_bytes, hgc_stream_t stream);

namespace {

// one thread per (vertex, slot): serial fp32 sum over the coordinates, 0 for a
// missing neighbour and for the vertex itself (order: the vertices are worked on in it)
__global__ __launch_bounds__(256) void local_distance_kernel(const int *__restrict__ idx,
                                                             const float *__restrict__ coord,
                                                             float *__restrict__ dist, int C, int n_in_vert,
                                                             long long total, int K, const int *__restrict__ order,
                                                             int n_out_vert) {
    long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= total) return;
    int i = (int)(t / K);
    if (order) {
        const int n = (int)(t - (long long)i * K);
        i = order[i];
        if ((uint32_t)i >= (uint32_t)n_out_vert) return;  // not a permutation: that vertex is left out
        t = (long long)i * K + n;
    }
    const int j = idx[t];
    float dsq = 0.f;
    if (j >= 0 && j < n_in_vert && j != i) {
        for (int c = 0; c < C; ++c) {
            const float d = coord[(size_t)i * C + c] - coord[(size_t)j * C + c];
            dsq = dsq + d * d;
        }
    }
    dist[t] = dsq;
}

// Gradient of push_knn, both outputs from one gather: a group of 16 lanes owns vertex v, fetches the
// upstream gradient rows of its K neighbours once and forms
//   feat_grad[v, f] = sum_n grad[idx[v,n], f] * w[v,n]   (serial, slot order: the reference's sum)
//   w_grad[v, n]    = sum_f grad[idx[v,n], f] * feat[v, f]
// the second as dot products per lane that a fixed exchange over the group adds up, four slots at a
// time. Lane l owns the VEC features from l*VEC on of each of the NB blocks of 16*VEC (rows of up to
// 256 features). Index and weight of 16 slots sit one per lane, slot s in lane entry_lane(s), which is
// the lane that ends up with the slot's dot product. Bound by vector issue like the accumulation's
// forward pass. On kNN tables (3-D Gaussian, processed in bin order) against one wave per vertex, or two
// separate passes where 64 does not divide the columns: 60,000 vertices, K = 24, F = 48 97 -> 23 us;
// 150,000, K = 64, F = 64 356 -> 125; 300,000, K = 64, F = 128 1346 -> 547; 200,000, K = 40, F = 256
// 1169 -> 477 (on tables that need no order 65 -> 21, 322 -> 123, 700 -> 527, 498 -> 438).
template <int VEC, int NB, acc::Tail TAIL>
__global__ __launch_bounds__(256) void push_grad_rows_kernel(const float *__restrict__ grad, const float *__restrict__ w,
                                                             const float *__restrict__ feat, const int *__restrict__ idx,
                                                             const int *__restrict__ order, float *__restrict__ feat_grad,
                                                             float *__restrict__ w_grad, int n_vert, int K, int F) {
    using namespace acc;
    const int lane = lane_id(), l = lane & (kRowLanes - 1);
    const GroupTask task = group_task(order, n_vert, 1);
    const bool live = task.vertex >= 0;
    const int v = live ? task.vertex : 0;
    const int *irow = idx + (size_t)v * K;
    const float *wrow = w + (size_t)v * K;
    const __amdgpu_buffer_rsrc_t rows = make_rows(grad, (unsigned long long)n_vert * F * 4ull);
    // Columns that a lane at the end of a row shares with its neighbour count in the neighbour's dot product only (see
    // Tail; only the last block of a row has any). owned[e]: the lanes whose element e of that block is theirs.
    uint32_t lane_bytes[NB];
    float own[NB][VEC], sum[NB][VEC];
    uint64_t owned[VEC];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int fb = (b * kRowLanes + l) * VEC, f = min(fb, F - VEC);
        lane_bytes[b] = (uint32_t)f * 4u;
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            const float x = feat[(size_t)v * F + f + e];
            own[b][e] = f + e >= fb ? x : 0.f;
            sum[b][e] = 0.f;
            if (b == NB - 1) owned[e] = __builtin_amdgcn_ballot_w64(f + e >= fb);
        }
    }
    const int mine = entry_lane(l);
    bool in_row = live && mine < K;
    int j_next = in_row ? irow[mine] : -1;
    float w_next = in_row ? wrow[mine] : 0.f;
    for (int c0 = 0; c0 < K; c0 += kRowLanes) {
        const bool store = in_row;
        const bool has_row = (uint32_t)j_next < (uint32_t)n_vert;
        const uint32_t offset = has_row ? (uint32_t)j_next * (uint32_t)(F * 4) : kNoRow;  // no row: 0 is read ...
        const float wn = has_row ? w_next : 0.f;                                           // ... and adds 0
        in_row = live && c0 + kRowLanes + mine < K;
        j_next = in_row ? irow[c0 + kRowLanes + mine] : -1;
        w_next = in_row ? wrow[c0 + kRowLanes + mine] : 0.f;
        float r[4] = {};
#define HGC_PUSH_SLOT(Q, U)                                                                                  \
    {                                                                                                        \
        const uint32_t row = group_bcast<entry_lane((Q) * 4 + (U))>(offset);                                 \
        _Pragma("unroll") for (int b = 0; b < NB; ++b) load_cols<VEC>(rows, row + lane_bytes[b], x[U][b]);    \
        ws[U] = group_bcast<entry_lane((Q) * 4 + (U))>(wn);                                                  \
    }
#define HGC_PUSH_FOUR(Q)                                                                                     \
    if (c0 + (Q) * 4 < K) {                                                                                  \
        float x[4][NB][VEC], ws[4], val[4];                                                                  \
        HGC_PUSH_SLOT(Q, 0)                                                                                  \
        HGC_PUSH_SLOT(Q, 1)                                                                                  \
        HGC_PUSH_SLOT(Q, 2)                                                                                  \
        HGC_PUSH_SLOT(Q, 3)                                                                                  \
        _Pragma("unroll") for (int u = 0; u < 4; ++u) {                                                      \
            val[u] = 0.f;                                                                                    \
            float before = 0.f;                                                                              \
            _Pragma("unroll") for (int b = 0; b < NB; ++b) {                                                 \
                if (b == NB - 1) before = val[u];                                                            \
                _Pragma("unroll") for (int e = 0; e < VEC; ++e) {                                            \
                    const bool counts = TAIL != kElements || b < NB - 1 || __builtin_amdgcn_inverse_ballot_w64(owned[e]);\
                    val[u] = __builtin_fmaf(own[b][e], counts ? x[u][b][e] : 0.f, val[u]);                   \
                    sum[b][e] = sum[b][e] + x[u][b][e] * ws[u];                                              \
                }                                                                                            \
            }                                                                                                \
            if (TAIL == kLanes) val[u] = __builtin_amdgcn_inverse_ballot_w64(owned[0]) ? val[u] : before;    \
        }                                                                                                    \
        r[Q] = group_sum_4(val, lane);                                                                       \
    }
        HGC_PUSH_FOUR(0)
        HGC_PUSH_FOUR(1)
        HGC_PUSH_FOUR(2)
        HGC_PUSH_FOUR(3)
#undef HGC_PUSH_FOUR
#undef HGC_PUSH_SLOT
        // lane l holds the sums of slot 4 q + (l >> 2) in r[q]; its own slot has q = l & 3
        const float dot = (l & 2) ? ((l & 1) ? r[3] : r[2]) : ((l & 1) ? r[1] : r[0]);
        if (store) w_grad[(size_t)v * K + c0 + mine] = has_row ? dot : 0.f;
    }
    if (!live) return;
#pragma unroll
    for (int b = 0; b < NB; ++b)
        if ((b * kRowLanes + l) * VEC < F) store_cols<VEC>(feat_grad + (size_t)v * F + (lane_bytes[b] >> 2), sum[b]);
}

// returns 1 when the shape is not covered
int launch_push_grad_rows(const float *grad, const float *w, const float *feat, const int *idx, const int *order,
                          float *feat_grad, float *w_grad, int n_vert, int K, int F, hipStream_t s) {
    using namespace acc;
    if (F > 256 || (unsigned long long)n_vert * (unsigned long long)F * 4ull > kMaxRowBytes) return 1;
    int vec, nb;
    row_shape(F, vec, nb);
    const Tail tail = row_tail(F, vec, nb);
    const dim3 grid(ceil_div(n_vert, 256 / kRowLanes)), block(256);
#define HGC_PUSH_TAIL(VEC, NB, TAIL) \
    push_grad_rows_kernel<VEC, NB, TAIL><<<grid, block, 0, s>>>(grad, w, feat, idx, order, feat_grad, w_grad, n_vert, K, F)
#define HGC_PUSH_GRAD(VEC, NB)                                   \
    case VEC * 10 + NB:                                          \
        if (tail == kFull) HGC_PUSH_TAIL(VEC, NB, kFull);        \
        else if (tail == kLanes) HGC_PUSH_TAIL(VEC, NB, kLanes); \
        else HGC_PUSH_TAIL(VEC, NB, kElements);                  \
        break
    switch (vec * 10 + nb) {
        HGC_PUSH_GRAD(1, 1);
        HGC_PUSH_GRAD(2, 1);
        HGC_PUSH_GRAD(3, 1);
        HGC_PUSH_GRAD(4, 1);
        HGC_PUSH_GRAD(3, 2);
        HGC_PUSH_GRAD(4, 2);
        HGC_PUSH_GRAD(3, 3);
        HGC_PUSH_GRAD(4, 3);
        HGC_PUSH_GRAD(4, 4);
        default: return 1;
    }
#undef HGC_PUSH_GRAD
#undef HGC_PUSH_TAIL
    return check_launch("push_grad_rows_kernel");
}

}  // namespace
}  // namespace hgc

using namespace hgc;

namespace {

// weights of AccumulateKnn, w = exp(-d) (modules/accknn_op.py:52), and the chain rule back to
// the distances, gd = -(gw * w): one pass each instead of two framework kernels
__global__ __launch_bounds__(256) void exp_neg_kernel(const float *__restrict__ d, float *__restrict__ w,
                                                      long long n) {
    const long long i = ((long long)blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (i + 4 <= n) {
        const float4 v = *reinterpret_cast<const float4 *>(d + i);
        *reinterpret_cast<float4 *>(w + i) = float4{expf(-v.x), expf(-v.y), expf(-v.z), expf(-v.w)};
    } else {
        for (long long j = i; j < n; ++j) w[j] = expf(-d[j]);
    }
}

// (gd may be gw)
__global__ __launch_bounds__(256) void exp_neg_grad_kernel(const float *gw, const float *__restrict__ w, float *gd,
                                                           long long n) {
    const long long i = ((long long)blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (i + 4 <= n) {
        const float4 a = *reinterpret_cast<const float4 *>(gw + i), b = *reinterpret_cast<const float4 *>(w + i);
        *reinterpret_cast<float4 *>(gd + i) = float4{-(a.x * b.x), -(a.y * b.y), -(a.z * b.z), -(a.w * b.w)};
    } else {
        for (long long j = i; j < n; ++j) gd[j] = -(gw[j] * w[j]);
    }
}


// ---- feature-weighted moments of the neighbours' coordinates ----------------------
//
// modules/neighbour_covariance_op.py:8-62 builds, with w = exp(-distsq) and a = the
// (activated) features,
//   S[v,f]       = sum_n w[v,n] a[j,f]
//   mean[v,f,c]  = sum_n w[v,n] a[j,f] x[j,c] / (S[v,f] + 1e-3)
//   cov[v,f,c,d] = sum_n w[v,n] a[j,f] (x[j,c] - mean[j,f,c]) (x[j,d] - mean[j,f,d]) / (S[v,f] + 1e-3)
// (j = idx[v,n]; every neighbour is centred on ITS OWN mean) out of three mean-only
// accumulations over matrices of F, F*C and F*C*C columns that it materialises first.
// Here two passes over the neighbour table do it, one thread per (vertex, feature): the
// first gathers a[j,f] and x[j,:], the second a[j,f], x[j,:] and mean[j,f,:] and forms the
// C*C products in registers. The sums run over the slots in order and every term is formed
// as the composition forms it -- ((x*a)*w, ((cen_c*cen_d)*a)*w, the sum divided by K and
// multiplied by K again as the accumulation's mean is) -- so the results are its bits.

__device__ __forceinline__ float divide_no_nan(float a, float b) { return b == 0.f ? 0.f : a / b; }

// A wave's 64 (vertex, feature) pairs belong to a few consecutive vertices of the processing order. It puts indices and
// weights of 32 of their slots (16 where a wave has more than 16 vertices) into its own part of LDS, one lane per slot,
// and each lane reads them there two slots per 16-byte load; the rows of four slots are gathered together.
// Index and weight as loads of every lane (the same address for the lanes of a vertex) cost as much of the L1's address
// rate as the gathers themselves: 40,000 vertices, K = 32, F = 8, C = 4 26 us for the means and 37 for the covariance
// before, the whole call with its search 161 -> 141 us. What bounds them now (18 and 29 us) is the latency of the gathered
// rows: 5000 waves are five per SIMD, a third to 44 % of their time is waiting, and vector issue is 45 and 56 % busy.
// Workgroups of one XCD take consecutive vertices.
constexpr int kMomentSlots = 4, kMomentWaves = 4;

struct alignas(8) Slot {
    int j;  // -1: no neighbour
    float w;
};

// vertices that 64 consecutive pairs can belong to, slots of each that are in LDS at a time
inline int moment_vertices(int n_feat) { return std::min(kWave, (kWave - 2 + n_feat) / n_feat + 1); }
inline int moment_chunk(int n_feat) { return moment_vertices(n_feat) > 16 ? 16 : 32; }
inline size_t moment_lds_bytes(int n_feat) {
    // two slots of padding: rows of 36 or 68 dwords, the 16-byte reads of up to 16 vertices meet no bank twice
    return (size_t)kMomentWaves * moment_vertices(n_feat) * (moment_chunk(n_feat) + 2) * sizeof(Slot);
}

// Calls term(j, w, valid) for the four slots of every step, in order, with the rows of a step requested by gather(u, j).
template <typename Gather, typename Term>
__device__ __forceinline__ void for_each_slot(Slot *const staged, const int lane, const int local, const int n_local,
                                              const int my_row, const int chunk_bits, const int *__restrict__ idx,
                                              const float *__restrict__ weights, const int n_neigh, const int n_vert,
                                              Gather gather, Term term) {
    const int chunk = 1 << chunk_bits, stride = chunk + 2;
    const Slot *const mine = staged + local * stride;
    for (int n0 = 0; n0 < n_neigh; n0 += chunk) {
        for (int e0 = 0; e0 < n_local << chunk_bits; e0 += kWave) {
            const int e = e0 + lane, v = e >> chunk_bits, n = n0 + (e & (chunk - 1));
            const int row = __shfl(my_row, v & (kWave - 1));
            if (v < n_local) {
                Slot slot{-1, 0.f};
                if (row >= 0 && n < n_neigh) {
                    const int at = row * n_neigh + n;
                    slot = {idx[at], weights[at]};
                    if ((unsigned)slot.j >= (unsigned)n_vert) slot.j = -1;
                }
                staged[v * stride + (e & (chunk - 1))] = slot;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const int n_steps = min(chunk, n_neigh - n0);
        for (int n = 0; n < n_steps; n += kMomentSlots) {
            Slot slot[kMomentSlots];
#pragma unroll
            for (int u = 0; u < kMomentSlots; u += 2) {
                const int4 two = *reinterpret_cast<const int4 *>(mine + n + u);
                slot[u] = {two.x, __int_as_float(two.y)};
                slot[u + 1] = {two.z, __int_as_float(two.w)};
            }
            int any_missing = 0;
#pragma unroll
            for (int u = 0; u < kMomentSlots; ++u) {
                gather(u, (unsigned)max(slot[u].j, 0));
                any_missing |= slot[u].j;
            }
            if (__all(any_missing >= 0)) {
#pragma unroll
                for (int u = 0; u < kMomentSlots; ++u) term(u, slot[u].w);
            } else {
#pragma unroll
                for (int u = 0; u < kMomentSlots; ++u)
                    if (slot[u].j >= 0) term(u, slot[u].w);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // the next chunk overwrites what was read here
        __builtin_amdgcn_wave_barrier();
    }
}

// the pair a lane owns: vertex (-1 past the end) and feature, and its place among the wave's vertices
struct MomentPair {
    int v, f, local, n_local, row_of_lane;
};

__device__ __forceinline__ MomentPair moment_pair(const int *__restrict__ order, const int lane, int n_vert, int n_feat) {
    const long long wave_first = ((long long)xcd_contiguous_block(blockIdx.x, gridDim.x) * kMomentWaves + (threadIdx.x >> 6)) * kWave;
    const long long t = wave_first + lane;
    const int first = (int)(wave_first / n_feat), i = (int)(t / n_feat);
    MomentPair m;
    m.f = (int)(t - (long long)i * n_feat);
    m.local = i - first;
    m.n_local = min((int)((wave_first + kWave - 1) / n_feat), n_vert - 1) - first + 1;
    // processing order with locality: results do not depend on it
    int row = -1;
    if (lane < m.n_local) row = order ? order[first + lane] : first + lane;
    if ((unsigned)row >= (unsigned)n_vert) row = -1;
    m.row_of_lane = row;
    const int v = __shfl(row, m.local & (kWave - 1));
    m.v = i < n_vert ? v : -1;
    return m;
}

template <int C>
__global__ __launch_bounds__(kMomentWaves *kWave) void neighbour_means_kernel(
    const float *__restrict__ coords, const float *__restrict__ weights, const float *__restrict__ feats,
    const int *__restrict__ idx, float *__restrict__ sumw, float *__restrict__ means, const int *__restrict__ order,
    int n_vert, int n_feat, int n_neigh, int chunk_bits, int wave_slots) {
    extern __shared__ __align__(16) char s_slots[];
    Slot *const staged = reinterpret_cast<Slot *>(s_slots) + (threadIdx.x >> 6) * wave_slots;
    const int lane = threadIdx.x & (kWave - 1);
    const MomentPair m = moment_pair(order, lane, n_vert, n_feat);
    if (m.n_local <= 0) return;
    const int local = m.v >= 0 ? m.local : 0;
    float s = 0.f, sc[C], a[kMomentSlots], x[kMomentSlots][C];
#pragma unroll
    for (int c = 0; c < C; ++c) sc[c] = 0.f;
    for_each_slot(
        staged, lane, local, m.n_local, m.row_of_lane, chunk_bits, idx, weights, n_neigh, n_vert,
        [&](int u, unsigned j) {
            a[u] = feats[j * (unsigned)n_feat + m.f];
#pragma unroll
            for (int c = 0; c < C; ++c) x[u][c] = coords[j * C + c];
        },
        [&](int u, float w) {
            s = s + a[u] * w;
#pragma unroll
            for (int c = 0; c < C; ++c) sc[c] = sc[c] + (x[u][c] * a[u]) * w;
        });
    if (m.v < 0) return;
    const float kf = (float)n_neigh;
    const float S = (s / kf) * kf;
    const size_t out = (size_t)m.v * n_feat + m.f;
    sumw[out] = S;
#pragma unroll
    for (int c = 0; c < C; ++c) means[out * C + c] = divide_no_nan((sc[c] / kf) * kf, S + 1e-3f);
}

template <int C>
__global__ __launch_bounds__(kMomentWaves *kWave) void neighbour_covariance_kernel(
    const float *__restrict__ coords, const float *__restrict__ weights, const float *__restrict__ feats,
    const int *__restrict__ idx, const float *__restrict__ sumw, const float *__restrict__ means, float *__restrict__ cov,
    const int *__restrict__ order, int n_vert, int n_feat, int n_neigh, int chunk_bits, int wave_slots) {
    extern __shared__ __align__(16) char s_slots[];
    Slot *const staged = reinterpret_cast<Slot *>(s_slots) + (threadIdx.x >> 6) * wave_slots;
    const int lane = threadIdx.x & (kWave - 1);
    const MomentPair m = moment_pair(order, lane, n_vert, n_feat);
    if (m.n_local <= 0) return;
    const int local = m.v >= 0 ? m.local : 0;
    // the lower triangle is accumulated, the products are symmetric bit for bit
    float acc[C][C], a[kMomentSlots], x[kMomentSlots][C], mean[kMomentSlots][C];
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int d = 0; d < C; ++d) acc[c][d] = 0.f;
    for_each_slot(
        staged, lane, local, m.n_local, m.row_of_lane, chunk_bits, idx, weights, n_neigh, n_vert,
        [&](int u, unsigned j) {
            const unsigned at = j * (unsigned)n_feat + m.f;
            a[u] = feats[at];
#pragma unroll
            for (int c = 0; c < C; ++c) x[u][c] = coords[j * C + c], mean[u][c] = means[(size_t)at * C + c];
        },
        [&](int u, float w) {
            float cen[C];
#pragma unroll
            for (int c = 0; c < C; ++c) cen[c] = x[u][c] - mean[u][c];
#pragma unroll
            for (int c = 0; c < C; ++c)
#pragma unroll
                for (int d = 0; d <= c; ++d) acc[c][d] = acc[c][d] + ((cen[c] * cen[d]) * a[u]) * w;
        });
    if (m.v < 0) return;
    const float kf = (float)n_neigh;
    const size_t at = (size_t)m.v * n_feat + m.f;
    const float den = sumw[at] + 1e-3f;
    float *out = cov + at * C * C;
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int d = 0; d < C; ++d) out[c * C + d] = divide_no_nan((acc[c > d ? c : d][c > d ? d : c] / kf) * kf, den);
}

template <int C>
int launch_neighbour_covariance(const float *coords, const float *weights, const float *feats, const int *idx, float *cov,
                                float *means, float *sumw, const int *order, int n_vert, int n_feat, int n_neigh,
                                hipStream_t s) {
    const int blocks = ceil_div((long long)n_vert * n_feat, kMomentWaves * kWave);
    const int chunk = moment_chunk(n_feat), chunk_bits = chunk == 32 ? 5 : 4;
    const int wave_slots = moment_vertices(n_feat) * (chunk + 2);
    const size_t lds = moment_lds_bytes(n_feat);
    neighbour_means_kernel<C><<<blocks, kMomentWaves * kWave, lds, s>>>(coords, weights, feats, idx, sumw, means, order,
                                                                        n_vert, n_feat, n_neigh, chunk_bits, wave_slots);
    int rc = check_launch("neighbour_means_kernel");
    if (rc) return rc;
    neighbour_covariance_kernel<C><<<blocks, kMomentWaves * kWave, lds, s>>>(
        coords, weights, feats, idx, sumw, means, cov, order, n_vert, n_feat, n_neigh, chunk_bits, wave_slots);
    return check_launch("neighbour_covariance_kernel");
}

}  // namespace

extern "C" {

int hgc_neighbour_covariance(const float *d_coords, const float *d_weights, const float *d_feats, const int *d_n_idxs,
                             const int *d_vertex_order, float *d_covariance, float *d_means, float *d_sum_weights,
                             int n_vert, int n_coords, int n_feat, int n_neigh, hgc_stream_t stream) {
    HGC_REQUIRE(n_vert >= 0 && n_coords >= 1 && n_feat >= 1 && n_neigh >= 1, "bad sizes");
    if (n_coords > 6) return fail(HGC_ERR_UNSUPPORTED, "neighbour covariance is built for up to 6 coordinates");
    HGC_REQUIRE((long long)n_vert * std::max(n_neigh, n_feat * n_coords * n_coords) < (1ll << 31),
                "tensor too large for int32 indexing");
    if (n_vert == 0) return HGC_OK;
    HGC_REQUIRE(d_coords && d_weights && d_feats && d_n_idxs && d_covariance && d_means && d_sum_weights, "null pointer");
    hipStream_t s = as_stream(stream);
#define HGC_COV(C)                                                                                                  \
    case C:                                                                                                         \
        return launch_neighbour_covariance<C>(d_coords, d_weights, d_feats, d_n_idxs, d_covariance, d_means,        \
                                              d_sum_weights, d_vertex_order, n_vert, n_feat, n_neigh, s)
    switch (n_coords) {
        HGC_COV(1);
        HGC_COV(2);
        HGC_COV(3);
        HGC_COV(4);
        HGC_COV(5);
        HGC_COV(6);
    }
#undef HGC_COV
    return HGC_ERR_UNSUPPORTED;
}

int hgc_local_distance_ordered(const int *d_neigh_idxs, const float *d_coords, const int *d_vertex_order,
                               float *d_distances, int n_coords, int n_in_vert, int n_out_vert, int n_neigh,
                               hgc_stream_t stream) {
    HGC_REQUIRE(n_in_vert >= 0 && n_out_vert >= 0 && n_out_vert <= n_in_vert && n_neigh >= 1 && n_coords >= 1,
                "bad sizes");
    HGC_REQUIRE((long long)n_out_vert * n_neigh < (1ll << 31), "tensor too large for int32 indexing");
    if (n_out_vert == 0) return HGC_OK;
    HGC_REQUIRE(d_neigh_idxs && d_coords && d_distances, "null pointer");
    const long long total = (long long)n_out_vert * n_neigh;
    local_distance_kernel<<<ceil_div(total, 256), 256, 0, as_stream(stream)>>>(
        d_neigh_idxs, d_coords, d_distances, n_coords, n_in_vert, total, n_neigh, d_vertex_order, n_out_vert);
    return check_launch("local_distance_kernel");
}

int hgc_local_distance(const int *d_neigh_idxs, const float *d_coords, float *d_distances, int n_coords, int n_in_vert,
                       int n_out_vert, int n_neigh, hgc_stream_t stream) {
    return hgc_local_distance_ordered(d_neigh_idxs, d_coords, nullptr, d_distances, n_coords, n_in_vert, n_out_vert,
                                      n_neigh, stream);
}

int hgc_push_knn_ordered(const float *d_weights, const float *d_feat, const int *d_idxs, const int *d_inv_offsets,
                         const int *d_inv_slots, const int *d_vertex_order, float *d_out_feat, int n_vert, int n_neigh,
                         int n_feat, hgc_stream_t stream) {
    (void)d_idxs;  // the inverse index carries all the op needs of the neighbour table
    HGC_REQUIRE(n_vert <= 0 || d_out_feat, "null pointer");
    // out[m, f] = sum over (v, n) naming m of feat[v, f] * w[v, n]: the mean-only
    // feature gradient of the accumulation with `feat` as upstream gradient, not divided by K
    return accumulate_gradient(d_feat, d_weights, nullptr, nullptr, nullptr, nullptr, d_inv_offsets, d_inv_slots,
                               nullptr, d_out_feat, n_vert, n_neigh, n_feat, n_feat, 0, 1.f, d_vertex_order, nullptr, 0,
                               false, nullptr, 0, stream);
}

int hgc_push_knn(const float *d_weights, const float *d_feat, const int *d_idxs, const int *d_inv_offsets,
                 const int *d_inv_slots, float *d_out_feat, int n_vert, int n_neigh, int n_feat, hgc_stream_t stream) {
    return hgc_push_knn_ordered(d_weights, d_feat, d_idxs, d_inv_offsets, d_inv_slots, nullptr, d_out_feat, n_vert,
                                n_neigh, n_feat, stream);
}

int hgc_push_knn_grad_ordered(const float *d_grad, const float *d_weights, const float *d_feat, const int *d_idxs,
                              const int *d_vertex_order, float *d_feat_grad, float *d_w_grad, int n_vert, int n_neigh,
                              int n_feat, hgc_stream_t stream) {
    HGC_REQUIRE(n_vert <= 0 || (d_feat_grad && d_w_grad), "null pointer");
    HGC_REQUIRE(n_vert >= 0 && n_neigh >= 1 && n_feat >= 1, "bad sizes");
    HGC_REQUIRE((long long)n_vert * n_neigh < (1ll << 31), "n_vert * n_neigh must stay below 2^31");
    if (n_vert == 0) return HGC_OK;
    HGC_REQUIRE(d_grad && d_weights && d_feat && d_idxs, "null pointer");
    {
        // both gradients from one gather pass where that kernel covers the shape
        const int rc = launch_push_grad_rows(d_grad, d_weights, d_feat, d_idxs, d_vertex_order, d_feat_grad, d_w_grad,
                                             n_vert, n_neigh, n_feat, as_stream(stream));
        if (rc <= 0) return rc;
    }
    // feat_grad[v, f] = sum_n grad[idx[v,n], f] * w[v,n]: the mean-only forward over `grad`, not divided by K
    int rc = accumulate_forward(d_weights, d_grad, d_idxs, d_feat_grad, nullptr, nullptr, n_vert, n_neigh, n_feat,
                                n_feat, 0, 1.f, d_vertex_order, nullptr, stream);
    if (rc) return rc;
    // w_grad[v, n] = sum_f grad[idx[v,n], f] * feat[v, f]: the weight gradient with the roles of the
    // vertex's own row (feat) and the gathered rows (grad) as in the accumulation's
    return accumulate_gradient(d_feat, nullptr, d_grad, nullptr, nullptr, d_idxs, nullptr, nullptr, d_w_grad, nullptr,
                               n_vert, n_neigh, n_feat, n_feat, 0, 1.f, nullptr, nullptr, 0, false, nullptr, 0, stream);
}

int hgc_push_knn_grad(const float *d_grad, const float *d_weights, const float *d_feat, const int *d_idxs,
                      float *d_feat_grad, float *d_w_grad, int n_vert, int n_neigh, int n_feat, hgc_stream_t stream) {
    return hgc_push_knn_grad_ordered(d_grad, d_weights, d_feat, d_idxs, nullptr, d_feat_grad, d_w_grad, n_vert, n_neigh,
                                     n_feat, stream);
}

int hgc_exp_neg(const float *d_distances, float *d_weights, long long n_values, hgc_stream_t stream) {
    HGC_REQUIRE(n_values >= 0, "bad sizes");
    if (n_values == 0) return HGC_OK;
    HGC_REQUIRE(d_distances && d_weights, "null pointer");
    HGC_REQUIRE(((reinterpret_cast<uintptr_t>(d_distances) | reinterpret_cast<uintptr_t>(d_weights)) & 15u) == 0,
                "arrays must start on a 16-byte boundary");
    exp_neg_kernel<<<ceil_div(ceil_div(n_values, 4), 256), 256, 0, as_stream(stream)>>>(d_distances, d_weights,
                                                                                       n_values);
    return check_launch("exp_neg");
}

int hgc_exp_neg_grad(const float *d_weight_grad, const float *d_weights, float *d_distance_grad, long long n_values,
                     hgc_stream_t stream) {
    HGC_REQUIRE(n_values >= 0, "bad sizes");
    if (n_values == 0) return HGC_OK;
    HGC_REQUIRE(d_weight_grad && d_weights && d_distance_grad, "null pointer");
    HGC_REQUIRE(((reinterpret_cast<uintptr_t>(d_weight_grad) | reinterpret_cast<uintptr_t>(d_weights) |
                  reinterpret_cast<uintptr_t>(d_distance_grad)) & 15u) == 0,
                "arrays must start on a 16-byte boundary");
    exp_neg_grad_kernel<<<ceil_div(ceil_div(n_values, 4), 256), 256, 0, as_stream(stream)>>>(
        d_weight_grad, d_weights, d_distance_grad, n_values);
    return check_launch("exp_neg_grad");
}

}  // extern "C"
