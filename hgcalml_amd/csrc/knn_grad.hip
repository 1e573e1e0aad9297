// Gradient of the kNN squared distances w.r.t. the coordinates (SelectKnnGrad).
//
// Reference behaviour restated here:
//   modules/compiled/select_knn_grad_kernel.cu.cc:81-164
//
//   grad[i,c] = - sum_n 2 g[i,n] (x[idx[i,n],c] - x[i,c])       (slot order)
//               + sum over (v,n) naming i of 2 g[v,n] (x[i,c] - x[v,c])   (ascending (v,n))
// every term rounded into the float sum one after the other. The reference's `2. * g * (x_k - x_i)` is exact in
// double; subtracted from the sum there and rounded to float it is a fused multiply-add (apart from
// roundings that the double subtraction moves onto the middle between two floats, one in 2^29), rounded to
// float and added it is a float product and a float sum. The factor 2 goes to the difference: coordinates whose
// differences it could take beyond the largest float have infinite distances, a gradient may be that large.
//
// Both sums are chains, so a lane owns one coordinate of one vertex and walks its slots and list entries
// serially; what it walks over is fetched by the wave together: 16 slots (entries) of its 16 vertices (8
// with more than 4 coordinates) at a time, one lane per slot for index, gradient and coordinate row,
// handed over through LDS as differences. (One thread per coordinate doing its own loads fetched every
// index and gradient C times and issued 16 distinct lines per load: Gaussian points in bin order, 150,000,
// K = 65, C = 4 224 -> 138 us (160 in a training step, with other kernels' data in the caches); 240,000,
// K = 41, C = 3 248 -> 127.) What bounds it is the L2: 24 M lines at
// 136 G/s for gathers of 4 and 16 bytes; vector issue 12 %. Consecutive workgroups of an XCD take
// consecutive vertices of the processing order, which keeps the scattered gradients of the second sum in
// that XCD's L2.
#include "accumulate_rows.hpp"

#include <algorithm>

namespace hgc {

namespace {

using namespace acc;

constexpr int kChunk = 16;  // slots per vertex and step
constexpr int kGradWaves = 4;

template <int C>
__device__ __forceinline__ void load_row(const float *__restrict__ coord, int row, float (&x)[C]) {
    typedef float vec_t __attribute__((ext_vector_type(C == 2 ? 2 : 4), aligned(4)));
    const float *p = coord + (size_t)row * C;
    if constexpr (C == 2 || C == 4) {
        const vec_t v = *reinterpret_cast<const vec_t *>(p);
#pragma unroll
        for (int c = 0; c < C; ++c) x[c] = v[c];
    } else {
#pragma unroll
        for (int c = 0; c < C; ++c) x[c] = p[c];
    }
}

template <int C>
__global__ __launch_bounds__(kGradWaves *kWave) void knn_grad_kernel(const float *__restrict__ grad_dist,
                                                                    const int *__restrict__ idx,
                                                                    const float *__restrict__ coord,
                                                                    const int *__restrict__ inv_off,
                                                                    const int *__restrict__ inv_slots,
                                                                    float *__restrict__ out, int n_vert, int K,
                                                                    const FastDiv div_k,
                                                                    const int *__restrict__ order) {
    constexpr int kLanes = C <= 4 ? 4 : 8;          // lanes per vertex
    constexpr int kVertices = kWave / kLanes;       // per wave
    constexpr int kPairs = kVertices * kChunk / kWave;
    constexpr int kRow = kChunk * kLanes + kLanes;  // padded: the lanes of a wave then read all banks
    __shared__ float s_diff[kGradWaves][kVertices * kRow];
    __shared__ float s_grad[kGradWaves][kVertices * (kChunk + 1)];
    const int wave = threadIdx.x >> 6, lane = lane_id();
    float *const diff = s_diff[wave], *const grad = s_grad[wave];
    const int tile = xcd_contiguous_block(blockIdx.x, gridDim.x);
    const int r0 = (tile * kGradWaves + wave) * kVertices;

    // of the pairs (vertex, slot) this lane fetches: pair p is slot lane % 16 of vertex p * 4 + lane / 16
    const int s = lane & (kChunk - 1);
    int vertex[kPairs], begin[kPairs], count[kPairs];
    float x[kPairs][C];
    int longest = 0;
#pragma unroll
    for (int p = 0; p < kPairs; ++p) {
        const int r = r0 + p * (kWave / kChunk) + lane / kChunk;
        int i = r < n_vert ? (order ? order[r] : r) : -1;
        if ((uint32_t)i >= (uint32_t)n_vert) i = -1;  // not a permutation: that vertex is left out
        vertex[p] = i;
        begin[p] = i >= 0 ? inv_off[i] : 0;
        count[p] = i >= 0 ? inv_off[i + 1] - begin[p] : 0;
        if (i >= 0) load_row<C>(coord, i, x[p]);
        else
#pragma unroll
            for (int c = 0; c < C; ++c) x[p][c] = 0.f;
        longest = max(longest, count[p]);
    }
    longest = max(max(readlane_i32(longest, 0), readlane_i32(longest, 16)),
                  max(readlane_i32(longest, 32), readlane_i32(longest, 48)));

    // the chain this lane adds up
    const int cv = lane / kLanes, cc = lane % kLanes;
    const float *const my_diff = diff + cv * kRow + cc, *const my_grad = grad + cv * (kChunk + 1);
    float sum = 0.f;
    // Steps: the indices (slots) of a chunk are requested two steps, gradients and rows one step before the
    // chunk is added up.
    int k_next[kPairs];
    float g_next[kPairs], x_next[kPairs][C];
    uint64_t counts[kPairs];  // lanes whose pair has a neighbour; the others hand over 0 (inf - inf is no 0)
    auto hand_over = [&](bool own) {  // own: neighbour minus vertex, otherwise vertex minus namer
        wave_lds_fence();
#pragma unroll
        for (int p = 0; p < kPairs; ++p) {
            const int v = p * (kWave / kChunk) + lane / kChunk;
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const float d = own ? x_next[p][c] - x[p][c] : x[p][c] - x_next[p][c];
                diff[v * kRow + s * kLanes + c] = __builtin_amdgcn_inverse_ballot_w64(counts[p]) ? 2.f * d : 0.f;
            }
            grad[v * (kChunk + 1) + s] = g_next[p];
        }
        wave_lds_fence();
    };
    auto request_indices = [&](int n0) {
#pragma unroll
        for (int p = 0; p < kPairs; ++p) k_next[p] = vertex[p] >= 0 && n0 + s < K ? idx[(size_t)vertex[p] * K + n0 + s] : -1;
    };
    auto request_neighbours = [&](int n0) {
#pragma unroll
        for (int p = 0; p < kPairs; ++p) {
            const bool ok = (uint32_t)k_next[p] < (uint32_t)n_vert;
            counts[p] = __builtin_amdgcn_ballot_w64(ok);
            const size_t at = (size_t)max(vertex[p], 0) * K + min(n0 + s, K - 1);
            g_next[p] = ok ? grad_dist[at] : 0.f;
            load_row<C>(coord, ok ? k_next[p] : max(vertex[p], 0), x_next[p]);
        }
    };
    auto request_slots = [&](int e0) {
#pragma unroll
        for (int p = 0; p < kPairs; ++p) k_next[p] = e0 + s < count[p] ? inv_slots[begin[p] + e0 + s] : -1;
    };
    auto request_namers = [&]() {
#pragma unroll
        for (int p = 0; p < kPairs; ++p) {
            const bool ok = k_next[p] >= 0;
            counts[p] = __builtin_amdgcn_ballot_w64(ok);
            g_next[p] = ok ? grad_dist[k_next[p]] : 0.f;
            load_row<C>(coord, ok ? fast_div(k_next[p], div_k) : max(vertex[p], 0), x_next[p]);
        }
    };
    request_indices(0);
    request_neighbours(0);
    request_indices(kChunk);
    for (int n0 = 0; n0 < K; n0 += kChunk) {
        hand_over(true);
        const bool more = n0 + kChunk < K;
        if (more) {
            request_neighbours(n0 + kChunk);
            request_indices(n0 + 2 * kChunk);
        } else {
            request_slots(0);
        }
        if (C == kLanes || cc < C) {
#pragma unroll
            for (int u = 0; u < kChunk; ++u)  // a slot without a neighbour subtracts 0
                sum = __builtin_fmaf(-my_grad[u], my_diff[u * kLanes], sum);
        }
    }
    request_namers();
    request_slots(kChunk);
    for (int e0 = 0; e0 < longest; e0 += kChunk) {
        hand_over(false);
        request_namers();
        request_slots(e0 + 2 * kChunk);
        if (C == kLanes || cc < C) {
#pragma unroll
            for (int u = 0; u < kChunk; ++u) {  // an entry beyond the list adds 0
                const float add = my_grad[u] * my_diff[u * kLanes];
                sum = sum + add;
            }
        }
    }
    const int r = r0 + cv;
    if (cc < C && r < n_vert) {
        const int i = order ? order[r] : r;
        if ((uint32_t)i < (uint32_t)n_vert) out[(size_t)i * C + cc] = sum;
    }
}

// More than 8 coordinates: one thread per coordinate. The loads of eight slots (list entries) are issued together; the
// additions stay in their order.
__global__ __launch_bounds__(256) void knn_grad_wide_kernel(const float *__restrict__ grad_dist,
                                                            const int *__restrict__ idx,
                                                            const float *__restrict__ coord,
                                                            const int *__restrict__ inv_off,
                                                            const int *__restrict__ inv_slots, float *__restrict__ out,
                                                            int n_vert, int K, int C,
                                                            const FastDiv div_k, const int *__restrict__ order) {
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const int r = (int)(t / C);
    if (r >= n_vert) return;
    const int c = (int)(t - (long long)r * C);
    const int i = order ? order[r] : r;
    if ((uint32_t)i >= (uint32_t)n_vert) return;
    const float xi = coord[(size_t)i * C + c];
    constexpr int U = 8;
    float sum = 0.f;
    for (int n0 = 0; n0 < K; n0 += U) {
        int k[U];
        float g[U], x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const size_t at = (size_t)i * K + min(n0 + u, K - 1);
            k[u] = idx[at];
            g[u] = grad_dist[at];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool ok = n0 + u < K && (uint32_t)k[u] < (uint32_t)n_vert;
            k[u] = ok ? k[u] : -1;
            x[u] = coord[(size_t)(ok ? k[u] : i) * C + c];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (k[u] < 0) continue;
            const float diff = x[u] - xi;
            sum = __builtin_fmaf(-g[u], 2.f * diff, sum);
        }
    }
    const int begin = inv_off[i], count = inv_off[i + 1] - begin;
    const int *const list = inv_slots + begin;
    for (int e0 = 0; e0 < count; e0 += U) {
        int slot[U];
        float g[U], x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) slot[u] = list[min(e0 + u, count - 1)];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            g[u] = grad_dist[slot[u]];
            x[u] = coord[(size_t)fast_div(slot[u], div_k) * C + c];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (e0 + u >= count) break;
            const float diff = xi - x[u];
            const float add = g[u] * (2.f * diff);
            sum = sum + add;
        }
    }
    out[(size_t)i * C + c] = sum;
}

}  // namespace

int launch_knn_grad(const float *grad_dist, const int *idx, const float *coord, const int *inv_off, const int *inv_slots,
                    const int *order, float *out, int n_vert, int K, int C, hipStream_t s) {
    const FastDiv div_k = make_fast_div(K);
#define HGC_KNN_GRAD(N)                                                                                              \
    case N:                                                                                                          \
        knn_grad_kernel<N><<<ceil_div(n_vert, kGradWaves * kWave / (N <= 4 ? 4 : 8)), kGradWaves * kWave, 0, s>>>(   \
            grad_dist, idx, coord, inv_off, inv_slots, out, n_vert, K, div_k, order);                                \
        break
    switch (C) {
        HGC_KNN_GRAD(1);
        HGC_KNN_GRAD(2);
        HGC_KNN_GRAD(3);
        HGC_KNN_GRAD(4);
        HGC_KNN_GRAD(5);
        HGC_KNN_GRAD(6);
        HGC_KNN_GRAD(7);
        HGC_KNN_GRAD(8);
        default: {
            const long long threads = (long long)n_vert * C;
            knn_grad_wide_kernel<<<ceil_div(threads, 256), 256, 0, s>>>(grad_dist, idx, coord, inv_off, inv_slots, out, n_vert,
                                                                       K, C, div_k, order);
        }
    }
#undef HGC_KNN_GRAD
    return check_launch("knn_grad_kernel");
}

}  // namespace hgc

using namespace hgc;

extern "C" {

int hgc_select_knn_grad_ordered(const float *d_grad_dist, const int *d_indices, const float *d_dist,
                                const float *d_coord, const int *d_inv_offsets, const int *d_inv_slots,
                                const int *d_vertex_order, float *d_grad_coord, int n_vert, int n_neigh, int n_coords,
                                hgc_stream_t stream) {
    (void)d_dist;  // carried by the reference op, not used by its kernels
    HGC_REQUIRE(n_vert >= 0 && n_neigh >= 1 && n_coords >= 1, "bad sizes");
    HGC_REQUIRE((long long)n_vert * std::max(n_neigh, n_coords) < (1ll << 31), "tensor too large for int32 indexing");
    if (n_vert == 0) return HGC_OK;
    HGC_REQUIRE(d_grad_dist && d_indices && d_coord && d_inv_offsets && d_inv_slots && d_grad_coord, "null pointer");
    return launch_knn_grad(d_grad_dist, d_indices, d_coord, d_inv_offsets, d_inv_slots, d_vertex_order, d_grad_coord, n_vert,
                           n_neigh, n_coords, as_stream(stream));
}

int hgc_select_knn_grad(const float *d_grad_dist, const int *d_indices, const float *d_dist, const float *d_coord,
                        const int *d_inv_offsets, const int *d_inv_slots, float *d_grad_coord, int n_vert, int n_neigh,
                        int n_coords, hgc_stream_t stream) {
    return hgc_select_knn_grad_ordered(d_grad_dist, d_indices, d_dist, d_coord, d_inv_offsets, d_inv_slots, nullptr,
                                       d_grad_coord, n_vert, n_neigh, n_coords, stream);
}

}  // extern "C"
