// The memory passes of the GravNet block around its search and accumulation
// (modules/GravNetLayersRagged.py:3095-3283): the neighbour table and distances without the self column, the update of
// the dynamic radius, the row [mean - p | max - p | x] that the last dense layer reads, and sums over the rows for the
// gradients of the dense layers. All of them stream; as single tensor operations they were 40 launches and, at 150k
// vertices, K = 64, F = 64, 0.6 of the 2.45 ms of a training step, most of it intermediates written and read again; the
// step took 2.19 ms with these (240k vertices, K = 40, F = 32 with the weights' sum: 2.97 -> 2.27). Reads and writes
// together run at what a large copy reaches (5.3 TB/s): at 150k vertices 42 and 49 us for the join and its gradient
// (269 MB each), 27 and 23 us for the table (155 MB) and its gradient (116 MB), 13 us for the radius (39 MB).
#include <algorithm>
#include <cmath>

#include "accumulate_rows.hpp"

namespace hgc {
namespace {

constexpr int kThreads = 256;

// ---- table and distances without column 0 -------------------------------------------------------------------------

// A thread moves four consecutive entries of the narrow table (16-byte stores); the wide rows start anywhere, their
// loads are four dwords each that neighbouring lanes complete to whole lines.
// (The block weights neighbours by exp(-10 d^2): its factor is taken here and in the gradient, where the values pass
// anyway. As products of their own 13 us each way at 150k vertices, K = 64.)
__global__ __launch_bounds__(kThreads) void drop_self_kernel(const int *__restrict__ idx, const float *__restrict__ dist,
                                                             unsigned total, unsigned narrow, float scale,
                                                             int *__restrict__ out_idx, float *__restrict__ out_dist) {
    const unsigned first = (blockIdx.x * kThreads + threadIdx.x) * 4u;
    if (first >= total) return;
    unsigned row = first / narrow, col = first - row * narrow;
    int ai[4];
    float di[4];
    const unsigned count = min(4u, total - first);
#pragma unroll
    for (unsigned u = 0; u < 4; ++u) {
        if (u < count) {
            ai[u] = idx[first + u + row + 1];  // row * (narrow + 1) + col + 1
            di[u] = scale * dist[first + u + row + 1];
        }
        if (++col == narrow) col = 0, ++row;
    }
    if (count == 4) {
        *reinterpret_cast<int4 *>(out_idx + first) = int4{ai[0], ai[1], ai[2], ai[3]};
        *reinterpret_cast<float4 *>(out_dist + first) = float4{di[0], di[1], di[2], di[3]};
    } else {
#pragma unroll
        for (unsigned u = 0; u < 3; ++u)
            if (u < count) out_idx[first + u] = ai[u], out_dist[first + u] = di[u];
    }
}

// gradient w.r.t. the wide distances: that of the narrow ones, times the factor, moved up by a column, plus that of the wide ones (if any)
__global__ __launch_bounds__(kThreads) void drop_self_grad_kernel(const float *__restrict__ g_narrow,
                                                                  const float *__restrict__ g_wide, unsigned total,
                                                                  unsigned wide, float scale, float *__restrict__ out) {
    const unsigned first = (blockIdx.x * kThreads + threadIdx.x) * 4u;
    if (first >= total) return;
    unsigned row = first / wide, col = first - row * wide;
    const unsigned count = min(4u, total - first);
    float vi[4] = {0.f, 0.f, 0.f, 0.f};
    if (g_wide && count == 4) {
        const float4 v = *reinterpret_cast<const float4 *>(g_wide + first);
        vi[0] = v.x, vi[1] = v.y, vi[2] = v.z, vi[3] = v.w;
    } else if (g_wide) {
#pragma unroll
        for (unsigned u = 0; u < 3; ++u)
            if (u < count) vi[u] = g_wide[first + u];
    }
#pragma unroll
    for (unsigned u = 0; u < 4; ++u) {
        if (u < count && col > 0) vi[u] += scale * g_narrow[first + u - row - 1];
        if (++col == wide) col = 0, ++row;
    }
    if (count == 4) {
        *reinterpret_cast<float4 *>(out + first) = float4{vi[0], vi[1], vi[2], vi[3]};
    } else {
#pragma unroll
        for (unsigned u = 0; u < 3; ++u)
            if (u < count) out[first + u] = vi[u];
    }
}

// ---- dynamic radius -----------------------------------------------------------------------------------------------

constexpr int kRadiusBlocks = 512;

struct MaxSum {
    double sum;
    float max;
};

__device__ __forceinline__ void fold(MaxSum &a, float max, double sum) {
    a.max = (max > a.max || max != max) ? max : a.max;  // NaN stays, as in torch's max
    a.sum += sum;
}

__device__ __forceinline__ MaxSum block_fold(MaxSum a) {
    __shared__ MaxSum s_wave[kThreads / kWave];
    for (int off = kWave / 2; off > 0; off >>= 1) {
        const float m = __shfl_xor(a.max, off);
        const double sum = __shfl_xor(a.sum, off);
        fold(a, m, sum);
    }
    if (lane_id() == 0) s_wave[threadIdx.x / kWave] = a;
    __syncthreads();
    a = s_wave[0];
    for (int w = 1; w < kThreads / kWave; ++w) fold(a, s_wave[w].max, s_wave[w].sum);
    return a;
}

// largest distance and sum of the distances (roots of the squares), one pair per workgroup
__global__ __launch_bounds__(kThreads) void radius_parts_kernel(const float *__restrict__ distsq, long long total,
                                                                MaxSum *__restrict__ parts) {
    MaxSum a{0.0, 0.f};  // no distance is negative
    const long long whole = total / 4;
    for (long long i = (long long)blockIdx.x * kThreads + threadIdx.x; i < whole; i += (long long)gridDim.x * kThreads) {
        const float4 v = reinterpret_cast<const float4 *>(distsq)[i];
        const float x = sqrtf(v.x), y = sqrtf(v.y), z = sqrtf(v.z), w = sqrtf(v.w);
        fold(a, x, 0.0);
        fold(a, y, 0.0);
        fold(a, z, 0.0);
        fold(a, w, (double)x + (double)y + ((double)z + (double)w));
    }
    if (blockIdx.x == 0 && threadIdx.x < total - whole * 4) {
        const float x = sqrtf(distsq[whole * 4 + threadIdx.x]);
        fold(a, x, x);
    }
    a = block_fold(a);
    if (threadIdx.x == 0) parts[blockIdx.x] = a;
}

// 0.05 (update - radius), update = max(min(1.05 largest, 2), 2 mean) + 1e-3
__global__ __launch_bounds__(kThreads) void radius_step_kernel(const MaxSum *__restrict__ parts, int n_parts,
                                                               long long total, const float *__restrict__ radius,
                                                               float *__restrict__ step) {
    MaxSum a{0.0, 0.f};
    for (int i = threadIdx.x; i < n_parts; i += kThreads) fold(a, parts[i].max, parts[i].sum);
    a = block_fold(a);
    if (threadIdx.x == 0) {
        const float reach = a.max * 1.05f;
        const float low = reach > 2.f ? 2.f : reach;  // NaN stays
        const float twice = 2.f * (float)(a.sum / (double)total);
        const float update = (low > twice ? low : twice) + 1e-3f;
        *step = 0.05f * (update - *radius);
    }
}

// ---- the last dense layer's input ---------------------------------------------------------------------------------

// VEC consecutive columns of a row per thread; a workgroup takes `rows` whole rows
template <int VEC>
struct Vec;
template <>
struct Vec<1> {
    using type = float;
};
template <>
struct Vec<4> {
    using type = float4;
};

__device__ __forceinline__ float minus(float a, float b) { return a - b; }
__device__ __forceinline__ float4 minus(float4 a, float4 b) { return {a.x - b.x, a.y - b.y, a.z - b.z, a.w - b.w}; }
__device__ __forceinline__ float minus_sum(float a, float b) { return -a - b; }
__device__ __forceinline__ float4 minus_sum(float4 a, float4 b) { return {-a.x - b.x, -a.y - b.y, -a.z - b.z, -a.w - b.w}; }

// out row: acc[0..F) - p | acc[F..2F) - p | x; widths in units of VEC columns
template <int VEC>
__global__ __launch_bounds__(kThreads) void join_rows_kernel(const float *__restrict__ acc, const float *__restrict__ p,
                                                             const float *__restrict__ x, int n, int rows, unsigned f,
                                                             unsigned w_x, float *__restrict__ out) {
    using V = typename Vec<VEC>::type;
    const unsigned width = 2 * f + w_x;
    const long long first = (long long)blockIdx.x * rows;
    const unsigned items = (unsigned)min((long long)rows, n - first) * width;
    const V *acc_v = reinterpret_cast<const V *>(acc) + first * 2 * f;
    const V *p_v = reinterpret_cast<const V *>(p) + first * f;
    const V *x_v = reinterpret_cast<const V *>(x) + first * w_x;
    V *out_v = reinterpret_cast<V *>(out) + first * width;
    for (unsigned t = threadIdx.x; t < items; t += kThreads) {
        const unsigned row = t / width, col = t - row * width;
        V v;
        if (col < 2 * f)
            v = minus(acc_v[row * 2 * f + col], p_v[row * f + (col < f ? col : col - f)]);
        else
            v = x_v[row * w_x + (col - 2 * f)];
        out_v[t] = v;
    }
}

// its gradient: to acc (2F columns), to p (-(first half) - (second half)), to x; outputs may be null
template <int VEC>
__global__ __launch_bounds__(kThreads) void join_rows_grad_kernel(const float *__restrict__ g, int n, int rows, unsigned f,
                                                                  unsigned w_x, float *__restrict__ g_acc,
                                                                  float *__restrict__ g_p, float *__restrict__ g_x) {
    using V = typename Vec<VEC>::type;
    const unsigned width = 2 * f + w_x, tasks = f + w_x;
    const long long first = (long long)blockIdx.x * rows;
    const unsigned items = (unsigned)min((long long)rows, n - first) * tasks;
    const V *g_v = reinterpret_cast<const V *>(g) + first * width;
    V *acc_v = reinterpret_cast<V *>(g_acc) + first * 2 * f;
    V *p_v = reinterpret_cast<V *>(g_p) + first * f;
    V *x_v = reinterpret_cast<V *>(g_x) + first * w_x;
    for (unsigned t = threadIdx.x; t < items; t += kThreads) {
        const unsigned row = t / tasks, col = t - row * tasks;
        if (col < f) {
            const V a = g_v[row * width + col], b = g_v[row * width + f + col];
            if (g_acc) acc_v[row * 2 * f + col] = a, acc_v[row * 2 * f + f + col] = b;
            if (g_p) p_v[row * f + col] = minus_sum(a, b);
        } else if (g_x) {
            x_v[row * w_x + (col - f)] = g_v[row * width + f + col];
        }
    }
}

// ---- mean over the weights' sum instead of the number of slots ------------------------------------------------------
//
// AccumulateKnnSumw (modules/GravNetLayersRagged.py:35-62) sends a column of ones through the accumulation and divides by
// what arrives there: the sum of the weights over the slots, divided by K. The sum needs the weights only, so here the
// features keep their own width (33 columns instead of 32 cost the accumulation 75 us forward and 155 us backward of 240,000
// vertices with K = 40) and three streaming passes do the rest. Same bits forward; backward the sum's share
// of a weight's gradient is added after the dot product instead of inside it.

constexpr int kGroup = acc::kRowLanes;  // lanes per vertex

template <int U>
__device__ __forceinline__ void add_slots(float mine, float &sum) {
    if constexpr (U < kGroup) {
        sum = sum + acc::group_bcast<U>(mine);
        add_slots<U + 1>(mine, sum);
    }
}

// norm[v] = (sum of the weights, slot after slot) / K; the mean columns of `out` [n, 2F] divided by it (0 where it is 0),
// and again to `kept` [n, F] (may be null): what the gradient reads, so that `out` may be written to by then
__global__ __launch_bounds__(kThreads) void sumw_normalise_kernel(const float *__restrict__ weights,
                                                                  const int *__restrict__ idx, int n, int K, int F, float kf,
                                                                  float *__restrict__ out, float *__restrict__ kept,
                                                                  float *__restrict__ norm) {
    const int v = blockIdx.x * (kThreads / kGroup) + threadIdx.x / kGroup, l = threadIdx.x % kGroup;
    const bool live = v < n;
    float sum = 0.f;
    for (int c0 = 0; c0 < K; c0 += kGroup) {
        const size_t at = (size_t)v * K + c0 + l;
        const bool in_row = live && c0 + l < K;
        const bool has = in_row && (uint32_t)idx[in_row ? at : 0] < (uint32_t)n;
        add_slots<0>(has ? weights[at] : 0.f, sum);  // a sum from +0 on: adding 0 changes nothing
    }
    if (!live) return;
    const float d = sum / kf;
    if (l == 0) norm[v] = d;
    float *row = out + (size_t)v * 2 * F;
    for (int c = l; c < F; c += kGroup) {
        const float mean = d == 0.f ? 0.f : row[c] / d;
        row[c] = mean;
        if (kept) kept[(size_t)v * F + c] = mean;
    }
}

// From the gradient g [n, 2F] of the normalised rows: that of the accumulation's rows, and 1/K of that of norm (means:
// rows of `pitch` floats)
__global__ __launch_bounds__(kThreads) void sumw_grad_kernel(const float *__restrict__ g, const float *__restrict__ means,
                                                             size_t pitch, const float *__restrict__ norm, int n, int F, float kf,
                                                             float *__restrict__ g_acc, float *__restrict__ g_norm) {
    const int v = blockIdx.x * (kThreads / kGroup) + threadIdx.x / kGroup, l = threadIdx.x % kGroup;
    if (v >= n) return;
    const float d = norm[v];
    const size_t row = (size_t)v * 2 * F;
    float part = 0.f;
    for (int c = l; c < F; c += kGroup) {
        const float gm = g[row + c], gx = g[row + F + c], mean = means[v * pitch + c];
        if (d != 0.f) part = part - gm * (mean / d);
        g_acc[row + c] = d == 0.f ? 0.f : gm / d;
        g_acc[row + F + c] = gx;
    }
    part += acc::dpp_from<0x128>(part);  // over the 16 lanes: ror 8, 4, 2, 1
    part += acc::dpp_from<0x124>(part);
    part += acc::dpp_from<0x122>(part);
    part += acc::dpp_from<0x121>(part);
    if (l == 0) g_norm[v] = part / kf;
}

// the weights' sum in the gradient of the distances, w = exp(-d): g_dist -= g_norm * w where there is a neighbour
__global__ __launch_bounds__(kThreads) void sumw_distance_grad_kernel(const float *__restrict__ g_norm,
                                                                      const float *__restrict__ weights,
                                                                      const int *__restrict__ idx, unsigned total,
                                                                      unsigned K, unsigned n, float *__restrict__ g_dist) {
    const unsigned first = (blockIdx.x * kThreads + threadIdx.x) * 4u;
    if (first >= total) return;
    unsigned row = first / K, col = first - row * K;
    const unsigned count = min(4u, total - first);
    float w[4], g[4];
    int j[4];
    if (count == 4) {
        const float4 a = *reinterpret_cast<const float4 *>(weights + first), b = *reinterpret_cast<float4 *>(g_dist + first);
        const int4 c = *reinterpret_cast<const int4 *>(idx + first);
        w[0] = a.x, w[1] = a.y, w[2] = a.z, w[3] = a.w;
        g[0] = b.x, g[1] = b.y, g[2] = b.z, g[3] = b.w;
        j[0] = c.x, j[1] = c.y, j[2] = c.z, j[3] = c.w;
    } else {
#pragma unroll
        for (unsigned u = 0; u < 4; ++u) {
            const unsigned at = min(first + u, total - 1);
            w[u] = weights[at], g[u] = g_dist[at], j[u] = idx[at];
        }
    }
#pragma unroll
    for (unsigned u = 0; u < 4; ++u) {
        if (u < count && (unsigned)j[u] < n) g[u] = g[u] - g_norm[row] * w[u];
        if (++col == K) col = 0, ++row;
    }
    if (count == 4) {
        *reinterpret_cast<float4 *>(g_dist + first) = float4{g[0], g[1], g[2], g[3]};
    } else {
#pragma unroll
        for (unsigned u = 0; u < 3; ++u)
            if (u < count) g_dist[first + u] = g[u];
    }
}

// ---- sums over the rows -------------------------------------------------------------------------------------------

// Columns are cut into tiles of `tile` vectors (grid.y), rows into grid.x slabs; a thread adds its columns of every
// (256 / tile)-th row of the slab, four loads under way at a time, the groups of a workgroup meet in LDS. With one slab the
// results are final, otherwise one row per slab is left and added by a second launch of the same kernel.
template <int VEC>
__global__ __launch_bounds__(kThreads) void column_sums_kernel(const float *__restrict__ x, int n_rows, int cols_v,
                                                               int tile_width, int slab, float *__restrict__ out) {
    using V = typename Vec<VEC>::type;
    __shared__ float s_part[kThreads * VEC];
    const int tile = blockIdx.y * tile_width;
    const int width = min(tile_width, cols_v - tile);
    const int groups = kThreads / width;
    const int group = threadIdx.x / width, col = threadIdx.x - group * width;
    // rows and what lies a step beyond a slab's end fit into 32 bits without a sign: up to 2^31 - 1 rows
    const unsigned begin = blockIdx.x * (unsigned)slab, end = min((unsigned)n_rows, begin + (unsigned)slab);
    const V *src = reinterpret_cast<const V *>(x) + tile + col;
    float sum[VEC] = {};
    auto add = [&](const V &v) {
        const float *f = reinterpret_cast<const float *>(&v);
#pragma unroll
        for (int e = 0; e < VEC; ++e) sum[e] += f[e];
    };
    if (group < groups) {
        unsigned r = begin + group;
        for (; r + 3 * groups < end; r += 4 * groups) {
            const V a = src[(size_t)r * cols_v], b = src[(size_t)(r + groups) * cols_v];
            const V c = src[(size_t)(r + 2 * groups) * cols_v], d = src[(size_t)(r + 3 * groups) * cols_v];
            add(a), add(b), add(c), add(d);
        }
        for (; r < end; r += groups) add(src[(size_t)r * cols_v]);
    }
#pragma unroll
    for (int e = 0; e < VEC; ++e) s_part[e * kThreads + threadIdx.x] = sum[e];
    __syncthreads();
    if (threadIdx.x < width) {
        float *o = out + ((size_t)blockIdx.x * cols_v + tile + col) * VEC;
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            float s = s_part[e * kThreads + threadIdx.x];
            for (int g = 1; g < groups; ++g) s += s_part[e * kThreads + g * width + threadIdx.x];
            o[e] = s;
        }
    }
}

struct SumsPlan {
    int vec, cols_v, tile, slab, slabs;
};

// First pass: tiles of 32 vectors (128 or 512 bytes of a row), 16 rows or more per thread, up to about 512 workgroups.
SumsPlan sums_plan(int n_rows, int cols, int vec) {
    SumsPlan p;
    p.vec = vec;
    p.cols_v = cols / vec;
    p.tile = std::min(32, p.cols_v);
    const int most = std::max(1, 512 / ceil_div(p.cols_v, p.tile));
    p.slab = std::max(16 * (kThreads / p.tile), ceil_div(n_rows, most));
    p.slabs = ceil_div(n_rows, p.slab);
    return p;
}

int launch_column_sums(const float *x, int n_rows, const SumsPlan &p, float *out, hipStream_t s) {
    const dim3 grid(p.slabs, ceil_div(p.cols_v, p.tile));
    if (p.vec == 4)
        column_sums_kernel<4><<<grid, kThreads, 0, s>>>(x, n_rows, p.cols_v, p.tile, p.slab, out);
    else
        column_sums_kernel<1><<<grid, kThreads, 0, s>>>(x, n_rows, p.cols_v, p.tile, p.slab, out);
    return check_launch("column_sums");
}

int rows_per_block(unsigned items_per_row) { return std::max(1, (int)(4 * kThreads / std::max(1u, items_per_row))); }

bool aligned16(std::initializer_list<const void *> pointers) {
    for (const void *p : pointers)
        if (reinterpret_cast<uintptr_t>(p) & 15u) return false;
    return true;
}

}  // namespace
}  // namespace hgc

using namespace hgc;

extern "C" {

int hgc_gravnet_drop_self_scaled(const int *d_idxs, const float *d_dist, int n_vert, int n_neigh, float scale, int *d_out_idxs,
                                 float *d_out_dist, hgc_stream_t stream) {
    HGC_REQUIRE(n_vert >= 0 && n_neigh >= 2, "n_vert >= 0, n_neigh >= 2");
    HGC_REQUIRE((long long)n_vert * n_neigh < (1ll << 31), "n_vert * n_neigh must stay below 2^31");
    if (n_vert == 0) return HGC_OK;
    HGC_REQUIRE(d_idxs && d_dist && d_out_idxs && d_out_dist, "null pointer");
    HGC_REQUIRE(aligned16({d_out_idxs, d_out_dist}), "outputs must lie on 16-byte boundaries");
    const unsigned total = (unsigned)n_vert * (unsigned)(n_neigh - 1);
    drop_self_kernel<<<ceil_div(total, 4 * kThreads), kThreads, 0, as_stream(stream)>>>(
        d_idxs, d_dist, total, (unsigned)(n_neigh - 1), scale, d_out_idxs, d_out_dist);
    return check_launch("gravnet_drop_self");
}

int hgc_gravnet_drop_self(const int *d_idxs, const float *d_dist, int n_vert, int n_neigh, int *d_out_idxs,
                          float *d_out_dist, hgc_stream_t stream) {
    return hgc_gravnet_drop_self_scaled(d_idxs, d_dist, n_vert, n_neigh, 1.f, d_out_idxs, d_out_dist, stream);
}

int hgc_gravnet_drop_self_grad_scaled(const float *d_grad_narrow, const float *d_grad_wide, int n_vert, int n_neigh, float scale,
                                      float *d_out_grad, hgc_stream_t stream) {
    HGC_REQUIRE(n_vert >= 0 && n_neigh >= 2, "n_vert >= 0, n_neigh >= 2");
    HGC_REQUIRE((long long)n_vert * n_neigh < (1ll << 31), "n_vert * n_neigh must stay below 2^31");
    if (n_vert == 0) return HGC_OK;
    HGC_REQUIRE(d_grad_narrow && d_out_grad, "null pointer");
    HGC_REQUIRE(aligned16({d_grad_wide, d_out_grad}), "wide gradients must lie on 16-byte boundaries");
    const unsigned total = (unsigned)n_vert * (unsigned)n_neigh;
    drop_self_grad_kernel<<<ceil_div(total, 4 * kThreads), kThreads, 0, as_stream(stream)>>>(
        d_grad_narrow, d_grad_wide, total, (unsigned)n_neigh, scale, d_out_grad);
    return check_launch("gravnet_drop_self_grad");
}

int hgc_gravnet_drop_self_grad(const float *d_grad_narrow, const float *d_grad_wide, int n_vert, int n_neigh,
                               float *d_out_grad, hgc_stream_t stream) {
    return hgc_gravnet_drop_self_grad_scaled(d_grad_narrow, d_grad_wide, n_vert, n_neigh, 1.f, d_out_grad, stream);
}

size_t hgc_gravnet_radius_step_workspace_bytes(void) { return align_up(kRadiusBlocks * sizeof(MaxSum)); }

int hgc_gravnet_radius_step(const float *d_distsq, long long total, const float *d_radius, float *d_step, void *workspace,
                            size_t workspace_bytes, hgc_stream_t stream) {
    HGC_REQUIRE(total >= 1, "the largest of no distances is not defined");
    HGC_REQUIRE(d_distsq && d_radius && d_step, "null pointer");
    HGC_REQUIRE(aligned16({d_distsq}), "distances must lie on a 16-byte boundary");
    if (!workspace || !aligned256(workspace) || workspace_bytes < hgc_gravnet_radius_step_workspace_bytes())
        return fail(HGC_ERR_WORKSPACE, "radius step workspace missing, misaligned or too small");
    MaxSum *parts = static_cast<MaxSum *>(workspace);
    const int blocks = (int)std::max(1ll, std::min<long long>(kRadiusBlocks, total / (16 * kThreads)));
    radius_parts_kernel<<<blocks, kThreads, 0, as_stream(stream)>>>(d_distsq, total, parts);
    radius_step_kernel<<<1, kThreads, 0, as_stream(stream)>>>(parts, blocks, total, d_radius, d_step);
    return check_launch("gravnet_radius_step");
}

int hgc_gravnet_join(const float *d_acc, const float *d_features, const float *d_x, int n_vert, int n_feat, int n_x,
                     float *d_out, hgc_stream_t stream) {
    HGC_REQUIRE(n_vert >= 0 && n_feat >= 1 && n_x >= 1 && n_feat <= 1 << 30 && n_x <= 1 << 30, "bad sizes");
    if (n_vert == 0) return HGC_OK;
    HGC_REQUIRE(d_acc && d_features && d_x && d_out, "null pointer");
    const bool wide = n_feat % 4 == 0 && n_x % 4 == 0 && aligned16({d_acc, d_features, d_x, d_out});
    const int vec = wide ? 4 : 1;
    const unsigned f = n_feat / vec, w = n_x / vec;
    const int rows = rows_per_block(2 * f + w);
    const int grid = ceil_div(n_vert, rows);
    if (wide)
        join_rows_kernel<4><<<grid, kThreads, 0, as_stream(stream)>>>(d_acc, d_features, d_x, n_vert, rows, f, w, d_out);
    else
        join_rows_kernel<1><<<grid, kThreads, 0, as_stream(stream)>>>(d_acc, d_features, d_x, n_vert, rows, f, w, d_out);
    return check_launch("gravnet_join");
}

int hgc_gravnet_join_grad(const float *d_grad, int n_vert, int n_feat, int n_x, float *d_grad_acc, float *d_grad_features,
                          float *d_grad_x, hgc_stream_t stream) {
    HGC_REQUIRE(n_vert >= 0 && n_feat >= 1 && n_x >= 1 && n_feat <= 1 << 30 && n_x <= 1 << 30, "bad sizes");
    if (n_vert == 0) return HGC_OK;
    HGC_REQUIRE(d_grad, "null pointer");
    const bool wide = n_feat % 4 == 0 && n_x % 4 == 0 && aligned16({d_grad, d_grad_acc, d_grad_features, d_grad_x});
    const int vec = wide ? 4 : 1;
    const unsigned f = n_feat / vec, w = n_x / vec;
    const int rows = rows_per_block(f + w);
    const int grid = ceil_div(n_vert, rows);
    if (wide)
        join_rows_grad_kernel<4><<<grid, kThreads, 0, as_stream(stream)>>>(d_grad, n_vert, rows, f, w, d_grad_acc,
                                                                          d_grad_features, d_grad_x);
    else
        join_rows_grad_kernel<1><<<grid, kThreads, 0, as_stream(stream)>>>(d_grad, n_vert, rows, f, w, d_grad_acc,
                                                                          d_grad_features, d_grad_x);
    return check_launch("gravnet_join_grad");
}

int hgc_sumw_normalise_keep(const float *d_weights, const int *d_idxs, int n_vert, int n_neigh, int n_feat,
                            float *d_out_feat, float *d_kept_mean, float *d_norm, hgc_stream_t stream) {
    HGC_REQUIRE(n_vert >= 0 && n_neigh >= 1 && n_feat >= 1, "bad sizes");
    if (n_vert == 0) return HGC_OK;
    HGC_REQUIRE(d_weights && d_idxs && d_out_feat && d_norm, "null pointer");
    sumw_normalise_kernel<<<ceil_div(n_vert, kThreads / kGroup), kThreads, 0, as_stream(stream)>>>(
        d_weights, d_idxs, n_vert, n_neigh, n_feat, (float)n_neigh, d_out_feat, d_kept_mean, d_norm);
    return check_launch("sumw_normalise");
}

int hgc_sumw_normalise(const float *d_weights, const int *d_idxs, int n_vert, int n_neigh, int n_feat, float *d_out_feat,
                       float *d_norm, hgc_stream_t stream) {
    return hgc_sumw_normalise_keep(d_weights, d_idxs, n_vert, n_neigh, n_feat, d_out_feat, nullptr, d_norm, stream);
}

static int sumw_grad(const float *d_grad, const float *d_means, size_t pitch, const float *d_norm, int n_vert, int n_neigh,
                     int n_feat, float *d_grad_accumulated, float *d_grad_norm, hgc_stream_t stream) {
    if (n_vert == 0) return HGC_OK;
    HGC_REQUIRE(d_grad && d_means && d_norm && d_grad_accumulated && d_grad_norm, "null pointer");
    sumw_grad_kernel<<<ceil_div(n_vert, kThreads / kGroup), kThreads, 0, as_stream(stream)>>>(
        d_grad, d_means, pitch, d_norm, n_vert, n_feat, (float)n_neigh, d_grad_accumulated, d_grad_norm);
    return check_launch("sumw_grad");
}

int hgc_sumw_grad(const float *d_grad, const float *d_out_feat, const float *d_norm, int n_vert, int n_neigh, int n_feat,
                  float *d_grad_accumulated, float *d_grad_norm, hgc_stream_t stream) {
    HGC_REQUIRE(n_vert >= 0 && n_neigh >= 1 && n_feat >= 1, "bad sizes");
    return sumw_grad(d_grad, d_out_feat, 2ull * n_feat, d_norm, n_vert, n_neigh, n_feat, d_grad_accumulated, d_grad_norm, stream);
}

int hgc_sumw_grad_kept(const float *d_grad, const float *d_kept_mean, const float *d_norm, int n_vert, int n_neigh, int n_feat,
                       float *d_grad_accumulated, float *d_grad_norm, hgc_stream_t stream) {
    HGC_REQUIRE(n_vert >= 0 && n_neigh >= 1 && n_feat >= 1, "bad sizes");
    return sumw_grad(d_grad, d_kept_mean, n_feat, d_norm, n_vert, n_neigh, n_feat, d_grad_accumulated, d_grad_norm, stream);
}

int hgc_sumw_distance_grad(const float *d_grad_norm, const float *d_weights, const int *d_idxs, int n_vert, int n_neigh,
                           float *d_grad_distances, hgc_stream_t stream) {
    HGC_REQUIRE(n_vert >= 0 && n_neigh >= 1, "bad sizes");
    HGC_REQUIRE((long long)n_vert * n_neigh < (1ll << 31), "n_vert * n_neigh must stay below 2^31");
    if (n_vert == 0) return HGC_OK;
    HGC_REQUIRE(d_grad_norm && d_weights && d_idxs && d_grad_distances, "null pointer");
    HGC_REQUIRE(aligned16({d_weights, d_idxs, d_grad_distances}), "arrays must lie on 16-byte boundaries");
    const unsigned total = (unsigned)n_vert * (unsigned)n_neigh;
    sumw_distance_grad_kernel<<<ceil_div(total, 4 * kThreads), kThreads, 0, as_stream(stream)>>>(
        d_grad_norm, d_weights, d_idxs, total, (unsigned)n_neigh, (unsigned)n_vert, d_grad_distances);
    return check_launch("sumw_distance_grad");
}

size_t hgc_column_sums_workspace_bytes(int n_rows, int n_cols) {
    if (n_rows < 1 || n_cols < 1) return 0;
    // one row of partial sums per slab, whichever vector width the call takes
    int slabs = sums_plan(n_rows, n_cols, 1).slabs;
    if (n_cols % 4 == 0) slabs = std::max(slabs, sums_plan(n_rows, n_cols, 4).slabs);
    return slabs > 1 ? align_up((size_t)slabs * n_cols * sizeof(float)) : 0;
}

int hgc_column_sums(const float *d_x, int n_rows, int n_cols, float *d_sums, void *workspace, size_t workspace_bytes,
                    hgc_stream_t stream) {
    HGC_REQUIRE(n_rows >= 1 && n_cols >= 1 && n_cols <= 1 << 20, "bad sizes");
    HGC_REQUIRE(d_x && d_sums, "null pointer");
    const size_t need = hgc_column_sums_workspace_bytes(n_rows, n_cols);
    if (need && (!workspace || !aligned256(workspace) || workspace_bytes < need))
        return fail(HGC_ERR_WORKSPACE, "column sums workspace missing, misaligned or too small");
    hipStream_t s = as_stream(stream);
    const SumsPlan p = sums_plan(n_rows, n_cols, n_cols % 4 == 0 && aligned16({d_x, d_sums}) ? 4 : 1);
    if (p.slabs == 1) return launch_column_sums(d_x, n_rows, p, d_sums, s);
    float *parts = static_cast<float *>(workspace);
    if (int rc = launch_column_sums(d_x, n_rows, p, parts, s)) return rc;
    SumsPlan last = p;  // few rows: narrow tiles, so that many groups share them
    last.tile = std::min(8, p.cols_v);
    last.slab = p.slabs;
    last.slabs = 1;
    return launch_column_sums(parts, p.slabs, last, d_sums, s);
}

}  // extern "C"
