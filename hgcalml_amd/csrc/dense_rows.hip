// Gradients of the dense layers of the GravNet block, rows in and rows out, with what stands around them in the same pass:
//   output's gradient g where y > 0 times W: to the accumulation's rows, to p (minus both halves) and to x; the masked g kept
//                     (y = relu([mean - p | max - p | x] W^T + b))
//   input's gradient  (g1 + g2 where the features are > 0) Wf + g_coordinates Ws + g_x; the masked sum kept
// The three layers themselves are library products: the last bits of coordinates decide between neighbours at nearly equal
// distances, those of features between neighbours with nearly equal maxima, and those in front of both activations which
// gradients pass. With the last layer as a pass of its own about one activation of 20 million fell on the other side of 0, and single
// rows of the gradients changed by up to 0.6 of their root mean square (10 of 34 steps by more than 0.01; none of them with the
// library's product: 9e-6 at the most). It took 113 and 117 us in the steps below, join, product and activation 154 and 173.
//
// A contraction over at most a few hundred columns, for very many rows. Its bound is the float32 matrix instruction
// (150,000 rows, 128 -> 192: 7.4 GFLOP, 47 us at its rate) or, for narrow layers, reading and writing the rows once.
// The weights of a workgroup's columns lie in LDS for its whole life, in the order in which the instruction takes them (a
// step of 16 columns of the input times 16 of the output is 64 lanes x 16 bytes, without bank conflicts), so nothing but
// the first barrier keeps its waves together: each takes 16 rows at a time, streams them from memory with one batch of
// steps requested ahead and has all output columns of the workgroup in registers. 16 rows a wave: many short tasks fill the
// four SIMDs of 256 CUs evenly (9375 tasks for 150,000 rows).
// Rows go in as the instruction's second operand, so that a lane holds four consecutive columns of one row in the end and
// stores 16 bytes. At the end of a width that is no multiple of four a lane moves back onto the row's last four columns
// (the ones it has twice count once), and behind the last row stands the last row again: no load or store is left out, so
// none stands in a branch, which would make waiting for a load mean waiting for everything after it.
// Measured next to the library products with mask, sums and the join's gradient as passes of their own, us, a gigabyte written
// between calls (inputs come from memory): 150,000 rows, 64 inputs, 64 features, 128 outputs: output's gradient 197 -> 134,
// input's 145 -> 80; 240,011 rows, 48, 32, 96: 248 -> 151, 173 -> 74; 20,000 rows, 64, 64, 128: 52 -> 30, 45 -> 17. In a training
// step of the block the two take 122 and 52 us, and 135 and 48. The step 1973 -> 1759 and 1999 -> 1735 (35 and 45 of it elsewhere),
// 2477 points 856 -> 730 (the host's time; runs of one side differ by 8 %). In the step of 150,000 points the matrix cores are busy
// for 37 and 14 % of the two passes, and 3.9 and 4.9 TB/s move past the L2 (470 and 254 MB, 384 and 233 needed). Error against 64 bits
// (2-norm, 150,000 rows), here and library: gradient of the accumulated rows 8.7e-8 and 1.5e-7, of the joined x the same, input's
// 5.6e-8 and 6.4e-8. Tried and taken back: 8 waves instead of 16, one chain of products over all columns (twice the error), higher
// priority while multiplying, whole ranges of rows per workgroup or XCD.
#include <algorithm>

#include "hgc_common.hpp"

namespace hgc {
namespace {

constexpr int kTile = 16, kStepCols = 16;
constexpr int kGroups = 256;               // workgroups at the most, one per CU
constexpr int kLdsBytes = 160 * 1024;

typedef float vec4 __attribute__((ext_vector_type(4)));

enum class Form { OutputGrad, InputGrad };

struct DenseRows {
    const float *a0, *a1, *a2, *a3, *add;  // rows in
    const float *w0, *w1;
    float *o0, *o1, *o2, *masked;          // rows out; masked: the operand as it was multiplied
    long long n;
    int F, I, O, C;
    int steps;                             // of 16 input columns
    int tiles;                             // of 16 output columns, all of them
    int relu, two;
};

__device__ __forceinline__ vec4 load4(const float *p) {
    vec4 v;
    __builtin_memcpy(&v, p, sizeof(v));
    return v;
}

// Past the caches: what is written here is read by other kernels, after more than the L2 holds. (Output's gradient, inputs in the
// caches, 150,000 rows 112 -> 87 us; 240,011 rows, 96 of 112 columns: 116 -> 83)
__device__ __forceinline__ void store4(float *p, const vec4 &v) {
    typedef vec4 vec4_any __attribute__((aligned(4)));
    __builtin_nontemporal_store(v, reinterpret_cast<vec4_any *>(p));
}

// the derivative of max(y, 0): NaN stays, as in torch
__device__ __forceinline__ float where_positive(float g, float y) { return y <= 0.f ? 0.f : g; }

// Four columns in sequence of a row of `width` >= 4, wanted from col on: the last ones move back onto the row's end.
// Columns in front of `col` are then held twice.
__device__ __forceinline__ int first_of_four(int col, int width) { return min(col, width - 4); }

// columns of a row that is multiplied
template <Form FORM>
__device__ __forceinline__ int width_in(const DenseRows &p) { return FORM == Form::OutputGrad ? p.O : p.F; }

// first weight of output column c of tile `tile` and the distance of its weights for consecutive input columns
template <Form FORM>
__device__ __forceinline__ const float *weights_of(const DenseRows &p, int tile, int c, size_t &pitch) {
    const int tiles_f = (p.F + kTile - 1) / kTile;
    auto column = [&](int tile, int width) { return first_of_four(tile * kTile + (c & ~3), width) + (c & 3); };
    if constexpr (FORM == Form::OutputGrad) {  // tiles of both halves in turn, then those of x
        pitch = 2 * p.F + p.I;
        return tile < 2 * tiles_f ? p.w0 + (tile & 1) * p.F + column(tile >> 1, p.F) : p.w0 + 2 * p.F + column(tile - 2 * tiles_f, p.I);
    } else {
        pitch = p.I;
        return p.w0 + column(tile, p.I);
    }
}

constexpr int sources(Form form) { return form == Form::InputGrad ? 3 : 2; }

template <int NSRC>
struct Raw {
    vec4 v[NSRC];
};

// Steps requested while as many are multiplied (three sources and many tiles: registers for one)
constexpr int steps_ahead(Form form, int tiles) { return tiles >= 6 && sources(form) == 3 ? 1 : 2; }
// 16 waves of 128 registers, or 12 of 168 for many tiles
constexpr int most_waves(int tiles) { return tiles <= 8 ? 16 : 12; }

// COORDS: the gradient of the coordinates takes part (at most four of them: one more step of the instruction).
template <Form FORM, int NT, bool COORDS>
__global__ __launch_bounds__(most_waves(NT) *kWave) void dense_rows_kernel(const DenseRows p) {
    constexpr int NSRC = sources(FORM), U = steps_ahead(FORM, NT);
    const int width = width_in<FORM>(p);
    extern __shared__ __align__(16) float s_weights[];
    vec4 *const s_w = reinterpret_cast<vec4 *>(s_weights);
    float *const s_coords = s_weights + (size_t)p.steps * NT * kWave * 4;  // weights of the coordinates
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = lane_id(), l = lane & 15, k = lane >> 4;
    const int waves = blockDim.x / kWave, tile0 = blockIdx.y * NT;
    const int tiles_f = (p.F + kTile - 1) / kTile;

    // lane: output column l of the tile, four input columns of group k of the step; columns held twice count once
    constexpr int kAtOnce = 4;
    const int pieces = p.steps * NT;
    for (int first = wave * kAtOnce; first < pieces; first += waves * kAtOnce) {
        vec4 w[kAtOnce];
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) {
            const int i = min(first + u, pieces - 1), step = i / NT;
            const int wanted = step * kStepCols + 4 * k, col = first_of_four(wanted, width);
            size_t pitch;
            const float *from = weights_of<FORM>(p, min(tile0 + i - step * NT, p.tiles - 1), l, pitch);
#pragma unroll
            for (int e = 0; e < 4; ++e) w[u][e] = from[(col + e) * pitch];
#pragma unroll
            for (int e = 0; e < 4; ++e) w[u][e] = col + e < wanted ? 0.f : w[u][e];
        }
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u)
            if (first + u < pieces) s_w[(size_t)(first + u) * kWave + lane] = w[u];
    }
    if constexpr (COORDS) {  // lane: output column l, coordinate k
        for (int i = threadIdx.x; i < NT * kWave; i += blockDim.x) {
            const int c = i & 15, coord = (i >> 4) & 3;
            const int col = first_of_four(min(tile0 + i / kWave, p.tiles - 1) * kTile + (c & ~3), p.I) + (c & 3);
            s_coords[i] = coord < p.C ? p.w1[(size_t)coord * p.I + col] : 0.f;
        }
    }
    __syncthreads();

    const long long tasks = (p.n + kTile - 1) / kTile, stride = (long long)waves * gridDim.x;
    long long task = (long long)wave * gridDim.x + blockIdx.x;
    if (task >= tasks) return;
    const int batches = (p.steps + U - 1) / U;

    // Rows behind the last one are the last one again, which is then written several times with the same values: loads and
    // stores stand in no branch, so that waiting for a load never means waiting for what was asked for after it.
    auto row_in = [&](long long task) { return (int)min((long long)l, p.n - 1 - task * kTile); };
    auto request = [&](Raw<NSRC> (&raw)[U], float &coord, long long task, int batch) {
        task = min(task, tasks - 1);
        const unsigned row = row_in(task);
        // (a base that is the same for all lanes and an offset of 32 bits)
        auto at = [&](const float *from, int pitch, int first) { return from + task * kTile * pitch + (row * (unsigned)pitch + first); };
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int col = first_of_four(min(batch * U + u, p.steps - 1) * kStepCols + 4 * k, width);
            raw[u].v[0] = load4(at(p.a0, width, col));
            raw[u].v[1] = load4(at(p.a1, width, col));
            if constexpr (FORM == Form::InputGrad) raw[u].v[2] = load4(at(p.a2, width, col));
        }
        if constexpr (COORDS) coord = *at(p.a3, p.C, min(k, p.C - 1));
        __builtin_amdgcn_sched_barrier(0);  // before what is multiplied meanwhile
    };

    vec4 acc[NT];
    auto clear = [&]() {
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = vec4{0.f, 0.f, 0.f, 0.f};
    };
    auto multiply = [&](const Raw<NSRC> (&raw)[U], long long task, int batch) {
        const unsigned row = row_in(task);
        const int here = min(U, p.steps - batch * U);
        vec4 a[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int first = min(batch * U + u, p.steps - 1) * kStepCols;
            const int wanted = first + 4 * k, col = first_of_four(wanted, width);
            a[u] = raw[u].v[0];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if constexpr (FORM == Form::OutputGrad) a[u][e] = where_positive(a[u][e], raw[u].v[1][e]);
                if constexpr (FORM == Form::InputGrad) {
                    a[u][e] = p.two ? a[u][e] + raw[u].v[1][e] : a[u][e];
                    a[u][e] = p.relu ? where_positive(a[u][e], raw[u].v[2][e]) : a[u][e];
                }
            }
            if (tile0 == 0) store4(p.masked + task * kTile * width + (row * (unsigned)width + col), a[u]);
            if (first + kStepCols > width) {
#pragma unroll
                for (int e = 0; e < 4; ++e) a[u][e] = col + e < wanted ? 0.f : a[u][e];
            }
        }
        // The sum over two steps first, then onto the others: less rounding than one chain over all columns.
#pragma unroll
        for (int u0 = 0; u0 < U; u0 += 2) {
            if (u0 > 0 && u0 >= here) break;
#pragma unroll
            for (int t0 = 0; t0 < NT; t0 += 4) {
                constexpr int kMost = 4;
                vec4 sum[kMost];
#pragma unroll
                for (int t = 0; t < kMost; ++t) sum[t] = vec4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int u = u0; u < u0 + 2 && u < U; ++u) {
                    if (u > u0 && u >= here) break;
                    vec4 w[kMost];
#pragma unroll
                    for (int t = 0; t < kMost && t0 + t < NT; ++t) w[t] = s_w[((batch * U + u) * NT + t0 + t) * kWave + lane];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int t = 0; t < kMost && t0 + t < NT; ++t)
                            sum[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[t][e], a[u][e], sum[t], 0, 0, 0);
                }
#pragma unroll
                for (int t = 0; t < kMost && t0 + t < NT; ++t)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[t0 + t][e] = acc[t0 + t][e] + sum[t][e];
            }
        }
    };
    // lane: columns 4 k .. 4 k + 3 of every tile of row l
    auto finish = [&](long long task, float coord) {
        const long long row = task * kTile + row_in(task);
        if constexpr (COORDS) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(s_coords[t * kWave + lane], k < p.C ? coord : 0.f, acc[t], 0, 0, 0);
        }
        auto column = [&](int tile, int width) { return first_of_four(tile * kTile + 4 * k, width); };
        if constexpr (FORM == Form::InputGrad) {
            if (p.add) {
#pragma unroll
                for (int t0 = 0; t0 < NT; t0 += 4) {
                    vec4 more[4];
#pragma unroll
                    for (int t = 0; t < 4 && t0 + t < NT; ++t)
                        more[t] = load4(p.add + row * p.I + column(min(tile0 + t0 + t, p.tiles - 1), p.I));
#pragma unroll
                    for (int t = 0; t < 4 && t0 + t < NT; ++t)
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[t0 + t][e] = acc[t0 + t][e] + more[t][e];
                }
            }
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            // (behind the last tile: that one again, weights and all)
            const int tile = min(tile0 + t, p.tiles - 1);
            if constexpr (FORM == Form::OutputGrad) {
                if (tile0 + t < 2 * tiles_f) {
                    if (t % 2 == 0) {
                        const int col = column(tile >> 1, p.F);
                        const vec4 &mean = acc[t], &max = acc[t + 1 < NT ? t + 1 : t];
                        store4(p.o0 + row * 2 * p.F + col, mean);
                        store4(p.o0 + (row * 2 + 1) * p.F + col, max);
                        vec4 v;
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = -mean[e] - max[e];
                        store4(p.o1 + row * p.F + col, v);
                    }
                } else {
                    store4(p.o2 + row * p.I + column(tile - 2 * tiles_f, p.I), acc[t]);
                }
            } else {
                store4(p.o0 + row * p.I + column(tile, p.I), acc[t]);
            }
        }
    };

    Raw<NSRC> now[U], ahead[U];
    float coord_now = 0.f, coord_ahead = 0.f;
    request(ahead, coord_ahead, task, 0);
    for (int batch = 0;;) {
#pragma unroll
        for (int u = 0; u < U; ++u) now[u] = ahead[u];
        coord_now = coord_ahead;
        const bool last = batch + 1 == batches;
        const long long next_task = last ? task + stride : task;
        const int next = last ? 0 : batch + 1;
        request(ahead, coord_ahead, next_task, next);  // (behind the last task: its last row once more)
        if (batch == 0) clear();
        multiply(now, task, batch);
        if (last) finish(task, coord_now);
        if (next_task >= tasks) break;
        task = next_task;
        batch = next;
    }
}

struct Plan {
    int tiles, chunks;  // tiles of a workgroup, workgroups along the output's columns
    size_t lds;
};

// Tiles of a workgroup: all output columns where registers and LDS hold them, otherwise equal shares.
bool make_plan(Form form, int steps, int tiles, bool coords, Plan &plan) {
    constexpr int offered[] = {1, 2, 3, 4, 5, 6, 8, 10, 12};
    const bool pairs = form == Form::OutputGrad;
    for (int chunks = 1; chunks <= tiles; ++chunks) {
        const int share = (tiles + chunks - 1) / chunks;
        for (int nt : offered) {
            if (nt < share || (pairs && nt % 2)) continue;
            const size_t lds = (size_t)steps * nt * kWave * sizeof(vec4) + (coords ? nt * kWave * sizeof(float) : 0);
            if (lds > kLdsBytes) break;
            plan.tiles = nt;
            plan.chunks = (tiles + nt - 1) / nt;
            plan.lds = lds;
            return true;
        }
    }
    return false;
}

template <Form FORM, int NT, bool COORDS>
int launch_kernel(const DenseRows &p, const Plan &plan, hipStream_t s) {
    const long long tasks = (p.n + kTile - 1) / kTile;
    const int groups = (int)std::min<long long>(tasks, std::max(1, kGroups / plan.chunks));
    const long long each = (tasks + groups - 1) / groups;
    const int waves = (int)std::min<long long>(most_waves(NT), (each + 3) / 4 * 4);
    if (plan.lds > 64 * 1024) {
        HGC_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&dense_rows_kernel<FORM, NT, COORDS>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes));
    }
    dense_rows_kernel<FORM, NT, COORDS><<<dim3(groups, plan.chunks), waves * kWave, plan.lds, s>>>(p);
    return check_launch("dense_rows_kernel");
}

template <Form FORM, bool COORDS>
int launch(DenseRows p, int tiles, hipStream_t s) {
    constexpr bool kPairs = FORM == Form::OutputGrad;
    Plan plan;
    p.tiles = tiles;
    if (!make_plan(FORM, p.steps, tiles, COORDS, plan)) return fail(HGC_ERR_INVALID_ARGUMENT, "layer too wide");
    switch (plan.tiles) {
        case 1: if constexpr (!kPairs) return launch_kernel<FORM, 1, COORDS>(p, plan, s); break;
        case 2: if constexpr (!kPairs) return launch_kernel<FORM, 2, COORDS>(p, plan, s); break;
        case 3: if constexpr (!kPairs) return launch_kernel<FORM, 3, COORDS>(p, plan, s); break;
        case 4: return launch_kernel<FORM, 4, COORDS>(p, plan, s);
        case 5: if constexpr (!kPairs) return launch_kernel<FORM, 5, COORDS>(p, plan, s); break;
        case 6: return launch_kernel<FORM, 6, COORDS>(p, plan, s);
        case 8: return launch_kernel<FORM, 8, COORDS>(p, plan, s);
        case 10: return launch_kernel<FORM, 10, COORDS>(p, plan, s);
        case 12: return launch_kernel<FORM, 12, COORDS>(p, plan, s);
    }
    return fail(HGC_ERR_INVALID_ARGUMENT, "no kernel for this number of tiles");
}

int steps_of(int width) { return ceil_div(width, kStepCols); }
int tiles_of(int width) { return ceil_div(width, kTile); }

// Rows of four columns and more, so that four in sequence exist; up to four coordinates, one step of the instruction. Wider
// layers are the library product's, whose workgroups share what they read of the weights. Up to the widest both gradients together
// are faster here, us here / library, inputs from memory: last layer 384 -> 256 20,000 rows 90 / 142, 60,000 218 / 315, 240,000
// 727 / 1138; 512 (256 of them x) -> 256 60,000 278 / 427, 150,000 627 / 1062, 240,000 959 / 1552; 512 (412 of them x) -> 255
// 60,000 397 / 557, 240,000 1502 / 2047; 512 -> 64 240,000 607 / 1036.
constexpr int kWidestIn = 512, kWidestOut = 256;

bool widths_fit(int f, int x, int o, int c) {
    return f >= 4 && x >= 4 && o >= 4 && c >= 1 && f <= kWidestIn && x <= kWidestIn && 2 * f + x <= kWidestIn && o <= kWidestOut &&
           c <= 4;
}

}  // namespace
}  // namespace hgc

using namespace hgc;

extern "C" {

int hgc_gravnet_dense_covers(int n_feat, int n_x, int n_out, int n_coords) {
    return widths_fit(n_feat, n_x, n_out, n_coords);
}

int hgc_gravnet_output_layer_grad(const float *d_grad, const float *d_out, int n_vert, int n_feat, int n_x, const float *d_w,
                                  int n_out, float *d_masked, float *d_grad_acc, float *d_grad_features, float *d_grad_x,
                                  hgc_stream_t stream) {
    HGC_REQUIRE(n_vert >= 0 && widths_fit(n_feat, n_x, n_out, 1), "bad sizes");
    if (n_vert == 0) return HGC_OK;
    HGC_REQUIRE(d_grad && d_out && d_w && d_masked && d_grad_acc && d_grad_features && d_grad_x, "null pointer");
    DenseRows p{};
    p.a0 = d_grad, p.a1 = d_out, p.w0 = d_w, p.masked = d_masked, p.o0 = d_grad_acc, p.o1 = d_grad_features, p.o2 = d_grad_x;
    p.n = n_vert, p.F = n_feat, p.I = n_x, p.O = n_out;
    p.steps = steps_of(n_out);
    return launch<Form::OutputGrad, false>(p, 2 * tiles_of(n_feat) + tiles_of(n_x), as_stream(stream));
}

int hgc_gravnet_input_layers_grad(const float *d_grad_features, const float *d_grad_features2, const float *d_features,
                                  const float *d_grad_coords, const float *d_grad_x, int n_vert, int n_x,
                                  const float *d_w_feat, int n_feat, const float *d_w_coords, int n_coords, int relu,
                                  float *d_masked, float *d_grad_in, hgc_stream_t stream) {
    HGC_REQUIRE(n_vert >= 0 && widths_fit(n_feat, n_x, 4, n_coords), "bad sizes");
    if (n_vert == 0) return HGC_OK;
    HGC_REQUIRE(d_grad_features && (d_features || !relu) && d_w_feat && (d_w_coords || !d_grad_coords) && d_masked && d_grad_in,
                "null pointer");
    DenseRows p{};
    p.a0 = d_grad_features, p.a1 = d_grad_features2 ? d_grad_features2 : d_grad_features, p.a2 = relu ? d_features : d_grad_features;
    p.a3 = d_grad_coords, p.add = d_grad_x, p.two = d_grad_features2 != nullptr;
    p.w0 = d_w_feat, p.w1 = d_w_coords, p.masked = d_masked, p.o0 = d_grad_in;
    p.n = n_vert, p.F = n_feat, p.I = n_x, p.C = n_coords, p.relu = relu;
    p.steps = steps_of(n_feat);
    return d_grad_coords ? launch<Form::InputGrad, true>(p, tiles_of(n_x), as_stream(stream))
                         : launch<Form::InputGrad, false>(p, tiles_of(n_x), as_stream(stream));
}

}  // extern "C"
