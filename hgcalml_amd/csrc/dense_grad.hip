// Weight and bias gradient of a dense layer over very many rows: W'[o, i] = sum_n g[n, o] x[n, i], b'[o] = sum_n g[n, o].
//
// A contraction over the rows with a small result, on the float32 matrix instruction (16 x 16 x 4, exact products,
// float32 sums). What bounds it is that instruction for wide layers (150,000 rows, 128 x 192: 7.4 GFLOP, 47 us at its
// rate) and reading g and x once for narrow ones (64 x 64: 77 MB, 15 us).
//
// A wave owns up to 64 x 64 of the result and a slab of rows and needs no LDS for its operands: a step takes four
// rows, lane l holds columns TM (l % 16) .. + TM of row l / 16 of the step in one load of TM floats, and column e of
// every lane is the operand of tile e. So a tile's columns are TM apart, and 16 lanes read whole lines. The waves of
// the result's blocks for one slab stand in one workgroup and share its rows in the L1; as many slabs as fit beside
// them are added through LDS, and one part of the result per workgroup is left to a second launch. Lanes at the end of
// a row that is no multiple of TM move back onto its last TM columns: they compute them twice, from the same values in
// the same order, and both write the same.
//
// Measured next to what it replaced, a batched library product over 64 slices of the rows, the slices' sum and the
// gradient's column sums, us: 150,000 rows, 128 x 192 99 -> 81, 64 x 64 68 -> 23; 240,011, 96 x 112 90 -> 59; 2477, 48 x 73
// 31 -> 10; its error against 64 bits is half as large. What keeps wide layers from the instruction's rate is the L1, in which
// the blocks of a slab meet: 150,000 rows, 128 x 192 read their rows 1.7 times from L2 and keep the matrix cores 60 % busy,
// 240,000 rows, 160 x 352 3.5 times and 57 % (393 us, the batched product 290). Tried and taken back:
// the rows through LDS, in lockstep (128 x 192 88 to 92 us, 240,000 rows, 96 x 112 72 to 77, 160 x 352 454).
#include <algorithm>

#include "hgc_common.hpp"

namespace hgc {

namespace {

constexpr int kTile = 16, kStepRows = 4, kMostTiles = 4, kMostWaves = 16;
// row slabs' parts: one workgroup per CU, half of that where the blocks of the result take more than one workgroup
constexpr int kMostParts = 256;
constexpr int kLeastRows = 16;  // of a wave, before they are made whole batches of kStepRows * steps_ahead() rows
constexpr int kWaves = 8;       // of a workgroup, or the next multiple of the four SIMDs that the blocks allow

typedef float acc_t __attribute__((ext_vector_type(4)));

template <int N>
struct Cols {
    float v[N];
};

template <int N>
__device__ __forceinline__ Cols<N> load_cols(const float *p) {
    Cols<N> out;
    if constexpr (N == 1) {
        out.v[0] = *p;
    } else {
        typedef float vec_t __attribute__((ext_vector_type(N == 3 ? 3 : N)));
        vec_t v;
        __builtin_memcpy(&v, p, N * sizeof(float));  // rows start on any multiple of four bytes
#pragma unroll
        for (int e = 0; e < N; ++e) out.v[e] = v[e];
    }
    return out;
}

struct WeightGrad {
    const float *g, *x;
    float *w_out, *b_out;  // parts of the result, `stride` floats apart; b_out may be null
    long long n, slab;     // rows, rows of a wave
    size_t stride;
    int O, I, blocks_n, blocks, blocks_here, splits;  // blocks_here: blocks of a workgroup, splits: slabs of it
};

// Steps that are under way while as many are multiplied: enough bytes for narrow tiles. With wide ones the waves of a
// slab drift apart the further they read ahead and miss each other's rows in the L1 (150,000 rows, 128 x 192, one, two
// and four steps: 76, 88 and 97 us with requests beyond the slab's end, which are gone).
constexpr int steps_ahead(int tiles) { return tiles > 8 ? 1 : tiles > 2 ? 4 : 8; }

template <int TM, int TN>
__global__ __launch_bounds__(kMostWaves *kWave) void weight_grad_kernel(const WeightGrad p) {
    constexpr int U = steps_ahead(TM * TN);
    extern __shared__ __align__(16) float s_parts[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = lane_id(), l = lane & 15, k = lane >> 4;
    const int split = wave / p.blocks_here, block = blockIdx.y * p.blocks_here + wave % p.blocks_here;
    const bool active = block < p.blocks;
    const int block_m = block / p.blocks_n, block_n = block - block_m * p.blocks_n;
    const int col_m = min(block_m * kTile * TM + l * TM, p.O - TM), col_n = min(block_n * kTile * TN + l * TN, p.I - TN);

    acc_t acc[TM][TN];
    float sums[TM];
#pragma unroll
    for (int a = 0; a < TM; ++a) {
        sums[a] = 0.f;
#pragma unroll
        for (int b = 0; b < TN; ++b) acc[a][b] = acc_t{0.f, 0.f, 0.f, 0.f};
    }
    auto multiply = [&](const Cols<TM> &a, const Cols<TN> &b) {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            sums[i] = sums[i] + a.v[i];
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.v[i], b.v[j], acc[i][j], 0, 0, 0);
        }
    };

    const long long first = ((long long)blockIdx.x * p.splits + split) * p.slab;
    const long long end = min(p.n, first + p.slab);
    if (active && first < end) {
        const float *const g = p.g + (size_t)(first + k) * p.O + col_m, *const x = p.x + (size_t)(first + k) * p.I + col_n;
        const long long batches = (end - first) / (kStepRows * U);
        Cols<TM> a[2][U];
        Cols<TN> b[2][U];
        auto request = [&](int at, long long batch) {
            const size_t row = (size_t)batch * (kStepRows * U);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                a[at][u] = load_cols<TM>(g + (row + u * kStepRows) * p.O);
                b[at][u] = load_cols<TN>(x + (row + u * kStepRows) * p.I);
            }
            __builtin_amdgcn_sched_barrier(0);  // before what is multiplied meanwhile
        };
        auto multiply_batch = [&](int at) {
#pragma unroll
            for (int u = 0; u < U; ++u) multiply(a[at][u], b[at][u]);
        };
        if (batches > 0) {
            request(0, 0);
            long long batch = 0;
            for (; batch + 2 < batches; batch += 2) {
                request(1, batch + 1);
                multiply_batch(0);
                request(0, batch + 2);
                multiply_batch(1);
            }
            // the last one or two, the first of them under way
            const bool another = batch + 1 < batches;
            if (another) request(1, batch + 1);
            multiply_batch(0);
            if (another) multiply_batch(1);
        }
        // what is left of the slab: rows behind it count as zeros
        for (long long row = first + batches * (kStepRows * U); row < end; row += kStepRows) {
            const bool there = row + k < end;
            const long long r = there ? row + k : end - 1;
            Cols<TM> left = load_cols<TM>(p.g + (size_t)r * p.O + col_m);
            Cols<TN> right = load_cols<TN>(p.x + (size_t)r * p.I + col_n);
#pragma unroll
            for (int i = 0; i < TM; ++i) left.v[i] = there ? left.v[i] : 0.f;
#pragma unroll
            for (int j = 0; j < TN; ++j) right.v[j] = there ? right.v[j] : 0.f;
            multiply(left, right);
        }
    }
#pragma unroll
    for (int a = 0; a < TM; ++a) {  // over the four rows of a step
        sums[a] += __shfl_xor(sums[a], 16);
        sums[a] += __shfl_xor(sums[a], 32);
    }

    // the workgroup's slabs: those of the first one get the others' sums through LDS, a row of tiles at a time
    if (p.splits > 1) {
        const int here = wave % p.blocks_here;
        const int others = (p.splits - 1) * p.blocks_here;
        acc_t *const tiles = reinterpret_cast<acc_t *>(s_parts);
#pragma unroll
        for (int a = 0; a < TM; ++a) {
            if (split > 0) {
                const int at = (split - 1) * p.blocks_here + here;
#pragma unroll
                for (int b = 0; b < TN; ++b) tiles[(at * TN + b) * kWave + lane] = acc[a][b];
                if (lane < kTile) s_parts[others * TN * kWave * 4 + at * kTile + lane] = sums[a];
            }
            __syncthreads();
            if (split == 0) {
                for (int s = 0; s < p.splits - 1; ++s) {
                    const int at = s * p.blocks_here + here;
#pragma unroll
                    for (int b = 0; b < TN; ++b) acc[a][b] = acc[a][b] + tiles[(at * TN + b) * kWave + lane];
                    sums[a] = sums[a] + s_parts[others * TN * kWave * 4 + at * kTile + l];
                }
            }
            __syncthreads();
        }
    }
    if (!active || split > 0) return;
    float *const w_out = p.w_out + blockIdx.x * p.stride;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = min(block_m * kTile * TM + (k * 4 + r) * TM, p.O - TM);
#pragma unroll
        for (int a = 0; a < TM; ++a)
#pragma unroll
            for (int b = 0; b < TN; ++b) w_out[(size_t)(row + a) * p.I + col_n + b] = acc[a][b][r];
    }
    if (p.b_out && block_n == 0 && k == 0) {
#pragma unroll
        for (int a = 0; a < TM; ++a) p.b_out[blockIdx.x * p.stride + col_m + a] = sums[a];
    }
}

constexpr int kSumCols = 32, kSumGroups = 8;

// the parts added up: 32 columns a workgroup, eight threads a column
__global__ __launch_bounds__(kSumCols *kSumGroups) void sum_parts_kernel(const float *__restrict__ parts, int n_parts,
                                                                        int stride, int n_weights, float *__restrict__ w,
                                                                        float *__restrict__ b) {
    __shared__ float s_sum[kSumGroups][kSumCols];
    const int lane = threadIdx.x % kSumCols, group = threadIdx.x / kSumCols;
    const int col = blockIdx.x * kSumCols + lane;
    float sum = 0.f;
    if (col < stride) {
        const float *at = parts + col;
        int part = group;
        for (; part + 7 * kSumGroups < n_parts; part += 8 * kSumGroups) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = at[(size_t)(part + u * kSumGroups) * stride];
#pragma unroll
            for (int u = 0; u < 8; ++u) sum = sum + v[u];
        }
        for (; part < n_parts; part += kSumGroups) sum = sum + at[(size_t)part * stride];
    }
    s_sum[group][lane] = sum;
    __syncthreads();
    if (group > 0 || col >= stride) return;
#pragma unroll
    for (int s = 1; s < kSumGroups; ++s) sum = sum + s_sum[s][lane];
    if (col < n_weights) w[col] = sum;
    else if (b) b[col - n_weights] = sum;
}

struct Plan {
    int tiles_m, tiles_n, blocks_n, blocks, blocks_here, groups, splits, parts;
    long long slab;
    size_t lds;
};

Plan make_plan(long long n, int O, int I) {
    Plan p;
    auto cut = [](int width, int &blocks) {  // into blocks of equal numbers of tiles, four at most
        blocks = ceil_div(width, kTile * kMostTiles);
        return ceil_div(ceil_div(width, blocks), kTile);
    };
    int blocks_m;
    p.tiles_m = cut(O, blocks_m);
    p.tiles_n = cut(I, p.blocks_n);
    p.blocks = blocks_m * p.blocks_n;
    p.groups = ceil_div(p.blocks, kMostWaves);
    p.blocks_here = ceil_div(p.blocks, p.groups);
    // 16 waves of one block each spend the time on their sums (20,000 rows, 64 x 64: 20 us with 16, 13 with 8); six
    // blocks without splits leave two SIMDs half empty (150,000 rows, 128 x 192: 88 us with 6 waves, 76 with 12)
    p.splits = ceil_div(kWaves, p.blocks_here);
    for (int more = p.splits; more * p.blocks_here <= kMostWaves; ++more)
        if (more * p.blocks_here % 4 == 0) {
            p.splits = more;
            break;
        }
    if (p.splits * p.blocks_here > kMostWaves) p.splits = 1;
    p.splits = (int)std::min<long long>(p.splits, std::max(1ll, n / kLeastRows));
    const long long most = std::max(1, kMostParts / p.groups);
    const long long rows = std::max<long long>(kLeastRows, (n + most * p.splits - 1) / (most * p.splits));
    const int batch = kStepRows * steps_ahead(p.tiles_m * p.tiles_n);
    p.slab = (rows + batch - 1) / batch * batch;
    p.parts = (int)((n + p.slab * p.splits - 1) / (p.slab * p.splits));
    p.lds = (size_t)(p.splits - 1) * p.blocks_here * (p.tiles_n * kWave * sizeof(acc_t) + kTile * sizeof(float));
    return p;
}

template <int TM>
void launch_tiles(const Plan &plan, const WeightGrad &p, hipStream_t s) {
    const dim3 grid(plan.parts, plan.groups), block(plan.blocks_here * plan.splits * kWave);
    switch (plan.tiles_n) {
        case 1: weight_grad_kernel<TM, 1><<<grid, block, plan.lds, s>>>(p); break;
        case 2: weight_grad_kernel<TM, 2><<<grid, block, plan.lds, s>>>(p); break;
        case 3: weight_grad_kernel<TM, 3><<<grid, block, plan.lds, s>>>(p); break;
        default: weight_grad_kernel<TM, 4><<<grid, block, plan.lds, s>>>(p); break;
    }
}

}  // namespace

}  // namespace hgc

using namespace hgc;

extern "C" {

size_t hgc_dense_weight_grad_workspace_bytes(long long n_rows, int n_out, int n_in) {
    if (n_rows < 1 || n_out < 1 || n_in < 1 || (long long)n_out * n_in > 1 << 20) return 0;
    const Plan plan = make_plan(n_rows, n_out, n_in);
    return plan.parts > 1 ? align_up((size_t)plan.parts * n_out * (n_in + 1) * sizeof(float)) : 0;
}

int hgc_dense_weight_grad(const float *d_grad, const float *d_x, long long n_rows, int n_out, int n_in, float *d_weight_grad,
                          float *d_bias_grad, void *workspace, size_t workspace_bytes, hgc_stream_t stream) {
    HGC_REQUIRE(n_rows >= 1 && n_rows < (1ll << 40) && n_out >= 1 && n_in >= 1 && (long long)n_out * n_in <= 1 << 20, "bad sizes");
    HGC_REQUIRE(d_grad && d_x && d_weight_grad, "null pointer");
    const size_t need = hgc_dense_weight_grad_workspace_bytes(n_rows, n_out, n_in);
    if (need && (!workspace || !aligned256(workspace) || workspace_bytes < need))
        return fail(HGC_ERR_WORKSPACE, "dense weight gradient workspace missing, misaligned or too small");
    hipStream_t s = as_stream(stream);
    const Plan plan = make_plan(n_rows, n_out, n_in);
    const int n_weights = n_out * n_in;
    float *const parts = static_cast<float *>(workspace);
    WeightGrad p;
    p.g = d_grad;
    p.x = d_x;
    p.w_out = need ? parts : d_weight_grad;
    p.b_out = need ? parts + n_weights : d_bias_grad;
    p.n = n_rows;
    p.slab = plan.slab;
    p.stride = need ? (size_t)n_weights + n_out : 0;
    p.O = n_out;
    p.I = n_in;
    p.blocks_n = plan.blocks_n;
    p.blocks = plan.blocks;
    p.blocks_here = plan.blocks_here;
    p.splits = plan.splits;
    switch (plan.tiles_m) {
        case 1: launch_tiles<1>(plan, p, s); break;
        case 2: launch_tiles<2>(plan, p, s); break;
        case 3: launch_tiles<3>(plan, p, s); break;
        default: launch_tiles<4>(plan, p, s); break;
    }
    int rc = check_launch("weight_grad_kernel");
    if (rc || !need) return rc;
    const int stride = n_weights + n_out;
    sum_parts_kernel<<<ceil_div(stride, kSumCols), kSumCols * kSumGroups, 0, s>>>(parts, plan.parts, stride, n_weights,
                                                                                 d_weight_grad, d_bias_grad);
    return check_launch("sum_parts_kernel");
}

}  // extern "C"
