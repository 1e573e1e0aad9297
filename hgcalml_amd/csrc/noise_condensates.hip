// keep_noise of the condensate wrapper (modules/assign_condensate_op.py:16-44): every noise hit becomes a
// condensation point of its own, numbered before the real ones of its event.
//
// All results are prefix counts: with P(i) = noise hits before hit i, a noise hit of event e gets the number
// P(i) - P(first hit of e), an assigned one is moved up by the event's noise hits, and the list of condensation points
// takes a noise hit at P(i) + (real points of the events before e), a real point j at j + (noise hits up to the end of
// e). Four short launches (block counts, their scan, counts at the event boundaries, one pass over the hits) with 9
// bytes per hit read twice and 13 written; bound by the launches at any size of use. As 30 tensor operations (a search,
// a scan, a radix sort and two compactions that the host waits for among them) it took 0.33 ms of the 0.55 ms of a call
// on 5000 hits; the four launches take 17 us.
#include <algorithm>

#include "hgc_common.hpp"

namespace hgc {
namespace {

constexpr int kPart = 1024;                 // hits per workgroup
constexpr int kPartThreads = 256;
constexpr int kPartWaves = kPartThreads / kWave;
constexpr int kWaveSteps = kPart / kPartThreads;  // a wave owns kWaveSteps * 64 consecutive hits

struct Counts {
    int noise, cond;  // noise hits, condensation points with the noise hits among them
};

struct HitFlags {
    bool noise, cond;
};

__device__ __forceinline__ HitFlags flags_of(const int *assignment, const int *association, const unsigned char *is_cond,
                                             int i, int end) {
    HitFlags f{false, false};
    if (i < end) {
        f.noise = assignment[i] < 0;
        f.cond = association[i] < 0 || is_cond[i] != 0;
    }
    return f;
}

// the two counts of every part of kPart hits
__global__ __launch_bounds__(kPartThreads) void part_counts_kernel(const int *__restrict__ assignment,
                                                                   const int *__restrict__ association,
                                                                   const unsigned char *__restrict__ is_cond, int n,
                                                                   Counts *__restrict__ parts) {
    __shared__ Counts s_wave[kPartWaves];
    const int wave = threadIdx.x / kWave, lane = lane_id();
    const int first = blockIdx.x * kPart + wave * (kWaveSteps * kWave);
    Counts c{0, 0};
#pragma unroll
    for (int t = 0; t < kWaveSteps; ++t) {
        const HitFlags f = flags_of(assignment, association, is_cond, first + t * kWave + lane, n);
        c.noise += __popcll(__ballot(f.noise));
        c.cond += __popcll(__ballot(f.cond));
    }
    if (lane == 0) s_wave[wave] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kPartWaves; ++w) c.noise += s_wave[w].noise, c.cond += s_wave[w].cond;
        parts[blockIdx.x] = c;
    }
}

// exclusive prefix of the parts in place, the totals behind them (one workgroup: 1000 parts are a million hits)
__global__ __launch_bounds__(1024) void part_scan_kernel(Counts *__restrict__ parts, int n_parts) {
    __shared__ Counts s_wave[16];
    const int tid = threadIdx.x, wave = tid / kWave;
    Counts run{0, 0};
    for (int base = 0; base < n_parts; base += 1024) {
        const int i = base + tid;
        const Counts mine = i < n_parts ? parts[i] : Counts{0, 0};
        const Counts upto{wave_inclusive_sum(mine.noise), wave_inclusive_sum(mine.cond)};
        if (lane_id() == kWave - 1) s_wave[wave] = upto;
        __syncthreads();
        Counts before = run;
        for (int w = 0; w < 16; ++w) {
            if (w < wave) before.noise += s_wave[w].noise, before.cond += s_wave[w].cond;
            run.noise += s_wave[w].noise, run.cond += s_wave[w].cond;
        }
        if (i < n_parts) parts[i] = Counts{before.noise + upto.noise - mine.noise, before.cond + upto.cond - mine.cond};
        __syncthreads();
    }
    if (tid == 0) parts[n_parts] = run;
}

// one wave per event boundary: noise hits before it, and the cumulative number of condensation points
__global__ __launch_bounds__(kPartThreads) void boundary_counts_kernel(
    const int *__restrict__ assignment, const int *__restrict__ association, const unsigned char *__restrict__ is_cond,
    int n, const int *__restrict__ row_splits, int num_rows, const Counts *__restrict__ parts, int n_parts,
    const int *__restrict__ n_condensates, int *__restrict__ noise_before, int *__restrict__ out_n_condensates,
    int *__restrict__ out_n_alpha) {
    const int e = blockIdx.x * kPartWaves + threadIdx.x / kWave;
    if (e > num_rows) return;
    const int at = min(max(row_splits[e], 0), n);
    Counts c = parts[at / kPart];  // at == n on a part's border: the totals
    const int first = at / kPart * kPart;
#pragma unroll  // the loads of all steps together: one after the other the chain took 10 us
    for (int t = 0; t < kPart / kWave; ++t) {
        const HitFlags f = flags_of(assignment, association, is_cond, first + t * kWave + lane_id(), at);
        c.noise += __popcll(__ballot(f.noise));
        c.cond += __popcll(__ballot(f.cond));
    }
    if (lane_id() == 0) {
        noise_before[e] = c.noise;
        out_n_condensates[e] = e == 0 ? n_condensates[0] : c.cond;
        if (e == 0) *out_n_alpha = parts[n_parts].noise + n_condensates[num_rows];
    }
}

// first e in [0, num_rows) with splits[e + 1] > at (the last one if there is none)
__device__ __forceinline__ int interval_of(const int *splits, int num_rows, int at) {
    int lo = 0, hi = num_rows - 1;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (splits[mid + 1] > at)
            hi = mid;
        else
            lo = mid + 1;
    }
    return lo;
}

__global__ __launch_bounds__(kPartThreads) void keep_noise_kernel(
    const int *__restrict__ row_splits, int n, int num_rows, const Counts *__restrict__ parts,
    const int *__restrict__ noise_before, const int *__restrict__ n_condensates, const int *__restrict__ alpha_idx,
    int *__restrict__ assignment, int *__restrict__ association, unsigned char *__restrict__ is_cond,
    int *__restrict__ out_alpha_idx) {
    __shared__ int s_noise[kPartWaves];
    const int wave = threadIdx.x / kWave, lane = lane_id();
    const int first = blockIdx.x * kPart + wave * (kWaveSteps * kWave);
    const int n_real = n_condensates[num_rows];
    uint64_t noise[kWaveSteps];
    int in_wave = 0;
#pragma unroll
    for (int t = 0; t < kWaveSteps; ++t) {
        const int i = first + t * kWave + lane;
        noise[t] = __ballot(i < n && assignment[i] < 0);
        in_wave += __popcll(noise[t]);
    }
    if (lane == 0) s_noise[wave] = in_wave;
    __syncthreads();
    int before = parts[blockIdx.x].noise;
    for (int w = 0; w < wave; ++w) before += s_noise[w];
#pragma unroll
    for (int t = 0; t < kWaveSteps; ++t) {
        const int i = first + t * kWave + lane;
        const int rank = before + __popcll(noise[t] & ((1ull << lane) - 1ull));
        before += __popcll(noise[t]);
        if (i >= n) continue;
        const int ev = interval_of(row_splits, num_rows, i);
        if ((noise[t] >> lane) & 1ull) {
            assignment[i] = rank - noise_before[ev];
            out_alpha_idx[rank + n_condensates[ev]] = i;
        } else {
            assignment[i] += noise_before[ev + 1] - (ev == 0 ? 0 : noise_before[ev]);
        }
        if (association[i] < 0) {
            association[i] = i;
            is_cond[i] = 1;
        }
        if (i < n_real) out_alpha_idx[i + noise_before[interval_of(n_condensates, num_rows, i) + 1]] = alpha_idx[i];
    }
}

}  // namespace
}  // namespace hgc

using namespace hgc;

extern "C" {

size_t hgc_keep_noise_condensates_workspace_bytes(int n_vert, int num_rows) {
    if (n_vert < 0 || num_rows < 0) return 0;
    return align_up((ceil_div(n_vert, kPart) + 1ull) * sizeof(Counts)) + align_up((num_rows + 1ull) * sizeof(int));
}

int hgc_keep_noise_condensates(const int *d_row_splits, int n_vert, int num_rows, const int *d_alpha_idx,
                               const int *d_n_condensates, int *d_assignment, int *d_association,
                               unsigned char *d_is_cond, int *d_out_alpha_idx, int *d_out_n_condensates,
                               int *d_out_n_alpha, void *workspace, size_t workspace_bytes, hgc_stream_t stream) {
    HGC_REQUIRE(n_vert >= 0 && num_rows >= 0, "bad sizes");
    HGC_REQUIRE(n_vert == 0 || num_rows >= 1, "hits without an event");
    HGC_REQUIRE(d_out_n_condensates && d_out_n_alpha, "null pointer");
    hipStream_t s = as_stream(stream);
    if (n_vert == 0) {
        if (int rc = launch_fill_i32(d_out_n_alpha, 0, 1, s)) return rc;
        return launch_fill_i32(d_out_n_condensates, 0, (long long)num_rows + 1, s);
    }
    HGC_REQUIRE(d_row_splits && d_alpha_idx && d_n_condensates && d_assignment && d_association && d_is_cond &&
                    d_out_alpha_idx, "null pointer");
    if (!workspace || !aligned256(workspace) ||
        workspace_bytes < hgc_keep_noise_condensates_workspace_bytes(n_vert, num_rows))
        return fail(HGC_ERR_WORKSPACE, "keep_noise workspace missing, misaligned or too small");
    const int n_parts = ceil_div(n_vert, kPart);
    Carver carve(workspace);
    Counts *parts = carve.take<Counts>(n_parts + 1ull);
    int *noise_before = carve.take<int>(num_rows + 1ull);
    part_counts_kernel<<<n_parts, kPartThreads, 0, s>>>(d_assignment, d_association, d_is_cond, n_vert, parts);
    part_scan_kernel<<<1, 1024, 0, s>>>(parts, n_parts);
    boundary_counts_kernel<<<ceil_div(num_rows + 1ll, kPartWaves), kPartThreads, 0, s>>>(
        d_assignment, d_association, d_is_cond, n_vert, d_row_splits, num_rows, parts, n_parts, d_n_condensates,
        noise_before, d_out_n_condensates, d_out_n_alpha);
    keep_noise_kernel<<<n_parts, kPartThreads, 0, s>>>(d_row_splits, n_vert, num_rows, parts, noise_before,
                                                      d_n_condensates, d_alpha_idx, d_assignment, d_association,
                                                      d_is_cond, d_out_alpha_idx);
    return check_launch("keep_noise");
}

}  // extern "C"
