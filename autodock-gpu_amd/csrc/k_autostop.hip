// k_autostop.hip -- the AutoStop test on the device.
//
// The reference tests the population every as_frequency generations on the
// host: AutoStop::check_if_satisfactory (host/inc/autostop.hpp:181-231) on the
// downloaded energies, leaving the generation loop when the test passes and
// total_evals > min_as_evals (host/src/performdocking.cpp.Cuda:687-696).  Here
// one workgroup runs the same test between two generations on the resident
// energies and raises the job's stop flag, so the host never has to drain the
// device to decide.
//
// The result must equal the reference host's bit for bit: its sums are float
// sums in population order, so each stays one chain of additions in that
// order.  What bounds the test is therefore one wavefront's latency, and the
// work beside the chains is taken off them: the workgroup finds the samples
// below the threshold, their bins (bisection over the monotone bin edges, in
// double) and their squares, and packs them in order; then every sum of every
// bin has a lane of its own, which adds each sample or -0.0, the number that
// changes no float it is added to -- a comparison, a select and an addition a
// sample, with no branch and with the next sixteen samples' reads under way.
// The three sums over all samples take a wavefront that only adds.
// A test of 20 x 150 energies takes 17 us (some 400 with one lane summing all
// three values of a bin under a branch a sample and one lane walking the
// bins), the first test of a docking 190, since the reference tabulates nine
// times there.  Division and square root go through double, which rounds to the
// correctly rounded float result.
#include "adgpu_internal.h"

namespace adgpu {

namespace {

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / 64;
constexpr int kPerThread = 2;
constexpr int kChunk = kThreads * kPerThread;   // energies staged in LDS per pass
constexpr int kStep = 16;                       // samples a sum's lane reads at once
constexpr int kRow = kChunk + 4;                // one value's row: the three rows start in different banks

struct Packed {                    // the samples of a chunk that are below the threshold, in order
    alignas(16) float v[3 * kRow]; // energy, square, one; -0.0 up to a multiple of kStep
    alignas(16) int bin[kChunk];   // -1 in the padding
    int count[kPerThread * kWaves];
    float best[kWaves];
    int best_at[kWaves];
};

__device__ __forceinline__ float div_rn(float a, float b) { return (float)((double)a / (double)b); }
__device__ __forceinline__ float sqrt_rn(float a) { return (float)__builtin_sqrt((double)a); }

// average(), autostop.hpp:62-67
__device__ float avg3(const float* s) {
    if (s[2] < 1.0f) return 0.0f;
    return div_rn(s[0], s[2]);
}

// stddev(), autostop.hpp:69-76
__device__ float std3(const float* s) {
#pragma clang fp contract(off)
    if (s[2] < 1.0f) return 0.0f;
    const float a = s[1] * s[2];
    const float b = s[0] * s[0];
    const float sq = a - b;
    if (((double)__builtin_fabsf(sq) <= 0.000001) || (sq < 0.0f)) return 0.0f;
    return div_rn(sqrt_rn(sq), s[2]);
}

// Index of the first bin m in [0, ntop) with e < lo + m * delta
// (autostop.hpp:88-95), ntop if none, -1 if e is not below the threshold.
// The edges lo + (double)((float)m * delta) do not decrease with m when
// delta >= 0, so the first one above e is found by bisection.
__device__ int bin_of(float e, float threshold, double lo, float delta, int ntop) {
#pragma clang fp contract(off)
    if (!(e < threshold)) return -1;
    const double ed = (double)e;
    if (!(delta >= 0.0f)) {
        for (int m = 0; m < ntop; ++m)
            if (ed < lo + (double)((float)m * delta)) return m;
        return ntop;
    }
    int a = 0, b = ntop;
    while (a < b) {
        const int m = (a + b) >> 1;
        if (ed < lo + (double)((float)m * delta)) b = m;
        else a = m + 1;
    }
    return a;
}

// tabulate_energies(), autostop.hpp:78-100, adding to acc (average_sd2_N in
// LDS): acc[0..2] are the sums over all samples, acc[3 m + 3 ..] those of bin
// m.  Returns the lowest energy to thread 0.
__device__ float tabulate(const float* ene, int n, int ntop, float threshold, float thres_stddev, float delta,
                          Packed& P, float* acc) {
#pragma clang fp contract(off)
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const double lo = (double)threshold - 2.0 * (double)thres_stddev;
    float best = 16777216.0f;
    int best_at = 0x7fffffff;
    for (int c0 = 0; c0 < n; c0 += kChunk) {
        float e[kPerThread];
        int bin[kPerThread], before[kPerThread];
#pragma unroll
        for (int k = 0; k < kPerThread; ++k) {
            const int i = c0 + k * kThreads + t;
            e[k] = 0.0f;
            bin[k] = -1;
            if (i < n) {
                e[k] = ene[i];
                if (e[k] < best) { best = e[k]; best_at = i; }
                bin[k] = bin_of(e[k], threshold, lo, delta, ntop);
            }
            const uint64_t in = __ballot(bin[k] >= 0);
            before[k] = __popcll(in & ((1ull << lane) - 1ull));
            if (lane == 0) P.count[k * kWaves + wave] = __popcll(in);
        }
        __syncthreads();
        int len = 0, base[kPerThread];
#pragma unroll
        for (int k = 0; k < kPerThread; ++k) {
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
                if (w == wave) base[k] = len;
                len += P.count[k * kWaves + w];
            }
        }
#pragma unroll
        for (int k = 0; k < kPerThread; ++k) {
            if (bin[k] < 0) continue;
            const int at = base[k] + before[k];
            P.v[at] = e[k];
            P.v[kRow + at] = e[k] * e[k];
            P.v[2 * kRow + at] = 1.0f;
            P.bin[at] = bin[k];
        }
        const int end = (len + kStep - 1) & ~(kStep - 1);
        if (len + t < end) {
            for (int q = 0; q < 3; ++q) P.v[q * kRow + len + t] = -0.0f;
            P.bin[len + t] = -1;
        }
        __syncthreads();
        if (t < 3) {
            float a = acc[t];
            const float4* v = (const float4*)(P.v + t * kRow);
            for (int i = 0; i < end / 4; i += kStep / 4) {
                float4 x[kStep / 4];
#pragma unroll
                for (int q = 0; q < kStep / 4; ++q) x[q] = v[i + q];
#pragma unroll
                for (int q = 0; q < kStep / 4; ++q) { a += x[q].x; a += x[q].y; a += x[q].z; a += x[q].w; }
            }
            acc[t] = a;
        } else if (t >= 64) {
            for (int id = t - 64; id < 3 * ntop; id += kThreads - 64) {
                const int m = id / 3;
                float a = acc[3 + id];
                const float4* v = (const float4*)(P.v + (id - 3 * m) * kRow);
                const int4* b = (const int4*)P.bin;
                for (int i = 0; i < end / 4; i += kStep / 4) {
                    float4 x[kStep / 4];
                    int4 y[kStep / 4];
#pragma unroll
                    for (int q = 0; q < kStep / 4; ++q) { x[q] = v[i + q]; y[q] = b[i + q]; }
#pragma unroll
                    for (int q = 0; q < kStep / 4; ++q) {
                        a += y[q].x == m ? x[q].x : -0.0f;
                        a += y[q].y == m ? x[q].y : -0.0f;
                        a += y[q].z == m ? x[q].z : -0.0f;
                        a += y[q].w == m ? x[q].w : -0.0f;
                    }
                }
                acc[3 + id] = a;
            }
        }
        __syncthreads();
    }
    // the first of the lowest energies, as a scan in population order finds it
    for (int d = 32; d > 0; d >>= 1) {
        const float o = __shfl_xor(best, d);
        const int at = __shfl_xor(best_at, d);
        if (o < best || (o == best && at < best_at)) { best = o; best_at = at; }
    }
    if (lane == 0) { P.best[wave] = best; P.best_at[wave] = best_at; }
    __syncthreads();
    if (t == 0)
        for (int w = 1; w < kWaves; ++w)
            if (P.best[w] < best || (P.best[w] == best && P.best_at[w] < best_at)) {
                best = P.best[w];
                best_at = P.best_at[w];
            }
    return best;
}

// set_stats(), autostop.hpp:102-126, by one wavefront: lane k holds bin
// m0 + k, and the bins that hold samples are taken in order.
__device__ void set_stats(AutoStopDev& S, float* acc, int ntop, uint32_t ncream, float stopstd) {
#pragma clang fp contract(off)
    const int lane = threadIdx.x;
    float cur[3] = {acc[0], acc[1], acc[2]};
    const float all_avg = avg3(cur), all_std = std3(cur);
    const uint32_t all_n = (uint32_t)cur[2];
    cur[0] = 0.0f; cur[1] = 0.0f; cur[2] = 0.0f;
    float cur_avg = 0.0f;
    uint32_t taken = 0;
    for (int m0 = 0; m0 < ntop && taken < ncream; m0 += 64) {
        float b[3] = {0.0f, 0.0f, 0.0f};
        if (m0 + lane < ntop)
            for (int q = 0; q < 3; ++q) b[q] = acc[3 * (m0 + lane + 1) + q];
        const float b_avg = avg3(b);
        for (uint64_t left = __ballot(b[2] >= 1.0f); left && taken < ncream; left &= left - 1) {
            const int k = __builtin_ctzll(left);
            if (cur[2] < 4.0f || (double)__builtin_fabsf(cur_avg - __shfl(b_avg, k)) < 2.0 * (double)stopstd) {
                for (int q = 0; q < 3; ++q) cur[q] += __shfl(b[q], k);
                cur_avg = avg3(cur);
                taken++;
            }
        }
    }
    if (lane == 0) {
        for (int q = 0; q < 3; ++q) acc[q] = cur[q];
        S.curr_avg = taken > 0 ? cur_avg : all_avg;
        S.curr_std = taken > 0 ? std3(cur) : all_std;
        S.best_n = taken > 0 ? (uint32_t)cur[2] : all_n;
    }
}

__device__ void fill_record(adgpu_autostop_record& r, const AutoStopDev& S, const float* sums, int64_t generation,
                            int64_t total, float threshold, int stop) {
    r.generation = generation;
    r.total_evals = total;
    r.threshold = threshold;
    r.average = S.curr_avg;
    r.stddev = S.curr_std;
    r.samples = (int32_t)S.best_n;
    r.best_energy = S.overall_best;
    r.autostopped = S.autostopped;
    r.stop = stop;
    r.roll_average = avg3(sums);
    r.roll_stddev = std3(sums);
    r.roll_samples = (int32_t)(uint32_t)sums[2];
}

}  // namespace

// mode 0: one test (check_if_satisfactory + the min_as_evals rule); a job
// whose stop flag is already raised is left unchanged.  mode 1: the final
// statistics of output_final_stddev (autostop.hpp:233-244) into *out.
__global__ __launch_bounds__(kThreads) void k_autostop(AutoStopParams P, const float* ene,
                                                       const int32_t* evals_runs, AutoStopDev* st, float* gbins,
                                                       adgpu_autostop_record* log, int32_t* stop, int64_t generation,
                                                       int mode, adgpu_autostop_record* out) {
#pragma clang fp contract(off)
    __shared__ Packed pk;
    __shared__ AutoStopDev S;
    __shared__ int64_t part[kWaves];
    extern __shared__ float acc[];   // average_sd2_N: 3 * (pop_size + 1)
    if (mode == 0 && *stop) return;
    const int t = threadIdx.x;
    const int ntop = P.pop_size, n = P.num_runs * P.pop_size, nb = 3 * (ntop + 1);
    int64_t s = 0;
    for (int r = t; r < P.num_runs; r += kThreads) s += evals_runs[r];
    for (int d = 32; d > 0; d >>= 1) s += __shfl_xor(s, d);
    if ((t & 63) == 0) part[t >> 6] = s;
    if (t == 0) S = *st;
    for (int i = t; i < nb; i += kThreads) acc[i] = gbins[i];
    __syncthreads();
    int64_t total = 0;
    for (int i = 0; i < kWaves; ++i) total += part[i];

    if (mode == 0) {
        const int reps = generation == 0 ? 9 : 1;
        for (int c = 0; c < reps; ++c) {
            if (!((double)__builtin_fabsf(S.curr_avg) > 0.00001)) break;   // S is uniform here
            for (int i = t; i < nb; i += kThreads) acc[i] = 0.0f;
            __syncthreads();
            if (t == 0) S.threshold_used = S.threshold;
            const float best = tabulate(ene, n, ntop, S.threshold, S.thres_stddev, S.delta_energy, pk, acc);
            if (t < 64 && !S.first_time) set_stats(S, acc, ntop, (uint32_t)P.ncream, P.stopstd);
            if (t == 0) {
                S.overall_best = best;
                if (S.first_time) {
                    S.curr_avg = avg3(acc);
                    S.curr_std = std3(acc);
                    S.best_n = (uint32_t)acc[2];
                    S.thres_stddev = S.curr_std;
                    S.threshold = S.curr_avg + S.thres_stddev;
                    S.first_time = 0;
                } else {
                    S.thres_stddev = (S.curr_std < 0.5f * P.stopstd) ? P.stopstd : S.curr_std;
                    const float num = (float)(uint32_t)P.ncream * S.thres_stddev;
                    S.threshold = S.curr_avg + div_rn(num, (float)S.best_n);
                }
                S.delta_energy = (float)(2.0 * (double)S.thres_stddev / (double)(uint32_t)(ntop - 1));
            }
            __syncthreads();
        }
        if (t == 0) {
            // rolling window of the last four tests, autostop.hpp:205-224
            float* r = S.rolling + 4 * S.roll_count;
            const float bn = (float)S.best_n;
            r[0] = S.curr_avg * bn;
            const float v2 = S.curr_std * S.curr_std;
            const float a2 = S.curr_avg * S.curr_avg;
            r[1] = (v2 + a2) * bn;
            r[2] = bn;
            r[3] = S.overall_best;
            S.roll_count = (S.roll_count + 1u) % 4u;
            const float* q = S.rolling;
            acc[0] = q[0] + q[4] + q[8] + q[12];
            acc[1] = q[1] + q[5] + q[9] + q[13];
            acc[2] = q[2] + q[6] + q[10] + q[14];
            float best_avg = q[3] + q[7] + q[11] + q[15];
            best_avg = div_rn(best_avg, 4.0f);
            const float b3 = q[3] * q[3], b7 = q[7] * q[7], b11 = q[11] * q[11], b15 = q[15] * q[15];
            float best_var = b3 + b7 + b11 + b15;
            best_var = div_rn(best_var, 4.0f);
            const float ba2 = best_avg * best_avg;
            best_var -= ba2;
            if ((std3(acc) < P.stopstd) && (generation >= (int64_t)(4u * (uint32_t)P.as_frequency)) &&
                (best_var <= 0.00002f))
                S.autostopped = 1;
            const int halt = S.autostopped && total > P.min_as_evals;
            adgpu_autostop_record rec;
            fill_record(rec, S, acc, generation, total, S.threshold_used, halt);
            log[S.num_tests % P.log_cap] = rec;
            S.num_tests++;
            if (halt) *stop = 1;
        }
    } else {
        if (!S.autostopped) {
            const float best = tabulate(ene, n, ntop, S.threshold, S.thres_stddev, S.delta_energy, pk, acc);
            if (t < 64) set_stats(S, acc, ntop, (uint32_t)P.ncream, P.stopstd);
            if (t == 0) S.overall_best = best;
        }
        if (t == 0) {
            adgpu_autostop_record rec;
            fill_record(rec, S, acc, generation, total, S.threshold, 0);
            *out = rec;
        }
    }
    __syncthreads();
    for (int i = t; i < nb; i += kThreads) gbins[i] = acc[i];
    if (t == 0) *st = S;
}

hipError_t launch_autostop(hipStream_t s, const AutoStopParams& p, const float* ene, const int32_t* evals_runs,
                           AutoStopDev* st, float* bins, adgpu_autostop_record* log, int32_t* stop,
                           int64_t generation, int mode, adgpu_autostop_record* out) {
    const size_t lds = sizeof(float) * 3 * ((size_t)p.pop_size + 1);
    hipLaunchKernelGGL(k_autostop, dim3(1), dim3(kThreads), lds, s, p, ene, evals_runs, st, bins, log, stop,
                       generation, mode, out);
    return hipGetLastError();
}

}  // namespace adgpu
