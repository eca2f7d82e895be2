// The two scalars around the linear cross-entropy's kernels: the valid-row count with its reciprocal, and the mean loss.
// Reference: src/sisa/kernels/linear_ce.py:138-191 (n_valid, the loss sum). One workgroup each: at the row counts a
// call has, a few thousand 4- or 8-byte values, the six torch launches they replace (compare, sum, cast, reciprocal;
// sum, divide) cost 4 to 5 us apiece and nothing else: evaluations of 1,023 rows of 512 120 -> 107 us, of 4,096 258 -> 249,
// of 16,384 793 -> 784. Callers bring at most 65,536 rows; beyond, one workgroup's loads cost more than the launches.
#include "common.h"
#include "host.h"
#include "sisa_hip_ce.h"

namespace {

constexpr int NT = 1024, AHEAD = 8;          // threads; loads in flight per thread

template <class V>
SISA_DEV V block_sum(V v, V* lds) {          // fixed order: lanes by halving, waves in order; the total in thread 0
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if (lane == 0) lds[w] = v;
    __syncthreads();
    V s = 0;
    if (threadIdx.x == 0)
        for (int k = 0; k < NT / 64; ++k) s += lds[k];
    return s;
}

__global__ __launch_bounds__(NT) void ce_count_kernel(const int64_t* labels, int64_t N, int64_t ignore, float* n_valid,
                                                      float* inv_n) {
    __shared__ int64_t part[NT / 64];
    int64_t c = 0;
    for (int64_t i0 = threadIdx.x; i0 < N; i0 += NT * AHEAD) {
        int64_t t[AHEAD];
#pragma unroll
        for (int e = 0; e < AHEAD; ++e) t[e] = i0 + e * NT < N ? labels[i0 + e * NT] : ignore;
#pragma unroll
        for (int e = 0; e < AHEAD; ++e) c += t[e] != ignore;
    }
    c = block_sum<int64_t>(c, part);
    if (threadIdx.x == 0) {
        *n_valid = (float)c;
        *inv_n = 1.f / (float)c;
    }
}

__global__ __launch_bounds__(NT) void ce_mean_kernel(const float* rows, int64_t N, const float* n_valid, float* mean) {
    __shared__ double part[NT / 64];
    double s = 0.0;
    for (int64_t i0 = threadIdx.x; i0 < N; i0 += NT * AHEAD) {
        float t[AHEAD];
#pragma unroll
        for (int e = 0; e < AHEAD; ++e) t[e] = i0 + e * NT < N ? rows[i0 + e * NT] : 0.f;
#pragma unroll
        for (int e = 0; e < AHEAD; ++e) s += (double)t[e];
    }
    s = block_sum<double>(s, part);
    if (threadIdx.x == 0) *mean = (float)s / *n_valid;
}

}  // namespace

extern "C" int sisa_ce_count(const int64_t* labels, int64_t N, int64_t ignore_index, float* n_valid, float* inv_n,
                             void* stream) {
    SISA_REQUIRE(N >= 0 && (labels || N == 0) && n_valid && inv_n, "sisa_ce_count: null pointer or N < 0");
    ce_count_kernel<<<1, NT, 0, (hipStream_t)stream>>>(labels, N, ignore_index, n_valid, inv_n);
    return sisa::launch_status("sisa_ce_count");
}

extern "C" int sisa_ce_mean(const float* rows, int64_t N, const float* n_valid, float* mean, void* stream) {
    SISA_REQUIRE(N >= 0 && (rows || N == 0) && n_valid && mean, "sisa_ce_mean: null pointer or N < 0");
    ce_mean_kernel<<<1, NT, 0, (hipStream_t)stream>>>(rows, N, n_valid, mean);
    return sisa::launch_status("sisa_ce_mean");
}
