// The two scalars around the linear cross-entropy's kernels: the valid-row count with its reciprocal, and the mean loss.
// Reference: src/sisa/kernels/linear_ce.py:138-191 (n_valid, the loss sum). One workgroup each: at the row counts a
// call has, a few thousand 4- or 8-byte values, the six torch launches they replace (compare, sum, cast, reciprocal;
// sum, divide) cost 4 to 5 us apiece and nothing else: evaluations of 1,023 rows of 512 120 -> 107 us, of 4,096 258 -> 249,
// of 16,384 793 -> 784. More rows than that are more than one workgroup reads well: the _wide forms give each workgroup up
// to 8,192 at a time and add their partial sums in order in a second launch. Evaluations of rows of 64 at 1,003 tokens, us,
// one workgroup, several, and torch's sums: 32,768 rows 57, 71, 65; 65,536 81, 70, 85; 131,072 155, 95, 114.
#include "common.h"
#include "host.h"
#include "sisa_hip_ce.h"

namespace {

constexpr int NT = 1024, AHEAD = 8;          // threads; loads in flight per thread
constexpr int PARTS = 256;                   // workgroups of the wide forms at most

template <class V, int THREADS = NT>
SISA_DEV V block_sum(V v, V* lds) {          // fixed order: lanes by halving, waves in order; the total in thread 0
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if (lane == 0) lds[w] = v;
    __syncthreads();
    V s = 0;
    if (threadIdx.x == 0)
        for (int k = 0; k < THREADS / 64; ++k) s += lds[k];
    return s;
}

// The rows of workgroup b of a grid, `per` each: the whole of a launch of one workgroup with per = N.
template <class F>
SISA_DEV void each_ahead(int64_t N, int64_t per, F body) {
    const int64_t begin = blockIdx.x * per, end = begin + per < N ? begin + per : N;
    for (int64_t i0 = begin + threadIdx.x; i0 < end; i0 += NT * AHEAD) body(i0, end);
}

SISA_DEV void store_count(int64_t c, float* n_valid, float* inv_n) {
    *n_valid = (float)c;
    *inv_n = 1.f / (float)c;
}

__global__ __launch_bounds__(NT) void ce_count_kernel(const int64_t* labels, int64_t N, int64_t ignore, float* n_valid,
                                                      float* inv_n, int64_t* parts, int64_t per) {
    __shared__ int64_t part[NT / 64];
    int64_t c = 0;
    each_ahead(N, per, [&](int64_t i0, int64_t end) {
        int64_t t[AHEAD];
#pragma unroll
        for (int e = 0; e < AHEAD; ++e) t[e] = i0 + e * NT < end ? labels[i0 + e * NT] : ignore;
#pragma unroll
        for (int e = 0; e < AHEAD; ++e) c += t[e] != ignore;
    });
    c = block_sum<int64_t>(c, part);
    if (threadIdx.x != 0) return;
    if (parts) parts[blockIdx.x] = c;
    else store_count(c, n_valid, inv_n);
}

__global__ __launch_bounds__(NT) void ce_mean_kernel(const float* rows, int64_t N, const float* n_valid, float* mean,
                                                     double* parts, int64_t per) {
    __shared__ double part[NT / 64];
    double s = 0.0;
    each_ahead(N, per, [&](int64_t i0, int64_t end) {
        float t[AHEAD];
#pragma unroll
        for (int e = 0; e < AHEAD; ++e) t[e] = i0 + e * NT < end ? rows[i0 + e * NT] : 0.f;
#pragma unroll
        for (int e = 0; e < AHEAD; ++e) s += (double)t[e];
    });
    s = block_sum<double>(s, part);
    if (threadIdx.x != 0) return;
    if (parts) parts[blockIdx.x] = s;
    else *mean = (float)s / *n_valid;
}

__global__ __launch_bounds__(PARTS) void ce_count_total_kernel(const int64_t* parts, int n, float* n_valid, float* inv_n) {
    __shared__ int64_t part[PARTS / 64];
    const int64_t c = block_sum<int64_t, PARTS>((int)threadIdx.x < n ? parts[threadIdx.x] : 0, part);
    if (threadIdx.x == 0) store_count(c, n_valid, inv_n);
}

__global__ __launch_bounds__(PARTS) void ce_mean_total_kernel(const double* parts, int n, const float* n_valid, float* mean) {
    __shared__ double part[PARTS / 64];
    const double s = block_sum<double, PARTS>((int)threadIdx.x < n ? parts[threadIdx.x] : 0.0, part);
    if (threadIdx.x == 0) *mean = (float)s / *n_valid;
}

// Rows per workgroup of the wide forms, whole batches of loads, and the workgroups that makes.
int64_t wide_per(int64_t N) { return sisa::cdiv(sisa::cdiv(N, PARTS), NT * AHEAD) * NT * AHEAD; }
int wide_parts(int64_t N) { return (int)sisa::cdiv(N, wide_per(N)); }

}  // namespace

extern "C" int sisa_ce_count(const int64_t* labels, int64_t N, int64_t ignore_index, float* n_valid, float* inv_n,
                             void* stream) {
    SISA_REQUIRE(N >= 0 && (labels || N == 0) && n_valid && inv_n, "sisa_ce_count: null pointer or N < 0");
    ce_count_kernel<<<1, NT, 0, (hipStream_t)stream>>>(labels, N, ignore_index, n_valid, inv_n, nullptr, N);
    return sisa::launch_status("sisa_ce_count");
}

extern "C" int sisa_ce_mean(const float* rows, int64_t N, const float* n_valid, float* mean, void* stream) {
    SISA_REQUIRE(N >= 0 && (rows || N == 0) && n_valid && mean, "sisa_ce_mean: null pointer or N < 0");
    ce_mean_kernel<<<1, NT, 0, (hipStream_t)stream>>>(rows, N, n_valid, mean, nullptr, N);
    return sisa::launch_status("sisa_ce_mean");
}

extern "C" int64_t sisa_ce_workspace_bytes(int64_t N) { return N < 1 ? 0 : wide_parts(N) * (int64_t)sizeof(double); }

extern "C" int sisa_ce_count_wide(const int64_t* labels, int64_t N, int64_t ignore_index, float* n_valid, float* inv_n,
                                  void* workspace, void* stream) {
    SISA_REQUIRE(N >= 1 && labels && n_valid && inv_n && workspace && ((uintptr_t)workspace & 7) == 0,
                 "sisa_ce_count_wide: null pointer, N < 1, or workspace not 8-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    ce_count_kernel<<<wide_parts(N), NT, 0, st>>>(labels, N, ignore_index, nullptr, nullptr, (int64_t*)workspace,
                                                  wide_per(N));
    const int rc = sisa::launch_status("sisa_ce_count_wide");
    if (rc) return rc;
    ce_count_total_kernel<<<1, PARTS, 0, st>>>((const int64_t*)workspace, wide_parts(N), n_valid, inv_n);
    return sisa::launch_status("sisa_ce_count_wide (total)");
}

extern "C" int sisa_ce_mean_wide(const float* rows, int64_t N, const float* n_valid, float* mean, void* workspace,
                                 void* stream) {
    SISA_REQUIRE(N >= 1 && rows && n_valid && mean && workspace && ((uintptr_t)workspace & 7) == 0,
                 "sisa_ce_mean_wide: null pointer, N < 1, or workspace not 8-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    ce_mean_kernel<<<wide_parts(N), NT, 0, st>>>(rows, N, nullptr, nullptr, (double*)workspace, wide_per(N));
    const int rc = sisa::launch_status("sisa_ce_mean_wide");
    if (rc) return rc;
    ce_mean_total_kernel<<<1, PARTS, 0, st>>>((const double*)workspace, wide_parts(N), n_valid, mean);
    return sisa::launch_status("sisa_ce_mean_wide (total)");
}
