// Sign codes for the search's pre-filter.
//
// The reference consumes them (swann/csrc/local_search.cu:205-243: bit b of
// word w stands for dimension 32w + b, set meaning +1 around the corpus mean;
// alpha scales the code back to the corpus's units) and loads them from
// codes_<name>.npy / alpha_<name>.npy / mu_<name>.npy (swann/_engine.py:320-337),
// but does not ship the builder.  This one follows the consumer's estimator:
//   mu[t]    = mean over rows of x[r, t]       (double sums, rounded to fp32)
//   bit      = x[r, t] - mu[t] > 0             (fp32 difference)
//   alpha[r] = sum_t |x[r, t] - mu[t]| / dim   (double sum, rounded to fp32)
//
// Two passes over X, both bound by reading it: column sums (row chunks in
// parallel, partials in a workspace, folded in chunk order so the mean does not
// depend on timing), then one wave per eight rows writing their words and
// alphas.  In both a lane reads 16 bytes of a row (VEC, element loads where the
// rows are not whole 16-byte chunks on a 16-byte boundary) and holds eight
// rows' loads in flight.  400,000 x 1,536 fp16 (1.23 GB):
// 0.21 ms for the sums and 0.29 ms for the words, 5.9 and 4.3 TB/s (a column, then
// a code word, a lane: 0.73 and 2.23 ms).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.h"

namespace swann {
namespace {

constexpr int kChunks = 256;
constexpr int kWaves = 4;                      // a workgroup
constexpr int kRows = 8;                       // rows a wave has in flight

// A lane's share of a row: 16 bytes, elements [16 / sizeof(XT) * lane, ...) of
// every 64-lane group.
template <typename XT>
struct Chunk {
    static constexpr int N = 16 / (int)sizeof(XT);
    static constexpr int kGroup = 64 * N;      // columns of a group
    XT v[N];
};

// Elements [t, t + N) of a row of `dim`, zero past it.
template <typename XT, bool VEC>
__device__ __forceinline__ Chunk<XT> load_chunk(const XT* __restrict__ x, int t, int dim) {
    Chunk<XT> c;
    if constexpr (VEC) {
        // dim is a multiple of N: a chunk is inside the row or past it
        const uint4 raw = *reinterpret_cast<const uint4*>(x + (t < dim ? t : 0));
        c = __builtin_bit_cast(Chunk<XT>, raw);
    } else {
#pragma unroll
        for (int i = 0; i < Chunk<XT>::N; ++i) c.v[i] = t + i < dim ? x[t + i] : (XT)0;
    }
    return c;
}

// Partial column sums: workgroup (g, c) sums group g's columns over the rows of
// chunk c, its waves taking every fourth row; the waves' sums meet in LDS in
// wave order.
template <typename XT, bool VEC>
__global__ __launch_bounds__(kWaves * 64) void col_partial(const XT* __restrict__ X, int64_t n,
                                                           int dim, int64_t rows_per,
                                                           double* __restrict__ part) {
    using C = Chunk<XT>;
    __shared__ double sum[kWaves][C::kGroup];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int t = blockIdx.x * C::kGroup + lane * C::N;
    const int64_t r0 = (int64_t)blockIdx.y * rows_per;
    const int64_t r1 = r0 + rows_per < n ? r0 + rows_per : n;
    double s[C::N];
#pragma unroll
    for (int i = 0; i < C::N; ++i) s[i] = 0.0;
    int64_t r = r0 + wave;
    for (; r + (kRows - 1) * kWaves < r1; r += kRows * kWaves) {
        C x[kRows];
#pragma unroll
        for (int k = 0; k < kRows; ++k) x[k] = load_chunk<XT, VEC>(X + (r + k * kWaves) * dim, t, dim);
#pragma unroll
        for (int k = 0; k < kRows; ++k)
#pragma unroll
            for (int i = 0; i < C::N; ++i) s[i] += (double)(float)x[k].v[i];
    }
    for (; r < r1; r += kWaves) {
        const C x = load_chunk<XT, VEC>(X + r * dim, t, dim);
#pragma unroll
        for (int i = 0; i < C::N; ++i) s[i] += (double)(float)x.v[i];
    }
#pragma unroll
    for (int i = 0; i < C::N; ++i) sum[wave][lane * C::N + i] = s[i];
    __syncthreads();
    for (int i = threadIdx.x; i < C::kGroup; i += kWaves * 64) {
        const int c = blockIdx.x * C::kGroup + i;
        if (c >= dim) break;
        double v = sum[0][i];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) v += sum[w][i];
        part[(int64_t)blockIdx.y * dim + c] = v;
    }
}

// mu of a column: its chunks' sums in chunk order, a wave's lanes 64 columns.
__global__ __launch_bounds__(64) void col_final(const double* __restrict__ part, int nchunk,
                                                int dim, int64_t n, float* __restrict__ mu) {
    const int c = blockIdx.x * 64 + threadIdx.x;
    if (c >= dim) return;
    double s = 0.0;
#pragma unroll 16
    for (int k = 0; k < nchunk; ++k) s += part[(int64_t)k * dim + c];
    mu[c] = (float)(s / (double)n);
}

// One wave per kRows rows: a lane sets the bits of its chunk, the 32 / N lanes of
// a word join theirs, and alpha folds over the wave.  Rows past n repeat row
// n - 1 (their results are not written).
template <typename XT, bool VEC>
__global__ __launch_bounds__(kWaves * 64) void code_rows(const XT* __restrict__ X, int64_t n,
                                                         int dim, int cwords,
                                                         const float* __restrict__ mu,
                                                         int32_t* __restrict__ codes,
                                                         float* __restrict__ alpha) {
    using C = Chunk<XT>;
    constexpr int kPer = 32 / C::N;            // lanes of a word: 4 (fp16) or 8 (fp32)
    const int lane = threadIdx.x & 63;
    const int64_t r0 = ((int64_t)blockIdx.x * kWaves + (threadIdx.x >> 6)) * kRows;
    if (r0 >= n) return;
    double l1[kRows];
#pragma unroll
    for (int k = 0; k < kRows; ++k) l1[k] = 0.0;
    for (int t0 = 0; t0 < dim; t0 += C::kGroup) {
        const int t = t0 + lane * C::N;
        C x[kRows];
#pragma unroll
        for (int k = 0; k < kRows; ++k)
            x[k] = load_chunk<XT, VEC>(X + (r0 + k < n ? r0 + k : n - 1) * dim, t, dim);
        float m[C::N];
#pragma unroll
        for (int i = 0; i < C::N; ++i) m[i] = t + i < dim ? mu[t + i] : 0.f;
#pragma unroll
        for (int k = 0; k < kRows; ++k) {
            unsigned bits = 0u;
#pragma unroll
            for (int i = 0; i < C::N; ++i) {
                const float df = t + i < dim ? (float)x[k].v[i] - m[i] : 0.f;
                bits |= (df > 0.f ? 1u : 0u) << i;
                l1[k] += (double)fabsf(df);
            }
            bits <<= (lane & (kPer - 1)) * C::N;
#pragma unroll
            for (int off = 1; off < kPer; off <<= 1) bits |= __shfl_xor(bits, off, 64);
            const int w = t / 32;
            if ((lane & (kPer - 1)) == 0 && w < cwords && r0 + k < n)
                codes[(r0 + k) * cwords + w] = (int32_t)bits;
        }
    }
#pragma unroll
    for (int k = 0; k < kRows; ++k) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) l1[k] += __shfl_down(l1[k], off, 64);
        if (lane == 0 && r0 + k < n) alpha[r0 + k] = (float)(l1[k] / (double)dim);
    }
}

template <typename XT, bool VEC>
void codes_run(const XT* X, int64_t n, int dim, bool mean, int32_t* codes, float* alpha, float* mu,
               double* part, int nchunk, hipStream_t st) {
    if (mean) {
        const unsigned g = (unsigned)((dim + Chunk<XT>::kGroup - 1) / Chunk<XT>::kGroup);
        hipLaunchKernelGGL((col_partial<XT, VEC>), dim3(g, nchunk), dim3(kWaves * 64), 0, st, X, n,
                           dim, (n + nchunk - 1) / nchunk, part);
        hipLaunchKernelGGL(col_final, dim3((unsigned)((dim + 63) / 64)), dim3(64), 0, st, part,
                           nchunk, dim, n, mu);
    }
    hipLaunchKernelGGL((code_rows<XT, VEC>),
                       dim3((unsigned)((n + kWaves * kRows - 1) / (kWaves * kRows))),
                       dim3(kWaves * 64), 0, st, X, n, dim, (dim + 31) / 32, mu, codes, alpha);
}

int nchunks_for(int64_t n) { return n < kChunks ? (int)n : kChunks; }

}  // namespace
}  // namespace swann

using namespace swann;

extern "C" {

int64_t swann_codes_workspace_size(int64_t n, int dim) {
    if (n <= 0 || dim <= 0) return 0;
    return (int64_t)nchunks_for(n) * dim * (int64_t)sizeof(double);
}

int swann_build_codes(const void* X, int x_dtype, int64_t n, int dim, const float* mu_in,
                      int32_t* codes, float* alpha, float* mu_out, void* workspace,
                      void* stream) {
    clear_error();
    SWANN_REQUIRE(n > 0 && dim > 0, "X must be a non-empty [n, dim] matrix");
    SWANN_REQUIRE(x_dtype == SWANN_DTYPE_F32 || x_dtype == SWANN_DTYPE_F16,
                  "X: float32 or float16");
    SWANN_REQUIRE(X && codes && alpha && mu_out, "build_codes: a required pointer is NULL");
    SWANN_REQUIRE(mu_in || workspace, "build_codes: computing the mean needs the workspace");
    hipStream_t st = (hipStream_t)stream;
    SWANN_REQUIRE((n + 3) / 4 <= (int64_t)INT32_MAX, "too many rows for one launch");
    if (mu_in && mu_in != mu_out) {
        const hipError_t e = hipMemcpyAsync(mu_out, mu_in, sizeof(float) * (size_t)dim,
                                            hipMemcpyDeviceToDevice, st);
        if (e != hipSuccess) return launch_status("build_codes (copy mu)");
    }
    const int nchunk = nchunks_for(n);
    double* part = static_cast<double*>(workspace);
    const bool f32 = x_dtype == SWANN_DTYPE_F32;
    const bool vec = dim % (f32 ? 4 : 8) == 0 && (uintptr_t)X % 16 == 0;
    if (f32)
        (vec ? codes_run<float, true> : codes_run<float, false>)(
            static_cast<const float*>(X), n, dim, !mu_in, codes, alpha, mu_out, part, nchunk, st);
    else
        (vec ? codes_run<_Float16, true> : codes_run<_Float16, false>)(
            static_cast<const _Float16*>(X), n, dim, !mu_in, codes, alpha, mu_out, part, nchunk,
            st);
    return launch_status("build_codes");
}

}  // extern "C"
