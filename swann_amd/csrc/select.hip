// Seed selection: the E nearest catalogue rows per query (swann/_select.py:93-128).
//
// Two steps: a tiled fp32 distance GEMM that writes the distance matrix
// D[q, p] (1 - <q,v> for IP; |v|^2 - 2<q,v> + |q|^2 for L2, the reference's
// formulas) into a caller-owned workspace, and a per-row top-E, ascending by
// (distance, index).  The reference folds slices of 8192 columns into a
// running best; the result is the exact top-E either way.
//
// Batches of up to 8 queries read the catalogue once in a wave-per-rows
// product (dist_gemv).  Larger batches that would still leave most of the
// chip idle (64 queries against a 4096-entry catalogue are 64 GEMM tiles)
// split the K dimension so the grid has >= 1024 workgroups: partial dot
// products go to the workspace, and a finishing pass sums them in split
// order and applies the formula.
// The top-E keeps a row of up to 16384 distances in the registers of 1024
// threads and finds the E-th smallest by a 4-pass radix select over the
// distances' order-preserving 32-bit keys (LDS histograms), then sorts only
// the E survivors; longer rows are streamed once against a running threshold.
#include <float.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <mutex>

#include "common.h"

namespace swann {
namespace {

constexpr int kTM = 64, kTN = 64;             // the tile that the K split is sized by
constexpr int kTopBuf = 4096;                 // twice the largest E
constexpr int kRadBlock = 1024, kRadPer = 16; // radix top-E: rows of up to 16384
constexpr int kRadMaxE = 2048;
constexpr int kMaxSplit = 16;

// K splits for a grid of `tiles` workgroups: enough for >= 1024 workgroups.
int split_for(int64_t tiles) {
    if (tiles >= 256) return 1;
    int64_t s = (1024 + tiles - 1) / tiles;
    return (int)(s < kMaxSplit ? s : kMaxSplit);
}

// Order-preserving key of a distance: -0 folded onto +0, so equal distances
// have equal keys; every NaN takes the largest key, so it ranks after every
// number (as torch.topk ranks NaN) and the order is total.
__device__ __forceinline__ unsigned dkey(float d) {
    if (d != d) return 0xFFFFFFFFu;
    const unsigned u = __float_as_uint(d + 0.0f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// (distance, index) order: on numbers the plain comparison; a NaN after
// every number, NaNs by index.  Total, so a sorting network run on it keeps
// every element once and sorts the padding (pad_d(), INT32_MAX) last.
__device__ __forceinline__ bool lt(float da, int ia, float db, int ib) {
    const unsigned ka = dkey(da), kb = dkey(db);
    return ka < kb || (ka == kb && ia < ib);
}

// The distance of a padding entry: a NaN, which with index INT32_MAX ranks
// after every real entry.
__device__ __forceinline__ float pad_d() { return __int_as_float(0x7fffffff); }

// Squared norms of rows (only the L2 metric needs them).
__global__ __launch_bounds__(256) void row_norms(const float* __restrict__ A, int64_t n, int dim,
                                                 float* __restrict__ out) {
    const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (r >= n) return;
    const float* a = A + r * dim;
    float s = 0.f;
    // eight loads in flight; the sum's order is the loop's
#pragma unroll 8
    for (int t = lane; t < dim; t += 64) s = __builtin_fmaf(a[t], a[t], s);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if (lane == 0) out[r] = s;
}

// D[m, n] = f(<A_m, B_n>) for A [M, dim], B [N, dim], both row-major fp32, on
// the fp32 matrix cores (32x32x2: fp32 products and sums, a fused
// multiply-add a term as the vector unit's).  With `kper` < dim, workgroup z
// covers k in [z*kper, (z+1)*kper) and writes the raw partial dot product to
// Dm + z*M*N (finished by split_finish).
//
// What bounds it is the fp32 MFMA rate (a large library product reaches 154
// TFLOP/s on this card).  Four waves share a T x T tile, each a quarter of it in
// 32 x 32 blocks; K advances 32 floats (128 bytes a row) a stage through two LDS
// buffers, with the loads of two stages ahead in flight in registers.  Chunk c
// of row r sits at chunk c ^ gswz(r), so the 32 rows of a fragment read fall in
// distinct banks.  In step t lane l reads chunk 2t + l/32 of its row, four
// consecutive k, and feeds them to four MFMAs (k = 4 (l/32) + s of the step's 8:
// a permutation of the order in which a step's terms enter the sum, the same
// for every row and column, so equal rows have equal distances to the bit).
// 2,000 x 131,072 x 1,024: 4.3 ms, 125 TFLOP/s (64 x 64 tiles on the vector
// unit: 15.3 ms); 500 x 4,096 x 960: 50 against 162 us; 4,096 x 4,096 x 1,536:
// 0.49 against 1.50 ms.
// T = 128 reads each operand half as often from L2 as T = 64; the smaller tiles keep
// more of the chip busy and pad a batch to fewer rows (gemm_run).
// The vector path of the loads (VEC) needs rows of whole 16-byte chunks on a
// 16-byte boundary; otherwise element loads fill the same stages.
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
constexpr int kGK = 32;                        // floats of K a stage
constexpr int kGRow = kGK * 4;                 // bytes of a row a stage

__device__ __forceinline__ int gswz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

template <int T, bool VEC>
__global__ __launch_bounds__(256) void dist_gemm(const float* __restrict__ A,
                                                 const float* __restrict__ B, int64_t M, int64_t N,
                                                 int dim, int metric,
                                                 const float* __restrict__ an,
                                                 const float* __restrict__ bn,
                                                 float* __restrict__ Dm, int kper) {
    constexpr int BI = T / 64;                 // 32 x 32 blocks a wave, each way
    constexpr int NL = T / 32;                 // 16-byte chunks a thread stages, each operand
    __shared__ __align__(16) unsigned char sA[2][T * kGRow];
    __shared__ __align__(16) unsigned char sB[2][T * kGRow];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = (wave >> 1) * (T / 2), wn = (wave & 1) * (T / 2);
    const int half = lane >> 5;
    // consecutive tiles of one XCD share their columns' rows (m runs fastest)
    const int64_t mt = (M + T - 1) / T;
    const int64_t id = xcd_remap(blockIdx.x, gridDim.x);
    const int64_t m0 = (id % mt) * T, n0 = (id / mt) * T;
    const int kb = blockIdx.z * kper;
    const int ke = (kb + kper < dim) ? kb + kper : dim;
    f32x16 acc[BI][BI];
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
        for (int j = 0; j < BI; ++j) acc[i][j] = (f32x16){};
    // rows past the matrix read its last row; their sums are not written
    const float* pa[NL];
    const float* pb[NL];
    int lds[NL];
    const int ch = tid & 7;
#pragma unroll
    for (int q = 0; q < NL; ++q) {
        const int r = q * 32 + (tid >> 3);
        pa[q] = A + (m0 + r < M ? m0 + r : M - 1) * dim;
        pb[q] = B + (n0 + r < N ? n0 + r : N - 1) * dim;
        lds[q] = r * kGRow + ((ch ^ gswz(r)) << 4);
    }
    // every load is issued, past the end of K from the row's first chunk, and
    // zeroed at staging: no branch for the loads in flight to be waited at
    f32x4 ra[NL], rb[NL];
    int left = 0;                              // elements of the fetched chunk inside K
    auto fetch = [&](int k0) {
        const int k = k0 + ch * 4;
        left = ke - k;
        const int kc = left > 0 ? k : kb;
#pragma unroll
        for (int q = 0; q < NL; ++q) {
            if constexpr (VEC) {
                ra[q] = *reinterpret_cast<const f32x4*>(pa[q] + kc);
                rb[q] = *reinterpret_cast<const f32x4*>(pb[q] + kc);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int ke1 = e < left ? kc + e : kb;
                    ra[q][e] = pa[q][ke1];
                    rb[q][e] = pb[q][ke1];
                }
            }
        }
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int q = 0; q < NL; ++q) {
            f32x4 va = ra[q], vb = rb[q];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                va[e] = (VEC ? 0 : e) < left ? va[e] : 0.f;
                vb[e] = (VEC ? 0 : e) < left ? vb[e] : 0.f;
            }
            *reinterpret_cast<f32x4*>(&sA[buf][lds[q]]) = va;
            *reinterpret_cast<f32x4*>(&sB[buf][lds[q]]) = vb;
        }
    };
    const int fsw = gswz(lane & 31);           // fragment rows are 32 x + lane % 32
    fetch(kb);
    stage(0);
    fetch(kb + kGK);
    __syncthreads();
    int buf = 0;
    f32x4 fga[2][BI], fgb[2][BI];
    auto frags = [&](int t, int slot) {
        const int co = ((2 * t + half) ^ fsw) << 4;
#pragma unroll
        for (int i = 0; i < BI; ++i) {
            const int r = i * 32 + (lane & 31);
            fga[slot][i] = *reinterpret_cast<const f32x4*>(&sA[buf][(wm + r) * kGRow + co]);
            fgb[slot][i] = *reinterpret_cast<const f32x4*>(&sB[buf][(wn + r) * kGRow + co]);
        }
    };
    for (int k0 = kb; k0 < ke; k0 += kGK) {
        frags(0, 0);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            // half way, the next stage goes to the other buffer (last read
            // before the barrier this stage began at) and the one after it is
            // fetched: both among the MFMAs, so the waves of a CU do not meet
            // at the stage's end with nothing to multiply
            if (t == 2) {
                stage(buf ^ 1);
                fetch(k0 + 2 * kGK);
            }
            // the next step's fragments are read while this one's multiply
            if (t < 3) frags(t + 1, (t + 1) & 1);
            // (in that order, where four blocks' MFMAs cover the reads)
            if (BI > 1) __builtin_amdgcn_sched_barrier(0);
            const f32x4* fa = fga[t & 1];
            const f32x4* fb = fgb[t & 1];
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int i = 0; i < BI; ++i)
#pragma unroll
                    for (int j = 0; j < BI; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i][s], fb[j][s],
                                                                         acc[i][j], 0, 0, 0);
        }
        __syncthreads();
        buf ^= 1;
    }
    // lane: column lane % 32 of a block, rows (e / 4) * 8 + 4 (lane / 32) + e % 4
#pragma unroll
    for (int j = 0; j < BI; ++j) {
        const int64_t nn = n0 + wn + j * 32 + (lane & 31);
        if (nn >= N) continue;
        const float b = metric == SWANN_METRIC_L2 && kper >= dim ? bn[nn] : 0.f;
#pragma unroll
        for (int i = 0; i < BI; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int64_t m = m0 + wm + i * 32 + (e >> 2) * 8 + half * 4 + (e & 3);
                if (m >= M) continue;
                const float s = acc[i][j][e];
                if (kper < dim)
                    Dm[(int64_t)blockIdx.z * M * N + m * N + nn] = s;
                else
                    Dm[m * N + nn] = metric == SWANN_METRIC_IP ? 1.0f - s : (b - 2.0f * s) + an[m];
            }
    }
}

// Small batches (nq <= kGvMaxQ): D[m, p] for every query m against catalogue
// rows p, the catalogue read once.  A wave takes kGvRows consecutive rows
// (one: a 4096-row catalogue is 4096 waves, with eight 16-byte loads of the
// row in flight a lane); lane l sums the 4-float blocks l, l + 64, ... of
// each row against each query, which the workgroup stages in LDS
// kGvLds / NQ dimensions at a time; then the wave folds each sum.  For l2 the
// row's |v|^2 is summed on the way.  The 64 x 64 tiles of dist_gemm would
// spend 63 of 64 products on padding at batch 1 and read the catalogue
// through 16 split-K passes.  (Measured at 4096 x 4096 with the top-E: 1
// row and 8 waves a workgroup beat 2 or 4 rows a wave and 4 waves.)
constexpr int kGvRows = 1, kGvWaves = 8, kGvMaxQ = 8;
constexpr int kGvLds = 8192;                  // staged query floats (32 KB)

template <int NQ>
__global__ __launch_bounds__(kGvWaves * 64) void dist_gemv(const float* __restrict__ Q,
                                                           const float* __restrict__ V, int nq,
                                                           int64_t P, int dim, int metric,
                                                           const float* __restrict__ qn,
                                                           float* __restrict__ Dm) {
    constexpr int KC = kGvLds / NQ;           // dimensions staged a pass
    __shared__ __align__(16) float qs[kGvLds];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t p0 = ((int64_t)blockIdx.x * kGvWaves + wave) * kGvRows;
    const bool vec = (dim & 3) == 0 && ((uintptr_t)V & 15) == 0;
    const bool qvec = (dim & 3) == 0 && ((uintptr_t)Q & 15) == 0;
    float acc[kGvRows][NQ], vv[kGvRows];
#pragma unroll
    for (int r = 0; r < kGvRows; ++r) {
        vv[r] = 0.f;
#pragma unroll
        for (int m = 0; m < NQ; ++m) acc[r][m] = 0.f;
    }
    // rows past P read row P - 1 (their sums are never written)
    const float* vr[kGvRows];
#pragma unroll
    for (int r = 0; r < kGvRows; ++r) vr[r] = V + (p0 + r < P ? p0 + r : P - 1) * (int64_t)dim;
    for (int k0 = 0; k0 < dim; k0 += KC) {
        const int kc = dim - k0 < KC ? dim - k0 : KC;
        __syncthreads();                      // the last pass's reads of qs are done
        if (qvec) {
            // 16-byte loads, four in flight a thread
            const int nv = NQ * (kc >> 2);
#pragma unroll 4
            for (int i = tid; i < nv; i += kGvWaves * 64) {
                const int m = i / (kc >> 2), t = (i - m * (kc >> 2)) << 2;
                const float4 v = m < nq ? *reinterpret_cast<const float4*>(Q + (int64_t)m * dim + k0 + t)
                                        : make_float4(0.f, 0.f, 0.f, 0.f);
                *reinterpret_cast<float4*>(&qs[m * KC + t]) = v;
            }
        } else {
            for (int i = tid; i < NQ * kc; i += kGvWaves * 64) {
                const int m = i / kc, t = i - m * kc;
                qs[m * KC + t] = m < nq ? Q[(int64_t)m * dim + k0 + t] : 0.f;
            }
        }
        __syncthreads();
        if (vec) {
#pragma unroll 8
            for (int t = lane * 4; t < kc; t += 256) {
                float4 x[kGvRows];
#pragma unroll
                for (int r = 0; r < kGvRows; ++r)
                    x[r] = *reinterpret_cast<const float4*>(vr[r] + k0 + t);
#pragma unroll
                for (int m = 0; m < NQ; ++m) {
                    const float4 q = *reinterpret_cast<const float4*>(&qs[m * KC + t]);
#pragma unroll
                    for (int r = 0; r < kGvRows; ++r) {
                        float s = acc[r][m];
                        s = __builtin_fmaf(x[r].x, q.x, s);
                        s = __builtin_fmaf(x[r].y, q.y, s);
                        s = __builtin_fmaf(x[r].z, q.z, s);
                        acc[r][m] = __builtin_fmaf(x[r].w, q.w, s);
                    }
                }
                if (metric == SWANN_METRIC_L2) {
#pragma unroll
                    for (int r = 0; r < kGvRows; ++r) {
                        float s = vv[r];
                        s = __builtin_fmaf(x[r].x, x[r].x, s);
                        s = __builtin_fmaf(x[r].y, x[r].y, s);
                        s = __builtin_fmaf(x[r].z, x[r].z, s);
                        vv[r] = __builtin_fmaf(x[r].w, x[r].w, s);
                    }
                }
            }
        } else {
            for (int t = lane; t < kc; t += 64) {
                float x[kGvRows];
#pragma unroll
                for (int r = 0; r < kGvRows; ++r) x[r] = vr[r][k0 + t];
#pragma unroll
                for (int m = 0; m < NQ; ++m) {
                    const float q = qs[m * KC + t];
#pragma unroll
                    for (int r = 0; r < kGvRows; ++r) acc[r][m] = __builtin_fmaf(x[r], q, acc[r][m]);
                }
#pragma unroll
                for (int r = 0; r < kGvRows; ++r) vv[r] = __builtin_fmaf(x[r], x[r], vv[r]);
            }
        }
    }
    // fold every sum over the wave (each lane ends with every total); lane
    // r * NQ + m writes D[m, p0 + r]
    float out = 0.f;
#pragma unroll
    for (int r = 0; r < kGvRows; ++r) {
        float n2 = vv[r];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) n2 += __shfl_xor(n2, off, 64);
#pragma unroll
        for (int m = 0; m < NQ; ++m) {
            float s = acc[r][m];
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
            if (lane == r * NQ + m)
                out = metric == SWANN_METRIC_IP ? 1.0f - s
                                                : (n2 - 2.0f * s) + (m < nq ? qn[m] : 0.f);
        }
    }
    const int r = lane / NQ, m = lane - r * NQ;
    if (lane < kGvRows * NQ && m < nq && p0 + r < P) Dm[(int64_t)m * P + p0 + r] = out;
}

// Sum the S partial dot products in split order, then the distance formula.
__global__ __launch_bounds__(256) void split_finish(const float* __restrict__ part, int S,
                                                    int64_t M, int64_t N, int metric,
                                                    const float* __restrict__ an,
                                                    const float* __restrict__ bn,
                                                    float* __restrict__ Dm) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= M * N) return;
    float s = part[i];
    for (int z = 1; z < S; ++z) s += part[(int64_t)z * M * N + i];
    const int64_t m = i / N, nn = i - m * N;
    Dm[i] = metric == SWANN_METRIC_IP ? 1.0f - s : (bn[nn] - 2.0f * s) + an[m];
}

// A wave's 64 (d, id) pairs in ascending order, in registers: a bitonic network
// over the lanes (padding entries sort last), no barriers.
__device__ __forceinline__ void wave_sort(float& d, int& id) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int size = 2; size <= 64; size <<= 1) {
#pragma unroll
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            const float d2 = __shfl_xor(d, stride, 64);
            const int id2 = __shfl_xor(id, stride, 64);
            // both lanes of a pair decide the same swap, from the lower
            // lane's element (so a pair the order cannot rank, NaN against
            // NaN, is swapped or kept whole, never duplicated)
            const bool up = (lane & size) == 0;
            const bool sw = (lane & stride) == 0 ? up != lt(d, id, d2, id2)
                                                 : up != lt(d2, id2, d, id);
            if (sw) { d = d2; id = id2; }
        }
    }
}

// Row top-E for rows of N <= kRadBlock*kRadPer: radix select of the E-th key,
// then a bitonic sort of the E survivors by (d, index).
__global__ __launch_bounds__(kRadBlock) void row_topk_radix(const float* __restrict__ Dm,
                                                           int64_t N, int E,
                                                           int32_t* __restrict__ oi,
                                                           float* __restrict__ od) {
    __shared__ unsigned hist[256];
    __shared__ unsigned s_bucket, s_before;
    __shared__ int s_nsel, s_wcnt[kRadBlock / 64], s_ebase;
    __shared__ float sd[kRadMaxE];
    __shared__ int si[kRadMaxE];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t r = blockIdx.x;
    const float* row = Dm + r * N;
    // slots i < nper hold keys (column tid + i * kRadBlock); the loops below
    // visit only those, and skip the padding columns c >= N
    const int nper = (int)((N + kRadBlock - 1) / kRadBlock);
    unsigned key[kRadPer];
#pragma unroll
    for (int i = 0; i < kRadPer; ++i) {
        const int64_t c = tid + (int64_t)i * kRadBlock;
        key[i] = (i < nper && c < N) ? dkey(row[c]) : 0xFFFFFFFFu;
    }
    // ---- the E-th smallest key, 8 bits at a time from the top ----
    unsigned prefix = 0u, pmask = 0u;
    int need = E;                       // how many to take from the current bucket
    for (int pass = 0; pass < 4; ++pass) {
        const int shift = 24 - 8 * pass;
        if (tid < 256) hist[tid] = 0u;
        __syncthreads();
        // Distances that share their leading bits (all of them, in the
        // first pass over a row of similar distances) fall into a few bins:
        // lanes of a wave that share the first two bins add with one atomic
        // each, the rest one by one.
#pragma unroll
        for (int i = 0; i < kRadPer; ++i) {
            if (i >= nper) break;
            const unsigned bin = (key[i] >> shift) & 255u;
            bool pend = tid + i * kRadBlock < N && (key[i] & pmask) == prefix;
#pragma unroll
            for (int peel = 0; peel < 2; ++peel) {
                const uint64_t act = __ballot(pend);
                if (act == 0) break;
                const unsigned b0 = __builtin_amdgcn_readlane(bin, __builtin_ctzll(act));
                const uint64_t same = __ballot(pend && bin == b0);
                if (pend && bin == b0) {
                    if (lane == __builtin_ctzll(same))
                        atomicAdd(&hist[b0], (unsigned)__builtin_popcountll(same));
                    pend = false;
                }
            }
            if (pend) atomicAdd(&hist[bin], 1u);
        }
        __syncthreads();
        if (wave == 0) {
            unsigned h[4], run = 0u;
#pragma unroll
            for (int j = 0; j < 4; ++j) { h[j] = hist[lane * 4 + j]; run += h[j]; }
            unsigned incl = run;        // inclusive scan of lane totals
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const unsigned o = __shfl_up(incl, off, 64);
                if (lane >= off) incl += o;
            }
            unsigned before = incl - run;
            const bool mine = before < (unsigned)need && incl >= (unsigned)need;
            if (mine) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (before + h[j] >= (unsigned)need) { s_bucket = lane * 4 + j; s_before = before; break; }
                    before += h[j];
                }
            }
        }
        __syncthreads();
        prefix |= s_bucket << shift;
        pmask |= 0xFFu << shift;
        need -= (int)s_before;
        __syncthreads();
    }
    const unsigned T = prefix;          // keys < T: all taken; keys == T: the `need` lowest indices
    if (tid == 0) { s_nsel = 0; s_ebase = 0; }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kRadPer; ++i) {
        if (i >= nper) break;
        if (key[i] < T) {
            const int pos = atomicAdd(&s_nsel, 1);
            const int c = tid + i * kRadBlock;
            sd[pos] = row[c]; si[pos] = c;
        }
    }
    __syncthreads();
    const int nless = s_nsel;           // == E - need
    // ties at T in index order (c = tid + i*kRadBlock: i-major, then tid)
    for (int i = 0; i < nper; ++i) {
        // padding slots (c >= N) carry the largest key and the largest
        // indices: never taken, even when a NaN distance ties them
        const bool eq = key[i] == T && tid + i * kRadBlock < N;
        const uint64_t m = __ballot(eq);
        if (lane == 0) s_wcnt[wave] = __builtin_popcountll(m);
        __syncthreads();
        int base = s_ebase;
        for (int w = 0; w < wave; ++w) base += s_wcnt[w];
        const int rank = base + __builtin_popcountll(m & ((1ull << lane) - 1ull));
        if (eq && rank < need) {
            const int c = tid + i * kRadBlock;
            sd[nless + rank] = row[c]; si[nless + rank] = c;
        }
        __syncthreads();
        if (tid == 0) {
            int tot = 0;
            for (int w = 0; w < kRadBlock / 64; ++w) tot += s_wcnt[w];
            s_ebase += tot;
        }
        __syncthreads();
        if (s_ebase >= need) break;     // uniform: every later tie ranks >= need
    }
    // ---- sort the E survivors by (d, index) ----
    if (E <= 64) {
        // one wave, in registers (lanes past E hold the padding entry)
        __syncthreads();
        if (wave != 0) return;
        float d = lane < E ? sd[lane] : pad_d();
        int id = lane < E ? si[lane] : INT32_MAX;
        wave_sort(d, id);
        if (lane < E) {
            oi[r * E + lane] = id;
            if (od) od[r * E + lane] = d;
        }
        return;
    }
    int n = 1;
    while (n < E) n <<= 1;
    for (int i = E + tid; i < n; i += kRadBlock) { sd[i] = pad_d(); si[i] = INT32_MAX; }
    __syncthreads();
    for (int size = 2; size <= n; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int i = tid; i < n; i += kRadBlock) {
                const int j = i ^ stride;
                if (j > i) {
                    const bool up = ((i & size) == 0);
                    if (up != lt(sd[i], si[i], sd[j], si[j])) {
                        const float td = sd[i]; sd[i] = sd[j]; sd[j] = td;
                        const int ti = si[i]; si[i] = si[j]; si[j] = ti;
                    }
                }
            }
            __syncthreads();
        }
    }
    for (int e = tid; e < E; e += kRadBlock) {
        oi[r * E + e] = si[e];
        if (od) od[r * E + e] = sd[e];
    }
}

// Row top-E for longer rows (an entry pool or a whole corpus): one pass over
// the row against a running threshold.  A workgroup streams its share of the
// row 2,048 distances at a time, the next two groups' loads in flight, appends
// those that rank below the E-th best so far to a buffer in LDS, and cuts the
// buffer back to its E best when another group might not fit (stream_cut: radix
// select, exact, ties to the lower index).  After the first cut only about
// E ln(N / 2048) of a row's N distances are appended, so the pass is bound by
// reading the matrix; 33 KB of LDS is four workgroups a CU, 64 KB of loads in
// flight on each.  (Sorting the row 4,096 at a time instead: 2,000 rows of
// 131,072, E = 32, took 17.2 ms; this takes 0.30 ms, 3.5 TB/s of the matrix;
// 1,024 rows of 400,003, E = 10: 26.8 against 0.35 ms, 4.6 TB/s.)
constexpr int kStBlock = 256, kStPer = 8, kStGroup = kStBlock * kStPer;
constexpr int kStBuf = 2 * kStGroup;
constexpr int kStOwn = kStBuf / kStBlock;      // buffer entries a thread holds in a cut
static_assert(kTopBuf / 2 + kStGroup <= kStBuf, "after a cut a group fits");

struct StreamLds {
    float d[kStBuf];
    int i[kStBuf];
    unsigned hist[256];
    unsigned bucket, before, tie;
    int cnt, wcnt[2][kStBlock / 64];
};

// One radix select over the workgroup's values u(j), j < kStOwn a thread, those
// with in(j): the value of rank `need` (from 1), and how many rank before it.
template <class U, class In>
__device__ __forceinline__ void stream_rank(StreamLds& L, U u, In in, int need, unsigned* value,
                                            int* less) {
    const int tid = threadIdx.x, lane = tid & 63;
    unsigned prefix = 0u, pmask = 0u;
    const int need0 = need;
    for (int shift = 24; shift >= 0; shift -= 8) {
        L.hist[tid] = 0u;
        __syncthreads();
        // values that share their leading bits fall into a few bins: a wave's
        // lanes of its first two bins add with one atomic each
#pragma unroll
        for (int j = 0; j < kStOwn; ++j) {
            const unsigned bin = (u(j) >> shift) & 255u;
            bool pend = in(j) && (u(j) & pmask) == prefix;
#pragma unroll
            for (int peel = 0; peel < 2; ++peel) {
                const uint64_t act = __ballot(pend);
                if (act == 0) break;
                const unsigned b0 = __builtin_amdgcn_readlane(bin, __builtin_ctzll(act));
                const uint64_t same = __ballot(pend && bin == b0);
                if (pend && bin == b0) {
                    if (lane == __builtin_ctzll(same))
                        atomicAdd(&L.hist[b0], (unsigned)__builtin_popcountll(same));
                    pend = false;
                }
            }
            if (pend) atomicAdd(&L.hist[bin], 1u);
        }
        __syncthreads();
        if (tid < 64) {
            unsigned h[4], run = 0u;
#pragma unroll
            for (int j = 0; j < 4; ++j) { h[j] = L.hist[lane * 4 + j]; run += h[j]; }
            unsigned incl = run;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const unsigned o = __shfl_up(incl, off, 64);
                if (lane >= off) incl += o;
            }
            unsigned before = incl - run;
            if (before < (unsigned)need && incl >= (unsigned)need) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (before + h[j] >= (unsigned)need) {
                        L.bucket = lane * 4 + j;
                        L.before = before;
                        break;
                    }
                    before += h[j];
                }
            }
        }
        __syncthreads();
        prefix |= L.bucket << shift;
        pmask |= 0xFFu << shift;
        need -= (int)L.before;
    }
    *value = prefix;
    *less = need0 - need;
}

// Cut the buffer's `n` entries (n >= E) to the E best in (distance, index)
// order, in place and unsorted; returns the E-th best's key.  Ends with a
// barrier and L.cnt == E.
__device__ __forceinline__ unsigned stream_cut(StreamLds& L, int n, int E) {
    const int tid = threadIdx.x, lane = tid & 63;
    float d[kStOwn];
    int id[kStOwn];
#pragma unroll
    for (int j = 0; j < kStOwn; ++j) {
        const int i = tid + j * kStBlock;
        d[j] = i < n ? L.d[i] : 0.f;
        id[j] = i < n ? L.i[i] : 0;
    }
    auto in = [&](int j) { return tid + j * kStBlock < n; };
    auto key = [&](int j) { return dkey(d[j]); };
    unsigned T;
    int less;
    stream_rank(L, key, in, E, &T, &less);
    // copies of T: the E - less lowest indices stay
    auto eq = [&](int j) { return in(j) && key(j) == T; };
    if (tid == 0) { L.tie = 0u; L.cnt = 0; }
    __syncthreads();
    int neq = 0;
#pragma unroll
    for (int j = 0; j < kStOwn; ++j) neq += __builtin_popcountll(__ballot(eq(j)));
    if (lane == 0 && neq) atomicAdd(&L.tie, (unsigned)neq);
    __syncthreads();
    unsigned last = 0xFFFFFFFFu;
    if ((int)L.tie > E - less) {                // uniform
        int unused;
        stream_rank(L, [&](int j) { return (unsigned)id[j]; }, eq, E - less, &last, &unused);
    }
#pragma unroll
    for (int j = 0; j < kStOwn; ++j) {
        const bool keep = in(j) && (key(j) < T || (key(j) == T && (unsigned)id[j] <= last));
        const uint64_t m = __ballot(keep);
        if (m == 0) continue;
        int base = 0;
        if (lane == 0) base = atomicAdd(&L.cnt, __builtin_popcountll(m));
        base = __builtin_amdgcn_readfirstlane(base);
        if (keep) {
            const int at = base + __builtin_popcountll(m & ((1ull << lane) - 1ull));
            L.d[at] = d[j];
            L.i[at] = id[j];
        }
    }
    __syncthreads();
    return T;
}

// Workgroup (row, part): the E best of columns [N part / parts, N (part + 1) /
// parts) of the row.  One part writes the sorted result.  With more, each
// leaves its E best, unsorted, at the start of the columns it has read (E
// distances, then E indices; a part has at least 4 E columns), and row_topk_join
// takes those (JOIN).
template <bool JOIN>
__device__ __forceinline__ void row_topk_body(float* __restrict__ row, int64_t N, int E, int parts,
                                              int part, int32_t* __restrict__ oi,
                                              float* __restrict__ od) {
    __shared__ StreamLds L;
    const int tid = threadIdx.x, lane = tid & 63;
    const int64_t c0 = JOIN ? 0 : N * part / parts;
    const int64_t c1 = JOIN ? (int64_t)parts * E : N * (part + 1) / parts;
    const int64_t len = c1 - c0;
    auto load = [&](int64_t g, float* v, int* id) {
#pragma unroll
        for (int j = 0; j < kStPer; ++j) {
            const int64_t c = g + tid + j * kStBlock;
            const bool ok = c < len;
            if constexpr (JOIN) {
                const int64_t p = ok ? c / E : 0, k = ok ? c - p * E : 0;
                const float* at = row + N * p / parts;
                v[j] = at[k];
                id[j] = reinterpret_cast<const int*>(at + E)[k];
            } else {
                v[j] = row[c0 + (ok ? c : 0)];
            }
        }
    };
    const int wave = tid >> 6;
    unsigned T = 0u;
    bool full = false;                          // T holds: E entries rank at or below it
    int have = 0;                               // entries in the buffer (uniform)
    const int limit = E + 512 < kStGroup ? (E + 512 > 1024 ? E + 512 : 1024) : kStGroup;
    float v[kStPer], v1[kStPer], v2[kStPer];
    int id[kStPer], i1[kStPer], i2[kStPer];
    load(0, v1, i1);
    load(kStGroup, v2, i2);
    int par = 0;
    for (int64_t g = 0; g < len || have > E; g += kStGroup) {
        if (have > limit || g >= len) {         // (the last cut: the row is read)
            __syncthreads();                    // the last group's entries are written
            T = stream_cut(L, have, E);
            full = true;
            have = E;
            if (g >= len) break;
        }
#pragma unroll
        for (int j = 0; j < kStPer; ++j) {
            v[j] = v1[j]; v1[j] = v2[j];
            if constexpr (JOIN) { id[j] = i1[j]; i1[j] = i2[j]; }
            else id[j] = (int)(c0 + g) + tid + j * kStBlock;
        }
        load(g + 2 * kStGroup, v2, i2);
        // an entry that ties the E-th best comes after it in the row and
        // ranks after it; joining parts, their entries are in no order, and
        // the cut decides
        unsigned on = 0u;
        int w = 0;
#pragma unroll
        for (int j = 0; j < kStPer; ++j) {
            const unsigned k = dkey(v[j]);
            const bool p = g + tid + j * kStBlock < len && (!full || (JOIN ? k <= T : k < T));
            on |= (p ? 1u : 0u) << j;
            w += __builtin_popcountll(__ballot(p));
        }
        // the waves' counts give each its slots (two sets, so that the next
        // group's are not written over counts a slower wave still reads)
        if (lane == 0) L.wcnt[par][wave] = w;
        __syncthreads();
        int at = have;
#pragma unroll
        for (int x = 0; x < kStBlock / 64; ++x) {
            const int c = L.wcnt[par][x];
            at += x < wave ? c : 0;
            have += c;
        }
        par ^= 1;
        if (w == 0) continue;                   // uniform in the wave
#pragma unroll
        for (int j = 0; j < kStPer; ++j) {
            const bool p = (on >> j) & 1u;
            const uint64_t m = __ballot(p);
            if (p) {
                const int o = at + __builtin_popcountll(m & ((1ull << lane) - 1ull));
                L.d[o] = v[j];
                L.i[o] = id[j];
            }
            at += __builtin_popcountll(m);
        }
    }
    __syncthreads();
    if (!JOIN && parts > 1) {
        float* at = row + c0;
        for (int e = tid; e < E; e += kStBlock) {
            at[e] = L.d[e];
            reinterpret_cast<int*>(at + E)[e] = L.i[e];
        }
        return;
    }
    // sort the E best by (distance, index)
    if (E <= 64) {
        if (tid >= 64) return;
        float d = lane < E ? L.d[lane] : pad_d();
        int id = lane < E ? L.i[lane] : INT32_MAX;
        wave_sort(d, id);
        if (lane < E) {
            oi[lane] = id;
            if (od) od[lane] = d;
        }
        return;
    }
    int n = 128;
    while (n < E) n <<= 1;                      // n <= 2048 < kStBuf
    for (int i = E + tid; i < n; i += kStBlock) { L.d[i] = pad_d(); L.i[i] = INT32_MAX; }
    __syncthreads();
    for (int size = 2; size <= n; size <<= 1)
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int i = tid; i < n; i += kStBlock) {
                const int j = i ^ stride;
                if (j > i) {
                    const bool up = (i & size) == 0;
                    if (up != lt(L.d[i], L.i[i], L.d[j], L.i[j])) {
                        const float td = L.d[i]; L.d[i] = L.d[j]; L.d[j] = td;
                        const int ti = L.i[i]; L.i[i] = L.i[j]; L.i[j] = ti;
                    }
                }
            }
            __syncthreads();
        }
    for (int e = tid; e < E; e += kStBlock) {
        oi[e] = L.i[e];
        if (od) od[e] = L.d[e];
    }
}

__global__ __launch_bounds__(kStBlock, 4) void row_topk_stream(float* __restrict__ Dm, int64_t N,
                                                            int E, int parts,
                                                            int32_t* __restrict__ oi,
                                                            float* __restrict__ od) {
    const int64_t r = blockIdx.x / parts;
    const int part = (int)(blockIdx.x - r * parts);
    row_topk_body<false>(Dm + r * N, N, E, parts, part, oi + r * E, od ? od + r * E : nullptr);
}

__global__ __launch_bounds__(kStBlock, 4) void row_topk_join(float* __restrict__ Dm, int64_t N, int E,
                                                          int parts, int32_t* __restrict__ oi,
                                                          float* __restrict__ od) {
    const int64_t r = blockIdx.x;
    row_topk_body<true>(Dm + r * N, N, E, parts, 0, oi + r * E, od ? od + r * E : nullptr);
}

// Parts a row of the streaming top-E is read in: enough workgroups for a few
// on every CU, none shorter than 16,384 columns (eight steps).
constexpr int kShortPart = 16384;
static_assert(kShortPart >= 4 * (kTopBuf / 2), "a part holds its E best and their indices");
int topk_parts(int64_t nq, int64_t N) {
    int64_t p = (1536 + nq - 1) / nq;
    if (nq >= 512) p = 1;
    if (p > N / kShortPart) p = N / kShortPart;
    return (int)(p < 1 ? 1 : p > 64 ? 64 : p);
}

}  // namespace
}  // namespace swann

using namespace swann;

// ---- the fixed workspace of swann_select_nearest_noalloc -------------------
// One array per GPU in the library's own device memory, reserved when the
// code object loads on that device and held until the process ends, so the
// no-alloc entry point never calls an allocator.  In host code `scratch` only
// names the symbol; its address on a device comes from hipGetSymbolAddress,
// looked up once per device (with that device current) and cached.
constexpr int64_t kScratchBytes = SWANN_SELECT_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::atomic<void*> g_scratch[kMaxDevices];
std::mutex g_scratch_mu;

int scratch_address(void** out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        set_error("select (no-alloc): hipGetDevice failed: %s", hipGetErrorString(e));
        return SWANN_E_NODEVICE;
    }
    if (dev < 0 || dev >= kMaxDevices) {
        set_error("select (no-alloc): device %d out of range", dev);
        return SWANN_E_UNSUPPORTED;
    }
    void* p = g_scratch[dev].load(std::memory_order_acquire);
    if (!p) {
        std::lock_guard<std::mutex> lock(g_scratch_mu);
        p = g_scratch[dev].load(std::memory_order_relaxed);
        if (!p) {
            e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
            if (e != hipSuccess || !p) {
                set_error("select (no-alloc): hipGetSymbolAddress(scratch) failed on device %d: %s",
                          dev, hipGetErrorString(e));
                return SWANN_E_LAUNCH;
            }
            g_scratch[dev].store(p, std::memory_order_release);
        }
    }
    *out = p;
    return SWANN_OK;
}
}  // namespace

// The distance matrix of a small batch: one pass over the catalogue.
static int gemv_run(const float* Q, int64_t nq, int dim, const float* Vp, int64_t P, int metric,
                    const float* qn, float* Dm, hipStream_t st) {
    const dim3 g((unsigned)((P + kGvRows * kGvWaves - 1) / (kGvRows * kGvWaves)));
    const dim3 b(kGvWaves * 64);
    const int q = (int)nq;
    if (nq == 1) hipLaunchKernelGGL(dist_gemv<1>, g, b, 0, st, Q, Vp, q, P, dim, metric, qn, Dm);
    else if (nq == 2) hipLaunchKernelGGL(dist_gemv<2>, g, b, 0, st, Q, Vp, q, P, dim, metric, qn, Dm);
    else if (nq <= 4) hipLaunchKernelGGL(dist_gemv<4>, g, b, 0, st, Q, Vp, q, P, dim, metric, qn, Dm);
    else hipLaunchKernelGGL(dist_gemv<8>, g, b, 0, st, Q, Vp, q, P, dim, metric, qn, Dm);
    return launch_status("select gemv");
}

// The distance matrix of a larger batch, K split when the tiles alone would not fill
// the chip.  128 x 128 tiles once they give every CU two workgroups, where they
// multiply at most a sixteenth more rows of padding than 64 x 64 tiles do and the
// rows allow 16-byte loads.  Whole selections, 128 to 64 tiles in ms, against 400,003
// x 768: 9 queries 0.78 to 0.46, 64 0.83 to 0.51, 100 0.853 to 0.855, 160 1.51 to
// 1.20, 256 1.59 to 1.61, 500 2.91 to 2.99, 1,000 5.51 to 5.84; element loads (131,072
// x 99): 64 0.177 to 0.130, 256 0.303 to 0.263, 1,000 0.90 to 0.71.
static int gemm_run(const float* Q, int64_t nq, int dim, const float* Vp, int64_t P, int metric,
                    const float* qn, float* vn, float* Dm, hipStream_t st) {
    if (metric == SWANN_METRIC_L2)
        hipLaunchKernelGGL(row_norms, dim3((unsigned)((P + 3) / 4)), dim3(256), 0, st, Vp, P, dim,
                           vn);
    const int64_t tiles = ((P + kTN - 1) / kTN) * ((nq + kTM - 1) / kTM);
    int S = split_for(tiles);
    int kper = dim;
    if (S > 1) {
        kper = (dim + S - 1) / S;
        kper = ((kper + 15) / 16) * 16;
        S = (dim + kper - 1) / kper;
    }
    float* out = Dm;
    if (S > 1) out = (float*)((char*)vn + ((P * 4 + 255) / 256) * 256);
    else kper = dim;
    const bool vec = dim % 4 == 0 && (uintptr_t)Q % 16 == 0 && (uintptr_t)Vp % 16 == 0;
    const int64_t b64 = (nq + 63) / 64, b128 = (nq + 127) / 128;
    const bool big = vec && ((P + 127) / 128) * b128 >= 512 && 32 * b128 <= 17 * b64;
    const int T = big ? 128 : 64;
    const dim3 grid((unsigned)(((P + T - 1) / T) * ((nq + T - 1) / T)), 1, (unsigned)S);
    auto* kernel = big ? dist_gemm<128, true> : vec ? dist_gemm<64, true> : dist_gemm<64, false>;
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, Q, Vp, nq, P, dim, metric, qn, vn, out,
                       kper);
    if (S > 1)
        hipLaunchKernelGGL(split_finish, dim3((unsigned)((nq * P + 255) / 256)), dim3(256), 0, st,
                           out, S, nq, P, metric, qn, vn, Dm);
    return launch_status("select gemm");
}

static int select_run(const float* Q, int64_t nq, int dim, const float* Vp, int64_t P, int E,
                      int metric, int32_t* out_idx, float* out_dist, void* workspace,
                      void* stream) {
    SWANN_REQUIRE(metric == SWANN_METRIC_IP || metric == SWANN_METRIC_L2,
                  "metric must be 0 (ip) or 1 (l2)");
    SWANN_REQUIRE(nq >= 0 && P >= 1 && dim >= 1, "select: need nq >= 0, P >= 1, dim >= 1");
    SWANN_REQUIRE(E >= 1 && E <= kTopBuf / 2, "select: E must be in 1..%d", kTopBuf / 2);
    SWANN_REQUIRE(E <= P, "select: E (%d) exceeds the catalogue size (%lld)", E, (long long)P);
    SWANN_REQUIRE(nq <= INT32_MAX && (P + kTN - 1) / kTN <= INT32_MAX &&
                      (nq + kTM - 1) / kTM <= 65535,
                  "select: batch of %lld queries too large for one call", (long long)nq);
    if (nq == 0) return SWANN_OK;
    SWANN_REQUIRE(Q && Vp && out_idx && workspace, "select: a required pointer is NULL");
    hipStream_t st = (hipStream_t)stream;
    char* ws = (char*)workspace;
    float* Dm = (float*)ws;
    float* qn = (float*)(ws + ((nq * P * 4 + 255) / 256) * 256);
    float* vn = (float*)((char*)qn + ((nq * 4 + 255) / 256) * 256);
    if (metric == SWANN_METRIC_L2)
        hipLaunchKernelGGL(row_norms, dim3((unsigned)((nq + 3) / 4)), dim3(256), 0, st, Q, nq, dim,
                           qn);
    const int rc = nq <= kGvMaxQ ? gemv_run(Q, nq, dim, Vp, P, metric, qn, Dm, st)
                                 : gemm_run(Q, nq, dim, Vp, P, metric, qn, vn, Dm, st);
    if (rc) return rc;
    if (P <= (int64_t)kRadBlock * kRadPer && E <= kRadMaxE)
        hipLaunchKernelGGL(row_topk_radix, dim3((unsigned)nq), dim3(kRadBlock), 0, st, Dm, P, E,
                           out_idx, out_dist);
    else {
        const int parts = topk_parts(nq, P);
        hipLaunchKernelGGL(row_topk_stream, dim3((unsigned)(nq * parts)), dim3(kStBlock), 0, st,
                           Dm, P, E, parts, out_idx, out_dist);
        if (parts > 1)
            hipLaunchKernelGGL(row_topk_join, dim3((unsigned)nq), dim3(kStBlock), 0, st, Dm, P, E,
                               parts, out_idx, out_dist);
    }
    return launch_status("select top-E");
}


extern "C" {

int64_t swann_select_workspace_size(int64_t nq, int64_t P) {
    // distance matrix + both norm vectors + (small batches) the split-K
    // partials, each 256-byte aligned
    const int64_t a = ((nq * P * 4 + 255) / 256) * 256;
    const int64_t b = ((nq * 4 + 255) / 256) * 256;
    const int64_t c = ((P * 4 + 255) / 256) * 256;
    const int S = split_for(((P + kTN - 1) / kTN) * ((nq + kTM - 1) / kTM));
    const int64_t d = S > 1 ? (int64_t)S * a : 0;
    return a + b + c + d;
}

int swann_select_nearest(const float* Q, int64_t nq, int dim, const float* Vp, int64_t P, int E,
                         int metric, int32_t* out_idx, float* out_dist, void* workspace,
                         void* stream) {
    clear_error();
    return select_run(Q, nq, dim, Vp, P, E, metric, out_idx, out_dist, workspace, stream);
}

int swann_select_nearest_noalloc(const float* Q, int64_t nq, int dim, const float* Vp, int64_t P,
                                 int E, int metric, int32_t* out_idx, float* out_dist,
                                 void* stream) {
    clear_error();
    SWANN_REQUIRE(nq >= 0 && P >= 1, "select: need nq >= 0, P >= 1");
    const int64_t need = swann_select_workspace_size(nq, P);
    SWANN_REQUIRE(need <= kScratchBytes,
                  "select (no-alloc): %lld queries x %lld catalogue rows need %lld bytes of "
                  "workspace; the built-in scratch holds %lld (use swann_select_nearest with a "
                  "workspace of swann_select_workspace_size bytes)",
                  (long long)nq, (long long)P, (long long)need, (long long)kScratchBytes);
    if (nq == 0) return select_run(Q, nq, dim, Vp, P, E, metric, out_idx, out_dist, nullptr,
                                   stream);
    void* ws = nullptr;
    const int rc = scratch_address(&ws);
    if (rc) return rc;
    return select_run(Q, nq, dim, Vp, P, E, metric, out_idx, out_dist, ws, stream);
}

}  // extern "C"
