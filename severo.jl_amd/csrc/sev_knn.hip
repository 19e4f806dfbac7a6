// Exact Euclidean k-nearest neighbours (brute force, bit-exact definition).
//
// Replaces the native FindNeighboursEuclidean32/64 called from
// src/neighbours.jl:32-63 (which the reference backs with an approximate
// multi-table search).  Here the neighbours are exact under a stated order of
// operations, so every implementation of the definition agrees bit for bit:
//   D(i,j) = sum_{t=0}^{d-1} (x_it - x_jt)^2, each difference and square
//            rounded in T, accumulated in t order, no FMA;
//   ranking by (D, j) lexicographically (lower index wins ties, the order of
//   the reference test's partialsortperm, test/test_nn.jl:33);
//   j == i skipped only when include_self == 0; distance = sqrt(D).
//
// One block handles kQB queries; every thread owns one candidate of a
// 256-candidate tile and computes its distance to all kQB queries (query
// coordinates broadcast from LDS, candidate coordinates read coalesced from
// the column-major X).  Candidates below a query's current k-th distance are
// appended to that query's LDS pending list; after each tile one wavefront
// per query merges the pending entries into a sorted list held one entry per
// lane (insertion by ballot + shift).
//
// The thresholds start from a first sweep over the head of the candidates
// (all of them up to kHeadTiles tiles, 4 tiles of a large search): every thread keeps its smallest distance to each query,
// the k-th smallest of the 64 lanes' minima is reached by k candidates, so
// only candidates up to that value are appended.  Without it the whole first
// tile is merged entry by entry, 256 serial steps per query, which took most
// of a small search: 2,003 x 15, k = 10: 0.27 ms, now 0.08; 5,000 x 50, k = 20:
// 0.69 ms, now 0.41.  Bound then: VALU (3 operations per coordinate pair).
#include "sev_kernels.hpp"

#include <algorithm>
#include <cfloat>
#include <climits>
#include <type_traits>

namespace sev {

namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / kWave;

template <class T>
__device__ __forceinline__ T inf_val();
template <>
__device__ __forceinline__ float inf_val<float>() {
    return __builtin_huge_valf();
}
template <>
__device__ __forceinline__ double inf_val<double>() {
    return __builtin_huge_val();
}

// the next value above a distance (+0 or positive; infinity stays)
__device__ __forceinline__ float next_up(float v) {
    return v < inf_val<float>() ? __uint_as_float(__float_as_uint(v) + 1u) : v;
}
__device__ __forceinline__ double next_up(double v) {
    return v < inf_val<double>() ? __longlong_as_double(__double_as_longlong(v) + 1ll) : v;
}

constexpr int kHeadTiles = 16;

template <class T, int kQB>
__global__ void __launch_bounds__(kBlock)
k_knn_exact(const T *X, int64_t n, int64_t d, int64_t ld, int k, int include_self,
            const int64_t *qidx, int64_t nq, int scatter, int32_t *oidx, T *odist,
            const int64_t *seg, const int32_t *row_sample) {
    extern __shared__ unsigned char smem_raw[];
    T *qx = (T *)smem_raw;  // kQB * d
    __shared__ T pendD[kQB][kBlock];
    __shared__ int32_t pendJ[kQB][kBlock];
    __shared__ int pendN[kQB];
    __shared__ T listD[kQB][kMaxK];
    __shared__ int32_t listJ[kQB][kMaxK];
    __shared__ int listN[kQB];
    __shared__ T thr[kQB];
    __shared__ int64_t qrow[kQB];

    const int64_t q0 = (int64_t)blockIdx.x * kQB;
    const int nqb = (int)((nq - q0) < kQB ? (nq - q0) : kQB);
    if (threadIdx.x < kQB) {
        const int q = threadIdx.x;
        qrow[q] = q < nqb ? (qidx ? qidx[q0 + q] : q0 + q) : -1;
        pendN[q] = 0;
        listN[q] = 0;
        thr[q] = inf_val<T>();
    }
    __syncthreads();
    for (int64_t e = threadIdx.x; e < (int64_t)kQB * d; e += kBlock) {
        const int q = (int)(e / d);
        const int64_t t = e % d;
        qx[e] = q < nqb ? X[t * ld + qrow[q]] : T(0);
    }
    __syncthreads();

    // candidates: all n points, or (batches) the rows of the sample of the
    // block's first query -- every query of a block is from that sample
    int64_t cb = 0, ce = n;
    if (seg) {
        const int32_t s = row_sample[qrow[0]];
        cb = seg[s];
        ce = seg[s + 1];
    }
    const int lane = lane_id(), w = threadIdx.x / kWave;
    if (k < kWave) {
        // the whole of a small search; fewer tiles the more there are
        const int64_t nt = (ce - cb + kBlock - 1) / kBlock;
        const int64_t ht = nt <= kHeadTiles ? nt : (kHeadTiles * kHeadTiles / nt > 4
                                                        ? kHeadTiles * kHeadTiles / nt
                                                        : 4);
        const int64_t he = cb + ht * kBlock < ce ? cb + ht * kBlock : ce;
        T mn[kQB];
#pragma unroll
        for (int q = 0; q < kQB; ++q) mn[q] = inf_val<T>();
        for (int64_t j = cb + threadIdx.x; j < he; j += kBlock) {
            T D[kQB];
#pragma unroll
            for (int q = 0; q < kQB; ++q) D[q] = T(0);
            for (int64_t t = 0; t < d; ++t) {
                const T xj = X[t * ld + j];
#pragma unroll
                for (int q = 0; q < kQB; ++q) {
                    const T diff = qx[q * d + t] - xj;
                    D[q] = D[q] + diff * diff;
                }
            }
#pragma unroll
            for (int q = 0; q < kQB; ++q)
                if (D[q] < mn[q] && (include_self || j != qrow[q])) mn[q] = D[q];
        }
#pragma unroll
        for (int q = 0; q < kQB; ++q) pendD[q][threadIdx.x] = mn[q];
        __syncthreads();
        for (int q = w; q < nqb; q += kWaves) {
            T v = pendD[q][lane];
            for (int u = 1; u < kWaves; ++u) {
                const T o = pendD[q][lane + u * kWave];
                v = o < v ? o : v;
            }
            for (int size = 2; size <= kWave; size <<= 1)
                for (int stride = size >> 1; stride > 0; stride >>= 1) {
                    const T o = __shfl_xor(v, stride, kWave);
                    const bool up = (lane & size) == 0, lower = (lane & stride) == 0;
                    if ((lower == up) ? o < v : v < o) v = o;
                }
            v = __shfl(v, k - 1, kWave);
            if (lane == 0) thr[q] = next_up(v);  // candidates at the bound itself pass
        }
        __syncthreads();
    }
    for (int64_t tile = cb; tile < ce; tile += kBlock) {
        const int64_t j = tile + threadIdx.x;
        if (j < ce) {
            T D[kQB];
#pragma unroll
            for (int q = 0; q < kQB; ++q) D[q] = T(0);
            for (int64_t t = 0; t < d; ++t) {
                const T xj = X[t * ld + j];
#pragma unroll
                for (int q = 0; q < kQB; ++q) {
                    const T diff = qx[q * d + t] - xj;
                    D[q] = D[q] + diff * diff;
                }
            }
#pragma unroll
            for (int q = 0; q < kQB; ++q) {
                if (q < nqb && D[q] < thr[q] && (include_self || j != qrow[q])) {
                    const int pos = atomicAdd(&pendN[q], 1);
                    pendD[q][pos] = D[q];
                    pendJ[q][pos] = (int32_t)j;
                }
            }
        }
        __syncthreads();
        for (int q = w; q < nqb; q += kWaves) {
            const int P = pendN[q];
            if (P == 0) continue;
            int cnt = listN[q];
            T ld_ = lane < cnt ? listD[q][lane] : inf_val<T>();
            int32_t lj = lane < cnt ? listJ[q][lane] : INT_MAX;
            for (int e = 0; e < P; ++e) {
                const T Dn = pendD[q][e];
                const int32_t jn = pendJ[q][e];
                const bool less = lane < cnt && (ld_ < Dn || (ld_ == Dn && lj < jn));
                const int pos = __popcll(__ballot(less));
                const T upD = __shfl_up(ld_, 1, kWave);
                const int32_t upJ = __shfl_up(lj, 1, kWave);
                if (pos < k) {
                    if (lane == pos) {
                        ld_ = Dn;
                        lj = jn;
                    } else if (lane > pos) {
                        ld_ = upD;
                        lj = upJ;
                    }
                    cnt = cnt + 1 < k ? cnt + 1 : k;
                }
            }
            if (lane < kMaxK) {
                listD[q][lane] = ld_;
                listJ[q][lane] = lj;
            }
            const T kth = __shfl(ld_, k - 1, kWave);
            if (lane == 0) {
                listN[q] = cnt;
                if (cnt == k) thr[q] = kth;
                pendN[q] = 0;
            }
        }
        __syncthreads();
    }
    for (int q = w; q < nqb; q += kWaves) {
        const int cnt = listN[q];
        if (lane < k) {
            const int64_t r = scatter ? qrow[q] : q0 + q;
            oidx[r * k + lane] = lane < cnt ? listJ[q][lane] : -1;
            odist[r * k + lane] = lane < cnt ? sqrt(listD[q][lane]) : inf_val<T>();
        }
    }
}

}  // namespace

template <class T>
void knn_exact_impl(const T *X, int64_t n, int64_t d, int64_t ld, int64_t k, int include_self,
                    const int64_t *qidx, int64_t nq, int scatter, int32_t *idx, T *dist,
                    hipStream_t st, const int64_t *seg = nullptr,
                    const int32_t *row_sample = nullptr) {
    SEV_REQUIRE(k >= 1 && k <= kMaxK, "knn: k must be in [1, 64]");
    SEV_REQUIRE(d >= 1, "knn: d must be >= 1");
    // 16 queries per block in FP32, 8 in FP64 (keeps LDS under 64 KB)
    constexpr int QB = sizeof(T) == 4 ? 16 : 8;
    SEV_REQUIRE(sizeof(T) * (size_t)QB * (size_t)d <= 16384,
                "knn: too many dimensions for the exact kernel");
    if (nq == 0) return;
    ProfScope ps("knn_exact", st, 0.0, 2.0 * (double)nq * (double)n * (double)d);
    auto go = [&](auto qb) {
        constexpr int B = decltype(qb)::value;
        hipLaunchKernelGGL((k_knn_exact<T, B>), dim3((unsigned)ceil_div(nq, B)), dim3(kBlock),
                           sizeof(T) * (size_t)B * (size_t)d, st, X, n, d, ld, (int)k,
                           include_self, qidx, nq, scatter, idx, dist, seg, row_sample);
    };
    // half the queries per block until that gives every compute unit 8 blocks:
    // twice the blocks and more of them resident (20,000 x 50: 4.2 -> 2.8 ms; a
    // batch's query blocks are cut at 16 rows, a multiple of both)
    if (ceil_div(nq, (int64_t)QB) < 8 * device_cu_count())
        go(std::integral_constant<int, QB / 2>());
    else
        go(std::integral_constant<int, QB>());
    SEV_LAUNCH_CHECK();
}

template <class T>
void knn_exact(const T *X, int64_t n, int64_t d, int64_t ld, int64_t k, int include_self,
               const int64_t *qidx, int64_t nq, int32_t *idx, T *dist, hipStream_t st) {
    knn_exact_impl<T>(X, n, d, ld, k, include_self, qidx, nq, 0, idx, dist, st);
}

template <class T>
void knn_exact_rows(const T *X, int64_t n, int64_t d, int64_t ld, int64_t k, int include_self,
                    const int64_t *qidx, int64_t nq, int32_t *idx, T *dist, hipStream_t st) {
    SEV_REQUIRE(qidx != nullptr, "knn_exact_rows needs row indices");
    knn_exact_impl<T>(X, n, d, ld, k, include_self, qidx, nq, 1, idx, dist, st);
}

void knn_exact_rows_batch(const float *X, int64_t n, int64_t d, int64_t ld, int64_t k,
                          int include_self, const int64_t *qidx, int64_t nq, const int64_t *seg,
                          const int32_t *row_sample, int32_t *idx, float *dist, hipStream_t st) {
    SEV_REQUIRE(qidx != nullptr && seg != nullptr, "knn_exact_rows_batch needs rows and samples");
    knn_exact_impl<float>(X, n, d, ld, k, include_self, qidx, nq, 1, idx, dist, st, seg,
                          row_sample);
}

// --------------------------------------------------------------------------
// Cosine neighbours (the CosineDist form of src/neighbours.jl:41-50 and
// :63-72).  Each row is scaled to unit length in T (sum of squares in t
// order, IEEE sqrt and division; an all-zero row stays zero); the exact
// Euclidean search then runs on the unit rows, whose D ranks pairs as
// 1 - cos does in exact arithmetic; the reported distance is D / 2, with D
// recomputed for the found pairs by the same definition.
// --------------------------------------------------------------------------
namespace {

template <class T>
__global__ void __launch_bounds__(kBlock)
k_unit_rows(T *X, int64_t n, int64_t d) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * kBlock) {
        T s = 0;
        for (int64_t t = 0; t < d; ++t) {
            const T v = X[t * n + i];
            s = s + v * v;
        }
        if (s > T(0)) {
            const T nrm = sqrt(s);
            for (int64_t t = 0; t < d; ++t) X[t * n + i] = X[t * n + i] / nrm;
        }
    }
}

template <class T>
__global__ void __launch_bounds__(kBlock)
k_half_pair_dist(const T *X, int64_t n, int64_t d, const int32_t *idx, int64_t k, T *dist) {
    for (int64_t p = (int64_t)blockIdx.x * kBlock + threadIdx.x; p < n * k;
         p += (int64_t)gridDim.x * kBlock) {
        const int64_t i = p / k;
        const int32_t j = idx[p];
        if (j < 0 || j >= n) continue;
        T D = 0;
        for (int64_t t = 0; t < d; ++t) {
            const T diff = X[t * n + i] - X[t * n + j];
            D = D + diff * diff;
        }
        dist[p] = T(0.5) * D;
    }
}

unsigned rows_grid(int64_t n) {
    const int64_t g = ceil_div(n > 0 ? n : 1, (int64_t)kBlock);
    return (unsigned)std::min<int64_t>(g, (int64_t)device_cu_count() * 16);
}

}  // namespace

template <class T>
void knn_unit_rows(T *X, int64_t n, int64_t d, hipStream_t st) {
    hipLaunchKernelGGL(k_unit_rows<T>, dim3(rows_grid(n)), dim3(kBlock), 0, st, X, n, d);
    SEV_LAUNCH_CHECK();
}

template <class T>
void knn_half_pair_dist(const T *X, int64_t n, int64_t d, const int32_t *idx, int64_t k, T *dist,
                        hipStream_t st) {
    hipLaunchKernelGGL(k_half_pair_dist<T>, dim3(rows_grid(n * k)), dim3(kBlock), 0, st, X, n, d,
                       idx, k, dist);
    SEV_LAUNCH_CHECK();
}

template void knn_unit_rows<float>(float *, int64_t, int64_t, hipStream_t);
template void knn_unit_rows<double>(double *, int64_t, int64_t, hipStream_t);
template void knn_half_pair_dist<float>(const float *, int64_t, int64_t, const int32_t *, int64_t,
                                        float *, hipStream_t);
template void knn_half_pair_dist<double>(const double *, int64_t, int64_t, const int32_t *,
                                         int64_t, double *, hipStream_t);

template void knn_exact<float>(const float *, int64_t, int64_t, int64_t, int64_t, int,
                               const int64_t *, int64_t, int32_t *, float *, hipStream_t);
template void knn_exact<double>(const double *, int64_t, int64_t, int64_t, int64_t, int,
                                const int64_t *, int64_t, int32_t *, double *, hipStream_t);
template void knn_exact_rows<float>(const float *, int64_t, int64_t, int64_t, int64_t, int,
                                    const int64_t *, int64_t, int32_t *, float *, hipStream_t);
template void knn_exact_rows<double>(const double *, int64_t, int64_t, int64_t, int64_t, int,
                                     const int64_t *, int64_t, int32_t *, double *, hipStream_t);

}  // namespace sev
