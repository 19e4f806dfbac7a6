// Exact kNN over cells of nearby points.
//
// The result is that of knn_exact (sev_knn.hip), as for the candidate search
// of sev_knn_mfma.hip, whose re-rank and certificate are used.  The search
// itself differs in three ways.
//
// Cells.  The points are sorted by their nearest of M centroids (two Lloyd
// steps on a sample, then ordered so that neighbouring centroids are close),
// each cell padded to whole groups of kGrp slots.  A group's points lie in the
// ball of radius r_b around their mean b.  A query block is one group, so its
// queries want the same candidates: it skips every group that the triangle
// inequality puts beyond the k-th neighbour of all of its queries.  On an
// embedding of clusters that leaves the query's own cluster and the close
// ones: 7% of the groups at 1,000,000 x 50 with 40 clusters, 11% at 100,000
// with 24 (40% with sampled points as centroids, which miss small clusters).
//
// Operands.  z is taken around the mean of a sample (the error of a score goes
// with the norms: 100,000 x 50, 300 from the origin, 24 groups, FP32: 70 ms, most
// rows without a certificate; now 2.1), scaled by a power of two (largest |z|^2 in
// (2^12, 2^14]) and rounded to FP16, relative error 2^-11 where BF16 has 2^-8, at
// the same rate:
// with BF16 the rounding exceeds the gap between the k-th neighbour and the
// end of the list wherever clusters lie far from the origin, and nearly every
// row lost its certificate (1,000,000 x 50, 40 clusters: a first pass of 251 ms,
// then 263 ms for the rows left).  The FP32 form splits z into two FP16 parts
// h + l (2^-22) and takes q.c as h.h' + l.h' + h.l': three products at a sixth of
// the time of one on the FP32 matrix instruction.  FP16 parts below the
// normal range are taken as zero, so their treatment by the MFMA does not
// matter.
//
// Measured, k = 20: 1,000,000 x 50, 40 clusters, one part: 526 -> 73 ms (65 of
// them k_knn_cell); 100,000 x 50, 24 clusters, two parts: 27.3 -> 3.6 ms; 20,000 x
// 50, 12 clusters: 4.9 -> 0.86.  Without clusters nothing is skipped and the two
// sweeps cost more than the one with insertion (1,000,000 Gaussian points: 165
// ms by sev_knn_mfma.hip), so the 16-bit form keeps that search there; the FP32
// form is faster this way in either case.
//
// Two sweeps and no insertion.  The largest score of each of the 64 residues
// of the tile position is kept in registers over a sweep; the r-th largest of
// the 64 is reached by r candidates.  A sweep over the nearest groups in slot
// order bounds the k-th neighbour (for the skip), a sweep over the groups left
// gives the final threshold, and a second one appends what exceeds it: about
// 64 ln(64 / (64 - r)) candidates, 40 at r = 30 for k = 20.  Sorted insertion of each
// passing pair, one at a time, had cost more than the products.
//
// A block holds 128 queries (4 wavefronts of 32) and 64-candidate tiles in
// two LDS buffers: 80 KB at KP = 160, so two blocks share a compute unit, three
// at KP <= 64.  Bound: the chain of a tile (rows from beyond L2, LDS, matrix
// instructions, maxima), 1.3 us per tile and block at KP = 160, 0.27 us of them
// MFMA; no unit is full (1,000,000 x 50: matrix cores 15% busy, VALU 37%, 72% of
// the L2 requests missing, at 2.1 TB/s).
#include "sev_kernels.hpp"

#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <climits>
#include <cmath>
#include <type_traits>
#include <vector>

namespace sev {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

constexpr int kBlock = 256;
constexpr int kNW = kBlock / kWave;
constexpr int kCT = 64;           // candidates per tile
constexpr int kGrp = 128;         // slots per group, queries per block
constexpr int kQW = 2;            // 16-query row blocks per wavefront
constexpr int kCap = 64;          // candidates kept per query
constexpr int kWindow = 32;       // groups of the first sweep
constexpr int kMaxGroups = 32768; // bits of the needed-group mask (4 KB of LDS)
constexpr int kMaxPivots = 512;
constexpr int kPivLd = 64;        // floats per pivot row (zero padded)
constexpr int kSample = 16384;    // points of the Lloyd steps
constexpr int kTestPivots = 1024; // structure test: pivots and queries
constexpr int kTestQueries = 256;
// Bound of the error of nq - 2 s from the norm's three parts: a part below 2^-14
// is taken as zero, once (2^-13), whatever the scale.  It matters where the scale
// stops at 2^60 (largest |z| below 2e-18) and the relative terms vanish.
constexpr double kNormErr = 0x1p-12;

// FP16 bits of x, 0 below the normal range
__device__ __forceinline__ uint16_t f2h(float x) {
    const _Float16 h = (_Float16)x;
    return fabsf((float)h) < 6.103515625e-5f ? (uint16_t)0 : __builtin_bit_cast(uint16_t, h);
}
__device__ __forceinline__ float h2f(uint16_t h) { return (float)__builtin_bit_cast(_Float16, h); }
__device__ __forceinline__ float ninf() { return -__builtin_huge_valf(); }

// the power of two that brings the largest |z|^2 (float bits n2) into
// (2^12, 2^14]
__device__ __forceinline__ float point_scale(unsigned n2) {
    const float v = __uint_as_float(n2);
    if (!(v > 0.0f) || !(v < 1e38f)) return 1.0f;
    int x;
    (void)frexpf(v, &x);
    const int e = (14 - x) >> 1;
    return ldexpf(1.0f, e > 60 ? 60 : (e < -60 ? -60 : e));
}

// cen[t] = mean of coordinate t over sampled points (0 if not finite), one block
// per coordinate; gmax[0..3] = 0.
template <class T>
__global__ void __launch_bounds__(kBlock)
k_cell_centre(const T *Z, int64_t n, int64_t ld, float *cen, unsigned *gmax) {
    __shared__ double part[kNW];
    const int t = blockIdx.x;
    if (t == 0 && threadIdx.x < 4) gmax[threadIdx.x] = 0u;
    double a = 0.0;
#pragma unroll
    for (int u = 0; u < kTestPivots / kBlock; ++u)
        a += (double)Z[t * ld + (int64_t)(threadIdx.x + u * kBlock) * n / kTestPivots];
    a = wave_sum(a);
    if (threadIdx.x % kWave == 0) part[threadIdx.x / kWave] = a;
    __syncthreads();
    if (threadIdx.x != 0) return;
    const float m = (float)((part[0] + part[1] + part[2] + part[3]) / kTestPivots);
    cen[t] = fabsf(m) < __builtin_huge_valf() ? m : 0.0f;
}

// z - cen rounded to FP32
__device__ __forceinline__ float centred(float z, float c) { return z - c; }
__device__ __forceinline__ float centred(double z, float c) { return (float)(z - (double)c); }

// Zr[i*d + t] = Z[t*ld + i], 64 points per block through LDS; n2 = max |z - cen|^2
template <class T>
__global__ void __launch_bounds__(kBlock)
k_cell_rows(const T *Z, int64_t n, int d, int64_t ld, const float *cen, T *Zr, unsigned *n2) {
    __shared__ T s[kWave * 65];
    __shared__ float nn[kNW][kWave];
    const int64_t i0 = (int64_t)blockIdx.x * kWave;
    const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
    const int nr = (int)(n - i0 < kWave ? n - i0 : kWave);
    float a = 0.0f;
    for (int t = w; t < d; t += kNW)
        if (lane < nr) {
            const T z = Z[(int64_t)t * ld + i0 + lane];
            s[lane * (d + 1) + t] = z;
            const float zc = centred(z, cen[t]);
            a = fmaf(zc, zc, a);
        }
    nn[w][lane] = a;
    __syncthreads();
    for (int e = threadIdx.x; e < nr * d; e += kBlock)
        Zr[i0 * d + e] = s[(e / d) * (d + 1) + e % d];
    if (w == 0) {
        unsigned b = __float_as_uint(nn[0][lane] + nn[1][lane] + nn[2][lane] + nn[3][lane]);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) b = max(b, (unsigned)__shfl_xor((int)b, o, kWave));
        if (lane == 0) atomicMax(n2, b);
    }
}

// piv[m*kPivLd + t] = centred coordinates of the point (m * n) / M, zero padded
template <class T>
__global__ void __launch_bounds__(kBlock)
k_cell_pivots(const T *Zr, const float *cen, int64_t n, int d, int M, float *piv) {
    for (int e = blockIdx.x * kBlock + threadIdx.x; e < M * kPivLd; e += gridDim.x * kBlock) {
        const int m = e / kPivLd, t = e % kPivLd;
        piv[e] = t < d ? centred(Zr[((int64_t)m * n / M) * d + t], cen[t]) : 0.0f;
    }
}

// S[t*ns + i] = coordinates of the point (i * n) / ns (less cen, if given);
// coordinate t of point j at X[j*ri + t*rt].  *zero (if given) is set to 0.
template <class T>
__global__ void __launch_bounds__(kBlock)
k_cell_sample(const T *X, int64_t ri, int64_t rt, const float *cen, int64_t n, int d, int ns,
              float *S, int *zero) {
    if (zero && blockIdx.x == 0 && threadIdx.x == 0) *zero = 0;
    for (int e = blockIdx.x * kBlock + threadIdx.x; e < ns * d; e += gridDim.x * kBlock) {
        const int t = e / ns, i = e % ns;
        S[e] = centred(X[((int64_t)i * n / ns) * ri + t * rt], cen ? cen[t] : 0.0f);
    }
}

__global__ void __launch_bounds__(kBlock) k_cell_half(const float *piv, int M, float *half) {
    const int m = blockIdx.x * kBlock + threadIdx.x;
    if (m >= M) return;
    float h = 0.0f;
    for (int t = 0; t < kPivLd; ++t) h = fmaf(piv[m * kPivLd + t], piv[m * kPivLd + t], h);
    half[m] = 0.5f * h;
}

// Mean of the sample points of each cell (an empty one keeps its pivot): one
// block per pivot, each wavefront a quarter of the sample, in order.
__global__ void __launch_bounds__(kBlock)
k_cell_means(const float *S, int ns, int d, const uint32_t *cell, float *piv, float *half) {
    __shared__ float acc[kNW][kWave];
    __shared__ int cnt[kNW];
    const int m = blockIdx.x, lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
    const int per = (ns + kNW - 1) / kNW;
    const int b = w * per, e = b + per < ns ? b + per : ns;
    float a = 0.0f;
    int c = 0;
    for (int i = b; i < e; i += kWave) {
        uint64_t mask = __ballot(i + lane < e && cell[i + lane] == (uint32_t)m);
        c += __popcll(mask);
        while (mask) {
            const int u = i + __builtin_ctzll(mask);
            mask &= mask - 1;
            if (lane < d) a += S[(int64_t)lane * ns + u];
        }
    }
    acc[w][lane] = a;
    if (lane == 0) cnt[w] = c;
    __syncthreads();
    if (w != 0) return;
    c = cnt[0] + cnt[1] + cnt[2] + cnt[3];
    if (c == 0) return;
    a = (acc[0][lane] + acc[1][lane] + acc[2][lane] + acc[3][lane]) / (float)c;
    a = lane < d ? a : 0.0f;
    piv[m * kPivLd + lane] = a;
    float h = a * a;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) h += __shfl_xor(h, o, kWave);
    if (lane == 0) half[m] = 0.5f * h;
}

// Structure test: the share of kTestPivots sampled points within 2.1 times
// the distance of the nearest one, for each of kTestQueries sampled queries.
// Within one Gaussian blob all distances are alike (a share near 1); among
// clusters the share is that of the query's own and the overlapping ones.
// It comes before anything else of this search, which points without clusters do
// not need, and its points lie coordinate by coordinate, one after the other for
// the lanes: 30 us of the 1.4 ms of such a search at 14,000 x 50 (60 after the
// rows, with a pivot's coordinates together).
template <class T>
__global__ void __launch_bounds__(kBlock)
k_cell_test(const T *Z, int64_t n, int d, int64_t ld, const float *S, int *share) {
    __shared__ float q[64];
    __shared__ float best[kNW];
    __shared__ int cnt;
    const int64_t i = ((int64_t)blockIdx.x * n) / kTestQueries + n / (2 * kTestQueries);
    if (threadIdx.x < d) q[threadIdx.x] = (float)Z[threadIdx.x * ld + (i < n ? i : n - 1)];
    if (threadIdx.x == 0) cnt = 0;
    __syncthreads();
    float D[kTestPivots / kBlock];
    float mn = __builtin_huge_valf();
#pragma unroll
    for (int u = 0; u < kTestPivots / kBlock; ++u) {
        const float *p = S + threadIdx.x + u * kBlock;
        float a = 0.0f;
        for (int t = 0; t < d; ++t) {
            const float x = q[t] - p[t * kTestPivots];
            a = fmaf(x, x, a);
        }
        D[u] = a;
        if (a > 0.0f) mn = fminf(mn, a);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mn = fminf(mn, __shfl_xor(mn, o, kWave));
    if (threadIdx.x % kWave == 0) best[threadIdx.x / kWave] = mn;
    __syncthreads();
    for (int u = 0; u < kNW; ++u) mn = fminf(mn, best[u]);
    int c = 0;
#pragma unroll
    for (int u = 0; u < kTestPivots / kBlock; ++u) c += !(D[u] > 4.4f * mn) ? 1 : 0;
    atomicAdd(&cnt, c);
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(share, cnt);
}

// Pivots put in the order of their nearest of up to 32 super-pivots, so that
// cells next to each other in slot order are close; one block.
__global__ void __launch_bounds__(kMaxPivots)
k_cell_order(const float *piv, const float *half, int M, int d, float *out, float *ohalf) {
    __shared__ float sp[32][kPivLd];
    __shared__ int key[kMaxPivots];
    const int m = threadIdx.x, ns = M >= 32 ? M / 16 : 1;
    for (int e = threadIdx.x; e < 32 * kPivLd; e += kMaxPivots) {
        const int s = e / kPivLd;
        sp[s][e % kPivLd] = s < ns ? piv[(s * M / ns) * kPivLd + e % kPivLd] : 0.0f;
    }
    __syncthreads();
    float a[32];
#pragma unroll
    for (int s = 0; s < 32; ++s) a[s] = 0.0f;
    if (m < M)
        for (int t = 0; t < d; ++t) {
            const float x = piv[m * kPivLd + t];
#pragma unroll
            for (int s = 0; s < 32; ++s) a[s] = fmaf(x - sp[s][t], x - sp[s][t], a[s]);
        }
    float bd = __builtin_huge_valf();
    int bs = 0;
#pragma unroll
    for (int s = 0; s < 32; ++s)
        if (s < ns && a[s] < bd) {
            bd = a[s];
            bs = s;
        }
    key[m] = m < M ? bs * kMaxPivots + m : INT_MAX;
    __syncthreads();
    if (m >= M) return;
    int r = 0;
    for (int u = 0; u < M; ++u) r += key[u] < key[m] ? 1 : 0;
    for (int t = 0; t < kPivLd; ++t) out[r * kPivLd + t] = piv[m * kPivLd + t];
    ohalf[r] = half[m];
}

// Nearest pivot of each point (any choice is correct: it only shapes the
// cells); counts per cell when asked for.  The pivots are read at uniform
// addresses, so they reach the FMAs as scalar operands.
template <int DP, class T>
__global__ void __launch_bounds__(kBlock)
k_cell_assign(const T *Z, int64_t n, int d, int64_t ld, const float *__restrict__ cen,
              const float *__restrict__ piv,
              const float *__restrict__ half, int M, uint32_t *cell, int32_t *id, int32_t *cnt) {
    __shared__ int lc[kMaxPivots];
    if (cnt)
        for (int m = threadIdx.x; m < M; m += kBlock) lc[m] = 0;
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    float z[DP];
#pragma unroll
    for (int t = 0; t < DP; ++t)
        z[t] = (t < d && i < n) ? -centred(Z[(int64_t)t * ld + i], cen ? cen[t] : 0.0f) : 0.0f;
    float best = __builtin_huge_valf();
    int bm = 0;
    for (int m = 0; m < M; ++m) {
        const float *p = piv + m * kPivLd;
        float a0 = half[m], a1 = 0.0f;
#pragma unroll
        for (int t = 0; t < DP; t += 2) {
            a0 = fmaf(z[t], p[t], a0);
            a1 = fmaf(z[t + 1], p[t + 1], a1);
        }
        const float a = a0 + a1;
        if (a < best) {
            best = a;
            bm = m;
        }
    }
    if (i < n) {
        cell[i] = (uint32_t)bm;
        if (id) id[i] = (int32_t)i;
    }
    if (!cnt) return;
    __syncthreads();
    if (i < n) atomicAdd(&lc[bm], 1);
    __syncthreads();
    for (int m = threadIdx.x; m < M; m += kBlock)
        if (lc[m]) atomicAdd(&cnt[m], lc[m]);
}

// First sorted position and first slot of each cell (one block); tot[0] =
// groups in use.
__global__ void __launch_bounds__(kMaxPivots)
k_cell_offsets(const int32_t *cnt, int M, int64_t *start, int64_t *off, int *tot) {
    __shared__ int64_t cs[2][kMaxPivots], gs[2][kMaxPivots];
    const int m = threadIdx.x;
    const int64_t c = m < M ? cnt[m] : 0, g = (c + kGrp - 1) / kGrp;
    cs[0][m] = c;
    gs[0][m] = g;
    __syncthreads();
    int b = 0;
    for (int o = 1; o < kMaxPivots; o <<= 1, b ^= 1) {
        cs[b ^ 1][m] = cs[b][m] + (m >= o ? cs[b][m - o] : 0);
        gs[b ^ 1][m] = gs[b][m] + (m >= o ? gs[b][m - o] : 0);
        __syncthreads();
    }
    if (m < M) {
        start[m] = cs[b][m] - c;
        off[m] = (gs[b][m] - g) * kGrp;
    }
    if (m == M - 1) tot[0] = (int)gs[b][m];
}

__global__ void __launch_bounds__(kBlock)
k_cell_slots(const uint32_t *scell, const int32_t *sid, int64_t n, const int64_t *start,
             const int64_t *off, int32_t *perm) {
    const int64_t p = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (p >= n) return;
    const uint32_t c = scell[p];
    perm[off[c] + p - start[c]] = sid[p];
}

// One block per group: rows in slot order (Zs), the operands, |y|^2 and |y - z|
// per slot (y the operand value, z the centred and scaled point), and the group's
// mean, radius and operand row.  One part: q rows [h, 1, 1, 1], candidate and
// centre rows [h, n1, n2, n3], n1 + n2 + n3 = -|y|^2 / 2; two parts: [h, l, h,
// 1, 1, 1] and [h, h, l, n1, n2, n3].  gmax: [0] max |y|^2 and [1] max error over
// the points, [2] max |y|^2 over the means, [3] max |z|^2 unscaled (centred).
template <int KP, bool SPLIT, class T>
__global__ void __launch_bounds__(kBlock)
k_cell_prep(const T *Zr, int d, const float *cen, const int32_t *perm, const int *tot, uint16_t *zq,
            uint16_t *zc, uint16_t *zb, float *Rb, T *Zs, float *nhat, float *eps,
            unsigned *gmax) {
    __shared__ float zt[kGrp * 65];
    __shared__ uint16_t nc[kGrp + 1][4];
    __shared__ float mean[kPivLd];
    __shared__ int32_t ids[kGrp];
    __shared__ int nval;
    const int g = blockIdx.x, tid = threadIdx.x, ldz = d + 1;
    if (g >= tot[0]) {
        if (tid == 0) Rb[g] = -1.0f;
        return;
    }
    const float sc = point_scale(gmax[3]);
    const int64_t s0 = (int64_t)g * kGrp;
    if (tid == 0) nval = 0;
    __syncthreads();
    if (tid < kGrp) {
        const int32_t id = perm[s0 + tid];
        ids[tid] = id;
        const int nv = __popcll(__ballot(id >= 0));
        if (tid % kWave == 0) atomicAdd(&nval, nv);
    }
    __syncthreads();
    for (int e = tid; e < kGrp * d; e += kBlock) {
        const int r = e / d, t = e - r * d;
        const T z = ids[r] >= 0 ? Zr[(int64_t)ids[r] * d + t] : T(0);
        Zs[s0 * d + e] = z;
        zt[r * ldz + t] = ids[r] >= 0 ? centred(z, cen[t]) * sc : 0.0f;
    }
    __syncthreads();
    if (tid < d) {
        float a = 0.0f;
        for (int i = 0; i < kGrp; ++i) a += zt[i * ldz + tid];
        mean[tid] = a / (float)nval;
    }
    __syncthreads();
    // thread r < kGrp: slot r; thread kGrp: the mean
    float nf = 0.0f, ef = 0.0f, rad = 0.0f;
    if (tid <= kGrp) {
        double nn = 0.0, ee = 0.0;
        float a = 0.0f;
        const float *zr = tid < kGrp ? zt + tid * ldz : mean;
        for (int t = 0; t < d; ++t) {
            const float z = zr[t];
            const uint16_t h = f2h(z);
            double y = (double)h2f(h);
            if constexpr (SPLIT) y += (double)h2f(f2h(z - h2f(h)));
            nn += y * y;
            double x = (double)z;
            if constexpr (sizeof(T) == 8)  // against the double, not its FP32 rounding
                if (tid < kGrp) x = (Zs[(s0 + tid) * d + t] - (double)cen[t]) * (double)sc;
            ee += (y - x) * (y - x);
            a = fmaf(z - mean[t], z - mean[t], a);
        }
        const bool live = tid == kGrp || ids[tid] >= 0;
        const double v = -0.5 * nn;
        uint16_t o[3];
        o[0] = f2h((float)v);
        const double r1 = v - (double)h2f(o[0]);
        o[1] = f2h((float)r1);
        o[2] = f2h((float)(r1 - (double)h2f(o[1])));
        if (!live) {  // never above a threshold
            o[0] = f2h(-65504.0f);
            o[1] = o[2] = 0;
        }
        for (int u = 0; u < 3; ++u) nc[tid][u] = o[u];
        if (live) {
            nf = (float)(nn * (1.0 + 1e-6)) + 1e-30f;
            ef = (float)(sqrt(ee) * (1.0 + 1e-6));
            // FP32 points: z - cen was rounded (2^-24 of each coordinate)
            if constexpr (sizeof(T) == 4)
                if (tid < kGrp) ef += 6e-8f * sqrtf(nf);
            rad = a == a ? sqrtf(a) * (1.0f + 1e-5f) : __builtin_huge_valf();
        }
        if (tid < kGrp) {
            nhat[s0 + tid] = nf;
            eps[s0 + tid] = ef;
        }
    }
    __syncthreads();
    const uint16_t one = f2h(1.0f);
    auto elem = [&](const float *zr, const uint16_t *nrm, int c, bool query) -> uint32_t {
        const int parts = SPLIT ? 3 : 1;
        if (c < parts * d) {
            const int q = SPLIT ? c / d : 0;
            const float z = zr[c - q * d];
            const uint16_t h = f2h(z);
            const bool low = SPLIT && (query ? q == 1 : q == 2);
            return low ? f2h(z - h2f(h)) : h;
        }
        const int u = c - parts * d;
        return u < 3 ? (query ? one : nrm[u]) : (uint16_t)0;
    };
    auto chunk = [&](const float *zr, const uint16_t *nrm, int c8, bool query) -> uint4 {
        uint32_t wv[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            wv[u] = elem(zr, nrm, 8 * c8 + 2 * u, query) |
                    (elem(zr, nrm, 8 * c8 + 2 * u + 1, query) << 16);
        return make_uint4(wv[0], wv[1], wv[2], wv[3]);
    };
    uint4 *q4 = (uint4 *)(zq + s0 * KP), *c4 = (uint4 *)(zc + s0 * KP);
    for (int e = tid; e < kGrp * KP / 8; e += kBlock) {
        const int r = e / (KP / 8), c = e % (KP / 8);
        q4[e] = chunk(zt + r * ldz, nc[r], c, true);
        c4[e] = chunk(zt + r * ldz, nc[r], c, false);
    }
    for (int c = tid; c < KP / 8; c += kBlock)
        ((uint4 *)(zb + (int64_t)g * KP))[c] = chunk(mean, nc[kGrp], c, false);
    // maxima: wavefronts 0 and 1 hold the slots, thread kGrp the mean (the
    // bits of non-negative floats order as integers, NaN above all)
    __shared__ unsigned red[3][kGrp / kWave];
    if (tid < kGrp) {
        unsigned a = __float_as_uint(nf), b = __float_as_uint(ef), r = __float_as_uint(rad);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            a = max(a, (unsigned)__shfl_xor((int)a, o, kWave));
            b = max(b, (unsigned)__shfl_xor((int)b, o, kWave));
            r = max(r, (unsigned)__shfl_xor((int)r, o, kWave));
        }
        if (tid % kWave == 0) {
            red[0][tid / kWave] = a;
            red[1][tid / kWave] = b;
            red[2][tid / kWave] = r;
        }
    }
    __syncthreads();
    if (tid == kGrp) {
        atomicMax(&gmax[0], max(red[0][0], red[0][1]));
        atomicMax(&gmax[1], max(red[1][0], red[1][1]));
        atomicMax(&gmax[2], __float_as_uint(nf));
        float r = __uint_as_float(max(red[2][0], red[2][1])) + ef;
        // the radius was taken of FP32 roundings
        r += 1.2e-7f * sqrtf(__uint_as_float(max(red[0][0], red[0][1])));
        Rb[g] = r * (1.0f + 1e-5f) + 1e-30f;
    }
}

// The 16-byte chunk c of LDS row r is stored at chunk swz(r, c): the 16 rows
// of a candidate block then meet 16 different bank groups.
template <int KP>
__device__ __forceinline__ int swz(int r, int c) {
    if constexpr (KP % 128 == 0)
        return c ^ (r & 15);
    else if constexpr (KP % 64 == 0)
        return c ^ ((r >> 1) & 7);
    else
        return c ^ ((r >> 2) & 3);
}

struct CellArgs {
    const uint16_t *zq, *zc, *zb;
    const float *Rb, *nhat, *eps;
    const unsigned *gmax;
    const int32_t *perm;
    const int *tot;
    int include_self, rank_k, rank_l;
    double eta, spec;
    int32_t *cidx, *ccnt;
    float *cthr;
};

template <int KP>
struct CellLds {
    uint16_t tiles[2][kCT * KP];
    int32_t list[kGrp][kCap];  // also the residue maxima (as floats)
    uint32_t need[kMaxGroups / 32];
    float thr[kGrp], ta[kGrp];
};

template <int KP>
__global__ void __launch_bounds__(kBlock, KP <= 64 ? 3 : 2)
k_knn_cell(CellArgs a) {
    static_assert(KP % 32 == 0, "whole MFMA steps");
    constexpr int KS = KP / 32, NCB = kCT / 16, CH = KP / 8;
    constexpr int NLD = (kCT * CH + kBlock - 1) / kBlock;
    extern __shared__ __attribute__((aligned(16))) unsigned char cell_lds[];
    CellLds<KP> &L = *(CellLds<KP> *)cell_lds;
    const int ng = a.tot[0];
    // consecutive groups on one XCD (blocks are dealt to the 8 XCDs in turn):
    // they sweep the same candidates
    const int per = (gridDim.x + 7) / 8;
    const int g = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    if (g >= ng) return;
    const int lane = lane_id();
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const int col = lane & 15, grp = lane >> 4;
    const int64_t q0 = (int64_t)g * kGrp;

    v8h ab[kQW][KS];
#pragma unroll
    for (int rb = 0; rb < kQW; ++rb)
#pragma unroll
        for (int s = 0; s < KS; ++s)
            ab[rb][s] = *(const v8h *)(a.zq + (q0 + w * kQW * 16 + rb * 16 + col) * KP + 32 * s +
                                        8 * grp);
    for (int i = threadIdx.x; i < (ng + 31) / 32; i += kBlock) L.need[i] = 0u;

    static_assert(NLD * kBlock == kCT * CH, "whole loads");
    auto fetch = [&](const uint16_t *rows, int64_t t0, v4u (&s)[NLD])
                     __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < NLD; ++u)
            s[u] = ((const v4u *)(rows + t0 * KP))[threadIdx.x + u * kBlock];
    };
    auto deposit = [&](int b, const v4u (&s)[NLD]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < NLD; ++u) {
            const int e = threadIdx.x + u * kBlock;
            const int r = e / CH, c = e % CH;
            *(v4u *)(&L.tiles[b][r * KP + swz<KP>(r, c) * 8]) = s[u];
        }
    };
    auto products = [&](int b, v4f (&acc)[NCB][kQW]) __attribute__((always_inline)) {
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb) {
            const int r = cb * 16 + col;
            v8h bb[KS];
#pragma unroll
            for (int s = 0; s < KS; ++s)
                bb[s] = *(const v8h *)(&L.tiles[b][r * KP + swz<KP>(r, 4 * s + grp) * 8]);
#pragma unroll
            for (int rb = 0; rb < kQW; ++rb) {
                v4f x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < KS; ++s)
                    x = __builtin_amdgcn_mfma_f32_16x16x32_f16(ab[rb][s], bb[s], x, 0, 0, 0);
                acc[cb][rb] = x;
            }
        }
    };
    // Runs body(t0, buf) over the tiles that next() yields (-1: no more), two
    // tiles of loads in flight; every wavefront sees the same tiles.
    auto sweep = [&](const uint16_t *rows, auto next, auto body) __attribute__((always_inline)) {
        int64_t t = next();
        if (t < 0) return;
        v4u s0[NLD], s1[NLD];
        fetch(rows, t, s0);
        int64_t t1 = next();
        if (t1 >= 0) fetch(rows, t1, s1);
        __syncthreads();  // the buffers' last readers are done
        deposit(0, s0);
        __syncthreads();
        for (;;) {
            const int64_t t2 = t1 >= 0 ? next() : -1;
            if (t2 >= 0) fetch(rows, t2, s0);
            body(t, 0);
            if (t1 < 0) break;
            deposit(1, s1);
            __syncthreads();
            const int64_t t3 = t2 >= 0 ? next() : -1;
            if (t3 >= 0) fetch(rows, t3, s1);
            body(t1, 1);
            if (t2 < 0) break;
            deposit(0, s0);
            __syncthreads();
            t = t2;
            t1 = t3;
        }
    };
    float mx[NCB][kQW][4];
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
        for (int rb = 0; rb < kQW; ++rb)
#pragma unroll
            for (int i = 0; i < 4; ++i) mx[cb][rb][i] = ninf();
    auto keep_max = [&](int64_t t0, int b) __attribute__((always_inline)) {
        v4f acc[NCB][kQW];
        products(b, acc);
        const bool own = !a.include_self && t0 >= q0 && t0 < q0 + kGrp;
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
            for (int rb = 0; rb < kQW; ++rb)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float v = acc[cb][rb][i];
                    if (own && t0 + cb * 16 + col == q0 + w * kQW * 16 + rb * 16 + 4 * grp + i)
                        v = ninf();
                    mx[cb][rb][i] = fmaxf(mx[cb][rb][i], v);
                }
    };
    // rank-th largest of each row's 64 residue maxima, through f(row, value)
    auto ranks = [&](int rank, auto f) {
        __syncthreads();
#pragma unroll
        for (int rb = 0; rb < kQW; ++rb)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int cb = 0; cb < NCB; ++cb)
                    L.list[w * kQW * 16 + rb * 16 + 4 * grp + i][cb * 16 + col] =
                        __float_as_int(mx[cb][rb][i]);
        __syncthreads();
        for (int r = 0; r < kQW * 16; ++r) {
            const int row = w * kQW * 16 + r;
            float v = __int_as_float(L.list[row][lane]);
            for (int size = 2; size <= kWave; size <<= 1)
                for (int stride = size >> 1; stride > 0; stride >>= 1) {
                    const float ov = __shfl_xor(v, stride, kWave);
                    const bool up = (lane & size) == 0, lower = (lane & stride) == 0;
                    if ((lower == up) ? ov > v : v > ov) v = ov;
                }
            f(row, __shfl(v, rank - 1, kWave));
        }
        __syncthreads();
    };

    // 1. the groups around this one in slot order: a bound of the k-th
    // neighbour of every query
    {
        int gb = g - kWindow / 2;
        if (gb + kWindow > ng) gb = ng - kWindow;
        if (gb < 0) gb = 0;
        const int ge = gb + kWindow < ng ? gb + kWindow : ng;
        int64_t t = (int64_t)gb * kGrp;
        const int64_t te = (int64_t)ge * kGrp;
        sweep(a.zc,
              [&]() {
                  const int64_t r = t < te ? t : -1;
                  t += kCT;
                  return r;
              },
              keep_max);
    }
    const double ncmax = (double)__uint_as_float(a.gmax[0]);
    const double emax = (double)__uint_as_float(a.gmax[1]);
    const double nbmax = (double)__uint_as_float(a.gmax[2]);
    ranks(a.rank_k, [&](int row, float sv) {
        if (lane != 0) return;
        const double nq = (double)a.nhat[q0 + row], eq = (double)a.eps[q0 + row];
        // |q - c| of rank_k candidates is at most U, their exact FP32
        // distance at most U^2 / spec
        const double dt = nq - 2.0 * (double)sv;
        const double U = sqrt((dt > 0.0 ? dt : 0.0) * (1.0 + 0x1p-21) + a.eta * (nq + ncmax) +
                              kNormErr) + eq + emax;
        const bool live = a.perm[q0 + row] >= 0;
        // a group is out of reach when nq - 2 s > (T + R)^2 with room for the
        // score's error
        float T = (float)((U / a.spec + eq) * (1.0 + 1e-5));
        if (!(sv > -6e4f) || !(T == T)) T = __builtin_huge_valf();
        float A = (float)(nq - (1.02 * a.eta + 4e-6) * (nq + nbmax) - kNormErr);
        L.thr[row] = live ? T : 0.0f;
        L.ta[row] = live ? A : __builtin_huge_valf();
    });
    // 2. the groups within reach of some query
    {
        float T[kQW][4], A[kQW][4];
#pragma unroll
        for (int rb = 0; rb < kQW; ++rb)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = w * kQW * 16 + rb * 16 + 4 * grp + i;
                T[rb][i] = L.thr[row];
                A[rb][i] = L.ta[row];
            }
        int64_t t = 0;
        const int64_t te = (ng + kCT - 1) / kCT * kCT;
        sweep(a.zb,
              [&]() {
                  const int64_t r = t < te ? t : -1;
                  t += kCT;
                  return r;
              },
              [&](int64_t t0, int b) __attribute__((always_inline)) {
                  float R[NCB];
#pragma unroll
                  for (int cb = 0; cb < NCB; ++cb) R[cb] = a.Rb[t0 + cb * 16 + col];
                  v4f acc[NCB][kQW];
                  products(b, acc);
                  uint64_t bits = 0;
#pragma unroll
                  for (int cb = 0; cb < NCB; ++cb) {
                      bool need = false;
#pragma unroll
                      for (int rb = 0; rb < kQW; ++rb)
#pragma unroll
                          for (int i = 0; i < 4; ++i) {
                              const float s = T[rb][i] + R[cb];
                              need |= !(A[rb][i] - 2.0f * acc[cb][rb][i] > s * s * 1.0001f) &&
                                      A[rb][i] < __builtin_huge_valf();
                          }
                      const uint64_t m = __ballot(need && R[cb] >= 0.0f);
                      const uint64_t f = (m | (m >> 16) | (m >> 32) | (m >> 48)) & 0xFFFFull;
                      bits |= f << (16 * cb);
                  }
                  if (lane < 2 && bits)
                      atomicOr(&L.need[t0 / 32 + lane], (uint32_t)(bits >> (32 * lane)));
              });
        __syncthreads();
    }
    // the tiles of the needed groups
    auto needed = [&]() {
        return [&L, ng, word = 0, cur = 0u, half = 0, gi = 0]() mutable -> int64_t {
            if (half) {
                half = 0;
                return (int64_t)gi * kGrp + kCT;
            }
            if (word == 0) cur = __builtin_amdgcn_readfirstlane(L.need[word++]);
            while (cur == 0u) {
                if (word * 32 >= ng) return -1;
                cur = __builtin_amdgcn_readfirstlane(L.need[word++]);
            }
            gi = (word - 1) * 32 + __builtin_ctz(cur);
            cur &= cur - 1;
            half = 1;
            return (int64_t)gi * kGrp;
        };
    };
    // 3. the threshold: the rank_l-th residue maximum over them (a candidate
    // seen twice, here and in the window, keeps its residue)
    sweep(a.zc, needed(), keep_max);
    ranks(a.rank_l, [&](int row, float sv) {
        if (lane == 0) L.thr[row] = sv;
    });
    // 4. everything above it
    {
        float thr[kQW][4];
        int cnt[kQW][4];
#pragma unroll
        for (int rb = 0; rb < kQW; ++rb)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = w * kQW * 16 + rb * 16 + 4 * grp + i;
                thr[rb][i] = a.perm[q0 + row] >= 0 ? L.thr[row] : __builtin_huge_valf();
                cnt[rb][i] = 0;
            }
        sweep(a.zc, needed(), [&](int64_t t0, int b) __attribute__((always_inline)) {
            v4f acc[NCB][kQW];
            products(b, acc);
            const bool own = !a.include_self && t0 >= q0 && t0 < q0 + kGrp;
#pragma unroll
            for (int rb = 0; rb < kQW; ++rb)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float m = fmaxf(fmaxf(acc[0][rb][i], acc[1][rb][i]),
                                          fmaxf(acc[2][rb][i], acc[3][rb][i]));
                    if (!__ballot(m > thr[rb][i])) continue;
                    const int row = w * kQW * 16 + rb * 16 + 4 * grp + i;
#pragma unroll
                    for (int cb = 0; cb < NCB; ++cb) {
                        const int32_t slot = (int32_t)t0 + cb * 16 + col;
                        const bool pass = acc[cb][rb][i] > thr[rb][i] &&
                                          !(own && slot == (int32_t)q0 + row);
                        const uint64_t mask = __ballot(pass);
                        if (!mask) continue;
                        const uint32_t mr = (uint32_t)(mask >> (16 * grp)) & 0xFFFFu;
                        const int pos = cnt[rb][i] + __popc(mr & ((1u << col) - 1u));
                        if (pass && pos < kCap) L.list[row][pos] = slot;
                        cnt[rb][i] += __popc(mr);
                    }
                }
        });
#pragma unroll
        for (int rb = 0; rb < kQW; ++rb)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = w * kQW * 16 + rb * 16 + 4 * grp + i;
                if (col == 0) {
                    a.ccnt[q0 + row] = cnt[rb][i];
                    a.cthr[q0 + row] = thr[rb][i];
                }
            }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < kGrp * kCap; e += kBlock)
        a.cidx[q0 * kCap + e] = (&L.list[0][0])[e];
}

// Exact distances of a query's candidates (unscaled rows), the k smallest under (distance,
// index), and the certificate of sev_knn_mfma.hip; one wavefront per slot.
template <class T>
__global__ void __launch_bounds__(kBlock)
k_cell_rerank(const T *Zs, const int32_t *perm, const int *tot, int d, int k,
              const int32_t *cidx, const int32_t *ccnt, const float *cthr, const float *nhat,
              const float *eps, const unsigned *gmax, double eta, double spec, int32_t *oidx,
              T *odist, int32_t *nfail, int64_t *fail) {
    const int lane = lane_id();
    const int64_t s = ((int64_t)blockIdx.x * kBlock + threadIdx.x) / kWave;
    if (s >= (int64_t)tot[0] * kGrp) return;
    const int32_t q = perm[s];
    if (q < 0) return;
    const int cnt = ccnt[s];
    const int32_t c = lane < cnt && cnt <= kCap ? cidx[s * kCap + lane] : -1;
    T D = (T)__builtin_huge_valf();
    int32_t ci = INT_MAX;
    if (c >= 0) {
        typedef T T2 __attribute__((ext_vector_type(2)));
        ci = perm[c];
        const T *zq = Zs + s * d, *zc = Zs + (int64_t)c * d;
        T acc = 0;
        if ((d & 1) == 0) {  // rows start at a multiple of two values
            const T2 *q2 = (const T2 *)zq, *c2 = (const T2 *)zc;
#pragma unroll 4
            for (int t = 0; t < d / 2; ++t) {
                const T2 x = q2[t], y = c2[t];
                const T d0 = x[0] - y[0];
                acc = acc + d0 * d0;
                const T d1 = x[1] - y[1];
                acc = acc + d1 * d1;
            }
        } else {
#pragma unroll 4
            for (int t = 0; t < d; ++t) {
                const T x = zq[t] - zc[t];
                acc = acc + x * x;
            }
        }
        D = acc;
    }
    for (int size = 2; size <= kWave; size <<= 1)
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            const T oD = __shfl_xor(D, stride, kWave);
            const int32_t oc = __shfl_xor(ci, stride, kWave);
            const bool up = (lane & size) == 0, lower = (lane & stride) == 0;
            const bool less = oD < D || (oD == D && oc < ci);
            const bool more = oD > D || (oD == D && oc > ci);
            if ((lower == up) ? less : more) {
                D = oD;
                ci = oc;
            }
        }
    const T Dk = __shfl(D, k - 1, kWave);
    const double nq = (double)nhat[s];
    const double dt = nq - 2.0 * (double)cthr[s];
    const double lb2 = dt * (1.0 - 0x1p-21) -
                       eta * (nq + (double)__uint_as_float(gmax[0])) - kNormErr;
    const double lb = lb2 > 0.0 ? sqrt(lb2) - (double)eps[s] - (double)__uint_as_float(gmax[1])
                                : -1.0;
    const double sc = (double)point_scale(gmax[3]);
    const bool ok = cnt >= k && cnt <= kCap && lb > 0.0 &&
                    lb * lb * spec > (double)Dk * sc * sc && Dk == Dk;
    if (ok) {
        if (lane < k) {
            oidx[(int64_t)q * k + lane] = ci;
            odist[(int64_t)q * k + lane] = sqrt(D);
        }
    } else if (lane == 0) {
        fail[atomicAdd(nfail, 1)] = q;
    }
}

template <int KP, bool SPLIT, class T>
void run_cell(int64_t n, int64_t d, int64_t k, int include_self, int M, KnnWork &w, int32_t *idx,
              T *dist, hipStream_t st) {
    const int64_t ngb = ceil_div(n, (int64_t)kGrp) + M;  // at least the groups in use
    const int64_t ns = ngb * kGrp;
    const int64_t ngt = ceil_div(ngb, (int64_t)kCT) * kCT;
    w.zq.ensure((size_t)ns * KP * 2);
    w.zc.ensure((size_t)ns * KP * 2);
    w.zcp.ensure((size_t)ngt * KP * 2);
    w.scf.ensure((size_t)ngt);
    w.zs.ensure((size_t)(ns * d) * sizeof(T));
    const T *zr = (const T *)w.zrb.get();
    T *zs = (T *)w.zs.get();
    w.nhat.ensure((size_t)ns);
    w.eps.ensure((size_t)ns);
    w.cidx.ensure((size_t)ns * kCap);
    w.cthr.ensure((size_t)ns);
    w.ccnt.ensure((size_t)ns);
    const int *tot = w.ctot.get();
    {
        ProfScope ps("knn_prep", st, 8.0 * n * d + 4.0 * n * KP);
        hipLaunchKernelGGL((k_cell_prep<KP, SPLIT, T>), dim3((unsigned)ngt), dim3(kBlock), 0, st,
                           zr, (int)d, w.piv.get(), w.perm.get(), tot, (uint16_t *)w.zq.get(),
                           (uint16_t *)w.zc.get(), (uint16_t *)w.zcp.get(), w.scf.get(),
                           zs, w.nhat.get(), w.eps.get(), w.gmax.get());
        SEV_LAUNCH_CHECK();
    }
    CellArgs a;
    a.zq = (const uint16_t *)w.zq.get();
    a.zc = (const uint16_t *)w.zc.get();
    a.zb = (const uint16_t *)w.zcp.get();
    a.Rb = w.scf.get();
    a.nhat = w.nhat.get();
    a.eps = w.eps.get();
    a.gmax = w.gmax.get();
    a.perm = w.perm.get();
    a.tot = tot;
    a.include_self = include_self;
    a.rank_k = (int)k;
    a.rank_l = knn_cell_rank(k);
    // FP32 accumulation over KP terms, the dropped l.l' (2^-22) and the
    // three-part norm
    a.eta = 4.0 * (KP + 2) * 0x1p-24 + 0x1p-20;
    a.spec = pow(1.0 - (sizeof(T) == 4 ? 0x1p-24 : 0x1p-53), (double)(d + 3));
    a.cidx = w.cidx.get();
    a.ccnt = w.ccnt.get();
    a.cthr = w.cthr.get();
    {
        ProfScope ps("knn_cell", st, 0.0, 2.0 * (double)n * (double)n * (double)d);
        const int lds = (int)sizeof(CellLds<KP>);
        SEV_HIP(hipFuncSetAttribute((const void *)&k_knn_cell<KP>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        hipLaunchKernelGGL(k_knn_cell<KP>, dim3((unsigned)(ceil_div(ngb, (int64_t)8) * 8)),
                           dim3(kBlock), lds, st, a);
        SEV_LAUNCH_CHECK();
    }
    ProfScope ps("knn_rerank", st, (double)n * (kCap * 0.6) * (4.0 + 4.0 * d));
    hipLaunchKernelGGL(k_cell_rerank<T>, dim3((unsigned)ceil_div(ns * kWave, (int64_t)kBlock)),
                       dim3(kBlock), 0, st, (const T *)zs, w.perm.get(), tot, (int)d, (int)k,
                       w.cidx.get(), w.ccnt.get(), w.cthr.get(), w.nhat.get(), w.eps.get(),
                       w.gmax.get(), a.eta, a.spec, idx, dist, w.nfail.get(), w.fail.get());
    SEV_LAUNCH_CHECK();
}

}  // namespace

bool knn_cell_fits(int64_t n, int64_t d, int64_t k) {
    // at k = 30 a list of 64 overflows for 2% of the rows; 3 d + 3 operand
    // columns of at most 192
    return n <= (int64_t)kGrp * (kMaxGroups - kMaxPivots - 64) && k <= 30 && d <= 63;
}

template <class T>
int64_t knn_cell(const T *Z, int64_t n, int64_t d, int64_t ld, int64_t k, int include_self,
                 bool split, KnnWork &w, int32_t *idx, T *dist, hipStream_t st) {
    // cells of 1024 to 2048 points (smaller ones below 16,384 points)
    int M = 16;
    while (M < kMaxPivots && (int64_t)M * 1024 < n) M <<= 1;
    const int nsam = (int)std::min<int64_t>(n, kSample);
    w.piv.ensure((size_t)(kPivLd + 2 * kMaxPivots * kPivLd + 2 * kMaxPivots + kSample * kPivLd));
    w.ctot.ensure(1);
    w.gmax.ensure(4);
    float *cen = w.piv.get(), *piv = cen + kPivLd, *pivo = piv + kMaxPivots * kPivLd,
          *half = pivo + kMaxPivots * kPivLd, *halfo = half + kMaxPivots,
          *sam = halfo + kMaxPivots;
    if (!split) {
        w.ccnt.ensure(1);
        hipLaunchKernelGGL(k_cell_sample<T>, dim3(128), dim3(kBlock), 0, st, Z, (int64_t)1, ld,
                           (const float *)nullptr, n, (int)d, kTestPivots, sam, w.ccnt.get());
        SEV_LAUNCH_CHECK();
        hipLaunchKernelGGL(k_cell_test<T>, dim3(kTestQueries), dim3(kBlock), 0, st, Z, n, (int)d,
                           ld, sam, w.ccnt.get());
        SEV_LAUNCH_CHECK();
        int32_t share = 0;
        SEV_HIP(hipMemcpyAsync(&share, w.ccnt.get(), sizeof share, hipMemcpyDeviceToHost, st));
        SEV_HIP(hipStreamSynchronize(st));
        if ((double)share > kCellMaxShare * kTestPivots * kTestQueries) return -1;
    }
    w.zrb.ensure((size_t)(n * d) * sizeof(T));
    T *zr = (T *)w.zrb.get();
    hipLaunchKernelGGL(k_cell_centre<T>, dim3((unsigned)d), dim3(kBlock), 0, st, Z, n, ld, cen,
                       w.gmax.get());
    SEV_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_cell_rows<T>, dim3((unsigned)ceil_div(n, (int64_t)kWave)), dim3(kBlock), 0,
                       st, Z, n, (int)d, ld, cen, zr, w.gmax.get() + 3);
    SEV_LAUNCH_CHECK();
    {
        ProfScope ps("knn_order", st, 4.0 * n * d + 24.0 * n);
        w.skey.ensure((size_t)n);
        w.skey2.ensure((size_t)n);
        w.sval.ensure((size_t)n);
        w.sval2.ensure((size_t)n);
        w.ccell.ensure((size_t)kMaxPivots);
        w.coff.ensure((size_t)2 * kMaxPivots);
        const int64_t ns = (ceil_div(n, (int64_t)kGrp) + M) * kGrp;
        w.perm.ensure((size_t)ns);
        SEV_HIP(hipMemsetAsync(w.ccell.get(), 0, sizeof(int32_t) * kMaxPivots, st));
        SEV_HIP(hipMemsetAsync(w.perm.get(), 0xFF, sizeof(int32_t) * (size_t)ns, st));
        auto assign = [&](const auto *X, int64_t nx, int64_t lx, const float *cn, const float *pv,
                          const float *hv, uint32_t *cell, int32_t *id, int32_t *cnt) {
            auto go = [&](auto dp) {
                constexpr int DP = decltype(dp)::value;
                typedef std::remove_const_t<std::remove_pointer_t<decltype(X)>> TX;
                hipLaunchKernelGGL((k_cell_assign<DP, TX>),
                                   dim3((unsigned)ceil_div(nx, (int64_t)kBlock)), dim3(kBlock), 0,
                                   st, X, nx, (int)d, lx, cn, pv, hv, M, cell, id, cnt);
            };
            if (d <= 16)
                go(std::integral_constant<int, 16>());
            else if (d <= 32)
                go(std::integral_constant<int, 32>());
            else if (d <= 52)
                go(std::integral_constant<int, 52>());
            else
                go(std::integral_constant<int, 64>());
            SEV_LAUNCH_CHECK();
        };
        hipLaunchKernelGGL(k_cell_pivots<T>, dim3(64), dim3(kBlock), 0, st, zr, cen, n,
                           (int)d, M, piv);
        hipLaunchKernelGGL(k_cell_half, dim3((unsigned)ceil_div((int64_t)M, (int64_t)kBlock)),
                           dim3(kBlock), 0, st, piv, M, half);
        hipLaunchKernelGGL(k_cell_sample<T>, dim3(256), dim3(kBlock), 0, st, zr, d, (int64_t)1, cen,
                           n, (int)d, nsam, sam, (int *)nullptr);
        SEV_LAUNCH_CHECK();
        for (int it = 0; it < 2; ++it) {
            assign((const float *)sam, nsam, nsam, nullptr, piv, half, w.skey2.get(), nullptr,
                   nullptr);
            hipLaunchKernelGGL(k_cell_means, dim3((unsigned)M), dim3(kBlock), 0, st, sam, nsam,
                               (int)d, w.skey2.get(), piv, half);
            SEV_LAUNCH_CHECK();
        }
        hipLaunchKernelGGL(k_cell_order, dim3(1), dim3(kMaxPivots), 0, st, piv, half, M, (int)d,
                           pivo, halfo);
        SEV_LAUNCH_CHECK();
        assign(Z, n, ld, cen, pivo, halfo, w.skey.get(), w.sval.get(), w.ccell.get());
        hipLaunchKernelGGL(k_cell_offsets, dim3(1), dim3(kMaxPivots), 0, st, w.ccell.get(), M,
                           w.coff.get(), w.coff.get() + kMaxPivots, w.ctot.get());
        SEV_LAUNCH_CHECK();
        int bits = 1;
        while ((1 << bits) < M) ++bits;
        size_t tb = 0;
        SEV_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, w.skey.get(), w.skey2.get(),
                                                   w.sval.get(), w.sval2.get(), (int)n, 0, bits,
                                                   st));
        w.stmp.ensure(tb);
        SEV_HIP(hipcub::DeviceRadixSort::SortPairs(w.stmp.get(), tb, w.skey.get(), w.skey2.get(),
                                                   w.sval.get(), w.sval2.get(), (int)n, 0, bits,
                                                   st));
        hipLaunchKernelGGL(k_cell_slots, dim3((unsigned)ceil_div(n, (int64_t)kBlock)), dim3(kBlock),
                           0, st, w.skey2.get(), w.sval2.get(), n, w.coff.get(),
                           w.coff.get() + kMaxPivots, w.perm.get());
        SEV_LAUNCH_CHECK();
    }
    w.nfail.ensure(4);
    w.fail.ensure((size_t)n);
    SEV_HIP(hipMemsetAsync(w.nfail.get(), 0, 4 * sizeof(int32_t), st));
    if (split) {
        const int64_t cols = 3 * d + 3;
        if (cols <= 64)
            run_cell<64, true, T>(n, d, k, include_self, M, w, idx, dist, st);
        else if (cols <= 96)
            run_cell<96, true, T>(n, d, k, include_self, M, w, idx, dist, st);
        else if (cols <= 128)
            run_cell<128, true, T>(n, d, k, include_self, M, w, idx, dist, st);
        else if (cols <= 160)
            run_cell<160, true, T>(n, d, k, include_self, M, w, idx, dist, st);
        else
            run_cell<192, true, T>(n, d, k, include_self, M, w, idx, dist, st);
    } else {
        const int64_t cols = d + 3;
        if (cols <= 32)
            run_cell<32, false, T>(n, d, k, include_self, M, w, idx, dist, st);
        else if (cols <= 64)
            run_cell<64, false, T>(n, d, k, include_self, M, w, idx, dist, st);
        else
            run_cell<96, false, T>(n, d, k, include_self, M, w, idx, dist, st);
    }
    int32_t nf = 0;
    SEV_HIP(hipMemcpyAsync(&nf, w.nfail.get(), sizeof nf, hipMemcpyDeviceToHost, st));
    SEV_HIP(hipStreamSynchronize(st));
    return nf;
}

template int64_t knn_cell<float>(const float *, int64_t, int64_t, int64_t, int64_t, int, bool,
                                 KnnWork &, int32_t *, float *, hipStream_t);

// FP64 points: their FP32 roundings in two parts propose the candidates (the
// rounding is part of each point's operand error), the exact FP64 distances
// rank them.
void knn_cell_f64(const double *Z, int64_t n, int64_t d, int64_t ld, int64_t k, int include_self,
                  KnnWork &w, int32_t *idx, double *dist, hipStream_t st, int64_t *n_fallback) {
    const int64_t nf = knn_cell<double>(Z, n, d, ld, k, include_self, true, w, idx, dist, st);
    if (nf > 0)
        knn_exact_rows<double>(Z, n, d, ld, k, include_self, w.fail.get(), nf, idx, dist, st);
    if (n_fallback) *n_fallback = nf;
}

}  // namespace sev
