// Blocked right-looking Cholesky (lower) for gfx950, row-major, in place.
// Only the lower triangle of A is read, as in scirs2-linalg/src/lapack.rs:632-679,
// and the strict upper triangle of the result is zeroed so the output is the
// reference's L.  Per block of kb columns at k0:
//   1. chol_panel — the diagonal block's factor and L21 = A21 L11^-T in one
//      launch; the reference's test `a_ii - sum <= 0` (lapack.rs:661-670) sets
//      info = row + 1 and stops.
//   2. syrk — A22 -= L21 L21^T on the matrix cores (lower tiles only).
#include "arrive.hpp"
#include "common.hpp"
#include "kernels.hpp"
#include "lanes.hpp"
#include <algorithm>
#include <cstdlib>
#include <type_traits>

namespace {
constexpr int NT = 256;

template <typename T>
__device__ __forceinline__ T readlane_t(T v, int k);
template <>
__device__ __forceinline__ float readlane_t<float>(float v, int k)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), k));
}
template <>
__device__ __forceinline__ double readlane_t<double>(double v, int k)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), k);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), k);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// A panel of kb <= 128 columns in one launch: the diagonal block's factor and the
// rows below, L21 = A21 L11^-T by substitution (lapack.rs:661-676: sqrt, true
// division).  Every workgroup factors the diagonal block for itself — 32 columns at a
// time, and a wave needs nothing from another while it does: its lanes 0..31 hold the
// 32 diagonal rows (the same in all waves), lanes 32..63 the rows it is responsible
// for, groups 1..3 of the diagonal block (waves 0..2) and 32 rows of A21 (wave 3).
// Column j: the diagonal by readlane, its square root and reciprocal, l = a / sqrt
// (one residual correction: correctly rounded), and a_c -= l l_c with l_c handed to all
// lanes by two permlane swaps and DPP (lanes.hpp).  Between the 32-column steps the
// waves exchange their L through LDS and update their later columns, which wait in
// registers in the matrix-core layout.  The last workgroup to have read the diagonal
// block (an arrival count, nobody waits) writes it back.
// Bound by the column chain.  Measured for one FP64 128-column panel: 45 to 50 us
// whatever the rows below (up to one workgroup per CU), against 78 (diagonal block) + 36
// (its inverse) + 23 us (product) in three launches before.
// One a_jj - sum <= 0 sets info = row + 1 and stops; a workgroup that starts after that
// still registers its arrival (arrive.hpp) before it leaves.
template <typename T> struct CholPanelArgs {
    T *A; long lda;
    int k0, kb, n;
    int *arrive;      // zero between launches
    int *info; double *info_val;
};
struct CholArrival {
    int *count;
    bool failed;   // info as it was when the workgroup started
    __device__ int add() { return __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
    __device__ void clear() { __hip_atomic_store(count, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
    __device__ bool stopped() const { return failed; }
};
// x's lanes 0..15 (lo) and 16..31 (hi) in every row of 16 lanes
__device__ __forceinline__ void spread(unsigned x, unsigned &lo, unsigned &hi)
{
    const auto p = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    lo = __builtin_amdgcn_permlane32_swap(p[0], p[0], false, false)[0];
    hi = __builtin_amdgcn_permlane32_swap(p[1], p[1], false, false)[0];
}
__device__ __forceinline__ void spread(double x, double (&pr)[2])
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(x);
    unsigned l0, l1, h0, h1;
    spread((unsigned)b, l0, l1);
    spread((unsigned)(b >> 32), h0, h1);
    pr[0] = __longlong_as_double((long long)(((unsigned long long)h0 << 32) | l0));
    pr[1] = __longlong_as_double((long long)(((unsigned long long)h1 << 32) | l1));
}
__device__ __forceinline__ void spread(float x, float (&pr)[2])
{
    unsigned l0, l1;
    spread(__float_as_uint(x), l0, l1);
    pr[0] = __uint_as_float(l0);
    pr[1] = __uint_as_float(l1);
}
// 1/p to an ulp, and a/p from it by residual corrections
__device__ __forceinline__ double recip(double p)
{
    double r = __builtin_amdgcn_rcp(p);
    r = fma(r, fma(-p, r, 1.0), r);
    return fma(r, fma(-p, r, 1.0), r);
}
__device__ __forceinline__ float recip(float p)
{
    const float r = __builtin_amdgcn_rcpf(p);
    return fmaf(r, fmaf(-p, r, 1.0f), r);
}
__device__ __forceinline__ double quot(double a, double p, double r)
{
    const double q = a * r;
    return fma(fma(-q, p, a), r, q);
}
__device__ __forceinline__ float quot(float a, float p, float r)
{
    float q = a * r;
    q = fmaf(fmaf(-q, p, a), r, q);
    return fmaf(fmaf(-q, p, a), r, q);
}

constexpr int CP_B = 32;   // columns of a step
// column J of the step; returns false when the diagonal is not positive
template <typename T, int J> __device__ __forceinline__ bool chol_column(T (&a)[CP_B], T &dv)
{
    dv = readlane_t<T>(a[J], J);
    if (__builtin_expect(!(dv > (T)0), 0)) return false;
    const T s = sqrt(dv), r = recip(s);   // (a root is neither tiny nor huge: no scaling)
    T q = quot(a[J], s, r);
    if (__builtin_expect(dv > (T)(sizeof(T) == 8 ? DBL_MAX : FLT_MAX), 0)) q = a[J] / s;   // infinite: no residual
    const T l = (threadIdx.x & 63) == J ? s : q;
    a[J] = l;
    T pr[2];
    spread(l, pr);
    constexpr int c0 = J + 1;
    if constexpr (c0 < CP_B) {
        // up to the next multiple of eight, then whole blocks
        constexpr int n0 = (8 - (c0 & 7)) & 7;
        if constexpr (n0 > 0) lanes::fmac_row<c0 & 15, n0 ? n0 : 1>(&a[c0], pr[c0 >> 4], l);
        constexpr int b0 = (c0 + 7) / 8;
        if constexpr (b0 < 1) lanes::fmac_row<0, 8>(&a[0], pr[0], l);
        if constexpr (b0 < 2) lanes::fmac_row<8, 8>(&a[8], pr[0], l);
        if constexpr (b0 < 3) lanes::fmac_row<0, 8>(&a[16], pr[1], l);
        if constexpr (b0 < 4) lanes::fmac_row<8, 8>(&a[24], pr[1], l);
    }
    return true;
}
// columns J .. 31 of a step with `cols` columns left (looked at every eighth: the others
// are the identity's); the failing column, or -1
template <typename T, int J> __device__ __forceinline__ int chol_columns(T (&a)[CP_B], T &dv, int cols)
{
    if constexpr (J < CP_B) {
        if constexpr (J > 0 && J % 8 == 0)
            if (J >= cols) return -1;
        if (!chol_column<T, J>(a, dv)) return J;
        return chol_columns<T, J + 1>(a, dv, cols);
    } else {
        return -1;
    }
}

template <typename T> __global__ __launch_bounds__(NT, 2) void chol_panel_kernel(CholPanelArgs<T> g)
{
    using lanes::Mf;
    typedef typename Mf<T>::V V4;
    typedef typename lanes::Vec16<T>::type V;
    typedef typename lanes::Vec16u<T>::type Vu;
    constexpr int B = CP_B, E = 16 / (int)sizeof(T), P = B + E;   // LDS pitch: 16-byte rows
    __shared__ __align__(16) T Ls[5][B * P];   // the waves' row groups; [4]: the diagonal rows
    __shared__ int s_last, s_stop, s_fail;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    // read once, by one thread: workgroup 0 of this very launch may be setting it
    const int info = t == 0 ? __hip_atomic_load(g.info, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
    const int l16 = lane & 15, grp = lane >> 4, l32 = lane & 31;
    const bool low = lane < 32;
    T *D = g.A + (long)g.k0 * g.lda + g.k0;
    const int chunk0 = g.kb + B * (int)blockIdx.x;   // first of this workgroup's rows of A21, from k0
    const int rows = g.n - g.k0;
    // row group of a wave's upper lanes: its first row from k0, and the rows that exist
    const int group0 = wave < 3 ? B * (wave + 1) : chunk0;
    const int glimit = wave < 3 ? g.kb : rows;
    // element (r, c) of the panel; outside the diagonal block the identity
    T a[B];
    {
        const int r = low ? l32 : group0 + l32;
        const bool ok = r < (low ? g.kb : glimit);
        const T *src = D + (long)min(r, rows - 1) * g.lda;
        if (g.kb >= B) {
#pragma unroll
            for (int c = 0; c < B; c += E) {
                const Vu v = *reinterpret_cast<const Vu *>(src + c);
#pragma unroll
                for (int e = 0; e < E; ++e) a[c + e] = ok ? v[e] : (T)0;
            }
        } else {
#pragma unroll
            for (int c = 0; c < B; ++c) a[c] = (ok && c < g.kb) ? src[c] : (T)0;
        }
#pragma unroll
        for (int c = 0; c < B; ++c) {
            if (low && c > l32) a[c] = (T)0;
            if (low && !ok && c == l32) a[c] = (T)1;
        }
    }
    // the later columns of the group, blocks 1 .. own, in the matrix-core layout
    const int own = wave < 3 ? wave + 1 : 3;
    V4 C[3][2][2];
#pragma unroll
    for (int b = 0; b < 3; ++b)
        if (b < own)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int r = group0 + 16 * i + Mf<T>::row(grp, q), c = B * (b + 1) + 16 * j + l16;
                        const bool ok = r < glimit && c < g.kb && (wave == 3 || c <= r);
                        const T v = D[(long)min(r, rows - 1) * g.lda + min(c, g.kb - 1)];
                        C[b][i][j][q] = ok ? v : (T)(wave < 3 && r == c ? 1 : 0);
                    }
    __builtin_amdgcn_s_waitcnt(0);
    if (t == 0) {
        s_fail = 0;
        s_stop = info != 0;
    }
    __syncthreads();
    if (t == 0) {
        CholArrival m{g.arrive, info != 0};
        s_last = arrive::enter(m, (int)gridDim.x).last;
    }
    if (s_stop) return;
#pragma unroll
    for (int jb = 0; jb < 4; ++jb) {
        if (B * jb >= g.kb) break;
        const bool active = wave == 3 || wave >= jb;   // the wave's group lies below the diagonal rows
        if (active) {
            T dv;
            const int f = chol_columns<T, 0>(a, dv, g.kb - B * jb);
            if (f >= 0) {
                if (lane == 0) s_fail = 1;
                if (wave == 3 && lane == 0 && blockIdx.x == 0) {
                    *g.info = g.k0 + B * jb + f + 1;
                    *g.info_val = (double)dv;
                }
            }
            if (!low || wave == 3) {
                T *dst = Ls[low ? 4 : wave] + l32 * P;
#pragma unroll
                for (int c = 0; c < B; c += E) {
                    V v;
#pragma unroll
                    for (int e = 0; e < E; ++e) v[e] = a[c + e];
                    *reinterpret_cast<V *>(dst + c) = v;
                }
            }
        }
        __syncthreads();
        if (s_fail) return;
        // out: 256-byte (FP64) row segments; the diagonal block by the last arrival
        auto write_out = [&](const T *src, int r0, int limit) {
            constexpr int LPR = B / E, RPI = 64 / LPR;   // lanes per row, rows per store
#pragma unroll
            for (int i = 0; i < B / RPI; ++i) {
                const int rr = RPI * i + lane / LPR, c = E * (lane % LPR), cc = B * jb + c;
                const V v = *reinterpret_cast<const V *>(src + rr * P + c);
                if (r0 + rr < limit) {
                    T *dst = D + (long)(r0 + rr) * g.lda + cc;
                    if (cc + E <= g.kb) *reinterpret_cast<Vu *>(dst) = v;
                    else
#pragma unroll
                        for (int e = 0; e < E; ++e)
                            if (cc + e < g.kb) dst[e] = v[e];
                }
            }
        };
        if (wave == 3) write_out(Ls[3], chunk0, rows);
        if (s_last) {
            if (wave == 3) write_out(Ls[4], B * jb, g.kb);
            else if (active) write_out(Ls[wave], group0, g.kb);
        }
        if (B * (jb + 1) >= g.kb) break;
        // C -= L L^T on the later blocks; k-order: lane group grp, step i -> k = 8 grp + i.
        // Summed from zero: one rounding at C's magnitude per step instead of eight (mean
        // error of a solve, 300 matrices: n = 64 5.68e-16 -> 5.24e-16, n = 128 7.39e-16 ->
        // 6.22e-16, n = 1000 7.72e-16 -> 6.84e-16).
        if (active) {
            T lf[2][8];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int k = 0; k < 8; k += E) {
                    const V v = *reinterpret_cast<const V *>(Ls[wave] + (16 * i + l16) * P + 8 * grp + k);
#pragma unroll
                    for (int e = 0; e < E; ++e) lf[i][k + e] = -v[e];
                }
#pragma unroll
            for (int b = jb; b < 3; ++b)
                if (b < own) {
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        T rf[8];
#pragma unroll
                        for (int k = 0; k < 8; k += E) {
                            const V v = *reinterpret_cast<const V *>(Ls[b] + (16 * j + l16) * P + 8 * grp + k);
#pragma unroll
                            for (int e = 0; e < E; ++e) rf[k + e] = v[e];
                        }
                        V4 sum[2] = {};
#pragma unroll
                        for (int k = 0; k < 8; ++k)
#pragma unroll
                            for (int i = 0; i < 2; ++i) sum[i] = Mf<T>::mac(lf[i][k], rf[k], sum[i]);
#pragma unroll
                        for (int i = 0; i < 2; ++i) C[b][i][j] += sum[i];
                    }
                }
        }
        __syncthreads();
        // the next step's columns back to rows, through LDS
        if (active && jb < own) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        Ls[wave][(16 * i + Mf<T>::row(grp, q)) * P + 16 * j + l16] = C[jb < 3 ? jb : 0][i][j][q];
        }
        __syncthreads();
        {
            // (waves that are done read along: their rows then need no registers across the
            // update, which spills 100 of them otherwise)
            const T *src = Ls[low ? jb : wave] + l32 * P;
#pragma unroll
            for (int c = 0; c < B; c += E) {
                const V v = *reinterpret_cast<const V *>(src + c);
#pragma unroll
                for (int e = 0; e < E; ++e) a[c + e] = low && c + e > l32 ? (T)0 : v[e];
            }
        }
        __syncthreads();
    }
}

template <typename T>
__global__ void zero_upper_kernel(T *A, long lda, int n)
{
    long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long)n * n) return;
    int i = (int)(idx / n), j = (int)(idx % n);
    if (j > i) A[(long)i * lda + j] = (T)0;
}
} // namespace

// Look-ahead as in the LU: after block k's TRSM the main stream updates only
// the next block column (rows below it) and goes on to block k+1; the rest of
// the trailing lower triangle is updated on the side stream meanwhile.  Block
// k's side-stream update also covers block k+2's columns, so block k+1's
// next-column update waits for it.
template <typename T>
int scirs_potrf_device(int n, T *A, long lda, int kb, ScirsWork &w, hipStream_t stream)
{
    if (n <= 0 || kb <= 0 || kb > 128) return SCIRS_ERR_ARG;
    const bool lookahead = w.lookahead && w.side_stream && n > 2 * kb;
    if (lookahead) {
        SCIRS_HIP_CHECK(hipEventRecord(w.ev_start, stream));
        SCIRS_HIP_CHECK(hipStreamWaitEvent(w.side_stream, w.ev_start, 0));
    }
    for (int k0 = 0, p = 0; k0 < n; k0 += kb, ++p) {
        const int kbw = std::min(kb, n - k0);
        const int rest = n - k0 - kbw;
        CholPanelArgs<T> pa;
        pa.A = A; pa.lda = lda; pa.k0 = k0; pa.kb = kbw; pa.n = n;
        pa.arrive = w.chol_arrive; pa.info = w.info; pa.info_val = w.info_val;
        hipLaunchKernelGGL(chol_panel_kernel<T>, dim3(std::max(1, (rest + CP_B - 1) / CP_B)), dim3(NT), 0,
                           stream, pa);
        SCIRS_HIP_CHECK(hipGetLastError());
        if (rest > 0) {
            const T *L21 = A + (long)(k0 + kbw) * lda + k0;
            T *A22 = A + (long)(k0 + kbw) * lda + k0 + kbw;
            const int nn = lookahead ? std::min(kb, rest) : rest;   // columns updated on the main stream
            if (lookahead) {
                // the previous block's side-stream update covers these columns
                if (p > 0) SCIRS_HIP_CHECK(hipStreamWaitEvent(stream, w.ev_upd, 0));
                if (rest > nn) {
                    SCIRS_HIP_CHECK(hipEventRecord(w.ev_trsm, stream));
                    SCIRS_HIP_CHECK(hipStreamWaitEvent(w.side_stream, w.ev_trsm, 0));
                    int rc = scirs_syrk_update<T>(rest - nn, kbw, L21 + (long)nn * lda, lda,
                                                  A22 + (long)nn * lda + nn, lda, w, w.side_stream);
                    if (rc) return rc;
                }
                SCIRS_HIP_CHECK(hipEventRecord(w.ev_upd, w.side_stream));
                // A22[:, 0:nn) for every row below the block, in one launch (the strict
                // upper part of the nn x nn corner is updated too: it is never read,
                // and the factorisation zeroes it at the end)
                int rc = scirs_launch_gemm_sub_t<T>(rest, nn, kbw, L21, lda, L21, lda, A22, lda, w, stream);
                if (rc) return rc;
            } else {
                int rc = scirs_syrk_update<T>(rest, kbw, L21, lda, A22, lda, w, stream);
                if (rc) return rc;
            }
        }
        SCIRS_HIP_CHECK(hipGetLastError());
    }
    if (lookahead) {
        SCIRS_HIP_CHECK(hipEventRecord(w.ev_upd, w.side_stream));
        SCIRS_HIP_CHECK(hipStreamWaitEvent(stream, w.ev_upd, 0));
    }
    long total = (long)n * n;
    hipLaunchKernelGGL(zero_upper_kernel<T>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, A, lda, n);
    SCIRS_HIP_CHECK(hipGetLastError());
    return SCIRS_OK;
}

template int scirs_potrf_device<double>(int, double *, long, int, ScirsWork &, hipStream_t);
template int scirs_potrf_device<float>(int, float *, long, int, ScirsWork &, hipStream_t);
