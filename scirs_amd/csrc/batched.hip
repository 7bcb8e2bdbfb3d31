// Batched solves of many independent small systems of uneven size
// (n <= 256) in one call.
//
// There is no batched solve in the reference (scirs2-linalg/src/batch/mod.rs
// offers matmul/matvec/add/sum only); each system follows the reference's
// per-system semantics: `solve` (scirs2-linalg/src/solve.rs:54-111) for the
// general systems and the cholesky + two triangular solves composition
// (decomposition.rs:44, solve.rs:139) for the SPD ones, with the same
// breakdown tests (|pivot| < eps, a_ii - sum <= 0).
//
// Arithmetic: the factor is computed in FP32 (blocked right-looking LU with
// partial pivoting, or lower Cholesky), then FP64 refinement — residual
// r = b - A x from the FP64 input, correction with the FP32 factors — until
// the normwise backward error of every right-hand side is <= tol.  A system
// whose FP32 factorisation breaks down, or whose refinement stalls, is
// factored again in FP64 (the breakdown is then decided in FP64, as the
// reference decides it).
//
// Scheduling: the host sorts the systems by decreasing n.  One launch takes
// every system through FP32 and the refinement, one wave each
// (batched_wave.hpp); it marks those that need FP64, and a second launch takes
// these from a queue: n > wave_max by a 256-thread workgroup, smaller ones one
// per wave.  Without any it ends at once.  Batches whose workspace passes
// BATCH_WORK_MB take these launches chunk by chunk.
#include "common.hpp"
#include "kernels.hpp"
#include "prof.hpp"
#include "batched_wave.hpp"

namespace {

constexpr int NT = 256;
constexpr int NB = 32;          // panel width
constexpr int NMAX = 256;       // largest system handled

struct BatchDesc {
    int n, nrhs, spd, pad;
    long offA, offB;            // element offsets of A (n x n) and B/X (n x nrhs) in the packed buffers
    long offW;                  // element offset (FP64 units) of the factor workspace
};

struct BatchArgs {
    const BatchDesc *desc;
    const int *order;           // queue: system indices sorted by decreasing n
    int batch;
    const double *A; const double *B; double *X;
    double *work;               // factor workspace, work_doubles(n) per system
    int *perm;                  // n ints per system (offset = offA / n ... use offB-like index: offP)
    const long *offP;
    int *status;                // per system: 0 ok, k>0 breakdown column/row, -5 not converged
    int *iters;                 // per system: refinement steps
    double *bwd;                // per system: final backward error
    unsigned *counter;          // [0] queue head, [1] a system needs FP64; cleared ahead of the launches
    int wave_max;               // FP64: n <= wave_max -> one wave per system
    int max_iter;
    double tol_scale;           // tol = tol_scale * n * 2^-53 (per system)
};

// ----------------------------------------------------------------- team ops
// A team is either the whole workgroup (TEAM = 256) or one wave (TEAM = 64).
template <int TEAM>
__device__ __forceinline__ void team_sync()
{
    if (TEAM == NT) __syncthreads();
    else __builtin_amdgcn_wave_barrier();
}

// arg-max of |v| over the team, lowest index on ties; result in all threads
template <int TEAM, typename T>
__device__ __forceinline__ void team_argmax(T &v, int &idx, T *red_v, int *red_i)
{
    wave_argmax(v, idx);
    if (TEAM == NT) {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        if (lane == 0) { red_v[wave] = v; red_i[wave] = idx; }
        __syncthreads();
        v = red_v[0]; idx = red_i[0];
        for (int w = 1; w < NT / 64; ++w) {
            const int oi = red_i[w]; const T ov = red_v[w];
            if (oi >= 0 && (idx < 0 || ov > v || (ov == v && oi < idx))) { v = ov; idx = oi; }
        }
        __syncthreads();
    } else {
        v = __shfl(v, 0, 64);
        idx = __shfl(idx, 0, 64);
    }
}

template <int TEAM, typename T>
__device__ __forceinline__ T team_max(T v, T *red_v)
{
    v = wave_max(v);
    if (TEAM == NT) {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        if (lane == 0) red_v[wave] = v;
        __syncthreads();
        v = fmax(fmax(red_v[0], red_v[1]), fmax(red_v[2], red_v[3]));
        __syncthreads();
    } else {
        v = __shfl(v, 0, 64);
    }
    return v;
}

// Blocked right-looking LU with partial pivoting of the n x n matrix M
// (row-major, ld n, global workspace).  The NB-column panel is factored in
// LDS (pan: n x (NB+1)), the trailing update reads the panel from LDS.
// Returns 0 or the 1-based breakdown column.
template <int TEAM, typename T>
__device__ int team_getrf(int n, T *M, int *perm, T *pan, T *red_v, int *red_i, int tid)
{
    for (int i = tid; i < n; i += TEAM) perm[i] = i;
    const T eps = num_limits<T>::eps();
    for (int k0 = 0; k0 < n; k0 += NB) {
        const int kb = min(NB, n - k0);
        const int mrows = n - k0;
        team_sync<TEAM>();
        // stage the panel rows k0..n, columns k0..k0+kb
        for (int idx = tid; idx < mrows * NB; idx += TEAM) {
            const int r = idx / NB, c = idx % NB;
            pan[r * (NB + 1) + c] = c < kb ? M[(long)(k0 + r) * n + k0 + c] : (T)0;
        }
        team_sync<TEAM>();
        for (int j = 0; j < kb; ++j) {
            T bv = (T)0; int bi = -1;
            for (int r = j + tid; r < mrows; r += TEAM) {
                const T v = fabs(pan[r * (NB + 1) + j]);
                if (bi < 0 || v > bv) { bv = v; bi = r; }
            }
            team_argmax<TEAM>(bv, bi, red_v, red_i);
            if (!(bv >= eps)) return k0 + j + 1;
            const int p = bi;
            if (p != j) {
                // swap inside the panel, and the whole row outside it
                for (int c = tid; c < NB; c += TEAM) {
                    const T a = pan[j * (NB + 1) + c];
                    pan[j * (NB + 1) + c] = pan[p * (NB + 1) + c];
                    pan[p * (NB + 1) + c] = a;
                }
                for (int c = tid; c < n; c += TEAM) {
                    if (c >= k0 && c < k0 + kb) continue;
                    const T a = M[(long)(k0 + j) * n + c];
                    M[(long)(k0 + j) * n + c] = M[(long)(k0 + p) * n + c];
                    M[(long)(k0 + p) * n + c] = a;
                }
                if (tid == 0) {
                    const int tmp = perm[k0 + j]; perm[k0 + j] = perm[k0 + p]; perm[k0 + p] = tmp;
                }
            }
            team_sync<TEAM>();
            const T piv = pan[j * (NB + 1) + j];
            for (int r = j + 1 + tid; r < mrows; r += TEAM) pan[r * (NB + 1) + j] /= piv;
            team_sync<TEAM>();
            const int ncol = kb - j - 1;
            if (ncol > 0)
                for (int w = tid; w < (mrows - j - 1) * ncol; w += TEAM) {
                    const int r = j + 1 + w / ncol, c = j + 1 + w % ncol;
                    pan[r * (NB + 1) + c] -= pan[r * (NB + 1) + j] * pan[j * (NB + 1) + c];
                }
            team_sync<TEAM>();
        }
        // write the panel back
        for (int idx = tid; idx < mrows * kb; idx += TEAM) {
            const int r = idx / kb, c = idx % kb;
            M[(long)(k0 + r) * n + k0 + c] = pan[r * (NB + 1) + c];
        }
        team_sync<TEAM>();
        const int c1 = k0 + kb;
        if (c1 >= n) continue;
        const int rows = n - c1, cols = n - c1;
        // U12 = L11^-1 A12 in memory (registers for 32 doubles would spill in this kernel)
        for (int c = c1 + tid; c < n; c += TEAM)
            for (int i = 1; i < kb; ++i) {
                T sv = M[(long)(k0 + i) * n + c];
                for (int q = 0; q < i; ++q) sv -= pan[i * (NB + 1) + q] * M[(long)(k0 + q) * n + c];
                M[(long)(k0 + i) * n + c] = sv;
            }
        team_sync<TEAM>();
        // A22 -= L21 U12
        for (int w = tid; w < rows * cols; w += TEAM) {
            const int r = w / cols, c = w % cols;
            const T *lr = pan + (kb + r) * (NB + 1);
            T sv = (T)0;
#pragma unroll 8
            for (int q = 0; q < NB; ++q)
                if (q < kb) sv += lr[q] * M[(long)(k0 + q) * n + c1 + c];
            M[(long)(c1 + r) * n + c1 + c] -= sv;
        }
    }
    team_sync<TEAM>();
    return 0;
}

// Lower Cholesky (right-looking, unblocked over NB-column panels in LDS), only
// the lower triangle of M is read.  Returns 0 or the 1-based failing row.
template <int TEAM, typename T>
__device__ int team_potrf(int n, T *M, T *pan, int tid)
{
    for (int k0 = 0; k0 < n; k0 += NB) {
        const int kb = min(NB, n - k0);
        const int mrows = n - k0;
        team_sync<TEAM>();
        for (int idx = tid; idx < mrows * NB; idx += TEAM) {
            const int r = idx / NB, c = idx % NB;
            pan[r * (NB + 1) + c] = (c < kb && c <= r) ? M[(long)(k0 + r) * n + k0 + c] : (T)0;
        }
        team_sync<TEAM>();
        for (int j = 0; j < kb; ++j) {
            const T d = pan[j * (NB + 1) + j];
            if (!(d > (T)0)) return k0 + j + 1;
            const T l = sqrt(d);
            team_sync<TEAM>();
            for (int r = j + tid; r < mrows; r += TEAM) pan[r * (NB + 1) + j] = (r == j) ? l : pan[r * (NB + 1) + j] / l;
            team_sync<TEAM>();
            const int ncol = kb - j - 1;
            if (ncol > 0)
                for (int w = tid; w < (mrows - j - 1) * ncol; w += TEAM) {
                    const int r = j + 1 + w / ncol, c = j + 1 + w % ncol;
                    if (c <= r) pan[r * (NB + 1) + c] -= pan[r * (NB + 1) + j] * pan[c * (NB + 1) + j];
                }
            team_sync<TEAM>();
        }
        for (int idx = tid; idx < mrows * kb; idx += TEAM) {
            const int r = idx / kb, c = idx % kb;
            if (c <= r) M[(long)(k0 + r) * n + k0 + c] = pan[r * (NB + 1) + c];
        }
        team_sync<TEAM>();
        const int c1 = k0 + kb;
        if (c1 >= n) continue;
        // A22 (lower) -= L21 L21^T
        const int rows = n - c1;
        for (int w = tid; w < rows * rows; w += TEAM) {
            const int r = w / rows, c = w % rows;
            if (c > r) continue;
            const T *lr = pan + (kb + r) * (NB + 1);
            const T *lc = pan + (kb + c) * (NB + 1);
            T sv = (T)0;
            // the panel's columns past kb are zero
#pragma unroll 8
            for (int q = 0; q < NB; ++q) sv += lr[q] * lc[q];
            M[(long)(c1 + r) * n + c1 + c] -= sv;
        }
    }
    team_sync<TEAM>();
    return 0;
}

// d <- op^-1 d with the factors in M, column by column (d in LDS, length n): every thread reads the finished d[i], then
// the team removes its contribution from the remaining entries (one sync per row).
// LU: L unit lower then U; Cholesky: L then L^T.
template <int TEAM, typename T, typename V>
__device__ void team_subst_cols(int n, const T *M, V *d, bool chol, int tid)
{
    for (int i = 0; i < n; ++i) {
        V xi = d[i];
        if (chol) xi /= (V)M[(long)i * n + i];
        for (int r = i + 1 + tid; r < n; r += TEAM) d[r] -= (V)M[(long)r * n + i] * xi;
        team_sync<TEAM>();
        if (tid == 0 && chol) d[i] = xi;
        team_sync<TEAM>();
    }
    for (int i = n - 1; i >= 0; --i) {
        const V xi = d[i] / (V)M[(long)i * n + i];
        for (int r = tid; r < i; r += TEAM)
            d[r] -= (V)(chol ? M[(long)i * n + r] : M[(long)r * n + i]) * xi;
        team_sync<TEAM>();
        if (tid == 0) d[i] = xi;
        team_sync<TEAM>();
    }
}

// Solve one system with a team, in FP64: factor + refinement.
template <int TEAM>
__device__ void team_solve(const BatchArgs &a, int sys, double *pan, double *vec, double *red, int *redi, int tid)
{
    const BatchDesc d = a.desc[sys];
    const int n = d.n, nrhs = d.nrhs;
    const double *A = a.A + d.offA;
    const double *B = a.B + d.offB;
    double *X = a.X + d.offB;
    int *perm = a.perm + a.offP[sys];
    double *W = a.work + d.offW;
    const double tol = a.tol_scale * n * 0x1p-53;

    // ||A||_inf
    double an = 0.0;
    for (int r = tid; r < n; r += TEAM) {
        double s = 0.0;
        for (int c = 0; c < n; ++c) s += fabs(A[(long)r * n + c]);
        an = fmax(an, s);
    }
    an = team_max<TEAM>(an, red);

    int it_used = 0;
    double worst = 0.0;
    const bool chol = d.spd != 0;
    // copy A into the workspace and factor
    for (int idx = tid; idx < n * n; idx += TEAM) W[idx] = A[idx];
    team_sync<TEAM>();
    const int status = chol ? team_potrf<TEAM, double>(n, W, pan, tid)
                            : team_getrf<TEAM, double>(n, W, perm, pan, red, redi, tid);
    if (status == 0) {
        // refinement for each right-hand side
        for (int j = 0; j < nrhs; ++j) {
            for (int r = tid; r < n; r += TEAM) X[(long)r * nrhs + j] = 0.0;
            team_sync<TEAM>();
            double bn = 0.0;
            for (int r = tid; r < n; r += TEAM) bn = fmax(bn, fabs(B[(long)r * nrhs + j]));
            bn = team_max<TEAM>(bn, red);
            double eta = 1.0, prev = INFINITY;
            int it = 0;
            for (; it <= a.max_iter; ++it) {
                // r = b - A x  (FP64), stored in vec: one wave per row, the
                // lanes over the columns (coalesced row reads)
                double rn = 0.0, xn = 0.0;
                {
                    const int lane = tid & 63;
                    for (int r = tid >> 6; r < n; r += TEAM / 64) {
                        double ax = 0.0;
                        for (int c = lane; c < n; c += 64) ax += A[(long)r * n + c] * X[(long)c * nrhs + j];
                        ax = wave_sum(ax);
                        const double rv = B[(long)r * nrhs + j] - ax;
                        if (lane == 0) vec[r] = rv;
                        rn = fmax(rn, fabs(rv));
                    }
                    for (int r = tid; r < n; r += TEAM) xn = fmax(xn, fabs(X[(long)r * nrhs + j]));
                }
                team_sync<TEAM>();
                rn = team_max<TEAM>(rn, red);
                xn = team_max<TEAM>(xn, red);
                const double den = an * xn + bn;
                eta = den > 0 ? rn / den : (rn > 0 ? INFINITY : 0.0);
                if (eta <= tol) break;
                if (it == a.max_iter || (it >= 2 && !(eta < 0.5 * prev))) break;
                prev = eta;
                // permute for LU: d = P r
                if (!chol) {
                    team_sync<TEAM>();
                    double *tmp = vec + NMAX;
                    for (int r = tid; r < n; r += TEAM) tmp[r] = vec[perm[r]];
                    team_sync<TEAM>();
                    for (int r = tid; r < n; r += TEAM) vec[r] = tmp[r];
                }
                team_sync<TEAM>();
                team_subst_cols<TEAM, double, double>(n, W, vec, chol, tid);
                for (int r = tid; r < n; r += TEAM) X[(long)r * nrhs + j] += vec[r];
                team_sync<TEAM>();
            }
            it_used = max(it_used, it);
            worst = fmax(worst, eta);
        }
    }
    if (tid == 0) {
        a.status[sys] = status;
        a.iters[sys] = it_used;
        a.bwd[sys] = worst;
    }
    team_sync<TEAM>();
}

__global__ void batched_reset_kernel(unsigned *counter) { counter[threadIdx.x] = 0u; }

// FP64 launch: systems up to this size one per wave, larger ones by a whole workgroup
// (NMAX / 4 is what a wave's slice of LDS holds; 4000 systems of 33 to 64 rows: 1.4 ms, by
// workgroups 3.1; 8000 of 8 to 32: 0.86 and 1.9)
constexpr int FP64_WAVE_MAX = NMAX / 4;
// Workspace of a batch, MiB: a padded system takes up to 40 times what its matrix does
// (5 KB for n <= 16), so larger batches run in several chunks that share it.  Half of
// the factors of 65,000 systems of 256 rows; a chunk of systems of 16 rows is 1.6 million.
constexpr long BATCH_WORK_MB = 8192;
constexpr int NEED_FP64 = -1000;     // status between the two launches

// systems order[0..gridDim.x), all of one kind
template <bool CHOL>
__global__ __launch_bounds__(64, 2) void batched_wave_kernel(BatchArgs a, const int *order)
{
    extern __shared__ __align__(16) char wave_lds[];
    const int sys = order[blockIdx.x];
    const BatchDesc d = a.desc[sys];
    int iters = 0;
    double bwd = 0.0;
    const bool ok = wave::solve<CHOL>(d.n, d.nrhs, a.A + d.offA, a.B + d.offB, a.X + d.offB, a.work + d.offW,
                                      a.tol_scale * d.n * 0x1p-53, a.max_iter, wave_lds, threadIdx.x, &iters, &bwd);
    if (threadIdx.x == 0) {
        a.status[sys] = ok ? 0 : NEED_FP64;
        a.iters[sys] = iters;
        a.bwd[sys] = bwd;
        if (!ok) __hip_atomic_store(a.counter + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// the systems that need FP64, one workgroup or wave each
__global__ __launch_bounds__(NT) void batched_solve_kernel(BatchArgs a)
{
    // one NMAX x (NB+1) FP64 panel for a whole-workgroup system, or four
    // (NMAX/4) x (NB+1) slices, one per wave, for small systems
    __shared__ double panbuf[NMAX * (NB + 1)];
    __shared__ double vec[4][2 * NMAX];
    __shared__ double red[8];
    __shared__ int redi[8];
    __shared__ int s_item;
    constexpr int SLICE = NMAX / 4 * (NB + 1);   // doubles per wave slice
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    if (a.counter[1] == 0u) return;
    while (true) {
        if (t == 0) s_item = (int)atomicAdd(a.counter, 4u);
        __syncthreads();
        const int item = s_item;
        __syncthreads();
        if (item >= a.batch) break;
        for (int q = 0; q < 4 && item + q < a.batch; ++q) {
            const int sys = a.order[item + q];
            if (a.desc[sys].n > a.wave_max) {
                const bool mine = a.status[sys] == NEED_FP64;
                __syncthreads();   // read by every wave before the result is written
                if (mine) team_solve<NT>(a, sys, panbuf, &vec[0][0], red, redi, t);
            } else {
                // the remaining small entries of this pop: one per wave
                const int qq = q + wave;
                if (qq < 4 && item + qq < a.batch) {
                    const int s2 = a.order[item + qq];
                    if (a.status[s2] == NEED_FP64)
                        team_solve<64>(a, s2, panbuf + (size_t)wave * SLICE, vec[wave], red + 2 * wave, redi + 2 * wave,
                                       lane);
                }
                __syncthreads();
                break;
            }
        }
        __syncthreads();
    }
}
} // namespace

// ===================================================================== host
#include "api_internal.hpp"
#include <string>
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

namespace {

// Systems that share the workspace: order[first .. first + count), of which `general` are
// general ones (kinds: those first, then the positive definite ones, each by size).
struct BatchChunk { int first, count, general; };

struct BatchPlan {
    uint64_t key = 0;
    int batch = 0;
    BatchDesc *d_desc = nullptr;
    int *d_order = nullptr, *d_kinds = nullptr;   // by size; within a chunk by kind and size
    std::vector<BatchChunk> chunks;
    long *d_offP = nullptr;
    int *d_status = nullptr, *d_iters = nullptr;
    double *d_bwd = nullptr;
    double *d_work = nullptr;
    int *d_perm = nullptr;
    unsigned *d_counter = nullptr;
    size_t cap_batch = 0, cap_work = 0, cap_perm = 0;
    hipGraphExec_t exec = nullptr;
    hipGraph_t graph = nullptr;
    int graph_wave_max = -1;
    int nmax = 0;
};

BatchPlan g_plan;
// FNV-1a over 8-byte words (a last partial word is padded with zeros)
uint64_t fnv1a(uint64_t h, const void *p, size_t n)
{
    const unsigned char *b = (const unsigned char *)p;
    for (size_t i = 0; i < n; i += 8) {
        uint64_t w = 0;
        memcpy(&w, b + i, std::min<size_t>(8, n - i));
        h ^= w;
        h *= 1099511628211ull;
        h ^= h >> 32;
    }
    return h;
}

template <typename T>
int grow(T **p, size_t *cap, size_t count)
{
    if (*cap >= count && *p) return SCIRS_OK;
    if (*p) {
        SCIRS_HIP_CHECK(hipDeviceSynchronize());
        SCIRS_HIP_CHECK(hipFree(*p));
        *p = nullptr;
    }
    if (hipMalloc((void **)p, std::max<size_t>(count, 1) * sizeof(T)) != hipSuccess) {
        scirs_set_error("batched: hipMalloc of %zu bytes failed", count * sizeof(T));
        *cap = 0;
        return SCIRS_ERR_NOMEM;
    }
    *cap = count;
    return SCIRS_OK;
}

int launch_batch(BatchPlan &pl, const double *dA, const double *dB, double *dX, int wave_max, int max_iter,
                 double tol_scale, hipStream_t s)
{
    BatchArgs a;
    a.desc = pl.d_desc;
    a.A = dA; a.B = dB; a.X = dX; a.work = pl.d_work; a.perm = pl.d_perm; a.offP = pl.d_offP;
    a.status = pl.d_status; a.iters = pl.d_iters; a.bwd = pl.d_bwd; a.counter = pl.d_counter;
    a.wave_max = wave_max; a.max_iter = max_iter; a.tol_scale = tol_scale;
    for (const BatchChunk &ch : pl.chunks) {
        a.order = pl.d_order + ch.first;
        a.batch = ch.count;
        const int *kinds = pl.d_kinds + ch.first;
        hipLaunchKernelGGL(batched_reset_kernel, dim3(1), dim3(2), 0, s, pl.d_counter);
        if (ch.general)
            hipLaunchKernelGGL(batched_wave_kernel<false>, dim3(ch.general), dim3(64), wave::lds_bytes(pl.nmax), s, a,
                               kinds);
        if (ch.general < ch.count)
            hipLaunchKernelGGL(batched_wave_kernel<true>, dim3(ch.count - ch.general), dim3(64),
                               wave::lds_bytes(pl.nmax), s, a, kinds + ch.general);
        // a persistent grid: one workgroup per CU (LDS allows one) pulls work from the queue
        const int grid = std::min(ch.count, scirs::ctx().cu_count);
        hipLaunchKernelGGL(batched_solve_kernel, dim3(grid), dim3(NT), 0, s, a);
    }
    SCIRS_HIP_CHECK(hipGetLastError());
    return SCIRS_OK;
}

} // namespace

extern "C" int scirs_gpu_dgesv_batched_dev(int batch, const int *n, const int *nrhs, const unsigned char *spd,
                                           const double *dA, const int64_t *offA, const double *dB,
                                           const int64_t *offB, double *dX, int *status, double *bwd,
                                           int max_iter, double tol_scale, void *stream, scirs_batch_info *info)
{
    using namespace scirs;
    const double t0 = now_ms();
    if (info) memset(info, 0, sizeof(*info));
    if (batch <= 0 || !n || !nrhs || !dA || !offA || !dB || !offB || !dX || !status) {
        scirs_set_error("dgesv_batched: invalid arguments");
        return SCIRS_ERR_ARG;
    }
    for (int i = 0; i < batch; ++i)
        if (n[i] < 1 || n[i] > NMAX || nrhs[i] < 1 || nrhs[i] > 16) {
            scirs_set_error("dgesv_batched: system %d has n=%d nrhs=%d (1 <= n <= %d, 1 <= nrhs <= 16)", i, n[i],
                            nrhs[i], NMAX);
            return SCIRS_ERR_ARG;
        }
    if (max_iter <= 0) max_iter = 10;
    if (!(tol_scale > 0)) tol_scale = 1.0;
    std::lock_guard<std::recursive_mutex> lk(ctx().mu);
    Context &c = ctx();
    int rc = c.init(0);
    if (rc) return rc;
    hipStream_t s = (hipStream_t)stream;   // NULL: the default stream, ordered after the caller's work on it
    BatchPlan &pl = g_plan;

    // ---- plan: descriptors, size-sorted queue, workspace (rebuilt when the batch changes)
    uint64_t key = 1469598103934665603ull;
    key = fnv1a(key, &batch, sizeof(batch));
    key = fnv1a(key, n, sizeof(int) * batch);
    key = fnv1a(key, nrhs, sizeof(int) * batch);
    if (spd) key = fnv1a(key, spd, batch);
    key = fnv1a(key, offA, sizeof(int64_t) * batch);
    key = fnv1a(key, offB, sizeof(int64_t) * batch);
    const void *ptrs[3] = {dA, dB, dX};
    key = fnv1a(key, ptrs, sizeof(ptrs));
    key = fnv1a(key, &max_iter, sizeof(max_iter));
    key = fnv1a(key, &tol_scale, sizeof(tol_scale));
    const char *wl = getenv("SCIRS_GPU_BATCH_WORK_MB");
    const long limit = (wl && *wl && atol(wl) > 0 ? atol(wl) : BATCH_WORK_MB) * (1l << 17);   // doubles
    key = fnv1a(key, &limit, sizeof(limit));
    const bool same = (pl.key == key && pl.batch == batch);
    if (!same) {
        pl.key = 0;       // no plan until this one is complete
        pl.batch = 0;
        std::vector<BatchDesc> desc(batch);
        std::vector<long> offP(batch);
        long work = 0, pw = 0;
        int nmax = 0;
        for (int i = 0; i < batch; ++i) {
            desc[i].n = n[i]; desc[i].nrhs = nrhs[i]; desc[i].spd = spd ? spd[i] : 0; desc[i].pad = 0;
            desc[i].offA = offA[i]; desc[i].offB = offB[i];
            offP[i] = pw; pw += n[i];
            nmax = std::max(nmax, n[i]);
        }
        std::vector<int> order(batch);
        for (int i = 0; i < batch; ++i) order[i] = i;
        std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return n[x] > n[y]; });
        std::vector<int> kinds;
        // chunks of at most lim doubles of workspace
        auto cut = [&](long lim) {
            kinds = order;
            pl.chunks.clear();
            work = 0;
            for (int first = 0; first < batch;) {
                int last = first;
                long used = 0;
                for (; last < batch; ++last) {
                    const int ni = n[order[last]];
                    const long need = std::max(((long)ni * ni + 15) & ~15L, wave::work_doubles(ni));
                    if (last > first && used + need > lim) break;
                    desc[order[last]].offW = used;
                    used += need;
                }
                work = std::max(work, used);
                const auto k0 = kinds.begin() + first;
                const auto mid = std::stable_partition(k0, kinds.begin() + last, [&](int x) { return !desc[x].spd; });
                pl.chunks.push_back(BatchChunk{first, last - first, (int)(mid - k0)});
                first = last;
            }
        };
        // smaller chunks where memory is short
        for (long lim = limit;; lim /= 4) {
            cut(lim);
            if (!(rc = grow(&pl.d_work, &pl.cap_work, (size_t)work))) break;
            (void)hipGetLastError();
            if (lim < (1l << 20)) return rc;
        }
        if ((rc = grow(&pl.d_desc, &pl.cap_batch, batch))) return rc;
        size_t cap1 = 0, cap2 = 0, cap3 = 0, cap4 = 0, cap5 = 0, cap6 = 0;
        // the per-system arrays are (re)allocated together with the descriptors
        if (pl.d_order) { (void)hipFree(pl.d_order); (void)hipFree(pl.d_kinds); pl.d_kinds = nullptr; (void)hipFree(pl.d_offP); (void)hipFree(pl.d_status);
                          (void)hipFree(pl.d_iters); (void)hipFree(pl.d_bwd); pl.d_order = nullptr; pl.d_offP = nullptr;
                          pl.d_status = nullptr; pl.d_iters = nullptr; pl.d_bwd = nullptr; }
        if ((rc = grow(&pl.d_order, &cap2, batch)) || (rc = grow(&pl.d_kinds, &cap1, batch)) || (rc = grow(&pl.d_offP, &cap3, batch)) ||
            (rc = grow(&pl.d_status, &cap4, batch)) || (rc = grow(&pl.d_iters, &cap5, batch)) ||
            (rc = grow(&pl.d_bwd, &cap6, batch)))
            return rc;
        if ((rc = grow(&pl.d_perm, &pl.cap_perm, (size_t)pw))) return rc;
        if (!pl.d_counter) {
            size_t cc = 0;
            if ((rc = grow(&pl.d_counter, &cc, 64))) return rc;
        }
        SCIRS_HIP_CHECK(hipMemcpy(pl.d_desc, desc.data(), sizeof(BatchDesc) * batch, hipMemcpyHostToDevice));
        SCIRS_HIP_CHECK(hipMemcpy(pl.d_order, order.data(), sizeof(int) * batch, hipMemcpyHostToDevice));
        SCIRS_HIP_CHECK(hipMemcpy(pl.d_kinds, kinds.data(), sizeof(int) * batch, hipMemcpyHostToDevice));
        SCIRS_HIP_CHECK(hipMemcpy(pl.d_offP, offP.data(), sizeof(long) * batch, hipMemcpyHostToDevice));
        if (pl.exec) { (void)hipGraphExecDestroy(pl.exec); pl.exec = nullptr; }
        if (pl.graph) { (void)hipGraphDestroy(pl.graph); pl.graph = nullptr; }
        pl.key = key;
        pl.batch = batch;
        pl.nmax = nmax;
    }

    // crossover of the FP64 launch; a wave's LDS slice holds systems up to NMAX / 4 rows
    int wave_max = FP64_WAVE_MAX;
    const char *wm = getenv("SCIRS_GPU_BATCH_WAVE_MAX");
    if (wm && *wm && atoi(wm) >= 0) wave_max = atoi(wm);
    wave_max = std::min(wave_max, NMAX / 4);

    // ---- one graph per plan and crossover: [reset queue, FP32 solve, FP64 solve], replayed
    bool replay = true;
    if (!pl.exec || pl.graph_wave_max != wave_max) {
        replay = false;
        if (pl.exec) { (void)hipGraphExecDestroy(pl.exec); pl.exec = nullptr; }
        if (pl.graph) { (void)hipGraphDestroy(pl.graph); pl.graph = nullptr; }
        SCIRS_HIP_CHECK(hipStreamSynchronize(s));
        SCIRS_HIP_CHECK(hipStreamBeginCapture(c.stream, hipStreamCaptureModeRelaxed));
        rc = launch_batch(pl, dA, dB, dX, wave_max, max_iter, tol_scale, c.stream);
        hipGraph_t g = nullptr;
        hipError_t ce = hipStreamEndCapture(c.stream, &g);
        if (rc) return rc;
        if (ce != hipSuccess) {
            scirs_set_error("batched: graph capture failed: %s", hipGetErrorString(ce));
            return SCIRS_ERR_HIP;
        }
        pl.graph = g;
        SCIRS_HIP_CHECK(hipGraphInstantiate(&pl.exec, pl.graph, nullptr, nullptr, 0));
        pl.graph_wave_max = wave_max;
    }
    scirs::CallEvents ev;
    if (int erc = ev.create(2)) return erc;
    hipEvent_t e0 = ev.e[0], e1 = ev.e[1];
    SCIRS_HIP_CHECK(hipEventRecord(e0, s));
    {
        scirs::ProfScope prof(SCIRS_PROF_OTHER, 0.0, 0.0, s);
        SCIRS_HIP_CHECK(hipGraphLaunch(pl.exec, s));
    }
    SCIRS_HIP_CHECK(hipEventRecord(e1, s));
    SCIRS_HIP_CHECK(hipEventSynchronize(e1));
    float ms = 0;
    SCIRS_HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));

    std::vector<int> iters(batch);
    std::vector<double> bw(batch);
    SCIRS_HIP_CHECK(hipMemcpy(status, pl.d_status, sizeof(int) * batch, hipMemcpyDeviceToHost));
    SCIRS_HIP_CHECK(hipMemcpy(iters.data(), pl.d_iters, sizeof(int) * batch, hipMemcpyDeviceToHost));
    SCIRS_HIP_CHECK(hipMemcpy(bw.data(), pl.d_bwd, sizeof(double) * batch, hipMemcpyDeviceToHost));
    if (bwd) memcpy(bwd, bw.data(), sizeof(double) * batch);
    int failed = 0, maxit = 0;
    double maxb = 0;
    for (int i = 0; i < batch; ++i) {
        failed += status[i] != 0;
        maxit = std::max(maxit, iters[i]);
        if (status[i] == 0) maxb = std::max(maxb, bw[i]);
    }
    if (info) {
        info->failed = failed;
        info->max_iters = maxit;
        info->max_backward_error = maxb;
        info->time_ms = ms;
        info->wave_max = wave_max;
        info->graph_replayed = replay ? 1 : 0;
        info->total_ms = now_ms() - t0;
    }
    return SCIRS_OK;
}

// ---------------------------------------------------------------- host memory
// Host-memory batched solve: the systems are packed into pinned staging, sent
// in one copy, solved by the device entry point above, and the solutions come
// back in one copy.  Staging (pinned and device) is kept between calls and
// grown on demand, so a repeated batch of the same shape replays the cached
// graph on the same device buffers.
namespace {
struct HostBatch {
    double *h = nullptr;   // pinned: packed A | packed B (X on the way back)
    size_t hcap = 0;
    double *d = nullptr;   // device: packed A | packed B | packed X
    size_t dcap = 0;
};
HostBatch g_hb;

int grow_pinned(double **p, size_t *cap, size_t count)
{
    if (*cap >= count && *p) return SCIRS_OK;
    if (*p) {
        SCIRS_HIP_CHECK(hipDeviceSynchronize());
        SCIRS_HIP_CHECK(hipHostFree(*p));
        *p = nullptr;
    }
    if (hipHostMalloc((void **)p, std::max<size_t>(count, 1) * sizeof(double), hipHostMallocDefault) != hipSuccess) {
        scirs_set_error("batched: pinned allocation of %zu bytes failed", count * sizeof(double));
        *cap = 0;
        return SCIRS_ERR_NOMEM;
    }
    *cap = count;
    return SCIRS_OK;
}
} // namespace

extern "C" int scirs_gpu_dgesv_batched(int batch, const int *n, const int *nrhs, const unsigned char *spd,
                                       const double *const *A, const int64_t *lda, const double *const *B,
                                       const int64_t *ldb, double *const *X, const int64_t *ldx, int *status,
                                       double *bwd, int max_iter, double tol_scale, scirs_batch_info *info)
{
    using namespace scirs;
    const double t0 = now_ms();
    if (info) memset(info, 0, sizeof(*info));
    if (batch <= 0 || !n || !nrhs || !A || !lda || !B || !ldb || !X || !ldx || !status) {
        scirs_set_error("dgesv_batched: invalid arguments");
        return SCIRS_ERR_ARG;
    }
    std::vector<int64_t> offA(batch), offB(batch);
    size_t na = 0, nb = 0;
    for (int i = 0; i < batch; ++i) {
        if (n[i] < 1 || n[i] > NMAX || nrhs[i] < 1 || nrhs[i] > 16 || !A[i] || !B[i] || !X[i] || lda[i] < n[i] ||
            ldb[i] < nrhs[i] || ldx[i] < nrhs[i]) {
            scirs_set_error("dgesv_batched: system %d has n=%d nrhs=%d lda=%lld ldb=%lld ldx=%lld or a null pointer "
                            "(1 <= n <= %d, 1 <= nrhs <= 16, leading dimensions >= the row length)",
                            i, n[i], nrhs[i], (long long)lda[i], (long long)ldb[i], (long long)ldx[i], NMAX);
            return SCIRS_ERR_ARG;
        }
        offA[i] = (int64_t)na;
        offB[i] = (int64_t)nb;
        na += (size_t)n[i] * n[i];
        nb += (size_t)n[i] * nrhs[i];
    }
    std::lock_guard<std::recursive_mutex> lk(ctx().mu);
    Context &c = ctx();
    if (int rc = c.init(0)) return rc;
    hipStream_t s = c.stream;
    HostBatch &hb = g_hb;
    if (int rc = grow_pinned(&hb.h, &hb.hcap, na + nb)) return rc;
    if (int rc = grow(&hb.d, &hb.dcap, na + 2 * nb)) return rc;
    double *hA = hb.h, *hB = hb.h + na;
    for (int i = 0; i < batch; ++i) {
        const int ni = n[i], ri = nrhs[i];
        for (int r = 0; r < ni; ++r) {
            memcpy(hA + offA[i] + (size_t)r * ni, A[i] + (size_t)r * lda[i], sizeof(double) * ni);
            memcpy(hB + offB[i] + (size_t)r * ri, B[i] + (size_t)r * ldb[i], sizeof(double) * ri);
        }
    }
    double *dA = hb.d, *dB = hb.d + na, *dX = hb.d + na + nb;
    SCIRS_HIP_CHECK(hipMemcpyAsync(dA, hA, sizeof(double) * (na + nb), hipMemcpyHostToDevice, s));
    int rc = scirs_gpu_dgesv_batched_dev(batch, n, nrhs, spd, dA, offA.data(), dB, offB.data(), dX, status, bwd,
                                         max_iter, tol_scale, s, info);
    if (rc) return rc;
    SCIRS_HIP_CHECK(hipMemcpyAsync(hB, dX, sizeof(double) * nb, hipMemcpyDeviceToHost, s));
    SCIRS_HIP_CHECK(hipStreamSynchronize(s));
    for (int i = 0; i < batch; ++i) {
        const int ni = n[i], ri = nrhs[i];
        for (int r = 0; r < ni; ++r)
            memcpy(X[i] + (size_t)r * ldx[i], hB + offB[i] + (size_t)r * ri, sizeof(double) * ri);
    }
    if (info) info->total_ms = now_ms() - t0;
    return SCIRS_OK;
}
