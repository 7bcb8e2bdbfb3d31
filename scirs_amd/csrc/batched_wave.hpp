// One system of a batch by one wave: FP32 factor (LU with partial pivoting or lower
// Cholesky) and FP64 refinement, the semantics described at the top of batched.hip.
//
// What bounds it: a small system is a chain of short dependent steps (one per column of
// the factor, one per 16 rows of each substitution), so the chip is filled with many
// systems rather than one system with many threads.  A wave needs no barrier and no
// exchange through LDS between steps, and eight waves per CU cover each other's
// waits.  Everything else is arranged in 16 x 16 blocks for the matrix cores:
//   - the factor runs over panels of 16 columns held in registers, one row per lane and
//     64 rows per register set; the pivot row is broadcast through scalar registers and
//     rows stay where they are in memory: `map` holds the row behind each position
//   - two panels share one trailing update (one update per panel: 5.6 and 4.7 ms instead of
//     4.8 and 3.4 for the two kinds); it computes the transposed product, so that
//     each lane holds four neighbouring elements of one row of A22 (16-byte accesses)
//   - the 16 x 16 diagonal blocks of the factors are inverted once, in FP64; the
//     substitutions are then products only, for up to four right-hand sides at a time
//   - residual rows come straight from A, 64 bytes per lane
// 20000 systems of n ~ U[8,256], half of them Cholesky, 1 or 4 right-hand sides (3.6 GB
// of input): 8.1 ms (general 4.7, SPD 3.4); 99.6 ms with a 256-thread workgroup per system,
// columns in LDS and substitutions in vector arithmetic.  What is left is HBM traffic: with
// 2048 systems under way nothing stays in L2, A is read once to convert it and once per
// refinement step, and the general systems moved 24.7 GB (4.2 TB/s; a copy reaches 4.8)
// while each panel had its own update.
#pragma once
#include "common.hpp"
#include "lanes.hpp"

namespace wave {

using lanes::d4;
using lanes::f4;
typedef unsigned u32;
constexpr int KB = 16;          // panel width and block size
constexpr int QR = 4;           // right-hand sides per pass
constexpr int LU_ROW = 68;      // LDS row of the staged U12 (32 x 64), padded off the banks

__host__ __device__ constexpr int pad16(int n) { return (n + 15) & ~15; }
// LDS of a wave whose systems have n <= nmax: two vector blocks of QR columns (together they
// double as the staged U12) and the two row maps
__host__ __device__ constexpr int ld_vec(int n) { return ((n + 31) & ~31) + 2; }
__host__ __device__ constexpr size_t vec_bytes(int n)
{
    return (size_t)QR * ld_vec(n) * 8 > KB * LU_ROW * 4 ? (size_t)QR * ld_vec(n) * 8 : KB * LU_ROW * 4;
}
__host__ __device__ constexpr size_t lds_bytes(int n) { return 2 * vec_bytes(n) + 2 * (size_t)pad16(n) * 4; }
// workspace of a system, in doubles: the padded FP32 factor and the inverses of the
// diagonal blocks of both triangles
__host__ __device__ constexpr long work_doubles(int n)
{
    return (long)pad16(n) * pad16(n) / 2 + 2L * pad16(n) * KB;
}

// orders the wave's own LDS and global accesses (they are performed in order; this keeps
// the compiler from moving them)
__device__ __forceinline__ void wsync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ float rl(float v, int k)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), k));
}
template <int CTRL, int RM> __device__ __forceinline__ u32 dmax(u32 v)
{
    return max(v, (u32)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, RM, 0xf, false));
}
__device__ __forceinline__ u32 max_u32(u32 v)
{
    v = dmax<0x111, 0xf>(v);
    v = dmax<0x112, 0xf>(v);
    v = dmax<0x114, 0xf>(v);
    v = dmax<0x118, 0xf>(v);
    v = dmax<0x142, 0xa>(v);
    v = dmax<0x143, 0xc>(v);
    return (u32)__builtin_amdgcn_readlane((int)v, 63);
}
// maximum over the four 16-lane groups, per lane of a group
__device__ __forceinline__ double max_groups(double v)
{
    v = fmax(v, __shfl_xor(v, 16, 64));
    return fmax(v, __shfl_xor(v, 32, 64));
}

// a / p from r ~ 1/p: one residual correction (Markstein, IBM J. Res. Dev. 34, 1990)
__device__ __forceinline__ float quot(float a, float p, float r)
{
    const float q = a * r;
    return fmaf(fmaf(-q, p, a), r, q);
}
__device__ __forceinline__ float recip(float p)
{
    const float r = __builtin_amdgcn_rcpf(p);
    return fmaf(r, fmaf(-p, r, 1.0f), r);
}

// Column J of a panel.  ok turns false at a pivot below FLT_EPSILON, a diagonal entry
// that is not positive, or NaN; the steps after that run on without a meaning, which keeps
// the panel free of branches.
template <int R, bool CHOL, int J>
__device__ __forceinline__ void panel_step(float (&p)[R][KB], int (&pos)[R], int lane, bool &ok)
{
    float s[KB];
    if constexpr (CHOL) {
        const float d = rl(p[0][J], J);
        ok = ok && d > 0.0f;
        const float l = sqrtf(d), r = 1.0f / l;
#pragma unroll
        for (int q = 0; q < R; ++q) p[q][J] = (q == 0 && lane == J) ? l : quot(p[q][J], l, r);
#pragma unroll
        for (int c = J + 1; c < KB; ++c) s[c] = rl(p[0][J], c);
#pragma unroll
        for (int q = 0; q < R; ++q)
#pragma unroll
            for (int c = J + 1; c < KB; ++c) p[q][c] = fmaf(-p[q][J], s[c], p[q][c]);
    } else {
        u32 key[R], kmax = 0u;
#pragma unroll
        for (int q = 0; q < R; ++q) {
            key[q] = pos[q] >= J ? __float_as_uint(fabsf(p[q][J])) : 0u;
            kmax = max(kmax, key[q]);
        }
        kmax = max_u32(kmax);
        ok = ok && kmax >= 0x34000000u && kmax <= 0x7f800000u;
        // the lowest row that holds the maximum (set qs, lane src) to scalar registers
        int qs = R - 1;
        unsigned long long hit = __ballot(key[R - 1] == kmax);
#pragma unroll
        for (int q = R - 2; q >= 0; --q) {
            const unsigned long long h = __ballot(key[q] == kmax);
            qs = h ? q : qs;
            hit = h ? h : hit;
        }
        const int src = (__ffsll(hit) - 1) & 63;
        int pp = pos[0];
#pragma unroll
        for (int q = 1; q < R; ++q) pp = qs == q ? pos[q] : pp;
        const int ppos = __builtin_amdgcn_readlane(pp, src);
#pragma unroll
        for (int c = J; c < KB; ++c) {
            float v = p[0][c];
#pragma unroll
            for (int q = 1; q < R; ++q) v = qs == q ? p[q][c] : v;
            s[c] = rl(v, src);
        }
        const float r = recip(s[J]);
#pragma unroll
        for (int q = 0; q < R; ++q) {
            pos[q] = (q == qs && lane == src) ? J : (pos[q] == J ? ppos : pos[q]);
            const bool below = pos[q] > J;
            const float l = below ? quot(p[q][J], s[J], r) : 0.0f;
            p[q][J] = below ? l : p[q][J];
#pragma unroll
            for (int c = J + 1; c < KB; ++c) p[q][c] = fmaf(-l, s[c], p[q][c]);
        }
    }
    if constexpr (J + 1 < KB) panel_step<R, CHOL, J + 1>(p, pos, lane, ok);
}

// One panel of 16 columns from position k0 (rows k0..np, at most 64 R of them); false on
// a breakdown.
template <int R, bool CHOL>
__device__ __forceinline__ bool panel(int np, int k0, float *W, int *map, int lane)
{
    float p[R][KB];
    int pos[R], phys[R];
    const int m = np - k0;
#pragma unroll
    for (int q = 0; q < R; ++q) {
        const int i = q * 64 + lane;
        const bool in = i < m;
        pos[q] = in ? i : -1;
        phys[q] = CHOL ? k0 + (in ? i : m - 1) : map[k0 + (in ? i : m - 1)];
        const f4 *src = reinterpret_cast<const f4 *>(W + (long)phys[q] * np + k0);
        const f4 v0 = src[0], v1 = src[1], v2 = src[2], v3 = src[3];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            p[q][e] = v0[e];
            p[q][4 + e] = v1[e];
            p[q][8 + e] = v2[e];
            p[q][12 + e] = v3[e];
        }
    }
    bool ok = true;
    panel_step<R, CHOL, 0>(p, pos, lane, ok);
    if (!ok) return false;
#pragma unroll
    for (int q = 0; q < R; ++q) {
        if (pos[q] >= 0) {
            if (!CHOL) map[k0 + pos[q]] = phys[q];
            f4 *dst = reinterpret_cast<f4 *>(W + (long)phys[q] * np + k0);
            dst[0] = f4{p[q][0], p[q][1], p[q][2], p[q][3]};
            dst[1] = f4{p[q][4], p[q][5], p[q][6], p[q][7]};
            dst[2] = f4{p[q][8], p[q][9], p[q][10], p[q][11]};
            dst[3] = f4{p[q][12], p[q][13], p[q][14], p[q][15]};
        }
    }
    wsync();
    return true;
}

// u[i] -= L11[i][k] u[k] for i > k, k = K..14; lane i of each 16-lane group holds row i of L11
template <int K> __device__ __forceinline__ void eliminate(float *u, const float *lq)
{
    if constexpr (K < KB - 1) {
        constexpr int N = KB - 1 - K;
        lanes::fmac_row<K + 1, (N > 8 ? 8 : N)>(u + K + 1, lq[K], u[K]);
        if constexpr (N > 8) lanes::fmac_row<K + 9, N - 8>(u + K + 9, lq[K], u[K]);
        eliminate<K + 1>(u, lq);
    }
}

// 16 elements of a row
__device__ __forceinline__ void load16(const float *row, float *v)
{
#pragma unroll
    for (int c = 0; c < KB / 4; ++c) {
        const f4 t = reinterpret_cast<const f4 *>(row)[c];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[4 * c + e] = t[e];
    }
}

// v[e], k = 4 grp + e, to k = 4 e + grp
__device__ __forceinline__ void column_order(f4 &v)
{
    float w[4] = {v[0], v[1], v[2], v[3]};
    lanes::swap_groups<32>(w[0], w[2]);
    lanes::swap_groups<32>(w[1], w[3]);
    lanes::swap_groups<16>(w[0], w[1]);
    lanes::swap_groups<16>(w[2], w[3]);
    v = f4{w[0], w[1], w[2], w[3]};
}

// The update of columns [k0 + KK, cend) behind KK = 16 or 32 finished columns, 64 of them
// at a time; LU first solves U12 = L11^-1 A12 (lane = column).
template <bool CHOL, int KK>
__device__ __forceinline__ void update(int np, int k0, int cend, float *W, const int *map, float *ush, int lane)
{
    const int l16 = lane & 15, grp = lane >> 4;
    const int k1 = k0 + KK;
    float lq[2][KK];              // rows l16 and 16 + l16 of L11
    if (!CHOL) {
#pragma unroll
        for (int h = 0; h < KK / KB; ++h)
#pragma unroll
            for (int c = 0; c <= h; ++c)
                load16(W + (long)map[k0 + h * KB + l16] * np + k0 + c * KB, lq[h] + c * KB);
    }
    for (int c0 = k1; c0 < cend; c0 += 64) {
        const int nct = min(4, (cend - c0) / KB);
        float ua[4][KK / 4];      // block ct: element (k, column l16) of U12, k = 4 i + grp, or of L21^T, k = 16 (i / 4) + 4 grp + i % 4
        if constexpr (CHOL) {
#pragma unroll
            for (int ct = 0; ct < 4; ++ct)
#pragma unroll
                for (int h = 0; h < KK / KB; ++h) {
                    const f4 v = *reinterpret_cast<const f4 *>(W + (long)min(c0 + ct * KB + l16, np - 1) * np + k0 +
                                                               h * KB + 4 * grp);
#pragma unroll
                    for (int i = 0; i < 4; ++i) ua[ct][4 * h + i] = v[i];
                }
        } else {
            const int c = min(c0 + lane, np - 1);
            float u[KK];
#pragma unroll
            for (int i = 0; i < KK; ++i) u[i] = W[(long)map[k0 + i] * np + c];
            eliminate<0>(u, lq[0]);
            if constexpr (KK > KB) {
#pragma unroll
                for (int k = 0; k < KB; ++k) {
                    lanes::fmac_row<0, 8>(u + KB, lq[1][k], u[k]);
                    lanes::fmac_row<8, 8>(u + KB + 8, lq[1][k], u[k]);
                }
                eliminate<0>(u + KB, lq[1] + KB);
            }
            if (c0 + lane < cend) {
#pragma unroll
                for (int i = 0; i < KK; ++i) W[(long)map[k0 + i] * np + c] = u[i];
            }
#pragma unroll
            for (int i = 0; i < KK; ++i) ush[i * LU_ROW + lane] = u[i];
            wsync();
#pragma unroll
            for (int ct = 0; ct < 4; ++ct)
#pragma unroll
                for (int i = 0; i < KK / 4; ++i)
                    ua[ct][i] = ush[(4 * i + grp) * LU_ROW + ct * KB + l16];
            wsync();
        }
        // RB row blocks at a time, all their loads ahead of the products
        constexpr int RB = 4;
        for (int r0 = CHOL ? c0 : k1; r0 < np; r0 += RB * KB) {
            float *row[RB];
            f4 lv[RB][KK / KB], old[RB][4];
#pragma unroll
            for (int h = 0; h < RB; ++h) {
                const int rr = min(r0 + h * KB, np - KB) + l16;
                row[h] = W + (long)(CHOL ? rr : map[rr]) * np;
#pragma unroll
                for (int g = 0; g < KK / KB; ++g)
                    lv[h][g] = *reinterpret_cast<const f4 *>(row[h] + k0 + g * KB + 4 * grp);
            }
            // LU: the products in the order of the columns, whose partial sums the pivoting
            // keeps small.  Lane group and register exchange their two bits of k.
            if (!CHOL) {
#pragma unroll
                for (int h = 0; h < RB; ++h)
#pragma unroll
                    for (int g = 0; g < KK / KB; ++g) column_order(lv[h][g]);
            }
#pragma unroll
            for (int h = 0; h < RB; ++h)
                if (r0 + h * KB < np) {
#pragma unroll
                    for (int ct = 0; ct < 4; ++ct)
                        if (ct < nct && (!CHOL || c0 + ct * KB <= r0 + h * KB))
                            old[h][ct] = *reinterpret_cast<const f4 *>(row[h] + c0 + ct * KB + 4 * grp);
                }
#pragma unroll
            for (int h = 0; h < RB; ++h)
                if (r0 + h * KB < np) {
#pragma unroll
                    for (int ct = 0; ct < 4; ++ct)
                        if (ct < nct && (!CHOL || c0 + ct * KB <= r0 + h * KB)) {
                            f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                            for (int i = 0; i < KK / 4; ++i)
                                acc = lanes::Mf<float>::mac(ua[ct][i], -lv[h][i / 4][i % 4], acc);
                            *reinterpret_cast<f4 *>(row[h] + c0 + ct * KB + 4 * grp) = old[h][ct] + acc;
                        }
                }
        }
        wsync();
    }
}

template <bool CHOL>
__device__ __forceinline__ bool panel_any(int np, int k0, float *W, int *map, int lane)
{
    const int m = np - k0;
    if (m > 192) return panel<4, CHOL>(np, k0, W, map, lane);
    if (m > 128) return panel<3, CHOL>(np, k0, W, map, lane);
    if (m > 64) return panel<2, CHOL>(np, k0, W, map, lane);
    return panel<1, CHOL>(np, k0, W, map, lane);
}

// Two panels, then the rest of the matrix once for both: half the passes over it (the
// waves' matrices together are far larger than L2).
template <bool CHOL>
__device__ __forceinline__ bool factor(int np, float *W, int *map, float *ush, int lane)
{
    for (int k0 = 0; k0 < np; k0 += KB) {
        if (!panel_any<CHOL>(np, k0, W, map, lane)) return false;
        if (k0 + KB == np) break;
        if (k0 % (2 * KB) == 0) update<CHOL, KB>(np, k0, k0 + 2 * KB, W, map, ush, lane);
        else update<CHOL, 2 * KB>(np, k0 - KB, np, W, map, ush, lane);
    }
    return true;
}

// Inverses of the 16 x 16 diagonal blocks, in FP64 from the FP32 factor: group = block,
// lane of a group = column.  Element (row, k) of a block sits at row * 16 + (k % 4) * 4 +
// k / 4, so that a lane reads the four it multiplies as one piece.  inv: the lower
// triangle's blocks, then the upper triangle's (Cholesky: the lower ones transposed).
template <bool CHOL>
__device__ __forceinline__ void invert_blocks(int np, const float *W, const int *map, double *inv, int lane)
{
    const int l16 = lane & 15, grp = lane >> 4, nb = np / KB;
    for (int b0 = 0; b0 < nb; b0 += 4) {
        const int b = min(b0 + grp, nb - 1);
        double *lo = inv + (long)b * KB * KB, *up = inv + (long)nb * KB * KB + (long)b * KB * KB;
        double y[KB];
#pragma unroll
        for (int i = 0; i < KB; ++i) {
            const int rr = CHOL ? b * KB + i : map[b * KB + i];
            const f4 *src = reinterpret_cast<const f4 *>(W + (long)rr * np + b * KB);
            double s = i == l16 ? 1.0 : 0.0;
            float v[KB];
#pragma unroll
            for (int c = 0; c <= i / 4; ++c) {
                const f4 t = src[c];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[4 * c + e] = t[e];
            }
#pragma unroll
            for (int q = 0; q < i; ++q) s = fma(-(double)v[q], y[q], s);
            y[i] = CHOL ? s / (double)v[i] : s;
            lo[i * KB + (l16 & 3) * 4 + (l16 >> 2)] = y[i];
            if (CHOL) up[l16 * KB + (i & 3) * 4 + (i >> 2)] = y[i];
        }
        if (!CHOL) {
#pragma unroll
            for (int ii = 0; ii < KB; ++ii) {
                const int i = KB - 1 - ii;
                const f4 *src = reinterpret_cast<const f4 *>(W + (long)map[b * KB + i] * np + b * KB);
                double s = i == l16 ? 1.0 : 0.0;
                float v[KB];
#pragma unroll
                for (int c = i / 4; c < 4; ++c) {
                    const f4 t = src[c];
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[4 * c + e] = t[e];
                }
#pragma unroll
                for (int q = i + 1; q < KB; ++q) s = fma(-(double)v[q], y[q], s);
                y[i] = s / (double)v[i];
                up[i * KB + (l16 & 3) * 4 + (l16 >> 2)] = y[i];
            }
        }
    }
    wsync();
}

// acc -= rows of one block of the factor times the finished vector block kb (16 x 16 by
// 16 x QR); element (k = 4 grp + t) of both operands
__device__ __forceinline__ d4 block_mac(const float (&lv)[4], const double *vec, bool col, d4 acc)
{
#pragma unroll
    for (int t = 0; t < 4; ++t) acc = lanes::Mf<double>::mac(-(double)lv[t], col ? vec[t] : 0.0, acc);
    return acc;
}
// a diagonal block's inverse (row l16, elements k = grp + 4 t) times acc (element k is acc[t])
__device__ __forceinline__ d4 block_solve(d4 inv, d4 acc)
{
    d4 x = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int t = 0; t < 4; ++t) x = lanes::Mf<double>::mac(inv[t], acc[t], x);
    return x;
}

// d <- (factors)^-1 d, positions 0..np, up to QR columns of pitch ldv in LDS
template <bool CHOL>
__device__ __forceinline__ void substitute(int np, const float *W, const int *map, const double *inv, double *d,
                                           int ldv, int nr, int lane)
{
    const int l16 = lane & 15, grp = lane >> 4, nb = np / KB;
    const bool col = l16 < nr;
    double *dc = d + (col ? l16 : 0) * ldv;
    for (int b = 0; b < nb; ++b) {
        const d4 iv = *reinterpret_cast<const d4 *>(inv + (long)b * KB * KB + l16 * KB + grp * 4);
        d4 acc;
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] = col ? dc[b * KB + grp + 4 * q] : 0.0;
        const int rr = b * KB + l16;
        const float *row = W + (long)(CHOL ? rr : map[rr]) * np + 4 * grp;
#pragma unroll 8
        for (int k = 0; k < b; ++k) {
            const f4 v = *reinterpret_cast<const f4 *>(row + k * KB);
            const float lv[4] = {v[0], v[1], v[2], v[3]};
            acc = block_mac(lv, dc + k * KB + 4 * grp, col, acc);
        }
        acc = block_solve(iv, acc);
        if (col) {
#pragma unroll
            for (int q = 0; q < 4; ++q) dc[b * KB + grp + 4 * q] = acc[q];
        }
        wsync();
    }
    for (int b = nb - 1; b >= 0; --b) {
        const d4 iv = *reinterpret_cast<const d4 *>(inv + (long)(nb + b) * KB * KB + l16 * KB + grp * 4);
        d4 acc;
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] = col ? dc[b * KB + grp + 4 * q] : 0.0;
        const int rr = b * KB + l16;
        const float *row = W + (long)(CHOL ? 4 * grp : map[rr]) * np + (CHOL ? rr : 4 * grp);
#pragma unroll 8
        for (int k = b + 1; k < nb; ++k) {
            float lv[4];
            if constexpr (CHOL) {
                // the transpose of L: rows are the k
#pragma unroll
                for (int t = 0; t < 4; ++t) lv[t] = row[(long)(k * KB + t) * np];
            } else {
                const f4 v = *reinterpret_cast<const f4 *>(row + k * KB);
#pragma unroll
                for (int t = 0; t < 4; ++t) lv[t] = v[t];
            }
            acc = block_mac(lv, dc + k * KB + 4 * grp, col, acc);
        }
        acc = block_solve(iv, acc);
        if (col) {
#pragma unroll
            for (int q = 0; q < 4; ++q) dc[b * KB + grp + 4 * q] = acc[q];
        }
        wsync();
    }
}

// Eight elements of a row of n from column kc on, zero past the end: element 2 t + e is
// column kc + 8 t + 2 grp + e, so that the four lanes of a row read 64 bytes at a time.
__device__ __forceinline__ void load8(const double *row, int kc, int grp, int n, double (&v)[8])
{
    if (kc + 32 <= n) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const auto w = *reinterpret_cast<const lanes::Vec16u<double>::type *>(row + kc + 8 * t + 2 * grp);
            v[2 * t] = w[0];
            v[2 * t + 1] = w[1];
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int k = kc + 8 * (i / 2) + 2 * grp + i % 2;
            v[i] = k < n ? row[k] : 0.0;
        }
    }
}

// A to the padded FP32 workspace (unit diagonal past n); the return value is ||A||_inf
__device__ __forceinline__ double convert(int n, int np, const double *A, float *W, int lane)
{
    const int l16 = lane & 15, grp = lane >> 4;
    double an = 0.0;
    for (int r0 = 0; r0 < np; r0 += KB) {
        const int r = r0 + l16;
        const double *row = A + (long)min(r, n - 1) * n;
        double s = 0.0;
#pragma unroll 4
        for (int kc = 0; kc < np; kc += KB) {
            const int k = kc + 4 * grp;
            double v[4];
            if (kc + KB <= n) {
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const auto w = *reinterpret_cast<const lanes::Vec16u<double>::type *>(row + k + 2 * t);
                    v[2 * t] = w[0];
                    v[2 * t + 1] = w[1];
                }
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = k + i < n ? row[k + i] : 0.0;
            }
            f4 o;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s += fabs(v[i]);
                o[i] = r < n && k + i < n ? (float)v[i] : (k + i == r ? 1.0f : 0.0f);
            }
            *reinterpret_cast<f4 *>(W + (long)r * np + k) = o;
        }
        s += __shfl_xor(s, 16, 64);
        s += __shfl_xor(s, 32, 64);
        an = fmax(an, s);
    }
    an = fmax(an, __shfl_xor(an, 1, 64));
    an = fmax(an, __shfl_xor(an, 2, 64));
    an = fmax(an, __shfl_xor(an, 4, 64));
    return fmax(an, __shfl_xor(an, 8, 64));
}

struct Result { bool ok; int iters; double bwd; };

// Right-hand sides j0..j0+nr of a factored system: refinement from zero until every
// column's backward error is <= tol (each column stops by itself).
template <bool CHOL>
__device__ __forceinline__ Result refine(int n, int np, int nrhs, int j0, int nr, const double *A, const double *B,
                                         double *X, const float *W, const int *map, const int *imap,
                                         const double *inv, double an, double tol, int max_iter, double *d, double *xs,
                                         int ldv, int lane)
{
    const int l16 = lane & 15, grp = lane >> 4;
    const bool col = l16 < nr;
    const double *Bc = B + j0 + (col ? l16 : 0);
    double *xc = xs + (col ? l16 : 0) * ldv, *dc = d + (col ? l16 : 0) * ldv;
    for (int i = lane; i < QR * ldv; i += 64) { xs[i] = 0.0; d[i] = 0.0; }
    wsync();
    // x = 0: the residual is b
    double bn = 0.0;
    bool nan = false;
    for (int r = grp; r < n; r += 4) {
        const double bv = Bc[(long)r * nrhs];
        bn = fmax(bn, fabs(bv));
        nan |= bv != bv;
        if (col) dc[CHOL ? r : imap[r]] = bv;
    }
    bn = max_groups(bn);
    double rn = bn, xn = 0.0, eta = 1.0, prev = INFINITY, worst = 0.0;
    bool done = !col, ok = true;
    int iters = 0;
    wsync();
    for (int it = 0;; ++it) {
        nan = __shfl_xor((int)nan, 16, 64) | (int)nan;
        nan = __shfl_xor((int)nan, 32, 64) | (int)nan;
        if (!done) {
            const double den = an * xn + bn;
            eta = nan ? INFINITY : den > 0 ? rn / den : (rn > 0 ? INFINITY : 0.0);
            const bool hit = eta <= tol;
            if (hit || it == max_iter || (it >= 2 && !(eta < 0.5 * prev))) {
                done = true;
                ok = hit;
                iters = it;
                worst = eta;
            }
            prev = eta;
        }
        if (__all(done) || __any(!ok)) break;
        substitute<CHOL>(np, W, map, inv, d, ldv, nr, lane);
        xn = 0.0;
        if (!done) {
            for (int r = grp; r < n; r += 4) {
                const double xv = xc[r] + dc[r];
                xc[r] = xv;
                xn = fmax(xn, fabs(xv));
            }
        }
        xn = max_groups(xn);
        wsync();
        // r = b - A x
        rn = 0.0;
        nan = false;
        for (int r0 = 0; r0 < n; r0 += 2 * KB) {
            // two row blocks; each 32 columns in eight sums of four products (Cholesky: four of
            // eight), added up in pairs.  A matrix-core step rounds after each of its products, so two
            // sums along the whole row round n times at their full size (mean error of general systems of 8 to
            // 256 rows, kappa = 1e3: 2.1e-14 so, 1.2e-14 as it is).
            const double *row[2] = {A + (long)min(r0 + l16, n - 1) * n, A + (long)min(r0 + KB + l16, n - 1) * n};
            d4 total[2] = {};
#pragma unroll 2
            for (int kc = 0; kc < n; kc += 32) {
                double v[2][8], xv[8];
                load8(row[0], kc, grp, n, v[0]);
                load8(row[1], kc, grp, n, v[1]);
#pragma unroll
                for (int i = 0; i < 8; ++i) xv[i] = col ? xc[kc + 8 * (i / 2) + 2 * grp + i % 2] : 0.0;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    constexpr int NS = CHOL ? 4 : 8;   // (eight cost the Cholesky kernel its third wave per SIMD)
                    d4 part[NS] = {};
#pragma unroll
                    for (int i = 0; i < 8; ++i) part[i % NS] = lanes::Mf<double>::mac(v[h][i], xv[i], part[i % NS]);
#pragma unroll
                    for (int s = 1; s < NS; s *= 2)
#pragma unroll
                        for (int i = 0; i < NS; i += 2 * s) part[i] += part[i + s];
                    total[h] += part[0];
                }
            }
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int r = r0 + h * KB + grp + 4 * q;
                    if (r < n && col) {
                        const double rv = Bc[(long)r * nrhs] - total[h][q];
                        rn = fmax(rn, fabs(rv));
                        nan |= rv != rv;
                        dc[CHOL ? r : imap[r]] = rv;
                    }
                }
        }
        rn = max_groups(rn);
        wsync();
    }
    // every column has a verdict, or one of them failed
    Result res;
    res.ok = !__any(!ok);
    for (int i = lane; i < n * nr; i += 64) {
        const int r = i / nr, c = i - r * nr;
        X[(long)r * nrhs + j0 + c] = xs[c * ldv + r];
    }
#pragma unroll
    for (int o = 1; o < 16; o *= 2) {
        iters = max(iters, __shfl_xor(iters, o, 64));
        worst = fmax(worst, __shfl_xor(worst, o, 64));
    }
    res.iters = iters;
    res.bwd = worst;
    wsync();
    return res;
}

// False: FP32 broke down or its refinement stalled.
template <bool CHOL>
__device__ __forceinline__ bool solve(int n, int nrhs, const double *A, const double *B, double *X, double *work,
                                      double tol, int max_iter, char *lds, int lane, int *iters, double *bwd)
{
    const int np = pad16(n), ldv = ld_vec(n);
    float *W = reinterpret_cast<float *>(work);
    double *inv = work + (long)np * np / 2;
    double *d = reinterpret_cast<double *>(lds);
    double *xs = reinterpret_cast<double *>(lds + vec_bytes(n));
    int *map = reinterpret_cast<int *>(lds + 2 * vec_bytes(n)), *imap = map + np;
    for (int i = lane; i < np; i += 64) map[i] = i;
    const double an = convert(n, np, A, W, lane);
    wsync();
    if (!factor<CHOL>(np, W, map, reinterpret_cast<float *>(d), lane)) return false;
    for (int i = lane; i < np; i += 64) imap[map[i]] = i;
    invert_blocks<CHOL>(np, W, map, inv, lane);
    *iters = 0;
    *bwd = 0.0;
    for (int j0 = 0; j0 < nrhs; j0 += QR) {
        const Result r = refine<CHOL>(n, np, nrhs, j0, min(QR, nrhs - j0), A, B, X, W, map, imap, inv, an, tol,
                                      max_iter, d, xs, ldv, lane);
        if (!r.ok) return false;
        *iters = max(*iters, r.iters);
        *bwd = fmax(*bwd, r.bwd);
    }
    return true;
}

} // namespace wave
