// Partial-pivot LU in 32-column sub-panels whose rows live in registers.
//
// Two launches per sub-panel:
//   sub_panel_kernel — the pivot search, the multipliers and the update of the
//       sub-panel's own 32 columns.  A lane holds R whole rows; rows never move,
//       each carries its position, and the finished rows are written to their
//       final positions.  Same pivots as scirs2-linalg/src/lapack.rs:95-131
//       (largest |a_ij|, the first position on ties), correctly rounded
//       multipliers (lapack.rs:138), the absolute test |pivot| < eps
//       (lapack.rs:106-120), a_ij - l_ik u_kj as one fused operation.
//   sub_apply_kernel — the other columns asked for: the sub-panel's row
//       interchanges, U12 = L11^-1 A12 by substitution and the rank-32 update on
//       the matrix cores, in one pass (and the composition of several
//       sub-panels' interchanges into one list).
//
// What bounds the panel is the dependent chain of one column: arg-max, exchange
// of the candidates, the pivot row to every lane, division, update of the next
// column.  A wave issues an instruction every four cycles at best and a taken
// branch costs about ten times that, so the 32 steps are straight-line code; the
// pivot row reaches the lanes as DPP operands (lane c % 16 of every 16-lane row
// holds element c, v_fmac's row_newbcast broadcasts it), which replaces sixteen
// 16-byte LDS broadcasts per wave and column by two 8-byte reads.  Two forms of
// the exchange:
//   - one workgroup (few rows): candidates and rows go through LDS;
//   - many single waves on ONE die (XCD): through that die's L2.  A store of
//     workgroup scope stays in the die's L2 and a load of agent scope passes the
//     L1, so a round among 64 waves takes 0.37 us, against 1.5 - 1.65 us when they
//     sit on all eight dies (measured, G = 64 and 128).  The launch offers
//     8 (g - 1) + 1 workgroups for g places: by the pigeonhole principle some die
//     receives g of them; they register per die, the first die to fill is elected
//     and the rest exit.
// Measured for one 32-column FP64 panel, launch included: 512 rows 33 us (65 us with
// one row per thread, LDS broadcasts and a rolled loop), 2000 rows 41 us and 8192
// rows 50 us (160 us with one exchange per column over the whole device).
#include "common.hpp"
#include "elect.hpp"
#include "kernels.hpp"
#include "lanes.hpp"
#include "prof.hpp"
#include "tags.hpp"

#include "api_internal.hpp"

#include <algorithm>
#include <type_traits>

namespace sub {

using namespace lanes;
typedef unsigned long long u64;
typedef unsigned u32;
constexpr int W = SCIRS_SUB_W;
constexpr int GMAX = SCIRS_SUB_AGENTS;
static_assert(W == 32, "two 16-lane rows of pivot-row elements");

template <int CTRL, int RM> __device__ __forceinline__ u32 dmax(u32 v)
{
    return max(v, (u32)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, RM, 0xf, false));
}
__device__ __forceinline__ u32 wave_max_u32(u32 v)
{
    v = dmax<0x111, 0xf>(v);
    v = dmax<0x112, 0xf>(v);
    v = dmax<0x114, 0xf>(v);
    v = dmax<0x118, 0xf>(v);
    v = dmax<0x142, 0xa>(v);
    v = dmax<0x143, 0xc>(v);
    return (u32)__builtin_amdgcn_readlane((int)v, 63);
}
// every lane of an aligned group of N lanes gets the group's maximum
template <int N> __device__ __forceinline__ u32 group_max(u32 v)
{
    if constexpr (N >= 2) v = dmax<0xB1, 0xf>(v);    // quad_perm 1 0 3 2
    if constexpr (N >= 4) v = dmax<0x4E, 0xf>(v);    // quad_perm 2 3 0 1
    if constexpr (N >= 8) v = dmax<0x141, 0xf>(v);   // row_half_mirror
    if constexpr (N >= 16) v = dmax<0x140, 0xf>(v);  // row_mirror
    return v;
}
__device__ __forceinline__ u32 rl(u32 v, int k) { return (u32)__builtin_amdgcn_readlane((int)v, k); }
__device__ __forceinline__ u64 bal(bool c) { return __builtin_amdgcn_ballot_w64(c); }

// The search key of a value is its top word without the sign, |v| ordered, except that
// FP64 values equal in their top 20 mantissa bits need the lower word too; minus (the word
// of infinity + 1), which wraps every number above the NaN: these compare with nothing
// (lapack.rs:95-104), so they are candidates only where nothing else is left.
template <typename T> struct Val;
template <> struct Val<double> {
    static __device__ __forceinline__ u32 hi(double v) { return (u32)((u64)__double_as_longlong(v) >> 32); }
    static __device__ __forceinline__ u32 lo(double v) { return (u32)(u64)__double_as_longlong(v); }
    static __device__ __forceinline__ double make(u32 h, u32 l)
    {
        return __longlong_as_double((long long)(((u64)h << 32) | l));
    }
    // 1/p to an ulp (Newton-Raphson) and a/p from it by one residual correction: the
    // correctly rounded quotient (Markstein, IBM J. Res. Dev. 34, 1990)
    static __device__ __forceinline__ double rcp(double p)
    {
        double r = __builtin_amdgcn_rcp(p);
        r = fma(r, fma(-p, r, 1.0), r);
        return fma(r, fma(-p, r, 1.0), r);
    }
    static __device__ __forceinline__ double div(double a, double p, double r)
    {
        const double q = a * r;
        return fma(fma(-q, p, a), r, q);
    }
    static constexpr u32 eps_hi = 0x3cb00000u, inf_hi = 0x7ff00000u;   // top words of eps and infinity
    static constexpr u32 big_hi = 0x7d000000u;   // from here on 1/p nears the subnormals: divide instead
};
template <> struct Val<float> {
    static __device__ __forceinline__ u32 hi(float v) { return __float_as_uint(v); }
    static __device__ __forceinline__ u32 lo(float) { return 0u; }
    static __device__ __forceinline__ float make(u32 h, u32) { return __uint_as_float(h); }
    static __device__ __forceinline__ float rcp(float p)
    {
        const float r = __builtin_amdgcn_rcpf(p);
        return fmaf(r, fmaf(-p, r, 1.0f), r);
    }
    static __device__ __forceinline__ float div(float a, float p, float r)
    {
        float q = a * r;
        q = fmaf(fmaf(-q, p, a), r, q);
        return fmaf(fmaf(-q, p, a), r, q);
    }
    static constexpr u32 eps_hi = 0x34000000u, inf_hi = 0x7f800000u;
    static constexpr u32 big_hi = 0x7c000000u;
};

template <typename T> __host__ __device__ constexpr u32 to_key(u32 hi) { return hi - Val<T>::inf_hi - 1u; }
template <typename T> __host__ __device__ constexpr u32 from_key(u32 key) { return key + Val<T>::inf_hi + 1u; }

__device__ __forceinline__ void put(u64 *p, u64 v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ u64 get(const u64 *p)
{
    return __hip_atomic_load(const_cast<u64 *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <typename T> struct PanelArgs {
    T *A; long lda;      // the sub-panel's first diagonal element
    int top;             // its row (and column) in the matrix
    int m, w;            // rows from the diagonal down, columns (<= 32)
    int G;               // waves that hold rows
    u64 *key, *row;      // [2][GMAX][2] candidates, [2][GMAX][32][2] their rows (tagged words)
    int *elect;          // per-die registration counts (128 bytes apart), then the elected die + 1; zeroed
    u32 seq;             // tag of column 0
    int *pairs, *npairs; // the moved rows (destination, source), absolute; *npairs zeroed
    int *info; double *info_val; int *abort;
    u32 spin_limit;
};

template <typename T, int R> struct Rows {
    T a[R][W];
    int pos[R];      // current position of the row
    u32 live[R];     // 31 while the row can still be picked, 0 after (the width of the key's bit field)
    T l[R];          // multipliers of the last column
    T pr[W / 16];    // its pivot row: lane l holds elements l % 16 and 16 + l % 16
    T odd;           // zero until a pivot row holds an infinity or a NaN
    bool stop;
};
template <typename T> struct Xch {
    alignas(16) T row[W][W];   // the pivot rows (many workgroups: each wave writes them all, the same)
    uint4 key[2][16];
};

// Several candidates share the top word: keep the largest lower word, then the first position.
template <int R> __device__ void tie_break(bool (&win)[R], const u32 (&lo)[R], const int (&pos)[R])
{
    u32 b = 0, q = 0;
#pragma unroll
    for (int x = 0; x < R; ++x) b = max(b, win[x] ? lo[x] : 0u);
    b = wave_max_u32(b);
#pragma unroll
    for (int x = 0; x < R; ++x) {
        win[x] = win[x] && lo[x] == b;
        q = max(q, win[x] ? ~(u32)pos[x] : 0u);
    }
    q = wave_max_u32(q);
#pragma unroll
    for (int x = 0; x < R; ++x) win[x] = win[x] && ~(u32)pos[x] == q;
}

// columns J + 1 .. of J's block of eight columns
template <typename T, int R, int J> __device__ __forceinline__ void update_block(Rows<T, R> &S)
{
    constexpr int c0 = J + 1, n = 7 - (J & 7);
    if constexpr (n > 0)
#pragma unroll
        for (int x = 0; x < R; ++x) fmac_row<c0 & 15, n>(&S.a[x][c0], S.pr[c0 >> 4], S.l[x]);
}
// the blocks from B on (without block B's first SKIP columns)
template <typename T, int R, int B, int SKIP = 0> __device__ __forceinline__ void update_rest(Rows<T, R> &S, int x)
{
    if constexpr (B < W / 8) {
        fmac_row<(8 * B + SKIP) & 15, 8 - SKIP>(&S.a[x][8 * B + SKIP], S.pr[(8 * B) >> 4], S.l[x]);
        update_rest<T, R, B + 1>(S, x);
    }
}
template <typename T, int R, int J> __device__ __forceinline__ void row_out(const Rows<T, R> &S, int x, T *lr)
{
    constexpr int E = 16 / (int)sizeof(T);
    typedef typename Vec16<T>::type V;
#pragma unroll
    for (int c = J & ~(E - 1); c < W; c += E) {
        V v;
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = S.a[x][c + e];
        *reinterpret_cast<V *>(lr + c) = v;
    }
}

// Column J.  NW > 0: one workgroup of at most NW waves, exchange through LDS.
// NW = 0: wave g of A.G, exchange through the die's L2 in 64-bit words that carry the
// column's tag (tags.hpp), NS candidates per lane.  Bounded polls: a wave that gives
// up stops the panel.  A wave's update of the columns beyond the current block waits
// until its candidate is on its way, so that it runs in the exchange's shadow.
template <typename T, int R, int NS, int NW, int J>
__device__ __forceinline__ void step(Rows<T, R> &S, const PanelArgs<T> &A, int g, T *lr, Xch<T> *L)
{
    typedef Val<T> V;
    const int lane = threadIdx.x & 63;
    constexpr int b = J & 1;
    u32 h[R], hm = 0;
    bool win[R];
#pragma unroll
    for (int x = 0; x < R; ++x) {
        h[x] = to_key<T>(__builtin_amdgcn_ubfe(V::hi(S.a[x][J]), 0, S.live[x]));
        hm = max(hm, h[x]);
    }
    const u32 gm = wave_max_u32(hm);
    int cnt = 0;
#pragma unroll
    for (int x = 0; x < R; ++x) {
        win[x] = h[x] == gm;
        cnt += __popcll(bal(win[x]));
    }
    if (__builtin_expect(cnt != 1, 0)) {
        u32 lo[R];
#pragma unroll
        for (int x = 0; x < R; ++x) {
            lo[x] = V::lo(S.a[x][J]);
            win[x] = win[x] && S.live[x] != 0;
        }
        tie_break<R>(win, lo, S.pos);
        if (gm <= to_key<T>(0)) {   // zeros and NaN, or no row left: still one candidate
            bool any = false;
#pragma unroll
            for (int x = 0; x < R; ++x) any = any || win[x];
            if (bal(any) == 0) win[0] = lane == 0;
        }
    }
    u32 khi;
    int p;
    if constexpr (NW == 0) {
        const u32 tag = A.seq + (u32)J;
        u64 *ks = A.key + ((size_t)b * GMAX + g) * 2;
#pragma unroll
        for (int x = 0; x < R; ++x)
            if (win[x]) {
                put(ks, tags::value_word(tag, gm));
                put(ks + 1, tags::position_word(tag, (u32)S.pos[x], V::lo(S.a[x][J])));
            }
#pragma unroll
        for (int x = 0; x < R; ++x) {
            if constexpr (J > 0) update_rest<T, R, (J - 1) / 8 + 1, (J & 7) == 0>(S, x);
            if (win[x]) row_out<T, R, J>(S, x, lr);
        }
        __builtin_amdgcn_wave_barrier();
        u32 spins = 0;
        u64 k0[NS], k1[NS];
        bool late = false;
        auto poll = [&]() {
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const u64 *q = A.key + ((size_t)b * GMAX + min(lane + 64 * s, A.G - 1)) * 2;
                k0[s] = get(q);
                k1[s] = get(q + 1);
            }
        };
        // a poll that did not succeed: give up after spin_limit tries or when another wave
        // did; now and then push this die's lines out, in case the waves sit on several
        auto give_up = [&]() -> bool {
            if (S.stop || ++spins > A.spin_limit) return true;
            if ((spins & 4095u) == 0) {
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
                return __hip_atomic_load(A.abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
            }
            return false;
        };
        poll();
        const T pv = lr[lane & (W - 1)];
        u64 *rs = A.row + ((size_t)b * GMAX + g) * 2 * W + 2 * lane;
        if (lane < W) {
            put(rs, ((u64)tag << 32) | V::hi(pv));
            if constexpr (sizeof(T) == 8) put(rs + 1, ((u64)tag << 32) | V::lo(pv));
        }
        while (true) {
            bool ok = true;
#pragma unroll
            for (int s = 0; s < NS; ++s) ok = ok && tags::current(k0[s], k1[s], tag);
            if (__builtin_expect(bal(ok) == ~0ull, 1)) break;
            if (give_up()) { late = true; break; }
            poll();
        }
        u32 kh = (u32)k0[0], kl = (u32)k1[0], kp = tags::position(k1[0]);
        int slot = 0;
#pragma unroll
        for (int s = 1; s < NS; ++s) {
            const u32 h2 = (u32)k0[s], l2 = (u32)k1[s], p2 = tags::position(k1[s]);
            const bool bt = h2 > kh || (h2 == kh && (l2 > kl || (l2 == kl && p2 < kp)));
            kh = bt ? h2 : kh;
            kl = bt ? l2 : kl;
            kp = bt ? p2 : kp;
            slot = bt ? s : slot;
        }
        khi = wave_max_u32(kh);
        bool w1[1] = {kh == khi};
        if (__builtin_expect(__popcll(bal(w1[0])) != 1, 0)) {
            const u32 lo1[1] = {kl};
            const int p1[1] = {(int)kp};
            tie_break<1>(w1, lo1, p1);
        }
        // (lanes past the last wave repeat its candidate: any of them names the same row)
        const int wl = __builtin_ctzll(bal(w1[0]) | (1ull << 63));
        int wg = wl;
        if constexpr (NS > 1) wg += 64 * (int)rl((u32)slot, wl);
        wg = min(wg, A.G - 1);
        p = (int)rl(kp, wl);
        const u64 *q = A.row + ((size_t)b * GMAX + wg) * 2 * W + 2 * (lane & 15);
        while (true) {
            bool ok = true;
#pragma unroll
            for (int k = J / 16; k < W / 16; ++k) {
                const u64 vh = get(q + 32 * k);
                ok = ok && (u32)(vh >> 32) == tag;
                u64 vl = 0;
                if constexpr (sizeof(T) == 8) {
                    vl = get(q + 32 * k + 1);
                    ok = ok && (u32)(vl >> 32) == tag;
                }
                S.pr[k] = V::make((u32)vh, (u32)vl);
            }
            if (__builtin_expect(bal(ok) == ~0ull, 1)) break;
            if (late || give_up()) { late = true; break; }
        }
#pragma unroll
        for (int k = J / 16; k < W / 16; ++k) L->row[J][16 * k + (lane & 15)] = S.pr[k];
        if (__builtin_expect(S.stop || late || khi < to_key<T>(V::eps_hi), 0)) {
            if (!S.stop && lane == 0) {
                if (late) {
                    // the 1-based column whose exchange timed out; info != 0 stops what is queued
                    __hip_atomic_store(A.abort, A.top + J + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    __hip_atomic_store(A.info, -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                } else if (g == 0) {
                    *A.info = A.top + J + 1;
                    *A.info_val = khi > to_key<T>(0) ? (double)V::make(from_key<T>(khi), rl(kl, wl)) : 0.0;
                }
            }
            S.stop = true;
        }
    } else {
        const int wave = threadIdx.x >> 6;
        if constexpr (J > 0) {
#pragma unroll
            for (int x = 0; x < R; ++x) update_rest<T, R, (J - 1) / 8 + 1, (J & 7) == 0>(S, x);
        }
        // the keys first; only the winner's row then crosses (a write of one lane's row
        // costs as much LDS time as one of 64 lanes: 14 cycles per 16 bytes)
#pragma unroll
        for (int x = 0; x < R; ++x)
            if (win[x]) L->key[b][wave] = uint4{gm, V::lo(S.a[x][J]), (u32)S.pos[x], 0u};
        __syncthreads();
        constexpr int NP = NW <= 1 ? 1 : NW <= 2 ? 2 : NW <= 4 ? 4 : NW <= 8 ? 8 : 16;
        const uint4 k = L->key[b][lane & (NP - 1)];
        const u32 km = group_max<NP>(k.x);
        bool w1[1] = {k.x == km};
        u64 wb = bal(w1[0]) & ((1ull << NP) - 1);
        if (__builtin_expect(__popcll(wb) != 1, 0)) {
            const u32 lo1[1] = {k.y};
            const int p1[1] = {(int)k.z};
            tie_break<1>(w1, lo1, p1);
            wb = bal(w1[0]) & ((1ull << NP) - 1);
        }
        const int wl = __builtin_ctzll(wb | (1ull << 63)) & (NP - 1);
        if (wl == wave) {
#pragma unroll
            for (int x = 0; x < R; ++x)
                if (win[x]) row_out<T, R, J>(S, x, L->row[J]);
        }
        khi = rl(k.x, wl);
        p = (int)rl(k.z, wl);
        if (__builtin_expect(S.stop || khi < to_key<T>(V::eps_hi), 0)) {
            if (!S.stop && threadIdx.x == 0) {
                *A.info = A.top + J + 1;
                *A.info_val = khi > to_key<T>(0) ? (double)V::make(from_key<T>(khi), rl(k.y, wl)) : 0.0;
            }
            S.stop = true;
        }
        __syncthreads();
#pragma unroll
        for (int q = J / 16; q < W / 16; ++q) S.pr[q] = L->row[J][16 * q + (lane & 15)];
    }
    if (__builtin_expect(S.stop, 0)) {
#pragma unroll
        for (int x = 0; x < R; ++x) S.l[x] = (T)0;
#pragma unroll
        for (int q = 0; q < W / 16; ++q) S.pr[q] = (T)0;
    } else {
        const T piv = V::make(rl(V::hi(S.pr[J / 16]), J & 15), rl(V::lo(S.pr[J / 16]), J & 15));
        const T r = V::rcp(piv);
#pragma unroll
        for (int x = 0; x < R; ++x) {
            const int ps = S.pos[x];
            const bool hit = ps == p;
            S.pos[x] = hit ? J : (ps == J ? p : ps);   // the interchange of positions J and p
            S.live[x] = hit ? 0u : S.live[x];
            T q = V::div(S.a[x][J], piv, r);
            if (__builtin_expect(khi >= to_key<T>(V::big_hi), 0)) q = S.a[x][J] / piv;
            S.a[x][J] = S.live[x] ? q : S.a[x][J];
            S.l[x] = S.live[x] ? q : (T)0;
        }
    }
    update_block<T, R, J>(S);
    if constexpr ((J & 7) == 7 && J + 1 < W) {   // the next column opens the next block
#pragma unroll
        for (int x = 0; x < R; ++x) fmac_row<(J + 1) & 15, 1>(&S.a[x][J + 1], S.pr[(J + 1) >> 4], S.l[x]);
    }
#pragma unroll
    for (int q = J / 16; q < W / 16; ++q) S.odd = fma((T)0, S.pr[q], S.odd);
}
template <typename T, int R, int NS, int NW, int J>
__device__ __forceinline__ void steps(Rows<T, R> &S, const PanelArgs<T> &A, int g, T *lr, Xch<T> *L)
{
    if constexpr (J < W) {
        if (J < A.w) step<T, R, NS, NW, J>(S, A, g, lr, L);
        steps<T, R, NS, NW, J + 1>(S, A, g, lr, L);
    }
}

// elect::place on the device: eight counts 128 bytes apart, then the elected die + 1
struct Ballot {
    int *count;
    int *info, *abort;
    int top, die;   // die: HW_REG_XCC_ID, bits 0..3
    __device__ bool stopped() const
    {
        return __hip_atomic_load(info, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
    }
    __device__ int add()
    {
        return __hip_atomic_fetch_add(count + 32 * die, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ void claim()
    {
        int none = 0;
        __hip_atomic_compare_exchange_strong(count + 32 * 8, &none, die + 1, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ int winner() const
    {
        return __hip_atomic_load(count + 32 * 8, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ int mine() const { return die + 1; }
    __device__ void timed_out()
    {
        __hip_atomic_store(abort, top + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(info, -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
};

// NW = 0: workgroups of 256 threads, each wave an agent of the exchange
template <typename T, int R, int NS, int NW>
__global__ __launch_bounds__(NW ? 64 * NW : 256, 2) void sub_panel_kernel(PanelArgs<T> A)
{
    constexpr int NWV = NW ? NW : 4;
    constexpr int E = 16 / (int)sizeof(T), NE = 128 / (int)sizeof(T), PE = NE + E;   // 128-byte row segments
    typedef typename Vec16<T>::type V;
    typedef typename Vec16u<T>::type Vu;
    __shared__ __align__(16) T seg[NWV][32 * PE];   // 32 rows of one segment, per wave
    __shared__ __align__(16) T lrow[NWV][W];
    __shared__ int dpos[NWV][32];
    __shared__ Xch<T> L;
    __shared__ int s_g;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    int g = wave;
    if constexpr (NW == 0) {
        if (t == 0) {
            Ballot m{A.elect, A.info, A.abort, A.top, (int)(__builtin_amdgcn_s_getreg(20 | (3 << 11)) & 7)};
            s_g = elect::place(m, (A.G + 3) / 4, A.spin_limit);
        }
        __syncthreads();
        if (s_g < 0) return;
        g = 4 * s_g + wave;
        if (g >= A.G) return;   // (no barrier follows: the waves are independent from here on)
    } else {
        // (one workgroup: nobody else sets info while it runs)
        if (*A.info != 0) return;
        if (t < 32) L.key[t >> 4][t & 15] = uint4{0, 0, 0, 0};
        __syncthreads();
    }
    T *sg = seg[wave];
    Rows<T, R> S;
    const int base = g * 64 * R;
    // rows in: 8 lanes read a 128-byte segment of a row, each lane then takes its row from LDS
    {
        V v[W / NE][R][8];
#pragma unroll
        for (int s = 0; s < W / NE; ++s)
#pragma unroll
            for (int x = 0; x < R; ++x)
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int row = min(base + 64 * x + 8 * i + (lane >> 3), A.m - 1), c = s * NE + E * (lane & 7);
                    const T *src = A.A + (long)row * A.lda + c;
                    if (c + E <= A.w) {
                        v[s][x][i] = *reinterpret_cast<const Vu *>(src);
                    } else {
#pragma unroll
                        for (int e = 0; e < E; ++e) v[s][x][i][e] = c + e < A.w ? src[e] : (T)0;
                    }
                }
#pragma unroll
        for (int s = 0; s < W / NE; ++s)
#pragma unroll
            for (int x = 0; x < R; ++x)
#pragma unroll
                for (int hf = 0; hf < 2; ++hf) {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        *reinterpret_cast<V *>(sg + (8 * i + (lane >> 3)) * PE + E * (lane & 7)) = v[s][x][4 * hf + i];
                    __builtin_amdgcn_wave_barrier();
                    const T *mine = sg + (lane & 31) * PE;
#pragma unroll
                    for (int c = 0; c < NE; c += E) {
                        const V q = *reinterpret_cast<const V *>(mine + c);
#pragma unroll
                        for (int e = 0; e < E; ++e)
                            if ((lane >> 5) == hf) S.a[x][s * NE + c + e] = q[e];
                    }
                    __builtin_amdgcn_wave_barrier();
                }
#pragma unroll
        for (int x = 0; x < R; ++x) {
            const int row = base + 64 * x + lane;
            S.pos[x] = row < A.m ? row : -1;
            S.live[x] = row < A.m ? 31u : 0u;
        }
    }
    S.stop = false;
    S.odd = (T)0;
    steps<T, R, NS, NW, 0>(S, A, g, lrow[wave], &L);
    // rows out, to their final positions, the same way (every row was read before the
    // first exchange of the panel ended)
#pragma unroll
    for (int x = 0; x < R; ++x)
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
#pragma unroll
            for (int s = 0; s < W / NE; ++s) {
                __builtin_amdgcn_wave_barrier();
                if ((lane >> 5) == hf) {
#pragma unroll
                    for (int c = 0; c < NE; c += E) {
                        V q;
#pragma unroll
                        for (int e = 0; e < E; ++e) q[e] = S.a[x][s * NE + c + e];
                        *reinterpret_cast<V *>(sg + (lane & 31) * PE + c) = q;
                    }
                    dpos[wave][lane & 31] = S.pos[x];
                }
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int r = 8 * i + (lane >> 3), c = s * NE + E * (lane & 7), d = dpos[wave][r];
                    const V q = *reinterpret_cast<const V *>(sg + r * PE + E * (lane & 7));
                    T *dst = A.A + (long)d * A.lda + c;
                    if (d >= 0) {
                        if (c + E <= A.w) {
                            *reinterpret_cast<Vu *>(dst) = q;
                        } else {
#pragma unroll
                            for (int e = 0; e < E; ++e)
                                if (c + e < A.w) dst[e] = q[e];
                        }
                    }
                }
            }
    // A finished row takes part in the later updates with multiplier zero, which changes it
    // if the pivot row of such an update is infinite or NaN: its later columns are those
    // that it had as the pivot row.
    if (__builtin_expect(bal(S.odd != (T)0) != 0, 0)) {
        __builtin_amdgcn_s_waitcnt(0);   // behind the rows as they went out
#pragma unroll
        for (int x = 0; x < R; ++x)
            if (S.live[x] == 0 && S.pos[x] >= 0)
#pragma unroll 1
                for (int d = S.pos[x], c = d + 1; c < A.w; ++c) A.A[(long)d * A.lda + c] = L.row[d][c];
    }
#pragma unroll
    for (int x = 0; x < R; ++x) {
        const int row = base + 64 * x + lane;
        if (S.pos[x] >= 0 && S.pos[x] != row) {
            const int at = atomicAdd(A.npairs, 1);
            A.pairs[2 * at] = A.top + S.pos[x];
            A.pairs[2 * at + 1] = A.top + row;
        }
    }
}

// ------------------------------------------------------------------ the other columns
template <typename T> struct ApplyArgs {
    long lda;
    int c0, w, rows;         // the sub-panel's first column and row, its width, rows of the matrix
    int ca, cb;              // columns to interchange, solve and update
    int la, lb;              // columns to interchange only
    int nstrip, nchunk, chunk, nleft;
    const int *pairs, *npairs;
    int *arrive;             // [strip] arrival counts, zero between launches
    int ncomp;               // lists to compose into out_pairs (0: none)
    const int *cpairs, *cn;  // the first of them (2 * SCIRS_SUB_PAIRS ints each) and their counts
    int *out_pairs, *out_n;
    int *label;              // [rows] identity between launches
    const int *info;
};
constexpr int ANT = 256, SC = 64, SP = SC + 2;   // threads, columns of a strip, LDS pitch

// A workgroup owns 64 columns and a chunk of the rows below the sub-panel.  Each
// forms the strip's U12 itself (the pivot rows' old contents, 2000 cycles of
// substitution) rather than wait for another launch to do so; the last of a strip's
// workgroups to have read those rows (an arrival count, nobody waits) writes the top
// rows and the rows that the interchanges displaced, so no row is overwritten while
// another workgroup may still read it.  Rank 32 per pass: latency-bound at small
// sizes (12 to 20 us a launch for FP64 of up to 7000 rows), HBM-bound above.
// A: the matrix; L11: the sub-panel's diagonal block (in columns that no workgroup writes).
// ZERO: the products summed from zero, else subtracted from the element one by one (the
// caller chooses; the sums' 16 registers more are kept out of the accumulation registers,
// for three workgroups per CU either way: n = 1999 solve 4.08 ms, with two 4.15 ms).
template <typename T, bool ZERO>
__global__ __launch_bounds__(ANT, 3) void sub_apply_kernel(T *__restrict__ A, const T *__restrict__ L11, ApplyArgs<T> a)
{
    if (*a.info != 0) return;
    typedef typename Mf<T>::V V4;
    __shared__ T Xs[W * SP], Us[W * SP];
    __shared__ int srow[W], ddst[SCIRS_SUB_PAIRS], dsrc[SCIRS_SUB_PAIRS], s_nd, s_last, skip[64];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int np = min(*a.npairs, (int)SCIRS_SUB_PAIRS);
    int bid = blockIdx.x;
    if (bid >= a.nstrip * a.nchunk + a.nleft) {
        // compose the lists: label[d] = original row now at d, then the moved rows
        for (int s = 0; s < a.ncomp; ++s) {
            const int *pp = a.cpairs + (size_t)s * 2 * SCIRS_SUB_PAIRS;
            const int n = min(a.cn[s * SCIRS_SUB_CTL], (int)SCIRS_SUB_PAIRS);
            const bool on = t < n;
            const int v = on ? a.label[pp[2 * t + 1]] : 0;
            __syncthreads();
            if (on) a.label[pp[2 * t]] = v;
            __syncthreads();
        }
        if (t == 0) s_nd = 0;
        __syncthreads();
        for (int s = 0; s < a.ncomp; ++s) {
            const int *pp = a.cpairs + (size_t)s * 2 * SCIRS_SUB_PAIRS;
            if (t < min(a.cn[s * SCIRS_SUB_CTL], (int)SCIRS_SUB_PAIRS)) {
                const int d = pp[2 * t], v = atomicExch(a.label + d, d);   // back to the identity; each moved row once
                if (v != d) {
                    const int at = atomicAdd(&s_nd, 1);
                    a.out_pairs[2 * at] = d;
                    a.out_pairs[2 * at + 1] = v;
                }
            }
        }
        __syncthreads();
        if (t == 0) *a.out_n = s_nd;
        return;
    }
    if (bid >= a.nstrip * a.nchunk) {
        // interchanges only: every read of the strip before its first write
        const int c = a.la + (bid - a.nstrip * a.nchunk) * SC + lane;
        const bool ok = c < a.lb;
        T v[SCIRS_SUB_PAIRS / 4];
#pragma unroll
        for (int u = 0; u < SCIRS_SUB_PAIRS / 4; ++u) {
            const int q = wave + 4 * u;
            v[u] = (ok && q < np) ? A[(long)a.pairs[2 * q + 1] * a.lda + c] : (T)0;
        }
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
#pragma unroll
        for (int u = 0; u < SCIRS_SUB_PAIRS / 4; ++u) {
            const int q = wave + 4 * u;
            if (ok && q < np) A[(long)a.pairs[2 * q] * a.lda + c] = v[u];
        }
        return;
    }
    const int strip = bid / a.nchunk, chunk = bid - strip * a.nchunk;
    const int cs = a.ca + strip * SC, c = cs + lane, top_end = a.c0 + a.w;
    const bool ok = c < a.cb;
    const int r0 = top_end + chunk * a.chunk, r1 = min(a.rows, r0 + a.chunk);
    if (t < W) srow[t] = a.c0 + t;
    if (t < 64) skip[t] = 0;
    if (t == 0) s_nd = 0;
    __syncthreads();
    if (t < np) {
        const int d = a.pairs[2 * t], s = a.pairs[2 * t + 1];
        if (d < top_end) {
            srow[d - a.c0] = s;
        } else {
            const int q = atomicAdd(&s_nd, 1);
            ddst[q] = d;
            dsrc[q] = s;
            if (d >= r0 && d < r1) atomicOr(&skip[(d - r0) >> 5], 1 << ((d - r0) & 31));
        }
    }
    __syncthreads();
    {
        T v[W / 4];
#pragma unroll
        for (int u = 0; u < W / 4; ++u) {
            const int i = wave + 4 * u;
            v[u] = (ok && i < a.w) ? A[(long)srow[i] * a.lda + c] : (T)0;
        }
#pragma unroll
        for (int u = 0; u < W / 4; ++u) Xs[(wave + 4 * u) * SP + lane] = v[u];
    }
    __syncthreads();
    if (t == 0) {
        int last = 1;
        if (a.nchunk > 1) {
            last = __hip_atomic_fetch_add(a.arrive + strip, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                   a.nchunk - 1;
            if (last) __hip_atomic_store(a.arrive + strip, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        s_last = last;
    }
    // U12: blocks of eight rows; every wave solves the 8 x 8 diagonal block itself (L11
    // at wave-uniform addresses: scalar loads), the rows below are split over the waves
    if (a.w == W) {
#pragma unroll 1
        for (int ib = 0; ib < W; ib += 8) {
            T x[8], ld[8][8];
#pragma unroll
            for (int q = 0; q < 8; ++q) x[q] = Xs[(ib + q) * SP + lane];
#pragma unroll
            for (int q = 1; q < 8; ++q)
#pragma unroll
                for (int pp = 0; pp < q; ++pp) ld[q][pp] = L11[(long)(ib + q) * a.lda + ib + pp];
#pragma unroll
            for (int q = 1; q < 8; ++q)
#pragma unroll
                for (int pp = 0; pp < q; ++pp) x[q] = fma(-ld[q][pp], x[pp], x[q]);
            if (wave == 0) {
#pragma unroll
                for (int q = 0; q < 8; ++q) Us[(ib + q) * SP + lane] = x[q];
            }
            for (int r = ib + 8 + wave; r < W; r += 4) {
                T acc = Xs[r * SP + lane];
                const T *lr = L11 + (long)r * a.lda + ib;
#pragma unroll
                for (int q = 0; q < 8; ++q) acc = fma(-lr[q], x[q], acc);
                Xs[r * SP + lane] = acc;
            }
            __syncthreads();
        }
    } else {   // a ragged last sub-panel
        if (wave == 0) {
            for (int i = 0; i < W; ++i) {
                T x = Xs[i * SP + lane];
                if (i < a.w)
                    for (int k = 0; k < i; ++k) x = fma(-L11[(long)i * a.lda + k], Us[k * SP + lane], x);
                Us[i * SP + lane] = x;
            }
        }
        __syncthreads();
    }
    // rank-32 update, the products in the order of the columns (lane group g, step i ->
    // k = 4 i + g): subtracted one after the other, every partial sum is then a Schur
    // complement, which the pivoting keeps small.  In the order that lets a lane load its
    // eight L entries as one piece (k = 8 g + i) the factors of N(0,1) matrices of 64 to
    // 400 rows had 7 to 17 % more error.
    const int l16 = lane & 15, grp = lane >> 4;
    T uf[SC / 16][8];
#pragma unroll
    for (int j = 0; j < SC / 16; ++j)
#pragma unroll
        for (int i = 0; i < 8; ++i) uf[j][i] = Us[(4 * i + grp) * SP + 16 * j + l16];
    auto load_l = [&](int row, T (&lf)[8]) {
        const T *src = A + (long)row * a.lda + a.c0;
        if (a.w == W) {
            // eight consecutive entries (k = 8 g + i), then the groups exchange: k's bits 4
            // and 3 (group) against bits 1 and 0 (register)
            constexpr int E = 16 / (int)sizeof(T);
            T v[8];
#pragma unroll
            for (int i = 0; i < 8; i += E) {
                const typename Vec16u<T>::type t = *reinterpret_cast<const typename Vec16u<T>::type *>(src + 8 * grp + i);
#pragma unroll
                for (int e = 0; e < E; ++e) v[i + e] = -t[e];
            }
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (!(i & 2)) swap_groups<32>(v[i], v[i + 2]);
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (!(i & 1)) swap_groups<16>(v[i], v[i + 1]);
#pragma unroll
            for (int i = 0; i < 8; ++i) lf[i] = v[4 * (i & 1) + (i >> 1)];
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) lf[i] = 4 * i + grp < a.w ? -src[4 * i + grp] : (T)0;
        }
    };
    // four tiles of one row block, two at a time where each needs a sum of its own
    auto update = [&](const T (&lf)[8], V4 (&c4)[SC / 16]) {
        if constexpr (ZERO) {
#pragma unroll
            for (int j = 0; j < SC / 16; j += 2) {
                V4 sum[2] = {};
#pragma unroll
                for (int i = 0; i < 8; ++i)
#pragma unroll
                    for (int h = 0; h < 2; ++h) sum[h] = Mf<T>::mac(lf[i], uf[j + h][i], sum[h]);
#pragma unroll
                for (int h = 0; h < 2; ++h) c4[j + h] += sum[h];
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
#pragma unroll
            for (int j = 0; j < SC / 16; ++j)
#pragma unroll
                for (int i = 0; i < 8; ++i) c4[j] = Mf<T>::mac(lf[i], uf[j][i], c4[j]);
        }
    };
    for (int rt = r0 + 16 * wave; rt < r1; rt += 64) {
        T lf[8];
        V4 acc[SC / 16];
        load_l(min(rt + l16, r1 - 1), lf);
#pragma unroll
        for (int j = 0; j < SC / 16; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int r = min(rt + Mf<T>::row(grp, q), r1 - 1), cc = min(cs + 16 * j + l16, a.cb - 1);
                acc[j][q] = A[(long)r * a.lda + cc];
            }
        update(lf, acc);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int r = rt + Mf<T>::row(grp, q);
            const bool st = r < r1 && !((skip[((r - r0) >> 5) & 63] >> ((r - r0) & 31)) & 1);
#pragma unroll
            for (int j = 0; j < SC / 16; ++j)
                if (st && cs + 16 * j + l16 < a.cb) A[(long)r * a.lda + cs + 16 * j + l16] = acc[j][q];
        }
    }
    if (!s_last) return;
    // the top rows' final contents, and the displaced rows (old contents from the top rows)
    const int nd = s_nd;
    V4 acc[SC / 16];
    const bool tile = 16 * wave < nd;
    if (tile) {
        T lf[8];
        load_l(ddst[min(16 * wave + l16, nd - 1)], lf);
#pragma unroll
        for (int j = 0; j < SC / 16; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int e = min(16 * wave + Mf<T>::row(grp, q), nd - 1), cc = min(cs + 16 * j + l16, a.cb - 1);
                acc[j][q] = A[(long)dsrc[e] * a.lda + cc];
            }
        update(lf, acc);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    for (int i = wave; i < a.w; i += 4)
        if (ok) A[(long)(a.c0 + i) * a.lda + c] = Us[i * SP + lane];
    if (tile) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int e = 16 * wave + Mf<T>::row(grp, q);
#pragma unroll
            for (int j = 0; j < SC / 16; ++j)
                if (e < nd && cs + 16 * j + l16 < a.cb) A[(long)ddst[e] * a.lda + cs + 16 * j + l16] = acc[j][q];
        }
    }
}

template <typename T, int R, int NS, int NW> int launch_panel(const PanelArgs<T> &pa, hipStream_t s)
{
    const int wgs = NW ? 1 : 8 * ((pa.G + 3) / 4 - 1) + 1;
    hipLaunchKernelGGL((sub_panel_kernel<T, R, NS, NW>), dim3(wgs), dim3(NW ? 64 * pa.G : 256), 0, s, pa);
    SCIRS_HIP_CHECK(hipGetLastError());
    return SCIRS_OK;
}

} // namespace sub

// Rows up to which sub_panel_kernel factors a panel (two FP64 or four FP32 rows
// per lane in 128 waves: their registers hold no more).
template <typename T> int scirs_sub_max_rows() { return 64 * SCIRS_SUB_AGENTS * (sizeof(T) == 8 ? 2 : 4); }
template int scirs_sub_max_rows<double>();
template int scirs_sub_max_rows<float>();

// Rows and waves: a workgroup exchanges through LDS up to 512 rows (FP64: 33 us
// there, 36 us through L2; at 1024 rows 44 against 37 us) or 1024 (FP32: 35
// against 37 us); beyond, as few rows per lane as 64 waves allow (each more costs
// 5 us a panel), 128 waves only past that (66 us at 16384 FP64 rows: the polls of
// 128 waves contend).
template <typename T>
int scirs_sub_panel(T *A, long lda, int rows, int c0, int w, int *pairs, int *npairs, int *elect, ScirsWork &wk,
                    hipStream_t s)
{
    using namespace sub;
    PanelArgs<T> pa;
    pa.A = A + (long)c0 * lda + c0; pa.lda = lda; pa.top = c0; pa.m = rows - c0; pa.w = w;
    pa.key = wk.sub_key; pa.row = wk.sub_row; pa.elect = elect;
    pa.seq = 0;
    pa.pairs = pairs; pa.npairs = npairs;
    pa.info = wk.info; pa.info_val = wk.info_val; pa.abort = wk.abort; pa.spin_limit = wk.spin_limit;
    auto waves = [&](int r) { return (pa.m + 64 * r - 1) / (64 * r); };
    constexpr bool f64 = std::is_same<T, double>::value;
    pa.G = waves(1);
    if (pa.G <= 4) return launch_panel<T, 1, 1, 4>(pa, s);
    if (pa.G <= 8) return launch_panel<T, 1, 1, 8>(pa, s);
    if constexpr (!f64) {
        if (waves(2) <= 8) { pa.G = waves(2); return launch_panel<T, 2, 1, 8>(pa, s); }
    }
    // from here on the waves exchange through the die's L2, by tags
    const tags::Range r = tags::draw(wk.sub_next, W, tags::CANDIDATE_TOP);
    if (r.clear)
        if (int rc = scirs_fill_int((int *)wk.sub_key, SCIRS_SUB_XCH_INTS, 0, s)) return rc;
    wk.sub_next = r.next;
    pa.seq = r.base;
    if (pa.G <= 64) return launch_panel<T, 1, 1, 0>(pa, s);
    pa.G = waves(2);
    if (pa.G <= 64) return launch_panel<T, 2, 1, 0>(pa, s);
    if constexpr (f64) {
        if (pa.G <= GMAX) return launch_panel<T, 2, 2, 0>(pa, s);
    } else {
        pa.G = waves(4);
        if (pa.G <= 64) return launch_panel<T, 4, 1, 0>(pa, s);
        if (pa.G <= GMAX) return launch_panel<T, 4, 2, 0>(pa, s);
    }
    scirs_set_error("sub-panel: %d rows exceed its registers", pa.m);
    return SCIRS_ERR_UNSUPPORTED;
}
template int scirs_sub_panel<double>(double *, long, int, int, int, int *, int *, int *, ScirsWork &, hipStream_t);
template int scirs_sub_panel<float>(float *, long, int, int, int, int *, int *, int *, ScirsWork &, hipStream_t);

template <typename T>
int scirs_sub_apply(T *A, long lda, int rows, int c0, int w, int ca, int cb, int la, int lb, bool from_zero,
                    const int *pairs, const int *npairs, int ncomp, const int *cpairs, const int *cn, int *out_pairs, int *out_n,
                    ScirsWork &wk, hipStream_t s)
{
    using namespace sub;
    ApplyArgs<T> a;
    a.lda = lda;
    a.c0 = c0; a.w = w; a.rows = rows;
    a.ca = ca; a.cb = cb; a.la = la; a.lb = lb;
    a.nstrip = cb > ca ? (cb - ca + SC - 1) / SC : 0;
    a.nleft = lb > la ? (lb - la + SC - 1) / SC : 0;
    if (a.nstrip > SCIRS_SUB_STRIPS) {
        scirs_set_error("sub-panel update: %d columns exceed the workspace", cb - ca);
        return SCIRS_ERR_ARG;
    }
    // 64 rows per workgroup until the device has two workgroups per CU, then longer
    // chunks (each workgroup forms U12 again); at most 2048 rows (the skip bits)
    const long tiles = (long)a.nstrip * ((rows - c0 - w + 63) / 64);
    a.chunk = 64 * (int)std::max(1l, std::min(32l, (tiles + 511) / 512));
    a.nchunk = std::max(1, (rows - c0 - w + a.chunk - 1) / a.chunk);
    a.pairs = pairs; a.npairs = npairs; a.arrive = wk.sub_arrive;
    a.ncomp = ncomp; a.cpairs = cpairs; a.cn = cn; a.out_pairs = out_pairs; a.out_n = out_n;
    a.label = wk.sub_label; a.info = wk.info;
    const int wgs = a.nstrip * a.nchunk + a.nleft + (ncomp > 0 ? 1 : 0);
    if (wgs == 0) return SCIRS_OK;
    const T *l11 = A + (long)c0 * lda + c0;
    if (from_zero) hipLaunchKernelGGL((sub_apply_kernel<T, true>), dim3(wgs), dim3(ANT), 0, s, A, l11, a);
    else hipLaunchKernelGGL((sub_apply_kernel<T, false>), dim3(wgs), dim3(ANT), 0, s, A, l11, a);
    SCIRS_HIP_CHECK(hipGetLastError());
    return SCIRS_OK;
}
template int scirs_sub_apply<double>(double *, long, int, int, int, int, int, int, int, bool, const int *, const int *,
                                     int, const int *, const int *, int *, int *, ScirsWork &, hipStream_t);
template int scirs_sub_apply<float>(float *, long, int, int, int, int, int, int, int, bool, const int *, const int *,
                                    int, const int *, const int *, int *, int *, ScirsWork &, hipStream_t);
