// Lane-level building blocks of the register-resident factorisations: products with
// a row of 16 lanes broadcast by DPP, 16-byte accesses, the 16 x 16 x 4 matrix-core
// operations.
#pragma once
#include <hip/hip_runtime.h>
#include <type_traits>

namespace lanes {

// acc[i] -= (element I0 + i of pr's 16-lane row) * l, i < K.  The s_nop covers a
// VALU write of pr right before its use as a DPP operand (two wait states).
#define SUB_L(TT, i, n) "v_fmac_" TT "_dpp %" #i ", %[p], -%[l] row_newbcast:%c[" #n "] row_mask:0xf bank_mask:0xf\n"
#define SUB_ASM(K_, TXT, ...)                                                                                  \
    if constexpr (K == K_)                                                                                     \
        asm("s_nop 1\n" TXT : __VA_ARGS__ : [p] "v"(pr), [l] "v"(l), [i0] "n"(I0), [i1] "n"(I0 + 1),           \
            [i2] "n"(I0 + 2), [i3] "n"(I0 + 3), [i4] "n"(I0 + 4), [i5] "n"(I0 + 5), [i6] "n"(I0 + 6),          \
            [i7] "n"(I0 + 7));
#define SUB_L2(TT) SUB_L(TT, 0, i0) SUB_L(TT, 1, i1)
#define SUB_L4(TT) SUB_L2(TT) SUB_L(TT, 2, i2) SUB_L(TT, 3, i3)
#define SUB_L6(TT) SUB_L4(TT) SUB_L(TT, 4, i4) SUB_L(TT, 5, i5)
#define SUB_O1 "+v"(a[0])
#define SUB_O2 SUB_O1, "+v"(a[1])
#define SUB_O3 SUB_O2, "+v"(a[2])
#define SUB_O4 SUB_O3, "+v"(a[3])
#define SUB_O5 SUB_O4, "+v"(a[4])
#define SUB_O6 SUB_O5, "+v"(a[5])
#define SUB_O7 SUB_O6, "+v"(a[6])
#define SUB_O8 SUB_O7, "+v"(a[7])
#define SUB_ALL(TT)                                                       \
    SUB_ASM(1, SUB_L(TT, 0, i0), SUB_O1)                                  \
    SUB_ASM(2, SUB_L2(TT), SUB_O2)                                        \
    SUB_ASM(3, SUB_L2(TT) SUB_L(TT, 2, i2), SUB_O3)                       \
    SUB_ASM(4, SUB_L4(TT), SUB_O4)                                        \
    SUB_ASM(5, SUB_L4(TT) SUB_L(TT, 4, i4), SUB_O5)                       \
    SUB_ASM(6, SUB_L6(TT), SUB_O6)                                        \
    SUB_ASM(7, SUB_L6(TT) SUB_L(TT, 6, i6), SUB_O7)                       \
    SUB_ASM(8, SUB_L6(TT) SUB_L(TT, 6, i6) SUB_L(TT, 7, i7), SUB_O8)
template <int I0, int K, typename T> __device__ __forceinline__ void fmac_row(T *a, T pr, T l)
{
    static_assert(K >= 1 && K <= 8 && I0 >= 0 && I0 + K <= 16, "one 16-lane row");
    if constexpr (std::is_same<T, double>::value) {
        SUB_ALL("f64")
    } else {
        SUB_ALL("f32")
    }
}

// a's lanes with bit N set <-> b's lanes with bit N clear
template <int N, typename T> __device__ __forceinline__ void swap_groups(T &a, T &b)
{
    auto word = [](unsigned &x, unsigned &y) {
        if constexpr (N == 32) {
            const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
            x = r[0]; y = r[1];
        } else {
            const auto r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
            x = r[0]; y = r[1];
        }
    };
    if constexpr (sizeof(T) == 8) {
        const unsigned long long p = (unsigned long long)__double_as_longlong(a), q = (unsigned long long)__double_as_longlong(b);
        unsigned pl = (unsigned)p, ph = (unsigned)(p >> 32), ql = (unsigned)q, qh = (unsigned)(q >> 32);
        word(pl, ql);
        word(ph, qh);
        a = __longlong_as_double((long long)(((unsigned long long)ph << 32) | pl));
        b = __longlong_as_double((long long)(((unsigned long long)qh << 32) | ql));
    } else {
        unsigned p = __float_as_uint(a), q = __float_as_uint(b);
        word(p, q);
        a = __uint_as_float(p);
        b = __uint_as_float(q);
    }
}

template <typename T> struct Vec16;
template <> struct Vec16<double> { typedef double type __attribute__((ext_vector_type(2))); };
template <> struct Vec16<float> { typedef float type __attribute__((ext_vector_type(4))); };
// a 16-byte access at an address aligned to an element only
template <typename T> struct Vec16u;
template <> struct Vec16u<double> { typedef double type __attribute__((ext_vector_type(2), aligned(8))); };
template <> struct Vec16u<float> { typedef float type __attribute__((ext_vector_type(4), aligned(4))); };

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
template <typename T> struct Mf;
template <> struct Mf<double> {
    typedef d4 V;
    static __device__ __forceinline__ V mac(double a, double b, V c)
    {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int grp, int q) { return grp + 4 * q; }
};
template <> struct Mf<float> {
    typedef f4 V;
    static __device__ __forceinline__ V mac(float a, float b, V c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int grp, int q) { return 4 * grp + q; }
};

} // namespace lanes
