// Device helpers shared by the FFT kernels (cg_fft.hip, cg_fftmix.hip): complex
// arithmetic, butterflies in registers, the live columns.
#pragma once
#include <type_traits>

#include "cg_internal.hpp"

namespace cg {

// max elements per thread: 16 complex64 or 8 complex128
template <typename T>
constexpr int fft_ept() { return sizeof(T) == 4 ? 16 : 8; }

template <typename T>
__device__ __forceinline__ cx_t<T> cmul(cx_t<T> a, cx_t<T> b)
{
    return mkc(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
template <typename T>
__device__ __forceinline__ cx_t<T> cadd(cx_t<T> a, cx_t<T> b) { return mkc(a.x + b.x, a.y + b.y); }
template <typename T>
__device__ __forceinline__ cx_t<T> csub(cx_t<T> a, cx_t<T> b) { return mkc(a.x - b.x, a.y - b.y); }
// multiply by dir*i
template <typename T, int DIR>
__device__ __forceinline__ cx_t<T> cmul_i(cx_t<T> a)
{
    return DIR > 0 ? mkc(-a.y, a.x) : mkc(a.y, -a.x);
}

// workgroup barrier that orders LDS only: outstanding global loads (the
// row prefetch) are not waited for
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// cos and sin of 2 pi k / n at compile time: the angle folded to within
// pi / 4 of a quarter turn, there the Taylor series
struct UnitRoot {
    double c, s;
};
constexpr UnitRoot unit_root(int k, int n)
{
    k %= n;
    const int q = (4 * k + n / 2) / n;  // nearest quarter turn
    const double x = 2.0 * kPi * (4 * k - q * n) / (4.0 * n);
    double c = 1.0, s = x, tc = 1.0, ts = x;
    for (int j = 1; j < 14; j++) {
        tc *= -x * x / ((2 * j - 1) * (2 * j));
        ts *= -x * x / ((2 * j) * (2 * j + 1));
        c += tc;
        s += ts;
    }
    switch (q & 3) {
    case 1: return UnitRoot{-s, c};
    case 2: return UnitRoot{-c, -s};
    case 3: return UnitRoot{s, -c};
    default: return UnitRoot{c, s};
    }
}
template <int K, int N>
struct Root {
    static constexpr UnitRoot w = unit_root(K, N);
};

template <typename T, int R, int DIR>
__device__ __forceinline__ void dft_small(cx_t<T> *a);

template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F &&f)
{
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// composite radix R = A B in registers.  Coprime A and B (6, 10, 12, 15, 20):
// Good's mapping x[(B i + A j) mod R], X[k] at (k mod A, k mod B), without
// twiddles; 9 = 3 x 3 and 25 = 5 x 5 with the twiddles w_R^(j k1).
template <typename T, int R, int DIR>
__device__ __forceinline__ void dft_split(cx_t<T> *a)
{
    constexpr int A = R == 25 ? 5 : R % 3 == 0 ? 3 : R == 20 ? 4 : 2, B = R / A;
    static_assert(A * B == R && (R == 6 || R == 9 || R == 10 || R == 12 || R == 15 || R == 20 || R == 25),
                  "radix");
    cx_t<T> y[B][A];
    if constexpr (A == B) {
        static_for<0, B>([&](auto J) {
            constexpr int j = decltype(J)::value;
            cx_t<T> t[A];
#pragma unroll
            for (int i = 0; i < A; i++) t[i] = a[B * i + j];
            dft_small<T, A, DIR>(t);
            y[j][0] = t[0];
            static_for<1, A>([&](auto K1) {
                constexpr int k1 = decltype(K1)::value;
                constexpr UnitRoot w = Root<j * k1, R>::w;
                const T wr = (T)w.c, wi = (T)(DIR * w.s);
                y[j][k1] = j == 0 ? t[k1] : mkc(t[k1].x * wr - t[k1].y * wi, t[k1].x * wi + t[k1].y * wr);
            });
        });
#pragma unroll
        for (int k1 = 0; k1 < A; k1++) {
            cx_t<T> t[B];
#pragma unroll
            for (int j = 0; j < B; j++) t[j] = y[j][k1];
            dft_small<T, B, DIR>(t);
#pragma unroll
            for (int k2 = 0; k2 < B; k2++) a[k1 + A * k2] = t[k2];
        }
    } else {
#pragma unroll
        for (int j = 0; j < B; j++) {
            cx_t<T> t[A];
#pragma unroll
            for (int i = 0; i < A; i++) t[i] = a[(B * i + A * j) % R];
            dft_small<T, A, DIR>(t);
#pragma unroll
            for (int k1 = 0; k1 < A; k1++) y[j][k1] = t[k1];
        }
        static_for<0, A>([&](auto K1) {
            constexpr int k1 = decltype(K1)::value;
            cx_t<T> t[B];
#pragma unroll
            for (int j = 0; j < B; j++) t[j] = y[j][k1];
            dft_small<T, B, DIR>(t);
            static_for<0, R>([&](auto K) {
                constexpr int k = decltype(K)::value;
                if constexpr (k % A == k1) a[k] = t[k % B];
            });
        });
    }
}

template <typename T, int R, int DIR>
__device__ __forceinline__ void dft_small(cx_t<T> *a)
{
    if constexpr (R == 2) {
        cx_t<T> t = a[0];
        a[0] = cadd<T>(t, a[1]);
        a[1] = csub<T>(t, a[1]);
    } else if constexpr (R == 4) {
        cx_t<T> t0 = cadd<T>(a[0], a[2]), t1 = csub<T>(a[0], a[2]);
        cx_t<T> t2 = cadd<T>(a[1], a[3]), t3 = cmul_i<T, DIR>(csub<T>(a[1], a[3]));
        a[0] = cadd<T>(t0, t2);
        a[2] = csub<T>(t0, t2);
        a[1] = cadd<T>(t1, t3);
        a[3] = csub<T>(t1, t3);
    } else if constexpr (R == 8) {
        const T r2 = (T)0.70710678118654752440084436210485;
        cx_t<T> e[4] = {a[0], a[2], a[4], a[6]};
        cx_t<T> o[4] = {a[1], a[3], a[5], a[7]};
        dft_small<T, 4, DIR>(e);
        dft_small<T, 4, DIR>(o);
        // W8^k o_k, W8 = (1 + dir i)/sqrt2
        cx_t<T> w1 = mkc(r2 * (o[1].x - DIR * o[1].y), r2 * (o[1].y + DIR * o[1].x));
        cx_t<T> w2 = cmul_i<T, DIR>(o[2]);
        cx_t<T> w3 = mkc(r2 * (-o[3].x - DIR * o[3].y), r2 * (-o[3].y + DIR * o[3].x));
        a[0] = cadd<T>(e[0], o[0]);
        a[4] = csub<T>(e[0], o[0]);
        a[1] = cadd<T>(e[1], w1);
        a[5] = csub<T>(e[1], w1);
        a[2] = cadd<T>(e[2], w2);
        a[6] = csub<T>(e[2], w2);
        a[3] = cadd<T>(e[3], w3);
        a[7] = csub<T>(e[3], w3);
    } else if constexpr (R == 16) {
        // 16 = 4 x 4: X[k1 + 4 k2] = sum_n2 w16^(n2 k1) [sum_n1 x[4 n1 + n2] w4^(n1 k1)] w4^(n2 k2)
        const T c1 = (T)0.92387953251128675612818318939679;  // cos(pi/8)
        const T s1 = (T)0.38268343236508977172845998403040;  // sin(pi/8)
        const T r2 = (T)0.70710678118654752440084436210485;
        cx_t<T> y[4][4];
#pragma unroll
        for (int n2 = 0; n2 < 4; n2++) {
            cx_t<T> t[4] = {a[n2], a[4 + n2], a[8 + n2], a[12 + n2]};
            dft_small<T, 4, DIR>(t);
#pragma unroll
            for (int k1 = 0; k1 < 4; k1++) y[n2][k1] = t[k1];
        }
        // w16^(DIR m) for m = n2 k1 in {1, 2, 3, 4, 6, 9}
        auto tw = [&](cx_t<T> v, T wr, T wi) { return mkc(v.x * wr - v.y * wi, v.x * wi + v.y * wr); };
        const T d = (T)DIR;
        y[1][1] = tw(y[1][1], c1, d * s1);
        y[1][2] = tw(y[1][2], r2, d * r2);
        y[1][3] = tw(y[1][3], s1, d * c1);
        y[2][1] = tw(y[2][1], r2, d * r2);
        y[2][2] = cmul_i<T, DIR>(y[2][2]);
        y[2][3] = tw(y[2][3], -r2, d * r2);
        y[3][1] = tw(y[3][1], s1, d * c1);
        y[3][2] = tw(y[3][2], -r2, d * r2);
        y[3][3] = tw(y[3][3], -c1, -d * s1);
#pragma unroll
        for (int k1 = 0; k1 < 4; k1++) {
            cx_t<T> t[4] = {y[0][k1], y[1][k1], y[2][k1], y[3][k1]};
            dft_small<T, 4, DIR>(t);
#pragma unroll
            for (int k2 = 0; k2 < 4; k2++) a[k1 + 4 * k2] = t[k2];
        }
    } else if constexpr (R == 3) {
        const T h = (T)0.86602540378443864676372317075294;  // sqrt(3)/2
        cx_t<T> t = cadd<T>(a[1], a[2]);
        cx_t<T> d = csub<T>(a[1], a[2]);
        cx_t<T> m = mkc(a[0].x - (T)0.5 * t.x, a[0].y - (T)0.5 * t.y);
        cx_t<T> e = cmul_i<T, DIR>(mkc(h * d.x, h * d.y));
        a[0] = cadd<T>(a[0], t);
        a[1] = cadd<T>(m, e);
        a[2] = csub<T>(m, e);
    } else if constexpr (R == 5) {
        const T c1 = (T)0.30901699437494742410229341718282;    // cos(2pi/5)
        const T c2 = (T)-0.80901699437494742410229341718282;   // cos(4pi/5)
        const T s1 = (T)0.95105651629515357211643933337938;    // sin(2pi/5)
        const T s2 = (T)0.58778525229247312916870595463907;    // sin(4pi/5)
        cx_t<T> t1 = cadd<T>(a[1], a[4]), t2 = cadd<T>(a[2], a[3]);
        cx_t<T> d1 = csub<T>(a[1], a[4]), d2 = csub<T>(a[2], a[3]);
        cx_t<T> b1 = mkc(a[0].x + c1 * t1.x + c2 * t2.x, a[0].y + c1 * t1.y + c2 * t2.y);
        cx_t<T> b2 = mkc(a[0].x + c2 * t1.x + c1 * t2.x, a[0].y + c2 * t1.y + c1 * t2.y);
        cx_t<T> e1 = cmul_i<T, DIR>(mkc(s1 * d1.x + s2 * d2.x, s1 * d1.y + s2 * d2.y));
        cx_t<T> e2 = cmul_i<T, DIR>(mkc(s2 * d1.x - s1 * d2.x, s2 * d1.y - s1 * d2.y));
        a[0] = mkc(a[0].x + t1.x + t2.x, a[0].y + t1.y + t2.y);
        a[1] = cadd<T>(b1, e1);
        a[4] = csub<T>(b1, e1);
        a[2] = cadd<T>(b2, e2);
        a[3] = csub<T>(b2, e2);
    } else {
        dft_split<T, R, DIR>(a);
    }
}

// fast-axis indices that carry image pixels: k < a or k >= b
struct Live {
    int a, b;
    __host__ __device__ bool operator()(int k) const { return k < a || k >= b; }
    __host__ __device__ int count(int n) const { return a + (n - b); }
    // k-th live index
    __host__ __device__ int at(int k) const { return k < a ? k : k - a + b; }
};

}  // namespace cg
