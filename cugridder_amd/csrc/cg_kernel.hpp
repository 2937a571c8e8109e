// Kernel values in device code (ES, per-tap polynomials, learned), shared by the
// gridding and degridding kernels.
#pragma once
#include "cg_internal.hpp"

namespace cg {

__device__ __forceinline__ uint32_t geo_bits(float w) { return __float_as_uint(w); }
__device__ __forceinline__ uint32_t geo_bits(double w) { return (uint32_t)__double_as_longlong(w); }

__device__ __forceinline__ double es_val(double d, double beta, double c, double hw)
{
    return fabs(d) < hw ? exp(beta * sqrt(1.0 - c * d * d)) : 0.0;
}

// FP32 kernel values divided by e^beta (the MFMA gridders scale their sums
// back once, the other FP32 kernels every value):
//   psi(d) / e^beta = exp(beta (sqrt(1 - u) - 1) + y) = 2^(-beta log2(e) u / (1 + sqrt(1 - u)) + log2(e) y),
// u = c d^2, y the learned kernel's polynomial in s = 2 u - 1 (0 for the ES
// kernel).  The rewritten exponent has no cancellation near the centre, so
// the hardware square root, reciprocal and exp2 (about ten instructions
// instead of the library's correctly rounded expf and sqrtf) keep the large
// central taps within a few ulp; only the taps near the support edge, whose
// values are ~e^-beta of the centre, see errors up to ~beta * 1e-7.
struct KernelEvalN {
    float nb, ec, hw;
    int learned;
    const float *q;  // the launch argument's polynomial coefficients
    __device__ __forceinline__ explicit KernelEvalN(const GridArgs &g, int kw)
        : nb(g.f_nb), ec(g.f_ec), hw(0.5f * (float)kw), learned(g.learned), q(g.kq)
    {
    }
    // LEARNED: -1 follows the launch's flag, 0 / 1 fix the kernel at compile
    // time (no learned-polynomial code in the ES instantiations)
    template <int LEARNED = -1>
    __device__ __forceinline__ float at(float off0, int t) const
    {
        const float d = off0 + (float)t;
        const float u = ec * d * d;
        float y = nb * u * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_sqrtf(1.0f - u));
        if (LEARNED == 1 || (LEARNED < 0 && learned)) {
            const float s = 2.0f * u - 1.0f;
            float p = q[LEARN_MAXDEG];
#pragma unroll
            for (int k = LEARN_MAXDEG - 1; k >= 0; k--) p = p * s + q[k];
            y += 1.4426950408889634f * p;
        }
        const float v = __builtin_amdgcn_exp2f(y);
        return fabsf(d) < hw ? v : 0.0f;
    }
    __device__ __forceinline__ float operator()(float off0, int t) const { return at(off0, t); }
};

// Kernel-value source of the complex64 MFMA kernels, fixed per
// instantiation: the ES exp2 form or the per-tap polynomials (tp_on; KernelEvalN
// also takes kKerLearned for the exact learned form).
enum : int { kKerES = 0, kKerLearned = 1, kKerPoly = 2 };
// the MFMA kernels are instantiated for the ES form and the polynomials: a
// learned kernel always comes with its polynomials (grid_args), so a
// learned launch without them is refused
inline int ker_mode(const GridArgs &g) { return g.tp_on ? kKerPoly : g.learned ? -1 : kKerES; }

// FP32 kernel values psi(off0 + t) / e^beta (the normalisation of
// KernelEvalN) from per-tap polynomials in x = 2 off0 + kw - 1 (host fit,
// tap_polynomials), coefficients in LDS; zero outside the taps.  Eleven FMAs
// instead of the square root, reciprocal and exp2 of KernelEvalN, and the
// same cost for the ES and the learned kernel.
struct TapPolyN {
    const float *tab;  // kw rows of kTapStride coefficients
    int kw;
    __device__ __forceinline__ float operator()(float off0, int t) const
    {
        if (t < 0 || t >= kw) return 0.f;
        const float x = 2.f * off0 + (float)(kw - 1);
        const float4 *c = reinterpret_cast<const float4 *>(tab + t * kTapStride);
        const float4 c0 = c[0], c1 = c[1], c2 = c[2];
        float p = c2.z;
        p = p * x + c2.y;
        p = p * x + c2.x;
        p = p * x + c1.w;
        p = p * x + c1.z;
        p = p * x + c1.y;
        p = p * x + c1.x;
        p = p * x + c0.w;
        p = p * x + c0.z;
        p = p * x + c0.y;
        p = p * x + c0.x;
        return p;
    }
};

// Kernel values of a point: the ES kernel exp(beta sqrt(1 - c d^2)) at the
// tap offsets d, or the learned kernel, whose exponent adds the network's
// polynomial sum_k q_k s^k in s = 2 c d^2 - 1 (c = (2/kw)^2).  The choice is
// uniform across a launch and the coefficients are launch arguments, so
// they stay in scalar registers.  FP64 evaluates the formula directly; FP32
// is KernelEvalN times e^beta.
template <typename T>
struct KernelEval {
    T beta, ec, hw;
    int learned;
    T q[LEARN_MAXDEG + 1];
    __device__ __forceinline__ explicit KernelEval(const GridArgs &g, int kw)
        : beta((T)g.beta), ec((T)g.es_c), hw((T)(0.5 * kw)), learned(g.learned)
    {
#pragma unroll
        for (int k = 0; k <= LEARN_MAXDEG; k++) q[k] = (T)g.kq[k];
    }
    // value of tap t of a point whose first tap sits at offset off0
    __device__ __forceinline__ T operator()(T off0, int t) const
    {
        const T d = off0 + (T)t;
        if (!learned) return es_val(d, beta, ec, hw);
        if (!(fabs(d) < hw)) return (T)0;
        const T r = (T)1 - ec * d * d;
        const T s = (T)1 - (T)2 * r;
        T y = q[LEARN_MAXDEG];
#pragma unroll
        for (int k = LEARN_MAXDEG - 1; k >= 0; k--) y = y * s + q[k];
        return exp(beta * sqrt(r) + y);
    }
};
template <>
struct KernelEval<float> : KernelEvalN {
    float eb;  // e^beta
    __device__ __forceinline__ explicit KernelEval(const GridArgs &g, int kw)
        : KernelEvalN(g, kw), eb(g.f_e1)
    {
    }
    __device__ __forceinline__ float operator()(float off0, int t) const
    {
        return KernelEvalN::operator()(off0, t) * eb;
    }
};

__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace cg
