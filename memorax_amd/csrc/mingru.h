// The MinGRU cell's element map: a = sigma(-z), b = sigma(z) g(x), g(x) = x + 0.5 (x >= 0) | sigma(x).
#pragma once
#include <hip/hip_runtime.h>

namespace mrx {
namespace {

struct MinGru {
    // s = sigma(z) and a = sigma(-z), each from exp(-|z|): neither is 1 - the other, so a small
    // gate keeps its relative precision (the cumulative decay is a product of them)
    // The hardware exponential and reciprocal (a few ulp) instead of the library routines: the
    // kernels stream at HBM rate only if a step costs a handful of instructions per element.
    static __device__ __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
    static __device__ __forceinline__ void gates(float z, float &s, float &a)
    {
        const float e = __expf(-fabsf(z)), r = rcp(1.0f + e), q = e * r;
        s = z >= 0.0f ? r : q;
        a = z >= 0.0f ? q : r;
    }
    // sigma(x) for x < 0 from exp(x) <= 1 (no overflow however negative x is)
    static __device__ __forceinline__ float g(float x)
    {
        const float e = __expf(-fabsf(x));
        return x >= 0.0f ? x + 0.5f : e * rcp(1.0f + e);
    }
    static __device__ __forceinline__ float dg(float x)
    {
        const float e = __expf(-fabsf(x)), r = rcp(1.0f + e);
        return x >= 0.0f ? 1.0f : e * r * r;  // sigma (1 - sigma) = e / (1 + e)^2
    }
    // (z, x) -> (a, b) in place
    static __device__ __forceinline__ void coeffs(float &za, float &xb)
    {
        float s, a;
        gates(za, s, a);
        xb = s * g(xb);
        za = a;
    }
    // gradients of one step: lam = dL/db_t, da = dL/da_t (0 at a reset) -> dz, dx
    static __device__ __forceinline__ void grads(float z, float x, float lam, float da, float &dz, float &dx)
    {
        float s, a;
        gates(z, s, a);
        dz = s * a * (g(x) * lam - da);  // sigma'(z) = s a; b = s g(x), a = 1 - s
        dx = lam * s * dg(x);
    }
};

}  // namespace
}  // namespace mrx
