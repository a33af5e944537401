// The polynomial of the GELU pass (dit.hip): P(u) = erfcx(t / sqrt(2)) / 2 with
// u = t / (1 + t / 2) and P(0) = 1/2, fitted here (weighted minimax) on
// 0 <= t <= 14.  exp(-t^2 / 2) times its error is at most 4.2e-9 (at t = 0.8); its
// relative error is at most 1e-7 to t = 2, 4e-6 to t = 6 and 6e-5 to t = 14.
// Compiled for the CPU too, where a test holds it to those figures in 64 bits.
#pragma once

#include <cmath>

namespace anima_hip {

template <typename T>
__host__ __device__ inline T gelu_poly(T u)
{
    constexpr float c[] = {-2.704118961e-04f, -2.087033645e-04f, -1.072004903e-03f,
                           6.642731605e-04f,  1.728924364e-02f,  5.052748695e-02f,
                           -3.989422023e-01f, 0.5f};
    T p = T(1.143050249e-04f);
#pragma unroll
    for (int i = 0; i < 8; ++i)
        p = std::fma(p, u, T(c[i]));
    return p;
}

}  // namespace anima_hip
