// csrc/gelu_poly.h against erfc, both in 64 bits, on 0 <= t <= 14: the largest of
// exp(-t^2 / 2) times its error, and of its relative error to t = 2, 6 and 14.
#define __host__
#define __device__
#include "gelu_poly.h"

#include <algorithm>
#include <cstdio>

int main()
{
    double weighted = 0, rel[3] = {0, 0, 0};
    for (int i = 0; i <= 1400000; ++i) {
        const double t = i * 1e-5;
        const double phi = std::erfc(t / std::sqrt(2.0)) / 2;  // exp(-t^2 / 2) P
        const double got = std::exp(-t * t / 2) * anima_hip::gelu_poly(t / (1 + t / 2));
        weighted = std::max(weighted, std::fabs(got - phi));
        double &r = rel[t <= 2 ? 0 : t <= 6 ? 1 : 2];
        r = std::max(r, std::fabs(got / phi - 1));
    }
    std::printf("%.3e %.3e %.3e %.3e\n", weighted, rel[0], rel[1], rel[2]);
    return 0;
}
