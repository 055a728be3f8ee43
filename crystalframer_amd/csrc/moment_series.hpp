// The angle basis as local moments: its mathematics, free of device code so that the host can evaluate it too.
//
// The Gaussian basis of the cosine has sigma = ws bins.  Around a node c (in bin units) the value of the basis function
// of bin m at u = c + half eps, eps in [-1, 1], is a power series in eps:
//     exp(-((m - u)/ws)^2 / 2) = sum_o eps^o D_o,  D_o = exp(-y^2/2) He_o(y) r^o / o!,  y = (m - c)/ws,  r = half/ws
// (generating function of the Hermite polynomials).  An image adds its NORD moments w eps^o at the node next to it, and
// the coefficients of eps^o are folded into the projection weights.
//
// Two sets of nodes:
//   every bin (training)    nodes at the 64 bins, half = 1/2, the series cut after NORD terms;
//   43 nodes (inference)    3/2 bins apart, half = 3/4; the terms of order NORD and more are folded into the lower ones
//                           modulo a quintic between the Legendre polynomial, whose mean square on [-1, 1] is the smallest,
//                           and the Chebyshev polynomial, whose maximum is: close to 1/8 of the cut series' error.
// Error over all u and bins, against 64 bits (ws = 4): every bin 1.43e-6 at most, 1.35e-7 rms; 43 nodes 1.22e-6, 1.31e-7.
// It is the mean square that a sum over many images shows: 38 nodes 5/3 bins apart, interpolated at the Chebyshev points, stay
// below 1.17e-6 but have 2.52e-7 rms.  And not all cosines are alike: the image that sets the first axis has the cosine 1 to
// it and 0 to the others, its opposite -1 and 0.  There the nodes of inference are exact (u = 63, 31.5 and 0 are nodes; with 42
// of them between the ends they were the ends of intervals), where the bins, for the cosine 0, are at their worst.  Output of
// one layer with large angle weights against float64, relative rms: every bin 8.0e-7, 43 nodes 3.0e-7; 42 nodes 9.0e-7, the 38
// nodes 8.1e-7.
#pragma once
#ifdef __HIPCC__
#define CFH_SERIES_FN __host__ __device__ __forceinline__
#else
#include <cmath>
#define CFH_SERIES_FN inline
#endif

namespace cfh {

#ifndef CFH_NORD
#define CFH_NORD 5
#endif
constexpr int NORD = CFH_NORD;                  // moments per axis
constexpr int LEAN_NUM = 3, LEAN_DEN = 2;       // distance of the nodes of inference in bins
constexpr int LEAN_NODES = 43;                  // node 0 at bin 0, node 42 at bin 63
constexpr double LEAN_FOLD_3 = 1.15, LEAN_FOLD_1 = 0.26;      // the quintic eps^5 - 1.15 eps^3 + 0.26 eps

CFH_SERIES_FN float series_exp(float x) {
#ifdef __HIP_DEVICE_COMPILE__
    return __expf(x);
#else
    return expf(x);
#endif
}
CFH_SERIES_FN double series_exp(double x) { return exp(x); }

// D_o for a node at every bin (half = 1/2), d = m - c
template <typename T>
CFH_SERIES_FN T moment_matrix(int o, T d, T ws) {
    const T y = d / ws;
    T h0 = (T)1, h1 = y;               // probabilists' Hermite polynomials
    T he = o == 0 ? h0 : h1;
    for (int n = 1; n < o; n++) { const T h2 = y * h1 - (T)n * h0; h0 = h1; h1 = h2; he = h2; }
    T coef = (T)1;
    for (int n = 1; n <= o; n++) coef /= (T)n * ((T)2 * ws);
    return series_exp((T)-0.5 * y * y) * he * coef;
}
// Coefficients of eps^0 ... eps^4 around a node of inference: D_0 ... D_8, those from D_5 on folded into the lower ones modulo
// the quintic.
template <typename T>
CFH_SERIES_FN void node_coefficients(T y, T r, T (&c)[NORD]) {
    static_assert(NORD == 5, "a quintic leaves five terms");
    constexpr double A = LEAN_FOLD_3, B = LEAN_FOLD_1;
    T D[9];
    D[0] = series_exp((T)-0.5 * y * y);
    D[1] = y * r * D[0];
#pragma unroll
    for (int o = 2; o < 9; o++) D[o] = (y * D[o - 1] - r * D[o - 2]) * (r * ((T)1 / (T)o));
    c[0] = D[0];
    c[1] = D[1] - (T)B * D[5] - (T)(A * B) * D[7];
    c[2] = D[2] - (T)B * D[6] - (T)(A * B) * D[8];
    c[3] = D[3] + (T)A * D[5] + (T)(A * A - B) * D[7];
    c[4] = D[4] + (T)A * D[6] + (T)(A * A - B) * D[8];
}

}  // namespace cfh
