// The weighted product of column sums shared by the repeated-row sweeps.
#pragma once

#include "pqb_device.h"

namespace pqb {

// p = w * prod_{s < NS-1} c_s, as up to four chains (w folded into the first factor).
template <int NS>
__device__ __forceinline__ void wprod_first(const double (&cr)[NS], const double (&ci)[NS], double w,
                                            double& pr, double& pi) {
    constexpr int M = NS - 1;
    constexpr int NCH = (M >= 12) ? 4 : ((M >= 4) ? 2 : 1);
    double qr[NCH], qi[NCH];
#pragma unroll
    for (int q = 0; q < NCH; ++q) {
        const int lo = q * M / NCH;
        const int hi = (q + 1) * M / NCH;
        if (q == 0) {
            qr[0] = w * cr[0];
            qi[0] = w * ci[0];
        } else {
            qr[q] = cr[lo];
            qi[q] = ci[lo];
        }
#pragma unroll
        for (int j = lo + 1; j < hi; ++j) cmul(qr[q], qi[q], cr[j], ci[j]);
    }
    if constexpr (NCH == 4) {
        cmul(qr[0], qi[0], qr[1], qi[1]);
        cmul(qr[2], qi[2], qr[3], qi[3]);
        cmul(qr[0], qi[0], qr[2], qi[2]);
    } else if constexpr (NCH == 2) {
        cmul(qr[0], qi[0], qr[1], qi[1]);
    }
    pr = qr[0];
    pi = qi[0];
}

// acc += w * prod_s c_s
template <int NS>
__device__ __forceinline__ void add_wterm(const double (&cr)[NS], const double (&ci)[NS], double w,
                                          double& ar, double& ai) {
    if constexpr (NS == 1) {
        ar = fma(w, cr[0], ar);
        ai = fma(w, ci[0], ai);
    } else {
        double pr, pi;
        wprod_first<NS>(cr, ci, w, pr, pi);
        const double lr = cr[NS - 1], li = ci[NS - 1];
        ar = fma(pr, lr, ar);
        ar = fma(-pi, li, ar);
        ai = fma(pr, li, ai);
        ai = fma(pi, lr, ai);
    }
}

}  // namespace pqb
