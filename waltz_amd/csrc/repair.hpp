// Native repair decisions of a wave whose lanes hold reconstructed samples, for
// the last inverse passes that detect them instead of storing.
#pragma once

#include "common.hpp"

namespace wz {

template <class T>
struct WaveRepair {
    const T* orig;
    double bound;
    T bound_lo;  // the largest T <= bound
    SegList rep;
};

// Lanes (of in_m, the ballot of `in`) whose sample v needs a record against
// `ref` (its value: v - ref); clears *ok where it cannot meet the bound. As in
// the fused finest level, the rounded difference of the final value and the
// original settles the strict bound unless it is not below it; a wave with
// such a lane (a tie, a non-finite sample) runs the full test.
template <class T>
WZ_D unsigned long long repair_mask(T v, T ref, bool in, unsigned long long in_m, const WaveRepair<T>& r, bool* ok) {
    const T nb = T(r.bound), e = v - ref;
    const bool p = abs_t(e) > nb;
    const T d = p ? (v - e) - ref : e;
    if (!(in_m & ~__ballot(abs_t(d) < r.bound_lo))) return __ballot(p) & in_m;
    bool okj = true;
    T ej;
    const bool pj = repair_decision<T>(v, ref, nb, r.bound, &ej, &okj);
    *ok = *ok && (!in || okj);
    return __ballot(pj) & in_m;
}

}  // namespace wz
