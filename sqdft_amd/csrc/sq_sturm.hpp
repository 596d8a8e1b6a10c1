// sq_sturm.hpp -- extreme eigenvalue of a symmetric tridiagonal, by one thread.
// No HIP in here, so that it can be tested on the CPU: constexpr functions are
// device functions too.
#pragma once

namespace sqk {

// Largest eigenvalue of the symmetric tridiagonal sg T (T: diagonal d(0..n-1),
// off-diagonal e(0..n-2) through the accessors) by Newton's method on
// det(xI - sg T).  With q_i = p_i/p_{i-1} (Sturm ratios) and r_i = q_i'/q_i,
// p'/p = sum_i q_i'/q_i; past the largest root the characteristic polynomial
// is monotone and convex, so iterates started outside the spectrum move
// monotonically onto the root; the iteration stops at the first step that is
// no longer inward by more than rounding, and keeps that step where it is inward
// at all (left out, the error of the eigenvalue against long double was 4.6e-17
// instead of 3.6e-17 of the spectrum's size, root mean square; 3.6e-17 also for
// divisions iterated until no step is inward).  A start x is outside iff every
// q_i(x) > 0.  It first tries the near start b + g (just past the previous
// pass's extreme, which the new one can only exceed), widening the gap 16-fold
// per failed sweep, and falls back to the far start f (a Weyl bound, always
// outside).  recip(q): 1/q.  Returns false after 200 sweeps.
template <typename D, typename E, typename R>
constexpr bool tridiag_largest(D d, E e, R recip, int n, double sg, double f, double b, double g, double *out)
{
    bool probe = b + g < f;
    double x = probe ? b + g : f;
    for (int it = 0; it < 200; ++it) {
        double q = x - sg * d(0), dq = 1.0, iq = recip(q), s = iq;
        bool outside = q > 0.0;
#pragma unroll 4
        for (int i = 1; i < n; ++i) {
            const double ei = e(i - 1), r = ei * ei * iq;
            dq = 1.0 + r * dq * iq;
            q = (x - sg * d(i)) - r;
            outside = outside && q > 0.0;
            iq = recip(q);
            s += dq * iq;
        }
        if (probe && !outside) {
            g *= 16.0;           // inside: widen, or take the far start
            x = b + g;
            if (!(x < f)) { x = f; probe = false; }
            continue;
        }
        probe = false;
        const double xn = x - recip(s);
        if (!(xn < x - 2.0e-16 * (x < 0.0 ? -x : x))) {
            *out = xn < x ? xn : x;
            return true;
        }
        x = xn;
    }
    return false;
}

}  // namespace sqk
