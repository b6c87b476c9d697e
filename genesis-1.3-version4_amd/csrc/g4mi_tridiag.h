// The radial tridiagonal of the short-range space-charge solver
// (EFieldSolver::tridiag, EFieldSolver.cpp:260-272) by parallel cyclic
// reduction, one row per thread: each pass eliminates the neighbours `d` rows
// away, so log2(n) passes with one barrier and one division each replace the
// forward and backward recurrences, whose 2 n dependent steps (a division and
// an LDS round trip in each) ran on one lane while the workgroup waited.  The
// operator is diagonally dominant (1 + |low| + |up| on the diagonal), which
// is what the reduction needs to be as accurate as the recurrence.
#pragma once

#include <hip/hip_runtime.h>

namespace g4mi {

// Row t of n (n at most the workgroup's threads): low x[t-1] + mid x[t] +
// up x[t+1] = rhs, low of row 0 and up of row n-1 zero.  Every thread of the
// workgroup calls it (rows t >= n pass anything); buf: 8 n doubles of LDS
// that nothing reads or writes meanwhile.  Returns x[t].
__device__ __forceinline__ double2 tridiag_pcr(int t, int n, double low, double mid, double up, double2 rhs,
                                               double *buf) {
    const bool row = t < n;
    double r = 1.0 / (row ? mid : 1.0);
    low *= r, up *= r, rhs.x *= r, rhs.y *= r;
    double *now = buf, *next = buf + 4 * n;
    for (int d = 1; d < n; d *= 2) {
        if (row) {
            now[t] = low;
            now[n + t] = up;
            now[2 * n + t] = rhs.x;
            now[3 * n + t] = rhs.y;
        }
        __syncthreads();
        if (row) {
            const int a = t - d, b = t + d;
            double la = 0, ua = 0, xa = 0, ya = 0, lb = 0, ub = 0, xb = 0, yb = 0;
            if (a >= 0) la = now[a], ua = now[n + a], xa = now[2 * n + a], ya = now[3 * n + a];
            if (b < n) lb = now[b], ub = now[n + b], xb = now[2 * n + b], yb = now[3 * n + b];
            r = 1.0 / (1.0 - low * ua - up * lb);
            rhs.x = (rhs.x - low * xa - up * xb) * r;
            rhs.y = (rhs.y - low * ya - up * yb) * r;
            low = -low * la * r;
            up = -up * ub * r;
        }
        double *s = now;  // the next pass writes the other buffer: this one's readers need no barrier
        now = next;
        next = s;
    }
    return rhs;
}

}  // namespace g4mi
