// Both ADI half steps of one strip of columns by one wavefront
// (FieldSolverADI::ADI, FieldSolverADI.cpp:60-122), FP64 arithmetic on a field
// stored in FP64 or FP32.
//
// x-implicit: away from the grid's edges the inverse of 1 - i a d^2 is the
// convolution g w^|m|, w the root of i a (w^2 + 1) = (1 + 2 i a) w inside the
// unit circle.  It factors into one-sided sums, sum_m w^m S^m, and each of
// those, cut off at m < B 2^L, into (1 + .. + w^(B-1) S^(B-1)) (1 + w^B S^B)
// (1 + w^2B S^2B)...; the two sides of one binary factor together are
// (1 + w^2j) + w^j (S^j + S^-j), one complex product for the cell and one for
// the sum of its two neighbours j away.  B = 3, L = 1 reaches m = 5 with 26
// operations a cell (32 with a single term at 6, X), B = 2, L = 2 m = 7 with
// 30, where the band of the inverse takes 7 to 9 products of the neighbours'
// sums (42 to 52); B = 5, L = 2 reaches m = 19 with 48.  At the edges the
// system is the same convolution of the right-hand side continued oddly about
// the cells -1 and ng (where the solution is zero), so every lane runs the same
// code: its column is a mirror image with a sign outside the grid.
//
// y-implicit: a lane walks its column down, so Thomas' elimination runs as it
// stands (the reference's factors, row after row); the back substitution
// starts 8 NB rows below the 8 rows it completes, where its start is off by
// w^(8 NB + 1).  14 operations a cell (NB = 1) for the band's 46.
//
// A wavefront owns U columns and H on each side that its neighbours own too;
// it shares nothing with other wavefronts, so there is no barrier.  Neighbours
// come through LDS, which serves a wavefront's accesses in order (those 1 away
// by a wavefront shift where the right-hand side is not in LDS anyway).  The
// number of terms also sets the number of strips: 255 columns are 5 strips of
// 52 with 7 terms, 6 of 50 with 8.
//
// us a launch (floor: one read and one write of the field), and what it replaces:
//   FP64  1024 slices of 151^2,  7 terms  164 (159)   whole-width band product 438
//          509 slices of 255^2,  9 terms  263 (225)   the same 458
//                               16 terms  354         window recurrence 785
//                               20 terms  476         band of 33 terms 1446, Thomas 2713
//   FP32  1024 slices of 151^2,  6 terms  114  (79)   FP32 band product with correction 198
//         4096 slices of 255^2,  7 terms 1171 (903)   the same 1697
//                               12 terms 1853         the same 2243
//                               16 terms 1968         the same 3243
// Up to 9 terms FP64 is bound by HBM; FP32 and the rest by FP64 arithmetic
// (86 to 100 vector instructions a cell, 3 wavefronts per SIMD) and the halo's
// share of the columns.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

namespace g4mi {

constexpr int kStripRows = 8;  // rows completed per back substitution

// B 2^L terms (and one more, X) of the x convolution on each side, 8 NB rows
// of look-ahead.
template <int B, int L, int X, int NB>
struct StripGeom {
    static constexpr int terms = (B << L) + X;
    static constexpr int H = terms - 1;  // halo: the farthest neighbour
    static constexpr int U = 64 - 2 * H;
    static constexpr bool taps = B > 2 || X;    // the right-hand side itself goes to LDS
    static constexpr int pitch = 64 + 2 * H;
    static constexpr int lds = (L + taps) * pitch;  // double2 cells per wavefront
};

// The forms of the kernel, from the cheapest to the farthest reaching.
constexpr int kStripForms = 8;  // 6, 7, 8, 9, 12, 16, 20, 24 terms
template <int N>
using StripInt = std::integral_constant<int, N>;
template <class F>
inline void strip_form(int form, F f) {
    switch (form) {
    case 0: f(StripInt<3>{}, StripInt<1>{}, StripInt<0>{}, StripInt<1>{}); break;
    case 1: f(StripInt<3>{}, StripInt<1>{}, StripInt<1>{}, StripInt<1>{}); break;
    case 2: f(StripInt<2>{}, StripInt<2>{}, StripInt<0>{}, StripInt<1>{}); break;
    case 3: f(StripInt<2>{}, StripInt<2>{}, StripInt<1>{}, StripInt<1>{}); break;
    case 4: f(StripInt<3>{}, StripInt<2>{}, StripInt<0>{}, StripInt<2>{}); break;
    case 5: f(StripInt<2>{}, StripInt<3>{}, StripInt<0>{}, StripInt<2>{}); break;
    case 6: f(StripInt<5>{}, StripInt<2>{}, StripInt<0>{}, StripInt<3>{}); break;
    default: f(StripInt<3>{}, StripInt<3>{}, StripInt<0>{}, StripInt<3>{}); break;
    }
}
struct StripDims {
    int B, L, X, NB, U;
    int reach() const { return std::min((B << L) + X, kStripRows * NB + 1); }  // the power of w left out
    int count(int ng) const { return (ng + U - 1) / U; }
};
inline StripDims strip_dims(int form) {
    StripDims d{};
    strip_form(form, [&](auto b, auto l, auto x, auto n) {
        d = {b(), l(), x(), n(), StripGeom<b(), l(), x(), n()>::U};
    });
    return d;
}

// Blocks of four wavefronts, one per SIMD: the strips of a slice in one block
// (6 wavefronts at 255^2) leave room for only one block on a CU, 1.5
// wavefronts per SIMD of the registers' 3.  Workgroups go to the 8 XCDs in
// turn, so each XCD takes a run of strips: neighbours share their halo in its L2.
constexpr int kStripWaves = 4;
inline unsigned strip_blocks(int ns, int nstrip) {
    const long long nb = ((long long)ns * nstrip + kStripWaves - 1) / kStripWaves;
    return (unsigned)((nb + 7) / 8 * 8);
}

// Coefficients of a step size: the x convolution's first factor at distances
// 0 .. 4, its binary factors (cell and neighbours), the single term, and the y
// elimination's tables (device): cbet[ng] and -cwet[ng + kStripPad] (zero from
// ng on: the back substitution reads up to 8 NB rows past the last).  The
// cell's coefficients are kept as their difference from 1: they lie close to
// it, and their rounding would be the same for every cell and step (2e-16 to
// 4e-16 of the power a step, several times Thomas').
constexpr int kStripPad = 32;
struct StripCoef {
    double a;  // Im(cstep)
    double2 e[5], c[3], s[3], x;
    const double2 *cbet, *ncwet;
};

namespace strip {

// this wavefront's strip of all slices' (may lie past the last)
__device__ __forceinline__ long long item() {
    const long long b = (long long)(blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    return b * kStripWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
}
template <int CTRL>
__device__ __forceinline__ double shift1(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
// the sum of both neighbours one lane away (0 beyond the wavefront)
__device__ __forceinline__ double2 beside(double2 v) {
    return make_double2(shift1<0x138>(v.x) + shift1<0x130>(v.x), shift1<0x138>(v.y) + shift1<0x130>(v.y));
}
__device__ __forceinline__ double2 sum(double2 p, double2 q) { return make_double2(p.x + q.x, p.y + q.y); }
__device__ __forceinline__ double2 mul(double2 k, double2 v) {
    return make_double2(__builtin_fma(k.x, v.x, -(k.y * v.y)), __builtin_fma(k.x, v.y, k.y * v.x));
}
__device__ __forceinline__ double2 fma2(double2 k, double2 v, double2 c) {
    return make_double2(__builtin_fma(k.x, v.x, __builtin_fma(-k.y, v.y, c.x)),
                        __builtin_fma(k.x, v.y, __builtin_fma(k.y, v.x, c.y)));
}
// orders a wavefront's LDS accesses for the compiler (the LDS keeps them in order)
__device__ __forceinline__ void lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
}
// entry i (uniform) of a table that nothing writes during the launch: by the
// scalar cache, whatever the kernel stores elsewhere
__device__ __forceinline__ double2 entry(const double2 *t, int i) {
    typedef const __attribute__((address_space(4))) double *Const;
    Const p = (Const)(unsigned long long)t;
    return make_double2(p[2 * i], p[2 * i + 1]);
}
// coefficients kept in device memory, read the same way
__device__ __forceinline__ StripCoef coef(const StripCoef *d) {
    static_assert(sizeof(StripCoef) % 8 == 0, "");
    typedef const __attribute__((address_space(4))) unsigned long long *Const;
    Const p = (Const)(unsigned long long)d;
    union U {
        StripCoef k;
        unsigned long long w[sizeof(StripCoef) / 8];
        __device__ U() {}
    } u;
#pragma unroll
    for (int i = 0; i < (int)(sizeof(StripCoef) / 8); i++) u.w[i] = p[i];
    return u.k;
}
__device__ __forceinline__ double2 wide(double2 v) { return v; }
__device__ __forceinline__ double2 wide(float2 v) { return make_double2(v.x, v.y); }
__device__ __forceinline__ void narrow(double2 v, double2 *o) { *o = v; }
__device__ __forceinline__ void narrow(double2 v, float2 *o) { *o = make_float2((float)v.x, (float)v.y); }

}  // namespace strip

// Strip `q` of one slice: field u, source S (inside bx only), result uo;
// lds: StripGeom::lds cells of this wavefront, finite values in all of them.
// dg[8]: this lane's field sums (power, x, x^2, y, y^2 moments, far field,
// on-axis power), zero on lanes that complete no column.
template <class T2, int B, int L, int X, int NB>
__device__ __forceinline__ void adi_strip(const T2 *__restrict__ u, T2 *__restrict__ uo, const T2 *__restrict__ S,
                                          const int4 bx, int ng, int q,
                                          const StripCoef &k, double2 *lds, double (&dg)[8]) {
    using namespace strip;
    using G = StripGeom<B, L, X, NB>;
    constexpr int H = G::H, R = kStripRows, RING = R * (NB + 1);
    const int lane = threadIdx.x & 63;
    const int x = q * G::U - H + lane;
    const bool mine = lane >= H && lane < 64 - H && x < ng;
    // the odd continuation: cells t = x + 1 mod 2 (ng + 1), zero at 0 and ng + 1
    const int per = 2 * (ng + 1);
    int t = (x + 1) % per;
    if (t < 0) t += per;
    const bool fixed = t == 0 || t == ng + 1, image = t > ng + 1;
    const int col = fixed ? 0 : image ? per - t - 1 : t - 1;
    const double sign = fixed ? 0.0 : image ? -1.0 : 1.0;
    const bool edge = __any(sign != 1.0);
    // rows are uniform, so a load is a scalar row address and the lane's column;
    // source rows outside the box load the nearest row inside and drop it
    const bool sin = col >= bx.x && col <= bx.z;
    const unsigned ucol = (unsigned)(col * sizeof(T2)), scol = sin ? ucol : 0u, ocol = (unsigned)(x * (int)sizeof(T2));
    auto uload = [&](int r) -> T2 { return *(const T2 *)((const char *)(u + (long long)min(r, ng - 1) * ng) + ucol); };
    auto sload = [&](int r) -> T2 {
        return *(const T2 *)((const char *)(S + (long long)max(0, min(max(r, bx.y), bx.w)) * ng) + scol);
    };
    auto inbox = [&](int r) -> bool { return sin && r >= bx.y && r <= bx.w; };
    double2 *const erow = lds + H + lane;  // the right-hand side, then each factor's input
    double2 *row[L];
#pragma unroll
    for (int l = 0; l < L; l++) row[l] = lds + (l + G::taps) * G::pitch + H + lane;
    const double2 z2 = make_double2(0, 0);
    // rows r - 1, r, r + 1 of u at the start of row r, the next ones in flight
    double2 um = z2, uc = wide(uload(0)), un = ng > 1 ? wide(uload(1)) : z2;
    T2 up1 = uload(2), up2 = uload(3);
    T2 sv = sload(0), sp1 = sload(1), sp2 = sload(2);
    double2 Y[RING], yprev = z2;  // eliminated rows k0 .. k0 + RING
#pragma unroll
    for (int j = 0; j < RING; j++) Y[j] = z2;
    double s_w = 0, s_yw = 0, s_yyw = 0, s_re = 0, s_im = 0, s_cen = 0;
    const double shift = -0.5 * (double)(ng - 1);
    double dy = shift;  // of the next row completed
    // eight rows of the elimination, then the back substitution that completes
    // the eight rows above them.  FULL: the rows and
    // the two below them exist.
    auto block = [&](auto full, const int k0) {
        constexpr bool FULL = decltype(full)::value;
#pragma unroll
        for (int j = 0; j < R; j++) {
            const int r = k0 + R * NB + j;
            double2 y = z2;
            if (FULL || r < ng) {  // uniform
                // E = S + u + i a (u(r+1) - 2 u(r) + u(r-1)), zero rows outside
                T2 sb = sv;
                if (!inbox(r)) sb.x = sb.y = 0;
                const double2 s = wide(sb);
                const double dx = __builtin_fma(-2.0, uc.x, un.x) + um.x, dy = __builtin_fma(-2.0, uc.y, un.y) + um.y;
                double2 E = make_double2(__builtin_fma(-k.a, dy, s.x + uc.x), __builtin_fma(k.a, dx, s.y + uc.y));
                if (edge) {  // uniform
                    E.x *= sign;
                    E.y *= sign;
                }
                double2 v = fma2(k.e[0], E, E), far = z2;
                if (!G::taps) {
                    v = fma2(k.e[1], beside(E), v);
                } else {
                    *erow = E;
                    lds_order();
#pragma unroll
                    for (int d = 1; d < B; d++) v = fma2(k.e[d], sum(erow[-d], erow[d]), v);
                    if (X) far = sum(erow[-(B << L)], erow[B << L]);
                }
#pragma unroll
                for (int l = 0; l < L; l++) {
                    const int d = B << l;
                    *row[l] = v;
                    lds_order();
                    v = fma2(k.s[l], sum(row[l][-d], row[l][d]), fma2(k.c[l], v, v));
                }
                if (X) v = fma2(k.x, far, v);
                lds_order();
                // F = S + (1 + i a d_x^2) u' = S + 2 u' - E, then Thomas' step
                const double fx = __builtin_fma(2.0, v.x, s.x - E.x), fy = __builtin_fma(2.0, v.y, s.y - E.y);
                const double2 e = make_double2(__builtin_fma(-k.a, yprev.y, fx), __builtin_fma(k.a, yprev.x, fy));
                y = mul(entry(k.cbet, r), e);
                yprev = y;
                um = uc;
                uc = un;
                un = FULL || r + 2 < ng ? wide(up1) : z2;
                up1 = up2;
                sv = sp1;
                sp1 = sp2;
                up2 = uload(r + 4);
                sp2 = sload(r + 3);
                // the row is finished here: left to itself, the compiler moves the
                // elimination down to the substitution and keeps its operands instead
                asm volatile("" : "+v"(y.x), "+v"(y.y));
            }
            Y[R * NB + j] = y;
        }
        if (k0 >= 0) {  // uniform
            double2 v = Y[RING - 1];
#pragma unroll
            for (int j = RING - 2; j >= 0; j--) {
                v = fma2(entry(k.ncwet, k0 + j + 1), v, Y[j]);
                if (j < R) Y[j] = v;
            }
            if (mine) {
#pragma unroll
                for (int j = 0; j < R; j++) {
                    if (FULL || k0 + j < ng) {
                        const double2 o = Y[j];
                        narrow(o, (T2 *)((char *)(uo + (long long)(k0 + j) * ng) + ocol));
                        const double wei = __builtin_fma(o.x, o.x, o.y * o.y), yw = dy * wei;
                        s_w += wei;
                        s_yw += yw;
                        s_yyw = __builtin_fma(dy, yw, s_yyw);
                        dy += 1.0;
                        s_re += o.x;
                        s_im += o.y;
                        if (k0 + j == ng / 2) s_cen = wei;
                    }
                }
            }
        }
#pragma unroll
        for (int j = 0; j < R * NB; j++) Y[j] = Y[j + R];
    };
    int k0 = -R * NB;
    for (; k0 + RING + 2 <= ng; k0 += R) block(std::true_type{}, k0);
    for (; k0 < ng; k0 += R) block(std::false_type{}, k0);
    const double dx = (double)x + shift;
    dg[0] = s_w;
    dg[1] = dx * s_w;
    dg[2] = dx * dx * s_w;
    dg[3] = s_yw;
    dg[4] = s_yyw;
    dg[5] = s_re;
    dg[6] = s_im;
    dg[7] = x == ng / 2 ? s_cen : 0.0;
}

}  // namespace g4mi
