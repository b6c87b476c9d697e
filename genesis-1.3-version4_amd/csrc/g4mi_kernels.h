// Launchers of the FP64 device kernels (defined in g4mi_kernels.hip).
#pragma once

#include "g4mi_adi_strip.h"
#include "g4mi_common.h"

namespace g4mi {

// Thomas factors of the constant-coefficient ADI systems (complex, ngrid
// entries each, device pointers) and cstep = (0, cstep).
struct AdiFactors {
    const double2 *c, *cbet, *cwet;
    double cstep;
    int ngrid;
};

void launch_transverse(hipStream_t s, long long n, const double *g, double *x, double *y,
                       double *px, double *py, const TransParams &p);
void launch_r56(hipStream_t s, long long n, const double *g, double *th, double r56, double g0);
// Energy kicks after the push (Beam::track, src/Core/Beam.cpp:105-106), in
// the reference's order: gamma += beamlet_dg[boff[s] + (i - off[s]) / nbins]
// (Incoherent::apply) when beamlet_dg is set, then gamma += slice_dg[s]
// (Collective::apply) when slice_dg is set.  One workgroup per slice.
void launch_kicks(hipStream_t s, int ns, const long long *off, double *g, const double *beamlet_dg,
                  const long long *boff, int nbins, const double *slice_dg);
void launch_slice_moments(hipStream_t s, int ns, const long long *off, const double *x,
                          const double *y, double *mom);
void launch_slice_sizes(hipStream_t s, int ns, const long long *off, const double *cur,
                        const double *mom, double *fsize, double *cen);
void launch_lsc_long(hipStream_t s, int ns, const double *cur, const double *fsize, double sl,
                     double gamma, double scl, double *esc);
void launch_sc_rbound(hipStream_t s, int ns, const long long *off, const double *x,
                      const double *y, const double *cen, double *rbound);
void launch_sc_scan(hipStream_t s, int ns, const long long *off, const double *rbound,
                    double *rmax_state, int ngr, double *dr);
void launch_sc_solve(hipStream_t s, int ns, const long long *off, const double *x,
                     const double *y, const double *th, const double *cur, const double *cen,
                     const double *dr, int ngr, int nz, int nphi, double ks, double gz2,
                     double *ez, double *efield);
void launch_push(hipStream_t s, int nblocks, const int *blk_slice, const long long *blk_begin,
                 const long long *off, double *g, double *th, const double *x, const double *y,
                 const double *px, const double *py, const double2 *field, const double *esc,
                 const double *ezsc, const PushParams &p);
// The step's particle passes in two kernels (one workgroup per slice).
// front: first transverse half step, moments mom[4 ns] (the same bits as
// launch_slice_moments), fsize, cen, rbound (when sc), the in-grid
// footprint box pbox[ns] of each slice and pmaxf[ns], the largest
// sqrt(faw2) / gamma of its in-grid particles (the deposit's fixed-point
// scale).
void launch_fp64_front(hipStream_t s, int ns, const long long *off, const double *g, double *x, double *y,
                       double *px, double *py, const double *cur, const TransParams &t1, bool moments, bool sc,
                       double gridmax, double dgrid, int ng, double *mom, double *fsize, double *cen,
                       double *rbound, int4 *pbox, const DepositParams &d, double *pmaxf);
// Parameters of the main kernel: the push (fundamental only), the second
// transverse half step, R56, the short-range solver and the deposit.
struct FuseParams {
    PushParams p;
    TransParams t2;
    DepositParams d;
    double r56, gamma0;            // R56 (chicane != 0)
    double ks, gz2;                // short-range solver
    int chicane, use_sc, ngr, nz, nphi;
};
// Mode-solution cells the main kernel holds: (2 nphi + 1) nz ngr must fit.
int fp64_main_modes();
// main: short-range solve, push, R56, second transverse half step, beam sums
// beamsum[8 ns] (the layout of launch_diag_beam) and the deposit of the
// slice's source (src, box) when f.d.enabled.
void launch_fp64_main(hipStream_t s, int ns, const long long *off, double *g, double *th, double *x, double *y,
                      double *px, double *py, const double2 *field, const double *esc, const double *cur,
                      const double *cen, const double *dr, double *efield, const int4 *pbox,
                      const double *pmaxf, double2 *src, int4 *box, double *beamsum, const FuseParams &f);
// The particle half of a step over blocks of particles (small windows).
// track: the push, R56 and second half step, the first half step before them
// when `first`; per-block sums part[8 nblocks], per-slice pmax.
struct TrackParams {
    PushParams p;
    TransParams t1, t2;
    DepositParams d;               // the fundamental's (its enabled and faw2 terms); gridmax: the widest field's
    double r56, gamma0;            // R56 (chicane != 0)
    int chicane, first;
};
void launch_track(hipStream_t s, int nblocks, const int *blk_slice, const long long *blk_begin,
                  const long long *off, double *g, double *th, double *x, double *y, double *px, double *py,
                  const double2 *field, const double *esc, const double *ezsc, const TrackParams &f, double *part,
                  unsigned long long *pmax);
// The deposit split over the slices' particles: acc (ns ngrid^2 fixed-point
// cells, all zero before and after) and corner (4 ns) of this step; leaves
// corner_next and, unless null, pmax_next empty for the next one.
void launch_deposit_split(hipStream_t s, int ns, long long ntot, long long maxn, const long long *off,
                          const double *g, const double *th, const double *x, const double *y, const double *cur,
                          const unsigned long long *pmax, unsigned long long *pmax_next, long long *acc,
                          int *corner, int *corner_next, double2 *src, int4 *box, const DepositParams &p);
void launch_deposit(hipStream_t s, int ns, const long long *off, const double *g,
                    const double *th, const double *x, const double *y, const double *cur,
                    double2 *src, int4 *box, const DepositParams &p);
void launch_adi(hipStream_t s, int ns, double2 *field, double2 *work, const double2 *src,
                const int4 *box, const AdiFactors &f, int first);
// The same with a wavefront per line and the lines' systems as a product of
// log2 convolutions (grids up to kLineMax, coefficients from the host); the
// field sums of every four columns to tilediag [ns][line_blocks(ng)][8] (null:
// none).
constexpr int kLineMax = 512, kLineLevels = 10;
struct LineCoef {
    double a;       // Im(cstep)
    int levels;     // 2^levels terms on each side
    int d[kLineLevels];
    double2 c[kLineLevels], s[kLineLevels];  // factor at distance d: cell (less 1) and neighbours
};
inline int line_blocks(int ng) { return (ng + 3) / 4; }
void launch_adi_lines(hipStream_t s, int ns, double2 *field, double2 *work, const double2 *src, const int4 *box,
                      const LineCoef &k, int ng, int first, double *tilediag);
// Fused two-sweep ADI (one workgroup per slice, ngrid <= 256) with
// register-window back substitution of `tile` cells (8 or 16), tiles
// prefetched into registers (prefetch=1) or loaded when needed (0), and the
// field diagnostics sums of every storage slice into diag[8*ns].
int launch_adi_fused(hipStream_t s, int ns, double2 *field, double2 *work, const double2 *src,
                     const int4 *box, const AdiFactors &f, int first, double *diag, int tile,
                     int prefetch);
// Banded-inverse ADI (both half steps, 32x32 output tiles, halo M+1):
// reads field `fin`, writes `fout` (the host swaps the buffers), band =
// [ngrid][2M+1] complex rows of A^-1 around the diagonal, a = Im(cstep).
// m: 7, 8 or 12.  Rows [klo, khi] of the band equal row (klo+khi)/2 to
// 2^-60.  tilediag: scratch [ns][adi_band_tiles(ngrid)][8], or null: no
// field sums; launch_tile_sums folds them.
int adi_band_tiles(int ng);
void launch_tile_sums(hipStream_t s, int ns, const double *tilediag, int ntiles, double *diag);
int launch_adi_band(hipStream_t s, int ns, const double2 *fin, double2 *fout, const double2 *src,
                    const int4 *box, const double2 *band, double a, int ng, int first, int m,
                    int klo, int khi, double *tilediag);
// Both half steps in strips of columns, one wavefront each (any grid):
// tilediag [ns][strip_dims(form).count(ng)][8] or null.
void launch_adi_strip(hipStream_t s, int ns, const double2 *fin, double2 *fout, const double2 *src, const int4 *box,
                      const StripCoef &k, int form, int ng, int first, double *tilediag);
void launch_zero(hipStream_t s, double2 *p, long long n);
// A record's slot (device address of pinned memory): beam sums [8 ns] from
// part (per block of the slices' blk_first ranges) or beam, or left alone;
// field sums [8 ns] from tiles (ntiles per slice) or field; with aux the
// auxiliary sums [16 ns] and the space-charge fields esc, ssc [ns each]; with
// mom the spectral moments [5 ns].
struct RecordSources {
    const double *part, *beam, *tiles, *field, *aux, *esc, *ssc, *mom;
    const long long *blk_first;
    int ntiles;
};
void launch_record(hipStream_t s, int ns, const RecordSources &r, double *slot);
// harmonic bunching sums for h0 .. h0 + cnt - 1 (cnt <= 8), out[ns][cnt][2]
void launch_diag_bunch(hipStream_t s, int ns, const long long *off, const double *th, int h0, int cnt,
                       double *out);
void launch_diag_beam(hipStream_t s, int ns, const long long *off, const double *g,
                      const double *th, const double *x, const double *y, double *out);
// px/py sums, coordinate extremes and the on-axis field value per beam
// slice, out[16 ns]
void launch_diag_aux(hipStream_t s, int ns, const long long *off, const double *g, const double *x,
                     const double *y, const double *px, const double *py, const double2 *field, int ng,
                     int first, double *out);
void launch_diag_field(hipStream_t s, int ns, const double2 *field, int ng, double *out);
void launch_sort_index(hipStream_t s, long long n, const double *th, double invslen, int *atar,
                       unsigned long long *moved);

}  // namespace g4mi
