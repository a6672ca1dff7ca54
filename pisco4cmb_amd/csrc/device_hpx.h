/*
 * device_hpx.h -- HEALPix RING geometry and the per-visit beam-frame mapping
 * for gfx950 kernels.
 *
 * Semantics follow the CPU path of PISCO (Convolver, convolver.cpp:74-183),
 * which takes pix2ang / ang2pix / query_disc from healpix_cxx's Healpix_Base
 * (RING scheme, non-inclusive disc), and the rotation of
 * SphericalTransformations::rho_sigma_chi_pix (sphtrigo.cpp:4-55).  The device
 * port of those routines in the reference (cudaHealpix.cu:30-259) differs from
 * the CPU library in three places (its fmod, its polar "sth" rule and the
 * missing imodulo); the CPU behaviour is the one reproduced here.
 *
 * All FP64 arithmetic is written so that, compiled with -ffp-contract=off and
 * evaluated with pisco_libm.h, it yields the same bits as the CPU oracle:
 * pixel indices are therefore bit-exact, not merely close.
 */
#ifndef PISCO_DEVICE_HPX_H
#define PISCO_DEVICE_HPX_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "pisco_libm.h"

#if defined(__clang__)
#pragma clang fp contract(off)
#endif

namespace pisco {

constexpr double kPi = 3.141592653589793238462643383279502884197;
constexpr double kTwoPi = 6.283185307179586476925286766559005768394;
constexpr double kHalfPi = 1.570796326794896619231321691639751442099;
constexpr double kInvHalfPi = 0.6366197723675813430755350534900574;
constexpr double kInvTwoPi = 1.0 / 6.283185307179586476925286766559005768394;
constexpr double kTwoThird = 2.0 / 3.0;

/* Geometry of one RING-ordered HEALPix map (NSIDE <= 8192, int32 pixels,
 * as Healpix_Base<int>). */
struct Hpx {
    int nside;
    int ncap;   /* pixels in the north polar cap */
    int npix;
    double fact1, fact2;
};

__host__ __device__ inline Hpx hpx_make(int nside)
{
    Hpx h;
    h.nside = nside;
    h.ncap = 2 * (nside * nside - nside);
    h.npix = 12 * nside * nside;
    h.fact2 = 4. / h.npix;
    h.fact1 = (nside << 1) * h.fact2;
    return h;
}

/* fmod(x, y) for finite x and y > 0, exact (IEEE fmod is exact, and so is
 * this: the candidate quotient k is off by at most one and x - k*y is
 * representable for the right k, so one fma returns it unrounded). */
__host__ __device__ inline double exact_fmod(double x, double y)
{
    double ax = fabs(x);
    if (ax < y)
        return x;
    double k = trunc(ax / y);
    double r = fma(-k, y, ax);
    if (r < 0.0) {
        k -= 1.0;
        r = fma(-k, y, ax);
    } else if (r >= y) {
        k += 1.0;
        r = fma(-k, y, ax);
    }
    return copysign(r, x);
}

/* healpix_cxx fmodulo: result in [0, v2). */
__host__ __device__ inline double fmodulo(double v1, double v2)
{
    if (v1 >= 0)
        return (v1 < v2) ? v1 : exact_fmod(v1, v2);
    double tmp = exact_fmod(v1, v2) + v2;
    return (tmp == v2) ? 0. : tmp;
}

__host__ __device__ inline int isqrt_i(int v)
{
    return (int)sqrt((double)v + 0.5);
}

/* Ring index (1..4N-1) of a RING pixel. */
__host__ __device__ inline int pix2ring(const Hpx &h, int pix)
{
    if (pix < h.ncap)
        return (1 + isqrt_i(1 + 2 * pix)) >> 1;
    if (pix < h.npix - h.ncap)
        return (pix - h.ncap) / (4 * h.nside) + h.nside;
    int ip = h.npix - pix;
    return 4 * h.nside - ((1 + isqrt_i(2 * ip - 1)) >> 1);
}

/* First pixel, number of pixels and shift flag of ring r
 * (Healpix_Base::get_ring_info_small). */
__host__ __device__ inline void ring_info(const Hpx &h, int r, int &startpix, int &ringpix,
                                 bool &shifted)
{
    if (r < h.nside) {
        shifted = true;
        ringpix = 4 * r;
        startpix = 2 * r * (r - 1);
    } else if (r < 3 * h.nside) {
        shifted = ((r - h.nside) & 1) == 0;
        ringpix = 4 * h.nside;
        startpix = h.ncap + (r - h.nside) * ringpix;
    } else {
        shifted = true;
        int nr = 4 * h.nside - r;
        ringpix = 4 * nr;
        startpix = h.npix - 2 * nr * (nr + 1);
    }
}

/* z and (if |z| > 0.99) sin(theta) of the pixels of ring r, as pix2loc
 * computes them. */
__host__ __device__ inline void ring_z(const Hpx &h, int r, double &z, double &sth,
                              bool &have_sth)
{
    have_sth = false;
    sth = 0.0;
    int n = h.nside;
    if (r < n) {
        double tmp = (r * r) * h.fact2;
        z = 1.0 - tmp;
        if (z > 0.99) {
            sth = sqrt(tmp * (2.0 - tmp));
            have_sth = true;
        }
    } else if (r <= 3 * n) {
        z = (2 * n - r) * h.fact1;
    } else {
        int ir = 4 * n - r;
        double tmp = (ir * ir) * h.fact2;
        z = tmp - 1.0;
        if (z < -0.99) {
            sth = sqrt(tmp * (2.0 - tmp));
            have_sth = true;
        }
    }
}

/* theta of ring r (pix2ang). */
__host__ __device__ inline double ring_theta(const Hpx &h, int r)
{
    double z, sth;
    bool hs;
    ring_z(h, r, z, sth, hs);
    return hs ? pl_atan2(sth, z) : pl_acos(z);
}

/* phi of pixel pix lying in ring r with first pixel startpix (pix2loc). */
__host__ __device__ inline double pixel_phi(const Hpx &h, int r, int pix, int startpix)
{
    int iphi = pix - startpix + 1;
    int n = h.nside;
    if (r < n)
        return (iphi - 0.5) * kHalfPi / r;
    if (r <= 3 * n) {
        double fodd = ((r + n) & 1) ? 1 : 0.5;
        return (iphi - fodd) * kPi * 0.75 * h.fact1;
    }
    return (iphi - 0.5) * kHalfPi / (4 * n - r);
}

__host__ __device__ inline void pix2ang(const Hpx &h, int pix, double &theta, double &phi)
{
    int r = pix2ring(h, pix);
    int sp, nr;
    bool sh;
    ring_info(h, r, sp, nr, sh);
    theta = ring_theta(h, r);
    phi = pixel_phi(h, r, pix, sp);
}

/* Per-ring constants the kernels read once per visit: cos and sin of the
 * ring's declination (dec = pi/2 - theta, exactly as pix2ang + the rotation
 * compute them), the first pixel, and for polar-cap rings the divisor of
 * the phi formula (ring index from the nearest pole) with its reciprocal. */
struct RingRec {
    double cdp, sdp;
    double inv;       /* 1.0 / rdiv (cap rings), 0 in the equatorial belt */
    int startpix;
    int rdiv;         /* r (north cap), 4N - r (south cap), 0 otherwise */
};

__host__ __device__ inline RingRec ring_record(const Hpx &h, int r)
{
    RingRec rr;
    double th = ring_theta(h, r);
    double dec = kPi / 2.0 - th;
    pl_sincos(dec, &rr.sdp, &rr.cdp);
    int nr;
    bool sh;
    ring_info(h, r, rr.startpix, nr, sh);
    rr.rdiv = (r < h.nside) ? r : ((r > 3 * h.nside) ? 4 * h.nside - r : 0);
    rr.inv = rr.rdiv ? 1.0 / rr.rdiv : 0.0;
    return rr;
}

/* pixel_phi from a ring record.  In the caps ((iphi - 0.5) * pi/2) / rdiv is
 * formed as q = x * inv, then q + (x - q*rdiv) * inv with fma: this equals
 * the IEEE quotient for every cap pixel of every NSIDE up to 8192 (checked
 * exhaustively, 134,201,344 cases), and costs no division. */
__host__ __device__ inline double ring_phi(const Hpx &h, const RingRec &rr, int r, int pix)
{
    int iphi = pix - rr.startpix + 1;
    if (rr.rdiv > 0) {
        double x = (iphi - 0.5) * kHalfPi;
        double q = x * rr.inv;
        double e = fma(-q, (double)rr.rdiv, x);
        return fma(e, rr.inv, q);
    }
    double fodd = ((r + h.nside) & 1) ? 1 : 0.5;
    return (iphi - fodd) * kPi * 0.75 * h.fact1;
}

/* Healpix_Base::loc2pix, RING. */
__host__ __device__ inline int loc2pix(const Hpx &h, double z, double phi, double sth,
                              bool have_sth)
{
    double za = fabs(z);
    double tt = fmodulo(phi * kInvHalfPi, 4.0);
    int nside = h.nside;
    if (za <= kTwoThird) {
        int nl4 = 4 * nside;
        double temp1 = nside * (0.5 + tt);
        double temp2 = nside * z * 0.75;
        int jp = (int)(temp1 - temp2);
        int jm = (int)(temp1 + temp2);
        int ir = nside + 1 + jp - jm;
        int kshift = 1 - (ir & 1);
        int t1 = jp + jm - nside + kshift + 1 + nl4 + nl4;
        int ip = (t1 >> 1) % nl4;
        return h.ncap + (ir - 1) * nl4 + ip;
    }
    double tp = tt - (int)tt;
    double tmp = ((za < 0.99) || (!have_sth)) ? nside * sqrt(3 * (1 - za))
                                              : nside * sth / sqrt((1. + za) / 3.);
    int jp = (int)(tp * tmp);
    int jm = (int)((1.0 - tp) * tmp);
    int ir = jp + jm + 1;
    int ip = (int)(tt * ir);
    return (z > 0) ? 2 * ir * (ir - 1) + ip : h.npix - 2 * ir * (ir + 1) + ip;
}

/* Healpix_Base::ang2pix(pointing): sin(theta) is used only within 0.01 rad
 * of a pole. */
__host__ __device__ inline int ang2pix(const Hpx &h, double theta, double phi)
{
    if ((theta < 0.01) || (theta > 3.14159 - 0.01)) {
        double s, c;
        pl_sincos(theta, &s, &c);
        return loc2pix(h, c, phi, s, true);
    }
    return loc2pix(h, pl_cos(theta), phi, 0., false);
}

__host__ __device__ inline int ring_above(const Hpx &h, double z)
{
    double az = fabs(z);
    if (az <= kTwoThird)
        return (int)(h.nside * (2 - 1.5 * z));
    int iring = (int)(h.nside * sqrt(3 * (1 - az)));
    return (z > 0) ? iring : 4 * h.nside - iring - 1;
}

__host__ __device__ inline double ring2z(const Hpx &h, int ring)
{
    if (ring < h.nside)
        return 1 - ring * ring * h.fact2;
    if (ring <= 3 * h.nside)
        return (2 * h.nside - ring) * h.fact1;
    ring = 4 * h.nside - ring;
    return ring * ring * h.fact2 - 1;
}

/* ---- query_disc, decomposed by ring ------------------------------------ */

/* Per-pointing part of the non-inclusive RING query_disc
 * (Healpix_Base::query_disc with fact = 0). Rings are r_first..r_last;
 * rings outside [irmin, irmax] are whole (the polar blocks). */
struct Disc {
    double phi;       /* normalised phi of the centre */
    double z0, xa;
    double cosr;
    int irmin, irmax;
    int r_first, r_last;
};

__host__ __device__ inline void disc_setup(const Hpx &h, double theta, double phi,
                                  double radius, double cosr, Disc &d)
{
    /* pointing::normalize */
    theta = fmodulo(theta, kTwoPi);
    if (theta > kPi) {
        phi += kPi;
        theta = kTwoPi - theta;
    }
    phi = fmodulo(phi, kTwoPi);
    d.phi = phi;
    d.cosr = cosr;
    if (radius >= kPi) {            /* whole sky */
        d.irmin = 4 * h.nside;
        d.irmax = 0;
        d.r_first = 1;
        d.r_last = 4 * h.nside - 1;
        d.z0 = 0;
        d.xa = 0;
        return;
    }
    d.z0 = pl_cos(theta);
    d.xa = 1. / sqrt((1 - d.z0) * (1 + d.z0));
    double rlat1 = theta - radius;
    d.irmin = ring_above(h, pl_cos(rlat1)) + 1;
    bool north = (rlat1 <= 0) && (d.irmin > 1);
    double rlat2 = theta + radius;
    d.irmax = ring_above(h, pl_cos(rlat2));
    bool south = (rlat2 >= kPi) && (d.irmax + 1 < 4 * h.nside);
    d.r_first = north ? 1 : d.irmin;
    d.r_last = south ? 4 * h.nside - 1 : d.irmax;
}

/* Pixel ranges of ring r inside the disc, in ascending order: returns the
 * number of ranges (0..2); range k is [pix0[k], pix0[k] + len[k]). */
__host__ __device__ inline int disc_ring(const Hpx &h, const Disc &d, int r, int pix0[2],
                                int len[2])
{
    int ipix1, nr;
    bool shifted;
    ring_info(h, r, ipix1, nr, shifted);
    if (r < d.irmin || r > d.irmax) {
        pix0[0] = ipix1;
        len[0] = nr;
        return 1;
    }
    double z = ring2z(h, r);
    double x = (d.cosr - z * d.z0) * d.xa;
    double ysq = 1 - z * z - x * x;
    double dphi = (ysq <= 0) ? 0.0 : pl_atan2(sqrt(ysq), x);
    if (!(dphi > 0))
        return 0;
    double shift = shifted ? 0.5 : 0.;
    double a = nr * kInvTwoPi * (d.phi - dphi) - shift;
    double b = nr * kInvTwoPi * (d.phi + dphi) - shift;
    int ip_lo = ((a >= 0) ? (int)a : (int)a - 1) + 1;
    int ip_hi = (b >= 0) ? (int)b : (int)b - 1;
    if (ip_lo > ip_hi)
        return 0;
    if (ip_hi >= nr) {
        ip_lo -= nr;
        ip_hi -= nr;
    }
    if (ip_lo < 0) {   /* (constant indices: a runtime index would put the arrays in scratch) */
        if (ip_hi + 1 > 0) {
            pix0[0] = ipix1;
            len[0] = ip_hi + 1;
            pix0[1] = ipix1 + ip_lo + nr;
            len[1] = -ip_lo;
            return 2;
        }
        pix0[0] = ipix1 + ip_lo + nr;
        len[0] = -ip_lo;
        return 1;
    }
    pix0[0] = ipix1 + ip_lo;
    len[0] = ip_hi - ip_lo + 1;
    return 1;
}

/* The same ring of the disc as one unwrapped index range: returns 0 (empty),
 * 1 (ring positions ip_lo..ip_hi, which may run below 0 or past nr-1 and
 * are taken modulo nr) or 2 (whole ring). */
__host__ __device__ inline int disc_ring_span(const Hpx &h, const Disc &d, int r, int &ip_lo,
                                              int &ip_hi, int &ipix1, int &nr)
{
    bool shifted;
    ring_info(h, r, ipix1, nr, shifted);
    if (r < d.irmin || r > d.irmax)
        return 2;
    double z = ring2z(h, r);
    double x = (d.cosr - z * d.z0) * d.xa;
    double ysq = 1 - z * z - x * x;
    double dphi = (ysq <= 0) ? 0.0 : pl_atan2(sqrt(ysq), x);
    if (!(dphi > 0))
        return 0;
    double shift = shifted ? 0.5 : 0.;
    double a = nr * kInvTwoPi * (d.phi - dphi) - shift;
    double b = nr * kInvTwoPi * (d.phi + dphi) - shift;
    ip_lo = ((a >= 0) ? (int)a : (int)a - 1) + 1;
    ip_hi = (b >= 0) ? (int)b : (int)b - 1;
    if (ip_lo > ip_hi)
        return 0;
    if (ip_hi - ip_lo + 1 >= nr)
        return 2;
    return 1;
}

/* disc_ring_span with the arc's half-width dphi from a float atan2, for
 * callers that need a superset (grow) or a subset (!grow) of the exact span
 * rather than the span itself.  The float dphi is within 4e-6 rad of the
 * FP64 one (float rounding of x and sqrt(ysq), <= 1.2e-7 rad; plf_atan2_core
 * with the hardware reciprocal, ~1e-6), which moves the floor arguments a, b
 * by at most m = nr/(2 pi) 4e-6 pixels.  A floor whose argument lies farther
 * than m from an integer equals the exact one; otherwise it is moved one
 * pixel outward (grow) or inward.  Everything else (the ring range, ysq and
 * the empty-arc test) is the exact path's.  Rings of more than 2^17 pixels
 * (m > 0.08) take the exact path. */
__host__ __device__ inline int disc_ring_span_cover(const Hpx &h, const Disc &d, int r, bool grow,
                                                    int &ip_lo, int &ip_hi, int &ipix1, int &nr)
{
    bool shifted;
    ring_info(h, r, ipix1, nr, shifted);
    if (nr > (1 << 17))
        return disc_ring_span(h, d, r, ip_lo, ip_hi, ipix1, nr);
    if (r < d.irmin || r > d.irmax)
        return 2;
    double z = ring2z(h, r);
    double x = (d.cosr - z * d.z0) * d.xa;
    double ysq = 1 - z * z - x * x;
    if (!(ysq > 0))
        return 0;   /* dphi = 0 on the exact path: empty */
    const float yf = (float)sqrt(ysq), xf = (float)x;
    /* The device's reciprocal estimate is within 1 ulp of the IEEE quotient
     * the host builds (the checks of the cover) use; through plf_atan2_core
     * that moves dphi by under 1e-7 rad, and the 4e-6 rad margin below
     * covers both forms. */
#if defined(__HIP_DEVICE_COMPILE__)
    const float rm = __builtin_amdgcn_rcpf(fmaxf(fabsf(xf), yf));
#else
    const float rm = 1.0f / fmaxf(fabsf(xf), yf);
#endif
    const float dphi = plf_atan2_core(yf, xf, rm);
    const double k = nr * kInvTwoPi, shift = shifted ? 0.5 : 0.;
    const double a = k * (d.phi - (double)dphi) - shift;
    const double b = k * (d.phi + (double)dphi) - shift;
    const double fa = floor(a), fb = floor(b), m = k * 4e-6;
    const double da = a - fa, db = b - fb;
    ip_lo = (int)fa + 1;
    ip_hi = (int)fb;
    if (da < m || da > 1.0 - m)
        ip_lo += grow ? -1 : 1;
    if (db < m || db > 1.0 - m)
        ip_hi += grow ? 1 : -1;
    if (ip_lo > ip_hi)
        return 0;
    if (ip_hi - ip_lo + 1 >= nr)
        return 2;
    return 1;
}

/* Pixel runs of ring r whose centres lie in the annulus dout minus din (two
 * discs about the same centre, din the smaller; inner == false: no inner
 * disc): up to two arcs, each split at the ring's first pixel, so up to 4
 * runs [p0[k], p0[k] + len[k]).  Returns the number of runs.  Both spans come
 * from disc_ring_span about the same centre, so the inner span lies inside
 * the outer one in the same unwrapped positions.  COVER: the spans come from
 * disc_ring_span_cover, the outer one grown and the inner one shrunk, so the
 * runs hold every pixel of the exact annulus (and, near a tie of a floor,
 * a pixel more); the nesting of the spans is kept. */
template <bool COVER = false>
__host__ __device__ inline int annulus_ring(const Hpx &h, const Disc &dout, const Disc &din,
                                            bool inner, int r, int p0[4], int len[4])
{
    int lo_o = 0, hi_o = -1, ip1 = 0, nr = 0;
    int kind_o;
    if constexpr (COVER)
        kind_o = disc_ring_span_cover(h, dout, r, true, lo_o, hi_o, ip1, nr);
    else
        kind_o = disc_ring_span(h, dout, r, lo_o, hi_o, ip1, nr);
    if (kind_o == 0)
        return 0;
    int kind_i = 0, lo_i = 0, hi_i = -1;
    if (inner && r >= din.r_first && r <= din.r_last) {
        int ip1b, nrb;
        if constexpr (COVER)
            kind_i = disc_ring_span_cover(h, din, r, false, lo_i, hi_i, ip1b, nrb);
        else
            kind_i = disc_ring_span(h, din, r, lo_i, hi_i, ip1b, nrb);
    }
    if (kind_i == 2)
        return 0;   /* the whole ring lies inside the inner disc */
    int ia[2], ib[2], ni = 0;
    if (kind_i == 0) {
        ia[0] = kind_o == 2 ? 0 : lo_o;
        ib[0] = kind_o == 2 ? nr - 1 : hi_o;
        ni = 1;
    } else if (kind_o == 2) {   /* the ring minus the inner span */
        ia[0] = hi_i + 1;
        ib[0] = lo_i - 1 + nr;
        ni = 1;
    } else {
        if (lo_i > lo_o) {
            ia[ni] = lo_o;
            ib[ni] = lo_i - 1;
            ni++;
        }
        if (hi_o > hi_i) {
            ia[ni] = hi_i + 1;
            ib[ni] = hi_o;
            ni++;
        }
    }
    int n = 0;
    for (int k = 0; k < ni; k++) {
        const int l = ib[k] - ia[k] + 1;   /* 1 .. nr */
        if (l <= 0)
            continue;
        int st = ia[k] % nr;
        if (st < 0)
            st += nr;
        if (st + l <= nr) {
            p0[n] = ip1 + st;
            len[n] = l;
            n++;
        } else {
            p0[n] = ip1 + st;
            len[n] = nr - st;
            n++;
            p0[n] = ip1;
            len[n] = l - (nr - st);
            n++;
        }
    }
    return n;
}

/* The annulus of sky radii that holds every visit whose beam pixel lies in
 * rows [lo, lo + nrow) of a beam map hb of support radius rho_max (cos_rmax
 * its cosine): a point in a pixel of beam ring R lies between the centres of
 * rings R-1 and R+1, so rows of rings Rf..Rl need rho in
 * [theta(Rf-1), theta(Rl+1)], widened by 1e-9 and clipped to rho_max.
 * inner == false: no inner disc (Rf is ring 1). */
__host__ __device__ inline void band_annulus_radii(const Hpx &hb, double rho_max, double cos_rmax,
                                                   int lo, int nrow, bool &inner, double &r_in,
                                                   double &c_in, double &r_out, double &c_out)
{
    const int rf = pix2ring(hb, lo), rl = pix2ring(hb, lo + nrow - 1);
    inner = rf > 1;
    r_in = inner ? ring_theta(hb, rf - 1) - 1e-9 : 0.0;
    r_out = rl + 1 <= 4 * hb.nside - 1 ? ring_theta(hb, rl + 1) + 1e-9 : rho_max;
    if (r_out >= rho_max) {
        r_out = rho_max;
        c_out = cos_rmax;
    } else {
        c_out = pl_cos(r_out);
    }
    c_in = pl_cos(r_in);
}

/* ---- the beam-frame mapping of one visit -------------------------------- */

/* Per-sample constants of the rotation (sphtrigo.cpp:29-30 evaluated once
 * per sample: they depend only on the beam centre). */
struct Centre {
    double ra, dec, psi;   /* ra, dec of the beam centre; psi = -pa */
    double cdc, sdc;
};

__host__ __device__ inline Centre centre_make(float ra, float dec, float pa)
{
    Centre c;
    c.ra = (double)ra;
    c.dec = (double)dec;
    c.psi = -(double)pa;
    pl_sincos(c.dec, &c.sdc, &c.cdc);
    return c;
}

/* rho, sigma and chi of the sky pixel at (ra_pix, cos/sin dec_pix) seen
 * from the beam centre c: rho_sigma_chi_pix (sphtrigo.cpp:27-54). */
__host__ __device__ inline void visit_rsc(const Centre &c, double ra_pix, double cdp, double sdp,
                                          double &rho, double &sigma, double &chi)
{
    double sd, cd;
    pl_sincos(ra_pix - c.ra, &sd, &cd);
    double crho = c.sdc * sdp + c.cdc * cdp * cd;
    rho = (crho >= 1.0) ? 0.0 : pl_acos(crho);
    double alpha, beta;
    if (rho > 1.0e-6) {
        beta = pl_atan2(sd * c.cdc, c.sdc * cdp - c.cdc * sdp * cd);
        alpha = pl_atan2(sd * cdp, sdp * c.cdc - cdp * c.sdc * cd);
    } else {
        beta = kHalfPi;
        alpha = kHalfPi;
    }
    sigma = kPi - alpha - c.psi;
    if (sigma < 0.0)
        sigma += 2.0 * kPi;
    else if (sigma > 2.0 * kPi)
        sigma -= 2.0 * kPi;
    chi = beta - sigma;
    if (chi < -kPi)
        chi += 2.0 * kPi;
}

/* Beam pixel (ang2pix of (rho, sigma) on the beam map) and chi for the sky
 * pixel at (ra_pix, cos/sin dec_pix): rho_sigma_chi_pix followed by
 * Healpix_Base::ang2pix (convolver.cpp:148-149). */
__host__ __device__ inline int beam_pixel(const Hpx &hb, const Centre &c, double ra_pix,
                                 double cdp, double sdp, double &chi)
{
    double rho, sigma;
    visit_rsc(c, ra_pix, cdp, sdp, rho, sigma, chi);
    return ang2pix(hb, rho, sigma);
}

/* ---- single-precision form of the same mapping, certified ---------------
 *
 * The kernels evaluate the visit geometry in float32 and keep the beam pixel
 * it gives only where no floor of ang2pix can flip; any other visit is
 * re-evaluated by the FP64 form below (beam_pixel_f64).  Either way the pixel
 * is the one the CPU path computes.
 *
 * What depends only on the ring and the sample is evaluated once per ring, in
 * FP64, when the walk's run table is built (run_geo), and rounded to float.
 * With dD = dec_p - dec_c, x = dra/2:
 *   1 - cos rho = (1 - cos dD) + 2 cos dec_c cos dec_p sin^2 x,
 *   ya = 2 sin x cos x cos dec_p,  xa = sin dD + 2 cos dec_p sin dec_c sin^2 x,
 * alpha = atan2(ya, xa) (sphtrigo.cpp:42).  x is linear in the pixel's
 * position in the ring: x = k b + a0 with k the (integer) distance from the
 * ring position nearest to the centre's right ascension, so that its relative
 * error stays at float rounding right up to the centre.
 *
 * In the polar branch of ang2pix (cos rho > 2/3) the floors are jp =
 * (int)(tp*tmp), jm = (int)((1-tp)*tmp) and ip = (int)(tt*(jp+jm+1)), with
 * tt = (2/pi) sigma mod 4, tp = frac(tt), tmp = nside*sqrt(3 (1 - cos rho)).
 * sigma = pi - (alpha + psi): the vector (xa, ya) is turned by psi and its
 * octant gives tt without a range reduction.
 *
 * Errors against FP64, from a float32 emulation over 2e6 visits for each of 21
 * combinations of sky NSIDE 64-2048, beam NSIDE 512-8192, caps 0.3-34 deg and
 * centres anywhere, near and at the poles, with the hardware's reciprocal and
 * square root within 1 ulp:
 *   tt <= 4.9e-7, tmp <= 4e-7 relative; no floor flipped that lay farther
 *   than 3.3e-7 tmp from an integer.
 * Bound used: kFloorMargin tmp + 2e-6 (for the batched kernels, which take
 * alpha before the turn by psi and reduce tt mod 4, kFloorMarginBatch).  The
 * CPU path's own rounding of acos(crho) (|crho error| <= 7e-16) moves tmp by
 * under 1e-7 of that bound for rho > 1e-4; closer visits (and those beyond the
 * polar branch) take the FP64 form, so the rho > 1e-6 rule of sphtrigo.cpp:40
 * never meets the float form. */
struct FastConsts {
    float k3;       /* 3 nside_beam^2 */
};

constexpr float kOmcLo = 5e-9f;           /* 1 - cos(1e-4) */
constexpr float kOmcHi = 0.33332f;        /* polar branch: cos rho > 2/3 */
constexpr float kFloorMargin = 2.5e-6f;
constexpr float kFloorMarginBatch = 4e-6f;
constexpr int kNeedExact = -2;            /* the floors are not certain */

/* Wave-uniform float constants of one sample. */
struct SampleF {
    float cdc, sdc;             /* cos, sin dec of the beam centre */
    float cps, sps;             /* cos, sin psi */
    float c2h, c2l, s2h, s2l;   /* cos, sin 2 psi as float pairs */
    float lim0;                 /* 1/2 - 2e-6, or -1: certify no visit */
};

/* Whether the float form's geometry holds for a beam centre: a declination
 * within [-pi/2, pi/2] (beyond it query_disc's centre is the reflected point)
 * and a right ascension small enough that its FP64 reduction is exact to
 * 1e-11.  Otherwise (NaN included) every visit takes the FP64 form. */
__host__ __device__ inline bool centre_regular(double ra, double dec)
{
    return fabs(ra) < 1e4 && fabs(dec) <= kHalfPi;
}

__host__ __device__ inline SampleF sample_f32(const Centre &c, double cpsi, double spsi,
                                              double c2psi, double s2psi)
{
    SampleF f;
    f.cdc = (float)c.cdc;
    f.sdc = (float)c.sdc;
    f.cps = (float)cpsi;
    f.sps = (float)spsi;
    f.c2h = (float)c2psi;
    f.c2l = (float)(c2psi - (double)f.c2h);
    f.s2h = (float)s2psi;
    f.s2l = (float)(s2psi - (double)f.s2h);
    f.lim0 = centre_regular(c.ra, c.dec) ? 0.5f - 2e-6f : -1.0f;
    return f;
}

/* 1/n to ~1e-15 relative: hardware reciprocal estimate + one Newton step
 * (used only where the value feeds float outputs, never an index). */
__device__ inline double recip_fast(double n)
{
    double r = __builtin_amdgcn_rcp(n);
    return fma(r, fma(-n, r, 1.0), r);
}

/* Float geometry of a run of consecutive pixels of one ring, positions j0 ..
 * j0+len-1, around one sample: x = dra/2 of position j is (j - kc) b + a0. */
struct RunGeo {
    double a0d, bd, kapd;   /* a0, b, kap before the rounding to float */
    float a0, b;
    int kc;
    float sD, omD;    /* sin dD, 1 - cos dD */
    float cdp2;       /* 2 cos dec_p */
    float kap;        /* sin((dec_p + dec_c)/2) / cos(dD/2) */
};

__device__ inline RunGeo run_geo(const Hpx &h, const RingRec &rr, int r, const Centre &c, int j0,
                                 int len)
{
    RunGeo g;
    /* pixel spacing 2 pi / nr and the ring's half-pixel shift */
    const bool cap = rr.rdiv > 0;
    const double tpn = cap ? kHalfPi * rr.inv : (kPi * 0.75) * h.fact1;
    const double nr = cap ? 4.0 * rr.rdiv : 4.0 * h.nside;
    const double shift = (cap || ((r - h.nside) & 1) == 0) ? 0.5 : 0.0;
    /* the centre's right ascension on the branch nearest the run's middle */
    const double mid = ((double)j0 + 0.5 * (double)(len - 1) + shift) * tpn;
    const double ra = c.ra + kTwoPi * rint((mid - c.ra) * kInvTwoPi);
    const double kc = rint(ra * (nr * kInvTwoPi) - shift);
    g.a0d = 0.5 * ((kc + shift) * tpn - ra);
    g.bd = 0.5 * tpn;
    g.a0 = (float)g.a0d;
    g.b = (float)g.bd;
    g.kc = (int)kc;
    const double sD = fma(rr.sdp, c.cdc, -(rr.cdp * c.sdc));
    const double rc = recip_fast(1.0 + fma(rr.cdp, c.cdc, rr.sdp * c.sdc));
    g.sD = (float)sD;
    g.omD = (float)(sD * sD * rc);
    g.cdp2 = (float)(2.0 * rr.cdp);
    g.kapd = (c.sdc + rr.sdp) * rc;
    g.kap = (float)g.kapd;
    return g;
}

/* Position angle free part of a visit. */
struct VisitGeo {
    float s2, sc;     /* sin^2 x, sin x cos x */
    float omc;        /* 1 - cos rho */
    float xa, ya;
};

__device__ inline VisitGeo visit_geo(float x, float sD, float omD, float cdp2, float cdc,
                                     float sdc)
{
    VisitGeo v;
    float sh, ch;
    plf_sincos(x, &sh, &ch);
    v.s2 = sh * sh;
    v.sc = sh * ch;
    v.omc = fmaf(v.s2, cdp2 * cdc, omD);
    v.xa = fmaf(v.s2, cdp2 * sdc, sD);
    v.ya = v.sc * cdp2;
    return v;
}

/* e^{2i(alpha + beta)} = (1 - d4, -s4), from Napier's analogy: alpha + beta =
 * pi - 2 eta (mod 2 pi) with tan eta = kap tan x, so no ill-conditioned
 * direction at the centre enters.  Error of the result after the turn by 2 psi
 * (visit_chi): 2.3e-6 |eta| + 4e-8 (float32 emulation). */
__device__ inline void visit_phase(const VisitGeo &v, float kap, float &d4, float &s4)
{
    const float w = (kap * kap) * v.s2, p = 1.0f - v.s2;
    const float inv = __builtin_amdgcn_rcpf(p + w);
    const float c = (p - w) * inv, s = (kap * v.sc) * inv;   /* cos 2 eta, sin(2 eta) / 2 */
    d4 = 8.0f * s * s;
    s4 = 4.0f * (s * c);
}

/* cos, sin 2 chi, chi = beta + alpha + psi - pi (sphtrigo.cpp:41-53), as the turn
 * by 2 psi and a correction that is small with eta: only the last addition rounds
 * at the size of the result.  (The low parts' products with d4 are below 3e-8
 * d4.) */
__device__ inline void visit_chi(const SampleF &f, float d4, float s4, float &c2, float &s2)
{
    c2 = f.c2h + fmaf(s4, f.s2h, fmaf(-d4, f.c2h, fmaf(s4, f.s2l, f.c2l)));
    s2 = f.s2h + fmaf(-s4, f.c2h, fmaf(-d4, f.s2h, fmaf(-s4, f.c2l, f.s2l)));
}

/* atan(min(ax, ay) / max(ax, ay)) 2/pi, in [0, 1/2]; fit error 5.6e-8. */
__device__ inline float quarter_turns(float ax, float ay)
{
    const float t = fminf(ax, ay) * __builtin_amdgcn_rcpf(fmaxf(ax, ay));
    const float z = t * t;
    float p = -0x1.8ee3fcp-9f;
    p = fmaf(p, z, 0x1.00234cp-6f);
    p = fmaf(p, z, -0x1.3869b6p-5f);
    p = fmaf(p, z, 0x1.03442ep-4f);
    p = fmaf(p, z, -0x1.6dd48ap-4f);
    p = fmaf(p, z, 0x1.0462e0p-3f);
    p = fmaf(p, z, -0x1.b2953cp-3f);
    p = fmaf(p, z, 0x1.45f304p-1f);
    return t * p;
}

/* A certified pixel of the polar cap: its ring, quadrant, and place in the
 * quadrant (whole numbers). */
struct CapPlace {
    float ring, quad, pos;
};

/* Beam pixel from tt in [0, 4] and tmp; kNeedExact unless every floor's
 * argument is farther than 1/2 - lim from an integer. */
__device__ inline int cap_floors(float tt, float tmp, float omc, float lim, CapPlace &place)
{
    const float tp = __builtin_amdgcn_fractf(tt);
    const float u1 = tp * tmp, u2 = tmp - u1;
    const float d1 = __builtin_amdgcn_fractf(u1), d2 = __builtin_amdgcn_fractf(u2);
    const float irf = ((u1 - d1) + (u2 - d2)) + 1.0f;
    const float vv = tt * irf;
    const float dv = __builtin_amdgcn_fractf(vv);
    place.ring = irf;
    place.quad = tt - tp;
    place.pos = fmaf(-place.quad, irf, vv - dv);
    const int ir = (int)irf, ip = (int)(vv - dv);
    const float e = fmaxf(fmaxf(fabsf(d1 - 0.5f), fabsf(d2 - 0.5f)), fabsf(dv - 0.5f));
    const bool ok = e < lim && omc > kOmcLo && omc < kOmcHi;
    return ok ? 2 * (int)__umul24((unsigned)ir, (unsigned)(ir - 1)) + ip : kNeedExact;
}

/* Beam pixel of a visit for the sample's position angle, or kNeedExact. */
__device__ inline int visit_pixel(const FastConsts &fc, const SampleF &f, const VisitGeo &v,
                                  CapPlace &place)
{
    const float xr = fmaf(v.xa, f.cps, -(v.ya * f.sps)), yr = fmaf(v.xa, f.sps, v.ya * f.cps);
    const float ax = fabsf(xr), ay = fabsf(yr);
    const float a = quarter_turns(ax, ay);
    /* sigma's vector is (-xr, yr): tt = 2 - copysign(1 + copysign(m, -xr), yr),
     * m the quarter turns from the y axis */
    const float m = ay > ax ? a : 1.0f - a;
    const float tt = 2.0f - copysignf(1.0f - copysignf(m, xr), yr);
    const float tmp = __builtin_amdgcn_sqrtf(fc.k3 * v.omc);
    return cap_floors(tt, tmp, v.omc, fmaf(tmp, -kFloorMargin, f.lim0), place);
}

/* The same for the batched kernels, whose pairs share a visit's alpha, in quarter
 * turns in [-2, 2], and turn it by their own psi: t0 = (pi - psi) 2/pi mod 4. */
__device__ inline float visit_alpha(const VisitGeo &v)
{
    const float ax = fabsf(v.xa), ay = fabsf(v.ya);
    const float a = quarter_turns(ax, ay);
    const float m = ay > ax ? a : 1.0f - a;   /* from the y axis */
    return copysignf(1.0f - copysignf(m, v.xa), v.ya);
}

__device__ inline float pair_t0(double psi)
{
    return (float)fmodulo((kPi - psi) * kInvHalfPi, 4.0);
}

__device__ inline int pair_pixel(float alpha, float x3y, float omc, float t0, float nside,
                                 float lim0, CapPlace &place)
{
    const float tt = 4.0f * __builtin_amdgcn_fractf(0.25f * (t0 - alpha));
    const float tmp = nside * x3y;
    return cap_floors(tt, tmp, omc, fmaf(tmp, -kFloorMarginBatch, lim0), place);
}

/* |eta| above which cos, sin 2 chi take the FP64 form (visit_phase64): the
 * forward and the sky adjoint with lane groups of discs below 1,000 pixels keep
 * them within 2.2e-7 of FP64, and the other adjoints, whose gradients are float
 * sums of many visits, within 1e-6.  Sky gradient over small discs, relative RMS of Q and U
 * against FP64 for the bounds 0.078 and 0.38, and an FP64 geometry with every
 * product rounded to float: 1.5 degrees at NSIDE 256, declination 29 degrees 5.2e-8,
 * 5.2e-8, 6.0e-8, 77 degrees 5.6e-8, 5.8e-8, 6.3e-8, 86 degrees 5.6e-8, 7.3e-8,
 * 6.5e-8. */
constexpr float kEtaForward = 0.078f;
constexpr float kEtaAdjoint = 0.38f;

/* visit_phase in FP64, rounded to float at the end (with visit_chi: within 1.2e-7),
 * from h = dra/4 and k2 = 2 kap of the visit: with t = tan h, tan eta = k2 t /
 * (1 - t^2).  t by a polynomial in h^2 up to h = pi/4 (Chebyshev interpolation,
 * relative error 1.2e-9). */
__device__ inline void visit_phase64(double h, double k2, float &d4, float &s4)
{
    const double z = h * h;
    double p = 0x1.21afd124822a5p-8;
    p = fma(p, z, -0x1.6e08157222680p-17);
    p = fma(p, z, 0x1.6612cdee32a5fp-7);
    p = fma(p, z, 0x1.5bfd2464feb1cp-6);
    p = fma(p, z, 0x1.baf2170033bf3p-5);
    p = fma(p, z, 0x1.110cd8e996eb4p-3);
    p = fma(p, z, 0x1.5555655f8048ap-2);
    p = fma(p, z, 0x1.fffffff6139bfp-1);
    const double t = h * p, num = k2 * t, den = fma(-t, t, 1.0);
    const double q = num * num, r = recip_fast(fma(den, den, q));
    const double ce = fma(den, den, -q) * r, se = 2.0 * (den * num) * r;
    d4 = (float)(2.0 * (se * se));
    s4 = (float)(2.0 * (ce * se));
}

/* The same from the visit's ring. */
__device__ inline void visit_phase64(const Centre &c, double ra_pix, double cdp, double sdp,
                                     float &d4, float &s4)
{
    double dra = ra_pix - c.ra;
    dra = fma(-kTwoPi, rint(dra * kInvTwoPi), dra);
    const double kap = (c.sdc + sdp) * recip_fast(1.0 + fma(cdp, c.cdc, sdp * c.sdc));
    visit_phase64(0.25 * dra, 2.0 * kap, d4, s4);
}

struct ExactVisit {
    int bp;
    float c2, s2;
};

/* The exact FP64 mapping (beam_pixel) of one visit, with (float)cos/sin 2chi
 * as the CPU path forms them.  Out of line, scalar arguments only (a
 * reference argument would force the caller's parameters into scratch). */
__device__ __noinline__ ExactVisit beam_visit_exact(int nside_beam, double ra_c, double psi,
                                                    double cdc, double sdc, double ra_pix,
                                                    double cdp, double sdp)
{
    Centre c;
    c.ra = ra_c;
    c.dec = 0.0;   /* not read by beam_pixel */
    c.psi = psi;
    c.cdc = cdc;
    c.sdc = sdc;
    double chi, s, co;
    ExactVisit e;
    e.bp = beam_pixel(hpx_make(nside_beam), c, ra_pix, cdp, sdp, chi);
    pl_sincos(2.0 * chi, &s, &co);
    e.c2 = (float)co;
    e.s2 = (float)s;
    return e;
}

/* ---- certified double-precision form of the same mapping -----------------
 *
 * Maps the visits that the single-precision form declines, and the visits of
 * the banded beam adjoint.  Its margins are ~1e-12 relative, so it practically
 * never needs the exact path, and it evaluates that path in place. */

/* The CPU path obtains the beam pixel from rho = acos(crho) through
 * z = cos(rho) (and sin(rho) within 0.01 rad of the pole); in the polar branch
 * of ang2pix the two floors that depend on rho are jp = (int)(tp*tmp) and
 * jm = (int)((1-tp)*tmp) with tmp = nside*sqrt(3*(1-z)) (or, within 0.01 rad,
 * nside*sin(rho)/sqrt((1+z)/3)).  Both forms equal nside*sqrt(3*(1-crho))
 * up to the rounding of acos/cos/sin, which is bounded by
 *     |tmp_exact - tmp_fast| <= nside*4.4e-16/sqrt(1-crho) + 2e-15*tmp
 * (pisco_libm's acos, cos and sin are within 2 ulp).  beam_pixel_f64
 * evaluates the cheap form and accepts its floors only if both fractional
 * parts are farther than 100 times that bound (plus 1e-10) from an integer;
 * otherwise it evaluates the exact path.  Either way the returned pixel is
 * the one beam_pixel returns.  sigma (hence tt, tp and ip) is computed with
 * the same operations as the exact path.
 *
 * chi is needed only as float cos(2 chi), sin(2 chi).  With
 * beta = atan2(yb, xb), alpha = atan2(ya, xa) and chi = beta + alpha + psi - pi
 * (mod 2 pi; sphtrigo.cpp:41-53), e^{2 i chi} = w^2/|w|^2 * e^{2 i psi} with
 * w = (xb + i yb)(xa + i ya): no transcendental is needed (FP64 algebra,
 * within ~1e-15 of cos/sin(2 chi) before rounding to float). */
struct FastConsts64 {
    double crho_big;    /* crho <  crho_big  => rho > 1e-6 for sure */
    double crho_small;  /* crho >= crho_small => rho <= 1e-6 for sure */
    double marg_k;      /* 100 * 4.4e-16 * nside * sqrt(3) */
};

/* Rare paths of beam_pixel_f64, kept out of line so that they do not
 * occupy registers in the hot loop. */
/* (NSIDE by value: a reference argument of an out-of-line call would force
 * the caller's parameter block into addressable scratch memory.) */
__device__ __noinline__ int beam_pixel_exact_rho(int nside_beam, double crho, double sigma)
{
    double rho = (crho >= 1.0) ? 0.0 : pl_acos(crho);
    return ang2pix(hpx_make(nside_beam), rho, sigma);
}

__device__ __noinline__ bool rho_above_1e6(double crho)
{
    return (crho >= 1.0) ? false : (pl_acos(crho) > 1.0e-6);
}

__device__ __noinline__ double2 e2i_angles(double yb, double xb, double alpha)
{
    double beta = pl_atan2(yb, xb);
    double s2c, c2c;
    pl_sincos(2.0 * (beta + alpha), &s2c, &c2c);
    return make_double2(c2c, s2c);
}

/* pl_sincos for a wavefront: when no lane needs argument reduction the
 * reduction step is skipped for the whole wave.  For |x| < 0.78 the
 * reduction computes n = rint(2x/pi) = 0 and returns y = x, ylo = +0 exactly,
 * so the results are the same bits either way. */
__device__ inline void wave_sincos(double x, double *s, double *c)
{
    if (__any(!(fabs(x) < 0.78))) {
        pl_sincos(x, s, c);
        return;
    }
    *s = pl_sin_kernel(x, 0.0);
    *c = pl_cos_kernel(x, 0.0);
}

/* sigma -> the polar-branch floors of loc2pix (beam_pixel_f64's tail); the
 * exact path's pixel where a floor is uncertain. */
__device__ inline int beam_floors(const Hpx &hb, double crho, double sigma, double tmp, double y,
                                  double marg_k)
{
    double tt = fmodulo(sigma * kInvHalfPi, 4.0);
    double tp = tt - (int)tt;
    double u1 = tp * tmp;
    double u2 = (1.0 - tp) * tmp;
    int jp = (int)u1, jm = (int)u2;
    double d1 = u1 - jp, d2 = u2 - jm;
    /* margin: nside * 4.4e-14 / sqrt(omc) + 3e-13 tmp + 1e-10, with
     * 1/sqrt(omc) = sqrt(3) * y */
    double md = fma(marg_k, y, fma(3e-13, tmp, 1e-10));
    bool ok = (crho > kTwoThird + 1e-12) && (d1 > md) && (d1 < 1.0 - md) && (d2 > md) &&
              (d2 < 1.0 - md);
    int ir = jp + jm + 1;
    int ip = (int)(tt * ir);
    if (ok)
        return 2 * ir * (ir - 1) + ip;
    return beam_pixel_exact_rho(hb.nside, crho, sigma);
}

__device__ inline double sigma_of(double alpha, double psi)
{
    double sigma = kPi - alpha - psi;
    if (sigma < 0.0)
        sigma += 2.0 * kPi;
    else if (sigma > 2.0 * kPi)
        sigma -= 2.0 * kPi;
    return sigma;
}

__device__ inline int beam_pixel_f64(const Hpx &hb, const FastConsts64 &fc, const Centre &c,
                                      double c2psi, double s2psi, double ra_pix,
                                      double cdp, double sdp, float &c2, float &s2)
{
    double sd, cd;
    wave_sincos(ra_pix - c.ra, &sd, &cd);
    double crho = c.sdc * sdp + c.cdc * cdp * cd;
    bool big;   /* rho > 1e-6 (sphtrigo.cpp:40) */
    if (crho < fc.crho_big)
        big = true;
    else if (crho >= fc.crho_small)
        big = false;
    else
        big = rho_above_1e6(crho);
    double yb = sd * c.cdc, xb = c.sdc * cdp - c.cdc * sdp * cd;
    double ya = sd * cdp, xa = sdp * c.cdc - cdp * c.sdc * cd;

    /* cos/sin 2chi */
    double er = 1.0, ei = 0.0;   /* e^{2i(alpha+beta)}; alpha = beta = pi/2 -> 1 */
    if (big) {
        double wr = xb * xa - yb * ya, wi = xb * ya + yb * xa;
        double n = wr * wr + wi * wi;
        if (n > 1e-280) {
            double inv = recip_fast(n);
            er = (wr * wr - wi * wi) * inv;
            ei = 2.0 * wr * wi * inv;
        } else {   /* degenerate geometry: take the angles themselves */
            double2 e = e2i_angles(yb, xb, pl_atan2(ya, xa));
            er = e.x;
            ei = e.y;
        }
    }
    c2 = (float)(er * c2psi - ei * s2psi);
    s2 = (float)(er * s2psi + ei * c2psi);

    /* beam pixel: polar branch of loc2pix with the certified floors.
     * sqrt(3 omc) from the hardware rsqrt estimate and two Newton steps:
     * within 1e-15 relative, an error the margin includes. */
    double omc = 1.0 - crho;
    omc = omc > 0.0 ? omc : 0.0;
    double x3 = 3.0 * omc;
    double y = __builtin_amdgcn_rsq(x3);
    y = y * fma(-0.5 * x3, y * y, 1.5);
    y = y * fma(-0.5 * x3, y * y, 1.5);
    double tmp = (x3 > 0.0) ? hb.nside * (x3 * y) : 0.0;
    /* alpha from the FP64 atan2, the CPU path's own (sphtrigo.cpp:42) */
    double alpha = big ? pl_atan2(ya, xa) : kHalfPi;
    return beam_floors(hb, crho, sigma_of(alpha, c.psi), tmp, y, fc.marg_k);
}

/* get_interpol (Healpix_Base::get_interpol; the device port in the reference
 * is cudaHealpix.cu:198-259). */
__host__ __device__ inline void ring_info2(const Hpx &h, int ring, int &startpix,
                                  int &ringpix, double &theta, bool &shifted)
{
    int northring = (ring > 2 * h.nside) ? 4 * h.nside - ring : ring;
    if (northring < h.nside) {
        double tmp = northring * northring * h.fact2;
        double costheta = 1 - tmp;
        double sintheta = sqrt(tmp * (2 - tmp));
        theta = pl_atan2(sintheta, costheta);
        ringpix = 4 * northring;
        shifted = true;
        startpix = 2 * northring * (northring - 1);
    } else {
        theta = pl_acos((2 * h.nside - northring) * h.fact1);
        ringpix = 4 * h.nside;
        shifted = ((northring - h.nside) & 1) == 0;
        startpix = h.ncap + (northring - h.nside) * ringpix;
    }
    if (northring != ring) {
        theta = kPi - theta;
        startpix = h.npix - startpix - ringpix;
    }
}

__host__ __device__ inline void get_interpol(const Hpx &h, double theta, double phi,
                                    int pix[4], double wgt[4])
{
    double z = pl_cos(theta);
    int ir1 = ring_above(h, z);
    int ir2 = ir1 + 1;
    double theta1 = 0, theta2 = 0, w1, tmp, dphi;
    int sp, nr, i1, i2;
    bool shift;
    if (ir1 > 0) {
        ring_info2(h, ir1, sp, nr, theta1, shift);
        dphi = kTwoPi / nr;
        tmp = (phi / dphi - .5 * shift);
        i1 = (tmp < 0) ? (int)tmp - 1 : (int)tmp;
        w1 = (phi - (i1 + .5 * shift) * dphi) / dphi;
        i2 = i1 + 1;
        if (i1 < 0) i1 += nr;
        if (i2 >= nr) i2 -= nr;
        pix[0] = sp + i1;
        pix[1] = sp + i2;
        wgt[0] = 1 - w1;
        wgt[1] = w1;
    }
    if (ir2 < (4 * h.nside)) {
        ring_info2(h, ir2, sp, nr, theta2, shift);
        dphi = kTwoPi / nr;
        tmp = (phi / dphi - .5 * shift);
        i1 = (tmp < 0) ? (int)tmp - 1 : (int)tmp;
        w1 = (phi - (i1 + .5 * shift) * dphi) / dphi;
        i2 = i1 + 1;
        if (i1 < 0) i1 += nr;
        if (i2 >= nr) i2 -= nr;
        pix[2] = sp + i1;
        pix[3] = sp + i2;
        wgt[2] = 1 - w1;
        wgt[3] = w1;
    }
    if (ir1 == 0) {
        double wtheta = theta / theta2;
        wgt[2] *= wtheta;
        wgt[3] *= wtheta;
        double fac = (1 - wtheta) * 0.25;
        wgt[0] = fac;
        wgt[1] = fac;
        wgt[2] += fac;
        wgt[3] += fac;
        pix[0] = (pix[2] + 2) & 3;
        pix[1] = (pix[3] + 2) & 3;
    } else if (ir2 == 4 * h.nside) {
        double wtheta = (theta - theta1) / (kPi - theta1);
        wgt[0] *= (1 - wtheta);
        wgt[1] *= (1 - wtheta);
        double fac = wtheta * 0.25;
        wgt[0] += fac;
        wgt[1] += fac;
        wgt[2] = fac;
        wgt[3] = fac;
        pix[2] = ((pix[0] + 2) & 3) + h.npix - 4;
        pix[3] = ((pix[1] + 2) & 3) + h.npix - 4;
    } else {
        double wtheta = (theta - theta1) / (theta2 - theta1);
        wgt[0] *= (1 - wtheta);
        wgt[1] *= (1 - wtheta);
        wgt[2] *= wtheta;
        wgt[3] *= wtheta;
    }
}

} /* namespace pisco */

#endif /* PISCO_DEVICE_HPX_H */
