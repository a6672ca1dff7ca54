/*
 * kernels.hip -- gfx950 kernels of the pixel-space beam convolution.
 *
 * Work mapping (CDNA4: 64-lane wavefronts, 4 waves per 256-thread block):
 *   a lane group (8, 16, 32 or 64 lanes) per pointing sample.  It first runs the
 *   ring part of query_disc with one ring per lane, turns the 0-2 pixel runs of
 *   each ring into a table in LDS with a prefix sum over its lanes, and then
 *   walks the flattened visit list lane-strided, so that consecutive lanes read
 *   consecutive sky pixels of a ring (coalesced) while the beam reads are
 *   gathers.  Each visit maps its pixel into the beam frame in certified single
 *   precision; a visit whose beam pixel that cannot certify is mapped in double
 *   precision or exactly as the CPU path does.  Sums are reduced across the
 *   lanes with shuffles, so the forward is deterministic and needs no global
 *   atomics.
 *
 * Blocks are remapped so that each of the 8 XCDs (each with its own L2) works
 * on one contiguous stretch of the scan: consecutive samples share most of
 * their disc pixels, and this keeps those reuses inside one L2.
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <cstring>

#include "device_hpx.h"
#include "kernels.hpp"
#include "visit_marks.h"
#include "work_items.h"

namespace pisco {

constexpr int kWaveSize = 64;
constexpr int kWavesPerBlock = 4;
constexpr int kBlock = kWaveSize * kWavesPerBlock;
constexpr int kMaxRuns = 2 * kWaveSize;   /* per ring pass: <= 2 runs per ring */

__device__ inline void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

/* A wave-uniform double moved to scalar registers (one wave = one sample,
 * so the sample's constants need no vector registers). */
__device__ inline double uni(double x)
{
    long long v = __double_as_longlong(x);
    int lo = __builtin_amdgcn_readfirstlane((int)(v & 0xffffffffLL));
    int hi = __builtin_amdgcn_readfirstlane((int)(v >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

__device__ inline int wave_incl_scan(int x, int lane)
{
#pragma unroll
    for (int d = 1; d < kWaveSize; d <<= 1) {
        int y = __shfl_up(x, d, kWaveSize);
        if (lane >= d)
            x += y;
    }
    return x;
}

__device__ inline double wave_sum(double x)
{
#pragma unroll
    for (int m = kWaveSize / 2; m > 0; m >>= 1)
        x += __shfl_xor(x, m, kWaveSize);
    return x;
}

/* Logical block index such that XCD x (hardware dispatches blocks round-robin
 * over the 8 XCDs) receives a contiguous range of logical blocks. */
__device__ inline long xcd_remap(long b, long nblk)
{
    const long nx = 8;
    long q = nblk / nx, r = nblk % nx;
    long x = b % nx, k = b / nx;
    return (x < r) ? x * (q + 1) + k : r * (q + 1) + (x - r) * q + k;
}

/* Run table of one wave for one pass over (up to) 64 rings (beam
 * interpolation). */
struct RunTable {
    int pref[kMaxRuns + 1];  /* visit offset of each run; pref[nrun] = total */
    int pix0[kMaxRuns];
    int ring[kMaxRuns];
};

/* Builds the run table for rings r0 .. r0+63 (clipped to the disc); returns
 * the number of visits of the pass. */
__device__ inline int build_runs(const Hpx &hs, const Disc &d, int r0, int lane,
                                 RunTable &t)
{
    int r = r0 + lane;
    int p0[2] = {0, 0}, ln[2] = {0, 0};
    int ns = 0;
    if (r <= d.r_last)
        ns = disc_ring(hs, d, r, p0, ln);
    int cnt = ns;
    int tot = (ns > 0 ? ln[0] : 0) + (ns > 1 ? ln[1] : 0);
    int cnt_in = wave_incl_scan(cnt, lane);
    int tot_in = wave_incl_scan(tot, lane);
    int cbase = cnt_in - cnt;
    int off = tot_in - tot;
#pragma unroll
    for (int k = 0; k < 2; k++) {   /* constant indices keep p0, ln in registers */
        if (k < ns) {
            t.pix0[cbase + k] = p0[k];
            t.ring[cbase + k] = r;
            t.pref[cbase + k] = off;
            off += ln[k];
        }
    }
    int nrun = __shfl(cnt_in, kWaveSize - 1, kWaveSize);
    int total = __shfl(tot_in, kWaveSize - 1, kWaveSize);
    if (lane == 0)
        t.pref[nrun] = total;
    wave_sync();
    return total;
}

/* ---- the walk over a disc's visits ----------------------------------------
 *
 * A lane group of SUB lanes (64: the whole wave) walks the visits of its
 * sample's disc SUB at a time, in passes of at most RPP runs of consecutive
 * pixels (0 to 2 per ring).  A pass's table holds, per run, the float geometry
 * of the ring around the sample (run_geo), so that a visit reads two LDS
 * records and does no FP64.  `bits` marks the visits that start a run: a lane
 * finds its run by counting the marks below it (its wave's visits are
 * consecutive), where a search through the run offsets would be a chain of
 * dependent LDS reads.  Per 64 visits the forward issues about 130 vector
 * instructions, where recomputing the ring's geometry per visit in mixed
 * precision took 279: 1e6 samples of 135 pixels 1.28 and 0.80 ms.  Bound by
 * vector issue and by the gather's lines, 2.15 cycles each per CU.  The marks
 * cover a segment of VCAP visits from seg0 on:
 * bit v - 1 - seg0 marks a run that starts at visit v > seg0. */
/* A wide run's constants for visit_phase64 (h of position j is (j - kc) b + a0).
 * With them a wide visit takes about 25 FP64 instructions more than another; from the
 * ring's record, with a sine and a cosine of full precision, it took a hundred and a
 * load from memory in the loop.  2e4 samples of 5 degrees at declination 69 degrees
 * 1.22 -> 0.82 ms (no wide runs 0.71; an FP64 geometry throughout 0.94).  The tables
 * of 8 lanes and of the sky adjoint have no room for them beside what they hold. */
struct WideRec {
    double a0, b, k2;
};
template <int N>
struct WideRecs {   /* of the wide runs, where the LDS has room for them */
    WideRec wide[N];
};
template <>
struct WideRecs<0> {
};

template <int SUB_, int RPP_, int VCAP_, bool WIDE_ = false>
struct VisitTable : WideRecs<WIDE_ ? RPP_ : 0> {
    static constexpr int SUB = SUB_, RPP = RPP_, VCAP = VCAP_;
    static constexpr bool WIDE = WIDE_;
    float4 rec[RPP][2];      /* a0, b, mid, pixoff (int bits); sD, omD, cdp2, kap */
    unsigned bits[VCAP / 32];
    int pref[RPP + 1];       /* visit offset of each run; pref[nrun] = total */
    int ring[RPP];
};

/* What a pass covers: its visits and runs, the first ring of the next pass,
 * and whether some run is wide: the |eta| of its visits may exceed the caller's
 * bound.  Wide runs hold ~ring: which form a visit takes does not depend on the
 * pass it is in. */
struct Pass {
    int total, nrun, next;
    bool wide;
};

template <int SUB>
__device__ inline int seg_incl_scan(int x, int sl)
{
#pragma unroll
    for (int d = 1; d < SUB; d <<= 1) {
        int y = __shfl_up(x, d, SUB);
        if (sl >= d)
            x += y;
    }
    return x;
}

/* The runs of ring r, as ring positions: query_disc's ranges, a whole ring
 * split where dra passes pi (each run then lies on one branch of dra). */
__device__ inline int disc_runs(const Hpx &h, const Disc &d, const Centre &c, int r, int startpix,
                                int j0[2], int len[2])
{
    int ns = disc_ring(h, d, r, j0, len);
    j0[0] -= startpix;
    j0[1] -= startpix;
    const int nr = 4 * (r < h.nside ? r : (r > 3 * h.nside ? 4 * h.nside - r : h.nside));
    if (ns == 1 && len[0] == nr) {
        const bool shifted = r < h.nside || r > 3 * h.nside || ((r - h.nside) & 1) == 0;
        double t = (c.ra + kPi) * kInvTwoPi;
        t -= floor(t);
        int ja = (int)ceil(t * nr - (shifted ? 0.5 : 0.0));
        ja = ja < 0 ? 0 : ja;
        if (ja > 0 && ja < nr) {
            len[0] = ja;
            j0[1] = ja;
            len[1] = nr - ja;
            ns = 2;
        }
    }
    return ns;
}

/* Builds the table of the pass that starts at ring r0 (up to d.r_last) for
 * the lane group; every lane of the group returns the same Pass. */
template <typename T>
__device__ inline Pass build_pass(const Hpx &hs, const RingRec *rings, const Disc &d,
                                  const Centre &c, int r0, int r_last, int sl, float eta_max, T &t)
{
    constexpr int SUB = T::SUB, RPP = T::RPP;
    constexpr int kWords = T::VCAP / 32;
    const int lane = (int)__lane_id();
    for (int w = sl; w < kWords; w += SUB)
        t.bits[w] = 0u;
    wave_sync();
    int carry = 0;            /* visits << 8 | runs of the rounds before */
    Pass ps;
    ps.next = r0;
    bool wide = false, more = true;
#pragma unroll 1
    for (int q = 0; q < (RPP + SUB - 1) / SUB; q++) {
        const int r = r0 + q * SUB + sl;
        const bool in = more && r <= r_last;
        if (q > 0 && !__any(in))
            break;   /* no lane group has more rings */
        RingRec rr;
        int j0[2] = {0, 0}, ln[2] = {0, 0};
        int ns = 0;
        if (in) {
            rr = rings[r];
            ns = disc_runs(hs, d, c, r, rr.startpix, j0, ln);
        }
        const int mine = ns + (((ns > 0 ? ln[0] : 0) + (ns > 1 ? ln[1] : 0)) << 8);
        const int incl = carry + seg_incl_scan<SUB>(mine, sl);
        /* the rings whose runs still fit the table (a prefix of the lanes) */
        const bool fit = more && (incl & 255) <= RPP;
        unsigned long long fm = __ballot(fit);
        if constexpr (SUB < kWaveSize)
            fm = (fm >> (lane & ~(SUB - 1))) & ((1ull << SUB) - 1ull);
        const int nfit = __popcll(fm);
        int run = (incl & 255) - ns;
        int off = (incl >> 8) - (mine >> 8);
#pragma unroll
        for (int k = 0; k < 2; k++) {   /* constant indices keep j0, ln in registers */
            if (fit && k < ns) {
                const RunGeo g = run_geo(hs, rr, r, c, j0[k], ln[k]);
                const int mid = off - j0[k] + g.kc;
                t.rec[run][0] = make_float4(g.a0, g.b, (float)mid,
                                            __int_as_float(rr.startpix + j0[k] - off));
                t.rec[run][1] = make_float4(g.sD, g.omD, g.cdp2, g.kap);
                t.pref[run] = off;
                const float x0 = fabsf(fmaf((float)(off - mid), g.b, g.a0));
                const float x1 = fabsf(fmaf((float)(off + ln[k] - mid), g.b, g.a0));
                const float xm = fmaxf(x0, x1);
                const bool w = !(fabsf(g.kap) * xm < eta_max) || xm > 0.7f;
                t.ring[run] = w ? ~r : r;
                if constexpr (T::WIDE) {
                    if (w)
                        t.wide[run] = {0.5 * g.a0d, 0.5 * g.bd, 2.0 * g.kapd};
                }
                wide = wide || w;
                if (off > 0 && off <= T::VCAP)   /* the first segment's marks */
                    atomicOr(&t.bits[mark_word(off)], mark_bit(off));
                run++;
                off += ln[k];
            }
        }
        const int last = __shfl(incl, nfit > 0 ? nfit - 1 : 0, SUB);
        carry = nfit > 0 ? last : carry;
        ps.next += nfit;
        more = more && nfit == SUB;
    }
    ps.nrun = carry & 255;
    ps.total = carry >> 8;
    unsigned long long wm = __ballot(wide);
    if constexpr (SUB < kWaveSize)   /* the group's own runs decide its form */
        wm = (wm >> (lane & ~(SUB - 1))) & ((1ull << SUB) - 1ull);
    ps.wide = wm != 0ull;
    if (sl == 0)
        t.pref[ps.nrun] = ps.total;
    wave_sync();
    return ps;
}

template <typename T>
__device__ inline int run_ring(const T &t, int i)
{
    const int r = t.ring[i];
    return r < 0 ? ~r : r;
}

/* Marks the runs of the segment that starts at visit seg0 > 0; returns the run
 * of its first visit. */
template <typename T>
__device__ inline int mark_segment(T &t, int nrun, int seg0, int sl)
{
    constexpr int SUB = T::SUB;
    wave_sync();
    for (int w = sl; w < T::VCAP / 32; w += SUB)
        t.bits[w] = 0u;
    wave_sync();
    int started = 0;
    for (int i0 = 0; i0 < T::RPP; i0 += SUB) {
        const bool in = i0 + sl < nrun;
        const int o = in ? t.pref[i0 + sl] - seg0 : 1;
        unsigned long long m = __ballot(in && o <= 0);
        if constexpr (SUB < kWaveSize)
            m = (m >> ((int)__lane_id() & ~(SUB - 1))) & ((1ull << SUB) - 1ull);
        started += __popcll(m);
        if (in && o > 0 && o <= T::VCAP)
            atomicOr(&t.bits[mark_word(o)], mark_bit(o));
    }
    wave_sync();
    return segment_base(started);
}

/* A visit whose beam pixel lies inside the beam, with what `use` needs. */
struct Pending {
    int v, s;         /* visit and run of the pass */
    int pix, bp;
    float c2, s2;
    float4 v0;        /* A0 A1 A2 B0 */
    float2 v1;        /* B1 B2 */
    float2 v2;        /* A3 B3 (forward with the V term only) */
    float sI, sQ, sU; /* sky of the visit (forward only) */
    float sV;         /* sky V of the visit (forward with the V term only) */
    bool live;
    CapPlace place;   /* WALK_PLACE only */
};

/* Adds the TOD terms of one visit, a and b (convolver.cpp:157-164; with VT
 * the V terms the reference's GPU kernel adds, V A3 and V B3,
 * cudaConv2.cu:204,214,217-218).  With X + iY = (Q + iU) e^{-2i chi} the
 * polarised part is A1 X + A2 Y for a and its negative with B for b.  The I
 * (and V) products are formed exactly in FP64: their float rounding would be
 * the sum's largest error. */
template <bool VT>
__device__ inline void visit_tod(const Pending &e, double &acc_a, double &acc_b)
{
    const float X = fmaf(e.sQ, e.c2, e.sU * e.s2), Y = fmaf(e.sU, e.c2, -(e.sQ * e.s2));
    const float pa = fmaf(e.v0.z, Y, e.v0.y * X), pb = fmaf(e.v1.y, Y, e.v1.x * X);
    const double I = e.sI;
    acc_a = fma(I, (double)e.v0.x, acc_a) + (double)pa;
    acc_b = fma(I, (double)e.v0.w, acc_b) - (double)pb;
    if constexpr (VT) {
        acc_a = fma((double)e.sV, (double)e.v2.x, acc_a);
        acc_b = fma((double)e.sV, (double)e.v2.y, acc_b);
    }
}

__device__ inline int lanes_below(unsigned long long m)
{
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                          __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

/* What a walk loads and computes per visit. */
enum {
    WALK_SKY = 1,      /* the sky values */
    WALK_BEAM = 2,     /* the beam row */
    WALK_V = 4,        /* the V columns and the sky's V */
    WALK_CHI = 8,      /* cos, sin 2 chi */
    WALK_PLACE = 16,   /* the beam pixel's ring, quadrant and position */
};

template <int F>
__device__ inline void load_visit(const PairParams &p, Pending &q, int bp, int pix)
{
    if constexpr (F & WALK_BEAM) {
        const float *row = p.beam + 8 * (long)bp;
        q.v0 = *(const float4 *)row;
        q.v1 = *(const float2 *)(row + 4);
        if constexpr (F & WALK_V)
            q.v2 = *(const float2 *)(row + 6);
    }
    if constexpr (F & WALK_SKY) {
        const float4 sv = p.sky4[pix];
        q.sI = sv.x;
        q.sQ = sv.y;
        q.sU = sv.z;
        q.sV = sv.w;
    }
}

__device__ inline void rec_make(const PairParams &p, float ra, float dec, float pa, SampleRec &r)
{
    const Centre c = centre_make(ra, dec, pa);
    double s, co;
    pl_sincos(c.psi, &s, &co);
    r.c2psi = fma(co, co, -(s * s));
    r.s2psi = 2.0 * (s * co);
    r.sf = sample_f32(c, co, s, r.c2psi, r.s2psi);
    r.ra = c.ra;
    r.cdc = c.cdc;
    r.sdc = c.sdc;
    r.psi = c.psi;
    Disc d;
    disc_setup(p.hs, kHalfPi - c.dec, c.ra, p.rho_max, p.cos_rmax, d);
    r.phi = d.phi;
    r.z0 = d.z0;
    r.xa = d.xa;
    r.irmin = d.irmin;
    r.irmax = d.irmax;
    r.r_first = d.r_first;
    r.r_last = d.r_last;
}

__device__ inline Centre rec_centre(const SampleRec &r)
{
    Centre c;
    c.ra = r.ra;
    c.dec = 0.0;   /* not read by the mappings */
    c.psi = r.psi;
    c.cdc = r.cdc;
    c.sdc = r.sdc;
    return c;
}

__device__ inline Disc rec_disc(const PairParams &p, const SampleRec &r)
{
    Disc d;
    d.phi = r.phi;
    d.z0 = r.z0;
    d.xa = r.xa;
    d.cosr = p.cos_rmax;
    d.irmin = r.irmin;
    d.irmax = r.irmax;
    d.r_first = r.r_first;
    d.r_last = r.r_last;
    return d;
}

/* Wave-uniform copy of a float (to scalar registers). */
__device__ inline float unif(float x)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, x)));
}

__device__ inline SampleF unif(const SampleF &f)
{
    SampleF u;
    u.cdc = unif(f.cdc);
    u.sdc = unif(f.sdc);
    u.cps = unif(f.cps);
    u.sps = unif(f.sps);
    u.c2h = unif(f.c2h);
    u.c2l = unif(f.c2l);
    u.s2h = unif(f.s2h);
    u.s2l = unif(f.s2l);
    u.lim0 = unif(f.lim0);
    return u;
}

/* A wave's samples (NS of them) and its queue of visits deferred to the FP64
 * form (sky pixel, sample); fewer than 64 entries between drains, and one
 * iteration adds at most 64. */
template <int NS_>
struct WaveState {
    static constexpr int NS = NS_;
    SampleRec rec[NS];
    int qpix[2 * kWaveSize];
    unsigned char qj[2 * kWaveSize];
};

/* Maps pixel pix for sample j with the certified double-precision form
 * (beam_pixel_f64, whose own fallback is the exact FP64 path; the beam pixel is
 * the exact path's either way) and hands a visit inside the beam to
 * use(q, ring, startpix, j). */
template <int F, typename Use>
__device__ inline void exact_visit(const PairParams &p, const SampleRec &sr, int pix, int j,
                                   Use &use)
{
    const int r = pix2ring(p.hs, pix);
    const RingRec rr = p.rings[r];
    Pending q;
    q.v = q.s = 0;
    q.pix = pix;
    q.live = true;
    q.bp = beam_pixel_f64(p.hb, p.fc64, rec_centre(sr), sr.c2psi, sr.s2psi,
                          ring_phi(p.hs, rr, r, pix), rr.cdp, rr.sdp, q.c2, q.s2);
    if ((unsigned)q.bp < (unsigned)p.npix_beam) {
        load_visit<F>(p, q, q.bp, pix);
        use(q, r, rr.startpix, j);
    }
}

/* Queue entries base .. base+cnt-1 (cnt <= 64), one per lane.  Called with
 * every lane of the wave active. */
template <int F, typename WS, typename Use>
__device__ inline void drain_queue(const PairParams &p, const WS &ws, int base, int cnt, int lane,
                                   Use &use)
{
    wave_sync();
    if (lane < cnt) {
        const int j = ws.qj[base + lane];
        exact_visit<F>(p, ws.rec[j], ws.qpix[base + lane], j, use);
    }
    wave_sync();
}

/* The lanes of m (visits of sample j) join the queue. */
template <typename WS>
__device__ inline void enqueue(WS &ws, int &qn, unsigned long long m, int pix, int j)
{
    if ((m >> __lane_id()) & 1ull) {
        const int pos = qn + lanes_below(m);
        ws.qpix[pos] = pix;
        ws.qj[pos] = (unsigned char)j;
    }
    qn += __popcll(m);
}

/* Where a walk of a pass is: its next visit, its segment, and the runs besides
 * the first that start at or before the next visit's block. */
struct WalkAt {
    int v0 = 0, seg0 = 0, base = 0;
};

/* The walk of one segment of a pass, visits at.v0 .. vend - 1.  Software
 * pipelined by hand: the next visit's records are read from LDS while the
 * current one is mapped (two sets of registers, the loop unrolled by two), and
 * the beam and sky loads of a visit are issued at the end of its iteration and
 * consumed (by `use`) after the next visit's mapping.  Loads two iterations
 * ahead measured slower: the L1 holds 256 lines and a wave's iteration takes
 * 72.  Every global load is issued unconditionally (lanes without a visit load
 * row 0 / pixel 0 and discard them): a load skipped on some path makes the
 * in-order load counter ambiguous at the loop head.  Visits whose floors the
 * float form cannot certify join the queue; the walk returns (at.v0 < vend)
 * when it holds a batch of 64, so that the FP64 drain, which needs many
 * registers, is outside the loop.  WIDE: cos, sin 2 chi in FP64 for the wide
 * runs of the lane groups with `wide`. */
template <int F, bool WIDE, typename T, typename WS, typename Use>
__device__ inline void walk_segment(const PairParams &p, const T &t, WS &ws, int total, int vend,
                                    bool wide, int sl, int j, const SampleF &sf, WalkAt &at,
                                    int &qn, Use &use)
{
    constexpr int SUB = T::SUB;
    struct Rec {
        float4 a, b;
        int run;
    };
    int v0 = at.v0, base = at.base, base0 = base;
    if (v0 >= vend || qn >= kWaveSize)
        return;
    auto fetch = [&](Rec &n, int v) {   /* the records of visit v + sl */
        const int k = v - at.seg0;
        if constexpr (SUB == kWaveSize) {
            const unsigned lo = t.bits[k >> 5], hi = t.bits[(k >> 5) + 1];
            n.run = (int)__builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, base));
            base += __popc(lo) + __popc(hi);
        } else {
            const unsigned m = t.bits[k >> 5] >> (k & 31);
            n.run = base + marks_below(m, sl);
            base += SUB == 32 ? __popc(m) : marks_below(m, SUB);
        }
        n.a = t.rec[n.run][0];
        n.b = t.rec[n.run][1];
    };
    Pending q;
    q.live = false;
    float vf = (float)(v0 + sl);
    auto step = [&](const Rec &r, Rec &n) {
        base0 = base;
        if (v0 + SUB < vend)
            fetch(n, v0 + SUB);
        const int v = v0 + sl;
        const bool act = v < total;
        const int pix = v + __float_as_int(r.a.w);
        const float at_run = vf - r.a.z;   /* ring positions from the run's kc */
        const VisitGeo g =
            visit_geo(fmaf(at_run, r.a.y, r.a.x), r.b.x, r.b.y, r.b.z, sf.cdc, sf.sdc);
        vf += (float)SUB;
        v0 += SUB;
        CapPlace place;
        int bp = visit_pixel(p.fc, sf, g, place);
        float c2 = 0.f, s2 = 0.f;
        if constexpr (F & WALK_CHI) {
            float d4, s4;
            visit_phase(g, r.b.w, d4, s4);
            if constexpr (WIDE) {
                const int rg = wide ? ~t.ring[r.run] : -1;   /* a wide pass has runs */
                if (rg >= 0) {
                    if constexpr (T::WIDE) {
                        const WideRec &wr = t.wide[r.run];
                        visit_phase64(fma((double)at_run, wr.b, wr.a0), wr.k2, d4, s4);
                    } else {
                        const RingRec rr = p.rings[rg];
                        visit_phase64(rec_centre(ws.rec[j]), ring_phi(p.hs, rr, rg, pix), rr.cdp,
                                      rr.sdp, d4, s4);
                    }
                }
            }
            visit_chi(sf, d4, s4, c2, s2);
        }
        bp = act ? bp : -1;
        const unsigned long long m = __ballot(bp == kNeedExact);
        if (q.live)
            use(q);
        if (m)
            enqueue(ws, qn, m, pix, j);
        q.live = (unsigned)bp < (unsigned)p.npix_beam;   /* rejects -1 and kNeedExact */
        q.v = v;
        q.s = r.run;
        q.pix = pix;
        q.bp = bp;
        q.c2 = c2;
        q.s2 = s2;
        if constexpr (F & WALK_PLACE)
            q.place = place;
        if constexpr ((F & (WALK_SKY | WALK_BEAM)) != 0)
            load_visit<F>(p, q, q.live ? bp : 0, q.live ? pix : 0);
    };
    Rec ra, rb;
    fetch(ra, v0);
    for (;;) {
        step(ra, rb);
        if (v0 >= vend || qn >= kWaveSize)
            break;
        step(rb, ra);
        if (v0 >= vend || qn >= kWaveSize)
            break;
    }
    if (q.live)
        use(q);
    at.v0 = v0;
    at.base = base0;
}

/* The largest x over the wave's lane groups, each of which holds one value.  By
 * lane reads: the lane addresses of shuffles, formed before the walk, were spilled,
 * and each of their six steps waited for scratch memory (forward, 2e4 samples of 5
 * pixels 17.0 and 15.6 us, 2e5 of 136 pixels 179 and 171; sky adjoint, 2e5 of 34
 * pixels 261 and 242). */
template <int SUB>
__device__ inline int group_max_uniform(int x)
{
    int m = __builtin_amdgcn_readlane(x, 0);
#pragma unroll
    for (int g = SUB; g < kWaveSize; g += SUB)
        m = max(m, __builtin_amdgcn_readlane(x, g));
    return m;
}

/* Rings r0 .. r_last of the disc of sample j of the lane group's wave state
 * (none if r_last < r0), in passes; wave-uniform control flow: groups with
 * fewer rings, visits or segments idle.  after(ps): called once per pass
 * between its build and its walk; use(q) per visit inside the beam, use_exact
 * per deferred one (see drain_queue). */
template <int F, typename T, typename WS, typename After, typename Use, typename UseExact>
__device__ inline void walk_rings(const PairParams &p, T &t, WS &ws, int j, int r0, int r_last,
                                  int sl, const SampleF &sf, float eta_max, int &qn, After &after,
                                  Use &use, UseExact &use_exact)
{
    constexpr int SUB = T::SUB;
    const int lane = (int)__lane_id();
    while (SUB == kWaveSize ? r0 <= r_last : (bool)__any(r0 <= r_last)) {
        const Pass ps = build_pass(p.hs, p.rings, rec_disc(p, ws.rec[j]), rec_centre(ws.rec[j]), r0,
                                   r_last, sl, eta_max, t);
        after(ps);
        int total = ps.total, wtot;
        if constexpr (SUB == kWaveSize) {
            total = __builtin_amdgcn_readfirstlane(total);
            wtot = total;
        } else {
            wtot = group_max_uniform<SUB>(total);
        }
        const bool any_wide = __any(ps.wide);
        WalkAt at;
        for (;;) {
            const int vend = min(wtot, at.seg0 + T::VCAP);
            if (any_wide)
                walk_segment<F, true>(p, t, ws, total, vend, ps.wide, sl, j, sf, at, qn, use);
            else
                walk_segment<F, false>(p, t, ws, total, vend, false, sl, j, sf, at, qn, use);
            if (qn >= kWaveSize) {
                drain_queue<F>(p, ws, qn - kWaveSize, kWaveSize, lane, use_exact);
                qn -= kWaveSize;
            }
            if (at.v0 >= vend) {
                if (vend >= wtot)
                    break;
                at.seg0 = vend;
                at.base = mark_segment(t, ps.nrun, vend, sl);
            }
        }
        wave_sync();
        r0 = ps.next;
        if constexpr (SUB == kWaveSize)
            r0 = __builtin_amdgcn_readfirstlane(r0);
    }
}

/* The constants of samples i0 .. i0+cnt-1 (cnt <= NS): from p.samples, or
 * computed, one sample per lane. */
template <typename WS>
__device__ inline void wave_samples(const PairParams &p, WS &ws, long i0, int cnt, float pa_off,
                                    bool offset, int lane)
{
    if (p.samples) {
        constexpr int W = sizeof(SampleRec) / sizeof(int);
        const int *src = (const int *)(p.samples + (i0 - p.s_begin));
        for (int k = lane; k < cnt * W; k += kWaveSize)
            ((int *)ws.rec)[k] = src[k];
    } else if (lane < cnt) {
        const float pa = p.pa[i0 + lane];
        rec_make(p, p.ra[i0 + lane], p.dec[i0 + lane], offset ? pa + pa_off : pa, ws.rec[lane]);
    }
    wave_sync();
}

template <int SUB>
using SubTable = VisitTable<SUB, (SUB < 16 ? 24 : SUB < 64 ? 32 : 64),
                            (SUB < 16 ? 256 : SUB < 64 ? 1024 : 4096), (SUB >= 16)>;
using WaveTable = SubTable<kWaveSize>;

/* ---- forward ---------------------------------------------------------------
 *
 * A wave holds G = 64/SUB samples of SUB lanes each, a block kWavesPerBlock
 * waves.  The deferred visits that do not fill a batch of 64 are mapped once per
 * block, by the last wave that finishes, so that no wave waits: the FP64 form
 * costs the same for one lane as for 64 (5-degree discs in 6 strips: 0.10 of the
 * time).  The first wave computing the constants of the whole block's samples
 * was no gain: the others wait for it.
 *
 * The runs of a table: 24 and 32 for 8 and 16 lanes (16: more passes, each with
 * a ragged end; 1.29 and 1.15 ms for 1e6 samples of 135 pixels with 16 lanes),
 * within the 40 KB of LDS that leave four blocks per CU. */
template <int SUB>
struct FwdBlock {
    static constexpr int G = kWaveSize / SUB, NS = kWavesPerBlock * G;
    SubTable<SUB> tables[NS];
    SampleRec rec[NS];
    int qpix[kWavesPerBlock][2 * kWaveSize];
    unsigned char qj[kWavesPerBlock][2 * kWaveSize];
    int qn[kWavesPerBlock], done;
    double sum[NS][2], dsum[NS][2];   /* of the walks, of the deferred visits */
};

/* A wave's view of its block: the samples of the block, its own queue. */
struct WaveView {
    SampleRec *rec;
    int *qpix;
    unsigned char *qj;
};

/* Samples i0 .. i0+ns-1 (ns <= NS), strip k of their discs: their sums to
 * put(sample, a, b).  Every thread of the block calls it.  With one wave
 * per sample a sample's sums do not depend on the samples it shares the block
 * with.  Lane groups share a wave's queue of deferred visits, so there the order
 * in which those few are added in FP64 does. */
template <int SUB, bool VT, typename Put>
__device__ inline void forward_block(const PairParams &p, FwdBlock<SUB> &B, long i0, int ns, int k,
                                     float pa_off, bool offset, Put &put)
{
    constexpr int G = FwdBlock<SUB>::G;
    constexpr int F = WALK_SKY | WALK_BEAM | WALK_CHI | (VT ? WALK_V : 0);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
    const int lane = threadIdx.x % kWaveSize;
    const int grp = lane / SUB, sl = lane % SUB;
    WaveView ws = {B.rec, B.qpix[wave], B.qj[wave]};
    if (threadIdx.x < 2 * ns)
        B.dsum[threadIdx.x >> 1][threadIdx.x & 1] = 0.0;
    if (threadIdx.x == 0)
        B.done = 0;
    const int j0 = wave * G;
    if (j0 < ns) {
        WaveView own = {B.rec + j0, nullptr, nullptr};
        wave_samples(p, own, i0 + j0, min(G, ns - j0), pa_off, offset, lane);
    }
    __syncthreads();
    if (j0 >= ns)
        return;
    const int j = j0 + grp < ns ? j0 + grp : j0;   /* a group without a sample idles */
    SampleF sf = B.rec[j].sf;
    int r0 = B.rec[j].r_first, r1 = B.rec[j].r_last;
    if constexpr (SUB == kWaveSize) {
        sf = unif(sf);
        r0 = __builtin_amdgcn_readfirstlane(r0);
        r1 = __builtin_amdgcn_readfirstlane(r1);
        const int m = (r1 - r0 + p.strips) / p.strips;   /* rings per strip */
        r0 += k * m;
        r1 = min(r1, r0 + m - 1);
    } else if (j0 + grp >= ns) {
        r1 = r0 - 1;
    }
    double acc_a = 0.0, acc_b = 0.0;
    auto use = [&](const Pending &q) { visit_tod<VT>(q, acc_a, acc_b); };
    auto use_exact = [&](const Pending &q, int, int, int jj) {
        double a = 0.0, b = 0.0;
        visit_tod<VT>(q, a, b);
        atomicAdd(&B.dsum[jj][0], a);
        atomicAdd(&B.dsum[jj][1], b);
    };
    auto after = [](const Pass &) {};
    int qn = 0;
    walk_rings<F>(p, B.tables[j0 + grp], ws, j, r0, r1, sl, sf, kEtaForward, qn, after, use,
                  use_exact);
#pragma unroll
    for (int m = SUB / 2; m > 0; m >>= 1) {
        acc_a += __shfl_xor(acc_a, m, SUB);
        acc_b += __shfl_xor(acc_b, m, SUB);
    }
    if (sl == 0 && j0 + grp < ns) {
        B.sum[j0 + grp][0] = acc_a;
        B.sum[j0 + grp][1] = acc_b;
    }
    if (lane == 0)
        B.qn[wave] = qn;
    const int waves = (ns + G - 1) / G;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    int arrived = 0;
    if (lane == 0)
        arrived = atomicAdd(&B.done, 1);
    if (__builtin_amdgcn_readfirstlane(arrived) != waves - 1)
        return;
    /* the last wave of the block */
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    int end[kWavesPerBlock], total = 0;
#pragma unroll
    for (int w = 0; w < kWavesPerBlock; w++) {
        total += w < waves ? __builtin_amdgcn_readfirstlane(B.qn[w]) : 0;
        end[w] = total;
    }
    for (int e0 = 0; e0 < total; e0 += kWaveSize) {
        const int e = e0 + lane;
        if (e < total) {
            int w = 0, first = 0;
#pragma unroll
            for (int x = 0; x < kWavesPerBlock - 1; x++) {
                w = e >= end[x] ? x + 1 : w;
                first = e >= end[x] ? end[x] : first;
            }
            const int jj = B.qj[w][e - first];
            exact_visit<F>(p, B.rec[jj], B.qpix[w][e - first], jj, use_exact);
        }
        wave_sync();
    }
    wave_sync();
    if (lane < ns)
        put(lane, B.sum[lane][0] + B.dsum[lane][0], B.sum[lane][1] + B.dsum[lane][1]);
}

/* The forward of one pair: consecutive samples, whole discs; or (SUB = 64,
 * p.strips > 1) a strip of each disc, in chunks of kStripChunk samples and
 * within a chunk by strip.  The beam rows that a strip of the sky meets are
 * about a strip of the beam, nearly the same one for samples close in the scan,
 * so that this part stays in the XCD's L2; with whole discs the waves gather
 * from all of a 12 MB beam.  The samples in flight have to be close: with 2, 4
 * and 8 samples per wave (1,024 to 4,096 in flight per XCD) the L2 hit rate fell
 * from 0.93 to 0.83, 0.71 and 0.56; hence one sample per wave, whose constants
 * k_samples computes once for all strips.
 *
 * Bound: a visit gathers a 128-byte line of the beam, 2.15 cycles each per CU
 * (140 cycles per 64 visits), and takes about 130 vector instructions per 64;
 * both units are 0.84 to 0.96 busy at 5 degrees. */
constexpr int kStripChunk = 4096;

template <int SUB, bool VT = false>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_fwd_sub(PairParams p)
{
    __shared__ FwdBlock<SUB> B;
    constexpr int NS = FwdBlock<SUB>::NS;
    const long lb = xcd_remap(blockIdx.x, gridDim.x);
    long i0 = p.s_begin + lb * NS;
    int k = 0;
    if (SUB == kWaveSize && p.strips > 1) {
        long strip, blk;
        if (!work_item(lb, (p.s_end - p.s_begin + NS - 1) / NS, p.strips, kStripChunk / NS, strip,
                       blk))
            return;
        k = (int)strip;
        i0 = p.s_begin + blk * NS;
    }
    if (i0 >= p.s_end)
        return;
    auto put = [&](int j, double a, double b) {
        const long i = i0 + j;
        if (SUB == kWaveSize && p.strips > 1) {
            const long n = p.s_end - p.s_begin;
            p.part[(2 * k) * n + i - p.s_begin] = a;
            p.part[(2 * k + 1) * n + i - p.s_begin] = b;
        } else {
            if (p.tod_a)
                p.tod_a[i] = (float)a;
            if (p.tod_b)
                p.tod_b[i] = (float)b;
        }
    };
    forward_block<SUB, VT>(p, B, i0, (int)min((long)NS, p.s_end - i0), k, 0.f, false, put);
}

/* The strips of a disc one after the other, where there is no workspace for their
 * sums (a captured graph holds the context's buffers): the same sums in the same
 * order as k_fwd_sub and k_strip_sum.  The waves drift apart over the beam. */
template <bool VT>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_fwd_strips(PairParams p)
{
    __shared__ FwdBlock<kWaveSize> B;
    constexpr int NS = FwdBlock<kWaveSize>::NS;
    __shared__ double total[NS][2];
    const long i0 = p.s_begin + xcd_remap(blockIdx.x, gridDim.x) * NS;
    const int ns = (int)min((long)NS, p.s_end - i0);
    if (threadIdx.x < 2 * NS)
        total[threadIdx.x >> 1][threadIdx.x & 1] = 0.0;
    auto put = [&](int j, double a, double b) {
        total[j][0] += a;
        total[j][1] += b;
    };
    for (int k = 0; k < p.strips; k++) {
        __syncthreads();
        forward_block<kWaveSize, VT>(p, B, i0, ns, k, 0.f, false, put);
    }
    __syncthreads();
    if ((int)threadIdx.x < ns) {
        const long i = i0 + threadIdx.x;
        if (p.tod_a)
            p.tod_a[i] = (float)total[threadIdx.x][0];
        if (p.tod_b)
            p.tod_b[i] = (float)total[threadIdx.x][1];
    }
}

/* The samples' constants, one per thread. */
__global__ void k_samples(PairParams p)
{
    const long i = p.s_begin + (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < p.s_end) {
        SampleRec r;
        rec_make(p, p.ra[i], p.dec[i], p.pa[i], r);
        p.samples[i - p.s_begin] = r;
    }
}

/* TOD = the sums of the strips, in strip order. */
__global__ void k_strip_sum(PairParams p)
{
    const long n = p.s_end - p.s_begin;
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (long)gridDim.x * blockDim.x) {
        double a = 0.0, b = 0.0;
        for (int k = 0; k < p.strips; k++) {
            a += p.part[(2 * k) * n + i];
            b += p.part[(2 * k + 1) * n + i];
        }
        if (p.tod_a)
            p.tod_a[p.s_begin + i] = (float)a;
        if (p.tod_b)
            p.tod_b[p.s_begin + i] = (float)b;
    }
}

/* The direct-atomic adjoints, one sample per wave. */
template <int OP>
__global__ __launch_bounds__(kBlock) void k_pair(PairParams p)
{
    constexpr int F = WALK_CHI | (OP == OP_ADJ_MAP ? WALK_BEAM : 0);
    __shared__ WaveTable tables[kWavesPerBlock];
    __shared__ WaveState<1> states[kWavesPerBlock];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
    const int lane = threadIdx.x % kWaveSize;
    const long i = p.s_begin + xcd_remap(blockIdx.x, gridDim.x) * kWavesPerBlock + wave;
    if (i >= p.s_end)
        return;
    auto &ws = states[wave];
    wave_samples(p, ws, i, 1, 0.f, false, lane);
    const double ga = uni(p.g_a ? (double)p.g_a[i] : 0.0);
    const double gb = uni(p.g_b ? (double)p.g_b[i] : 0.0);
    auto use = [&](const Pending &q) {
        if constexpr (OP == OP_ADJ_MAP) {
            const float A0 = q.v0.x, A1 = q.v0.y, A2 = q.v0.z;
            const float B0 = q.v0.w, B1 = q.v1.x, B2 = q.v1.y;
            double cc = q.c2, ss = q.s2;
            double vI = ga * A0 + gb * B0;
            double vQ = ga * (A1 * cc - A2 * ss) + gb * (-B1 * cc + B2 * ss);
            double vU = ga * (A2 * cc + A1 * ss) + gb * (-B2 * cc - B1 * ss);
            unsafeAtomicAdd(&p.gI[q.pix], vI);
            unsafeAtomicAdd(&p.gQ[q.pix], vQ);
            unsafeAtomicAdd(&p.gU[q.pix], vU);
        } else {
            double cc = q.c2, ss = q.s2;
            double qq = p.Q[q.pix], u = p.U[q.pix], sI = p.I[q.pix];
            double *g = p.gbeam + 8 * (long)q.bp;
            unsafeAtomicAdd(&g[0], ga * sI);
            unsafeAtomicAdd(&g[1], ga * (qq * cc + u * ss));
            unsafeAtomicAdd(&g[2], ga * (-qq * ss + u * cc));
            unsafeAtomicAdd(&g[3], gb * sI);
            unsafeAtomicAdd(&g[4], gb * (-qq * cc - u * ss));
            unsafeAtomicAdd(&g[5], gb * (qq * ss - u * cc));
        }
    };
    auto use_exact = [&](const Pending &q, int, int, int) { use(q); };
    auto after = [](const Pass &) {};
    int qn = 0;
    walk_rings<F>(p, tables[wave], ws, 0, __builtin_amdgcn_readfirstlane(ws.rec[0].r_first),
                  __builtin_amdgcn_readfirstlane(ws.rec[0].r_last), lane, unif(ws.rec[0].sf),
                  kEtaAdjoint, qn, after, use, use_exact);
    if (qn > 0)
        drain_queue<F>(p, ws, 0, qn, lane, use_exact);
}

/* ---- beam interpolation mode ----------------------------------------------
 *
 * The convolution with the beam interpolated at (rho, sigma) from the four
 * get_interpol neighbours that lie inside the beam map, normalised by the
 * sum of their weights: the interpolating form of convolver.cpp:124-147
 * (commented out there), in its precision (float values accumulated from
 * double products, divided by the double weight sum), with the values
 * starting from zero at every visit.  A visit with no neighbour in the beam
 * contributes nothing.  The mapping is the exact FP64 rho_sigma_chi of the
 * sky pixel; one wave per sample walks the disc as k_fwd_sub does, without the
 * pipelining of the nearest-pixel kernels.  Sky adjoint and beam adjoint use
 * FP64 atomics; the beam adjoint spreads each visit over the neighbours used
 * with weights w / sum(w). */
template <int OP>
__global__ __launch_bounds__(kBlock) void k_pair_interp(PairParams p)
{
    __shared__ RunTable tables[kWavesPerBlock];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
    const int lane = threadIdx.x % kWaveSize;
    const long lb = xcd_remap(blockIdx.x, gridDim.x);
    const long i = p.s_begin + lb * kWavesPerBlock + wave;
    if (i >= p.s_end)
        return;
    RunTable &t = tables[wave];
    Centre c = centre_make(p.ra[i], p.dec[i], p.pa[i]);
    c.ra = uni(c.ra);
    c.psi = uni(c.psi);
    c.cdc = uni(c.cdc);
    c.sdc = uni(c.sdc);
    Disc d;
    disc_setup(p.hs, kHalfPi - uni(c.dec), c.ra, p.rho_max, p.cos_rmax, d);
    double ga = 0.0, gb = 0.0;
    if (OP != OP_FWD) {
        ga = p.g_a ? (double)p.g_a[i] : 0.0;
        gb = p.g_b ? (double)p.g_b[i] : 0.0;
    }
    double acc_a = 0.0, acc_b = 0.0;
    for (int r0 = d.r_first; r0 <= d.r_last; r0 += kWaveSize) {
        const int total = build_runs(p.hs, d, r0, lane, t);
        int s = 0;
        for (int v = lane; v < total; v += kWaveSize) {
            while (v >= t.pref[s + 1])
                s++;
            const int pix = t.pix0[s] + (v - t.pref[s]);
            const int r = t.ring[s];
            const RingRec rr = p.rings[r];
            const double ra_pix = ring_phi(p.hs, rr, r, pix);
            double rho, sigma, chi;
            visit_rsc(c, ra_pix, rr.cdp, rr.sdp, rho, sigma, chi);
            int nb[4];
            double w[4];
            get_interpol(p.hb, rho, sigma, nb, w);
            float va[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            double ws = 0.0;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                if ((unsigned)nb[k] < (unsigned)p.npix_beam) {
                    ws += w[k];
                    const float *row = p.beam + 8 * (long)nb[k];
#pragma unroll
                    for (int b = 0; b < 6; b++)
                        va[b] = (float)((double)va[b] + (double)row[b] * w[k]);
                }
            }
            if (!(ws > 0.0))
                continue;
#pragma unroll
            for (int b = 0; b < 6; b++)
                va[b] = (float)((double)va[b] / ws);
            double c2d, s2d;
            pl_sincos(2.0 * chi, &s2d, &c2d);
            const float c2 = (float)c2d, s2 = (float)s2d;
            const float A0 = va[0], A1 = va[1], A2 = va[2];
            const float B0 = va[3], B1 = va[4], B2 = va[5];
            if (OP == OP_FWD) {
                const float sI = p.I[pix], sQ = p.Q[pix], sU = p.U[pix];
                float ta = sI * (A0) + sQ * (A1 * c2 - A2 * s2) + sU * (A2 * c2 + A1 * s2);
                float tb = sI * (B0) + sQ * (-B1 * c2 + B2 * s2) + sU * (-B2 * c2 - B1 * s2);
                acc_a += ta;
                acc_b += tb;
            } else if (OP == OP_ADJ_MAP) {
                double cc = c2, ss = s2;
                unsafeAtomicAdd(&p.gI[pix], ga * A0 + gb * B0);
                unsafeAtomicAdd(&p.gQ[pix], ga * (A1 * cc - A2 * ss) + gb * (-B1 * cc + B2 * ss));
                unsafeAtomicAdd(&p.gU[pix], ga * (A2 * cc + A1 * ss) + gb * (-B2 * cc - B1 * ss));
            } else {
                double cc = c2, ss = s2;
                double qq = p.Q[pix], u = p.U[pix], sI = p.I[pix];
                const double v6[6] = {ga * sI, ga * (qq * cc + u * ss), ga * (-qq * ss + u * cc),
                                      gb * sI, gb * (-qq * cc - u * ss), gb * (qq * ss - u * cc)};
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    if ((unsigned)nb[k] < (unsigned)p.npix_beam) {
                        const double f = w[k] / ws;
                        double *g = p.gbeam + 8 * (long)nb[k];
#pragma unroll
                        for (int b = 0; b < 6; b++)
                            unsafeAtomicAdd(&g[b], v6[b] * f);
                    }
                }
            }
        }
        wave_sync();
    }
    if (OP == OP_FWD) {
        acc_a = wave_sum(acc_a);
        acc_b = wave_sum(acc_b);
        if (lane == 0) {
            if (p.tod_a)
                p.tod_a[i] = (float)acc_a;
            if (p.tod_b)
                p.tod_b[i] = (float)acc_b;
        }
    }
}

/* Samples per chunk of the batched launches (work_item): every XCD sees every
 * pair, whose discs differ widely in size. */
constexpr long kBatchChunk = 1024;

/* PairParams of one pair of a batch: its beam, beam-map geometry, disc and
 * outputs (TOD rows 2 out, 2 out + 1 of [pairs][2][nsamples]). */
__device__ inline PairParams batch_pair_params(const BatchParams &b, const BatchPair &q)
{
    PairParams p;
    p.hs = b.hs;
    p.rings = b.rings;
    p.sky4 = b.sky4;
    p.I = b.I;
    p.Q = b.Q;
    p.U = b.U;
    p.hb = hpx_make(q.nside);
    p.npix_beam = q.npix;
    p.rho_max = q.rho_max;
    p.cos_rmax = q.cos_rmax;
    p.fc.k3 = 3.0f * q.nside_f * q.nside_f;
    p.fc64.crho_big = b.fc64.crho_big;
    p.fc64.crho_small = b.fc64.crho_small;
    p.fc64.marg_k = 100.0 * 4.4e-16 * q.nside * 1.7320508075688772;
    p.beam = q.beam;
    p.beam_last = nullptr;
    p.strips = 1;
    p.samples = nullptr;
    p.part = nullptr;
    /* a pointing per pair (ptg_stride > 0) is found by the pair's caller index */
    const long po = (long)(q.out < 0 ? 0 : q.out) * b.ptg_stride;
    p.ra = b.ra + po;
    p.dec = b.dec + po;
    p.pa = b.pa + po;
    p.s_begin = b.s_begin;
    p.s_end = b.s_end;
    const long row = 2 * (long)(q.out < 0 ? 0 : q.out) * b.nsamples;
    p.tod_a = b.tod ? b.tod + row : nullptr;
    p.tod_b = b.tod ? b.tod + row + b.nsamples : nullptr;
    p.g_a = b.g ? b.g + row : nullptr;
    p.g_b = b.g ? b.g + row + b.nsamples : nullptr;
    p.gI = b.gI;
    p.gQ = b.gQ;
    p.gU = b.gU;
    p.gbeam = nullptr;
    return p;
}

/* Batched form of k_fwd_sub: a block per (pair, NS samples) item in the order
 * of work_item; each sample is the single-pair computation with
 * pa = (float)(pa + pa_offset). */
template <int SUB>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4, 8)))
void k_batch_pair(BatchParams b)
{
    __shared__ FwdBlock<SUB> B;
    constexpr int NS = FwdBlock<SUB>::NS;
    const long lb = xcd_remap(blockIdx.x, gridDim.x);
    const long n = b.s_end - b.s_begin;
    long k, j;
    if (!work_item(lb, (n + NS - 1) / NS, b.npairs, b.turn > 0 ? b.turn : kBatchChunk, k, j))
        return;
    const BatchPair &q = b.pairs[k];
    if (q.out < 0)
        return;   /* inert padding */
    const long i0 = b.s_begin + j * NS;
    const PairParams p = batch_pair_params(b, q);
    auto put = [&](int l, double x, double y) {
        p.tod_a[i0 + l] = (float)x;
        p.tod_b[i0 + l] = (float)y;
    };
    forward_block<SUB, false>(p, B, i0, (int)min((long)NS, b.s_end - i0), 0, q.pa_off, true, put);
}

/* ---- batched forward: many detector pairs on one pointing ----------------
 *
 * Detector pairs that share the boresight pointing (each with its own beam,
 * disc radius and position-angle offset) are convolved in one launch.  A wave
 * takes one (sample, group of G pairs), in the item order of work_item; the
 * pairs are sorted by disc radius,
 * so the group's union disc is the disc of its first pair.  Lanes walk the
 * visits of that disc as in k_fwd_sub; per visit the parts that do not depend on
 * the pair (sky values, the float geometry: 1 - cos rho, alpha, the chi
 * phase) are computed once and each pair runs only its tail: disc membership
 * (its own rho_max), beam pixel for its position angle, beam gather, sum.
 * Membership is decided in float away from the disc edge and by the exact
 * query_disc ring test (disc_ring at the pair's radius) within 4e-6 of it;
 * like uncertain beam pixels, such visits go to the per-wave queue and are
 * evaluated exactly, their sums kept in LDS.  The pair table is padded to a
 * multiple of G with inert pairs (npix 0, never members). */

/* Per-wave LDS of a group of G pairs.  A queue entry is a sky pixel (below
 * 2^30) with the pair in the group in its top two bits; the queue holds < 64
 * entries between drains and one visit adds at most G x 64. */
template <int G, typename T>
struct BatchTable {
    T vt;
    unsigned queue[(G + 1) * kWaveSize];
    double acc[G][2];                  /* forward: exact-path sums of each pair */
    double psi[G];                     /* psi of each pair at this sample */
    float ga[G], gb[G];                /* adjoint: cotangents of each pair */
};

/* Exact mapping of a queued visit for one pair: membership by the query_disc
 * ring test at the pair's radius, then the exact beam pixel and chi; the
 * visit's beam row (and its ring's first pixel) when it is inside the beam. */
__device__ inline bool batch_exact_visit(const BatchParams &p, const BatchPair &bp_,
                                         const Centre &c, double psi, int pix, int r,
                                         ExactVisit &e, float4 &v0, float2 &v1, int &sp)
{
    Disc dk;
    disc_setup(p.hs, kHalfPi - c.dec, c.ra, bp_.rho_max, bp_.cos_rmax, dk);
    if (r < dk.r_first || r > dk.r_last)
        return false;
    int p0[2] = {0, 0}, ln[2] = {0, 0};
    const int nrun = disc_ring(p.hs, dk, r, p0, ln);
    bool in = false;
#pragma unroll
    for (int k = 0; k < 2; k++)
        in = in || (k < nrun && (unsigned)(pix - p0[k]) < (unsigned)ln[k]);
    if (!in)
        return false;
    const RingRec rr = p.rings[r];
    const double ra_pix = ring_phi(p.hs, rr, r, pix);
    e = beam_visit_exact(bp_.nside, c.ra, psi, c.cdc, c.sdc, ra_pix, rr.cdp, rr.sdp);
    if ((unsigned)e.bp >= (unsigned)bp_.npix)
        return false;
    const float *row = bp_.beam + 8 * (long)e.bp;
    v0 = *(const float4 *)row;
    v1 = *(const float2 *)(row + 4);
    sp = rr.startpix;
    return true;
}

/* Wave-uniform constants of the pairs d0 .. d0+G-1 at one sample. */
template <int G>
struct BatchConsts {
    float T0[G];                   /* (pi - psi) 2/pi mod 4 */
    float C2H[G], C2L[G], S2H[G], S2L[G];   /* cos, sin 2 psi as float pairs */
    float GA[G], GB[G];            /* adjoint cotangents */
    float NSF[G], CUT_IN[G], CUT_OUT[G];
    float lim0;
    int NPIX[G];
    const float *BEAM[G];
};

__device__ inline float lane_float(float x, int k)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), k));
}

template <int G, bool ADJ, typename BT>
__device__ inline void batch_consts(const BatchParams &p, BT &bt, long i, int d0, int lane,
                                    const Centre &c, BatchConsts<G> &K)
{
    float t0l = 0.f, gal = 0.f, gbl = 0.f;
    double s2 = 0.0, c2 = 1.0;
    if (lane < G) {   /* lane k: pair d0 + k */
        const BatchPair &q = p.pairs[d0 + lane];
        const float pa_k = p.pa[i] + q.pa_off;   /* the pair's own pa */
        const double psi = -(double)pa_k;
        pl_sincos(2.0 * psi, &s2, &c2);
        t0l = pair_t0(psi);
        if (ADJ && q.out >= 0) {
            const long row = 2 * (long)q.out * p.nsamples;
            gal = p.g[row + i];
            gbl = p.g[row + p.nsamples + i];
        }
        bt.psi[lane] = psi;
        bt.acc[lane][0] = 0.0;
        bt.acc[lane][1] = 0.0;
        bt.ga[lane] = gal;
        bt.gb[lane] = gbl;
    }
    const float c2h = (float)c2, s2h = (float)s2;
    const float c2l = (float)(c2 - (double)c2h), s2l = (float)(s2 - (double)s2h);
    /* an irregular centre: every visit of every pair to the exact path */
    const bool reg = centre_regular(c.ra, c.dec);
    K.lim0 = reg ? 0.5f - 2e-6f : -1.0f;
#pragma unroll
    for (int k = 0; k < G; k++) {
        K.T0[k] = lane_float(t0l, k);
        K.C2H[k] = lane_float(c2h, k);
        K.C2L[k] = lane_float(c2l, k);
        K.S2H[k] = lane_float(s2h, k);
        K.S2L[k] = lane_float(s2l, k);
        K.GA[k] = lane_float(gal, k);
        K.GB[k] = lane_float(gbl, k);
        const BatchPair &q = p.pairs[d0 + k];
        K.NSF[k] = q.nside_f;
        K.CUT_IN[k] = reg ? q.omc_cut * (1.0f - 4e-6f) : -1.0f;
        K.CUT_OUT[k] = reg ? q.omc_cut * (1.0f + 4e-6f) : INFINITY;
        K.NPIX[k] = q.npix;
        K.BEAM[k] = q.beam;
    }
    wave_sync();
}

/* A visit of the group waiting for its loads: per pair the beam row, and the
 * visit's sky values, phase e^{2i(alpha+beta)} = (c4, -s4) and place. */
template <int G>
struct BatchPend {
    float4 q0[G];
    float2 q1[G];
    float c4, s4;
    float sI, sQ, sU;
    int pix, v, s;
    unsigned live;   /* bit k: pair k has this visit inside its beam */
};

/* The walk over the visits of the group's union disc (the disc of its first
 * pair; d clipped by the caller), pipelined as walk_segment: per visit the shared
 * float geometry, then each pair's tail (membership, beam pixel, gather);
 * consume(q) receives a visit once its loads are due (after the next visit's
 * geometry).  Queued visits (uncertain membership or beam pixel) are drained
 * 64 at a time by the whole wave; exact(k, pix, r, sp, e, v0, v1) receives
 * those inside pair k's disc and beam. */
template <int G, bool LOAD_SKY, typename BT, typename After, typename Consume, typename Exact>
__device__ inline void batch_walk(const BatchParams &p, BT &bt, const Disc &d, int lane,
                                  const Centre &c, const BatchConsts<G> &K, int d0, float eta_max,
                                  After &after, Consume &consume, Exact &exact)
{
    auto &t = bt.vt;
    using T = typename std::remove_reference<decltype(t)>::type;
    constexpr int VCAP = T::VCAP;
    const float cdc = unif((float)c.cdc), sdc = unif((float)c.sdc);
    int qn = 0;
    auto drain = [&](int base, int cnt) {
        wave_sync();
        if (lane < cnt) {
            const unsigned e_ = bt.queue[base + lane];
            const int pix = (int)(e_ & 0x3fffffffu), k = (int)(e_ >> 30);
            const int r = pix2ring(p.hs, pix);
            ExactVisit e;
            float4 v0;
            float2 v1;
            int sp;
            if (batch_exact_visit(p, p.pairs[d0 + k], c, bt.psi[k], pix, r, e, v0, v1, sp))
                exact(k, pix, r, sp, e, v0, v1);
        }
        __builtin_amdgcn_s_waitcnt(0);
        wave_sync();
    };
    for (int r0 = d.r_first; r0 <= d.r_last;) {
        const Pass ps = build_pass(p.hs, p.rings, d, c, r0, d.r_last, lane, eta_max, t);
        after(ps);
        r0 = __builtin_amdgcn_readfirstlane(ps.next);
        const int total = __builtin_amdgcn_readfirstlane(ps.total);
        if (total <= 0)
            continue;
        const bool marked = total <= VCAP;
        int base = 0, s = 0;
        float4 n0, n1;
        auto fetch = [&](int v0) {   /* as walk_segment */
            if (marked) {
                const unsigned lo = t.bits[v0 >> 5], hi = t.bits[(v0 >> 5) + 1];
                s = (int)__builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, base));
                base += __popc(lo) + __popc(hi);
            } else {
                const int v = v0 + lane;
                if (v < total)
                    while (v >= t.pref[s + 1])
                        s++;
            }
            n0 = t.rec[s][0];
            n1 = t.rec[s][1];
        };
        fetch(0);
        BatchPend<G> q;
        q.live = 0;
        q.sI = q.sQ = q.sU = 0.f;
        q.pix = q.v = q.s = 0;
        float vf = (float)lane;
        for (int v0 = 0; v0 < total; v0 += kWaveSize, vf += (float)kWaveSize) {
            const float4 r0_ = n0, r1_ = n1;
            const int run = s;
            if (v0 + kWaveSize < total)
                fetch(v0 + kWaveSize);
            const int v = v0 + lane;
            const bool act = v < total;
            const int pix = v + __float_as_int(r0_.w);
            const float at_run = vf - r0_.z;
            const VisitGeo g =
                visit_geo(fmaf(at_run, r0_.y, r0_.x), r1_.x, r1_.y, r1_.z, cdc, sdc);
            float d4, s4;
            visit_phase(g, r1_.w, d4, s4);
            const int r = ps.wide ? ~t.ring[run] : -1;
            if (r >= 0) {
                if constexpr (T::WIDE) {
                    const WideRec &wr = t.wide[run];
                    visit_phase64(fma((double)at_run, wr.b, wr.a0), wr.k2, d4, s4);
                } else {
                    const RingRec rr = p.rings[r];
                    visit_phase64(c, ring_phi(p.hs, rr, r, pix), rr.cdp, rr.sdp, d4, s4);
                }
            }
            const float c4 = 1.0f - d4;
            const float al = visit_alpha(g);
            const float x3y = __builtin_amdgcn_sqrtf(3.0f * g.omc);

            if (q.live)
                consume(q);
            /* the only drain site of the loop: the previous visit is consumed
             * and the next loads are not issued yet */
            while (qn >= kWaveSize) {
                drain(qn - kWaveSize, kWaveSize);
                qn -= kWaveSize;
            }
            /* this visit, per pair (the queue holds < 64 entries here and
             * grows by at most G x 64 below) */
            q.live = 0;
#pragma unroll
            for (int k = 0; k < G; k++) {
                const bool in = act && g.omc < K.CUT_IN[k];
                const bool edge = act && !in && !(g.omc > K.CUT_OUT[k]);
                CapPlace place;
                int bp = pair_pixel(al, x3y, g.omc, K.T0[k], K.NSF[k], K.lim0, place);
                bp = in ? bp : -1;
                const bool defer = edge || bp == kNeedExact;
                const unsigned long long md = __ballot(defer);
                if (md) {
                    if (defer)
                        bt.queue[qn + lanes_below(md)] = (unsigned)pix | ((unsigned)k << 30);
                    qn += __popcll(md);
                }
                const bool live = (unsigned)bp < (unsigned)K.NPIX[k];
                q.live |= live ? (1u << k) : 0u;
                const float *row = K.BEAM[k] + 8 * (long)(live ? bp : 0);
                q.q0[k] = *(const float4 *)row;
                q.q1[k] = *(const float2 *)(row + 4);
            }
            q.c4 = c4;
            q.s4 = s4;
            q.pix = pix;
            q.v = v;
            q.s = run;
            if (LOAD_SKY) {
                const float4 sv = p.sky4[act ? pix : 0];
                q.sI = sv.x;
                q.sQ = sv.y;
                q.sU = sv.z;
            }
        }
        if (q.live)
            consume(q);
        wave_sync();
    }
    while (qn > 0) {
        const int cnt = qn < kWaveSize ? qn : kWaveSize;
        drain(qn - cnt, cnt);
        qn -= cnt;
    }
}

template <int G>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4, 8)))
void k_batch_fwd(BatchParams p)
{
    using BT = BatchTable<G, VisitTable<kWaveSize, kWaveSize, 4096, true>>;
    __shared__ BT tabs[kWavesPerBlock];
    /* each lane's FP64 TOD sums of the group's pairs in LDS, one slot per
     * lane (the same additions in the same order as in registers).  In
     * registers they spilled, and the spill traffic went through the vector
     * memory path this gather-bound kernel is limited by. */
    __shared__ double accb_s[kWavesPerBlock][G][kWaveSize];
    __shared__ double acca_s[kWavesPerBlock][G][kWaveSize];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
    const int lane = threadIdx.x % kWaveSize;
    BT &bt = tabs[wave];
    double (*accb)[kWaveSize] = accb_s[wave];
    double (*acca)[kWaveSize] = acca_s[wave];

    const long lb = xcd_remap(blockIdx.x, gridDim.x);
    const long w = lb * kWavesPerBlock + wave;
    long grp, j;
    if (!work_item(w, p.s_end - p.s_begin, p.ngroups, kBatchChunk, grp, j))
        return;
    const long i = p.s_begin + j;
    const int d0 = (int)grp * G;

    Centre c = centre_make(p.ra[i], p.dec[i], p.pa[i]);
    c.ra = uni(c.ra);
    c.dec = uni(c.dec);
    c.cdc = uni(c.cdc);
    c.sdc = uni(c.sdc);
    BatchConsts<G> K;
    batch_consts<G, false>(p, bt, i, d0, lane, c, K);
    Disc d;
    disc_setup(p.hs, kHalfPi - c.dec, c.ra, p.pairs[d0].rho_max, p.pairs[d0].cos_rmax, d);

#pragma unroll
    for (int k = 0; k < G; k++) {
        acca[k][lane] = 0.0;
        accb[k][lane] = 0.0;
    }
    /* as visit_tod, the sky turned by the visit's phase once for the group
     * and by each pair's 2 psi */
    auto consume = [&](const BatchPend<G> &q) {
        const float Qr = fmaf(q.sQ, q.c4, -(q.sU * q.s4)), Ur = fmaf(q.sU, q.c4, q.sQ * q.s4);
        const double I = q.sI;
#pragma unroll
        for (int k = 0; k < G; k++) {
            if (q.live & (1u << k)) {
                const float X = fmaf(Qr, K.C2H[k],
                                     fmaf(Ur, K.S2H[k], fmaf(Qr, K.C2L[k], Ur * K.S2L[k])));
                const float Y = fmaf(Ur, K.C2H[k],
                                     fmaf(-Qr, K.S2H[k], fmaf(Ur, K.C2L[k], -(Qr * K.S2L[k]))));
                const float ta = fmaf(q.q0[k].z, Y, q.q0[k].y * X);
                const float tb = fmaf(q.q1[k].y, Y, q.q1[k].x * X);
                acca[k][lane] = fma(I, (double)q.q0[k].x, acca[k][lane]) + (double)ta;
                accb[k][lane] = fma(I, (double)q.q0[k].w, accb[k][lane]) - (double)tb;
            }
        }
    };
    auto exact = [&](int k, int pix, int r, int sp, const ExactVisit &e, const float4 &v0,
                     const float2 &v1) {
        (void)r;
        (void)sp;
        const float4 sv = p.sky4[pix];
        Pending q;
        q.sI = sv.x;
        q.sQ = sv.y;
        q.sU = sv.z;
        q.c2 = e.c2;
        q.s2 = e.s2;
        q.v0 = v0;
        q.v1 = v1;
        double ta = 0.0, tb = 0.0;
        visit_tod<false>(q, ta, tb);
        atomicAdd(&bt.acc[k][0], ta);
        atomicAdd(&bt.acc[k][1], tb);
    };
    auto after = [](const Pass &) {};
    batch_walk<G, true>(p, bt, d, lane, c, K, d0, kEtaForward, after, consume, exact);
    wave_sync();
#pragma unroll
    for (int k = 0; k < G; k++) {
        const double ta = wave_sum(acca[k][lane]) + bt.acc[k][0];
        const double tb = wave_sum(accb[k][lane]) + bt.acc[k][1];
        const int out = p.pairs[d0 + k].out;
        if (lane == 0 && out >= 0) {
            p.tod[(2 * (long)out) * p.nsamples + i] = (float)ta;
            p.tod[(2 * (long)out + 1) * p.nsamples + i] = (float)tb;
        }
    }
}

/* ---- adjoint with respect to the sky, LDS-privatised ---------------------
 *
 * A block (8 waves) owns a chunk of K consecutive samples.  Their discs
 * overlap almost entirely, so the block first computes, per ring, the pixel
 * window that covers every disc of the chunk (pass 1: ring spans unwrapped
 * around the chunk's first centre, atomic min/max in LDS), lays the windows
 * out contiguously in LDS (prefix sum), accumulates every visit's I,Q,U
 * gradient into LDS (pass 2: a wave or a lane group per sample, as the forward;
 * ds_add_f32, or ds_add_u64 of 64-bit integers in the deterministic mode), and
 * finally adds the non-zero window entries to the global gradient (one global
 * atomic per pixel and chunk instead of one per visit).  Windows larger than the
 * LDS are taken in slabs of whole rings, one walk each; a chunk with too many
 * rings, or whose samples lie far apart, adds to the global gradient directly. */

struct AdjLayout {
    int chunk;       /* samples per chunk */
    int cap;         /* LDS pixel capacity of the window */
    int rw;          /* ring capacity of the window tables */
    int group;       /* samples per wave at a time, one wave per sample (at most kAdjSamples) */
    long nchunks;
    /* strips of rings that a chunk's discs are cut into (p.strips), taken in
     * groups of strip_group chunks and within a group by strip */
    int strips, strip_group;
    /* batch mode (pairs != NULL): every pair of b.pairs adds into the same
     * windows; the windows use radius rho_w (the pairs' union support) */
    const BatchPair *pairs;
    int npairs;
    double rho_w, cos_w;
    BatchParams b;
    /* deterministic mode: contributions are rounded to multiples of
     * 1 / *fx_scale and summed as 64-bit integers (LDS windows and the global
     * accumulators, whose FP64 planes then hold int64 bits) */
    const double *fx_scale;
};

__host__ __device__ inline long adj_items(const AdjLayout &L)
{
    return work_items(L.nchunks, L.strips);
}

constexpr int kAdjBlock = kAdjWaves * kWaveSize;
/* The beam adjoint's band kernels: one block per CU. */
constexpr int kBandWaves = 16;
constexpr int kBandBlock = kBandWaves * kWaveSize;

/* rint(v * s) as a two's-complement 64-bit integer, for |v * s| < 2^51 and s
 * a power of two (v * s is then exact): adding 1.5 * 2^52 rounds it to the
 * nearest integer, ties to even as rint does (1.5 * 2^52 is even), and
 * leaves that integer in the low bits of the sum's mantissa, whose exponent
 * is fixed (its low word is zero, so the subtraction is one of the high
 * words).  Two instructions instead of rint and a 64-bit conversion. */
__device__ inline unsigned long long fix64(float v, double s)
{
    const unsigned long long t = (unsigned long long)__double_as_longlong(fma((double)v, s, 0x1.8p52));
    return (unsigned long long)((unsigned)(t >> 32) - 0x43380000u) << 32 | (unsigned)t;
}
/* An add to LDS.  The scope differs from that of the global atomics beside it:
 * with the same one the compiler merged the last add of both branches into one
 * flat atomic, which waits for all memory. */
template <typename V>
__device__ inline void lds_add(V *x, V v)
{
    __hip_atomic_fetch_add(x, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
constexpr int kBigI = 0x3fffffff;
/* A chunk whose window exceeds the LDS capacity is split into at most this
 * many slabs of consecutive window rings (see k_adjmap_lds). */
constexpr int kMaxSlabs = 63;
constexpr int kAdjCtl = 4 + kMaxSlabs + 1;   /* ints of the control block */

/* I,Q,U gradient of one visit, in float: each is rounded to the windows'
 * resolution (or accumulated in float) anyway.  The polarised part is
 * (P + iR) e^{2i chi} with P + iR = ga (A1 + iA2) - gb (B1 + iB2). */
__device__ inline void adj_visit_values(float ga, float gb, float4 v0, float2 v1, float c2,
                                        float s2, float &vI, float &vQ, float &vU)
{
    vI = fmaf(gb, v0.w, ga * v0.x);
    const float P = fmaf(-gb, v1.x, ga * v0.y), R = fmaf(-gb, v1.y, ga * v0.z);
    vQ = fmaf(P, c2, -(R * s2));
    vU = fmaf(R, c2, P * s2);
}

/* Where a run's visits lie in the chunk's LDS window: visit v is entry v + x
 * of the window of its ring, which has (y >> 16) entries and starts at slot
 * y & 0xffff (the slab's capacity and a ring's pixels are below 2^16). */
template <typename T>
struct WindowTable : T {
    int2 win[T::RPP];
};

/* Samples that a wave of the sky adjoint takes one after the other. */
constexpr int kAdjSamples = 2;

/* Per-wave LDS of the sky adjoint. */
template <int BG, int SUB>
struct AdjWave {   /* BG >= 2: a group of BG pairs */
    using VT = WindowTable<VisitTable<kWaveSize, 32, 3072>>;
    BatchTable<BG, VT> bt;
};
template <int SUB>
struct AdjWave<0, SUB> {   /* several samples per wave */
    using VT = WindowTable<VisitTable<SUB, SUB, 32 * SUB>>;
    VT vt[kWaveSize / SUB];
    WaveState<kWaveSize / SUB> ws;
    float g[kWaveSize / SUB][2];   /* cotangents */
};
template <>
struct AdjWave<0, kWaveSize> {
    using VT = WindowTable<VisitTable<kWaveSize, 40, 1536>>;
    VT vt;
    WaveState<kAdjSamples> ws;
    float g[kAdjSamples][2];
};
template <>
struct AdjWave<1, kWaveSize> : AdjWave<0, kWaveSize> {
};

/* BG: 0 one pair; 1 a batch, one wave per (pair, sample); 2, 4 a batch, one
 * wave per (group of BG pairs, sample) sharing each visit's geometry.
 * DET: deterministic mode: every contribution (with BG >= 2, each visit's
 * sum over the group's pairs, formed in pair order) is rounded once to a
 * multiple of 1 / scale and all sums are 64-bit integer sums, which do not
 * depend on the order of the additions; the result is the same bits for any
 * schedule and launch shape (for a given grouping of the pairs). */
template <int BG, bool DET = false, int SUB = kWaveSize>
__global__ __launch_bounds__(kAdjBlock) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_adjmap_lds(PairParams p, AdjLayout L)
{
    static_assert(SUB == kWaveSize || BG == 0, "several samples per wave: single pair");
    constexpr bool BATCH = BG > 0;
    using WT = AdjWave<BG, SUB>;
    extern __shared__ __align__(16) unsigned char smem[];
    WT *wtab = (WT *)smem;
    int *win_lo = (int *)(wtab + kAdjWaves);
    int *win_hi = win_lo + L.rw;
    int *win_base = win_hi + L.rw;          /* rw + 1 */
    int *ctl = win_base + L.rw + 1;         /* 0 R0, 1 R1, 2 W, 3 slabs, 4.. slab starts */
    int *slab = ctl + 4;                    /* first window ring of each slab, then nring */
    float *acc = (float *)(ctl + kAdjCtl);
    /* deterministic mode: int64 windows, 8-byte aligned after ctl.  Formed
     * by indexing smem (16-byte aligned), not through an integer: a pointer
     * that passes through an integer loses its LDS address space, and its
     * atomics compile to flat instead of ds_add_u64 (which measured the
     * same here: the window's adds are off the critical path). */
    const size_t acc_off = (size_t)((unsigned char *)(ctl + kAdjCtl) - smem);
    unsigned long long *acc64 = (unsigned long long *)(smem + ((acc_off + 7) & ~(size_t)7));
    const double fxs = DET ? *L.fx_scale : 0.0;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWaveSize);
    const int lane = tid % kWaveSize;

    /* Window radius.  A visit adds a non-zero value only if its beam pixel
     * is at or before row `last`, i.e. lies in a beam ring <= R of that row.
     * A point in a ring-R pixel has colatitude below the centre colatitude of
     * ring R+1 (pixel vertices lie on the neighbouring rings), so every
     * contributing sky pixel is within theta(R+1) of the sample; the windows
     * use theta(R+2), one more ring of margin.  Visits outside a window still
     * take the global-atomic path below, so the windows only need to be
     * right for speed, not for the result. */
    double rho_w = p.rho_max, cos_w = p.cos_rmax;
    if (BATCH) {
        rho_w = L.rho_w;
        cos_w = L.cos_w;
    } else if (p.beam_last) {
        int last = __builtin_amdgcn_readfirstlane(*p.beam_last);
        int rq = (last < 0 ? 0 : pix2ring(p.hb, last)) + 2;
        if (rq < 4 * p.hb.nside) {
            double th = ring_theta(p.hb, rq);
            if (th < rho_w) {
                rho_w = th;
                cos_w = pl_cos(th);
            }
        }
    }

    long lb = xcd_remap(blockIdx.x, gridDim.x);
    const long nitems = adj_items(L);
    for (long item = lb; item < nitems; item += gridDim.x) {
        long unit, ch;
        if (!work_item(item, L.nchunks, L.strips, L.strip_group, unit, ch))
            continue;
        const int strip = (int)unit;
        long s0 = p.s_begin + ch * L.chunk;
        long s1 = s0 + L.chunk < p.s_end ? s0 + L.chunk : p.s_end;
        int ns = (int)(s1 - s0);

        /* pass 0: ring range of the chunk */
        if (tid == 0) {
            ctl[0] = kBigI;
            ctl[1] = -1;
        }
        __syncthreads();
        for (int j = tid; j < ns; j += kAdjBlock) {
            Centre c = centre_make(p.ra[s0 + j], p.dec[s0 + j], 0.f);
            Disc d;
            disc_setup(p.hs, kHalfPi - c.dec, c.ra, rho_w, cos_w, d);
            if (d.r_first <= d.r_last) {
                atomicMin(&ctl[0], d.r_first);
                atomicMax(&ctl[1], d.r_last);
            }
        }
        __syncthreads();
        int R0 = __builtin_amdgcn_readfirstlane(ctl[0]);
        int nring = __builtin_amdgcn_readfirstlane(ctl[1]) - R0 + 1;
        const bool scattered = nring > L.rw;   /* samples all over the sky */
        /* this strip of the window rings; the first strip also takes the disc
         * rings before them and the last one those after */
        const int per_strip = (nring + L.strips - 1) / L.strips;
        int first = -kBigI, last = kBigI;
        if (L.strips > 1) {
            __syncthreads();   /* every wave has read ctl before the next item sets it */
            if (nring <= 0 || scattered) {   /* global atomics: the discs uncut */
                if (strip > 0)
                    continue;
            } else {
                const int a = R0 + min(strip * per_strip, nring);
                const int b = R0 + min((strip + 1) * per_strip, nring);   /* one past */
                if (strip > 0)
                    first = a;
                if (strip < L.strips - 1)
                    last = b - 1;
                R0 = a;
                nring = b - a;
                if (first > last)
                    continue;
            }
        }
        /* no window ring (a disc of radius rho_w can miss every ring centre
         * while the rho_max discs still have visits) or too many: global
         * atomics for this chunk */
        bool fallback = nring <= 0 || scattered;
        double phi_ref;
        {
            Centre c = centre_make(p.ra[s0], p.dec[s0], 0.f);
            Disc d;
            disc_setup(p.hs, kHalfPi - c.dec, c.ra, rho_w, cos_w, d);
            phi_ref = d.phi;
        }
        if (!fallback) {
            for (int k = tid; k < nring; k += kAdjBlock) {
                win_lo[k] = kBigI;
                win_hi[k] = -kBigI;
            }
            __syncthreads();
            /* pass 1: windows (SUB lanes per sample, 64/SUB samples per wave) */
            for (int j0 = wave * (kWaveSize / SUB); j0 < ns; j0 += kAdjWaves * (kWaveSize / SUB)) {
                const int j = j0 + lane / SUB;
                Centre c = centre_make(p.ra[s0 + (j < ns ? j : j0)], p.dec[s0 + (j < ns ? j : j0)],
                                       0.f);
                Disc d;
                disc_setup(p.hs, kHalfPi - c.dec, c.ra, rho_w, cos_w, d);
                const int r_end = j < ns ? min(d.r_last, R0 + nring - 1) : -1;
                for (int r = max(d.r_first, R0) + lane % SUB; r <= r_end; r += SUB) {
                    int lo, hi, ipix1, nr;
                    int kind = disc_ring_span(p.hs, d, r, lo, hi, ipix1, nr);
                    if (kind == 0)
                        continue;
                    if (kind == 2) {
                        lo = -kBigI;
                        hi = kBigI;
                    } else {
                        double ref = nr * kInvTwoPi * phi_ref;
                        double mid = 0.5 * (lo + hi);
                        int sh = (int)rint((ref - mid) / nr);
                        lo += sh * nr;
                        hi += sh * nr;
                    }
                    atomicMin(&win_lo[r - R0], lo);
                    atomicMax(&win_hi[r - R0], hi);
                }
            }
            __syncthreads();
            /* finalise: window start (mod nr) and length per ring; prefix sum */
            if (wave == 0) {
                int carry = 0;
                for (int k0 = 0; k0 < nring; k0 += kWaveSize) {
                    int k = k0 + lane;
                    int len = 0;
                    if (k < nring) {
                        int lo = win_lo[k], hi = win_hi[k];
                        int sp, nr;
                        bool shf;
                        ring_info(p.hs, R0 + k, sp, nr, shf);
                        if (lo == kBigI) {
                            len = 0;
                            lo = 0;
                        } else if (lo <= -kBigI / 2 || hi - lo + 1 >= nr) {
                            len = nr;
                            lo = 0;
                        } else {
                            len = hi - lo + 1;
                            lo %= nr;
                            if (lo < 0)
                                lo += nr;
                        }
                        win_lo[k] = lo;
                        win_hi[k] = len;
                    }
                    int inc = wave_incl_scan(len, lane);
                    if (k < nring)
                        win_base[k] = carry + inc - len;
                    carry += __shfl(inc, kWaveSize - 1, kWaveSize);
                }
                if (lane == 0) {
                    win_base[nring] = carry;
                    ctl[2] = carry;
                }
            }
            __syncthreads();
            /* Samples far apart (a ring's window spans the gaps): windows with more
             * pixels than the discs have visits save no atomics, and with a quarter of
             * that they are not worth more than a few slabs.  Pointings all over the
             * sky, NSIDE 512, 5 degrees: 3,000 samples 1.54 ms in windows, 0.61; 5e4
             * samples 15.7, 7.2. */
            const float disc = 0.5f * (float)p.hs.npix * (float)(1.0 - cos_w);
            const float visits = disc * (float)ns * (BATCH ? (float)L.npairs : 1.0f);
            const float W = (float)__builtin_amdgcn_readfirstlane(ctl[2]);
            const float all = W * (float)L.strips;
            fallback = all > visits || (4.0f * all > visits && W > 4.0f * (float)L.cap);
        }
        if (!fallback) {
            /* slabs: consecutive window rings whose windows add up to at
             * most cap pixels (one slab, the whole window, when it fits) */
            if (tid == 0) {
                const int W = ctl[2];
                int n = 1;
                slab[0] = 0;
                if (W > L.cap) {
                    int k0 = 0;
                    n = 0;
                    while (k0 < nring && n < kMaxSlabs) {
                        int k1 = k0 + 1;
                        while (k1 < nring && win_base[k1 + 1] - win_base[k0] <= L.cap)
                            k1++;
                        slab[n++] = k0;
                        k0 = k1;
                    }
                    /* beyond kMaxSlabs slabs the last one takes the remaining
                     * rings: it exceeds cap, and its visits use global atomics */
                }
                slab[n] = nring;
                ctl[3] = n;
            }
            __syncthreads();
        }
        /* block-uniform slab bounds, read from LDS into scalar registers */
        const int nslab = fallback ? 1 : __builtin_amdgcn_readfirstlane(ctl[3]);
        for (int si = 0; si < nslab; si++) {
        /* this slab: window rings [k0, k1) and their Ws window pixels; the
         * first slab also walks the disc rings before the window rings and
         * the last slab those after (their visits take global atomics) */
        const int k0 = fallback ? 0 : __builtin_amdgcn_readfirstlane(slab[si]);
        const int k1 = fallback ? 0 : __builtin_amdgcn_readfirstlane(slab[si + 1]);
        const int base0 = fallback ? 0 : __builtin_amdgcn_readfirstlane(win_base[k0]);
        const int Ws = fallback ? 0 : __builtin_amdgcn_readfirstlane(win_base[k1]) - base0;
        const bool sfall = fallback || Ws > L.cap;
        const int rlo = (fallback || si == 0) ? first : R0 + k0;
        const int rhi = (fallback || si == nslab - 1) ? last : R0 + k1 - 1;
        auto clamp = [&](Disc &d) {
            d.r_first = d.r_first > rlo ? d.r_first : rlo;
            d.r_last = d.r_last < rhi ? d.r_last : rhi;
        };
        if (!sfall) {
            for (int k = tid; k < 3 * Ws; k += kAdjBlock) {
                if constexpr (DET)
                    acc64[k] = 0ull;
                else
                    acc[k] = 0.f;
            }
        }
        __syncthreads();

        /* pass 2: visits; adds I,Q,U of one visit to the LDS window (or, when no
         * window holds the pixel, to the global FP64 gradient) */
        const int W = sfall ? 0 : Ws;
        auto add = [&](int slot, int pix, float vI, float vQ, float vU) {
            if constexpr (DET) {
                const unsigned long long fI = fix64(vI, fxs);
                const unsigned long long fQ = fix64(vQ, fxs);
                const unsigned long long fU = fix64(vU, fxs);
                if (slot >= 0) {
                    lds_add(&acc64[slot], fI);
                    lds_add(&acc64[W + slot], fQ);
                    lds_add(&acc64[2 * W + slot], fU);
                } else {   /* no window holds the pixel: global int64 atomics */
                    atomicAdd((unsigned long long *)&p.gI[pix], fI);
                    atomicAdd((unsigned long long *)&p.gQ[pix], fQ);
                    atomicAdd((unsigned long long *)&p.gU[pix], fU);
                }
            } else if (slot >= 0) {
                lds_add(&acc[slot], vI);
                lds_add(&acc[W + slot], vQ);
                lds_add(&acc[2 * W + slot], vU);
            } else {   /* no window holds the pixel: global FP64 atomics */
                unsafeAtomicAdd(&p.gI[pix], (double)vI);
                unsafeAtomicAdd(&p.gQ[pix], (double)vQ);
                unsafeAtomicAdd(&p.gU[pix], (double)vU);
            }
        };
        /* the windows of a pass's runs (`n` lanes of a lane group fill them).
         * A ring's window may hold a second copy of the run's positions, nr
         * pixels away; visits there (a run nearly a ring long) take the
         * global atomics. */
        auto fill_windows = [&](auto &vt, const Pass &ps, int l, int n) {
            for (int i = l; i < ps.nrun; i += n) {
                const int r = run_ring(vt, i), k = r - R0;
                int2 w = make_int2(0, 0);
                if (!sfall && k >= k0 && k < k1) {
                    int sp, nr;
                    bool shf;
                    ring_info(p.hs, r, sp, nr, shf);
                    const int off = vt.pref[i];
                    const int j0 = __float_as_int(vt.rec[i][0].w) + off - sp;
                    const int len = win_hi[k];
                    int lo = win_lo[k];
                    const int dm = j0 + (vt.pref[i + 1] - off) / 2 - (lo + len / 2);
                    lo += dm > nr / 2 ? nr : (dm < -(nr / 2) ? -nr : 0);
                    w = make_int2(j0 - off - lo, (len << 16) | (win_base[k] - base0));
                }
                vt.win[i] = w;
            }
            wave_sync();
        };
        /* a visit of the walk, through its run's window */
        auto scatter = [&](const int2 w, int v, int pix, float vI, float vQ, float vU) {
            const int off = v + w.x;
            const int slot = (unsigned)off < (unsigned)w.y >> 16 ? (w.y & 0xffff) + off : -1;
            add(slot, pix, vI, vQ, vU);
        };
        /* a deferred visit, by its pixel and ring */
        auto scatter_pix = [&](int pix, int r, int sp, float vI, float vQ, float vU) {
            if (vI == 0.f && vQ == 0.f && vU == 0.f)
                return;   /* adds nothing */
            const int k = r - R0;
            int slot = -1;
            if (!sfall && k >= k0 && k < k1) {
                int nr = 4 * (r < p.hs.nside ? r
                              : (r > 3 * p.hs.nside ? 4 * p.hs.nside - r : p.hs.nside));
                int off = pix - sp - win_lo[k];
                if (off < 0)
                    off += nr;
                if (off < win_hi[k])   /* inside the ring's window */
                    slot = win_base[k] - base0 + off;
            }
            add(slot, pix, vI, vQ, vU);
        };
        if constexpr (BG >= 2) {
            /* one wave per (group, sample), groups outermost */
            auto &bt = wtab[wave].bt;
            const int ngr = L.npairs / BG;
            for (int j = wave; j < ns * ngr; j += kAdjWaves) {
                const int jg = j / ns;
                const long i = s0 + (j - jg * ns);
                const int d0 = jg * BG;
                Centre c = centre_make(p.ra[i], p.dec[i], p.pa[i]);
                c.ra = uni(c.ra);
                c.dec = uni(c.dec);
                c.cdc = uni(c.cdc);
                c.sdc = uni(c.sdc);
                BatchConsts<BG> K;
                batch_consts<BG, true>(L.b, bt, i, d0, lane, c, K);
                Disc d;
                disc_setup(p.hs, kHalfPi - c.dec, c.ra, L.pairs[d0].rho_max,
                           L.pairs[d0].cos_rmax, d);
                clamp(d);
                /* the pairs' gradients are summed in the frame turned by the
                 * visit's phase, which is undone once */
                auto consume = [&](const BatchPend<BG> &q) {
                    float vI = 0.f, zr = 0.f, zi = 0.f;
#pragma unroll
                    for (int k = 0; k < BG; k++) {
                        if (q.live & (1u << k)) {
                            const float4 v0 = q.q0[k];
                            const float2 v1 = q.q1[k];
                            const float ga = K.GA[k], gb = K.GB[k];
                            vI = fmaf(gb, v0.w, fmaf(ga, v0.x, vI));
                            const float P = fmaf(-gb, v1.x, ga * v0.y);
                            const float R = fmaf(-gb, v1.y, ga * v0.z);
                            zr = fmaf(P, K.C2H[k], fmaf(-R, K.S2H[k], zr));
                            zi = fmaf(R, K.C2H[k], fmaf(P, K.S2H[k], zi));
                        }
                    }
                    if (vI != 0.f || zr != 0.f || zi != 0.f)
                        scatter(bt.vt.win[q.s], q.v, q.pix, vI, fmaf(zr, q.c4, zi * q.s4),
                                fmaf(zi, q.c4, -(zr * q.s4)));
                };
                auto exact = [&](int k, int pix, int r, int sp, const ExactVisit &e,
                                 const float4 &v0, const float2 &v1) {
                    float vI, vQ, vU;
                    adj_visit_values(bt.ga[k], bt.gb[k], v0, v1, e.c2, e.s2, vI, vQ, vU);
                    scatter_pix(pix, r, sp, vI, vQ, vU);
                };
                auto after = [&](const Pass &ps) { fill_windows(bt.vt, ps, lane, kWaveSize); };
                batch_walk<BG, false>(L.b, bt, d, lane, c, K, d0, kEtaAdjoint, after, consume,
                                      exact);
            }
        } else if constexpr (SUB < kWaveSize) {
            /* single pair, small discs: 64/SUB samples per wave, SUB lanes
             * each (as k_fwd_sub) */
            constexpr int G = kWaveSize / SUB;
            const int grp = lane / SUB, sl = lane % SUB;
            auto &tg = wtab[wave].vt[grp];
            auto &ws = wtab[wave].ws;
            for (int j0 = wave * G; j0 < ns; j0 += kAdjWaves * G) {
                const int cnt = min(G, ns - j0);
                const long i0 = s0 + j0;
                wave_samples(p, ws, i0, cnt, 0.f, false, lane);
                const int j = grp < cnt ? grp : 0;
                const SampleF sf = ws.rec[j].sf;
                const float ga = p.g_a ? p.g_a[i0 + j] : 0.f;
                const float gb = p.g_b ? p.g_b[i0 + j] : 0.f;
                if (sl == 0) {
                    wtab[wave].g[grp][0] = ga;
                    wtab[wave].g[grp][1] = gb;
                }
                auto use = [&](const Pending &q) {
                    float vI, vQ, vU;
                    adj_visit_values(ga, gb, q.v0, q.v1, q.c2, q.s2, vI, vQ, vU);
                    if (vI != 0.f || vQ != 0.f || vU != 0.f)
                        scatter(tg.win[q.s], q.v, q.pix, vI, vQ, vU);
                };
                auto use_exact = [&](const Pending &q, int r, int sp, int g) {
                    float vI, vQ, vU;
                    adj_visit_values(wtab[wave].g[g][0], wtab[wave].g[g][1], q.v0, q.v1, q.c2,
                                     q.s2, vI, vQ, vU);
                    scatter_pix(q.pix, r, sp, vI, vQ, vU);
                };
                auto after = [&](const Pass &ps) { fill_windows(tg, ps, sl, SUB); };
                const int r0 = max(ws.rec[j].r_first, rlo);
                const int r1 = grp < cnt ? min(ws.rec[j].r_last, rhi) : r0 - 1;
                int qn = 0;
                constexpr int F = WALK_BEAM | WALK_CHI;
                walk_rings<F>(p, tg, ws, j, r0, r1, sl, sf, p.eta, qn, after, use,
                              use_exact);
                if (qn > 0)
                    drain_queue<F>(p, ws, 0, qn, lane, use_exact);
                wave_sync();   /* the next samples' constants replace these */
            }
        } else {
        /* one wave per (pair, kAdjSamples samples), pairs outermost */
        auto &t = wtab[wave].vt;
        auto &ws = wtab[wave].ws;
        const int np = BATCH ? L.npairs : 1;
        const int nq = (ns + L.group - 1) / L.group;
        for (int jq = wave; jq < nq * np; jq += kAdjWaves) {
            const int jp = jq / nq;
            const int j0 = (jq - jp * nq) * L.group, cnt = min(L.group, ns - j0);
            const long i0 = s0 + j0;
            PairParams pp;
            if constexpr (BATCH) {
                const BatchPair &q = L.pairs[jp];
                if (q.out < 0)
                    continue;   /* inert padding (uniform per wave) */
                pp = batch_pair_params(L.b, q);
                wave_samples(pp, ws, i0, cnt, q.pa_off, true, lane);
            } else {
                pp = p;
                wave_samples(p, ws, i0, cnt, 0.f, false, lane);
            }
            if (lane < cnt) {
                wtab[wave].g[lane][0] = pp.g_a ? pp.g_a[i0 + lane] : 0.f;
                wtab[wave].g[lane][1] = pp.g_b ? pp.g_b[i0 + lane] : 0.f;
            }
            wave_sync();
            float ga = 0.f, gb = 0.f;
            auto use = [&](const Pending &q) {
                float vI, vQ, vU;
                adj_visit_values(ga, gb, q.v0, q.v1, q.c2, q.s2, vI, vQ, vU);
                if (vI != 0.f || vQ != 0.f || vU != 0.f)
                    scatter(t.win[q.s], q.v, q.pix, vI, vQ, vU);
            };
            auto use_exact = [&](const Pending &q, int r, int sp, int g) {
                float vI, vQ, vU;
                adj_visit_values(wtab[wave].g[g][0], wtab[wave].g[g][1], q.v0, q.v1, q.c2, q.s2, vI,
                                 vQ, vU);
                scatter_pix(q.pix, r, sp, vI, vQ, vU);
            };
            auto after = [&](const Pass &ps) { fill_windows(t, ps, lane, kWaveSize); };
            int qn = 0;
            constexpr int F = WALK_BEAM | WALK_CHI;
            for (int j = 0; j < cnt; j++) {
                const SampleF sf = unif(ws.rec[j].sf);
                ga = unif(wtab[wave].g[j][0]);
                gb = unif(wtab[wave].g[j][1]);
                const int r0 = max(__builtin_amdgcn_readfirstlane(ws.rec[j].r_first), rlo);
                const int r1 = min(__builtin_amdgcn_readfirstlane(ws.rec[j].r_last), rhi);
                walk_rings<F>(pp, t, ws, j, r0, r1, lane, sf, kEtaAdjoint, qn, after, use,
                              use_exact);
            }
            if (qn > 0)
                drain_queue<F>(pp, ws, 0, qn, lane, use_exact);
            wave_sync();   /* the next samples' constants replace these */
        }
        }
        __syncthreads();

        /* flush the slab's window */
        if (!sfall) {
            for (int slot = tid; slot < W; slot += kAdjBlock) {
                float vI = 0.f, vQ = 0.f, vU = 0.f;
                unsigned long long fI = 0, fQ = 0, fU = 0;
                if constexpr (DET) {
                    fI = acc64[slot];
                    fQ = acc64[W + slot];
                    fU = acc64[2 * W + slot];
                    if ((fI | fQ | fU) == 0ull)
                        continue;
                } else {
                    vI = acc[slot];
                    vQ = acc[W + slot];
                    vU = acc[2 * W + slot];
                    if (vI == 0.f && vQ == 0.f && vU == 0.f)
                        continue;
                }
                int lo = k0, hi = k1;   /* win_base[lo] <= base0 + slot < win_base[hi] */
                while (hi - lo > 1) {
                    int mid = (lo + hi) >> 1;
                    if (win_base[mid] - base0 <= slot)
                        lo = mid;
                    else
                        hi = mid;
                }
                int sp, nr;
                bool shf;
                ring_info(p.hs, R0 + lo, sp, nr, shf);
                int ip = win_lo[lo] + (slot - (win_base[lo] - base0));
                if (ip >= nr)
                    ip -= nr;
                int pix = sp + ip;
                if constexpr (DET) {
                    if (fI)
                        atomicAdd((unsigned long long *)&p.gI[pix], fI);
                    if (fQ)
                        atomicAdd((unsigned long long *)&p.gQ[pix], fQ);
                    if (fU)
                        atomicAdd((unsigned long long *)&p.gU[pix], fU);
                } else {
                    if (vI != 0.f)
                        unsafeAtomicAdd(&p.gI[pix], (double)vI);
                    if (vQ != 0.f)
                        unsafeAtomicAdd(&p.gQ[pix], (double)vQ);
                    if (vU != 0.f)
                        unsafeAtomicAdd(&p.gU[pix], (double)vU);
                }
            }
        }
        __syncthreads();
        }   /* slabs */
    }
}

/* ---- beam adjoint in LDS bands --------------------------------------------
 *
 * The beam adjoint adds six values per visit to the visit's beam row.  With
 * global FP64 atomics that is bound by the atomic rate (every sample's disc
 * touches the whole beam support, so no short span of samples repeats a
 * row).  Here the beam rows are split into bands of `rows` consecutive rows
 * that fit the LDS; a work item is (band, chunk of samples).  A point in a
 * pixel of beam ring R lies between the centres of rings R-1 and R+1, so the
 * visits whose beam pixel falls in rows [lo, hi) of rings Rf..Rl have
 * rho in [theta(Rf-1), theta(Rl+1)]: the item walks only that annulus of each
 * sample's disc (annulus_ring), keeps the visits whose exact beam pixel is in
 * the band, sums their values in float in LDS and adds the band to the FP64
 * gradient once per item. */
constexpr int kBandRuns = 4 * kWaveSize;   /* <= 4 runs per ring, 64 rings per pass */

struct BandRunTable {
    int pref[kBandRuns + 1];
    int pix0[kBandRuns];
    int ring[kBandRuns];
    int spare[7];   /* room for eight 8-lane tables (SubBandTable<8>) in the same slot */
};

struct BeamBands {
    int rows;      /* rows per band */
    int nband;
    int chunk;     /* samples per work item */
    long nchunks;
};

__device__ inline int build_band_runs(const Hpx &hs, const Disc &dout, const Disc &din,
                                      bool inner, int r0, int lane, BandRunTable &t)
{
    const int r = r0 + lane;
    int p0[4] = {0, 0, 0, 0}, ln[4] = {0, 0, 0, 0};
    int ns = 0;
    if (r <= dout.r_last)
        ns = annulus_ring<true>(hs, dout, din, inner, r, p0, ln);
    int tot = 0;
#pragma unroll
    for (int k = 0; k < 4; k++)
        tot += k < ns ? ln[k] : 0;
    const int cnt_in = wave_incl_scan(ns, lane);
    const int tot_in = wave_incl_scan(tot, lane);
    const int cbase = cnt_in - ns;
    int off = tot_in - tot;
#pragma unroll
    for (int k = 0; k < 4; k++) {   /* constant indices keep p0, ln in registers */
        if (k < ns) {
            t.pix0[cbase + k] = p0[k];
            t.ring[cbase + k] = r;
            t.pref[cbase + k] = off;
            off += ln[k];
        }
    }
    const int nrun = __shfl(cnt_in, kWaveSize - 1, kWaveSize);
    const int total = __shfl(tot_in, kWaveSize - 1, kWaveSize);
    if (lane == 0)
        t.pref[nrun] = total;
    wave_sync();
    return total;
}

/* The walk of one annulus pass: FP64 certified mapping, software pipelined
 * as walk_segment; every load of the loop issued unconditionally.  use(q) is
 * called for each visit whose beam pixel lies in rows [lo, lo + nrow). */
template <typename Use>
__device__ inline void walk_band(const PairParams &p, const BandRunTable &t, int total, int lane,
                                 const Centre &c, double c2psi, double s2psi, int lo, int nrow,
                                 Use &use)
{
    if (total <= 0)
        return;
    int s = 0;
    int v = lane;
    if (v < total)
        while (v >= t.pref[s + 1])
            s++;
    RingRec rr = p.rings[t.ring[s]];
    __builtin_amdgcn_s_waitcnt(0);   /* the counter is 0 at the loop head */
    Pending q;
    q.live = false;
    for (int v0 = 0; v0 < total; v0 += kWaveSize, v += kWaveSize) {
        const bool act = v < total;
        const int pix = t.pix0[s] + (act ? v - t.pref[s] : 0);
        const int r = t.ring[s];
        const RingRec cur = rr;
        const int vn = v + kWaveSize;
        if (vn < total)
            while (vn >= t.pref[s + 1])
                s++;
        rr = p.rings[t.ring[s]];
        float c2, s2;
        const int bp = beam_pixel_f64(p.hb, p.fc64, c, c2psi, s2psi,
                                      ring_phi(p.hs, cur, r, pix), cur.cdp, cur.sdp, c2, s2);
        if (q.live)
            use(q);
        q.live = act && (unsigned)(bp - lo) < (unsigned)nrow;
        q.pix = pix;
        q.bp = bp;
        q.c2 = c2;
        q.s2 = s2;
        const float4 sv = p.sky4[q.live ? pix : 0];
        q.sI = sv.x;
        q.sQ = sv.y;
        q.sU = sv.z;
    }
    if (q.live)
        use(q);
}

/* Several samples per wave (64/SUB, SUB lanes each) for the band walks:
 * per (band, sample) the annulus holds few visits and its set-up is a long
 * dependent chain, so lane groups keep several chains in flight. */
template <int SUB>
struct SubBandTable {
    int pref[4 * SUB + 1];
    int pix0[4 * SUB];
    int ring[4 * SUB];
};

template <int SUB>
__device__ inline int build_band_sub(const Hpx &hs, const Disc &dout, const Disc &din, bool inner,
                                     int nrings, int ps, int sl, SubBandTable<SUB> &t)
{
    const int r = dout.r_first + ps * SUB + sl;
    int p0[4] = {0, 0, 0, 0}, ln[4] = {0, 0, 0, 0};
    int ns = 0;
    if (ps * SUB + sl < nrings)
        ns = annulus_ring<true>(hs, dout, din, inner, r, p0, ln);
    int tot = 0;
#pragma unroll
    for (int k = 0; k < 4; k++)
        tot += k < ns ? ln[k] : 0;
    const int cnt_in = seg_incl_scan<SUB>(ns, sl);
    const int tot_in = seg_incl_scan<SUB>(tot, sl);
    const int cbase = cnt_in - ns;
    int off = tot_in - tot;
#pragma unroll
    for (int k = 0; k < 4; k++) {   /* constant indices keep p0, ln in registers */
        if (k < ns) {
            t.pix0[cbase + k] = p0[k];
            t.ring[cbase + k] = r;
            t.pref[cbase + k] = off;
            off += ln[k];
        }
    }
    const int nrun = __shfl(cnt_in, SUB - 1, SUB);
    const int total = __shfl(tot_in, SUB - 1, SUB);
    if (sl == 0)
        t.pref[nrun] = total;
    wave_sync();
    return total;
}

/* walk_band for a lane group: its `total` visits SUB at a time, for wtot
 * (the wave's largest total) iterations' worth; a lane without a visit
 * computes the first visit of its run (or pixel 0 of ring 1) and discards
 * it. */
template <int SUB, typename Use>
__device__ inline void walk_band_sub(const PairParams &p, const SubBandTable<SUB> &t, int total,
                                     int wtot, int sl, const Centre &c, double c2psi,
                                     double s2psi, int lo, int nrow, Use &use)
{
    if (wtot <= 0)
        return;
    const bool any = total > 0;
    int s = 0;
    int v = sl;
    if (v < total)
        while (v >= t.pref[s + 1])
            s++;
    RingRec rr = p.rings[any ? t.ring[s] : 1];
    __builtin_amdgcn_s_waitcnt(0);   /* the counter is 0 at the loop head */
    Pending q;
    q.live = false;
    for (int v0 = 0; v0 < wtot; v0 += SUB, v += SUB) {
        const bool act = v < total;
        const int r = any ? t.ring[s] : 1;
        const int pix = any ? t.pix0[s] + (act ? v - t.pref[s] : 0) : 0;
        const RingRec cur = rr;
        const int vn = v + SUB;
        if (vn < total)
            while (vn >= t.pref[s + 1])
                s++;
        rr = p.rings[any ? t.ring[s] : 1];
        float c2, s2;
        const int bp = beam_pixel_f64(p.hb, p.fc64, c, c2psi, s2psi,
                                      ring_phi(p.hs, cur, r, pix), cur.cdp, cur.sdp, c2, s2);
        if (q.live)
            use(q);
        q.live = act && (unsigned)(bp - lo) < (unsigned)nrow;
        q.pix = pix;
        q.bp = bp;
        q.c2 = c2;
        q.s2 = s2;
        const float4 sv = p.sky4[q.live ? pix : 0];
        q.sI = sv.x;
        q.sQ = sv.y;
        q.sU = sv.z;
    }
    if (q.live)
        use(q);
}

template <int SUB>
__global__ __launch_bounds__(kBandBlock) void k_adjbeam_band_sub(PairParams p, BeamBands B)
{
    constexpr int G = kWaveSize / SUB;
    static_assert(sizeof(SubBandTable<SUB>) * G <= sizeof(BandRunTable),
                  "lane-group tables within the wave's run table");
    extern __shared__ __align__(16) unsigned char smem[];
    BandRunTable *tabs = (BandRunTable *)smem;
    float *acc = (float *)(tabs + kBandWaves);
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWaveSize);
    const int lane = tid % kWaveSize;
    const int grp = lane / SUB, sl = lane % SUB;
    SubBandTable<SUB> &t = ((SubBandTable<SUB> *)&tabs[wave])[grp];
    const long nitems = B.nchunks * B.nband;
    for (long it = xcd_remap(blockIdx.x, gridDim.x); it < nitems; it += gridDim.x) {
        const long ch = it / B.nband;
        const int k = (int)(it - ch * B.nband);
        const int lo = k * B.rows;
        const int nrow = min(p.npix_beam - lo, B.rows);
        bool inner;
        double r_in, c_in, r_out, c_out;
        band_annulus_radii(p.hb, p.rho_max, p.cos_rmax, lo, nrow, inner, r_in, c_in, r_out, c_out);
        for (int i = tid; i < 6 * nrow; i += kBandBlock)
            acc[i] = 0.f;
        __syncthreads();
        const long s0 = p.s_begin + ch * B.chunk;
        const long s1 = s0 + B.chunk < p.s_end ? s0 + B.chunk : p.s_end;
        for (long j0 = s0 + (long)wave * G; j0 < s1; j0 += (long)kBandWaves * G) {
            const long i = j0 + grp;
            const bool valid = i < s1;
            const long iv = valid ? i : j0;
            const float ga = valid && p.g_a ? p.g_a[iv] : 0.f;
            const float gb = valid && p.g_b ? p.g_b[iv] : 0.f;
            const Centre c = centre_make(p.ra[iv], p.dec[iv], p.pa[iv]);
            double s2psi, c2psi;
            pl_sincos(2.0 * c.psi, &s2psi, &c2psi);
            Disc dout, din;
            disc_setup(p.hs, kHalfPi - c.dec, c.ra, r_out, c_out, dout);
            if (inner)
                disc_setup(p.hs, kHalfPi - c.dec, c.ra, r_in, c_in, din);
            else
                din = dout;   /* not read */
            const bool work = valid && (ga != 0.f || gb != 0.f);
            const int nrings = work && dout.r_last >= dout.r_first ? dout.r_last - dout.r_first + 1
                                                                    : 0;
            auto use = [&](const Pending &q) {
                const float X = q.sQ * q.c2 + q.sU * q.s2;
                const float Y = -q.sQ * q.s2 + q.sU * q.c2;
                float *a = acc + 6 * (q.bp - lo);
                atomicAdd(&a[0], ga * q.sI);
                atomicAdd(&a[1], ga * X);
                atomicAdd(&a[2], ga * Y);
                atomicAdd(&a[3], gb * q.sI);
                atomicAdd(&a[4], -(gb * X));
                atomicAdd(&a[5], -(gb * Y));
            };
            const int npass = (group_max_uniform<SUB>(nrings) + SUB - 1) / SUB;
            for (int ps = 0; ps < npass; ps++) {
                const int total = build_band_sub<SUB>(p.hs, dout, din, inner, nrings, ps, sl, t);
                walk_band_sub<SUB>(p, t, total, group_max_uniform<SUB>(total), sl, c, c2psi, s2psi, lo,
                                   nrow, use);
                wave_sync();
            }
        }
        __syncthreads();
        for (int rr = tid; rr < nrow; rr += kBandBlock) {
            const float *a = acc + 6 * rr;
            double *g = p.gbeam + 8 * (long)(lo + rr);
#pragma unroll
            for (int m = 0; m < 6; m++)
                if (a[m] != 0.f)
                    unsafeAtomicAdd(&g[m], (double)a[m]);
        }
        __syncthreads();
    }
}

__global__ __launch_bounds__(kBandBlock) void k_adjbeam_band(PairParams p, BeamBands B)
{
    extern __shared__ __align__(16) unsigned char smem[];
    BandRunTable *tabs = (BandRunTable *)smem;
    float *acc = (float *)(tabs + kBandWaves);
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWaveSize);
    const int lane = tid % kWaveSize;
    BandRunTable &t = tabs[wave];
    const long nitems = B.nchunks * B.nband;
    for (long it = xcd_remap(blockIdx.x, gridDim.x); it < nitems; it += gridDim.x) {
        /* consecutive items: the bands of one chunk (its samples stay in L2) */
        const long ch = it / B.nband;
        const int k = (int)(it - ch * B.nband);
        const int lo = k * B.rows;
        const int nrow = min(p.npix_beam - lo, B.rows);
        /* the annulus of rows [lo, lo + nrow) */
        bool inner;
        double r_in, c_in, r_out, c_out;
        band_annulus_radii(p.hb, p.rho_max, p.cos_rmax, lo, nrow, inner, r_in, c_in, r_out,
                           c_out);
        for (int i = tid; i < 6 * nrow; i += kBandBlock)
            acc[i] = 0.f;
        __syncthreads();
        const long s0 = p.s_begin + ch * B.chunk;
        const long s1 = s0 + B.chunk < p.s_end ? s0 + B.chunk : p.s_end;
        for (long i = s0 + wave; i < s1; i += kBandWaves) {
            const float ga = unif(p.g_a ? p.g_a[i] : 0.f);
            const float gb = unif(p.g_b ? p.g_b[i] : 0.f);
            if (ga == 0.f && gb == 0.f)
                continue;   /* adds nothing (wave-uniform) */
            Centre c = centre_make(p.ra[i], p.dec[i], p.pa[i]);
            c.ra = uni(c.ra);
            c.dec = uni(c.dec);
            c.psi = uni(c.psi);
            c.cdc = uni(c.cdc);
            c.sdc = uni(c.sdc);
            double s2psi, c2psi;
            pl_sincos(2.0 * c.psi, &s2psi, &c2psi);
            c2psi = uni(c2psi);
            s2psi = uni(s2psi);
            Disc dout, din;
            disc_setup(p.hs, kHalfPi - c.dec, c.ra, r_out, c_out, dout);
            if (inner)
                disc_setup(p.hs, kHalfPi - c.dec, c.ra, r_in, c_in, din);
            else
                din = dout;   /* not read */
            auto use = [&](const Pending &q) {
                const float X = q.sQ * q.c2 + q.sU * q.s2;
                const float Y = -q.sQ * q.s2 + q.sU * q.c2;
                float *a = acc + 6 * (q.bp - lo);
                atomicAdd(&a[0], ga * q.sI);
                atomicAdd(&a[1], ga * X);
                atomicAdd(&a[2], ga * Y);
                atomicAdd(&a[3], gb * q.sI);
                atomicAdd(&a[4], -(gb * X));
                atomicAdd(&a[5], -(gb * Y));
            };
            for (int r0 = dout.r_first; r0 <= dout.r_last; r0 += kWaveSize) {
                const int total = build_band_runs(p.hs, dout, din, inner, r0, lane, t);
                walk_band(p, t, total, lane, c, c2psi, s2psi, lo, nrow, use);
                wave_sync();
            }
        }
        __syncthreads();
        /* add the band to the FP64 gradient */
        for (int rr = tid; rr < nrow; rr += kBandBlock) {
            const float *a = acc + 6 * rr;
            double *g = p.gbeam + 8 * (long)(lo + rr);
#pragma unroll
            for (int m = 0; m < 6; m++)
                if (a[m] != 0.f)
                    unsafeAtomicAdd(&g[m], (double)a[m]);
        }
        __syncthreads();
    }
}

/* ---- beam adjoint through visit records -----------------------------------
 *
 * The banded kernels above map each sample's annulus once per band of beam
 * rows and set up every (band, sample) pair.  Here each visit is mapped
 * twice, once per pass, and the gradient is formed from 16-byte visit
 * records, per chunk of samples:
 *  1. k_beamrec<false> (one wave per sample, the sky adjoint's walk and
 *     certified mapping) counts the sample's visits inside the beam per band
 *     of `rows` consecutive beam rows;
 *  2. k_band_scan + k_scan_excl: per band, the offsets of the samples' records
 *     within the band; the bands' starts;
 *  3. k_beamrec<true> maps the visits again and writes each one's record
 *     (row within the band | sample << kRecRowBits, I, X = Q c2 + U s2,
 *     Y = -Q s2 + U c2) into its band, within the range of the samples of
 *     its block;
 *  4. k_beamrec_sum: a block per (band, part: the records of a share of the
 *     chunk's samples) sums its records, times the cotangents of each
 *     record's sample, into the band's
 *     rows in LDS as 64-bit fixed-point integers, then adds them to its own
 *     FP64 partial rows (a (band, part) slice belongs to one block in every
 *     chunk: no global atomics).
 * k_beamrec_reduce adds the parts into the FP64 gradient at the end.
 * Integers because float atomic adds to random LDS addresses ran about ten
 * times slower than 64-bit integer ones here (6.8 against 1.0 ms per chunk
 * of 41,000 samples at the 5-degree, beam NSIDE 4096 shape); integer sums
 * also make the result independent of the order of the additions. */
struct BeamRec {
    unsigned key;   /* row within the band | sample within the chunk << kRecRowBits */
    float sI, X, Y;
};
constexpr int kRecRowBits = 13;
constexpr int kRecUnroll = 4;
constexpr int kRecWriteWaves = 8;   /* samples per block of the write pass (shared cursors) */
constexpr int kScanBlock = 1024;

/* In-place exclusive scan of x[0 .. n) (one block); x[n] receives the total. */
__global__ __launch_bounds__(kScanBlock) void k_scan_excl(long *x, long n)
{
    __shared__ long part[kScanBlock];
    const int t = threadIdx.x;
    const long seg = (n + kScanBlock - 1) / kScanBlock;
    const long a = std::min<long>(n, t * seg), b = std::min<long>(n, a + seg);
    long s = 0;
    for (long k = a; k < b; k++)
        s += x[k];
    part[t] = s;
    __syncthreads();
    for (int o = 1; o < kScanBlock; o <<= 1) {
        const long v = t >= o ? part[t - o] : 0;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    long run = part[t] - s;
    for (long k = a; k < b; k++) {
        const long v = x[k];
        x[k] = run;
        run += v;
    }
    if (t == kScanBlock - 1)
        x[n] = part[t];
}

/* Band and row of a beam pixel.  tile == 0: consecutive rows.  Otherwise a band
 * is a patch of the polar cap: `tile` rings by `tile` pixels of a quadrant (ring
 * i has i pixels per quadrant), block t of rings and column c <= t, numbered
 * 2 t (t + 1) + quadrant (t + 1) + c.  A sky pixel is several beam pixels, so
 * along a sky ring each visit is in another block of consecutive rows (1.5 outer
 * rings hold 3,400 pixels) and the 64 records of a wave went to 64 lines; of a
 * patch it crosses about seven visits at a time. */
__device__ inline int rec_band(const RecParams &R, int bp, int &row)
{
    if (R.tile == 0) {
        int b = (int)((float)bp * R.inv_rows);
        if (b * R.rows > bp)
            b--;
        else if ((b + 1) * R.rows <= bp)
            b++;
        row = bp - b * R.rows;
        return b;
    }
    /* ring i = 1, 2, ... starts at 2 i (i - 1); the estimate is off by at most 1 */
    int i = (int)(0.5f * (1.0f + __builtin_amdgcn_sqrtf(fmaf(2.0f, (float)bp, 1.0f))));
    int j = bp - 2 * i * (i - 1);
    if (j < 0) {
        i--;
        j += 4 * i;
    } else if (j >= 4 * i) {
        j -= 4 * i;
        i++;
    }
    const int q = (j >= i) + (j >= 2 * i) + (j >= 3 * i);
    j -= q * i;
    const int t = (int)(((float)i - 0.5f) * R.inv_tile);   /* (i - 1) / tile */
    const int c = (int)(((float)j + 0.5f) * R.inv_tile);
    row = (i - 1 - t * R.tile) * R.tile + (j - c * R.tile);
    return (2 * t + q) * (t + 1) + c;
}

/* The same from a visit's certified place: whole numbers in float. */
__device__ inline int rec_band(const RecParams &R, int bp, const CapPlace &e, int &row)
{
    if (R.tile == 0)
        return rec_band(R, bp, row);
    const float w = (float)R.tile;
    const float t = floorf((e.ring - 0.5f) * R.inv_tile), c = floorf((e.pos + 0.5f) * R.inv_tile);
    row = (int)fmaf(fmaf(-t, w, e.ring - 1.0f), w, fmaf(-c, w, e.pos));
    return (int)fmaf(fmaf(2.0f, t, e.quad), t + 1.0f, c);
}

/* The beam pixel of a row of band b, or -1 if it has none. */
__device__ inline int rec_pixel(const RecParams &R, int b, int row, int npix)
{
    int bp = b * R.rows + row;
    if (R.tile) {
        int t = (int)(0.5f * (__builtin_amdgcn_sqrtf(fmaf(2.0f, (float)b, 1.0f)) - 1.0f));
        t += 2 * (t + 1) * (t + 2) <= b;
        t -= 2 * t * (t + 1) > b;
        const int rem = b - 2 * t * (t + 1), q = rem / (t + 1), c = rem - q * (t + 1);
        const int u = row / R.tile, i = t * R.tile + u + 1, j = c * R.tile + (row - u * R.tile);
        bp = j < i ? 2 * i * (i - 1) + q * i + j : npix;
    }
    return bp < npix ? bp : -1;
}

/* Steps 1 and 3: one wave per sample of the chunk [p.s_begin, p.s_end),
 * the sky adjoint's walk and certified single-precision mapping (every
 * visit's beam pixel is the exact one; cos/sin 2chi within 1e-6), with the
 * deferred visits mapped by the FP64-alpha form.  The count pass loads no
 * beam rows; the write pass loads each visit's sky values, pipelined. */
template <bool WRITE>
__global__ __launch_bounds__(WRITE ? kRecWriteWaves * kWaveSize : kBlock)
__attribute__((amdgpu_waves_per_eu(4, 8)))
void k_beamrec(PairParams p, RecParams R)
{
    constexpr int NW = WRITE ? kRecWriteWaves : kWavesPerBlock;   /* waves (samples) per block */
    __shared__ WaveTable tables[NW];
    __shared__ WaveState<1> states[NW];
    /* counts: one row per wave (sample); write cursors: one row per block */
    __shared__ unsigned curs[WRITE ? 1 : NW][kRecMaxBands];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
    const int lane = threadIdx.x % kWaveSize;
    WaveTable &t = tables[wave];
    const long j0 = xcd_remap(blockIdx.x, gridDim.x) * NW;
    const long j = j0 + wave;
    const long i = p.s_begin + j;
    unsigned *cur;
    if constexpr (WRITE) {
        /* The block's samples j0 .. j0+NW-1 own adjacent ranges in every
         * band (the offsets are an exclusive scan over samples), so the
         * block fills each band's range through one shared cursor: a
         * 128-byte line of records is completed by the block's waves
         * together, while it is still in L2, instead of by one wave over
         * many iterations (partly written lines left L2 and doubled the
         * pass's HBM writes). */
        cur = curs[0];
        for (int b = threadIdx.x; b < R.nband; b += NW * kWaveSize)
            cur[b] = (unsigned)(R.bbase[b] + R.bcnt[b * R.chunk + j0]);
        __syncthreads();
        if (i >= p.s_end)
            return;
    } else {
        if (i >= p.s_end)
            return;
        cur = curs[wave];
        for (int b = lane; b < R.nband; b += kWaveSize)
            cur[b] = 0u;
        wave_sync();
    }
    const float ga = unif(p.g_a ? p.g_a[i] : 0.f);
    const float gb = unif(p.g_b ? p.g_b[i] : 0.f);
    if (ga != 0.f || gb != 0.f) {   /* else it adds nothing (wave-uniform) */
        auto &ws = states[wave];
        wave_samples(p, ws, i, 1, 0.f, false, lane);
        const SampleF sf = unif(ws.rec[0].sf);
        const int r0 = __builtin_amdgcn_readfirstlane(ws.rec[0].r_first);
        const int r1 = __builtin_amdgcn_readfirstlane(ws.rec[0].r_last);
        auto after = [](const Pass &) {};
        int qn = 0;
        if constexpr (WRITE) {
            const unsigned smp_key = (unsigned)j << kRecRowBits;
            auto put = [&](const Pending &q, int b, int row) {
                const unsigned slot = atomicAdd(&cur[b], 1u);
                if (slot >= (unsigned)R.nrec_cap)
                    return;   /* never: both passes count the same visits */
                BeamRec r;
                r.key = (unsigned)row | smp_key;
                r.sI = q.sI;
                r.X = fmaf(q.sQ, q.c2, q.sU * q.s2);
                r.Y = fmaf(q.sU, q.c2, -(q.sQ * q.s2));
                R.brec[slot] = r;
            };
            auto write = [&](const Pending &q) {
                int row;
                const int b = rec_band(R, q.bp, q.place, row);
                put(q, b, row);
            };
            auto write_exact = [&](const Pending &q, int, int, int) {
                int row;
                const int b = rec_band(R, q.bp, row);
                put(q, b, row);
            };
            constexpr int F = WALK_SKY | WALK_CHI | WALK_PLACE;
            walk_rings<F>(p, t, ws, 0, r0, r1, lane, sf, kEtaAdjoint, qn, after, write,
                          write_exact);
            if (qn > 0)
                drain_queue<F>(p, ws, 0, qn, lane, write_exact);
        } else {
            auto count = [&](const Pending &q) {
                int row;
                atomicAdd(&cur[rec_band(R, q.bp, q.place, row)], 1u);
            };
            auto count_exact = [&](const Pending &q, int, int, int) {
                int row;
                atomicAdd(&cur[rec_band(R, q.bp, row)], 1u);
            };
            walk_rings<WALK_PLACE>(p, t, ws, 0, r0, r1, lane, sf, kEtaAdjoint, qn, after, count,
                          count_exact);
            if (qn > 0)
                drain_queue<0>(p, ws, 0, qn, lane, count_exact);
        }
    }
    if constexpr (!WRITE) {
        wave_sync();
        for (int b = lane; b < R.nband; b += kWaveSize)
            R.bcnt[b * R.chunk + j] = cur[b];
    }
}

/* Step 2: per band (one block each), the exclusive offsets of the samples'
 * records within the band (in place) and the band's total in bbase[b].
 * Each thread scans kScanItems consecutive samples per round. */
constexpr int kScanItems = 16;
__global__ __launch_bounds__(kScanBlock) void k_band_scan(RecParams R, long nsamp)
{
    __shared__ long part[kScanBlock];
    const int b = blockIdx.x, t = threadIdx.x;
    long *x = R.bcnt + (long)b * R.chunk;
    long carry = 0;
    for (long r0 = 0; r0 < nsamp; r0 += (long)kScanBlock * kScanItems) {
        long v[kScanItems];
        long s = 0;
#pragma unroll
        for (int q = 0; q < kScanItems; q++) {
            const long k = r0 + (long)t * kScanItems + q;
            v[q] = k < nsamp ? x[k] : 0;
            s += v[q];
        }
        part[t] = s;
        __syncthreads();
        for (int o = 1; o < kScanBlock; o <<= 1) {
            const long w = t >= o ? part[t - o] : 0;
            __syncthreads();
            part[t] += w;
            __syncthreads();
        }
        long run = carry + part[t] - s;
#pragma unroll
        for (int q = 0; q < kScanItems; q++) {
            const long k = r0 + (long)t * kScanItems + q;
            if (k < nsamp)
                x[k] = run;
            run += v[q];
        }
        carry += part[kScanBlock - 1];
        __syncthreads();
    }
    if (t == 0)
        R.bbase[b] = carry;
}

/* Step 4: block (band, part) of nsplit.  Each value v = g * (I, X or Y) is
 * rounded once to a multiple of 2^-k and summed as a 64-bit integer, with k
 * the largest integer such that the block's records, each |v| <= gmax *
 * smax * (1 + 1e-3), cannot sum past 2^62 in magnitude. */
__global__ __launch_bounds__(kBandBlock) void k_beamrec_sum(PairParams p, RecParams R)
{
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned long long *acc = (unsigned long long *)smem;
    const int tid = threadIdx.x;
    const int b = blockIdx.x / R.nsplit, part = blockIdx.x % R.nsplit;
    const int nrow = R.tile ? R.rows : min(p.npix_beam - b * R.rows, R.rows);
    const long r0 = R.bbase[b], cnt = R.bbase[b + 1] - r0;
    /* the part's samples: a share of the chunk's, cut at multiples of the
     * write pass's samples per block, so that the records of a part are the
     * same set however the block's waves interleaved them */
    const long ns = p.s_end - p.s_begin;
    const long sa = (ns * part / R.nsplit) / kRecWriteWaves * kRecWriteWaves;
    const long sb = part + 1 == R.nsplit
                        ? ns
                        : (ns * (part + 1) / R.nsplit) / kRecWriteWaves * kRecWriteWaves;
    const long k0 = sa < ns ? R.bcnt[b * R.chunk + sa] : cnt;
    const long j1 = sb < ns ? R.bcnt[b * R.chunk + sb] : cnt;
    if (k0 >= j1)
        return;   /* no records (uniform per block) */
    const double vmax = (double)R.vmax[0] * (double)R.vmax[1] * (1.0 + 1e-3);
    if (!(vmax > 0.0))
        return;   /* every value is zero */
    /* every sum below 2^62 and (for fix64) every single value below 2^50 */
    const int e = (int)std::ceil(std::log2((double)(j1 - k0) * vmax));
    const double scale = std::ldexp(1.0, std::min(62 - e, 49 - ilogb(vmax)));
    for (int k = tid; k < 6 * nrow; k += kBandBlock)
        acc[k] = 0ull;
    __syncthreads();
    /* an absent cotangent reads the other one and adds zeros (with neither
     * there are no records) */
    const bool has_a = p.g_a != nullptr, has_b = p.g_b != nullptr;
    const float *gA = has_a ? p.g_a : p.g_b, *gB = has_b ? p.g_b : p.g_a;
    if (gA == nullptr)
        return;
    /* records of the next batch are loaded while the current one is summed */
    BeamRec nx[kRecUnroll];
#pragma unroll
    for (int u = 0; u < kRecUnroll; u++) {
        const long k = k0 + u * kBandBlock + tid;
        nx[u] = R.brec[r0 + (k < j1 ? k : k0)];
    }
    for (long kk = k0; kk < j1; kk += (long)kRecUnroll * kBandBlock) {
        BeamRec r[kRecUnroll];
        float ga[kRecUnroll], gb[kRecUnroll];
#pragma unroll
        for (int u = 0; u < kRecUnroll; u++) {
            const long k = kk + u * kBandBlock + tid;
            r[u] = nx[u];
            if (k >= j1)
                r[u].sI = r[u].X = r[u].Y = 0.f;   /* adds zeros */
        }
        /* the cotangents first, then the prefetch: loads complete in order,
         * so waiting for the cotangents does not wait for the prefetch */
#pragma unroll
        for (int u = 0; u < kRecUnroll; u++) {
            const long i = p.s_begin + (long)(r[u].key >> kRecRowBits);
            const float a = gA[i], bb = gB[i];   /* unconditional: no branch between loads */
            ga[u] = has_a ? a : 0.f;
            gb[u] = has_b ? bb : 0.f;
        }
#pragma unroll
        for (int u = 0; u < kRecUnroll; u++) {
            const long kn = kk + u * kBandBlock + tid + (long)kRecUnroll * kBandBlock;
            nx[u] = R.brec[r0 + (kn < j1 ? kn : k0)];
        }
#pragma unroll
        for (int u = 0; u < kRecUnroll; u++) {
            unsigned long long *a = acc + 6 * (int)(r[u].key & ((1u << kRecRowBits) - 1));
            const float v[6] = {ga[u] * r[u].sI, ga[u] * r[u].X,    ga[u] * r[u].Y,
                                gb[u] * r[u].sI, -(gb[u] * r[u].X), -(gb[u] * r[u].Y)};
#pragma unroll
            for (int m = 0; m < 6; m++)
                if (v[m] != 0.f)
                    atomicAdd(&a[m], fix64(v[m], scale));
        }
    }
    __syncthreads();
    const double inv = 1.0 / scale;
    double *dst = R.part + (long)part * p.npix_beam * 6;
    if (R.tile == 0) {
        dst += (long)b * R.rows * 6;
        for (int k = tid; k < 6 * nrow; k += kBandBlock)
            dst[k] += (double)(long long)acc[k] * inv;
        return;
    }
    for (int k = tid; k < 6 * nrow; k += kBandBlock) {
        const int row = k / 6, bp = rec_pixel(R, b, row, p.npix_beam);
        if (bp >= 0)
            dst[6 * (long)bp + (k - 6 * row)] += (double)(long long)acc[k] * inv;
    }
}

/* The parts' sums into the FP64 gradient (rows of eight, columns 0..5), in
 * part order. */
__global__ void k_beamrec_reduce(const double *part, int nsplit, long npix, double *gbeam)
{
    long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    for (; k < 6 * npix; k += (long)gridDim.x * blockDim.x) {
        double s = 0.0;
        for (int q = 0; q < nsplit; q++)
            s += part[(long)q * 6 * npix + k];
        const long row = k / 6;
        gbeam[8 * row + (k - 6 * row)] += s;
    }
}

/* Blocks of the maxima over long arrays: an atomic to one address takes about
 * 12 ns, so each block makes one per maximum (one per wave of 8,192 blocks took
 * 0.37 ms over 3.8e6 floats). */
constexpr int kMaxBlocks = 512;

/* The block's maximum of v >= 0 onto *out, as float bits.  Every thread of a
 * block of at most 1024 calls it. */
__device__ inline void block_max(float v, unsigned *out)
{
    __shared__ float part[16];
#pragma unroll
    for (int m = kWaveSize / 2; m > 0; m >>= 1)
        v = fmaxf(v, __shfl_xor(v, m, kWaveSize));
    __syncthreads();   /* part may be in use by a call before */
    if (threadIdx.x % kWaveSize == 0)
        part[threadIdx.x / kWaveSize] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < (int)blockDim.x / kWaveSize; w++)
            v = fmaxf(v, part[w]);
        if (v > 0.f)
            atomicMax(out, __float_as_uint(v));
    }
}

/* vmax[0] = max |g_a|, |g_b| over the samples; vmax[1] = max over sky
 * pixels of max(|I|, |Q| + |U|) (bounds |I|, |X| and |Y| of every record).
 * vmax must hold zeros on entry; non-negative floats order as their bits. */
__global__ void k_rec_vmax(PairParams p, float *vmax)
{
    float g = 0.f, sk = 0.f;
    long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long n = p.s_end - p.s_begin, stride = (long)gridDim.x * blockDim.x;
    for (long j = k; j < n; j += stride) {
        if (p.g_a)
            g = fmaxf(g, fabsf(p.g_a[p.s_begin + j]));
        if (p.g_b)
            g = fmaxf(g, fabsf(p.g_b[p.s_begin + j]));
    }
    for (long j = k; j < p.hs.npix; j += stride) {
        const float4 v = p.sky4[j];
        sk = fmaxf(sk, fmaxf(fabsf(v.x), fabsf(v.y) + fabsf(v.z)));
    }
    block_max(g, (unsigned *)&vmax[0]);
    block_max(sk, (unsigned *)&vmax[1]);
}

__global__ void k_fill_f64_n(double *x, long n)
{
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (long)gridDim.x * blockDim.x)
        x[i] = 0.0;
}

__global__ void k_fill_i32(int *x, int v) { *x = v; }

/* Last row with a non-zero value in columns 0..5 (block max, one atomic
 * per block). */
__global__ void k_beam_support(const float4 *beam8, long npix, int *last)
{
    __shared__ int part[16];
    int best = -1;
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < npix; i += (long)gridDim.x * blockDim.x) {
        float4 a = beam8[2 * i];
        float4 b = beam8[2 * i + 1];
        if (a.x != 0.f || a.y != 0.f || a.z != 0.f || a.w != 0.f || b.x != 0.f || b.y != 0.f)
            best = (int)i;
    }
#pragma unroll
    for (int m = kWaveSize / 2; m > 0; m >>= 1)
        best = max(best, __shfl_xor(best, m, kWaveSize));
    if (threadIdx.x % kWaveSize == 0)
        part[threadIdx.x / kWaveSize] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < (int)blockDim.x / kWaveSize; w++)
            best = max(best, part[w]);
        if (best >= 0)
            atomicMax(last, best);
    }
}

/* Ring records of every ring, indexed by ring number 1 .. 4N-1 (entry 0
 * unused). */
__global__ void k_ring_table(Hpx h, RingRec *out)
{
    int r = blockIdx.x * blockDim.x + threadIdx.x + 1;
    if (r >= 4 * h.nside)
        return;
    out[r] = ring_record(h, r);
}

__global__ void k_fill_f64(double *x, long n)
{
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (long)gridDim.x * blockDim.x)
        x[i] = 0.0;
}

__global__ void k_add_offset(const float *x, float off, float *y, long n)
{
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (long)gridDim.x * blockDim.x)
        y[i] = x[i] + off;
}

__global__ void k_pack_sky(const float *I, const float *Q, const float *U, const float *V, long n,
                           float4 *out)
{
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (long)gridDim.x * blockDim.x)
        out[i] = make_float4(I[i], Q[i], U[i], V ? V[i] : 0.f);
}

/* Deterministic sky adjoint: out[0] = max over beam rows of the sum of |A0
 * A1 A2 B0 B1 B2|, out[1] = max |g| (as float bits; atomicMax on the bits of
 * non-negative floats orders them as the values).  gridDim.y: the beams. */
__global__ void k_absmax(FixSource f, unsigned *out)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long stride = (long)gridDim.x * blockDim.x;
    const float *beam8 = f.beam8;
    long npix = f.npix;
    if (f.pairs) {
        const BatchPair &q = f.pairs[blockIdx.y];
        beam8 = q.beam;
        npix = q.out < 0 ? 0 : q.npix;   /* inert padding */
    }
    float rows = 0.f, g = 0.f;
    for (long i = t; i < npix; i += stride) {
        const float4 r = *(const float4 *)(beam8 + 8 * i);
        const float2 s = *(const float2 *)(beam8 + 8 * i + 4);
        rows = fmaxf(rows, fabsf(r.x) + fabsf(r.y) + fabsf(r.z) + fabsf(r.w) + fabsf(s.x) +
                               fabsf(s.y));
    }
    for (long i = blockIdx.y * stride + t; i < f.n; i += gridDim.y * stride) {
        if (f.g_a)
            g = fmaxf(g, fabsf(f.g_a[i]));
        if (f.g_b)
            g = fmaxf(g, fabsf(f.g_b[i]));
    }
    block_max(rows, out);
    block_max(g, out + 1);
}

/* scale = 2^k, the largest power of two with count * bound * scale <= 2^62,
 * bound = max row sum * max |g| (the largest |contribution| of a visit) and
 * count the most contributions one pixel can receive (one per sample and
 * pair); every pixel's sum then fits a signed 64-bit integer. */
__global__ void k_fix_scale(const unsigned *m, long count, double *scale)
{
    const double one = (double)__uint_as_float(m[0]) * (double)__uint_as_float(m[1]);
    const double bound = one * (double)(count > 0 ? count : 1);
    double s = 1.0;
    if (bound > 0.0 && bound < INFINITY) {
        /* every sum below 2^62, and (for fix64) every single value below
         * 2^50: one value is at most m[0] m[1] */
        int k = min(62 - ilogb(bound) - 1, 49 - ilogb(one));
        k = k > 1000 ? 1000 : (k < -1000 ? -1000 : k);
        s = ldexp(1.0, k);
    }
    *scale = s;
}

__global__ void k_fix_to_f32(const unsigned long long *x, const double *scale, F32Planes y, long n)
{
    const double inv = 1.0 / *scale;
    float *out = y.p[blockIdx.y];
    x += blockIdx.y * n;
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (long)gridDim.x * blockDim.x)
        out[i] = (float)((double)(long long)x[i] * inv);
}

__global__ void k_fill_u32(unsigned *x, int n, unsigned v)
{
    if ((int)threadIdx.x < n)
        x[threadIdx.x] = v;
}

__global__ void k_f64_to_f32(const double *x, float *y, long n)
{
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (long)gridDim.x * blockDim.x)
        y[i] = (float)x[i];
}

/* eight float maps -> rows A0 A1 A2 B0 B1 B2 A3 B3 */
__global__ void k_pack_beam(long npix, const float *a0, const float *a1, const float *a2,
                            const float *a3, const float *b0, const float *b1,
                            const float *b2, const float *b3, float4 *out)
{
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < npix; i += (long)gridDim.x * blockDim.x) {
        out[2 * i] = make_float4(a0[i], a1[i], a2[i], b0[i]);
        out[2 * i + 1] = make_float4(b1[i], b2[i], a3 ? a3[i] : 0.f, b3 ? b3[i] : 0.f);
    }
}

/* ---- test kernels: the HEALPix and matching primitives on their own ---- */

__global__ void k_pix2ang(Hpx h, long n, const int *pix, double *th, double *ph)
{
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (long)gridDim.x * blockDim.x)
        pix2ang(h, pix[i], th[i], ph[i]);
}

__global__ void k_ang2pix(Hpx h, long n, const double *th, const double *ph, int *pix)
{
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (long)gridDim.x * blockDim.x)
        pix[i] = ang2pix(h, th[i], ph[i]);
}

__global__ void k_interpol(Hpx h, long n, const double *th, const double *ph, int *pix,
                           double *wgt)
{
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (long)gridDim.x * blockDim.x)
        get_interpol(h, th[i], ph[i], pix + 4 * i, wgt + 4 * i);
}

/* Disc of each pointing, one thread per pointing: count (pixels == NULL) or
 * fill pixels at offsets[i]. */
__global__ void k_disc(Hpx h, long n, const float *ra, const float *dec, double radius,
                       double cosr, const long *offsets, int *counts, int *pixels)
{
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    Centre c = centre_make(ra[i], dec[i], 0.f);
    Disc d;
    disc_setup(h, kHalfPi - c.dec, c.ra, radius, cosr, d);
    long k = pixels ? offsets[i] : 0;
    int cnt = 0;
    for (int r = d.r_first; r <= d.r_last; r++) {
        int p0[2] = {0, 0}, ln[2] = {0, 0};
        int ns = disc_ring(h, d, r, p0, ln);
#pragma unroll
        for (int j = 0; j < 2; j++) {
            if (j < ns) {
                if (pixels)
                    for (int q = 0; q < ln[j]; q++)
                        pixels[k + cnt + q] = p0[j] + q;
                cnt += ln[j];
            }
        }
    }
    if (counts)
        counts[i] = cnt;
}

/* Sky pixel -> (beam pixel, chi) for pixel lists laid out as offsets/pixels
 * (the quantity kernel 1 of the reference computes, cudaConv2.cu:59-128).
 * mode 0: the exact FP64 mapping, chi[k] = chi.
 * mode 1: what the adjoint kernels use: the float form, and the FP64 form
 *         where the float form cannot certify the pixel; chi[k] receives
 *         float cos(2chi), sin(2chi) packed as two floats.
 * mode 2: the float form alone; bpix[k] = kNeedExact (-2) where it declines.
 * mode 3: the FP64 form of the deferred-visit drain (output as mode 1).
 * modes 4, 5: as 1 and 2 with the bound of the forward and of the sky adjoint
 *         with lane groups for cos(2chi), sin(2chi) in float.
 * mode 6: the batched kernels' float form alone (as mode 2; chi as mode 5). */
__global__ void k_match(Hpx hs, const RingRec *rings, Hpx hb, FastConsts fc, FastConsts64 fc64,
                        int mode, long n,
                        const float *ra, const float *dec, const float *pa,
                        const long *offsets, const int *pixels, int *bpix, double *chi)
{
    long i = (long)blockIdx.x;
    if (i >= n)
        return;
    const Centre c = centre_make(ra[i], dec[i], pa[i]);
    double spsi, cpsi;
    pl_sincos(c.psi, &spsi, &cpsi);
    const double c2psi = fma(cpsi, cpsi, -(spsi * spsi)), s2psi = 2.0 * (spsi * cpsi);
    const SampleF sf = sample_f32(c, cpsi, spsi, c2psi, s2psi);
    for (long k = offsets[i] + threadIdx.x; k < offsets[i + 1]; k += blockDim.x) {
        int pix = pixels[k];
        int r = pix2ring(hs, pix);
        RingRec rr = rings[r];
        if (mode > 0) {
            float c2 = 0.f, s2 = 0.f;
            const double ra_pix = ring_phi(hs, rr, r, pix);
            int bp = kNeedExact;
            if (mode != 3) {
                const int j = pix - rr.startpix;
                const RunGeo g = run_geo(hs, rr, r, c, j, 1);
                const float x = fmaf((float)(j - g.kc), g.b, g.a0);
                const VisitGeo v = visit_geo(x, g.sD, g.omD, g.cdp2, sf.cdc, sf.sdc);
                CapPlace place;
                bp = mode == 6 ? pair_pixel(visit_alpha(v), __builtin_amdgcn_sqrtf(3.0f * v.omc),
                                            v.omc, pair_t0(c.psi), (float)hb.nside, sf.lim0, place)
                               : visit_pixel(fc, sf, v, place);
                float d4, s4;
                visit_phase(v, g.kap, d4, s4);
                if (!(fabsf(g.kap * x) < (mode >= 4 ? kEtaForward : kEtaAdjoint)) ||
                    fabsf(x) > 0.7f)
                    visit_phase64(c, ra_pix, rr.cdp, rr.sdp, d4, s4);
                visit_chi(sf, d4, s4, c2, s2);
            }
            if (bp == kNeedExact && (mode == 1 || mode == 3 || mode == 4))
                bp = beam_pixel_f64(hb, fc64, c, c2psi, s2psi, ra_pix, rr.cdp, rr.sdp, c2, s2);
            bpix[k] = bp;
            float2 *o = (float2 *)&chi[k];
            *o = make_float2(c2, s2);
        } else {
            int sp, nr;
            bool sh;
            ring_info(hs, r, sp, nr, sh);
            double ra_pix = pixel_phi(hs, r, pix, sp);
            double x;
            bpix[k] = beam_pixel(hb, c, ra_pix, rr.cdp, rr.sdp, x);
            chi[k] = x;
        }
    }
}

/* Element-wise FP64 primitives, for checking host/device bit equality. */
__global__ void k_libm(int op, long n, const double *x, const double *y, double *o)
{
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (long)gridDim.x * blockDim.x) {
        double a = x[i], b = y ? y[i] : 0.0, r = 0.0;
        switch (op) {
        case 0: r = pl_sin(a); break;
        case 1: r = pl_cos(a); break;
        case 2: r = pl_acos(a); break;
        case 3: r = pl_atan2(a, b); break;
        case 4: r = sqrt(a); break;
        case 5: r = a / b; break;
        case 6: r = fmodulo(a, b); break;
        case 7: { double s, c; pl_sincos(a, &s, &c); r = s + 2.0 * c; } break;
        case 8: r = __longlong_as_double((long long)fix64((float)a, b)); break;
        default: r = 0.0;
        }
        o[i] = r;
    }
}

/* ---- launchers ---------------------------------------------------------- */

static inline unsigned nblocks(long n, int per)
{
    long b = (n + per - 1) / per;
    if (b < 1)
        b = 1;
    return (unsigned)b;
}

static inline unsigned gs_blocks(long n)
{
    long b = (n + 255) / 256;
    if (b > 8192)
        b = 8192;
    if (b < 1)
        b = 1;
    return (unsigned)b;
}

hipError_t launch_pair(int op, const PairParams &p, hipStream_t st)
{
    long n = p.s_end - p.s_begin;
    if (n <= 0)
        return hipSuccess;
    unsigned g = nblocks(n, kWavesPerBlock);
    switch (op) {
    case OP_ADJ_MAP: hipLaunchKernelGGL(k_pair<OP_ADJ_MAP>, dim3(g), dim3(kBlock), 0, st, p); break;
    case OP_ADJ_BEAM: hipLaunchKernelGGL(k_pair<OP_ADJ_BEAM>, dim3(g), dim3(kBlock), 0, st, p); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int SUB>
static void launch_fwd_lanes(const PairParams &p, hipStream_t st, bool vterm)
{
    constexpr int NS = FwdBlock<SUB>::NS;
    const long n = p.s_end - p.s_begin;
    const unsigned nb = (unsigned)work_items(nblocks(n, NS), p.strips);
    if (vterm)
        hipLaunchKernelGGL((k_fwd_sub<SUB, true>), dim3(nb), dim3(kBlock), 0, st, p);
    else
        hipLaunchKernelGGL((k_fwd_sub<SUB, false>), dim3(nb), dim3(kBlock), 0, st, p);
}

hipError_t launch_forward(int lanes, const PairParams &p0, hipStream_t st, bool vterm)
{
    const long n = p0.s_end - p0.s_begin;
    if (n <= 0)
        return hipSuccess;
    PairParams p = p0;
    if (lanes != kWaveSize)
        p.strips = 1;
    if (p.strips > 1 && !p.samples) {
        const dim3 g(nblocks(n, FwdBlock<kWaveSize>::NS));
        if (vterm)
            hipLaunchKernelGGL(k_fwd_strips<true>, g, dim3(kBlock), 0, st, p);
        else
            hipLaunchKernelGGL(k_fwd_strips<false>, g, dim3(kBlock), 0, st, p);
        return hipGetLastError();
    }
    if (p.strips > 1)
        hipLaunchKernelGGL(k_samples, dim3(nblocks(n, 64)), dim3(64), 0, st, p);
    switch (lanes) {
    case 8: launch_fwd_lanes<8>(p, st, vterm); break;
    case 16: launch_fwd_lanes<16>(p, st, vterm); break;
    case 32: launch_fwd_lanes<32>(p, st, vterm); break;
    case 64: launch_fwd_lanes<64>(p, st, vterm); break;
    default: return hipErrorInvalidValue;
    }
    if (p.strips > 1)
        hipLaunchKernelGGL(k_strip_sum, dim3(gs_blocks(n)), dim3(256), 0, st, p);
    return hipGetLastError();
}

hipError_t launch_pair_interp(int op, const PairParams &p, hipStream_t st)
{
    long n = p.s_end - p.s_begin;
    if (n <= 0)
        return hipSuccess;
    unsigned g = nblocks(n, kWavesPerBlock);
    switch (op) {
    case OP_FWD: hipLaunchKernelGGL(k_pair_interp<OP_FWD>, dim3(g), dim3(kBlock), 0, st, p); break;
    case OP_ADJ_MAP:
        hipLaunchKernelGGL(k_pair_interp<OP_ADJ_MAP>, dim3(g), dim3(kBlock), 0, st, p);
        break;
    case OP_ADJ_BEAM:
        hipLaunchKernelGGL(k_pair_interp<OP_ADJ_BEAM>, dim3(g), dim3(kBlock), 0, st, p);
        break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int SUB>
static void launch_batch_pairs(const BatchParams &p, long n, hipStream_t st)
{
    constexpr int NS = FwdBlock<SUB>::NS;
    hipLaunchKernelGGL(k_batch_pair<SUB>, dim3((unsigned)work_items((n + NS - 1) / NS, p.npairs)),
                       dim3(kBlock), 0, st, p);
}

hipError_t launch_batch_forward(int group, const BatchParams &p, hipStream_t st, int lanes)
{
    const long n = p.s_end - p.s_begin;
    if (n <= 0)
        return hipSuccess;
    const unsigned g = nblocks(work_items(n, p.ngroups), kWavesPerBlock);
    switch (group) {
    case 1:
        switch (lanes) {
        case 8: launch_batch_pairs<8>(p, n, st); break;
        case 16: launch_batch_pairs<16>(p, n, st); break;
        case 32: launch_batch_pairs<32>(p, n, st); break;
        case 64: launch_batch_pairs<64>(p, n, st); break;
        default: return hipErrorInvalidValue;
        }
        break;
    case 2: hipLaunchKernelGGL(k_batch_fwd<2>, dim3(g), dim3(kBlock), 0, st, p); break;
    case 4: hipLaunchKernelGGL(k_batch_fwd<4>, dim3(g), dim3(kBlock), 0, st, p); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

/* The limits of cap and rw allow for the tables. */
static_assert(sizeof(AdjWave<0, kWaveSize>) * kAdjWaves <= kAdjTableBytes);
size_t adjmap_lds_bytes(int cap, int rw, int group, bool det, int lanes)
{
    const size_t wt = group == 2   ? sizeof(AdjWave<2, kWaveSize>)
                      : group == 4 ? sizeof(AdjWave<4, kWaveSize>)
                      : lanes == 8 ? sizeof(AdjWave<0, 8>)
                      : lanes == 16 ? sizeof(AdjWave<0, 16>)
                                    : sizeof(AdjWave<0, kWaveSize>);
    return wt * kAdjWaves + sizeof(int) * (3 * (size_t)rw + 1 + kAdjCtl) +
           (det ? 8 + 8 * 3 * (size_t)cap : sizeof(float) * 3 * (size_t)cap);
}

/* Raises the dynamic-LDS limit of kernel fn on the current device to at
 * least `bytes`.  `configured[dev]` holds the largest limit set so far for
 * that kernel and device, so a later launch that needs more LDS than an
 * earlier one raises the limit again (it is never lowered). */
constexpr int kDevs = 64;
static hipError_t ensure_dyn_lds(const void *fn, size_t bytes, std::atomic<size_t> *configured)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess)
        return e;
    if (dev >= 0 && dev < kDevs && bytes <= configured[dev].load())
        return hipSuccess;
    e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    if (e != hipSuccess)
        return e;
    if (dev >= 0 && dev < kDevs) {
        size_t cur = configured[dev].load();
        while (bytes > cur && !configured[dev].compare_exchange_weak(cur, bytes)) {
        }
    }
    return hipSuccess;
}

template <int BG, bool DET, int SUB = kWaveSize>
static hipError_t launch_adjmap_bg(const PairParams &p, const AdjLayout &L, size_t bytes,
                                   long g, hipStream_t st)
{
    static std::atomic<size_t> configured[kDevs];
    hipError_t e = ensure_dyn_lds((const void *)k_adjmap_lds<BG, DET, SUB>, bytes, configured);
    if (e != hipSuccess)
        return e;
    hipLaunchKernelGGL((k_adjmap_lds<BG, DET, SUB>), dim3((unsigned)g), dim3(kAdjBlock), bytes, st,
                       p, L);
    return hipGetLastError();
}

hipError_t launch_adjmap_lds(const PairParams &p, int chunk, int cap, int rw, int nblocks,
                             hipStream_t st, const BatchParams *batch, double rho_w, int group,
                             const double *fx_scale, int lanes)
{
    long n = p.s_end - p.s_begin;
    if (n <= 0)
        return hipSuccess;
    AdjLayout L;
    memset(&L, 0, sizeof L);
    L.chunk = chunk;
    L.cap = cap;
    L.rw = rw;
    L.group = std::max(1, std::min(kAdjSamples, chunk / kAdjWaves));
    L.nchunks = (n + chunk - 1) / chunk;
    L.strips = 1;
    L.strip_group = 1;
    if (p.samples) {
        L.strips = p.strips;
        L.strip_group = std::max(1, kStripChunk / chunk);
        hipLaunchKernelGGL(k_samples, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, st, p);
    }
    if (batch) {
        L.pairs = batch->pairs;
        L.npairs = batch->npairs;
        L.rho_w = rho_w;
        L.cos_w = pl_cos(rho_w);
        L.b = *batch;
    }
    const int bg = batch ? group : 0;
    const bool det = fx_scale != nullptr;
    L.fx_scale = fx_scale;
    const size_t bytes = adjmap_lds_bytes(cap, rw, bg, det, bg == 0 ? lanes : kWaveSize);
    /* nblocks 0: one block per window.  Blocks start in index order, so the
     * windows in flight on an XCD stay consecutive in the scan; persistent
     * blocks (one per CU) drift apart over the launch, and measured 10%
     * slower on the 5-degree, NSIDE 512 sky adjoint. */
    const long g = nblocks > 0 ? std::min<long>(adj_items(L), nblocks) : adj_items(L);
    if (bg == 0 && lanes != kWaveSize) {   /* several samples per wave */
        switch (lanes) {
        case 8:
            return det ? launch_adjmap_bg<0, true, 8>(p, L, bytes, g, st)
                       : launch_adjmap_bg<0, false, 8>(p, L, bytes, g, st);
        case 16:
            return det ? launch_adjmap_bg<0, true, 16>(p, L, bytes, g, st)
                       : launch_adjmap_bg<0, false, 16>(p, L, bytes, g, st);
        default: return hipErrorInvalidValue;
        }
    }
    if (det) {
        switch (bg) {
        case 0: return launch_adjmap_bg<0, true>(p, L, bytes, g, st);
        case 1: return launch_adjmap_bg<1, true>(p, L, bytes, g, st);
        case 2: return launch_adjmap_bg<2, true>(p, L, bytes, g, st);
        case 4: return launch_adjmap_bg<4, true>(p, L, bytes, g, st);
        default: return hipErrorInvalidValue;
        }
    }
    switch (bg) {
    case 0: return launch_adjmap_bg<0, false>(p, L, bytes, g, st);
    case 1: return launch_adjmap_bg<1, false>(p, L, bytes, g, st);
    case 2: return launch_adjmap_bg<2, false>(p, L, bytes, g, st);
    case 4: return launch_adjmap_bg<4, false>(p, L, bytes, g, st);
    default: return hipErrorInvalidValue;
    }
}

int adjbeam_band_rows()
{
    return (int)((163840 - sizeof(BandRunTable) * kBandWaves) / (6 * sizeof(float)));
}

hipError_t launch_adjbeam_bands(const PairParams &p, int chunk, int rows, int nblocks, int ncu,
                                int lanes, hipStream_t st)
{
    const long n = p.s_end - p.s_begin;
    if (n <= 0 || p.npix_beam <= 0)
        return hipSuccess;
    if (chunk < 1)
        return hipErrorInvalidValue;
    BeamBands B;
    B.rows = adjbeam_band_rows();
    if (rows > 0 && rows < B.rows)
        B.rows = rows;
    B.rows = std::min<long>(B.rows, p.npix_beam);   /* no LDS for rows past the beam */
    B.nband = (p.npix_beam + B.rows - 1) / B.rows;
    /* smaller items when there are too few to give every block two */
    const long fill = n * B.nband / (2L * std::max(ncu, 1));
    B.chunk = (int)std::max<long>(std::min<long>(chunk, std::max<long>(fill, 64)), 1);
    B.nchunks = (n + B.chunk - 1) / B.chunk;
    const size_t bytes = sizeof(BandRunTable) * kBandWaves + 6 * sizeof(float) * (size_t)B.rows;
    if (lanes != 64 && lanes != 8)
        return hipErrorInvalidValue;
    const void *fn = lanes == 8 ? (const void *)k_adjbeam_band_sub<8> : (const void *)k_adjbeam_band;
    static std::atomic<size_t> configured[2][kDevs];
    hipError_t e = ensure_dyn_lds(fn, bytes, configured[lanes == 8 ? 1 : 0]);
    if (e != hipSuccess)
        return e;
    const long items = B.nchunks * B.nband;
    const long g = nblocks > 0 ? std::min<long>(items, nblocks) : items;   /* 0: one per item */
    if (lanes == 8)
        hipLaunchKernelGGL(k_adjbeam_band_sub<8>, dim3((unsigned)g), dim3(kBandBlock), bytes, st, p,
                           B);
    else
        hipLaunchKernelGGL(k_adjbeam_band, dim3((unsigned)g), dim3(kBandBlock), bytes, st, p, B);
    return hipGetLastError();
}

bool adjbeam_rec_plan(const PairParams &p, int rows, size_t pool_bytes, int ncu, RecPlan &pl)
{
    const long n = p.s_end - p.s_begin;
    /* six 64-bit sums per row in the band sums' LDS */
    const int max_rows = std::min<int>(1 << kRecRowBits, 163840 / (6 * 8));
    pl.rows = rows > 0 && rows < max_rows ? rows : max_rows;
    pl.rows = (int)std::max<long>(1, std::min<long>(pl.rows, p.npix_beam));
    pl.nband = (int)((p.npix_beam + pl.rows - 1) / pl.rows);
    if (pl.nband > kRecMaxBands || n <= 0)
        return false;
    /* patches, where the beam lies in the polar cap and has several */
    pl.tile = 0;
    const long nb = p.hb.nside;
    if (pl.nband > 8 && p.npix_beam <= 2 * nb * (nb + 1)) {
        const int tile = (int)std::sqrt((double)pl.rows);
        long rings = 1;
        while (2 * rings * (rings + 1) < p.npix_beam)
            rings++;
        const long blocks = (rings + tile - 1) / tile;
        if (tile >= 8 && 2 * blocks * (blocks + 1) <= kRecMaxBands) {
            pl.tile = tile;
            pl.rows = tile * tile;
            pl.nband = (int)(2 * blocks * (blocks + 1));
        }
    }
    /* Visits per sample, at most: the sky pixels whose centres lie within
     * rho_max are disjoint, each of area 4 pi / npix, and lie inside the cap
     * of radius rho_max + 2 s, s = sqrt(4 pi / npix) (more than any HEALPix
     * pixel's centre-to-boundary distance). */
    const double om = 4.0 * M_PI / (double)p.hs.npix;
    const double rc = std::min(M_PI, p.rho_max + 2.0 * std::sqrt(om));
    pl.bound = (long)(2.0 * M_PI * (1.0 - std::cos(rc)) / om) + 1;
    pl.bound = std::min<long>(pl.bound, p.hs.npix);
    /* per sample: its records and its offsets per band */
    const double per_sample = (double)sizeof(BeamRec) * pl.bound + 8.0 * pl.nband;
    double chunk = (double)pool_bytes / per_sample;
    chunk = std::max(chunk, (double)kBlock);
    chunk = std::min(chunk, (double)((1L << (32 - kRecRowBits)) - 1));
    chunk = std::min(chunk, (double)(0x7fffffffL / pl.bound));   /* 32-bit record positions */
    pl.chunk = std::max<long>(1, std::min<long>((long)chunk, n));
    /* parts per band: about eight blocks per CU (one fits a CU at a time),
     * so that the last round of blocks is a small part of the launch */
    pl.nsplit = (int)std::max<long>(1, std::min<long>(64, (8L * std::max(ncu, 1) + pl.nband - 1) /
                                                               pl.nband));
    pl.nrec = (size_t)pl.chunk * (size_t)pl.bound;
    pl.nidx = (size_t)pl.chunk * pl.nband + pl.nband + 1;
    pl.npart = (size_t)pl.nsplit * 6 * (size_t)p.npix_beam;
    return true;
}

hipError_t launch_adjbeam_records(const PairParams &p0, const RecPlan &pl, void *recs, long *idx,
                                  float *vmax, double *part, hipStream_t st)
{
    if (p0.s_end <= p0.s_begin || p0.npix_beam <= 0)
        return hipSuccess;
    RecParams R;
    R.rows = pl.rows;
    R.nband = pl.nband;
    R.inv_rows = 1.0f / (float)pl.rows;
    R.tile = pl.tile;
    R.inv_tile = pl.tile ? 1.0f / (float)pl.tile : 0.f;
    R.brec = (BeamRec *)recs;
    R.nrec_cap = (long)pl.nrec;
    R.bcnt = idx;
    R.bbase = idx + (size_t)pl.chunk * pl.nband;
    R.chunk = pl.chunk;
    R.vmax = vmax;
    R.part = part;
    R.nsplit = pl.nsplit;
    const size_t bytes = 6 * sizeof(unsigned long long) * (size_t)pl.rows;
    static std::atomic<size_t> configured[kDevs];
    hipError_t e = ensure_dyn_lds((const void *)k_beamrec_sum, bytes, configured);
    if (e != hipSuccess)
        return e;
    hipLaunchKernelGGL(k_fill_f64_n, dim3(gs_blocks((long)pl.npart)), dim3(256), 0, st, part,
                       (long)pl.npart);
    hipLaunchKernelGGL(k_fill_f64_n, dim3(1), dim3(64), 0, st, (double *)vmax, 1L);
    hipLaunchKernelGGL(k_rec_vmax, dim3(kMaxBlocks), dim3(256), 0, st, p0, vmax);
    for (long s0 = p0.s_begin; s0 < p0.s_end; s0 += pl.chunk) {
        PairParams p = p0;
        p.s_begin = s0;
        p.s_end = std::min(s0 + pl.chunk, p0.s_end);
        const long ns = p.s_end - p.s_begin;
        const dim3 g1((unsigned)((ns + kWavesPerBlock - 1) / kWavesPerBlock));
        hipLaunchKernelGGL(k_beamrec<false>, g1, dim3(kBlock), 0, st, p, R);
        hipLaunchKernelGGL(k_band_scan, dim3((unsigned)pl.nband), dim3(kScanBlock), 0, st, R, ns);
        hipLaunchKernelGGL(k_scan_excl, dim3(1), dim3(kScanBlock), 0, st, R.bbase,
                           (long)pl.nband);
        const dim3 g3((unsigned)((ns + kRecWriteWaves - 1) / kRecWriteWaves));
        hipLaunchKernelGGL(k_beamrec<true>, g3, dim3(kRecWriteWaves * kWaveSize), 0, st, p, R);
        hipLaunchKernelGGL(k_beamrec_sum, dim3((unsigned)(pl.nband * pl.nsplit)), dim3(kBandBlock),
                           bytes, st, p, R);
    }
    hipLaunchKernelGGL(k_beamrec_reduce, dim3(gs_blocks(6 * (long)p0.npix_beam)), dim3(256), 0, st,
                       part, pl.nsplit, (long)p0.npix_beam, p0.gbeam);
    return hipGetLastError();
}

int adjmap_describe(char *buf, size_t n, int cap, int rw)
{
    hipFuncAttributes a;
    hipError_t e = hipFuncGetAttributes(&a, (const void *)k_adjmap_lds<0, false>);
    if (e != hipSuccess)
        return snprintf(buf, n, "hipFuncGetAttributes: %s", hipGetErrorString(e));
    return snprintf(buf, n,
                    "block %d threads, kernel max %d, regs %d, static LDS %zu, dynamic LDS "
                    "%zu (max %d), private %zu",
                    kAdjBlock, a.maxThreadsPerBlock, a.numRegs, a.sharedSizeBytes,
                    adjmap_lds_bytes(cap, rw, 0, false), a.maxDynamicSharedSizeBytes,
                    a.localSizeBytes);
}

hipError_t launch_beam_support(const float *beam8, long npix, int *last, hipStream_t st)
{
    hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(1), 0, st, last, -1);
    if (npix > 0)
        hipLaunchKernelGGL(k_beam_support, dim3(std::min<unsigned>(gs_blocks(npix), kMaxBlocks)), dim3(256), 0, st,
                           (const float4 *)beam8, npix, last);
    return hipGetLastError();
}

hipError_t launch_ring_table(const Hpx &h, RingRec *out, hipStream_t st)
{
    long n = 4L * h.nside - 1;
    hipLaunchKernelGGL(k_ring_table, dim3(nblocks(n, 256)), dim3(256), 0, st, h, out);
    return hipGetLastError();
}

hipError_t launch_zero_f64(double *x, long n, hipStream_t st)
{
    if (n <= 0)
        return hipSuccess;
    hipLaunchKernelGGL(k_fill_f64, dim3(gs_blocks(n)), dim3(256), 0, st, x, n);
    return hipGetLastError();
}

hipError_t launch_add_offset(const float *x, float off, float *y, long n, hipStream_t st)
{
    if (n <= 0)
        return hipSuccess;
    hipLaunchKernelGGL(k_add_offset, dim3(gs_blocks(n)), dim3(256), 0, st, x, off, y, n);
    return hipGetLastError();
}

hipError_t launch_pack_sky(const float *I, const float *Q, const float *U, long npix,
                           float4 *sky4, hipStream_t st, const float *V)
{
    if (npix <= 0)
        return hipSuccess;
    hipLaunchKernelGGL(k_pack_sky, dim3(gs_blocks(npix)), dim3(256), 0, st, I, Q, U, V, npix,
                       sky4);
    return hipGetLastError();
}

hipError_t launch_fix_scale(const FixSource &f, long count, unsigned *work, double *scale,
                            hipStream_t st)
{
    const int ny = f.pairs ? f.npairs : 1;
    const long most = std::max(f.pairs ? 1L << 20 : f.npix, (f.n + ny - 1) / ny);
    const unsigned nx = std::min<unsigned>(gs_blocks(most), std::max(1, kMaxBlocks / ny));
    hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(64), 0, st, work, 2, 0u);
    hipLaunchKernelGGL(k_absmax, dim3(nx, ny), dim3(256), 0, st, f, work);
    hipLaunchKernelGGL(k_fix_scale, dim3(1), dim3(1), 0, st, (const unsigned *)work, count,
                       scale);
    return hipGetLastError();
}

hipError_t launch_fix_to_f32(const double *x, const double *scale, const F32Planes &y, long n,
                             hipStream_t st)
{
    if (n <= 0)
        return hipSuccess;
    /* Small planes in one launch; large ones one after the other, as blocks of two
     * planes at a time slow each other down (50e6 pixels 0.390 and 0.359 ms; 12.6e6, whole
     * call 0.235 and 0.239). */
    const int per = n < (1L << 24) ? 3 : 1;
    for (int k = 0; k < 3; k += per) {
        const F32Planes out = {{y.p[k], y.p[(k + 1) % 3], y.p[(k + 2) % 3]}};
        hipLaunchKernelGGL(k_fix_to_f32, dim3(gs_blocks(n), per), dim3(256), 0, st,
                           (const unsigned long long *)x + k * n, scale, out, n);
    }
    return hipGetLastError();
}

hipError_t launch_f64_to_f32(const double *x, float *y, long n, hipStream_t st)
{
    if (n <= 0)
        return hipSuccess;
    hipLaunchKernelGGL(k_f64_to_f32, dim3(gs_blocks(n)), dim3(256), 0, st, x, y, n);
    return hipGetLastError();
}

hipError_t launch_pack_beam(long npix, const float *const in[8], float *out, hipStream_t st)
{
    hipLaunchKernelGGL(k_pack_beam, dim3(gs_blocks(npix)), dim3(256), 0, st, npix, in[0],
                       in[1], in[2], in[3], in[4], in[5], in[6], in[7], (float4 *)out);
    return hipGetLastError();
}

hipError_t launch_pix2ang(const Hpx &h, long n, const int *pix, double *th, double *ph,
                          hipStream_t st)
{
    hipLaunchKernelGGL(k_pix2ang, dim3(gs_blocks(n)), dim3(256), 0, st, h, n, pix, th, ph);
    return hipGetLastError();
}

hipError_t launch_ang2pix(const Hpx &h, long n, const double *th, const double *ph,
                          int *pix, hipStream_t st)
{
    hipLaunchKernelGGL(k_ang2pix, dim3(gs_blocks(n)), dim3(256), 0, st, h, n, th, ph, pix);
    return hipGetLastError();
}

hipError_t launch_interpol(const Hpx &h, long n, const double *th, const double *ph,
                           int *pix, double *wgt, hipStream_t st)
{
    hipLaunchKernelGGL(k_interpol, dim3(gs_blocks(n)), dim3(256), 0, st, h, n, th, ph, pix,
                       wgt);
    return hipGetLastError();
}

hipError_t launch_disc(const Hpx &h, long n, const float *ra, const float *dec,
                       double radius, double cosr, const long *offsets, int *counts,
                       int *pixels, hipStream_t st)
{
    hipLaunchKernelGGL(k_disc, dim3(nblocks(n, 64)), dim3(64), 0, st, h, n, ra, dec, radius,
                       cosr, offsets, counts, pixels);
    return hipGetLastError();
}

hipError_t launch_match(const Hpx &hs, const RingRec *rings, const Hpx &hb, int mode, long n,
                        const float *ra, const float *dec, const float *pa,
                        const long *offsets, const int *pixels, int *bpix, double *chi,
                        hipStream_t st)
{
    if (n <= 0)
        return hipSuccess;
    hipLaunchKernelGGL(k_match, dim3((unsigned)n), dim3(256), 0, st, hs, rings, hb,
                       fast_consts(hb), fast_consts64(hb), mode, n, ra, dec, pa, offsets, pixels,
                       bpix, chi);
    return hipGetLastError();
}

FastConsts fast_consts(const Hpx &hb)
{
    FastConsts f;
    f.k3 = 3.0f * (float)hb.nside * (float)hb.nside;
    return f;
}

/* Constants of beam_pixel_f64: thresholds of the rho > 1e-6 test on crho
 * (rho >= 1.5e-6 is surely above 1e-6, rho <= 0.5e-6 surely below) and the
 * floor margin factor. */
FastConsts64 fast_consts64(const Hpx &hb)
{
    FastConsts64 f;
    f.crho_big = pl_cos(1.5e-6);
    f.crho_small = pl_cos(0.5e-6);
    f.marg_k = 100.0 * 4.4e-16 * hb.nside * 1.7320508075688772;
    return f;
}

hipError_t launch_libm(int op, long n, const double *x, const double *y, double *o,
                       hipStream_t st)
{
    hipLaunchKernelGGL(k_libm, dim3(gs_blocks(n)), dim3(256), 0, st, op, n, x, y, o);
    return hipGetLastError();
}

} /* namespace pisco */
