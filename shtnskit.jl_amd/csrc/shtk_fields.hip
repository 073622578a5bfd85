// FP64 Legendre stage of batches of fields, for gfx950: the recurrence of one
// order is run once for a group of fields (the single-field kernels of
// shtk_legendre.hip run it again for every field).
//
// Reference behaviour: analysis_batch / synthesis_batch
// (src/batch_transforms.jl:312-655), whose inner loops contract one Legendre
// row per (order, latitude) with all fields (:400-425, :519-535).
//
// FP64 matrix and vector instructions share one pipeline on this chip (a wave
// that issues both takes the sum of their times), so matrix instructions do not
// raise the FP64 rate; they are used where they save work around the FMAs.
#include <algorithm>

#include "shtk_internal.h"

namespace shtk {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr double kHi = 0x1p100;
constexpr double kDown = 0x1p-512;

template <typename T>
using cptr = const __attribute__((address_space(4))) T *;
template <typename T>
__device__ __forceinline__ cptr<T> as_const(const T *p) {
    return (cptr<T>)p;
}

__device__ __forceinline__ double mfac_of(int mode, int m) {
    if (m == 0 || mode == 0) return 1.0;
    return mode == 1 ? 2.0 : 0.5;
}

// ---------------------------------------------------------------------------
// Analysis of field groups: out[l, c] = sum_p P[l, p] G[p, c] over the latitude
// pairs p, c = 16 real columns (8 fields x re/im), as v_mfma_f64_16x16x4_f64
// with the degrees of one parity as rows, so the sum over pairs needs no
// cross-lane reduction (most of the LDS traffic of k_anal_w).
//
// One wavefront per (64-degree segment, field group).  It takes the pairs 64 at
// a time (one chain per lane, from the segment's seeds): 32 degrees of the
// recurrence go to the wave's LDS tile [16 even | 16 odd degrees][64 pairs] and
// come back as A operands (a lane reads two pairs, 16 bytes, of one degree)
// against the field operand of those pairs in registers, whose Fourier rows were
// loaded during the previous 64 pairs.  The products of all pairs stay in the
// accumulators, so waves share nothing and there are no barriers; every
// coefficient is stored once.
//
// Bound: FP64 issue (a matrix instruction holds the FP64 pipeline 64 cycles, 48 % of
// the kernel's cycles for 16 fields at lmax 1023, vector instructions 16 %), then LDS
// (operand staging) at 2 waves per SIMD.  16 fields at lmax 1023: 918 us (k_anal_w) -> 425 us;
// 37 fields at lmax 255: 86 -> 35 us; 16 at 511: 167 -> 81 us.  Tried, at 410 us: the pairs of a 512-pair block dealt to 4 waves with
// field operands held over 8 segments and the partial sums of every 32 degrees
// added through LDS (445 us: barriers), 16 fields per wave (478 us), operand
// loads straight from the Fourier columns (434 us: four times the cache lines).
// ---------------------------------------------------------------------------
constexpr int MX_ROW = 66;   // LDS row stride in doubles: 16 rows of one column pair fall on 16 different bank quads
constexpr int MX_DEG = 32;   // degrees per chunk (16 rows per parity)
constexpr int MX_FIELDS = 8; // fields per group

// Degrees N .. 31 of a chunk for one chain: value of the degree to the tile
// (row: parity, then degree / 2), then the Q-form step.  The per-degree beta
// sit in two VGPR pairs, lane n of each 16-lane row holding degree n (b0) and
// 16 + n (b1), broadcast by DPP.  cm: 0 for lanes still in the scaled range.
template <bool FAST, int N>
__device__ __forceinline__ void mx_steps(double b0, double b1, double x, double cm, double &prev, double &cur,
                                         double *tl) {
    if constexpr (N < MX_DEG) {
        tl[((N & 1) * 16 + (N >> 1)) * MX_ROW] = FAST ? cur : cur * cm;
        double t = x * cur;
        if (N < 16) SHTK_FMAC_BC(t, b0, prev, (N & 15), "-");
        else SHTK_FMAC_BC(t, b1, prev, (N & 15), "-");
        prev = cur;
        cur = t;
        mx_steps<FAST, N + 1>(b0, b1, x, cm, prev, cur, tl);
    }
}

template <typename OT>
__global__ __launch_bounds__(64, 2) void k_anal_mx(const LegArgs a) {
    __shared__ __align__(16) double tile[MX_DEG * MX_ROW];
    // blocks go round-robin over the XCDs; a.seglist holds every order's segments on one
    // XCD, so its Fourier columns are read into one L2
    const int xcd = blockIdx.x % kXcds, fg = blockIdx.x / kXcds % a.gz;
    const cptr<int> item = as_const((const int *)a.seglist) + 4 * (size_t)(blockIdx.x / kXcds / a.gz * kXcds + xcd);
    int gs = item[0], coff = item[3];  // one load, short waves
    const int im = item[1], s = item[2];
    if (gs < 0 || (a.skip_m0 && im == 0)) return;
    const int m = im * a.mres, np = a.np, nlat = a.nlat, lmax = a.lmax;
    const bool one = a.m0_one && im == 0;  // order 0 on the tables of order 1
    const double *wlat = one ? a.wlat0 : a.wlat;
    const int mt = one ? 1 : m;
    if (one) {
        gs = min(as_const(a.segbase)[1] + s, a.nseg_total - 1);
        coff = (int)as_const(a.coff)[1];
    }
    const int l0 = mt + s * DSEG, lend = min(l0 + DSEG, lmax + 1), lstop = min(lend, a.ltr + 1);
    if (l0 >= lend) return;  // order 1 can have one segment fewer
    const int lane = threadIdx.x;
    const int f0 = fg * MX_FIELDS, nfl = min(MX_FIELDS, a.nf - f0);
    OT *col = (OT *)a.out0 + 2 * ((size_t)f0 * a.spec_fstride + (size_t)(lmax + 1) * m);
    // coefficients of this order that no degree writes: l < m, and the orders up
    // to the next multiple of mres
    if (s == 0) {
        for (int f = 0; f < nfl; ++f) {
            OT *d = col + 2 * (size_t)f * a.spec_fstride;
            for (int l = lane; l < m; l += 64) {
                d[2 * l] = (OT)0;
                d[2 * l + 1] = (OT)0;
            }
            const int nx = (min(m + a.mres, a.mmax + 1) - m - 1) * (lmax + 1);
            for (int l = lmax + 1 + lane; l < lmax + 1 + nx; l += 64) {
                d[2 * l] = (OT)0;
                d[2 * l + 1] = (OT)0;
            }
        }
    }
    const int pfirst = as_const(a.pfirst)[gs], pfast = as_const(a.pfast)[gs];
    const int nch = l0 < lstop ? (np - min(pfirst, np) + 63) / 64 : 0;  // 64-pair chains, ending at the equator
    const int pst = np - 64 * nch;
    const long long co = (long long)coff - mt;
    const double *qbv = a.qb + co + l0 + 1 + (lane & 15);  // padded past lmax
    const double b0 = qbv[0], b1 = qbv[16], b2 = qbv[32], b3 = qbv[48];
    const cptr<double> qcm = as_const(a.qcc) + co;
    d4 acc[2][2] = {};
    const double *at = tile + (lane & 15) * MX_ROW + 2 * (lane >> 4);
    // Fourier rows of the next 64 pairs: lane = pair, 16 bytes (re, im) per field and
    // hemisphere (a load covers 1 KB of one row; loading the operand layout below directly
    // takes four times the cache lines per byte)
    const double2 *Fn = a.F0 + ((size_t)f0 * a.nm + im) * nlat;
    const size_t fst = (size_t)a.nm * nlat;
    double2 RN[8], RS[8];
    double nq0 = 0.0, nq1 = 0.0, nx = 0.0, nw = 0.0;
    int nk = 0;
    auto load = [&](int ch) {
        // lanes before the first live pair carry weight zero over that pair's values: what the
        // field holds at rows that count for nothing (an infinity, a NaN) stays out of the sums
        const int p0 = pst + 64 * ch + lane, p = max(p0, pfirst);
#pragma unroll
        for (int f = 0; f < 8; ++f) {
            const double2 *Ff = Fn + min(f, nfl - 1) * fst;
            RN[f] = Ff[p];
            RS[f] = Ff[nlat - 1 - p];
        }
        const size_t q = (size_t)gs * np + p;
        nq0 = a.seedq0[q];
        nq1 = a.seedq1[q];
        nk = a.seedk[q];
        nx = a.x[p];
        nw = wlat ? wlat[p] : 1.0;
        if (2 * p == nlat - 1) nw *= 0.5;  // the equator's latitude is both halves of its pair
        if (p0 < pfirst) nw = 0.0;
    };
    // sums and differences of the hemispheres through the tile, as [16 columns][64 pairs] per
    // half: lane (column c = lane & 15, k = lane >> 4) reads pairs 8 t + 2 k + 0, 1 of column c
    double *sw = tile + lane;
    const double *sr = tile + (lane & 15) * MX_ROW + 2 * (lane >> 4);
    if (nch > 0) load(0);
    for (int ch = 0; ch < nch; ++ch) {
        double B[2][16];
#pragma unroll
        for (int f = 0; f < 8; ++f) {
            sw[(2 * f) * MX_ROW] = RN[f].x + RS[f].x;
            sw[(2 * f + 1) * MX_ROW] = RN[f].y + RS[f].y;
            sw[(16 + 2 * f) * MX_ROW] = RN[f].x - RS[f].x;
            sw[(16 + 2 * f + 1) * MX_ROW] = RN[f].y - RS[f].y;
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const double2 v = *(const double2 *)(sr + 16 * MX_ROW * q + 8 * t);
                B[q][2 * t] = v.x;
                B[q][2 * t + 1] = v.y;
            }
        __builtin_amdgcn_wave_barrier();
        // the weights go into the recurrence's starting values
        const double x = nx;
        double prev = nq0 * nw, cur = nq1 * nw;
        int kk = nk;
        const int pc = pst + 64 * ch, t0 = max(pfirst - pc, 0) >> 3;
        bool slow = pc < pfast;
        if (ch + 1 < nch) load(ch + 1);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const double bl = h ? b2 : b0, bh = h ? b3 : b1;
            if (h == 1 && l0 + MX_DEG >= lstop) break;
            dpp_wait(bl, bh);
            if (slow) {
                const double cm = kk == 0 ? 1.0 : 0.0;
                mx_steps<false, 0>(bl, bh, x, cm, prev, cur, tile + lane);
                // one check per chunk: a chain grows by less than 2^230 over 32 degrees, so
                // what it misses before it counts is below 2^(100 + 230 - 512)
                const double cl = qcm[l0 + MX_DEG * h + MX_DEG - 1];
                if (kk > 0 && fmax(fabs(cur), fabs(prev)) * cl > kHi) {
                    cur *= kDown;
                    prev *= kDown;
                    kk -= 1;
                }
                slow = __any(kk > 0);
            } else {
                mx_steps<true, 0>(bl, bh, x, 1.0, prev, cur, tile + lane);
            }
            __builtin_amdgcn_wave_barrier();
            auto mul = [&](int t, const double2 &ae, const double2 &ao) {
                acc[h][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(ae.x, B[0][2 * t], acc[h][0], 0, 0, 0);
                acc[h][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(ao.x, B[1][2 * t], acc[h][1], 0, 0, 0);
                acc[h][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(ae.y, B[0][2 * t + 1], acc[h][0], 0, 0, 0);
                acc[h][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(ao.y, B[1][2 * t + 1], acc[h][1], 0, 0, 0);
            };
            auto lda = [&](int t, int par) { return *(const double2 *)(at + 16 * MX_ROW * par + 8 * t); };
            if (t0 == 0) {
                // (with an exit test per step the reads could not move ahead of the products)
                double2 ae = lda(0, 0), ao = lda(0, 1);
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    double2 ne = ae, no = ao;
                    if (t < 7) {
                        ne = lda(t + 1, 0);
                        no = lda(t + 1, 1);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    mul(t, ae, ao);
                    ae = ne;
                    ao = no;
                }
            } else {
#pragma unroll
                for (int t = 0; t < 8; ++t)
                    if (t >= t0) mul(t, lda(t, 0), lda(t, 1));
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
    // sums to the tile, [chunk, parity, register][lane]: degree 32 chunk + 2 i + parity, i =
    // lane / 16 + 4 register, column lane & 15; lane d then stores degree l0 + d
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r) tile[(8 * h + 4 * q + r) * 64 + lane] = acc[h][q][r];
    __builtin_amdgcn_wave_barrier();
    const int l = l0 + lane, i = (lane & 31) >> 1;
    if (l >= lend) return;
    const double sc = l < lstop ? a.g * mfac_of(a.mfac_mode, m) * (a.raw_q ? 1.0 : a.qcc[co + l]) : 0.0;
    const double *src = tile + (8 * (lane >> 5) + 4 * (lane & 1) + (i >> 2)) * 64 + (i & 3) * 16;
    for (int f = 0; f < nfl; ++f) {
        const double2 v = *(const double2 *)(src + 2 * f);
        OT *d = col + 2 * ((size_t)f * a.spec_fstride + l);
        d[0] = (OT)(sc * v.x);
        d[1] = (OT)(sc * v.y);
    }
}

// ---------------------------------------------------------------------------
// Synthesis of field groups.  One wavefront per (order, 64 latitude pairs, group
// of NG fields) runs the order's recurrence once, from the seeds of its first
// live segment to the last degree, and adds every degree to the NG fields' sums
// (even and odd degrees, re and im: 4 NG accumulators per lane).  The operands of
// 16 degrees, beta_{l+1} and c_l a_l of every field, sit in VGPRs, lane n of each
// 16-lane row holding degree n, and reach the FMAs by DPP broadcast as in
// k_synth_d; the next 16 degrees are loaded meanwhile.  Per degree and pair: one
// multiply, one FMA and 2 NG FMAs.
// NW waves per block take equal runs of the order's live segments, each from its own
// seeds, and add their sums through LDS.
//
// Bound: FP64 issue (VALU 78 % of the cycles for 16 fields at lmax 1023, at 2.1 GHz).
// 16 fields at lmax 1023: 735 us (k_synth_d) -> 379; 3 fields: 152 -> 98; 16 at 511:
// 114 -> 61; 37 at 255: 40 -> 30; 5 at 340: 29 -> 17; 8 at 63: 5.7 -> 4.8.
// ---------------------------------------------------------------------------
template <int NG, typename CT = double2>
struct SFRec {
    double b, c;      // beta_{l+1}, c_l
    CT v[NG];         // a_l of the fields
};

// Degrees N .. 15 of a record group.
template <int NG, bool FAST, int N>
__device__ __forceinline__ void sf_steps(const SFRec<NG> &r, double x, double cm, double &prev, double &cur,
                                         double (*acc)[NG][2]) {
    if constexpr (N < 16) {
        double t = x * cur;
        const double u = FAST ? cur : cur * cm;
#pragma unroll
        for (int f = 0; f < NG; ++f) {
            SHTK_FMAC_BC(acc[N & 1][f][0], r.v[f].x, u, N, "");
            SHTK_FMAC_BC(acc[N & 1][f][1], r.v[f].y, u, N, "");
        }
        SHTK_FMAC_BC(t, r.b, prev, N, "-");
        prev = cur;
        cur = t;
        sf_steps<NG, FAST, N + 1>(r, x, cm, prev, cur, acc);
    }
}

// The degree before (N = 0, odd) or after (N = 1, even) a segment, operands in lane N of
// each row.
template <int NG, int N>
__device__ __forceinline__ void sf_edge(const double2 *eg, double (*acc)[NG][2], double u) {
#pragma unroll
    for (int f = 0; f < NG; ++f) {
        SHTK_FMAC_BC(acc[1 - N][f][0], eg[f].x, u, N, "");
        SHTK_FMAC_BC(acc[1 - N][f][1], eg[f].y, u, N, "");
    }
}

// CT: the type of the coefficients (float2: scalar transforms of FP32 arrays).
template <int NG, int NW, bool VEC, typename CT>
__global__ __launch_bounds__(64 * NW, NG <= 4 ? 4 : 3) void k_synth_sf(const LegArgs a) {
    __shared__ double red[NW > 1 ? NW - 1 : 1][NW > 1 ? 4 * NG : 1][64];
    // units lowest order first for every pair block and group: the long columns start first
    const int unit = blockIdx.x, b = unit % a.gx, fg = unit / a.gx % a.gz, im = unit / (a.gx * a.gz);
    if (a.skip_m0 && im == 0) return;
    const int m = im * a.mres, np = a.np, lmax = a.lmax, ltr = a.ltr;
    const int lane = threadIdx.x & 63;
    const int w = NW > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
    const int f0 = fg * NG, nfl = min(NG, a.nf - f0);
    const int p = b * 64 + lane, pc = min(p, np - 1), pb1 = min(b * 64 + 64, np);
    const bool one = VEC && a.m0_one && im == 0;  // order 0 on the tables of order 1
    const int mt = one ? 1 : m, segb = as_const(a.segbase)[one ? 1 : im];
    const long long co = as_const(a.coff)[one ? 1 : im] - mt;
    double acc[2][NG][2];
#pragma unroll
    for (int f = 0; f < NG; ++f) acc[0][f][0] = acc[0][f][1] = acc[1][f][0] = acc[1][f][1] = 0.0;
    // first segment with a live pair of this block
    const int nseg = ltr >= mt ? (ltr - mt) / DSEG + 1 : 0;
    int s0 = nseg;
    for (int q = 0; q < nseg; q += 64) {
        const unsigned long long live = __ballot(q + lane < nseg && pb1 > a.pfirst[segb + min(q + lane, nseg - 1)]);
        if (live) {
            s0 = q + __builtin_ctzll(live);
            break;
        }
    }
    s0 = __builtin_amdgcn_readfirstlane(s0);
    const int sa = s0 + w * (nseg - s0) / NW, sb = s0 + (w + 1) * (nseg - s0) / NW;
    if (sa < sb) {
        const double x = a.x[pc];
        const size_t q = (size_t)(segb + sa) * np + pc;
        double prev = a.seedq0[q], cur = a.seedq1[q];
        int kk = a.seedk[q];
        const double *qb = a.qb + co + 1, *qc = a.qcc + co;  // padded past lmax
        const cptr<double> qcm = as_const(a.qcc) + co;
        const CT *av = (const CT *)a.in0 + (size_t)f0 * a.spec_fstride + (size_t)(lmax + 1) * m;
        const int l1 = min(mt + sb * DSEG, ltr + 1);  // VEC: ltr is the degree after the last S, T
        SFRec<NG, CT> n;
        auto load = [&](int l0) {
            // uniform bases and one 32-bit lane offset (64-bit addresses per field would
            // take the registers of a wave)
            const unsigned l = l0 + (lane & 15), lc = (unsigned)sizeof(CT) * min(l, (unsigned)lmax);
            n.b = qb[l];
            n.c = qc[l];
#pragma unroll
            for (int f = 0; f < NG; ++f)
                n.v[f] = *(const CT *)((const char *)(av + (size_t)min(f, nfl - 1) * a.spec_fstride) + lc);
        };
        int l = mt + sa * DSEG;
        load(l);
        bool slow = __any(kk > 0);
        // VEC: the terms that reach past the segments (a.edge): the degree before segment
        // s (its Q is prev there) and the degree after the one that ends (cur)
        const double2 *ev = VEC ? a.edge + 2 * ((size_t)f0 * a.nseg_total + as_const(a.segbase)[im]) : nullptr;
        double2 eg[VEC ? NG : 1];
        auto load_edges = [&]([[maybe_unused]] int s) {  // lane 0 of a row: before segment s, lane 1: after segment s - 1
            if constexpr (VEC) {
                const unsigned o = 16u * ((lane & 15) == 0 ? 2 * min(s, nseg - 1) : max(2 * s - 1, 0));
#pragma unroll
                for (int f = 0; f < NG; ++f)
                    eg[f] = *(const double2 *)((const char *)(ev + 2 * (size_t)min(f, nfl - 1) * a.nseg_total) + o);
#pragma unroll
                for (int f = 0; f < NG; ++f) {
                    dpp_written(eg[f].x);
                    dpp_written(eg[f].y);
                }
                dpp_wait();
            }
        };
        if constexpr (VEC)
            if (sa > 0) {
                load_edges(sa);
                sf_edge<NG, 0>(eg, acc, kk == 0 ? prev : 0.0);
            }
        // the group's operands, and the loads of the next group (the last one reads clamped
        // positions and is not used)
        auto take = [&](SFRec<NG> &r) {
            if (l + 16 > l1) {  // degrees past the last one contribute nothing
                const bool in = l + (lane & 15) < l1;
#pragma unroll
                for (int f = 0; f < NG; ++f) {
                    n.v[f].x = in ? n.v[f].x : 0;
                    n.v[f].y = in ? n.v[f].y : 0;
                }
            }
            r.b = n.b;
            const double sc = a.qscale_in ? n.c : 1.0;
#pragma unroll
            for (int f = 0; f < NG; ++f) r.v[f] = make_double2((double)n.v[f].x * sc, (double)n.v[f].y * sc);
            load(l + 16);
#pragma unroll
            for (int f = 0; f < NG; ++f) {
                dpp_written(r.v[f].x);
                dpp_written(r.v[f].y);
            }
            dpp_wait(r.b);
        };
        // groups with scaled lanes first (a lane never becomes scaled again), then the rest in
        // a loop of its own, whose registers hold one body
        for (; l < l1 && slow; l += 16) {
            SFRec<NG> r;
            take(r);
            sf_steps<NG, false, 0>(r, x, kk == 0 ? 1.0 : 0.0, prev, cur, acc);
            // one check per 16 degrees: growth below 2^120, so what a chain misses before it
            // counts is below 2^(100 + 120 - 512)
            const double cl = qcm[l + 15];
            if (kk > 0 && fmax(fabs(cur), fabs(prev)) * cl > kHi) {
                cur *= kDown;
                prev *= kDown;
                kk -= 1;
            }
            slow = __any(kk > 0);
            if (((l - mt + 16) & (DSEG - 1)) == 0 && l + 16 <= l1) {  // the Q form of the next segment
                const int s = (l - mt + 16) / DSEG;
                if constexpr (VEC) load_edges(s);
                if constexpr (VEC) sf_edge<NG, 1>(eg, acc, kk == 0 ? cur : 0.0);
                prev *= cl;
                cur *= cl;
                if constexpr (VEC)
                    if (s < sb) sf_edge<NG, 0>(eg, acc, kk == 0 ? prev : 0.0);
            }
        }
        // once every lane is live each segment starts from its own seeds, loaded a segment ahead
        size_t qn = (size_t)(segb + (l - mt) / DSEG + 1) * np + pc;
        double nq0 = 0.0, nq1 = 0.0;
        auto load_seeds = [&] {
            if (mt + ((l - mt) / DSEG + 1) * DSEG < l1) {
                nq0 = a.seedq0[qn];
                nq1 = a.seedq1[qn];
                qn += np;
            }
        };
        load_seeds();
        for (; l < l1; l += 16) {
            SFRec<NG> r;
            take(r);
            sf_steps<NG, true, 0>(r, x, 1.0, prev, cur, acc);
            if (((l - mt + 16) & (DSEG - 1)) == 0 && l + 16 <= l1) {
                const int s = (l - mt + 16) / DSEG;
                if constexpr (VEC) load_edges(s);
                if constexpr (VEC) sf_edge<NG, 1>(eg, acc, cur);
                prev = nq0;
                cur = nq1;
                if constexpr (VEC)
                    if (s < sb) sf_edge<NG, 0>(eg, acc, prev);
                l += 16;
                load_seeds();
                l -= 16;
            }
        }
    }
    if constexpr (NW > 1) {
        if (w > 0)
#pragma unroll
            for (int f = 0; f < NG; ++f)
#pragma unroll
                for (int k = 0; k < 4; ++k) red[w - 1][4 * f + k][lane] = acc[k >> 1][f][k & 1];
        __syncthreads();
        if (w > 0) return;
#pragma unroll
        for (int f = 0; f < NG; ++f)
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int v = 0; v < NW - 1; ++v) acc[k >> 1][f][k & 1] += red[v][4 * f + k][lane];
    }
    if (p >= np) return;
    const double *wlat = one ? a.wlat0 : a.wlat;
    const double sc = a.g * mfac_of(a.mfac_mode, m) * (wlat ? wlat[p] : 1.0);
    double2 *Fo = a.F0 + ((size_t)f0 * a.nm + im) * a.nlat;
    const int ps = a.nlat - 1 - p;
#pragma unroll
    for (int f = 0; f < NG; ++f) {
        if (f >= nfl) break;
        double2 *Ff = Fo + (size_t)f * a.nm * a.nlat;
        Ff[p] = make_double2((acc[0][f][0] + acc[1][f][0]) * sc, (acc[0][f][1] + acc[1][f][1]) * sc);
        if (ps != p) Ff[ps] = make_double2((acc[0][f][0] - acc[1][f][0]) * sc, (acc[0][f][1] - acc[1][f][1]) * sc);
    }
}

template <int NG, bool VEC, typename CT>
void launch_synth_sf(const LegArgs &a, hipStream_t st) {
    const long long units = (long long)(a.nm_run > 0 ? std::min(a.nm_run, a.nm) : a.nm) * a.gx * a.gz;
    // 2 waves per unit where one would leave the chip short of waves (4096 units, 16
    // fields at lmax 511: 65 -> 62 us; 16384, 16 at 1023: 429 against 432; 4 waves lose
    // the accumulator traffic through LDS: 98 us at 511)
    const dim3 grid((unsigned)units);
    if (units >= 8192 || a.lmax < DSEG) hipLaunchKernelGGL((k_synth_sf<NG, 1, VEC, CT>), grid, dim3(64), 0, st, a);
    else hipLaunchKernelGGL((k_synth_sf<NG, 2, VEC, CT>), grid, dim3(128), 0, st, a);
}

// ---------------------------------------------------------------------------
// Vector synthesis as two scalar ones of degree lmax + 1: with d_l = sqrt((l^2 - m^2) /
// (4 l^2 - 1)) the coefficients of sin(theta) V_theta and sin(theta) V_phi are
//     (l-1) d_l S_{l-1} - (l+2) d_{l+1} S_{l+1} - i m T_l
//     i m S_l + (l-1) d_l T_{l-1} - (l+2) d_{l+1} T_{l+1}
// (src/legendre.jl:542-546 applied to the sums of src/kernels.jl:155-169).  Written
// times c_l, the form k_synth_sf takes: c_l d_l = c_{l-1} and d_l^2 = beta_{l+1}, so
// they need no root, and both degrees that one S_l reaches carry the same c_l.  The
// two terms cancel near the poles, so they also have to come from one segment's
// recurrence: where S_l reaches past its segment the term goes to E instead, which
// k_synth_sf adds with that segment's own Q at the degree before or after it (with
// the neighbour segment's Q the error of the grid was 10 to 17 % larger).
// m0_one: dP_l/dtheta of order 0 is sqrt(l(l+1)) P_l^1, so order 0 needs no division by
// sin(theta): its column holds sqrt(l(l+1)) S_l (and T_l) for the recurrence of order 1, and
// its rows take their own factor (LegArgs.wlat0).  That is the differentiated recurrence of the
// zonal kernel in one more order of the same launch, instead of a kernel on a second stream
// (two events and two waits: 20 to 30 us of a call of 70).
// One block per (order, field); [theta fields][phi fields], columns of lmax + 2 and
// E[field][segment][before, after].
// ---------------------------------------------------------------------------
template <typename IT>
__global__ __launch_bounds__(256) void k_vcoef(const IT *S, const IT *T, double2 *C, double2 *E, const int *segbase,
                                               int nseg_total, const double *scale, int divide, int ll1,
                                               const double *qb, const double *qcc, const long long *coff,
                                               int lmax, int mres, int nm, int ltr, int m0_one, long long in_fstride,
                                               long long out_fstride, int nf) {
    const int im = blockIdx.x % nm, f = blockIdx.x / nm, m = im * mres;
    const size_t col = (size_t)(lmax + 1) * m;
    const IT *Sm = S + 2 * ((size_t)f * in_fstride + col), *Tm = T + 2 * ((size_t)f * in_fstride + col);
    const double *sm = scale ? scale + col : nullptr;
    const double *cq = qcc + coff[im] - m, *bq = qb + coff[im] - m;
    double2 *Ct = C + (size_t)f * out_fstride + (size_t)(lmax + 2) * m;
    double2 *Cp = Ct + (size_t)nf * out_fstride;
    const int lo = max(1, m), hi = min(ltr, lmax);
    for (int l = m + (int)threadIdx.x; l <= lmax + 1; l += 256) {
        const int t = l - m;
        // S_k, T_k times k's factor, zero outside [lo, hi] (clamped reads)
        auto at = [&](int k, double fac, double2 *s, double2 *q) {
            const bool in = k >= lo && k <= hi;
            const int kc = min(max(k, m), lmax);
            if (sm) fac = divide ? fac / sm[kc] : fac * sm[kc];
            if (ll1 && in) fac /= (double)k * (k + 1);
            *s = in ? make_double2(fac * (double)Sm[2 * kc], fac * (double)Sm[2 * kc + 1]) : make_double2(0.0, 0.0);
            *q = in ? make_double2(fac * (double)Tm[2 * kc], fac * (double)Tm[2 * kc + 1]) : make_double2(0.0, 0.0);
        };
        const bool first = t % DSEG == 0, last = t % DSEG == DSEG - 1;  // in the segment
        double2 s1, t1, s0, t0, s2, t2, q, r;
        if (m0_one && m == 0) {
            const int l1 = max(l, 1);
            at(l, sqrt((double)l1 * (l1 + 1)) * qcc[coff[1] + l1 - 1], &Ct[l], &Cp[l]);
            if (first || last) {
                const size_t e = 2 * ((size_t)f * nseg_total + segbase[0] + t / DSEG) + (last ? 1 : 0);
                E[e] = E[e + 2 * (size_t)nf * nseg_total] = make_double2(0.0, 0.0);
            }
            continue;
        }
        const double cl = cq[l];
        at(first ? -1 : l - 1, (l - 1) * cq[max(l - 1, m)], &s1, &t1);
        at(l, m * cl, &s0, &t0);
        at(last ? -1 : l + 1, (l + 2) * bq[min(l, lmax - 1) + 2] * cq[min(l, lmax) + 1], &s2, &t2);
        Ct[l] = make_double2(s1.x - s2.x + t0.y, s1.y - s2.y - t0.x);
        Cp[l] = make_double2(t1.x - t2.x - s0.y, t1.y - t2.y + s0.x);
        if (first || last) {  // S_l at degree l - 1 (before), at degree l + 1 (after)
            at(l, first ? -(l + 1) * bq[min(l, lmax) + 1] * cl : l * cl, &q, &r);
            const size_t e = 2 * ((size_t)f * nseg_total + segbase[im] + t / DSEG) + (last ? 1 : 0);
            E[e] = q;
            E[e + 2 * (size_t)nf * nseg_total] = r;
        }
    }
}

// ---------------------------------------------------------------------------
// Vector analysis from two scalar ones of degree lmax + 1 with the weights w / sin(theta):
//     S_l = [l d_{l+1} Gt_{l+1} - (l+1) d_l Gt_{l-1} - i m Gp_l] / (l(l+1))
//     T_l = [i m Gt_l + l d_{l+1} Gp_{l+1} - (l+1) d_l Gp_{l-1}] / (l(l+1))
// (src/kernels.jl:205-215; ll1 = 0: without the division).  H: the sums against Q_l = P_l /
// c_l (LegArgs.raw_q), so with the identities of k_vcoef the factors are table entries:
// d_{l+1} c_{l+1} = c_l, or 1 where l + 1 starts a segment, and d_l c_{l-1} = beta_{l+1} c_l,
// times c_{l-1} of its own segment where l starts one.  One block per (column,
// field); columns that are not orders and rows l < max(1, m) or l > ltr are written
// as zero.  skip_m0: the zonal kernel writes the degrees to ltr of order 0.  m0_one: order 0
// has S_l = c_l Gt_l sqrt(l(l+1)) / (l(l+1)), T_l the same of Gp, on order 1's tables.
// ---------------------------------------------------------------------------
template <typename OT>
__global__ __launch_bounds__(256) void k_vout(const double2 *H, OT *S, OT *T, const double *scale, int divide, int ll1,
                                              int skip_m0, int m0_one, const double *qb, const double *qcc, const long long *coff,
                                              int lmax, int mmax, int mres, int ltr, long long h_fstride,
                                              long long out_fstride, int nf) {
    const int m = blockIdx.x % (mmax + 1), f = blockIdx.x / (mmax + 1), im = m / mres;
    const bool order = im * mres == m;
    const size_t col = (size_t)(lmax + 1) * m;
    OT *So = S + 2 * ((size_t)f * out_fstride + col), *To = T + 2 * ((size_t)f * out_fstride + col);
    const double2 *Ht = H + (size_t)f * h_fstride + (size_t)(lmax + 2) * m, *Hp = Ht + (size_t)nf * h_fstride;
    const double *cq = qcc + coff[im] - im * mres, *bq = qb + coff[im] - im * mres;
    const int lo = max(1, m), hi = min(ltr, lmax);
    for (int l = (int)threadIdx.x + (skip_m0 && m == 0 ? hi + 1 : 0); l <= lmax; l += 256) {
        double2 s = make_double2(0.0, 0.0), t = s;
        if (order && l >= lo && l <= hi) {
            const int lm = max(l - 1, m), r = l - m;
            const double c = cq[l];
            double k = ll1 ? 1.0 / ((double)l * (l + 1)) : 1.0;
            if (scale) k = divide ? k / scale[col + l] : k * scale[col + l];
            if (m0_one && m == 0) {
                const double fac = sqrt((double)l * (l + 1)) * qcc[coff[1] + l - 1] * k;
                const double2 t0 = Ht[l], p0 = Hp[l];
                s = make_double2(fac * t0.x, fac * t0.y);
                t = make_double2(fac * p0.x, fac * p0.y);
            } else {
                const double up = l * ((r + 1) % DSEG == 0 ? 1.0 : c) * k, mc = m * c * k;
                const double dn = (l + 1) * bq[l + 1] * c * (r % DSEG == 0 ? cq[lm] : 1.0) * k;  // 0 for l = m
                const double2 t2 = Ht[l + 1], t0 = Ht[l], t1 = Ht[lm], p2 = Hp[l + 1], p0 = Hp[l], p1 = Hp[lm];
                s = make_double2(up * t2.x - dn * t1.x + mc * p0.y, up * t2.y - dn * t1.y - mc * p0.x);
                t = make_double2(up * p2.x - dn * p1.x - mc * t0.y, up * p2.y - dn * p1.y + mc * t0.x);
            }
        }
        So[2 * l] = (OT)s.x;
        So[2 * l + 1] = (OT)s.y;
        To[2 * l] = (OT)t.x;
        To[2 * l + 1] = (OT)t.y;
    }
}

}  // namespace

// A group costs the same for 1 to 8 fields.  Against the single-field kernel, lmax
// 1023: 4 fields 228 (one group) against 256 us, 3 fields 228 against 192; so fewer
// than 4 fields go to the single-field kernel.  Beside other groups that is a launch of
// its own, which one field is worth from lmax 400 and two from 600 (whole calls, single
// kernel against a group more: 9 fields at 127 22.7 and 15.2 us, at 255 36.6 and 31.0, at
// 511 92.5 and 99.0; 10 at 511 103.8 and 96.4, at 700 310 and 317, at 1023 464 and 510; 11
// at 1023 541 and 528).
int fields_anal_count(const LegArgs &a, int nfields) {
    if (a.seg != DSEG) return 0;
    const int rest = nfields % MX_FIELDS;
    const bool single = nfields < MX_FIELDS ? rest < 4 : rest < 3 && a.lmax >= 200 * (rest + 1);
    return single ? nfields - rest : nfields;
}

hipError_t launch_fields_anal(const LegArgs &a0, int nfields, hipStream_t st) {
    LegArgs a = a0;
    a.nf = nfields;
    a.gz = (nfields + MX_FIELDS - 1) / MX_FIELDS;
    const dim3 grid((unsigned)a.nlist * a.gz);
    if (a.io_f32) hipLaunchKernelGGL(k_anal_mx<float>, grid, dim3(64), 0, st, a);
    else hipLaunchKernelGGL(k_anal_mx<double>, grid, dim3(64), 0, st, a);
    return hipGetLastError();
}

bool fields_synth_ok(const LegArgs &a, int nfields) { return nfields >= 2 && a.seg == DSEG; }

template <bool VEC, typename CT>
static void launch_synth_groups(const LegArgs &a, int ng, hipStream_t st) {
    switch (ng) {
        case 2: launch_synth_sf<2, VEC, CT>(a, st); break;
        case 3: launch_synth_sf<3, VEC, CT>(a, st); break;
        case 4: launch_synth_sf<4, VEC, CT>(a, st); break;
        case 5: launch_synth_sf<5, VEC, CT>(a, st); break;
        case 6: launch_synth_sf<6, VEC, CT>(a, st); break;
        case 7: launch_synth_sf<7, VEC, CT>(a, st); break;
        default: launch_synth_sf<8, VEC, CT>(a, st); break;
    }
}

hipError_t launch_fields_synth(const LegArgs &a0, int nfields, hipStream_t st) {
    LegArgs a = a0;
    a.nf = nfields;
    a.gx = (a.np + 63) / 64;
    // equal groups of at most 8 fields, 4 or 2 where these would leave fewer than 1024 units
    // (a short launch takes as long as one unit, whose time goes with the fields: whole calls
    // in groups of 8, 4 and 2, 8 fields at lmax 127 14.6, 13.3 and 13.3 us, at 255 24.2, 21.3
    // and 21.1; 16 at 191 25.4, 22.3 and 23.8; 32 at 127 19.3, 16.1 and 18.5; from 1024 units
    // of 8 on 8 at 511 60.5, 60.5 and 67.2, 32 at 340 193, 194 and 205)
    const int nm = a.nm_run > 0 ? std::min(a.nm_run, a.nm) : a.nm;
    int most = 8;
    while (most > 2 && (long long)nm * a.gx * ((nfields + most - 1) / most) < 1024) most /= 2;
    a.gz = (nfields + most - 1) / most;
    const int ng = (nfields + a.gz - 1) / a.gz;
    if (a.edge) launch_synth_groups<true, double2>(a, ng, st);
    else if (a.io_f32) launch_synth_groups<false, float2>(a, ng, st);
    else launch_synth_groups<false, double2>(a, ng, st);
    return hipGetLastError();
}

hipError_t launch_vcoef(const void *S, const void *T, void *C, void *E, int in_f32, const double *scale, int divide, int ll1,
                        const LegArgs &v, int nf, hipStream_t st) {
    const int lmax = v.lmax - 1, ltr = v.ltr - 1;
    const long long in_fs = (long long)(lmax + 1) * (v.mmax + 1);
    const int nm = v.nm_run > 0 ? std::min(v.nm_run, v.nm) : v.nm;
    const dim3 grid((unsigned)nm * nf);
    if (in_f32)
        hipLaunchKernelGGL(k_vcoef<float>, grid, dim3(256), 0, st, (const float *)S, (const float *)T, (double2 *)C,
                           (double2 *)E, v.segbase, v.nseg_total, scale, divide, ll1, v.qb, v.qcc, v.coff, lmax, v.mres,
                           nm, ltr, v.m0_one, in_fs, v.spec_fstride, nf);
    else
        hipLaunchKernelGGL(k_vcoef<double>, grid, dim3(256), 0, st, (const double *)S, (const double *)T, (double2 *)C,
                           (double2 *)E, v.segbase, v.nseg_total, scale, divide, ll1, v.qb, v.qcc, v.coff, lmax, v.mres,
                           nm, ltr, v.m0_one, in_fs, v.spec_fstride, nf);
    return hipGetLastError();
}

hipError_t launch_vout(const void *H, void *S, void *T, int out_f32, const double *scale, int divide, int ll1,
                       int skip_m0, const LegArgs &v, int nf, hipStream_t st) {
    const int lmax = v.lmax - 1, ltr = v.ltr - 1;
    const long long out_fs = (long long)(lmax + 1) * (v.mmax + 1);
    const dim3 grid((unsigned)(v.mmax + 1) * nf);
    if (out_f32)
        hipLaunchKernelGGL(k_vout<float>, grid, dim3(256), 0, st, (const double2 *)H, (float *)S, (float *)T, scale,
                           divide, ll1, skip_m0, v.m0_one, v.qb, v.qcc, v.coff, lmax, v.mmax, v.mres, ltr, v.spec_fstride, out_fs,
                           nf);
    else
        hipLaunchKernelGGL(k_vout<double>, grid, dim3(256), 0, st, (const double2 *)H, (double *)S, (double *)T, scale,
                           divide, ll1, skip_m0, v.m0_one, v.qb, v.qcc, v.coff, lmax, v.mmax, v.mres, ltr, v.spec_fstride, out_fs,
                           nf);
    return hipGetLastError();
}

}  // namespace shtk
