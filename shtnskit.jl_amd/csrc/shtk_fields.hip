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
// Bound: FP64 issue (a matrix instruction holds the FP64 pipeline 64 cycles, 52 % of
// the kernel's cycles at lmax 1023), then LDS (operand staging) at 2 waves per
// SIMD.  16 fields at lmax 1023: 912 us (k_anal_w) -> 410 us; 37 fields at lmax 255: 85 -> 35 us; 16 at
// 511: 175 -> 79 us.  Tried: the pairs of a 512-pair block dealt to 4 waves with
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
    const int gs = item[0], im = item[1], s = item[2], coff = item[3];  // one load, short waves
    if (gs < 0) return;
    const int m = im * a.mres, np = a.np, nlat = a.nlat, lmax = a.lmax;
    const int l0 = m + s * DSEG, lend = min(l0 + DSEG, lmax + 1), lstop = min(lend, a.ltr + 1);
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
    const long long co = (long long)coff - m;
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
        const int p = max(pst + 64 * ch + lane, 0);
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
        nw = a.wlat ? a.wlat[p] : 1.0;
        if (2 * p == nlat - 1) nw *= 0.5;  // the equator's latitude is both halves of its pair
        if (pst + 64 * ch + lane < 0) nw = 0.0;
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
            asm volatile("s_nop 4");
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
    const double sc = l < lstop ? a.g * mfac_of(a.mfac_mode, m) * a.qcc[co + l] : 0.0;
    const double *src = tile + (8 * (lane >> 5) + 4 * (lane & 1) + (i >> 2)) * 64 + (i & 3) * 16;
    for (int f = 0; f < nfl; ++f) {
        const double2 v = *(const double2 *)(src + 2 * f);
        OT *d = col + 2 * ((size_t)f * a.spec_fstride + l);
        d[0] = (OT)(sc * v.x);
        d[1] = (OT)(sc * v.y);
    }
}

}  // namespace

// A group costs the same for 1 to 8 fields.  Against the single-field kernel, lmax
// 1023: 4 fields 228 (one group) against 256 us, 3 fields 228 against 192; so a
// last group of fewer than 4 fields goes to the single-field kernel.
int fields_anal_count(const LegArgs &a, int nfields) {
    if (a.seg != DSEG) return 0;
    const int rest = nfields % MX_FIELDS;
    return rest < 4 ? nfields - rest : nfields;
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

}  // namespace shtk
