// wr_kernels.h -- kernels of the MI355X RRTMG radiation path (templated on the optics precision R).
//
// Per column tile (n columns starting at col0), after the layer records of wr_rec.h:
//   k_colprep   column scalars: LW laytrop, precipitable water, cloud flag; SW day flag, column cloud
//               cover (max-random), SW laytrop
//   k_sflux     solar source of the 112 g-points of the day columns
//   k_day*      ordered compaction of the day columns (count, scan, scatter; deterministic order)
//   k_lw<B>, k_lwl64<B>  FP64: one lane per column, all g-points of band B in registers: the rtrnmc down
//               sweep and up sweep; the band's level fluxes go to its own planes
//   k_lwc<B>, k_lwl<B>  FP32: the same, with each layer's upward transmittance and source kept in the pool slot
//               by the down sweep, so that the up sweep needs no optics
//   k_sw<B>, k_swl<B>  one lane per day column: for each g-point of band B the two-stream adding method
//               as one bottom-up sweep (reflectance of the atmosphere below each level, to the pool
//               slot) and one top-down sweep (direct and diffuse beams, level fluxes)
//   k_post      level fluxes -> heating rates, top-first outputs
// (the kernels with an l read the band's tables from LDS).
#pragma once
#include <type_traits>

#include "wr_rec.h"

namespace wr {

typedef float f32x2v __attribute__((ext_vector_type(2)));
typedef float f32x4v __attribute__((ext_vector_type(4)));
typedef double f64x2v __attribute__((ext_vector_type(2)));

// Level fluxes of ONE band for one tile ([nrl+1][n] planes, written once per level; sw_clr0 [n]), in
// the band kernel's precision P: FP64 planes for the FP64 kernels; FP32 planes for the FP32 kernels,
// whose band sums are FP32 values, so that nothing is lost and k_post reads half the bytes.
template <typename P> struct AccT {
    WR_G P *lw_up, *lw_dn, *sw_up, *sw_dn, *sw_clr0;
};
// All band planes of a tile: LW band b at planes 2b, 2b+1; SW band b at planes 32+2b, 33+2b; the
// clear-sky surface SW of SW band b at base + 60 P + b n (in elements of the plane type; the space is
// sized for FP64).  k_post sums the bands in band order in FP64, which reproduces the sequential
// accumulation of the reference bit for bit.
struct BandAcc {
    WR_G double *base;
    long long P;  // (nrl + 1) * n
    int n;
    unsigned lw_mask, sw_mask;  // bands present (bit b)
};
template <typename P>
__host__ __device__ inline AccT<P> band_acc(const BandAcc &ba, int id)  // id 0..15 LW, 16..29 SW
{
    AccT<P> a = {nullptr, nullptr, nullptr, nullptr, nullptr};
    WR_G P *base = (WR_G P *)ba.base;
    if (id < 16) {
        a.lw_up = base + (size_t)(2 * id) * ba.P;
        a.lw_dn = base + (size_t)(2 * id + 1) * ba.P;
    } else {
        const int b = id - 16;
        a.sw_up = base + (size_t)(32 + 2 * b) * ba.P;
        a.sw_dn = base + (size_t)(33 + 2 * b) * ba.P;
        a.sw_clr0 = base + (size_t)60 * ba.P + (size_t)b * ba.n;
    }
    return a;
}

// Column scalars of a tile, one thread per column; the layer logs come from k_layers.
static __global__ void __launch_bounds__(256) k_colprep(ColIn in, int col0, int n, ColScal cs)
{
#pragma clang fp contract(off)
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    if (t >= valid_cols(in, col0, n)) {  // padding column of a shorter tile: not in the day list
        cs.day[t] = 0;
        return;
    }
    const int i = col0 + t;
    const RadCol rc{in, i, in.nlay + 1};
    const int nrl = rc.nrl;
    const double tem1g = 100.0 * CON_G;
    const double tem2c = 1.0e-20 * 1.0e3 * CON_AVGD;
    double tem1 = 0.0, tem2 = 0.0, z0 = 1.0, z1 = 1.0;
    int lt = 0, lcf = 0, swlt = nrl;
    uint32_t blocks = 0;
    double pb = rc.plvl(nrl);
#pragma unroll 4
    for (int k = 0; k < nrl; ++k) {
        const int kin = nrl - 1 - k;
        const double pt = rc.plvl(kin);
        const double dlp = pb - pt;
        pb = pt;
        const double qv = rc.qlyr(kin);
        const double h2ovmr = fmax(0.0, qv * AMDW / (1.0 - qv));
        const double tem0 = (1.0 - h2ovmr) * CON_AMD + h2ovmr * CON_AMW;
        const double cdry = tem2c * dlp / (tem1g * tem0 * (1.0 + h2ovmr));
        const double ca0 = fmax(0.0, cdry * h2ovmr);
        tem1 = tem1 + cdry + ca0;
        tem2 = tem2 + ca0;
        if (cs.la[(size_t)kin * n + t] > 4.56) {
            lt += 1;
            swlt = k + 1;
        }
        const double ct = rc.cfrac(kin);
        if (ct > EPS) lcf = 1;
        if (ct > 0.0) blocks |= 1u << (k >> 2);
        if (ct > FTINY) {
            z1 = fmin(z1, 1.0 - ct);
        } else if (z1 < 1.0) {
            z0 = z0 * z1;
            z1 = 1.0;
        }
    }
    cs.lw_laytrop[t] = lt;
    cs.lcf1[t] = lcf;
    cs.cblk[t] = blocks;
    const double tem0p = 10.0 * tem2 / (AMDW * tem1 * CON_G);
    cs.pwv[t] = tem0p * rc.plvl(nrl);
    const int day = in.cosz[i] >= 1.0e-4;
    cs.day[t] = day;
    if (!day) return;
    z0 = z0 * z1;
    if (z0 <= FTINY) z0 = 0.0;
    if (z0 > ONEMINUS) z0 = 1.0;
    cs.zcf1[t] = 1.0 - z0;
    cs.zcf0[t] = z0;
    cs.sw_laytrop[t] = swlt;
}

// Solar source per g-point (phys_rrtm_sw_taumol.cu:59-120), one thread per (day-list entry, band).
template <typename R>
__global__ void __launch_bounds__(64) k_sflux(const Tabs<R> *__restrict__ T, ColIn in, RunPar par, int col0, int n, ColScal cs,
                                              R *__restrict__ sflux)
{
    const int tt = blockIdx.x * 64 + threadIdx.x, b = blockIdx.y;
    if (tt >= *cs.nday) return;
    const int t = cs.dlist[tt];
    const RadCol rc{in, col0 + t, in.nlay + 1};
    const int nrl = rc.nrl, swlt = cs.sw_laytrop[t];
    const int jb = b + 16, ibd = T->ibx[b], njb = SW_NG[b], ns = SW_NS[b], lr = T->layreffr[b];
    if (jb == 16 || jb == 20 || jb == 23 || jb == 25 || jb == 26 || jb == 29) {
        for (int j = 0; j < njb; ++j) sflux[(size_t)(ns + j) * n + t] = T->sf01[(ibd - 1) * 16 + j];
        return;
    }
    if (jb == 27) {
        for (int j = 0; j < njb; ++j) sflux[(size_t)(ns + j) * n + t] = T->scalekur * T->sf01[(ibd - 1) * 16 + j];
        return;
    }
    auto jp = [&](int k) {  // reference pressure index of surface-first layer k
        return imax(1, imin(58, (int)(36.0 - 5.0 * (cs.la[(size_t)(nrl - 1 - k) * n + t] + 0.04))));
    };
    const bool upper = jb == 17 || jb == 28;
    const WR_G R *tab = upper ? T->sf02 : T->sf03;
    const int mfs = upper ? 5 : 9, k0 = upper ? swlt : 1, k1 = upper ? nrl - 1 : swlt - 1;
    int ks = upper ? nrl : swlt;
    bool found = false;  // no early exit, so that the loads of several layers are in flight
    int prev = jp(k0 - 1);
#pragma unroll 8
    for (int k = k0; k <= k1; ++k) {
        const int cur = jp(k);
        if (!found && prev < lr && cur >= lr) ks = k + 1, found = true;
        prev = cur;
    }
    SwLay<R> L;
    const int kin = nrl - 1 - (ks - 1);
    sw_layer<R>(T, rc, par, kin, cs.la[(size_t)kin * n + t], L);
    const int i1 = T->ix1[b] - 1, i2 = T->ix2[b] - 1;
    R colm1 = (R)0, colm2 = (R)0;
#pragma unroll
    for (int m = 0; m < 6; ++m) {
        colm1 = m == i1 ? L.colamt[m] : colm1;
        colm2 = m == i2 ? L.colamt[m] : colm2;
    }
    const R speccomb = colm1 + T->sw_strrat[b] * colm2;
    const R specmult = T->sw_specwt[b] * fmin((R)0.999999, rdiv<R>(colm1, speccomb));
    const int jsi = (int)specmult;
    const int js = 1 + jsi;
    const R fs = specmult - (R)jsi;
    const int base = ((ibd - 1) * mfs) * 16;
    for (int j = 0; j < njb; ++j) {
        const R a = tab[base + (js - 1) * 16 + j];
        const R c = tab[base + js * 16 + j];
        sflux[(size_t)(ns + j) * n + t] = a + fs * (c - a);
    }
}

// ---- ordered compaction of the day columns of a tile --------------------------------------------
// Three small kernels, all reads coalesced: per-segment day counts (DAY_SEG columns per 256-thread
// block), one workgroup's exclusive scan of the counts, then each segment writes its day columns in
// column order.  The result is the same ordered list whatever the launch shape.
constexpr int DAY_T = 256, DAY_IT = 8, DAY_SEG = DAY_T * DAY_IT;

// the whole list of a tile of up to DAY_SMALL columns by one workgroup
constexpr int DAY_SMALL = 16384;
static __global__ void __launch_bounds__(1024) k_daylist_small(const int *__restrict__ day, int n, int *__restrict__ nday,
                                                               int *__restrict__ dlist)
{
    __shared__ int cnt[16];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int base = 0;
    for (int j0 = 0; j0 < n; j0 += 1024) {
        const int j = j0 + (int)threadIdx.x;
        const bool f = j < n && day[j] != 0;
        const uint64_t m = __ballot(f);
        if (lane == 0) cnt[w] = __popcll(m);
        __syncthreads();
        int before = 0, total = 0;
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            before += q < w ? cnt[q] : 0;
            total += cnt[q];
        }
        if (f) dlist[base + before + __popcll(m & (((uint64_t)1 << lane) - 1))] = j;
        base += total;
        __syncthreads();
    }
    if (threadIdx.x == 0) *nday = base;
}

// exclusive prefix of v over the 256 threads of the block (4 waves); total = the block sum
__device__ __forceinline__ int block_excl_scan256(int v, int *lds, int &total)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63) lds[w] = x;
    __syncthreads();
    int before = 0;
    total = 0;
#pragma unroll
    for (int q = 0; q < DAY_T / 64; ++q) {
        const int c = lds[q];
        before += (q < w) ? c : 0;
        total += c;
    }
    __syncthreads();  // lds is reused by the next call
    return before + x - v;
}

static __global__ void __launch_bounds__(DAY_T) k_daycount(const int *__restrict__ day, int n, int *__restrict__ seg)
{
    __shared__ int lds[DAY_T / 64];
    const int j0 = blockIdx.x * DAY_SEG + threadIdx.x;
    int c = 0;
#pragma unroll
    for (int it = 0; it < DAY_IT; ++it) {
        const int j = j0 + it * DAY_T;
        c += (j < n && day[j] != 0) ? 1 : 0;
    }
    int tot;
    (void)block_excl_scan256(c, lds, tot);
    if (threadIdx.x == 0) seg[blockIdx.x] = tot;
}

// in place: segment counts -> exclusive segment offsets; *nday = the total
static __global__ void __launch_bounds__(1024) k_dayscan(int *__restrict__ seg, int nseg, int *__restrict__ nday)
{
    __shared__ int part[1024];
    const int tid = threadIdx.x;
    int carry = 0;
    for (int base = 0; base < nseg; base += 1024) {
        const int v = (base + tid < nseg) ? seg[base + tid] : 0;
        part[tid] = v;
        __syncthreads();
        for (int off = 1; off < 1024; off <<= 1) {  // Hillis-Steele inclusive scan
            const int u = (tid >= off) ? part[tid - off] : 0;
            __syncthreads();
            part[tid] += u;
            __syncthreads();
        }
        if (base + tid < nseg) seg[base + tid] = carry + part[tid] - v;
        const int tot = part[1023];
        __syncthreads();
        carry += tot;
    }
    if (tid == 0) *nday = carry;
}

static __global__ void __launch_bounds__(DAY_T) k_dayscatter(const int *__restrict__ day, int n, const int *__restrict__ seg,
                                                         int *__restrict__ dlist)
{
    __shared__ int lds[DAY_T / 64];
    const int j0 = blockIdx.x * DAY_SEG + threadIdx.x;
    int run = seg[blockIdx.x];
    for (int it = 0; it < DAY_IT; ++it) {
        const int j = j0 + it * DAY_T;
        const int f = (j < n && day[j] != 0) ? 1 : 0;
        int tot;
        const int r = block_excl_scan256(f, lds, tot);
        if (f) dlist[run + r] = j;
        run += tot;
    }
}

// ---- LW band kernel (rtrnmc, McICA) -------------------------------------------------------------
constexpr double LW_A0[16] = {1.66, 1.55, 1.58, 1.66, 1.54, 1.454, 1.89, 1.33, 1.668, 1.66, 1.66, 1.66, 1.66, 1.66, 1.66, 1.66};
constexpr double LW_A1[16] = {0.00, 0.25, 0.22, 0.00, 0.13, 0.446, -0.10, 0.40, -0.006, 0.00, 0.00, 0.00, 0.00, 0.00, 0.00, 0.00};
constexpr double LW_A2[16] = {0.00, -12.0, -11.7, 0.00, -0.72, -0.243, 0.19, -0.062, 0.414, 0.00, 0.00, 0.00, 0.00, 0.00, 0.00, 0.00};

template <typename R> struct GasT {  // rtrnmc gas transmittance and source factor of one g, one layer
    R trng, atrgas, gasfac, odepth;
};
template <typename R> __device__ __forceinline__ GasT<R> lw_gas(const Tabs<R> *__restrict__ T, R sdif, R tau)
{
    GasT<R> q;
    R od = fmax((R)0, sdif * tau);
    if (od <= (R)0.06) {
        q.atrgas = od - (R)0.5 * od * od;
        q.trng = (R)1 - q.atrgas;
        q.gasfac = (R)0.166667 * od;
    } else {
        const R tblind = od / ((R)(1.0 / 0.278) + od);
        const int itgas = imin(NTBL, (int)((R)10000 * tblind + (R)0.5));
        if constexpr (sizeof(R) == 4) {
            const LutF l = lut_f32(itgas, true);
            q.trng = l.e, q.gasfac = l.tfn, od = l.tau;
        } else {
            q.trng = T->exp_tbl[itgas];
            q.gasfac = T->tfn_tbl[itgas];
            od = T->tau_tbl[itgas];
        }
        q.atrgas = (R)1 - q.trng;
    }
    q.odepth = od;
    return q;
}
template <typename R> __device__ __forceinline__ void lw_tot(const Tabs<R> *__restrict__ T, R odtot, R &totfac, R &atrtot)
{
    if (odtot < (R)0.06) {
        totfac = (R)0.166667 * odtot;
        atrtot = odtot - (R)0.5 * odtot * odtot;
    } else {
        const R tblind = odtot / ((R)(1.0 / 0.278) + odtot);
        const int ittot = imin(NTBL, (int)((R)10000 * tblind + (R)0.5));
        if constexpr (sizeof(R) == 4) {
            const LutF l = lut_f32(ittot, true);
            totfac = l.tfn, atrtot = (R)1 - l.e;
        } else {
            totfac = T->tfn_tbl[ittot];
            atrtot = (R)1 - T->exp_tbl[ittot];
        }
    }
}

// Learned gas optics of one tile (surrogate path): normalised network outputs Y[j * S + k * n + t] (BF16;
// S the padded row stride)
// (j < 504 outputs, surface-first layer k, tile column t), de-normalised as y * tstd[j] + tmean[j];
// flag[t] != 0 sends column t back to the table optics (inputs outside the training envelope);
// bands: bit b set when band b uses the network (LW bands at bits 0..15, SW bands at 16..29).
struct Surr {
    const WR_G __bf16 *Y;
    const WR_G float *tmean, *tstd;
    const WR_G int *flag;
    long long S;
    uint32_t bands;
    __device__ __forceinline__ int table(int t, int bit) const { return ((bands >> bit) & 1u) ? flag[t] : 1; }
};

__device__ __forceinline__ float surr_out(const Surr &sg, int j, size_t s)
{
    return (float)sg.Y[(size_t)j * sg.S + s] * sg.tstd[j] + sg.tmean[j];
}

template <typename R, int B, int NGL = LW_NG[B]>
__device__ __forceinline__ void surr_lw(const Surr &sg, size_t s, R *tau, R *fr, int g0 = 0)
{
#pragma unroll
    for (int jj = 0; jj < NGL; ++jj) {
        const int g = g0 + jj;
        tau[jj] = (R)__expf(surr_out(sg, LW_NS[B] + g, s));
        fr[jj] = (R)fminf(1.0f, fmaxf(0.0f, surr_out(sg, 140 + LW_NS[B] + g, s)));
    }
}

// ---- per-wave level slots of the band kernels -------------------------------------------------------
// What a column's second sweep takes over from its first lives in a slot of the context's pool, not in
// per-lane private arrays (which would need kilobytes of scratch per lane, backed by the runtime on every
// HIP queue): one slot per resident 64-lane wave (the kernels loop over column blocks, so the slot count
// bounds the memory), laid out [level][g][lane][value], so that every access is one contiguous run of the
// wave and the offset of a g-point within a level is a compile-time constant.  A slot holds nk = nlay + 2
// levels of nv values per g-point.
__host__ __device__ constexpr size_t cache_slot_bytes(int nv, int ng, int nk, int rbytes)
{
    return (size_t)64 * nv * ng * nk * rbytes;
}

// Optics chunks and wave bounds of the LW band kernels, per band.  These kernels wait on memory most of the time
// (0.65 to 0.8 of the wave cycles on the 954x835x60 grid), so more resident waves per SIMD pay as far as the
// registers allow:
// * chunk: g-points whose optics are evaluated together, about four.  A scheduling barrier between chunks keeps
//   the gathers of one from being hoisted above the arithmetic of the one before, which bounds the registers; within
//   a chunk nothing branches per g-point, so that its chains overlap.  The arithmetic of every g-point is
//   that of the whole band at once;
// * waves: waves per SIMD the compiler must fit.  FP32: three in the bands of two gases with 12 or more g-points (3, 5,
//   7 and 9 still have 96 to 132 bytes of scratch a lane there), four in the others, of which 6, 8, 12 and 13 have 20 to
//   140 bytes that three waves do not need.  Alone on 796,590 columns, four waves / three: band 1 2.54 / 2.62 ms, 2 2.75
//   / 2.84, 6 2.30 / 2.32, 8 2.46 / 2.41, 10 1.74 / 1.79, 11 2.18 / 2.22, 12 2.25 / 2.35, 15 1.22 / 1.28, 16 1.11 / 1.19;
//   only band 13, with 4 g-points, is much the slower at four: 2.64 / 1.70.  FP64: two everywhere; at three the LW
//   kernels of a 796,590-column call took 205 ms in place of 147, from up to 530 bytes of scratch a lane.
// WR_LWC_WAVES / WR_LW64_WAVES > 0 or WR_LW_CHUNK / WR_LW64_CHUNK >= 0 override the tables for every
// band (tuning builds).
constexpr int LWC_WAVES[16] = {4, 4, 3, 3, 3, 4, 3, 4, 3, 4, 4, 4, 4, 4, 4, 4};
constexpr int LWC_CHUNK[16] = {5, 4, 4, 2, 4, 4, 4, 4, 4, 3, 4, 4, 4, 2, 2, 2};
constexpr int LW64_WAVES[16] = {2, 2, 2, 2, 2, 2, 2, 2, 2, 2, 2, 2, 2, 2, 2, 2};
constexpr int LW64_CHUNK[16] = {5, 4, 4, 2, 4, 4, 4, 4, 4, 3, 4, 4, 4, 2, 2, 2};
#ifndef WR_LWC_WAVES
#define WR_LWC_WAVES 0
#endif
#ifndef WR_LW_CHUNK
#define WR_LW_CHUNK -1
#endif
#ifndef WR_LW64_WAVES
#define WR_LW64_WAVES 0
#endif
#ifndef WR_LW64_CHUNK
#define WR_LW64_CHUNK -1
#endif
template <int B> constexpr int lwc_waves() { return WR_LWC_WAVES > 0 ? WR_LWC_WAVES : LWC_WAVES[B]; }
template <int B> constexpr int lw64_waves() { return WR_LW64_WAVES > 0 ? WR_LW64_WAVES : LW64_WAVES[B]; }
// the smallest divisor of ngl that is >= want (ngl when want <= 0)
constexpr int chunk_of(int ngl, int want)
{
    if (want <= 0) return ngl;
    for (int c = want; c < ngl; ++c)
        if (ngl % c == 0) return c;
    return ngl;
}
template <int B> constexpr int lw_chunk() { return chunk_of(LW_NG[B], WR_LW_CHUNK >= 0 ? WR_LW_CHUNK : LWC_CHUNK[B]); }
template <int B> constexpr int lw64_chunk() { return chunk_of(LW_NG[B], WR_LW64_CHUNK >= 0 ? WR_LW64_CHUNK : LW64_CHUNK[B]); }
// ---- level sums over the g-points of a band ---------------------------------------------------------
// A band's level flux is the sum of its g-points' contributions in g order.  A lane either holds all NG
// g-points of its column (GW = NG) and adds them itself, or GW of them, the others being with the other
// waves of its workgroup (k_sweep): then the contributions of SUM_LEVELS levels are left in LDS, and after a
// barrier each wave adds those of its levels, again in g order, so that the sums are the same bits.
// NQ: quantities per level (4: two skies, with half as many levels between barriers).  The levels come in order
// row0, row0 + step, ...; emit(row, sums) stores one.
constexpr int SUM_LEVELS = 4;
template <typename R> constexpr size_t sum_lds_bytes() { return sizeof(R) * SUM_LEVELS * 64 * 24; }  // LW 16 g, SW 2 x 12 g
template <typename R> struct Share {  // a wave's part of a column's g-points (split bands)
    R *xs;         // LDS of the workgroup, sum_lds_bytes
    int g0, wave;  // first g-point, wave index
};
template <typename R, int NG, int GW, int NQ> struct LevelSum {
    static constexpr int SL = NQ > 2 ? SUM_LEVELS / 2 : SUM_LEVELS;
    Share<R> sh;
    int lane, row, step, cnt;
    __device__ __forceinline__ void begin(int row0, int step_) { row = row0, step = step_, cnt = 0; }
    template <typename EMIT> __device__ __forceinline__ void put(const R (&v)[NQ][GW], EMIT &&emit)
    {
        if constexpr (GW == NG) {
            R sum[NQ];
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                sum[q] = (R)0;
#pragma unroll
                for (int j = 0; j < GW; ++j) sum[q] = sum[q] + v[q][j];
            }
            emit(row, sum);
            row += step;
        } else {
#pragma unroll
            for (int q = 0; q < NQ; ++q)
#pragma unroll
                for (int j = 0; j < GW; ++j) sh.xs[((cnt * NQ + q) * NG + sh.g0 + j) * 64 + lane] = v[q][j];
            if (++cnt == SL) finish(emit);
        }
    }
    template <typename EMIT> __device__ __forceinline__ void finish(EMIT &&emit)
    {
        if constexpr (GW < NG) {
            __syncthreads();
            for (int l = sh.wave; l < cnt; l += NG / GW) {
                R sum[NQ];
#pragma unroll
                for (int q = 0; q < NQ; ++q) {
                    sum[q] = (R)0;
#pragma unroll
                    for (int g = 0; g < NG; ++g) sum[q] = sum[q] + sh.xs[((l * NQ + q) * NG + g) * 64 + lane];
                }
                emit(row + step * l, sum);
            }
            __syncthreads();
            row += step * cnt;
            cnt = 0;
        }
    }
};

// ---- LW band kernels (rtrnmc, McICA) ------------------------------------------------------------
// One lane per column, one wave per 64-column block; the layer's set-up comes from its record row
// (wr_rec.h), the McICA bits of the band's g-points from one word per layer.  The g-points of a layer run
// in chunks: a chunk's table gathers, its transmittances and its radiances are done before the next
// chunk's gathers are issued (a scheduling barrier stands between), which bounds the registers.  Inside a chunk
// nothing branches per g-point: both forms of the transmittance are evaluated and selected, so that the
// chunk's chains (division, table gather or exponential) overlap; a form that no lane of the wave needs
// is skipped as a whole.

// Transmittance, source factor and optical depth of the LW tables at od (rtrnmc's tblind quantisation).
// FP64 takes the transmittance from the table etab that the oracle reproduces (LDS in the staged kernels) and evaluates
// the rest of the entry (lut_rest): the gather of whole entries from L2, 64 lanes on 64 lines, bound the FP64 kernels
// (15 TB/s of L2 reads at 0.34 of the issue slots).  FP32 evaluates the entry.  FP32: tblind of the largest
// depths rounds to 1, where the table ends in (1e-20, 1, 1e10); the index stops just below it, which gives
// those values to FP32 accuracy.  tau and 1 / tau share one reciprocal.
template <typename R, typename PE> __device__ __forceinline__ void lw_lut(PE etab, R od, R &e, R &tfn, R &tau)
{
    if constexpr (sizeof(R) == 4) {
        const R tb = od * __builtin_amdgcn_rcpf((R)(1.0 / 0.278) + od);
        const R fi = fmin(floorf(__builtin_fmaf((R)NTBL, tb, (R)0.5)), (R)9999.999);
        const R ci = (R)NTBL - fi;
        const R r = __builtin_amdgcn_rcpf(fi * ci);
        tau = ((R)(1.0 / 0.278) * fi) * (fi * r);
        const R it = (ci * r) * (ci * (R)0.278);
        e = fmax(M<R>::exp(-tau), (R)1.0e-20);
        const R big = __builtin_fmaf((R)-2, it - e * __builtin_amdgcn_rcpf((R)1 - e), (R)1);
        tfn = tau < (R)0.06 ? tau * (R)(1.0 / 6.0) : big;
    } else {
        const R tb = od / ((R)(1.0 / 0.278) + od);
        const int i = imin(NTBL, (int)((R)NTBL * tb + (R)0.5));
        e = etab[i];
        lut_rest(i, NTBL, e, tfn, tau);
    }
}

template <typename R, int CH> struct GasV {  // CH g-points: transmittance, absorptance, source factor, optical depth
    R tr[CH], at[CH], gf[CH], od[CH];
};
template <typename R, int CH, typename PE>
__device__ __forceinline__ void lw_gas_v(PE etab, R sdif, R taer, const R *tau, GasV<R, CH> &q)
{
    bool any = false;
#pragma unroll
    for (int j = 0; j < CH; ++j) {
        const R od = fmax((R)0, sdif * (tau[j] + taer));
        q.od[j] = od;
        q.at[j] = od - (R)0.5 * od * od;
        q.tr[j] = (R)1 - q.at[j];
        q.gf[j] = (R)0.166667 * od;
        any |= !(od <= (R)0.06);
    }
    if (__any(any)) {
#pragma unroll
        for (int j = 0; j < CH; ++j) {
            R e, tfn, ta;
            lw_lut<R>(etab, q.od[j], e, tfn, ta);
            const bool big = !(q.od[j] <= (R)0.06);
            q.tr[j] = big ? e : q.tr[j];
            q.at[j] = big ? (R)1 - e : q.at[j];
            q.gf[j] = big ? tfn : q.gf[j];
            q.od[j] = big ? ta : q.od[j];
        }
    }
}
// the same for the total (gas plus cloud) optical depth: transmittance, absorptance, source factor
template <typename R, int CH, typename PE>
__device__ __forceinline__ void lw_tot_v(PE etab, const R *od, R odcld, R *tr, R *at, R *gf)
{
    bool any = false;
#pragma unroll
    for (int j = 0; j < CH; ++j) {
        const R x = od[j] + odcld;
        at[j] = x - (R)0.5 * x * x;
        tr[j] = (R)1 - at[j];
        gf[j] = (R)0.166667 * x;
        any |= !(x < (R)0.06);
    }
    if (__any(any)) {
#pragma unroll
        for (int j = 0; j < CH; ++j) {
            const R x = od[j] + odcld;
            R e, tfn, ta;
            lw_lut<R>(etab, x, e, tfn, ta);
            const bool big = !(x < (R)0.06);
            tr[j] = big ? e : tr[j];
            at[j] = big ? (R)1 - e : at[j];
            gf[j] = big ? tfn : gf[j];
        }
    }
}

// What the LW transfer of one column needs besides its layers.
template <typename R> struct LwCol {
    int i, t, nrl, table;
    R sdif, semis, reflct;
};
template <typename R, int B, bool SURR>
__device__ __forceinline__ LwCol<R> lw_col(const ColIn &in, int col0, const ColScal &cs, const Surr &sg, int t)
{
    LwCol<R> c;
    c.i = col0 + t, c.t = t, c.nrl = in.nlay + 1;
    c.table = SURR ? sg.table(t, B) : 1;
    const double pwv = cs.pwv[t];
    c.sdif = (R)((B == 0 || B == 3 || B == 9) ? 1.66 : fmin(1.80, fmax(1.50, LW_A0[B] + LW_A1[B] * exp_d(LW_A2[B] * pwv))));
    const double sfe = in.emis[c.i];
    c.semis = (R)((sfe > EPS && sfe <= 1.0) ? sfe : 1.0);
    c.reflct = (R)1 - c.semis;
    return c;
}

// A layer of a column as the sweeps use it: Planck sources of the layer and of the level below, cloud.
template <typename R> struct LwLayer {
    LwLay<R> L;
    R blay, bbot;   // Planck function at the layer and at the level below it
    R taer, odcld;  // aerosol absorption depth; cloud depth times the diffusivity secant
    bool cloudy;    // this lane's layer holds cloud
};
template <typename R, int B>
__device__ __forceinline__ void lw_get(const Tabs<R> *__restrict__ T, const ColIn &in, const RunPar &par, const RecPtrs &rp,
                                       const LwCol<R> &c, int blk, int lane, int k, LwLayer<R> &y)
{
    const LRow<R> row = lrow<R>(rp, blk, k, lane);
    const uint32_t w0 = row.w(0), w1 = row.w(1);
    lrow_get<R>(row, w0, par, y.L);
    y.blay = planck_of<R>(T, B, (int)(w0 >> 22), row.f(LF_PL));
    y.bbot = planck_of<R>(T, B, (int)(w1 & 255u), row.f(LF_PB));
    y.cloudy = (w1 & 256u) != 0;
    const RadCol rc{in, c.i, c.nrl};
    y.taer = (R)rc.aer_lw_tau(B, c.nrl - 1 - k);  // tautot = taug + tauaer
    y.odcld = (R)0;
    if (__any(y.cloudy)) {
        double rl = par.re_liq, ri = par.re_ice, rain = 0.0;
        if (y.cloudy) rc.props(c.nrl - 1 - k, par.re_liq, par.re_ice, rl, ri, rain);
        const R tc = lw_taucld_r<R>(T, B, row.f(LF_LIQ), row.f(LF_ICE), rl, ri, rain);
        y.odcld = c.sdif * (y.cloudy ? tc : (R)0);
    }
}
// gas optical depth and Planck fraction of g-points g0 .. g0 + CH - 1 of a layer
template <typename R, int B, bool SURR, int CH, typename BT>
__device__ __forceinline__ void lw_taufr(const Tabs<R> *__restrict__ T, const BT &Bt, const Surr &sg, const LwCol<R> &c, int n,
                                         int k, const LwLay<R> &L, int g0, R *tau, R *fr)
{
    if (SURR && !c.table)
        surr_lw<R, B, CH>(sg, (size_t)k * n + c.t, tau, fr, g0);
    else
        lw_optics_t<R, B, CH>(T, Bt, L, tau, fr, g0);
}

// One column of LW band B in FP64, optics from the band tables Bt: the down sweep also forms each layer's
// upward gas source and, where a g-point has cloud, the cloud correction, and leaves them with the transmittance
// in the wave's pool slot, so that the up sweep needs no optics.  Every sum and product in the reference's order.
// Slot, per lane: [layer][g] {transmittance, upward gas source}; [layer][g] cloud minus gas source, written and
// read only where a chunk has cloud; [layer] cloud transmittance.
__host__ __device__ constexpr size_t lw64_slot_bytes(int ng, int nk) { return (size_t)64 * sizeof(double) * nk * (3 * ng + 1); }
template <typename R, int B, bool SURR, typename BT>
__device__ __forceinline__ void lw_column(const Tabs<R> *__restrict__ T, const BT &Bt, const ColIn &in, const RunPar &par,
                                          int col0, int n, const ColScal &cs, const RecPtrs &rp, const AccT<R> &acc,
                                          const Surr &sg, int blk, int lane, WR_G char *slot)
{
    constexpr int NG = LW_NG[B], GW = NG, CH = lw64_chunk<B>();
    const Share<R> sh{nullptr, 0, 0};
    const int nv = valid_cols(in, col0, n);
    if (blk * 64 >= nv) return;
    const bool ok = blk * 64 + lane < nv;  // lanes past the last column repeat it and store nothing
    const int rl = ok ? lane : nv - 1 - blk * 64, t = blk * 64 + rl;
    const LwCol<R> c = lw_col<R, B, SURR>(in, col0, cs, sg, t);
    const int nrl = c.nrl;
    WR_G f64x2v *const tg = (WR_G f64x2v *)slot + lane;
    WR_G R *const cg = (WR_G R *)((WR_G f64x2v *)slot + (size_t)nrl * NG * 64) + lane, *const ef = cg + (size_t)nrl * NG * 64;
    if (ok) acc.lw_dn[(size_t)nrl * n + t] = (R)0;  // no downward LW at the top
    R rad[1][GW];
#pragma unroll
    for (int g = 0; g < GW; ++g) rad[0][g] = (R)0;
    LevelSum<R, NG, GW, 1> sum{sh, lane, 0, 0, 0};
    auto dn = [&](int row, const R *s) {
        if (ok) acc.lw_dn[(size_t)row * n + t] = s[0];
    };
    auto up = [&](int row, const R *s) {
        if (ok) acc.lw_up[(size_t)row * n + t] = s[0];
    };
    R btop = (R)0;  // Planck function at the level above the layer; above the top layer its own temperature's
    sum.begin(nrl - 1, -1);
    for (int k = nrl - 1; k >= 0; --k) {  // down sweep, top to surface
        LwLayer<R> y;
        lw_get<R, B>(T, in, par, rp, c, blk, rl, k, y);
        const uint32_t bits = y.cloudy ? mword(rp.mlw, rp.row(blk, k), MROW_LW, B, rl) : 0u;
        if (k == nrl - 1) btop = y.blay;
        const R dd = y.bbot - y.blay, du = btop - y.blay;
        R efclrfr = (R)1;
        if (__any(y.cloudy)) {
            efclrfr = (R)1 - ((R)1 - M<R>::exp(-y.odcld));
            ef[(size_t)k * 64] = efclrfr;
        }
        R sfc0[GW];
#pragma unroll
        for (int g0 = 0; g0 < GW; g0 += CH) {
            R tau[CH], fr[CH];
            lw_taufr<R, B, SURR, CH>(T, Bt, sg, c, n, k, y.L, g0, tau, fr);
            GasV<R, CH> q;
            lw_gas_v<R, CH>(Bt.etab, c.sdif, y.taer, tau, q);
            R nr[CH], gas[CH], gup[CH];
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                gas[j] = fr[j] * (y.blay + dd * q.gf[j]) * q.at[j];
                gup[j] = fr[j] * (y.blay + du * q.gf[j]) * q.at[j];
                tg[((size_t)k * NG + g0 + j) * 64] = (f64x2v){q.tr[j], gup[j]};
                nr[j] = rad[0][g0 + j] * q.tr[j] + gas[j];
            }
            const uint32_t cb = bits >> g0;
            if (__any(cb & ((1u << CH) - 1u))) {
                R tr[CH], at[CH], gf[CH];
                lw_tot_v<R, CH>(Bt.etab, q.od, y.odcld, tr, at, gf);
#pragma unroll
                for (int j = 0; j < CH; ++j) {
                    const R td = fr[j] * (y.blay + dd * gf[j]) * at[j], tu = fr[j] * (y.blay + du * gf[j]) * at[j];
                    cg[((size_t)k * NG + g0 + j) * 64] = tu - gup[j];
                    const R rc = rad[0][g0 + j] * q.tr[j] * efclrfr + gas[j] + (td - gas[j]);
                    nr[j] = (cb >> j) & 1u ? rc : nr[j];
                }
            }
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                rad[0][g0 + j] = nr[j];
                if (k == 0) {  // surface emission and reflection start the upward sweep
                    const R rad0 = c.semis * fr[j] * y.bbot;
                    sfc0[g0 + j] = rad0 + c.reflct * nr[j];
                }
            }
            if constexpr (CH < GW) __builtin_amdgcn_sched_barrier(0);
        }
        sum.put(rad, dn);
        if (k == 0) {
#pragma unroll
            for (int g = 0; g < GW; ++g) rad[0][g] = sfc0[g];
        }
        btop = y.bbot;
    }
    sum.finish(dn);
    sum.begin(0, 1);
    sum.put(rad, up);
    for (int k = 0; k < nrl; ++k) {  // up sweep, surface to top
        const bool cloudy = (lrow<R>(rp, blk, k, rl).w(1) & 256u) != 0;
        uint32_t bits = 0;
        R efclrfr = (R)1;
        if (__any(cloudy)) {
            efclrfr = ef[(size_t)k * 64];
            if (cloudy) bits = mword(rp.mlw, rp.row(blk, k), MROW_LW, B, rl);
        }
#pragma unroll
        for (int g0 = 0; g0 < GW; g0 += CH) {
            const uint32_t cb = bits >> g0;
            f64x2v v[CH];
            R nr[CH];
#pragma unroll
            for (int j = 0; j < CH; ++j) v[j] = tg[((size_t)k * NG + g0 + j) * 64];
#pragma unroll
            for (int j = 0; j < CH; ++j) nr[j] = rad[0][g0 + j] * v[j].x + v[j].y;
            if (__any(cb & ((1u << CH) - 1u))) {
#pragma unroll
                for (int j = 0; j < CH; ++j) {
                    const R rc = rad[0][g0 + j] * v[j].x * efclrfr + v[j].y + cg[((size_t)k * NG + g0 + j) * 64];
                    nr[j] = (cb >> j) & 1u ? rc : nr[j];
                }
            }
#pragma unroll
            for (int j = 0; j < CH; ++j) rad[0][g0 + j] = nr[j];
        }
        sum.put(rad, up);
    }
    sum.finish(up);
}

template <typename R, int B, bool SURR = false, bool EXT = true>
__global__ void __launch_bounds__(64, lw64_waves<B>()) k_lw(const Tabs<R> *__restrict__ T, ColIn in_, RunPar par, int col0,
                                           int n, ColScal cs, RecPtrs rp, AccT<R> acc, Surr sg, char *__restrict__ pool)
{
    const ColIn in = band_in<EXT>(in_);
    WR_G char *slot = (WR_G char *)(pool + (size_t)blockIdx.x * lw64_slot_bytes(LW_NG[B], in.nlay + 2));
    for (int blk = blockIdx.x; blk * 64 < n; blk += gridDim.x)
        lw_column<R, B, SURR>(T, T->lw[B], in, par, col0, n, cs, rp, acc, sg, blk, (int)threadIdx.x, slot);
}

// The band tables of an LDS image (the LwImg order), absb from PB: the image's when the image holds it,
// the global table otherwise.  A table the band does not have points at the image start and is never
// read.  The offsets are multiples of 4 elements (the & ~3 states it, so that 4 g-points of a row
// load as one 16-byte read).
template <typename R, int B, typename PB>
__device__ __forceinline__ auto lds_band(const WR_L R *lt, const LwImg<R> &im, const LwBand<R> &G, PB absb)
{
    constexpr bool MINOR = sizeof(R) == 4 || lw64_minor(B);
    LwBandT<R, const WR_L R *, PB, typename std::conditional<MINOR, const WR_L R *, const WR_G R *>::type> Bl;
    auto at = [&](int j) { return lt + (imax(0, im.off[j]) & ~3); };
    Bl.absa = at(0), Bl.absb = absb, Bl.selfref = at(2), Bl.forref = at(3), Bl.fracrefa = at(4), Bl.fracrefb = at(5);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        if constexpr (MINOR)
            Bl.ka_m[i] = at(6 + i), Bl.kb_m[i] = at(9 + i);
        else
            Bl.ka_m[i] = G.ka_m[i], Bl.kb_m[i] = G.kb_m[i];
    }
    Bl.etab = lt + im.n;  // FP64: behind the image (lds_fill_lw); FP32 reads none
    Bl.x1 = at(12), Bl.x2 = at(13);
    Bl.refrat_planck_a = G.refrat_planck_a, Bl.refrat_planck_b = G.refrat_planck_b;
    Bl.refrat_m_a = G.refrat_m_a, Bl.refrat_m_b = G.refrat_m_b, Bl.refrat_m_a3 = G.refrat_m_a3;
    return Bl;
}
// the wave's index in its workgroup, as the wave-uniform value it is
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x / 64)); }

// The wave's number in a grid of persistent workgroups, workgroups first: consecutive numbers are on different
// CUs, so that the last round of a large tile spreads over the whole chip instead of filling a few workgroups
// (796,590 columns are 12,447 blocks, 159 more than six rounds of 2,048 waves).  A tile of fewer blocks than the grid
// could hold keeps few and full workgroups, so that the band streams share the chip (one wave on each CU
// instead: 40,000 columns of the FP64 NAM route in 44 ms, not 26).
__device__ __forceinline__ int wave_slot() { return wave_id() * (int)gridDim.x + (int)blockIdx.x; }

// copies the image into the workgroup's LDS (16-byte words) and waits for the whole workgroup
template <typename R, typename I> __device__ __forceinline__ void lds_fill(float4 *dst, const I &im)
{
    const WR_G float4 *src = (const WR_G float4 *)im.base;
    const int n4 = (int)((size_t)im.n * sizeof(R) / 16);
    for (int q = threadIdx.x; q < n4; q += blockDim.x) dst[q] = src[q];
    __syncthreads();
}
// LW: FP64 with exp_tbl behind the image (ETAB_LDS bytes; the last word holds one entry)
template <typename R> __device__ __forceinline__ void lds_fill_lw(float4 *dst, const LwImg<R> &im, const WR_G R *etab)
{
    if constexpr (sizeof(R) == 8) {
        WR_L R *e = (WR_L R *)dst + im.n;
        for (int q = threadIdx.x; q <= NTBL; q += blockDim.x) e[q] = etab[q];
    }
    lds_fill<R>(dst, im);
}

// k_lw (FP64, one lane per column) with the band's tables and the transmittance table in LDS (absb, the table
// of the layers above laytrop, and the minor gases of bands 3 and 5 stay in global memory: the rest of every
// band then fits).  Persistent workgroups of 4 x lw64_waves waves, as many as the CUs hold; each copies the tables
// into LDS once and its waves then run 64-column blocks.  Same arithmetic as k_lw.  Bound by memory latency at two
// waves per SIMD (0.3 to 0.4 of the issue slots): the LW kernels of a 954x835x60 call take 124 ms alone on the GPU, 144
// with the optics evaluated in both sweeps and whole entries gathered from L2.
template <int B> constexpr int lwl64_wpg() { return 4 * lw64_waves<B>(); }
template <int B, bool SURR = false, bool EXT = true>
__global__ void __launch_bounds__(64 * lwl64_wpg<B>(), lw64_waves<B>())
    k_lwl64(const Tabs<double> *__restrict__ T, ColIn in_, RunPar par, int col0, int n, ColScal cs, RecPtrs rp,
            AccT<double> acc, Surr sg, char *__restrict__ pool)
{
    extern __shared__ float4 lwl64_tab[];
    const ColIn in = band_in<EXT>(in_);
    const LwImg<double> &im = T->lw_img[B];
    lds_fill_lw<double>(lwl64_tab, im, T->exp_tbl);
    const auto Bl = lds_band<double, B>((const WR_L double *)lwl64_tab, im, T->lw[B], T->lw[B].absb);
    constexpr int WPG = lwl64_wpg<B>();
    const int lane = threadIdx.x % 64, w = wave_slot();
    WR_G char *slot = (WR_G char *)(pool + (size_t)w * lw64_slot_bytes(LW_NG[B], in.nlay + 2));
    for (int blk = w; blk * 64 < n; blk += gridDim.x * WPG)
        lw_column<double, B, SURR>(T, Bl, in, par, col0, n, cs, rp, acc, sg, blk, lane, slot);
}

// FP32 LW band kernel with a cached upward sweep.  The down sweep also forms, per layer and g-point,
// the upward transmittance a = trng * efclrfr and source b (gas plus cloud term) and keeps them in the
// lane's pool slot (8 bytes per layer and g-point, one store); the up sweep is then rad = rad * a + b,
// with no optics.  Bound by HBM: 2.5 TB/s read and 1.4 TB/s written on the 954x835x60 grid.
constexpr int LW_NV_F32 = 2;
// transmittance a and the downward and upward sources (gas plus cloud) of CH g-points of a layer
template <int CH>
__device__ __forceinline__ void lw_chunk_f32(const LwLayer<float> &y, float sdif, float dd, float du,
                                             float ecld, uint32_t cb, const float *tau, const float *fr, float *a, float *bd,
                                             float *bu)
{
    using R = float;
    GasV<R, CH> q;
    lw_gas_v<R, CH>(nullptr, sdif, y.taer, tau, q);
#pragma unroll
    for (int j = 0; j < CH; ++j) {
        const R fa = fr[j] * q.at[j];
        bd[j] = fa * (y.blay + dd * q.gf[j]);
        bu[j] = fa * (y.blay + du * q.gf[j]);
        a[j] = q.tr[j];
    }
    if (__any(cb & ((1u << CH) - 1u))) {
        R tr[CH], at[CH], gf[CH];
        lw_tot_v<R, CH>(nullptr, q.od, y.odcld, tr, at, gf);
#pragma unroll
        for (int j = 0; j < CH; ++j) {
            const bool cl = (cb >> j) & 1u;
            const R fa = fr[j] * at[j];
            const R td = fa * (y.blay + dd * gf[j]), tu = fa * (y.blay + du * gf[j]);
            a[j] = cl ? q.tr[j] * ecld : a[j];
            bd[j] = cl ? td : bd[j];
            bu[j] = cl ? tu : bu[j];
        }
    }
}

template <int B, bool SURR, typename BT>
__device__ __forceinline__ void lw_column_f32c(const Tabs<float> *__restrict__ T, const BT &Bt, const ColIn &in,
                                               const RunPar &par, int col0, int n, const ColScal &cs, const RecPtrs &rp,
                                               const AccT<float> &acc, const Surr &sg, int blk, int lane, WR_G char *slot)
{
    using R = float;
    constexpr int NG = LW_NG[B], GW = NG, CH = lw_chunk<B>();
    const Share<R> sh{nullptr, 0, 0};
    const int nv = valid_cols(in, col0, n);
    if (blk * 64 >= nv) return;
    const bool ok = blk * 64 + lane < nv;  // lanes past the last column repeat it and store nothing
    const int rl = ok ? lane : nv - 1 - blk * 64, t = blk * 64 + rl;
    const LwCol<R> c = lw_col<R, B, SURR>(in, col0, cs, sg, t);
    const int nrl = c.nrl;
    WR_G f32x2v *ab = (WR_G f32x2v *)slot + lane;  // [layer][g][lane]
    if (ok) acc.lw_dn[(size_t)nrl * n + t] = (R)0;  // no downward LW at the top
    R rad[1][GW];
#pragma unroll
    for (int g = 0; g < GW; ++g) rad[0][g] = (R)0;
    LevelSum<R, NG, GW, 1> sum{sh, lane, 0, 0, 0};
    auto dn = [&](int row, const R *s) {
        if (ok) acc.lw_dn[(size_t)row * n + t] = s[0];
    };
    auto up = [&](int row, const R *s) {
        if (ok) acc.lw_up[(size_t)row * n + t] = s[0];
    };
    R btop = (R)0;  // Planck function at the level above the layer
    sum.begin(nrl - 1, -1);
    for (int k = nrl - 1; k >= 0; --k) {
        LwLayer<R> y;
        lw_get<R, B>(T, in, par, rp, c, blk, rl, k, y);
        const uint32_t bits = y.cloudy ? mword(rp.mlw, rp.row(blk, k), MROW_LW, B, rl) : 0u;
        if (k == nrl - 1) btop = y.blay;
        const R dd = y.bbot - y.blay, du = btop - y.blay;
        R ecld = (R)1;
        if (__any(y.cloudy)) ecld = M<R>::exp(-y.odcld);
        R sfc0[GW];
#pragma unroll
        for (int g0 = 0; g0 < GW; g0 += CH) {
            R tau[CH], fr[CH];
            lw_taufr<R, B, SURR, CH>(T, Bt, sg, c, n, k, y.L, g0, tau, fr);
            R a[CH], bd[CH], bu[CH];
            lw_chunk_f32<CH>(y, c.sdif, dd, du, ecld, bits >> g0, tau, fr, a, bd, bu);
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                rad[0][g0 + j] = rad[0][g0 + j] * a[j] + bd[j];
                ab[((size_t)k * NG + g0 + j) * 64] = (f32x2v){a[j], bu[j]};
            }
            if (k == 0) {  // surface emission and reflection start the upward sweep
#pragma unroll
                for (int j = 0; j < CH; ++j) {
                    const R rad0 = c.semis * fr[j] * y.bbot;
                    sfc0[g0 + j] = rad0 + c.reflct * rad[0][g0 + j];
                }
            }
            if constexpr (CH < GW) __builtin_amdgcn_sched_barrier(0);
        }
        sum.put(rad, dn);
        if (k == 0) {
#pragma unroll
            for (int g = 0; g < GW; ++g) rad[0][g] = sfc0[g];
        }
        btop = y.bbot;
    }
    sum.finish(dn);
    sum.begin(0, 1);
    sum.put(rad, up);
    for (int k = 0; k < nrl; ++k) {  // up sweep over the cached layers
#pragma unroll
        for (int g = 0; g < GW; ++g) {
            const f32x2v v = ab[((size_t)k * NG + g) * 64];
            rad[0][g] = rad[0][g] * v.x + v.y;
        }
        sum.put(rad, up);
    }
    sum.finish(up);
}

template <int B, bool SURR = false, bool EXT = true>
__global__ void __launch_bounds__(64, lwc_waves<B>()) k_lwc(const Tabs<float> *__restrict__ T, ColIn in_, RunPar par,
                                                         int col0, int n, ColScal cs, RecPtrs rp, AccT<float> acc, Surr sg,
                                                         char *__restrict__ pool)
{
    const ColIn in = band_in<EXT>(in_);
    WR_G char *slot = (WR_G char *)(pool + (size_t)blockIdx.x * cache_slot_bytes(LW_NV_F32, LW_NG[B], in.nlay + 2, 4));
    for (int blk = blockIdx.x; blk * 64 < n; blk += gridDim.x)
        lw_column_f32c<B, SURR>(T, T->lw[B], in, par, col0, n, cs, rp, acc, sg, blk, (int)threadIdx.x, slot);
}

// k_lwc with the band's tables in LDS.  Persistent workgroups of one wave per SIMD times the band's
// wave bound (LWC_WAVES; 1 where the registers alone set the waves, so a CU then holds several); each
// copies the band's packed table image (T->lw_img[B], up to about 130 KB) into LDS once, and each wave
// then runs 64-column blocks with its own pool slot, so the optics' table reads are LDS reads instead
// of L2/HBM gathers.  Same arithmetic as k_lwc.
template <int B> constexpr int lwl_wpg() { return 4 * lwc_waves<B>(); }
template <int B, bool SURR = false, bool EXT = true>
__global__ void __launch_bounds__(64 * lwl_wpg<B>(), lwc_waves<B>())
    k_lwl(const Tabs<float> *__restrict__ T, ColIn in_, RunPar par, int col0, int n, ColScal cs, RecPtrs rp, AccT<float> acc,
          Surr sg, char *__restrict__ pool)
{
    extern __shared__ float4 lwl_tab[];
    const ColIn in = band_in<EXT>(in_);
    const LwImg<float> &im = T->lw_img[B];
    lds_fill<float>(lwl_tab, im);
    const WR_L float *lt = (const WR_L float *)lwl_tab;
    const auto Bl = lds_band<float, B>(lt, im, T->lw[B], lt + (imax(0, im.off[1]) & ~3));
    constexpr int WPG = lwl_wpg<B>();
    const int lane = threadIdx.x % 64, w = wave_slot();
    WR_G char *slot = (WR_G char *)(pool + (size_t)w * cache_slot_bytes(LW_NV_F32, LW_NG[B], in.nlay + 2, 4));
    for (int blk = w; blk * 64 < n; blk += gridDim.x * WPG)
        lw_column_f32c<B, SURR>(T, Bl, in, par, col0, n, cs, rp, acc, sg, blk, lane, slot);
}

// Waves per SIMD the SW kernels are compiled for, per band: what the registers allow without much scratch; two
// g-points a chunk in both precisions.  FP64 McICA, one wave -> two, alone on 796,590 columns: bands 18, 19, 24, 27
// 5.45 -> 5.10, 5.45 -> 5.22, 5.55 -> 5.38, 5.98 -> 5.00 ms; bands 17, 20, 21, 23, 29 lose (17: 8.9 -> 13.0 ms with
// 628 bytes of scratch a lane).  The NAM route holds two skies, hence its own row.
// WR_SW64_WAVES / WR_SW32_WAVES > 0 override the tables for every band (tuning builds).
constexpr int SW64_WAVES[14] = {2, 1, 2, 2, 1, 1, 2, 1, 2, 2, 2, 2, 2, 1};
constexpr int SWR64_WAVES[14] = {2, 1, 1, 1, 1, 1, 2, 1, 1, 2, 2, 1, 2, 1};
constexpr int SW32_WAVES[14] = {3, 2, 2, 2, 2, 2, 4, 2, 2, 3, 3, 2, 3, 2};
constexpr int SWR32_WAVES[14] = {3, 2, 2, 2, 2, 2, 4, 2, 2, 3, 3, 2, 3, 2};
// g-points per chunk of the layer R/T (0: the whole band), by precision and route
constexpr int SW_CHUNK64 = 2, SW_CHUNK32 = 2, SWR_CHUNK64 = 2, SWR_CHUNK32 = 2;
template <typename R, int B, bool NAM = false> constexpr int sw_chunk()
{
    return chunk_of(SW_NG[B], sizeof(R) == 8 ? (NAM ? SWR_CHUNK64 : SW_CHUNK64) : (NAM ? SWR_CHUNK32 : SW_CHUNK32));
}
#ifndef WR_SW64_WAVES
#define WR_SW64_WAVES 0
#endif
#ifndef WR_SW32_WAVES
#define WR_SW32_WAVES 0
#endif
template <typename R, int B, bool NAM = false> constexpr int sw_waves()
{
    if (sizeof(R) == 8) return WR_SW64_WAVES > 0 ? WR_SW64_WAVES : (NAM ? SWR64_WAVES[B] : SW64_WAVES[B]);
    return WR_SW32_WAVES > 0 ? WR_SW32_WAVES : (NAM ? SWR32_WAVES[B] : SW32_WAVES[B]);
}

// ---- SW band kernels (McICA two-stream) ------------------------------------------------------------
// One lane per day column, one wave per block of 64 day-list entries, layer set-up and McICA words from the
// records.  Per layer the g-points run in chunks as in the LW kernels: layer R/T of a chunk without
// per-g-point branches, so that its chains of divisions, square roots and exponentials overlap.

// single-scattering albedo above which the mixed path evaluates the SW layer R/T in FP64
constexpr double W0_FP64 = 0.999999;


template <typename R, int CH> struct RtV {  // layer reflectances, transmittances and direct transmission of CH g-points
    R rb[CH], rd[CH], tb[CH], td[CH], ld[CH];
};

// exp(-z) of the SW table for CH arguments: the series below 0.06, the table entry above
template <typename R, int CH>
__device__ __forceinline__ void expm_v(const R *z, const WR_G R *__restrict__ tbl, R *e)
{
    bool any = false;
#pragma unroll
    for (int j = 0; j < CH; ++j) {
        e[j] = (R)1 - z[j] + (R)0.5 * z[j] * z[j];
        any |= !(z[j] <= (R)0.06);
    }
    if (__any(any)) {
#pragma unroll
        for (int j = 0; j < CH; ++j) {
            R v;
            if constexpr (sizeof(R) == 4) {
                const R tb = z[j] * __builtin_amdgcn_rcpf((R)(1.0 / 0.278) + z[j]);
                const R fi = fmin(floorf(__builtin_fmaf((R)NTBL, tb, (R)0.5)), (R)9999.999);
                v = M<R>::exp(-(((R)(1.0 / 0.278) * fi) * __builtin_amdgcn_rcpf((R)NTBL - fi)));
            } else {
                const R ft = z[j] / ((R)(1.0 / 0.278) + z[j]);
                v = tbl[imax(0, imin(10000, (int)((R)0.5 + (R)10000 * ft)))];
            }
            e[j] = !(z[j] <= (R)0.06) ? v : e[j];
        }
    }
}

// layer_rt (delta scaling, PIFM, layer R/T) for CH g-points; FP32 flags a g-point near the two-stream
// singularity k mu = 1, where numerator and denominator of the direct-beam terms both vanish
template <typename R, int CH>
__device__ __forceinline__ void layer_rt_v(const R *ztau0, const R *zssa0, const R *zasy0, R cz, R snt,
                                           const WR_G R *__restrict__ tbl, RtV<R, CH> &o, bool *ill)
{
    R zb1[CH], zb2[CH], zb3[CH], e1[CH], e2[CH];
    R g1[CH], g2[CH], g3[CH], rk[CH], w1[CH];
    bool far = false;
    // FP32: cap the exponents at 80 so exp(-zb) stays a normal number and 1/exp(-zb) finite (the R/T
    // expressions depend on the capped terms only through factors below exp(-160))
    const R zcap = (sizeof(R) < sizeof(double)) ? (R)80 : (R)500;
#pragma unroll
    for (int j = 0; j < CH; ++j) {
        const R zssaw = fmin((R)ONEMINUS, rdiv<R>(zssa0[j], ztau0[j]));
        const R zasyw = rdiv<R>(zasy0[j], fmax((R)FTINY, zssa0[j]));
        const R za1s = zasyw * zasyw;
        const R za2s = zssaw * za1s;
        const R ztau1 = ((R)1 - za2s) * ztau0[j];
        w1[j] = rdiv<R>(zssaw - za2s, (R)1 - za2s);
        const R zasy1 = rdiv<R>(zasyw, (R)1 + zasyw);
        const R zasy3 = (R)0.75 * zasy1;
        g1[j] = (R)2 - w1[j] * ((R)1.25 + zasy3);
        g2[j] = (R)0.75 * w1[j] * ((R)1 - zasy1);
        g3[j] = (R)0.5 - zasy3 * cz;
        rk[j] = sqrt((g1[j] - g2[j]) * (g1[j] + g2[j]));
        zb1[j] = fmin(rk[j] * ztau1, zcap);
        zb3[j] = ztau1 * snt;
        zb2[j] = fmin(zb3[j], zcap);
        far |= zb3[j] > zcap;
    }
    expm_v<R, CH>(zb1, tbl, e1);
    expm_v<R, CH>(zb2, tbl, e2);
#pragma unroll
    for (int j = 0; j < CH; ++j) o.ld[j] = e2[j];
    if (__any(far)) {
        R e3[CH];
        expm_v<R, CH>(zb3, tbl, e3);
#pragma unroll
        for (int j = 0; j < CH; ++j) o.ld[j] = zb3[j] > zcap ? e3[j] : o.ld[j];
    }
#pragma unroll
    for (int j = 0; j < CH; ++j) {
        const R zgam1 = g1[j], zgam2 = g2[j], zgam3 = g3[j], zrk = rk[j];
        const R zgam4 = (R)1 - zgam3;
        const R eps1 = (R)1.0e-8;
        const R za1 = zgam1 * zgam4 + zgam2 * zgam3;
        const R za2 = zgam1 * zgam3 + zgam2 * zgam4;
        const R zrk2 = (R)2 * zrk;
        const R zrp = zrk * cz;
        const R zrp1 = (R)1 + zrp;
        const R zrm1 = (R)1 - zrp;
        R zrpp = (R)1 - zrp * zrp;
        if constexpr (sizeof(R) == 4) ill[j] = fabs(zrpp) < (R)1.0e-2;
        if (fabs(zrpp) < eps1) zrpp = (zrpp < (R)0) ? -eps1 : eps1;
        const R zrkg1 = zrk + zgam1;
        const R zrkg3 = zrk * zgam3;
        const R zrkg4 = zrk * zgam4;
        const R zr1 = zrm1 * (za2 + zrkg3);
        const R zr2 = zrp1 * (za2 - zrkg3);
        const R zr3 = zrk2 * (zgam3 - za2 * cz);
        const R zr4 = zrpp * zrkg1;
        const R zr5 = zrpp * (zrk - zgam1);
        const R zt1 = zrp1 * (za1 + zrkg4);
        const R zt2 = zrm1 * (za1 - zrkg4);
        const R zt3 = zrk2 * (zgam4 + za1 * cz);
        const R zexm1 = e1[j], zexm2 = e2[j];
        const R zexp1 = rdiv<R>((R)1, zexm1);
        const R zexp2 = rdiv<R>((R)1, zexm2);
        const R ze1r45 = zr4 * zexp1 + zr5 * zexm1;
        const R zden1 = rdiv<R>(w1[j], ze1r45);
        const R rb = fmax((R)0, fmin((R)1, (zr1 * zexp1 - zr2 * zexm1 - zr3 * zexm2) * zden1));
        const R tb = fmax((R)0, fmin((R)1, zexm2 * ((R)1 - (zt1 * zexp1 - zt2 * zexm1 - zt3 * zexp2) * zden1)));
        const bool tiny = ze1r45 >= -eps1 && ze1r45 <= eps1;
        o.rb[j] = tiny ? eps1 : rb;
        o.tb[j] = tiny ? zexm2 : tb;
        const R zden1d = rdiv<R>(zr4, ze1r45 * zrkg1);
        o.rd[j] = fmax((R)0, fmin((R)1, zgam2 * (zexp1 - zexm1) * zden1d));
        o.td[j] = fmax((R)0, fmin((R)1, zrk2 * zden1d));
    }
}

// What a layer's two-stream solution of one column needs besides the g-point optics.
template <typename R> struct SwSky {
    R ta, sa, ya;         // aerosol optical depth, single-scattering albedo, asymmetry
    R ctau, cssa, casy;   // cloud tau, tau w, tau w g
    R cz, snt;
};

// LDS of one wave for the FP64 evaluations of the FP32 kernels
struct alignas(16) Fix64 {
    double t0[64], s0[64], g0[64];
    float cz[64], snt[64];
};

// Layer R/T of CH g-points from their gas (tg) and Rayleigh (tr) optical depths, the aerosol and, where
// bit j of cld is set, the cloud.  FP32 evaluates in FP64 where FP32 loses the answer: near-conservative
// scattering (w0 > 1 - 1e-6: 1 - w0 and gamma1 - gamma2 cancel; an FP32 pre-test with a 10x wider
// margin skips the FP64 test for most layers) and near the two-stream singularity.  About one g-point
// and layer in a hundred is of that kind, so nearly every wave has some in every chunk: the (lane,
// g-point) pairs of the chunk are gathered through LDS and evaluated together, one per lane, where a
// branch per g-point took the FP64 evaluation (about 200 operations) once for each g-point with any.
template <typename R, int CH>
__device__ __forceinline__ void layer_rt_sky(const Tabs<R> *__restrict__ T, const R *tr, const R *tg, const SwSky<R> &y,
                                             uint32_t cld, RtV<R, CH> &o, Fix64 *fx)
{
    R t0[CH], s0[CH], a0[CH];
    bool ill[CH];
#pragma unroll
    for (int j = 0; j < CH; ++j) {
        // clear-sky optical parameters with the aerosol (phys_rrtm_sw_spcvrtc.cu:323-329)
        t0[j] = fmax((R)FTINY, tr[j] + tg[j] + y.ta);
        s0[j] = tr[j] + y.ta * y.sa;
        a0[j] = y.ya * y.sa * y.ta;
        const bool c = (cld >> j) & 1u;
        t0[j] = c ? t0[j] + y.ctau : t0[j];
        s0[j] = c ? s0[j] + y.cssa : s0[j];
        a0[j] = c ? a0[j] + y.casy : a0[j];
    }
    layer_rt_v<R, CH>(t0, s0, a0, y.cz, y.snt, T->sw_exp_tbl, o, ill);
    if constexpr (sizeof(R) == 4) {
        auto wide = [&](int j, double &t, double &s, double &a) {  // the optical parameters summed in FP64
            const double ta = (double)y.ta, sa = (double)y.sa, ya = (double)y.ya;
            const bool c = (cld >> j) & 1u;
            t = fmax(FTINY, (double)tr[j] + (double)tg[j] + ta) + (c ? (double)y.ctau : 0.0);
            s = (double)tr[j] + ta * sa + (c ? (double)y.cssa : 0.0);
            a = ya * sa * ta + (c ? (double)y.casy : 0.0);
        };
        bool any = false;
#pragma unroll
        for (int j = 0; j < CH; ++j) {
            const bool pre = s0[j] > (R)0.99999 * t0[j];
            if (__any(pre)) {
                double t, s, a;
                wide(j, t, s, a);
                ill[j] |= pre && s > W0_FP64 * t;
            }
            any |= ill[j];
        }
        if (__any(any)) {
            const uint64_t active = __ballot(1);
            const uint64_t below = ((uint64_t)1 << (threadIdx.x & 63)) - 1;
            int total = 0, pos[CH];
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                const uint64_t m = __ballot(ill[j]);
                pos[j] = total + __popcll(m & below);
                total += __popcll(m);
            }
            const int rank = __popcll(active & below);
            const int lanes = __popcll(active);
            for (int first = 0; first < total; first += lanes) {  // one round, unless most of the chunk is of that kind
#pragma unroll
                for (int j = 0; j < CH; ++j) {
                    const int p = pos[j] - first;
                    if (ill[j] && p >= 0 && p < lanes) {
                        double t, s, a;
                        wide(j, t, s, a);
                        fx->t0[p] = t, fx->s0[p] = s, fx->g0[p] = a, fx->cz[p] = y.cz, fx->snt[p] = y.snt;
                    }
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
                if (first + rank < total) {
                    const double t = fx->t0[rank], s = fx->s0[rank], a = fx->g0[rank];
                    RtV<double, 1> d;
                    layer_rt_v<double, 1>(&t, &s, &a, (double)fx->cz[rank], (double)fx->snt[rank], T->sw_exp_tbl64, d, nullptr);
                    float *q0 = (float *)&fx->t0[rank], *q1 = (float *)&fx->s0[rank], *q2 = (float *)&fx->g0[rank];
                    q0[0] = (R)d.rb[0], q0[1] = (R)d.rd[0], q1[0] = (R)d.tb[0], q1[1] = (R)d.td[0], q2[0] = (R)d.ld[0];
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int j = 0; j < CH; ++j) {
                    const int p = pos[j] - first;
                    if (ill[j] && p >= 0 && p < lanes) {
                        const float *q0 = (const float *)&fx->t0[p], *q1 = (const float *)&fx->s0[p], *q2 = (const float *)&fx->g0[p];
                        o.rb[j] = q0[0], o.rd[j] = q0[1], o.tb[j] = q1[0], o.td[j] = q1[1], o.ld[j] = q2[0];
                    }
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
        }
    }
}

// One layer of a day column: optics record and sky.
template <typename R> struct SwLayer {
    SwLay<R> L;
    SwSky<R> y;
    bool cloudy;
};
template <typename R, int B>
__device__ __forceinline__ void sw_get(const Tabs<R> *__restrict__ T, const ColIn &in, const RunPar &par, const RecPtrs &rp,
                                       int i, R cz, R snt, int blk, int lane, int k, SwLayer<R> &a)
{
    const LRow<R> row = srow<R>(rp, blk, k, lane);
    srow_get<R>(row, row.w(0), par, a.L);
    a.cloudy = row.w(1) != 0;
    const RadCol rc{in, i, rp.nrl};
    double ta, sa, ya;
    rc.aer_sw3(B, rp.nrl - 1 - k, ta, sa, ya);
    a.y = {(R)ta, (R)sa, (R)ya, (R)0, (R)1, (R)0, cz, snt};
    if (__any(a.cloudy)) {
        double rl = par.re_liq, ri = par.re_ice, rain = 0.0;
        if (a.cloudy) rc.props(rp.nrl - 1 - k, par.re_liq, par.re_ice, rl, ri, rain);
        sw_cloud<R>(T, B, (double)row.f(SF_LIQ), rl, (double)row.f(SF_ICE), ri, a.y.ctau, a.y.cssa, a.y.casy, rain);
    }
}
// gas and Rayleigh optical depths of g-points g0 .. g0 + CH - 1
template <typename R, int B, bool SURR, int CH, typename BT>
__device__ __forceinline__ void sw_tgtr(const Tabs<R> *__restrict__ T, const BT &Bt, const Surr &sg, int table, size_t s, int k,
                                        int lt, const SwLay<R> &L, int g0, R *tg, R *tr)
{
    if (SURR && !table) {
#pragma unroll
        for (int j = 0; j < CH; ++j) {
            const R tau = (R)__expf(surr_out(sg, 280 + SW_NS[B] + g0 + j, s));
            const R ssa = (R)fminf(1.0f, fmaxf(0.0f, surr_out(sg, 392 + SW_NS[B] + g0 + j, s)));
            tr[j] = tau * ssa;
            tg[j] = tau - tr[j];
        }
    } else {
        sw_optics_t<R, B, CH>(T, Bt, L, k + 1, lt, tg, tr, g0);
    }
}

// What the bottom-up sweep leaves per layer and g-point for the top-down one: the reflectances (direct pb,
// diffuse pd) of everything below the layer and, in FP32, what carries the beams through it.  With S the direct
// and F the diffuse radiation that enter at the layer's top, those that leave at its bottom are
//   S' = ld S,   F' = al F + be S,   al = td / (1 - rd pd),   be = ((tb - ld) + rd ld pb) / (1 - rd pd)
// (the diffuse beam is transmitted, gains what the layer scatters out of the direct one, and what the layer
// reflects back of S' pb + F' pd), and the fluxes at that level are S' pb + F' pd up and S' + F' down.  The
// denominator is the one that the bottom-up step divides by anyway, so FP32 spends one reciprocal per layer where
// the reference's order (the reflectance of everything above, vrtqdr) takes three, and 5 values per g-point
// and layer where that needs 7.  FP64 keeps the reference's order, which its outputs reproduce bit for
// bit, and evaluates the layer's R/T again (the bytes cost more than the evaluation).
template <typename R> constexpr int sw_nv() { return sizeof(R) == 4 ? 5 : 2; }
// Pool slot of one SW wave.
template <typename R, int NG> struct SwSlot {
    WR_G char *p;
    int lane, nk;
    // sky 1 (NAM route: the total sky beside the clear one) lies behind sky 0
    __device__ __forceinline__ void put(int k, int sky, int g, const R (&v)[sw_nv<R>()]) const  // pb, pd; FP32 al, be, ld
    {
        WR_G char *const p = this->p + (size_t)sky * nk * NG * 64 * sw_nv<R>() * sizeof(R);
        const size_t e = ((size_t)k * NG + g) * 64 + lane;
        if constexpr (sizeof(R) == 4) {
            ((WR_G f32x4v *)p)[e] = (f32x4v){v[0], v[1], v[2], v[3]};
            ((WR_G float *)(p + (size_t)nk * NG * 64 * 16))[e] = v[4];
        } else {
            ((WR_G f64x2v *)p)[e] = (f64x2v){v[0], v[1]};
        }
    }
    __device__ __forceinline__ void get(int k, int sky, int g, R (&v)[sw_nv<R>()]) const
    {
        const WR_G char *const p = this->p + (size_t)sky * nk * NG * 64 * sw_nv<R>() * sizeof(R);
        const size_t e = ((size_t)k * NG + g) * 64 + lane;
        if constexpr (sizeof(R) == 4) {
            const f32x4v q = ((const WR_G f32x4v *)p)[e];
            v[0] = q.x, v[1] = q.y, v[2] = q.z, v[3] = q.w;
            v[4] = ((const WR_G float *)(p + (size_t)nk * NG * 64 * 16))[e];
        } else {
            const f64x2v q = ((const WR_G f64x2v *)p)[e];
            v[0] = q.x, v[1] = q.y;
        }
    }
};

// The adding method over one column: bottom-up reflectances to the slot, then the direct and diffuse beams
// top-down with the level fluxes.  NP skies at once (the NAM route's clear and total sky, whose layers differ only
// where there is cloud: one evaluation of the optics serves both; the second is skipped as a whole where two is
// false).  layer(k, step) gives a layer (step: the sweep's direction), rt_at(layer, k, g0, o) its R/T of a chunk of
// the lane's g-points in each sky, sun(g) the solar source of one; emit(level, {up, down of each sky}) takes
// a level's fluxes, top first.
template <typename R, int NG, int GW, int CH, int NP, typename SLOT, typename LAYER, typename RT, typename SUN, typename EMIT>
__device__ __forceinline__ void sw_adding(int nrl, R asfc, bool two, SLOT &&slot, int lane, const Share<R> &sh, LAYER &&layer,
                                          RT &&rt_at, SUN &&sun, EMIT &&emit)
{
    R pb[NP][GW], pd[NP][GW];
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int g = 0; g < GW; ++g) pb[p][g] = asfc, pd[p][g] = asfc;
    for (int k = 0; k < nrl; ++k) {
        auto a = layer(k, 1);
#pragma unroll
        for (int g0 = 0; g0 < GW; g0 += CH) {
            RtV<R, CH> os[NP];
            rt_at(a, k, g0, os);
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                if (p > 0 && !two) break;
                const RtV<R, CH> &o = os[p];
#pragma unroll
                for (int j = 0; j < CH; ++j) {
                    const int g = g0 + j;
                    R &b = pb[p][g], &d = pd[p][g];
                    const R zden1 = rdiv<R>((R)1, (R)1 - d * o.rd[j]);
                    if constexpr (sizeof(R) == 4) {
                        const R sc = o.tb[j] - o.ld[j], lb = o.ld[j] * b, al = o.td[j] * zden1;
                        slot.put(k, p, g, {b, d, al, (sc + o.rd[j] * lb) * zden1, o.ld[j]});
                        b = o.rb[j] + al * (sc * d + lb);
                        d = o.rd[j] + al * o.td[j] * d;
                    } else {
                        slot.put(k, p, g, {b, d});
                        const R nb = o.rb[j] + (o.td[j] * ((o.tb[j] - o.ld[j]) * d + o.ld[j] * b)) * zden1;
                        const R nd = o.rd[j] + o.td[j] * o.td[j] * d * zden1;
                        b = nb, d = nd;
                    }
                }
            }
            if constexpr (CH < GW) __builtin_amdgcn_sched_barrier(0);
        }
    }
    R zsolar[GW], f[2 * NP][GW];
    LevelSum<R, NG, GW, 2 * NP> sum{sh, lane, 0, 0, 0};
    sum.begin(nrl, -1);
#pragma unroll
    for (int g = 0; g < GW; ++g) {
        zsolar[g] = sun(g);
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            f[2 * p][g] = zsolar[g] * pb[p][g];
            f[2 * p + 1][g] = zsolar[g];
        }
    }
    sum.put(f, emit);
    if constexpr (sizeof(R) == 4) {
        R s[NP][GW], d[NP][GW];  // direct and diffuse beams
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
            for (int g = 0; g < GW; ++g) s[p][g] = zsolar[g], d[p][g] = (R)0;
        for (int k = nrl - 1; k >= 0; --k) {
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                if (p > 0 && !two) break;
#pragma unroll
                for (int g = 0; g < GW; ++g) {
                    R v[5];
                    slot.get(k, p, g, v);
                    d[p][g] = v[2] * d[p][g] + v[3] * s[p][g];
                    s[p][g] = v[4] * s[p][g];
                    f[2 * p][g] = s[p][g] * v[0] + d[p][g] * v[1];
                    f[2 * p + 1][g] = s[p][g] + d[p][g];
                }
            }
            sum.put(f, emit);
        }
    } else {
        R tdbt[NP][GW], tdn[NP][GW], rdnd[NP][GW];
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
            for (int g = 0; g < GW; ++g) tdbt[p][g] = (R)1, tdn[p][g] = (R)1, rdnd[p][g] = (R)0;
        for (int k = nrl - 1; k >= 0; --k) {
            auto a = layer(k, -1);
#pragma unroll
            for (int g0 = 0; g0 < GW; g0 += CH) {
                RtV<R, CH> os[NP];
                rt_at(a, k, g0, os);
#pragma unroll
                for (int p = 0; p < NP; ++p) {
                    if (p > 0 && !two) break;
                    const RtV<R, CH> &o = os[p];
#pragma unroll
                    for (int j = 0; j < CH; ++j) {
                        const int g = g0 + j;
                        R z[2];
                        slot.get(k, p, g, z);
                        const R db = tdbt[p][g], dn = tdn[p][g], rn = rdnd[p][g];
                        const R tdbt_s = o.ld[j] * db;
                        const R zden0 = (R)1 / ((R)1 - o.rd[j] * rn);
                        const R tdn_s = db * o.tb[j] + (o.td[j] * ((dn - db) + db * o.rb[j] * rn)) * zden0;
                        const R rdnd_s = o.rd[j] + o.td[j] * o.td[j] * rn * zden0;
                        tdbt[p][g] = tdbt_s, tdn[p][g] = tdn_s, rdnd[p][g] = rdnd_s;
                        const R zden1 = (R)1 / ((R)1 - rdnd_s * z[1]);
                        const R zfu = (tdbt_s * z[0] + (tdn_s - tdbt_s) * z[1]) * zden1;
                        const R zfd = tdbt_s + (tdn_s - tdbt_s + tdbt_s * z[0] * rdnd_s) * zden1;
                        f[2 * p][g] = zsolar[g] * zfu;
                        f[2 * p + 1][g] = zsolar[g] * zfd;
                    }
                }
                if constexpr (CH < GW) __builtin_amdgcn_sched_barrier(0);
            }
            sum.put(f, emit);
        }
    }
    sum.finish(emit);
}

// What the SW sweeps of one day column need besides its layers.
template <typename R> struct SwCol {
    int i, t, lt;
    R cz, snt, asfc, ssolar;
};
template <typename R, int B>
__device__ __forceinline__ void sw_col(const ColIn &in, const RunPar &par, int col0, const ColScal &cs, int t, SwCol<R> &c)
{
    c.i = col0 + t, c.t = t;
    const double czd = in.cosz[c.i];
    c.cz = (R)czd, c.snt = (R)(1.0 / czd);
    c.ssolar = (R)((par.solcon / S0) * czd);
    const double alb = in.alb[c.i];
    c.asfc = (R)((SW_IDXSFC[B] != 0) ? alb : 0.5 * (alb + alb));
    c.lt = cs.sw_laytrop[t];
}

// One day column of one SW band (spcvrtc, McICA).
template <typename R, int B, bool SURR, typename BT>
__device__ __forceinline__ void sw_column(const Tabs<R> *__restrict__ T, const BT &Bt, const ColIn &in, const RunPar &par, int col0,
                                          int n, const ColScal &cs, const RecPtrs &rp, const R *__restrict__ sflux,
                                          const AccT<R> &acc, const Surr &sg, int blk, int lane, WR_G char *slot, Fix64 *fx)
{
    constexpr int NG = SW_NG[B], CH = sw_chunk<R, B>();
    const int nday = *cs.nday;
    if (blk * 64 >= nday) return;
    const bool ok = blk * 64 + lane < nday;  // lanes past the last day column repeat it and store nothing
    const int rl = ok ? lane : nday - 1 - blk * 64;
    const int t = cs.dlist[blk * 64 + rl], nrl = rp.nrl;
    SwCol<R> c;
    sw_col<R, B>(in, par, col0, cs, t, c);
    const int table = SURR ? sg.table(t, 16 + B) : 1;
    if (ok) acc.sw_clr0[t] = (R)0;  // clear-sky surface flux: NAM route only
    struct Lay {
        SwLayer<R> y;
        uint32_t bits;
    };
    sw_adding<R, NG, NG, CH, 1>(
        nrl, c.asfc, false, SwSlot<R, NG>{slot, lane, in.nlay + 2}, lane, Share<R>{nullptr, 0, 0},
        [&](int k, int) {
            Lay a;
            sw_get<R, B>(T, in, par, rp, c.i, c.cz, c.snt, blk, rl, k, a.y);
            a.bits = a.y.cloudy ? mword(rp.msw, rp.row(blk, k), MROW_SW, B, rl) : 0u;
            return a;
        },
        [&](const Lay &a, int k, int g0, RtV<R, CH> (&o)[1]) {
            R tg[CH], tr[CH];
            sw_tgtr<R, B, SURR, CH>(T, Bt, sg, table, (size_t)k * n + t, k, c.lt, a.y.L, g0, tg, tr);
            layer_rt_sky<R, CH>(T, tr, tg, a.y.y, a.bits >> g0, o[0], fx);
        },
        [&](int g) { return c.ssolar * sflux[(size_t)(SW_NS[B] + g) * n + t]; },
        [&](int lev, const R *f) {
            if (ok) {
                acc.sw_up[(size_t)lev * n + t] = f[0];
                acc.sw_dn[(size_t)lev * n + t] = f[1];
            }
        });
}

// SW band kernel: blocks of 64 day-list entries, a grid no larger than the pool's slot count.
template <typename R, int B, bool SURR = false, bool EXT = true>
__global__ void __launch_bounds__(64, (sw_waves<R, B>())) k_sw(const Tabs<R> *__restrict__ T, ColIn in_, RunPar par, int col0,
                                           int n, ColScal cs, RecPtrs rp, const R *__restrict__ sflux, AccT<R> acc, Surr sg,
                                           char *__restrict__ pool)
{
    __shared__ Fix64 fx[1];
    const ColIn in = band_in<EXT>(in_);
    WR_G char *slot = (WR_G char *)(pool + (size_t)blockIdx.x * cache_slot_bytes(sw_nv<R>(), SW_NG[B], in.nlay + 2, (int)sizeof(R)));
    const int nday = *cs.nday;
    for (int blk = blockIdx.x; blk * 64 < nday; blk += gridDim.x)
        sw_column<R, B, SURR>(T, T->sw[B], in, par, col0, n, cs, rp, sflux, acc, sg, blk, (int)threadIdx.x, slot, fx);
}

// The SW band tables of an LDS image (the SwImg order); FP64 keeps absb in global memory.  A table the
// band does not have points at the image start and is never read; offsets are multiples of 4 elements.
template <typename R>
__device__ __forceinline__ SwBandT<R, const WR_L R *,
                                   typename std::conditional<sizeof(R) == 4, const WR_L R *, const WR_G R *>::type>
sw_lds_band(const WR_L R *lt, const SwImg<R> &im, const SwBand<R> &G)
{
    SwBandT<R, const WR_L R *, typename std::conditional<sizeof(R) == 4, const WR_L R *, const WR_G R *>::type> Bl;
    auto at = [&](int j) { return lt + (imax(0, im.off[j]) & ~3); };
    Bl.absa = at(0);
    if constexpr (sizeof(R) == 4)
        Bl.absb = at(1);
    else
        Bl.absb = G.absb;
    Bl.selfref = at(2), Bl.forref = at(3), Bl.rayl_v = at(4), Bl.rayla = at(5), Bl.raylb = at(6);
    Bl.abso3a = at(7), Bl.abso3b = at(8), Bl.absch4 = at(9), Bl.absh2o = at(10), Bl.absco2 = at(11);
    Bl.rayl = G.rayl, Bl.strrat = G.strrat;
    return Bl;
}

// k_sw with the band's tables in LDS (absb in global memory in FP64), as k_lwl / k_lwl64 do for LW:
// persistent workgroups of 4 x sw_waves waves, as many as the CUs hold at once; each copies the band's
// packed table image (T->sw_img[B]) into LDS once and each wave then runs blocks of 64 day-list
// entries with its own pool slot.  Same arithmetic as k_sw.
template <typename R, int B> constexpr int swl_wpg() { return 4 * sw_waves<R, B>(); }
template <typename R, int B, bool SURR = false, bool EXT = true>
__global__ void __launch_bounds__((64 * swl_wpg<R, B>()), (sw_waves<R, B>()))
    k_swl(const Tabs<R> *__restrict__ T, ColIn in_, RunPar par, int col0, int n, ColScal cs, RecPtrs rp,
          const R *__restrict__ sflux, AccT<R> acc, Surr sg, char *__restrict__ pool)
{
    extern __shared__ float4 swl_tab[];
    const ColIn in = band_in<EXT>(in_);
    lds_fill<R>(swl_tab, T->sw_img[B]);
    const auto Bl = sw_lds_band<R>((const WR_L R *)swl_tab, T->sw_img[B], T->sw[B]);
    constexpr int WPG = swl_wpg<R, B>();
    __shared__ Fix64 fx[sizeof(R) == 4 ? WPG : 1];
    const int lane = threadIdx.x % 64, wv = wave_id(), w = wave_slot();
    WR_G char *slot = (WR_G char *)(pool + (size_t)w * cache_slot_bytes(sw_nv<R>(), SW_NG[B], in.nlay + 2, (int)sizeof(R)));
    const int nday = *cs.nday;
    for (int blk = w; blk * 64 < nday; blk += gridDim.x * WPG)
        sw_column<R, B, SURR>(T, Bl, in, par, col0, n, cs, rp, sflux, acc, sg, blk, lane, slot, fx + (sizeof(R) == 4 ? wv : 0));
}

// ---- post: FP64 fluxes -> heating rates, top-first outputs -------------------------------------------
struct OutPtrs {
    WR_G double *hr_lw, *hr_sw, *flw_up, *flw_dn, *fsw_up, *fsw_dn, *fsw_dn_sfc_clr;
};
// One thread per column and segment of levels (gridDim.y segments; one for large tiles, whose planes bound the
// kernel: 13 GB in FP32, 26 GB in FP64 for 796,590 columns).  A segment after the first evaluates the level
// below it once more.  Small tiles take 16: a column's 62 levels one after the other were 139 us.
template <typename P>
__global__ void __launch_bounds__(256) k_post(ColIn in, int col0, int n, ColScal cs, BandAcc ba, OutPtrs out)
{
#pragma clang fp contract(off)
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= valid_cols(in, col0, n)) return;
    const int i = col0 + t;
    const RadCol rc{in, i, in.nlay + 1};
    const int nrl = rc.nrl, nm = in.nlay;
    const size_t nc = (size_t)in.ncol;
    const double flxfac = 0.5 * FLUXFAC;
    const WR_G P *pl = (const WR_G P *)ba.base;
    // band sums in band order (the order the reference accumulates them).  Every plane is loaded and
    // the sum is selected per band, not branched on, so that the loads of a level are all in flight
    // at once; a band that is absent (single-band runs) keeps the sum unchanged, as skipping it would.
    auto lwsum = [&](int plane0, int k) {
        double v = 0.0;
#pragma unroll
        for (int b = 0; b < 16; ++b) {
            const double x = (double)pl[(size_t)(2 * b + plane0) * ba.P + (size_t)k * n + t];
            v = ((ba.lw_mask >> b) & 1) ? v + x : v;
        }
        return v;
    };
    auto swsum = [&](int plane0, int k) {
        double v = 0.0;
#pragma unroll
        for (int b = 0; b < 14; ++b) {
            const double x = (double)pl[(size_t)(32 + 2 * b + plane0) * ba.P + (size_t)k * n + t];
            v = ((ba.sw_mask >> b) & 1) ? v + x : v;
        }
        return v;
    };
    const int len = (nrl + (int)gridDim.y - 1) / (int)gridDim.y, k0 = (int)blockIdx.y * len, k1 = imin(nrl, k0 + len);
    const bool first = blockIdx.y == 0;
    if (k0 >= k1) return;
    const double up0 = lwsum(0, k0), dn0 = lwsum(1, k0);
    double fprev = up0 * flxfac - dn0 * flxfac;
    if (first) {
        out.flw_up[(size_t)nrl * nc + i] = up0 * flxfac;
        out.flw_dn[(size_t)nrl * nc + i] = dn0 * flxfac;
    }
    for (int k = k0 + 1; k <= k1; ++k) {
        const double fu = lwsum(0, k) * flxfac, fd = lwsum(1, k) * flxfac;
        out.flw_up[(size_t)(nrl - k) * nc + i] = fu;
        out.flw_dn[(size_t)(nrl - k) * nc + i] = fd;
        const double fnet = fu - fd;
        const int kin = nrl - k;  // surface-first layer k-1
        const double rfdelp = HEATFAC / (rc.plvl(kin + 1) - rc.plvl(kin));
        const double h = (fprev - fnet) * rfdelp;
        if (k - 1 < nm) out.hr_lw[(size_t)(nm - 1 - (k - 1)) * nc + i] = h;
        fprev = fnet;
    }
    if (cs.day[t]) {
        double fu0 = swsum(0, k0), fd0 = swsum(1, k0);
        if (first) {
            out.fsw_up[(size_t)nrl * nc + i] = fu0;
            out.fsw_dn[(size_t)nrl * nc + i] = fd0;
        }
        for (int k = k0; k < k1; ++k) {
            const double fu1 = swsum(0, k + 1), fd1 = swsum(1, k + 1);
            out.fsw_up[(size_t)(nrl - 1 - k) * nc + i] = fu1;
            out.fsw_dn[(size_t)(nrl - 1 - k) * nc + i] = fd1;
            const int kin = nrl - 1 - k;
            const double rf = HEATFAC / (rc.plvl(kin + 1) - rc.plvl(kin));
            const double h = ((fd1 - fu1) - (fd0 - fu0)) * rf;
            if (k < nm) out.hr_sw[(size_t)(nm - 1 - k) * nc + i] = h;
            fu0 = fu1, fd0 = fd1;
        }
        if (first && out.fsw_dn_sfc_clr) {
            double v = 0.0;
#pragma unroll
            for (int b = 0; b < 14; ++b) {
                const double x = (double)pl[(size_t)60 * ba.P + (size_t)b * n + t];
                v = ((ba.sw_mask >> b) & 1) ? v + x : v;
            }
            out.fsw_dn_sfc_clr[i] = v;
        }
    } else {
        for (int L = first ? k0 : k0 + 1; L <= k1; ++L)
            out.fsw_up[(size_t)L * nc + i] = 0.0, out.fsw_dn[(size_t)L * nc + i] = 0.0;
        for (int q = k0; q < imin(k1, nm); ++q) out.hr_sw[(size_t)q * nc + i] = 0.0;
        if (first && out.fsw_dn_sfc_clr) out.fsw_dn_sfc_clr[i] = 0.0;
    }
}

}  // namespace wr
