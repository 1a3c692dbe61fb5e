// wr_nam.h -- the NAM route (mcica = 0): LW transfer with maximum-random overlap of fractional
// clouds (rtrnmr, phys_rrtm_lw_rtrnmr_body.cuh:9-365) and the SW two-stream with cloud-fraction
// mixing and column-cover weighting (spcvrtc, phys_rrtm_sw_spcvrtc.cu:217-547).
#pragma once
#include "wr_kernels.h"

namespace wr {

// Overlap factors of one tile (rtrnmr:50-172): f[q][idx][t], idx 0..nl+2 as in the reference;
// q = 0 faccld1u, 1 faccld2u, 2 facclr1u, 3 facclr2u, 4 faccmb1u, 5 faccmb2u, 6..11 the same
// downward; lstu/lstd bit (idx - 1) set for idx = 1..nl.
template <typename R> struct Rtr {
    WR_G R *f;
    WR_G uint64_t *lstu, *lstd;
    int n;
    __device__ __forceinline__ R &at(int q, int idx, int t) const { return f[((size_t)q * (NL + 3) + idx) * n + t]; }
};
enum { FCLD1U = 0, FCLD2U, FCLR1U, FCLR2U, FCMB1U, FCMB2U, FCLD1D, FCLD2D, FCLR1D, FCLR2D, FCMB1D, FCMB2D };

// layer cloud fraction cldfrc(kk) of the LW route (1-based surface-first, cldfrc(0) = 1, (nl+1) = 0)
__device__ __forceinline__ double lw_cldfrc(const RadCol &rc, int kk)
{
    if (kk == 0) return 1.0;
    if (kk > rc.nrl) return 0.0;
    return rc.cfrac(rc.nrl - kk);
}

// The six factors of one index while the sweep that sets them is at it.
struct Fac6 {
    double cld1 = 0.0, cld2 = 0.0, clr1 = 0.0, clr2 = 0.0, cmb1 = 0.0, cmb2 = 0.0;
};

// Step k of a sweep sets the factors of the next index (k + 1 upward, k - 1 downward) and may clear
// clr2/cld2 of index k itself; no later step touches index k.  So the sweeps keep two indices in
// registers (cur = k, nxt) and three cloud fractions (cfm, cfk, cfp), and write each index as soon as
// its step is done: no per-lane arrays, no private memory.
template <typename R>
__global__ void __launch_bounds__(64) k_rtr_fac(ColIn in, int col0, int n, Rtr<R> rt)
{
#pragma clang fp contract(off)
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= valid_cols(in, col0, n)) return;
    const RadCol rc{in, col0 + t, in.nlay + 1};
    const int nl = rc.nrl;
    const double eps = 1.0e-6;
    auto put = [&](int base, int idx, const Fac6 &f) {
        rt.at(base + 0, idx, t) = (R)f.cld1, rt.at(base + 1, idx, t) = (R)f.cld2, rt.at(base + 2, idx, t) = (R)f.clr1;
        rt.at(base + 3, idx, t) = (R)f.clr2, rt.at(base + 4, idx, t) = (R)f.cmb1, rt.at(base + 5, idx, t) = (R)f.cmb2;
    };
    // one step of either sweep: k's own fraction cfk, the one it moves to (cfn) and the one it came
    // from (cfo); cur = index k, nxt = the index the step sets
    auto step = [&](double cfo, double cfk, double cfn, bool lk, double &rat1, double &rat2, Fac6 &cur, Fac6 &nxt) {
        if (!(cfk > eps)) return;
        if (cfn >= cfk) {
            if (lk) {
                if (cfk < 1.0) nxt.clr2 = (cfn - cfk) / (1.0 - cfk);
                cur.clr2 = 0.0;
                cur.cld2 = 0.0;
            } else {
                const double fmx = fmax(cfk, cfo);
                if (cfn > fmx) {
                    nxt.clr1 = rat2;
                    nxt.clr2 = (cfn - fmx) / (1.0 - fmx);
                } else if (cfn < fmx) {
                    nxt.clr1 = (cfn - cfk) / (cfo - cfk);
                } else {
                    nxt.clr1 = rat2;
                }
            }
            if (nxt.clr1 > 0.0 || nxt.clr2 > 0.0) rat1 = 1.0, rat2 = 0.0;
            else rat1 = 0.0, rat2 = 0.0;
        } else {
            if (lk) {
                nxt.cld2 = (cfk - cfn) / cfk;
                cur.clr2 = 0.0;
                cur.cld2 = 0.0;
            } else {
                const double fmn = fmin(cfk, cfo);
                if (cfn <= fmn) {
                    nxt.cld1 = rat1;
                    nxt.cld2 = (fmn - cfn) / fmn;
                } else {
                    nxt.cld1 = (cfk - cfn) / (cfk - fmn);
                }
            }
            if (nxt.cld1 > 0.0 || nxt.cld2 > 0.0) rat1 = 0.0, rat2 = 1.0;
            else rat1 = 0.0, rat2 = 0.0;
        }
        nxt.cmb1 = nxt.clr1 * cur.cld2 * cfo;
        nxt.cmb2 = nxt.cld1 * cur.clr2 * (1.0 - cfo);
    };
    const Fac6 zero;
    // upward factors: index 0 stays zero, step k = 1..nl-1 sets index k + 1
    {
        uint64_t lst = 0;
        double cfm = lw_cldfrc(rc, 0), cfk = lw_cldfrc(rc, 1);
        bool lk = cfk > eps;
        if (lk) lst |= 1ull;
        double rat1 = 0.0, rat2 = 0.0;
        Fac6 cur;
        put(FCLD1U, 0, zero);
        for (int k = 1; k <= nl - 1; ++k) {
            const double cfp = lw_cldfrc(rc, k + 1);
            const bool lk1 = cfp > eps && cfk <= eps;
            if (lk1) lst |= 1ull << k;
            Fac6 nxt;
            step(cfm, cfk, cfp, lk, rat1, rat2, cur, nxt);
            put(FCLD1U, k, cur);
            cur = nxt;
            lk = lk1;
            cfm = cfk;
            cfk = cfp;
        }
        put(FCLD1U, nl, cur);
        put(FCLD1U, nl + 1, zero);
        put(FCLD1U, nl + 2, zero);
        rt.lstu[t] = lst;
    }
    // downward factors: indices nl+1, nl+2 stay zero, step k = nl..2 sets index k - 1
    {
        uint64_t lst = 0;
        double cfp = lw_cldfrc(rc, nl + 1), cfk = lw_cldfrc(rc, nl);
        bool lk = cfk > eps;
        if (lk) lst |= 1ull << (nl - 1);
        double rat1 = 0.0, rat2 = 0.0;
        Fac6 cur;
        put(FCLD1D, nl + 2, zero);
        put(FCLD1D, nl + 1, zero);
        for (int k = nl; k >= 2; --k) {
            const double cfm = lw_cldfrc(rc, k - 1);
            const bool lkm = cfm > eps && cfk <= eps;
            if (lkm) lst |= 1ull << (k - 2);
            Fac6 nxt;
            step(cfp, cfk, cfm, lk, rat1, rat2, cur, nxt);
            put(FCLD1D, k, cur);
            cur = nxt;
            lk = lkm;
            cfp = cfk;
            cfk = cfm;
        }
        put(FCLD1D, 1, cur);
        put(FCLD1D, 0, zero);
        rt.lstd[t] = lst;
    }
}

// ---- LW band kernel of the NAM route (rtrnmr) ---------------------------------------------------
// Per-band optics chunks and wave bounds, by precision, as for the McICA route's LW kernels (same reasons); the
// three radiances a g-point of a cloudy layer has (clear, cloudy, their overlap) leave room for fewer waves.
// WR_LWR_WAVES > 0 or WR_LWR_CHUNK >= 0 override the tables for every band (tuning builds).
constexpr int LWR64_WAVES[16] = {1, 1, 1, 1, 1, 2, 1, 2, 1, 2, 2, 2, 2, 2, 2, 2};
constexpr int LWR64_CHUNK[16] = {5, 4, 4, 2, 4, 4, 4, 4, 4, 3, 4, 4, 4, 2, 2, 2};
constexpr int LWR32_WAVES[16] = {3, 2, 2, 2, 2, 3, 2, 3, 2, 4, 3, 3, 4, 4, 4, 4};
constexpr int LWR32_CHUNK[16] = {5, 4, 4, 2, 4, 4, 4, 4, 4, 3, 4, 4, 4, 2, 2, 2};
#ifndef WR_LWR_WAVES
#define WR_LWR_WAVES 0
#endif
#ifndef WR_LWR_CHUNK
#define WR_LWR_CHUNK -1
#endif
template <typename R, int B> constexpr int lwr_waves()
{
    return WR_LWR_WAVES > 0 ? WR_LWR_WAVES : (sizeof(R) == 8 ? LWR64_WAVES[B] : LWR32_WAVES[B]);
}
template <typename R, int B> constexpr int lwr_chunk()
{
    return chunk_of(LW_NG[B], WR_LWR_CHUNK >= 0 ? WR_LWR_CHUNK : (sizeof(R) == 8 ? LWR64_CHUNK[B] : LWR32_CHUNK[B]));
}

// the overlap factors of one step of a sweep and the layer's cloud fraction
template <typename R> struct RtrStep {
    R clfr, cld1, cld2, clr1, clr2, cmb1, cmb2;
    bool start;  // a cloud block starts here
};
template <typename R>
__device__ __forceinline__ RtrStep<R> rtr_step(const Rtr<R> &rt, int q0, int idx, int t, R clfr, bool start)
{
    return {clfr, rt.at(q0, idx, t), rt.at(q0 + 1, idx, t), rt.at(q0 + 2, idx, t), rt.at(q0 + 3, idx, t), rt.at(q0 + 4, idx, t),
            rt.at(q0 + 5, idx, t), start};
}
// radiances of one g-point through a layer with cloud in some lane: total (tot), its cloudy and clear parts,
// the overlap correction; gas and src the clear and cloudy sources, tr and trc the transmittances
template <typename R>
__device__ __forceinline__ void rtr_update(const RtrStep<R> &f, bool cloudy, R gas, R src, R tr, R trc, R &tot, R &cld, R &clr, R &rad)
{
    const R clear = tot * tr + gas;
    R a = cld, b = clr, r = rad;
    if (f.start) {
        a = f.clfr * tot;
        b = tot - a;
        r = (R)0;
    }
    R na = a * trc + f.clfr * src;
    R nb = b * tr + ((R)1 - f.clfr) * gas;
    const R ntot = na + nb;
    const R mod = r * (f.clr1 * tr + f.cld1 * trc) - f.cmb1 * gas + f.cmb2 * src;
    const R nr = -mod + f.clr2 * (nb + mod) - f.cld2 * (na - mod);
    na = na + nr;
    nb = nb - nr;
    tot = cloudy ? ntot : clear;
    cld = cloudy ? na : a;
    clr = cloudy ? nb : b;
    rad = cloudy ? nr : r;
}

// One column of LW band B on the NAM route (rtrnmr), optics from the band tables Bt: down sweep, surface, up
// sweep with the optics evaluated again, in chunks of g-points without per-g-point branches (as lw_column).
template <typename R, int B, typename BT>
__device__ __forceinline__ void lwr_column(const Tabs<R> *__restrict__ T, const BT &Bt, const ColIn &in, const RunPar &par,
                                           int col0, int n, const ColScal &cs, const RecPtrs &rp, const AccT<R> &acc,
                                           const Rtr<R> &rt, int blk, int lane)
{
    constexpr int NG = LW_NG[B], GW = NG, CH = lwr_chunk<R, B>();
    const Share<R> sh{nullptr, 0, 0};
    const int nv = valid_cols(in, col0, n);
    if (blk * 64 >= nv) return;
    const bool ok = blk * 64 + lane < nv;  // lanes past the last column repeat it and store nothing
    const int rl = ok ? lane : nv - 1 - blk * 64, t = blk * 64 + rl;
    const Surr none{};
    const LwCol<R> c = lw_col<R, B, false>(in, col0, cs, none, t);
    const int nrl = c.nrl;
    const RadCol rcol{in, c.i, nrl};
    const uint64_t lstu = rt.lstu[t], lstd = rt.lstd[t];
    if (ok) acc.lw_dn[(size_t)nrl * n + t] = (R)0;  // no downward LW at the top
    // radiances per g-point: total, its cloudy and clear parts, the overlap correction between them
    R tot[1][GW], cld[GW], clr[GW], rad[GW], sfc0[1][GW];
#pragma unroll
    for (int g = 0; g < GW; ++g) tot[0][g] = cld[g] = clr[g] = rad[g] = (R)0;
    // one layer of a sweep; q0, idx: the overlap factors of its direction; start: a cloud block starts here
    auto sweep = [&](int k, const LwLayer<R> &y, R dplnk, int q0, int idx, bool start, bool sfc, R pk0) {
        const bool some = __any(y.cloudy);
        RtrStep<R> f{};
        if (some) f = rtr_step<R>(rt, q0, idx, t, (R)rcol.cfrac(nrl - 1 - k), start);
#pragma unroll
        for (int g0 = 0; g0 < GW; g0 += CH) {
            R tau[CH], fr[CH];
            lw_taufr<R, B, false, CH>(T, Bt, none, c, n, k, y.L, g0, tau, fr);
            GasV<R, CH> q;
            lw_gas_v<R, CH>(Bt.etab, c.sdif, y.taer, tau, q);
            if (sfc) {  // surface emission and reflection
#pragma unroll
                for (int j = 0; j < CH; ++j) {
                    const int g = g0 + j;
                    const R r0 = c.semis * fr[j] * pk0;
                    tot[0][g] = r0 + c.reflct * tot[0][g];
                    cld[g] = clr[g] = rad[g] = (R)0;
                    sfc0[0][g] = tot[0][g];
                }
            }
            R gas[CH];
#pragma unroll
            for (int j = 0; j < CH; ++j) gas[j] = fr[j] * (y.blay + dplnk * q.gf[j]) * q.at[j];
            if (some) {
                R trc[CH], at[CH], gf[CH];
                lw_tot_v<R, CH>(Bt.etab, q.od, y.odcld, trc, at, gf);
#pragma unroll
                for (int j = 0; j < CH; ++j) {
                    const int g = g0 + j;
                    const R src = fr[j] * (y.blay + dplnk * gf[j]) * at[j];
                    rtr_update<R>(f, y.cloudy, gas[j], src, q.tr[j], trc[j], tot[0][g], cld[g], clr[g], rad[g]);
                }
            } else {
#pragma unroll
                for (int j = 0; j < CH; ++j) tot[0][g0 + j] = tot[0][g0 + j] * q.tr[j] + gas[j];
            }
            if constexpr (CH < GW) __builtin_amdgcn_sched_barrier(0);
        }
    };
    LevelSum<R, NG, GW, 1> sum{sh, lane, 0, 0, 0};
    auto dn = [&](int row, const R *s) {
        if (ok) acc.lw_dn[(size_t)row * n + t] = s[0];
    };
    auto up = [&](int row, const R *s) {
        if (ok) acc.lw_up[(size_t)row * n + t] = s[0];
    };
    sum.begin(nrl - 1, -1);
    for (int k = nrl - 1; k >= 0; --k) {  // down sweep, top to surface
        LwLayer<R> y;
        lw_get<R, B>(T, in, par, rp, c, blk, rl, k, y);
        sweep(k, y, y.bbot - y.blay, FCLD1D, k, (lstd >> k) & 1, false, (R)0);
        sum.put(tot, dn);
    }
    sum.finish(dn);
    sum.begin(0, 1);
    for (int k = 0; k < nrl; ++k) {  // up sweep, surface to top
        LwLayer<R> y;
        lw_get<R, B>(T, in, par, rp, c, blk, rl, k, y);
        R btop = y.blay;  // above the top layer, its own temperature
        if (k + 1 < nrl) {
            const LRow<R> nx = lrow<R>(rp, blk, k + 1, rl);
            btop = planck_of<R>(T, B, (int)(nx.w(1) & 255u), nx.f(LF_PB));
        }
        sweep(k, y, btop - y.blay, FCLD1U, k + 2, (lstu >> k) & 1, k == 0, y.bbot);
        if (k == 0) sum.put(sfc0, up);
        sum.put(tot, up);
    }
    sum.finish(up);
}

template <typename R, int B, bool EXT = true>
__global__ void __launch_bounds__(64, (lwr_waves<R, B>())) k_lwr(const Tabs<R> *__restrict__ T, ColIn in_, RunPar par, int col0,
                                            int n, ColScal cs, RecPtrs rp, AccT<R> acc, Rtr<R> rt)
{
    const ColIn in = band_in<EXT>(in_);
    lwr_column<R, B>(T, T->lw[B], in, par, col0, n, cs, rp, acc, rt, (int)blockIdx.x, (int)threadIdx.x);
}

// k_lwr with the band's tables in LDS (the image of k_lwl / k_lwl64: FP64 keeps absb in global
// memory): persistent workgroups of 4 x lwr_waves waves, as many as the CUs hold at once, each
// copying the image into LDS once.  Same arithmetic as k_lwr.
template <typename R, int B> constexpr int lwrl_wpg() { return 4 * lwr_waves<R, B>(); }
template <typename R, int B, bool EXT = true>
__global__ void __launch_bounds__((64 * lwrl_wpg<R, B>()), (lwr_waves<R, B>()))
    k_lwrl(const Tabs<R> *__restrict__ T, ColIn in_, RunPar par, int col0, int n, ColScal cs, RecPtrs rp, AccT<R> acc,
           Rtr<R> rt)
{
    extern __shared__ float4 lwrl_tab[];
    const ColIn in = band_in<EXT>(in_);
    const LwImg<R> &im = T->lw_img[B];
    lds_fill_lw<R>(lwrl_tab, im, T->exp_tbl);
    const WR_L R *lt = (const WR_L R *)lwrl_tab;
    constexpr int WPG = lwrl_wpg<R, B>();
    const int lane = threadIdx.x % 64;
    if constexpr (sizeof(R) == 4) {
        const auto Bl = lds_band<R, B>(lt, im, T->lw[B], lt + (imax(0, im.off[1]) & ~3));
        for (int blk = wave_slot(); blk * 64 < n; blk += gridDim.x * WPG)
            lwr_column<R, B>(T, Bl, in, par, col0, n, cs, rp, acc, rt, blk, lane);
    } else {
        const auto Bl = lds_band<R, B>(lt, im, T->lw[B], T->lw[B].absb);
        for (int blk = wave_slot(); blk * 64 < n; blk += gridDim.x * WPG)
            lwr_column<R, B>(T, Bl, in, par, col0, n, cs, rp, acc, rt, blk, lane);
    }
}

// ---- SW band kernel of the NAM route (spcvrtc with cldfrc mixing and zcf1/zcf0 weighting) -------
// o = zc0 o + zc1 d: the cloudy R/T of a layer mixed into the clear ones
template <typename R, int CH> __device__ __forceinline__ void rt_mix(bool mix, R zc0, R zc1, const RtV<R, CH> &d, RtV<R, CH> &o)
{
#pragma unroll
    for (int j = 0; j < CH; ++j) {
        o.rb[j] = mix ? zc0 * o.rb[j] + zc1 * d.rb[j] : o.rb[j];
        o.rd[j] = mix ? zc0 * o.rd[j] + zc1 * d.rd[j] : o.rd[j];
        o.tb[j] = mix ? zc0 * o.tb[j] + zc1 * d.tb[j] : o.tb[j];
        o.td[j] = mix ? zc0 * o.td[j] + zc1 * d.td[j] : o.td[j];
        o.ld[j] = mix ? zc0 * o.ld[j] + zc1 * d.ld[j] : o.ld[j];
    }
}

// The fluxes of a level, {clear up, clear down, total up, total down}, to the band planes.
template <typename R>
__device__ __forceinline__ void swr_emit(const AccT<R> &acc, bool ok, bool total, double cf1, double cf0, int lev, int n, int t,
                                         const R *f)
{
    if (!ok) return;
    const size_t p = (size_t)lev * n + t;
    if (lev == 0) acc.sw_clr0[t] = f[1];
    acc.sw_up[p] = total ? (R)(cf1 * (double)f[2] + cf0 * (double)f[0]) : f[0];
    acc.sw_dn[p] = total ? (R)(cf1 * (double)f[3] + cf0 * (double)f[1]) : f[1];
}

// One day column of one SW band on the NAM route: the clear sky and, for cloudy columns, the total sky,
// whose layers mix the cloudy R/T with the clear ones by the layer's cloud fraction over the column's
// cover, zc1 = cfrac / zcf1 (phys_rrtm_sw_spcvrtc.cu, cloudy block).  Both skies go through the adding method
// together, on one evaluation of the optics; the column's fluxes are cf1 x total + cf0 x clear.
template <typename R, int B, typename BT>
__device__ __forceinline__ void swr_column(const Tabs<R> *__restrict__ T, const BT &Bt, const ColIn &in, const RunPar &par, int col0,
                                           int n, const ColScal &cs, const RecPtrs &rp, const R *__restrict__ sflux,
                                           const AccT<R> &acc, int blk, int lane, WR_G char *slot, Fix64 *fx)
{
    constexpr int NG = SW_NG[B], CH = sw_chunk<R, B, true>();
    const int nday = *cs.nday;
    if (blk * 64 >= nday) return;
    const bool ok = blk * 64 + lane < nday;  // lanes past the last day column repeat it and store nothing
    const int rl = ok ? lane : nday - 1 - blk * 64;
    const int t = cs.dlist[blk * 64 + rl], nrl = rp.nrl;
    SwCol<R> c;
    sw_col<R, B>(in, par, col0, cs, t, c);
    const RadCol rcol{in, c.i, nrl};
    const double cf1 = cs.zcf1[t], cf0 = cs.zcf0[t];
    const bool total = cf1 > EPS;
    const Surr none{};
    struct Lay {
        SwLayer<R> y;
        R zc1, zc0;
        bool mix;
    };
    const bool two = __any(total);
    sw_adding<R, NG, NG, CH, 2>(
        nrl, c.asfc, two, SwSlot<R, NG>{slot, lane, in.nlay + 2}, lane, Share<R>{nullptr, 0, 0},
        [&](int k, int) {
            Lay a;
            sw_get<R, B>(T, in, par, rp, c.i, c.cz, c.snt, blk, rl, k, a.y);
            a.mix = false, a.zc1 = (R)0, a.zc0 = (R)1;
            if (two && __any(a.y.cloudy)) {
                const double zc1 = rcol.cfrac(nrl - 1 - k) / cf1;
                a.mix = total && zc1 > FTINY, a.zc1 = (R)zc1, a.zc0 = (R)(1.0 - zc1);
            }
            return a;
        },
        [&](const Lay &a, int k, int g0, RtV<R, CH> (&o)[2]) {
            R tg[CH], tr[CH];
            sw_tgtr<R, B, false, CH>(T, Bt, none, 1, 0, k, c.lt, a.y.L, g0, tg, tr);
            layer_rt_sky<R, CH>(T, tr, tg, a.y.y, 0u, o[0], fx);
            o[1] = o[0];
            if (__any(a.mix)) {
                RtV<R, CH> d;
                layer_rt_sky<R, CH>(T, tr, tg, a.y.y, ~0u, d, fx);
                rt_mix<R, CH>(a.mix, a.zc0, a.zc1, d, o[1]);
            }
        },
        [&](int g) { return c.ssolar * sflux[(size_t)(SW_NS[B] + g) * n + t]; },
        [&](int lev, const R *f) { swr_emit<R>(acc, ok, total, cf1, cf0, lev, n, t, f); });
}

// SW band kernel of the NAM route: blocks of 64 day-list entries looped over a pool-sized grid.
template <typename R, int B, bool EXT = true>
__global__ void __launch_bounds__(64, (sw_waves<R, B, true>())) k_swr(const Tabs<R> *__restrict__ T, ColIn in_, RunPar par, int col0,
                                            int n, ColScal cs, RecPtrs rp, const R *__restrict__ sflux, AccT<R> acc,
                                            char *__restrict__ pool)
{
    __shared__ Fix64 fx[1];
    const ColIn in = band_in<EXT>(in_);
    WR_G char *slot = (WR_G char *)(pool + (size_t)blockIdx.x * cache_slot_bytes(2 * sw_nv<R>(), SW_NG[B], in.nlay + 2, (int)sizeof(R)));
    const int nday = *cs.nday;
    for (int blk = blockIdx.x; blk * 64 < nday; blk += gridDim.x)
        swr_column<R, B>(T, T->sw[B], in, par, col0, n, cs, rp, sflux, acc, blk, (int)threadIdx.x, slot, fx);
}

// k_swr with the band's tables in LDS (the images of k_swl): persistent workgroups of 4 x the band's
// waves, as many as the CUs hold at once, each wave with its own pool slot.  Same arithmetic as k_swr.
template <typename R, int B> constexpr int swrl_wpg() { return 4 * sw_waves<R, B, true>(); }
template <typename R, int B, bool EXT = true>
__global__ void __launch_bounds__((64 * swrl_wpg<R, B>()), (sw_waves<R, B, true>()))
    k_swrl(const Tabs<R> *__restrict__ T, ColIn in_, RunPar par, int col0, int n, ColScal cs, RecPtrs rp,
           const R *__restrict__ sflux, AccT<R> acc, char *__restrict__ pool)
{
    extern __shared__ float4 swrl_tab[];
    const ColIn in = band_in<EXT>(in_);
    lds_fill<R>(swrl_tab, T->sw_img[B]);
    const auto Bl = sw_lds_band<R>((const WR_L R *)swrl_tab, T->sw_img[B], T->sw[B]);
    constexpr int WPG = swrl_wpg<R, B>();
    __shared__ Fix64 fx[sizeof(R) == 4 ? WPG : 1];
    const int lane = threadIdx.x % 64, wv = wave_id(), w = wave_slot();
    WR_G char *slot = (WR_G char *)(pool + (size_t)w * cache_slot_bytes(2 * sw_nv<R>(), SW_NG[B], in.nlay + 2, (int)sizeof(R)));
    const int nday = *cs.nday;
    for (int blk = w; blk * 64 < nday; blk += gridDim.x * WPG)
        swr_column<R, B>(T, Bl, in, par, col0, n, cs, rp, sflux, acc, blk, lane, slot, fx + (sizeof(R) == 4 ? wv : 0));
}

}  // namespace wr
