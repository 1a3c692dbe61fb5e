// wr_many.h -- the bands of a small tile, in two launches for all of them.
//
// A tile of some thousand columns gives each of the 30 band kernels only n / 64 waves, far fewer than
// the 1,024 SIMDs hold, and a wave's time is one column's serial chain: for each of 61 layers (twice, where
// a sweep evaluates the optics again) the loads of its record, the table gathers that depend on them and
// the arithmetic, about 9 us a layer.  Only the radiances and the adding method need one layer after
// the other; the optics do not.  So the small tiles run
//   k_lay    the optics of every (64-column block, band, layer): transmittances and sources (LW), layer
//            R/T (SW) to the pool, one wave each, all of them independent;
//   k_sweep  the sweeps of every (block, band) over those values, MANY_GW g-points per wave; the level sums over
//            the waves of a band meet in LDS in g order.
// Both use the expressions of the per-band kernels, so the outputs are the same bits.
//
// Values that only clouds need are written and read only for the layers of a block that hold cloud.  The NAM
// route's two skies share a sweep.  Bound by latency at a few hundred columns (257 columns FP64: optics 83,
// sweeps 140 us), by the optics' issue and the pool's traffic at several thousand (4,096: 1,040 and 900 us);
// above many_cols the per-band kernels, which keep a column's values in registers, are faster.
#pragma once
#include "wr_launch.h"

namespace wr {

// g-points per wave of a sweep (every band's count is a multiple), waves per workgroup (the widest band's 16)
constexpr int MANY_GW = 2, MANY_W = 16 / MANY_GW;
constexpr int MANY_LAYERS = 4;  // layers (waves) per k_lay workgroup

// band ids, the ones with most g-points first
constexpr int MANY_ORDER[30] = {17, 29, 21, 20, 23, 2,  4,  3,  24, 8,  6,  19, 18, 27, 1,
                                11, 0,  28, 16, 25, 26, 12, 10, 7,  5,  9,  14, 15, 22, 13};

// Pool values per layer and g-point.  LW: FP32 McICA {a, b down, b up}; FP64 McICA {transmittance, gas source
// and cloud minus gas source, down and up}; NAM {clear transmittance, clear and cloudy source, down and up,
// cloudy transmittance}.  SW: R/T (NAM: of the clear sky, then of the mixed sky).
template <typename R, bool NAM> constexpr int many_vl() { return NAM ? 6 : sizeof(R) == 4 ? 3 : 5; }
template <bool NAM> constexpr int many_vs() { return NAM ? 10 : 5; }
// pool values of one 64-column block, per lane: [140][nrl][VL], surface source [140], cloud transmittance
// [16][nrl], SW [112][nrl][VS], FP64 reflectances [112][nrl][2] of each sky (the FP32
// sweep leaves its 5 values in the place of the layer's R/T)
template <typename R, bool NAM> constexpr size_t many_lane_values(int nrl)
{
    return (size_t)140 * nrl * many_vl<R, NAM>() + 140 + (size_t)16 * nrl + (size_t)112 * nrl * many_vs<NAM>() +
           (sizeof(R) == 8 ? (size_t)112 * nrl * sw_nv<R>() * (NAM ? 2 : 1) : 0);
}
template <typename R, bool NAM> constexpr size_t many_block_bytes(int nrl)
{
    return many_lane_values<R, NAM>(nrl) * 64 * sizeof(R);
}

template <typename R> struct ManyArgs {
    const Tabs<R> *T;
    const R *sflux;
    ColIn in;
    RunPar par;
    int col0, n, blk0, nblk;  // blocks blk0 .. blk0 + nblk - 1 of 64 columns
    ColScal cs;
    RecPtrs rp;
    BandAcc ba;
    Surr sg;
    Rtr<R> rt;
    char *pool;
};

// One block's part of the pool.
template <typename R, bool NAM> struct ManyBlk {
    WR_G R *p;
    int nrl;
    static constexpr int VL = many_vl<R, NAM>(), VS = many_vs<NAM>();
    __device__ __forceinline__ WR_G R *lw(int g, int k, int lane) const { return p + ((size_t)g * nrl + k) * VL * 64 + lane; }
    __device__ __forceinline__ WR_G R *sfc(int g, int lane) const { return p + ((size_t)140 * nrl * VL + g) * 64 + lane; }
    __device__ __forceinline__ WR_G R *ef(int b, int k, int lane) const
    {
        return p + ((size_t)140 * nrl * VL + 140 + (size_t)b * nrl + k) * 64 + lane;
    }
    __device__ __forceinline__ WR_G R *sw(int g, int k, int lane) const
    {
        return p + ((size_t)140 * nrl * VL + 140 + (size_t)16 * nrl + ((size_t)g * nrl + k) * VS) * 64 + lane;
    }
    __device__ __forceinline__ WR_G R *refl(int g, int k, int sky, int lane) const
    {
        return p + ((size_t)140 * nrl * VL + 140 + (size_t)16 * nrl + (size_t)112 * nrl * VS +
                    ((size_t)g * nrl + k) * (NAM ? 4 : 2) + 2 * sky) * 64 + lane;
    }
};
template <typename R, bool NAM>
__device__ __forceinline__ ManyBlk<R, NAM> many_blk(const ManyArgs<R> &a, int b)
{
    return {(WR_G R *)a.pool + many_lane_values<R, NAM>(a.rp.nrl) * 64 * b, a.rp.nrl};
}

// ---- optics of one layer of one block ----------------------------------------------------------
template <typename R, int B, bool NAM, bool SURR>
__device__ __forceinline__ void lay_lw(const ManyArgs<R> &a, int b, int k, int lane)
{
    constexpr int NG = LW_NG[B], NS = LW_NS[B], CH = chunk_of(NG, NG == 14 ? 2 : 4);
    const int blk = a.blk0 + b, nv = valid_cols(a.in, a.col0, a.n);
    if (blk * 64 >= nv) return;
    const int rl = imin(lane, nv - 1 - blk * 64), t = blk * 64 + rl;
    const LwCol<R> c = lw_col<R, B, SURR>(a.in, a.col0, a.cs, a.sg, t);
    const ManyBlk<R, NAM> m = many_blk<R, NAM>(a, b);
    LwLayer<R> y;
    lw_get<R, B>(a.T, a.in, a.par, a.rp, c, blk, rl, k, y);
    uint32_t bits = 0;
    if (!NAM && y.cloudy) bits = mword(a.rp.mlw, a.rp.row(blk, k), MROW_LW, B, rl);
    R btop = y.blay;
    if (k + 1 < c.nrl) {
        const LRow<R> nx = lrow<R>(a.rp, blk, k + 1, rl);
        btop = planck_of<R>(a.T, B, (int)(nx.w(1) & 255u), nx.f(LF_PB));
    }
    const R dd = y.bbot - y.blay, du = btop - y.blay;
    R ecld = (R)1;
    if (!NAM && __any(y.cloudy)) ecld = M<R>::exp(-y.odcld);
    // what only clouds need is stored where the block's layer has any (many_cloud tells the sweeps)
    const bool some = __any(y.cloudy);
    if constexpr (!NAM && sizeof(R) == 8)
        if (some) *m.ef(B, k, lane) = (R)1 - ((R)1 - ecld);
#pragma unroll
    for (int g0 = 0; g0 < NG; g0 += CH) {
        R tau[CH], fr[CH];
        lw_taufr<R, B, SURR, CH>(a.T, a.T->lw[B], a.sg, c, a.n, k, y.L, g0, tau, fr);
        if (k == 0) {
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                const R rad0 = c.semis * fr[j] * y.bbot;
                *m.sfc(NS + g0 + j, lane) = rad0;
            }
        }
        if constexpr (!NAM && sizeof(R) == 4) {
            R ta[CH], bd[CH], bu[CH];
            lw_chunk_f32<CH>(y, c.sdif, dd, du, ecld, bits >> g0, tau, fr, ta, bd, bu);
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                WR_G R *q = m.lw(NS + g0 + j, k, lane);
                q[0] = ta[j], q[64] = bd[j], q[128] = bu[j];
            }
        } else {
            GasV<R, CH> q;
            lw_gas_v<R, CH>(a.T->exp_tbl, c.sdif, y.taer, tau, q);
            R gd[CH], gu[CH], trc[CH], sd[CH], su[CH];
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                gd[j] = fr[j] * (y.blay + dd * q.gf[j]) * q.at[j];
                gu[j] = fr[j] * (y.blay + du * q.gf[j]) * q.at[j];
                trc[j] = q.tr[j], sd[j] = (R)0, su[j] = (R)0;
            }
            const uint32_t cb = NAM ? (y.cloudy ? ~0u : 0u) : bits >> g0;
            if (__any(cb & ((1u << CH) - 1u))) {
                R at[CH], gf[CH];
                lw_tot_v<R, CH>(a.T->exp_tbl, q.od, y.odcld, trc, at, gf);
#pragma unroll
                for (int j = 0; j < CH; ++j) {
                    const R td = fr[j] * (y.blay + dd * gf[j]) * at[j], tu = fr[j] * (y.blay + du * gf[j]) * at[j];
                    if constexpr (NAM) {
                        sd[j] = td, su[j] = tu;
                    } else {
                        const bool cl = (cb >> j) & 1u;
                        sd[j] = cl ? td - gd[j] : (R)0, su[j] = cl ? tu - gu[j] : (R)0;
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                WR_G R *w = m.lw(NS + g0 + j, k, lane);
                w[0] = q.tr[j], w[64] = gd[j], w[192] = gu[j];
                if (some) {
                    w[128] = sd[j], w[256] = su[j];
                    if constexpr (NAM) w[320] = trc[j];
                }
            }
        }
        if constexpr (CH < NG) __builtin_amdgcn_sched_barrier(0);
    }
}

template <typename R, int B, bool NAM, bool SURR>
__device__ __forceinline__ void lay_sw(const ManyArgs<R> &a, int b, int k, int lane, Fix64 *fx)
{
    constexpr int NG = SW_NG[B], NS = SW_NS[B], CH = 2;
    const int blk = a.blk0 + b, nday = *a.cs.nday;
    if (blk * 64 >= nday) return;
    const int rl = imin(lane, nday - 1 - blk * 64), t = a.cs.dlist[blk * 64 + rl];
    SwCol<R> c;
    sw_col<R, B>(a.in, a.par, a.col0, a.cs, t, c);
    const int table = SURR ? a.sg.table(t, 16 + B) : 1;
    const ManyBlk<R, NAM> m = many_blk<R, NAM>(a, b);
    SwLayer<R> y;
    sw_get<R, B>(a.T, a.in, a.par, a.rp, c.i, c.cz, c.snt, blk, rl, k, y);
    uint32_t bits = 0;
    bool mix = false;
    R zc1 = (R)0, zc0 = (R)1;
    const bool some = __any(y.cloudy);
    if constexpr (NAM) {
        if (some) {
            const RadCol rcol{a.in, c.i, a.rp.nrl};
            const double cf1 = a.cs.zcf1[t], z = rcol.cfrac(a.rp.nrl - 1 - k) / cf1;
            mix = cf1 > EPS && z > FTINY, zc1 = (R)z, zc0 = (R)(1.0 - z);
        }
    } else if (y.cloudy) {
        bits = mword(a.rp.msw, a.rp.row(blk, k), MROW_SW, B, rl);
    }
    auto put = [&](WR_G R *q, const RtV<R, CH> &o, int j) {
        q[0] = o.rb[j], q[64] = o.rd[j], q[128] = o.tb[j], q[192] = o.td[j], q[256] = o.ld[j];
    };
#pragma unroll
    for (int g0 = 0; g0 < NG; g0 += CH) {
        R tg[CH], tr[CH];
        sw_tgtr<R, B, SURR, CH>(a.T, a.T->sw[B], a.sg, table, (size_t)k * a.n + t, k, c.lt, y.L, g0, tg, tr);
        RtV<R, CH> o;
        layer_rt_sky<R, CH>(a.T, tr, tg, y.y, bits >> g0, o, fx);
#pragma unroll
        for (int j = 0; j < CH; ++j) put(m.sw(NS + g0 + j, k, lane), o, j);
        if constexpr (NAM) {
            if (some) {
                RtV<R, CH> d;
                layer_rt_sky<R, CH>(a.T, tr, tg, y.y, ~0u, d, fx);
                rt_mix<R, CH>(mix, zc0, zc1, d, o);
#pragma unroll
                for (int j = 0; j < CH; ++j) put(m.sw(NS + g0 + j, k, lane) + 320, o, j);
            }
        }
        if constexpr (CH < NG) __builtin_amdgcn_sched_barrier(0);
    }
}

template <typename R, bool NAM, bool SURR, int P>
__device__ __forceinline__ void lay_run(const ManyArgs<R> &a, int pos, int b, int k, int lane, Fix64 *fx)
{
    if constexpr (P < 30) {
        constexpr int id = MANY_ORDER[P];
        if (pos != P) return lay_run<R, NAM, SURR, P + 1>(a, pos, b, k, lane, fx);
        if constexpr (id < 16)
            lay_lw<R, id, NAM, SURR>(a, b, k, lane);
        else
            lay_sw<R, id - 16, NAM, SURR>(a, b, k, lane, fx);
    }
}
// grid: nblk blocks x layer groups x 30 bands
template <typename R, bool NAM, bool SURR>
__global__ void __launch_bounds__(64 * MANY_LAYERS, sizeof(R) == 4 ? 3 : 2) k_lay(ManyArgs<R> a)
{
    __shared__ Fix64 fx[sizeof(R) == 4 ? MANY_LAYERS : 1];
    const int w = wave_id(), k = (int)blockIdx.y * MANY_LAYERS + w;
    if (k >= a.rp.nrl) return;
    lay_run<R, NAM, SURR, 0>(a, (int)blockIdx.z, (int)blockIdx.x, k, (int)(threadIdx.x & 63), fx + (sizeof(R) == 4 ? w : 0));
}

// ---- sweeps of one block and band ----------------------------------------------------------------
// The layers of a block that hold cloud in any of its columns (bit k).
template <bool SW, typename R> __device__ __forceinline__ uint64_t many_cloud(const RecPtrs &rp, int blk, int lane)
{
    uint64_t m = 0;
#pragma unroll 8
    for (int k = 0; k < rp.nrl; ++k) {
        const uint32_t w = SW ? srow<R>(rp, blk, k, lane).w(1) : lrow<R>(rp, blk, k, lane).w(1) & 256u;
        m |= (uint64_t)(__any(w != 0) ? 1 : 0) << k;
    }
    return m;
}

template <typename R, int B, bool NAM>
__device__ __forceinline__ void sweep_lw(const ManyArgs<R> &a, int b, int lane, const Share<R> &sh)
{
    constexpr int NG = LW_NG[B], NS = LW_NS[B], GW = MANY_GW;
    const int blk = a.blk0 + b, nv = valid_cols(a.in, a.col0, a.n);
    if (blk * 64 >= nv) return;
    const bool ok = blk * 64 + lane < nv;
    const int rl = ok ? lane : nv - 1 - blk * 64, t = blk * 64 + rl, nrl = a.rp.nrl;
    const LwCol<R> c = lw_col<R, B, false>(a.in, a.col0, a.cs, Surr{}, t);
    const ManyBlk<R, NAM> m = many_blk<R, NAM>(a, b);
    const AccT<R> acc = band_acc<R>(a.ba, B);
    const int gs = NS + sh.g0;
    if (ok) acc.lw_dn[(size_t)nrl * a.n + t] = (R)0;  // no downward LW at the top
    LevelSum<R, NG, GW, 1> sum{sh, lane, 0, 0, 0};
    auto dn = [&](int row, const R *s) {
        if (ok) acc.lw_dn[(size_t)row * a.n + t] = s[0];
    };
    auto up = [&](int row, const R *s) {
        if (ok) acc.lw_up[(size_t)row * a.n + t] = s[0];
    };
    R rad[1][GW], cld[GW], clr[GW], cor[GW];
#pragma unroll
    for (int j = 0; j < GW; ++j) rad[0][j] = cld[j] = clr[j] = cor[j] = (R)0;
    uint64_t lstu = 0, lstd = 0;
    if constexpr (NAM) lstu = a.rt.lstu[t], lstd = a.rt.lstd[t];
    const RadCol rcol{a.in, c.i, nrl};
    const uint64_t clouds = NAM || sizeof(R) == 8 ? many_cloud<false, R>(a.rp, blk, rl) : 0;
    // one layer; v: 0 the downward values, 1 the upward ones
    auto step = [&](int k, int v) {
        if constexpr (NAM) {
            RtrStep<R> f{};
            const bool some = (clouds >> k) & 1;
            const R clfr = some ? (R)rcol.cfrac(nrl - 1 - k) : (R)0;
            const bool cloudy = clfr > (R)0;
            if (some) f = rtr_step<R>(a.rt, v ? FCLD1U : FCLD1D, v ? k + 2 : k, t, clfr, ((v ? lstu : lstd) >> k) & 1);
#pragma unroll
            for (int j = 0; j < GW; ++j) {
                const WR_G R *q = m.lw(gs + j, k, lane);
                const R tr = q[0], gas = q[v ? 192 : 64];
                if (some)
                    rtr_update<R>(f, cloudy, gas, q[v ? 256 : 128], tr, q[320], rad[0][j], cld[j], clr[j], cor[j]);
                else
                    rad[0][j] = rad[0][j] * tr + gas;
            }
        } else if constexpr (sizeof(R) == 4) {
#pragma unroll
            for (int j = 0; j < GW; ++j) {
                const WR_G R *q = m.lw(gs + j, k, lane);
                rad[0][j] = rad[0][j] * q[0] + q[v ? 128 : 64];
            }
        } else {
            if ((clouds >> k) & 1) {
                // a clear g-point: cloud transmittance 1 and cloud source 0, which leave the value as it is
                const R ef = *m.ef(B, k, lane);
                const uint32_t w1 = lrow<R>(a.rp, blk, k, rl).w(1);
                const uint32_t word = mword(a.rp.mlw, a.rp.row(blk, k), MROW_LW, B, rl);
                const uint32_t bits = (w1 & 256u) ? word >> sh.g0 : 0u;
#pragma unroll
                for (int j = 0; j < GW; ++j) {
                    const WR_G R *q = m.lw(gs + j, k, lane);
                    const R e = (bits >> j) & 1u ? ef : (R)1;
                    rad[0][j] = rad[0][j] * q[0] * e + q[v ? 192 : 64] + q[v ? 256 : 128];
                }
            } else {
#pragma unroll
                for (int j = 0; j < GW; ++j) {
                    const WR_G R *q = m.lw(gs + j, k, lane);
                    rad[0][j] = rad[0][j] * q[0] + q[v ? 192 : 64];
                }
            }
        }
    };
    sum.begin(nrl - 1, -1);
#pragma unroll 4
    for (int k = nrl - 1; k >= 0; --k) {
        step(k, 0);
        sum.put(rad, dn);
    }
    sum.finish(dn);
    sum.begin(0, 1);
#pragma unroll
    for (int j = 0; j < GW; ++j) {  // surface emission and reflection
        rad[0][j] = *m.sfc(gs + j, lane) + c.reflct * rad[0][j];
        cld[j] = clr[j] = cor[j] = (R)0;
    }
    sum.put(rad, up);
#pragma unroll 4
    for (int k = 0; k < nrl; ++k) {
        step(k, 1);
        sum.put(rad, up);
    }
    sum.finish(up);
}

// The slot of a sweep's g-points: FP32 in the place of the layer's R/T.  Reading the layers ahead of their use into
// registers gained nothing (FP32 within 2 %; in FP64 the registers cost more than it gave).
template <typename R, bool NAM, int GW> struct ManySlot {
    static constexpr int NV = sw_nv<R>();
    ManyBlk<R, NAM> m;
    int g0, lane;
    __device__ __forceinline__ WR_G R *at(int k, int sky, int g) const
    {
        return sizeof(R) == 4 ? m.sw(g0 + g, k, lane) + sky * 320 : m.refl(g0 + g, k, sky, lane);
    }
    __device__ __forceinline__ void put(int k, int sky, int g, const R (&x)[NV]) const
    {
        WR_G R *q = at(k, sky, g);
#pragma unroll
        for (int i = 0; i < NV; ++i)
            if (i < 4 || sky) q[64 * i] = x[i];  // the fifth, the direct transmission, is in place already in sky 0
    }
    __device__ __forceinline__ void get(int k, int sky, int g, R (&x)[NV]) const
    {
        const WR_G R *q = at(k, sky, g);
#pragma unroll
        for (int i = 0; i < NV; ++i) x[i] = q[64 * i];
    }
};

template <typename R, int B, bool NAM>
__device__ __forceinline__ void sweep_sw(const ManyArgs<R> &a, int b, int lane, const Share<R> &sh)
{
    constexpr int NG = SW_NG[B], NS = SW_NS[B], GW = MANY_GW;
    const int blk = a.blk0 + b, nday = *a.cs.nday, nrl = a.rp.nrl;
    if (blk * 64 >= nday) return;
    const bool ok = blk * 64 + lane < nday;
    const int rl = ok ? lane : nday - 1 - blk * 64, t = a.cs.dlist[blk * 64 + rl];
    SwCol<R> c;
    sw_col<R, B>(a.in, a.par, a.col0, a.cs, t, c);
    const ManyBlk<R, NAM> m = many_blk<R, NAM>(a, b);
    const AccT<R> acc = band_acc<R>(a.ba, 16 + B);
    const double cf1 = a.cs.zcf1[t], cf0 = a.cs.zcf0[t];
    const bool total = NAM && cf1 > EPS;
    if (!NAM && ok) acc.sw_clr0[t] = (R)0;  // clear-sky surface flux: NAM route only
    const bool two = NAM && __any(total);
    constexpr int NP = NAM ? 2 : 1;
    const uint64_t clouds = two ? many_cloud<true, R>(a.rp, blk, rl) : 0;  // layers whose total-sky R/T differ
    sw_adding<R, NG, GW, GW, NP>(
        nrl, c.asfc, two, ManySlot<R, NAM, GW>{m, NS + sh.g0, lane}, lane, sh, [](int k, int) { return k; },
        [&](int, int k, int, RtV<R, GW> (&o)[NP]) {
            auto one = [&](int sky) {
#pragma unroll
                for (int j = 0; j < GW; ++j) {
                    const WR_G R *q = m.sw(NS + sh.g0 + j, k, lane) + sky * 320;
                    RtV<R, GW> &r = o[sky];
                    r.rb[j] = q[0], r.rd[j] = q[64], r.tb[j] = q[128], r.td[j] = q[192], r.ld[j] = q[256];
                }
            };
            one(0);
            if constexpr (NAM) {
                if ((clouds >> k) & 1)
                    one(1);
                else
                    o[1] = o[0];
            }
        },
        [&](int g) { return c.ssolar * a.sflux[(size_t)(NS + sh.g0 + g) * a.n + t]; },
        [&](int lev, const R *f) {
            if constexpr (NAM) {
                swr_emit<R>(acc, ok, total, cf1, cf0, lev, a.n, t, f);
            } else if (ok) {
                acc.sw_up[(size_t)lev * a.n + t] = f[0];
                acc.sw_dn[(size_t)lev * a.n + t] = f[1];
            }
        });
}

template <typename R, bool NAM, int P>
__device__ __forceinline__ void sweep_run(const ManyArgs<R> &a, int pos, int b, int lane, const Share<R> &sh)
{
    if constexpr (P < 30) {
        constexpr int id = MANY_ORDER[P];
        if (pos != P) return sweep_run<R, NAM, P + 1>(a, pos, b, lane, sh);
        if constexpr (id < 16) {
            if (sh.wave < LW_NG[id] / MANY_GW) sweep_lw<R, id, NAM>(a, b, lane, sh);
        } else {
            if (sh.wave < SW_NG[id - 16] / MANY_GW) sweep_sw<R, id - 16, NAM>(a, b, lane, sh);
        }
    }
}
// grid: nblk blocks x 30 bands; waves beyond the band's g-points leave at once
template <typename R, bool NAM>
__global__ void __launch_bounds__(64 * MANY_W, 4) k_sweep(ManyArgs<R> a)
{
    __shared__ __attribute__((aligned(16))) R xs[sum_lds_bytes<R>() / sizeof(R)];
    const int w = wave_id();
    sweep_run<R, NAM, 0>(a, (int)blockIdx.y, (int)blockIdx.x, (int)(threadIdx.x & 63), Share<R>{xs, w * MANY_GW, w});
}

// The bands of a tile, as many 64-column blocks at once as the pool has room for.
template <typename R, bool NAM, bool SURR> int launch_many(const BandJob<R> &j, hipStream_t s)
{
    ManyArgs<R> a{j.tabs, j.sflux, j.in, j.par, j.col0, j.n, 0, 0, j.cs, j.rp, j.ba, j.sg, j.rt, j.c->pool[0]};
    const int nb = (j.n + 63) / 64, nrl = j.rp.nrl;
    const size_t room = j.c->pool_all / many_block_bytes<R, NAM>(nrl);
    const int per = (size_t)nb < room ? nb : (int)room;
    if (per < 1) return WR_ERR_NOMEM;
    tbeg(j.c, KID_MANY, s);
    for (a.blk0 = 0; a.blk0 < nb; a.blk0 += per) {
        a.nblk = nb - a.blk0 < per ? nb - a.blk0 : per;
        hipLaunchKernelGGL((k_lay<R, NAM, SURR>), dim3((unsigned)a.nblk, (unsigned)((nrl + MANY_LAYERS - 1) / MANY_LAYERS), 30),
                           dim3(64 * MANY_LAYERS), 0, s, a);
        hipLaunchKernelGGL((k_sweep<R, NAM>), dim3((unsigned)a.nblk, 30), dim3(64 * MANY_W), 0, s, a);
    }
    tend(j.c, s);
    return hipGetLastError() == hipSuccess ? WR_OK : WR_ERR_HIP;
}

}  // namespace wr
