// wr_rec.h -- layer records and McICA words of a tile, computed once and read by every band kernel.
//
// A band kernel's per-layer set-up (lwrad / swrad prep and setcoef: about 300 VALU operations in FP64
// with a dozen divisions, and two logs) is the same for all bands; so are the indices and weights of the
// Planck interpolation.  k_layers evaluates them once per layer and column, one thread each, and leaves
// them in rows of 64 columns: [block of 64 columns][layer][field][64], so that a wave reads a field as
// one contiguous run at a constant offset from a wave-uniform address (no per-lane address arithmetic)
// and loads only the fields its band uses.  The values are those the band kernels computed for
// themselves, rounded to the optics precision R, so the FP64 results stay the same bits.
// SW records hold day columns only, in day-list order.
//
// McICA sub-columns: one word per (band, layer, column), bit g set when g-point g of the band is
// cloudy there.  A lane evaluates only the 4-layer Philox blocks of its own column that hold cloud (the
// draws of a clear layer decide nothing: a cloud deck's first layer takes its own draw), and writes the
// words of those blocks; readers mask the words of clear layers away.
#pragma once
#include "wr_lw.h"
#include "wr_sw.h"

namespace wr {

struct ColScal {
    WR_G int *lw_laytrop, *lcf1, *day, *sw_laytrop, *dlist, *nday;
    WR_G uint32_t *cblk;  // 4-layer blocks (from the surface) that hold cloud
    WR_G double *pwv, *zcf1, *zcf0;
    // per tile column, written by k_layers: la[kin * n + t] = log of the layer pressure (layer kin,
    // top-first); tz[L * n + t] = LW level temperature, L = 0 the top layer's temperature, L = kin + 1
    // the interface below layer kin, L = nrl the skin temperature
    WR_G double *la, *tz;
};

// Fields of a row.  The last ones are for FP32 only: column amounts that follow from the dry column and the
// call's mixing ratios, which the FP64 kernels form themselves (the same two operations) instead of loading
// 8 bytes each; in FP32 they are roundings of FP64 products, so they are kept.
enum { LF_F00 = 0, LF_F01, LF_F10, LF_F11, LF_SF, LF_SFR, LF_FF, LF_FFR, LF_MF, LF_SCM, LF_SCN2, LF_CA0, LF_CA2, LF_DRY, LF_BRD,
       LF_P, LF_PL, LF_PB, LF_LIQ, LF_ICE, LF_N64, LF_CA1 = LF_N64, LF_CA3, LF_WX = LF_CA3 + 4, LF_N32 = LF_WX + 4 };
// SF_MOL: FP32 dry plus water vapour column, FP64 the dry column
enum { SF_F00 = 0, SF_F01, SF_F10, SF_F11, SF_SF, SF_SFR, SF_FF, SF_FFR, SF_CA0, SF_CA2, SF_MOL, SF_LIQ, SF_ICE, SF_N64,
       SF_CA1 = SF_N64, SF_CA3, SF_N32 = SF_CA3 + 3 };

// bytes of a row (one layer of one 64-column block): index words, then the fields
constexpr int lrow_size(int rbytes) { return 64 * (2 * 4 + (rbytes == 4 ? LF_N32 : LF_N64) * rbytes); }
constexpr int srow_size(int rbytes) { return 64 * (2 * 4 + (rbytes == 4 ? SF_N32 : SF_N64) * rbytes); }
template <typename R> constexpr int lrow_bytes() { return lrow_size((int)sizeof(R)); }
template <typename R> constexpr int srow_bytes() { return srow_size((int)sizeof(R)); }
constexpr int MROW_LW = 16 * 64 * 2, MROW_SW = 14 * 64 * 2;  // McICA words of a row
// bytes of a tile's records per 64-column block and layer, in the larger precision, and of its words
constexpr size_t rec_row_bytes(int rbytes) { return (size_t)lrow_size(rbytes) + srow_size(rbytes); }
constexpr size_t mrow_bytes() { return MROW_LW + MROW_SW; }

struct RecPtrs {
    WR_G char *lw, *sw, *mlw, *msw;  // [block][layer, surface first] rows
    int nrl;
    __device__ __forceinline__ size_t row(int blk, int k) const { return (size_t)blk * nrl + k; }
};
inline RecPtrs rec_ptrs(char *rec, char *words, int n, int nrl, int rbytes)
{
    RecPtrs r;
    const size_t rows = (size_t)((n + 63) / 64) * nrl;
    r.lw = gptr(rec);
    r.sw = r.lw + rows * lrow_size(rbytes);
    r.mlw = gptr(words);
    r.msw = r.mlw + rows * MROW_LW;
    r.nrl = nrl;
    return r;
}

// One LW record row as a lane of the block reads it.
template <typename R> struct LRow {
    const WR_G char *p;
    int lane;
    __device__ __forceinline__ uint32_t w(int i) const { return ((const WR_G uint32_t *)p)[i * 64 + lane]; }
    __device__ __forceinline__ R f(int i) const { return ((const WR_G R *)(p + 512))[i * 64 + lane]; }
};
template <typename R> __device__ __forceinline__ LRow<R> lrow(const RecPtrs &rp, int blk, int k, int lane)
{
    return {rp.lw + rp.row(blk, k) * lrow_bytes<R>(), lane};
}
template <typename R> __device__ __forceinline__ LRow<R> srow(const RecPtrs &rp, int blk, int k, int lane)
{
    return {rp.sw + rp.row(blk, k) * srow_bytes<R>(), lane};
}
// McICA word of band b (0-based) of a row
__device__ __forceinline__ uint32_t mword(const WR_G char *m, size_t row, int rowbytes, int b, int lane)
{
    return ((const WR_G uint16_t *)(m + row * rowbytes))[b * 64 + lane];
}

// index word 0: jp | (jt - 1) << 6 | (jt1 - 1) << 8 | inds << 10 | indf << 14 | indm << 16 | lower << 21 |
// planck index of the layer << 22 (0..179); word 1 (LW): planck index of the level below | cloudy << 8;
// word 1 (SW): cloudy
template <typename R> __device__ __forceinline__ uint32_t lw_word0(const LwLay<R> &L, int ipl)
{
    return (uint32_t)L.jp | (uint32_t)(L.jt - 1) << 6 | (uint32_t)(L.jt1 - 1) << 8 | (uint32_t)L.indself << 10 |
           (uint32_t)L.indfor << 14 | (uint32_t)L.indminor << 16 | (uint32_t)L.lower << 21 | (uint32_t)ipl << 22;
}
// planck()'s table index (0-based lower entry) and weight of a temperature
template <typename R> __device__ __forceinline__ int planck_at(double t, R &fr)
{
    fr = (R)(t - (double)((int)t));
    return imin(180, imax(1, (int)(t - 159.0))) - 1;
}
template <typename R>
__device__ __forceinline__ R planck_of(const Tabs<R> *__restrict__ T, int b, int i, R fr)
{
    const WR_G R *tp = T->totplnk + b * 181;
    return T->delwave[b] * (tp[i] + fr * (tp[i + 1] - tp[i]));
}

// the layer quantities the band optics use, from a record row (unused fields are never loaded)
template <typename R>
__device__ __forceinline__ void lrow_get(const LRow<R> &r, uint32_t w, const RunPar &par, LwLay<R> &L)
{
    L.jp = w & 63, L.jt = ((w >> 6) & 3) + 1, L.jt1 = ((w >> 8) & 3) + 1, L.indself = (w >> 10) & 15;
    L.indfor = (w >> 14) & 3, L.indminor = (w >> 16) & 31, L.lower = (w >> 21) & 1;
    L.fac00 = r.f(LF_F00), L.fac01 = r.f(LF_F01), L.fac10 = r.f(LF_F10), L.fac11 = r.f(LF_F11);
    L.selffac = r.f(LF_SF), L.selffrac = r.f(LF_SFR), L.forfac = r.f(LF_FF), L.forfrac = r.f(LF_FFR);
    L.minorfrac = r.f(LF_MF), L.scaleminor = r.f(LF_SCM), L.scaleminorn2 = r.f(LF_SCN2);
    L.coldry = r.f(LF_DRY), L.colbrd = r.f(LF_BRD), L.pavel = r.f(LF_P);
    L.colamt[0] = r.f(LF_CA0), L.colamt[2] = r.f(LF_CA2);
    if constexpr (sizeof(R) == 4) {
        L.colamt[1] = r.f(LF_CA1);
#pragma unroll
        for (int m = 3; m < 7; ++m) L.colamt[m] = r.f(LF_CA3 + m - 3);
#pragma unroll
        for (int m = 0; m < 4; ++m) L.wx[m] = r.f(LF_WX + m);
    } else {  // lw_layer's operations on the same dry column
        const double floor = 1.0e-12 * L.coldry;
        L.colamt[1] = fmax(floor, L.coldry * par.vmr[0]);
        L.colamt[3] = fmax(floor, L.coldry * par.vmr[1]), L.colamt[4] = fmax(floor, L.coldry * par.vmr[2]);
        L.colamt[5] = fmax(0.0, L.coldry * par.vmr[3]), L.colamt[6] = fmax(0.0, L.coldry * par.vmr[4]);
        L.wx[0] = fmax(0.0, L.coldry * par.vmr[8]), L.wx[1] = fmax(0.0, L.coldry * par.vmr[5]);
        L.wx[2] = fmax(0.0, L.coldry * par.vmr[6]), L.wx[3] = fmax(0.0, L.coldry * par.vmr[7]);
    }
}
template <typename R>
__device__ __forceinline__ void srow_get(const LRow<R> &r, uint32_t w, const RunPar &par, SwLay<R> &L)
{
    L.jp = w & 63, L.jt = ((w >> 6) & 3) + 1, L.jt1 = ((w >> 8) & 3) + 1, L.indself = (w >> 10) & 15;
    L.indfor = (w >> 14) & 3;
    L.fac00 = r.f(SF_F00), L.fac01 = r.f(SF_F01), L.fac10 = r.f(SF_F10), L.fac11 = r.f(SF_F11);
    L.selffac = r.f(SF_SF), L.selffrac = r.f(SF_SFR), L.forfac = r.f(SF_FF), L.forfrac = r.f(SF_FFR);
    L.colamt[0] = r.f(SF_CA0), L.colamt[2] = r.f(SF_CA2);
    if constexpr (sizeof(R) == 4) {
        L.colmol = r.f(SF_MOL);
        L.colamt[1] = r.f(SF_CA1);
#pragma unroll
        for (int m = 3; m < 6; ++m) L.colamt[m] = r.f(SF_CA3 + m - 3);
    } else {  // sw_layer's operations on the same dry column
        const double cd = r.f(SF_MOL), floor = 1.0e-12 * cd;
        L.colmol = cd + L.colamt[0];
        L.colamt[1] = fmax(floor, cd * par.vmr[0]);
        L.colamt[3] = fmax(floor, cd * par.vmr[1]), L.colamt[4] = fmax(floor, cd * par.vmr[2]);
        L.colamt[5] = fmax(floor, cd * par.vmr[3]);
    }
}

// ---- LW records, layer logs and level temperatures: one thread per (column, layer) ----------------
// Bound by the stores (124 bytes per layer and column in FP32, 168 in FP64).
template <typename R>
__global__ void __launch_bounds__(256) k_layers(const Tabs<R> *__restrict__ T, ColIn in, RunPar par, int col0, int n,
                                                ColScal cs, RecPtrs rp)
{
#pragma clang fp contract(off)
    const int lane = threadIdx.x, blk = blockIdx.x, kin = blockIdx.y * 4 + threadIdx.y;
    const int t = blk * 64 + lane, nrl = rp.nrl, k = nrl - 1 - kin;
    if (kin >= nrl || t >= valid_cols(in, col0, n)) return;
    const RadCol rc{in, col0 + t, nrl};
    const LayV v = rc.lay(kin);
    const double la = log_d(v.pl);
    cs.la[(size_t)kin * n + t] = la;
    double tb;  // temperature of the level below the layer
    if (kin + 1 < nrl)
        tb = tlvl_v(rc.tlyr(kin + 1), v.t, log_d(v.pb), log_d(rc.plyr(kin + 1)), la);
    else
        tb = rc.tskn();
    cs.tz[(size_t)(kin + 1) * n + t] = tb;
    if (kin == 0) cs.tz[t] = v.t;
    LwLay<R> L;
    lw_layer<R>(T, v, par, la, L);
    R fl, fb;
    const int il = planck_at<R>(L.tavel, fl), ib = planck_at<R>(tb, fb);
    WR_G char *row = rp.lw + rp.row(blk, k) * lrow_bytes<R>();
    WR_G uint32_t *w = (WR_G uint32_t *)row;
    w[lane] = lw_word0<R>(L, il);
    w[64 + lane] = (uint32_t)ib | (L.ct > 0.0 ? 256u : 0u);
    WR_G R *f = (WR_G R *)(row + 512) + lane;
    auto put = [&](int i, R x) { f[i * 64] = x; };
    put(LF_F00, L.fac00), put(LF_F01, L.fac01), put(LF_F10, L.fac10), put(LF_F11, L.fac11);
    put(LF_SF, L.selffac), put(LF_SFR, L.selffrac), put(LF_FF, L.forfac), put(LF_FFR, L.forfrac);
    put(LF_MF, L.minorfrac), put(LF_SCM, L.scaleminor), put(LF_SCN2, L.scaleminorn2);
    put(LF_CA0, L.colamt[0]), put(LF_CA2, L.colamt[2]);
    if constexpr (sizeof(R) == 4) {
        put(LF_CA1, L.colamt[1]);
#pragma unroll
        for (int m = 3; m < 7; ++m) put(LF_CA3 + m - 3, L.colamt[m]);
#pragma unroll
        for (int m = 0; m < 4; ++m) put(LF_WX + m, L.wx[m]);
    }
    put(LF_DRY, L.coldry), put(LF_BRD, L.colbrd), put(LF_P, L.pavel), put(LF_PL, fl), put(LF_PB, fb);
    put(LF_LIQ, (R)L.clwp), put(LF_ICE, (R)L.ciwp);
}

// ---- SW records of the day columns: one thread per (day-list entry, layer) -------------------------
template <typename R>
__global__ void __launch_bounds__(256) k_layers_sw(const Tabs<R> *__restrict__ T, ColIn in, RunPar par, int col0, int n,
                                                   ColScal cs, RecPtrs rp)
{
    const int lane = threadIdx.x, blk = blockIdx.x, kin = blockIdx.y * 4 + threadIdx.y;
    const int tt = blk * 64 + lane, nrl = rp.nrl, k = nrl - 1 - kin;
    if (kin >= nrl || tt >= *cs.nday) return;
    const int t = cs.dlist[tt];
    const RadCol rc{in, col0 + t, nrl};
    SwLay<R> L;
    sw_layer<R>(T, rc, par, kin, cs.la[(size_t)kin * n + t], L);
    WR_G char *row = rp.sw + rp.row(blk, k) * srow_bytes<R>();
    WR_G uint32_t *w = (WR_G uint32_t *)row;
    w[lane] = (uint32_t)L.jp | (uint32_t)(L.jt - 1) << 6 | (uint32_t)(L.jt1 - 1) << 8 | (uint32_t)L.indself << 10 |
              (uint32_t)L.indfor << 14;
    w[64 + lane] = L.ct > FTINY ? 1u : 0u;
    WR_G R *f = (WR_G R *)(row + 512) + lane;
    auto put = [&](int i, R x) { f[i * 64] = x; };
    put(SF_F00, L.fac00), put(SF_F01, L.fac01), put(SF_F10, L.fac10), put(SF_F11, L.fac11);
    put(SF_SF, L.selffac), put(SF_SFR, L.selffrac), put(SF_FF, L.forfac), put(SF_FFR, L.forfrac);
    put(SF_CA0, L.colamt[0]), put(SF_CA2, L.colamt[2]);
    if constexpr (sizeof(R) == 4) {
        put(SF_CA1, L.colamt[1]);
#pragma unroll
        for (int m = 3; m < 6; ++m) put(SF_CA3 + m - 3, L.colamt[m]);
    }
    put(SF_MOL, sizeof(R) == 4 ? L.colmol : L.coldry), put(SF_LIQ, (R)L.cwp), put(SF_ICE, (R)L.cip);
}

// ---- McICA words: one thread per (column or day-list entry, band) ----------------------------------
// The same draws and rule as mcica_g.  Bound by the Philox multiplies of the cloudy blocks.
template <int NG>
__device__ __forceinline__ void mcica_words(const RadCol &rc, uint32_t blocks, uint64_t col, uint64_t seed, int kind, int g0, int iovr,
                                            WR_G char *m, size_t row0, int rowbytes, int b, int lane)
{
    const int nrl = rc.nrl;
    double prev[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) prev[g] = 0.0;
    while (blocks) {
        const int kb = __builtin_ctz(blocks);
        blocks &= blocks - 1;
        double cf[5];  // the layer below the block, then its layers
#pragma unroll
        for (int q = 0; q < 5; ++q) {
            const int k = kb * 4 + q - 1;
            cf[q] = (k >= 0 && k < nrl) ? rc.cfrac(nrl - 1 - k) : 0.0;
        }
        uint32_t word[4] = {0, 0, 0, 0};
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            uint32_t u[4];
            philox4x32_10((uint32_t)col, (uint32_t)(col >> 32), (uint32_t)(g0 + g) | ((uint32_t)kind << 16),
                          iovr == 2 ? 0u : (uint32_t)kb, (uint32_t)seed, (uint32_t)(seed >> 32), u);
            double pv = prev[g];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const double r = (double)u[iovr == 2 ? 0 : q] * 0x1p-32;
                double cd = r;
                if (iovr == 1) {
                    const double tem1 = 1.0 - cf[q];
                    cd = (kb == 0 && q == 0) ? r : (pv > tem1 ? pv : r * tem1);
                    pv = cd;
                }
                if (cd >= 1.0 - cf[q + 1]) word[q] |= 1u << g;
            }
            prev[g] = pv;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (kb * 4 + q < nrl)
                ((WR_G uint16_t *)(m + (row0 + kb * 4 + q) * rowbytes))[b * 64 + lane] = (uint16_t)word[q];
    }
}
template <int B>
__device__ __forceinline__ void mcica_band(int b, const RadCol &rc, uint32_t blocks, uint64_t col, uint64_t seed, int iovr, const RecPtrs &rp,
                                           size_t row0, int lane)
{
    if constexpr (B < 30) {
        if (b != B) return mcica_band<B + 1>(b, rc, blocks, col, seed, iovr, rp, row0, lane);
        if constexpr (B < 16)
            mcica_words<LW_NG[B]>(rc, blocks, col, seed, 0, LW_NS[B], iovr, rp.mlw, row0, MROW_LW, B, lane);
        else
            mcica_words<SW_NG[B - 16]>(rc, blocks, col, seed, 1, SW_NS[B - 16], iovr, rp.msw, row0, MROW_SW, B - 16, lane);
    }
}
static __global__ void __launch_bounds__(64) k_mcica(ColIn in, RunPar par, int col0, int n, ColScal cs,
                                                     RecPtrs rp)
{
    const int lane = threadIdx.x, blk = blockIdx.x, b = blockIdx.y;
    int t = blk * 64 + lane;
    if (t >= (b < 16 ? valid_cols(in, col0, n) : *cs.nday)) return;
    if (b >= 16) t = cs.dlist[t];
    const RadCol rc{in, col0 + t, rp.nrl};
    const uint64_t col = in.col_id ? in.col_id[col0 + t] : (uint64_t)(col0 + t);
    const uint64_t seed = in.seed_dev ? *in.seed_dev : par.seed;
    mcica_band<0>(b, rc, cs.cblk[t], col, seed, par.iovr, rp, rp.row(blk, 0), lane);
}

}  // namespace wr
