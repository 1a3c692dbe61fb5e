// wr_many.h -- every band of a small tile in one launch.
//
// A tile of a few thousand columns gives each of the 30 band kernels only n / 64 waves, far fewer than
// the 1,024 SIMDs hold, and a wave's time is one column's serial chain over the layers.  Launched one
// after another on the four hardware queues of a process, the band kernels of such a tile take the sum of
// eight such chains.  Here one grid holds a 64-lane workgroup per (band, 64-column block), the
// longest bands first, so the whole tile takes about the longest chain (FP64, 257 columns of 60
// layers: 12.8 ms per call with the per-band launches).  The workgroups run the same column functions as
// the per-band kernels, from the band tables in global memory, so the results are the same bits.
#pragma once
#include "wr_launch.h"

namespace wr {

// band ids by falling duration of one wave (serialised FP64 and FP32 timings; the order matters little)
constexpr int MANY_ORDER[30] = {17, 29, 21, 20, 23, 4,  2,  3,  24, 8,  6,  19, 18, 27, 28,
                                16, 11, 1,  0,  25, 26, 12, 10, 7,  5,  9,  14, 15, 22, 13};

template <typename R, bool NAM> constexpr size_t many_slot(int id, int nk)  // pool bytes of one block of band id
{
    return id >= 16 ? cache_slot_bytes(sw_nv_mc<R>(), SW_NG[id - 16], nk, (int)sizeof(R))
                    : (sizeof(R) == 4 && !NAM ? cache_slot_bytes(LW_NV_F32, LW_NG[id], nk, 4) : 0);
}
template <typename R, bool NAM> constexpr size_t many_block_bytes(int nk)  // pool bytes of one block of every band
{
    size_t b = 0;
    for (int id = 0; id < 30; ++id) b += many_slot<R, NAM>(id, nk);
    return b;
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
    char *pool;  // nblk slots of the first band in MANY_ORDER, nblk of the second, ...
};

template <typename R, bool NAM, bool SURR, int P>
__device__ __forceinline__ void many_run(const ManyArgs<R> &a, int pos, int b, size_t before, Fix64 *fx)
{
    if constexpr (P < 30) {
        constexpr int id = MANY_ORDER[P];
        if (pos != P) {
            many_run<R, NAM, SURR, P + 1>(a, pos, b, before + many_slot<R, NAM>(id, 1), fx);
            return;
        }
        const int nk = a.in.nlay + 2;
        const AccT<R> acc = band_acc<R>(a.ba, id);
        WR_G char *slot = (WR_G char *)(a.pool + (before * a.nblk + many_slot<R, NAM>(id, 1) * b) * nk);
        const int blk = a.blk0 + b, lane = (int)threadIdx.x;
        if constexpr (id < 16) {
            if constexpr (NAM)
                lwr_column<R, id>(a.T, a.T->lw[id], a.in, a.par, a.col0, a.n, a.cs, a.rp, acc, a.rt, blk, lane);
            else if constexpr (sizeof(R) == 4)
                lw_column_f32c<id, SURR>(a.T, a.T->lw[id], a.in, a.par, a.col0, a.n, a.cs, a.rp, acc, a.sg, blk, lane, slot);
            else
                lw_column<R, id, SURR>(a.T, a.T->lw[id], a.in, a.par, a.col0, a.n, a.cs, a.rp, acc, a.sg, blk, lane);
        } else {
            constexpr int S = id - 16;
            if constexpr (NAM)
                swr_column<R, S>(a.T, a.T->sw[S], a.in, a.par, a.col0, a.n, a.cs, a.rp, a.sflux, acc, blk, lane, slot, fx);
            else
                sw_column<R, S, SURR>(a.T, a.T->sw[S], a.in, a.par, a.col0, a.n, a.cs, a.rp, a.sflux, acc, a.sg, blk, lane, slot, fx);
        }
    }
}

template <typename R, bool NAM, bool SURR>
__global__ void __launch_bounds__(64, sizeof(R) == 4 && !NAM ? 2 : 1) k_many(ManyArgs<R> a)
{
    __shared__ Fix64 fx[1];
    many_run<R, NAM, SURR, 0>(a, (int)(blockIdx.x / a.nblk), (int)(blockIdx.x % a.nblk), 0, fx);
}

// The bands of a tile, as many 64-column blocks at once as the pool has room for.
template <typename R, bool NAM, bool SURR> int launch_many(const BandJob<R> &j, hipStream_t s)
{
    ManyArgs<R> a{j.tabs, j.sflux, j.in, j.par, j.col0, j.n, 0, 0, j.cs, j.rp, j.ba, j.sg, j.rt, j.c->pool[0]};
    const int nb = (j.n + 63) / 64;
    const size_t room = j.c->pool_all / many_block_bytes<R, NAM>(j.in.nlay + 2);
    const int per = (size_t)nb < room ? nb : (int)room;
    if (per < 1) return WR_ERR_NOMEM;
    tbeg(j.c, KID_MANY, s);
    for (a.blk0 = 0; a.blk0 < nb; a.blk0 += per) {
        a.nblk = nb - a.blk0 < per ? nb - a.blk0 : per;
        hipLaunchKernelGGL((k_many<R, NAM, SURR>), dim3((unsigned)a.nblk * 30u), dim3(64), 0, s, a);
    }
    tend(j.c, s);
    return hipGetLastError() == hipSuccess ? WR_OK : WR_ERR_HIP;
}

}  // namespace wr
