"""Small tiles: all bands of a tile in two launches against the per-band launches.

WR_MANY_COLS=0 (read when a context is created) keeps the per-band kernels; both run the same column
functions, so every output is the same bits, at the edges of a 64-column block, for both precisions and
routes, with and without the optional column inputs."""
from pathlib import Path

import numpy as np
import pytest
import torch

from woof_nam_amd import abi, gen
from woof_nam_amd import surrogate as S
from woof_nam_amd.radiation import Radiation

pytestmark = pytest.mark.gpu


def columns(n, seed, ext, device):
    c = gen.columns(n, seed=seed)
    if ext:
        rng = np.random.default_rng(seed)
        dp = np.diff(c["p_lev"], axis=0) * (1000.0 / 9.80665)
        c["cwp"], c["cip"], c["crp"] = c["qc"] * dp, c["qi"] * dp, 0.1 * c["qc"] * dp
        c["rew"] = rng.uniform(5.0, 14.0, size=c["t_lay"].shape)
        c["rei"] = rng.uniform(20.0, 100.0, size=c["t_lay"].shape)
        c["o3_top"] = 0.5 * c["o3_lay"][0]
        for k, nb in abi.AER_BANDS.items():
            a = np.empty((3, nb, c["t_lay"].shape[0] + 1, n), dtype=np.float32)
            a[0], a[1], a[2] = rng.uniform(0.0, 0.02, size=a[0].shape), 0.9, 0.65
            c[k] = a
    return {k: torch.from_numpy(np.ascontiguousarray(v)).to(device) for k, v in c.items()}


@pytest.mark.parametrize("mcica,ext", [(1, False), (0, False), (1, True), (0, True)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_two_launches_equal_per_band_launches(gpu_device, monkeypatch, precision, mcica, ext):
    p = Radiation.default_params(mcica=mcica, seed=11)
    rads = []
    for env in ("0", None):
        monkeypatch.setenv("WR_MANY_COLS", env) if env else monkeypatch.delenv("WR_MANY_COLS")
        rads.append(Radiation(0, max_cols=700))
    try:
        for n in (1, 63, 64, 65, 701):              # 701: a full tile and a one-column tile
            print(f"case two launches {precision} mcica={mcica} ext={ext} ncol={n}", flush=True)
            cols = columns(n, 50 + n, ext, gpu_device)
            a, b = (r.run(cols, params=p, precision=precision)[0] for r in rads)
            torch.cuda.synchronize()
            for k in abi.OUTPUT_FIELDS:
                assert torch.equal(a[k].view(torch.int64), b[k].view(torch.int64)), (k, n)
    finally:
        for r in rads:
            r.close()


def test_surrogate_two_launches_equal_per_band_launches(gpu_device, monkeypatch):
    """The learned optics in both forms: columns inside the training envelope, every third one outside it (table
    optics), alone in a tile, at the edges of a block and in two tiles."""
    net = S.MLP.load(Path(S.__file__).resolve().parent / "data" / "surrogate_rrtmg.npz", gpu_device)
    rads = []
    for env in ("0", None):
        monkeypatch.setenv("WR_MANY_COLS", env) if env else monkeypatch.delenv("WR_MANY_COLS")
        rads.append(Radiation(0, max_cols=700))
        rads[-1].attach_surrogate(net)
    try:
        for n in (1, 63, 65, 701):
            print(f"case two launches surrogate ncol={n}", flush=True)
            cols = columns(n, 150 + n, False, gpu_device)
            cols["t_lay"][:, 2::3] = 345.0              # far outside the training temperatures
            (a, fa), (b, fb) = (r.run(cols, params=Radiation.default_params(seed=9), precision="surrogate") for r in rads)
            torch.cuda.synchronize()
            fa, fb = fa["fallback"], fb["fallback"]
            assert torch.equal(fa, fb) and bool((fa[2::3] == 1).all()) and (n == 1 or int(fa.sum()) < n)
            for k in abi.OUTPUT_FIELDS:
                assert torch.equal(a[k].view(torch.int64), b[k].view(torch.int64)), (k, n)
    finally:
        for r in rads:
            r.close()


@pytest.mark.parametrize("mcica", [1, 0])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_tiles_of_any_size_agree(gpu_device, monkeypatch, precision, mcica):
    """One set of columns in large and in smaller tiles: the band kernels over more blocks than their grid has
    waves (several rounds and a ragged last one), and the two launches over more blocks than the pool holds."""
    n, p = 140_001, Radiation.default_params(mcica=mcica, seed=5)
    cols = columns(n, 77, False, gpu_device)
    out = []
    for max_cols, env in ((n, "0"), (30_000, None), (9_000, "0")):
        monkeypatch.setenv("WR_MANY_COLS", env) if env else monkeypatch.delenv("WR_MANY_COLS")
        print(f"case tiles {precision} mcica={mcica} max_cols={max_cols} many={env}", flush=True)
        rad = Radiation(0, max_cols=max_cols)
        try:
            out.append(rad.run(cols, params=p, precision=precision)[0])
            torch.cuda.synchronize()
        finally:
            rad.close()
    for other in out[1:]:
        for k in abi.OUTPUT_FIELDS:
            assert torch.equal(out[0][k].view(torch.int64), other[k].view(torch.int64)), k


@pytest.mark.parametrize("mcica", [1, 0])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_small_pools_give_the_same_bits(gpu_device, monkeypatch, precision, mcica):
    """WR_POOL_GB: 4 x 0.03 GB hold one or a few blocks of the two launches at once; 4 x 0.01 GB hold none, and the
    band kernels then loop over the few slots that there are."""
    n, p = 705, Radiation.default_params(mcica=mcica, seed=3)
    cols = columns(n, 91, False, gpu_device)
    out = []
    for gb in (None, "0.03", "0.01"):
        monkeypatch.setenv("WR_POOL_GB", gb) if gb else monkeypatch.delenv("WR_POOL_GB", raising=False)
        print(f"case small pools {precision} mcica={mcica} gb={gb}", flush=True)
        rad = Radiation(0, max_cols=n)
        try:
            out.append(rad.run(cols, params=p, precision=precision)[0])
            torch.cuda.synchronize()
        finally:
            rad.close()
    for other in out[1:]:
        for k in abi.OUTPUT_FIELDS:
            assert torch.equal(out[0][k].view(torch.int64), other[k].view(torch.int64)), k
