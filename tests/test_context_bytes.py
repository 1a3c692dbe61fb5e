"""Device bytes of a context (wr_context_bytes, what wr_create allocates), computed on the host."""
import pytest

from woof_nam_amd import _lib


@pytest.fixture
def context_bytes(monkeypatch):
    """wr_context_bytes under the given settings; every other WR_* setting that it reads unset."""
    L = _lib.load()

    def get(max_cols, **env):
        for k in ("WR_POOL_GB", "WR_BAND_STREAMS", "WR_MANY_COLS", "WR_LW_GLANE"):
            monkeypatch.setenv(k, str(env[k])) if k in env else monkeypatch.delenv(k, raising=False)
        return L.wr_context_bytes(max_cols)
    return get


@pytest.mark.parametrize("gb", [0.3, 2.01, 2.03, 2.999999999])
def test_stream_pools_start_on_aligned_addresses(context_bytes, gb):
    """The four streams' pools lie one after another and hold 16-byte vectors, so each must take a multiple of 256
    bytes whatever WR_POOL_GB says: the difference to a limit that is such a multiple (2.048 GB) is one of 4 x 256.
    WR_MANY_COLS=0: the pools are the streams' alone."""
    whole = context_bytes(262144, WR_POOL_GB=2.048, WR_MANY_COLS=0)
    assert (whole - context_bytes(262144, WR_POOL_GB=gb, WR_MANY_COLS=0)) % 1024 == 0


def test_small_contexts_stay_small(context_bytes):
    """Column work space of at most 70 KB a column, 10 MB of tables and the pools: 2 GB for the two-launch form, or
    what four band kernels' slots take (2.0 MB per 64-column block each), or one block of the two-launch form."""
    for m in (1, 64, 257, 1000, 4096, 8192, 16384, 40_000, 65_536):
        blocks = (m + 63) // 64
        assert context_bytes(m) <= 10e6 + 70e3 * 64 * blocks + min(80e6 * blocks, max(2e9, 4 * 2.0e6 * blocks)), m
    assert context_bytes(4096) < 2.5e9


@pytest.mark.parametrize("m", [1000, 4096, 32_768, 65_536, 65_537, 262_144])
@pytest.mark.parametrize("gb", [0.05, 0.5, 3.0])
def test_pool_limit_bounds_every_pool(context_bytes, gb, m):
    """WR_POOL_GB limits the pools of the four streams, and with them the two-launch form that uses their space."""
    assert context_bytes(m, WR_POOL_GB=gb) <= 10e6 + 70e3 * (m + 63) + 4 * gb * 1e9


def test_context_bytes_grow_with_the_tile(context_bytes):
    """Callers bisect on them; past WR_MANY_COLS each band stream has its own pool."""
    for env in ({}, {"WR_MANY_COLS": 0}, {"WR_POOL_GB": 0.5}, {"WR_BAND_STREAMS": 0}):
        b = [context_bytes(m, **env) for m in (1, 64, 65, 1000, 4096, 20_000, 65_535, 65_536, 65_537, 131_072, 800_000)]
        assert b == sorted(b), env
