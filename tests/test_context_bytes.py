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
