"""When the prepared-tile path of the gated delta rule is taken (host rule, no GPU): its workspace is
nonzero exactly for bf16 128 x 128 heads, chunks dividing 32, at least ten tiles, at most 64
(sequence, head) pairs and a bounded tile step; a workspace that is too small is refused before any
launch, and one for a shape the path does not take is ignored."""

import pytest

from dllm_qwen38_amd import _lib

BF, F32 = _lib.DT_BF16, _lib.DT_F32
MB = 1 << 20


def _bytes(B=1, T=2048, Hk=16, Hv=48, Dk=128, Dv=128, chunk=32, dtype=BF, streams=2, states=0):
    return _lib.lib().dllm_gdn_scan_workspace_bytes(B, T, Hk, Hv, Dk, Dv, chunk, dtype, streams, states)


@pytest.mark.parametrize("kw", [
    {}, {"streams": 1}, {"states": 1}, {"T": 320}, {"T": 80, "chunk": 8}, {"T": 10, "chunk": 1}, {"Hv": 64}, {"Hk": 1, "Hv": 1},
    {"B": 3, "Hv": 16}, {"T": 32 * 1000},
])
def test_taken_and_bounded(kw):
    n = _bytes(**kw)
    assert 0 < n <= 96 * MB + 64 * 65536


@pytest.mark.parametrize("kw", [
    {"dtype": F32}, {"Dk": 64}, {"Dv": 64}, {"chunk": 64}, {"chunk": 24}, {"T": 288}, {"T": 72, "chunk": 8}, {"T": 2047},
    {"B": 2}, {"B": 4, "Hv": 16}, {"B": 3, "Hv": 16, "states": 1}, {"Hk": 5}, {"streams": 3}, {"B": 0}, {"T": 0}, {"chunk": 0},
])
def test_not_taken(kw):
    assert _bytes(**kw) == 0


def test_ranges_share_one_workspace():
    """A long sequence is walked in ranges of tiles: the workspace stays under its bound and gains the
    state carried between them."""
    per = 16 * 5 * 8192 + 48 * 2 * (3 * 2048 + 512)
    assert _bytes() == 64 * per
    assert _bytes(T=4096) == 64 * per + 48 * 128 * 128 * 4


def test_small_workspace_is_refused():
    L = _lib.lib()
    import ctypes

    st = (ctypes.c_int64 * 3)(320 * 10240, 10240, 128)
    sg = (ctypes.c_int64 * 3)(320 * 48, 48, 1)
    need = _bytes(T=320, streams=1)
    P = 4096
    for nbytes, ws in ((need - 1, P), (need, P + 16)):
        rc = L.dllm_gdn_chunk_ws_fwd(P, st, P, st, P, st, P, sg, P, sg, None, P, None, 1, 320, 16, 48, 128, 128, 32, BF, 1,
                                     0.1, ws, nbytes, None)
        assert rc == -1 and "workspace" in _lib.last_error()
