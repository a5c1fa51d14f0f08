"""The fp32 state fork by prepared tiles (csrc/gdn_scan_f32.hip): outputs, states and tails against the
oracle over head sizes, blocks (full, half, one-row tiles), grouped heads, one to several tiles and sequences,
states kept or not, and a sequence walked in ranges against one walked whole. The workspace holds NaN
before the direct calls: every operand read was written by the same call."""

import pytest
import torch

from dllm_qwen38_amd import _lib, gdn, inputs
from oracle import gdn_ref

pytestmark = pytest.mark.gpu

# fp32 sums of at most 128 terms with the oracle's own operands, as for the chunk kernel's fp32 results
F32_TOL = 1e-4


@pytest.mark.parametrize("B,L,block,Hk,Hv,D", [
    (1, 64, 32, 4, 4, 64),
    (2, 96, 32, 2, 6, 64),    # an odd number of tiles
    (1, 32, 32, 2, 2, 128),   # one tile
    (1, 160, 32, 2, 6, 128),
    (3, 48, 16, 1, 5, 128),   # half tiles, five heads on one key head
    (1, 56, 8, 2, 2, 64),
    (2, 5, 1, 1, 3, 128),     # one row per tile
])
@pytest.mark.parametrize("states", [True, False])
def test_fork_matches_oracle(dev, B, L, block, Hk, Hv, D, states):
    s = inputs.GdnShape("f32", B, L, block, Hk, Hv, D, 4, torch.float32, 1.0, 7700 + L)
    x = inputs.gdn_layer_inputs(s)
    o0, ot, st, tails = gdn_ref.state_fork_layer(x["raw0"], x["rawt"], x["conv_w"], x["beta0"], x["betat"], x["g0"],
                                                 x["gt"], Hk=Hk, Hv=Hv, Dk=D, Dv=D, block=block)
    r = gdn.gdn_state_fork(*(x[n].to(dev) for n in ("raw0", "rawt", "conv_w", "beta0", "betat", "g0", "gt")),
                           num_k_heads=Hk, num_v_heads=Hv, head_k_dim=D, head_v_dim=D, block=block, need_states=states)
    torch.cuda.synchronize()
    assert "prepared" in gdn.last_impl()[1]
    assert torch.equal(r["tails"].cpu(), tails)
    for name, ref in (("o0", o0), ("ot", ot), ("states", st)):
        if r[name] is None:
            assert not states
            continue
        assert (r[name].cpu() - ref).abs().max().item() <= F32_TOL, name


@pytest.mark.parametrize("states", [True, False])
def test_ranges_equal_one_walk(dev, states):
    """B = 3 sequences of 14 tiles pass the workspace's bound and are walked in ranges; each alone is one
    walk: the same bits."""
    B, L, block, Hk, Hv, D = 3, 448, 32, 16, 48, 128
    lib = _lib.lib()
    per = Hv * 2 * (9 * 4096 + 512) + Hk * 4 * 4096 + (0 if states else Hv * D * D * 4)
    n1 = lib.dllm_gdn_fork_f32_workspace_bytes(1, L, Hk, Hv, D, D, block, int(states))
    n3 = lib.dllm_gdn_fork_f32_workspace_bytes(B, L, Hk, Hv, D, D, block, int(states))
    assert n1 == per * 14 and 0 < n3 < 3 * n1
    g = torch.Generator().manual_seed(11)
    C = (2 * Hk + Hv) * D
    y0, yt = (torch.randn(B, L, C, generator=g).to(dev) for _ in range(2))
    b0, bt = (torch.sigmoid(torch.randn(B, L, Hv, generator=g)).to(dev) for _ in range(2))
    g0, gt = (-torch.nn.functional.softplus(torch.randn(B, L, Hv, generator=g)).to(dev) for _ in range(2))

    def run(sl, nbytes):
        t = [x[sl].contiguous() for x in (y0, yt, b0, bt, g0, gt)]
        n = t[0].shape[0]
        ws = torch.empty(nbytes, dtype=torch.uint8, device=dev).fill_(0xFF)
        o = [torch.full((n, L, Hv, D), float("nan"), device=dev) for _ in range(2)]
        st = torch.full((n, L // block, Hv, D, D), float("nan"), device=dev) if states else None
        _lib.check(lib.dllm_gdn_state_fork_ws_fwd(
            t[0].data_ptr(), t[1].data_ptr(), L * C, C, *(x.data_ptr() for x in t[2:]), o[0].data_ptr(), o[1].data_ptr(),
            _lib.ptr(st), n, L, Hk, Hv, D, D, block, _lib.DT_F32, D ** -0.5, ws.data_ptr(), nbytes,
            _lib.stream_handle(dev)), "fork")
        torch.cuda.synchronize()
        return o + ([st] if states else [])

    whole = run(slice(0, B), n3)
    for b in range(B):
        for x, y in zip(whole, run(slice(b, b + 1), n1)):
            assert torch.isfinite(y).all() and torch.equal(x[b:b + 1], y)
