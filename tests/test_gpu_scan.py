"""The prepared-tile path of the gated delta rule (csrc/gdn_scan.hip) against the pipelined kernel: the
same bits, for one and two streams, every block size, initial states, kept states or none, tile counts
around the least that takes the path, sequences walked in ranges, and head counts that leave XCDs
uneven. The workspace holds NaN before each call: every operand read was written by the same call."""

import pytest
import torch

from dllm_qwen38_amd import _lib, gdn

pytestmark = pytest.mark.gpu


def _gates(g, *shape):
    beta = torch.sigmoid(torch.randn(shape, generator=g))
    return beta.cuda(), (-torch.nn.functional.softplus(torch.randn(shape, generator=g) - 3.0)).cuda()


def _ws(n, poison=True):
    w = torch.empty(n, dtype=torch.uint8, device="cuda")
    return w.fill_(0xFF) if poison else w


def _same(a, b, what):
    for k in a:
        if a[k] is None:
            assert b[k] is None
            continue
        assert torch.isfinite(b[k].float()).all(), (what, k)
        assert torch.equal(a[k], b[k]), (what, k)


@pytest.mark.parametrize("B,T,chunk,Hk,Hv,init,states,l2norm", [
    (1, 320, 32, 16, 48, True, True, 1),    # ten tiles: the least
    (1, 352, 32, 2, 6, False, True, 0),     # no l2norm, eleven tiles
    (3, 176, 16, 1, 5, True, False, 1),     # five heads on one key head: two rounds of the prep waves
    (1, 88, 8, 4, 4, True, True, 1),        # quarter tiles
    (2, 13, 1, 2, 2, False, True, 1),       # one row per tile
    (1, 6400, 32, 16, 48, True, True, 1),   # two ranges, the second from the snapshot before it
    (1, 6400, 32, 16, 48, False, False, 1),  # two ranges, the state carried in the workspace
])
def test_rule_is_bit_identical(dev, B, T, chunk, Hk, Hv, init, states, l2norm):
    g = torch.Generator().manual_seed(T + chunk + Hv)
    C = 2 * Hk * 128 + Hv * 128
    x = torch.randn(B, T, C, generator=g).to(torch.bfloat16).cuda()
    q, k, v = (t.unflatten(-1, (-1, 128)) for t in (x[..., :Hk * 128], x[..., Hk * 128:2 * Hk * 128], x[..., 2 * Hk * 128:]))
    if not l2norm:
        k.mul_(0.05)
    beta, gg = _gates(g, B, T, Hv)
    s0 = torch.randn(B, Hv, 128, 128, generator=g).cuda() * 0.1 if init else None
    L = _lib.lib()
    n = L.dllm_gdn_scan_workspace_bytes(B, T, Hk, Hv, 128, 128, chunk, _lib.DT_BF16, 1, int(states))
    assert n > 0
    got = []
    for ws in (None, _ws(n)):
        out = torch.full((B, T, Hv, 128), float("nan"), dtype=torch.bfloat16, device=dev)
        st = torch.full((B, T // chunk, Hv, 128, 128), float("nan"), device=dev) if states else None
        _lib.check(L.dllm_gdn_chunk_ws_fwd(
            q.data_ptr(), _lib.strides3(q), k.data_ptr(), _lib.strides3(k), v.data_ptr(), _lib.strides3(v), gg.data_ptr(),
            _lib.strides3(gg), beta.data_ptr(), _lib.strides3(beta), _lib.ptr(s0), out.data_ptr(), _lib.ptr(st), B, T, Hk,
            Hv, 128, 128, chunk, _lib.DT_BF16, l2norm, 128 ** -0.5, _lib.ptr(ws), n, _lib.stream_handle(dev)), "rule")
        torch.cuda.synchronize()
        got.append({"out": out, "states": st})
    _same(got[0], got[1], f"rule T={T} chunk={chunk}")


@pytest.mark.parametrize("B,L,block,Hk,Hv,states", [
    (1, 320, 32, 16, 48, True),
    (1, 416, 32, 1, 7, False),
    (2, 192, 16, 4, 8, True),
    (1, 96, 8, 2, 2, False),
    (2, 22, 2, 1, 3, True),
    (1, 4128, 32, 16, 48, False),  # two ranges, the state carried
    (1, 4128, 32, 16, 48, True),
])
def test_fork_is_bit_identical(dev, B, L, block, Hk, Hv, states):
    g = torch.Generator().manual_seed(L + block + Hv)
    C = 2 * Hk * 128 + Hv * 128
    y0, yt = (torch.randn(B, L, C, generator=g).to(torch.bfloat16).cuda() for _ in range(2))
    (b0, g0), (bt, gt) = _gates(g, B, L, Hv), _gates(g, B, L, Hv)
    lib = _lib.lib()
    n = lib.dllm_gdn_scan_workspace_bytes(B, L, Hk, Hv, 128, 128, block, _lib.DT_BF16, 2, int(states))
    assert n > 0
    got = []
    for ws in (None, _ws(n)):
        o0, ot = (torch.full((B, L, Hv, 128), float("nan"), dtype=torch.bfloat16, device=dev) for _ in range(2))
        st = torch.full((B, L // block, Hv, 128, 128), float("nan"), device=dev) if states else None
        _lib.check(lib.dllm_gdn_state_fork_ws_fwd(
            y0.data_ptr(), yt.data_ptr(), L * C, C, b0.data_ptr(), bt.data_ptr(), g0.data_ptr(), gt.data_ptr(),
            o0.data_ptr(), ot.data_ptr(), _lib.ptr(st), B, L, Hk, Hv, 128, 128, block, _lib.DT_BF16, 128 ** -0.5,
            _lib.ptr(ws), n, _lib.stream_handle(dev)), "fork")
        torch.cuda.synchronize()
        got.append({"o0": o0, "ot": ot, "states": st})
    _same(got[0], got[1], f"fork L={L} block={block}")


def test_two_streams_do_not_share_a_workspace(dev):
    """Calls on two streams at once, each with the workspace its stream's allocator gave it."""
    g = torch.Generator().manual_seed(3)
    B, T, Hk, Hv = 1, 640, 4, 8
    xs = [torch.randn(B, T, (2 * Hk + Hv) * 128, generator=g).to(torch.bfloat16).cuda() for _ in range(2)]
    ga = [_gates(g, B, T, Hv) for _ in range(2)]

    def run(i):
        q, k, v = (t.unflatten(-1, (-1, 128)) for t in
                   (xs[i][..., :Hk * 128], xs[i][..., Hk * 128:2 * Hk * 128], xs[i][..., 2 * Hk * 128:]))
        return gdn.chunk_gated_delta_rule_with_states(q, k, v, ga[i][1], ga[i][0], 32)

    ref = [run(i) for i in range(2)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    for _ in range(3):
        got = []
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                got.append(run(i))
        torch.cuda.synchronize()
        for (o, st), (ro, rst) in zip(got, ref):
            assert torch.equal(o, ro) and torch.equal(st, rst)
