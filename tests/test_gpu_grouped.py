"""Grouped (prefill / batched) expert FFN on the GPU.

The grouped kernels and the per-pair GEMV kernels are built to compute every
(token, expert) row with the same MFMA slices, scale order and combine order,
so their outputs must be bit-identical; both are also checked against the
oracle's W8A8 restatement within the reference's own tolerance, max rel err
<= 2e-2 (bin/test_cache.py:51).  On the devtest input below one intermediate
activation sits on an e4m3 rounding boundary: fp32-level (2e-7) noise in the
oracle's own block sums moves its output by 1.17e-2 in 3 of 20 draws, and
the kernels land on the other side of that boundary."""
import numpy as np
import pytest
import torch

from conftest import say
from oracle import moe as omoe

pytestmark = pytest.mark.gpu
TOL = 2e-2


def _experts(seed, E, H, I, dev, recipe="blockq"):
    import synth
    w13 = torch.empty((E, 2 * I, H), dtype=torch.uint8)
    s13 = torch.empty((E, 2 * I // 128, H // 128), dtype=torch.float32)
    w2 = torch.empty((E, H, I), dtype=torch.uint8)
    s2 = torch.empty((E, H // 128, I // 128), dtype=torch.float32)
    for e in range(E):
        a, b, c, d = synth.expert_tensors(seed, 0, e, H, I, recipe)
        w13[e], s13[e], w2[e], s2[e] = a, b, c, d
    host = (w13, s13, w2, s2)
    return host, tuple(t.to(dev) for t in host)


def _fwd(x, ids, w, devt, mode, residual=None):
    import hipfetch
    lib = hipfetch.require()
    w13, s13, w2, s2 = devt
    T, H = x.shape
    out = torch.empty_like(x)
    ws = torch.empty(lib.fp8_moe_workspace(T, ids.shape[1], w13.shape[0], H, w2.shape[2]),
                     dtype=torch.uint8, device=x.device)
    lib.fp8_moe_forward(x, ids, w, w13.view(torch.float8_e4m3fn), s13,
                        w2.view(torch.float8_e4m3fn), s2, out, ws, mode=mode, residual=residual)
    return out


def _routing(T, E, K, seed, dev):
    rng = np.random.default_rng(seed)
    ids = torch.tensor(np.stack([rng.choice(E, K, replace=False) for _ in range(T)]), device=dev)
    w = torch.rand((T, K), generator=torch.Generator().manual_seed(seed)).to(dev)
    return ids, w / w.sum(-1, keepdim=True)


@pytest.mark.parametrize("T,E", [(3, 16), (16, 64), (64, 256), (512, 256)])
def test_grouped_equals_gemv(lib, dev, T, E):
    import synth
    H, I, K = 2048, 512, 8
    _, devt = _experts(T, E, H, I, dev)
    x = synth.hidden_states(T, T).to(dev)
    ids, w = _routing(T, E, K, T, dev)
    say(f"grouped: T={T} E={E}")
    a = _fwd(x, ids, w, devt, mode=1)
    b = _fwd(x, ids, w, devt, mode=2)
    torch.cuda.synchronize()
    if not torch.equal(a, b):
        d = (a.float() - b.float()).abs()
        pytest.fail(f"grouped != GEMV: {int((d > 0).sum())} elements differ, max {float(d.max())}")


def test_grouped_matches_oracle(lib, dev):
    import synth
    T, E, H, I, K = 6, 12, 2048, 512, 8
    host, devt = _experts(21, E, H, I, dev, recipe="devtest")
    x = synth.hidden_states(21, T).to(dev)
    ids, w = _routing(T, E, K, 21, dev)
    got = _fwd(x, ids, w, devt, mode=2)
    torch.cuda.synchronize()
    want = omoe.forward_w8a8(x.float().cpu().numpy(), ids.cpu().numpy(),
                             w.cpu().numpy().astype(np.float64), *(t.numpy() for t in host))
    err = omoe.max_rel_err(got.float().cpu().numpy(), want)
    print(f"grouped max rel err vs W8A8 oracle {err:.2e}")
    assert err <= TOL


def test_grouped_reference_prefill_ids(lib, dev, traces):
    """The reference's recorded prefill routing (55 tokens x 8 of 256, layer 0)."""
    import synth
    rows = traces["trace_prefill_rows"]
    ids = torch.from_numpy(traces["trace_prefill_ids"][:rows[0]].astype(np.int64)).to(dev)
    T = ids.shape[0]
    _, devt = _experts(5, 256, 2048, 512, dev)
    x = synth.hidden_states(5, T).to(dev)
    w = torch.full((T, 8), 0.125, device=dev)
    a = _fwd(x, ids, w, devt, mode=1)
    b = _fwd(x, ids, w, devt, mode=2)
    torch.cuda.synchronize()
    assert torch.equal(a, b)


def test_grouped_residual_and_bad_ids(lib, dev):
    import synth
    T, E, H, I, K = 9, 16, 256, 128, 4
    _, devt = _experts(8, E, H, I, dev)
    x = synth.hidden_states(8, T, H).to(dev)
    ids, w = _routing(T, E, K, 8, dev)
    res = synth.hidden_states(9, T, H).to(dev)
    plain = _fwd(x, ids, w, devt, mode=2)
    fused = _fwd(x, ids, w, devt, mode=2, residual=res)
    bad = ids.clone()
    bad[4, 2] = E + 3
    nanrow = _fwd(x, bad, w, devt, mode=2)
    torch.cuda.synchronize()
    assert torch.equal(fused, res + plain)
    assert torch.isnan(nanrow[4].float()).all()
    assert torch.equal(torch.cat([nanrow[:4], nanrow[5:]]), torch.cat([plain[:4], plain[5:]]))


@pytest.mark.parametrize("H,I", [(2048, 512), (4096, 384), (2560, 256), (1024, 1024)])
@pytest.mark.parametrize("mode", [1, 2])
def test_grouped_packed_record_views(lib, dev, mode, H, I):
    """Tile-ordered packed records against the same experts as dense
    row-major buffers: bit for bit, on the GEMV and the grouped path, at
    several hidden / intermediate sizes (K-block counts 2 to 32)."""
    import hostpool
    import synth
    T, E = 33 if mode == 2 else 5, 24
    lay = hostpool.RecordLayout(H, I)
    host, devt = _experts(31, E, lay.hidden, lay.inter, dev)
    rec = lay.pack(devt[0].view(torch.float8_e4m3fn), devt[1], devt[2].view(torch.float8_e4m3fn),
                   devt[3])
    v13, vs13, v2, vs2 = lay.views(rec)
    x = synth.hidden_states(31, T, H).to(dev)
    ids, w = _routing(T, E, 8, 31, dev)
    from fp8_moe import fp8_moe_forward
    say(f"packed record views: tile order, mode {mode}, H {H} I {I}")
    a = fp8_moe_forward(x, ids, w, v13, vs13, v2, vs2, mode=mode, layout=lay.code)
    b = _fwd(x, ids, w, devt, mode=mode)
    torch.cuda.synchronize()
    assert torch.equal(a, b)


@pytest.mark.parametrize("H,I,T,E,K", [(4096, 384, 40, 8, 4), (2560, 256, 70, 6, 3),
                                       (4096, 512, 512, 64, 8)])
def test_grouped_long_rows_equal_gemv(lib, dev, H, I, T, E, K):
    """Hidden sizes above 2048 (gate/up activations staged 16 K-blocks at a
    time: 2 stages at 4096, 16 + 4 blocks at 2560) and odd K-block counts of
    the down projection (inter 384 = 3 blocks).  The last case is large
    enough for the host to pick the 512-row down items and 128-row gate/up
    items."""
    import synth
    _, devt = _experts(H + I, E, H, I, dev)
    x = synth.hidden_states(H + T, T, H).to(dev)
    ids, w = _routing(T, E, K, H + E, dev)
    say(f"grouped long rows: H={H} I={I} T={T} E={E} K={K}")
    a = _fwd(x, ids, w, devt, mode=1)
    b = _fwd(x, ids, w, devt, mode=2)
    torch.cuda.synchronize()
    assert torch.isfinite(b.float()).all()
    if not torch.equal(a, b):
        d = (a.float() - b.float()).abs()
        pytest.fail(f"grouped != GEMV: {int((d > 0).sum())} elements differ, max {float(d.max())}")


def test_grouped_long_rows_match_oracle(lib, dev):
    import synth
    T, E, H, I, K = 6, 5, 4096, 384, 4
    host, devt = _experts(77, E, H, I, dev)
    x = synth.hidden_states(77, T, H).to(dev)
    ids, w = _routing(T, E, K, 77, dev)
    got = _fwd(x, ids, w, devt, mode=2)
    torch.cuda.synchronize()
    want = omoe.forward_w8a8(x.float().cpu().numpy(), ids.cpu().numpy(),
                             w.cpu().numpy().astype(np.float64), *(t.numpy() for t in host))
    err = omoe.max_rel_err(got.float().cpu().numpy(), want)
    print(f"grouped (H={H}, I={I}) max rel err vs W8A8 oracle {err:.2e}")
    assert err <= TOL


def _device_experts(seed, E, H, I, dev):
    """Random e4m3 weights and scales made on the device."""
    g = torch.Generator(device=dev).manual_seed(seed)
    def rnd(*s):
        return (torch.randn(s, generator=g, device=dev) * 80).clamp_(-448, 448).to(
            torch.float8_e4m3fn)

    def sc(*s):
        return torch.rand(s, generator=g, device=dev) * 1e-4 + 1e-4

    w13 = torch.cat([rnd(1, 2 * I, H) for _ in range(E)])
    w2 = torch.cat([rnd(1, H, I) for _ in range(E)])
    return (w13.view(torch.uint8), sc(E, 2 * I // 128, H // 128), w2.view(torch.uint8),
            sc(E, H // 128, I // 128))


@pytest.mark.parametrize("T,E,K,H,I", [
    # too few items for the wide tiles: 32-row ones
    (18, 1, 1, 256, 128),        # one K-block of down, two of gate/up
    (64, 1, 1, 2048, 512), (65, 1, 1, 512, 256), (129, 1, 1, 1024, 512),   # around whole tiles
    (100, 5, 3, 768, 384),       # a row block to spare, windows that end inside K
    (40, 6, 4, 8192, 2048),      # the largest expert
    # wide tiles
    (300, 16, 8, 2048, 512), (90, 4, 4, 4096, 1152),      # three windows of down
    # several placement passes: the last of one pair, wide and streamed tiles, 1000 experts
    (4097, 2, 1, 256, 128), (1100, 300, 8, 128, 128), (1300, 1000, 7, 256, 128),
    (6145, 3, 1, 256, 128), (8193, 2, 1, 256, 128),   # ... side by side, the last of one pair
    (4000, 1100, 8, 256, 128),   # wide tiles listed by the placement of more than 1024 experts
    # few rows per expert: 16-row tiles, most of one row; one expert with several
    (220, 450, 6, 256, 128), (40, 130, 8, 2048, 512), (64, 160, 6, 768, 384),
])
@pytest.mark.parametrize("tiled", [False, True])
def test_wide_tiles_equal_gemv(lib, dev, T, E, K, H, I, tiled):
    """Token tiles of 64, 32 and 16 rows, bit-identical to the per-pair GEMV for
    full, ragged and single-row column tiles, an expert without rows and picks
    of no expert (their tokens are NaN)."""
    from hostpool import RecordLayout
    import hipfetch
    devt = _device_experts(T + E, E, H, I, dev)
    rng = np.random.default_rng(T)
    ids = np.stack([rng.permutation(E)[:K] for _ in range(T)])
    if E > 4:
        ids[:, 0] = np.where(rng.random(T) < 0.6, 0, ids[:, 0])    # a crowded expert
        ids[ids == E - 1] = 1                                      # one nobody picks
    if T > 64 and E > 1:
        ids[3, 0], ids[T - 1, K - 1] = -1, E
    ids = torch.from_numpy(ids).to(dev)
    w = torch.rand((T, K), generator=torch.Generator().manual_seed(T)).to(dev)
    g = torch.Generator(device=dev).manual_seed(T)
    x = torch.randn((T, H), generator=g, device=dev).to(torch.bfloat16)
    if tiled:
        lay = RecordLayout(H, I)
        devt = lay.views(torch.cat([lay.pack(*(t[e:e + 1] for t in devt)) for e in range(E)]))
    code = hipfetch.LAYOUT_TILES if tiled else hipfetch.LAYOUT_ROWS
    say(f"wide tiles: T={T} E={E} K={K} H={H} I={I} tiled={tiled}")
    outs = []
    for mode in (1, 2):
        out = torch.full((T + 1, H), 7.0, dtype=torch.bfloat16, device=dev)
        ws = torch.empty(lib.fp8_moe_workspace(T, K, E, H, I), dtype=torch.uint8, device=dev)
        lib.fp8_moe_forward(x, ids, w, devt[0].view(torch.float8_e4m3fn), devt[1],
                            devt[2].view(torch.float8_e4m3fn), devt[3], out[:T], ws, mode=mode,
                            residual=x, layout=code)
        torch.cuda.synchronize()
        assert bool((out[T] == 7).all())
        outs.append(out[:T].view(torch.int16))
    assert torch.equal(*outs)
    bad = torch.isnan(outs[0].view(torch.bfloat16)).any(1).nonzero().view(-1).tolist()
    assert bad == ([3, T - 1] if T > 64 and E > 1 else [])


# rows per expert around whole tiles and column tiles of 16, one expert without
# any; repeated to the number of experts
_SEGMENTS = (64, 65, 128, 129, 63, 1, 17, 0, 16, 33, 48, 127)


@pytest.mark.parametrize("E,used,H,I", [
    (60, 60, 256, 128),          # one K-block of the down projection, two of gate/up
    (24, 24, 768, 384),          # a row block to spare, windows that end inside K
    (12, 12, 2048, 512), (12, 12, 8192, 2048),   # the largest expert
    (240, 180, 1024, 512),       # weights past the caches, in tile order
])
@pytest.mark.parametrize("tiled", [False, True])
def test_wide_tiles_segment_edges(lib, dev, E, used, H, I, tiled):
    """Wide tiles of segments that fill, miss and overrun them by a row,
    bit-identical to the per-pair GEMV."""
    from hostpool import RecordLayout
    import hipfetch
    counts = [_SEGMENTS[e % len(_SEGMENTS)] if e < used else 0 for e in range(E)]
    g = torch.Generator().manual_seed(E + H)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    ids = ids[torch.randperm(len(ids), generator=g)].view(-1, 1).to(dev)
    T = len(ids)
    devt = _device_experts(E, E, H, I, dev)
    if tiled:
        lay = RecordLayout(H, I)
        devt = lay.views(torch.cat([lay.pack(*(t[e:e + 1] for t in devt)) for e in range(E)]))
    x = torch.randn((T, H), generator=g).to(torch.bfloat16).to(dev)
    w = torch.rand((T, 1), generator=g).to(dev)
    say(f"wide tiles, segment edges: T={T} E={E} H={H} I={I} tiled={tiled}")
    outs = []
    for mode in (1, 2):
        out = torch.empty((T, H), dtype=torch.bfloat16, device=dev)
        ws = torch.empty(lib.fp8_moe_workspace(T, 1, E, H, I), dtype=torch.uint8, device=dev)
        lib.fp8_moe_forward(x, ids, w, devt[0].view(torch.float8_e4m3fn), devt[1],
                            devt[2].view(torch.float8_e4m3fn), devt[3], out, ws, mode=mode,
                            layout=hipfetch.LAYOUT_TILES if tiled else hipfetch.LAYOUT_ROWS)
        torch.cuda.synchronize()
        outs.append(out.view(torch.int16))
    assert torch.equal(*outs)


# (tokens, experts, top_k, hidden, inter) -> (chunk, row blocks per down item)
# of the wide plan (tests/test_dispatch.py holds the plans to it)
WIDE_PLANS = {
    (800, 64, 8, 1024, 1024): (4, 2),    # two K windows of down kept over two row blocks
    (800, 64, 8, 1024, 1152): (4, 2),    # three, staged again for the second block
    (900, 64, 8, 1280, 640): (4, 2),     # an odd number of row blocks: the last item has one
    (900, 64, 8, 1280, 1152): (4, 2),
    (1560, 520, 8, 256, 128): (8, 1),   # runs of 8 tiles
    (1560, 520, 8, 512, 256): (8, 2),
}


@pytest.mark.parametrize("case", list(WIDE_PLANS), ids=lambda c: "-".join(map(str, c)))
@pytest.mark.parametrize("tiled", [False, True])
def test_wide_down_row_blocks(lib, dev, case, tiled):
    """Wide down items of two row blocks and runs of 8 tiles, bit-identical to
    the per-pair GEMV."""
    from hostpool import RecordLayout
    import hipfetch
    T, E, K, H, I = case
    devt = _device_experts(T + H, E, H, I, dev)
    if tiled:
        lay = RecordLayout(H, I)
        devt = lay.views(torch.cat([lay.pack(*(t[e:e + 1] for t in devt)) for e in range(E)]))
    g = torch.Generator().manual_seed(T + I)
    ids = torch.rand((T, E), generator=g).topk(K, 1).indices.to(torch.int32).to(dev)
    w = torch.rand((T, K), generator=g).to(dev)
    x = torch.randn((T, H), generator=g).to(torch.bfloat16).to(dev)
    say(f"wide down: T={T} E={E} K={K} H={H} I={I} tiled={tiled}")
    outs = []
    for mode in (1, 2):
        out = torch.empty((T, H), dtype=torch.bfloat16, device=dev)
        ws = torch.empty(lib.fp8_moe_workspace(T, K, E, H, I), dtype=torch.uint8, device=dev)
        lib.fp8_moe_forward(x, ids, w, devt[0].view(torch.float8_e4m3fn), devt[1],
                            devt[2].view(torch.float8_e4m3fn), devt[3], out, ws, mode=mode,
                            layout=hipfetch.LAYOUT_TILES if tiled else hipfetch.LAYOUT_ROWS)
        torch.cuda.synchronize()
        outs.append(out.view(torch.int16))
    assert torch.equal(*outs)
