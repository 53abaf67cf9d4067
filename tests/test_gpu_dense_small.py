"""GPU parity of the Dense kernels that serve what the 128- and 256-wide tiles do not: any shape and alignment.

Bound of every comparison: the fp32 sum of K products in any order is off by at most K 2^-24 sum |x w|, and one rounding
to fp16 adds half an ulp of the result (2^-11 relative, 2^-25 below the normal range)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def dev(a):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def make(dthip, oracle, rng, N, K, q, nib):
    """(QxTensor, its weights as float64)."""
    if q == 16:
        w = (rng.standard_normal((N, K)) * 0.05).astype(np.float16)
        return dthip.QxTensor.from_f16(w), w.astype(np.float64)
    packed, _, _ = oracle.synth_qx_weight(rng, N, K, q, nib, 0.05)
    return dthip.QxTensor.from_packed(packed, q, nib, (N, K)), oracle.C.depalettize(q, nib, N * K, packed).reshape(N, K).astype(np.float64)


def check(got, X, W, bias=None):
    X = X.astype(np.float64)
    want = X @ W.T + (0 if bias is None else bias.astype(np.float64))
    sums = X.shape[1] * 2.0 ** -24 * (np.abs(X) @ np.abs(W).T + (0 if bias is None else np.abs(bias.astype(np.float64))))
    tol = (np.abs(want) + sums) * 2.0 ** -11 + 2.0 ** -25 + sums
    bad = np.abs(got.astype(np.float64) - want) > tol
    assert not bad.any(), (int(bad.sum()), np.argwhere(bad)[:4])


def _groups(dthip, x, ws, outs, bias=None, epi=None, post=None):
    """One problem as the C entry points take it, and what keeps it alive."""
    import ctypes

    n, at = len(ws), ctypes.addressof
    W = (dthip._QxWeight * n)(*[w._c() for w in ws])
    B = (ctypes.c_void_p * n)(*[None if bias is None or b is None else b.data_ptr() for b in bias or ws])
    Y, LDY = (ctypes.c_void_p * n)(*[o.data_ptr() for o in outs]), (ctypes.c_int64 * n)(*[o.stride(0) for o in outs])
    tails = [None if t is None else ctypes.create_string_buffer(t, len(t)) for t in (epi, post)]
    G = (dthip._DenseGroup * 1)(dthip._DenseGroup(x.shape[0], x.shape[1], x.data_ptr(), x.stride(0), at(W), n, at(B), at(Y), at(LDY),
                                                  *[None if t is None else at(t) for t in tails]))
    return G, (W, B, Y, LDY, tails)


@pytest.mark.parametrize("M,N,K,q,nib", [
    (1, 1, 1, 6, 1),            # the smallest there is: one block per weight
    (33, 31, 100, 6, 32),       # blocks that end inside a thread's run of 16
    (32, 32, 128, 5, 24),       # a block stride that is no multiple of 4
    (31, 65, 129, 7, 4096),     # an odd row length: every row starts at another bit
    (5, 40, 16, 4, 512),        # less than a K-tile
    (231, 1001, 1000, 8, 16384),
    (130, 70, 127, 16, 0), (40, 33, 72, 16, 0),  # plain fp16, without and with 16-byte rows
    (70, 90, 2500, 8, 512),     # more palettes than the LDS holds: looked up in memory
    (1500, 1400, 200, 6, 4096), (1450, 1470, 77, 4, 64), (1500, 1400, 100, 16, 0),  # enough tiles for the 64 x 64 form
])
def test_dense_any_shape(dthip, oracle, M, N, K, q, nib):
    rng = np.random.default_rng(M * 7 + N * 5 + K + q)
    X = rng.standard_normal((M, K)).astype(np.float16)
    w, W = make(dthip, oracle, rng, N, K, q, nib)
    bias = (rng.standard_normal(N) * 0.1).astype(np.float16)
    print("dense any shape", M, N, K, q, nib, flush=True)
    check(dthip.dense_multi(dev(X), [w], [dev(bias)])[0].cpu().numpy(), X, W, bias)
    # X as a view that starts at an odd element of rows of odd length
    wide = np.zeros((M, K + 3 - (K & 1)), np.float16)
    wide[:, 1:1 + K] = X
    check(dthip.dense_multi(dev(wide)[:, 1:1 + K], [w], [None])[0].cpu().numpy(), X, W)


@pytest.mark.parametrize("M,N,K,q,nib", [
    (1, 1, 64, 6, 64),             # one output; half of a 128-wide stretch of K
    (1, 3072, 3072, 8, 16384), (16, 17, 128, 4, 512), (17, 33, 192, 5, 1024), (33, 100, 1216, 6, 4096),
    (64, 48, 2112, 7, 8192), (64, 70, 64, 16, 0), (3, 9000, 320, 6, 4096),  # (the last: 32 features per workgroup)
    (20, 8200, 192, 16, 0),
    (2, 40, 3072, 8, 64),          # palettes that do not fit: the tiled kernel
])
def test_dense_few_rows(dthip, oracle, M, N, K, q, nib):
    rng = np.random.default_rng(M * 7 + N * 5 + K + q)
    X = rng.standard_normal((M, K)).astype(np.float16)
    wide = np.zeros((M, K + 8), np.float16)  # rows that do not follow each other
    wide[:, :K] = X
    pairs = [make(dthip, oracle, rng, n, K, q, nib) for n in (N, 16, N)]
    bias = [(rng.standard_normal(w.shape[0]) * 0.1).astype(np.float16) for w, _ in pairs]
    print("dense few rows", M, N, K, q, nib, flush=True)
    outs = dthip.dense_multi(dev(wide)[:, :K], [w for w, _ in pairs], [dev(bias[0]), None, dev(bias[2])])
    for i, (_, W) in enumerate(pairs):
        check(outs[i].cpu().numpy(), X, W, None if i == 1 else bias[i])
    # the tails act on the same Dense results, bit for bit
    gate = dev((1 + 0.3 * rng.standard_normal(N)).astype(np.float16))
    res = dev(rng.standard_normal((M, N)).astype(np.float32))
    want = res + (outs[0].float() * gate.float()).half().float()
    dthip.dense_post(dev(X), [w for w, _ in pairs], [dev(bias[0]), None, dev(bias[2])],
                     [dthip.DensePost(gate=gate, residual=res, keep_output=False), None, None])
    assert bool((res == want).all())


@pytest.mark.parametrize("M,K,rank,N", [(1, 1, 1, 1), (15, 33, 3, 7), (17, 100, 16, 129), (65, 320, 17, 128), (130, 257, 33, 200),
                                        (300, 3072, 128, 96), (33, 64, 70, 1001), (4099, 96, 20, 136), (4100, 40, 130, 130)])
def test_lora_branch_fp32_shapes(dthip, M, K, rank, N):
    """fp16(up(scale * down(float(x)))) at the edges of both kernels' blocks and of their K steps, X an unaligned view:
    both sums in fp32 (K 2^-24 and rank 2^-24 of the sums of magnitudes), one rounding to fp16."""
    import torch

    rng = np.random.default_rng(M + K + rank + N)
    X = rng.standard_normal((M, K)).astype(np.float16)
    wide = np.zeros((M, K + 2 + (K & 1)), np.float16)
    wide[:, 1:1 + K] = X
    down = (rng.standard_normal((rank, K)) * 0.1).astype(np.float32)
    up = (rng.standard_normal((N, rank)) * 0.1).astype(np.float32)
    xd, dd, ud = dev(wide), dev(down), dev(up)
    T = torch.empty((M, rank), dtype=torch.float32, device="cuda")
    out = torch.empty((M, N), dtype=torch.float16, device="cuda")
    print("lora branch", M, K, rank, N, flush=True)
    st = dthip.lib().dt_lora_branch_f32_f16(None, M, K, xd.data_ptr() + 2, wide.shape[1], dd.data_ptr(), rank, ud.data_ptr(), N, 0.75,
                                            T.data_ptr(), out.data_ptr(), N)
    assert st == 0
    X, down, up = (a.astype(np.float64) for a in (X, down, up))
    t, t_abs = 0.75 * (X @ down.T), 0.75 * (np.abs(X) @ np.abs(down).T)
    assert np.all(np.abs(T.cpu().numpy() - t) <= (K + 2) * 2.0 ** -24 * t_abs)
    want, sums = t @ up.T, (K + rank + 2) * 2.0 ** -24 * (t_abs @ np.abs(up).T)
    assert np.all(np.abs(out.cpu().numpy().astype(np.float64) - want) <= sums + (np.abs(want) + sums) * 2.0 ** -11 + 2.0 ** -25)


@pytest.mark.parametrize("M,N,K,q,nib", [
    (65, 256, 128, 6, 4096), (128, 300, 192, 5, 1024),    # 128 x 256 tiles; 2 and 3 shares
    (129, 257, 320, 4, 512), (300, 600, 448, 6, 64),      # 256 x 256 tiles; 5 and 7 shares, ragged edges, a block per 64 columns
    (257, 256, 576, 8, 16384), (200, 130, 704, 16, 0),    # 8 shares of unequal length; shared palettes, plain fp16
    (200, 140, 512, 8, 512), (130, 300, 512, 7, 512),     # palettes that only fit beside 256 x 128 tiles
    (130, 300, 1088, 7, 4096),                            # ... and that fit beside 256 x 256 tiles, shared
])
def test_dense_cut_along_k(dthip, oracle, monkeypatch, M, N, K, q, nib):
    import torch

    rng = np.random.default_rng(M * 7 + N * 5 + K + q)
    X = rng.standard_normal((M, K)).astype(np.float16)
    pairs = [make(dthip, oracle, rng, n, K, q, nib) for n in (N, 128)]
    ws, bias = [w for w, _ in pairs], dev((rng.standard_normal(N) * 0.1).astype(np.float16))
    x, gate = dev(X), dev((1 + 0.3 * rng.standard_normal(N)).astype(np.float16))
    gamma, rot = dev((1 + 0.1 * rng.standard_normal(128)).astype(np.float16)), dev(rng.standard_normal((M + 3, 128)).astype(np.float16))
    epi = [None, dthip.HeadEpilogue(gamma, rot, 3)]
    print("dense cut along K", M, N, K, q, nib, flush=True)
    monkeypatch.setenv("DT_DENSE_EXPAND", "never")
    monkeypatch.setenv("DT_DENSE_SPLIT", "never")
    whole = dthip.dense_multi(x, ws, [bias, None])
    monkeypatch.setenv("DT_DENSE_SPLIT", "always")
    # every tile is cut into as many shares as there are pairs of K-tiles, up to eight, of a slot of its fp32 sums each
    bm = 256 if M > 128 or (q == 7 and nib == 512) or (q == 8 and nib == 512) else 128
    bn = 128 if (q == 7 and nib == 512) or (q == 8 and nib == 512) else 256
    tiles, shares = sum(-(-M // bm) * -(-w.shape[0] // bn) for w in ws), min(8, K // 64)
    G, keep = _groups(dthip, x, ws, [torch.empty((M, w.shape[0]), dtype=torch.float16, device="cuda") for w in ws])
    assert dthip.lib().dt_dense_workspace_bytes(1, G) == (tiles * 32 + 255) // 256 * 256 + tiles * shares * bm * bn * 4
    outs = dthip.dense_multi(x, ws, [bias, None])
    assert not all(torch.equal(a, b) for a, b in zip(outs, whole))  # (the sums were added up in another order)
    again = dthip.dense_multi(x, ws, [bias, None])
    check(outs[0].cpu().numpy(), X, pairs[0][1], bias.cpu().numpy())
    check(outs[1].cpu().numpy(), X, pairs[1][1])
    assert all(torch.equal(a, b) for a, b in zip(outs, again))
    # the tails act on the same sums, bit for bit
    res = dev(rng.standard_normal((M, N)).astype(np.float32))
    want = res + (outs[0].float() * gate.float()).half().float()
    dthip.dense_post(x, ws, [bias, None], [dthip.DensePost(gate=gate, residual=res, keep_output=False), None])
    assert torch.equal(res, want)
    if bn == 256:  # (the head epilogue's tiles are 256 wide)
        fused = dthip.dense_multi(x, ws, [bias, None], epilogues=epi)
        lead = dthip.dense_multi(x, ws, [bias, None])[1]
        assert torch.equal(fused[0], outs[0])
        v = lead.float()
        n = (v * torch.rsqrt((v * v).mean(-1, keepdim=True) + 1e-6) * gamma.float()).half().float()
        r = rot[3:].float()
        turned = torch.stack([n[:, ::2] * r[:, ::2] - n[:, 1::2] * r[:, 1::2], n[:, ::2] * r[:, 1::2] + n[:, 1::2] * r[:, ::2]], -1).reshape(M, 128)
        # one fp16 rounding more or less of a normalised value, turned: 2^-10 of the pair's magnitude, plus the last rounding
        mag = torch.hypot(n[:, ::2], n[:, 1::2]).repeat_interleave(2, -1) * torch.hypot(r[:, ::2], r[:, 1::2]).repeat_interleave(2, -1)
        assert bool(((fused[1].float() - turned).abs() <= mag * 2.0 ** -9 + 2.0 ** -24).all())


@pytest.mark.parametrize("K", [64, 128, 192, 256, 320, 704])
def test_dense_plain_pair_slots(dthip, oracle, K):
    """Plain fp16 weights with fewer K-tile pairs than the 128 x 128 tile's four slots, as many, and more; the 128 x 256
    tile's three, which a fused head epilogue beside it asks for; and the two that launches of many tiles keep."""
    rng = np.random.default_rng(K)
    print("dense plain pair slots", K, flush=True)
    for M, N in ((130, 200), (300, 256), (2050, 2100)):
        X = rng.standard_normal((M, K)).astype(np.float16)
        (w, W), (head, _) = make(dthip, oracle, rng, N, K, 16, 0), make(dthip, oracle, rng, 128, K, 16, 0)
        check(dthip.dense_multi(dev(X), [w], [None])[0].cpu().numpy(), X, W)
        if M < 1024:
            epi = dthip.HeadEpilogue(dev(np.ones(128, np.float16)), None, 0)
            check(dthip.dense_multi(dev(X), [head, w], [None, None], epilogues=[epi, None])[1].cpu().numpy(), X, W)


@pytest.mark.parametrize("M,N,K", [(65, 8, 320), (128, 128, 384), (129, 257, 448), (300, 600, 512), (1000, 3900, 576)])
def test_dense_plain_tile_per_compute_unit(dthip, oracle, M, N, K):
    """Plain fp16 weights on up to 256 tiles of 128 x 128, five pairs of K-tiles and more: every remainder of the rounds of
    four slots, ragged edges, two weights; and the kernel with the tail, whose tail does nothing, bit for bit."""
    import torch

    rng = np.random.default_rng(M + N + K)
    X = rng.standard_normal((M, K)).astype(np.float16)
    pairs = [make(dthip, oracle, rng, n, K, 16, 0) for n in (N, 128)]
    ws, bias = [w for w, _ in pairs], dev((rng.standard_normal(N) * 0.1).astype(np.float16))
    print("dense plain tile per compute unit", M, N, K, flush=True)
    outs = dthip.dense_multi(dev(X), ws, [bias, None])
    check(outs[0].cpu().numpy(), X, pairs[0][1], bias.cpu().numpy())
    check(outs[1].cpu().numpy(), X, pairs[1][1])
    zero = torch.zeros((M, N), dtype=torch.float16, device="cuda")
    tails = dthip.dense_post(dev(X), ws, [bias, None], [dthip.DensePost(addend=zero), dthip.DensePost()])
    assert all(torch.equal(a, b) for a, b in zip(outs, tails))


@pytest.mark.parametrize("K", [64, 128, 192])
def test_dense_plain_brief(dthip, oracle, K):
    """Many tiles of one or two K-tile pairs stay 128 x 128; with three they are 256 x 256."""
    rng = np.random.default_rng(K)
    X = rng.standard_normal((4099, K)).astype(np.float16)
    w, W = make(dthip, oracle, rng, 3080, K, 16, 0)
    check(dthip.dense_multi(dev(X), [w], [None])[0].cpu().numpy(), X, W)


@pytest.mark.parametrize("K", [64, 128, 192, 256, 320, 704])
@pytest.mark.parametrize("q,nib", [(4, 512), (5, 1024), (6, 4096), (7, 8192), (8, 16384), (8, 512)])
def test_dense_small_tile_pairs(dthip, oracle, K, q, nib):
    """The 128 x 128 tile's K-tile pairs, from one to several rounds of its index registers, palettes per row and shared,
    one workgroup per compute unit and two."""
    rng = np.random.default_rng(K + q + nib)
    for M, N in ((131, 260), (1300, 4096)) if K in (64, 320) else ((131, 260),):
        X = rng.standard_normal((M, K)).astype(np.float16)
        w, W = make(dthip, oracle, rng, N, K, q, nib)
        check(dthip.dense_multi(dev(X), [w], [None])[0].cpu().numpy(), X, W)


@pytest.mark.parametrize("M,N,K,nib", [
    (200, 300, 64, 4096), (200, 300, 1600, 4096),  # 128 x 128 tiles, a block's end at every second K-tile
    (200, 300, 640, 4096), (200, 300, 768, 4096),  # at every fourth: shared palettes still; every eighth: per row
    (200, 300, 6080, 4096), (200, 300, 6208, 4096),  # as many palettes as 24 KB hold, and more
    (70, 300, 320, 64),                            # small blocks
    (8100, 1600, 192, 4096), (6200, 2000, 4032, 4096), (6200, 2000, 4160, 4096),  # 256 x 256 tiles: up to 32 KB, and beyond
])
def test_dense_shared_palettes_of_64(dthip, oracle, M, N, K, nib):
    import torch

    rng = np.random.default_rng(M + N + K)
    w, W = make(dthip, oracle, rng, N, K, 6, nib)
    X = rng.standard_normal((M, K)).astype(np.float16)
    got = dthip.dense_multi(dev(X), [w], [None])[0]
    rows = np.unique(np.concatenate([np.arange(min(M, 130)), np.arange(M - 130, M).clip(0)]))
    check(got[torch.from_numpy(rows).cuda()].cpu().numpy(), X[rows], W)


@pytest.mark.parametrize("K,q", [(512, 7), (1024, 8), (1536, 7), (2048, 8)])
def test_dense_row_palettes_on_a_unit_of_ones_own(dthip, oracle, monkeypatch, K, q):
    """128 x 128 tiles with 128- and 256-entry palettes: up to 256 of them look every row's palette up in a table of its
    own, more share the palettes with a neighbour.  The same bits, at ragged edges of either; and against the oracle."""
    import torch

    rng = np.random.default_rng(K + q)
    monkeypatch.setenv("DT_DENSE_SPLIT", "never")  # (a cut tile's sums are added up in another order)
    monkeypatch.setenv("DT_DENSE_EXPAND", "never")
    nib = {7: 8192, 8: 16384}[q]
    N, few, many = 2433, 200, 1790  # 2 and 14 tiles by 20: 40 and 280
    X = rng.standard_normal((many, K)).astype(np.float16)
    w, W = make(dthip, oracle, rng, N, K, q, nib)
    x = dev(X)
    print("dense row palettes", K, q, flush=True)
    got = dthip.dense_multi(x[:few], [w], [None])[0]
    assert torch.equal(got, dthip.dense_multi(x, [w], [None])[0][:few])
    check(got[150:].cpu().numpy(), X[150:few], W)


def test_dense_workspace_is_optional(dthip, oracle, monkeypatch):
    """A launch of few tiles is cut without being told to; too little workspace, or none, gives the uncut result, a
    misaligned one is refused; and a captured graph replays the cut launch, its counters zeroed each time."""
    import torch

    monkeypatch.delenv("DT_DENSE_SPLIT", raising=False)
    rng = np.random.default_rng(12)
    X = rng.standard_normal((300, 3072)).astype(np.float16)
    w, W = make(dthip, oracle, rng, 512, 3072, 6, 4096)
    x, out = dev(X), torch.zeros((300, 512), dtype=torch.float16, device="cuda")
    G, keep = _groups(dthip, x, [w], [out])
    L, s = dthip.lib(), torch.cuda.current_stream().cuda_stream
    need = L.dt_dense_workspace_bytes(1, G)
    assert need > 0
    ws = torch.full((need + 256,), 0xff, dtype=torch.uint8, device="cuda")
    assert L.dt_dense_qx_grouped_f16(s, 1, G, 0) == 0
    whole = out.clone()
    check(whole.cpu().numpy(), X, W)
    for give in (0, 256):
        out.zero_()
        assert L.dt_dense_qx_grouped_ws_f16(s, 1, G, 0, ws.data_ptr() if give else None, give) == 0
        assert torch.equal(out, whole)
    assert L.dt_dense_qx_grouped_ws_f16(s, 1, G, 0, ws.data_ptr() + 64, need) == dthip.DT_INVALID
    assert L.dt_dense_qx_grouped_ws_f16(s, 1, G, 0, ws.data_ptr(), need) == 0
    cut = out.clone()
    check(cut.cpu().numpy(), X, W)
    print("dense cut along K as hip graph", flush=True)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        L.dt_dense_qx_grouped_ws_f16(torch.cuda.current_stream().cuda_stream, 1, G, 0, ws.data_ptr(), need)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, cut)
        assert L.dt_dense_qx_grouped_ws_f16(s, 1, G, 0, ws.data_ptr(), need) == 0


@pytest.mark.parametrize("M,q,nib", [(5, 6, 4096), (70, 6, 4096), (1100, 8, 16384), (70, 16, 0), (300, 6, 24)])
def test_dense_c_entry_points_without_workspace(dthip, oracle, monkeypatch, M, q, nib):
    """The Dense entry points that take no workspace do what the operators, which go through the one that takes it, do when
    nothing is cut: bit for bit, plain, with head epilogues, with tails, and as a group."""
    import ctypes

    import torch

    monkeypatch.setenv("DT_DENSE_SPLIT", "never")
    monkeypatch.setenv("DT_DENSE_EXPAND", "never")
    rng = np.random.default_rng(M + q)
    K, N = 320, 256
    x = dev(rng.standard_normal((M, K)).astype(np.float16))
    ws = [make(dthip, oracle, rng, N, K, q, nib)[0] for _ in range(2)]
    bias = [dev((rng.standard_normal(N) * 0.1).astype(np.float16)), None]
    gamma, rot = dev((1 + 0.1 * rng.standard_normal(128)).astype(np.float16)), dev(rng.standard_normal((M, 128)).astype(np.float16))
    epi = [dthip.HeadEpilogue(gamma, rot), None]
    gate, res0 = dev((1 + 0.3 * rng.standard_normal(N)).astype(np.float16)), dev(rng.standard_normal((M, N)).astype(np.float32))
    res = [res0.clone(), res0.clone()]
    posts = [[dthip.DensePost(dthip.ACT_GELU_TANH, gate=gate, residual=r), dthip.DensePost(scale=0.5)] for r in res]
    want = [dthip.dense_multi(x, ws, bias), dthip.dense_multi(x, ws, bias, epilogues=epi), dthip.dense_post(x, ws, bias, posts[0])]
    L, s = dthip.lib(), torch.cuda.current_stream().cuda_stream
    new = lambda: [torch.zeros((M, N), dtype=torch.float16, device="cuda") for _ in ws]
    packed_epi = dthip._pack_epilogues(epi, M)
    print("dense entry points without workspace", M, q, nib, flush=True)

    def call(fn, outs, *tail):
        (g,), keep = _groups(dthip, x, ws, outs, bias)
        W, B, Y, LDY, _ = keep
        return fn(s, g.M, g.K, g.X, g.ldx, W, g.n_weights, B, Y, LDY, *tail, 0)

    outs = new()
    assert call(L.dt_dense_qx_f16, outs) == 0
    assert all(torch.equal(a, b) for a, b in zip(outs, want[0]))
    outs, held = new(), ctypes.create_string_buffer(packed_epi, len(packed_epi))
    assert call(L.dt_dense_qx_heads_f16, outs, ctypes.cast(held, L.dt_dense_qx_heads_f16.argtypes[10])) == 0
    assert all(torch.equal(a, b) for a, b in zip(outs, want[1]))
    outs = new()
    packed_post = dthip._pack_posts(posts[1], ws, M, [o.data_ptr() for o in outs], list(outs))
    held = ctypes.create_string_buffer(packed_post, len(packed_post))
    assert call(L.dt_dense_qx_post_f16, outs, ctypes.cast(held, L.dt_dense_qx_post_f16.argtypes[10])) == 0
    assert all(torch.equal(a, b) for a, b in zip(outs, want[2])) and torch.equal(res[0], res[1])
    for kind, tails in enumerate([{}, {"epi": packed_epi}]):
        outs = new()
        G, keep = _groups(dthip, x, ws, outs, bias, **tails)
        assert L.dt_dense_qx_grouped_f16(s, 1, G, 0) == 0
        assert all(torch.equal(a, b) for a, b in zip(outs, want[kind]))


@pytest.mark.parametrize("M,N,K,q,nib", [
    (70, 8, 64, 6, 4096),                                # less than one block, two granules per row
    (129, 257, 320, 4, 512), (200, 130, 448, 5, 1024),   # the smallest blocks; a last tile of granules that is not full
    (300, 600, 704, 7, 8192), (1100, 520, 576, 8, 16384), (260, 300, 640, 8, 544),  # a block per 17 granules
])
def test_dense_on_copies_of_the_weights(dthip, oracle, monkeypatch, M, N, K, q, nib):
    """Weights written out as fp16 ahead of the launch: the same bits as looked up in it, with every kind of tail; cut along K
    as well; not with less scratch than the copies take; and replayed from a graph."""
    import torch

    rng = np.random.default_rng(M + N * 3 + K + q)
    X = rng.standard_normal((M, K)).astype(np.float16)
    pairs = [make(dthip, oracle, rng, n, K, q, nib) for n in (N, 128)]
    ws, bias = [w for w, _ in pairs], dev((rng.standard_normal(N) * 0.1).astype(np.float16))
    x, gamma = dev(X), dev((1 + 0.1 * rng.standard_normal(128)).astype(np.float16))
    epi, res = [None, dthip.HeadEpilogue(gamma, None, 0)], torch.zeros((M, N), dtype=torch.float32, device="cuda")
    print("dense on copies", M, N, K, q, nib, flush=True)
    outs = [torch.empty((M, w.shape[0]), dtype=torch.float16, device="cuda") for w in ws]
    G, keep = _groups(dthip, x, ws, outs)
    L, s = dthip.lib(), torch.cuda.current_stream().cuda_stream
    monkeypatch.setenv("DT_DENSE_SPLIT", "never")
    got = {}
    for knob in ("never", "always"):
        monkeypatch.setenv("DT_DENSE_EXPAND", knob)
        res.zero_()
        got[knob] = dthip.dense_multi(x, ws, [bias, None]) + dthip.dense_multi(x, ws, [bias, None], epilogues=epi)
        got[knob] += dthip.dense_post(x, ws, [bias, None], [dthip.DensePost(dthip.ACT_GELU_TANH, residual=res), None]) + [res.clone()]
    check(got["always"][0].cpu().numpy(), X, pairs[0][1], bias.cpu().numpy())
    assert all(torch.equal(a, b) for a, b in zip(got["always"], got["never"]))
    need = L.dt_dense_scratch_bytes(1, G)
    assert need == sum((w.count * 2 + 255) // 256 * 256 for w in ws) and L.dt_dense_workspace_bytes(1, G) == 0
    scratch = torch.full((need + 256,), 0xff, dtype=torch.uint8, device="cuda")
    at = (scratch.data_ptr() + 255) & ~255
    assert L.dt_dense_qx_grouped_scratch_f16(s, 1, G, 0, at + 64, need) == dthip.DT_INVALID
    assert L.dt_dense_qx_grouped_scratch_f16(s, 1, G, 0, at, need - 256) == 0 and bool((scratch == 0xff).all())
    plain = dthip.dense_multi(x, ws, [None, None])
    assert all(torch.equal(a, b) for a, b in zip(outs, plain))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        assert L.dt_dense_qx_grouped_scratch_f16(torch.cuda.current_stream().cuda_stream, 1, G, 0, at, need) == 0
    for _ in range(3):
        outs[0].zero_()
        scratch.fill_(0xff)
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(outs, plain))
    for w, copy in zip(ws, torch.split(scratch[at - scratch.data_ptr():][:need], [(w.count * 2 + 255) // 256 * 256 for w in ws])):
        assert torch.equal(copy[:w.count * 2].view(torch.float16).view(w.shape), w.dequantize())
    monkeypatch.setenv("DT_DENSE_SPLIT", "always")
    cut = dthip.dense_multi(x, ws, [bias, None])
    check(cut[0].cpu().numpy(), X, pairs[0][1], bias.cpu().numpy())
    check(cut[1].cpu().numpy(), X, pairs[1][1])


@pytest.mark.parametrize("M,N,K,q,nib,rank", [(130, 260, 320, 6, 4096, 16), (300, 512, 448, 8, 16384, 64), (1100, 600, 704, 4, 512, 100)])
def test_lora_base_and_down_in_one_launch(dthip, oracle, monkeypatch, M, N, K, q, nib, rank):
    """The base projection on a copy of its weight and the plain down projection go out together: the same bits as one after
    the other, with and without a tail."""
    import torch

    rng = np.random.default_rng(M + N + rank)
    op = dthip.LoRADense(N, dthip.LoRANetworkConfiguration(rank, 0.75, False))
    op.weight, op.bias = make(dthip, oracle, rng, N, K, q, nib)[0], dev((rng.standard_normal(N) * 0.1).astype(np.float16))
    op.down, op.up = make(dthip, oracle, rng, rank, K, 16, 0)[0], make(dthip, oracle, rng, N, rank, 16, 0)[0]
    x, got = dev(rng.standard_normal((M, K)).astype(np.float16)), {}
    print("lora in one launch", M, N, K, q, nib, rank, flush=True)
    monkeypatch.setenv("DT_DENSE_SPLIT", "never")
    for knob in ("never", "always"):
        monkeypatch.setenv("DT_DENSE_EXPAND", knob)
        got[knob] = [op(x), op(x, dthip.DensePost(dthip.ACT_SWISH))]
    assert all(torch.equal(a, b) for a, b in zip(got["never"], got["always"]))


@pytest.mark.parametrize("formats,together", [
    ([(16, 0), (6, 4096)], [1]),                          # the plain weight first: the launch's format is another weight's
    ([(6, 4096), (16, 0), (6, 4096)], [0, 2]),
    ([(6, 4096), (16, 0), (8, 16384), (16, 0), (8, 16384)], [2, 4]),  # two launches, a plain weight in each
])
def test_palettized_and_plain_weights_in_one_launch(dthip, oracle, monkeypatch, formats, together):
    """One launch on the copies of all palettized weights and the plain ones between them, which the scratch asked for shows: the
    same bits as one launch after the other; cut along K as well, the counters behind the copies."""
    import torch

    rng = np.random.default_rng(len(formats))
    M, K = 300, 448
    X, Ns = rng.standard_normal((M, K)).astype(np.float16), [260, 72, 130, 128, 300][:len(formats)]
    pairs = [make(dthip, oracle, rng, n, K, q, nib) for n, (q, nib) in zip(Ns, formats)]
    ws, bias = [w for w, _ in pairs], [(rng.standard_normal(n) * 0.1).astype(np.float16) for n in Ns]
    x, b = dev(X), [dev(t) for t in bias]
    print("palettized and plain weights in one launch", formats, flush=True)
    monkeypatch.setenv("DT_DENSE_SPLIT", "never")
    monkeypatch.setenv("DT_DENSE_EXPAND", "never")
    apart = dthip.dense_multi(x, ws, b)
    monkeypatch.setenv("DT_DENSE_EXPAND", "always")
    G, keep = _groups(dthip, x, ws, apart)
    assert dthip.lib().dt_dense_scratch_bytes(1, G) == sum((ws[i].count * 2 + 255) // 256 * 256 for i in together)
    assert all(torch.equal(a, c) for a, c in zip(apart, dthip.dense_multi(x, ws, b)))
    monkeypatch.setenv("DT_DENSE_SPLIT", "always")
    for got, (_, W), t in zip(dthip.dense_multi(x, ws, b), pairs, bias):
        check(got.cpu().numpy(), X, W, t)


@pytest.mark.parametrize("M,N,K,q,nib", [(64, 256, 3072, 8, 16384), (64, 128, 13824, 6, 4096), (130, 260, 3072, 4, 256)])
def test_lora_down_beside_the_base_in_a_graph(dthip, oracle, M, N, K, q, nib):
    """The down projection on its own stream: captured, replayed and beside other work, the same bits as in one call."""
    import torch

    rng = np.random.default_rng(M + N + K)
    op = dthip.LoRADense(N, dthip.LoRANetworkConfiguration(16, 0.75, False))
    op.weight, op.bias = make(dthip, oracle, rng, N, K, q, nib)[0], dev((rng.standard_normal(N) * 0.1).astype(np.float16))
    op.down, op.up = make(dthip, oracle, rng, 16, K, 16, 0)[0], make(dthip, oracle, rng, N, 16, 16, 0)[0]
    x = dev((0.1 * rng.standard_normal((M, K))).astype(np.float16))
    print("lora side by side", M, N, K, q, nib, flush=True)
    dn, up = op._padded()
    base, down = dthip.dense_post(x, [op.weight, dn], [op.bias, None], [None, dthip.DensePost(scale=0.75)])
    want = dthip.dense_post(down, [up], [None], [dthip.DensePost(addend=base)])[0]
    assert torch.equal(op(x), want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = op(x)
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        assert torch.equal(op(x), want)


def test_dense_last_round_cut_along_k(dthip, oracle, monkeypatch):
    """288 tiles: 256 stay whole, the 32 of the second round are cut; against the uncut launch, one fp16 rounding apart."""
    import torch

    rng = np.random.default_rng(13)
    M, N, K = 1530, 12288, 3072
    w, _ = make(dthip, oracle, rng, N, K, 6, 4096)
    x = dev(rng.standard_normal((M, K)).astype(np.float16))
    monkeypatch.setenv("DT_DENSE_EXPAND", "never")
    monkeypatch.setenv("DT_DENSE_SPLIT", "never")
    whole = dthip.dense_multi(x, [w], [None])[0].float()
    monkeypatch.delenv("DT_DENSE_SPLIT")
    G, keep = _groups(dthip, x, [w], [torch.empty((M, N), dtype=torch.float16, device="cuda")])
    print("dense last round cut along K", flush=True)
    assert dthip.lib().dt_dense_workspace_bytes(1, G) > 0
    cut = dthip.dense_multi(x, [w], [None])[0].float()
    # the two sums differ by at most 2 K 2^-24 sum |x w| <= 2 K 2^-24 |x| |w| (row norms), the roundings by 2^-10 of the value
    sums = 2 * K * 2.0 ** -24 * x.float().norm(dim=1)[:, None] * w.dequantize().float().norm(dim=1)[None]
    assert bool(((cut - whole).abs() <= whole.abs() * 2.0 ** -10 + sums + 2.0 ** -24).all())
    assert not torch.equal(cut, whole)


def test_lists_shorter_than_the_weights(dthip, oracle):
    """Biases, head epilogues and tails that are not given stand for none; more of them than weights are refused."""
    import torch

    rng = np.random.default_rng(23)
    M, K, N = 70, 128, 256
    x = dev(rng.standard_normal((M, K)).astype(np.float16))
    ws = [make(dthip, oracle, rng, N, K, 6, 4096)[0] for _ in range(3)]
    b = dev((rng.standard_normal(N) * 0.1).astype(np.float16))
    gamma = dev((1 + 0.1 * rng.standard_normal(128)).astype(np.float16))
    e, p = dthip.HeadEpilogue(gamma), dthip.DensePost(dthip.ACT_GELU_TANH)
    for short, full in [
        (dthip.dense_multi(x, ws, [b]), dthip.dense_multi(x, ws, [b, None, None])),
        (dthip.dense_multi(x, ws, [b, b], epilogues=[e]), dthip.dense_multi(x, ws, [b, b, None], epilogues=[e, None, None])),
        (dthip.dense_post(x, ws, [], [p]), dthip.dense_post(x, ws, [None] * 3, [p, None, None])),
    ]:
        assert len(short) == 3 and all(torch.equal(s, f) for s, f in zip(short, full))
    with pytest.raises(IndexError):
        dthip.dense_multi(x, ws[:1], [b, b])
    with pytest.raises(IndexError):
        dthip.dense_multi(x, ws[:1], [b], epilogues=[e, e])
    with pytest.raises(IndexError):
        dthip.dense_post(x, ws[:1], [b], [p, p])


@pytest.mark.parametrize("K,N", [(64, 96), (77, 33)])
def test_single_row_of_any_stride(dthip, oracle, K, N):
    """One row of X: its stride, which torch leaves at any value (1 in a [K, 1] tensor's transpose), does not matter."""
    import torch

    rng = np.random.default_rng(K)
    w, W = make(dthip, oracle, rng, N, K, 6, 4096)
    X = rng.standard_normal((1, K)).astype(np.float16)
    for x in (dev(X.reshape(K, 1)).t(), torch.as_strided(dev(X), (1, K), (7, 1)), dev(X)[:, None].transpose(0, 1)):
        check(dthip.dense_multi(x, [w], [None])[0].reshape(1, N).cpu().numpy(), X, W)
    col = torch.zeros((K, 2), dtype=torch.float16, device="cuda")
    col[:, :1] = dev(X.reshape(K, 1))
    check(dthip.dense_multi(col[:, :1].t(), [w], [None])[0].cpu().numpy(), X, W)  # (elements two apart: a copy)


def test_given_outputs_come_back_in_the_shape_of_x(dthip, oracle):
    """Contiguous outputs of one row per row of X are returned with X's leading dimensions, for a 2-D X as for any other."""
    import torch

    rng = np.random.default_rng(3)
    M, K, N = 6, 64, 40
    w, W = make(dthip, oracle, rng, N, K, 6, 4096)
    X = rng.standard_normal((M, K)).astype(np.float16)
    for shape, given in (((M, K), (M, N)), ((M, K), (M, 1, N)), ((2, 3, K), (M, N)), ((2, 3, K), (M, 1, N))):
        out = torch.zeros(given, dtype=torch.float16, device="cuda")
        for got in (dthip.dense_multi(dev(X).view(shape), [w], [None], outs=[out]),
                    dthip.dense_post(dev(X).view(shape), [w], [None], [None], outs=[out])):
            assert got[0].shape == shape[:-1] + (N,) and got[0].data_ptr() == out.data_ptr()
        check(out.view(M, N).cpu().numpy(), X, W)


@pytest.mark.parametrize("kind", ["dense", "attention", "attention staged"])
def test_optional_scratch_is_not_insisted_on(dthip, oracle, monkeypatch, kind):
    """Where torch may not allocate any more, calls run uncut instead of failing: the scratch that cutting takes is
    optional, the staging of prepared keys is not."""
    import torch

    monkeypatch.delenv("DT_DENSE_SPLIT", raising=False)
    monkeypatch.delenv("DT_SDPA_KEY_SPLIT", raising=False)
    monkeypatch.setenv("DT_DENSE_EXPAND", "never")  # (the uncut launch on copies of the weights gives the uncut one's bits)
    rng = np.random.default_rng(9)
    L = dthip.lib()
    staged = 0
    if kind == "dense":
        M, K, N = 512, 5120, 5120
        w, _ = make(dthip, oracle, rng, N, K, 6, 4096)
        x, out = dev(rng.standard_normal((M, K)).astype(np.float16)), torch.empty((M, N), dtype=torch.float16, device="cuda")
        need = L.dt_dense_workspace_bytes(1, _groups(dthip, x, [w], [out])[0])
        call = lambda: dthip.dense_multi(x, [w], [None], outs=[out])
    else:
        B, S, H, D = 1, 1500, 4, 128
        q, k, v = (torch.randn((B, S, H, D), device="cuda").half() for _ in range(3))
        more = {} if kind == "attention" else {"gamma_k": [torch.ones(D, device="cuda").half()]}
        staged = B * S * H * D * 2 if more else 0
        need = L.dt_sdpa_workspace_bytes(B, H, H, D, S, S, int(bool(more)), 0)
        out = torch.empty((B, S, H, D), dtype=torch.float16, device="cuda")
        call = lambda: dthip.sdpa_segments([q], [k], [v], D ** -0.5, out=out, **more)
    assert need > (22 << 20) + staged  # (more than torch can have left over in a block)
    call()
    cut = out.clone()
    monkeypatch.setenv("DT_DENSE_SPLIT", "never")
    monkeypatch.setenv("DT_SDPA_KEY_SPLIT", "never")
    call()
    whole = out.clone()
    monkeypatch.delenv("DT_DENSE_SPLIT")
    monkeypatch.delenv("DT_SDPA_KEY_SPLIT")
    assert not torch.equal(cut, whole)
    print("scratch that cannot be had:", kind, flush=True)
    torch.cuda.empty_cache()
    total = torch.cuda.mem_get_info()[1]
    keep = torch.empty(staged, dtype=torch.uint8, device="cuda")
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (1 << 20)) / total)
    try:
        del keep  # room for the staging, and for no more
        with pytest.raises(torch.OutOfMemoryError):
            torch.empty(need, dtype=torch.uint8, device="cuda")
        out.zero_()
        call()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(out, whole)


def test_refused_dense_names_the_call_that_was_made(dthip, oracle):
    rng = np.random.default_rng(4)
    w = make(dthip, oracle, rng, 260, 64, 6, 4096)[0]
    x, gamma = dev(rng.standard_normal((5, 64)).astype(np.float16)), dev(np.ones(130, np.float16))
    with pytest.raises(dthip.DtError, match="dt_dense_qx_grouped_ws_f16"):
        dthip.dense_multi(x, [w], [None], epilogues=[dthip.HeadEpilogue(gamma, head_dim=130)])


@pytest.mark.parametrize("M", [1024, 16])  # the tiled kernel and the one for few rows
def test_gelu_erf_of_every_fp16_value(dthip, M):
    """The tail's GELU against float64 for every finite fp16 value, passed through a Dense with the identity; infinities and NaN
    through its bias.  Bound: the exponent is below 28 and p below 5, so the last rounding of p, times a, and that of the product are
    2^-22 x 5.8 + 2^-20 at most, 1.6e-6 in the result, those before them and the polynomial (5e-8) 4e-7, the exponential and the last
    two operations 2.4e-7; then fp16's own rounding.  (Past -5.8: 1.9e-8 instead of less.)"""
    import math

    import torch

    x = np.arange(1 << 16, dtype=np.uint16).view(np.float16).reshape(-1, M, 64)
    x = np.where(np.isfinite(x), x, np.float16(0))
    eye = dthip.QxTensor.from_f16(np.eye(64, dtype=np.float16))
    tail = [dthip.DensePost(dthip.ACT_GELU_ERF)]
    got = np.concatenate([dthip.dense_post(dev(p), [eye], [None], tail)[0].cpu().numpy() for p in x]).astype(np.float64).ravel()
    x = x.astype(np.float64).ravel()
    want = 0.5 * x * np.vectorize(math.erfc)(x * -math.sqrt(0.5))
    slack = 2.3e-6 * np.abs(want) + np.where(x < -5.8, 2e-8, 0.0)
    with np.errstate(over="ignore"):
        lo, hi = (want - slack).astype(np.float16).astype(np.float64), (want + slack).astype(np.float16).astype(np.float64)
    assert ((got >= lo) & (got <= hi)).all(), x[~((got >= lo) & (got <= hi))][:8]
    bias = torch.zeros(64, dtype=torch.float16, device="cuda")
    bias[:3] = torch.tensor([float("inf"), float("-inf"), float("nan")])
    out = dthip.dense_post(torch.zeros((M, 64), dtype=torch.float16, device="cuda"), [eye], [bias], tail)[0].cpu().numpy()
    assert (out[:, 0] == np.inf).all() and np.isnan(out[:, 1:3]).all() and (out[:, 3:] == 0).all()


@pytest.mark.parametrize("M,N,K", [
    (128, 128, 128),               # one whole tile
    (129, 136, 128), (127, 120, 192),  # a row / eight features into the next tile, and as much short of one
    (333, 652, 320),               # a width off the grid of 8 (it lies on that of 4)
    (300, 1001, 128),              # an odd one
    (200, 64, 320),                # half a tile of features
    (4100, 3080, 128), (4099, 3076, 192),  # 256 x 256 tiles
])
@pytest.mark.parametrize("q", [16, 6])
def test_dense_tails_at_the_edges(dthip, oracle, M, N, K, q):
    """Bias and every tail on slices that end inside a row of tiles: the tails act on the Dense's own results, bit for bit, and
    nothing behind a row or below the last one is written."""
    import torch

    rng = np.random.default_rng(M + N + K + q)
    X = rng.standard_normal((M, K)).astype(np.float16)
    w, W = make(dthip, oracle, rng, N, K, q, 4096)
    b = (rng.standard_normal(N) * 0.1).astype(np.float16)
    x, bias = dev(X), dev(b)

    def wide(dtype):  # [M, N] inside a buffer of sentinels, rows on the 16-byte grid
        buf = torch.full((M + 3, (N + 15) // 8 * 8), -77.0, dtype=dtype, device="cuda")
        return buf, buf[:M, :N]

    def untouched(buf):
        return bool((buf[M:] == -77).all()) and bool((buf[:, N:] == -77).all())

    print("dense tails at the edges", M, N, K, q, flush=True)
    buf, plain = wide(torch.float16)
    dthip.dense_multi(x, [w], [bias], outs=[plain])
    assert untouched(buf)
    check(plain.cpu().numpy(), X, W, b)
    rnd = lambda *s: dev(rng.standard_normal(s).astype(np.float16))
    other, gate = rnd(M, N), rnd(N)
    abuf, addend = wide(torch.float16)
    addend.copy_(other)
    res0 = rnd(M, N).float()
    half = plain.float()
    for post, want in ((dict(addend=addend), half + other.float()), (dict(multiplicand=addend), half * other.float()),
                       (dict(gate=gate), half * gate.float())):
        buf, y = wide(torch.float16)
        dthip.dense_post(x, [w], [bias], [dthip.DensePost(**post)], outs=[y])
        assert untouched(buf) and bool((y == want.half()).all()), post.keys()
    for g, product in ((gate, (half * gate.float()).half().float()), (gate.float() + 2.0 ** -13, half * (gate.float() + 2.0 ** -13))):
        rbuf, res = wide(torch.float32)
        res.copy_(res0)
        dthip.dense_post(x, [w], [bias], [dthip.DensePost(gate=g, residual=res, keep_output=False)])
        assert untouched(rbuf) and bool((res == res0 + product).all())


def test_cuts_where_copies_of_the_weights_do_not_fit(dthip, oracle, monkeypatch):
    """512 x 5120 -> 5120 runs on a 52 MB copy of its weight; where the device has no room for that, the call is cut along K as it is
    without copies, for which 27 MB do."""
    import torch

    monkeypatch.delenv("DT_DENSE_SPLIT", raising=False)
    monkeypatch.delenv("DT_DENSE_EXPAND", raising=False)
    rng = np.random.default_rng(10)
    M, K, N = 512, 5120, 5120
    w, _ = make(dthip, oracle, rng, N, K, 6, 4096)
    x, out = dev(rng.standard_normal((M, K)).astype(np.float16)), torch.empty((M, N), dtype=torch.float16, device="cuda")
    G, keep = _groups(dthip, x, [w], [out])
    copies, cut = dthip.lib().dt_dense_scratch_bytes(1, G), dthip.lib().dt_dense_workspace_bytes(1, G)
    assert copies >= 2 * N * K > cut > 0
    call = lambda: dthip.dense_multi(x, [w], [None])[0]
    print("scratch that takes cuts and no copies", flush=True)
    monkeypatch.setenv("DT_DENSE_EXPAND", "never")
    want = call()
    monkeypatch.setenv("DT_DENSE_SPLIT", "never")
    assert not torch.equal(call(), want)
    monkeypatch.delenv("DT_DENSE_SPLIT")
    monkeypatch.delenv("DT_DENSE_EXPAND")
    asked, scratch = [], dthip._scratch

    def tight(like, need, least):  # a device with room for `cut` bytes
        asked.append(need)
        return scratch(like, need if need <= cut else least, least)

    monkeypatch.setattr(dthip, "_scratch", tight)
    assert torch.equal(call(), want) and asked[0] == copies


@pytest.mark.parametrize("x_in,down_in", [(128, 64), (64, 128), (128, 128)])
def test_lora_in_fp32_refuses_widths_that_differ(dthip, oracle, x_in, down_in):
    """Inputs and down weights that are not as wide as the base weight (64) are refused before anything is launched on them."""
    import torch

    rng = np.random.default_rng(1)
    op = dthip.LoRADense(128, dthip.LoRANetworkConfiguration(4, 0.75, True))
    op.weight, op.bias = make(dthip, oracle, rng, 128, 64, 6, 4096)[0], None
    op.down = dthip.QxTensor(torch.zeros((4, down_in), device="cuda"), 16, 0, (4, down_in))
    op.up = dthip.QxTensor(torch.zeros((128, 4), device="cuda"), 16, 0, (128, 4))
    with pytest.raises(ValueError, match="input width"):
        op(torch.zeros((8, x_in), dtype=torch.float16, device="cuda"))
