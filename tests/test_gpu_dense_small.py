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
