"""GPU: the any-shape Dense where groups of waves share out K: K-tiles that do not divide among the groups, a last one of a few
columns, and both tile sizes, against float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [
    (33, 65, 129), (70, 96, 257), (31, 130, 641), (5, 33, 767), (64, 100, 1025), (231, 1001, 1000),  # 32 x 32: two groups, four, a tile short of both
    (515, 1001, 519), (700, 1001, 1153), (1020, 1010, 770),                                          # 64 x 64, four groups: 9, 19, 13 K-tiles
    (515, 1001, 511), (1030, 1030, 600),                                                             # ... and where one group has all of K
    (300, 1001, 1155), (297, 1030, 1051), (290, 1001, 1000), (512, 513, 1153),                       # 257 .. 512 small tiles: one or two groups on them, or 64 x 64
])
@pytest.mark.parametrize("q,nib", [(16, 0), (4, 1024), (8, 4096), (6, 50), (5, 8)])
def test_groups_of_waves_share_out_k(dthip, oracle, M, N, K, q, nib):
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    rng = np.random.default_rng(M + N + K)
    if q == 16:
        w = dthip.QxTensor.from_f16((rng.standard_normal((N, K)) * 0.05).astype(np.float16))
        W = w.data.view(N, K)
    else:
        w = dthip.QxTensor.from_packed(oracle.synth_qx_weight(rng, N, K, q, nib, 0.05)[0], q, nib, (N, K))
        W = w.dequantize()
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float16)).cuda()
    b = torch.from_numpy((rng.standard_normal(N) * 0.1).astype(np.float16)).cuda()
    print("dense any groups", M, N, K, q, nib, flush=True)
    got = dthip.dense_multi(x, [w], [b])[0].double()
    want = x.double() @ W.double().T + b.double()
    # sums in fp32 (K 2^-24 of the magnitudes at most), rounded to fp16 once
    sums = (K + 2) * 2.0 ** -24 * (x.double().abs() @ W.double().abs().T + b.double().abs())
    assert bool(((got - want).abs() <= sums + (want.abs() + sums) * 2.0 ** -11 + 2.0 ** -25).all())
