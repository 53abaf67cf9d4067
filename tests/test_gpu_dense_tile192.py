"""GPU: tiles of 192 tokens, which plain fp16 weights and fp16 copies take where they fill the chip better than others.  Every tile sums
over K in the same order, so a launch that is not cut has to give the bits of the same rows in calls of few enough of them to run on other tiles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def on_192_tokens(torch, call):
    """call(), whose Dense has to be a launch of that tile."""
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as seen:
        out = call()
        torch.cuda.synchronize()
    names = [e.key for e in seen.key_averages() if "dense_" in e.key]
    assert len(names) == 1 and ", 192, 256, " in names[0], names
    return out


# (rows and features at the ends of tiles and off them, odd ones too; sizes at which the estimates take the tile)
@pytest.mark.parametrize("M,N,K,q", [(3265, 3584, 512, 16), (2304, 5120, 2048, 16), (3200, 3839, 1984, 16), (2113, 4991, 1984, 16), (4108, 2816, 2048, 8),
                                     (4097, 2687, 1984, 8), (1900, 5504, 2176, 6), (1901, 5503, 2176, 6)])
def test_tiles_of_192_tokens(dthip, oracle, monkeypatch, M, N, K, q):
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    rng = np.random.default_rng(M + N)
    if q == 16:
        w = dthip.QxTensor.from_f16((rng.standard_normal((N, K)) * 0.05).astype(np.float16))
    else:
        w = dthip.QxTensor.from_packed(oracle.synth_qx_weight(rng, N, K, q, 4096, 0.05)[0], q, 4096, (N, K))
    wf = w.dequantize() if q != 16 else w.data.view(N, K)
    dev = lambda a: torch.from_numpy(a.astype(np.float16)).cuda()
    x, b, gate = dev(rng.standard_normal((M, K))), dev(rng.standard_normal(N) * 0.1), dev(1 + 0.3 * rng.standard_normal(N))
    res = torch.from_numpy(rng.standard_normal((M, N)).astype(np.float32)).cuda()
    print("dense 192", M, N, K, q, flush=True)
    monkeypatch.setenv("DT_DENSE_SPLIT", "never")  # (what is cut along K adds its shares up otherwise)
    ends = [M * i // (M // 100) for i in range(M // 100 + 1)]  # 100 .. 110 rows each: more than the kernel for few rows takes
    parts = list(zip(ends, ends[1:]))
    plain = on_192_tokens(torch, lambda: dthip.dense_multi(x, [w], [b])[0])
    want = torch.cat([dthip.dense_multi(x[i:j], [dthip.QxTensor(wf, 16, 0, (N, K))], [b])[0] for i, j in parts])
    assert torch.equal(plain, want)
    exact = x[:64].double() @ wf.double().T + b.double()
    assert float((plain[:64].double() - exact).abs().max()) <= 2.0 ** -10 * float(exact.abs().max())
    r, rw = res.clone(), res.clone()
    got = on_192_tokens(torch, lambda: dthip.dense_post(x, [w], [b], [dthip.DensePost(dthip.ACT_GELU_TANH, gate=gate, residual=r)])[0])
    want = torch.cat([dthip.dense_post(x[i:j], [dthip.QxTensor(wf, 16, 0, (N, K))], [b],
                                       [dthip.DensePost(dthip.ACT_GELU_TANH, gate=gate, residual=rw[i:j])])[0] for i, j in parts])
    assert torch.equal(got, want) and torch.equal(r, rw)
    if N % 128 == 0 and K > 1024:  # norm and rotation fused (which short K leaves on 256 x 256)
        gamma, rot = dev(1 + 0.1 * rng.standard_normal(128)), dev(rng.standard_normal((M + 3, 128)))
        epi = lambda p: dthip.HeadEpilogue(gamma, rot, p, 1e-6, 128)
        got = on_192_tokens(torch, lambda: dthip.dense_multi(x, [w], [b], epilogues=[epi(3)])[0])
        want = torch.cat([dthip.dense_multi(x[i:j], [dthip.QxTensor(wf, 16, 0, (N, K))], [b], epilogues=[epi(3 + i)])[0] for i, j in parts])
        assert torch.equal(got, want)
