"""GPU: a LoRA layer through dt_lora_dense_f16 -- the down projection, then the base projection with the branch in its epilogue --
against the Dense calls that it stands for, bit for bit: both round the intermediate, the branch and the sum to fp16 at the same
places (highPrecision: the branch and the sum), and sum in the same order wherever the base projection is laid out alike."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def layer_of(dthip, oracle, torch, rng, N, K, q, nib, rank, high, bias=True):
    if q == 16:
        w = dthip.QxTensor.from_f16((rng.standard_normal((N, K)) * 0.05).astype(np.float16))
    else:
        w = dthip.QxTensor.from_packed(oracle.synth_qx_weight(rng, N, K, q, nib, 0.05)[0], q, nib, (N, K))
    op = dthip.LoRADense(N, dthip.LoRANetworkConfiguration(rank, 0.75, high), noBias=not bias)
    op.weight, op.bias = w, torch.from_numpy((rng.standard_normal(N) * 0.1).astype(np.float16)).cuda() if bias else None
    pair = [(rng.standard_normal(s) * 0.1).astype(np.float32 if high else np.float16) for s in ((rank, K), (N, rank))]
    op.down, op.up = (dthip.QxTensor(torch.from_numpy(p).cuda(), 32 if high else 16, 0, p.shape) for p in pair)
    return op


def pair_of(dthip, op):
    c = op.configuration
    dn, up = (op.down, op.up) if c.highPrecision else op._padded()
    rank = c.rank if c.highPrecision else (c.rank + 15) // 16 * 16
    return dthip._LoraPair(dn.data.data_ptr(), up.data.data_ptr(), up.shape[1], rank, int(c.highPrecision), c.scale)


@pytest.mark.parametrize("M,N,K,q,nib,rank,high", [
    (65, 130, 64, 6, 512, 1, False), (129, 257, 128, 8, 4096, 17, False), (300, 512, 832, 4, 1024, 32, False),   # part of a wave's steps, of the waves
    (1100, 640, 1536, 6, 4096, 32, False), (257, 384, 1600, 5, 2048, 8, False), (4099, 256, 448, 16, 0, 16, False),  # whole rounds, a round and a share
    (4099, 300, 192, 7, 4096, 31, False), (16400, 128, 128, 6, 4096, 20, False), (70, 320, 192, 8, 256, 16, False),   # 32 rows a workgroup; blocks too small to copy
    (65, 130, 64, 6, 512, 1, True), (300, 257, 832, 4, 1024, 20, True), (1100, 512, 192, 8, 4096, 33, True),    # ranks of no multiple of 16, of 4
    (4099, 256, 320, 16, 0, 70, True), (16400, 130, 128, 6, 4096, 31, True), (129, 256, 256, 5, 512, 130, True),
])
def test_fused_layer_equals_its_dense_calls(dthip, oracle, torch_cuda, monkeypatch, M, N, K, q, nib, rank, high):
    torch = torch_cuda
    rng = np.random.default_rng(M + N + rank)
    op = layer_of(dthip, oracle, torch, rng, N, K, q, nib, rank, high, bias=rank % 2 == 0)
    wide = torch.from_numpy(rng.standard_normal((M, K + 8)).astype(np.float16)).cuda()
    x = wide[:, :K]  # rows further apart than they are long
    gate = torch.from_numpy((1 + 0.3 * rng.standard_normal(N)).astype(np.float16)).cuda()
    res = torch.from_numpy(rng.standard_normal((M, N)).astype(np.float32)).cuda()
    print("lora fused", M, N, K, q, nib, rank, high, flush=True)
    for split, expand in (("never", "never"), ("never", "always"), ("always", "always")):
        monkeypatch.setenv("DT_DENSE_SPLIT", split)
        monkeypatch.setenv("DT_DENSE_EXPAND", expand)

        def run(fused):
            with monkeypatch.context() as m:
                if not fused:
                    m.setattr(dthip.LoRADense, "_fused", lambda *a: None)
                r = res.clone()
                outs = [op(x), op(x, post=dthip.DensePost(dthip.ACT_GELU_TANH)), r]
                assert op(x, post=dthip.DensePost(gate=gate, residual=r, keep_output=False)) is None
                return outs

        assert type(op._fused(x, op.bias, None, None)) is list  # the call itself is what answers
        for got, want in zip(run(True), run(False)):
            if split == "never":
                assert torch.equal(got, want)
            else:  # (the Dense calls may lay the base projection out together with the down projection)
                assert float((got.float() - want.float()).norm() / want.float().norm()) <= 2.0 ** -11


@pytest.mark.parametrize("high", [False, True])
def test_scratch_of_a_fused_layer(dthip, oracle, torch_cuda, high):
    """All of the scratch, the intermediate's alone (the weight then stays packed: the same values), and less; replays of a graph."""
    torch = torch_cuda
    rng = np.random.default_rng(7)
    M, N, K, rank = 1200, 1024, 512, 24
    op = layer_of(dthip, oracle, torch, rng, N, K, 6, 4096, rank, high)
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float16)).cuda()
    L, pair, w = dthip.lib(), pair_of(dthip, op), dthip._QxWeight(op.weight.data.data_ptr(), 6, 4096, N * K)
    y = torch.empty((M, N), dtype=torch.float16, device="cuda")

    def call(scratch, size, rows=M):
        return L.dt_lora_dense_f16(torch.cuda.current_stream().cuda_stream, rows, K, x.data_ptr(), K, ctypes.byref(w), op.bias.data_ptr(),
                                   y.data_ptr(), N, None, ctypes.byref(pair), 0, scratch, size)

    size = lambda rows=M: L.dt_lora_dense_scratch_bytes(rows, K, x.data_ptr(), K, ctypes.byref(w), y.data_ptr(), N, None, ctypes.byref(pair))
    least = (M * pair.rank * (4 if high else 2) + 255) // 256 * 256
    assert size() >= least and size(32) == 0 and size(-1) == 0
    buf = torch.empty(size() + 256, dtype=torch.uint8, device="cuda")
    at = (buf.data_ptr() + 255) & ~255
    print("lora scratch", high, flush=True)
    want = op(x)
    for n in (size(), least):
        y.zero_()
        assert call(at, n) == 0 and torch.equal(y, want)
    assert call(at, least - 1) == -3 and call(None, 0) == -3 and call(at + 16, size()) == -1 and call(at, size(), 32) == -2
    pair.ld_up = pair.rank - 1
    assert call(at, size()) == -1
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = op(x)
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want) and torch.equal(op(x), want)
