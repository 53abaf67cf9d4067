"""The Python operators' native way to the library (csrc/dt_host.cpp) against the way through ctypes: the same bits, outputs of the
same shapes, and the same refusals."""
import numpy as np
import pytest


def _weights(dthip, oracle, rng, N, K, q, nib, n=1):
    return [dthip.QxTensor.from_packed(oracle.synth_qx_weight(rng, N, K, q, nib)[0], q, nib, (N, K)) for _ in range(n)]


def test_native_module_leaves_other_calls_alone(dthip):
    """Runs without a GPU: host tensors, and arguments that are no tensors, are not its business."""
    import torch

    host = dthip._host()
    assert host is not None
    x = torch.zeros((4, 64), dtype=torch.float16)
    w = dthip.QxTensor(torch.zeros((8, 64), dtype=torch.float16), 16, 0, (8, 64))
    scratch = lambda *a: pytest.fail("nothing was to be asked for")
    for problem in ((x, [w], [None], None, None, None), (None, [w], [None], None, None, None), ("x",), 3):
        assert host.dense([problem], 0, scratch) is None
    assert host.dense([], 0, scratch) is None and host.dense() is None
    assert host.layernorm16(x, None, None, 1e-5) is None
    assert host.sdpa([x], [x], [x], 1.0, None, None, None, None, 1e-6, None, scratch) is None


@pytest.fixture
def both(dthip, monkeypatch):
    """call -> its results the native way, which has to have been taken (natively=False: nowhere), and the other one."""
    import torch

    def run(call, natively=True):
        native = dthip._host()
        assert native is not None
        answers = []

        class Watched:
            def __getattr__(self, name):
                def called(*args):
                    answers.append(getattr(native, name)(*args))
                    return answers[-1]

                return called

        monkeypatch.setattr(dthip, "_native", Watched())
        got = call()
        monkeypatch.undo()
        assert answers and all((a is not None) == natively for a in answers), answers
        monkeypatch.setattr(dthip, "_native", False)
        monkeypatch.setattr(dthip, "_host", lambda: None)
        want = call()
        monkeypatch.undo()
        assert dthip._native is native
        flat = lambda r: [r] if isinstance(r, torch.Tensor) or r is None else [t for e in r for t in flat(e)]
        got, want = flat(got), flat(want)
        assert len(got) == len(want)
        for a, b in zip(got, want):
            assert (a is None) == (b is None)
            if a is not None:
                assert a.shape == b.shape and a.dtype == b.dtype and a.stride() == b.stride() and torch.equal(a, b)
        return got

    return run


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(5, 128), (2, 40, 128), (3, 1, 128), (1, 128), (512, 1280)])
def test_dense_calls(dthip, oracle, both, shape):
    import torch

    rng = np.random.default_rng(sum(shape))
    K, N = shape[-1], 256
    M = int(np.prod(shape[:-1]))
    dev = lambda *s, t=torch.float16: torch.from_numpy(rng.standard_normal(s)).cuda().to(t)
    x, b = dev(*shape), dev(N)
    ws = _weights(dthip, oracle, rng, N, K, 6, 4096, 2)
    print("native dense", shape, flush=True)
    both(lambda: dthip.dense_multi(x, ws, [b]))
    both(lambda: dthip.dense_multi(x, ws, (None, b)))
    both(lambda: dthip.dense_multi(x, ws, [b], stream=torch.cuda.current_stream()))
    out = torch.zeros((M, 3 * N), dtype=torch.float16, device="cuda")
    got = both(lambda: dthip.dense_multi(x, ws, [b], outs=[out[:, :N], out[:, 2 * N:]]))
    assert got[0].data_ptr() == out.data_ptr()
    rot = dev(M + 3, 128)
    epi = [dthip.HeadEpilogue(dev(128), rot, 3), None]
    both(lambda: dthip.dense_multi(x, ws, [b, b], epilogues=epi))
    res = dev(*shape[:-1], N, t=torch.float32)
    posts = lambda: [dthip.DensePost(dthip.ACT_GELU_TANH, gate=b, scale=0.5, addend=torch.ones((M, N), device="cuda").half()),
                     dthip.DensePost(residual=res.clone(), keep_output=False, gate=b.float())]
    both(lambda: dthip.dense_post(x, ws, [b, None], posts()))

    def accumulated():
        p = posts()
        dthip.dense_post(x, ws, [b, None], p)
        return p[1].residual

    both(accumulated)
    both(lambda: dthip.dense_grouped([dict(x=x, weights=ws, biases=[b]), dict(x=x, weights=ws[:1], biases=[None], posts=[None])]))
    # (a copy is the other way's)
    for view in (x.transpose(0, 1) if x.dim() == 3 else x[:, ::1], dev(K, 70).t()):
        both(lambda: dthip.dense_multi(view, ws, [b]), natively=view.is_contiguous())


@pytest.mark.gpu
def test_attention_and_norm_calls(dthip, both):
    import torch

    g = torch.Generator(device="cuda").manual_seed(3)
    r = lambda *s: torch.randn(s, generator=g, device="cuda").half()
    q, k, v = [r(1, 70, 4, 64), r(1, 200, 4, 64)], [r(1, 70, 2, 64), r(1, 200, 2, 64)], [r(1, 70, 2, 64), r(1, 200, 2, 64)]
    gam, rot = [r(64), None], r(270, 64)
    print("native attention and norms", flush=True)
    both(lambda: dthip.sdpa_segments(q, k, v, 0.125))
    both(lambda: dthip.sdpa_segments(q, k, v, 0.125, gamma_q=gam, gamma_k=gam, rot_q=rot, rot_k=rot, eps=1e-5))
    out = torch.empty((1, 270, 2, 4, 64), dtype=torch.float16, device="cuda")
    both(lambda: dthip.sdpa_segments(q, k, v, 0.125, out=out[:, :, 1], stream=torch.cuda.current_stream()))
    x = r(3, 50, 320)
    both(lambda: dthip.layernorm16(x, r(320).fill_(1), None, 1e-5))
    both(lambda: dthip.layernorm16(x[0, :, :64].contiguous().expand(50, 64)))


@pytest.mark.gpu
def test_refusals_are_the_same(dthip, oracle, monkeypatch):
    import torch

    rng = np.random.default_rng(8)
    w = _weights(dthip, oracle, rng, 256, 128, 6, 4096)[0]
    x = torch.zeros((70, 128), dtype=torch.float16, device="cuda")
    layers = []
    for high in (False, True):  # (a base weight of fewer rows than the layer's)
        op = dthip.LoRADense(320, dthip.LoRANetworkConfiguration(16, 0.5, high))
        dtype = torch.float32 if high else torch.float16
        op.down, op.up = (dthip.QxTensor(torch.zeros(s, dtype=dtype, device="cuda"), 16, 0, s) for s in ((16, 128), (320, 16)))
        op.weight = w
        layers.append(op)
    calls = [lambda: layers[0](x), lambda: layers[1](x), lambda: dthip.dense_multi(x.float(), [w], [None]), lambda: dthip.dense_multi(x[:, :64], [w], [None]),
             lambda: dthip.dense_multi(x, [w], [None, None]), lambda: dthip.dense_multi(x, [w], [x.float()]),
             lambda: dthip.dense_multi(x, [w], [None], epilogues=[dthip.HeadEpilogue(x[0], x[:1])]),
             lambda: dthip.dense_multi(x, [w], [None], epilogues=[dthip.HeadEpilogue(x[0, :100].contiguous(), None, head_dim=100)]),
             lambda: dthip.dense_post(x, [w], [None], [dthip.DensePost(scale=0.0)]),
             lambda: dthip.dense_post(x, [w], [None], [dthip.DensePost(7)]),
             lambda: dthip.dense_post(x, [w], [None], [dthip.DensePost(gate=x[0])]),
             lambda: dthip.sdpa_segments([x.view(1, 70, 1, 128)], [x.view(1, 70, 1, 128)[:, :0]], [x.view(1, 70, 1, 128)[:, :0]], 1.0),
             lambda: dthip.sdpa_segments([x], [x], [x], 1.0),
             lambda: dthip.layernorm16(x, x[:, 0])]
    print("native refusals", flush=True)
    for i, call in enumerate(calls):
        seen = []
        for native in (True, False):
            with monkeypatch.context() as m:
                if not native:
                    m.setattr(dthip, "_native", False)
                    m.setattr(dthip, "_host", lambda: None)
                with pytest.raises(Exception) as e:
                    call()
                seen.append((type(e.value), str(e.value)))
        assert seen[0] == seen[1], (i, seen)
