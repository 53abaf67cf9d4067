"""CPU-side checks of the product's host logic and of the C-ABI library as a binary:
it loads, exports every declared symbol, and its pure-host entry points answer.
No kernel is launched here."""
import ctypes
import os
import re

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_library_exports_every_declared_symbol(dthip):
    header = open(os.path.join(ROOT, "include", "dt_hip.h")).read()
    declared = set(re.findall(r"\b(dt_[a-z0-9_]+)\s*\(", header))
    declared -= {"dt_status", "dt_stream"}
    assert declared == set(dthip.ABI_SYMBOLS), declared ^ set(dthip.ABI_SYMBOLS)
    L = ctypes.CDLL(dthip.LIB_PATH)
    for name in declared:
        assert hasattr(L, name), name


def test_host_only_entry_points(dthip, oracle):
    L = dthip.lib()
    assert b"gfx950" in L.dt_version()
    for q, nib in [(4, 512), (5, 1024), (6, 4096), (7, 64), (8, 16384)]:
        for count in (0, 1, nib - 1, nib, 5 * nib + 3, 3072 * 3072):
            assert dthip.qx_bytes(q, nib, count) == oracle.C.qx_bytes(q, nib, count)
    assert dthip.qx_bytes(3, 32, 10) == -1 and dthip.qx_bytes(9, 32, 10) == -1 and dthip.qx_bytes(6, 0, 10) == -1
    # workspace sizing: nothing needed for the plain call, K' for the fused prep (the queries are normalised and
    # rotated inside the kernel), O for the fused projection
    assert L.dt_sdpa_workspace_bytes(1, 24, 24, 128, 4608, 4608, 0, 0) == 0
    one = 4608 * 24 * 128 * 2
    assert L.dt_sdpa_workspace_bytes(1, 24, 24, 128, 4608, 4608, 1, 0) == one
    assert L.dt_sdpa_workspace_bytes(1, 24, 24, 128, 4608, 4608, 1, 1) == 2 * one


def test_key_split_planning(dthip, monkeypatch):
    """Which attention launches get room for the key-split form (host arithmetic; without a device the plan assumes
    256 compute units): launches of whole or several rounds of workgroups never, launches well under one round with
    enough key tiles do, and the environment knob overrides the estimate either way."""
    L = dthip.lib()
    ws = lambda B, H, D, Sq, Skv: L.dt_sdpa_workspace_bytes(B, H, H, D, Sq, Skv, 0, 0)
    monkeypatch.delenv("DT_SDPA_KEY_SPLIT", raising=False)
    assert ws(1, 24, 128, 4608, 4608) == 0         # 432 workgroups = 1.69 rounds: measured slower when split
    assert ws(1, 24, 128, 16896, 16896) == 0       # 6.19 rounds
    assert ws(2, 8, 40, 4096, 4096) == 0           # exactly one round
    assert ws(2, 8, 40, 4096, 77) == 0             # two key tiles: nothing to cut
    # 64 workgroups of 64 key tiles: one run per compute unit, two partial-result slots each, plus the counters
    slot = (128 // 32 * 16 * 512 + 2 * 512) * 4
    assert ws(1, 4, 128, 4096, 4096) == 256 + 2 * 256 * slot
    # 8 workgroups: at most 8 pieces per task
    assert ws(1, 1, 128, 2048, 16384) == 256 + 2 * 64 * slot
    assert ws(1, 1, 64, 2048, 16384) == 256 + 2 * 64 * (64 // 32 * 16 * 512 + 2 * 512) * 4
    monkeypatch.setenv("DT_SDPA_KEY_SPLIT", "never")
    assert ws(1, 4, 128, 4096, 4096) == 0
    monkeypatch.setenv("DT_SDPA_KEY_SPLIT", "always")
    assert ws(1, 24, 128, 4608, 4608) == 1792 + 2 * 256 * slot   # 432 counters (1728 bytes), 256-byte aligned
    assert ws(1, 1, 128, 1, 64) == 0                # a single key tile cannot be cut


def test_key_split_room_beside_full_rounds(dthip, monkeypatch):
    """Launches with full rounds in front bring a slot for every part of their cut tasks and no more."""
    L = dthip.lib()
    ws = lambda H, D, S: L.dt_sdpa_workspace_bytes(1, H, H, D, S, S, 0, 0)
    monkeypatch.delenv("DT_SDPA_KEY_SPLIT", raising=False)
    slot = lambda dp: (dp // 32 * 16 * 512 + 2 * 512) * 4
    assert ws(24, 128, 2637) == 256 + 8 * 8 * slot(128)    # 264 tasks: 8 of them in 8 parts
    assert ws(20, 128, 4096) == 2048 + 64 * 4 * slot(128)  # 320 tasks: 64 in 4 parts, whose counters fill 2 KB
    assert ws(33, 64, 2000) == 256 + 8 * 8 * slot(64)


def test_dense_tiles_that_cannot_share_a_compute_unit_are_cut(dthip, monkeypatch):
    """Two 128 x 128 tiles with per-row palettes of 128 entries (88 KB of LDS each) do not run side by side: 460 of them are
    two rounds, where 256 x 128 tiles that are cut take three quarters of the time.  With 64 entries they do, and nothing is cut."""
    monkeypatch.delenv("DT_DENSE_SPLIT", raising=False)
    addr = ctypes.addressof
    M, K, N, nib = 590, 7936, 5888, 8192

    def ws(q):
        W = (dthip._QxWeight * 2)(*[dthip._QxWeight(4096, q, nib, N * K)] * 2)  # (addresses are not looked at)
        Y, ldy = (ctypes.c_void_p * 2)(4096, 4096), (ctypes.c_int64 * 2)(N, N)
        G = (dthip._DenseGroup * 1)(dthip._DenseGroup(M, K, 4096, K, addr(W), 2, None, addr(Y), addr(ldy), None, None))
        return dthip.lib().dt_dense_workspace_bytes(1, G)

    assert ws(7) > 0
    assert ws(6) == 0


@pytest.mark.parametrize("M,K,N,n,q,nib,cut", [
    (571, 4288, 7872, 3, 7, 8192, False),   # 256 x 128 tiles would rewrite their palettes at every other K-tile: 342 us against 251
    (1000, 1792, 4096, 1, 7, 8192, False),  # 48 against 42
    (721, 7168, 2560, 1, 16, 0, False),     # plain fp16 weights on four pair slots: 52 against 46
    (2391, 2688, 1600, 1, 6, 4096, False),  # 66 against 61
    (512, 5120, 5120, 2, 5, 1024, True),    # 88 against 117
    (128, 5120, 1152, 1, 8, 16384, True),   # 37 against 90
])
def test_dense_is_cut_where_that_is_faster(dthip, monkeypatch, M, K, N, n, q, nib, cut):
    """The plan follows what cut and uncut launches measured (us at the right, cut first)."""
    monkeypatch.delenv("DT_DENSE_SPLIT", raising=False)
    addr = ctypes.addressof
    W = (dthip._QxWeight * n)(*[dthip._QxWeight(4096, q, nib, N * K)] * n)  # (addresses are not looked at)
    Y, ldy = (ctypes.c_void_p * n)(*[4096] * n), (ctypes.c_int64 * n)(*[N] * n)
    G = (dthip._DenseGroup * 1)(dthip._DenseGroup(M, K, 4096, K, addr(W), n, None, addr(Y), addr(ldy), None, None))
    assert (dthip.lib().dt_dense_workspace_bytes(1, G) > 0) == cut


@pytest.mark.parametrize("M,K,N,n,q,nib,copied", [
    (4608, 3072, 3072, 3, 6, 4096, True), (300, 3072, 3072, 1, 8, 16384, True), (2016, 1280, 5120, 1, 4, 512, True),
    (512, 5120, 5120, 2, 5, 1024, False),    # 100 MB of copies for 512 rows
    (4096, 320, 320, 1, 6, 4096, False),     # a second launch would cost more than it gains
    (4608, 3072, 3072, 1, 6, 64, False),     # small blocks are not copied, nor are plain weights
    (4608, 3072, 3072, 1, 16, 0, False), (64, 3072, 3072, 1, 6, 4096, False), (32760, 5120, 51200, 2, 6, 4096, False),
])
def test_dense_scratch_for_copies(dthip, monkeypatch, M, K, N, n, q, nib, copied):
    """dt_dense_scratch_bytes asks for room for fp16 copies of the weights where the launch is estimated to gain by them."""
    monkeypatch.delenv("DT_DENSE_SPLIT", raising=False)
    monkeypatch.delenv("DT_DENSE_EXPAND", raising=False)
    addr = ctypes.addressof
    W = (dthip._QxWeight * n)(*[dthip._QxWeight(4096, q, nib, N * K)] * n)  # (addresses are not looked at)
    Y, ldy = (ctypes.c_void_p * n)(*[4096] * n), (ctypes.c_int64 * n)(*[N] * n)
    G = (dthip._DenseGroup * 1)(dthip._DenseGroup(M, K, 4096, K, addr(W), n, None, addr(Y), addr(ldy), None, None))
    cut, scratch = dthip.lib().dt_dense_workspace_bytes(1, G), dthip.lib().dt_dense_scratch_bytes(1, G)
    assert (scratch >= n * N * K * 2) == copied
    assert copied or scratch == cut
    monkeypatch.setenv("DT_DENSE_EXPAND", "never")
    assert dthip.lib().dt_dense_scratch_bytes(1, G) == cut


@pytest.mark.parametrize("M,q,cut", [
    (3112, 8, True), (2791, 6, True),  # 238 against 269 on tiles of 192 x 256, 244 against 274
    (4608, 6, False),                  # 349 against 313 on tiles of 256 x 256
    (3112, 16, False),                 # no copies come between the launch and its X: 220 against 212
])
def test_dense_on_copies_with_an_x_that_left_the_cache(dthip, monkeypatch, M, q, cut):
    """Big tiles wait for an X of over 48 MB that was written ahead of the copies: a Flux block's second feed-forward projection (us in the
    block, cut first) is cut on 128 x 256 tiles, which have more on their way."""
    monkeypatch.delenv("DT_DENSE_SPLIT", raising=False)
    monkeypatch.delenv("DT_DENSE_EXPAND", raising=False)
    addr, K, N, nib = ctypes.addressof, 12288, 3072, 0 if q == 16 else 16384 if q == 8 else 4096
    W = (dthip._QxWeight * 1)(dthip._QxWeight(4096, q, nib, N * K))  # (addresses are not looked at)
    Y, ldy = (ctypes.c_void_p * 1)(4096), (ctypes.c_int64 * 1)(N)
    G = (dthip._DenseGroup * 1)(dthip._DenseGroup(M, K, 4096, K, addr(W), 1, None, addr(Y), addr(ldy), None, None))
    copies = 0 if q == 16 else N * K * 2
    scratch = dthip.lib().dt_dense_scratch_bytes(1, G)
    assert scratch >= copies and (scratch > copies) == cut


@pytest.mark.parametrize("M,K,N,n,q,nib,copied", [
    (91, 448, 64, 6, 8, 16384, False), (1215, 448, 128, 6, 8, 16384, False),  # 18.8 against 12.6, 19.3 against 13.8: the host
    (127, 1024, 3776, 3, 5, 1024, False), (346, 704, 3264, 6, 5, 1024, False),  # 27.7 against 19.7, 40.0 against 32.5: the copies
    (3795, 640, 192, 1, 5, 1024, True), (82, 640, 192, 2, 5, 1024, True), (203, 704, 1664, 1, 6, 4096, True),  # 11.1 against 15.6, 11.2 / 15.3, 12.7 / 16.2
])
def test_dense_copies_for_small_gains(dthip, monkeypatch, M, K, N, n, q, nib, copied):
    """Calls whose estimated gain is a few us: what the copies cost beyond the estimate grows with the weights and their size (us a call
    at the right, copied first)."""
    monkeypatch.delenv("DT_DENSE_SPLIT", raising=False)
    monkeypatch.delenv("DT_DENSE_EXPAND", raising=False)
    addr = ctypes.addressof
    W = (dthip._QxWeight * n)(*[dthip._QxWeight(4096, q, nib, N * K)] * n)  # (addresses are not looked at)
    Y, ldy = (ctypes.c_void_p * n)(*[4096] * n), (ctypes.c_int64 * n)(*[N] * n)
    G = (dthip._DenseGroup * 1)(dthip._DenseGroup(M, K, 4096, K, addr(W), n, None, addr(Y), addr(ldy), None, None))
    assert (dthip.lib().dt_dense_scratch_bytes(1, G) >= n * N * K * 2) == copied


@pytest.mark.parametrize("M,K,N", [(219, 1024, 7808), (103, 1536, 10240), (108, 1024, 7296)])
def test_dense_copies_where_palettes_would_be_looked_up_in_memory(dthip, monkeypatch, M, K, N):
    """A head epilogue needs tiles of 256 features, and q8 palettes of small blocks do not fit the LDS beside one: looked up in
    memory the launch takes four times what its estimate says (153 .. 221 us against 37 .. 51 on copies)."""
    monkeypatch.delenv("DT_DENSE_SPLIT", raising=False)
    monkeypatch.delenv("DT_DENSE_EXPAND", raising=False)
    addr, n = ctypes.addressof, 3
    W = (dthip._QxWeight * n)(*[dthip._QxWeight(4096, 8, 2048, N * K)] * n)  # (addresses are not looked at)
    Y, ldy = (ctypes.c_void_p * n)(*[4096] * n), (ctypes.c_int64 * n)(*[N] * n)
    epi = (dthip._HeadEpilogue * n)(*[dthip._HeadEpilogue(4096, None, 0, 1e-6, 128)] * n)
    G = (dthip._DenseGroup * 1)(dthip._DenseGroup(M, K, 4096, K, addr(W), n, None, addr(Y), addr(ldy), addr(epi), None))
    assert dthip.lib().dt_dense_scratch_bytes(1, G) >= n * N * K * 2


@pytest.mark.parametrize("split", ["never", "always", ""])
def test_dense_copies_do_not_hang_on_the_knob_for_cuts(dthip, monkeypatch, split):
    monkeypatch.delenv("DT_DENSE_EXPAND", raising=False)
    monkeypatch.setenv("DT_DENSE_SPLIT", split)
    addr, M, K, N, n = ctypes.addressof, 4608, 3072, 3072, 3
    W = (dthip._QxWeight * n)(*[dthip._QxWeight(4096, 6, 4096, N * K)] * n)  # (addresses are not looked at)
    Y, ldy = (ctypes.c_void_p * n)(*[4096] * n), (ctypes.c_int64 * n)(*[N] * n)
    G = (dthip._DenseGroup * 1)(dthip._DenseGroup(M, K, 4096, K, addr(W), n, None, addr(Y), addr(ldy), None, None))
    assert dthip.lib().dt_dense_scratch_bytes(1, G) >= n * N * K * 2


@pytest.mark.parametrize("K,N,n,q,nib,copied", [
    (5120, 5120, 1, 6, 4096, True), (12288, 3072, 1, 8, 16384, True),  # 52 and 75 MB
    (10368, 6144, 2, 5, 1024, False),                                  # 255 MB
])
def test_dense_scratch_for_copies_with_few_rows(dthip, monkeypatch, K, N, n, q, nib, copied):
    """Few rows copy weights that the memory-side cache holds, larger ones do not."""
    monkeypatch.delenv("DT_DENSE_SPLIT", raising=False)
    monkeypatch.delenv("DT_DENSE_EXPAND", raising=False)
    addr = ctypes.addressof
    for M in (400, 512, 640):
        W = (dthip._QxWeight * n)(*[dthip._QxWeight(4096, q, nib, N * K)] * n)  # (addresses are not looked at)
        Y, ldy = (ctypes.c_void_p * n)(*[4096] * n), (ctypes.c_int64 * n)(*[N] * n)
        G = (dthip._DenseGroup * 1)(dthip._DenseGroup(M, K, 4096, K, addr(W), n, None, addr(Y), addr(ldy), None, None))
        assert (dthip.lib().dt_dense_scratch_bytes(1, G) >= n * N * K * 2) == copied, M


@pytest.mark.parametrize("M,K,N,q,nib,captured,otherwise", [
    (64, 13824, 5120, 6, 4096, True, True), (64, 5120, 5120, 8, 16384, True, False), (64, 12288, 3072, 8, 16384, True, False),
    (32, 13824, 5120, 6, 4096, False, False), (48, 3072, 3072, 6, 4096, False, False), (64, 13824, 5120, 16, 0, False, False),
    (1024, 12288, 3072, 6, 128, True, True), (1024, 3072, 3072, 6, 256, True, False), (4608, 1280, 1280, 6, 256, False, False),
    (933, 2816, 1152, 6, 256, True, False), (4608, 2048, 1280, 6, 256, True, False), (1300, 1984, 640, 6, 256, False, False),
    (4608, 3072, 3072, 6, 4096, False, False), (512, 5120, 5120, 5, 1024, False, False),  # copied: one launch
])
def test_lora_down_projection_beside_the_base(dthip, monkeypatch, M, K, N, q, nib, captured, otherwise):
    """The down projection gets a stream of its own where it is long and not part of the base projection's launch."""
    monkeypatch.delenv("DT_DENSE_SPLIT", raising=False)
    monkeypatch.delenv("DT_DENSE_EXPAND", raising=False)
    w = dthip.QxTensor(None, q, nib, (N, K))
    assert dthip.LoRADense._down_beside_base(M, K, w, 64, lambda: True) == captured
    assert dthip.LoRADense._down_beside_base(M, K, w, 64, lambda: False) == otherwise


def test_gelu_erf_polynomial_is_as_exact_as_erfcf():
    """The tail's GELU in the kernel's fp32 steps, over every fp16 value from -5.8 on: no further from float64 than with the library
    function (9.7e-8 rms, 2.49e-6 at most, measured on the GPU).  The steps leave out the exponential's own last bit."""
    import math

    src = open(os.path.join(ROOT, "draw-things-community_amd", "csrc", "dt_dense_kernel.h")).read()
    coef = re.search(r"kP\[11\] = \{([^}]*)\}", src).group(1)
    c = [np.float32(float.fromhex(t.strip().rstrip("f"))) for t in coef.split(",")]
    x = np.arange(1 << 16, dtype=np.uint16).view(np.float16)
    x = x[np.isfinite(x)].astype(np.float32)
    x = x[(x >= -5.8) & (x != 0)]
    fma = lambda u, v, w: (u.astype(np.float64) * v.astype(np.float64) + np.asarray(w, np.float64)).astype(np.float32)
    a = np.minimum(np.abs(x), np.float32(5.8))
    p = np.full_like(a, c[10])
    for k in range(9, -1, -1):
        p = fma(p, a, c[k])
    e = np.exp2((p * a).astype(np.float64)).astype(np.float32)
    got = (np.float32(0.5) * fma(-a, e, x + np.abs(x))).astype(np.float64)
    want = np.array([0.5 * v * math.erfc(-v * math.sqrt(0.5)) for v in x.astype(np.float64)])
    rel = np.abs(got - want) / np.abs(want)
    assert np.sqrt((rel ** 2).mean()) <= 9e-8 and rel.max() <= 2.2e-6


def test_rows_that_need_no_workspace(dthip):
    """The operators do not ask for workspace up to the rows that the library's streaming kernel takes: one number, twice."""
    import re

    header = open(os.path.join(ROOT, "draw-things-community_amd", "csrc", "dt_dense_rows.h")).read()
    assert dthip._ROWS_MAX == int(re.search(r"kRowsMax = (\d+);", header).group(1))


def test_eager_lora_layers_are_decided_without_the_library(dthip, monkeypatch):
    """Its answer takes the host 6 us, which layers that wait for the host do not have; what it copies at most is stated twice."""
    csrc = os.path.join(ROOT, "draw-things-community_amd", "csrc")
    text = lambda name: open(os.path.join(csrc, name)).read()
    assert dthip._COPIED_NIB == int(re.search(r"kDepalMinNib = (\d+);", text("dt_depalettize.h")).group(1))
    assert dthip._COPIED_BYTES >> 20 == int(re.search(r"kDenseMaxExpand = \(size_t\)(\d+) << 20;", text("dt_dense.hip")).group(1))
    monkeypatch.setattr(dthip, "lib", lambda: pytest.fail("the library was asked"))
    for M, K, q, nib, beside in ((2800, 3072, 6, 4096, False), (4608, 12288, 8, 16384, False), (1024, 12288, 6, 256, True),
                                 (64, 13824, 6, 4096, True), (64, 3072, 6, 4096, False)):
        assert dthip.LoRADense._down_beside_base(M, K, dthip.QxTensor(None, q, nib, (512, K)), 64, lambda: False) == beside


def test_missing_library_fails_loudly(dthip, monkeypatch):
    monkeypatch.setattr(dthip, "_lib", None)
    monkeypatch.setattr(dthip, "LIB_PATH", os.path.join(ROOT, "no_such_dir", "libdthip.so"))
    with pytest.raises(RuntimeError, match="no CPU or PyTorch fallback"):
        dthip.lib()


def test_native_calls_that_do_not_load(dthip, monkeypatch, tmp_path):
    """A module built against another torch: said once, and every call goes through ctypes, the first one too."""
    import warnings

    (tmp_path / "_dthost.so").write_bytes(b"no library")
    monkeypatch.setattr(dthip, "_HERE", str(tmp_path))
    monkeypatch.setattr(dthip, "_native", None)
    with pytest.warns(RuntimeWarning, match="_dthost.so does not load"):
        assert dthip._host() is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert dthip._host() is None


def test_native_calls_are_seen_whole(dthip, monkeypatch):
    """Threads that come while the module is being loaded find nothing, or all of it."""
    import importlib.util
    import types

    seen = []

    class Loader:
        create_module = staticmethod(lambda spec: None)

        @staticmethod
        def exec_module(module):
            seen.append(dthip._native)
            module.classes = lambda *c: seen.append(dthip._native)

    spec = lambda name, path: importlib.util.spec_from_loader(name, Loader())
    monkeypatch.setattr(importlib.util, "spec_from_file_location", spec)
    monkeypatch.setattr(dthip, "_native", None)
    host = dthip._host()
    assert isinstance(host, types.ModuleType) and host is dthip._native and not any(seen) and len(seen) == 2


def test_library_builds_without_python(dthip):
    """What a C, C++ or Swift host runs names neither Python nor torch; the package's own build makes its native calls as well."""
    import subprocess

    recipe = lambda *goals: subprocess.run(["make", "-n", "-B", "-C", dthip.CSRC, "PYTHON=no-such-python", *goals], capture_output=True, text=True,
                                           check=True).stdout
    plain = recipe()
    assert "libdthip.so" in plain and "dt_cpp_check" in plain
    assert "no-such-python" not in plain and "torch" not in plain
    assert "no-such-python" in recipe("python") and "libdthip.so" in recipe("python")


@pytest.mark.parametrize("q", [4, 5, 6, 7, 8])
def test_host_packer_matches_oracle(dthip, oracle, q):
    rng = np.random.default_rng(q)
    for n in (0, 1, 7, 8, 9, 31, 32, 33, 1000):
        idx = rng.integers(0, 1 << q, size=n, dtype=np.uint8)
        assert np.array_equal(dthip.pack_indices(q, idx), oracle.C.pack_indices(q, idx))
    for nib, count in [(32, 0), (32, 31), (32, 96), (64, 64 * 3 + 5), (512, 512 * 4)]:
        nblocks = (count + nib - 1) // nib
        pal = (rng.standard_normal((nblocks, 1 << q)) * 0.02).astype(np.float16)
        idx = rng.integers(0, 1 << q, size=count, dtype=np.uint8)
        assert np.array_equal(dthip.pack_qx(q, nib, pal, idx), oracle.C.palettize_pack(q, nib, pal, idx))


def test_rotary_tables_match_oracle(dthip, oracle):
    a = dthip.Flux1RotaryPositionEmbedding(6, 5, 4, channels=128)
    assert np.array_equal(a, oracle.C.rope_flux(6, 5, 4, 128))
    a = dthip.Flux1RotaryPositionEmbedding(4, 4, 2, referenceSizes=[(2, 3), (3, 2), (5, 1)], channels=128)
    assert np.array_equal(a, oracle.C.rope_flux(4, 4, 2, 128, ref_sizes=[(2, 3), (3, 2), (5, 1)]))
    a = dthip.Flux1RotaryPositionEmbedding(3, 7, 0, channels=64)
    assert np.array_equal(a, oracle.C.rope_flux(3, 7, 0, 64))
    w = dthip.WanRotaryPositionEmbedding(4, 5, 3, channels=128)
    assert np.array_equal(w, oracle.C.rope_wan(4, 5, 3, 128))


def test_instruction_counts(dthip, oracle):
    assert dthip.DenseInstructionCount(4608, 3072, 9216) == oracle.C.dense_instruction_count(4608, 3072, 9216)
    assert dthip.ScaledDotProductAttentionInstructionCount(1, 24, 128, 4608, 4608) == \
        oracle.C.sdpa_instruction_count(1, 24, 128, 4608, 4608)


def test_operator_surface_argument_checks(dthip):
    with pytest.raises(dthip.DtError):
        dthip.ScaledDotProductAttention(scale=1.0, isCausal=True)
    d = dthip.Dense(count=8, noBias=True, name="x_q")
    with pytest.raises(RuntimeError, match="weight not loaded"):
        d(None)


def test_header_is_plain_c_and_links(dthip, tmp_path):
    """include/dt_hip.h is what a C (or Swift, through the module map) caller sees: it must compile as C99 on its
    own, and a C program linked against libdthip.so must be able to call the host-only entry points."""
    import shutil
    import subprocess

    cc = shutil.which("gcc") or shutil.which("cc")
    if cc is None:
        pytest.skip("no C compiler")
    src = tmp_path / "abi.c"
    src.write_text(r'''
#include "dt_hip.h"
#include <stdio.h>
#include <string.h>
int main(void) {
  dt_qx_weight w; dt_view4 v; dt_seq_segment s; dt_head_epilogue e; dt_dense_post p; dt_dense_group g;
  memset(&w, 0, sizeof w); memset(&v, 0, sizeof v); memset(&s, 0, sizeof s); memset(&e, 0, sizeof e);
  memset(&p, 0, sizeof p); memset(&g, 0, sizeof g);
  (void)w; (void)v; (void)s; (void)e; (void)p; (void)g;
  /* every entry point is declared with C linkage and takes only plain pointers and sizes */
  typedef void (*fn_t)(void);
  fn_t fns[] = {FNS};
  if (sizeof fns / sizeof fns[0] != NFNS) return 2;
  if (DT_OK != 0 || DT_INVALID != -1 || DT_NO_KERNEL != -2 || DT_OOM != -3) return 3;  /* ccv's exec status values */
  printf("%s %lld %zu\n", dt_version(), (long long)dt_qx_bytes(6, 4096, 3072LL * 3072),
         dt_sdpa_workspace_bytes(1, 24, 24, 128, 4608, 4608, 1, 0));
  return 0;
}
''')
    inc = os.path.join(ROOT, "include")
    text = src.read_text().replace("FNS", ", ".join(f"(fn_t){name}" for name in dthip.ABI_SYMBOLS), 1)
    src.write_text(text.replace("NFNS", str(len(dthip.ABI_SYMBOLS))))
    subprocess.check_call([cc, "-std=c99", "-Wall", "-Werror", "-pedantic", "-fsyntax-only", "-I", inc, str(src)])
    libdir = os.path.dirname(dthip.LIB_PATH)
    exe = tmp_path / "abi"
    subprocess.check_call([cc, "-std=c99", "-I", inc, str(src), "-o", str(exe), "-L", libdir, "-ldthip",
                           "-Wl,-rpath," + libdir, "-Wl,-rpath,/opt/rocm/lib"])
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stderr
    ver, qx, ws = out.stdout.split()[-3:] if len(out.stdout.split()) >= 3 else (None, None, None)
    assert "gfx950" in out.stdout
    assert int(qx) == dthip.qx_bytes(6, 4096, 3072 * 3072)
    assert int(ws) == 4608 * 24 * 128 * 2


def test_cpp_operator_mirror_compiles(dthip, tmp_path):
    """include/dt_hip.hpp (the C++ operator objects above the C ABI) compiles on its own as C++17 with warnings as
    errors, and the check program built from it exists beside the library after a build."""
    import shutil
    import subprocess

    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    src = tmp_path / "mirror.cpp"
    src.write_text('#include "dt_hip.hpp"\nint main() { dt::Dense d(8, true); return d.count == 8 ? 0 : 1; }\n')
    subprocess.check_call([cxx, "-std=c++17", "-Wall", "-Wextra", "-Werror", "-fsyntax-only", "-I",
                           os.path.join(ROOT, "include"), str(src)])
    assert os.path.exists(os.path.join(os.path.dirname(dthip.LIB_PATH), "dt_cpp_check"))


def test_any_shape_dense_stays_inside_its_buffers(tmp_path):
    """The any-shape Dense kernel's index arithmetic, walked on the host for every tile, row and run of ragged shapes:
    every palette slot that a thread looks up is one that the tile has loaded into its LDS, which holds them, every word
    lies in the packed buffer, and a run starts at the weight it stands for."""
    import shutil
    import subprocess

    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    src = tmp_path / "walk.cpp"
    src.write_text(r'''
#include <cstdio>
#include <cstdlib>
#include "dt_dense_any_index.h"
using namespace dt;
#define CHECK(c) do { if (!(c)) { printf("%s: n %lld k %lld q %d nib %d tile %d row %lld k0 %lld\n", #c, (long long)n, (long long)k, q, nib, bt, (long long)row, (long long)k0); return 1; } } while (0)
static int walk(int64_t n, int64_t k, int q, int nib, int bt) {
  const int bka = 4096 / bt, words = (q + 1) / 2 + 1;
  const QxLayout lay = make_layout(q, nib);
  const int64_t bytes = qx_total_bytes(q, nib, n * k), last = (n * k - 1) / nib;
  const bool shared = any_pal_shared(bt, k, q, nib), by_words = any_by_words(words, bytes, nib);
  for (int64_t n0 = 0; n0 < n; n0 += bt) {
    const AnyBlocks held = any_blocks(n0, bt, n, k, nib);
    for (int tr = 0; tr < bt; tr++)
      for (int run = 0; run < bka / 16; run++) {
        const int64_t row = any_row(n0 + tr, n);
        int64_t k0 = run * 16;
        CHECK(held.first >= 0 && held.first + held.count - 1 <= last && row >= 0 && row < n);
        CHECK(!shared || (held.count << q) * 2 <= kAnyPalBytes);
        AnyCursor c = any_cursor(row, k, run * 16, nib);
        for (int64_t kt = 0; kt * bka < k; kt++, k0 += bka, any_advance(c, bka, nib)) {
          const int left = any_run(k0, k), head = any_run_head(c, left, nib);
          CHECK(left >= 0 && left <= 16 && head <= left && (left == 0 || head > 0));
          if (left == 0) continue;  // (such a lane looks at the tile's first palette)
          CHECK(c.blk * nib + c.r == row * k + k0);
          if (!by_words) continue;
          CHECK(c.blk >= held.first && c.blk < held.first + held.count);
          int64_t at = any_words_at(index_byte_offset(lay, c.blk, c.r), words, bytes);
          CHECK(at >= 0 && at + 4 * words <= bytes);
          if (head < left) {
            CHECK(c.blk + 1 < held.first + held.count);
            at = any_words_at(any_rest_bit(lay, c, head) >> 3, words, bytes);
            CHECK(at >= 0 && at + 4 * words <= bytes);
          }
        }
      }
  }
  return 0;
}
int main(int argc, char** argv) {
  for (int i = 1; i + 3 < argc; i += 4)
    for (int bt = 32; bt <= 64; bt += 32)
      if (walk(atoll(argv[i]), atoll(argv[i + 1]), atoi(argv[i + 2]), atoi(argv[i + 3]), bt)) return 1;
  return 0;
}
''')
    exe = tmp_path / "walk"
    subprocess.check_call([cxx, "-std=c++17", "-O2", "-Wall", "-Wextra", "-Werror", "-I",
                           os.path.join(ROOT, "draw-things-community_amd", "csrc"), str(src), "-o", str(exe)])
    # N, K, index width, block size: the shapes of the GPU's parity test, and random ones
    shapes = [(1, 1, 6, 1), (31, 100, 6, 32), (32, 128, 5, 24), (65, 129, 7, 4096), (40, 16, 4, 512), (1001, 1000, 8, 16384),
              (90, 2500, 8, 512), (1400, 200, 6, 4096), (1470, 77, 4, 64), (33, 2560, 8, 16384), (97, 5121, 6, 4096)]
    rng = np.random.default_rng(88)
    for _ in range(300):
        n, k, nib = (int(np.exp(rng.uniform(np.log(lo), np.log(hi)))) for lo, hi in ((1, 600), (1, 1500), (1, 20000)))
        shapes.append((n, k, int(rng.integers(4, 9)), nib))
    out = subprocess.run([str(exe)] + [str(v) for s in shapes for v in s], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr


@pytest.mark.parametrize("high", [False, True])
@pytest.mark.parametrize("current", [0, 1])
def test_lora_layer_runs_where_its_input_is(dthip, monkeypatch, high, current):
    """x on the second device, whichever is current: the layer is enqueued on the current stream of x's device, made current for the
    call where its device is not.  (The tensors are host ones that say they are there, the native call a stand-in.)"""
    import contextlib

    import torch

    class There(torch.Tensor):
        is_cuda = property(lambda self: True)
        device = property(lambda self: torch.device("cuda", 1))

    entered, calls = [], []

    @contextlib.contextmanager
    def on(stream):
        entered.append(stream)
        yield
        entered.pop()

    class Host:
        @staticmethod
        def lora(*args):
            calls.append(list(entered))
            return ["out"]

    monkeypatch.setattr(dthip, "_native", Host)
    monkeypatch.setattr(dthip, "_on", on)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: current)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: ("stream of", str(device)))
    dtype = torch.float32 if high else torch.float16
    op = dthip.LoRADense(128, dthip.LoRANetworkConfiguration(16, 0.5, high))
    op.weight = dthip.QxTensor(torch.zeros((128, 64), dtype=torch.float16), 16, 0, (128, 64))
    op.down, op.up = (dthip.QxTensor(torch.zeros(s, dtype=dtype), 16, 0, s) for s in ((16, 64), (128, 16)))
    x = torch.zeros((80, 64), dtype=torch.float16).as_subclass(There)
    assert op(x) == "out" and op(x, stream="mine") == "out"
    assert calls == [[] if current == 1 else [("stream of", "cuda:1")], ["mine"]]


@pytest.mark.parametrize("high", [False, True])
@pytest.mark.parametrize("rows", [64, 192])
def test_lora_layer_refuses_a_weight_of_other_rows_than_count(dthip, monkeypatch, high, rows):
    """Before anything is enqueued: the base projection's result and the branch have to be of one width."""
    import torch

    class Host:
        @staticmethod
        def lora(*args):
            return ["out"]

        @staticmethod
        def dense(*args):
            return [["plain"]]

    monkeypatch.setattr(dthip, "_native", Host)
    dtype = torch.float32 if high else torch.float16
    op = dthip.LoRADense(128, dthip.LoRANetworkConfiguration(16, 0.5, high))
    op.weight = dthip.QxTensor(torch.zeros((rows, 64), dtype=torch.float16), 16, 0, (rows, 64))
    op.down, op.up = (dthip.QxTensor(torch.zeros(s, dtype=dtype), 16, 0, s) for s in ((16, 64), (128, 16)))
    x = torch.zeros((80, 64), dtype=torch.float16)
    with pytest.raises(ValueError, match="rows"):
        op(x)
    op.configuration.scale = 0  # no branch: a plain Dense, of whatever rows its weight has
    assert op(x) == "plain"


@pytest.mark.parametrize("M,K,N,rank,fused", [
    (1334, 832, 2816, 128, True), (2182, 384, 3008, 96, True), (3844, 960, 4096, 128, True), (1331, 1088, 3072, 64, True),  # 42 against 44, 49 / 53, 111 / 121
    (1331, 1088, 3072, 128, False), (2305, 1536, 1856, 128, False), (1617, 320, 3712, 128, False), (4371, 640, 4672, 96, False),  # 65 / 51, 79 / 69, 57 / 50, 143 / 127
])
def test_lora_layers_in_high_precision_that_run_as_calls(dthip, monkeypatch, M, K, N, rank, fused):
    """Many ranks stay Dense calls where few compute units have a second tile and are alone with the fp32 products of its epilogue (us, in
    one call first)."""
    monkeypatch.delenv("DT_DENSE_SPLIT", raising=False)
    monkeypatch.delenv("DT_DENSE_EXPAND", raising=False)
    w = dthip._QxWeight(4096, 6, 4096, N * K)  # (addresses are not looked at)
    pair = dthip._LoraPair(4096, 4096, rank, rank, 1, 0.5)
    got = dthip.lib().dt_lora_dense_scratch_bytes(M, K, 4096, K, ctypes.byref(w), 4096, N, None, ctypes.byref(pair))
    assert (got > 0) == fused
