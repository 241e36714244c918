"""Host-side layout helpers of the fused kernels (CPU): the weight-row regrouping of the SwiGLU GEMMs, the pair-mask
scope, and the kernels' own index maps and 32-bit buffer ranges built on the host."""

from __future__ import annotations

import pytest
import torch


def test_group_swiglu_rows():
    """Block q of the grouped matrix is [W_0 rows 32q..32q+31; W_1 same (; W_2 same)], every source row once."""
    from boltz_mlx_amd import kernels as K

    H, Kd = 96, 5
    ws = [torch.arange(H * Kd, dtype=torch.float32).view(H, Kd) + 1000 * p for p in range(3)]
    g3 = K.group_swiglu3_rows(*ws)
    assert g3.shape == (3 * H, Kd)
    for q in range(H // 32):
        for p in range(3):
            assert torch.equal(g3[96 * q + 32 * p:96 * q + 32 * (p + 1)], ws[p][32 * q:32 * (q + 1)])
    g2 = K.group_swiglu_rows(ws[0], ws[1])
    for q in range(H // 32):
        assert torch.equal(g2[64 * q:64 * q + 32], ws[0][32 * q:32 * (q + 1)])
        assert torch.equal(g2[64 * q + 32:64 * (q + 1)], ws[1][32 * q:32 * (q + 1)])
    assert torch.equal(torch.sort(g3.flatten())[0], torch.sort(torch.cat(ws).flatten())[0])


def test_pair_mask_scope_extent_and_transpose():
    """mask_transposed: nothing is kept outside a scope (a fresh transposed copy per call); inside, it is made once per
    mask, and an in-place change of the mask (a new version) is seen. The tests' own key extent is 1 + the last live
    token (columns for outgoing, rows for incoming), checked by brute force on an asymmetric mask."""
    from boltz_mlx_amd import kernels as K
    from conftest import mask_key_extent

    N = 70
    g = torch.Generator().manual_seed(5)
    m = (torch.rand((N, N), generator=g) > 0.4).float()
    m[:, 61:] = 0  # columns past 60 dead (outgoing extent 61)
    m[55:, :] = 0  # rows past 54 dead (incoming extent 55)
    brute_out = 1 + max(k for k in range(N) if any(m[i, k] != 0 for i in range(N)))
    brute_in = 1 + max(k for k in range(N) if any(m[k, i] != 0 for i in range(N)))
    assert (brute_out, brute_in) == (61, 55)
    assert mask_key_extent(m, False) == brute_out and mask_key_extent(m, True) == brute_in
    assert mask_key_extent(torch.zeros(N, N), False) == 0
    t0 = K.mask_transposed(m, N)
    assert torch.equal(t0, m.t()) and t0.is_contiguous() and K.mask_transposed(m, N) is not t0
    with K.pair_mask_scope():
        t1 = K.mask_transposed(m, N)
        assert torch.equal(t1, m.t()) and K.mask_transposed(m.view(N, N), N) is t1  # a view of the same storage
        m[:, 69] = 1  # in place: a new version
        assert torch.equal(K.mask_transposed(m, N), m.t())
        with K.pair_mask_scope():  # nested scopes start empty and restore the outer one
            assert not K._MASK_SCOPE.entries
        assert K.mask_transposed(m, N) is K.mask_transposed(m, N)
    assert K.mask_transposed(m, N) is not K.mask_transposed(m, N)


def test_stream_without_torchs_raw_handle(monkeypatch):
    """A torch without the private calls gives the same handle through its public Stream."""
    from boltz_mlx_amd import kernels as K

    class Stream:
        cuda_stream = 1234

    monkeypatch.setattr(torch.cuda, "current_stream", Stream)
    for name in ("_raw_stream", "_device"):
        with monkeypatch.context() as mp:
            mp.setattr(K, name, None)
            assert K._stream() == 1234


class _HalfLN:
    """LayerNorm parameters that the kernels cannot read as they are."""

    def __init__(self, d):
        self.weight, self.bias, self.eps = torch.ones(d, dtype=torch.float16), torch.zeros(d, dtype=torch.float16), 1e-5


def _ln_calls():
    from boltz_mlx_amd import kernels as K

    N, h = 3, torch.float16
    ld = K.row_pitch(N)
    z, o = torch.zeros(N, N, 128), torch.zeros(128, N, ld, dtype=h)
    xn, w, w12, w3 = (torch.zeros(*s, dtype=h) for s in ((N * N, 128), (128, 128), (512, 128), (128, 256)))
    z64, o64, xn64, w64 = torch.zeros(N, N, 64), o[:64], xn[:, :64].contiguous(), torch.zeros(64, 64, dtype=h)
    ln, ln64, pw = _HalfLN(128), _HalfLN(64), torch.zeros(4, 128, dtype=h)
    return {
        "layer_norm": lambda: K.layer_norm(xn, ln.weight, ln.bias),
        "add_ln": lambda: K.add_ln(z, z, ln),
        "trimul_tail": lambda: K.trimul_tail(o, ln, 1e-5, w, xn, w, z, True, ln, N),
        "trimul_tail64": lambda: K.trimul_tail64(o64, ln64, 1e-5, w64, xn64, w64, z64, True, ln64, N),
        "linear_resid_ln": lambda: K.linear_resid_ln(xn, w, False, z, True, ln, N),
        "linear_resid_ln64": lambda: K.linear_resid_ln64(xn, w[:64], False, z64, True, ln64, N),
        "transition": lambda: K.transition(xn, w12, w3, z, True, ln, (ln, pw)),
        "attn_out_transition": lambda: K.attn_out_transition(xn, w, True, z, ln, w12, w3, ln, (ln, pw)),
        "transition64_f16": lambda: K.transition64_f16(z64.view(-1, 64), ln64, w12[:, :64].contiguous(), w3[:64]),
        "ln_linear_f32": lambda: K.ln_linear_f32(z64.view(-1, 64), ln64, torch.zeros(256, 64)),
        "opm_ln_split": lambda: K.opm_ln_split(torch.zeros(2, N, 64), ln64, torch.zeros(64, 64), torch.zeros(2, N)),
        "pair_bias": lambda: K.pair_bias(z, ln, pw),
    }


@pytest.mark.parametrize("name", _ln_calls())
def test_converted_parameters_outlive_the_launch(monkeypatch, name):
    """A LayerNorm parameter that is not fp32 is converted for the call; the copy has to live until the launch is made,
    or the allocator gives its block to the next parameter's copy and the kernel reads one for the other."""
    import weakref

    from boltz_mlx_amd import kernels as K

    copies, calls = [], []

    def f32c(t):
        c = t.float()
        copies.append(weakref.ref(c))
        return c

    monkeypatch.setattr(K, "f32c", f32c)
    monkeypatch.setattr(K, "_dev", lambda *ts: None)
    monkeypatch.setattr(K, "_stream", lambda: 0)
    monkeypatch.setattr(K, "call", lambda *args: calls.append([c() is not None for c in copies]))
    _ln_calls()[name]()
    assert len(calls) == 1 and len(copies) >= 2 and all(calls[0])


class _DeviceMask(torch.Tensor):
    """A CPU tensor that says it is on the GPU, so that what a scope shares can be followed without one."""

    is_cuda = True


@pytest.fixture
def fake_device(monkeypatch):
    """Streams and captures as the wrappers see them, and the launches they make, without a GPU."""
    from boltz_mlx_amd import kernels as K

    state = {"stream": 1, "capturing": False, "calls": []}
    monkeypatch.setattr(K, "_stream", lambda: state["stream"])
    monkeypatch.setattr(torch.cuda, "is_available", lambda: True)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: state["capturing"])
    monkeypatch.setattr(K, "call", lambda name, *args: state["calls"].append((name, args[-1])))
    return state


def _mask(n=70):
    return torch.ones((n, n)).as_subclass(_DeviceMask)


def test_pair_mask_scope_shares_within_one_stream(fake_device):
    """A mask's device values have no order but their stream's: a reader on another stream makes its own."""
    from boltz_mlx_amd import kernels as K

    m = _mask()
    with K.pair_mask_scope():
        a, t = K.key_extent_device(m, 70, False), K.mask_transposed(m, 70)
        assert K.key_extent_device(m, 70, True).data_ptr() == a.data_ptr() + 4 and K.mask_transposed(m, 70) is t
        fake_device["stream"] = 2
        b, u = K.key_extent_device(m, 70, False), K.mask_transposed(m, 70)
        assert b.data_ptr() != a.data_ptr() and u is not t
        fake_device["stream"] = 1
        assert K.key_extent_device(m, 70, False).data_ptr() == a.data_ptr()
    assert fake_device["calls"] == [("bzpf_key_extents", 1), ("bzpf_key_extents", 2)]


@pytest.mark.parametrize("bad", [torch.ones(70, 70, dtype=torch.bool), torch.ones(70, 70, dtype=torch.float16),
                                 torch.ones(69, 70), torch.ones(70)])
def test_key_extent_device_checks_its_mask(fake_device, bad):
    """Its kernel reads N * N floats: nothing else gets there, inside a scope or outside."""
    from boltz_mlx_amd import kernels as K

    bad = bad.as_subclass(_DeviceMask)
    with pytest.raises(ValueError):
        K.key_extent_device(bad, 70, False)
    with K.pair_mask_scope(), pytest.raises(ValueError):
        K.key_extent_device(bad, 70, False)
    assert fake_device["calls"] == []


def test_pair_mask_scope_and_captures(fake_device):
    """A scope that outlives a capture shares nothing with it (a replay would read the mask of the capture, work outside
    it a value that only a replay computes); one entered inside it does, as a captured module run enters."""
    from boltz_mlx_amd import kernels as K

    m = _mask()
    with K.pair_mask_scope():
        t = K.mask_transposed(m, 70)
        fake_device["capturing"] = True
        assert K.mask_transposed(m, 70) is not t
        assert K.key_extent_device(m, 70, False) == 0  # every key
        with K.pair_mask_scope():
            a = K.key_extent_device(m, 70, False)
            assert K.key_extent_device(m, 70, False).data_ptr() == a.data_ptr()
            assert K.mask_transposed(m, 70) is K.mask_transposed(m, 70)
            fake_device["capturing"] = False
            assert K.key_extent_device(m, 70, False) == 0
        assert K.mask_transposed(m, 70) is t


def test_pair_mask_scope_is_the_threads_own(fake_device):
    """A scope of one thread is not another's, and leaving them in any order leaves none behind."""
    import threading

    from boltz_mlx_amd import kernels as K

    m, seen = _mask(), []
    entered, left = threading.Event(), threading.Event()

    def other():
        seen.append(K.key_extent_device(m, 70, False))  # outside: every key
        with K.pair_mask_scope():
            entered.set()
            left.wait(10)
        seen.append(K.key_extent_device(m, 70, False))

    t = threading.Thread(target=other)
    with K.pair_mask_scope():
        K.key_extent_device(m, 70, False)
        t.start()
        assert entered.wait(10)
    left.set()
    t.join()
    seen.append(K.key_extent_device(m, 70, False))
    assert not any(isinstance(v, torch.Tensor) for v in seen)


def test_pair_mask_scope_keeps_its_masks(fake_device):
    """A scope knows a mask by its address, so it holds the mask: one made where a dropped one was is not taken for it."""
    import gc
    import weakref

    from boltz_mlx_amd import kernels as K

    m = _mask()
    alive = weakref.ref(m)
    with K.pair_mask_scope():
        K.mask_transposed(m, 70)
        del m
        gc.collect()
        assert alive() is not None
    gc.collect()
    assert alive() is None


# ---------------------------------------------------------------- kernel index maps and buffer ranges (host build)

@pytest.fixture(scope="module")
def layout_lib(tmp_path_factory):
    """tests/layout_check.cpp built with g++ against boltz_mlx_amd/csrc/bzpf_layout.h (the header the kernels and
    their launchers use; it needs no HIP)."""
    import ctypes
    import os
    import subprocess

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = str(tmp_path_factory.mktemp("layout") / "layout_check.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(root, "boltz_mlx_amd", "csrc"),
                    os.path.join(root, "tests", "layout_check.cpp"), "-o", out], check=True)
    lib = ctypes.CDLL(out)
    lib.lc_check.argtypes = [ctypes.c_char_p, ctypes.c_int]
    lib.lc_tb_offsets.argtypes = [ctypes.c_int64, ctypes.c_int, ctypes.c_void_p]
    return lib


def test_kernel_layouts_and_buffer_ranges(layout_lib):
    """The fragment-ordered triangle bias is a bijection onto its buffer with the core's 1 KB load runs; the
    contraction's LDS swizzle permutes each row and makes the fragment reads conflict-free; every buffer resource of
    the attention core, the contraction and the fp16 sequence attention keeps its extent and largest offset below
    2^31 at the launchers' size limits, which refuse the first size past them."""
    import ctypes

    buf = ctypes.create_string_buffer(1 << 17)
    failures = layout_lib.lc_check(buf, len(buf))
    report = buf.value.decode()
    print(report)
    assert failures == 0, [line for line in report.splitlines() if line.startswith("FAIL")]
    assert report.count("ok") > 100


@pytest.mark.parametrize("N,H", [(1, 1), (37, 4), (130, 3), (257, 4)])
def test_tb_offset_matches_the_host_wrapper(layout_lib, N, H):
    """The kernels' tb_offset (bzpf_layout.h) and kernels.tri_bias_offsets (the host's map of a dense bias into the
    layout, used by the tests and the layout kernels' callers) agree element for element."""
    import numpy as np

    from boltz_mlx_amd import kernels as K

    got = np.empty((H, N, N), dtype=np.int64)
    layout_lib.lc_tb_offsets(N, H, got.ctypes.data)
    assert np.array_equal(got, K.tri_bias_offsets(N, H))
