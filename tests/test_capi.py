"""CPU checks of the C-ABI library: it loads, exports every symbol the header
declares, and its argument validation rejects bad calls before touching the GPU."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "rwkv6_amd.h")


def _declared():
    text = open(HEADER).read()
    return sorted(set(re.findall(r"\b(rwkv6_\w+)\s*\(", text)))


def test_header_declares_entry_points():
    names = _declared()
    for must in ("rwkv6_wkv_fwd", "rwkv6_wkv_bwd", "rwkv6_shift_lerp_fwd", "rwkv6_ddlerp_lora_fwd",
                 "rwkv6_ddlerp_lora_bwd", "rwkv6_lora_bias_fwd", "rwkv6_gn_gate_fwd",
                 "rwkv6_gn_gate_bwd", "rwkv6_strerror"):
        assert must in names


def test_library_exports_every_declared_symbol(pkg):
    lib = ctypes.CDLL(pkg._lib.LIB_PATH)
    missing = [n for n in _declared() if not hasattr(lib, n)]
    assert not missing, missing
    # and the ctypes signature table covers exactly the header
    assert sorted(pkg._lib.SIGNATURES) == _declared()


def test_version_and_strerror(pkg):
    L = pkg._lib.load()
    assert L.rwkv6_abi_version() == pkg._lib.ABI_VERSION == 3
    assert L.rwkv6_strerror(0) == b"ok"
    assert b"64" in L.rwkv6_strerror(2)
    assert L.rwkv6_strerror(12345) == b"unknown rwkv6 status code"


def test_workspace_sizes(pkg):
    L = pkg._lib.load()
    B, H, T = 8, 32, 4096
    NT = T // 64
    saved = L.rwkv6_wkv_saved_bytes(B, H, T, 64, 64)
    assert saved >= B * H * (NT + 1) * 64 * 64 * 2                  # bf16 state per chunk + final
    # forward: no per-chunk state (the walk carries it); per-segment states only when B*H
    # is far below the device's workgroup count (config 5: 32 sequences of 512 chunks)
    assert 0 < L.rwkv6_wkv_workspace_bytes(B, H, T, 64, 64, 0) < 16 << 20
    assert L.rwkv6_wkv_workspace_bytes(1, 32, 32768, 64, 64, 0) >= 32 * 64 * 64 * 4
    # backward, one reverse walk per sequence (B*H fills the device): only the fp32 du
    # partials of each (b,h); config 5 (B*H = 32, 8 segments of 64 chunks): du partials per
    # (b,h, segment), the 7 later segments' piece states (fp32 dS and decay) and the 7
    # segment-start state gradients, all far below a per-chunk state
    assert 0 < L.rwkv6_wkv_workspace_bytes(B, H, T, 64, 64, 1) < 1 << 20
    assert L.rwkv6_wkv_workspace_bytes(B, H, T, 64, 64, 1) >= B * H * 64 * 4
    c5 = L.rwkv6_wkv_workspace_bytes(1, 32, 32768, 64, 64, 1)
    assert 32 * (8 * 64 * 4 + 7 * (64 * 64 * 4 + 64 * 4) + 7 * 64 * 64 * 4) <= c5 < 16 << 20
    assert L.rwkv6_wkv_saved_bytes(B, H, T, 32, 64) == 0          # unsupported head size


def test_backward_plans_of_long_and_many_sequences(pkg):
    """The chunk-parallel backward serves few sequences of a bounded number of chunks: with more
    sequences than half the CUs each is one walk whatever its length, whose workspace holds the du
    partials alone, and one or a few very long sequences are walked in segments (the scan over the
    chunks is serial).  Both keep the workspace far below a state a chunk."""
    L = pkg._lib.load()
    for BH in (129, 132, 144, 150, 158, 200, 256, 1000):
        for NT in (1, 15, 29, 64, 512, 4096):
            assert L.rwkv6_wkv_plan(1, BH, 64 * NT, 1) == 1
            assert L.rwkv6_wkv_workspace_bytes(1, BH, 64 * NT, 64, 64, 1) <= 256 * BH + 256
    for BH in (1, 2, 4, 7, 8, 64, 128):
        for NT in (1024, 2048, 4096):
            assert L.rwkv6_wkv_plan(1, BH, 64 * NT, 1) > 1
            assert L.rwkv6_wkv_workspace_bytes(1, BH, 64 * NT, 64, 64, 1) < 24 << 20
    assert L.rwkv6_wkv_plan(1, 8, 64 * 32, 1) == 0 == L.rwkv6_wkv_plan(1, 1, 64 * 512, 1)


def _fake(addr):
    return ctypes.c_void_p(addr)


def test_validation_rejects_before_launch(pkg):
    """Bad calls return an error code without dereferencing anything (the pointers are fake)."""
    L = pkg._lib.load()
    p = _fake(0x100000)
    args = lambda K=64, u_dt=1, r=p, saved=p: (r, p, p, p, p, u_dt, None, p, None, saved, p,
                                               2, 2, 64, K, 64, 1.0, None)
    assert L.rwkv6_wkv_fwd(*args(K=32)) == pkg._lib.RWKV6_ERR_UNSUPPORTED
    assert L.rwkv6_wkv_fwd(*args(u_dt=7)) == pkg._lib.RWKV6_ERR_INVALID_ARG
    assert L.rwkv6_wkv_fwd(*args(r=None)) == pkg._lib.RWKV6_ERR_INVALID_ARG
    assert L.rwkv6_wkv_fwd(*args(saved=None)) == pkg._lib.RWKV6_ERR_INVALID_ARG
    assert L.rwkv6_wkv_fwd(*args(r=_fake(0x100002))) == pkg._lib.RWKV6_ERR_ALIGNMENT
    assert L.rwkv6_shift_lerp_fwd(p, p, 1, p, 4, 2, 12, None) == pkg._lib.RWKV6_ERR_UNSUPPORTED
    assert L.rwkv6_lora_bias_fwd(p, p, p, 3, p, 4, 1, 64, 32, None) == pkg._lib.RWKV6_ERR_INVALID_ARG
    assert L.rwkv6_lora_bias_fwd(p, p, p, 1, p, 4, 3, 64, 32, None) == pkg._lib.RWKV6_ERR_UNSUPPORTED
    assert L.rwkv6_lora_bias_fwd(p, p, p, 1, p, 4, 0, 64, 32, None) == pkg._lib.RWKV6_ERR_INVALID_ARG
    assert L.rwkv6_gn_gate_fwd(p, 1, p, p, p, 0, 1e-5, p, p, p, 4, 2, 2, 32, None) == \
        pkg._lib.RWKV6_ERR_UNSUPPORTED
    assert L.rwkv6_gn_gate_fwd(None, 1, p, p, p, 0, 1e-5, p, p, p, 4, 2, 2, 64, None) == \
        pkg._lib.RWKV6_ERR_INVALID_ARG
    E = pkg._lib
    assert L.rwkv6_cmix_lerp_fwd(p, p, 1, p, 4, 2, 12, None) == E.RWKV6_ERR_UNSUPPORTED
    assert L.rwkv6_cmix_lerp_fwd(p, None, 1, p, 4, 2, 16, None) == E.RWKV6_ERR_INVALID_ARG
    assert L.rwkv6_cmix_lerp_bwd(p, p, 1, p, p, p, None, 4, 2, 16, None) == E.RWKV6_ERR_INVALID_ARG
    assert L.rwkv6_relu_sq_fwd(p, p, 12, None) == E.RWKV6_ERR_UNSUPPORTED
    assert L.rwkv6_relu_sq_fwd(p, p, -8, None) == E.RWKV6_ERR_INVALID_ARG
    assert L.rwkv6_relu_sq_bwd(p, None, p, 16, None) == E.RWKV6_ERR_INVALID_ARG
    assert L.rwkv6_sigmoid_gate_fwd(p, _fake(0x100008), p, 16, None) == E.RWKV6_ERR_ALIGNMENT
    assert L.rwkv6_sigmoid_gate_bwd(p, p, p, p, None, 16, None) == E.RWKV6_ERR_INVALID_ARG
    assert L.rwkv6_relu_sq_fwd(None, None, 0, None) == E.RWKV6_OK       # empty: nothing to do


def test_overlapping_outputs_are_rejected(pkg):
    """An output that overlaps an input (or another output) is refused before any launch:
    several kernels re-load a clamped last piece after other threads stored theirs, and the
    walks read chunk c + 1 before storing chunk c (the pointers are fake; nothing is read)."""
    L = pkg._lib.load()
    E = pkg._lib
    a, b, c, d = (_fake(0x100000 * i) for i in (1, 2, 3, 4))
    inside = _fake(0x100000 + 16)                                   # 16 bytes into a
    assert L.rwkv6_relu_sq_fwd(a, a, 16, None) == E.RWKV6_ERR_INVALID_ARG
    assert L.rwkv6_relu_sq_fwd(a, inside, 16, None) == E.RWKV6_ERR_INVALID_ARG
    assert L.rwkv6_sigmoid_gate_bwd(a, b, c, d, d, 16, None) == E.RWKV6_ERR_INVALID_ARG
    assert L.rwkv6_sigmoid_gate_fwd(a, b, inside, 16, None) == E.RWKV6_ERR_INVALID_ARG
    assert L.rwkv6_shift_lerp_fwd(a, b, 1, a, 4, 2, 16, None) == E.RWKV6_ERR_INVALID_ARG
    # WKV forward: o on top of v
    assert L.rwkv6_wkv_fwd(a, b, c, d, _fake(0x500000), 1, None, c, None, _fake(0x600000),
                           _fake(0x700000), 1, 1, 64, 64, 64, 1.0, None) == E.RWKV6_ERR_INVALID_ARG
    # GroupNorm backward: a gate gradient without a gate input
    assert L.rwkv6_gn_gate_bwd(a, 1, None, b, b, 0, p_ := _fake(0x500000), p_, c, d, _fake(0x600000),
                               _fake(0x700000), _fake(0x800000), _fake(0x900000), 4, 2, 2, 64,
                               None) == E.RWKV6_ERR_INVALID_ARG


@pytest.mark.parametrize("E,R", [(5, 32), (1, 64), (5, 64), (1, 32), (2, 32)])
def test_bottleneck_calls_agree_on_what_they_take(pkg, E, R):
    """The backward's workspace query, by which a caller chooses these kernels, is nonzero exactly for
    the shapes that the forward and the backward take (null tensors: a shape they take is refused for
    those, after the shape)."""
    L, e = pkg._lib.load(), pkg._lib
    maa = _fake(0x100000) if E > 1 else None
    seen = set()
    for T in (0, 1, 63, 4096, (1 << 28) - 1, 1 << 28, (1 << 28) + 1, (1 << 30) + 1):
        for B in (1, 2, 4, 4097, 65535, 65536, 70000, 131072, 131073):
            for C in (8, 64, 96, 128, 2048, 1 << 23, (1 << 23) + 64):
                took = L.rwkv6_lora_bwd_workspace_bytes(T, B, C, E, R) != 0
                want = e.RWKV6_ERR_INVALID_ARG if took else e.RWKV6_ERR_UNSUPPORTED
                assert L.rwkv6_lora_bwd(None, maa, 0, None, None, None, None, 0, None, 0, None, None, None, 0, None, 0,
                                        None, None, T, B, C, E, R, None) == want, (T, B, C)
                if T:
                    assert L.rwkv6_lora_down_fwd(None, maa, 0, None, 0, None, T, B, C, E, R, None) == want, (T, B, C)
                seen.add(took)
    assert seen == ({True, False} if (E, R) in ((5, 32), (1, 64)) else {False})


def test_bottleneck_workspace_follows_the_device(pkg):
    """The token shift's backward keeps a full set of fp32 partial parameter gradients for each of a
    number of ranges that fills the device, (2 160 + 6) C floats each, whatever the batch: eight at C =
    2048, and d_pre of the tokens."""
    L = pkg._lib.load()
    part = 326 * 2048 * 4
    for N, shapes in ((16384, [(4096, 4), (256, 64), (64, 256), (32, 512), (16, 1024), (4, 4096)]),
                      (4096, [(1, 4096), (2, 2048), (33, 124), (4096, 1)])):
        for T, B in shapes:
            n = L.rwkv6_lora_bwd_workspace_bytes(T, B, 2048, 5, 32)
            assert part <= n - T * B * 160 * 2 <= 8 * part + 256, (T, B, n)
    # narrow layers: at most 256 ranges
    assert L.rwkv6_lora_bwd_workspace_bytes(1, 131072, 64, 5, 32) <= 131072 * 320 + 256 * 326 * 64 * 4 + 256


def test_layer_norm_takes_the_rows_that_a_launch_covers(pkg):
    """256 threads for four rows, below 2^32 threads: more rows are refused by the workspace query (by
    which a module falls back to torch) and by both entries (null tensors are refused after the shape)."""
    L, e = pkg._lib.load(), pkg._lib
    for N in (0, 1, (1 << 26) - 4, (1 << 26) - 3, 1 << 26, 1 << 32):
        took = -(-N // 4) * 256 < 1 << 32
        assert (L.rwkv6_layer_norm_bwd_workspace_bytes(N, 8) != 0) == took
        want = e.RWKV6_ERR_INVALID_ARG if took else e.RWKV6_ERR_UNSUPPORTED
        assert L.rwkv6_layer_norm_bwd(None, None, 0, None, None, None, None, None, None, 0, None, N, 8, None) == want
        if N:
            assert L.rwkv6_layer_norm_fwd(None, None, None, 0, 1e-5, None, None, None, None, N, 8, None) == want


def test_python_checker_maps_codes(pkg):
    with pytest.raises(NotImplementedError):
        pkg._lib.check(2, "x")
    with pytest.raises(ValueError):
        pkg._lib.check(1, "x")
    with pytest.raises(pkg._lib.Rwkv6Error):
        pkg._lib.check(3, "x")
    pkg._lib.check(0, "x")


def test_native_checker_maps_codes(pkg):
    """The C++ functions raise the same types, from a thread without the interpreter lock too (as a
    backward runs them)."""
    check, E = pkg._lib.native().check, pkg._lib
    check(E.RWKV6_OK, "x")
    for status, kind in ((E.RWKV6_ERR_UNSUPPORTED, NotImplementedError), (E.RWKV6_ERR_INVALID_ARG, ValueError),
                         (E.RWKV6_ERR_ALIGNMENT, ValueError), (E.RWKV6_ERR_LAUNCH, E.Rwkv6Error)):
        with pytest.raises(kind, match="^x: ") as e:
            check(status, "x")
        assert type(e.value) is kind


def test_a_forward_leaves_the_interpreter_to_other_threads(pkg):
    """While a function of the extension runs (here one product on the CPU, a hundred milliseconds),
    another thread goes on: with the lock held it could run once before and once after the call."""
    import threading
    import time

    import torch

    x = torch.randn(3000, 3000)
    count, stop = [0], threading.Event()

    def work():
        while not stop.is_set():
            time.sleep(0.001)
            count[0] += 1

    t = threading.Thread(target=work)
    t.start()
    try:
        before = count[0]
        pkg._lib.native().linear(x, x)
        inside = count[0] - before
    finally:
        stop.set()
        t.join()
    assert inside > 3, inside


def test_wrapper_rejects_cpu_tensors(pkg):
    import torch
    x = torch.zeros(1, 1, 4, 64, dtype=torch.bfloat16)
    with pytest.raises(ValueError):
        pkg.chunk_rwkv6(x, x, x, x, torch.zeros(1, 64))
    with pytest.raises(NotImplementedError):
        pkg.chunk_rwkv6(x, x, x, x, torch.zeros(1, 64), cu_seqlens=torch.tensor([0, 4]))


@pytest.mark.parametrize("version,msg", [(2, "ABI version 2"), (None, "lacks")])
def test_stale_library_gets_the_rebuild_message(pkg, tmp_path, version, msg):
    """A stub library built here with gcc: an older ABI version, or the current version with
    symbols missing, must fail with the rebuild hint, not a ctypes AttributeError."""
    import shutil
    import subprocess

    if shutil.which("gcc") is None:
        pytest.skip("gcc not available")
    v = pkg._lib.ABI_VERSION if version is None else version
    src = tmp_path / "stub.c"
    src.write_text(f"int rwkv6_abi_version(void) {{ return {v}; }}\n"
                   "const char* rwkv6_strerror(int c) { (void)c; return \"ok\"; }\n")
    so = tmp_path / "libstub.so"
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(so), str(src)], check=True)
    with pytest.raises(RuntimeError, match="rebuild") as e:
        pkg._lib.bind(ctypes.CDLL(str(so)), str(so))
    assert msg in str(e.value)
