"""CPU checks of the C-ABI boundary: libythip.so loads (no GPU needed to dlopen
it) and exports every function include/ythip.h declares; argument errors are
reported without touching the GPU."""
from __future__ import annotations

import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "ythip.h")


def _declared() -> list[str]:
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(ythip_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_entry_points():
    names = _declared()
    for n in ("ythip_gemm", "ythip_attn_prefill", "ythip_attn_decode", "ythip_rmsnorm_rope", "ythip_last_error"):
        assert n in names


def test_library_exports_every_declared_symbol():
    from ytensor_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.fail("libythip.so is not built (python -m ytensor_amd.build)")
    lib = ctypes.CDLL(_lib.LIB_PATH)
    missing = [n for n in _declared() if not hasattr(lib, n)]
    assert not missing, f"declared but not exported: {missing}"
    assert set(_declared()) == set(_lib.SIGNATURES), "ctypes signature table out of sync with the header"


def test_abi_version_and_argument_errors():
    import ytensor_amd
    lib = ytensor_amd.load()
    assert lib.ythip_abi_version() == 3
    # invalid dtype / negative sizes are rejected before any HIP call
    st = lib.ythip_gemm(7, 0, 1, 2, 2, 2, None, 0, 2, 1, None, 0, 2, 1, None, 0, 2, 1, 1.0, 0.0, None)
    assert st == -1 and b"dtype" in lib.ythip_last_error()
    st = lib.ythip_gemm(0, 0, 1, -2, 2, 2, None, 0, 2, 1, None, 0, 2, 1, None, 0, 2, 1, 1.0, 0.0, None)
    assert st == -1
    # m == 0: a no-op that succeeds (src/kernel/avx2/sgemm.inl:594)
    assert lib.ythip_gemm(0, 0, 1, 0, 2, 2, None, 0, 2, 1, None, 0, 2, 1, None, 0, 2, 1, 1.0, 0.0, None) == 0
    st = lib.ythip_rmsnorm_rope(2, 1, 1, 1, 1, 96, None, 0, None, None, 1e-6, None, None, 0, 0, 0,
                                None, None, None, None, None, None, 0, 0, None, None)
    assert st == -2  # head dim 96 unsupported


def test_decode_noalloc_rejects_oversize_without_a_launch():
    """ythip_attn_decode_noalloc refuses a shape whose split-K partials exceed
    its fixed per-GPU array before touching the GPU (the pointers are never
    dereferenced). B=128, Hq=64, d=128 needs 128*64*1*(128+2)*4 bytes > 4 MiB."""
    import ytensor_amd
    from ytensor_amd import _lib
    lib = ytensor_amd.load()
    cap = int(lib.ythip_attn_decode_noalloc_max_bytes())
    assert cap == 4 << 20
    need = int(lib.ythip_attn_decode_workspace_size(128, 64, 16, 128))
    assert need == 128 * 64 * 130 * 4 > cap
    fake = ctypes.c_void_p(256)
    st = lib.ythip_attn_decode_noalloc(_lib.BF16, 128, 64, 8, 128, 16, fake, _lib.i64array([64 * 128, 128]),
                                       fake, fake, _lib.i64array([8 * 16 * 128, 16 * 128, 128]), None,
                                       fake, _lib.i64array([64 * 128, 128]), 0.0, None)
    assert st == _lib.YTHIP_EINVAL
    assert b"fixed array" in lib.ythip_last_error()


def test_cpp_mirror_compiles_and_reports_errors(tmp_path):
    """The C++ host's kernel-level API (yt::kernel::hip in include/yt/ytensor.hpp)
    builds with the host C++ compiler against libythip.so and maps argument
    errors to exceptions."""
    import shutil
    import subprocess
    from ytensor_amd import _lib
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = tmp_path / "abi_errors"
    lib_dir = os.path.dirname(_lib.LIB_PATH)
    subprocess.check_call([gxx, "-std=c++20", "-O1", f"-I{os.path.join(ROOT, 'include')}", "-I/opt/rocm/include",
                           "-D__HIP_PLATFORM_AMD__", os.path.join(ROOT, "tests", "cpp", "abi_errors.cpp"),
                           "-o", str(exe), f"-L{lib_dir}", "-lythip", f"-Wl,-rpath,{lib_dir}", "-L/opt/rocm/lib",
                           "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib"])
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr
    assert "ok:" in out.stdout


def test_prefill_workspace_size_and_short_workspace():
    """ythip_attn_prefill_workspace_size: one byte per 32-row x 64-key tile of
    the bool mask, in 256-byte units; a bool-mask call given fewer bytes is an
    argument error before any launch (the pointers are never dereferenced)."""
    import ytensor_amd
    from ytensor_amd import _lib
    lib = ytensor_amd.load()
    assert lib.ythip_attn_prefill_workspace_size(8192, 8192) == 256 * 128
    assert lib.ythip_attn_prefill_workspace_size(33, 65) == 256
    assert lib.ythip_attn_prefill_workspace_size(2000, 2096) == 63 * 33 // 256 * 256 + 256
    assert lib.ythip_attn_prefill_workspace_size(0, 64) == 0
    assert lib.ythip_attn_prefill_workspace_size(64, 0) == 0
    fake = ctypes.c_void_p(256)
    st4 = _lib.i64array([16 * 64 * 128, 64 * 128, 128, 1])
    st = lib.ythip_attn_prefill_ws(_lib.BF16, 1, 16, 8, 64, 64, 128, 128, fake, st4, fake,
                                   _lib.i64array([8 * 64 * 128, 64 * 128, 128, 1]), fake,
                                   _lib.i64array([8 * 64 * 128, 64 * 128, 128, 1]), fake, st4, 0.0,
                                   _lib.MASK_BOOL, fake, 64, None, 0, 0, fake, 255, None)
    assert st == _lib.YTHIP_EINVAL
    assert b"workspace of 256 bytes" in lib.ythip_last_error()


def _math_call(lib, dtype, H, Hkv, Sq, Skv, D, at, strides=None, B=1, mask=0):
    """ythip_attn_math_workspace_needed for [B, H, S, D] operands at byte addresses `at`
    (Q, K, V, O; nothing is read)."""
    from ytensor_amd import _lib
    q4 = _lib.i64array([H * Sq * D, Sq * D, D, 1])
    k4 = _lib.i64array(strides or [Hkv * Skv * D, Skv * D, D, 1])
    q, k, v, o = (ctypes.c_void_p(x) for x in at)
    args = (dtype, B, H, Hkv, Sq, Skv, D, D, q, q4, k, k4, v, k4, o, q4)
    return args, int(lib.ythip_attn_math_workspace_needed(*args, mask, ctypes.c_void_p(1 << 40), Skv, None, 0, 0))


def test_math_workspace_only_where_it_is_written():
    """A MATH call that runs in one launch needs no workspace; one whose layout or whose
    output (over Q or K) sends it through the separate launches needs all of it, and
    is refused without (before any launch: the pointers are never dereferenced)."""
    import ytensor_amd
    from ytensor_amd import _lib
    lib = ytensor_amd.load()
    step = 1 << 30
    at = [step, 2 * step, 3 * step, 4 * step]
    for dtype in (_lib.F32, _lib.BF16, _lib.F16):
        full = int(lib.ythip_attn_math_workspace_size(dtype, 1, 16, 2048, 2048))
        assert _math_call(lib, dtype, 16, 8, 2048, 2048, 128, at)[1] == 0
        assert _math_call(lib, dtype, 16, 8, 2048, 2048, 128, [step + 2] + at[1:])[1] == full     # unaligned rows
        assert _math_call(lib, dtype, 16, 8, 2048, 2048, 128, at, [8 * 2048 * 128, 2048 * 128, 1, 2048])[1] == full
        assert _math_call(lib, dtype, 16, 8, 2048, 2048, 128, at[:3] + at[:1])[1] == full         # O over Q
        args, need = _math_call(lib, dtype, 16, 8, 2048, 2048, 128, at[:3] + [2 * step + 256])    # O into K
        assert need == full
        assert lib.ythip_attn_math(*args, 0.0, 0, None, 0, None, 0, 0, None, 0, None) == _lib.YTHIP_EINVAL
        assert b"workspace of" in lib.ythip_last_error()
    assert _math_call(lib, _lib.BF16, 16, 8, 2048, 0, 128, at)[1] == 0


def test_math_one_launch_rule():
    """Few workgroups over many keys take the separate launches (one launch measured 1.5 to 5 times
    their time there), a filled chip, few keys and large batches one launch."""
    import ytensor_amd
    from ytensor_amd import _lib
    lib = ytensor_amd.load()
    at = [i << 40 for i in range(1, 5)]
    one = lambda dt, *a, **k: _math_call(lib, dt, *a, at, **k)[1] == 0  # noqa: E731
    for dt in (_lib.BF16, _lib.F16):
        for Sq in (1, 16, 64):
            assert not one(dt, 16, 8, Sq, 4096, 128)
            assert not one(dt, 1, 1, Sq, 16384, 64)
            assert not one(dt, 1, 1, Sq, 8192, 128, mask=_lib.MASK_BOOL)
        assert not one(dt, 16, 8, 128, 4096, 128, mask=_lib.MASK_BOOL)
        assert one(dt, 16, 8, 512, 512, 128) and one(dt, 16, 8, 1024, 1024, 128, mask=_lib.MASK_BOOL)
        assert one(dt, 16, 8, 256, 4096, 128) and one(dt, 16, 8, 4096, 4096, 64)
        assert one(dt, 16, 8, 1, 256, 128) and one(dt, 16, 8, 1, 4096, 128, B=16)
    assert not one(_lib.F32, 16, 8, 1, 4096, 128) and not one(_lib.F32, 16, 8, 256, 4096, 128)
    assert not one(_lib.F32, 1, 1, 2048, 2048, 64)
    assert one(_lib.F32, 16, 8, 2048, 2048, 128) and one(_lib.F32, 16, 16, 4096, 4096, 64)


def _masked_call(din, dout, m, n, k, at=(1 << 40, 2 << 40, 3 << 40), nt=False, alpha=1.0, kind=2, mask_ld=0, fill=1, batch=1):
    """(needed bytes, operand arguments) of a masked product at byte addresses `at`; nothing is read."""
    import ytensor_amd
    a, b, c = (ctypes.c_void_p(x) for x in at)
    bs = (1, k) if nt else (n, 1)
    args = (din, dout, batch, m, n, k, a, m * k, k, 1, b, n * k, *bs, c, m * n, n, 1, alpha)
    return int(ytensor_amd.load().ythip_gemm_masked_workspace_needed(*args, kind, mask_ld or n, fill)), args


def test_masked_workspace_only_where_it_is_written():
    """A masked product in one launch needs no workspace; a C of another type or over an
    input needs m n floats, and is refused without (before any launch)."""
    import ytensor_amd
    from ytensor_amd import _lib
    lib = ytensor_amd.load()
    m, n, k = 200, 300, 128
    for dt in (_lib.F32, _lib.BF16, _lib.F16):
        assert _masked_call(dt, dt, m, n, k)[0] == 0
        assert _masked_call(dt, _lib.F32, m, n, k)[0] == 0
        for at in ((1 << 40, 2 << 40, 1 << 40), (1 << 40, 2 << 40, (2 << 40) + 64), (1 << 40, 2 << 40, (1 << 40) - 64)):
            need, args = _masked_call(dt, dt, m, n, k, at)
            assert need == m * n * 4 == lib.ythip_gemm_masked_workspace_size(1, m, n)
            st = lib.ythip_gemm_masked(*args, 0.0, 2, ctypes.c_void_p(1 << 44), n, 1, 0.0, None, 0, None)
            assert st == _lib.YTHIP_EINVAL and b"workspace of" in lib.ythip_last_error()
        assert _masked_call(dt, dt, m, n, k, (1 << 40, 2 << 40, 1 << 40), alpha=0.0)[0] == 0
        assert _masked_call(dt, dt, m, n, 0)[0] == 0
    assert _masked_call(_lib.F32, _lib.BF16, m, n, k)[0] == m * n * 4
    assert _masked_call(_lib.BF16, _lib.F16, m, n, k)[0] == m * n * 4


def test_masked_store_rule():
    """Masked products that are faster as a product in the workspace and a blend: few rows with
    a long k, 256-wide tiles with a long k, operands of 2 GiB; the others keep the one launch."""
    from ytensor_amd import _lib
    need = lambda *a, **k: _masked_call(*a, **k)[0] > 0  # noqa: E731
    causal, bytes_, diag = _lib.MASK_CAUSAL, _lib.MASK_BOOL, _lib.MASK_DIAG
    H, F = _lib.BF16, _lib.F32
    for m in (1, 16):
        assert need(H, H, m, 1024, 8192, nt=True) and not need(H, H, m, 1024, 1024, nt=True)
        assert need(F, F, m, 1024, 1024, nt=True) and not need(F, F, m, 1024, 256, nt=True)
    assert need(H, H, 1, 1024, 8192) and need(F, F, 2, 1024, 1024) and not need(H, H, 2, 1024, 8192)
    assert not need(H, H, 17, 1024, 8192, nt=True)
    for n in (512, 2048, 3072):
        for kind in (causal, bytes_):
            assert not need(H, H, n, n, n, kind=kind) and not need(H, H, n, n, n, kind=kind, fill=0)
    assert need(H, H, 4096, 4096, 4096) and need(H, H, 4096, 4096, 4096, fill=0) and need(H, H, 8192, 8192, 8192, kind=causal)
    assert not need(H, H, 4096, 4096, 1024) and not need(H, H, 4096, 4096, 512, fill=0)
    assert not need(H, H, 4096, 4096, 4096, kind=diag, mask_ld=-4000)
    assert not need(F, F, 4096, 4096, 4096) and not need(F, F, 8192, 8192, 8192, kind=causal)
    assert need(H, H, 131200, 256, 8192) and not need(H, H, 131200, 64, 8192)
    assert not need(H, H, 131200, 256, 8192, kind=causal) and need(H, H, 256, 131200, 8192, nt=True, kind=causal)
    assert not need(H, H, 4096, 4096, 4096, kind=_lib.MASK_NONE)


def test_probe_library_loads_and_rejects_bad_shapes():
    """The roofline probe library (libythip_probe.so, measurement support for
    bench.py) loads and refuses shapes it does not take before any launch
    (the pointers are never dereferenced)."""
    from ytensor_amd import probe
    if not os.path.exists(probe.PROBE_LIB_PATH):
        pytest.fail("libythip_probe.so is not built (python -m ytensor_amd.build)")
    lib = probe.load()
    fake = 256
    assert lib.ythip_probe_dma(fake, fake, 300, 256, 128, fake, None) == -1  # M not a multiple of 256
    assert lib.ythip_probe_dma(fake, fake, 256, 256, 64, fake, None) == -1   # fewer than two k steps
    assert lib.ythip_probe_mfma(fake, fake, fake, 0, 1, None) == -1
    assert lib.ythip_probe_mfma(fake, fake, fake, 1, 0, None) == -1
