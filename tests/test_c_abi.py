"""C-ABI surface and host-side routines (CPU only; no kernel is launched here)."""

import ctypes
import json
import re
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

from cornserve_amd import lib, ops
from oracle import vit_index as vi

ROOT = Path(__file__).resolve().parent.parent


def declared_symbols() -> list[str]:
    text = (ROOT / "include" / "cornserve_amd.h").read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\bint\s+(cs_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    names = declared_symbols()
    assert len(names) >= 14
    dll = ctypes.CDLL(str(lib.LIB_PATH))
    for n in names:
        assert hasattr(dll, n), f"{n} is declared in include/cornserve_amd.h but not exported"
    assert sorted(lib.EXPORTED_SYMBOLS) == names, "ctypes binding and header disagree"
    assert lib.load().cs_abi_version() == lib.ABI_VERSION


def test_gemm_args_struct_layout_matches_header():
    # 64-bit pointers / int64 / int32 fields in header order; sizeof must match the C struct (8-byte aligned)
    text = (ROOT / "include" / "cornserve_amd.h").read_text()
    body = re.search(r"typedef struct CsGemmArgs \{(.*?)\} CsGemmArgs;", text, flags=re.S).group(1)
    body = re.sub(r"/\*.*?\*/", "", body, flags=re.S)
    fields = []
    for decl in body.split(";"):
        decl = decl.strip()
        if not decl:
            continue
        names = [n.strip().lstrip("*") for n in decl.split(",")]
        first = names[0].split()[-1].lstrip("*")
        fields += [first] + names[1:]
    assert fields == [f[0] for f in lib.CsGemmArgs._fields_]
    assert ctypes.sizeof(lib.CsGemmArgs) % 8 == 0


def test_status_mapping():
    lib.check(lib.CS_OK, "x")
    with pytest.raises(ValueError):
        lib.check(lib.CS_ERR_INVALID_ARG, "x")
    with pytest.raises(RuntimeError):
        lib.check(lib.CS_ERR_UNSUPPORTED, "x")
    with pytest.raises(lib.KernelLibraryError):
        lib.check(lib.CS_ERR_LAUNCH, "x")


def test_invalid_arguments_are_rejected_without_a_gpu():
    l = lib.load()
    assert l.cs_gemm(None, None) == lib.CS_ERR_INVALID_ARG
    args = lib.CsGemmArgs()
    assert l.cs_gemm(ctypes.byref(args), None) == lib.CS_ERR_INVALID_ARG
    assert l.cs_rmsnorm(None, 0, None, None, 0, 1, 8, 1e-6, 0, None) == lib.CS_ERR_INVALID_ARG
    assert l.cs_attn_varlen(None, None, None, 0, None, 0, None, 0, 16, 80, 0.1, None, 64, None) == lib.CS_ERR_INVALID_ARG
    assert l.cs_rope_qk(None, 0, None, 0, 16, 80, None) == lib.CS_ERR_INVALID_ARG
    # the entry point that allocates nothing refuses what its folded-norm GEMM cannot take before it touches the GPU
    # (fake, suitably aligned addresses: nothing is dereferenced on the way to the refusal)
    na = lib.CsGemmArgs()
    na.A, na.W, na.C = 0x1000, 0x2000, 0x3000
    na.lda = na.ldw = 1280
    na.ldc = na.N = 3840
    na.M, na.K, na.epilogue = 256, 1240, lib.EPI_BIAS
    assert l.cs_gemm_rmsnorm_noalloc(ctypes.byref(na), None) == lib.CS_ERR_UNSUPPORTED      # K not a multiple of 64
    na.K, na.epilogue = 1280, lib.EPI_RESIDUAL
    assert l.cs_gemm_rmsnorm_noalloc(ctypes.byref(na), None) == lib.CS_ERR_UNSUPPORTED      # no folded form of it
    na.epilogue, na.M = lib.EPI_BIAS, 65537
    assert l.cs_gemm_rmsnorm_noalloc(ctypes.byref(na), None) == lib.CS_ERR_TOO_LARGE
    # a prefetch hint must start on a 16-byte boundary and carry a size (and no size without an address)
    pa = lib.CsGemmArgs()
    pa.A, pa.W, pa.C = 0x1000, 0x2000, 0x3000
    pa.lda = pa.ldw = pa.K = 1280
    pa.ldc = pa.N = 3840
    pa.M, pa.epilogue = 256, lib.EPI_BIAS
    pa.prefetch, pa.prefetch_bytes = 0x4008, 4096
    assert l.cs_gemm(ctypes.byref(pa), None) == lib.CS_ERR_INVALID_ARG
    pa.prefetch, pa.prefetch_bytes = 0x4000, -1
    assert l.cs_gemm(ctypes.byref(pa), None) == lib.CS_ERR_INVALID_ARG
    pa.prefetch, pa.prefetch_bytes = None, 4096
    assert l.cs_gemm(ctypes.byref(pa), None) == lib.CS_ERR_INVALID_ARG
    g = np.array([[1, 3, 4]], np.int64)  # odd height cannot be merged 2x2
    with pytest.raises(ValueError):
        ops.vit_seqlens_host(g, 2, 4)


def test_seqlens_host_matches_oracle_and_golden(golden_dir):
    golden = json.loads((golden_dir / "index_golden.json").read_text())
    for name, rec in golden.items():
        sl = ops.vit_seqlens_host(np.array(rec["grids"]), 2, 4)
        assert sl.cu_window.dtype == np.int32
        assert sl.cu_window.tolist() == rec["cu_window_seqlens"], name
        assert sl.cu_full.tolist() == rec["cu_seqlens"], name
        assert sl.total_patches == rec["pos_ids_shape"][0], name
    rng = np.random.default_rng(0)
    for _ in range(50):
        n = int(rng.integers(1, 6))
        grids = [(int(rng.integers(1, 4)), int(rng.integers(1, 50)) * 2, int(rng.integers(1, 50)) * 2) for _ in range(n)]
        sl = ops.vit_seqlens_host(np.array(grids), 2, 4)
        _, cu = vi.get_window_index(grids)
        assert sl.cu_window.tolist() == cu.tolist()
        assert sl.cu_full.tolist() == vi.full_cu_seqlens(grids).tolist()
        units = np.array([t * (h // 2) * (w // 2) for t, h, w in grids])
        assert sl.item_meta[:, 3].tolist() == np.concatenate([[0], np.cumsum(units)[:-1]]).tolist()


def test_empty_batch():
    sl = ops.vit_seqlens_host(np.zeros((0, 3), np.int64), 2, 4)
    assert sl.cu_window.tolist() == [0] and sl.cu_full.tolist() == [0] and sl.total_patches == 0


def test_attention_work_list_host():
    l = lib.load()
    assert l.cs_attn_block_q(64) == 64 and l.cs_attn_block_q(65) == 128
    cu = np.array([0, 64, 64 + 300, 64 + 300 + 128], np.int32)
    work = np.empty((16, 4), np.int32)
    n = ctypes.c_int32(0)
    assert l.cs_attn_work_host(cu.ctypes.data, 3, 128, work.ctypes.data, 16, ctypes.byref(n)) == 0
    w = work[: n.value]
    assert w.tolist() == [[0, 64, 0, 64], [64, 364, 64, 128], [64, 364, 192, 128], [64, 364, 320, 44], [364, 492, 364, 128]]
    # every query row is covered exactly once and stays inside its segment
    cover = np.zeros(cu[-1], int)
    for s, e, q0, nq in w:
        assert s <= q0 and q0 + nq <= e
        cover[q0 : q0 + nq] += 1
    assert (cover == 1).all()
    assert l.cs_attn_work_host(cu.ctypes.data, 3, 128, work.ctypes.data, 2, ctypes.byref(n)) == lib.CS_ERR_TOO_LARGE


def _window_attn_args(K: int, windows: int = 2, heads: int = 16) -> lib.CsGemmArgs:
    """A cs_qkv_window_attn call that is valid but for what the test changes (pointers that nothing follows on the host)."""
    a = lib.CsGemmArgs()
    a.A = a.W = a.C = a.bias = 1 << 20
    a.M, a.N, a.K = 64 * windows, 256 * heads, K
    a.lda = a.ldw = K
    a.ldc = 80 * heads
    return a


def _gemm_args(M: int, N: int, K: int, *, epilogue: int = lib.EPI_BIAS, split: bool = False) -> lib.CsGemmArgs:
    a = lib.CsGemmArgs()
    a.A = a.W = a.C = 1 << 20
    a.M, a.N, a.K = M, N, K
    a.lda = a.ldw = K
    a.ldc = N
    a.epilogue = epilogue
    if epilogue == lib.EPI_RESIDUAL:
        a.residual, a.ldr = 1 << 20, N
    if split:
        a.residual_lo = a.c_lo = 1 << 20
    return a


def test_few_row_kernel_takes_launches_of_at_most_two_rounds():
    """The few-row kernel's times hold for launches of one or two rounds of 256 workgroups: 4097 to 4480 rows x 1152 x 1152,
    which it would run in five, belong to the 256-row tiles."""
    groups = lambda *a, **kw: lib.load().cs_gemm_few_row_workgroups(ctypes.byref(_gemm_args(*a, **kw)))  # noqa: E731
    for M in (4100, 4160, 4374, 4480):
        for split in (False, True):
            assert groups(M, 1152, 1152, epilogue=lib.EPI_RESIDUAL, split=split) == 0
    for N in (1152, 1280, 3456, 3840, 4352, 5120, 6912):
        for K in (256, 1152, 1280, 3456, 4352, 5120):
            for epilogue, split in ((lib.EPI_BIAS, False), (lib.EPI_RESIDUAL, False), (lib.EPI_RESIDUAL, True)):
                for M in (1, 96, 250, 500, 1000, 1450, 2196, 3000, 4200, 6000, 9000, 20000):
                    assert groups(M, N, K, epilogue=epilogue, split=split) <= 512
    assert groups(96, 1280, 1280) == 3 * 40                                          # 32x32 tiles
    assert groups(1000, 1280, 1280, epilogue=lib.EPI_RESIDUAL, split=True) == 16 * 16    # 64x80
    assert groups(200, 4352, 1152, epilogue=lib.EPI_GELU_TANH) == 7 * 68             # 32x64, two rounds
    assert groups(96, 1280, 1216) == groups(8192, 1280, 1280) == 0                   # K % 128; many rows


def test_fp8_activation_products_take_the_forms_that_are_fast_with_them():
    """GELU products with fp8 weights, whose times are their own column of the table of forms: 1458 rows x 4352 x 1152 21.4 us in
    256x128 tiles (23.9 in the next form), 10000 rows 104.5 in 256x256 (109.6 in 192x192), 7290 rows x 5120 x 1280 93.8 in 256x256 tiles
    over 4352 columns and 128x192 over the rest (109.6 in 192x160)."""
    def plan(M, N, K, epilogue):
        a = _gemm_args(M, N, K, epilogue=epilogue)
        a.w_fp8, a.w_scale = 1, 1 << 20
        form = (ctypes.c_int32 * 3)()
        assert lib.load().cs_gemm_big_form(ctypes.byref(a), form) == 0
        return tuple(form)

    assert plan(1458, 4352, 1152, lib.EPI_GELU_TANH) == (256, 128, 0)
    assert plan(10000, 4352, 1152, lib.EPI_GELU_TANH) == (256, 256, 0)
    assert plan(7290, 5120, 1280, lib.EPI_QUICK_GELU) == (128, 192, 4352)


def test_few_row_launches_read_their_prefetch_hint():
    """A launch of at most 192 tiles starts workgroups on idle compute units that read the hint: up to 128, none without a
    hint or time.  Where a few-row form of nearly the big form's time is too full for that and the big form is not, the big
    form gets the launch."""
    def groups(M, N, K, nbytes, **kw):
        a = _gemm_args(M, N, K, **kw)
        plain = lib.load().cs_gemm_few_row_workgroups(ctypes.byref(a))
        a.prefetch, a.prefetch_bytes = (1 << 20, nbytes) if nbytes else (None, 0)
        return plain, lib.load().cs_gemm_few_row_workgroups(ctypes.byref(a)) - plain

    split = {"epilogue": lib.EPI_RESIDUAL, "split": True}
    assert groups(96, 1280, 1280, 8 << 20, **split) == (120, 128)
    assert groups(500, 1280, 3456, 10 << 20, **split) == (160, 96)
    assert groups(1000, 1280, 1280, 8 << 20, **split) == (256, 0)      # one tile for every compute unit
    assert groups(200, 4352, 1152, 8 << 20, epilogue=lib.EPI_GELU_TANH) == (476, 0)
    assert groups(40, 320, 256, 8 << 20, **split)[1] == 128 and groups(2400, 1280, 5120, 3 << 20, **split) == (190, 66)
    for M in (2700, 3024):                                             # 128x128 tiles without a hint, 128x160 with one
        assert groups(M, 1280, 5120, 3 << 20, **split) == ((M + 127) // 128 * 10, -((M + 127) // 128 * 10))
    assert groups(3248, 1280, 5120, 3 << 20, **split) == (0, 0)
    for nbytes in (0, 8):                                              # no hint, none of a whole piece
        assert groups(96, 1280, 1280, nbytes, **split) == (120, 0)
        assert groups(2700, 1280, 5120, nbytes, **split) == (220, 0)


@pytest.mark.parametrize("K", [1408, 2048, 3456, 1280 + 64, 192])
def test_window_attn_refuses_inline_norms_of_a_width_they_do_not_have(K):
    """Inline norms keep eight parts of 160 columns in LDS and exist for K a multiple of 128: any other width is refused
    before a launch (a ninth part would lie behind the launch's LDS)."""
    a = _window_attn_args(K)
    a.a_norm_inline = 1
    for windows in (2, 64):
        a.M = 64 * windows
        assert lib.load().cs_qkv_window_attn(ctypes.byref(a), 1 << 20, 0.1, 16, 80, None) == lib.CS_ERR_UNSUPPORTED
    assert lib.load().cs_gemm_norm_inline_pays(64, 4096, K, 1) == 0


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("M", [1, 200, 1450, 8192])
def test_gemm_refuses_row_sums_it_would_not_write(M, fp8):
    """c_row_sum needs c_row_sumsq: whatever the row count, a call with the sums alone is refused before a launch."""
    a = lib.CsGemmArgs()
    a.A = a.W = a.C = a.residual = a.c_row_sum = 1 << 20
    a.M, a.N, a.K = M, 1280, 1280
    a.lda = a.ldw = a.ldc = a.ldr = 1280
    if fp8:
        a.w_fp8, a.w_scale = 1, 1 << 20
    for epilogue in range(6):
        for byte_plane in (None, 1 << 20) if epilogue == lib.EPI_RESIDUAL else (None,):
            a.epilogue, a.c_lo = epilogue, byte_plane
            assert lib.load().cs_gemm(ctypes.byref(a), None) == lib.CS_ERR_UNSUPPORTED, epilogue


def test_resize_taps_host_matches_the_oracle_bit_for_bit():
    """cs_resize_bicubic_taps_host is host arithmetic (doubles, then 22-bit fixed point): no GPU needed."""
    from oracle import qwen_preprocess as qp

    for a, b in [(4000, 1344), (3000, 1008), (100, 250), (37, 37), (5, 3), (3, 300), (1080, 1092), (299, 28), (1, 7), (7, 1),
                 (9000, 28)]:
        bounds, taps = ops.resize_bicubic_taps_host(a, b)
        rb, rt = qp.pillow_bicubic_taps(a, b)
        assert bounds.dtype == np.int32 and taps.dtype == np.int32
        assert np.array_equal(bounds, rb) and np.array_equal(taps, rt), (a, b)
    dll = lib.load()
    k = ctypes.c_int32(0)
    assert dll.cs_resize_bicubic_taps_host(0, 5, None, None, 0, ctypes.byref(k)) == lib.CS_ERR_INVALID_ARG
    assert dll.cs_resize_bicubic_taps_host(10, 5, None, None, 0, ctypes.byref(k)) == 0 and k.value == 9
    small = np.zeros((5, 4), dtype=np.int32)
    b = np.zeros((5, 2), dtype=np.int32)
    assert dll.cs_resize_bicubic_taps_host(10, 5, b.ctypes.data, small.ctypes.data, 4, ctypes.byref(k)) == lib.CS_ERR_INVALID_ARG
    assert dll.cs_resize_u8_pass(None, 1, 4, 4, 3, None, None, 5, None, None) == lib.CS_ERR_INVALID_ARG


_LATE_BUILD = """
import sys
from pathlib import Path
import torch
from cornserve_amd import lib
built, built_torch, version = lib.LIB_PATH, lib.TORCH_LIB_PATH, lib.ABI_VERSION
lib.LIB_PATH, lib.TORCH_LIB_PATH = Path("/nonexistent/k.so"), Path("/nonexistent/t.so")
from cornserve_amd import ops
a = torch.zeros((4, 8), dtype=torch.bfloat16)
f, work = a.float(), torch.zeros((1, 4), dtype=torch.int32)
calls = [lambda: ops.gemm(a, a), lambda: ops.gemm(a, a, out=a), lambda: ops.rmsnorm(a, a[0], 1e-6),
         lambda: ops.layernorm(a, a[0], a[0], 1e-6), lambda: ops.rope_qk_(a, f, 1, 4),
         lambda: ops.attn_varlen(a, a, a, ops.AttnPlan(work, 1, 4), 1, 8, 1.0), lambda: ops.qkv_window_attn(a, a, a[0], f, 1, 1.0),
         lambda: torch.ops.cornserve_amd.rmsnorm_(a, a, a[0], 1e-6, False)]

def all_raise(kind, words):
    for n, call in enumerate(calls):
        try:
            call()
        except kind as e:
            assert any(w in str(e) for w in words), (n, str(e))
        else:
            sys.exit(f"call {n} did not raise {kind}")

all_raise(lib.KernelLibraryError, ["python -m cornserve_amd.build"])        # nothing built
lib.LIB_PATH = built
all_raise(lib.KernelLibraryError, ["python -m cornserve_amd.build"])        # the kernel library alone
lib.TORCH_LIB_PATH = Path(__import__("os").devnull)
all_raise(lib.KernelLibraryError, ["rebuild"])                              # not a library
lib.TORCH_LIB_PATH, lib.ABI_VERSION = built_torch, version + 1
all_raise(lib.KernelLibraryError, ["mismatch"])                             # of another version
lib.ABI_VERSION = version
all_raise(ValueError, ["device tensor", "2-D"])                             # built after the import: loaded by the call
print("late build ok")
"""


def test_a_missing_or_late_library_is_reported_and_loaded_by_the_call():
    """Importing the operators needs no library; a call names the build command while one is missing, refuses one of another
    version, and loads what was built after the import."""
    run = subprocess.run([sys.executable, "-c", _LATE_BUILD], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert run.returncode == 0 and "late build ok" in run.stdout, run.stdout + run.stderr
    assert "verrid" not in run.stderr, run.stderr


def test_native_operators_refuse_what_their_kernels_cannot_take():
    """The natively implemented operators raise the exception categories of the model API (ValueError for bad input)."""
    import torch

    a = torch.zeros((4, 8), dtype=torch.bfloat16)
    f = a.float()
    work = torch.zeros((1, 4), dtype=torch.int32)
    plan = ops.AttnPlan(work, 1, 4)
    for call in (lambda: ops.gemm(a, a), lambda: ops.gemm(a, a, out=a), lambda: ops.gemm(a[0], a), lambda: ops.gemm(a, a[0]),
                 lambda: ops.gemm(a, a, conv_patch=2), lambda: ops.rmsnorm(a, a[0], 1e-6), lambda: ops.layernorm(a, a[0], a[0], 1e-6),
                 lambda: ops.rope_qk_(a, f, 1, 4), lambda: ops.attn_varlen(a, a, a, plan, 1, 8, 1.0),
                 lambda: ops.qkv_window_attn(a, a, a[0], f, 1, 1.0)):
        with pytest.raises(ValueError, match="device tensor|2-D|NCHW"):
            call()
    # every operator has an implementation, here or in the native library
    for name in ops._OPERATORS:
        assert torch._C._dispatch_has_kernel_for_dispatch_key(f"cornserve_amd::{name}", "CompositeExplicitAutograd"), name
