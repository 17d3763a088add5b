"""CPU-side checks of the drop-in boundary: the shared library loads and exports exactly what
include/crow_hip.h declares, host-side types refuse bad shapes with the reference's messages, and
nothing computes without a GPU (no CPU fallback)."""
import os
import re

import numpy as np
import pytest

from conftest import ROOT
from crow_nest_amd import lib as L
from crow_nest_amd.weights import Nvfp4Matrix


def _declared(header="crow_hip.h"):
    text = open(os.path.join(ROOT, "include", header)).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(crow_hip_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    assert os.path.exists(L.library_path()), "libcrow_hip.so is not built: run __graft_entry__.build()"
    lib = L.lib()
    declared = _declared()
    assert declared, "no declarations found"
    for name in declared:
        assert hasattr(lib, name), f"{name} is declared in include/crow_hip.h but not exported"
    assert sorted(L.EXPORTS) == declared
    # the timing and tuning helpers of the benchmark and the tests live in a header of their own, outside the product ABI
    bench = _declared("crow_hip_bench.h")
    assert bench == sorted(L.BENCH_EXPORTS) and not set(bench) & set(declared)
    for name in bench:
        assert hasattr(lib, name), f"{name} is declared in include/crow_hip_bench.h but not exported"


def test_kernel_table_names_without_a_device():
    lib = L.lib()
    n = lib.crow_hip_function_count()
    names = [lib.crow_hip_function_name(i).decode() for i in range(n)]
    for want in ["gemv_nvfp4_w", "gemv_nvfp4_gu", "gemv_nvfp4_gu_bf16", "gemv_nvfp4_wm", "gemv_nvfp4_gum", "gemv_fp4", "gemv_fp4_b", "gemv_fp4_bs",
                 "gemv_fp4_b1k", "gemv_fp4_ptrb", "router_top10", "silu_mul_combo", "acc_combo", "argmax_k",
                 "dequant_fp4_flat", "gemv_nvfp4_w_argmax", "moe_gate_up_silu", "moe_down_combine", "moe_route_gate_up_silu", "moe_group", "moe_gate_up_silu_grouped", "moe_down_grouped", "gemm_nvfp4_bf16",
                 "gemm_nvfp4_bf16_m16", "gemm_nvfp4_bf16_m32", "gemm_nvfp4_bf16_m64", "gemv_bf16_w", "gemv_bf16", "gemv_bf16_b", "gemv_b", "gemv_bf16_ws", "gemv_bf16_bs"]:
        assert want in names, want
    import ctypes as C
    out = C.c_void_p()
    assert lib.crow_hip_get_function(b"no_such_kernel", C.byref(out)) == -2  # CROW_ERR_KERNEL_MISSING
    assert b"kernel missing" in lib.crow_hip_error_string(-2)
    assert lib.crow_hip_tiled_bytes(17408, 5120) == 17408 * 5120 // 64 * 36 == lib.crow_hip_container_bytes(17408, 5120)
    assert lib.crow_hip_tiled_bytes(1, 64) == 2304  # one padded group: 16 rows x 256 columns
    assert lib.crow_hip_tiled_bytes(151936, 5120) == lib.crow_hip_container_bytes(151936, 5120)


def test_kernel_header_is_the_library_table():
    """include/crow_kernels.h lists every kernel name with the number of values its launch takes: same set, same counts."""
    import ctypes as C
    text = open(os.path.join(ROOT, "include", "crow_kernels.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    listed = {m.group(1): int(m.group(2)) for m in re.finditer(r"^CROW_KERNEL\((\w+),\s*(\d+)\)", text, flags=re.M)}
    lib = L.lib()
    table = {}
    for i in range(lib.crow_hip_function_count()):
        name = lib.crow_hip_function_name(i)
        f = C.c_void_p()
        assert lib.crow_hip_get_function(name, C.byref(f)) == 0
        table[name.decode()] = lib.crow_hip_function_arg_count(f)
    assert listed == table


def test_gemm_kernel_choice_names_table_entries():
    lib = L.lib()
    n = lib.crow_hip_function_count()
    names = {lib.crow_hip_function_name(i).decode() for i in range(n)}
    picks = {m: lib.crow_hip_gemm_kernel(17408, m).decode() for m in (1, 16, 17, 96, 97, 128, 256, 512, 1024, 4096)}
    assert set(picks.values()) <= names
    assert picks[16] == "gemm_nvfp4_bf16_m16" and picks[17] == picks[96] == "gemm_nvfp4_bf16_m32"
    assert all(v != "gemm_nvfp4_bf16_m16" for m, v in picks.items() if m > 16)  # that entry point refuses m > 16


def test_gemm_kernel_choice_by_the_fullest_compute_unit():
    """Few row tiles stay with the K-split blocks well beyond 96 tokens; large products go to the tall tiles, whose grid is
    one block per (320 rows, tokens per block) tile."""
    import ctypes as C
    lib = L.lib()
    pick = lambda rows, m: lib.crow_hip_gemm_kernel(rows, m).decode()[len("gemm_nvfp4_bf16_"):]
    assert [pick(1024, m) for m in (17, 512, 1024)] == ["m32"] * 3
    assert pick(17408, 96) == "m32" and [pick(17408, m) for m in (97, 128, 144)] == ["m48"] * 3  # one round of 256 x 48 blocks
    assert pick(5120, 1024) == "t64" and pick(2816, 2048) == "t96" and pick(17408, 512) == pick(5120, 1999) == "t128"
    assert pick(16, 32 * 65535) == "m32" and pick(16, 32 * 65535 + 1) != "m32"  # the end of a grid's second dimension
    for name, mt in (("t64", 64), ("t96", 96), ("t128", 128)):
        for rows, m in ((1, 1), (320, mt), (321, mt + 1), (17408, 2048)):
            d = L.Dims()
            assert lib.crow_hip_launch_dims(f"gemm_nvfp4_bf16_{name}".encode(), rows, 5120, m, C.byref(d)) == 0
            assert (d.gx, d.gy, d.gz, d.bx) == (-(-rows // 320) * -(-m // mt), 1, 1, 256)


def test_gemm_kernel_choice_names_an_entry_point_that_takes_the_product():
    """Where any entry point does: the K-split and shared-X kernels count activations from the start of X in 32 bits and token
    blocks in the grid's second dimension, the tall tiles count from a block's first token row (K < 2^25)."""
    lib = L.lib()
    for rows in (16, 64, 256, 1024, 17408, 151936):
        for m in (17, 64, 128, 129, 12288, 246923, 839000, 32 * 65535 + 1, 1 << 22):
            for k in (64, 1024, 5120, 17408, (1 << 32) // m // 64 * 64, ((1 << 32) // m // 64 + 1) * 64, (1 << 25) - 64, 1 << 25):
                name = lib.crow_hip_gemm_kernel_for(rows, m, k).decode()[len("gemm_nvfp4_bf16_"):]
                counted = m * k <= 0xFFFFFFFF
                if name[0] == "t":
                    assert k < 1 << 25, (rows, m, k, name)
                elif counted or k < 1 << 25:  # (else none takes it, and the one named refuses)
                    assert counted and -(-m // int(name[1:])) <= 65535, (rows, m, k, name)


# (sizes at which a choice that does not know K, or leaves out the eight-wave blocks, names a kernel that takes 3 to 59 % longer)
@pytest.mark.parametrize("rows,m,k,want", [
    (17408, 1999, 1024, "w96"), (17408, 300, 1024, ("w48", "m48")), (5120, 300, 1024, "m48"), (8192, 200, 1024, "m48"), (1024, 1999, 1024, "m48"),
    (12288, 300, 512, ("m64", "m48")), (4096, 300, 256, "m48"), (8192, 1536, 5120, "w96"), (8192, 1536, 8192, "w96"), (12288, 1999, 5120, "w96"),
    (17408, 512, 5120, "t128"), (5120, 1999, 17408, "t128"), (17408, 1999, 2048, ("w96", "t128")), (5120, 1999, 1024, "t128"), (1024, 512, 5120, "m32")])
def test_gemm_kernel_choice_knows_k(rows, m, k, want):
    name = L.lib().crow_hip_gemm_kernel_for(rows, m, k).decode()[len("gemm_nvfp4_bf16_"):]
    assert name in ((want,) if isinstance(want, str) else want)


def test_a_shape_word_made_by_two_threads_at_once_is_one_word(monkeypatch):
    """A second thread asks for the same value while the first is making its word: both get the same address, of a tensor that
    the object keeps - never one that nothing holds any more."""
    import ctypes as C
    import torch
    from crow_nest_amd import weights as W
    monkeypatch.setattr(W, "_device", lambda: torch.device("cpu"))
    p, made, other = W.Params(), [], []

    def store(ptr, v):
        made.append(ptr)
        C.c_int32.from_address(ptr).value = v
        if len(made) == 1:
            other.append(p.i32(7))  # what the second thread does meanwhile

    monkeypatch.setattr(W, "_store_word", store)
    ptr = p.i32(7)
    assert ptr == other[0] == p.i32(7) and len(set(made)) == 2 and ptr in made
    # every word stays what it is, in memory that the object keeps, across more than one block of words
    words = {v: p.i32(v) for v in range(-3, 2 * p.BLOCK)}
    assert words[7] == ptr and len(set(words.values())) == len(words)
    assert all(C.c_int32.from_address(at).value == v == C.c_int32.from_address(p.i32(v)).value for v, at in words.items())
    assert all(any(0 <= at - t.data_ptr() < 4 * p.BLOCK for t in p._blocks.values()) for at in words.values())


def test_native_launch_call_arguments():
    """The package's native launch call hands its integers to the library and returns the library's codes; what is not an
    integer, or too much, raises.  (Nothing is launched: the library is not initialised here.)"""
    import ctypes as C
    import torch
    from crow_nest_amd import _launch
    lib = L.lib()
    _launch.bind(C.cast(lib.crow_hip_launch_dims_split, C.c_void_p).value, C.cast(lib.crow_hip_launch, C.c_void_p).value)
    f = C.c_void_p()
    assert lib.crow_hip_get_function(b"gemv_nvfp4_w", C.byref(f)) == 0
    vals = [16] * 6
    assert _launch.launch(b"no_such_kernel", f.value, 16, 256, 1, *vals) == -2
    assert _launch.launch(b"gemv_nvfp4_w", f.value, 16, 100, 1, *vals) == -7  # K is no whole block
    assert _launch.launch(b"gemv_nvfp4_w", 0, 16, 256, 1, *vals) == -2 and _launch.launch_at(0, 1, 1, 1, 64, *vals) == -2
    if not torch.cuda.is_available():
        assert _launch.launch(b"gemv_nvfp4_w", f.value, np.int64(16), 256, 1, *vals) == -1  # not initialised
        assert _launch.launch_at(f.value, 1, 4, 1, 64, *vals) == -1
    for bad in ((b"gemv_nvfp4_w", f.value, 16, 256, 1, 1.5), ("gemv_nvfp4_w", f.value, 16, 256, 1), (b"gemv_nvfp4_w", f.value, 16), (b"x",) + (1,) * 40):
        with pytest.raises(TypeError):
            _launch.launch(*bad)
    for bad in (-1, 1 << 32):
        with pytest.raises(OverflowError):
            _launch.launch(b"gemv_nvfp4_w", f.value, bad, 256, 1, *vals)


def test_launches_without_the_native_launch_module(monkeypatch):
    """An interpreter that the module was not built for launches through ctypes, says so once, and gets the same errors."""
    import ctypes as C
    import sys
    import warnings
    import torch
    import crow_nest_amd
    from crow_nest_amd import kernels as K

    class Loaded:
        def get(self, name):
            out = C.c_void_p()
            assert L.lib().crow_hip_get_function(name.encode(), C.byref(out)) == 0
            return out.value

    with warnings.catch_warnings():
        warnings.simplefilter("error")
        native = K.Kernels(Loaded())
    monkeypatch.setitem(sys.modules, "crow_nest_amd._launch", None)
    monkeypatch.delattr(crow_nest_amd, "_launch", raising=False)
    with pytest.warns(RuntimeWarning, match="launches go through ctypes"):
        plain = K.Kernels(Loaded())
    for k in (native, plain):
        with pytest.raises(K.KernelMissing):
            k.run("no_such_kernel", 16, 256, 1, *[16] * 6)
        with pytest.raises(L.CrowHipError) as ei:
            k.run("gemv_nvfp4_w", 16, 100, 1, *[16] * 6)
        assert ei.value.code == -7
        if not torch.cuda.is_available():
            for call in (lambda: k.run("gemv_nvfp4_w", 16, 256, 1, *[16] * 6), lambda: k.run_at("gemv_nvfp4_w", 1, 4, 1, 64, *[16] * 6)):
                with pytest.raises(L.CrowHipError) as ei:
                    call()
                assert ei.value.code == -1  # not initialised


def test_launch_dims_depend_on_the_matrix_only():
    import ctypes as C
    lib = L.lib()
    d1, d4 = L.Dims(), L.Dims()
    assert lib.crow_hip_launch_dims(b"gemv_nvfp4_w", 17408, 5120, 1, C.byref(d1)) == 0
    assert lib.crow_hip_launch_dims(b"gemv_nvfp4_wm", 17408, 5120, 1, C.byref(d4)) == 0
    # verify rows == decode row, bit for bit: same split of K over waves and slices (it fixes the order of the sums); the verify
    # kernel's blocks take two strips each, and the row hint differs
    assert (d1.gy & 0xFF0FFFFF, d1.gz, d1.bx) == (d4.gy & 0xFF0FFFFF, d4.gz, d4.bx) and d4.gx == (d1.gx + 1) // 2
    assert d1.gx == 17408 // 16 and d1.bx == 3 * 64 and d1.gy == (5120 // 64) | (1 << 24)  # one block per strip, whole K inside it
    assert (d4.gy >> 20) & 0xF == 1
    assert lib.crow_hip_launch_dims(b"gemv_nvfp4_w", 5120, 17408, 1, C.byref(d1)) == 0
    assert d1.gy >> 24 > 1 and d1.gy & 0xFFFFF == 17408 // 64  # a strip of 68 groups is cut into slices
    assert lib.crow_hip_launch_dims(b"gemv_nvfp4_gu_bf16", 17408, 5120, 1, C.byref(d1)) == 0
    assert d1.bx == 2 * 2 * 64 and d1.gy >> 24 == 1
    assert lib.crow_hip_launch_dims(b"gemv_nvfp4_w", 8, 96, 1, C.byref(d1)) == -7  # 96 columns: not whole blocks


@pytest.mark.parametrize("rows,cols", [(512, 2048), (4096, 2560), (8192, 3584), (2048, 5120)])
def test_routed_launches_keep_long_walks(rows, cols):
    """One wave per seven groups of a strip: a routed launch has a strip per combo or tile and needs no more waves."""
    import ctypes as C
    d = L.Dims()
    for name in (b"gemv_fp4_ptrb", b"moe_down_grouped"):
        assert L.lib().crow_hip_launch_dims(name, rows, cols, 64, C.byref(d)) == 0
        assert d.bx == 64 * -(-cols // (7 * 256)), name
    assert L.lib().crow_hip_launch_dims(b"gemv_nvfp4_w", rows, cols, 1, C.byref(d)) == 0 and d.bx == 64 * 4


def test_bf16_rows_keep_three_waves_on_long_strips():
    """Decode row and verify rows alike (they share the order of the sums)."""
    import ctypes as C
    d = L.Dims()
    for rows, cols, waves in ((8192, 4608, 3), (4112, 5376, 3), (4096, 5376, 4), (8192, 4096, 4), (8208, 4096, 3), (512, 5376, 4)):
        for name, m in ((b"gemv_nvfp4_w_bf16", 1), (b"gemv_nvfp4_wm_bf16", 3)):
            assert L.lib().crow_hip_launch_dims(name, rows, cols, m, C.byref(d)) == 0 and d.bx == 64 * waves, (name, rows, cols)


def test_matrix_shapes_are_checked_like_the_reference():
    b = np.zeros(Nvfp4Matrix.byte_len(3, 128), np.uint8)
    Nvfp4Matrix.new(b, 3, 128, 1.0)
    with pytest.raises(ValueError, match="96 columns are not whole 64-value NVFP4 blocks"):
        Nvfp4Matrix.new(b, 3, 96, 1.0)
    with pytest.raises(ValueError, match=r"\[3, 128\] needs 216 B, got 215"):
        Nvfp4Matrix.new(b[1:], 3, 128, 1.0)


def test_expert_block_is_cut_out_of_a_unit_like_the_reference():
    """ExpertBlock::new / from_unit (engine/src/cpu_nvfp4.rs:153-178): gate | up | down back to back, the three global scales
    in that order, the reference's refusal texts."""
    from crow_nest_amd.weights import ExpertBlock
    hidden, inter = 128, 64
    gu, dn = Nvfp4Matrix.byte_len(inter, hidden), Nvfp4Matrix.byte_len(hidden, inter)
    unit = (np.arange(2 * gu + dn) % 251).astype(np.uint8)
    e = ExpertBlock.from_unit(unit, hidden, inter, (1.0, 2.0, 3.0))
    assert (e.hidden, e.inter) == (hidden, inter)
    assert np.array_equal(e.gate.bytes, unit[:gu]) and np.array_equal(e.up.bytes, unit[gu:2 * gu]) and np.array_equal(e.down.bytes, unit[2 * gu:])
    assert (e.gate.global_scale, e.up.global_scale, e.down.global_scale) == (1.0, 2.0, 3.0)
    assert (e.down.rows, e.down.cols) == (hidden, inter)
    with pytest.raises(ValueError, match=f"expert unit H 128 I 64 needs {2 * gu + dn} B, got {2 * gu + dn - 1}"):
        ExpertBlock.from_unit(unit[1:], hidden, inter, (1.0, 2.0, 3.0))
    with pytest.raises(ValueError, match=r"expert shapes gate \[64, 128\], up \[64, 128\], down \[64, 128\] do not fit together"):
        ExpertBlock.new(e.gate, e.up, e.gate)


def test_no_cpu_fallback():
    import torch
    if torch.cuda.is_available():
        pytest.skip("a GPU is visible")
    from crow_nest_amd.weights import load_fp4
    m = Nvfp4Matrix.new(np.zeros(Nvfp4Matrix.byte_len(64, 256), np.uint8), 64, 256, 1.0)
    with pytest.raises(RuntimeError, match="no HIP device"):
        load_fp4(m)


def test_product_does_not_import_the_oracle():
    pkg = os.path.join(ROOT, "crow_nest_amd")
    for dirpath, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".h", ".hip", ".cpp", "Makefile")):
                text = open(os.path.join(dirpath, f)).read()
                assert "oracle" not in text.lower(), (dirpath, f)


def test_group_layout_is_a_bijection_and_matches_the_matrix_operand_shape():
    """Every byte of a 2304-byte group (16 rows x 256 columns) is owned by exactly one (row, column) item, and the placement is
    the one the kernels assume: a lane's dword d of code half h is strip row lane % 16, pair 2 h + d / 2, segment d % 2, columns
    8 (lane / 16) .. + 7 of that segment; a lane's scale byte jj is row lane % 16, pair jj, segment g & 1, half g >> 1."""
    lib = L.lib()
    seen = set()
    for row in range(16):
        for wp in range(32):
            o = lib.crow_hip_tile_code_offset(row, wp)
            pair, seg, g = wp >> 3, (wp >> 2) & 1, wp & 3
            lane, h, d = 16 * g + row, pair >> 1, 2 * (pair & 1) + seg
            assert o == 256 + 1024 * h + 16 * lane + 4 * d and o % 4 == 0
            for b in range(4):
                assert o + b not in seen
                seen.add(o + b)
        for sb in range(16):
            o = lib.crow_hip_tile_scale_offset(row, sb)
            pair, seg, half = sb >> 2, (sb >> 1) & 1, sb & 1
            g = 2 * half + seg
            assert o == 4 * (16 * g + row) + pair and o < 256
            assert o not in seen
            seen.add(o)
    assert seen == set(range(2304))
    assert lib.crow_hip_tile_code_offset(16, 0) == 0xFFFFFFFF and lib.crow_hip_tile_scale_offset(0, 16) == 0xFFFFFFFF
