"""C-ABI checks that need no GPU: the library loads, exports every symbol the
header declares, its structs match the ctypes mirror, and invalid calls are
rejected with the documented status before anything is launched."""
import ctypes as C
import os
import re
import subprocess

import pytest
import torch

from ma import _hip_lib as L

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "ma_hip.h")


def declared_functions():
    src = open(HEADER).read()
    src = re.sub(r"/\*.*?\*/", "", src, flags=re.S)
    return sorted(set(re.findall(r"^\s*(?:const\s+char\s*\*|int|uint64_t)\s+(ma_\w+)\s*\(", src, flags=re.M)))


def test_header_declares_the_expected_entry_points():
    names = declared_functions()
    assert set(L.EXPORTS) <= set(names), names
    assert "ma_fwd" in names and "ma_r_step" in names


def test_library_exports_every_declared_symbol():
    lib = L.load()
    for name in declared_functions():
        assert hasattr(lib, name), f"libma_hip.so does not export {name}"
    assert lib.ma_abi_version() == L.ABI_VERSION


def test_struct_layout_matches_header(tmp_path):
    prog = tmp_path / "sz.c"
    prog.write_text(
        '#include <stdio.h>\n#include <stddef.h>\n#include "ma_hip.h"\n'
        "int main(void){printf(\"%zu %zu %zu %zu %zu %zu %zu %zu\\n\", sizeof(ma_fwd_params), offsetof(ma_fwd_params,E),"
        " offsetof(ma_fwd_params,q_stride), offsetof(ma_fwd_params,mask_stride), offsetof(ma_fwd_params,eps),"
        " offsetof(ma_fwd_params,error_word), sizeof(ma_bwd_params), sizeof(ma_ws_layout)); return 0;}\n")
    exe = tmp_path / "sz"
    subprocess.run(["gcc", "-std=c99", "-Wall", "-Werror", "-I", os.path.join(ROOT, "include"), str(prog), "-o", str(exe)],
                   check=True)
    got = [int(x) for x in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()]
    F = L.FwdParams
    assert got == [C.sizeof(F), F.E.offset, F.q_stride.offset, F.mask_stride.offset, F.eps.offset,
                   F.error_word.offset, C.sizeof(L.BwdParams), C.sizeof(L.WsLayout)]


def good_params(**kw):
    p = L.FwdParams()
    p.E, p.H, p.N, p.D, p.Dv, p.B, p.T = 2, 3, 50, 16, 16, 8, 2
    p.dtype_qk = p.dtype_v = L.MA_F16
    for name, inner in (("q_stride", 16), ("k_stride", 16), ("v_stride", 16), ("out_stride", 16)):
        setattr(p, name, (C.c_int64 * 3)(3 * 50 * inner, 50 * inner, inner))
    p.eps = 1e-12
    for k, v in kw.items():
        setattr(p, k, v)
    return p


def test_workspace_layout_is_ordered_and_aligned():
    lib = L.load()
    p = good_params()
    lay = L.WsLayout()
    assert lib.ma_fwd_workspace_layout(p, lay) == L.MA_OK
    offs = [lay.sync, lay.aR, lay.cR, lay.aL, lay.cL, lay.Y, lay.stats, lay.total]
    assert lay.sync == 0 and offs == sorted(offs) and all(o % 256 == 0 for o in offs)
    rows = 2 * 3 * 7 * 8                       # E*H*Np with Np = ceil(50/8)*8
    assert lay.cR - lay.aR >= rows * 16 * 2 and lay.aL - lay.cR >= rows * 4
    assert lib.ma_fwd_workspace_bytes(p) == lay.total


@pytest.mark.parametrize("field,value,status", [
    ("E", 0, L.MA_ERR_SHAPE), ("N", -3, L.MA_ERR_SHAPE), ("B", 0, L.MA_ERR_SHAPE), ("T", 0, L.MA_ERR_SHAPE),
    ("Dv", 0, L.MA_ERR_SHAPE), ("dtype_qk", 7, L.MA_ERR_DTYPE), ("dtype_v", -1, L.MA_ERR_DTYPE),
    ("variant", 9, L.MA_ERR_VARIANT), ("variant", -1, L.MA_ERR_VARIANT),
])
def test_invalid_problem_is_rejected(field, value, status):
    lib = L.load()
    p = good_params(**{field: value})
    assert lib.ma_fwd_workspace_layout(p, L.WsLayout()) == status
    assert lib.ma_fwd_workspace_bytes(p) == 0
    assert lib.ma_fwd(p, None) == status
    assert L.strerror(status)


def test_overlapping_rows_and_negative_strides_are_rejected():
    lib = L.load()
    p = good_params()
    p.q_stride = (C.c_int64 * 3)(2400, 800, 8)       # row stride < D
    assert lib.ma_fwd_workspace_bytes(p) == 0
    assert lib.ma_fwd(p, None) == L.MA_ERR_STRIDE
    p = good_params()
    p.v_stride = (C.c_int64 * 3)(-1, 800, 16)
    assert lib.ma_fwd(p, None) == L.MA_ERR_STRIDE
    p = good_params()
    if p.H > 1:                                       # output slices of different heads may not coincide
        p.out_stride = (C.c_int64 * 3)(p.out_stride[0], 0, p.out_stride[2])
        assert lib.ma_fwd(p, None) == L.MA_ERR_STRIDE
    p = good_params()
    p.k_stride = (C.c_int64 * 3)(0, 0, p.k_stride[2])  # inputs may be broadcast over batch and heads
    assert lib.ma_fwd_workspace_bytes(p) > 0


def test_pointer_and_workspace_checks_precede_any_launch():
    lib = L.load()
    p = good_params()
    assert lib.ma_fwd(p, None) == L.MA_ERR_NULL                      # q/k/v/out NULL
    p.q = p.k = p.v = p.out = 0x10000
    assert lib.ma_fwd(p, None) == L.MA_ERR_WORKSPACE                 # no workspace
    need = lib.ma_fwd_workspace_bytes(p)
    p.workspace, p.workspace_bytes = 0x100000, need - 1
    assert lib.ma_fwd(p, None) == L.MA_ERR_WORKSPACE                 # too small
    p.workspace, p.workspace_bytes = 0x100010, need
    assert lib.ma_fwd(p, None) == L.MA_ERR_WORKSPACE                 # misaligned
    p.workspace = 0x100000
    p.q = 0x10001                                                    # fp16 pointer must be 2-byte aligned
    assert lib.ma_fwd(p, None) == L.MA_ERR_STRIDE
    for fn in (lib.ma_l_step, lib.ma_z_step):
        assert fn(good_params(), None) == L.MA_ERR_NULL
    assert lib.ma_r_step(good_params(), 1, 0, None) == L.MA_ERR_NULL
    assert lib.ma_fwd(None, None) == L.MA_ERR_NULL
    # ma_matrix: NULL output, NULL q / k, missing workspace, one-launch variants
    assert lib.ma_matrix(good_params(), None, None) == L.MA_ERR_NULL
    assert lib.ma_matrix(good_params(), 0x20000, None) == L.MA_ERR_NULL
    pm = good_params()
    pm.q = pm.k = 0x10000
    assert lib.ma_matrix(pm, 0x20002, None) == L.MA_ERR_STRIDE         # fp32 output must be 4-byte aligned
    assert lib.ma_matrix(pm, 0x20000, None) == L.MA_ERR_WORKSPACE      # v / out are not needed
    for name in ("fused", "resident", "chained"):
        pm.variant = L.VARIANTS[name]
        assert lib.ma_matrix(pm, 0x20000, None) == L.MA_ERR_UNSUPPORTED
    pm.variant = 99
    assert lib.ma_matrix(pm, 0x20000, None) == L.MA_ERR_VARIANT


def test_select_variant_reports_a_known_variant():
    lib = L.load()
    v = lib.ma_fwd_select_variant(good_params())
    assert v in (L.VARIANTS["generic"], L.VARIANTS["staged"], L.VARIANTS["chained"], L.VARIANTS["resident"], L.VARIANTS["fused"])
    p32 = good_params(dtype_qk=L.MA_F32, dtype_v=L.MA_F32)
    assert lib.ma_fwd_select_variant(p32) in (L.VARIANTS["generic"], L.VARIANTS["staged"], L.VARIANTS["resident"])


def test_auto_resolves_to_a_variant_that_takes_the_problem():
    """Over a random sample of problems: what AUTO resolves to is a variant that accepts the problem when it is asked for
    by name, the answer does not depend on the device-ownership flag unless it is the team kernel, and a kernel name exists."""
    import random
    lib = L.load()
    rnd = random.Random(11)
    seen = set()
    for _ in range(4000):
        E, H = rnd.choice([1, 1, 2, 3, 4, 8, 16, 32, 64]), rnd.choice([1, 2, 3, 4, 6, 8, 12, 16])
        B = rnd.choice([8, 14, 16, 24, 32, 45, 48, 64, 80, 96, 128, 160, 256])
        M = rnd.choice([1, 2, 3, 4, 8, 13, 16, 24, 32, 46, 64, 90, 128, 200])
        N = max(1, M * B - rnd.randint(0, B - 1))
        D = rnd.choice([32, 40, 48, 60, 64, 72, 80, 96, 128])
        if E * H * N * D > 3e8:
            continue
        p = good_params()
        p.E, p.H, p.N, p.D, p.Dv, p.B, p.T = E, H, N, D, D, B, rnd.randint(1, 3)
        p.dtype_qk = p.dtype_v = rnd.choice([L.MA_F16, L.MA_BF16, L.MA_F32])
        for field in ("q_stride", "k_stride", "v_stride", "out_stride"):
            setattr(p, field, (C.c_int64 * 3)(H * N * D, N * D, D))
        p.variant, p.flags = L.VARIANTS["auto"], 0
        shared = lib.ma_fwd_select_variant(p)
        p.flags = L.MA_FLAG_DEVICE_EXCLUSIVE
        owned = lib.ma_fwd_select_variant(p)
        assert shared >= 0 and owned >= 0, (E, H, N, D, B)
        assert shared != L.VARIANTS["fused"]
        assert owned == shared or owned == L.VARIANTS["fused"], (E, H, N, D, B)
        assert lib.ma_fwd_kernel_name(p) is not None
        for v in (shared, owned):
            p.variant = v
            assert lib.ma_fwd_select_variant(p) == v, (E, H, N, D, B, v)
            seen.add(v)
    assert seen == {L.VARIANTS[n] for n in ("generic", "staged", "fused", "resident", "chained")}


def test_kernel_name_follows_the_resolved_variant():
    lib = L.load()

    def name(E, H, N, D, B, dt=L.MA_F16, T=2, variant="auto", flags=0):
        p = good_params()
        p.E, p.H, p.N, p.D, p.Dv, p.B, p.T, p.flags = E, H, N, D, D, B, T, flags
        p.dtype_qk = p.dtype_v = dt
        p.variant = L.VARIANTS[variant]
        for field in ("q_stride", "k_stride", "v_stride", "out_stride"):
            setattr(p, field, (C.c_int64 * 3)(H * N * D, N * D, D))
        got = lib.ma_fwd_kernel_name(p)
        return got.decode() if got is not None else None

    assert name(1, 16, 4096, 64, 64) == "chain_fwd_mfma"
    assert name(1, 16, 4096, 64, 64, flags=L.MA_FLAG_DEVICE_EXCLUSIVE) == "fused_fwd_mfma"
    assert name(64, 12, 256, 64, 16) == "resident_head_mfma"      # the head fits in LDS with its inputs
    assert name(64, 4, 197, 64, 16) == "resident_head_mfma"       # ... a head per compute unit: the widest workgroup
    assert name(64, 12, 197, 64, 16) == "resident_head2_mfma"     # three short heads per compute unit: narrow workgroups, two tiles each
    assert name(128, 12, 64, 64, 16, T=1) == "resident_head_mfma"    # ... and four tiles where four fit a share of the LDS
    assert name(128, 12, 64, 128, 16) == "resident_head2_mfma"        # (not in the 128-column class)
    assert name(16, 12, 512, 64, 32) == "resident_head2_mfma"     # twice that length: the state and one input tile at a time
    assert name(16, 12, 512, 64, 32, T=1) == "resident_head2_mfma"
    assert name(8, 12, 512, 64, 32) == "chain_fwd_mfma"           # ... 96 heads do not fill the device
    assert name(16, 12, 1000, 32, 32, variant="resident") == "resident_fwd_mfma"   # state only
    assert name(1, 16, 4096, 64, 256) == "r_step_long"            # stage kernels by the rows of a block
    assert name(1, 16, 4096, 64, 128, variant="staged") == "r_step_pair"
    assert name(1, 16, 4096, 64, 64, variant="staged") == "r_step_mfma"
    assert name(1, 1, 256, 64, 16, dt=L.MA_F32, T=1) == "head_t1_f32"
    assert name(1, 1, 256, 64, 16, dt=L.MA_F32, T=2) == "r_step_f32"
    assert name(8, 8, 197, 64, 16, dt=L.MA_F32) == "head_fwd_f32"
    assert name(1, 16, 4096, 60, 64) == "r_step_kernel"           # D % 8 != 0: the FMA kernels
    assert name(1, 16, 0, 64, 64) is None                         # invalid problem


def test_sliced_by_name():
    """The slice-resident kernel by name: wherever AUTO runs it, and beyond; refused outside of its sizes, by the paths that keep
    the state of the steps or run them as stages, and with operands of 32 bits."""
    lib = L.load()

    def params(heads, N, D, B, T=2, variant="sliced", dt=L.MA_F16):
        p = good_params()
        p.E, p.H, p.N, p.D, p.Dv, p.B, p.T, p.variant = heads, 1, N, D, D, B, T, L.VARIANTS[variant]
        p.dtype_qk = p.dtype_v = dt
        for field in ("q_stride", "k_stride", "v_stride", "out_stride"):
            setattr(p, field, (C.c_int64 * 3)(N * D, N * D, D))
        return p

    ran = 0
    for heads in (8, 64, 128, 192, 256, 512):
        for N, B in ((197, 14), (400, 20), (512, 32), (1024, 32), (1500, 40), (2304, 48), (3000, 60)):
            for D in (32, 48, 64, 72, 80):
                for T in (1, 2, 3):
                    if lib.ma_fwd_kernel_name(params(heads, N, D, B, T, "auto")) != b"resident_slice_mfma":
                        continue
                    ran += 1
                    p = params(heads, N, D, B, T)
                    assert lib.ma_fwd_select_variant(p) == L.VARIANTS["sliced"], (heads, N, D, B, T)
                    assert lib.ma_fwd_kernel_name(p) == b"resident_slice_mfma"
                    assert lib.ma_fwd_workspace_bytes(p) == lib.ma_fwd_workspace_bytes(params(heads, N, D, B, T, "chained"))
    assert ran > 100
    assert lib.ma_fwd_select_variant(params(1, 512, 64, 32)) == L.VARIANTS["sliced"]      # one head: AUTO would not
    for refused in (params(64, 1024, 96, 32), params(64, 1024, 64, 65), params(64, 2080, 64, 32), params(64, 1000, 60, 32),
                    params(64, 4096, 80, 64), params(64, 512, 64, 32, dt=L.MA_F32)):
        assert lib.ma_fwd_select_variant(refused) == L.MA_ERR_UNSUPPORTED
        assert lib.ma_fwd_kernel_name(refused) is None
    p = params(1, 512, 64, 32)
    p.q = p.k = p.v = p.out = p.workspace = 0x100000
    p.workspace_bytes = 1 << 40
    assert lib.ma_matrix(p, 0x20000, None) == L.MA_ERR_UNSUPPORTED
    assert lib.ma_fwd_keep(p, 0x100000, 1 << 40, None) == L.MA_ERR_UNSUPPORTED
    assert lib.ma_r_step(p, 1, 0, None) == L.MA_ERR_UNSUPPORTED
    b = L.BwdParams()
    b.fwd = p
    b.dq_stride = b.dk_stride = b.dv_stride = b.dout_stride = (C.c_int64 * 3)(512 * 64, 512 * 64, 64)
    assert lib.ma_bwd_workspace_bytes(b) == 0


def test_auto_runs_slices_where_they_are_faster():
    """AUTO's choice between the slice-resident kernel and the one it stands in for, at shapes where one of the two took at most
    0.92 of the other's time (us on an MI355X: slices, the other)."""
    lib = L.load()
    for heads, N, D, B, T, slices, other in (
            # few blocks, more slices than compute units
            (768, 71, 32, 43, 2, 47.9, 22.1), (512, 36, 32, 37, 2, 32.5, 13.9), (512, 36, 32, 41, 3, 45.0, 18.7), (320, 127, 32, 33, 3, 32.3, 22.8),
            (384, 246, 32, 43, 1, 19.8, 16.0), (128, 29, 72, 18, 3, 16.8, 12.3), (128, 4, 80, 23, 2, 12.2, 10.2),
            # a last round of few waves or a last pass of few slices
            (224, 1234, 40, 20, 2, 125.0, 87.2), (320, 885, 72, 25, 2, 152.7, 125.6), (320, 749, 48, 20, 2, 108.9, 87.0), (256, 712, 72, 20, 4, 192.6, 160.6),
            (320, 548, 72, 15, 4, 187.5, 147.8), (128, 2002, 32, 34, 4, 181.1, 149.8), (192, 254, 72, 14, 6, 59.3, 52.6),
            # a single pass; few heads at a single step
            (78, 470, 32, 48, 1, 7.6, 9.4), (80, 300, 32, 40, 1, 7.1, 8.5), (128, 214, 72, 32, 1, 10.4, 11.6), (2, 192, 48, 15, 1, 7.4, 6.5),
            (4, 192, 48, 14, 1, 7.2, 6.6),
            # 33 .. 48 rows, which the chained kernel runs in workgroups of three waves
            (96, 1361, 32, 41, 4, 95.7, 73.3), (97, 1243, 32, 37, 3, 70.1, 57.2), (626, 423, 64, 40, 2, 104.1, 90.6), (456, 418, 48, 13, 2, 66.6, 58.7),
            (256, 1503, 64, 45, 2, 123.2, 160.7), (512, 1523, 32, 45, 2, 153.7, 220.5),
            # the slices' own ground
            (128, 1024, 72, 32, 3, 46.3, 77.6), (112, 260, 40, 20, 1, 8.7, 10.2), (128, 384, 40, 24, 1, 9.4, 10.9), (128, 512, 64, 32, 2, 17.1, 26.0)):
        p = good_params()
        p.E, p.H, p.N, p.D, p.Dv, p.B, p.T, p.variant = heads, 1, N, D, D, B, T, L.VARIANTS["auto"]
        p.dtype_qk = p.dtype_v = L.MA_F16
        for field in ("q_stride", "k_stride", "v_stride", "out_stride"):
            setattr(p, field, (C.c_int64 * 3)(N * D, N * D, D))
        assert (lib.ma_fwd_kernel_name(p) == b"resident_slice_mfma") == (slices < other), (heads, N, D, B, T)


def test_auto_records_with_slices_where_they_are_faster():
    """The same choice for recorded calls, which write the states of all steps (us on an MI355X: slices, chained)."""
    lib = L.load()
    for heads, N, D, B, T, slices, chained in (
            (38, 834, 64, 32, 3, 35.5, 28.0), (180, 1351, 64, 39, 4, 240.2, 173.3), (192, 59, 64, 43, 4, 63.2, 29.6), (88, 1572, 32, 27, 1, 30.8, 20.9),
            (1, 103, 72, 7, 2, 14.6, 12.3), (12, 218, 40, 14, 2, 14.4, 12.8), (18, 143, 80, 16, 2, 15.7, 14.4), (192, 1385, 64, 64, 2, 110.7, 92.2), (16, 673, 40, 16, 2, 40.4, 14.5), (12, 512, 64, 32, 2, 15.3, 13.3), (64, 1024, 64, 32, 2, 28.8, 24.3),
            (768, 197, 64, 14, 2, 40.4, 51.5), (384, 256, 64, 16, 2, 26.5, 33.5), (1411, 144, 32, 7, 4, 113.5, 157.4), (61, 63, 32, 5, 4, 16.5, 23.2),
            (453, 173, 80, 14, 4, 54.9, 74.7), (1244, 255, 48, 16, 1, 43.7, 66.4), (221, 42, 40, 5, 2, 12.3, 15.7), (512, 716, 32, 32, 4, 130.0, 171.5)):
        name = lib.ma_fwd_keep_kernel_name(call_params(heads, N, D, B, T).fwd)
        assert name == (b"resident_slice_mfma" if slices < chained else b"chain_fwd_mfma"), (heads, N, D, B, T)


def call_params(heads, N, D, B, T=2, variant="auto", dt=L.MA_BF16):
    """A backward call on contiguous tensors (its `fwd`: the recorded forward and the matrix call), with addresses that are never read."""
    b = L.BwdParams()
    b.fwd = good_params()
    p = b.fwd
    p.E, p.H, p.N, p.D, p.Dv, p.B, p.T, p.variant = heads, 1, N, D, D, B, T, L.VARIANTS[variant]
    p.dtype_qk = p.dtype_v = dt
    for field in ("q_stride", "k_stride", "v_stride", "out_stride"):
        setattr(p, field, (C.c_int64 * 3)(N * D, N * D, D))
    b.dout_stride = b.dq_stride = b.dk_stride = b.dv_stride = (C.c_int64 * 3)(N * D, N * D, D)
    p.q = p.k = p.v = p.out = b.dout = b.dq = b.dk = b.dv = 0x100000
    return b


def matrix_kernel(b):
    return L.load().ma_matrix_kernel_name(b.fwd, 0x100000)


def test_kernel_names_of_recorded_matrix_and_backward_calls():
    lib = L.load()
    assert lib.ma_fwd_keep_kernel_name(call_params(768, 197, 64, 14).fwd) == b"resident_slice_mfma"
    assert lib.ma_fwd_keep_kernel_name(call_params(192, 512, 64, 32).fwd) == b"chain_fwd_mfma"
    assert lib.ma_fwd_keep_kernel_name(call_params(192, 512, 64, 32, variant="staged").fwd) == b"r_step_mfma"
    assert lib.ma_fwd_keep_kernel_name(call_params(192, 512, 64, 32, dt=L.MA_F32).fwd) == b"r_step_f32"
    assert lib.ma_fwd_keep_kernel_name(call_params(192, 512, 60, 32, variant="generic").fwd) == b"r_step_kernel"
    assert lib.ma_fwd_keep_kernel_name(call_params(192, 512, 64, 32, variant="resident").fwd) is None
    assert matrix_kernel(call_params(12, 1024, 64, 32)) == b"matrix_slice_mfma"
    assert matrix_kernel(call_params(12, 1024, 64, 32, variant="staged")) == b"matrix_tile"
    assert matrix_kernel(call_params(12, 1024, 64, 32, dt=L.MA_F32)) == b"matrix_tile"
    assert matrix_kernel(call_params(12, 1024, 64, 32, variant="generic")) == b"matrix_kernel"
    assert matrix_kernel(call_params(12, 1024, 64, 32, variant="chained")) is None
    assert lib.ma_bwd_kernel_name(call_params(192, 512, 64, 32)) == b"head_bwd"
    assert lib.ma_bwd_kernel_name(call_params(192, 2048, 64, 64)) == b"r_bwd_tile"
    assert lib.ma_bwd_kernel_name(call_params(192, 512, 64, 32, variant="generic")) == b"r_bwd_kernel"
    assert lib.ma_bwd_kernel_name(call_params(192, 512, 64, 32, variant="chained")) is None
    without = call_params(192, 512, 64, 32)
    without.dq = None
    assert lib.ma_bwd_kernel_name(without) == b"r_bwd_kernel"


def test_staged_backward_of_short_heads_runs_the_stage_launches():
    """The one-launch backward is AUTO's; STAGED asks for the stage launches and their workspace, where AUTO would not choose them."""
    lib = L.load()
    for heads, N, D, B, T in ((192, 512, 64, 32, 2), (768, 197, 64, 14, 2), (12, 256, 64, 16, 3)):
        assert lib.ma_bwd_kernel_name(call_params(heads, N, D, B, T)) == b"head_bwd"
        assert lib.ma_bwd_kernel_name(call_params(heads, N, D, B, T, "staged")) == b"r_bwd_tile"
        one, stages = (lib.ma_bwd_kept_workspace_bytes(call_params(heads, N, D, B, T, v)) for v in ("auto", "staged"))
        state = heads * N * D * 2
        assert 0 < one and stages >= one + 3 * state   # gaL, gY and gaR


def test_head_counts_beyond_the_work_items_of_one_launch():
    """A dispatch counts its work items in 32 bits: workgroups of 512 and 1024 threads run out of them before the stage launches' do."""
    lib = L.load()
    most = (2 ** 32 - 1) // 512 // 8 * 8
    assert lib.ma_bwd_kernel_name(call_params(most, 64, 24, 8)) == b"head_bwd"
    assert lib.ma_bwd_kernel_name(call_params(most + 1, 64, 24, 8)) == b"r_bwd_tile"
    most = (2 ** 32 - 1) // 1024 // 8 * 8
    assert matrix_kernel(call_params(most, 12, 32, 4)) == b"matrix_slice_mfma"   # (four positions: one workgroup a head)
    assert matrix_kernel(call_params(most + 1, 12, 32, 4)) == b"matrix_tile"


def test_chained_launches_of_more_than_2_to_the_32_work_items_are_refused():
    """Many steps of many heads: the sync words have room for them, a dispatch of eight-wave workgroups has not."""
    lib = L.load()
    for heads, N, D, B, T, fits in ((2728, 10240, 72, 128, 16, False), (2728, 10240, 128, 80, 16, False), (2400, 10240, 72, 128, 16, True),
                                    (2728, 10240, 64, 128, 16, True), (2728, 16384, 72, 128, 16, True)):   # (the last two: workgroups of four waves)
        p = call_params(heads, N, D, B, T, "chained").fwd
        assert lib.ma_fwd_kernel_name(p) == (b"chain_fwd_mfma" if fits else None), (heads, N, D, B, T)
        if not fits:
            p.eps, p.workspace, p.workspace_bytes = 1e-12, 0x100000, 1 << 50
            assert lib.ma_fwd(p, None) == L.MA_ERR_UNSUPPORTED
            assert lib.ma_fwd_keep(p, 0x100000, 1 << 50, None) == L.MA_ERR_UNSUPPORTED
            p.variant = L.VARIANTS["auto"]
            assert lib.ma_fwd_kernel_name(p) == b"r_step_pair" and lib.ma_fwd_keep_kernel_name(p) == b"r_step_pair"


def test_auto_runs_the_one_launch_backward_where_it_is_faster():
    """AUTO's choice for the backward of short heads, at shapes where one side took at most 0.85 of the other's time (us of the backward
    alone on an MI355X: one launch, stage launches)."""
    lib = L.load()
    for heads, N, D, B, T, one, stages in (
            # few heads of 17 .. 32 rows one way; few blocks, of which most waves have none
            (10, 460, 8, 30, 2, 28.0, 15.8), (14, 332, 24, 31, 2, 25.9, 16.7), (2, 249, 8, 12, 2, 22.5, 15.0), (27, 161, 64, 7, 2, 27.7, 20.2),
            (21, 422, 8, 32, 2, 28.6, 17.5), (640, 14, 24, 19, 2, 43.0, 30.7), (1024, 37, 8, 30, 1, 39.1, 30.3), (768, 3, 96, 22, 2, 96.4, 67.4),
            (1937, 16, 40, 7, 2, 79.4, 50.8), (2886, 3, 72, 12, 1, 88.9, 49.5), (2, 214, 96, 14, 1, 15.9, 10.8),
            # its own ground
            (192, 512, 64, 32, 2, 58.0, 84.0), (768, 197, 64, 14, 2, 72.0, 142.0), (23, 10, 96, 1, 3, 19.5, 27.4), (287, 178, 24, 15, 3, 39.0, 57.5),
            (420, 281, 24, 32, 4, 96.6, 129.1), (1082, 557, 24, 20, 1, 124.7, 161.1), (224, 243, 48, 32, 2, 35.7, 49.5), (256, 53, 8, 26, 3, 27.4, 37.1),
            (212, 567, 32, 31, 2, 51.6, 71.7), (192, 148, 24, 6, 3, 28.6, 47.9)):
        name = lib.ma_bwd_kernel_name(call_params(heads, N, D, B, T))
        assert name == (b"head_bwd" if one < stages else b"r_bwd_tile"), (heads, N, D, B, T)


def test_auto_writes_the_matrix_in_one_launch_where_it_is_faster():
    """AUTO's choice for the matrix of short sequences, at shapes where one side took at most 0.91 of the other's time (us on an MI355X, mean
    of a replayed graph, calls from the host and calls that are waited for: one launch, stage launches)."""
    for heads, N, D, B, T, one, stages in (
            # workgroups with work for few waves; large matrices of one step; few heads of wide rows
            (1500, 3, 72, 1, 2, 46.3, 26.7), (1551, 28, 72, 18, 4, 209.6, 129.2), (1379, 10, 48, 1, 1, 33.7, 22.0), (1550, 13, 40, 1, 2, 60.2, 42.3),
            (85, 975, 32, 32, 1, 112.1, 89.5), (2, 321, 128, 13, 1, 19.5, 14.7), (11, 122, 128, 4, 2, 29.0, 23.1), (20, 162, 72, 6, 1, 16.9, 14.2),
            # its own ground
            (12, 1024, 64, 32, 2, 21.9, 25.1), (243, 76, 128, 11, 2, 13.7, 34.4), (5, 19, 32, 14, 3, 8.7, 19.0), (65, 12, 64, 6, 3, 9.9, 20.8),
            (192, 348, 72, 15, 1, 33.7, 46.4), (595, 60, 64, 9, 2, 29.6, 43.0)):
        name = matrix_kernel(call_params(heads, N, D, B, T))
        assert name == (b"matrix_slice_mfma" if one < stages else b"matrix_tile"), (heads, N, D, B, T)


def test_check_maps_status_to_python_exceptions():
    with pytest.raises(ValueError):
        L.check(L.MA_ERR_SHAPE, "x")
    with pytest.raises(NotImplementedError):
        L.check(L.MA_ERR_UNSUPPORTED, "x")
    with pytest.raises(RuntimeError):
        L.check(L.MA_ERR_WORKSPACE, "x")
    L.check(L.MA_OK, "x")


def test_auto_variant_policy():
    """AUTO: generic when the MFMA kernels do not apply; resident for many heads of small problems
    whose state fits in LDS; the fused kernel for 8 or 16 heads of ~4096 tokens in 64-row problems, but
    only for callers that state that they own the device (MA_FLAG_DEVICE_EXCLUSIVE);
    per-stage launches where the one-launch kernels are at a disadvantage (uneven head counts of 128-row problems, wide heads with many blocks,
    very few long heads); the chained kernel otherwise."""
    lib = L.load()

    def auto(E, H, N, D, B, dt=L.MA_F16, Dv=None, T=2, exclusive=False):
        p = L.FwdParams()
        p.flags = L.MA_FLAG_DEVICE_EXCLUSIVE if exclusive else 0
        p.E, p.H, p.N, p.D, p.Dv, p.B, p.T = E, H, N, D, Dv or D, B, T
        p.dtype_qk = p.dtype_v = dt
        for name, w in (("q_stride", D), ("k_stride", D), ("v_stride", p.Dv), ("out_stride", p.Dv)):
            setattr(p, name, (C.c_int64 * 3)(H * N * w, N * w, w))
        p.eps = 1e-12
        return L.VARIANT_NAMES[lib.ma_fwd_select_variant(p)]

    ex = dict(exclusive=True)
    assert auto(1, 16, 4096, 64, 64, **ex) == "fused"         # 16 heads x 64 workgroups: every head has a full team at once
    assert auto(1, 16, 4096, 64, 64, T=1, **ex) == "fused"
    assert auto(2, 16, 4096, 64, 64, **ex) == "chained"
    assert auto(1, 8, 8192, 64, 64, **ex) == "fused"          # with more than one step also 128 tasks per phase: 8 heads of 8192 tokens,
    assert auto(1, 16, 4096, 64, 128, **ex) == "fused"        # 16 heads of 4096 in 128-row blocks (two positions per workgroup)
    assert auto(1, 8, 8192, 72, 128, **ex) == "fused"         # 8 heads also with head dims up to 80
    # the fused kernel's workgroups wait for each other: without the caller's word that the device is its
    # own, AUTO stays with kernels that make progress beside any other work
    for T_ in (1, 2, 3):
        for shape in ((1, 16, 4096, 64, 64), (1, 8, 8192, 64, 64), (1, 16, 4096, 64, 128), (1, 8, 8192, 72, 128)):
            assert auto(*shape, T=T_) in ("chained", "staged"), (shape, T_)
    assert auto(1, 16, 4096, 64, 64) == "chained"
    assert auto(1, 16, 4096, 64, 64, T=1) == "chained"
    assert auto(1, 16, 4096, 72, 64) == "chained"       # ... 16 heads not
    assert auto(1, 8, 6144, 64, 64) == "chained"        # 96 blocks: the team kernel would run them as 128
    assert auto(1, 8, 8192, 64, 64, T=1) == "staged"    # a single step: two launches
    assert auto(1, 8, 4096, 64, 64, T=1) == "chained"   # ... and teams only when they fill every workgroup slot (16 heads)
    assert auto(1, 8, 2048, 64, 128, T=1) == "staged"   # few 128-row problems: the stage launches run them as halves
    assert auto(1, 16, 2048, 64, 128, T=1) == "chained" # ... 256 of them on 16 heads: one launch again
    assert auto(1, 4, 4096, 64, 128) == "staged"        # more steps: only very few problems, or at most 4 heads
    assert auto(1, 8, 2048, 64, 128) == "chained"
    assert auto(1, 8, 1024, 64, 32) == "chained"        # teams of 16 workgroups: the chained kernel is ahead
    assert auto(1, 12, 4096, 64, 64) == "chained"       # 12 heads do not sit evenly on 8 XCDs: no teams
    assert auto(1, 12, 4096, 64, 64, T=1) == "staged"   # ... and with a single step two launches beat an unbalanced one
    assert auto(1, 16, 16384, 64, 128) == "chained"     # 128-row problems both ways, heads even over the XCDs
    assert auto(1, 12, 16384, 64, 128) == "staged"      # 12 heads on 8 XCDs: uneven
    assert auto(16, 12, 512, 64, 128) == "chained"      # 192 heads of four 128-row blocks: several positions per L / Z tile
    assert auto(16, 12, 384, 64, 96) == "chained"       # ... also for 96-row blocks
    assert auto(1, 16, 8192, 64, 90) == "chained"       # 92 blocks of 90 rows: the chained kernel has the 96-row class too
    assert auto(64, 12, 197, 64, 16) == "resident"
    assert auto(16, 12, 512, 64, 32) == "resident"     # 512-token heads: the state and one input tile at a time in LDS
    assert auto(8, 12, 512, 64, 32) == "chained"       # ... when there are enough heads for the compute units (a head has one to itself)
    assert auto(32, 12, 512, 64, 32) == "resident"     # (384 heads, 1.5 passes over 256 CUs: still 0.85 of the chained kernel's time)
    assert auto(16, 12, 512, 64, 32, T=1) == "resident"
    assert auto(8, 16, 512, 64, 32) == "resident"      # 128 heads: for long heads that are a single strip one way
    assert auto(8, 16, 500, 64, 24) == "chained"
    assert auto(8, 16, 512, 64, 32, T=1) == "chained"
    assert auto(8, 24, 256, 128, 16) == "resident"     # head dim 128: 256 tokens are a two-tile head
    assert auto(8, 24, 272, 128, 16) == "chained"      # ... longer ones only in whole passes over the compute units
    assert auto(8, 32, 272, 128, 16) == "resident"
    assert auto(16, 12, 512, 64, 64) == "chained"      # 64-row blocks (eight waves per workgroup)
    assert auto(16, 12, 768, 64, 32) == "chained"      # beyond two tiles: the one-tile form is no match for the chained kernel here
    assert auto(16, 12, 512, 64, 64) == "chained"      # ... and for problems of one or two strips
    assert auto(32, 12, 256, 64, 64) == "chained"      # 64-row blocks never run resident
    assert auto(16, 12, 256, 64, 32) == "resident"     # 256-token heads fit in LDS with their inputs: from 128 heads on
    assert auto(2, 16, 256, 64, 32) == "chained"       # ... fewer heads of 32-row blocks stay with the chained kernel
    assert auto(1, 2, 256, 64, 16) == "resident"       # ... those of 16-row blocks do not when there is more than one step
    assert auto(1, 2, 256, 64, 16, T=1) == "chained"
    assert auto(16, 12, 197, 64, 16, T=1) == "resident"
    assert auto(8, 16, 1024, 72, 32) == "chained"
    assert auto(4, 16, 16384, 64, 128) == "chained"
    assert auto(512, 16, 1024, 64, 32) == "staged"      # more heads than the chained kernel has flag words for
    assert auto(2, 16, 8192, 64, 64) == "chained"       # 128 blocks of 64 rows (long documents), head dim 64
    assert auto(2, 16, 8192, 128, 64) == "staged"       # ... but not for wide heads
    assert auto(1, 16, 8192, 128, 64) == "chained"      # ... under 48 MB a tensor
    assert auto(8, 8, 8192, 72, 64) == "staged"         # D = 72, 128 blocks, 72 MB a tensor: with more than one step
    assert auto(8, 8, 8192, 72, 64, T=1) == "chained"
    assert auto(8, 8, 8192, 72, 96) == "chained"        # 65 .. 96 rows: only at the head dims of the 96-column class
    assert auto(8, 8, 8192, 96, 96) == "staged"
    assert auto(4, 8, 8192, 128, 96) == "chained"
    assert auto(2, 16, 5000, 64, 64) == "chained"       # 79 blocks: the 96-row class
    assert auto(1, 2, 8192, 64, 64) == "staged"         # two long heads would run on two of the eight XCDs
    assert auto(2, 2, 197, 64, 16) == "resident"        # few short heads in 16-row blocks, two steps: whole in LDS
    assert auto(2, 2, 197, 64, 16, T=1) == "chained"    # ... a single step: one launch of the chained kernel
    assert auto(1, 1, 16, 64, 4) == "resident"
    assert auto(1, 1, 16, 64, 4, T=1) == "chained"
    assert auto(1, 16, 4096, 64, 64, dt=L.MA_F32) == "staged"       # fp32 MFMA stage kernels
    assert auto(1, 2, 7600, 48, 128, dt=L.MA_F32) == "staged"
    assert auto(1, 1, 256, 64, 16, dt=L.MA_F32, T=1) == "resident"  # few small fp32 heads, one step: a workgroup per (head, position)
    assert auto(1, 1, 256, 64, 16, dt=L.MA_F32, T=2) == "staged"    # ... more steps: spread over compute units by the stage launches
    assert auto(1, 17, 256, 64, 16, dt=L.MA_F32, T=1) == "staged"   # ... more than 256 workgroups likewise
    assert auto(8, 8, 197, 64, 16, dt=L.MA_F32) == "resident"       # from 64 heads on: one workgroup per head, one launch
    assert auto(64, 12, 197, 64, 16, dt=L.MA_F32) == "resident"
    assert auto(1, 2, 128, 32, 16, dt=L.MA_F32) == "resident"       # ... and for very small heads always
    assert auto(8, 8, 272, 64, 16, dt=L.MA_F32) == "staged"         # 17 blocks
    assert auto(8, 8, 256, 80, 16, dt=L.MA_F32) == "staged"         # head dim above 64
    assert auto(1, 16, 16384, 128, 128, dt=L.MA_F32) == "staged"    # fp32 stage kernels up to 256 rows and 128 columns (tiles in chunks)
    assert auto(1, 16, 65536, 128, 256, dt=L.MA_F32) == "staged"
    assert auto(1, 16, 4096, 128, 257, dt=L.MA_F32) == "generic"
    assert auto(1, 16, 4096, 62, 64, dt=L.MA_F32) == "generic"      # D % 4 != 0
    assert auto(1, 16, 4096, 64, 64, Dv=128) == "generic"
    assert auto(1, 16, 4096, 60, 64) == "generic"       # D % 8 != 0
    assert auto(1, 16, 4096, 64, 256) == "staged"       # blocks of 129 .. 256 rows: per-stage launches only
    assert auto(1, 16, 32768, 64, 128) == "staged"      # 129 .. 256 blocks likewise (heads of up to 65536 tokens)
    assert auto(1, 16, 65536, 64, 256) == "staged"
    assert auto(1, 16, 4096, 64, 257) == "generic"      # B > 256
    for name in ("fused", "chained", "resident"):       # the one-launch kernels stop at 128 rows
        p = L.FwdParams()
        p.E, p.H, p.N, p.D, p.Dv, p.B, p.T = 1, 16, 4096, 64, 64, 256, 2
        p.dtype_qk = p.dtype_v = L.MA_F16
        for field in ("q_stride", "k_stride", "v_stride", "out_stride"):
            setattr(p, field, (C.c_int64 * 3)(4096 * 64, 4096 * 64, 64))
        p.eps = 1e-12
        p.variant = L.VARIANTS[name]
        assert lib.ma_fwd_select_variant(p) == L.MA_ERR_UNSUPPORTED
    assert auto(1, 16, 65537, 64, 256) == "generic"     # more than 256 blocks


def good_bwd_params(**kw):
    b = L.BwdParams()
    b.fwd = good_params(**kw)
    for name, inner in (("dout_stride", 16), ("dq_stride", 16), ("dk_stride", 16), ("dv_stride", 16)):
        setattr(b, name, (C.c_int64 * 3)(3 * 50 * inner, 50 * inner, inner))
    return b


def test_backward_workspace_and_argument_checks_precede_any_launch():
    """ma_bwd validates before it launches: everything here runs without a GPU."""
    lib = L.load()
    b = good_bwd_params()
    need = lib.ma_bwd_workspace_bytes(b)
    rows, T, D = 2 * 3 * 7 * 8, 2, 16
    # every step's state (T aL + T-1 aR slots of 16-bit rows), fp32 state gradients and fp32 dq, dk, dv
    assert need >= (2 * T - 1) * rows * D * 2 + 3 * rows * D * 4 + 3 * rows * D * 4
    assert need % 256 == 0
    assert lib.ma_bwd_workspace_bytes(good_bwd_params(T=3)) > need
    assert lib.ma_bwd(None, None) == L.MA_ERR_NULL
    assert lib.ma_bwd(b, None) == L.MA_ERR_NULL                        # q / k / v / dout / dq / dk / dv NULL
    b.fwd.q = b.fwd.k = b.fwd.v = b.dout = b.dq = b.dk = b.dv = 0x10000
    assert lib.ma_bwd(b, None) == L.MA_ERR_WORKSPACE                   # fwd.out is not needed; no workspace
    b.fwd.workspace, b.fwd.workspace_bytes = 0x100000, need - 1
    assert lib.ma_bwd(b, None) == L.MA_ERR_WORKSPACE                   # too small
    b.fwd.workspace, b.fwd.workspace_bytes = 0x100010, need
    assert lib.ma_bwd(b, None) == L.MA_ERR_WORKSPACE                   # misaligned
    b.fwd.workspace = 0x100000
    b.dq = 0x10001                                                     # fp16 pointer must be 2-byte aligned
    assert lib.ma_bwd(b, None) == L.MA_ERR_STRIDE
    b.dq = 0x10000
    for name in ("fused", "resident", "chained"):                      # the T steps run as separate launches
        b.fwd.variant = L.VARIANTS[name]
        assert lib.ma_bwd(b, None) == L.MA_ERR_UNSUPPORTED
        assert lib.ma_bwd_workspace_bytes(b) == 0
    b.fwd.variant = L.VARIANTS["auto"]
    b.dk_stride = (C.c_int64 * 3)(0, 50 * 16, 16)                      # gradient slices of batch entries coincide
    assert lib.ma_bwd(b, None) == L.MA_ERR_STRIDE
    b.dk_stride = (C.c_int64 * 3)(3 * 50 * 16, 50 * 16, 8)             # rows of dk overlap
    assert lib.ma_bwd(b, None) == L.MA_ERR_STRIDE
    bad = good_bwd_params(B=5000)                                      # beyond the backward kernels' block size
    bad.fwd.N = 20000
    bad.fwd.q = bad.fwd.k = bad.fwd.v = bad.dout = bad.dq = bad.dk = bad.dv = 0x10000
    for name in ("q_stride", "k_stride", "v_stride", "out_stride"):
        setattr(bad.fwd, name, (C.c_int64 * 3)(3 * 20000 * 16, 20000 * 16, 16))
    for name in ("dout_stride", "dq_stride", "dk_stride", "dv_stride"):
        setattr(bad, name, (C.c_int64 * 3)(3 * 20000 * 16, 20000 * 16, 16))
    need = lib.ma_bwd_workspace_bytes(bad)
    bad.fwd.workspace, bad.fwd.workspace_bytes = 0x100000, need
    assert need > 0 and lib.ma_bwd(bad, None) == L.MA_ERR_UNSUPPORTED


def test_workspaces_hold_what_the_path_uses():
    """Bytes a row: what the tiled backward kernels keep (state gradients in the operand type, fp32 dq and, with more than one
    step, dk) and nothing for the other kernels; the matrix call's probabilities only where they are kept."""
    lib = L.load()
    E, H, N, D, B, es = 1, 16, 8192, 64, 64, 2
    rows = H * N

    def params(T, align, variant="auto"):
        b = L.BwdParams()
        p = b.fwd
        p.E, p.H, p.N, p.D, p.Dv, p.B, p.T = E, H, N, D, D, B, T
        p.dtype_qk = p.dtype_v = L.MA_BF16
        p.eps, p.variant = 1e-12, L.VARIANTS[variant]
        for name in ("q_stride", "k_stride", "v_stride", "out_stride"):
            setattr(p, name, (C.c_int64 * 3)(H * N * D, N * D, D))
        for name in ("dout_stride", "dq_stride", "dk_stride", "dv_stride"):
            setattr(b, name, (C.c_int64 * 3)(H * N * D, N * D, D))
        if align:
            p.q = p.k = p.v = b.dout = b.dq = b.dk = b.dv = align
        return b

    slack = 16 * 256
    for T, per_row in ((1, 2 * D * es + 4 + 16 + 4 * D), (2, 3 * D * es + 8 + 16 + 2 * 4 * D), (3, 3 * D * es + 8 + 16 + 2 * 4 * D)):
        need = lib.ma_bwd_kept_workspace_bytes(params(T, 0x10000))
        assert rows * per_row <= need <= rows * per_row + slack
        assert lib.ma_bwd_kept_workspace_bytes(params(T, 0x10002)) > need         # other kernels: fp32 throughout
        assert lib.ma_bwd_kept_workspace_bytes(params(T, 0)) >= lib.ma_bwd_kept_workspace_bytes(params(T, 0x10002))
        b = params(T, 0x10000)
        b.fwd.workspace, b.fwd.workspace_bytes = 0x100000, need - 1
        assert lib.ma_bwd_kept(b, 0x200000, lib.ma_fwd_state_bytes(b.fwd), None) == L.MA_ERR_WORKSPACE
    p = params(2, 0).fwd
    assert lib.ma_matrix_workspace_bytes(p) == lib.ma_fwd_workspace_bytes(p) + rows * B * 4
    p.D = 60   # D % 8 != 0: the FMA writer
    p.Dv = 60
    assert lib.ma_matrix_workspace_bytes(p) == lib.ma_fwd_workspace_bytes(p)
    assert lib.ma_matrix_workspace_bytes(params(2, 0, "generic").fwd) == lib.ma_fwd_workspace_bytes(params(2, 0).fwd)


def test_workspace_of_the_one_launch_backward():
    """fp32 rows of dq and dk only where they go through memory: dq from ~ 270 tokens of 64 columns on, dk where a wave's strips of it outgrow
    64 registers, with more than one step.  dv and the state's gradients never do."""
    lib = L.load()
    for heads, N, D, B, T, arrays in ((768, 197, 64, 14, 2, 0), (192, 512, 64, 32, 2, 1), (256, 512, 64, 32, 1, 1), (192, 1000, 32, 32, 2, 1),
                                      (192, 250, 96, 16, 2, 1), (192, 480, 64, 24, 3, 2), (224, 243, 48, 32, 2, 0), (16 * 16, 323, 96, 17, 1, 1)):
        b = call_params(heads, N, D, B, T)
        assert lib.ma_bwd_kernel_name(b) == b"head_bwd"
        rows = heads * -(-N // B) * B
        assert arrays * rows * D * 4 <= lib.ma_bwd_kept_workspace_bytes(b) <= arrays * rows * D * 4 + 16 * 256, (heads, N, D, B, T)


@pytest.mark.parametrize("variant,D,dt", [("staged", 8, L.MA_F16), ("staged", 8, L.MA_F32), ("generic", 3, L.MA_F16), ("sliced", 32, L.MA_F16)])
def test_launches_of_more_than_2_to_the_32_work_items_are_refused(variant, D, dt):
    """The runtime would run some of the workgroups and report nothing.  2^27 heads of one token."""
    lib = L.load()
    b = call_params(2 ** 27, 1, D, 1, 2, variant, dt)
    p = b.fwd
    p.eps = 1e-12
    p.workspace = 0x100000
    p.workspace_bytes = 1 << 50
    assert lib.ma_fwd(p, None) == L.MA_ERR_UNSUPPORTED
    if variant == "sliced":
        return
    for fn in (lambda: lib.ma_r_step(p, 1, 1, None), lambda: lib.ma_l_step(p, None), lambda: lib.ma_z_step(p, None),
               lambda: lib.ma_fwd_keep(p, 0x100000, 1 << 50, None), lambda: lib.ma_matrix(p, 0x100000, None)):
        assert fn() == L.MA_ERR_UNSUPPORTED
    if variant == "staged":   # (GENERIC clears its accumulators first)
        assert lib.ma_bwd_kept(b, 0x100000, 1 << 50, None) == L.MA_ERR_UNSUPPORTED
