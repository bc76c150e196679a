"""Properties of the compiled device code that the sources rely on but the compiler does not check (CPU only: the
kernels are cross-compiled to assembly, nothing runs).  The library's Makefile runs the first check on every build."""
import importlib.util
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flash-3-way-attention_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def _checker():
    spec = importlib.util.spec_from_file_location("check_m0", os.path.join(CSRC, "check_m0.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod.check


_compiled = {}


def _assembly(tmp_path, unit):
    if unit in _compiled:
        return _compiled[unit]
    out = tmp_path / "unit.s"
    flags = ["-O3", "-std=c++20", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
             "-Wno-unused-command-line-argument", "--cuda-device-only", "-S"]
    subprocess.run([HIPCC, *flags, os.path.join(CSRC, unit), "-o", str(out)], check=True,
                   stderr=subprocess.DEVNULL, cwd=CSRC)
    _compiled[unit] = out.read_text()
    return _compiled[unit]


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
@pytest.mark.parametrize("unit", ["tdp_bwd_mfma.hip", "dps_mfma.hip", "tdp_f32_mfma.hip"])
def test_direct_lds_loads_own_m0(tmp_path, unit):
    """The direct-to-LDS loads set M0 in inline assembly; nothing the compiler emits in those kernels may use M0, and
    the LDS waits must stay counted (csrc/check_m0.py states the conditions)."""
    assert _checker()(_assembly(tmp_path, unit)) is None


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_passes_ahead_of_the_backward_use_no_scratch(tmp_path):
    """The pass that prepares the triple-dot backward's operands is a copy: pointers that the compiler keeps in scratch memory and loads
    back by an index cost it more than its registers ever would."""
    kernels = re.findall(r"\.amdhsa_kernel (\S+)(.*?)\.end_amdhsa_kernel", _assembly(tmp_path, "tdp_bwd_mfma.hip"), re.S)
    scratch = {name: int(re.search(r"\.amdhsa_private_segment_fixed_size (\d+)", body)[1])
               for name, body in kernels if "bwd_prep" in name or "bwd_finish" in name}
    assert len(scratch) == 10 and set(scratch.values()) == {0}, scratch


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_dot_product_sum_forward_keeps_its_waves(tmp_path):
    """The dot-product-sum forward of small grids: a SIMD holds four of its waves at D = 32 (128 registers a lane), three at D = 64 (168) and two at
    D = 128 (256), without scratch memory."""
    kernels = re.findall(r"\.amdhsa_kernel (\S*attn_fwd_mfma_kernel\S*)(.*?)\.end_amdhsa_kernel", _assembly(tmp_path, "dps_mfma.hip"), re.S)
    assert len(kernels) == 16
    for name, body in kernels:
        registers, scratch = (int(re.search(rf"\.amdhsa_{what} (\d+)", body)[1]) for what in ("next_free_vgpr", "private_segment_fixed_size"))
        assert scratch == 0 and registers <= (128 if "Li32E" in name else 168 if "Li64E" in name else 256), (name, registers, scratch)


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_buffer_loads_keep_their_offset_in_the_range_check(tmp_path):
    """The fp32 dot-product-sum kernels rely on buffer loads to return zeros for rows past the end of a head.  The range
    check of a raw buffer leaves the scalar offset out, so that offset is zero in every one of them."""
    loads = re.findall(r"^\s*buffer_load_dword\w*\s+(.*)$", _assembly(tmp_path, "dps_f32_mfma.hip"), re.M)
    assert len(loads) > 100
    assert [x for x in loads if not re.search(r"s\[\d+:\d+\], 0 offen\b", x)] == []


def test_checker_rejects_foreign_users_of_m0():
    check = _checker()
    ours = ("s_mov_b32 m0, s4\ns_nop 0\nglobal_load_lds_dwordx4 v1, s[2:3]\n" * 120 +
            "s_mov_b32 m0, s5\ns_nop 0\nglobal_load_lds_dword v2, s[2:3]\n" + "s_waitcnt lgkmcnt(4)\n")
    assert check(ours) is None
    assert "expected" in check(ours.replace("s_mov_b32 m0, s4\ns_nop 0\nglobal_load_lds_dwordx4 v1, s[2:3]\n", "", 40))
    assert "not ours" in check(ours + "s_movk_i32 m0, 0x100\n")
    assert "indirect" in check(ours + "s_set_gpr_idx_on s3, gpr_idx(SRC0)\n")
    assert "flushed" in check(ours.replace("lgkmcnt(4)", "lgkmcnt(0)"))
