"""Products of many rows in 16 bits: what can be checked without a GPU - the plan over all sizes, the refusals of the entry points, tensors that
are torch's, and the wait states behind products whose sums the compiler does not follow."""
import ctypes
import os
import re
import shutil

import pytest
import torch
import torch.nn.functional as F

from tools import isa_lint
from triforce_amd import hip, ops_rows

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "triforce_amd", "csrc")


def _libs():
    return (hip.lib().tf_rows_gemm, hip.lib().tf_rows_gemm_plan, 1), (hip.tile_lib().tfl_rows_gemm, hip.tile_lib().tfl_rows_gemm_plan, 2)


def test_every_part_of_a_plan_has_steps():
    for _, plan, _ in _libs():
        for rows in (1, 33, 129, 200, 700, 1500, 4096, 33000):
            for n in (16, 96, 1136, 4096, 22016):
                for k in (64, 128, 320, 1536, 4096, 11008, 65536):
                    shape, splits = ctypes.c_int32(), ctypes.c_int32()
                    floats = plan(rows, n, k, ctypes.byref(shape), ctypes.byref(splits))
                    steps, s = k // 64, splits.value
                    assert 0 <= shape.value < 8 and 1 <= s <= 16 and (s - 1) * -(-steps // s) < steps
                    assert floats == (s * rows * n if s > 1 else 0)
        assert plan(0, 16, 64, ctypes.byref(shape), ctypes.byref(splits)) < 0


def test_entry_points_refuse_what_the_kernel_does_not_take():
    at = 1 << 20                                                # (never read: every call is refused)
    good = dict(x=at, ld_x=128, w=at, out=at, ld_out=64, ws=None, floats=0, rows=40, n=64, k=128, form=0, shape=0, splits=1)
    for entry, _, unit in _libs():
        bad = [dict(x=None), dict(w=None), dict(out=None), dict(x=at + 8), dict(w=at + 2), dict(out=at + 4), dict(ld_x=120), dict(ld_x=132), dict(ld_out=56),
               dict(ld_out=68), dict(rows=0), dict(n=72, ld_out=72), dict(n=0), dict(k=96), dict(k=0), dict(form=3 - unit), dict(form=3), dict(shape=8), dict(shape=-1),
               dict(splits=0), dict(splits=3), dict(splits=-1), dict(n=48, form=unit), dict(rows=1 << 25), dict(k=1 << 26, ld_x=1 << 26)]
        for change in bad:
            a = dict(good, **change)
            assert entry(a["x"], a["ld_x"], a["w"], a["out"], a["ld_out"], a["ws"], a["floats"], a["rows"], a["n"], a["k"], a["form"], a["shape"], a["splits"],
                         None) == -22, change
        assert entry(at, 128, at, at, 64, None, 0, 40, 64, 128, 0, 0, 2, None) == -28
        assert entry(at, 128, at, at, 64, at, 2 * 40 * 64 - 1, 40, 64, 128, 0, 0, 2, None) == -28


def test_host_tensors_are_torchs():
    x, w = torch.randn(40, 128).half(), torch.randn(64, 128).half()
    assert not ops_rows.takes(x, w) and torch.equal(ops_rows.linear(x, w), F.linear(x, w))


def test_the_librarys_sizes():
    assert ops_rows.library_fills(4096, 4096) and ops_rows.library_fills(8000, 4096) and not ops_rows.library_fills(3100, 4096)
    assert not ops_rows.library_fills(4096, 22016) and not ops_rows.library_fills(3900, 4096)


# rows, n, k, form -> is the library's product the faster one: sizes where one of the two was by 5 % or more
@pytest.mark.parametrize("rows,n,k,form,library", [(112, 12288, 4096, 0, True), (384, 12320, 4096, 0, True), (768, 4096, 4096, 0, True), (560, 15360, 5120, 0, True),
                                                   (128, 32000, 4096, 0, True), (512, 6144, 1536, 0, True), (100, 768, 3072, 0, True), (100, 22016, 4096, 1, True),
                                                   (160, 4096, 4096, 0, False), (160, 5120, 5120, 0, False), (6000, 12288, 4096, 0, False),
                                                   (2048, 18784, 4096, 0, False), (700, 4096, 11008, 0, False), (160, 4096, 15104, 0, False), (100, 256, 4096, 0, False),
                                                   (700, 2304, 768, 0, False), (4096, 8192, 512, 0, False), (33, 22016, 4096, 1, False), (1500, 22016, 4096, 2, False)])
def test_sizes_of_the_kernel_and_of_the_library(rows, n, k, form, library):
    assert ops_rows.library_is_faster(rows, n, k, form) == library


@pytest.mark.skipif(shutil.which("hipcc") is None and not os.path.exists("/opt/rocm/bin/hipcc"), reason="hipcc not available")
@pytest.mark.parametrize("source", ["rows_gemm.hip", "tile_rows_gemm.hip"])
def test_sums_are_read_behind_the_wait_states_of_their_products(source):
    """Products in inline asm: nothing else may touch their sums within eleven cycles of the last of them in the text (they all lie in one
    loop, whose last instructions wait)."""
    def registers(token):
        return {r for lo, hi in re.findall(r"\ba\[(\d+):(\d+)\]", token) for r in range(int(lo), int(hi) + 1)} | {int(r) for r in re.findall(r"\ba(\d+)\b", token)}

    seen, kernels = 0, re.split(r"^(?=_Z\w+:)", isa_lint.compile_to_asm(os.path.join(CSRC, source)), flags=re.M)
    for kernel in kernels:
        lines = [t.strip() for t in kernel.split("\n")]
        asm = [i + 1 for i, t in enumerate(lines) if "ASMSTART" in t and lines[i + 1].startswith("v_mfma")]
        sums = set().union(*(registers(lines[i].split(",")[0]) for i in asm))
        seen, since, asm = seen + len(asm), None, set(asm)
        for i, t in enumerate(lines):
            if i in asm:
                since = 0
            elif since is not None and t and t[0] not in ";." and not t.endswith(":"):
                assert since >= 11 or not registers(t) & sums, (kernel[:60], t)
                since += isa_lint.cost(t)
    assert seen == 2 * 2 * (64 + 56 + 48)                      # two forms, two half steps, the three largest tiles
