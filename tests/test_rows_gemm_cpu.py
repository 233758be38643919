"""Products of many rows in 16 bits: what can be checked without a GPU - the plan over all sizes, the refusals of the entry points, tensors that
are torch's, and the wait states behind products whose sums the compiler does not follow."""
import ctypes
import functools
import os
import re
import shutil

import pytest
import torch
import torch.nn.functional as F

from tools import isa_lint
from triforce_amd import hip, ops_rows
from triforce_amd.build import FLAGS

NEEDS_HIPCC = pytest.mark.skipif(shutil.which("hipcc") is None and not os.path.exists("/opt/rocm/bin/hipcc"), reason="hipcc not available")
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


# is the library's product the one to take: sizes on either side of each line
@pytest.mark.parametrize("rows,n,k,library", [(128, 32000, 4096, True), (160, 32000, 5120, True), (96, 32000, 4096, False), (193, 32000, 4096, False), (128, 27648, 4096, False),
                                              (128, 28672, 8192, True), (128, 128256, 4096, False), (128, 40960, 4096, False), (128, 8192, 28672, False), (128, 16384, 16384, False),
                                              (64, 768, 3072, True), (320, 768, 3072, True), (321, 768, 3072, False), (64, 512, 4096, False), (64, 1536, 4096, False),
                                              (64, 768, 1536, False), (64, 640, 8192, False), (4096, 4096, 4096, True), (4096, 4096, 1152, False), (4096, 8192, 512, False),
                                              (512, 32768, 4096, False), (1024, 16384, 4096, False), (3100, 4096, 4096, False), (112, 12288, 4096, False),
                                              (700, 4096, 11008, False)])
def test_sizes_of_the_kernel_and_of_the_library(rows, n, k, library):
    assert ops_rows.library_is_faster(rows, n, k) == library


@functools.lru_cache(maxsize=None)
def _kernels(source):
    """(name, text) of the kernels, compiled as the library is."""
    text = isa_lint.compile_to_asm(os.path.join(CSRC, source), extra=tuple(f for f in FLAGS if f not in ("-fPIC", "-shared")))
    return re.findall(r"^(_Z\w+):\s*;\s*@\1\n([\s\S]*?)\n\.Lfunc_end\d+:", text, re.M)


@NEEDS_HIPCC
@pytest.mark.parametrize("source", ["rows_gemm.hip", "tile_rows_gemm.hip"])
def test_sums_are_read_behind_the_wait_states_of_their_products(source):
    """Products in inline asm: nothing else may touch their sums within eleven cycles of the last of them in the text (they all lie in one
    loop, whose last instructions wait)."""
    def registers(token):
        return {r for lo, hi in re.findall(r"\ba\[(\d+):(\d+)\]", token) for r in range(int(lo), int(hi) + 1)} | {int(r) for r in re.findall(r"\ba(\d+)\b", token)}

    seen = 0
    for name, kernel in _kernels(source):
        lines = [t.strip() for t in kernel.split("\n")]
        asm = [i + 1 for i, t in enumerate(lines) if "ASMSTART" in t and lines[i + 1].startswith("v_mfma")]
        sums = set().union(*(registers(lines[i].split(",")[0]) for i in asm))
        seen, since, asm = seen + len(asm), None, set(asm)
        for i, t in enumerate(lines):
            if i in asm:
                since = 0
            elif since is not None and t and t[0] not in ";." and not t.endswith(":"):
                assert since >= 11 or not registers(t) & sums, (name, t)
                since += isa_lint.cost(t)
    assert seen == 2 * 2 * (64 + 56 + 48)                      # two forms, two half steps, the three largest tiles


def _dma_steps(kernel):
    """The kernel's LDS-DMA, waits for vector memory, barriers, labels and jumps in the order of the text: ("dma", its scalar pointer), ("wait", loads left),
    ("barrier",), ("label", l), ("jump", l), ("memory",) for any other access to memory."""
    out = []
    for line in kernel.split("\n"):
        t = line.strip()
        for kind, pattern in (("label", r"(\.LBB\w+):"), ("dma", r"global_load_lds\S*\s.*?(s\[\d+:\d+\]|off)"), ("wait", r"s_waitcnt.*vmcnt\((\d+)\)"), ("barrier", r"(s_barrier)"),
                              ("jump", r"s_c?branch\w*\s+(\.LBB\w+)"), ("memory", r"((?:global|flat|buffer|scratch)_\w+)")):
            m = re.match(pattern, t)
            if m:
                out.append((kind, int(m.group(1)) if kind == "wait" else m.group(1)))
                break
    return out


def _check_counted_waits(steps, mt, nt, nb):
    """A step's x is asked for before the waves meet, its weights behind, nothing else in its loop: then all but (nb - 2)(mt + nt) + mt loads have landed
    exactly when the next step's x and weights have, and no buffer that a wave may still read is written."""
    kinds = [k for k, _ in steps]
    assert kinds.count("barrier") == 2
    first = kinds.index("barrier")
    begin = kinds.index("dma")
    assert kinds[begin:first].count("dma") == nb * (mt + nt) and "memory" not in kinds[begin:first]
    assert [v for k, v in steps[begin:first] if k == "wait"] == [(nb - 1) * (mt + nt)] and kinds[first - 1] == "wait"
    meet = first + 1 + kinds[first + 1:].index("barrier")
    head = max(i for i in range(meet) if kinds[i] == "label")
    back = next(i for i in range(meet, len(steps)) if kinds[i] == "jump")
    assert steps[back][1] == steps[head][1], "the step is one loop without a branch"
    body = steps[head + 1:back]
    x, w = body[0][1], body[-1][1]
    assert x != w and body == [("dma", x)] * mt + [("wait", (nb - 2) * (mt + nt) + mt), ("barrier", "s_barrier")] + [("dma", w)] * nt
    assert not {"dma", "barrier"} & set(kinds[first + 1:head] + kinds[back:])


def test_the_check_of_counted_waits_sees_a_load_out_of_place():
    x, w, meet = ("dma", "s[0:1]"), ("dma", "s[2:3]"), ("barrier", "s_barrier")

    def kernel(*step, prologue=(x, x, w) * 2 + (("wait", 3), meet)):
        return [*prologue, ("label", "a"), *step, ("jump", "a"), ("memory", "global_store_dwordx4"), ("wait", 0)]
    _check_counted_waits(kernel(x, x, ("wait", 2), meet, w), 2, 1, 2)
    for bad in (kernel(x, w, ("wait", 2), meet, x), kernel(w, x, ("wait", 2), meet, x), kernel(x, ("wait", 1), meet, x, w), kernel(x, x, ("wait", 3), meet, w),
                kernel(x, ("memory", "global_load_dword"), x, ("wait", 2), meet, w), kernel(x, ("wait", 2), meet, w), kernel(x, x, meet, w),
                kernel(x, x, ("wait", 2), meet, w, prologue=(x, x, w) * 2 + (("wait", 4), meet)),
                kernel(x, x, ("wait", 2), meet, w, prologue=(x, x, w, x, x, ("wait", 3), meet)), kernel(x, x, ("wait", 2), meet, w, meet)):
        with pytest.raises(AssertionError):
            _check_counted_waits(bad, 2, 1, 2)


@NEEDS_HIPCC
@pytest.mark.parametrize("source", ["rows_gemm.hip", "tile_rows_gemm.hip"])
def test_counted_waits_hold_for_the_order_of_the_loads(source):
    seen = 0
    for name, kernel in _kernels(source):
        m = re.search(r"rows_gemm_kernelI\w+?Li(\d+)ELi(\d+)ELi(\d+)ELi\d+ELi\d+E", name)
        if m:
            _check_counted_waits(_dma_steps(kernel), *map(int, m.groups()))
            seen += 1
    assert seen == 2 * 8
