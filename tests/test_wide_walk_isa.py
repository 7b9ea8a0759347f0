"""The wide tiled kernels (wide.hip) write their MFMAs in assembly with the accumulators in place, so
the compiler does not see the waits those need, and fill their LDS stages by DMA behind a plain
barrier. This test compiles wide.hip for gfx950 with the library's own flags and checks the loops
of the K walk in the compiled code (two steps per iteration, one loop per token-tile count):

  - no vector instruction besides the MFMAs (a move of an operand or accumulator next to an MFMA
    would need wait states), and every MFMA accumulates in place;
  - at least two instructions before the first MFMA, and `s_nop 15` after the last one, before
    anything can read an accumulator;
  - each of the two barriers directly follows a wait for every DMA and LDS read of the wave, and
    each is followed by one step's DMA (8 weight and 2, 4, 6 or 8 token instructions);

and that no kernel spills registers to scratch memory. Runs on the CPU: hipcc cross-compiles; no GPU
is used."""
import os
import re
import shutil
import subprocess

import pytest

from ae_amd import build as libbuild

KERNEL_RE = re.compile(r"^(_ZN3smx\d+wide_(gateup|down)_kernelILi([12])E(Lb[01]E)?EEvNS_10ExpertArgsE):")


@pytest.fixture(scope="module")
def wide_loops(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc is not installed")
    out = tmp_path_factory.mktemp("isa") / "wide.s"
    cmd = [hipcc, *libbuild.HIPCC_FLAGS, "--cuda-device-only", "-S",
           os.path.join(libbuild.CSRC, "wide.hip"), "-o", str(out)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr
    loops, spills, kernel, label, body = {}, {}, None, None, []
    for line in out.read_text().split("\n"):
        m = KERNEL_RE.match(line)
        if m:
            kernel, label, body = m.group(1), None, []
            loops[kernel], spills[kernel] = [], []
        elif line.startswith(".Lfunc_end"):
            kernel = None
        elif kernel and re.match(r"^\.LBB\w+:", line):
            label, body = line.split(":")[0], []
        elif kernel:
            t = line.split(";")[0].strip()
            if t and not t.startswith("."):
                body.append(t)
                if t.startswith("scratch_"):
                    spills[kernel].append(t)
                if t.startswith("s_cbranch") and t.split()[-1] == label and any("v_mfma" in b for b in body):
                    loops[kernel].append(body)
    return loops, spills


def test_no_spills(wide_loops):
    assert len(wide_loops[1]) == 6
    assert {k: v for k, v in wide_loops[1].items() if v} == {}


def test_walk_loops(wide_loops):
    wide_loops = wide_loops[0]
    assert len(wide_loops) == 6, sorted(wide_loops)  # gate/up, down of partials and of terms; fp16 and bf16
    for name, loops in wide_loops.items():
        tiles = sorted(sum("v_mfma" in t for t in b) // 32 for b in loops)
        # (the kernel of terms holds the loops twice: the shared expert's items write partials)
        assert tiles == sorted([2, 4, 6, 8] * (2 if "Lb1" in name else 1)), (name, tiles)
        for body in loops:
            nt = sum("v_mfma" in t for t in body) // 32
            mfma = [i for i, t in enumerate(body) if t.startswith("v_mfma")]
            assert [t for t in body if t.startswith("v_") and "mfma" not in t] == [], name
            for i in mfma:
                ops = re.findall(r"[av]\[\d+:\d+\]", body[i])
                assert ops[0] == ops[3] and ops[0][0] == "a", (name, body[i])
            assert mfma[0] >= 2 and body[mfma[-1] + 1] == "s_nop 15", name
            bars = [i for i, t in enumerate(body) if t == "s_barrier"]
            assert len(bars) == 2, name
            for k, i in enumerate(bars):
                w = body[i - 1]
                assert w.startswith("s_waitcnt") and "vmcnt(0)" in w and "lgkmcnt(0)" in w, (name, w)
                end = bars[k + 1] if k + 1 < len(bars) else len(body)
                assert sum(t.endswith(" lds") for t in body[i:end]) == 8 + nt, name
            assert not any(t.endswith(" lds") for t in body[:bars[0]]), name
