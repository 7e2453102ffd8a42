"""The machine code of the weight-streaming kernel's launches of a few workgroups: the look-ahead that the source describes is
really there. A wavefront requests the weights of step s + 5 at the head of step s; the instruction scheduler, left alone, gathers
the requests of a whole round at its end and waits for nearly all of them at once, which costs a launch of this kind up to 8 %
and changes with unrelated edits. Compiles one file for the device (no GPU needed) and reads the main loops."""
import functools
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dmlx_amd", "csrc")
STEPS = 6  # of a round: the ring's stages


@functools.lru_cache(maxsize=None)
def _device_asm(source):
    with open(os.path.join(CSRC, "Makefile")) as f:
        text = f.read().replace("\\\n", " ")
    flags = re.search(r"^FLAGS\s*:=(.*)$", text, re.M).group(1).replace("$(ARCH)", "gfx950").split()
    out = subprocess.run([os.environ.get("HIPCC", "hipcc")] + flags + ["-S", "--offload-device-only", source, "-o", "-"], cwd=CSRC,
                         capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stderr[-2000:]
    return out.stdout


def _functions(asm):
    name, body = None, []
    for line in asm.split("\n"):
        line = line.split(";")[0].strip()
        m = re.match(r"^(_Z\w+):", line)
        if m and name is None:
            name, body = m.group(1), []
        elif line.startswith(".Lfunc_end") and name is not None:
            yield name, body
            name = None
        elif name is not None and line:
            body.append(line)


def _rounds(body):
    """bodies of the loops that request one weight chunk per step of a round and never branch inside"""
    at = {line[:-1]: i for i, line in enumerate(body) if re.match(r"^\.LBB\w+:$", line)}
    for i, line in enumerate(body):
        m = re.match(r"s_c?branch\w*\s+(\.LBB\w+)", line)
        if m and at.get(m.group(1), i) < i:
            loop = body[at[m.group(1)]:i]
            if sum("global_load_dwordx4" in x for x in loop) == STEPS and not any("branch" in x for x in loop):
                yield loop


@pytest.mark.skipif(shutil.which(os.environ.get("HIPCC", "hipcc")) is None, reason="needs hipcc")
def test_few_workgroup_launches_keep_their_look_ahead():
    seen = {}
    for name, body in _functions(_device_asm("qgemm_skinny.hip")):
        # template arguments: format, FACTORED, PACKED, MBLK, KSPLIT, FEW
        m = re.match(r"_ZN4dmoe19qgemm_skinny_kernelINS_\d+Fmt(\w+?)ELb([01])ELb1ELb0ELb([01])ELb([01])EEE", name)
        if not m or m.group(3) == m.group(4) or m.group(1) == "Bf16":
            continue
        rounds = list(_rounds(body))
        assert len(rounds) == 1, (name, len(rounds))
        loop = rounds[0]
        mfma = [i for i, x in enumerate(loop) if "mfma" in x]
        loads = [i for i, x in enumerate(loop) if "global_load_dwordx4" in x]
        per_step = len(mfma) // STEPS
        for k, i in enumerate(loads):  # the request of step k: among that step's matrix instructions, or just ahead of them
            done = sum(j < i for j in mfma)
            assert (k - 1) * per_step <= done <= (k + 1) * per_step, (name, k, done)
        # every wait leaves at least four of the five younger steps' requests (chunk, and scale unless it is per row) in flight
        per_stage = sum("global_load" in x for x in loop) // STEPS
        waits = [int(x) for line in loop for x in re.findall(r"vmcnt\((\d+)\)", line)]
        assert waits and min(waits) >= 4 * per_stage, (name, waits)
        seen[m.groups()] = True
    # split reduction and few-workgroup launch of: 4-bit affine (scales factored out, and not), 8-bit affine, MXFP4, FP8 per row
    assert len(seen) == 10, sorted(seen)


@pytest.mark.skipif(shutil.which(os.environ.get("HIPCC", "hipcc")) is None, reason="needs hipcc")
def test_eight_bit_launches_leave_registers_for_three_workgroups():
    """The packed 8-bit kernel of launches that fill the chip: six wavefronts per SIMD (512 registers, handed out by eight), three
    workgroups of eight wavefronts on a compute unit, and nothing spilled for it. The LDS side is asserted in the source."""
    seen = 0
    for entry in _device_asm("qgemm_skinny.hip").split("  - .agpr_count:")[1:]:
        if "qgemm_skinny_kernelINS_10FmtAffine8ELb0ELb1ELb0ELb0ELb0EEE" not in entry:
            continue
        get = lambda key: int(re.search(rf"\.{key}:\s*(\d+)", entry).group(1))
        assert get("vgpr_count") <= 512 // 6 // 8 * 8 and get("vgpr_spill_count") == 0 and get("private_segment_fixed_size") == 0
        seen += 1
    assert seen == 1


@pytest.mark.skipif(shutil.which(os.environ.get("HIPCC", "hipcc")) is None, reason="needs hipcc")
def test_checkpoint_layout_kernel_keeps_its_scalar_registers():
    """The 4-bit kernels on the checkpoint's own arrays run out of scalar registers. What is spilled at their head is waited for load by
    load (about 0.1 us each on calls of 20): no more of it than the 30 and 35 registers it was measured with."""
    seen = {}
    for entry in _device_asm("qgemm_skinny.hip").split("  - .agpr_count:")[1:]:
        m = re.search(r"qgemm_skinny_kernelINS_10FmtAffine4ELb1ELb0ELb([01])ELb0ELb0EEE", entry)
        if m:
            seen[m.group(1)] = int(re.search(r"\.sgpr_spill_count:\s*(\d+)", entry).group(1))
    assert set(seen) == {"0", "1"} and seen["1"] <= 30 and seen["0"] <= 35, seen
