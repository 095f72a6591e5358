"""The wait states between a matrix instruction and the vector code on its result, read off the assembly of the
kernels that touch their accumulators behind a branch (fp32 folds).  The hardware does not interlock them, and the
compiler counts them along one of the paths into a block; a sum that takes a register too early is wrong only now and
then, so no run on the GPU is a test of it.

An instruction counts one wait state, s_nop n n + 1, a matrix instruction its passes (the pipe is busy that long);
needed are the passes + 2 of fp32 and + 3 of bf16 products."""
import re
import subprocess

import pytest

from mind_amd import _build

MFMA = {"32x32x2_f32": (16, 18), "16x16x4_f32": (8, 10), "32x32x16_bf16": (8, 11), "16x16x32_bf16": (4, 7)}


def _regs(text):
    out = set()
    for one, lo, hi in re.findall(r"\bv(\d+)\b|\bv\[(\d+):(\d+)\]", text):
        out |= {int(one)} if one else set(range(int(lo), int(hi) + 1))
    return out


def _kind(op):
    return next((v for k, v in MFMA.items() if k in op), None) if op.startswith("v_mfma") else None


def early_uses(lines):
    """(matrix instruction, instruction that reads or writes its result too early) of one kernel's assembly lines."""
    seq, label = [], {}
    for line in lines:
        line = line.split(";")[0].strip()
        m = re.match(r"(\.LBB\d+_\d+):", line)
        if m:
            label[m.group(1)] = len(seq)
        elif line and not line.startswith(".") and not line.endswith(":"):
            seq.append(line)

    def following(i):
        op = seq[i].split()[0]
        nxt = [] if op in ("s_endpgm", "s_branch") else [i + 1]
        return nxt + ([label[seq[i].split()[-1]]] if op.startswith(("s_branch", "s_cbranch")) else [])
    found = []
    for i, line in enumerate(seq):
        op, _, operands = line.partition(" ")
        if not op.startswith("v_mfma"):
            continue
        need, result = _kind(op)[1], _regs(operands.split(",")[0])
        best, todo = {}, [(j, 0) for j in following(i)]
        while todo:
            j, waited = todo.pop()
            if j >= len(seq) or waited >= need or best.get(j, need) <= waited:
                continue
            best[j] = waited
            op, _, operands = seq[j].partition(" ")
            if op.startswith("v_mfma"):   # that one's own result is looked at from there
                if _regs(operands.split(",")[0]) >= result:
                    continue
                waited += _kind(op)[0]
            else:
                if op.startswith(("v_", "ds_", "buffer_", "global_", "flat_", "scratch_")) and _regs(operands) & result:
                    found.append((line, seq[j]))
                waited += int(operands, 0) + 1 if op == "s_nop" else 1
            todo += [(k, waited) for k in following(j)]
    return found


def test_early_use_is_seen():
    kernel = ["v_mfma_f32_32x32x2_f32 v[2:17], v40, v44, v[2:17]", "s_cbranch_scc0 .LBB0_2", "s_nop 15", "s_nop 1",
              ".LBB0_2:", "s_add_i32 s4, s47, 9", "v_add_f32_e32 v21, v21, v17", "s_endpgm"]
    assert early_uses(kernel) == [(kernel[0], kernel[6])]           # along the branch
    assert not early_uses(kernel[:1] + kernel[2:])                  # waits written out on the one path
    assert not early_uses([kernel[0], "v_add_f32_e32 v21, v21, v18", "s_endpgm"])


@pytest.mark.parametrize("source", ["esa_linear_gemm", "esa_wgrad"])
def test_no_early_use_in(source, tmp_path):
    out = tmp_path / "kernels.txt"
    run = subprocess.run([_build.hipcc(), *_build.HIPFLAGS, "--cuda-device-only", "-S", str(_build.CSRC / f"{source}.hip"),
                          "-o", str(out)], capture_output=True, text=True)
    assert run.returncode == 0, run.stderr[-2000:]
    kernels = [part.split("\n.Lfunc_end")[0].split("\n")[1:] for part in re.split(r"\n(?=_Z\w+:)", out.read_text())[1:]]
    kernels = [k for k in kernels if any("v_mfma" in line for line in k)]
    assert len(kernels) >= 4 and not any(early_uses(k) for k in kernels)
