"""No kernel uses the result of a matrix instruction before it is written.

The hardware does not wait for an MFMA's result when another kind of instruction reads
or overwrites its registers (or a later MFMA takes them as A or B): the code has to
keep the distance.  The compiler does on straight-line code, but counts the distance
along the fall-through path only, so a use behind a short taken branch can come too
early; the kernels keep their accumulators away from such branches.  Here every path
through the assembly of every kernel is checked against the distances that the
compiler itself keeps on straight-line code."""
import os
import re
import subprocess
from concurrent.futures import ProcessPoolExecutor

import pytest

from quantax_amd import build

# wait states (instructions and s_nop counts) between an MFMA and a use of its result
NEED = {"v_mfma_f32_16x16x32_bf16": 8, "v_mfma_f32_16x16x4_f32": 10, "v_mfma_f64_16x16x4_f64": 19}
FAR = max(NEED.values())
JUMPS = ("s_cbranch", "s_branch", "s_endpgm", "s_setpc")


def registers(text):
    out = set()
    for m in re.finditer(r"\b([va])\[(\d+):(\d+)\]|\b([va])(\d+)\b", text):
        if m.group(1):
            out |= {(m.group(1), i) for i in range(int(m.group(2)), int(m.group(3)) + 1)}
        else:
            out.add((m.group(4), int(m.group(5))))
    return out


def functions(text):
    """{name: [(line, op, operands)]}, labels as op 'label'."""
    out, cur = {}, None
    for ln, line in enumerate(text.splitlines(), 1):
        line = line.split(";")[0].rstrip()
        if line.startswith(".Lfunc_end"):
            cur = None
        elif (m := re.match(r"^([A-Za-z_]\w*):", line)):
            cur = out.setdefault(m.group(1), [])
        elif cur is not None and (m := re.match(r"^(\.LBB\w+):", line)):
            cur.append((ln, "label", m.group(1)))
        elif cur is not None and (line := line.strip()) and not line.startswith("."):
            op, _, arg = line.partition(" ")
            cur.append((ln, op, arg.strip()))
    return out


def step(state, ins, report=None):
    """state {register: (distance, mfma)} after one instruction."""
    ln, op, arg = ins
    if op == "label":
        return state
    mfma = op.startswith("v_mfma")
    ops = arg.split(", ")
    if mfma:
        assert op in NEED, f"add the wait states of {op}"
        used = registers(ops[1]) | registers(ops[2])
    else:
        used = set() if op.startswith("s_") else registers(arg)
    if report is not None:
        for r in used & state.keys():
            if state[r][0] < NEED[state[r][1]]:
                report.append(f"line {ln}: {op} uses {r[0]}{r[1]} {state[r][0]} wait states after {state[r][1]}")
    n = int(arg, 0) + 1 if op == "s_nop" else 1
    written = registers(ops[0]) if op.startswith("v_") and not mfma else set()
    out = {r: (d + n, m) for r, (d, m) in state.items() if d + n <= FAR and r not in written}
    if mfma:
        out.update({r: (0, op) for r in registers(ops[0])})
    return out


def too_early(code):
    """Uses of MFMA results before their time, over all paths through a function."""
    starts = {0} | {i for i, x in enumerate(code) if x[1] == "label"}
    starts |= {i + 1 for i, x in enumerate(code) if x[1].startswith(JUMPS)}
    starts = sorted(s for s in starts if s < len(code))
    at = {s: k for k, s in enumerate(starts)}
    label = {x[2]: i for i, x in enumerate(code) if x[1] == "label"}
    ends = starts[1:] + [len(code)]
    inn = [None] * len(starts)
    inn[0], work = {}, [0]
    while work:
        k = work.pop()
        state = inn[k]
        for i in range(starts[k], ends[k]):
            state = step(state, code[i])
        op, arg = code[ends[k] - 1][1:]
        nxt = [at[label[arg]]] if op.startswith(("s_cbranch", "s_branch")) else []
        if not op.startswith(("s_branch", "s_endpgm", "s_setpc")) and ends[k] in at:
            nxt.append(at[ends[k]])
        for t in nxt:
            if inn[t] is None:
                inn[t] = dict(state)
                work.append(t)
                continue
            changed = False
            for r, v in state.items():
                if r not in inn[t] or v[0] < inn[t][r][0]:
                    inn[t][r], changed = v, True
            if changed:
                work.append(t)
    found = []
    for k, state in enumerate(inn):
        if state is not None:
            for i in range(starts[k], ends[k]):
                state = step(state, code[i], found)
    return found


def check(src):
    r = subprocess.run([build.HIPCC, *build.FLAGS, "-w", "-S", "--offload-device-only", os.path.join(build.CSRC, src),
                        "-o", "-"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    out, kernels = [], 0
    for name, code in functions(r.stdout).items():
        if any(x[1].startswith("v_mfma") for x in code):
            kernels += 1
            out += [f"{src} {name} {e}" for e in too_early(code)]
    return src, kernels, out


def _uses_mfma(src):
    text = open(os.path.join(build.CSRC, src)).read()
    return "mfma" in text or "resconv_wave.hpp" in text


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="needs the compiler")
def test_every_kernel_waits_for_its_matrix_results():
    with ProcessPoolExecutor(max_workers=8) as ex:
        done = list(ex.map(check, [s for s in build.SOURCES if _uses_mfma(s)]))
    assert all(kernels > 0 for _, kernels, _ in done), done
    found = [e for _, _, out in done for e in out]
    assert not found, "\n".join(found[:20])


F64 = "\tv_mfma_f64_16x16x4_f64 v[0:7], v[8:9], v[10:11], 0\n"


@pytest.mark.parametrize("body,bad", [
    (F64 + "\ts_nop 15\n\ts_nop 2\n\tv_add_f64 v[12:13], v[0:1], v[14:15]\n", False),  # 16 + 3 = 19
    (F64 + "\ts_nop 15\n\ts_nop 1\n\tv_add_f64 v[12:13], v[0:1], v[14:15]\n", True),
    (F64 + "\ts_cbranch_scc1 .LBB0_2\n\ts_nop 15\n\ts_nop 15\n.LBB0_2:\n\tv_add_f64 v[12:13], v[0:1], v[14:15]\n", True),
    (F64 + "\ts_cbranch_scc1 .LBB0_2\n\ts_nop 3\n.LBB0_2:\n\ts_nop 15\n\ts_nop 2\n\tds_write_b64 v20, v[6:7]\n", False),
    (F64 + "\ts_nop 8\n\tglobal_store_dwordx2 v[20:21], v[2:3], off\n", True),
    (F64 + "\ts_nop 8\n\tv_mov_b32_e32 v3, 0\n", True),  # overwritten
    (F64 + F64.replace(", 0\n", ", v[0:7]\n"), False),  # accumulating needs no wait of the code's
    (F64 + "\tv_mfma_f64_16x16x4_f64 v[30:37], v[0:1], v[10:11], 0\n", True),
    (".LBB0_1:\n\tv_mov_b32_e32 v5, v22\n" + F64 + "\ts_cbranch_scc1 .LBB0_1\n", True),  # around a loop
])
def test_the_check_itself(body, bad):
    code = functions("kernel:\n" + body + "\ts_endpgm\n.Lfunc_end0:\n")["kernel"]
    assert bool(too_early(code)) == bad
