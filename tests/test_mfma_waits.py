"""Inline assembly of the tail's kernels never reads an MFMA result that did not settle.  The
hardware needs wait states between an MFMA and an instruction that reads its result, and the
compiler inserts them only before instructions it knows, not before inline assembly.  The
device assembly of the two sources is built here and followed along its control flow: for each
inline vector instruction, no path may reach it from an MFMA that wrote one of its sources
without at least as many wait states as the compiler itself takes (one per instruction, s_nop n
n + 1; 8 after the 16x16 fp16 MFMAs of these files, 10 after v_mfma_f32_16x16x4_f32)."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rust-ppocrv6_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
NEED = {"v_mfma_f32_16x16x4_f32": 10}
NEED_DEFAULT, NEED_32 = 8, 18  # 32x32 tiles: 16 passes


def _regs(token):
    m = re.match(r"^[-|]*v\[(\d+):(\d+)\]", token)
    if m:
        return range(int(m[1]), int(m[2]) + 1)
    m = re.match(r"^[-|]*v(\d+)\b", token)
    return [int(m[1])] if m else []


def unsettled_reads(text):
    """(function, line, instruction) of each inline vector instruction that a path reaches with too
    few wait states after an MFMA that wrote one of its sources, and how many were looked at."""
    bad, seen = [], 0
    for part in re.split(r"^(?=_Z\S+:)", text, flags=re.M)[1:]:
        body = part.split("\t.section")[0].splitlines()
        code, labels, inline = [], {}, False
        for ln, line in enumerate(body):
            s = line.strip()
            if "#ASMSTART" in s or "#ASMEND" in s:
                inline = "#ASMSTART" in s
                continue
            m = re.match(r"^(\.LBB\S+|_Z\S+):", s)
            if m:
                labels[m[1]] = len(code)
                continue
            s = s.split(";")[0].strip()
            if s and s[0] not in ".;":
                code.append((s, inline, ln))
        # pending[i]: register -> wait states still missing before code[i]
        pending, work = {0: {}}, [0]
        hits = set()
        while work:
            i = work.pop()
            state = dict(pending[i])
            while i < len(code):
                s, inl, ln = code[i]
                op, _, rest = s.partition(" ")
                toks = [t.strip() for t in rest.split(",")]
                if op.startswith("v_"):
                    if inl:
                        seen += 1
                        if any(state.get(r, 0) > 0 for t in toks[1:] for r in _regs(t)):
                            hits.add((body[0].split(":")[0], ln, s))
                    spent = 1
                else:
                    spent = int(toks[0]) + 1 if op == "s_nop" else 1
                state = {r: w - spent for r, w in state.items() if w > spent}
                if op.startswith("v_mfma"):
                    need = NEED_32 if "32x32" in op else NEED.get(op, NEED_DEFAULT)
                    state.update((r, need) for r in _regs(toks[0]))
                elif op.startswith("v_"):
                    for r in _regs(toks[0]):
                        state.pop(r, None)  # the compiler's own instructions wait before they write
                if op == "s_endpgm":
                    break
                targets = []
                if op.startswith(("s_cbranch", "s_branch")):
                    targets.append(labels[toks[0]])
                if op == "s_branch":
                    nxt = targets
                elif targets or i + 1 in labels.values():
                    nxt = targets + [i + 1]
                else:
                    i += 1
                    continue
                for t in nxt:
                    old = pending.get(t)
                    new = dict(old or {})
                    for r, w in state.items():
                        new[r] = max(new.get(r, 0), w)
                    if old is None or new != old:
                        pending[t] = new
                        work.append(t)
                break
        bad += sorted(hits)
    return bad, seen


SYNTHETIC = """_Z1k:
\tv_mfma_f32_16x16x16_f16 v[2:5], v[2:3], v[6:7], 0
\ts_cbranch_vccz .LBB0_2
\tv_mov_b32_e32 v2, 0
\tv_mov_b32_e32 v3, 0
.LBB0_2:
%s\t;;#ASMSTART
\tv_max3_f32 v8, v2, v3, v9
\t;;#ASMEND
\ts_endpgm
\t.section"""


def test_the_scan_itself():
    assert len(unsettled_reads(SYNTHETIC % "")[0]) == 1  # along the branch only one instruction lies between
    assert len(unsettled_reads(SYNTHETIC % "\ts_nop 5\n")[0]) == 1
    assert unsettled_reads(SYNTHETIC % "\ts_nop 7\n") == ([], 1)


@pytest.mark.parametrize("name", ["neck.hip", "neck_fused.hip"])
def test_inline_assembly_reads_no_unsettled_mfma_result(name, tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    out = tmp_path / "k.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++20", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-mllvm", "-amdgpu-mfma-vgpr-form=1", "-S", "--cuda-device-only",
                    os.path.join(CSRC, name), "-o", str(out)], check=True, capture_output=True, timeout=600)
    bad, seen = unsettled_reads(out.read_text())
    assert seen > 0
    assert not bad, f"{len(bad)} inline instructions read unsettled MFMA results, e.g. {bad[:3]}"
