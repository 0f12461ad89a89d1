"""The hand-written instructions of csrc/prefill_q.hip in its compiled form (no GPU).

The compiler tracks no hazard of an inline-asm matrix instruction and does not
see its latency. Checked for every instance built: no operand is written by a
vector instruction within two wait states before the instruction, an
accumulator leaves it through the statements after acc_wait alone, and a counted
wait for the loads into LDS leaves no more in flight than was asked for after
them."""
import os
import re
import subprocess

import pytest

from alveare_amd import build

SRC = os.path.join(build.CSRC, "prefill_q.hip")
WAIT_STATES = 2  # vector write of a matrix instruction's operand to its read


def _emit(tmp, *flags):
    out = str(tmp / "out")
    r = subprocess.run([build._hipcc(), *build.HIPCC_FLAGS, "--offload-device-only", "-S", *flags, SRC, "-o", out],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return open(out).read()


@pytest.fixture(scope="module")
def compiled(tmp_path_factory):
    try:
        build._hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    tmp = tmp_path_factory.mktemp("prefill")
    return _emit(tmp), _emit(tmp, "-emit-llvm")


def _regs(op):
    m = re.match(r"([va])(?:\[(\d+):(\d+)\]|(\d+))$", op)
    if not m:
        return set()
    lo = int(m.group(2) or m.group(4))
    return {(m.group(1), i) for i in range(lo, int(m.group(3) or lo) + 1)}


def hazards(body):
    """Inline-asm matrix instructions of one kernel's assembly that read a
    register written by a vector instruction fewer than WAIT_STATES before, or
    that stand so close behind a label that the path there is not seen.
    Returns (instructions checked, those found)."""
    checked, bad = 0, []
    written = []  # per wait state back: registers written, None behind a label
    inline = False
    for line in body.splitlines():
        if ";#ASM" in line:
            inline = "#ASMSTART" in line
            continue
        text = line.split(";")[0].split("//")[0].strip()
        if re.match(r"[.\w$]+:$", text):
            written.append(None)
            continue
        if not text or text.startswith("."):
            continue
        op, _, rest = text.partition(" ")
        op, _, more = op.partition("\t")
        args = [a.strip() for a in (more or rest).split(",")]
        if inline and op.startswith("v_mfma"):
            checked += 1
            reads = _regs(args[1]) | _regs(args[2]) | _regs(args[3])
            for w in written[-WAIT_STATES:]:
                if w is None or w & reads:
                    bad.append(text)
                    break
        if op == "s_nop":
            written += [set()] * (int(args[0], 0) + 1)
        else:
            written.append(_regs(args[0]) if op.startswith("v_") and not op.startswith("v_mfma") else set())
    return checked, bad


def open_waits(body):
    """Counted (nonzero) hand-written load waits of one kernel's assembly that a
    load into LDS could still be pending behind: fewer vector memory
    instructions than the count, or a label, stand between the last such load
    and the wait. Returns (waits checked, those found)."""
    checked, bad = 0, []
    since = None  # vector memory instructions since the last load into LDS
    inline = False
    for line in body.splitlines():
        if ";#ASM" in line:
            inline = "#ASMSTART" in line
            continue
        text = line.split(";")[0].strip()
        if re.match(r"[.\w$]+:$", text):
            since = None
        elif re.match(r"buffer_load\w* .*\blds$", text):
            since = 0
        elif re.match(r"(buffer|global|flat|scratch)_(load|store|atomic)", text) and since is not None:
            since += 1
        m = re.match(r"s_waitcnt vmcnt\((\d+)\)$", text)
        if inline and m and int(m.group(1)):
            checked += 1
            if since is None or since < int(m.group(1)):
                bad.append(f"{text} after {since}")
    return checked, bad


def early_reads(ir):
    """Uses of an inline-asm matrix instruction's result, itself or through
    phis, by anything but another inline-asm statement, in one IR function."""
    live = set(re.findall(r"(%\d+) = .*\basm sideeffect \"v_mfma", ir))
    lines = ir.splitlines()
    uses = [(m.group(1), m.group(2)) for m in (re.match(r"\s*(%\d+) = (.*)", l) for l in lines) if m]
    grown = True
    while grown:
        grown = False
        for name, text in uses:
            if name not in live and text.startswith("phi") and live & set(re.findall(r"%\d+", text)):
                live.add(name)
                grown = True
    bad = []
    for line in lines:
        text = line.split(" = ", 1)[-1].strip()
        if not text.startswith("phi") and " asm " not in text and live & set(re.findall(r"%\d+", text)):
            bad.append(text)
    return len(live), bad


def test_matrix_operands_settle(compiled):
    kernels = re.findall(r"^(\w+prefill_kernel\w+):(.*?)\.end_amdhsa_kernel", compiled[0], re.S | re.M)
    assert len(kernels) == 10
    total = 0
    for name, body in kernels:
        checked, bad = hazards(body)
        total += checked
        assert not bad, f"{name}: {bad[:3]}"
    assert total > 0


def test_lds_loads_land_before_the_barrier(compiled):
    total = 0
    for name, body in re.findall(r"^(\w+prefill_kernel\w+):(.*?)\.end_amdhsa_kernel", compiled[0], re.S | re.M):
        checked, bad = open_waits(body)
        total += checked
        assert not bad, f"{name}: {bad[:3]}"
    assert total >= 20  # at least one per stage of a super-step


def test_accumulators_read_after_the_wait(compiled):
    found = 0
    for m in re.finditer(r"^define [^\n]*@(\w*prefill_kernel\w*)\(.*?^}", compiled[1], re.S | re.M):
        n, bad = early_reads(m.group(0))
        found += n
        assert not bad, f"{m.group(1)}: {bad[:3]}"
    assert found > 0


def test_checks_find_planted_faults():
    asm = ("\tv_mov_b32_e32 v8, v1\n\ts_nop 0\n\t;;#ASMSTART\n\tv_mfma_f32_16x16x32_bf16 a[0:3], v[4:7], v[8:11], a[0:3]\n"
           "\t;;#ASMEND\n")
    assert hazards(asm) == (1, ["v_mfma_f32_16x16x32_bf16 a[0:3], v[4:7], v[8:11], a[0:3]"])
    assert hazards(asm.replace("s_nop 0", "s_nop 1")) == (1, [])
    assert len(hazards(asm.replace("s_nop 0", "s_nop 1\n.LBB0_1:"))[1]) == 1
    load = "\tbuffer_load_dwordx4 v1, s[0:3], s4 offen lds\n\tbuffer_load_dwordx4 v[2:5], v1, s[0:3], 0 offen\n"
    wait = "\t;;#ASMSTART\n\ts_waitcnt vmcnt(%d)\n\t;;#ASMEND\n"
    assert open_waits(load + wait % 1) == (1, [])
    assert open_waits(load + wait % 2) == (1, ["s_waitcnt vmcnt(2) after 1"])
    assert len(open_waits(load + ".LBB0_1:\n" + wait % 1)[1]) == 1
    ir = ('  %1 = call <4 x float> asm sideeffect "v_mfma $0", "=a"()\n  %2 = phi <4 x float> [ %1, %3 ]\n'
          "  %4 = extractelement <4 x float> %2, i64 0\n")
    assert early_reads(ir)[1] == ["extractelement <4 x float> %2, i64 0"]
    through = ir.replace("  %4 = extract", '  %5 = call <4 x float> asm sideeffect "", "=a,0"(<4 x float> %2)\n  %4 = extract')
    assert early_reads(through.replace("%2, i64", "%5, i64"))[1] == []
