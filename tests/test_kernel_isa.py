"""Properties of the compiled code that no numerical test pins reliably.  In the pipelined gather
kernel the registers written by the hand-issued table loads must not be read by any instruction
before the ``s_waitcnt`` that releases them (a read before it returns whatever the register held,
sometimes the right value).  In the attention and GEMM kernels whose matrix products are inline assembly, which
the compiler takes for any other statement, the issue slots that such a product needs before and behind
it must be there.  The checks compile the source to gfx950 assembly and walk it."""

import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "speculators_amd", "csrc")


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
@pytest.mark.parametrize("source", sorted(f for f in os.listdir(CSRC) if f.endswith(".hip")))
def test_sources_compile_without_warnings(source):
    """An index past the end of a register array, for one, is a warning and nothing else."""
    subprocess.run(["hipcc", "-std=c++17", "--offload-arch=gfx950", "-fsyntax-only", "-Werror", "-Wno-unused-command-line-argument",
                    os.path.join(CSRC, source)], check=True, capture_output=True)


def _assembly(source, tmp_path):
    out = tmp_path / (source + ".s")
    subprocess.run(["hipcc", "-O3", "-std=c++17", "--offload-arch=gfx950", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", "-Wno-unused-command-line-argument", "-S",
                    "--cuda-device-only", "-o", str(out), os.path.join(CSRC, source)],
                   check=True, capture_output=True)
    return out.read_text()


def _registers(text):
    out = set()
    for kind, one, lo, hi in re.findall(r"\b([va])(?:(\d+)\b|\[(\d+):(\d+)\])", text):
        out.update((kind, i) for i in range(int(one or lo), int(one or hi) + 1))
    return out


class _Instruction:
    def __init__(self, text, in_asm):
        self.text, self.in_asm = text, in_asm
        self.op, _, rest = text.partition(" ")
        args = [a.strip() for a in re.split(r",(?![^\[]*\])", rest)] if rest else []
        self.target = args[0] if args else None
        self.product = self.op.startswith("v_mfma")
        self.passes = 8 if "32x32x16" in self.op else 4  # (16 x 16 x 32)
        self.slots = int(args[0], 0) + 1 if self.op == "s_nop" else self.passes if self.product else 1
        self.all = _registers(rest)
        if self.product:
            self.d, self.a, self.b, self.c = (_registers(a) for a in args[:4])
        both = self.op.startswith(("v_permlane16_swap", "v_permlane32_swap", "v_swap"))
        vector = self.op.startswith("v_") and not self.product
        self.writes = _registers(" ".join(args[:2 if both else 1])) if vector else set()


def _flow(body):
    """(instructions, the indexes that may come next of each)"""
    code, labels, in_asm = [], {}, False
    for line in body:
        if "#ASMSTART" in line or "#ASMEND" in line:
            in_asm = "#ASMSTART" in line
            continue
        text = line.split(";")[0].strip()
        if text.endswith(":"):
            labels[text[:-1]] = len(code)
        elif text and not text.startswith("."):
            code.append(_Instruction(text, in_asm))
    after = [[] for _ in code]
    for n, ins in enumerate(code):
        if ins.op.startswith(("s_branch", "s_cbranch")):
            after[n].append(labels[ins.target])
        if ins.op not in ("s_branch", "s_endpgm") and n + 1 < len(code):
            after[n].append(n + 1)
    return code, after


def _walk(start, edges, code, reach, visit):
    """visit(instruction, issue slots between) along every path from the instructions next to one, until it says so."""
    stack, seen = [(n, 0) for n in start], {}
    while stack:
        n, between = stack.pop()
        if between < reach and seen.get(n, reach) > between:
            seen[n] = between
            if not visit(code[n], between):
                stack += [(m, between + code[n].slots) for m in edges[n]]


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
@pytest.mark.parametrize("source,products", [
    # forward at head_dim 256 (V transposed beforehand or read transposing), dQ at 256 and 64
    ("attn_kernels.hip", {("attn_fwd_kernel", "256"): 256, ("attn_bwd_dq_kernel", "256"): 96, ("attn_bwd_dq_kernel", "64"): 24}),
    # two copies of a slab of 128 products each; with and without row statistics, row factors, whole leading dimensions
    ("gemm_bf16.hip", {("gemm_bf16_nt_kernel", "0"): 5 * 256, ("gemm_bf16_nt_kernel", "1"): 5 * 256}),
    # three copies; four kinds of result, with and without groups
    ("gemm_bf16_tn.hip", {("gemm_bf16_tn_kernel", str(out)): 2 * 384 for out in range(4)})])
def test_inline_products_have_their_issue_slots(source, products, tmp_path):
    """Two slots from a vector instruction that writes an operand to the product; behind it four more than its passes to whatever
    else touches its result, one less than its passes to a vector instruction that writes a C operand it only reads."""
    text = _assembly(source, tmp_path)
    counts = {}
    for m in re.finditer(r"^_ZN3spx\w*?\d+([a-z]+_\w+?_kernel)IL[ib](\d+)\w+:.*?^\.Lfunc_end", text, flags=re.S | re.M):
        code, after = _flow(m.group(0).splitlines()[1:-1])
        before = [[] for _ in code]
        for n, nexts in enumerate(after):
            for s in nexts:
                before[s].append(n)
        for n, p in enumerate(code):
            if not (p.product and p.in_asm):
                continue
            counts[m.groups()] = counts.get(m.groups(), 0) + 1
            operands, held = p.a | p.b | p.c, p.c - p.d

            def ahead(ins, between):
                assert not (ins.writes & operands and between < 2), (m.group(1), ins.text, between, p.text)

            def behind(ins, between):
                assert not ins.writes & held or between >= p.passes - 1, (m.group(1), p.text, between, ins.text)
                if ins.product and ins.c == ins.d == p.d and not (ins.a | ins.b) & p.d:
                    return True  # the next product onto it: it has a walk of its own
                assert not ins.all & p.d or between >= p.passes + 4, (m.group(1), p.text, between, ins.text)

            _walk(before[n], before, code, 2, ahead)
            _walk(after[n], after, code, 12, behind)
    assert counts == products


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
def test_hand_issued_loads_are_not_read_before_their_wait(tmp_path):
    text = _assembly("fused_loss.hip", tmp_path)
    kernels = re.findall(r"^(_ZN3spx27loss_fwd_gather_pipe_kernel\w+):", text, flags=re.M)
    assert len(kernels) == 2, kernels
    for name in kernels:
        body = text[text.index(name + ":"):]
        body = body[:body.index(".Lfunc_end")].splitlines()
        pending, loads, waits = set(), 0, 0
        for line in body:
            ins = line.strip()
            m = re.match(r"buffer_load_dword (v\d+), v\d+, s\[", ins)
            if m:
                pending.add(m.group(1))
                loads += 1
                continue
            if ins.startswith("s_waitcnt") and "vmcnt" in ins:
                pending.clear()
                waits += 1
                continue
            for reg in pending:
                assert not re.search(rf"\b{reg}\b", ins), f"{name}: {reg} read before its wait: {ins}"
            # a register range that covers a pending register counts as a read too
            for lo, hi in re.findall(r"v\[(\d+):(\d+)\]", ins):
                for reg in pending:
                    assert not int(lo) <= int(reg[1:]) <= int(hi), f"{name}: {reg} inside {ins}"
        # the prologue and the two unrolled tiles issue eight loads each
        assert loads == 24 and waits >= 3, (name, loads, waits)


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
@pytest.mark.parametrize("source,name,count", [("gemm_bf16_walk.hip", "gemm_bf16_walk_kernel", 6),
                                               ("gemm_bf16_tn_walk.hip", "gemm_bf16_tn_walk_kernel", 2)])
def test_named_accumulators_are_nobody_elses(source, name, count, tmp_path):
    """The kernels that walk their tiles hold the accumulators in a0 .. a255 by name: no statement of the compiler's own touches
    an accumulation register, none spills, and around every product lie the issue slots that it needs (as above; a fresh
    product's result has no C operand)."""
    text = _assembly(source, tmp_path)

    def decimal(m):
        return "a[" + ":".join(str(int(x, 0)) for x in m.group(1).split(":")) + "]" if ":" in m.group(1) else f"a{int(m.group(1), 0)}"

    text = re.sub(r"\ba\[([\w:]+)\]", decimal, text)
    kernels = 0
    for m in re.finditer(rf"^_ZN3spx\w*\d{name}\w+:.*?^\.Lfunc_end", text, flags=re.S | re.M):
        kernels += 1
        code, after = _flow(m.group(0).splitlines()[1:-1])
        before = [[] for _ in code]
        for n, nexts in enumerate(after):
            for s in nexts:
                before[s].append(n)
        fresh = 0
        for n, p in enumerate(code):
            assert p.in_asm or not any(kind == "a" for kind, _ in p.all), p.text
            assert not p.op.startswith("scratch_"), p.text
            if not p.product:
                continue
            assert p.in_asm and (not p.c or p.c == p.d) and len(p.d) == 4
            fresh += not p.c

            def ahead(ins, between):
                assert not (ins.writes & (p.a | p.b) and between < 2), (ins.text, between, p.text)

            def behind(ins, between):
                if ins.product and ins.d == p.d and not (ins.a | ins.b) & p.d:
                    return True
                assert not ins.all & p.d or between >= p.passes + 4, (p.text, between, ins.text)

            _walk(before[n], before, code, 2, ahead)
            _walk(after[n], after, code, 12, behind)
        assert fresh == 64 and sum(p.product for p in code) == 256
    assert kernels == count
