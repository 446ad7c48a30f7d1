#!/usr/bin/env python3
"""Build-time check of the device assembly of kernels whose matrix instructions are inline assembly.

The pipelined GEMM loops write v_mfma as inline assembly with the accumulator as one read-and-written
operand (Traits::mfma16_inplace).  The compiler's hazard recogniser does not look into inline assembly, so
the wait states that a matrix instruction needs are not inserted for it:
  * its result may be touched by any other kind of instruction only some wait states later (7 for the
    16x16x32 shape; SETTLE are asked for here);
  * the result of a matrix instruction that the compiler issued may be its operand no sooner either, other than as
    the accumulator in the very same registers;
  * a vector register that an ordinary vector instruction wrote may be its operand only 2 wait states later
    (FEED are asked for).
In the source the accumulators are zeroed long before the loop, operands come from LDS reads (which the
compiler does wait for) and mfma_settle() stands behind the last product.  What remains are copies that the
register allocator may insert anywhere.  This scan follows every path of SETTLE wait states behind each
MFMA, and of FEED behind each vector instruction, and fails if it finds one too close.

A file in which no kernel with such instructions is recognised fails too, and so does a pipelined kernel whose loops do
not have them all: the last reduction tile, which the compiler issues, repeats the loop's tile, so there are as many
of one kind as of the other (none in the stream-K kernels, which leave all products to the compiler).

usage: check_mfma.py file.s     (exit status 1 on a violation)
"""
import re
import sys

SETTLE, FEED = 18, 3
REG = re.compile(r"\b([av])(\d+)\b|\b([av])\[(\d+):(\d+)\]")


def registers(text):
    out = set()
    for m in REG.finditer(text):
        if m.group(1):
            out.add((m.group(1), int(m.group(2))))
        else:
            out.update((m.group(3), r) for r in range(int(m.group(4)), int(m.group(5)) + 1))
    return out


def operands(text):
    parts = text.split(None, 1)
    return [p.strip() for p in parts[1].split(",")] if len(parts) > 1 else []


def parse(lines):
    """(text, inline assembly, line number) of a kernel's instructions, and the index behind each label."""
    code, labels, in_asm = [], {}, False
    for n, raw in lines:
        raw = raw.strip()
        if re.match(r";+#ASMSTART", raw):
            in_asm = True
        elif re.match(r";+#ASMEND", raw):
            in_asm = False
        else:
            text = raw.split(";")[0].strip()
            if text.endswith(":"):
                labels[text[:-1]] = len(code)
            elif text and not text.startswith("."):
                code.append((text, in_asm, n))
    return code, labels


def states(text):
    m = re.match(r"s_nop (\d+)", text)
    return int(m.group(1)) + 1 if m else 1


def follow(code, labels, start, budget, visit):
    """Calls visit(text, asm, line) for every instruction less than `budget` wait states behind `start`."""
    todo, seen = [(start, budget)], {}
    while todo:
        i, left = todo.pop()
        while left > 0 and i < len(code) and seen.get(i, 0) < left:
            seen[i] = left
            text, asm, line = code[i]
            visit(text, asm, line)
            if text.startswith("s_endpgm"):
                break
            m = re.match(r"s_c?branch\S*\s+(\S+)", text)
            left -= states(text)
            if m and m.group(1) in labels:
                todo.append((labels[m.group(1)], left))
                if text.startswith("s_branch"):
                    break
            i += 1


# instructions that write both of their operands
SWAPS = re.compile(r"v_(swap_|permlane(16|32)_swap_)")
PIPELINED = re.compile(r"gemm_(group_|dx_dw_)?kernel_pipelined")
STREAM_K = re.compile(r"gemm_kernel_pipelined.*Lb1ELb[01]EEEv")


def check(path):
    lines = open(path).read().split("\n")
    starts = [i for i, l in enumerate(lines) if re.match(r"^_Z\w+:", l)] + [len(lines)]
    failures = kernels = products = 0
    for begin, end in zip(starts, starts[1:]):
        name = lines[begin].split(":")[0]
        code, labels = parse([(n + 1, lines[n]) for n in range(begin + 1, end)])
        matrix = [i for i, (text, _, _) in enumerate(code) if text.startswith("v_mfma")]
        mine = sum(code[i][1] for i in matrix)
        if PIPELINED.search(name) and 2 * mine != (0 if STREAM_K.search(name) else len(matrix)):
            print(f"{path}: {name}: {mine} of {len(matrix)} matrix instructions are inline assembly")
            failures += 1
        if not mine:
            continue
        kernels += 1
        products += mine
        found = set()
        for i in matrix:
            text, inline, line = code[i]
            dst = registers(operands(text)[0])

            def near(other, asm, at):
                if other.startswith("v_mfma"):
                    if not (inline or asm):
                        return
                    ops = operands(other)
                    used = [registers(o) for o in ops[:4]]
                    # (in place on the same registers is what the hardware orders by itself)
                    if used[0] == dst and used[3] == dst and not (used[1] | used[2]) & dst:
                        return
                    if any(u & dst for u in used):
                        found.add((line, at, other))
                elif inline and registers(other) & dst:
                    found.add((line, at, other))

            follow(code, labels, i + 1, SETTLE, near)
        for i, (text, asm, line) in enumerate(code):
            if not text.startswith("v_") or text.startswith(("v_mfma", "v_cmp", "v_readfirstlane")):
                continue
            dst = registers(",".join(operands(text)[: 2 if SWAPS.match(text) else 1]))
            if not dst:
                continue

            def feeds(other, other_asm, at):
                if other_asm and other.startswith("v_mfma") and registers(",".join(operands(other)[1:])) & dst:
                    found.add((line, at, other))

            follow(code, labels, i + 1, FEED, feeds)
        for line, at, other in sorted(found):
            print(f"{path}:{line}: {name}: too few wait states before line {at}: {other}")
        failures += len(found)
    print(f"check_mfma: {products} inline-assembly matrix instructions in {kernels} kernels of {path}, {failures} violation(s)")
    if kernels == 0:
        print(f"{path}: no kernel with inline-assembly matrix instructions recognised: nothing was verified")
        failures += 1
    return failures


if __name__ == "__main__":
    sys.exit(1 if check(sys.argv[1]) else 0)
