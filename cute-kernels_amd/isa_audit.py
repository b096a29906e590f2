"""Checks the hand-counted waits of the streaming grouped-GEMM kernels against the compiler's assembly output.

Usage: python cute-kernels_amd/isa_audit.py [file.s]

The kernels of csrc/ragged_kernel.h wait for their operand loads with `s_waitcnt vmcnt(N)` where N is a constant
that counts the vector-memory instructions a wavefront has issued after the loads it waits for (loads and stores complete
in issue order). The constants are derived in the source from the number of loads per K step, the number of stores an
epilogue issues and whether a bias load or a request for row_index entries follows a step's loads. This script
compiles the sources that instantiate them to assembly (device code only; or reads a file made with `hipcc ... --cuda-device-only -S`) and checks,
for every instantiation of ragged_gemm_kernel, that the instruction stream has the shape those constants assume:

 * a K step issues four operand loads behind its first barrier, then the wait and the second barrier, then four more (tall kernels: four
   or five) and the request, if the kernel has one, and nothing else up to the next step's first barrier;
 * that wait allows exactly the four loads, the request of a step in the loop, or in a tile's first step the epilogue's stores and the
   bias load;
 * in the tall kernels both steps of a loop body of two issue the same number of loads, and there are eight steps with eight: the middle
   of the K loops for eight, four, two and one row blocks, which fetch no rows past 256 (every other step does);
 * the cold start issues sixteen operand loads (tall kernels: eighteen), as many stand-in stores as an epilogue issues stores, and
   waits for all but the loads of the second step and the stores;
 * the three-stage loop of groups of few rows issues five loads per step, and without a bias a second one six, and waits for all but as
   many;
 * there are exactly as many of each as the source has, and of the waits for everything in front of a barrier, and no operand load is
   outside of them;
 * no instantiation touches scratch memory, and none contains a loop over the distinct values of an operand that the
   hardware wants in scalar registers (what the compiler generates around a vector-memory instruction whose descriptor or
   scalar offset it cannot prove to be the same in every lane: each costs a dozen instructions and a branch per use).

For these kernels and those of csrc/grouped_gemm.hip it checks as well that a wavefront reaches every barrier with all of its LDS
reads returned. Behind a barrier the other wavefronts' loads may fill the stage that was read, and the compiler is free to move a matrix
instruction, and with it the wait for its fragments, past the barrier: only a wait of its own in front of the barrier keeps the reads there.

The kernels of csrc/grouped_gemm_f32.hip store four results as 16 bytes: none of their stores may be of 12 bytes, which is what the
compiler makes of four separate values next to an element-wise branch, with a store of the fourth shared by both.
"""

import os
import re
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
SOURCES = [os.path.join(CSRC, name) for name in ("grouped_gemm_ragged.hip", "grouped_gemm_ragged_tall.hip")]
# stores per wavefront and tile: plain, SwiGLU with h, SwiGLU, SwiGLU backward, fp32 sums of a split reduction
EPI_STORES = {0: 16, 1: 24, 2: 8, 3: 32, 4: 32}


def compile_to_assembly(source: str, path: str) -> None:
    from build import FLAGS, HIPCC  # the flags the library is built with

    cmd = [HIPCC] + FLAGS + ["--cuda-device-only", "-S", source, "-o", path]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(proc.stderr[-2000:])


def tokens(lines):
    """The vector-memory instructions, waits and barriers of a kernel in program order, and the number of loops over the
    distinct values of a scalar operand (readfirstlane, compare, s_and_saveexec, the instruction, s_xor exec, branch)."""
    cur, waterfalls = [], 0
    for k, line in enumerate(lines):
        s = line.strip()
        if s.startswith("s_cbranch_execnz") and any("s_xor_b64 exec, exec" in x for x in lines[max(0, k - 3):k]):
            waterfalls += 1
        if re.match(r"^\.LBB\d+_\d+:", line):
            cur.append(" ")
        elif s.startswith("s_barrier"):
            cur.append("|")
        elif s.startswith("s_waitcnt") and "vmcnt" in s:
            cur.append("w%s," % re.search(r"vmcnt\((\d+)\)", s).group(1))
        elif s.startswith("buffer_load_dwordx4") and " lds" in s:
            cur.append("O")  # sixteen bytes per lane into LDS: an operand load
        elif s.startswith("buffer_load_dword ") and " lds" in s:
            cur.append("p")  # four bytes per lane into LDS: bias, row table, row_index request across a tile boundary
        elif s.startswith("buffer_load") or s.startswith("global_load"):
            cur.append("L")  # a load into registers
        elif s.startswith("buffer_store") or s.startswith("global_store"):
            cur.append("s")
        elif s.startswith("scratch_"):
            cur.append("X")
    return [b for b in "".join(cur).split(" ") if b], waterfalls


# a K step: the loads behind its first barrier, the wait, the loads behind its second one and the request; waits that the compiler adds
# beside the counted one only wait for more
STEP = re.compile(r"\|(O*)(?:w\d+,)*w(\d+),\|(?:w\d+,)*(O*)([Lp]?)")
COLD = re.compile(r"((?:[OLp]|w\d+,)*O)(s+)w(\d+),\|")


def audit_kernel(name: str, body) -> list:
    """The problems of one instantiation of ragged_gemm_kernel. Every operand load has to belong to one of the four shapes (K step,
    step and start of the three-stage loop, cold start), and there has to be the exact number of each."""
    m = re.search(r"ragged_gemm_kernelINS0_(\w+?)ELb(\d)ELb(\d)ELi(\d)ELb(\d)ELb(\d)ELb(\d)ELb(\d)E", name)
    el, a_kc, b_kc, epi, vary_k, bias, gather, tall = m.group(1), *[int(x) for x in m.groups()[1:]]
    blocks, waterfalls = tokens(body)
    request = 1 if (vary_k and gather) else 0
    stores = EPI_STORES[epi]
    wait_step, wait_first = 4 + request, 4 + stores + bias
    tag = f"{el} A_KC={a_kc} B_KC={b_kc} epilogue={epi} reduction_varies={vary_k} bias={bias} gather={gather} tall={tall}"
    found = {"steps": 0, "first steps": 0, "steps of eight loads": 0, "cold starts": 0, "three-stage steps of 5": 0,
             "three-stage steps of 6": 0, "three-stage starts": 0, "drains": 0}  # fmt: skip
    # The versions of the K loop have their first step, and behind it the second one and a body of two; those of full tiles two steps more, for
    # the loads of the next tile, and so have those of tiles of few rows in the tall kernels. Three-stage: a body of three and
    # two more, for four versions of up to 64 rows and two of up to 128.
    # Drains (a wait for everything and a barrier): behind the kernel's first load, which fetches nothing, a tile that nothing streams behind,
    # the three-stage loop, and in front of a gathered tile's cold start.
    expected = {"steps": 28 if tall else 17, "first steps": 6 if tall else 5, "steps of eight loads": 8 if tall else 22, "cold starts": 1,
                "three-stage steps of 5": a_kc * 5 * 4, "three-stage steps of 6": 0 if bias else a_kc * 5 * 2,
                "three-stage starts": a_kc * (1 if bias else 2), "drains": 2 + a_kc + (gather and not vary_k)}  # fmt: skip
    problems = []

    def fail(what, block=""):
        problems.append(f"{tag}: {what}: {block[:120]}")

    if waterfalls:
        fail(f"{waterfalls} loops over the distinct values of a scalar operand")
    for blk in blocks:
        if "X" in blk:
            fail("scratch access", blk)
        if "O" not in blk:
            found["drains"] += len(re.findall(r"w0,\|", blk))
            continue
        cold = COLD.search(blk)
        if cold:
            loads = 8 + tall
            if cold.group(1).count("O") != 2 * loads or len(cold.group(2)) != stores or int(cold.group(3)) != loads + stores:
                fail(f"cold start: {cold.group(1).count('O')} loads, {len(cold.group(2))} stores, wait {cold.group(3)}; "
                     f"expected {2 * loads}, {stores}, {loads + stores}", blk)
            found["cold starts"] += 1
        elif re.match(r"(?:w\d+,)*\|O{1,4}w", blk):
            # steps, and nothing else that counts
            seconds = []
            for first, wait, second, asked in STEP.findall(blk):
                if len(first) != 4:
                    fail(f"{len(first)} operand loads between the barriers of a step, expected 4", blk)
                if int(wait) not in (wait_step, wait_first):
                    fail(f"a step waits for all but {wait}, expected {wait_step} or {wait_first}", blk)
                if len(second) not in (4, 4 + tall) or len(asked) != request:
                    fail(f"{second + asked} behind the second barrier, expected {4} or {4 + tall} operand loads and {request} requests", blk)
                found["first steps" if int(wait) == wait_first else "steps"] += 1
                found["steps of eight loads"] += len(second) == 4
                seconds.append(len(second))
            if len(set(seconds)) != 1:
                fail(f"steps of {seconds} loads behind the second barrier in one body", blk)
            if not re.fullmatch(r"(?:w\d+,)*#+(?:w\d+,)*", STEP.sub("#", blk)):
                fail("more than K steps in a block of K steps", blk)
        else:
            # the start of the three-stage loop with the loads of two steps in front, or a step or a body of it
            shape = re.match(r"(O*)((?:w\d+,\|O+)+)(?:w\d+,)*$", blk)
            runs = re.findall(r"w(\d+),\|(O+)", shape.group(2)) if shape else []
            thin = len(runs[0][1]) if runs else 0
            if thin not in (5, 6) or len(shape.group(1)) not in (0, 2 * thin):
                fail("operand loads of no known shape", blk)
                continue
            for wait, loads in runs:
                if len(loads) != thin or int(wait) != thin:
                    fail(f"a three-stage step of {len(loads)} loads waits for all but {wait}, expected {thin}", blk)
            start = 1 if shape.group(1) else 0
            found["three-stage starts"] += start
            found[f"three-stage steps of {thin}"] += len(runs) - start
    for what, n in expected.items():
        if found[what] != n:
            fail(f"{found[what]} {what}, expected {n}")
    if not problems:
        print(f"ok  {tag}: " + ", ".join(f"{n} {what}" for what, n in found.items()))
    return problems


def kernels(asm_path: str, pattern: str):
    """(name, lines) of the functions of a listing whose names match"""
    lines = open(asm_path).read().split("\n")
    found = [i for i, line in enumerate(lines) if re.match(rf"^{pattern}\w*:", line)]
    if not found:
        raise RuntimeError(f"no {pattern} in {asm_path}")
    for a in found:
        end = next(i for i in range(a, len(lines)) if lines[i].startswith(".Lfunc_end"))
        yield lines[a].split(":")[0], [line.split(";")[0] for line in lines[a:end]]


def audit(asm_path: str) -> int:
    problems = []
    for name, body in kernels(asm_path, r"_ZN6fmahip4gemm6ragged18ragged_gemm_kernel"):
        problems += audit_kernel(name, body)
    for p in problems:
        print("PROBLEM " + p)
    return len(problems)


def reads_out_at_barriers(body):
    """How many barriers of a kernel (its instructions, without comments) some path reaches with LDS operations outstanding: of every
    block the most that are out where it begins, over all its predecessors, until nothing changes."""
    labels, starts = {}, {0}
    for i, s in enumerate(body):
        m = re.match(r"^(\.LBB\d+_\d+):", s)
        if m:
            labels[m.group(1)] = i
            starts.add(i)
        elif s.startswith(("s_cbranch", "s_branch", "s_endpgm")) and i + 1 < len(body):
            starts.add(i + 1)
    starts = sorted(starts)
    end_of = dict(zip(starts, starts[1:] + [len(body)]))
    most, todo, flagged = {0: 0}, [0], set()
    while todo:
        start = todo.pop()
        out, end = most[start], end_of[start]
        for i in range(start, end):
            s = body[i]
            if s.startswith("ds_"):
                out += 1
            elif s.startswith("s_waitcnt"):
                m = re.search(r"lgkmcnt\((\d+)\)", s)
                out = min(out, int(m.group(1))) if m else out
            elif s.startswith("s_barrier") and out:
                flagged.add(i)
        out = min(out, 16)  # (the counter's range)
        last = body[end - 1]
        to = [labels[last.split()[-1]]] if last.startswith(("s_cbranch", "s_branch")) else []
        if not last.startswith(("s_branch", "s_endpgm")) and end < len(body):
            to.append(end)
        for t in to:
            if out > most.get(t, -1):
                most[t] = out
                todo.append(t)
    return len(flagged)


def audit_barriers(asm_path: str) -> int:
    """Every grouped-GEMM kernel of a listing: no barrier with LDS reads outstanding."""
    problems, seen = 0, 0
    for name, body in kernels(asm_path, r"_ZN6fmahip4gemm\w*(?:ragged|grouped)_gemm_kernel"):
        seen += 1
        out = reads_out_at_barriers([line.strip() for line in body])
        if out:
            problems += 1
            print(f"PROBLEM {name}: {out} barriers with LDS reads outstanding")
    print(f"{os.path.basename(asm_path)}: LDS reads at the barriers of {seen} kernels, {problems} with some outstanding")
    return problems


def audit_f32(asm_path: str) -> int:
    text = open(asm_path).read()
    whole, cut = len(re.findall(r"\bglobal_store_dwordx4\b", text)), len(re.findall(r"\bglobal_store_dwordx3\b", text))
    if whole == 0 or cut:
        print(f"PROBLEM fp32 products: {whole} stores of 16 bytes, {cut} of 12")
        return 1
    print(f"ok  fp32 products: {whole} stores of 16 bytes")
    return 0


def main() -> int:
    if len(sys.argv) > 1:
        return audit(sys.argv[1]) + audit_barriers(sys.argv[1])
    problems = 0
    sys.path.insert(0, HERE)
    with tempfile.TemporaryDirectory() as tmp:
        for source in SOURCES:
            path = os.path.join(tmp, os.path.basename(source) + ".s")
            compile_to_assembly(source, path)
            problems += audit(path) + audit_barriers(path)
        path = os.path.join(tmp, "grouped_gemm.hip.s")
        compile_to_assembly(os.path.join(CSRC, "grouped_gemm.hip"), path)
        problems += audit_barriers(path)
        path = os.path.join(tmp, "f32.s")
        compile_to_assembly(os.path.join(CSRC, "grouped_gemm_f32.hip"), path)
        problems += audit_f32(path)
    return problems


if __name__ == "__main__":
    n = main()
    print("audit passed" if n == 0 else f"{n} problem(s)")
    sys.exit(0 if n == 0 else 1)
