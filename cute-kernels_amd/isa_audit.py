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
 * in the tall kernels both steps of a loop body of two issue the same number of loads, and there are four bodies with eight: the middle of
   the K loops for eight, four, two and one row blocks, which fetch no rows past 256 (every other step does);
 * the cold start issues sixteen operand loads (tall kernels: eighteen), as many stand-in stores as an epilogue issues stores, and
   waits for all but the loads of the second step and the stores;
 * the three-stage loop of groups of few rows issues five loads per step with a bias and otherwise six, and waits for all but as many;
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


def audit(asm_path: str) -> int:
    lines = open(asm_path).read().split("\n")
    starts = [i for i, line in enumerate(lines) if re.match(r"^_ZN6fmahip4gemm6ragged18ragged_gemm_kernel.*:", line)]
    if not starts:
        raise RuntimeError("no ragged_gemm_kernel in " + asm_path)
    starts.append(len(lines))
    problems = 0
    for a, b in zip(starts[:-1], starts[1:]):
        name = lines[a].split(":")[0]
        m = re.search(r"ragged_gemm_kernelINS0_(\w+?)ELb(\d)ELb(\d)ELi(\d)ELb(\d)ELb(\d)ELb(\d)ELb(\d)E", name)
        el, a_kc, b_kc, epi, vary_k, bias, gather, tall = m.group(1), *[int(x) for x in m.groups()[1:]]
        body = lines[a:b]
        end = next((k for k, line in enumerate(body) if "s_endpgm" in line), len(body))
        blocks, waterfalls = tokens(body[:end])
        request = 1 if (vary_k and gather) else 0
        stores = EPI_STORES[epi]
        wait_step, wait_first = 4 + request, 4 + stores + bias
        tag = f"{el} A_KC={a_kc} B_KC={b_kc} epilogue={epi} reduction_varies={vary_k} bias={bias} gather={gather} tall={tall}"
        found = {"step": 0, "first": 0, "body": 0, "eight": 0, "cold": 0, "thin": 0}

        def fail(what, block):
            nonlocal problems
            problems += 1
            print(f"PROBLEM {tag}: {what}: {block[:120]}")

        if waterfalls:
            fail(f"{waterfalls} loops over the distinct values of a scalar operand", "")
        for blk in blocks:
            if "X" in blk:
                fail("scratch access", blk)
            # the steps: in front of the second barrier four operand loads since the first
            for before, w, after in re.findall(r"\|([OLp]+|(?:[OLp]|w\d+,)*?)w(\d+),\|((?:[OLp]|w\d+,)*)", blk):
                n, count = int(w), before.count("O")
                if count != 4:
                    continue
                if len(re.sub(r"w\d+,", "", before)) != 4:
                    fail(f"{before} between the barriers of a step, expected four operand loads", blk)
                if n == wait_step:
                    found["step"] += 1
                elif n == wait_first:
                    found["first"] += 1
                else:
                    fail(f"a step waits for all but {n}, expected {wait_step} or {wait_first}", blk)
                behind = after.count("O")
                if behind not in (4, 4 + tall):
                    fail(f"{behind} operand loads behind the second barrier", blk)
            # the three-stage loop
            for w, loads in re.findall(r"w(\d+),\|(O+)", blk):
                if len(loads) in (5, 6) and int(w) == len(loads) and "|OOOOw" not in blk:
                    found["thin"] += 1
            # a loop body of two steps in one block: what is issued from the first step's second barrier to the second step's first
            # barrier, and behind the second step's second barrier
            for between, second in re.findall(r"\|O{4}w\d+,\|([^|]*)\|O{4}w\d+,\|((?:[OLp]|w\d+,)*)", blk):
                if between.count("O") != second.count("O"):
                    fail(f"{between.count('O')} and {second.count('O')} operand loads in the second halves of a body's steps", blk)
                found["eight"] += second.count("O") == 4
                issued = len(re.sub(r"w\d+,", "", between))
                if issued in (4 + request, 4 + tall + request):
                    found["body"] += 1
                else:
                    fail(f"{issued} instructions between two steps, expected {4 + request}" + (f" or {5 + request}" if tall else ""), blk)
            # the cold start: sixteen operand loads (the gathered kinds mix loads of row_index entries in), the stand-in
            # stores, the wait
            cold = re.search(r"((?:[OLp]|w\d+,)*O)(s+)w(\d+),\|", blk)
            if cold and cold.group(1).count("O") >= 16:
                found["cold"] += 1
                loads = 8 + tall
                if cold.group(1).count("O") != 2 * loads or len(cold.group(2)) != stores or int(cold.group(3)) != loads + stores:
                    fail(f"cold start: {cold.group(1).count('O')} loads, {len(cold.group(2))} stores, wait {cold.group(3)}; "
                         f"expected {2 * loads}, {stores}, {loads + stores}", blk)
        if found["step"] == 0 or found["first"] == 0 or found["cold"] != 1:
            fail(f"expected shapes not found ({found})", "")
        if a_kc and found["thin"] == 0:
            fail("no three-stage loop found", "")
        if tall and (found["eight"] != 4 or found["body"] == 4):
            fail(f"{found['eight']} of {found['body']} loop bodies with eight operand loads, expected 4 and some with nine", "")
        print(f"ok  {tag}: steps {found['step']}, first steps {found['first']}, two-step bodies {found['body']}, "
              f"three-stage steps {found['thin']}")
    return problems


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
    lines = open(asm_path).read().split("\n")
    starts = [i for i, line in enumerate(lines) if re.match(r"^_ZN6fmahip4gemm\w*(ragged|grouped)_gemm_kernel\w*:", line)]
    if not starts:
        raise RuntimeError("no grouped-GEMM kernel in " + asm_path)
    problems = 0
    for a in starts:
        end = next(i for i in range(a, len(lines)) if lines[i].startswith(".Lfunc_end"))
        out = reads_out_at_barriers([line.split(";")[0].strip() for line in lines[a:end]])
        if out:
            problems += 1
            print(f"PROBLEM {lines[a].split(':')[0]}: {out} barriers with LDS reads outstanding")
    print(f"{os.path.basename(asm_path)}: LDS reads at the barriers of {len(starts)} kernels, {problems} with some outstanding")
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
