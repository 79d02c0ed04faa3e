"""Guard against register spills inside the K loops of the large-tile kernels, and against loads that read a
scalar register too soon.

``python -m tileccl_amd.csrc.check_spills`` compiles ``tccl_api.hip`` and ``tccl_kmajor.hip`` to
assembly (about two minutes) and, for every ``gemm256_kernel`` / ``fused256_kernel``
instantiation, counts the scratch-memory instructions that lie between the kernel's first and last
MFMA, i.e. inside its K loops.  A register that the compiler keeps in scratch memory there is
reloaded through the same queue as the operand loads, so the reload waits for all of them: a
handful of such reloads per K step has cost the fused launches more than a third of their time.
The fused kernels run at the register limit; changes to the K step or to the background transfer
should be followed by this check.  Exit status 1 if any count exceeds ``--allow`` (default: the
two reloads of the rarely taken block-change path of the all-gather kernels).

The count over the whole kernel is printed as well.  In an all-gather kernel the accesses outside
the K loops sit on rarely taken paths; in a reduce-scatter kernel (third template argument true)
they sit in the reduction phases, between loads of the addends, and are marked: 32 of them made
the 8192 x 4096 x 2048 reduce-scatter 4 % slower.

A vector memory instruction must not read a scalar register within five wait states of the vector
instruction (v_readlane, v_readfirstlane, a compare) that wrote it: the hardware does not wait.  The compiler
pads its own accesses but does not look inside inline assembly, which is how the large-tile kernels issue their
global -> LDS loads.  Every such load of the listing is checked, backwards through every block it can be reached from; a
load that comes too soon is printed and makes the exit status 1.
"""

from __future__ import annotations

import argparse
import re
import subprocess
import sys
import tempfile
from pathlib import Path

from tileccl_amd.csrc.build import FLAGS, HERE, SOURCES


def kernels(asm: str):
    """(name, vgprs, scratch instructions in the K loops, scratch instructions in all) per large-tile kernel."""
    counts = dict(re.findall(r"\.name:\s+(\S+)\n(?:.*\n)*?\s+\.vgpr_count:\s+(\d+)", asm))
    for match in re.finditer(r"^(_ZN4tccl1[45](?:gemm|fused)256_kernel\w*):", asm, flags=re.M):
        name = match.group(1)
        body = asm[match.end(): asm.index(".Lfunc_end", match.end())].split("\n")
        mfma = [i for i, line in enumerate(body) if "v_mfma" in line]
        scratch = [i for i, line in enumerate(body) if "scratch_" in line]
        inside = [i for i in scratch if mfma and mfma[0] < i < mfma[-1]]
        yield name, int(counts.get(name, 0)), len(inside), len(scratch)


def is_reduce(name: str) -> bool:
    """Whether the mangled name is a fused kernel instantiated for reduce-scatter (first bool argument)."""
    match = re.search(r"fused256_kernelI.*?Lb([01])E", name)
    return bool(match) and match.group(1) == "1"


WAIT_STATES = 5  # between a vector instruction that writes a scalar register and a vector memory instruction that reads it


def scalars(operand: str) -> set[int]:
    """Numbers of the scalar registers an operand names: s12 or s[4:7]."""
    match = re.fullmatch(r"s(?:(\d+)|\[(\d+):(\d+)\])", operand)
    if not match:
        return set()
    first = int(match.group(1) or match.group(2))
    return set(range(first, int(match.group(3) or first) + 1))


def decode(line: str) -> tuple[str, list[str]] | None:
    """(mnemonic, operands) of a line that holds an instruction."""
    text = line.split(";")[0].split("//")[0].strip()
    if not text or text.startswith((".", "#")) or text.endswith(":"):
        return None
    name, _, rest = text.partition(" " if " " in text else "\t")
    return name, [o.split()[0] for o in rest.replace("\t", " ").split(",") if o.strip()]


def states(name: str, operands: list[str]) -> int:
    return int(operands[0], 0) + 1 if name == "s_nop" else 1


def vector_written(name: str, operands: list[str]) -> set[int]:
    """Scalar registers that a vector instruction writes."""
    if not name.startswith("v_") or not operands:
        return set()
    out = scalars(operands[0])
    if len(operands) > 1 and ("_co_" in name or name.startswith(("v_mad_u64", "v_mad_i64", "v_div_scale"))):
        out |= scalars(operands[1])
    return out


def early_reads(body: list[str]) -> list[tuple[int, int]]:
    """(line of a global -> LDS load, line of the vector instruction that wrote a register it reads) with fewer than
    WAIT_STATES wait states between the two, on any way to the load."""
    code = [decode(line) for line in body]
    labels = {m.group(1): i for i, line in enumerate(body) if (m := re.match(r"(\.?\w+):", line))}
    sources: dict[int, list[int]] = {}
    for i, ins in enumerate(code):
        if ins and ins[0].startswith(("s_branch", "s_cbranch")) and ins[1] and ins[1][0] in labels:
            sources.setdefault(labels[ins[1][0]], []).append(i)
    found = set()
    for at, ins in enumerate(code):
        if not ins or not ins[0].startswith("buffer_load") or not re.search(r"\blds\b", body[at]):
            continue
        reads = set().union(*(scalars(o) for o in ins[1]))
        todo, seen = [(at - 1, 0, frozenset(reads), False)], set()
        while todo:
            i, gone, wanted, jumped = todo.pop()
            while i >= 0 and gone < WAIT_STATES and wanted and (i, gone, wanted) not in seen:
                if code[i]:
                    name, operands = code[i]
                    if name in ("s_branch", "s_endpgm", "s_setpc_b64") and not jumped:
                        break  # nothing falls through this line
                    if vector_written(name, operands) & wanted:
                        found.add((at, i))
                        break
                    if name.startswith("s_") and operands:
                        wanted -= scalars(operands[0])  # (a scalar write is waited for by the hardware)
                    gone += states(name, operands)
                else:
                    seen.add((i, gone, wanted))
                    todo += [(j, gone, wanted, True) for j in sources.get(i, ())]
                jumped = False
                i -= 1
    return sorted(found)


def bodies(asm: str):
    """(name, lines) of every function of the listing."""
    for match in re.finditer(r"^(_Z\w+):.*$", asm, flags=re.M):
        end = asm.find(".Lfunc_end", match.end())
        if end >= 0:
            yield match.group(1), asm[match.end(): end].split("\n")


def report(asm: str, allow: int) -> bool:
    """Print what is found; whether all of it is as it should be."""
    good = True
    for name, vgprs, inside, total in kernels(asm):
        good &= inside <= allow
        flag = "  <-- spills in the K loop" if inside > allow else ""
        if not flag and total and is_reduce(name):
            flag = "  (scratch accesses in a reduce-scatter kernel)"
        print(f"{name}: {vgprs} VGPRs, scratch instructions {inside} in K loops / {total} in all{flag}")
    for name, body in bodies(asm):
        early = early_reads(body)
        if early:
            good = False
            load, write = early[0]
            print(f"{name}: {len(early)} loads read a scalar register too soon, first:\n{body[write]}\n    ...\n{body[load]}")
    return good


def main() -> int:
    ap = argparse.ArgumentParser(description=__doc__.split("\n\n")[0])
    ap.add_argument("--allow", type=int, default=2, help="scratch instructions tolerated inside a kernel's K loops")
    ap.add_argument("asm", nargs="*", help="check these assembly files instead of compiling the sources")
    args = ap.parse_args()
    good = True
    for path in args.asm:
        good &= report(Path(path).read_text(), args.allow)
    if args.asm:
        return 0 if good else 1
    with tempfile.TemporaryDirectory(prefix="tccl_spills_") as tmp:
        for src in SOURCES:
            out = Path(tmp) / (src.stem + ".s")
            cmd = ["hipcc", *FLAGS, "-S", "--cuda-device-only", str(src), "-o", str(out)]
            subprocess.run(cmd, check=True, capture_output=True, text=True, cwd=HERE)
            good &= report(out.read_text(), args.allow)
    return 0 if good else 1


if __name__ == "__main__":
    sys.exit(main())
