"""Refuses device code whose register allocator stores a spill under the wrong lane mask.

    python3 check_exec_mask.py <device assembly (.s)> ...

Where control flow of diverging lanes joins, the compiler first restores the
lane mask (``s_or_b64 exec, exec, ..``) and then goes on.  Under register
pressure its allocator can put the store of a spilled vector register before
that restore, when writes of spilled scalar registers to lanes
(``v_writelane``) already stand there: the store then reaches only the lanes
of the branch, or none where the branch was skipped with an empty mask, and
the reload hands the others whatever the scratch slot held.  That is how the
4-slot aerosol integrator, compiled with plain loads of its stream, lost the
largest step length ``_dtmax`` of every cell with at most 192 unknowns: the
only such store in that build, at the join after the load of unknowns 192 to
255.  The compiler gives no diagnostic, so the build looks for it.

Reported are, between the start of a block and the restore of its mask,
  * any vector instruction, in a block that a branch on an empty mask
    (``s_cbranch_execz``) leads to;
  * any access to scratch memory, in every other block.

Kernels that spill vector registers at all are named, without an error: they
are where such a store can appear.
"""
import re
import sys

_RESTORE = re.compile(r"s_or_b64 exec, exec|s_or_saveexec|s_andn2_saveexec")
_MASK = re.compile(r"s_\w+ exec\b|s_\w+saveexec")
_VECTOR = re.compile(r"v_(?!writelane|readlane|readfirstlane)|scratch_|ds_|global_|buffer_|flat_")


def find(lines):
    """(function, block, line number, instruction) of every misplaced instruction."""
    lines = list(lines)
    joins = {m.group(1) for m in (re.match(r"\s*s_cbranch_execz (\S+)", ln) for ln in lines) if m}
    out, function, block, before, open_ = [], "", "", [], False
    for no, line in enumerate(lines, 1):
        start = re.match(r"(\.LBB\w+):|; (%bb\.\d+):", line)
        if start:
            block, before, open_ = start.group(1) or start.group(2), [], True
            continue
        label = re.match(r"([A-Za-z_]\w*):", line)
        if label:
            function, open_ = label.group(1), False
            continue
        text = line.split(";")[0].strip()
        if not open_ or not text:
            continue
        if _MASK.match(text):
            open_ = False
            if _RESTORE.match(text):
                out += [(function, block, n, t) for n, t in before]
        elif _VECTOR.match(text) and (block in joins or text.startswith("scratch_")):
            before.append((no, text))
    return out


def spills(lines):
    """{kernel: spilled vector registers} of the kernels that spill any, from the code object's metadata."""
    out, name = {}, ""
    for line in lines:
        m = re.match(r"\s*\.name:\s+'?(_Z\w+)|\s*\.vgpr_spill_count:\s+(\d+)", line)
        if m and m.group(1):
            name = m.group(1)
        elif m and int(m.group(2)):
            out[name] = int(m.group(2))
    return out


def main(paths):
    bad = 0
    for path in paths:
        with open(path) as f:
            lines = f.readlines()
        for kernel, n in spills(lines).items():
            print(f"note: {n} vector registers spilled: {kernel}")
        for function, block, no, text in find(lines):
            bad += 1
            print(f"{path}:{no}: {function}: {block}: before the lane mask is restored: {text}")
    if bad:
        print("This compiler stored registers under the wrong lane mask; change the kernel's register pressure.")
    return 1 if bad else 0


if __name__ == "__main__":
    sys.exit(main(sys.argv[1:]))
