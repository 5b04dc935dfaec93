#!/usr/bin/env python3
"""Reads the compiler's kernel-resource-usage remarks of one translation unit (hipcc -Rpass-analysis=kernel-resource-usage,
stderr saved by the Makefile) and fails when a four-wave GEMM kernel uses scratch memory; and reads the assembly the
compiler wrote for the same translation unit (-save-temps) and fails when, in such a kernel, an accumulator register
(a0..a255) appears outside the kernel's own asm statements.

Those kernels keep 256 accumulators in a[0:255] across separate asm statements and pass the K loop ~28 operands; the
registers around the loop are tight by design.  A kernel that touches scratch at all pays for it at every dispatch (a
256-workgroup launch costs ~4 us more), and a lambda that stops being inlined, or address arithmetic hoisted out of the
tile loop, shows up here first: as bytes of scratch per lane.

The accumulators stay in a[0:255] from the statements that set them up, through the K loop, to the statements of the
write-back; the compiler is told that those statements clobber them, not that they carry values, so it must not use
the accumulator file for anything of its own in between (copies of vector registers it has run out of, say).  It does
not today -- the kernels ask for all 256 vector registers and the allocator prefers them -- and the check keeps it so.

And the register-staged edge kernels: a CU holds four workgroups of the 64 x 64 tiles, which is 128 vector registers each and
no scratch; the 128 x 128 ones (two) use no scratch; the 256 x 256 ones none for 16-bit inputs and up to 20 bytes per lane for int8.  The other
32x32-shape kernels: no scratch for 16-bit and fp32 inputs, up to 76 bytes for int8.

And the short-K kernels: two workgroups to a CU, which is 256 vector registers each, and no scratch.

    python3 check_resources.py <remarks .txt | assembly .s> [...]
"""
import re
import sys


def kernels(text):
    """(function name, {field: value}) per kernel of the remarks text."""
    out, cur = [], None
    for line in text.splitlines():
        # (the place in the source stands before "remark:" or after it, as the compiler's version has it)
        m = re.search(r"remark:\s+(?:\S+:\d+:\d+:\s+)?(.*?)(?:\s+\[-Rpass-analysis=kernel-resource-usage\])?$", line)
        if not m:
            continue
        body = m.group(1).strip()
        if body.startswith("Function Name:"):
            cur = (body.split(":", 1)[1].strip(), {})
            out.append(cur)
        elif cur and ":" in body:
            k, v = body.split(":", 1)
            cur[1][k.strip()] = v.strip()
    return out


# register-staged edge kernels: (edge length of the tile) -> most vector registers, most bytes of scratch per lane
_STAGED = re.compile(r"gemm_mfma_kernelINS_10MfmaConfigILi(\d+)ELi(\d+)ELi\d+ELi\d+ELi\d+ELb[01]ELb[01]ELb0ELb1E")
_STAGED_LIMITS = {64: (128, 0), 128: (256, 0), 256: (256, 0)}
_I8 = 2  # (number of the input type in a kernel's name)
# every other 32x32-shape kernel, and the short-K kernels: most bytes of scratch per lane
_OTHERS = re.compile(r"gemm_mfma_kernelINS_10MfmaConfigILi(\d+)E")
_SHORT_K = "gemm_short_k_kernel"

_AREG = re.compile(r"(?<![\w.$])a(\d+|\[\d+:\d+\])(?!\w)")


def agpr_uses_outside_asm(text):
    """{kernel: [lines]} of compiler-written instructions that name an accumulator register, per four-wave kernel of an
    assembly listing; and the number of such kernels seen."""
    cur, in_asm, bad, seen = None, False, {}, set()
    for line in text.splitlines():
        m = re.match(r"^(_ZN6acc950\w+):", line)
        if m:
            cur, in_asm = m.group(1), False
        elif line.startswith(".Lfunc_end"):
            cur = None
        if cur is None or "gemm_mfma16w4_kernel" not in cur:
            continue
        seen.add(cur)
        if ";;#ASMSTART" in line:
            in_asm = True
        elif ";;#ASMEND" in line:
            in_asm = False
        elif not in_asm:
            code = line.split(";")[0]
            if _AREG.search(code) or "v_accvgpr" in code:
                bad.setdefault(cur, []).append(line.strip())
    return bad, len(seen)


def main(paths):
    bad, staged_bad, seen = [], [], {}
    for path in [p for p in paths if p.endswith(".s")]:
        uses, seen[path] = agpr_uses_outside_asm(open(path, errors="replace").read())
        for name, lines in uses.items():
            bad.append(f"{name}: the compiler uses accumulator registers outside the asm statements, e.g. `{lines[0]}` ({len(lines)} places)")
    for path in [p for p in paths if not p.endswith(".s")]:
        seen[path] = 0
        for name, f in kernels(open(path, errors="replace").read()):
            scratch = int(f.get("ScratchSize [bytes/lane]", "0"))
            staged, other = _STAGED.search(name), _OTHERS.search(name)
            if staged or other or _SHORT_K in name:
                vgprs, most = _STAGED_LIMITS[int(staged.group(2))] if staged else (256, 0)
                if other and int(other.group(1)) == _I8:
                    most = (20 if int(staged.group(2)) == 256 else 0) if staged else 76
                if int(f.get("VGPRs", "0")) > vgprs or scratch > most:
                    staged_bad.append(f"{name}: {f.get('VGPRs')} vector registers (at most {vgprs}), {scratch} bytes of scratch per lane (at most {most})")
            if _SHORT_K in name:
                seen[path] += 1
            if "gemm_mfma16w4_kernel" not in name:
                continue
            seen[path] += 1
            if scratch:
                bad.append(f"{name}: {scratch} bytes of scratch per lane (VGPRs spilled: {f.get('VGPRs Spill')}, SGPRs spilled: {f.get('SGPRs Spill')})")
    if bad:
        print("four-wave GEMM kernels must not use scratch memory, nor the compiler their accumulator registers:\n  " + "\n  ".join(bad), file=sys.stderr)
        return 1
    if staged_bad:
        print("kernels take more than they may:\n  " + "\n  ".join(staged_bad), file=sys.stderr)
        return 1
    unread = [path for path, n in seen.items() if not n] # (a file in which nothing is found is one that was not understood)
    if unread:
        print("no four-wave or short-K GEMM kernel found in " + ", ".join(unread), file=sys.stderr)
        return 1
    return 0


if __name__ == "__main__":
    sys.exit(main(sys.argv[1:]))
