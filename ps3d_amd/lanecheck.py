"""Check of the compiler's gfx950 listings for register spills with lanes switched off.

Where the paths of a divergent branch meet, the first thing to run is `s_or_b64 exec, exec,
...`, which switches the other path's lanes on again.  The register allocator of ROCm 7.2's
compiler can put a spill store or reload ahead of it: only the lanes of the branch then save
(or get back) a value that all of them use afterwards.  Seen in a build of the z pass at
nz = 1024 (204 bytes per lane of scratch): one value per thread was saved by the lane that
holds the upper lid alone, and the step came out 3e-3 off with no error.  Whether a kernel is
hit changes with any edit near it, so the build looks at every kernel each time.

A store is reported if the value was not formed since the lanes were last switched, a reload
if nothing reads it before they are switched on again: both belong after the restore.
"""
import re

_FUNC = re.compile(r"^([\w.$]+):\s*;\s*@\1\b(.*?)^\.Lfunc_end", re.S | re.M)
_BLOCK = re.compile(r"^(?:\.LBB\w+:.*|; %bb\.\d+:.*)$", re.M)
_REG = re.compile(r"\b([va])\[(\d+):(\d+)\]|\b([va])(\d+)\b")
_EXEC = re.compile(r"\bexec\b|saveexec")
_RESTORE = re.compile(r"s_or_b64 exec, exec|s_or_saveexec")


def _regs(text):
    out = set()
    for kind, lo, hi, kind1, n in _REG.findall(text):
        out |= {(kind, i) for i in range(int(lo), int(hi) + 1)} if kind else {(kind1, int(n))}
    return out


def _written(ins):
    return _regs(ins.split(",")[0]) if ins.startswith(("v_", "ds_read", "ds_bpermute", "global_load", "scratch_load",
                                                       "buffer_load")) else set()


def _read(ins):
    if ins.startswith(("ds_", "global_store", "scratch_store", "buffer_store")) or "mac" in ins.split()[0]:
        return _regs(ins)
    return _regs(ins.partition(",")[2])


def _block(ins):
    for i, (code, note) in enumerate(ins):
        spill = code.startswith("scratch_store") and "Spill" in note or code.startswith("v_accvgpr_write") and "Reuse" in note
        reload = code.startswith("scratch_load") and "Reload" in note or code.startswith("v_accvgpr_read") and "Reuse" in note
        if not (spill or reload):
            continue
        after = next((j for j in range(i + 1, len(ins)) if _EXEC.search(ins[j][0])), None)
        if after is None or not _RESTORE.match(ins[after][0]):
            continue
        if spill:
            formed = set()
            for code1, _ in reversed(ins[:i]):
                if _EXEC.search(code1):
                    break
                formed |= _written(code1)
            bad = not _read(code) <= formed
        else:
            bad = not any(_read(c) & _written(code) for c, _ in ins[i + 1:after])
        if bad:
            yield code


def misplaced_spills(listing):
    """[(kernel, instruction)] of an assembly listing."""
    out = []
    for m in _FUNC.finditer(listing):
        for block in _BLOCK.split(m.group(2)):
            ins = []
            for line in block.splitlines():
                code, _, note = line.partition(";")
                code = code.strip()
                if code and not code.startswith("."):
                    ins.append((code, note))
            out += [(m.group(1), code) for code in _block(ins)]
    return out
