"""Build-time guards on the gfx950 device code.

Compiles every .hip source of this directory to device assembly (with the per-file flags the
Makefile gives it) and fails if
  * a scalar instruction appears that is not one of those known to leave memory as it is (scalar loads,
    arithmetic, branches, waits): the device code must not write through the scalar data cache;
  * LDS stores of one block through one address register go out in another order than ascending
    (lds_stores_out_of_order).  The step loops store a lane's cell at the lane's own column, so the
    lanes store to one column a step apart and the last lane's store has to come last; the compiler
    sees one lane, whose addresses all differ, and may reorder its stores.  A column then keeps another
    lane's row: FP64 results were wrong at columns 4 mod 8 from a build that had swapped two steps.
Run by __graft_entry__.build() in the build container only.
"""
import os
import re
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
# Loads; operations on registers, whose names end in their type; program control.
HARMLESS = re.compile(r"s_(?:(?:buffer_)?load_dword(?:x\d+)?|\w+_[biuf](?:16|32|64)|c?branch\w*|waitcnt\w*|nop|sleep|"
                      r"barrier|endpgm|setprio)\Z")
SCALAR = re.compile(r"^\s*(s_\w+)", re.M)
FLAGS = ["-O3", "-std=c++17", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang",
         "-packed-fp32-ops", "--cuda-device-only", "-S"]
# Per-file flags of the Makefile's object rules.
FILE_FLAGS = {"pairhmm_fwd.hip": ["-mllvm", "-enable-post-misched=false"]}
WIDE_LDS_STORE = re.compile(r"^ds_(write|store)_b(96|128)\b")
LDS_STORE = re.compile(r"^ds_(?:write|store)(2)?(st64)?_b(8|16|32|64|96|128)\s+(v\d+)")
ORDER_WINDOW = 256  # bytes: 16 steps of up to 16 bytes; planes lie further apart


def _vgprs(operand):
    out = set()
    for m in re.finditer(r"v\[(\d+):(\d+)\]", operand):
        out.update(range(int(m.group(1)), int(m.group(2)) + 1))
    out.update(int(m.group(1)) for m in re.finditer(r"\bv(\d+)\b", operand))
    return out


def _lds_store(line):
    """(address register, byte offsets) of an LDS store, or None."""
    m = LDS_STORE.match(line)
    if not m:
        return None
    if not m.group(1):
        off = re.search(r"offset:(\d+)", line)
        return m.group(4), [int(off.group(1)) if off else 0]
    unit = int(m.group(3)) // 8 * (64 if m.group(2) else 1)
    offs = [re.search(rf"offset{k}:(\d+)", line) for k in (0, 1)]
    return m.group(4), [int(o.group(1)) * unit if o else 0 for o in offs]


def lds_stores_out_of_order(asm):
    """(function, address register, offset, later lower offset): within a basic block, an LDS store through the
    same unchanged address register up to ORDER_WINDOW bytes below one before it."""
    hits, name, seen = [], None, {}
    for line in asm.split("\n"):
        label = re.match(r"^([\w$.]+):", line)
        if label:
            if not label.group(1).startswith(".L"):
                name = label.group(1)
            seen = {}
            continue
        if not line.startswith("\t") or line.startswith("\t."):
            continue
        ins = line.split(";")[0].strip()
        if ins.startswith(("s_cbranch", "s_branch")):
            seen = {}
            continue
        store = _lds_store(ins)
        if store:
            reg, offs = store
            before = seen.setdefault(reg, [])
            for o in offs:
                above = [b for b in before if 0 < b - o <= ORDER_WINDOW]
                if above:
                    hits.append((name, reg, above[0], o))
                before.append(o)
        elif re.match(r"^(v_|ds_|global_load|buffer_load|scratch_load|flat_load)", ins):
            written = _vgprs(ins.split(None, 1)[1].split(",")[0]) if " " in ins else set()
            for reg in [r for r in seen if int(r[1:]) in written]:
                del seen[reg]
    return hits


def wide_lds_store_overwrites(asm):
    """(store, overwriting instruction) pairs where a VALU op within two instructions after a
    ds_write_b96/b128 writes one of the store's data VGPRs.  Not an error: builds with 252 such pairs in the FP64
    forward, 32 in the adjoint and 2 in the PD kernel give the bits of builds without any."""
    ins = [l.split(";")[0].strip() for l in asm.split("\n")
           if l.startswith("\t") and not l.startswith("\t.")]
    hits = []
    for k, line in enumerate(ins):
        if not WIDE_LDS_STORE.match(line):
            continue
        data = set()
        for operand in line.split(None, 1)[1].split(",")[1:]:
            data |= _vgprs(operand)
        for nxt in ins[k + 1:k + 3]:
            if nxt.startswith("v_") and _vgprs(nxt.split(",")[0]) & data:
                hits.append((line, nxt))
    return hits


def unknown_scalar_ops(asm):
    """Scalar instructions that are not known to leave memory as it is."""
    return sorted({op for op in SCALAR.findall(asm) if not HARMLESS.match(op)})


def main() -> int:
    bad = []
    for name in sorted(os.listdir(HERE)):
        if not name.endswith(".hip"):
            continue
        with tempfile.TemporaryDirectory() as td:
            out = os.path.join(td, name + ".s")
            subprocess.run(["/opt/rocm/bin/hipcc", *FLAGS, *FILE_FLAGS.get(name, []), "-o", out,
                            os.path.join(HERE, name)], check=True, stderr=subprocess.DEVNULL)
            asm = open(out).read()
        unknown = unknown_scalar_ops(asm)
        if unknown:
            bad.append(f"{name}: scalar instructions that may write memory: {unknown}")
        swapped = lds_stores_out_of_order(asm)
        if swapped:
            bad.append(f"{name}: {len(swapped)} LDS stores out of order, e.g. {swapped[0]}")
    for msg in bad:
        print(f"check_isa: {msg}", file=sys.stderr)
    return 1 if bad else 0


if __name__ == "__main__":
    sys.exit(main())
