"""The machine code of the built kernels.

Where a vector register is spilled just before a lane mask is widened again, the
lanes outside the mask lose its value; the compiler has done that to registers
that every lane needs (an LDS address, by the exit of a loop over a site's
mouths), so the built code is looked over for it."""
import os
import re
import shutil
import subprocess

import pytest

from casim_amd import abi

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
WRITES = re.compile(r"v_(?!cmp|readlane|readfirstlane)|ds_read|ds_bpermute|(global|flat|scratch|buffer)_load")


def registers(text):
    out = {int(r) for r in re.findall(r"\bv(\d+)\b", text)}
    for a, b in re.findall(r"\bv\[(\d+):(\d+)\]", text):
        out |= set(range(int(a), int(b) + 1))
    return out


def written(ins):
    op, _, rest = ins.partition(" ")
    return registers(rest.split(",")[0]) if WRITES.match(op) else set()


def slot(ins):
    """The scratch bytes of a spill or reload: its first offset."""
    return re.search(r"offset:(\d+)|$", ins).group(1) or "0"


def lost_spills(code, before=None):
    """Spill stores right before an exec mask is restored, of registers that
    nothing has written since the mask was saved, into slots that no other
    store fills and a load outside the mask reads.  before: the instructions
    that may run before each one (by default the one above it)."""
    before = before or [[i - 1] if i else [] for i in range(len(code))]
    stores, loads = {}, {}
    for i, ins in enumerate(code):
        if ins.startswith("scratch_store"):
            stores.setdefault(slot(ins), []).append(i)
        elif ins.startswith("scratch_load"):
            loads.setdefault(slot(ins), []).append(i)
    bad = []
    for i, ins in enumerate(code):
        m = re.match(r"s_or_b64 exec, exec, (s\[\d+:\d+\])", ins)
        if not m:
            continue
        k, late = i - 1, []
        while k >= 0 and not code[k].startswith(("s_branch", "s_cbranch", "s_endpgm")) and \
                not re.search(r"\bexec\b|saveexec", code[k].partition(",")[0]):
            if code[k].startswith("scratch_store") and stores[slot(code[k])] == [k]:
                late.append(k)
            k -= 1
        if not late:
            continue
        # what runs under the mask: everything from its save to here
        save = re.compile(r"s_\w*saveexec_b64 " + re.escape(m.group(1)) + ",")
        masked, todo = set(), list(before[i])
        while todo:
            n = todo.pop()
            if n not in masked and not save.match(code[n]):
                masked.add(n)
                todo += before[n]
        since = set().union(*(written(code[n]) for n in masked))
        for k in reversed(late):
            if registers(code[k]) - since and any(n not in masked for n in loads.get(slot(code[k]), [])):
                bad.append(code[k])
    return bad


def kernels(tmp_path):
    """(name, instructions, what may run before each) of every kernel in the
    built library that spills vector registers."""
    lib = shutil.copy(abi.LIB_PATH, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True, cwd=tmp_path)
    for f in sorted(os.listdir(tmp_path)):
        if "gfx950" not in f:
            continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(tmp_path / f)], check=True, capture_output=True,
                              text=True).stdout
        for part in re.split(r"\n[0-9a-f]+ <", text)[1:]:
            name, _, body = part.partition(">:\n")
            if "scratch_store" not in body:
                continue
            lines = [line.split("//") for line in body.split("\n") if line.startswith("\t") and "//" in line]
            code = [a.strip() for a, _ in lines]
            at = {int(b.split(":")[0], 16): i for i, (_, b) in enumerate(lines)}
            start = min(at)
            before = [[] for _ in code]
            for i, ins in enumerate(code):
                target = re.search(r"\+0x([0-9a-f]+)>", lines[i][1])
                if ins.startswith(("s_branch", "s_cbranch")):
                    before[at[start + int(target.group(1), 16)] if target else 0].append(i)
                if not ins.startswith(("s_branch", "s_endpgm")) and i + 1 < len(code):
                    before[i + 1].append(i)
            yield name, code, before


def test_lost_spills_are_found():
    loop = ["v_mov_b32_e32 v20, v3", "s_and_saveexec_b64 s[0:1], vcc", "s_cbranch_execz 12", "v_add_u32_e32 v7, 64, v7",
            "s_cbranch_execnz 65000"]
    spill, restore = ["scratch_store_dwordx2 off, v[20:21], off offset:148"], ["s_or_b64 exec, exec, s[0:1]"]
    load = ["scratch_load_dwordx2 v[2:3], off, off offset:148"]
    assert lost_spills(loop + spill + restore + load) == spill
    assert lost_spills(loop + restore + spill + load) == []  # after the restore every lane stores
    assert lost_spills(loop + ["v_mov_b64_e32 v[20:21], v[4:5]"] + spill + restore + load) == []  # these lanes' own value
    assert lost_spills(loop + spill + load + restore) == []  # back in the register before the restore
    assert lost_spills(spill + loop + spill + restore + load) == []  # the other lanes' value is there


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler")
def test_no_spill_is_lost(tmp_path):
    names = []
    for name, code, before in kernels(tmp_path):
        names.append(name)
        assert lost_spills(code, before) == [], name
    assert names
