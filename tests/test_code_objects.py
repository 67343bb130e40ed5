"""The machine code of the kernels that hold a site's state over many steps.

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
ENDS = re.compile(r"s_cbranch|s_branch|s_endpgm|s_setpc")


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


def lost_spills(code):
    """Spill stores right before an exec mask is restored, of registers that
    nothing has written since the mask was saved, into slots that no other
    store fills and a load outside the mask reads."""
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
        save = j = i - 1
        while save > 0 and not re.match(r"s_\w*saveexec_b64 " + re.escape(m.group(1)) + r",", code[save]):
            save -= 1
        while j > save and not ENDS.match(code[j]):
            k, j = j, j - 1
            if not code[k].startswith("scratch_store") or stores[slot(code[k])] != [k]:
                continue
            if not any(not save < n < i for n in loads.get(slot(code[k]), [])):
                continue
            if registers(code[k]) - set().union(*(written(c) for c in code[save:k])):
                bad.insert(0, code[k])
    return bad


def kernels(tmp_path):
    """(name, instructions) of every kernel in the built library."""
    lib = shutil.copy(abi.LIB_PATH, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True, cwd=tmp_path)
    for f in sorted(os.listdir(tmp_path)):
        if "gfx950" not in f:
            continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(tmp_path / f)], check=True, capture_output=True,
                              text=True).stdout
        for part in re.split(r"\n[0-9a-f]+ <", text)[1:]:
            name, _, body = part.partition(">:\n")
            yield name, [line.split("//")[0].strip() for line in body.split("\n") if line.startswith("\t")]


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
def test_no_spill_is_lost_in_the_step_kernels(tmp_path):
    names = []
    for name, code in kernels(tmp_path):
        if re.search(r"k_resident|k_site2d", name):
            names.append(name)
            assert lost_spills(code) == [], name
    assert len(names) >= 20
