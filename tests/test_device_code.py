"""The device code in the built libraries, read as assembly."""
import os
import re
import shutil
import subprocess

import pytest

from memfabric_hybrid_amd import native

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
WIDE_STORE = re.compile(r"(global|flat|buffer)_store_dwordx[34] ")
VECTOR = re.compile(r"v(?:\[(\d+):(\d+)\]|(\d+))(?: |$)")


def registers(operand):
    """First and last vector register that an operand names, or None."""
    m = VECTOR.match(operand.strip())
    return None if m is None else (int(m[1] or m[3]), int(m[2] or m[3]))


def overwritten(code, states):
    """Stores of more than 64 bits whose data a vector instruction writes with fewer than `states` wait states in between."""
    found = []
    for i, line in enumerate(code):
        m = WIDE_STORE.match(line)
        if m is None:
            continue
        operands = line[m.end():].split(",")
        low, high = registers(operands[0 if m[1] == "buffer" else 1])
        passed = 0
        for after in code[i + 1:]:
            if passed >= states or after.startswith(("s_branch", "s_endpgm", "s_setpc")):
                break
            name, _, rest = after.partition(" ")
            written = registers(rest.split(",")[0]) if name.startswith("v_") else None
            if written is not None and written[0] <= high and low <= written[1]:
                found.append((line, after))
                break
            passed += int(rest, 0) + 1 if name == "s_nop" else 1
    return found


def test_what_counts_as_overwritten():
    store = "global_store_dwordx4 v[20:21], v[2:5], off sc0 sc1 nt"
    write = "v_lshl_add_u64 v[2:3], v[22:23], 0, s[46:47]"
    assert overwritten([store, write], 2) == [(store, write)]
    assert overwritten([store, "s_nop 0", write], 2) == [(store, write)]
    assert overwritten([store, "s_nop 1", write], 2) == []
    assert overwritten([store, "s_mov_b32 s0, 0", "s_mov_b32 s1, 0", write], 2) == []
    assert overwritten([store, "s_branch 100", write], 2) == []
    assert overwritten([store, "v_mov_b32_e32 v20, 0", "v_mov_b32_e32 v6, 0"], 2) == []      # the address may be written at once
    held = "buffer_store_dwordx4 v[4:7], v1, s[0:3], 0 offen"
    assert overwritten([held, "v_mov_b32_e32 v7, 0"], 2) == [(held, "v_mov_b32_e32 v7, 0")]
    assert overwritten([held, "v_mov_b32_e32 v1, 0"], 2) == []


@pytest.mark.parametrize("library", ["libmf_hip_dataplane.so", "libmf_hybm_copy_extend.so", "libmf_hip_yardstick.so"])
def test_data_of_wide_stores_stays_until_it_is_read(library, tmp_path):
    """A store of more than 64 bits reads its data late: a vector instruction may write those registers only two wait states later.  The
    hardware does not see to it, and the compiler does for its own stores only, not for those in inline assembly."""
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    built = os.path.join(os.path.dirname(native.__file__), "lib", library)
    copy = shutil.copy(built, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", copy], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    stores = 0
    found = []
    for name in sorted(os.listdir(tmp_path)):
        if "gfx950" not in name:
            continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", name], cwd=tmp_path, check=True, stdout=subprocess.PIPE, text=True).stdout
        code = [line.split("//")[0].strip() for line in text.splitlines() if line.startswith("\t")]
        stores += sum(WIDE_STORE.match(line) is not None for line in code)
        found += overwritten(code, 2)
    assert stores > 0, "no device code was found"
    assert not found, found[:4]
