"""No compiled kernel copies vector registers ahead of the execution mask.

Behind a divergent branch the join restores the mask of active lanes
(s_or_b64 exec, exec, ...).  Where scalar registers are spilled at such a join
and the allocator also moves a vector register there, clang has put the move
before the restore: the lanes that skipped the branch keep what the target held
(so O3's recrossing parents lost dt/2 on all lanes but one in sixteen).  The
disassembly of the library built here is read for joins that begin with moves
between vector registers."""
import os
import re
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "caracal_amd", "libcaracal_amd.so")
OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
MOVE = re.compile(r"v_accvgpr_(write|read|mov)|v_mov_b(32|64)\w* (v\S+), (v|a)")
SCALAR = re.compile(r"v_writelane|v_readlane|s_nop|s_mov|s_waitcnt")


def bad_joins(lines):
    """(kernel, moves) of every branch target that moves vector registers and
    then restores the mask, with nothing but scalar spills between."""
    kernel, moves, out = "", None, []
    for line in lines:
        if line.startswith("<"):
            if line.startswith("<_Z"):
                kernel, moves = line[1:line.index(">")], None
            else:
                moves = []
            continue
        if moves is None:
            continue
        op = line.strip()
        if MOVE.match(op):
            moves.append(op.split("//")[0].strip())
        elif op.startswith("s_or_b64 exec, exec"):
            if moves:
                out.append((kernel, moves))
            moves = None
        elif not SCALAR.match(op):
            moves = None
    return out


def test_a_join_that_moves_first_is_seen():
    good = ["<_Zk>:", "\tv_mov_b32_e32 v1, v2", "<L1>:", "\ts_or_b64 exec, exec, s[0:1]", "\tv_accvgpr_write_b32 a1, v1",
            "<L2>:", "\tv_mov_b32_e32 v1, v2", "\tv_add_f64 v[0:1], v[0:1], v[2:3]", "\ts_or_b64 exec, exec, s[2:3]"]
    assert bad_joins(good) == []
    bad = ["<_Zk>:", "<L1>:", "\tv_writelane_b32 v255, s20, 49", "\tv_accvgpr_write_b32 a20, v96   // 00: 00",
           "\tv_writelane_b32 v255, s21, 50", "\ts_or_b64 exec, exec, s[0:1]"]
    assert bad_joins(bad) == [("_Zk", ["v_accvgpr_write_b32 a20, v96"])]


@pytest.mark.skipif(not os.path.exists(LIB) or not os.path.exists(OBJDUMP), reason="library or llvm-objdump not there")
def test_no_join_of_the_library_moves_before_the_mask(tmp_path):
    os.symlink(LIB, tmp_path / "lib.so")       # the code objects are written beside it
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    objects = sorted(f for f in os.listdir(tmp_path) if f.endswith("gfx950"))
    assert objects

    def scan(name):
        p = subprocess.Popen([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", "--symbolize-operands", name],
                             cwd=tmp_path, stdout=subprocess.PIPE, text=True)
        found = bad_joins(p.stdout)
        assert p.wait() == 0
        return found

    with ThreadPoolExecutor(4) as pool:
        found = [x for part in pool.map(scan, objects) for x in part]
    assert not found, found
