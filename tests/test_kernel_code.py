"""What the compiled kernels must not contain, read from the disassembly of the built library (no GPU)."""
import os
import re
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "tiny-dpcpp-nn_amd", "lib", "libtnn_hip.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler")
def test_no_wide_buffer_store_takes_its_offset_from_a_scalar_register(tmp_path):
    """The compiler lets the instruction behind such a store overwrite its data, which the processor is still reading: rows of width-128 activations held, now and
    then, what the next instruction wrote (Tile::store_staged_at)."""
    os.symlink(LIB, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    objects = sorted(p for p in os.listdir(tmp_path) if p.endswith("gfx950"))
    store = re.compile(r"\bbuffer_store_dwordx[34] [^,]*, [^,]*, s\[[0-9:]*\], (\S+)")

    def offsets(name):
        dump = subprocess.Popen([OBJDUMP, "-d", "--no-show-raw-insn", name], cwd=tmp_path, stdout=subprocess.PIPE, text=True)
        found = [m.group(1) for line in dump.stdout if "buffer_store_dwordx" in line for m in [store.search(line)] if m]
        assert dump.wait() == 0
        return found

    with ThreadPoolExecutor(8) as pool:
        found = [o for part in pool.map(offsets, objects) for o in part]
    assert len(objects) >= 15 and len(found) > 1000
    assert not [o for o in found if re.match(r"s\d|m0|ttmp|vcc", o)]
