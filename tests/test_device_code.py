"""What the compiled tiled kernel must keep to between its memory operations, read off the
disassembly of the library built from this tree (no GPU needed)."""
import os
import re
import shutil
import subprocess

import pytest

from flash_distributed_moe_amd import _lib

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.fixture(scope="module")
def gemm_task(tmp_path_factory):
    """The instructions of tiled_gemm_task in address order."""
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    where = tmp_path_factory.mktemp("code")
    lib = shutil.copy(_lib.LIB_PATH, where)
    subprocess.run([OBJDUMP, "--offloading", lib], cwd=where, check=True, capture_output=True)
    for name in sorted(os.listdir(where)):
        if "gfx950" not in name:
            continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", os.path.join(where, name)], check=True,
                              capture_output=True, text=True).stdout
        for part in re.split(r"^[0-9a-f]+ <", text, flags=re.M)[1:]:
            if "tiled_gemm_task" in part.split(">:", 1)[0]:
                lines = (line.split("//")[0].strip() for line in part.split("\n")[1:])
                return [line for line in lines if line]
    raise AssertionError("tiled_gemm_task is not in the library")


def test_a_task_is_signalled_behind_a_full_wait_for_its_stores(gemm_task):
    """A GEMM task's completion counter is raised by the workgroup's next task, once the stores of
    the finished one have reached memory. Loads and stores are not assumed to complete in order
    with each other, so a wait that leaves younger loads in flight says nothing about older stores:
    in front of every signal (an add whose result nobody reads) the next task must have waited for
    everything, as its first wait; only waits of its k-loop may leave loads in flight behind that."""
    signals = [i for i, ins in enumerate(gemm_task)
               if ins.startswith("global_atomic_add") and "sc0" not in ins.split()]
    # both pipelines: JT 2..10 through LDS (two ways into the first hand-over at least), 2..8 direct, up and down
    assert len(signals) >= 2 * (9 + 7)
    for at in signals:
        partial = None   # a wait that leaves loads in flight, not (yet) seen to stand inside the k-loop
        for ins in reversed(gemm_task[:at]):
            op = ins.split()[0]
            assert not op.startswith("global_store"), "no wait for stores in front of instruction %d" % at
            if op.startswith("v_mfma"):
                partial = None
            wait = re.search(r"vmcnt\((\d+)\)", ins) if op == "s_waitcnt" else None
            start = op in ("s_branch", "s_setpc_b64")  # of this piece of the code
            if wait or start or op.startswith("global_load"):
                assert partial is None, "instruction %d is signalled behind `%s`" % (at, partial)
            if start or (wait and wait.group(1) == "0"):
                break
            if wait:
                partial = ins
        else:
            raise AssertionError("no wait in front of instruction %d" % at)
