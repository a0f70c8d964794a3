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
def functions(tmp_path_factory):
    """name -> [(address, instruction, branch target or None)] of every device function."""
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    where = tmp_path_factory.mktemp("code")
    lib = shutil.copy(_lib.LIB_PATH, where)
    subprocess.run([OBJDUMP, "--offloading", lib], cwd=where, check=True, capture_output=True)
    found = {}
    for name in sorted(os.listdir(where)):
        if "gfx950" not in name:
            continue
        text = subprocess.run([OBJDUMP, "-d", os.path.join(where, name)], check=True, capture_output=True, text=True).stdout
        for part in re.split(r"^(?=[0-9a-f]+ <)", text, flags=re.M)[1:]:
            start, symbol = re.match(r"([0-9a-f]+) <([^>]*)>:", part).groups()
            code = found.setdefault(symbol, [])
            for m in re.finditer(r"^\s+(\S.*?)\s*// ([0-9A-F]+):[0-9A-F ]*(?:<[^>+]*\+0x([0-9a-f]+)>)?$", part, flags=re.M):
                target = int(start, 16) + int(m.group(3), 16) if m.group(3) else None
                code.append((int(m.group(2), 16), m.group(1), target))
    return found


@pytest.fixture(scope="module")
def gemm_task(functions):
    """The instructions of tiled_gemm_task in address order."""
    (code,) = [v for k, v in functions.items() if "tiled_gemm_task" in k]
    return [ins for _, ins, _ in code]


def test_streaming_tasks_lie_on_4096_byte_boundaries(functions):
    """The streaming tasks' times depend on where they lie among each other by a percent or two (build.py)."""
    tasks = [(name, code[0][0]) for name, code in functions.items() if re.search(r"fmoe\d+(gateup|gateup_early|down)_taskI", name)]
    assert len(tasks) == 6 + 4 + 6
    assert not [t for t in tasks if t[1] % 4096]


def test_float32_sweeps_lie_on_64_byte_boundaries(functions):
    """The float32 streaming tasks lose about a percent to where their k-loops happen to lie
    (build.py), so those loops are aligned: every backward branch over the 256 matrix instructions of a round."""
    loops = 0
    for name, code in functions.items():
        if not re.search(r"(gateup|down)_task\w*3F32ELi4", name):
            continue
        for at, ins, target in code:
            if ins.startswith("s_cbranch") and target is not None and target < at:
                if sum(1 for a, i, _ in code if target <= a < at and i.startswith("v_mfma")) >= 256:
                    loops += 1
                    assert target % 64 == 0, "%s: a loop at 0x%x" % (name, target)
    assert loops >= 6  # packed weights and row-major ones, read once or shared


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


def _registers(text):
    found = set()
    for bank, lo, hi, bank1, one in re.findall(r"\b([va])\[(\d+):(\d+)\]|\b([va])(\d+)\b", text):
        found |= {(bank, r) for r in range(int(lo), int(hi) + 1)} if bank else {(bank1, int(one))}
    return found


def _check_accumulators(functions, tasks):
    checked = 0
    for name, code in functions.items():
        if not re.search(tasks, name):
            continue
        ins = [i for _, i, _ in code]
        for at, op in enumerate(ins):
            if not op.startswith("v_mfma"):
                continue
            checked += 1
            result, waited = _registers(op.split(None, 1)[1].split(", ")[0]), 0
            for later in ins[at + 1:at + 40]:
                if waited >= 16 or later.startswith(("s_branch", "s_cbranch", "s_setpc")):
                    break
                if later.startswith("s_nop"):
                    waited += int(later.split()[1]) + 1
                elif later.startswith("v_mfma"):
                    a, b = later.split(None, 1)[1].split(", ")[1:3]
                    assert not result & (_registers(a) | _registers(b)), "%s: %s | %s" % (name, op, later)
                    waited += 4
                else:
                    if later.startswith(("v_", "ds_", "global_", "buffer_", "scratch_")) and " " in later:
                        assert not result & _registers(later.split(None, 1)[1]), "%s: %s | %s" % (name, op, later)
                    waited += 1
    return checked


def test_accumulators_are_left_alone_until_they_are_written(functions):
    """The tiled kernel's matrix instructions stand in assembly, so the compiler does not know that their
    results take a while: wherever it copies an accumulator between registers (it may where two ways
    through the code meet) it would read the old value. So nothing but matrix instructions may touch a
    result for 16 wait states (a 16x16x32 product takes four passes of four cycles, and the wait the
    hardware does not make by itself is less), along the straight line behind it."""
    assert _check_accumulators(functions, "tiled_gemm_task|tiled_odd_down_task|tiled_ragged_(gate_up|down)_task") > 10000


def test_router_chains_are_left_alone_until_they_are_written(functions):
    """The same for the router's chains, which stand in assembly too: 16x16x4 float products of eight passes, ten wait
    states."""
    # 16 groups of 4 and of 2 instructions a stage
    assert _check_accumulators(functions, "tiled_router_task") == 16 * 4 + 16 * 2


def test_every_look_at_the_posts_reads_them_again(functions):
    """wait_posts polls with a load that is not atomic: it has to stand inside the loop around the wait's s_sleep 24."""
    loops = 0
    for name, code in functions.items():
        if "moe_split_kernel" not in name:
            continue
        for at in [a for a, ins, _ in code if ins == "s_sleep 24"]:
            back = [(a - target, target, a) for a, ins, target in code
                    if ins.startswith(("s_cbranch", "s_branch")) and target is not None and target <= at < a]
            assert back, "%s: no loop around 0x%x" % (name, at)
            _, first, last = min(back)
            assert any(first <= a < last and ins.startswith("buffer_load_dwordx4") and "sc1" in ins for a, ins, _ in code)
            loops += 1
    assert loops == 3 * 6  # routing, gate/up and down, in every instantiation


def test_a_kernel_waits_for_no_more_lines_of_its_arguments_than_params_has(functions):
    """Arguments are fetched anew for every launch, 64 bytes at a time. Params fills five such lines; gridDim and blockDim lie
    behind it, and a kernel that asks for a sixth line starts later (1 to 3 us with small batches)."""
    kernels = 0
    for name, code in functions.items():
        if re.search(r"moe_(split|stream|tiled|tiled_f32)_kernelI", name):
            loads = [re.match(r"s_load_dword(x\d+)? \S+, s\[\d+:\d+\], 0x([0-9a-f]+)", ins) for _, ins, _ in code]
            last = max(int(m.group(2), 16) + 4 * int((m.group(1) or "x1")[1:]) for m in loads if m)
            assert 256 < last <= 320, "%s reads %d bytes of arguments" % (name, last)
            kernels += 1
    assert kernels == 6 + 2 + 2 + 6
