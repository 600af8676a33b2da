"""What the kernels rely on in the compiled library, read from its disassembly.

The direct-to-LDS requests are inline assembly, for which the compiler inserts none of the wait states that the
hardware asks for: one between a scalar write of M0 (the LDS address) and the load, five between a vector
instruction that writes a scalar register and a load that takes its address from it.

The blocks of dK / dV keep 64 MFMAs and what stands between them in one order: nothing moves between the two
halves of the register file there (one wavefront per SIMD, nothing hides such moves and the waits they bring)."""
import os
import re
import shutil
import subprocess

import pytest

from intra_amd import build


def llvm_tool(name):
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(build.hipcc_path())))
    path = os.path.join(rocm, "llvm", "bin", name)
    return path if os.path.exists(path) else shutil.which(name)


@pytest.fixture(scope="module")
def code_object(tmp_path_factory):
    """The gfx950 code of libintra_hip.so"""
    try:
        tools = [llvm_tool(t) for t in ("llvm-objcopy", "clang-offload-bundler", "llvm-objdump")]
    except RuntimeError:
        tools = [None]
    if None in tools:
        pytest.skip("needs ROCm's llvm tools")
    if not os.path.exists(build.LIB):
        build.build()
    tmp = tmp_path_factory.mktemp("code")
    fat, code = str(tmp / "fat.bin"), str(tmp / "gfx950.co")
    subprocess.run([tools[0], "-O", "binary", "--only-section=.hip_fatbin", build.LIB, fat], check=True)
    subprocess.run([tools[1], "--type=o", f"--input={fat}", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950",
                    f"--output={code}", "--unbundle"], check=True)
    return code


def scalar_registers(operand):
    """Numbers of the scalar registers that an operand such as s7 or s[2:3] names"""
    m = re.match(r"s\[(\d+):(\d+)\]$", operand)
    if m:
        return set(range(int(m[1]), int(m[2]) + 1))
    m = re.match(r"s(\d+)$", operand)
    return {int(m[1])} if m else set()


def request_faults(lines):
    """(loads to LDS, those of them without their wait states) in a disassembly, read in program order"""
    n, faults, since_m0, since_vector = 0, [], 99, {}
    for line in lines:
        if line.endswith(">:\n"):  # next kernel
            since_m0, since_vector = 99, {}
        if not line.startswith("\t"):
            continue
        op, *rest = line.split("//")[0].split()
        args = " ".join(rest).split(", ") if rest else []
        if op.startswith("global_load_lds_"):
            n += 1
            states = [since_vector.get(r, 99) for r in scalar_registers(args[1].split()[0])]
            if since_m0 < 1 or min(states, default=99) < 5:
                faults.append(line.strip())
        passed = 1 + (int(args[0], 0) if op == "s_nop" else 0)
        since_m0 = since_m0 + passed
        since_vector = {r: d + passed for r, d in since_vector.items() if d < 5}
        if args and args[0] == "m0":
            since_m0 = 0
        if op.startswith("v_"):
            for a in args[:2]:  # (a carry or a comparison's result is the second operand; reading more only errs on the safe side)
                since_vector.update((r, 0) for r in scalar_registers(a))
    return n, faults


def test_the_check_itself():
    load = "\tglobal_load_lds_dwordx4 v1, s[2:3] // 0: 0\n"
    assert request_faults(["\ts_mov_b32 m0, s9\n", load])[1] != []
    assert request_faults(["\ts_mov_b32 m0, s9\n", "\ts_nop 0\n", load]) == (1, [])
    assert request_faults(["\tv_readlane_b32 s3, v9, 1\n", "\ts_mov_b32 m0, s9\n", "\ts_nop 2\n", load])[1] != []
    assert request_faults(["\tv_readlane_b32 s3, v9, 1\n", "\ts_mov_b32 m0, s9\n", "\ts_nop 3\n", load])[1] == []


def disassembly(code_object):
    with subprocess.Popen([llvm_tool("llvm-objdump"), "-d", "--no-show-raw-insn", code_object], text=True,
                          stdout=subprocess.PIPE) as dump:
        yield from dump.stdout
    assert dump.returncode == 0


def test_every_request_has_its_wait_states(code_object):
    n, faults = request_faults(disassembly(code_object))
    assert n > 1000
    assert not faults, (len(faults), faults[:4])


def blocks(lines, kernel, mfmas):
    """The instructions from the first to the last of the `mfmas` MFMAs in front of a branch, where there are as
    many without a branch between them, in the kernels whose name contains `kernel`"""
    inside, run = False, []
    for line in lines:
        if line.endswith(">:\n"):
            inside, run = kernel in line, []
        elif inside and line.startswith("\t"):
            op = line.split()[0]
            if not op.startswith(("s_cbranch", "s_branch", "s_endpgm")):
                run.append(op)
                continue
            at = [i for i, o in enumerate(run) if o.startswith("v_mfma")]
            if len(at) >= mfmas:
                yield run[at[-mfmas]:at[-1] + 1]
            run = []


def test_no_moves_between_register_halves_in_the_blocks_of_dk_and_dv(code_object):
    moves = [sum(op.startswith("v_accvgpr") for op in block) for block in blocks(disassembly(code_object), "intra_bwd_kernel", 64)]
    assert len(moves) >= 30 and not any(moves), moves


def test_ordinary_backward_kernels_keep_their_scalars(code_object):
    """What only tensors beyond 32-bit offsets and single tiles need stays out of the other kernels' registers: more
    scalars than this move to lanes of vector registers and back inside the tile loop."""
    notes = subprocess.run([llvm_tool("llvm-readelf"), "--notes", code_object], check=True, capture_output=True, text=True).stdout
    kernels = {}
    for entry in notes.split("- .agpr_count:")[1:]:
        fields = dict(re.findall(r"\.(name|sgpr_spill_count|vgpr_spill_count):\s+(\S+)", entry))
        if "intra_bwd_kernel" in fields["name"]:
            kernels[fields["name"]] = (int(fields["sgpr_spill_count"]), int(fields["vgpr_spill_count"]))
    near = {name: n for name, n in kernels.items() if "Lb0EEEv" in name}
    assert len(near) >= 30 and len(kernels) == 2 * len(near), (len(near), len(kernels))
    assert all(vector == 0 and scalar <= 40 for scalar, vector in near.values()), near
