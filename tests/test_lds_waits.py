"""The kernels that load tiles straight into LDS and drain them at every barrier: a workgroup's barrier does not wait for such loads, so
each one needs a wait for all of the wave's own in its own block of the built code, also on the way back to the loop's head."""
import os
import re
import subprocess

import pytest

import nvmai_amd.build as build

LLVM = "/opt/rocm/llvm/bin/"
KERNELS = ("window_flash_kernel", "latent_flash_kernel")


def unguarded(lines):
    """The barriers, by their place, without a vmcnt(0) between them and the last load into LDS, branch or branch target."""
    guarded, bad, barriers = False, [], 0
    for n, line in enumerate(lines):
        if re.match(r"\s*(<L\d+>:|s_c?branch|buffer_load_\S+ .*\blds\b)", line):
            guarded = False
        elif re.match(r"\s*s_waitcnt\b.*\bvmcnt\(0\)", line):
            guarded = True
        elif re.match(r"\s*s_barrier\b", line):
            barriers += 1
            if not guarded:
                bad.append(n)
    return barriers, bad


def test_the_check_sees_a_wait_only_on_the_way_in():
    loop = ["buffer_load_dwordx4 v0, s[0:3], 0 offen lds", "s_waitcnt vmcnt(0)", "<L0>:", "s_barrier", "s_branch L0"]
    assert unguarded(loop) == (1, [3])
    assert unguarded(loop[:3] + ["s_waitcnt vmcnt(0) lgkmcnt(0)"] + loop[3:]) == (1, [])


@pytest.mark.skipif(not os.path.exists(LLVM + "llvm-objdump"), reason="no llvm-objdump")
def test_every_barrier_of_the_flash_kernels_waits_for_the_loads_into_lds(tmp_path):
    library = tmp_path / "lib.so"
    os.symlink(build.LIB, library)
    subprocess.run([LLVM + "llvm-objdump", "--offloading", str(library)], check=True, stdout=subprocess.DEVNULL, cwd=tmp_path)
    seen = {}
    for path in sorted(tmp_path.glob("lib.so.*gfx950")):
        if not any(k.encode() in path.read_bytes() for k in KERNELS):
            continue
        text = subprocess.run([LLVM + "llvm-objdump", "-d", "--no-show-raw-insn", "--no-leading-addr", "--symbolize-operands", str(path)], check=True,
                              stdout=subprocess.PIPE, text=True).stdout
        for name, body in re.findall(r"^<(_Z\w+)>:\n(.*?)(?=^<_Z|\Z)", text, re.S | re.M):
            if any(k in name for k in KERNELS):
                seen[name] = unguarded(body.splitlines())
    assert len(seen) == 10 + 9                       # the sizes of the windowed kernel, and of the latent one
    for name, (barriers, bad) in seen.items():
        assert barriers >= 2 and not bad, (name, bad)
