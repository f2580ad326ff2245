"""The flash kernels whose waves share a block's keys: every barrier waits for the loads into LDS before it, as test_lds_waits.py asks of the
others."""
import os
import re
import subprocess

import pytest

import nvmai_amd.build as build
from test_lds_waits import LLVM, unguarded


@pytest.mark.skipif(not os.path.exists(LLVM + "llvm-objdump"), reason="no llvm-objdump")
def test_every_barrier_waits_for_the_loads_into_lds(tmp_path):
    library = tmp_path / "lib.so"
    os.symlink(build.LIB, library)
    subprocess.run([LLVM + "llvm-objdump", "--offloading", str(library)], check=True, stdout=subprocess.DEVNULL, cwd=tmp_path)
    seen = {}
    for path in sorted(tmp_path.glob("lib.so.*gfx950")):
        if b"flash_halves_kernel" not in path.read_bytes():
            continue
        text = subprocess.run([LLVM + "llvm-objdump", "-d", "--no-show-raw-insn", "--no-leading-addr", "--symbolize-operands", str(path)], check=True,
                              stdout=subprocess.PIPE, text=True).stdout
        for name, body in re.findall(r"^<(_Z\w+flash_halves_kernel\w+)>:\n(.*?)(?=^<_Z|\Z)", text, re.S | re.M):
            seen[name] = unguarded(body.splitlines())
    for kernel in ("window_flash_halves_kernel", "latent_flash_halves_kernel"):
        assert any(kernel in name for name in seen), kernel
    for name, (barriers, bad) in seen.items():
        assert barriers >= 4 and not bad, (name, bad)
