"""No verify kernel of the built library spills a vector register: a spilled one
shares the vector-memory counter with the state's loads and is memory traffic of
its own (kernels of K = 256 held to three waves took 1.4 to 2.3 times as long).
Read from the metadata the compiler writes beside each kernel."""

import os
import re
import shutil
import subprocess

import pytest

from gdn_recoverssm_ascend._build import LIB_PATH, hipcc


def _llvm(tool):
    root = os.path.dirname(os.path.dirname(os.path.realpath(hipcc())))
    for path in (os.path.join(root, "lib", "llvm", "bin", tool), os.path.join(root, "llvm", "bin", tool),
                 "/opt/rocm/llvm/bin/" + tool):
        if os.path.exists(path):
            return path
    pytest.skip(f"{tool} is not installed")


def _spills(folder):
    """{kernel name: spilled vector registers} of every code object of the library."""
    lib = shutil.copy(LIB_PATH, folder / "lib.so")
    subprocess.run([_llvm("llvm-objdump"), "--offloading", lib], check=True, stdout=subprocess.DEVNULL, cwd=folder)
    found = {}
    for name in sorted(os.listdir(folder)):
        if "amdgcn" in name:
            notes = subprocess.run([_llvm("llvm-readelf"), "--notes", str(folder / name)], check=True,
                                   stdout=subprocess.PIPE).stdout.decode()
            found.update((k, int(n)) for k, n in re.findall(r"\.name: +(_ZN\S+)\n(?:(?! +- ).*\n)*?"
                                                            r" +\.vgpr_spill_count: +(\d+)", notes))
    return found


@pytest.mark.skipif(not os.path.exists(LIB_PATH), reason="the library is built by __graft_entry__.build()")
def test_verify_kernels_spill_no_vector_register(tmp_path):
    spills = {k: n for k, n in _spills(tmp_path).items() if "verify_kernel" in k}
    assert len(spills) > 100
    assert not {k: n for k, n in spills.items() if n}
