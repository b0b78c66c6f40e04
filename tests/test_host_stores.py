"""Kernels that store to host memory behind a mark release their stores to the system themselves: a mark set by a later launch
says that they have ended, and its own release is of its own XCD's cache.  Read from the library's code for gfx950."""
import os
import re
import subprocess

import pytest

from cachegen_amd.build import LIBRARY

OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")


@pytest.fixture(scope="module")
def code_object(tmp_path_factory):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    if not os.path.exists(LIBRARY):
        from cachegen_amd.build import build_library
        build_library()
    at = tmp_path_factory.mktemp("code")
    os.symlink(LIBRARY, at / "library.so")
    subprocess.run([OBJDUMP, "--offloading", "library.so"], cwd=at, check=True, stdout=subprocess.DEVNULL)
    found = [f for f in os.listdir(at) if "gfx950" in f]
    assert len(found) == 1, os.listdir(at)
    symbols = subprocess.run([OBJDUMP, "-t", found[0]], cwd=at, check=True, capture_output=True, text=True).stdout
    return at, found[0], [line.split()[-1] for line in symbols.splitlines() if " .text" in line]


@pytest.mark.parametrize("kernel", ["mark_kernel", "read_words_kernel", "largest_kernel", "scan_collect_kernel", "collect_sizes_kernel",
                                    "wire_meta_kernel", "counts_to_tables_kernel"])
def test_stores_are_released_to_the_system(code_object, kernel):
    at, name, symbols = code_object
    found = [s for s in symbols if re.search(r"\d%s" % kernel, s)]
    assert len(found) == 1, found
    text = subprocess.run([OBJDUMP, "-d", "--disassemble-symbols=" + found[0], name], cwd=at, check=True, capture_output=True, text=True).stdout
    assert "s_endpgm" in text
    assert re.search(r"buffer_wbl2 .*sc0.*sc1|buffer_wbl2 .*sc1.*sc0", text), "no write-back at system scope"
