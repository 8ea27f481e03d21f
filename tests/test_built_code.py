"""What the built library's gfx950 code holds: hints that the sources give and a compiler may drop without a word."""
import collections
import os
import re
import shutil
import subprocess

import pytest

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.fixture(scope="module")
def stores(tmp_path_factory):
    """{kernel: {(width of a global store, non-temporal): how many}} of libbi8.so"""
    from blockwise_int8_linear_amd import _lib
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    _lib.load()
    at = tmp_path_factory.mktemp("code")
    shutil.copy(os.path.join(os.path.dirname(_lib.__file__), "libbi8.so"), at / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=at, check=True, capture_output=True)
    found = {}
    for part in sorted(p for p in os.listdir(at) if "gfx950" in p):
        code = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--demangle", part], cwd=at, check=True, capture_output=True, text=True).stdout
        count = None
        for line in code.splitlines():
            head = re.match(r"[0-9a-f]+ <(.*)>:", line)
            if head:
                name = head.group(1).replace("(anonymous namespace)::", "").replace("void ", "").split("(")[0]
                count = found.setdefault(name, collections.Counter())
                continue
            store = re.match(r"\s+global_store_(\w+)(.*)", line)
            if store and count is not None:
                count[store.group(1), re.search(r"\bnt\b", store.group(2).split("//")[0]) is not None] += 1
    return found


def test_last_tile_leaves_non_temporally(stores):
    """gemm_wide's workgroups store their last tile non-temporally and the tiles before it plainly: as many stores of either kind"""
    kernels = {n: c for n, c in stores.items() if n.startswith("gemm_wide<") and n.split(", ")[3] == "false"}
    assert len(kernels) == 30                      # two blocks, three output types, five tiles
    for name, count in kernels.items():
        assert count["dwordx4", True] == count["dwordx4", False] > 0, name
