"""What the built library's gfx950 code holds: hints and orders that the sources give and a compiler may drop without a word."""
import os
import re
import shutil
import subprocess

import pytest

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{kernel: its instructions} of libbi8.so"""
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
        lines = None
        for line in code.splitlines():
            head = re.match(r"[0-9a-f]+ <(.*)>:", line)
            if head:
                lines = found.setdefault(head.group(1).replace("(anonymous namespace)::", "").replace("void ", "").split("(")[0], [])
            elif lines is not None:
                lines.append(line.split("//")[0].strip())
    return found


def test_last_tile_leaves_non_temporally(kernels):
    """gemm_wide's workgroups store their last tile non-temporally and the tiles before it plainly: as many stores of either kind"""
    wide = {n: c for n, c in kernels.items() if n.startswith("gemm_wide<") and n.split(", ")[3] == "false"}
    assert len(wide) == 30                         # two blocks, three output types, five tiles
    for name, code in wide.items():
        stores = [line.split()[-1] == "nt" for line in code if line.startswith("global_store_dwordx4")]
        assert 2 * sum(stores) == len(stores) > 0, name


def test_early_bias_is_not_waited_for(kernels):
    """the few-row kernels ask for a 16-bit bias in front of their streams and convert it behind them: loads of the streams are issued
    between the bias' load and the first wait for loads after it"""
    few = {n: c for n, c in kernels.items() if n.startswith(("gemv_rows<", "gemv_staged<"))}
    assert few
    for name, code in few.items():
        bias = next(i for i, line in enumerate(code) if line.startswith("global_load_ushort"))
        wait = next(i for i in range(bias, len(code)) if line_waits_for_loads(code[i]))
        assert any(line.startswith("buffer_load") for line in code[bias:wait]), name


def line_waits_for_loads(line):
    return line.startswith("s_waitcnt") and "vmcnt" in line
