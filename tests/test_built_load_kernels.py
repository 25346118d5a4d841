"""The kernels that pick their tiles by the load hold every form of the persistent grouped GEMM and use its accumulators by number as
the kernels of test_built_kernels.py do: the same check on the built code."""

import os
import re
import shutil
import subprocess

from test_built_kernels import _foreign, _objdump


def _kernels(tmp_path):
    """(name, instructions) of every kernel of the built library"""
    from dolomite_engine_amd import _lib, build, is_built

    if not is_built():
        build()
    shutil.copy(os.path.realpath(_lib.load()._name), tmp_path / "lib.so")
    objdump = _objdump()
    subprocess.run([objdump, "--offloading", str(tmp_path / "lib.so")], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    for image in sorted(p for p in tmp_path.iterdir() if "gfx950" in p.name):
        text = subprocess.run([objdump, "-d", "--no-show-raw-insn", "--no-leading-addr", str(image)], check=True,
                              capture_output=True, text=True).stdout
        for part in re.split(r"^(?=(?:[0-9a-f]+ )?<\w+>:$)", text, flags=re.M):
            name, _, body = part.partition("\n")
            yield name, [line.split("//")[0].strip() for line in body.splitlines()]


def test_nothing_else_in_the_accumulators(tmp_path):
    seen = 0
    for name, instructions in _kernels(tmp_path):
        if "grouped_gemm_by_load_kernelI" in name:
            seen += 1
            assert sum("v_mfma" in i for i in instructions) >= 3 * 64, name
            assert _foreign(instructions) == [], name
    assert seen == 8


def test_no_register_in_memory(tmp_path):
    """The four-wave kernels have a whole register file per wave and address a half of it by number: what does not fit the other half
    would be spilled to memory, in kernels whose loads and stores are waited for by count."""
    seen = 0
    for name, instructions in _kernels(tmp_path):
        if re.search("grouped_gemm_(persistent|even|by_load)_kernelI", name):
            seen += 1
            assert [i for i in instructions if i.startswith("scratch_")] == [], name
    assert seen == 8 + 28 + 8
