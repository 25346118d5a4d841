"""The four-wave matrix kernels address their accumulators a0 .. a255 by number, which the compiler does not know to be live
between the points at which they are declared lost.  What it made of them is checked here on the built library: in these
kernels only matrix instructions write an accumulator register and only v_accvgpr_read reads one elsewhere."""

import os
import re
import shutil
import subprocess

import pytest

KERNELS = {"grouped_gemm_persistent_kernel": 8, "grouped_gemm_fp8_persistent_kernel": 4, "grouped_wgrad_kernel": 8}
AGPR = re.compile(r"(?<![\w.])a(\d+|\[\d+:\d+\])(?!\w)")


def _objdump():
    for path in (shutil.which("llvm-objdump"), os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm/bin/llvm-objdump")):
        if path and os.path.exists(path):
            return path
    pytest.skip("no llvm-objdump")


def _foreign(instructions):
    """Instructions that touch an accumulator register and are not the kernels' own."""
    out = []
    for text in instructions:
        mnemonic, _, operands = text.partition(" ")
        if not AGPR.search(operands):
            continue
        first = operands.split(",")[0]
        if mnemonic.startswith("v_mfma_f32_16x16x32") or (mnemonic.startswith("v_accvgpr_read") and not AGPR.search(first)):
            continue
        out.append(text)
    return out


def test_checker_sees_foreign_writes():
    own = ["v_mfma_f32_16x16x32_bf16 a[0:3], v[4:7], v[8:11], a[0:3]", "v_accvgpr_read_b32 v1, a17", "v_mov_b32_e32 v1, v2"]
    planted = ["v_accvgpr_write_b32 a3, v1", "v_accvgpr_mov_b32 a1, a2", "scratch_load_dword a5, off, off",
               "ds_read_b128 a[4:7], v1 offset:16", "global_store_dwordx4 v[0:1], a[0:3], off"]
    assert _foreign(own) == []
    assert _foreign(own + planted) == planted


def test_nothing_else_in_the_accumulators(tmp_path):
    from dolomite_engine_amd import _lib, build, is_built

    if not is_built():
        build()
    lib = os.path.realpath(_lib.load()._name)
    copy = tmp_path / "lib.so"
    shutil.copy(lib, copy)
    objdump = _objdump()
    subprocess.run([objdump, "--offloading", str(copy)], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    seen = dict.fromkeys(KERNELS, 0)
    for image in sorted(p for p in tmp_path.iterdir() if "gfx950" in p.name):
        text = subprocess.run([objdump, "-d", "--no-show-raw-insn", "--no-leading-addr", str(image)], check=True,
                              capture_output=True, text=True).stdout
        kernel, body = None, []
        for line in text.splitlines() + ["<end>:"]:
            label = re.match(r"^(?:[0-9a-f]+ )?<(\w+)>:$", line)
            if label is None:
                body.append(line.split("//")[0].strip())
                continue
            if kernel is not None:
                assert sum("v_mfma" in i for i in body) >= 128, label
                assert _foreign(body) == [], kernel
                seen[kernel] += 1
            kernel = next((k for k in KERNELS if re.search(rf"\d{k}I", label.group(1))), None)
            body = []
    assert seen == KERNELS
