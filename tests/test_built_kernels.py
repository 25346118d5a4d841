"""What the compiler made of the four-wave matrix kernels, checked on the built library.

They address their accumulators a0 .. a255 by number, which the compiler does not know to be live between the points at
which they are declared lost: only matrix instructions may write an accumulator register and only v_accvgpr_read may read
one elsewhere.  The weight gradient requests its row indices in assembly and waits for them later, by count: nothing may
touch their registers in between."""

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


def test_foreign_writes_are_seen():
    own = ["v_mfma_f32_16x16x32_bf16 a[0:3], v[4:7], v[8:11], a[0:3]", "v_accvgpr_read_b32 v1, a17", "v_mov_b32_e32 v1, v2"]
    planted = ["v_accvgpr_write_b32 a3, v1", "v_accvgpr_mov_b32 a1, a2", "scratch_load_dword a5, off, off",
               "ds_read_b128 a[4:7], v1 offset:16", "global_store_dwordx4 v[0:1], a[0:3], off"]
    assert _foreign(own) == []
    assert _foreign(own + planted) == planted


def _early_uses(instructions):
    """Instructions that touch the result of a plain buffer load before the next wait for one."""
    def regs(text):
        for lo, hi in re.findall(r"(?<!\w)v(?:\[(\d+):(\d+)\]|(?=\d))", text):
            if lo:
                yield from range(int(lo), int(hi) + 1)
        yield from map(int, re.findall(r"(?<![\w\[])v(\d+)\b", text))

    out, pending = [], set()
    for text in instructions:
        if text.startswith("s_waitcnt") and "vmcnt" in text:
            pending.clear()
            continue
        if text.startswith("buffer_load") and not text.endswith(" lds"):
            dst, _, rest = text.partition(" ")[2].partition(",")
            if not pending.isdisjoint(regs(rest)):
                out.append(text)
            pending.update(regs(dst))
        elif pending and not pending.isdisjoint(regs(text)):
            out.append(text)
    return out


def test_early_uses_are_seen():
    own = ["buffer_load_dwordx4 v[4:7], v1, s[0:3], s4 offen", "buffer_load_dwordx4 v8, s[0:3], s4 offen lds",
           "v_mov_b32_e32 v2, v3", "s_waitcnt vmcnt(8)", "v_mul_lo_u32 v9, v5, s3"]
    assert _early_uses(own) == []
    for planted in ("v_mul_lo_u32 v9, v5, s3", "v_mov_b64_e32 v[20:21], v[6:7]", "v_add_u32_e32 v4, v1, v2"):
        assert _early_uses(own[:2] + [planted] + own[2:]) == [planted]


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """(name, instructions) of the four-wave kernels in the built library."""
    from dolomite_engine_amd import _lib, build, is_built

    if not is_built():
        build()
    tmp = tmp_path_factory.mktemp("code")
    shutil.copy(os.path.realpath(_lib.load()._name), tmp / "lib.so")
    objdump = _objdump()
    subprocess.run([objdump, "--offloading", str(tmp / "lib.so")], cwd=tmp, check=True, stdout=subprocess.DEVNULL)
    found = []
    for image in sorted(p for p in tmp.iterdir() if "gfx950" in p.name):
        text = subprocess.run([objdump, "-d", "--no-show-raw-insn", "--no-leading-addr", str(image)], check=True,
                              capture_output=True, text=True).stdout
        kernel, body = None, []
        for line in text.splitlines() + ["<end>:"]:
            label = re.match(r"^(?:[0-9a-f]+ )?<(\w+)>:$", line)
            if label is None:
                body.append(line.split("//")[0].strip())
                continue
            if kernel is not None:
                found.append((kernel, body))
            kernel = next((k for k in KERNELS if re.search(rf"\d{k}I", label.group(1))), None)
            body = []
    assert {k: sum(name == k for name, _ in found) for k in KERNELS} == KERNELS
    return found


def test_nothing_else_in_the_accumulators(kernels):
    for name, body in kernels:
        assert sum("v_mfma" in i for i in body) >= 128, name
        assert _foreign(body) == [], name


def test_row_indices_are_not_touched_before_their_wait(kernels):
    loads = 0
    for name, body in kernels:
        if name == "grouped_wgrad_kernel":
            loads += sum(i.startswith("buffer_load") and not i.endswith(" lds") for i in body)
            assert _early_uses(body) == []
    assert loads > 0
