"""What the built kernels' code holds, read from the code objects of the last build (CPU only; the
tools are the ROCm toolchain's)."""
import os
import re
import subprocess

import pytest

from shaderous_amd import build

LLVM = "/opt/rocm/llvm/bin"


@pytest.fixture(scope="module")
def code_objects(tmp_path_factory):
    """The gfx950 code object of each translation unit, by its source's name."""
    out = {}
    folder = tmp_path_factory.mktemp("code")
    for src in build.sources():
        obj = os.path.join(build.BUILD, src + ".o")
        if not src.endswith(".hip") or not os.path.exists(obj):
            continue
        fat, co = str(folder / (src + ".fat")), str(folder / (src + ".co"))
        subprocess.run([f"{LLVM}/llvm-objcopy", "--dump-section", f".hip_fatbin={fat}", obj, os.devnull], check=True)
        subprocess.run([f"{LLVM}/clang-offload-bundler", "--unbundle", "--type=o", f"--input={fat}",
                        "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--output={co}"], check=True)
        out[src] = co
    if not out:
        pytest.skip("no objects: build first (python -m shaderous_amd.build)")
    return out


def kernels(co):
    """{kernel: bytes of code} of a code object."""
    text = subprocess.run([f"{LLVM}/llvm-readelf", "-sW", co], check=True, capture_output=True, text=True).stdout
    rows = [line.split() for line in text.splitlines() if " FUNC " in line]
    return {r[-1]: int(r[2], 0) for r in rows}


def test_second_flat_launch_stores_the_state_alone(code_objects):
    """k_amr_flat with MATCH reads the flux register that the launch before it wrote: its only stores
    are the leaf's two state vectors."""
    co = code_objects["amr2d_f32.hip"]
    found = [k for k in kernels(co) if re.match(r"_ZN3shx10k_amr_flatIfLi\dELi\dELb\dELb1E", k)]
    assert len(found) == 20   # ten schemes, means compensated or not
    text = subprocess.run([f"{LLVM}/llvm-objdump", "-d", "--no-show-raw-insn",
                           "--disassemble-symbols=" + ",".join(found), co], check=True, capture_output=True,
                          text=True).stdout
    stores, name = {k: [] for k in found}, None
    for line in text.splitlines():
        head = re.match(r"[0-9a-f]+ <(\S+)>:", line)
        if head:
            name = head.group(1)
        elif re.search(r"\b(global|buffer|flat)_(store|atomic)", line):
            stores[name].append(line.split()[0])
    bad = {k: v for k, v in stores.items() if v != ["global_store_dwordx4"] * 2}
    assert not bad, bad


def test_kernels_stay_small(code_objects):
    """A role kernel of 348 KB (FP64, Koren with the density reconstruction along the adiabat, walls;
    pow inlined at its 24 uses, 1452 B of scratch per lane) computed wrong values where the same source
    with pow as a call computed the plain path's. So pow stays a call, the uniform kernels stay
    within a branch's reach (2^15 words, 128 KiB: no branch through a register), and
    no kernel grows past the sizes that the GPU tests have covered."""
    found = {src: kernels(co) for src, co in code_objects.items()}
    assert "_ZN3shx4tpowEdd" in found["uniform_f64.hip"]
    for src, sizes in found.items():
        most = 128 << 10 if src.startswith(("uniform", "ens")) else 160 << 10
        big = {k: v for k, v in sizes.items() if v >= most}
        assert not big, (src, big)


def test_transcendentals_are_not_read_in_the_next_slot(code_objects):
    """On gfx950 a vector instruction must not read the result of a transcendental one (v_rcp, v_sqrt, v_exp,
    ...) right behind it. The compiler sees to that, but not for the operands of inline assembly
    (raw_min, raw_max in hydro.hpp), so it is checked over the whole code."""
    trans = re.compile(r"v_(rcp|sqrt|rsq|log|exp|sin|cos)_")

    def regs(text):
        out = {int(a) for a in re.findall(r"\bv(\d+)\b", text)}
        for a, b in re.findall(r"\bv\[(\d+):(\d+)\]", text):
            out |= set(range(int(a), int(b) + 1))
        return out

    seen, bad = 0, []
    for src, co in code_objects.items():
        text = subprocess.run([f"{LLVM}/llvm-objdump", "-d", "--no-show-raw-insn", "--no-leading-addr", co], check=True,
                              capture_output=True, text=True).stdout
        last = None
        for line in text.splitlines():
            op, _, rest = line.split("//")[0].strip().partition(" ")
            if last and op.startswith("v_") and not trans.match(op):
                first, _, others = rest.partition(",")
                read = regs(others) | (regs(first) if op.startswith(("v_fmac", "v_cmp")) else set())
                if last & read:
                    bad.append((src, line.strip()))
            last = None
            if trans.match(op):
                last = regs(rest.partition(",")[0])
                seen += 1
    assert seen > 10000 and not bad, bad[:5]
