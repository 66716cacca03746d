"""Builds libdecaes_amd.so (gfx950 kernels + C ABI) in-tree with hipcc."""
from __future__ import annotations

import os
import re
import subprocess
import tempfile
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent            # decaes.jl_amd/
REPO = ROOT.parent
CSRC = ROOT / "csrc"
LIB = PKG / "libdecaes_amd.so"
# a C host program of the C ABI (csrc/dmi_run.c), linked against LIB
RUN = PKG / "dmi_run"
# Same sources built with -DDMI_PHASE_PROFILE: per-phase shader-clock counters (decaes_amd.phase_profile)
PHASE_LIB = PKG / "libdecaes_amd_phase.so"

# dmi_kernels_split.hip: the voxel kernel of the split schedule (dmi_kernels.hip compiled once more); the instrumented
# build keeps both schedules in dmi_kernels.hip
# dmi_kernels_reg.hip: once per size class of the register-resident kernel (kRegClasses of dmi_internal.h)
REG_CLASSES = (80, 72, 64, 48)
SOURCES = [*(f"dmi_kernels_reg.hip:{s}" for s in REG_CLASSES), "dmi_kernels.hip", "dmi_kernels_split.hip", "dmi_host.cpp", "dmi_api.cpp", "dmi_server.cpp", "dmi_synth.cpp"]

HIPCC_FLAGS = [
    "-O3", "--offload-arch=gfx950", "-fPIC", "-shared", "-std=c++17",
    # fma only where the reference writes muladd; never contract elsewhere
    "-ffp-contract=off",
    # no packed FP32 instructions (v_pk_*_f32) anywhere in device code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]
# the register-resident kernels set the waves attribute for its register limit, not for that occupancy; their device
# assembly is kept for check_bank
REG_FLAGS = ["-Wno-pass-failed", "--save-temps=obj"]


def hipcc() -> str:
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    return str(Path(rocm) / "bin" / "hipcc")


def _vgprs(text: str) -> set[int]:
    out = set()
    for lo, hi, one in re.findall(r"\bv(?:\[(\d+):(\d+)\]|(\d+))(?![\w\[])", text):
        out |= {int(one)} if one else set(range(int(lo), int(hi) + 1))
    return out


def check_bank(asm: str, rows: int) -> None:
    """The register-resident solver addresses the registers from 256 - 2 rows on by name in inline assembly, which the
    compiler does not know of, and writes its DPP reads there too, past the compiler's hazard checks. In the device
    assembly of a size class: no instruction of the compiler's names a register of the bank, and every DPP read comes at
    least two wait states after a VALU write of its source."""
    bank, inline, recent = 256 - 2 * rows, False, []  # recent: registers written in each of the last two wait states
    for no, line in enumerate(asm.splitlines(), 1):
        if line.lstrip().startswith((";;#ASMSTART", ";;#ASMEND")):
            inline = "ASMSTART" in line
            continue
        text = line.split(";")[0].strip()
        if not text or text.startswith(".") or text.endswith(":"):
            continue
        op, _, args = text.replace("\t", " ").partition(" ")
        args = [a.strip() for a in args.split(",")]
        if not inline and max(_vgprs(text), default=0) >= bank:
            raise RuntimeError(f"{rows}-row class: the compiler uses the solver's registers (v{bank} on) in line {no}: {text}")
        if "_dpp" in op and any(_vgprs(args[1].split()[0]) & w for w in recent):
            raise RuntimeError(f"{rows}-row class: a DPP read follows the write of its source too closely in line {no}: {text}")
        states = int(args[0], 0) + 1 if op == "s_nop" else 1
        recent = (recent + [set()] * (states - 1) + [_vgprs(args[0]) if op.startswith("v_") else set()])[-2:]


def _compile(cmd: list[str], obj: Path, rows: str) -> None:
    if not rows:
        subprocess.run([*cmd, "-o", str(obj)], check=True)
        return
    with tempfile.TemporaryDirectory(dir=obj.parent) as tmp:
        subprocess.run([*cmd, *REG_FLAGS, "-o", str(Path(tmp) / obj.name)], check=True)
        check_bank(next(Path(tmp).glob("*gfx950.s")).read_text(), int(rows))
        os.replace(Path(tmp) / obj.name, obj)


def build(verbose: bool = False, phase_profile: bool = False) -> Path:
    """Compile every source into decaes_amd/libdecaes_amd.so (always recompiles). With phase_profile, build the
    instrumented variant decaes_amd/libdecaes_amd_phase.so instead."""
    objs, cmds = [], []
    obj_dir = ROOT / ("_build_phase" if phase_profile else "_build")
    obj_dir.mkdir(exist_ok=True)
    out = PHASE_LIB if phase_profile else LIB
    extra = ["-DDMI_PHASE_PROFILE"] if phase_profile else []
    for src in SOURCES:
        src, _, rows = src.partition(":")
        if phase_profile and src == "dmi_kernels_split.hip":
            continue
        obj = obj_dir / (src + rows + ".o")
        cmd = [hipcc(), *HIPCC_FLAGS, *extra, "-c", "-I", str(REPO / "include"), "-I", str(CSRC), str(CSRC / src)]
        if rows:
            cmd.insert(1, f"-DDMI_REG_S={rows}")
        if src.endswith(".cpp"):
            cmd = [c for c in cmd if c not in ("--offload-arch=gfx950",)]
        if verbose:
            print(" ".join(cmd), flush=True)
        cmds.append((cmd, obj, rows))
        objs.append(str(obj))
    # the sources compile independently: one hipcc process each, at most MAX_JOBS (or the CPU count) at once
    jobs = max(1, min(len(cmds), int(os.environ.get("MAX_JOBS", 0)) or os.cpu_count() or 1))
    with ThreadPoolExecutor(jobs) as pool:
        for f in [pool.submit(_compile, *c) for c in cmds]:
            f.result()
    tmp = out.with_suffix(".so.tmp")
    link = [hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", str(tmp), "-lpthread"]
    if verbose:
        print(" ".join(link), flush=True)
    subprocess.run(link, check=True)
    os.replace(tmp, out)
    if not phase_profile:
        run = [os.environ.get("CC", "gcc"), "-O2", "-std=c11", "-Wall", "-I", str(REPO / "include"),
               str(CSRC / "dmi_run.c"), "-o", str(RUN.with_suffix(".tmp")), "-L", str(PKG), "-ldecaes_amd",
               "-Wl,-rpath,$ORIGIN", "-Wl,--allow-shlib-undefined", "-lm"]
        if verbose:
            print(" ".join(run), flush=True)
        subprocess.run(run, check=True)
        os.replace(RUN.with_suffix(".tmp"), RUN)
    return out


if __name__ == "__main__":
    import sys

    print(build(verbose=True, phase_profile="--phase" in sys.argv[1:]))
