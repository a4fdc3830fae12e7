"""Build libtimeviper_hip.so (gfx950) from timeviper_amd/csrc with plain hipcc.

The library is a C-ABI shared object (include/timeviper_hip.h); it does not link
against torch.  Objects are cached by CONTENT: every object carries a sidecar with the
hash of its source, the shared headers and the compiler flags, and the library embeds the
hash of the whole source set (`tv_build_id()`), so a kernel edit can never be benchmarked
through a stale binary — not even on a box whose file mtimes were reset by a copy.

    python -m timeviper_amd.build [--force] [--jobs N]
"""
from __future__ import annotations

import argparse
import hashlib
import os
import subprocess
import sys
import sysconfig
import tempfile
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

ROOT = Path(__file__).resolve().parent
CSRC = ROOT / "csrc"
OBJ = ROOT / "lib" / "obj"
LIB = ROOT / "lib" / "libtimeviper_hip.so"
LIB_ID = ROOT / "lib" / "libtimeviper_hip.id"
NATIVE = ROOT / "lib" / f"_tv_native{sysconfig.get_config_var('EXT_SUFFIX') or '.so'}"      # the operators' host side: a Python extension on torch's headers, no device code
NATIVE_ID = NATIVE.with_suffix(".id")
NATIVE_SRC = CSRC / "host" / "native_ops.cpp"
ARCH = "gfx950"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = ["-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-ffp-contract=off",
         "-Wno-unused-result", "-DNDEBUG",
         # no packed fp32 arithmetic (v_pk_{add,mul,fma}_f32): some of its forms give wrong results now and then on this pool
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
if os.environ.get("TV_MARCH_ABLATE"):   # dev only: compile the scan kernel's ablation switches in
    FLAGS.append("-DTV_MARCH_ABLATE")
if os.environ.get("TV_FA_STAMP"):       # dev only: per-phase stamps in the streaming attention kernel
    FLAGS.append("-DTV_FA_STAMP")
if os.environ.get("TV_DRIP_STAMP"):     # dev only: per-phase cycle sums in the 256 x 192 GEMM (gemm_drip.hip)
    FLAGS.append("-DTV_DRIP_STAMP")
if os.environ.get("TV_SLICE_STAMP"):    # dev only: per-wave barrier-wait stamps in ssd_slice.hip
    FLAGS.append("-DTV_SLICE_STAMP")


FLAGS += os.environ.get("TV_EXTRA_HIPCC_FLAGS", "").split()   # dev only

# per-file flags.  gemm_drip.hip names its accumulator registers (a[0:119], csrc/gemm_drip_regs.inc) instead of handing
# them to the register allocator: the compiler must then never park a spilled vector register in an accumulator register.
FILE_FLAGS = {"gemm_drip.hip": ["-mllvm", "-amdgpu-spill-vgpr-to-agpr=0"]}


def _sources():
    return sorted(list(CSRC.glob("*.hip")) + list(CSRC.glob("*.cpp")))


def _headers():
    incs = [p for p in CSRC.glob("*.inc") if not p.name.endswith("_stamp.inc")]      # generated asm bodies (devtools/gen_head_step.py)
    return sorted(list(CSRC.glob("*.hpp")) + incs + list((ROOT.parent / "include").glob("*.h")))


def _hash(paths, extra: str = "") -> str:
    h = hashlib.sha256(extra.encode())
    for p in paths:
        h.update(p.name.encode())
        h.update(p.read_bytes())
    return h.hexdigest()[:16]


def source_id() -> str:
    """Hash of every source, header and compiler flag the library is built from."""
    return _hash(_sources() + _headers(), " ".join(FLAGS) + repr(sorted(FILE_FLAGS.items())))


def _compile(src: Path, force: bool, build_id: str) -> Path:
    obj = OBJ / (src.name + ".o")
    tag = OBJ / (src.name + ".hash")
    flags = list(FLAGS) + FILE_FLAGS.get(src.name, [])
    if src.name == "capi.cpp":                    # the one translation unit that carries the id
        flags.append(f'-DTV_BUILD_ID="{build_id}"')
    want = _hash([src] + _headers(), " ".join(flags))
    if not force and obj.exists() and tag.exists() and tag.read_text() == want:
        return obj
    cmd = [HIPCC, *flags, "-x", "hip", "-c", str(src), "-o", str(obj)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{r.stdout}\n{r.stderr}")
    # (the host pass does not know the device feature that FLAGS turn off and says so once per pass)
    err = "".join(ln for ln in r.stderr.splitlines(keepends=True) if "packed-fp32-ops" not in ln)
    if err.strip():
        sys.stderr.write(err)
    tag.write_text(want)
    return obj


def build(force: bool = False, jobs: int = 0) -> Path:
    jobs = jobs or max(1, min(16, int(os.environ.get("MAX_JOBS") or 8), os.cpu_count() or 1))
    OBJ.mkdir(parents=True, exist_ok=True)
    srcs = _sources()
    bid = source_id()
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(lambda s: _compile(s, force, bid), srcs))
    if force or not LIB.exists() or not LIB_ID.exists() or LIB_ID.read_text() != bid:
        cmd = [HIPCC, "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", str(LIB), *map(str, objs)]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
        LIB_ID.write_text(bid)
    try:
        build_native(force)
    except (OSError, RuntimeError) as e:          # (no C++ compiler for the host, no Python.h): the operators' other host side serves
        sys.stderr.write(f"{NATIVE.name} cannot be built, operators go through ctypes: {e}\n")
    return LIB


CXX = os.environ.get("CXX", "g++")
NATIVE_FLAGS = ["-O2", "-std=c++17", "-fPIC", "-shared", "-w", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1"]
NATIVE_LIBS = ["-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python"]


def _native_paths():
    import torch
    t = Path(torch.__file__).resolve().parent
    rocm = Path(HIPCC).resolve().parent.parent if Path(HIPCC).is_absolute() else Path("/opt/rocm")
    return [f"-I{p}" for p in (ROOT.parent / "include", t / "include", t / "include" / "torch" / "csrc" / "api" / "include", "/opt/rocm/include", rocm / "include",
                               sysconfig.get_paths()["include"])], [f"-L{t / 'lib'}"]


def native_id() -> str:
    """Hash of all that the host operators are built from: source, the C ABI's header, flags, compiler, Python's ABI, torch's version (not the paths: a tree may be copied)"""
    import torch
    return _hash([NATIVE_SRC, ROOT.parent / "include" / "timeviper_hip.h"],
                 " ".join([CXX, *NATIVE_FLAGS, *NATIVE_LIBS, NATIVE.name, torch.__version__, str(torch.version.hip)]))


def native_is_current() -> bool:
    """By the file beside it; what is loaded is asked itself (_native.py)"""
    return NATIVE.exists() and NATIVE_ID.exists() and NATIVE_ID.read_text() == native_id()


def build_native(force: bool = False) -> Path:
    if force or not native_is_current():
        want, (includes, paths) = native_id(), _native_paths()
        NATIVE.parent.mkdir(parents=True, exist_ok=True)
        # linked beside its place and moved there whole: another process may load it, or build it too, at any time
        with tempfile.TemporaryDirectory(dir=NATIVE.parent) as work:
            out, tag = Path(work) / NATIVE.name, Path(work) / NATIVE_ID.name
            r = subprocess.run([CXX, *NATIVE_FLAGS, f'-DTV_NATIVE_ID="{want}"', *includes, str(NATIVE_SRC), "-o", str(out), *paths, *NATIVE_LIBS], capture_output=True, text=True)
            if r.returncode != 0:
                raise RuntimeError(f"host operators: {r.stdout}\n{r.stderr}")
            tag.write_text(want)
            os.replace(out, NATIVE)
            os.replace(tag, NATIVE_ID)
    return NATIVE


def ensure_built() -> Path:
    """Make `lib/libtimeviper_hip.so` match the sources in the tree: a no-op when the library's
    recorded build id equals the hash of csrc/ + include/ (+ flags), else an incremental rebuild.
    This is a BUILD step, not a fallback: without a working hipcc it raises, and the operators
    keep failing loudly.  (`_capi.lib()` checks `tv_build_id()` of the loaded library against the
    same hash, so a stale binary cannot be used silently either.)"""
    if LIB.exists() and LIB_ID.exists() and LIB_ID.read_text() == source_id() and native_is_current():
        return LIB
    return build()


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--force", action="store_true")
    ap.add_argument("--jobs", type=int, default=0, help="parallel compilations (0: MAX_JOBS, else 8)")
    a = ap.parse_args()
    print(build(a.force, a.jobs))
