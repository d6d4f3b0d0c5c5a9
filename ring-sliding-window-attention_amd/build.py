"""Build librswa.so (HIP, gfx950 only) in-tree with hipcc, and the module that calls it from
PyTorch (host code) with the C++ compiler.

Usage: ``python build.py [--force]``.  Objects go to ``build/``, the shared
library to ``lib/librswa.so`` next to this file, the module to ``lib/rswa_torch.so``.  hipcc cross-compiles, so no
GPU is needed to build.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import re
import shutil
import struct
import subprocess
import sys
import tempfile
from typing import List

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "build")
LIBDIR = os.path.join(HERE, "lib")
LIB = os.path.join(LIBDIR, "librswa.so")
# the same library with every MFMA issued through the compiler builtin (hazards padded by the
# compiler): the cross-check of the hand-kept hazard distance of the inline-assembly MFMAs
LIB_BUILTIN_MFMA = os.path.join(LIBDIR, "librswa_builtin_mfma.so")
ASM_MFMA_SOURCES = ("attn_bwd.hip",)  # sources that issue MFMAs, and loads into LDS, as inline assembly

ARCH = "gfx950"
FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fno-gpu-rdc",
    "-Wall",
    "-Wno-unused-function",
    "-Wno-unknown-attributes",
    # packed fp32 VALU forms are kept out of generated code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # per-kernel register / scratch report on stderr (checked below)
    "-Rpass-analysis=kernel-resource-usage",
]


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found")


def sources() -> List[str]:
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))


def _headers() -> List[str]:
    hs = [os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".h")]
    hs.append(os.path.join(os.path.dirname(HERE), "include", "rswa.h"))
    return hs


def _stale(target: str, deps: List[str]) -> bool:
    if not os.path.exists(target):
        return True
    t = os.path.getmtime(target)
    return any(os.path.getmtime(d) > t for d in deps)


def _compile(src: str, force: bool, builtin_mfma: bool = False) -> str:
    stem = os.path.basename(src)[:-4]
    obj = os.path.join(OBJ, stem + (".builtin_mfma.o" if builtin_mfma else ".o"))
    if force or _stale(obj, [src] + _headers()):
        extra = ["-DRSWA_MFMA_BUILTIN_ONLY"] if builtin_mfma else []
        cmd = [_hipcc(), *FLAGS, *extra, "-c", src, "-o", obj]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"hipcc failed for {src}:\n{r.stdout}\n{r.stderr}")
        if not builtin_mfma:  # the cross-check build may spill: it is never timed
            _check_no_scratch(src, r.stderr)
            warn = _real_warnings(r.stderr)
            if warn:
                sys.stderr.write(warn + "\n")
    return obj


def _real_warnings(stderr: str) -> str:
    """Compiler output minus the resource-usage remarks (each followed by a source line and
    a caret line) and the host pass's note about the device-only target feature."""
    out, skip = [], 0
    for line in stderr.splitlines():
        if skip:
            skip -= 1
            continue
        if "-Rpass-analysis=kernel-resource-usage" in line:
            skip = 2 if "Function Name" in line else 0
            continue
        if "packed-fp32-ops" in line or not line.strip():
            continue
        out.append(line)
    return "\n".join(out)


def _check_no_scratch(src: str, stderr: str) -> None:
    """No kernel may use scratch memory: a register spilled inside a tile loop comes back
    through a load whose wait also waits for every tile load in flight."""
    name, bad = None, []
    for line in stderr.splitlines():
        m = re.search(r"remark:\s+(.*?): (.*?) \[-Rpass-analysis=kernel-resource-usage\]", line)
        if not m:
            continue
        key, val = m.group(1).strip(), m.group(2).strip()
        if key == "Function Name":
            name = val
        elif key.startswith("ScratchSize") and val != "0":
            bad.append(f"{name}: {val} bytes of scratch per lane")
    if bad:
        raise RuntimeError(f"{src}: kernels spill registers to scratch memory:\n  " + "\n  ".join(bad))


def _code_objects(fat: bytes):
    """The code objects for ARCH in a fatbin section (bundles one behind the other)."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = fat.find(magic)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", fat, at + 24)
        p = at + 32
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", fat, p)
            if ARCH.encode() in fat[p + 24:p + 24 + n] and size:
                yield fat[at + off:at + off + size]
            p += 24 + n
        at = fat.find(magic, at + 24)


_LDS_LOAD_WAIT = 5  # wait states from a vector instruction's write of an SGPR to its use by a memory instruction


def _sgprs(operand: str) -> set:
    m = re.fullmatch(r"s\[(\d+):(\d+)\]|s(\d+)", operand)
    if not m:
        return {operand} & {"m0"}
    return set(range(int(m[1]), int(m[2]) + 1)) if m[1] else {int(m[3])}


def close_sgpr_writes(listing: List[str]) -> List[str]:
    """Loads into LDS of one kernel (disassembled, branch targets as ``<L0>:`` lines) that a vector
    instruction's write of one of their scalar registers comes too close to, along any path: the
    hand-written ones are invisible to the compiler's hazard pass."""
    code = [line.split("//")[0].split(";")[0].strip() for line in listing]
    jumps = {}
    for i, x in enumerate(code):
        m = re.match(r"s_c?branch\S* (\S+)$", x)
        if m:
            jumps.setdefault(m[1].strip("<>"), []).append(i)
    bad = []

    def writer(i: int, left: int, used: set, load: str):
        """Walk back from line i (not included) with ``left`` wait states to go."""
        while left > 0 and i > 0:
            i -= 1
            x = code[i]
            label = re.fullmatch(r"(?:[0-9a-f]+ )?<(L\d+)>:", x)
            if label:
                for j in jumps.get(label[1], ()):
                    writer(j, left - 1, used, load)
                continue
            if not x:
                continue
            if x.startswith(("s_branch", "s_endpgm", "s_setpc")):
                return  # not reached from here
            name, _, rest = x.partition(" ")
            if name.startswith("v_"):
                ops = [o.strip() for o in rest.split(",")]
                out = ops[:2] if "_co_" in name or "div_scale" in name else ops[:1]
                if any(_sgprs(o) & used for o in out):
                    bad.append(f"{x}  ...  {load}")
                    return
            left -= int(rest) + 1 if name == "s_nop" else 1

    for i, x in enumerate(code):
        if x.startswith("buffer_load") and x.endswith(" lds"):
            ops = [o.strip() for o in x.partition(" ")[2].replace(" offen", ",").split(",")]
            writer(i, _LDS_LOAD_WAIT, set().union({"m0"}, *(_sgprs(o) for o in ops)), x)
    return bad


def close_m0_writes(listing: List[str]) -> List[str]:
    """Loads into LDS with no instruction between a scalar write of m0 and them (one wait state is needed; the
    hand-written loads that carry an offset take m0 as an earlier one left it, and have no ``s_nop`` of their own)."""
    code = [line.split("//")[0].split(";")[0].strip() for line in listing]
    code = [x for x in code if x and not x.endswith(">:")]
    return [f"{w}  ...  {x}" for w, x in zip(code, code[1:])
            if x.startswith("buffer_load") and x.endswith(" lds") and re.match(r"s_\w+ m0,", w)]


def _check_lds_loads(obj: str) -> None:
    """No load into LDS may follow a write of its scalar registers too closely."""
    llvm = os.path.join(os.path.dirname(os.path.realpath(_hipcc())), "..", "llvm", "bin")
    with tempfile.TemporaryDirectory() as tmp:
        fat = os.path.join(tmp, "fat")
        subprocess.run([os.path.join(llvm, "llvm-objcopy"), "--dump-section", ".hip_fatbin=" + fat, obj, os.devnull],
                       check=True)
        for i, code in enumerate(_code_objects(open(fat, "rb").read())):
            path = os.path.join(tmp, f"{i}.co")
            with open(path, "wb") as f:
                f.write(code)
            text = subprocess.run([os.path.join(llvm, "llvm-objdump"), "-d", "--no-show-raw-insn",
                                   "--symbolize-operands", path], check=True, capture_output=True, text=True).stdout
            for name, body in re.findall(r"^[0-9a-f]+ <(_Z\w+)>:\n(.*?)(?=^[0-9a-f]+ <_Z|\Z)", text, re.M | re.S):
                bad = close_sgpr_writes(body.splitlines()) + close_m0_writes(body.splitlines())
                if bad:
                    raise RuntimeError(f"{name}: scalar registers written too close to a load into LDS:\n  "
                                       + "\n  ".join(bad))


def _torch_build() -> str:
    """The same text as ring_swa._lib.torch_build() (the build imports nothing of the package)."""
    import torch

    return (f"{torch.__version__} {torch.version.git_version} hip {torch.version.hip} "
            f"python {sys.version_info[0]}.{sys.version_info[1]}")


def _build_torch_calls(force: bool) -> str:
    """The module of csrc/torch_calls.cpp, against the installed PyTorch (build/rswa_torch.for: which it was)."""
    src, out = os.path.join(CSRC, "torch_calls.cpp"), os.path.join(LIBDIR, "rswa_torch.so")
    made_for, now = os.path.join(OBJ, "rswa_torch.for"), _torch_build()
    same = os.path.exists(made_for) and open(made_for).read() == now
    if force or not same or _stale(out, [src] + _headers()):
        import sysconfig

        import torch

        root = os.path.dirname(torch.__file__)
        inc = [os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"),
               os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"), sysconfig.get_paths()["include"]]
        cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1",
               "-DUSE_ROCM=1", f'-DRSWA_TORCH_BUILD="{now}"', f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
               *[x for i in inc for x in ("-isystem", i)], src, "-o", out, "-L" + os.path.join(root, "lib"),
               *["-l" + n for n in ("c10", "c10_hip", "torch_cpu", "torch_hip", "torch", "torch_python")]]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"C++ compiler failed for {src}:\n{r.stdout}\n{r.stderr}")
        with open(made_for, "w") as f:
            f.write(now)
    return out


def build(force: bool = False, jobs: int = 8) -> str:
    os.makedirs(OBJ, exist_ok=True)
    os.makedirs(LIBDIR, exist_ok=True)
    srcs = sources()
    asm_srcs = [s for s in srcs if os.path.basename(s) in ASM_MFMA_SOURCES]
    with cf.ThreadPoolExecutor(max_workers=min(jobs, len(srcs) + len(asm_srcs) + 1)) as ex:
        calls = ex.submit(_build_torch_calls, force)
        futs = [ex.submit(_compile, s, force) for s in srcs]
        alt_futs = {s: ex.submit(_compile, s, force, True) for s in asm_srcs}
        objs = [f.result() for f in futs]
        alt = {s: f.result() for s, f in alt_futs.items()}
        calls.result()
    for o in objs:
        if os.path.basename(o)[:-2] + ".hip" in ASM_MFMA_SOURCES and (force or _stale(LIB, [o])):
            _check_lds_loads(o)
    alt_objs = [alt.get(s, o) for s, o in zip(srcs, objs)]
    for lib, members in ((LIB, objs), (LIB_BUILTIN_MFMA, alt_objs)):
        if force or _stale(lib, members):
            cmd = [_hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", lib, *members]
            r = subprocess.run(cmd, capture_output=True, text=True)
            if r.returncode != 0:
                raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    return LIB


if __name__ == "__main__":
    print(build(force="--force" in sys.argv))
