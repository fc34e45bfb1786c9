#!/usr/bin/env python3
"""Builds vkzg_amd/libvkzg.so for gfx950 with hipcc (no cmake needed).

Each HIP translation unit compiles in parallel; the mainnet setup is linked
in through embed_setup.S.  Run:  python3 vkzg_amd/build.py [-j N]
"""
import argparse
import concurrent.futures as cf
import os
import struct
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
OUT_DIR = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libvkzg.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("VKZG_AMD_ARCH", "gfx950")

SOURCES = ["setup.hip", "setup_fft.hip", "setup_tables.hip", "fk20_scalars.hip", "phase_a.hip",
           "ladder.hip", "phase_b.hip", "reduce.hip", "recover.hip", "copy.hip", "msm.hip", "pairing.hip",
           "verify.hip", "prover.cpp", "noalloc.cpp", "server.cpp", "verify.cpp", "tables_v1.cpp", "sha256.cc"]
HOST_FLAGS = ["-O3", "-fPIC", "-std=c++17", "-Wall"]  # plain host C++ (.cc): g++
HIP_FLAGS = [
    "--offload-arch=" + ARCH,
    "-O3",
    "-fPIC",
    "-std=c++17",
    "-Wall",
    "-Wno-unused-function",
    # Packed FP32 instructions are kept out of every device code object.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I" + os.path.join(REPO, "include"),
]


def run(cmd):
    r = subprocess.run(cmd, capture_output=True, text=True)
    out = "\n".join(line for line in (r.stdout + r.stderr).splitlines()
                    if "packed-fp32-ops" not in line and "is not a recognized feature" not in line)
    if r.returncode != 0:
        raise RuntimeError("command failed: %s\n%s" % (" ".join(cmd), out))
    return out


def compile_one(src):
    obj = os.path.join(OUT_DIR, os.path.basename(src) + ".o")
    if src.endswith(".cc"):
        run(["g++"] + HOST_FLAGS + ["-c", os.path.join(CSRC, src), "-o", obj])
        return obj
    cmd = [HIPCC] + HIP_FLAGS + ["-c", os.path.join(CSRC, src), "-o", obj]
    if src.endswith(".cpp"):
        cmd.insert(1, "-x")
        cmd.insert(2, "hip")
    run(cmd)
    return obj


# A branch of the device's instruction set reaches +-32767 words.  In a function
# past that the compiler goes through a register pair for a far branch, and may
# take the one that holds the return address of a function that saves none: the
# function then returns into itself.  Kernels do not return and may be longer.
BRANCH_REACH = 32767 * 4


def device_functions(lib):
    """{name: bytes} of the functions in the library's device code that are not kernels."""
    data = open(lib, "rb").read()
    out = {}
    at = data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + 24)
        entry = at + 32
        for _ in range(n):
            off, size, name = struct.unpack_from("<QQQ", data, entry)
            triple = data[entry + 24:entry + 24 + name]
            entry += 24 + name
            if triple.startswith(b"hip") and size:
                out.update(_functions(data[at + off:at + off + size]))
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)
    return out


def _functions(elf):
    """{name: bytes} of an ELF64 code object's functions without a kernel descriptor (name.kd)."""
    shoff, = struct.unpack_from("<Q", elf, 40)
    shentsize, shnum = struct.unpack_from("<HH", elf, 58)
    sections = [struct.unpack_from("<IIQQQQIIQQ", elf, shoff + k * shentsize) for k in range(shnum)]
    functions, kernels = {}, set()
    for kind, offset, size, link in [(s[1], s[4], s[5], s[6]) for s in sections]:
        if kind != 2:  # SHT_SYMTAB
            continue
        names = sections[link][4]
        for at in range(offset, offset + size, 24):
            name, info, _, shndx, _, bytes_ = struct.unpack_from("<IBBHQQ", elf, at)
            text = elf[names + name:elf.index(b"\0", names + name)].decode()
            if text.endswith(".kd"):
                kernels.add(text[:-3])
            elif info & 15 == 2 and shndx:  # STT_FUNC, defined
                functions[text] = bytes_
    return {f: b for f, b in functions.items() if f not in kernels}


def check_device_functions(lib, limit=BRANCH_REACH):
    far = sorted("%s (%d bytes)" % (f, b) for f, b in device_functions(lib).items() if b > limit)
    if far:
        raise RuntimeError("device functions longer than a branch reaches: " + ", ".join(far))


def build(jobs=8, verbose=True):
    os.makedirs(OUT_DIR, exist_ok=True)
    setup_file = os.path.join(HERE, "data", "g1_monomial_mainnet.bin")
    embed_obj = os.path.join(OUT_DIR, "embed_setup.o")
    run(["gcc", "-c", os.path.join(CSRC, "embed_setup.S"), "-o", embed_obj,
         '-DVKZG_SETUP_FILE="%s"' % setup_file])
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(compile_one, SOURCES))
    tmp = LIB + ".tmp"
    # Export only the C ABI (vkzg_* and vkzg_amd_*): a version script, so the
    # extern "C" functions keep default visibility in the objects.
    run([HIPCC, "--offload-arch=" + ARCH, "-shared", "-fPIC", "-o", tmp] + objs + [embed_obj] +
        ["-Wl,--version-script=" + os.path.join(CSRC, "exports.map")])
    check_device_functions(tmp)
    os.replace(tmp, LIB)
    if verbose:
        print("built", LIB)
    return LIB


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("-j", type=int, default=8)
    a = ap.parse_args()
    try:
        build(a.j)
    except RuntimeError as e:
        print(e, file=sys.stderr)
        sys.exit(1)
