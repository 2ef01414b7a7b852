"""Build-time guard over this repository's own gfx950 code: compiles every
HIP source to AMD assembly and fails if any instruction writes through the
scalar data cache (scalar stores, scalar atomics, scalar cache write-back or
discard) or any packed-FP32 arithmetic appears.  Runs in build() on the
build host only.

usage: python check_isa.py [libpetar_hip.so]   (the argument is informational)
"""
import os
import re
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
SOURCES = ["pth_kernels.hip", "pth_gtree.hip", "pth_noalloc.hip"]
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fno-slp-vectorize", "-Xclang", "-target-feature",
         "-Xclang", "-packed-fp32-ops", "-S", "--cuda-device-only", "-o", "-"]
# by class, not by name: scalar instructions that are stores or atomics or write
# the scalar cache back or discard it, and packed FP32 arithmetic
INSTRUCTION = re.compile(r"^\s+([sv]_\w+)", re.M)
SCALAR_WRITE = re.compile(r"^s_(\w*_)?(store|atomic|wb|discard)(_|$)")
PACKED_FP32 = re.compile(r"^v_pk_(add|mul|fma)_f32")


def forbidden(asm):
    """The forbidden instructions of an assembly listing."""
    ins = set(INSTRUCTION.findall(asm))
    return sorted(i for i in ins if SCALAR_WRITE.match(i) or PACKED_FP32.match(i))


def main():
    bad = []
    for src in SOURCES:
        asm = subprocess.run(["/opt/rocm/bin/hipcc"] + FLAGS + [os.path.join(HERE, src)], capture_output=True,
                             text=True, check=True).stdout
        hits = forbidden(asm)
        if hits:
            bad.append((src, hits))
        print(f"check_isa: {src}: {len(INSTRUCTION.findall(asm))} instructions scanned, forbidden forms: {hits or 'none'}")
    if bad:
        sys.exit(f"check_isa: forbidden instructions in {bad}")


if __name__ == "__main__":
    main()
