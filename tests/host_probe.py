"""Host builds of the library's headers for CPU tests: the device headers
leave OA_HD open, so a C++ probe can include them and run a rule or a formula
as the kernels do, without a GPU.  A probe may also call the host functions
that liboaxis.so exports (they stay unresolved in the probe and bind to the
loaded library)."""
import ctypes
import os
import subprocess

from oaxis import _abi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "ollinaxis-bib_amd", "csrc")


def build(folder, text, flags=("-O2", "-ffp-contract=off")):
    """Compile the C++ source text and load it."""
    src, out = os.path.join(str(folder), "probe.cpp"), os.path.join(str(folder), "probe.so")
    with open(src, "w") as f:
        f.write(text)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-w", *flags, "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-I" + CSRC, "-I" + os.path.join(ROOT, "include"), src, "-o", out],
                   check=True)
    ctypes.CDLL(_abi.LIBPATH, mode=ctypes.RTLD_GLOBAL)
    return ctypes.CDLL(out)
