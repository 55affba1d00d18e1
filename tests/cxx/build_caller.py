"""Build recipe of the C++ test programs (run by __graft_entry__.build()).

mwg_caller: a program that includes include/mwgreen.hpp and links
mrchem_amd/libmwgreen.so, the way a C++ code such as MRChem would.
band_table.so: calls of the library's own device interface
(mrchem_amd/csrc/mw_device.hpp) for tests/test_gpu_band_table.py.
The rpath finds the library relative to the program, so the built tree can
move.
"""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))


def _build(name, out, *flags):
    src = os.path.join(HERE, name)
    out = os.path.join(HERE, out)
    cmd = (["g++", "-O2", "-std=c++17", "-Wall", "-Wextra"] + list(flags) +
           [src, "-o", out + ".tmp", "-L" + os.path.join(ROOT, "mrchem_amd"), "-lmwgreen",
            "-Wl,-rpath,$ORIGIN/../../mrchem_amd"])
    print("+", " ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    os.replace(out + ".tmp", out)
    return out


def build():
    _build("band_table.cpp", "band_table.so", "-shared", "-fPIC",
           "-I" + os.path.join(ROOT, "mrchem_amd", "csrc"))
    return _build("mwg_caller.cpp", "mwg_caller", "-I" + os.path.join(ROOT, "include"))


if __name__ == "__main__":
    build()
