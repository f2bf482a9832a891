"""Builds wide_main.cpp (both traversal walks on the CPU) and runs it on a scene's nodes and triangles. The device
headers use vector and address-space types, so the ROCm clang compiles them, for the host."""
import ctypes
import os
import shutil
import subprocess

import numpy as np

from photon_amd.types import HIT_DTYPE, RAY_DTYPE

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
SRC = os.path.join(ROOT, "photon_amd", "csrc", "hip")


def build(out_dir):
    text = open(os.path.join(SRC, "internal.h")).read()
    head, tail = text.split("// ---- render.hip")[0], text.split("// ---- wide_build.hip")[1].split("// Guide tables")[0]
    with open(os.path.join(out_dir, "internal.h"), "w") as f:
        f.write(head.replace('#include "dpath.h"', '#include "dwide.h"') + "//" + tail + "\n}  // namespace phk\n")
    shutil.copyfile(os.path.join(SRC, "wide_build.hip"), os.path.join(out_dir, "wide_build.cpp"))
    so = os.path.join(out_dir, "wide_cpu.so")
    clang = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "clang++")
    subprocess.run([clang, "-std=c++20", "-O2", "-mavx2", "-mfma", "-ffp-contract=off", "-fPIC", "-shared", "-fvisibility=hidden", "-pthread", "-Wall", "-Wno-unused-function",
                    f"-I{out_dir}", f"-I{HERE}", f"-I{SRC}", f"-I{os.path.join(ROOT, 'include')}", os.path.join(HERE, "wide_main.cpp"), "-o", so], check=True)
    return ctypes.CDLL(so)


def scene_arrays(scene):
    """(nodes, triangles) of a built scene as float32 rows of 16 and 12."""
    d = scene.desc()

    def rows(p, n, k):
        return np.frombuffer((ctypes.c_uint8 * (4 * k * n)).from_address(ctypes.addressof(p.contents)), np.float32).reshape(n, k).copy()

    return rows(d.nodes, d.num_nodes, 16), rows(d.tris, d.num_tris, 12)


def walk(lib, nodes, tris, rays, anyhit=False):
    """(whether there are wide nodes, binary hits, wide hits, traced again) of every ray."""
    rays = np.ascontiguousarray(rays, RAY_DTYPE)
    n = len(rays)
    hits, again = np.zeros((n, 2), HIT_DTYPE), np.zeros(n, np.int32)
    ptr = [ctypes.c_void_p(np.ascontiguousarray(a).ctypes.data) for a in (nodes, tris, rays, hits, again)]
    count = lib.walk_both(ptr[0], len(nodes), ptr[1], len(tris), ptr[2], n, int(anyhit), ptr[3], ptr[4])
    return count, hits[:, 0], hits[:, 1], again != 0
