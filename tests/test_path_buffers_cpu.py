"""The wavefront engine's path-state memory and chunks on the CPU (tests/hipcpu), under AddressSanitizer, with allocations
that fail."""
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "hipcpu"))

import hipcpu_build  # noqa: E402


def test_path_memory_after_failed_allocations(tmp_path):
    (tmp_path / "internal.h").write_text(hipcpu_build.internal_header())
    for header in ("path_buffers.h", "chunks.h"):
        shutil.copy(os.path.join(hipcpu_build.SRC, header), tmp_path)  # next to that internal.h
    exe = str(tmp_path / "path_buffers")
    subprocess.run(["g++", "-std=c++20", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=undefined", "-pthread", f"-I{tmp_path}",
                    f"-I{os.path.join(HERE, 'hipcpu')}", f"-I{os.path.join(hipcpu_build.ROOT, 'include')}",
                    os.path.join(HERE, "hipcpu", "path_buffers_main.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-3000:]
