"""The staged download (csrc/download.cpp) on the CPU, against host memory in place of the GPU:
whole fields, one pinned ring per device that is given back, contexts of another device than
the current one, threads, failing copies (download_host.cpp)."""
import os
import subprocess

from imogen_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


def test_download_host(tmp_path):
    objs = []
    for src in (os.path.join(build.CSRC, "download.cpp"), os.path.join(HERE, "download_host.cpp")):
        objs.append(str(tmp_path / (os.path.basename(src) + ".o")))
        subprocess.run([build.HIPCC, "-x", "hip", "--cuda-host-only", "-O1", "-fPIC", "-std=c++17", "-w",
                        "-I" + build.CSRC, "-I" + os.path.join(HERE, "..", "include"), "-c", src,
                        "-o", objs[-1]], check=True)
    exe = str(tmp_path / "download_host")
    subprocess.run(["g++", "-o", exe] + objs + ["-lpthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
