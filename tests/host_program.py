"""Builds a small host program against the library's own objects, so that its
internal host rules (plans, dispatch) can be tested on the CPU."""

import os
import subprocess

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nova-wino-amd_amd")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def build(directory, source):
    """Compiles ``source`` (one translation unit that may include
    nova_internal.h) and returns a function from rows of integers, fed to its
    standard input, to the rows of integers it prints."""
    src, obj, exe = (os.path.join(str(directory), f) for f in ("rule.hip", "rule.o", "rule"))
    with open(src, "w") as f:
        f.write(source)
    build_dir = os.path.join(PKG, "_build")
    if not os.path.exists(os.path.join(PKG, "nova_winograd", "lib", "libnova_winograd.so")):
        subprocess.run(["make", "-C", PKG], check=True)
    if not os.path.isdir(build_dir):
        subprocess.run(["make", "-B", "-C", PKG], check=True)
    objs = [os.path.join(build_dir, f) for f in sorted(os.listdir(build_dir)) if f.endswith(".o")]
    subprocess.run([HIPCC, "-std=c++17", "--offload-host-only", "-I", os.path.join(PKG, "csrc"),
                    "-c", "-o", obj, src], check=True)
    subprocess.run([HIPCC, "-o", exe, obj, *objs, "-Wl,-rpath,/opt/rocm/lib"], check=True)

    def run(rows):
        text = "\n".join(" ".join(str(v) for v in r) for r in rows)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True)
        got = [tuple(int(v) for v in line.split()) for line in out.stdout.split("\n") if line]
        assert len(got) == len(rows)
        return got

    return run
