"""Build recipe for the fastmat_amd HIP library (gfx950).

Compiles every ``csrc/*.hip`` source into ``fastmat_amd/libfastmat_amd.so``
with hipcc.  Packed-FP32 instruction selection is disabled for device code
(``-packed-fp32-ops``); the host pass of hipcc warns that it does not know the
feature, which is harmless.

Usage: ``python -m fastmat_amd.build`` (also called by ``__graft_entry__.build``).
"""
import glob
import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "libfastmat_amd.so")
ARCH = os.environ.get("FASTMAT_AMD_ARCH", "gfx950")


def hipcc():
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found")


def flags():
    return [
        "--offload-arch=" + ARCH,
        "-O3",
        "-std=c++17",
        "-fPIC",
        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
        "-Wno-unused-result",
        "-Wno-unused-command-line-argument",
        "-Wno-unused-value",
    ]


def build(verbose=False, jobs=8):
    # largest source first (fm_batch.hip compiles longest), a new one as one ends
    srcs = sorted(glob.glob(os.path.join(CSRC, "*.hip")), key=lambda s: (-os.path.getsize(s), s))
    objdir = os.path.join(HERE, "_build")
    os.makedirs(objdir, exist_ok=True)
    cc = hipcc()

    def compile_one(src):
        obj = os.path.join(objdir, os.path.basename(src) + ".o")
        cmd = [cc] + flags() + ["-c", src, "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        return obj, src, subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)

    with ThreadPoolExecutor(jobs) as pool:
        done = list(pool.map(compile_one, srcs))
    _check(done)
    tmp = OUT + ".tmp"
    cmd = [cc] + flags() + ["-shared", "-o", tmp] + sorted(obj for obj, _, _ in done)
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    os.replace(tmp, OUT)
    return OUT


def _check(done):
    errors = []
    for _, src, p in done:
        text = p.stdout.decode(errors="replace")
        # drop the host pass's notice about the device-only target feature
        lines = [l for l in text.splitlines() if "packed-fp32-ops" not in l
                 and "is not a recognized feature" not in l]
        if p.returncode != 0:
            errors.append("%s failed:\n%s" % (src, "\n".join(lines)))
        elif any(l.strip() for l in lines):
            sys.stderr.write("\n".join(lines) + "\n")
    if errors:
        raise RuntimeError("\n".join(errors))


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
