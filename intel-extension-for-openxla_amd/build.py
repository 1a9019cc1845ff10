"""Builds libxmk.so (the C-ABI kernel library) for gfx950 with hipcc and _xmk_native.so (its torch binding)
with the host compiler, in-tree.

Usage: python build.py [-j N] [--force]   (without --force: incremental)
Each translation unit under csrc/ is compiled to an object file and the objects
are linked into one shared library next to this file.
"""
import concurrent.futures
import importlib.metadata
import importlib.util
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")
OBJ = os.path.join(HERE, "build")
LIB = os.path.join(HERE, "libxmk.so")
NATIVE_SRC = os.path.join(CSRC, "python", "native.cc")
NATIVE = os.path.join(HERE, "_xmk_native.so")
NATIVE_STAMP = os.path.join(OBJ, "native.stamp")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-I", INCLUDE, "-I", CSRC,
         # packed-fp32 VALU forms are kept out of generated code on purpose
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "-Wall", "-Wno-unused-function", "-Wno-unknown-attributes"] + os.environ.get("XMK_CXXFLAGS", "").split()


# Per-file flags.  Attention forward: matrix instructions write VGPRs, so that the softmax reads the
# scores where they were produced (the whole register budget is then one file of 256 per wave).
EXTRA = {f: ["-mllvm", "-amdgpu-mfma-vgpr-form"] for f in ("fmha_fwd.hip", "fmha_fwd_h48.hip", "fmha_fwd_h80.hip", "fmha_fwd_h96.hip", "fmha_fwd_h160.hip", "fmha_short.hip", "int4_tile.hip")}


def sources():
    return sorted(f for f in os.listdir(CSRC) if f.endswith((".hip", ".cc")))


def _deps_mtime():
    hdrs = [os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".h")]
    hdrs += [os.path.join(INCLUDE, f) for f in os.listdir(INCLUDE)]
    return max(os.path.getmtime(h) for h in hdrs)


def _compile(args):
    src, force = args
    obj = os.path.join(OBJ, os.path.splitext(src)[0] + ".o")
    spath = os.path.join(CSRC, src)
    if (not force and os.path.exists(obj)
            and os.path.getmtime(obj) > max(os.path.getmtime(spath), _deps_mtime())):
        return src, obj, 0, ""
    cmd = [HIPCC] + FLAGS + EXTRA.get(src, []) + (["-x", "hip"] if src.endswith(".cc") else []) + \
          ["-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    out = "\n".join(l for l in (r.stdout + r.stderr).splitlines()
                    if "packed-fp32-ops" not in l and l.strip())
    return src, obj, r.returncode, out


def _native_command():
    t = os.path.dirname(importlib.util.find_spec("torch").origin)
    return [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__",
            "-DUSE_ROCM", "-I", INCLUDE, "-isystem", "/opt/rocm/include", "-isystem", os.path.join(t, "include"),
            "-isystem", sysconfig.get_paths()["include"], NATIVE_SRC, "-o", NATIVE, "-L", os.path.join(t, "lib"),
            "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip"]


def _compile_native(force):
    """The host-only module between torch tensors and the C ABI.  It links to nothing of libxmk.so (bound by
    path when the package loads it).  Built for one Python and one torch, whose versions the stamp beside the
    object files holds: with others it is built again."""
    cmd = _native_command()
    stamp = "\n".join([sys.version, importlib.metadata.version("torch")] + cmd)
    if (not force and os.path.exists(NATIVE) and os.path.exists(NATIVE_STAMP) and open(NATIVE_STAMP).read() == stamp
            and os.path.getmtime(NATIVE) > max(os.path.getmtime(NATIVE_SRC), _deps_mtime())):
        return 0, ""
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode == 0:
        with open(NATIVE_STAMP, "w") as f:
            f.write(stamp)
    return r.returncode, r.stdout + r.stderr


def build(jobs=None, verbose=False, force=True):
    """force=False recompiles only sources newer than their object file."""
    os.makedirs(OBJ, exist_ok=True)
    jobs = jobs or min(8, os.cpu_count() or 1)
    objs = []
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as pool:
        native = pool.submit(_compile_native, force)
        for src, obj, rc, out in pool.map(_compile, [(s, force) for s in sources()]):
            if out and (verbose or rc != 0):
                print(f"--- {src}\n{out}", file=sys.stderr)
            if rc != 0:
                raise RuntimeError(f"hipcc failed on {src}")
            objs.append(obj)
        rc, out = native.result()
        if rc != 0:
            raise RuntimeError(f"the native binding does not compile:\n{out}")
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB] + objs
    subprocess.check_call(cmd)
    return LIB


if __name__ == "__main__":
    j = int(sys.argv[sys.argv.index("-j") + 1]) if "-j" in sys.argv else None
    print(build(j, verbose=True, force="--force" in sys.argv))
