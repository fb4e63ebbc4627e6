"""Builds the HIP libraries for gfx950, in-tree.

    python -m loongforge_amd.csrc.build [--force]

libdsa_hip.so    the C-ABI library of kernels (include/dsa_hip.h): every csrc/*.hip
_dsa_host.so     the native host layer of loongforge_amd/ops.py (a torch extension): csrc/host/*.cpp
libdsa_bench.so  measurement aids that only the benchmark loads (include/dsa_hip_bench.h):
                 csrc/bench/*.hip plus the error-state object

hipcc cross-compiles without a GPU.  Objects and the shared libraries are written next to the
package (`loongforge_amd/*.so`) so that they travel with the source tree.
"""
import concurrent.futures
import glob
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.dirname(HERE)
LIB = os.path.join(PKG, "libdsa_hip.so")
BENCH_LIB = os.path.join(PKG, "libdsa_bench.so")
HOST_LIB = os.path.join(PKG, "_dsa_host.so")
OBJ_DIR = os.path.join(HERE, "build")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-fPIC", "-std=c++17", "-Wno-unused-result", "-Wno-unused-value",
    # packed fp32 VALU ops are kept out of the generated code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def _sources():
    return sorted(glob.glob(os.path.join(HERE, "*.hip")))


def _bench_sources():
    return sorted(glob.glob(os.path.join(HERE, "bench", "*.hip")))


def _deps():
    return (glob.glob(os.path.join(HERE, "*.h")) + glob.glob(os.path.join(os.path.dirname(PKG), "include", "*.h"))
            + [os.path.join(HERE, "mla_bwd.hip")])          # csrc/bench/bwd_profile.hip includes it


def _run_if_stale(cmd, obj, inputs, force, built_for=""):
    """Runs the compiler unless ``obj`` is newer than its inputs and came out of the same command (and of the same ``built_for``:
    what it depends on besides); returns the result or None."""
    made, record = "\n".join([built_for] + cmd), obj + ".cmd"
    if not force and os.path.exists(obj) and os.path.getmtime(obj) >= max(os.path.getmtime(p) for p in inputs):
        if os.path.exists(record) and open(record).read() == made:
            return None
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode == 0:
        with open(record, "w") as f:
            f.write(made)
    return res


def _compile(src, force):
    prefix = "bench_" if os.path.basename(os.path.dirname(src)) == "bench" else ""
    obj = os.path.join(OBJ_DIR, prefix + os.path.basename(src)[:-4] + ".o")
    res = _run_if_stale([HIPCC] + FLAGS + ["-c", src, "-o", obj], obj, [src] + _deps(), force)
    if res is None:
        return obj, ""
    log = "\n".join(l for l in (res.stdout + res.stderr).splitlines() if "not a recognized feature" not in l)
    if res.returncode != 0:
        raise RuntimeError("hipcc failed for %s:\n%s" % (src, log))
    return obj, log


def _compile_host(force):
    """csrc/host/host.cpp -> object file (host code only: g++).  An extension works with the torch it was compiled against."""
    import torch
    from torch.utils.cpp_extension import include_paths

    src, obj = os.path.join(HERE, "host", "host.cpp"), os.path.join(OBJ_DIR, "host.o")
    includes = include_paths() + ["/opt/rocm/include", sysconfig.get_paths()["include"]]
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__",
           "-DUSE_ROCM", "-DTORCH_API_INCLUDE_EXTENSION_H", "-DTORCH_EXTENSION_NAME=_dsa_host"]
    cmd += ["-I" + p for p in includes] + ["-c", src, "-o", obj]
    res = _run_if_stale(cmd, obj, [src, os.path.join(os.path.dirname(PKG), "include", "dsa_hip.h")], force,
                        "torch %s, python %s" % (torch.__version__, sys.version))
    if res is not None and res.returncode != 0:
        raise RuntimeError("compiling host.cpp failed:\n" + res.stdout + res.stderr)
    return obj


def _link_host(obj):
    from torch.utils.cpp_extension import library_paths

    libs = ["-l" + n for n in ("dsa_hip", "c10", "c10_hip", "torch", "torch_cpu", "torch_hip", "torch_python", "amdhip64")]
    res = subprocess.run([os.environ.get("CXX", "g++"), "-shared", "-o", HOST_LIB, obj, "-L" + PKG]
                         + ["-L" + p for p in library_paths()] + ["-L/opt/rocm/lib"] + libs + ["-Wl,-rpath,$ORIGIN"],
                         capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("link failed:\n" + res.stdout + res.stderr)


def build(force=False, verbose=True):
    os.makedirs(OBJ_DIR, exist_ok=True)
    srcs, bench_srcs = _sources(), _bench_sources()
    with concurrent.futures.ThreadPoolExecutor(max_workers=8) as ex:
        host = ex.submit(_compile_host, force)
        results = list(ex.map(lambda s: _compile(s, force), srcs + bench_srcs))
        host_obj = host.result()
    objs = [o for o, _ in results[:len(srcs)]]
    bench_objs = [o for o, _ in results[len(srcs):]] + [os.path.join(OBJ_DIR, "api.o")]
    for _, log in results:
        if verbose and log.strip():
            print(log)
    for lib, members in ((LIB, objs), (BENCH_LIB, bench_objs)):
        newest = max(os.path.getmtime(o) for o in members)
        if force or not os.path.exists(lib) or os.path.getmtime(lib) < newest:
            cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", lib] + members
            res = subprocess.run(cmd, capture_output=True, text=True)
            if res.returncode != 0:
                raise RuntimeError("link failed:\n" + res.stdout + res.stderr)
    if force or not os.path.exists(HOST_LIB) or os.path.getmtime(HOST_LIB) < max(os.path.getmtime(host_obj), os.path.getmtime(LIB)):
        _link_host(host_obj)
    return LIB


if __name__ == "__main__":
    print(build(force="--force" in sys.argv))
