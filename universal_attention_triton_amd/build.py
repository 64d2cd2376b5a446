"""Builds libua_hip.so (gfx950, hipcc) and the host module _ua_host.so (g++) from csrc/.  `python -m universal_attention_triton_amd.build`."""
import concurrent.futures
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libua_hip.so")
HOST = os.path.join(HERE, "_ua_host.so")
UNITS = ["ua_capi", "ua_inst_fwd", "ua_inst_bwd", "ua_inst_bwd4", "ua_inst_aff"]
# packed-fp32 instructions are disabled for every device compile of this library
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fno-honor-nans", "-Wall", "-Wno-unused-function", "-Wno-unused-variable", "-Wno-unused-but-set-variable", "-Wno-unused-local-typedef", "-Wno-unused-value", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]


def source_hash():
    """Hash of everything the library is compiled from; the library reports the hash it was built with
    (ua_source_hash) and _lib.load refuses a library whose sources have changed since."""
    import hashlib
    h = hashlib.sha256()
    files = sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith((".hip", ".hpp", ".inc", ".cpp")))
    files.append(os.path.join(HERE, "..", "include", "ua.h"))
    for f in files:
        h.update(os.path.basename(f).encode())
        with open(f, "rb") as fh:
            h.update(fh.read())
    return h.hexdigest()[:16]


def _compile(unit, objdir, extra):
    src, obj = os.path.join(CSRC, unit + ".hip"), os.path.join(objdir, unit + ".o")
    cmd = ["hipcc", *FLAGS, *extra, "-c", src, "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    log = "\n".join(l for l in res.stderr.splitlines() if "not a recognized feature" not in l)
    if res.returncode != 0:
        raise RuntimeError("hipcc failed for %s:\n%s" % (unit, log))
    return obj, log


def _compile_host(objdir, tag):
    """The host module (plain C++ over torch's headers and the C ABI); linked once the library is."""
    import sysconfig
    import torch
    from torch.utils import cpp_extension
    obj = os.path.join(objdir, "ua_host.o")
    inc = [*cpp_extension.include_paths(), sysconfig.get_paths()["include"], "/opt/rocm/include"]
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-function", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           "-D_GLIBCXX_USE_CXX11_ABI=%d" % int(torch._C._GLIBCXX_USE_CXX11_ABI), *tag,
           *sum((["-isystem", i] for i in inc), []), "-c", os.path.join(CSRC, "ua_host.cpp"), "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("g++ failed for ua_host:\n" + res.stderr)
    return obj, res.stderr


def _link_host(obj):
    import torch
    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    res = subprocess.run(["g++", "-shared", "-o", HOST, obj, LIB, "-L" + lib, "-ltorch_python", "-ltorch_cpu", "-ltorch", "-lc10", "-lc10_hip",
                          "-Wl,-rpath,$ORIGIN"], capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("link of the host module failed:\n" + res.stderr)


def build(verbose=False, extra=()):
    objdir = os.path.join(HERE, "build")
    os.makedirs(objdir, exist_ok=True)
    tag = ['-DUA_SOURCE_HASH="%s"' % source_hash()]
    with concurrent.futures.ThreadPoolExecutor(max_workers=len(UNITS) + 1) as ex:
        host = ex.submit(_compile_host, objdir, tag)
        results = list(ex.map(lambda u: _compile(u, objdir, list(extra) + (tag if u == "ua_capi" else [])), UNITS))
    objs = [o for o, _ in results]
    res = subprocess.run(["hipcc", "--offload-arch=gfx950", "-shared", "-fPIC", "-Wl,-soname,libua_hip.so", "-o", LIB, *objs], capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("link failed:\n" + res.stderr)
    host_obj, host_log = host.result()
    _link_host(host_obj)
    for _, log in [*results, (None, host_log)]:      # compiler warnings are always shown: an uninitialised pointer on the host side faults the GPU
        if log.strip() and (verbose or "warning:" in log):
            print(log)
    return LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
