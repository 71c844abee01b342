"""The library's HIP sources built against a runtime that records launches instead of running them
(record_runtime.cpp) -- TEST INFRASTRUCTURE ONLY.  recorder() returns that library through ctypes, built
into _build/ (not committed) when a source is newer; `ops(lib)` its log."""
import concurrent.futures as cf
import ctypes as C
import functools
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
CSRC = os.path.join(ROOT, "grassmanntn_amd", "csrc")
OUT = os.path.join(HERE, "_build", "libgtn_record.so")
CXX = "/opt/rocm/llvm/bin/clang++"
FLAGS = ["-std=c++20", "-O0", "-g1", "-fPIC", "-w", "-Wno-unused-result", "-I", os.path.join(HERE, "include")]


def build():
    srcs = [os.path.join(CSRC, f) for f in sorted(os.listdir(CSRC)) if f.endswith(".hip")]
    srcs.append(os.path.join(HERE, "record_runtime.cpp"))
    deps = srcs + [os.path.join(CSRC, "gtn_common.h"), os.path.join(ROOT, "include", "gtn_hip.h"),
                   os.path.join(HERE, "include", "hip", "hip_runtime.h")]
    if os.path.exists(OUT) and os.path.getmtime(OUT) > max(os.path.getmtime(d) for d in deps):
        return OUT
    os.makedirs(os.path.dirname(OUT), exist_ok=True)

    def compile_(src):
        obj = os.path.join(os.path.dirname(OUT), "rec_%d_%s.o" % (os.getpid(), os.path.basename(src)))
        subprocess.run([CXX] + FLAGS + ["-x", "c++", "-c", src, "-o", obj], check=True)
        return obj

    with cf.ThreadPoolExecutor(4) as ex:
        objs = list(ex.map(compile_, srcs))
    tmp = "%s.%d" % (OUT, os.getpid())
    subprocess.run([CXX, "-shared", "-Wl,-Bsymbolic", "-o", tmp] + objs + ["-lpthread", "-ldl"], check=True)
    os.replace(tmp, OUT)
    for o in objs:
        os.remove(o)
    return OUT


@functools.lru_cache(maxsize=1)
def recorder():
    lib = C.CDLL(build())
    lib.rec_kernel.restype = C.c_char_p
    lib.rec_kernel.argtypes = [C.c_void_p]
    lib.rec_hold.argtypes = [C.c_void_p, C.c_char_p, C.c_int]
    lib.gtn_svd_workspace_bytes.restype = C.c_int64
    return lib


def ops(lib):
    """[(kind, stream, event, address or kernel, workgroups, lanes a workgroup)] since the last rec_reset."""
    out = []
    for i in range(lib.rec_count()):
        k, s, w, g, b = C.c_char(), C.c_void_p(), C.c_void_p(), C.c_ulonglong(), C.c_uint()
        lib.rec_op(i, C.byref(k), C.byref(s), C.byref(w), C.byref(g), C.byref(b))
        out.append((k.value.decode(), s.value, w.value, g.value, b.value))
    return out
