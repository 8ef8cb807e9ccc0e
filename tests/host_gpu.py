"""The library's host side over a HIP runtime on host memory
(host/fake_hip.cpp), for CPU tests of what the host does around launches:
`load()` gives the package bound to a library of its own, with the fake's
counters and limits on `.lib`.  No kernel runs."""
import ctypes
import importlib.util
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "herbert-metal-bf16_amd")
SOURCES = ["hb_runtime.cpp", "hb_emit.cpp", "hb_select.cpp", "hb_fill.cpp", "hb_checkpoint.cpp", "hb_moe.cpp"]


def build(out):
    """Compiles the host sources and the fake runtime into `out`/libherbert_hip.so."""
    sys.path.insert(0, PKG)
    try:
        import build as b
    finally:
        sys.path.remove(PKG)
    b.embed_sources(out_dir=out)
    flags = ["-O1", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-isystem", os.path.join(os.path.dirname(os.path.dirname(b.HIPCC)), "include"),
             "-I", b.CSRC, "-I", b.INCLUDE, "-I", out]
    srcs = [os.path.join(b.CSRC, s) for s in SOURCES] + [os.path.join(ROOT, "tests", "host", "fake_hip.cpp")]
    procs = [subprocess.Popen(["g++", *flags, "-c", s, "-o", os.path.join(out, "%d.o" % i)], stderr=subprocess.PIPE, text=True)
             for i, s in enumerate(srcs)]
    for s, p in zip(srcs, procs):
        err = p.communicate()[1]
        assert p.returncode == 0, (s, err)
    lib = os.path.join(out, "libherbert_hip.so")
    subprocess.run(["g++", "-shared", "-Wl,-Bsymbolic", "-Wl,-z,defs", "-o", lib, *(os.path.join(out, "%d.o" % i) for i in range(len(srcs))),
                    "-lpthread", "-ldl"], check=True)
    return lib


def load(out):
    """The package (herbert_hip/__init__.py) over the library built in `out`."""
    out = str(out)
    build(out)
    pkg = os.path.join(out, "herbert_hip")
    os.makedirs(pkg)
    with open(os.path.join(PKG, "herbert_hip", "__init__.py")) as f, open(os.path.join(pkg, "__init__.py"), "w") as g:
        g.write(f.read())
    spec = importlib.util.spec_from_file_location("herbert_hip_on_host", os.path.join(pkg, "__init__.py"))
    hb = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(hb)
    for name in ("fake_in_use", "fake_malloc_tries", "fake_launch_span"):
        getattr(hb.lib, name).restype = ctypes.c_uint64
    hb.lib.fake_limit.argtypes = hb.lib.fake_fail_reads.argtypes = [ctypes.c_uint64]
    hb.lib.fake_launch_name.restype = ctypes.c_char_p
    hb.lib.fake_launches.restype = hb.lib.fake_launch_rows.restype = ctypes.c_uint32
    return hb
