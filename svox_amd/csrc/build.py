"""Build libsvox_hip.so for gfx950 with hipcc, in-tree (next to the sources): one object for the entry points and one
per policy of the march kernels, compiled side by side and linked; and, beside them, the host extension _host_shim.so
(host_shim.cpp: plain C++ against torch's headers, no device code)."""
import os
import shutil
import subprocess
import sys
import sysconfig
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_NAME = "libsvox_hip.so"
SHIM_NAME = "_host_shim.so"

# -ffp-contract=off: the kernels spell their fused multiply-adds out; the compiler adds none.
# -munsafe-fp-atomics: floating-point atomicAdd becomes the hardware global_atomic_add.
# -packed-fp32-ops off: no packed fp32 instructions are generated from scalar code.
HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fvisibility=hidden",
    "-ffp-contract=off", "-munsafe-fp-atomics",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]

# (format, basis size) of every policy svox_hip.hip dispatches to (SVOX_DISPATCH_OCTREE); the longest compilations first
POLICIES = [("SH", 25), ("SG", 25), ("SH", 16), ("SG", 16), ("SH", 9), ("SG", 9), ("SH", 4), ("SG", 4), ("SH", 1), ("SG", 1),
            ("RGBA", 0)]


def library_path():
    return os.path.join(HERE, LIB_NAME)


def _units():
    """(name, source, extra flags) of every object."""
    for fmt, basis in POLICIES:
        yield (f"march_{fmt.lower()}{basis}", "march_policy.hip",
               [f"-DSVOX_POLICY_FORMAT=SVOX_FORMAT_{fmt}", f"-DSVOX_POLICY_BASIS={basis}"])
    yield "march_double", "march_double.hip", []
    yield "svox_hip", "svox_hip.hip", []


def _run(cmd):
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    log = "\n".join(l for l in proc.stdout.splitlines() if "packed-fp32-ops" not in l)
    if proc.returncode != 0:
        raise RuntimeError("build failed: " + " ".join(cmd) + "\n" + log)
    return log


def _shim_command(out):
    import torch
    root = os.path.dirname(torch.__file__)
    includes = [os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"),
                "/opt/rocm/include", sysconfig.get_paths()["include"]]
    libs = ["c10", "c10_hip", "torch_cpu", "torch_hip", "torch", "torch_python", "dl"]
    return (["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__",
             "-DTORCH_EXTENSION_NAME=" + SHIM_NAME[:-3], f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}"]
            + [f for i in includes for f in ("-isystem", i)] + [os.path.join(HERE, "host_shim.cpp"), "-o", out]
            + ["-L" + os.path.join(root, "lib")] + ["-l" + name for name in libs])


def build_library(verbose=True):
    """Compile the sources into svox_amd/csrc/libsvox_hip.so and _host_shim.so.  Raises on failure."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    out = library_path()
    with tempfile.TemporaryDirectory(prefix="svox_build_") as scratch:
        def compile_unit(unit):
            name, source, extra = unit
            obj = os.path.join(scratch, name + ".o")
            return obj, _run([hipcc] + HIPCC_FLAGS + extra + ["-c", "-o", obj, os.path.join(HERE, source)])

        if verbose:
            print(" ".join([hipcc] + HIPCC_FLAGS), "-c: one object per policy of the march kernels", flush=True)
        workers = int(os.environ.get("MAX_JOBS", 0)) or min(8, os.cpu_count() or 1)
        shim = os.path.join(HERE, SHIM_NAME)
        with ThreadPoolExecutor(max_workers=workers) as pool:
            host = pool.submit(_run, _shim_command(shim + ".tmp"))
            made = list(pool.map(compile_unit, list(_units())))
            log = host.result()
        if verbose and log.strip():
            print(log)
        for _, log in made:
            if verbose and log.strip():
                print(log)
        _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", out + ".tmp"] + [obj for obj, _ in made])
    os.replace(out + ".tmp", out)
    os.replace(shim + ".tmp", shim)
    return out


if __name__ == "__main__":
    build_library()
    sys.exit(0)
