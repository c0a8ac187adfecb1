"""Build libsvox_hip.so for gfx950 with hipcc, in-tree (next to the sources): one object for the entry points and one
per policy of the march kernels, compiled side by side and linked."""
import os
import shutil
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_NAME = "libsvox_hip.so"

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
    yield "svox_hip", "svox_hip.hip", []


def _run(cmd):
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    log = "\n".join(l for l in proc.stdout.splitlines() if "packed-fp32-ops" not in l)
    if proc.returncode != 0:
        raise RuntimeError("hipcc failed: " + " ".join(cmd) + "\n" + log)
    return log


def build_library(verbose=True):
    """Compile the HIP sources into svox_amd/csrc/libsvox_hip.so.  Raises on failure."""
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
        with ThreadPoolExecutor(max_workers=workers) as pool:
            made = list(pool.map(compile_unit, list(_units())))
        for _, log in made:
            if verbose and log.strip():
                print(log)
        _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", out + ".tmp"] + [obj for obj, _ in made])
    os.replace(out + ".tmp", out)
    return out


if __name__ == "__main__":
    build_library()
    sys.exit(0)
