"""Build the CPU suite's programs with AddressSanitizer and
UndefinedBehaviorSanitizer.  Host code only: no GPU code is built with a
sanitizer.

tests/cpp/host_sanitize: the library's host sources (capi.cpp,
kernel_shims.cpp, pjrt.cpp, cblas_sgemm.cpp) and a driver compiled by g++,
linked with the library's compiled .hip objects (device code and launchers,
built by jules_amd/build.py into _build/, not sanitized) and the HIP runtime.

tests/cpp/host_launch: those sources, the host side of every .hip source
(launchers and kernel stubs, without device code) and a driver compiled by
ROCm's clang, linked with hip_stub.cpp in the place of the HIP runtime."""
import concurrent.futures as cf
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
CSRC = os.path.join(ROOT, "jules_amd", "csrc")
INCLUDE = os.path.join(ROOT, "include")
OBJDIR = os.path.join(ROOT, "_build")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
CLANG = f"{ROCM}/lib/llvm/bin/clang++"
BINARY = os.path.join(HERE, "host_sanitize")
LAUNCH_BINARY = os.path.join(HERE, "host_launch")
HOST_SOURCES = ["capi.cpp", "kernel_shims.cpp", "pjrt.cpp", "cblas_sgemm.cpp"]
SANITIZE = ["-fsanitize=address,undefined", "-fno-sanitize-recover=all", "-fno-omit-frame-pointer"]
CXXFLAGS = ["-O1", "-g", "-std=c++17", "-fPIC", "-Wall", f"-I{INCLUDE}", f"-I{CSRC}",
            "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include"]


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed:\n{' '.join(cmd)}\n{r.stdout}\n{r.stderr}")


def build(verbose=False):
    sys.path.insert(0, ROOT)
    from jules_amd import build as lib_build

    os.makedirs(OBJDIR, exist_ok=True)
    dev_objs = [os.path.join(OBJDIR, s + ".o") for s in lib_build.SOURCES if s.endswith(".hip")]
    missing = [o for o in dev_objs if not os.path.exists(o)]
    if missing:
        raise RuntimeError(f"library objects missing (run jules_amd/build.py first): {missing}")
    host = [os.path.join(CSRC, s) for s in HOST_SOURCES]
    hips = [os.path.join(CSRC, s) for s in lib_build.SOURCES if s.endswith(".hip")]
    cpp = [os.path.join(HERE, s) for s in ("host_launch.cpp", "hip_stub.cpp")]

    def gxx(src):
        obj = os.path.join(OBJDIR, "san_" + os.path.basename(src) + ".o")
        _run(["g++", *CXXFLAGS, *SANITIZE, "-c", src, "-o", obj], verbose)
        return obj

    def clang(src):
        obj = os.path.join(OBJDIR, "stub_" + os.path.basename(src) + ".o")
        hip = [f"--offload-arch={lib_build.ARCH}", "--cuda-host-only", "-fuse-cuid=none", "-Wno-unused-function", "-x", "hip"]
        _run([CLANG, *CXXFLAGS, *SANITIZE, *(hip if src.endswith(".hip") else []), "-c", src, "-o", obj], verbose)
        return obj

    def link(cxx, objs, libs, out):
        tmp = out + ".tmp"
        _run([cxx, *SANITIZE, *objs, *libs, "-o", tmp], verbose)
        os.replace(tmp, out)

    with cf.ThreadPoolExecutor(max_workers=8) as ex:
        san = ex.map(gxx, [*host, os.path.join(HERE, "host_sanitize.cpp")])
        stub = ex.map(clang, [*hips, *host, *cpp])
        san, stub = list(san), list(stub)
    link("g++", [*san, *dev_objs], [f"-L{ROCM}/lib", "-lamdhip64", f"-Wl,-rpath,{ROCM}/lib"], BINARY)
    # the objects share the name of the device code that they are without
    link(CLANG, stub, ["-Wl,--allow-multiple-definition", "-lpthread"], LAUNCH_BINARY)
    return BINARY


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
