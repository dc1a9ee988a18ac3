"""Builds librefrakt_amd.so (HIP kernels for gfx950 + host library) in-tree.

Run as ``python -m refrakt_amd.build`` or through ``__graft_entry__.build()``.
"""
import concurrent.futures
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "librefrakt_amd.so")
SOURCES = ["rf_k_compat.hip", "rf_k_fast.hip", "rf_k_misc.hip", "rf_host.cpp", "rf_stage.cpp", "rf_flam3.cpp", "rf_output.cpp",
           "rf_k_batch.hip", "rf_batch.cpp", "rf_k_nn.hip", "rf_denoiser.cpp", "rf_k_sort.hip", "rf_jit.cpp"]
# Device headers of the fast engine's kernel body, embedded in the library so
# that flame programs (rf_jit.cpp) can be compiled at run time with hiprtc;
# the names are those of the #include lines.
JIT_HEADERS = ["rf_device.hpp", "rf_sort.hpp", "rf_internal.hpp", "rf_kern_common.hpp", "rf_k_fast_body.hpp",
               "rf_batch.hpp", "rf_k_batch_body.hpp", "gen/variation_cases.inc"]
ARCH = os.environ.get("RF_OFFLOAD_ARCH", "gfx950")

HIP_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    # determinism: no implicit contraction; fmaf is written where the reference uses fma
    "-ffp-contract=off",
    # division and sqrt within the ~2.5 ulp GLSL allows; the few results that
    # must match the CPU bit for bit call the correctly rounded forms explicitly
    "-fno-hip-fp32-correctly-rounded-divide-sqrt",
    # packed FP32 ops are kept out of the generated code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # host functions start on cache lines: the weight initialisation's
    # std::normal_distribution takes 47 ms on one and 81 ms, in the same
    # instructions, where linking left it 48 bytes behind one
    "-Xarch_host", "-falign-functions=64",
    "-Wno-unused-command-line-argument",
]


def _run(cmd, cwd=None):
    r = subprocess.run(cmd, cwd=cwd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in r.stdout.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"command failed ({r.returncode}): {' '.join(cmd)}\n{out}")
    return out


def generate():
    try:
        import yaml  # noqa: F401
    except ImportError:
        return  # generated files are committed
    sys.path.insert(0, HERE)
    try:
        import gen_variations
        gen_variations.main([])
    finally:
        sys.path.pop(0)


def generate_jit_headers():
    out = ["// Generated by refrakt_amd/build.py: device headers embedded for hiprtc.\n",
           "static const char* const k_jit_headers[][2] = {\n"]
    for name in JIT_HEADERS:
        with open(os.path.join(CSRC, name)) as f:
            text = f.read()
        if ')RFJIT"' in text:
            raise RuntimeError(f"{name} contains the raw-string delimiter")
        out.append(f'  {{"{name}", R"RFJIT({text})RFJIT"}},\n')
    out.append("};\n")
    path = os.path.join(CSRC, "gen", "jit_headers.inc")
    body = "".join(out)
    if not os.path.exists(path) or open(path).read() != body:
        with open(path, "w") as f:
            f.write(body)


def build(verbose=False):
    generate()
    generate_jit_headers()
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    build_dir = os.path.join(HERE, "_build")
    os.makedirs(build_dir, exist_ok=True)
    jobs = []
    for src in SOURCES:
        obj = os.path.join(build_dir, src.rsplit(".", 1)[0] + ".o")
        jobs.append(([hipcc] + HIP_FLAGS + ["-c", os.path.join(CSRC, src), "-o", obj], obj))
    with concurrent.futures.ThreadPoolExecutor(max_workers=min(len(jobs), os.cpu_count() or 4)) as ex:
        outs = list(ex.map(lambda j: _run(j[0]), jobs))
    if verbose:
        for o in outs:
            if o.strip():
                print(o)
    objs = [j[1] for j in jobs]
    tmp = LIB + ".tmp"
    _run([hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp] + objs + ["-lz", "-lhiprtc"])
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
