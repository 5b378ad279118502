"""Builds liblily_sampler_hip.so for gfx950 with hipcc (cross-compiles without a GPU).

    python lily-qwen3.8-flash-next_amd/build.py [--strict-handover]

--strict-handover builds liblily_sampler_hip_strict.so instead: the same library without the
relaxed form of the hand-over between the workgroups of a row (-DLILY_STRICT_HANDOVER, see
last_to_arrive() in csrc/device_common.h; the default build picks the form by the launch's size,
and LILY_SAMPLER_HANDOVER=strict picks the strict one at run time).  LILY_SAMPLER_LIBRARY=<path>
makes the Python mirror load it.

The row kernel is compiled once per (logits type, kernel kind) pair from rows_variant.hip, in
parallel; the objects are linked with the small kernels and the C-ABI layer.
"""
import concurrent.futures
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "build")
LIB = os.path.join(HERE, "liblily_sampler_hip.so")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    # Token ids depend on exact f32 arithmetic: no contraction into FMAs, IEEE division
    # (hipcc's default), denormals kept (hipcc's default).
    "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-command-line-argument",
]
VARIANTS = [(dt, kind) for dt in (0, 1) for kind in (0, 1, 2)]
NOISE = "is not a recognized feature for this target"


def units():
    """(source, object, extra flags) of every translation unit."""
    out = [("rows_variant.hip", f"rows_dt{dt}_kind{kind}.o", [f"-DLILY_DT={dt}", f"-DLILY_KIND={kind}"])
           for dt, kind in VARIANTS]
    out += [("rows_held.hip", f"rows_held_dt{dt}_blocks{nb}.o", [f"-DLILY_DT={dt}", f"-DLILY_BLOCKS={nb}"])
            for dt in (0, 1) for nb in (2, 1)]
    out += [("rows_blocks.hip", f"rows_blocks_dt{dt}.o", [f"-DLILY_DT={dt}"]) for dt in (0, 1)]
    out += [("rows_masked.hip", f"rows_masked_dt{dt}.o", [f"-DLILY_DT={dt}"]) for dt in (0, 1)]
    out.append(("scratch_kernels.hip", "scratch_kernels.o", []))
    out.append(("static_entry.hip", "static_entry.o", []))
    out.append(("lm_head.hip", "lm_head.o", []))
    out.append(("lm_head_codes.hip", "lm_head_codes.o", []))
    out.append(("lm_head_codes_rows.hip", "lm_head_codes_rows.o", []))
    out.append(("head_library.hip", "head_library.o", []))
    out.append(("rows_tiles.hip", "rows_tiles.o", []))
    out.append(("rows_wide.hip", "rows_wide.o", []))
    out.append(("rows_argmax.hip", "rows_argmax.o", []))
    out.append(("sampler_api.cpp", "sampler_api.o", []))
    return out


def _run(cmd):
    res = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in res.stderr.splitlines() if NOISE not in l)
    if res.returncode != 0:
        raise RuntimeError("hipcc failed: " + " ".join(cmd) + "\n" + err)
    return err


LIB_STRICT = os.path.join(HERE, "liblily_sampler_hip_strict.so")


def build(verbose=False, jobs=None, strict_handover=False):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    obj_dir = OBJ + ("_strict" if strict_handover else "")
    lib = LIB_STRICT if strict_handover else LIB
    flags = FLAGS + (["-DLILY_STRICT_HANDOVER"] if strict_handover else [])
    os.makedirs(obj_dir, exist_ok=True)
    jobs = jobs or min(8, os.cpu_count() or 1)
    cmds = [[hipcc] + flags + extra + ["-c", os.path.join(CSRC, src), "-o", os.path.join(obj_dir, obj)]
            for src, obj, extra in units()]
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as pool:
        for err in pool.map(_run, cmds):
            if verbose and err.strip():
                sys.stderr.write(err + "\n")
    objs = [os.path.join(obj_dir, obj) for _, obj, _ in units()]
    _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC"] + objs + ["-o", lib])
    if not strict_handover:
        build_harness(hipcc)
    return lib


HARNESS_SRC = os.path.join(os.path.dirname(HERE), "tests", "abi_harness", "harness.cpp")
HARNESS_BIN = os.path.join(os.path.dirname(HERE), "tests", "abi_harness", "harness.bin")


def build_harness(hipcc):
    """The C++ caller of the library that the tests run: host code only, written against the
    public header, linked against the library by a path relative to the binary."""
    if not os.path.exists(HARNESS_SRC):
        return None
    _run([hipcc, "-O1", "-std=c++17", "-Wall", "-Wno-unused-command-line-argument",
          "-I", os.path.join(os.path.dirname(HERE), "include"), HARNESS_SRC, "-o", HARNESS_BIN,
          "-L", HERE, "-llily_sampler_hip", "-Wl,-rpath,$ORIGIN/../../" + os.path.basename(HERE)])
    return HARNESS_BIN


if __name__ == "__main__":
    print(build(verbose=True, strict_handover="--strict-handover" in sys.argv[1:]))
