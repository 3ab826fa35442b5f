"""Build of the native libraries (no cmake/ninja: hipcc and gcc directly).

    python -m cpvulkan_amd.build            # everything
    python -m cpvulkan_amd.build libcpv     # one target (libcpv, oracle, icd, programs)

Products (git-ignored, built in-tree so they travel with the source tree):
    cpvulkan_amd/lib/libcpv.so              HIP draw path + C-ABI (include/cpv.h)
    cpvulkan_amd/lib/libcpvulkan_amd_icd.so Vulkan ICD front end
    oracle/build/libcpvref.so               CPU oracle (test infrastructure)
    cpvulkan_amd/lib/rtc_cache/             code objects of the precompiled SPIR-V programs
"""
from __future__ import annotations

import concurrent.futures
import os
import subprocess
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent
PKG = ROOT / "cpvulkan_amd"
CSRC = PKG / "csrc"
LIB = PKG / "lib"
ORACLE = ROOT / "oracle"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

# Strict IEEE fp32: no contraction, correctly rounded divide/sqrt, denormals
# kept, and packed-fp32 instructions disabled.
HIP_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-ffp-contract=off", "-fno-fast-math",
    "-fhip-fp32-correctly-rounded-divide-sqrt", "-fno-gpu-flush-denormals-to-zero",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
    f"-I{ROOT / 'include'}", f"-I{CSRC}",
]
HOST_FLAGS = ["-O2", "-std=c++17", "-fPIC", "-ffp-contract=off", "-fno-fast-math", f"-I{ROOT / 'include'}", f"-I{CSRC}"]


def _run(cmd: list[str]) -> None:
    res = subprocess.run(cmd, cwd=ROOT, capture_output=True, text=True)
    if res.returncode != 0:
        sys.stderr.write(res.stdout + res.stderr)
        raise RuntimeError(f"build step failed: {' '.join(cmd[:3])} ... (exit {res.returncode})")


def _obj(src: Path, out_dir: Path, hip: bool, defines: tuple = (), tag: str = "") -> Path:
    out_dir.mkdir(parents=True, exist_ok=True)
    obj = out_dir / (src.name + tag + ".o")
    if hip:
        _run([HIPCC, *HIP_FLAGS, *[f"-D{d}" for d in defines], "-c", str(src), "-o", str(obj)])
    else:
        _run([HIPCC, *HOST_FLAGS, "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-x", "c++", "-c", str(src), "-o", str(obj)])
    return obj


# Kernel headers a translated SPIR-V program is compiled against (hiprtc has
# no file system access to the source tree, so the library carries them).
RTC_HEADERS = ["cpv_types.h", "index_math.h", "raster_device.h", "raster_kernels.h", "raster_tile.h"]


def write_embedded_headers(out: Path) -> Path:
    """A C++ source holding the kernel headers as string literals."""
    delim = "CPVRTC"
    parts = ["// Generated by cpvulkan_amd/build.py: kernel headers for hiprtc.",
             f"extern const int cpv_rtc_header_count = {len(RTC_HEADERS)};",
             "extern const char* const cpv_rtc_header_names[] = {" + ", ".join(f'"{h}"' for h in RTC_HEADERS) + "};",
             "extern const char* const cpv_rtc_header_sources[] = {"]
    for h in RTC_HEADERS:
        text = (CSRC / h).read_text()
        if f"){delim}\"" in text:
            raise RuntimeError(f"{h} contains the raw-string delimiter")
        parts.append(f'R"{delim}({text}){delim}",')
    parts.append("};")
    out.parent.mkdir(parents=True, exist_ok=True)
    new = "\n".join(parts) + "\n"
    if not out.exists() or out.read_text() != new:
        out.write_text(new)
    return out


BUILTIN_FRAGMENT_SHADERS = ["FsColor", "FsTexLambert", "FsColorDiscard", "FsColorFlat", "FsColorNoPerspective"]


def build_libcpv() -> Path:
    objdir = PKG / "_build" / "libcpv"
    emb = write_embedded_headers(objdir / "rtc_headers.cpp")
    srcs = [(CSRC / "cpv_runtime.hip", True, (), ""), (CSRC / "cpv_launch.hip", True, (), ""),
            (CSRC / "cpv_mlp.hip", True, (), ""), (CSRC / "cpv_transfer.hip", True, (), ""),
            (CSRC / "spirv_compile.cpp", False, (), ""), (emb, False, (), "")]
    # the raster kernels of each built-in fragment shader in a unit of their own
    for fs in BUILTIN_FRAGMENT_SHADERS:
        srcs.append((CSRC / "raster_instances.hip", True, (f"CPV_RASTER_FS={fs}",), "." + fs))
    with concurrent.futures.ThreadPoolExecutor(max_workers=min(len(srcs), os.cpu_count() or 8)) as ex:
        objs = list(ex.map(lambda s: _obj(s[0], objdir, s[1], s[2], s[3]), srcs))
    LIB.mkdir(parents=True, exist_ok=True)
    out = LIB / "libcpv.so"
    tmp = LIB / "libcpv.so.tmp"
    _run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs), "-lhiprtc"])
    os.replace(tmp, out)
    return out


def build_oracle() -> Path:
    out_dir = ORACLE / "build"
    out_dir.mkdir(parents=True, exist_ok=True)
    out = out_dir / "libcpvref.so"
    _run(["gcc", "-O2", "-std=c11", "-ffp-contract=off", "-fno-fast-math", "-fPIC", "-shared", "-fopenmp",
          "-Wall", "-o", str(out), str(ORACLE / "cpvref.c"), "-lm"])
    return out


# SPIR-V programs the tests and the benchmark create: translated and
# compiled once here so that their code objects sit in the in-tree program
# cache (cpvulkan_amd/lib/rtc_cache) that travels with the built library.
PRECOMPILED_PROGRAMS = [("vs_mvp_color", "fs_color"), ("vs_passthrough", "fs_color"),
                        ("vs_mvp_lambert", "fs_tex_lambert"), ("vs_passthrough", "fs_discard_dark"),
                        ("vs_flat_inputs", "fs_alu_ops"), ("vs_point_size", "fs_color"),
                        ("vs_passthrough", "fs_color_flat"), ("vs_passthrough", "fs_color_noperspective")]


def build_programs() -> None:
    """Compile the programs the workloads and tests use into the code-object
    cache next to the library (the cache is emptied first, so it holds no
    code objects of older kernel headers)."""
    lib_path = LIB / "libcpv.so"
    if not lib_path.exists():
        build_libcpv()
    cache = LIB / "rtc_cache"
    if cache.is_dir():
        for p in cache.iterdir():
            if p.suffix in (".co", ".names"):
                p.unlink()
    # one process per program: hiprtc compiles of one process run one at a time
    with concurrent.futures.ThreadPoolExecutor(max_workers=min(len(PRECOMPILED_PROGRAMS), os.cpu_count() or 8)) as ex:
        list(ex.map(_build_program, PRECOMPILED_PROGRAMS))


def _build_program(pair: tuple) -> None:
    code = ("import sys; sys.path.insert(0, %r); import cpvulkan_amd; from cpvulkan_amd import spirv as S; "
            "cpvulkan_amd.spirv_build(S.SHADERS[%r](), S.SHADERS[%r]())") % (str(ROOT), pair[0], pair[1])
    _run([sys.executable, "-c", code])


def build_icd() -> Path:
    """The Vulkan ICD (C++ on the C-ABI, linked against libcpv.so) and the
    test application that drives it through vk_icdGetInstanceProcAddr."""
    LIB.mkdir(parents=True, exist_ok=True)
    out = LIB / "libcpvulkan_amd_icd.so"
    tmp = LIB / "libcpvulkan_amd_icd.so.tmp"
    if not (LIB / "libcpv.so").exists():
        build_libcpv()
    _run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-fvisibility=hidden", f"-I{ROOT / 'include'}",
          "-o", str(tmp), str(CSRC / "icd" / "cpv_icd.cpp"), f"-L{LIB}", "-lcpv", "-Wl,-rpath,$ORIGIN"])
    os.replace(tmp, out)
    app_dir = ROOT / "tests" / "icd" / "build"
    app_dir.mkdir(parents=True, exist_ok=True)
    for app in ("icd_cube", "icd_transfer"):
        _run(["g++", "-O2", "-std=c++17", "-Wall", f"-I{ROOT / 'include'}", "-o", str(app_dir / app),
              str(ROOT / "tests" / "icd" / f"{app}.cpp"), "-ldl"])
    return out


TARGETS = {"libcpv": build_libcpv, "oracle": build_oracle}


def build_all(targets: list[str] | None = None) -> None:
    names = targets or list(TARGETS) + ["icd", "programs"]
    lib_targets = [n for n in names if n in TARGETS]
    with concurrent.futures.ThreadPoolExecutor(max_workers=max(len(lib_targets), 1)) as ex:
        for fut in [ex.submit(TARGETS[n]) for n in lib_targets]:
            fut.result()
    if "icd" in names:
        build_icd()
    if "programs" in names:
        build_programs()


if __name__ == "__main__":
    build_all(sys.argv[1:] or None)
