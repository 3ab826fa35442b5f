"""A translated SPIR-V program compiles with the hiprtc that torch's wheel brings, which a process that has imported torch
has loaded and which may be older than the toolkit's (with that one the build compiles programs).  One raster kernel and
the vertex kernel, no GPU."""
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent

CODE = """
import ctypes as C, sys
sys.path.insert(0, {root!r})
import cpvulkan_amd
from cpvulkan_amd import build, spirv as S
src = cpvulkan_amd.spirv_translate(S.SHADERS["vs_passthrough"](), S.SHADERS["fs_color"]())
rtc = C.CDLL({lib!r})
names = [h.encode() for h in build.RTC_HEADERS]
texts = [(build.CSRC / h).read_bytes() for h in build.RTC_HEADERS]
prog = C.c_void_p()
n = len(names)
assert rtc.hiprtcCreateProgram(C.byref(prog), src.encode(), b"program.hip", n, (C.c_char_p * n)(*texts), (C.c_char_p * n)(*names)) == 0
for k in (b"cpv::vertex_kernel<cpv::SpvVs>", b"cpv::raster_kernel<cpv::SpvFs, 8, 1, false, true>"):
    assert rtc.hiprtcAddNameExpression(prog, k) == 0
opts = [b"--offload-arch=gfx950", b"-O1", b"-std=c++17", b"-ffp-contract=off", b"-Xclang", b"-target-feature", b"-Xclang", b"-packed-fp32-ops"]
rc = rtc.hiprtcCompileProgram(prog, len(opts), (C.c_char_p * len(opts))(*opts))
size = C.c_size_t()
rtc.hiprtcGetProgramLogSize(prog, C.byref(size))
log = C.create_string_buffer(size.value + 1)
rtc.hiprtcGetProgramLog(prog, log)
assert rc == 0, log.value.decode()[:2000]
"""


def test_program_compiles_with_the_wheels_hiprtc():
    torch = pytest.importorskip("torch")
    lib = Path(torch.__file__).parent / "lib" / "libhiprtc.so"
    if not lib.exists():
        pytest.skip("this torch brings no hiprtc")
    # a process of its own: a loaded hiprtc stays loaded
    r = subprocess.run([sys.executable, "-c", CODE.format(root=str(ROOT), lib=str(lib))], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
