"""wide_tile.hpp as the compiler takes it (hipcc cross-compiles the kernel; nothing runs)."""
import importlib.util
import pathlib
import re
import subprocess

import pytest

CSRC = pathlib.Path(__file__).resolve().parents[1] / "comfyui-drama3_amd" / "csrc"

KERNEL = """
#include "wide_tile.hpp"
__global__ void k(const void* base, int v) {
  __shared__ uint8_t lds[4096];
  asm volatile("; first use of %0" ::"{m0}"(v));
  d3::dma16(d3::lds_address(lds), base, 16 * threadIdx.x);
  asm volatile("; second use of %0" ::"{m0}"(v));
  d3::dma_wait();
}
"""


def _build():
    spec = importlib.util.spec_from_file_location("csrc_build", CSRC / "build.py")
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


def test_dma16_tells_the_compiler_that_it_writes_m0(tmp_path):
    """A value that the compiler keeps in m0 on both sides of a copy to LDS, whose LDS address the copy puts there: m0
    is set again before the second use."""
    build = _build()
    if not build.HIPCC.exists():
        pytest.skip("no hipcc")
    src, out = tmp_path / "k.hip", tmp_path / "k.s"
    src.write_text(KERNEL)
    subprocess.run([str(build.HIPCC), *build.FLAGS, f"-I{CSRC}", "--cuda-device-only", "-S", str(src), "-o", str(out)],
                   check=True, capture_output=True)
    text = out.read_text()
    copy, second = text.index("global_load_lds_dwordx4"), text.index("; second use of m0")
    assert text.index("; first use of m0") < copy < second
    assert re.search(r"s_mov_b32 m0, s\d+", text[copy:second])
