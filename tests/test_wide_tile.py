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


def _assembly(tmp_path, source):
    build = _build()
    if not build.HIPCC.exists():
        pytest.skip("no hipcc")
    src, out = tmp_path / "k.hip", tmp_path / "k.s"
    src.write_text(source)
    subprocess.run([str(build.HIPCC), *build.FLAGS, f"-I{CSRC}", "--cuda-device-only", "-S", str(src), "-o", str(out)],
                   check=True, capture_output=True)
    return out.read_text()


def test_dma16_tells_the_compiler_that_it_writes_m0(tmp_path):
    """A value that the compiler keeps in m0 on both sides of a copy to LDS, whose LDS address the copy puts there: m0
    is set again before the second use."""
    text = _assembly(tmp_path, KERNEL)
    copy, second = text.index("global_load_lds_dwordx4"), text.index("; second use of m0")
    assert text.index("; first use of m0") < copy < second
    assert re.search(r"s_mov_b32 m0, s\d+", text[copy:second])


BASE_IN_VECTOR_REGISTERS = """
#include "wide_tile.hpp"
__global__ void k(const char* const* bases, const int* lds_at) {
  __shared__ uint8_t lds[4096];
  const char* base = bases[threadIdx.x >> 6];
  d3::dma16(d3::lds_address(lds) + lds_at[threadIdx.x >> 6], base, 16 * (threadIdx.x & 63));
  d3::dma_wait();
}
"""


def _written(op):
    """The scalar registers that an instruction (its words) writes: its first operand's."""
    if len(op) < 2 or op[0] == "global_load_lds_dwordx4":
        return set()
    m = re.fullmatch(r"s\[(\d+):(\d+)\],?", op[1])
    return set(range(int(m[1]), int(m[2]) + 1)) if m else {int(op[1][1:].rstrip(","))} if re.fullmatch(
        r"s\d+,?", op[1]) else {"m0"} if op[1].rstrip(",") == "m0" else set()


def test_dma16_waits_for_scalar_registers_written_by_vector_instructions(tmp_path):
    """A base and an LDS address that come from vector registers: the base's two registers and m0, as the copy reads them,
    are written by scalar instructions or five wait states before (an instruction is one, s_nop n is n + 1)."""
    lines = [line.split(";")[0].split() for line in _assembly(tmp_path, BASE_IN_VECTOR_REGISTERS).splitlines()]
    ops = [line for line in lines if line and not line[0].startswith(".") and not line[0].endswith(":")]
    copy = next(i for i, op in enumerate(ops) if op[0] == "global_load_lds_dwordx4")
    assert sum(op[0] == "v_readfirstlane_b32" for op in ops[:copy]) >= 3
    first, last = map(int, re.fullmatch(r"s\[(\d+):(\d+)\]", ops[copy][2]).groups())
    for register in (first, last, "m0"):
        writer = max(i for i in range(copy) if register in _written(ops[i]))
        states = sum(int(op[1]) + 1 if op[0] == "s_nop" else 1 for op in ops[writer + 1:copy])
        assert states >= (5 if ops[writer][0].startswith("v_") else 1 if register == "m0" else 0)
