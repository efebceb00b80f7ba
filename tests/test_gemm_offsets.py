"""The addresses of the GEMM's stage DMAs (csrc/gemm_offsets.hpp), evaluated by the host compiler.

Everything is a static_assert over constexpr functions, so a wrong value, a read in range that
should be out of it, or a signed overflow stops the compilation."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "slang_amd", "csrc")


def holds(tmp_path, body):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    src = tmp_path / "offsets.cpp"
    src.write_text('#include <initializer_list>\n#include "gemm_offsets.hpp"\nusing namespace g4a;\n' + body)
    p = subprocess.run([cxx, "-std=c++17", "-fsyntax-only", f"-I{CSRC}", str(src)], capture_output=True, text=True)
    assert p.returncode == 0, p.stderr


def test_dma_past_the_range_reads_nothing(tmp_path):
    """A raw buffer load is out of range where its vector offset reaches the resource's bytes;
    descriptions differ in whether the scalar offset counts, and on which side. Past the last
    k-stage no description may let an address through; before it every one must."""
    holds(tmp_path, """
constexpr bool reads(StageDma d, uint32_t voff) {
    return voff < d.records || voff < d.records - d.soff || (uint64_t)voff + d.soff < d.records;
}
constexpr bool always_reads(StageDma d, uint32_t voff) {
    return voff < d.records && voff < d.records - d.soff && (uint64_t)voff + d.soff < d.records;
}
constexpr bool check() {
    for (uint32_t K : {64u, 192u, 1536u, 12288u})
        for (uint32_t rows : {1u, 65u, 2047u})
            for (uint32_t stage = 0; stage < K / 64 + 6; ++stage)
                for (uint32_t row : {0u, rows - 1, rows, rows + 255}) {
                    const bool more = stage < K / 64;
                    const StageDma d = stage_dma(rows * K * 2, (int)stage, more);
                    for (uint32_t c = 0; c < 128; c += 16) {
                        if (!more || row >= rows ? reads(d, row * K * 2 + c) : !always_reads(d, row * K * 2 + c)) return false;
                    }
                }
    return true;
}
static_assert(check(), "a DMA out of its matrix's k-stages");
""")
