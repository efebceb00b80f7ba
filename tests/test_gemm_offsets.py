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


def test_row_offsets_at_the_ends_of_what_is_accepted(tmp_path):
    """Rows of a tile past the matrix get offsets past its bytes: formed in 32 bits they neither
    overflow nor wrap back into it, for every tile height (tokens to 256; weight rows to 256, the
    gate/up form's outputs to 128) and the largest K and row counts that g4a_gemm16 and
    g4a_gemm16_geglu take: (M + 127) K 2 and n K 2 up to 2^31 - 1, n in steps of 128 (64)."""
    holds(tmp_path, """
constexpr uint64_t kMost = 0x7fffffff;
constexpr bool rows_ok(uint64_t rows, uint64_t K, uint64_t tile) {
    const uint64_t bytes = rows * K * 2, end = (rows + tile - 1) / tile * tile;
    for (uint64_t r = rows > 2 ? rows - 2 : 0; r < end; ++r) {
        const uint64_t off = row_offset((int)r, (int)K) + (uint64_t)(kStageBytes - 16), exact = r * K * 2 + kStageBytes - 16;
        if (off != exact || (r >= rows && off < bytes) || off + K * 2 > 0xffffffffu) return false;
    }
    return true;
}
constexpr bool check() {
    for (uint64_t tile : {64, 96, 128, 192, 256})
        for (uint64_t K = 64; K * 2 * 128 <= kMost; K *= 2) {
            for (uint64_t k : {K, K * 2 - 64}) {
                if (k * 2 * 128 > kMost) continue;
                if (!rows_ok(kMost / (k * 2) - 127, k, tile) || !rows_ok(1, k, tile)) return false;
                if (!rows_ok(kMost / (k * 2) / 128 * 128, k, tile)) return false;
                if (tile <= 128 && !rows_ok(kMost / (k * 2) / 64 * 64, k, tile)) return false;
            }
        }
    return true;
}
static_assert(check(), "an offset that wraps");
""")
