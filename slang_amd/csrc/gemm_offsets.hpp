// Addresses of the GEMM's stage DMAs (gemm.hip), apart from the kernel so that a host compiler
// can evaluate them at the ends of what the launch checks accept (tests/test_gemm_offsets.py).
#pragma once

#include <stdint.h>

namespace g4a {

constexpr int kStageBytes = 128;  // of a row in a 64-deep k-stage

// The range and scalar offset of a DMA of k-stage `stage` out of a matrix of `bytes` bytes; more =
// false: past the last stage, where no memory may be read. An empty range alone does not say so:
// a range check that takes the scalar offset from the range's bytes wraps around below zero.
struct StageDma {
    uint32_t records, soff;
};
constexpr StageDma stage_dma(uint32_t bytes, int stage, bool more) {
    return more ? StageDma{bytes, (uint32_t)stage * kStageBytes} : StageDma{0, 0};
}

// Byte offset of row `row` of a matrix of rows of K f16 values. A tile's rows past the matrix reach
// up to 255 rows beyond it, past 2^31 where the matrix ends just below (the launch checks leave 127
// rows), but never past 2^32: they read as zeros.
constexpr uint32_t row_offset(int row, int K) { return (uint32_t)row * (uint32_t)K * 2u; }

}  // namespace g4a
