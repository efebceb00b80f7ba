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

}  // namespace g4a
