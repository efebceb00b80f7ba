// Which output tile and k split a GEMM launch takes (gemm.hip), apart from the kernel so that a
// host compiler can evaluate the plan of any shape (tests/test_gemm_plan.py).
#pragma once

#include <stddef.h>

#include <algorithm>

namespace g4a {

constexpr int kCUs = 256;
constexpr size_t kGemmTicketBytes = 2048;  // G4A_GEMM_TICKET_BYTES

// The tiles a launch can take (tokens x weight rows) and what a workgroup of one costs in us: per
// 64-deep k-stage, and once for filling the pipeline and the epilogue. Tiles of 112 to 160 KiB of
// stages run one workgroup a CU; those of two or three stages (64 and 72 KiB) run two, and `step2`,
// `fixed2` are their costs then. A launch costs its rounds of 256 (512) workgroups, the last of
// them at one a CU where that holds it, and the plan takes the cheapest. Products that the larger
// tiles leave at just over one round share the CUs instead, and few k-stages fill a shallow pipeline
// sooner: us a call without -> with the shared tiles, N 4096 K 1536 M 2047 33.0 -> 28.4; N 2048
// K 1536 M 4000 31.8 -> 28.1; N 1536 K 256 M 2047 6.7 -> 6.2; N 1536 K 4096 M 200, split,
// 17.5 -> 13.8. The six-stage 64 x 128 tile stays for long k (N 1536 K 4096 M 512: 19.6, three
// stages 21.2).
//
// The costs are a fit to 448 products (M 1 to 8000, K 256 to 12288, N 256 to 24576, one to three
// matrices and the gate/up form, with and without a workspace): the time that the plan expects is off
// by 8 % in the mean, and its choice is 0.5 % slower than the fastest tile and split in the mean, 9 %
// at most. Against 128 x 128 and 128 x 64 tiles of two and three stages alone it is slower for one of
// them, N 4096 K 256 from M 3000 on (14.6 -> 16.0 us at M 4000). `runs`: consecutive tiles on one XCD
// (128 x 128 at M 2047 N 2048: 21.4 -> 19.4 us); the 256 x 256 tiles measured faster dealt round-robin
// (M 2047 N 24576: 152 against 160 us).
struct TileCfg {
    int bm, bn;
    float step, fixed;
    int runs;
    float step2, fixed2;  // two workgroups a CU; 0: one
};
constexpr TileCfg kTiles[] = {
    {256, 256, 1.35f, 5.5f, 0, 0.0f, 0.0f},   {256, 192, 1.04f, 6.6f, 1, 0.0f, 0.0f},
    {192, 128, 0.58f, 5.6f, 1, 0.0f, 0.0f},   {128, 128, 0.46f, 2.4f, 1, 1.02f, 1.3f},
    {128, 128, 0.33f, 5.5f, 1, 0.0f, 0.0f},   {64, 128, 0.27f, 3.0f, 1, 0.0f, 0.0f},
    {64, 128, 0.285f, 2.6f, 1, 0.58f, 2.5f},
};
constexpr int kTileCount = sizeof(kTiles) / sizeof(kTiles[0]);
constexpr int kFirstSplit = 4;  // the tiles from here on have a split form
// A split adds the tile's partials through memory: 0.73 us for each of a tile's, and 0.0155 us for
// every 64 x 128 part that a workgroup of the launch stores (same fit): N 256 K 1536 M 1 8.1 ->
// 7.1 us, M 1024 9.0 -> 8.7; N 1536 K 2048 M 300 11.5 -> 10.2.
constexpr float kMergeEach = 0.73f, kMergePart = 0.0155f;

// The workspace contract (g4a_gemm16_ws_bytes): launches of fewer 128 x 64 output tiles than
// CUs may split k up to `max_splits` times, at least four k-stages each, and are asked for that
// many f32 copies of their (padded) output behind the ticket words. The plan below splits
// fewer times or not at all where that is faster, and never needs more.
constexpr int kSplitBelow = 256, kSplitTarget = 768, kSplitMinSteps = 4;
static_assert(kSplitBelow * 4 <= kGemmTicketBytes, "a ticket word per split tile");

struct SplitRoom {
    int max_splits;
    size_t ws_bytes;  // tickets + partials, 0 without a split
};
inline SplitRoom split_room(int M, int K, int n_mats, const int* rows) {
    long tiles = 0;
    for (int i = 0; i < n_mats; ++i) tiles += (long)(rows[i] / 64) * ((M + 127) / 128);
    SplitRoom r{1, 0};
    if (tiles < kSplitBelow) r.max_splits = (int)std::max(1l, std::min((long)K / 64 / kSplitMinSteps, kSplitTarget / tiles));
    if (r.max_splits > 1) r.ws_bytes = kGemmTicketBytes + (size_t)tiles * r.max_splits * 128 * 64 * 4;
    return r;
}

struct GemmPlan {
    int cfg, tiles, splits;
};
// rows: weight rows of each matrix (2 n for the gate/up pair, whose tiles hold rows of both)
inline GemmPlan gemm_plan(int M, int K, int n_mats, const int* rows, int max_splits) {
    GemmPlan best{0, 0, 1};
    float least = 0;
    for (int c = 0; c < kTileCount; ++c) {
        const TileCfg& t = kTiles[c];
        long tiles = 0;
        for (int i = 0; i < n_mats; ++i) tiles += (long)((rows[i] + t.bn - 1) / t.bn) * ((M + t.bm - 1) / t.bm);
        for (int s = 1; s <= (c >= kFirstSplit && tiles <= (long)(kGemmTicketBytes / 4) ? max_splits : 1); ++s) {
            const long wgs = tiles * s, round = t.step2 > 0.0f ? 2 * kCUs : kCUs, last = wgs % round;
            const int stages = (K / 64 + s - 1) / s;
            const float one = stages * t.step + t.fixed, full = t.step2 > 0.0f ? stages * t.step2 + t.fixed2 : one;
            float cost = wgs / round * full + (last == 0 ? 0.0f : last <= kCUs ? one : full);
            if (s > 1) cost += kMergeEach * s + kMergePart * (t.bm / 64) * wgs;
            if (!best.tiles || cost < least) {
                best = {c, (int)tiles, s};
                least = cost;
            }
        }
    }
    return best;
}

}  // namespace g4a
