// The f16 GEMMs of the batched prefill, for gfx950: out = A . W^T over S token rows.
//
// Reference semantics: gemm_tiled (gemma4_150/kernels_dsl.py:34-136: f32 accumulation, f16
// result f16(alpha * sum)), srq_b on the q path (:246-255), and geglu_b (:259-290) behind the
// gate and up products; dispatched by PrefillGPU._gemm (prefill_gpu.py:151-184, 327-395).
//
// MI355X design. At these shapes (K 1536 .. 12288, N 256 .. 24576) the products are bound by
// how many bytes a CU moves per MFMA: a tile of BM tokens x BN outputs takes (BM + BN) * 128
// bytes into LDS per 64-deep k-stage for BM * BN / 32 MFMA cycles, so the tile is as large as
// the output allows, and the kernel keeps the loads away from the MFMAs:
//  * k-stages come straight from HBM / L2 into LDS (buffer_load .. lds, 1 KiB per wave
//    instruction, whole 128-byte row segments), ST stages deep. The DMAs are inline asm: as
//    builtins the compiler waits for all of them (vmcnt(0)) before every LDS read that
//    follows, so no stage is ever in flight behind another.
//  * operands are read 32 k ahead of their MFMAs, one LDS read after each MFMA, and the next
//    stage's DMAs go out between the MFMAs of the second half of a stage: issued in a block,
//    the reads of every wave queue at the LDS at once while the matrix cores idle (8192^3,
//    256 x 256 tiles: 1169 -> 1259 TFLOP/s).
//  * one barrier a stage, in its middle: there the wave's own DMAs of the next stage have
//    landed and all its operand reads of this one have returned, so after it the next stage
//    is readable and this one's buffer can be refilled.
// Under such a load the clock falls to about 1.5 GHz (power): 8192^3 keeps the matrix cores
// 80 % busy at 1.26 PFLOP/s, the vendor library's kernel 89 % at 1.47.
#include <stdio.h>
#include <stdlib.h>

#include "common.hpp"
#include "gemm_offsets.hpp"
#include "gemm_plan.hpp"

namespace g4a {

typedef float float16v __attribute__((ext_vector_type(16)));
typedef int int4v __attribute__((ext_vector_type(4)));
typedef unsigned v4u32 __attribute__((ext_vector_type(4)));

constexpr int kCpolSC1 = 16;  // device scope: the access bypasses the per-XCD caches

struct Gemm16Args {
    const half_t* a;  // [M][K] f16
    int M, K;
    const half_t* w[3];  // [N_p][K] f16
    void* out[3];        // [M][N_p] f16, or f32 (srq'd with out_q) when out_f32
    int n[3], out_f32[3];
    float out_q[3], alpha[3];
    int tile_end[3];  // cumulative tiles
    int tiles, mtiles, splits, runs;
    unsigned* ticket;  // [tiles], zero between calls
    float* part;       // [tiles][splits][NB * MB * 4][threads] float4: the f32 partial tiles
    float gq, uq, oq;  // the gate/up form: geglu_b's steps
    const float* lut;  // ... and the layer's GELU table of the gq grid (gelu_srq), or NULL
};

// compile-time loop: f(0), f(1), .. with the index a constant expression
template <int I>
struct Idx {
    static constexpr int value = I;
};
template <int N, int I = 0, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(Idx<I>{});
        static_for<N, I + 1>(f);
    }
}
constexpr int cmin(int a, int b) { return a < b ? a : b; }

// A raw buffer resource as four scalars, for the asm DMA (reads at or past `bytes` give zeros).
__device__ __forceinline__ int4v rsrc4(const void* p, uint32_t bytes) {
    const uint64_t u = (uint64_t)p;
    int4v r;
    r[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)u);
    r[1] = __builtin_amdgcn_readfirstlane((int)(uint32_t)(u >> 32) & 0xffff);
    r[2] = __builtin_amdgcn_readfirstlane((int)bytes);
    r[3] = 0x00020000;
    return r;
}
// 16 bytes a lane from rs + voff + soff to LDS address lds + 16 lane. No output register: the
// data is in LDS once vmcnt has counted it (wait_barrier).
__device__ __forceinline__ void dma16(int4v rs, uint32_t voff, uint32_t soff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds), "v"(voff), "s"(rs),
                 "s"(soff));
}
// At most N of this wave's DMAs still out, its LDS reads returned, then the workgroup's barrier.
template <int N>
__device__ __forceinline__ void wait_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}
// LDS written by other lanes of this wave: in order in hardware, kept in order by the compiler.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

enum GemmMode { kPlain, kSplitK, kGeglu };

// One tile of BM tokens x BN weight rows per workgroup of WM x WN waves (wave tile TM x TN,
// v_mfma_f32_32x32x16_f16 computed transposed, D^T = W . A^T, so a lane holds 4 consecutive
// outputs of one token). LDS rows are 128 B; chunk c of row r sits at c ^ ((r >> 1) & 7), so
// the 16 rows of a quarter-wave operand read fall in 16 distinct bank groups.
//
// kSplitK: k is cut into g.splits ranges, one workgroup each. Every workgroup stores its f32
// partial tile device-coherently, waits for the stores and takes the tile's ticket (a relaxed
// agent-scope atomic); the last to take it adds the partials in split order (whichever
// workgroup that is, so the result does not depend on arrival order), resets the ticket to
// zero for the next call and runs the epilogue.
//
// kGeglu: w[0] is the gate matrix, w[1] the up matrix. Of every 32 tile rows the first 16 are
// gate rows and the last 16 the up rows of the same outputs, so a lane holds both products of
// its outputs and the epilogue stores geglu_b's code of them.
template <int BM, int BN, int WM, int WN, int ST, int MINW, GemmMode MODE>
__global__ __launch_bounds__(64 * WM * WN, MINW) void gemm16_kernel(Gemm16Args g) {
    constexpr int NW = WM * WN, TM = BM / WM, TN = BN / WN, MB = TM / 32, NB = TN / 32;
    constexpr int ROWB = kStageBytes, STB = (BM + BN) * ROWB;
    constexpr int DW = BN / 8 / NW, DA = BM / 8 / NW, D = DW + DA;  // 1 KiB DMAs per wave and stage
    static_assert(TM % 32 == 0 && TN % 32 == 0 && DW * 8 * NW == BN && DA * 8 * NW == BM, "even shares");
    static_assert(ST >= 2 && (ST - 1) * D < 64 && ST * STB <= 160 * 1024, "vmcnt holds 6 bits; LDS holds 160 KiB");
    constexpr bool GEGLU = MODE == kGeglu;
    auto swz = [](int r) { return (r >> 1) & 7; };
    __shared__ __attribute__((aligned(1024))) char lds[ST * STB];  // [stage]{W rows, A rows}
    const uint32_t lbase = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave % WN, wm = wave / WN, l32 = lane & 31, h = lane >> 5;

    // ---- this workgroup's k range, matrix and tile
    const int unit = g.runs ? xcd_run_index() : blockIdx.x;
    const int split = MODE == kSplitK ? unit / g.tiles : 0, tile = MODE == kSplitK ? unit % g.tiles : unit;
    int p = 0, t0 = tile;
    if (!GEGLU && t0 >= g.tile_end[0]) p = t0 >= g.tile_end[1] ? 2 : 1;
    if (p > 0) t0 -= g.tile_end[p - 1];
    const int N = g.n[p], K = g.K;
    constexpr int TNO = GEGLU ? BN / 2 : BN;  // outputs a tile covers
    const int ntiles = (N + TNO - 1) / TNO;
    int tn, tm;
    if (g.runs) {  // four n-tiles wide, then down the tokens: an XCD's run shares W and A rows
        const int per = 4 * g.mtiles, grp = t0 / per, in = t0 % per, gn = min(4, ntiles - 4 * grp);
        tn = 4 * grp + in % gn;
        tm = in / gn;
    } else {
        tn = t0 % ntiles;
        tm = t0 / ntiles;
    }
    const int n0 = tn * TNO, m0 = tm * BM;
    const int nkall = K / 64;
    const int kt0 = MODE == kSplitK ? split * nkall / g.splits : 0;
    const int nk = MODE == kSplitK ? (split + 1) * nkall / g.splits - kt0 : nkall;

    // ---- the stage DMAs: wave w moves W rows 8 (DW w + j) .. and A rows 8 (DA w + j) .., eight
    // rows an instruction; rows past M or N read as zeros
    const int4v ra = rsrc4(g.a, (uint32_t)g.M * K * 2), rw = rsrc4(g.w[p], (uint32_t)N * K * 2);
    const int4v ru = GEGLU ? rsrc4(g.w[1], (uint32_t)N * K * 2) : rw;
    uint32_t vw[DW], va[DA];
#pragma unroll
    for (int j = 0; j < DW; ++j) {
        const int i = wave * DW + j, r = 8 * i + lane / 8;
        const int row = n0 + (GEGLU ? 16 * (i / 4) + r % 16 : r);
        vw[j] = row_offset(row, K) + 16 * ((lane % 8) ^ swz(r));
    }
#pragma unroll
    for (int j = 0; j < DA; ++j) {
        const int r = 8 * (wave * DA + j) + lane / 8;
        va[j] = row_offset(m0 + r, K) + 16 * ((lane % 8) ^ swz(r));
    }
    // DMA d of k-stage t into buffer buf; more = 0: past the range, an empty resource at offset 0 (no
    // memory is read and zeros go into a buffer that nobody reads any more)
    auto dma = [&](auto dc, int t, int buf, bool more) {
        constexpr int d = decltype(dc)::value;
        const uint32_t b = lbase + buf * STB;
        int4v q = d >= DW ? ra : GEGLU && ((wave * DW + d) / 2) % 2 ? ru : rw;
        const StageDma at = stage_dma((uint32_t)q[2], kt0 + t, more);
        q[2] = (int)at.records;
        if constexpr (d < DW)
            dma16(q, vw[d], at.soff, b + (wave * DW + d) * 1024);
        else
            dma16(q, va[d - DW], at.soff, b + BN * ROWB + (wave * DA + d - DW) * 1024);
    };

    float lut_entry = 0.0f;  // out before the stages, used after them
    if (GEGLU && g.lut && tid < 256) lut_entry = g.lut[tid];
    float16v acc[NB][MB];
#pragma unroll
    for (int a = 0; a < NB; ++a)
#pragma unroll
        for (int b = 0; b < MB; ++b) acc[a][b] = float16v{};
    // the operands of half a stage (32 k): k-step s holds k 16s + 8h .. +7 in lane (l32, h)
    struct Frag {
        half8 w[2][NB], a[2][MB];
    };
    constexpr int NR = 2 * (NB + MB), NM = 2 * NB * MB;  // operand reads and MFMAs per half stage
    constexpr int RPM = (NR + NM - 1) / NM;              // reads after each MFMA
    auto rd = [&](auto ic, const char* st, int half, Frag& f) {
        constexpr int s = decltype(ic)::value / (NB + MB), b = decltype(ic)::value % (NB + MB);
        const int c = 16 * ((2 * (2 * half + s) + h) ^ swz(l32));
        if constexpr (b < NB)
            f.w[s][b] = *reinterpret_cast<const half8*>(st + (TN * wn + 32 * b + l32) * ROWB + c);
        else
            f.a[s][b - NB] = *reinterpret_cast<const half8*>(st + (BN + TM * wm + 32 * (b - NB) + l32) * ROWB + c);
    };
    // half a stage: the MFMAs of `use`, each followed by its share of the reads of `fill` (half
    // `half` of the stage at st) and, with DMA, of stage t's DMAs into buffer buf
    auto phase = [&](const Frag& use, Frag& fill, const char* st, int half, auto dmac, int t, int buf, bool more) {
        static_for<NM>([&](auto ic) {
            constexpr int i = decltype(ic)::value, s = i / (MB * NB), b = (i / NB) % MB, a = i % NB;
            acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(use.w[s][a], use.a[s][b], acc[a][b], 0, 0, 0);
            constexpr int r0 = cmin(NR, i * RPM), r1 = cmin(NR, (i + 1) * RPM);
            static_for<r1 - r0>([&](auto rc) { rd(Idx<r0 + decltype(rc)::value>{}, st, half, fill); });
            if constexpr (decltype(dmac)::value) {
                constexpr int d0 = (i * D + NM - 1) / NM, d1 = ((i + 1) * D + NM - 1) / NM;
                static_for<d1 - d0>([&](auto dc) { dma(Idx<d0 + decltype(dc)::value>{}, t, buf, more); });
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    };

#pragma unroll
    for (int i = 0; i < ST; ++i)
        if (i < nk) static_for<D>([&](auto dc) { dma(dc, i, i, true); });
    if (nk >= ST)
        wait_barrier<(ST - 1) * D>();
    else
        wait_barrier<0>();  // a short range: all of it
    Frag f0, f1;
    static_for<NR>([&](auto ic) { rd(ic, lds, 0, f0); });
    int buf = 0;
    for (int t = 0; t < nk; ++t) {
        phase(f0, f1, lds + buf * STB, 1, Idx<0>{}, 0, 0, false);
        wait_barrier<(ST - 2) * D>();  // stage t + 1 has landed; stage t is in registers
        const int next = buf + 1 == ST ? 0 : buf + 1;
        phase(f1, f0, lds + next * STB, 0, Idx<1>{}, t + ST, buf, t + ST < nk);
        buf = next;
    }
    wait_barrier<0>();  // LDS is free

    if constexpr (MODE == kSplitK) {
        // publish this split's partial: float4 v of thread tid at [tile][split][v][tid]
        constexpr int NV = NB * MB * 4, NT = 64 * NW;
        const size_t tbytes = (size_t)g.splits * NV * NT * 16;
        const rsrc_t rp = make_rsrc(reinterpret_cast<char*>(g.part) + tile * tbytes, (uint32_t)tbytes);
#pragma unroll
        for (int a = 0; a < NB; ++a)
#pragma unroll
            for (int b = 0; b < MB; ++b)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int v = (a * MB + b) * 4 + q;
                    const float4v x{acc[a][b][4 * q], acc[a][b][4 * q + 1], acc[a][b][4 * q + 2], acc[a][b][4 * q + 3]};
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u32, x), rp,
                                                           ((split * NV + v) * NT + tid) * 16, 0, kCpolSC1);
                }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's partial stores are done
        int* s_last = reinterpret_cast<int*>(lds);
        __syncthreads();
        if (tid == 0) {
            const unsigned old = __hip_atomic_fetch_add(g.ticket + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const bool last = old == (unsigned)g.splits - 1;
            if (last) __hip_atomic_store(g.ticket + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *s_last = last;
        }
        __syncthreads();
        if (!*s_last) return;
        // the sum in split order, this workgroup's own partial from its registers
        float16v sum[NB][MB];
        for (int j = 0; j < g.splits; ++j) {
#pragma unroll
            for (int a = 0; a < NB; ++a)
#pragma unroll
                for (int b = 0; b < MB; ++b) {
                    float16v x;
                    if (j == split) {
                        x = acc[a][b];
                    } else {
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const int v = (a * MB + b) * 4 + q;
                            const float4v y = __builtin_bit_cast(
                                float4v, __builtin_amdgcn_raw_buffer_load_b128(rp, ((j * NV + v) * NT + tid) * 16, 0, kCpolSC1));
#pragma unroll
                            for (int e = 0; e < 4; ++e) x[4 * q + e] = y[e];
                        }
                    }
                    sum[a][b] = j == 0 ? x : sum[a][b] + x;
                }
        }
#pragma unroll
        for (int a = 0; a < NB; ++a)
#pragma unroll
            for (int b = 0; b < MB; ++b) acc[a][b] = sum[a][b];
        __syncthreads();  // s_last's bytes are staged over below
    }

    // ---- epilogue: D^T[n][m], acc[r] is output n = 8(r/4) + 4h + r%4, token m = l32 of the
    // 32x32 block. The product, times alpha, rounds to f16 (gemm_tiled's f16(alpha * acc)); the q
    // path then applies srq_b. A wave stages 32 tokens of its outputs at a time in LDS (its own
    // region, rows padded by 16 bytes so an instruction's writes spread over the banks) and
    // stores whole row segments, 16 bytes a lane.
    constexpr int WO = GEGLU ? TN / 2 : TN;  // outputs of a wave
    const int nw0 = n0 + WO * wn, mw0 = m0 + TM * wm;
    auto store_rows = [&](auto ec, const char* sg, int b, void* out) {
        constexpr int E = decltype(ec)::value, SR = WO * E + 16, CH = WO * E / 16;
        wave_lds_fence();
#pragma unroll
        for (int i = 0; i < CH / 2; ++i) {
            const int idx = 64 * i + lane, r = idx / CH, ch = idx % CH;
            const int m = mw0 + 32 * b + r, n = nw0 + ch * (16 / E);
            if (m < g.M && n < N)
                *reinterpret_cast<float4v*>(reinterpret_cast<char*>(out) + ((size_t)m * N + n) * E) =
                    *reinterpret_cast<const float4v*>(sg + r * SR + 16 * ch);
        }
        wave_lds_fence();
    };
    if constexpr (GEGLU) {
        constexpr int SR = WO * 2 + 16;
        static_assert(NW * 32 * SR + 1024 <= ST * STB && 64 * NW >= 256, "the staged rows and the table fit the stages");
        char* sg = lds + wave * 32 * SR;
        float* table = reinterpret_cast<float*>(lds + NW * 32 * SR);
        auto blocks = [&](auto&& code) {
#pragma unroll
            for (int b = 0; b < MB; ++b) {
#pragma unroll
                for (int a = 0; a < NB; ++a)
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        half4 y;
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            y[i] = code((float)(half_t)pin(acc[a][b][4 * q + i]), (float)(half_t)pin(acc[a][b][8 + 4 * q + i]));
                        *reinterpret_cast<half4*>(sg + l32 * SR + (16 * a + 8 * q + 4 * h) * 2) = y;
                    }
                store_rows(Idx<2>{}, sg, b, g.out[0]);
            }
        };
        if (g.lut && srq_fast(g.gq) && srq_fast(g.uq) && srq_fast(g.oq)) {
            // geglu_code's arithmetic with srq_index for its three divisions and the GELU table in
            // LDS: read from memory, each of a lane's lookups was a dependent 64-address gather
            const SrqStep tg = srq_step(g.gq), tu = srq_step(g.uq), to = srq_step(g.oq);
            if (tid < 256) table[tid] = lut_entry;
            __syncthreads();
            blocks([&](float gv, float uv) {
                const float y = pin(table[(int)srq_index(gv, tg) + 128] * pin(srq_index(uv, tu) * tu.s));
                return (half_t)srq_index(y, to);
            });
        } else {
            blocks([&](float gv, float uv) { return geglu_code(gv, uv, g.gq, g.uq, g.oq, g.lut); });
        }
        return;
    }
    const float oq = g.out_q[p], alpha = g.alpha[p];
    if (g.out_f32[p]) {
        constexpr int SR = WO * 4 + 16;
        static_assert(NW * 32 * SR <= ST * STB, "the staged rows fit the operand stages");
        char* sg = lds + wave * 32 * SR;
        auto blocks = [&](auto&& quant) {
#pragma unroll
            for (int b = 0; b < MB; ++b) {
#pragma unroll
                for (int a = 0; a < NB; ++a)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        float4v v;
#pragma unroll
                        for (int i = 0; i < 4; ++i) v[i] = quant((float)(half_t)pin(alpha * acc[a][b][4 * q + i]));
                        *reinterpret_cast<float4v*>(sg + l32 * SR + (32 * a + 8 * q + 4 * h) * 4) = v;
                    }
                store_rows(Idx<4>{}, sg, b, g.out[p]);
            }
        };
        if (srq_fast(oq)) {
            const SrqStep t = srq_step(oq);
            blocks([&](float x) { return srq_index(x, t) * oq; });
        } else {
            blocks([&](float x) { return srq(x, oq); });
        }
        return;
    }
    constexpr int SR = WO * 2 + 16;
    char* sg = lds + wave * 32 * SR;
#pragma unroll
    for (int b = 0; b < MB; ++b) {
#pragma unroll
        for (int a = 0; a < NB; ++a)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                half4 y;
#pragma unroll
                for (int i = 0; i < 4; ++i) y[i] = (half_t)pin(alpha * acc[a][b][4 * q + i]);
                *reinterpret_cast<half4*>(sg + l32 * SR + (32 * a + 8 * q + 4 * h) * 2) = y;
            }
        store_rows(Idx<2>{}, sg, b, g.out[p]);
    }
}

}  // namespace g4a

using namespace g4a;

namespace {

static_assert(kGemmTicketBytes == G4A_GEMM_TICKET_BYTES, "the header's ticket words");

int gemm_check(int M, int K, const void* a_f16, int n_mats, const g4a_gemm_mat* mats) {
    if (M <= 0 || K <= 0 || K % 64) {
        set_error("M (%d) must be positive and K (%d) a positive multiple of 64", M, K);
        return G4A_EINVAL;
    }
    if (n_mats < 1 || n_mats > 3 || !mats) {
        set_error("n_mats (%d) must be 1, 2 or 3 with a matrix table", n_mats);
        return G4A_EINVAL;
    }
    if (!a_f16 || ((uintptr_t)a_f16 & 15) || (int64_t)(M + 127) * K * 2 > 0x7fffffff) {
        set_error("a must be non-NULL, 16-byte aligned and within 32-bit buffer offsets");
        return G4A_EINVAL;
    }
    for (int i = 0; i < n_mats; ++i) {
        const g4a_gemm_mat* m = &mats[i];
        if (m->n <= 0 || m->n % 128 || !m->w_f16 || !m->out || (((uintptr_t)m->w_f16 | (uintptr_t)m->out) & 15) ||
            (int64_t)m->n * K * 2 > 0x7fffffff || (int64_t)M * m->n > 0x7fffffff || !(m->out_q >= 0.0f)) {
            set_error("matrix %d: n (%d) a positive multiple of 128, w/out non-NULL and 16-byte aligned, "
                      "within 32-bit offsets, out_q >= 0", i, m->n);
            return G4A_EINVAL;
        }
    }
    return G4A_OK;
}

template <GemmMode MODE>
void gemm_launch(const GemmPlan& pl, const Gemm16Args& g, hipStream_t s) {
    const dim3 grid(pl.tiles * pl.splits);
    if constexpr (MODE != kSplitK) {
        if (pl.cfg == 0) hipLaunchKernelGGL((gemm16_kernel<256, 256, 2, 4, 2, 2, MODE>), grid, dim3(512), 0, s, g);
        if (pl.cfg == 1) hipLaunchKernelGGL((gemm16_kernel<256, 192, 2, 2, 2, 1, MODE>), grid, dim3(256), 0, s, g);
        if (pl.cfg == 2) hipLaunchKernelGGL((gemm16_kernel<192, 128, 2, 2, 4, 1, MODE>), grid, dim3(256), 0, s, g);
        if (pl.cfg == 3) hipLaunchKernelGGL((gemm16_kernel<128, 128, 2, 2, 2, 2, MODE>), grid, dim3(256), 0, s, g);
    }
    if (pl.cfg == 4) hipLaunchKernelGGL((gemm16_kernel<128, 128, 2, 2, 4, 1, MODE>), grid, dim3(256), 0, s, g);
    if (pl.cfg == 5) hipLaunchKernelGGL((gemm16_kernel<64, 128, 2, 4, 6, 2, MODE>), grid, dim3(512), 0, s, g);
    if (pl.cfg == 6) hipLaunchKernelGGL((gemm16_kernel<64, 128, 2, 4, 3, 4, MODE>), grid, dim3(512), 0, s, g);
}

int gemm_run(int M, int K, const void* a_f16, int n_mats, const g4a_gemm_mat* mats, void* ws, size_t ws_bytes,
             void* stream) {
    const int rc = gemm_check(M, K, a_f16, n_mats, mats);
    if (rc != G4A_OK) return rc;
    int rows[3];
    for (int i = 0; i < n_mats; ++i) rows[i] = mats[i].n;
    const SplitRoom room = split_room(M, K, n_mats, rows);
    if (ws && ws_bytes < room.ws_bytes) {
        set_error("workspace of %zu bytes, this product needs %zu (g4a_gemm16_ws_bytes)", ws_bytes, room.ws_bytes);
        return G4A_EWORKSPACE;
    }
    if (ws && room.ws_bytes && ((uintptr_t)ws & 255)) {
        set_error("the workspace must be 256-byte aligned");
        return G4A_EINVAL;
    }
    const GemmPlan pl = gemm_plan(M, K, n_mats, rows, ws ? room.max_splits : 1);
    const TileCfg& tc = kTiles[pl.cfg];
    Gemm16Args g = {};
    g.a = reinterpret_cast<const half_t*>(a_f16);
    g.M = M;
    g.K = K;
    g.mtiles = (M + tc.bm - 1) / tc.bm;
    g.runs = tc.runs;
    int tiles = 0;
    for (int i = 0; i < 3; ++i) {
        const g4a_gemm_mat* m = i < n_mats ? &mats[i] : nullptr;
        if (m) tiles += ((m->n + tc.bn - 1) / tc.bn) * g.mtiles;
        g.w[i] = m ? reinterpret_cast<const half_t*>(m->w_f16) : nullptr;
        g.out[i] = m ? m->out : nullptr;
        g.n[i] = m ? m->n : tc.bn;
        g.out_f32[i] = m ? m->out_f32 : 0;
        g.out_q[i] = m ? m->out_q : 0.0f;
        g.alpha[i] = m && m->alpha != 0.0f ? m->alpha : 1.0f;
        g.tile_end[i] = tiles;
    }
    g.tiles = tiles;
    g.splits = pl.splits;
    if (pl.splits > 1) {
        g.ticket = reinterpret_cast<unsigned*>(ws);
        g.part = reinterpret_cast<float*>(reinterpret_cast<char*>(ws) + kGemmTicketBytes);
        gemm_launch<kSplitK>(pl, g, (hipStream_t)stream);
    } else {
        gemm_launch<kPlain>(pl, g, (hipStream_t)stream);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_error(e, "gemm16 launch");
    return G4A_OK;
}
}  // namespace

extern "C" int g4a_gemm16(int M, int K, const void* a_f16, int n_mats, const g4a_gemm_mat* mats, void* stream) {
    return gemm_run(M, K, a_f16, n_mats, mats, nullptr, 0, stream);
}

extern "C" int g4a_gemm16_geglu(int M, int K, const void* a_f16, const void* w_gate_f16, const void* w_up_f16, int n,
                                float gate_q, float up_q, float out_q, void* out_f16, const float* gelu_lut,
                                void* stream) {
    if (M <= 0 || K <= 0 || K % 64 || n <= 0 || n % 64) {
        set_error("M (%d) positive, K (%d) a positive multiple of 64, n (%d) a positive multiple of 64", M, K, n);
        return G4A_EINVAL;
    }
    if (!a_f16 || !w_gate_f16 || !w_up_f16 || !out_f16 ||
        (((uintptr_t)a_f16 | (uintptr_t)w_gate_f16 | (uintptr_t)w_up_f16 | (uintptr_t)out_f16) & 15) ||
        (int64_t)(M + 127) * K * 2 > 0x7fffffff || (int64_t)n * K * 2 > 0x7fffffff || (int64_t)M * n > 0x7fffffff) {
        set_error("a, w_gate, w_up, out non-NULL, 16-byte aligned and within 32-bit offsets");
        return G4A_EINVAL;
    }
    if (!(gate_q >= 0.0f) || !(up_q >= 0.0f) || !(out_q >= 0.0f)) {
        set_error("gate_q, up_q and out_q must be >= 0");
        return G4A_EINVAL;
    }
    const int rows = 2 * n;
    const GemmPlan pl = gemm_plan(M, K, 1, &rows, 1);
    const TileCfg& tc = kTiles[pl.cfg];
    Gemm16Args g = {};
    g.a = reinterpret_cast<const half_t*>(a_f16);
    g.M = M;
    g.K = K;
    g.mtiles = (M + tc.bm - 1) / tc.bm;
    g.runs = tc.runs;
    g.w[0] = reinterpret_cast<const half_t*>(w_gate_f16);
    g.w[1] = reinterpret_cast<const half_t*>(w_up_f16);
    g.out[0] = out_f16;
    g.n[0] = n;
    g.alpha[0] = 1.0f;
    g.tiles = pl.tiles;
    g.tile_end[0] = g.tile_end[1] = g.tile_end[2] = g.tiles;
    g.splits = 1;
    g.gq = gate_q;
    g.uq = up_q;
    g.oq = out_q;
    g.lut = gelu_lut;
    gemm_launch<kGeglu>(pl, g, (hipStream_t)stream);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_error(e, "gemm16_geglu launch");
    return G4A_OK;
}

extern "C" size_t g4a_gemm16_ws_bytes(int M, int K, int n_mats, const g4a_gemm_mat* mats) {
    if (M <= 0 || K <= 0 || K % 64 || n_mats < 1 || n_mats > 3 || !mats) return 0;
    int rows[3];
    for (int i = 0; i < n_mats; ++i) {
        if (mats[i].n <= 0 || mats[i].n % 128) return 0;
        rows[i] = mats[i].n;
    }
    return split_room(M, K, n_mats, rows).ws_bytes;
}

extern "C" int g4a_gemm16_ws(int M, int K, const void* a_f16, int n_mats, const g4a_gemm_mat* mats, void* ws,
                             size_t ws_bytes, void* stream) {
    return gemm_run(M, K, a_f16, n_mats, mats, ws, ws_bytes, stream);
}
