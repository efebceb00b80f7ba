// The q/k/v producer in front of the attention path, for gfx950: QAT-weight projections.
//
// Reference semantics:
//  * dq_f16 (gemma4_150/kernels_dsl.py:2101-2138): packed rows, value i of a row at bit
//    8*(i / (8/BITS)) + BITS*(i % (8/BITS)) of the row's bytes, w = f16(s_row * (q - 2^(BITS-1))).
//  * qkv_70 (kernels_dsl.py:1384-1480): decode GEMVs of q, k and v over one input a, 4-bit
//    rows, out[o] = srq(scale[o] * (sum_i q[o][i] a[i] - 8 sum_a), out_scale) with the zero
//    point folded into the input sum; one dispatch partitioned over the three matrices.
//  * prefill (prefill_gpu.py:327-342): srqh_b (a -> f16(srq(a, s)), kernels_dsl.py:233-242),
//    dq_f16, gemm_tiled (f32 accumulation, f16 result, :34-136), srq_b on the q path (:246-255).
//
// MI355X design (not the reference's):
//  * Decode reads the 4-bit rows straight from HBM (the bytes QAT saves are the bytes decode
//    pays for). A lane owns 16-byte chunks of a row (32 values) and keeps the matching 32
//    inputs in registers for every row it visits; values come out of the packed words with
//    byte masks and v_cvt_f32_ubyte*, and a row is one wave-wide DPP/permlane sum.
//  * Prefill is MFMA work. Weights are static, and 288 GB of HBM holds every layer's f16
//    weights many times over, so dequantisation is its own pass (g4a_dequant, run at load
//    or per call as the reference does) rather than VALU work repeated inside every GEMM
//    tile. srqh_b runs once per layer input (g4a_srqh); the q, k and v GEMMs then share
//    that f16 activation in one grouped launch (g4a_gemm16, gemm.hip).
#include <stdio.h>
#include <stdlib.h>

#include <algorithm>

#include "common.hpp"

namespace g4a {

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------- dequantisation
// One thread per 16 bytes of packed row (4 words): 128/BITS values, f16(s * (q - zp)).
template <int BITS>
__global__ __launch_bounds__(256) void dequant_kernel(const uint32_t* __restrict__ bits,
                                                      const float* __restrict__ scale,
                                                      half_t* __restrict__ out, int n_in,
                                                      int n_quads) {
    constexpr int VPQ = 128 / BITS;  // values per 16 bytes
    constexpr uint32_t MASK = (1u << BITS) - 1;
    const float zp = (float)(1 << (BITS - 1));
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n_quads) return;
    const int qpr = n_in / VPQ;  // quads per row
    const int o = i / qpr;
    const u32x4 w = *reinterpret_cast<const u32x4*>(bits + 4 * (size_t)i);
    const float s = scale[o];
    half_t* dst = out + (size_t)i * VPQ;
#pragma unroll
    for (int g = 0; g < VPQ / 8; ++g) {  // 8 values per 16-byte store
        half8 h;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int v = 8 * g + j;                      // value within the 16 bytes
            const int bit = 32 * (v / (32 / BITS)) + 8 * ((v % (32 / BITS)) / (8 / BITS)) +
                            BITS * (v % (8 / BITS));      // word, byte, then low bits first
            const uint32_t q = (w[bit / 32] >> (bit % 32)) & MASK;
            h[j] = (half_t)pin(s * ((float)q - zp));  // f16 of the f32 product, as dq_f16 rounds
        }
        *reinterpret_cast<half8*>(dst + 8 * g) = h;
    }
}

// ---------------------------------------------------------------- decode q/k/v GEMV
struct GemvArgs {
    const float* a;
    const float* sum_a;
    const uint32_t* bits[3];
    const float* scales;  // [q_dim + 2 kv_dim]: q rows, then k, then v
    float* out[3];
    float out_scale[3];
    int hidden, q_dim, kv_dim;
    // norm prologue (PRO): a = srq(rms((pres + rms(pa) * pw1) * pmult) * pw2, pq2) made by
    // every wave from the previous layer's tail; workgroup 0 stores x, a and sum_a
    const float* pa;
    const float* pres;
    const float* pw1;
    const float* pw2;
    float* pxout;
    float* pzout;
    float* psum;
    float pq2, peps, pmult;
};

// NJ chunks of 32 values per lane (hidden <= 2048 * NJ); RPW rows per wave, 4 waves.
// PRO: the input a and its sum come from the norm prologue instead of memory (NJ 1).
// sum over the 256 threads of a workgroup (per wave, then the 4 wave sums in order); every
// thread gets it. Two barriers: red may still be read by the previous call.
__device__ __forceinline__ float wg_sum(float v, float* red) {
    v = wave_sum(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
}

template <int NJ, int RPW, bool PRO>
__global__ __launch_bounds__(256) void qkv_gemv_kernel(GemvArgs g) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row0 = (blockIdx.x * 4 + wave) * RPW;  // over [q rows | k rows | v rows]
    const int mat = row0 < g.q_dim ? 0 : row0 < g.q_dim + g.kv_dim ? 1 : 2;
    const int r0 = row0 - (mat == 0 ? 0 : mat == 1 ? g.q_dim : g.q_dim + g.kv_dim);
    const int nrows = mat == 0 ? g.q_dim : g.kv_dim;
    const int row_bytes = g.hidden / 2;
    // every operand load first: the prologue's operands, the packed rows, then the input
    // chunks and the sum. Loads return in issue order, so the prologue's operands go out
    // before the rows: its norms and barriers then run while the rows are in flight.
    const rsrc_t ra = make_rsrc(g.a, (uint32_t)g.hidden * 4);
    const rsrc_t rw = make_rsrc(g.bits[mat], (uint32_t)nrows * row_bytes);
    constexpr int PER = 8;  // prologue: thread t holds elements t + 256k of each operand
    float pv[PER], rv[PER], w1v[PER], w2v[PER];
    if constexpr (PRO) {
        const uint32_t nb = (uint32_t)g.hidden * 4;  // past hidden: zeros
        const rsrc_t rpa = make_rsrc(g.pa, nb), rpr = make_rsrc(g.pres, nb), rp1 = make_rsrc(g.pw1, nb),
                     rp2 = make_rsrc(g.pw2, nb);
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int o = 4 * ((int)threadIdx.x + 256 * k);
            pv[k] = bload_f32(rpa, o);
            rv[k] = bload_f32(rpr, o);
            w1v[k] = bload_f32(rp1, o);
            w2v[k] = bload_f32(rp2, o);
        }
    }
    float av[NJ][32];
    u32x4 wv[RPW][NJ];
#pragma unroll
    for (int r = 0; r < RPW; ++r)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int c = lane + 64 * j;  // chunk of the row; past the row end reads zeros
            const int off = c < row_bytes / 16 ? (r0 + r) * row_bytes + 16 * c : 0x7fffffff;
            wv[r][j] = __builtin_amdgcn_raw_buffer_load_b128(rw, off, 0, kCpolNT);  // read once: non-temporal
        }
    __builtin_amdgcn_sched_barrier(0);  // no prologue arithmetic (and its waits) above the row loads
    float sa;
    if constexpr (PRO) {
        // once per workgroup: the sums run per thread, then over the workgroup (block_sum); a
        // is staged in LDS, from which lane c of every wave takes elements 32c .. 32c+31. The
        // arithmetic is the rms_kernel's: y = (res + pa / d1 * w1) * mult, z = y / d2 * w2,
        // a = srq(z, q2).
        static_assert(NJ == 1, "the norm prologue covers hidden <= 2048");
        __shared__ float s_a[2048];
        __shared__ float pred[4];
        const int tid = threadIdx.x, n = g.hidden;
        float ss = 0.0f;
#pragma unroll
        for (int k = 0; k < PER; ++k) ss = __builtin_fmaf(pv[k], pv[k], ss);
        const float d1 = sqrtf(wg_sum(ss, pred) / (float)n + g.peps);
        float ss2 = 0.0f;
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            rv[k] = (rv[k] + pv[k] / d1 * w1v[k]) * g.pmult;  // x, zeros past hidden
            ss2 = __builtin_fmaf(rv[k], rv[k], ss2);
        }
        const float d2 = sqrtf(wg_sum(ss2, pred) / (float)n + g.peps);
        float s2 = 0.0f;
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int i = tid + 256 * k;
            const float z = srq(rv[k] / d2 * w2v[k], g.pq2);
            if (i < 2048) s_a[i] = i < n ? z : 0.0f;
            s2 += i < n ? z : 0.0f;
            if (blockIdx.x == 0 && i < n) {
                if (g.pxout) g.pxout[i] = rv[k];
                if (g.pzout) g.pzout[i] = z;
            }
        }
        sa = wg_sum(s2, pred);  // its barriers also publish s_a
        if (blockIdx.x == 0 && tid == 0 && g.psum) g.psum[0] = sa;
#pragma unroll
        for (int q4 = 0; q4 < 8; ++q4) {
            const float4v v = *reinterpret_cast<const float4v*>(&s_a[32 * lane + 4 * q4]);
#pragma unroll
            for (int i = 0; i < 4; ++i) av[0][4 * q4 + i] = v[i];
        }
    } else {
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int q4 = 0; q4 < 8; ++q4) {
                const float4v v = bload_f32x4(ra, 128 * (lane + 64 * j) + 16 * q4);
#pragma unroll
                for (int i = 0; i < 4; ++i) av[j][4 * q4 + i] = v[i];
            }
        sa = g.sum_a[0];
    }
    float sc[RPW];
#pragma unroll
    for (int r = 0; r < RPW; ++r) sc[r] = g.scales[(row0 + r)];
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
        float acc = 0.0f;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint32_t lo = wv[r][j][k] & 0x0F0F0F0Fu, hi = (wv[r][j][k] >> 4) & 0x0F0F0F0Fu;
#pragma unroll
                for (int b = 0; b < 4; ++b) {  // byte b: low nibble = value 2b, high = 2b + 1
                    acc = __builtin_fmaf((float)((lo >> (8 * b)) & 0xFFu), av[j][8 * k + 2 * b], acc);
                    acc = __builtin_fmaf((float)((hi >> (8 * b)) & 0xFFu), av[j][8 * k + 2 * b + 1], acc);
                }
            }
        acc = wave_sum(acc);
        if (lane == 0) g.out[mat][r0 + r] = srq(sc[r] * (acc - 8.0f * sa), g.out_scale[mat]);
    }
}

// ---------------------------------------------------------------- the GEMMs' activation
// srqh_b (kernels_dsl.py:232-242): out = f16(srq(a, s)), 8 values per thread.
__global__ __launch_bounds__(256) void srqh_kernel(const float* __restrict__ a, float s, half_t* __restrict__ out,
                                                   int n8) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n8) return;
    const float4v x0 = reinterpret_cast<const float4v*>(a)[2 * i];
    const float4v x1 = reinterpret_cast<const float4v*>(a)[2 * i + 1];
    half8 h;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        h[j] = (half_t)srq(x0[j], s);
        h[4 + j] = (half_t)srq(x1[j], s);
    }
    reinterpret_cast<half8*>(out)[i] = h;
}

}  // namespace g4a

using namespace g4a;

extern "C" int g4a_srqh(int n, const float* a, float a_in_q, void* out_f16, void* stream) {
    if (n <= 0 || n % 8) {
        set_error("n (%d) must be a positive multiple of 8", n);
        return G4A_EINVAL;
    }
    if (!a || !out_f16 || (((uintptr_t)a | (uintptr_t)out_f16) & 15)) {
        set_error("a and out must be non-NULL and 16-byte aligned");
        return G4A_EINVAL;
    }
    if (!(a_in_q >= 0.0f)) {
        set_error("a_in_q must be >= 0");
        return G4A_EINVAL;
    }
    const int n8 = n / 8;
    hipLaunchKernelGGL(srqh_kernel, dim3((n8 + 255) / 256), dim3(256), 0, (hipStream_t)stream, a, a_in_q,
                       reinterpret_cast<half_t*>(out_f16), n8);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_error(e, "srqh launch");
    return G4A_OK;
}

extern "C" int g4a_dequant(int bits, int n_in, int n_out, const uint32_t* w_bits, const float* w_scale,
                           void* out_f16, void* stream) {
    if (bits != 2 && bits != 4 && bits != 8) {
        set_error("bits %d not supported (2, 4 or 8)", bits);
        return G4A_EUNSUPPORTED;
    }
    if (n_in <= 0 || n_out <= 0 || n_in % (128 / bits) || (int64_t)n_in * n_out > 0x7fffffff) {
        set_error("n_in (%d) must be a positive multiple of %d and n_in*n_out < 2^31 (n_out %d)", n_in,
                  128 / bits, n_out);
        return G4A_EINVAL;
    }
    if (!w_bits || !w_scale || !out_f16) {
        set_error("w_bits, w_scale and out must be non-NULL");
        return G4A_EINVAL;
    }
    if (((uintptr_t)w_bits | (uintptr_t)out_f16) & 15) {
        set_error("w_bits and out must be 16-byte aligned");
        return G4A_EINVAL;
    }
    const int n_quads = (int)((int64_t)n_out * n_in / (128 / bits));
    const dim3 grid((n_quads + 255) / 256);
    half_t* o = reinterpret_cast<half_t*>(out_f16);
    if (bits == 2) hipLaunchKernelGGL(dequant_kernel<2>, grid, dim3(256), 0, (hipStream_t)stream, w_bits, w_scale, o, n_in, n_quads);
    if (bits == 4) hipLaunchKernelGGL(dequant_kernel<4>, grid, dim3(256), 0, (hipStream_t)stream, w_bits, w_scale, o, n_in, n_quads);
    if (bits == 8) hipLaunchKernelGGL(dequant_kernel<8>, grid, dim3(256), 0, (hipStream_t)stream, w_bits, w_scale, o, n_in, n_quads);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_error(e, "dequant launch");
    return G4A_OK;
}

static int qkv_run(int hidden, int q_dim, int kv_dim, const float* a, const float* sum_a,
                   const g4a_norm_in* pro, float* sum_out, const uint32_t* q_bits, const uint32_t* k_bits,
                   const uint32_t* v_bits, const float* scales, float q_out, float k_out, float v_out,
                   float* out_q, float* out_k, float* out_v, void* stream) {
    if (hidden <= 0 || hidden % 32 || hidden > (pro ? 2048 : 4096)) {
        set_error("hidden (%d) must be a positive multiple of 32, at most %d", hidden, pro ? 2048 : 4096);
        return G4A_EINVAL;
    }
    if (pro) {
        if (!pro->a || !pro->res || !pro->w1 || !pro->w2 || pro->f16 || !(pro->q2 >= 0.0f) || !(pro->eps >= 0.0f)) {
            set_error("qkv norm prologue: a, res, w1 and w2 non-NULL, f16 0, q2 and eps >= 0");
            return G4A_EINVAL;
        }
        if (((uintptr_t)pro->a | (uintptr_t)pro->res | (uintptr_t)pro->w1 | (uintptr_t)pro->w2 |
             (uintptr_t)pro->x_out | (uintptr_t)pro->z_out) & 15) {
            set_error("qkv norm prologue: vectors must be 16-byte aligned");
            return G4A_EINVAL;
        }
        // workgroup 0 stores x and z while the others still read a, res and w1
        const size_t vb = (size_t)hidden * sizeof(float);
        for (const void* out : {(const void*)pro->x_out, (const void*)pro->z_out})
            if (overlaps(out, pro->a, vb) || overlaps(out, pro->res, vb) || overlaps(out, pro->w1, vb)) {
                set_error("qkv norm prologue: x_out and z_out must not overlap a, res or w1");
                return G4A_EINVAL;
            }
        a = pro->a;  // checked as the input below; the prologue makes the real one
        sum_a = pro->a;
    }
    if (q_dim <= 0 || q_dim % 8 || kv_dim < 0 || kv_dim % 8) {
        set_error("q_dim (%d) must be a positive and kv_dim (%d) a non-negative multiple of 8", q_dim, kv_dim);
        return G4A_EINVAL;
    }
    if (!a || !sum_a || !q_bits || !scales || !out_q || (kv_dim && (!k_bits || !v_bits || !out_k || !out_v))) {
        set_error("a, sum_a, q_bits, scales, out_q (and with kv_dim > 0 k_bits, v_bits, out_k, out_v) "
                  "must be non-NULL");
        return G4A_EINVAL;
    }
    if (((uintptr_t)a | (uintptr_t)q_bits | (uintptr_t)k_bits | (uintptr_t)v_bits) & 15) {
        set_error("a and the packed weights must be 16-byte aligned");
        return G4A_EINVAL;
    }
    if ((int64_t)q_dim * hidden / 2 > 0x7fffffff) {
        set_error("q rows beyond 32-bit buffer offsets");
        return G4A_EINVAL;
    }
    if (!(q_out >= 0.0f) || !(k_out >= 0.0f) || !(v_out >= 0.0f)) {
        set_error("q_out/k_out/v_out must be >= 0");
        return G4A_EINVAL;
    }
    GemvArgs g;
    g.a = a;
    g.sum_a = sum_a;
    g.bits[0] = q_bits;
    g.bits[1] = k_bits;
    g.bits[2] = v_bits;
    g.scales = scales;
    g.out[0] = out_q;
    g.out[1] = out_k;
    g.out[2] = out_v;
    g.out_scale[0] = q_out;
    g.out_scale[1] = k_out;
    g.out_scale[2] = v_out;
    g.hidden = hidden;
    g.q_dim = q_dim;
    g.kv_dim = kv_dim;
    g.pa = pro ? pro->a : nullptr;
    g.pres = pro ? pro->res : nullptr;
    g.pw1 = pro ? pro->w1 : nullptr;
    g.pw2 = pro ? pro->w2 : nullptr;
    g.pxout = pro ? pro->x_out : nullptr;
    g.pzout = pro ? pro->z_out : nullptr;
    g.psum = sum_out;
    g.pq2 = pro ? pro->q2 : 0.0f;
    g.peps = pro ? pro->eps : 0.0f;
    g.pmult = pro && pro->mult != 0.0f ? pro->mult : 1.0f;
    const int total = q_dim + 2 * kv_dim;  // rows; 2 per wave, 8 per workgroup
    const dim3 grid(total / 8);
    if (pro)
        hipLaunchKernelGGL((qkv_gemv_kernel<1, 2, true>), grid, dim3(256), 0, (hipStream_t)stream, g);
    else if (hidden <= 2048)
        hipLaunchKernelGGL((qkv_gemv_kernel<1, 2, false>), grid, dim3(256), 0, (hipStream_t)stream, g);
    else
        hipLaunchKernelGGL((qkv_gemv_kernel<2, 2, false>), grid, dim3(256), 0, (hipStream_t)stream, g);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_error(e, "qkv_gemv launch");
    return G4A_OK;
}

extern "C" int g4a_qkv_gemv(int hidden, int q_dim, int kv_dim, const float* a, const float* sum_a,
                            const uint32_t* q_bits, const uint32_t* k_bits, const uint32_t* v_bits,
                            const float* scales, float q_out, float k_out, float v_out, float* out_q,
                            float* out_k, float* out_v, void* stream) {
    return qkv_run(hidden, q_dim, kv_dim, a, sum_a, nullptr, nullptr, q_bits, k_bits, v_bits, scales, q_out, k_out,
                   v_out, out_q, out_k, out_v, stream);
}

extern "C" int g4a_qkv_gemv_norm(int hidden, int q_dim, int kv_dim, const g4a_norm_in* pro, float* sum_out,
                                 const uint32_t* q_bits, const uint32_t* k_bits, const uint32_t* v_bits,
                                 const float* scales, float q_out, float k_out, float v_out, float* out_q,
                                 float* out_k, float* out_v, void* stream) {
    if (!pro) {
        set_error("pro must be non-NULL (g4a_qkv_gemv takes a made input)");
        return G4A_EINVAL;
    }
    return qkv_run(hidden, q_dim, kv_dim, nullptr, nullptr, pro, sum_out, q_bits, k_bits, v_bits, scales, q_out,
                   k_out, v_out, out_q, out_k, out_v, stream);
}
