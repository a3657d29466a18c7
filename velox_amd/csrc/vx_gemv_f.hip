// vx_gemv_f.hip -- the decode step's GEMV over unquantized weights: the reference's quant_mode 0
// (fp32) and 1 (fp16) rows, stored row-major [rows][k] as the reference's weight arena holds them
// (src/codegen.rs:1024-1028; its emitted velox_cuda_matmul_vec_kernel, src/codegen.rs:1154, and
// velox_cuda_matmul_vec_kernel_f16 / velox_warp_dot_f16, src/codegen.rs:2267-2311, 2412-2420).
// Benchmark configuration 1, the fp32 SmolLM, runs on this kernel.
//
// Same contract as the Q4_0 GEMV (vx_launch_gemv picks this kernel from the matrix format): the
// input (or the LSE merge of split attention partials) goes into LDS as fp32 (RMSNorm: times the
// gain, 1 / rms applied to each row's result); each wave takes single logical rows (SwiGLU: a gate
// row and its up row, stored as n gate rows followed by n up rows), its lanes stride over the row in
// 16-byte words (4 fp32 or 8 fp16 weights), fp32 FMAs, then a 64-lane sum. Epilogues: store (+bias),
// residual add, SwiGLU, or the per-workgroup (max, index) candidate of the LM head.
//
// What bounds it: HBM for wide matrices, the first bytes' latency for SmolLM's (0.3-7 MB a launch).
// Both want every CU to hold loads from the start: one row per wave puts SmolLM's 576-1536 rows on
// 192-256 workgroups (tiles of 4 rows filled 18-48), each wave's first U words are requested
// before the input is staged (they arrive while it is), and the ring of words in flight runs on over
// row ends.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "vx_common.h"

namespace {

constexpr int kFWaves = 8, kFThreads = 64 * kFWaves;  // at most; the launcher picks 1..8 waves
constexpr uint32_t kFPad = 8;                          // zeros after the row's activations: one word's worth
constexpr uint32_t vf_lds(uint32_t k) { return (k + kFPad + 2u * kFWaves) * 4u; }

typedef uint32_t vf_u4 __attribute__((ext_vector_type(4)));
typedef float vf_f4 __attribute__((ext_vector_type(4)));

template <int CTRL>
__device__ __forceinline__ float vf_dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}

// Sum over the 64 lanes (in every lane): quad_perm xor 1 / xor 2, row half mirror, row mirror, then
// two lane exchanges across the 16-lane rows.
__device__ __forceinline__ float vf_wave_sum(float v) {
    v += vf_dpp<0xB1>(v);
    v += vf_dpp<0x4E>(v);
    v += vf_dpp<0x141>(v);
    v += vf_dpp<0x140>(v);
    v += __shfl_xor(v, 16);
    return v + __shfl_xor(v, 32);
}

__device__ __forceinline__ bool vf_better(float v, uint32_t i, float bv, uint32_t bi) {
    return v > bv || (v == bv && i < bi);
}

// 16 bytes of weights times the matching activations in LDS, accumulated in fp32 (one sum per
// 16-byte column: four independent chains)
template <typename T>
__device__ __forceinline__ void vf_dot16(const vf_u4& w, const float* x, vf_f4& acc);

template <>
__device__ __forceinline__ void vf_dot16<float>(const vf_u4& w, const float* x, vf_f4& acc) {
    const float4 xv = *(const float4*)x;
    acc.x = fmaf(__uint_as_float(w.x), xv.x, acc.x);
    acc.y = fmaf(__uint_as_float(w.y), xv.y, acc.y);
    acc.z = fmaf(__uint_as_float(w.z), xv.z, acc.z);
    acc.w = fmaf(__uint_as_float(w.w), xv.w, acc.w);
}

template <>
__device__ __forceinline__ void vf_dot16<__half>(const vf_u4& w, const float* x, vf_f4& acc) {
    const float4 x0 = *(const float4*)x, x1 = *(const float4*)(x + 4);
    const uint32_t d[4] = {w.x, w.y, w.z, w.w};
    const float xv[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        acc[i] = fmaf(__half2float(__ushort_as_half((unsigned short)(d[i] & 0xFFFFu))), xv[2 * i], acc[i]);
        acc[i] = fmaf(__half2float(__ushort_as_half((unsigned short)(d[i] >> 16))), xv[2 * i + 1], acc[i]);
    }
}

template <typename T, int EPI, bool NORM, int SPL>
__global__ __launch_bounds__(kFThreads) void vx_gemv_f_kernel(VxMat m, VxGemvArgs a) {
    extern __shared__ __align__(16) float vf_smem[];
    if ((a.active_mask & 1ULL) == 0ULL) return;
    constexpr uint32_t E = 16u / sizeof(T);     // weights per 16-byte word
    constexpr int PR = EPI == VX_EPI_SWIGLU ? 2 : 1;
    constexpr int U = PR == 2 ? 4 : 8;          // items in flight per wave: 8 KiB
    constexpr int GX = SPL > 0 ? 1 : NORM ? 2 : 4;  // float4 of x per thread requested before the weights
    const uint32_t K = m.k, K4 = K / 4u;
    float* xs = vf_smem;
    float* red = vf_smem + K + kFPad;  // [kFWaves] partial sums, then the argmax candidates
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t nwv = blockDim.x >> 6, nth = blockDim.x;

    // ---- x (or the splits' partials) requested first: loads return in order ----
    float4 xv[GX], gv[GX], po[GX][SPL ? SPL : 1];
    float2 pml[GX][SPL ? SPL : 1];
    auto load_x = [&](int g, uint32_t i) {
        if constexpr (SPL == 0) {
            xv[g] = ((const float4*)a.x)[i];
        } else {
            const uint32_t k = 4u * i, h = k / a.att_d, e0 = k - h * a.att_d;
#pragma unroll
            for (int sp = 0; sp < SPL; ++sp) {
                pml[g][sp] = *(const float2*)(a.part_ml + ((size_t)h * SPL + sp) * 2u);
                po[g][sp] = *(const float4*)(a.part_o + ((size_t)h * SPL + sp) * a.att_d + e0);
            }
        }
        if constexpr (NORM) gv[g] = ((const float4*)a.gain)[i];
    };
#pragma unroll
    for (int g = 0; g < GX; ++g) load_x(g, min((uint32_t)tid + (uint32_t)g * nth, K4 - 1u));
    __builtin_amdgcn_sched_barrier(0);

    // ---- the wave's rows: workgroup b owns a contiguous block, dealt to its waves; items are the
    // (row, 64 words) pairs in order ----
    const uint32_t b0 = (uint32_t)(((uint64_t)blockIdx.x * m.n) / gridDim.x);
    const uint32_t b1 = (uint32_t)(((uint64_t)(blockIdx.x + 1u) * m.n) / gridDim.x);
    const uint32_t nw = K / E, nit = (nw + 63u) / 64u;
    const uint32_t r0 = b0 + (uint32_t)wave, total = r0 < b1 ? (b1 - r0 + nwv - 1u) / nwv * nit : 0u;
    const uint8_t* wbase = (const uint8_t*)m.codes;
    const size_t row_bytes = (size_t)K * sizeof(T);
    vf_u4 w[U][PR];
    uint32_t nr = r0, ni = 0;  // next item
    // unconditional: past the wave's last item the block's first row is read again, past a row's
    // last word that word (in bounds, the value unused)
    auto issue = [&](int u) {
        const uint32_t row = __builtin_amdgcn_readfirstlane(nr < b1 ? nr : b0);
        const uint32_t c = min(ni * 64u + (uint32_t)lane, nw - 1u);
#pragma unroll
        for (int p = 0; p < PR; ++p)
            w[u][p] = __builtin_nontemporal_load((const vf_u4*)(wbase + (size_t)(p ? m.n + row : row) * row_bytes) + c);
        if (++ni == nit) {
            ni = 0;
            nr += nwv;
        }
    };
#pragma unroll
    for (int u = 0; u < U; ++u) issue(u);
    __builtin_amdgcn_sched_barrier(0);

    // ---- x into LDS (RMSNorm: x * gain, and the sum of squares; src/runtime.rs:588-601) ----
    float ss = 0.0f;
    auto stage = [&](int g, uint32_t i) {
        float4 v;
        if constexpr (SPL == 0) {
            v = xv[g];
        } else {
            // LSE merge of the splits (m, l in the log2 domain; an empty split has m = -inf, l = 0),
            // the merge of tests/empirical_challenge_phase2/test2_split_k_flashdecoding_parity.cu:23-125
            float M = -INFINITY;
#pragma unroll
            for (int sp = 0; sp < SPL; ++sp) M = fmaxf(M, pml[g][sp].x);
            float L = 0.0f, wt[SPL ? SPL : 1];
#pragma unroll
            for (int sp = 0; sp < SPL; ++sp) {
                wt[sp] = pml[g][sp].x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(pml[g][sp].x - M);
                L += wt[sp] * pml[g][sp].y;
            }
            const float invl = L > 0.0f ? 1.0f / L : 0.0f;
            v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int sp = 0; sp < SPL; ++sp) {
                const float ws = wt[sp] * invl;
                v.x += ws * po[g][sp].x; v.y += ws * po[g][sp].y; v.z += ws * po[g][sp].z; v.w += ws * po[g][sp].w;
            }
        }
        if constexpr (NORM) {
            ss += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
            v = make_float4(v.x * gv[g].x, v.y * gv[g].y, v.z * gv[g].z, v.w * gv[g].w);
        }
        ((float4*)xs)[i] = v;
    };
#pragma unroll
    for (int g = 0; g < GX; ++g)
        if ((uint32_t)tid + (uint32_t)g * nth < K4) stage(g, (uint32_t)tid + (uint32_t)g * nth);
    for (uint32_t i = (uint32_t)tid + GX * nth; i < K4; i += nth) {
        load_x(0, i);
        stage(0, i);
    }
    if (tid < (int)kFPad) xs[K + tid] = 0.0f;
    if constexpr (NORM) {
        ss = vf_wave_sum(ss);
        if (lane == 0) red[wave] = ss;
    }
    __syncthreads();
    float inv_rms = 1.0f;
    if constexpr (NORM) {
        float tot = 0.0f;
        for (uint32_t v = 0; v < nwv; ++v) tot += red[v];
        inv_rms = 1.0f / sqrtf(tot / (float)K + a.eps);
        if (!(tot < 1e30f)) {  // (workgroup-uniform) x may pass 1e15: 1 / rms goes first, or the sums overflow before it
            for (uint32_t i = (uint32_t)tid; i < K4; i += nth) {
                const float4 v = ((const float4*)a.x)[i], g = ((const float4*)a.gain)[i];
                ((float4*)xs)[i] = make_float4((v.x * inv_rms) * g.x, (v.y * inv_rms) * g.y, (v.z * inv_rms) * g.z,
                                               (v.w * inv_rms) * g.w);
            }
            inv_rms = 1.0f;
            __syncthreads();
        }
    }

    // ---- stream: consume item u, refill it with the item U ahead, finish rows on the fly ----
    float best_v = -INFINITY;
    uint32_t best_i = 0xFFFFFFFFu;
    vf_f4 acc[PR];
#pragma unroll
    for (int p = 0; p < PR; ++p) acc[p] = vf_f4{0.f, 0.f, 0.f, 0.f};
    uint32_t ci = 0, j = r0;  // current item
    auto consume = [&](int u) {
        const uint32_t c = ci * 64u + (uint32_t)lane;
        const bool in = c < nw;  // past the row's end: zero weights, and the zeros after xs (0 times infinity is no 0)
        const float* x = xs + min(c, nw) * E;
#pragma unroll
        for (int p = 0; p < PR; ++p) {
            vf_u4 q = w[u][p];
            q.x = in ? q.x : 0u; q.y = in ? q.y : 0u; q.z = in ? q.z : 0u; q.w = in ? q.w : 0u;
            vf_dot16<T>(q, x, acc[p]);
        }
        if (++ci == nit) {
            float v[PR];
#pragma unroll
            for (int p = 0; p < PR; ++p) {
                v[p] = vf_wave_sum((acc[p].x + acc[p].y) + (acc[p].z + acc[p].w));
                if constexpr (NORM) v[p] *= inv_rms;
                acc[p] = vf_f4{0.f, 0.f, 0.f, 0.f};
            }
            if (lane == 0) {
                if constexpr (EPI == VX_EPI_STORE) {
                    a.y[j] = a.bias ? v[0] + a.bias[j] : v[0];
                } else if constexpr (EPI == VX_EPI_RESID) {
                    a.y[j] = a.res[j] + v[0];
                } else if constexpr (EPI == VX_EPI_SWIGLU) {
                    a.y[j] = (v[0] / (1.0f + expf(-v[0]))) * v[PR - 1];  // src/runtime.rs:1064-1066
                } else {  // VX_EPI_ARGMAX
                    a.y[j] = v[0];
                    if (vf_better(v[0], j, best_v, best_i)) { best_v = v[0]; best_i = j; }
                }
            }
            ci = 0;
            j += nwv;
        }
    };
    uint32_t f0 = 0;
    for (; f0 + 2u * U <= total; f0 += U) {  // steady state: every refill is a real item of this wave
#pragma unroll
        for (int u = 0; u < U; ++u) {
            consume(u);
            issue(u);
        }
    }
    for (; f0 < total; f0 += U) {  // the last (< 2 U) items
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (f0 + u < total) {
                consume(u);
                if (f0 + u + U < total) issue(u);
            }
        }
    }
    if constexpr (EPI == VX_EPI_ARGMAX) {
        __syncthreads();  // red[] is reused
        if (lane == 0) {
            red[wave] = best_v;
            ((uint32_t*)red)[kFWaves + wave] = best_i;
        }
        __syncthreads();
        if (tid == 0) {
            float bv = red[0];
            uint32_t bi = ((const uint32_t*)red)[kFWaves];
            for (uint32_t v = 1; v < nwv; ++v)
                if (vf_better(red[v], ((const uint32_t*)red)[kFWaves + v], bv, bi)) {
                    bv = red[v];
                    bi = ((const uint32_t*)red)[kFWaves + v];
                }
            a.cand_v[blockIdx.x] = bv;
            a.cand_i[blockIdx.x] = bi;
        }
    }
}

}  // namespace

// Grid: 1..8 waves per workgroup so that up to 2048 rows, one per wave, make at most 256 workgroups
// (SmolLM's 576-1536 rows: 192-256); up to 8192 rows one row per wave in 8-wave workgroups (the wave's
// first U words of its row, all of a short one, are then requested at once: Llama-3-8B's 4096-row down
// projection in fp16 20.6 us on 512 workgroups, 21.0 with max_wgs = 256), where a CU's LDS and 32 waves hold
// them all in one round; otherwise, and for more rows, max_wgs workgroups, each wave streaming several rows
// (Llama-3-8B's gate/up, 28672 rows: 36.1 us, 6.5 TB/s; Qwen2-72B's down, 8192 rows of 29568 in 118 KB of LDS:
// four rounds of 256 workgroups, each staging the activations again, 83.7 us, one 80.0; its o_proj, 8192 rows of
// 8192, is one round of 1024, 27.8 us, 27.3 on 256). The LM head's grid is the caller's (its finalize
// kernel reads one candidate per workgroup). Against tiles of 4 rows per wave, kernel trace: SmolLM
// fp32 gate/up 7.0 -> 3.2 us, down 6.9 -> 2.8, QKV 5.2 -> 2.9, o_proj 5.4 -> 3.2; Llama-3-8B fp16
// gate/up 43.8 -> 36.1, down 28.7 -> 20.6, QKV 14.2 -> 10.6, o_proj 11.6 -> 9.0 us; Qwen2-72B fp16 o_proj
// 32.6 -> 27.8, down 81.0 -> 80.0.
extern "C" void vx_gemv_f_grid(uint32_t n, uint32_t k, int epi, uint32_t head_wgs, uint32_t max_wgs, uint32_t* wgs,
                               uint32_t* waves) {
    *waves = min((n + 255u) / 256u, (uint32_t)kFWaves);
    if (epi == VX_EPI_ARGMAX) {
        *waves = kFWaves;
        *wgs = head_wgs;
        return;
    }
    *wgs = (n + *waves - 1u) / *waves;
    const uint32_t per_cu = min(160u * 1024u / vf_lds(k), 4u);
    if (n > 8192u || *wgs > 256u * per_cu) *wgs = min(*wgs, max_wgs ? max_wgs : 1u);
}

namespace {

template <typename T, int EPI, bool NORM, int SPL>
hipError_t vx_gemv_f_launch_t(const VxMat& m, const VxGemvArgs& a, dim3 grid, hipStream_t st) {
    const size_t lds = vf_lds(m.k);
    // rows wider than 16360 need more than the default 64 KiB of dynamic LDS (up to 128 KiB + 96 B
    // at kVxFloatMaxK, of the 160 KiB a CU has): raised once per instantiation to the widest row
    static bool attr_set = false;
    if (lds > 65536u && !attr_set) {
        if (hipFuncSetAttribute((const void*)vx_gemv_f_kernel<T, EPI, NORM, SPL>,
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)vf_lds(kVxFloatMaxK)) != hipSuccess) {
            (void)hipGetLastError();
            return hipErrorInvalidValue;
        }
        attr_set = true;
    }
    hipLaunchKernelGGL((vx_gemv_f_kernel<T, EPI, NORM, SPL>), dim3(grid.x), dim3(64 * grid.y), lds, st, m, a);
    return hipGetLastError();
}

template <typename T, int EPI>
hipError_t vx_gemv_f_dispatch(const VxMat& m, const VxGemvArgs& a, dim3 grid, hipStream_t st) {
    if constexpr (EPI == VX_EPI_RESID) {
        if (a.gain) return hipErrorInvalidValue;  // the residual epilogue takes raw activations
        if (!a.part_o) return vx_gemv_f_launch_t<T, EPI, false, 0>(m, a, grid, st);
        if (!a.part_ml || a.att_d == 0 || (a.att_d & 3u) || m.k % a.att_d) return hipErrorInvalidValue;
        switch (a.att_splits) {
            case 1: return vx_gemv_f_launch_t<T, EPI, false, 1>(m, a, grid, st);
            case 2: return vx_gemv_f_launch_t<T, EPI, false, 2>(m, a, grid, st);
            case 4: return vx_gemv_f_launch_t<T, EPI, false, 4>(m, a, grid, st);
            case 8: return vx_gemv_f_launch_t<T, EPI, false, 8>(m, a, grid, st);
            default: return hipErrorInvalidValue;
        }
    } else {
        if (a.part_o) return hipErrorInvalidValue;
        return a.gain ? vx_gemv_f_launch_t<T, EPI, true, 0>(m, a, grid, st)
                      : vx_gemv_f_launch_t<T, EPI, false, 0>(m, a, grid, st);
    }
}

template <typename T>
hipError_t vx_gemv_f_epi(const VxMat& m, const VxGemvArgs& a, int epi, dim3 grid, hipStream_t st) {
    switch (epi) {
        case VX_EPI_STORE: return vx_gemv_f_dispatch<T, VX_EPI_STORE>(m, a, grid, st);
        case VX_EPI_RESID: return vx_gemv_f_dispatch<T, VX_EPI_RESID>(m, a, grid, st);
        case VX_EPI_SWIGLU: return vx_gemv_f_dispatch<T, VX_EPI_SWIGLU>(m, a, grid, st);
        case VX_EPI_ARGMAX: return vx_gemv_f_dispatch<T, VX_EPI_ARGMAX>(m, a, grid, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

hipError_t vx_launch_gemv_f(const VxMat& m, const VxGemvArgs& a, int epi, uint32_t head_wgs, uint32_t max_wgs,
                            hipStream_t st) {
    if (m.k == 0 || (m.k & 7u) || m.k > kVxFloatMaxK || m.n == 0) return hipErrorInvalidValue;
    if ((epi == VX_EPI_SWIGLU) != (m.paired != 0)) return hipErrorInvalidValue;
    if (epi == VX_EPI_ARGMAX && (!a.cand_v || !a.cand_i)) return hipErrorInvalidValue;
    uint32_t wgs, waves;
    vx_gemv_f_grid(m.n, m.k, epi, head_wgs, max_wgs, &wgs, &waves);
    const dim3 grid(wgs, waves);  // (workgroups, waves per workgroup)
    if (m.fmt == VX_FMT_F32) return vx_gemv_f_epi<float>(m, a, epi, grid, st);
    if (m.fmt == VX_FMT_F16) return vx_gemv_f_epi<__half>(m, a, epi, grid, st);
    return hipErrorInvalidValue;
}
