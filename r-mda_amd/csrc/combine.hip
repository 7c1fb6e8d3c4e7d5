// Weighted gather-sum of expert outputs back to token order.
//
// combine_ref_kernel restates shader/moe_combine.comp:26-40 (fp32 expert
// rows `y`, shared-expert term, hyper-connection streams h += acc * 2 *
// sigmoid(inj / hc)), plus a plain fp16 output mode.  One thread per output
// element, like the reference.
//
// combine32_kernel is its bandwidth version for the drop-in entry points
// (d % 4 == 0; combine_ref_kernel remains for other d).
//
// combine16_kernel is the fused layer's version: fp16 expert rows, fp16
// output and/or the hyper-connection streams.  Each thread handles 8
// consecutive columns of a token with 16-byte loads of every selected row,
// accumulating in fp32 in j order (the reference's order, :32-34) before the
// shared-expert term (:35).
#include <algorithm>

#include "common.h"

namespace {

__device__ __forceinline__ float sigmoidf(float v) {
    return rmda_sigmoidf(v);
}

__global__ __launch_bounds__(256) void combine_ref_kernel(rmda_pc_moe_combine_t pc,
                                                          const float *__restrict__ wt,
                                                          const uint32_t *__restrict__ slot,
                                                          const float *__restrict__ y,
                                                          const float *__restrict__ proj,
                                                          const float *__restrict__ sh,
                                                          const float *__restrict__ inj,
                                                          float *__restrict__ h,
                                                          uint16_t *__restrict__ out) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (uint64_t)pc.rows * pc.d) {
        return;
    }
    const uint32_t r = (uint32_t)(i / pc.d);
    const uint32_t c = (uint32_t)(i % pc.d);
    float acc = 0.0f;
    for (uint32_t j = 0; j < pc.topk; j += 1) {
        const uint32_t s = slot[(size_t)r * pc.topk + j];
        if (s != RMDA_NONE) {
            acc += wt[(size_t)r * pc.topk + j] * y[(size_t)s * pc.d + c];
        }
    }
    if (sh != nullptr) {
        acc += sigmoidf(proj[(size_t)r * pc.pstride + pc.sg_off]) * sh[i];
    }
    if (out != nullptr) {
        out[i] = rmda_f2h(acc);
        return;
    }
    for (uint32_t s = 0; s < pc.hc; s += 1) {
        const float gte = sigmoidf(inj[(size_t)r * pc.inj_stride + pc.inj_off + s] / (float)pc.hc);
        h[(size_t)r * pc.hc * pc.d + (size_t)s * pc.d + c] += acc * 2.0f * gte;
    }
}

// The drop-in combine (rmda_moe_combine / _plain) at bandwidth: the same
// arithmetic as combine_ref_kernel per element (fp32 y rows, acc += wt*y in
// j order, then the shared term, then the hc streams and/or the fp16 output),
// one wave per token and 256 columns, 4 columns per lane.  Needs d % 4 == 0.
//
// What bounds it: HBM; y is read once, the streams read and written once.  All
// of a wave's loads (the streams, the shared row, up to KB rows of y) are in
// flight before the first sum, and y and the streams pass the caches as
// non-temporal.  A workgroup per token that read its rows one after another
// took (MI355X) 62 us for 2048 tokens of hidden 2048, top-8, four streams (268
// MB), 44 us now; with the plain output 36 -> 23 us.  Non-temporal pays where
// the rows come from HBM, as they do after the GEMM that writes them (the same
// call on three sets of buffers in turn 45 us, with ordinary accesses 55); on
// one set, which the Infinity Cache holds, ordinary accesses take 40 us.
template <bool HC, uint32_t KB>
__global__ __launch_bounds__(256) void combine32_kernel(rmda_pc_moe_combine_t pc, uint32_t waves,
                                                        const float *__restrict__ wt,
                                                        const uint32_t *__restrict__ slot,
                                                        const float *__restrict__ y,
                                                        const float *__restrict__ proj,
                                                        const float *__restrict__ sh,
                                                        const float *__restrict__ inj,
                                                        float *__restrict__ h,
                                                        uint16_t *__restrict__ out) {
    const uint32_t d4 = pc.d / 4;
    const uint32_t cw = (d4 + RMDA_WAVE - 1) / RMDA_WAVE;  // waves per token
    const uint32_t wid =
        blockIdx.x * (blockDim.x / RMDA_WAVE) + __builtin_amdgcn_readfirstlane(threadIdx.x / RMDA_WAVE);
    const uint32_t r = wid / cw;
    const uint32_t c = (wid - r * cw) * RMDA_WAVE + threadIdx.x % RMDA_WAVE;
    if (wid >= waves || c >= d4) {
        return;
    }
    constexpr uint32_t HB = 4;  // streams read ahead
    floatx4_t hv[HB];
    auto stream = [&](uint32_t st) __attribute__((always_inline)) {
        return reinterpret_cast<floatx4_t *>(h + ((size_t)r * pc.hc + st) * pc.d) + c;
    };
    auto load_streams = [&](uint32_t st0) __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t i = 0; i < HB; i += 1) {
            if (st0 + i < pc.hc) {
                hv[i] = __builtin_nontemporal_load(stream(st0 + i));
            }
        }
    };
    if (HC) {
        load_streams(0);
    }
    floatx4_t sv = {0.0f, 0.0f, 0.0f, 0.0f};
    float sg = 0.0f;
    if (sh != nullptr) {
        sv = __builtin_nontemporal_load(reinterpret_cast<const floatx4_t *>(sh + (size_t)r * pc.d) + c);
        sg = sigmoidf(proj[(size_t)r * pc.pstride + pc.sg_off]);
    }
    const floatx4_t *const yc = reinterpret_cast<const floatx4_t *>(y) + c;
    floatx4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for (uint32_t j0 = 0; j0 < pc.topk; j0 += KB) {
        floatx4_t q[KB];
        uint32_t s[KB];
        float w[KB];
#pragma unroll
        for (uint32_t j = 0; j < KB; j += 1) {
            const size_t i = (size_t)r * pc.topk + min(j0 + j, pc.topk - 1u);
            s[j] = slot[i];
            w[j] = wt[i];
        }
#pragma unroll
        for (uint32_t j = 0; j < KB; j += 1) {
            if (j0 + j < pc.topk && s[j] != RMDA_NONE) {
                q[j] = __builtin_nontemporal_load(yc + (size_t)s[j] * d4);
            }
        }
#pragma unroll
        for (uint32_t j = 0; j < KB; j += 1) {
            if (j0 + j < pc.topk && s[j] != RMDA_NONE) {
#pragma unroll
                for (int v = 0; v < 4; v += 1) {
                    acc[v] += w[j] * q[j][v];
                }
            }
        }
    }
    if (sh != nullptr) {
#pragma unroll
        for (int v = 0; v < 4; v += 1) {
            acc[v] += sg * sv[v];
        }
    }
    if (out != nullptr) {
        uint2 o;
        o.x = (uint32_t)rmda_f2h(acc[0]) | ((uint32_t)rmda_f2h(acc[1]) << 16);
        o.y = (uint32_t)rmda_f2h(acc[2]) | ((uint32_t)rmda_f2h(acc[3]) << 16);
        reinterpret_cast<uint2 *>(out + (size_t)r * pc.d)[c] = o;
    }
    if (HC) {
        for (uint32_t st0 = 0; st0 < pc.hc; st0 += HB) {
            if (st0 > 0) {
                load_streams(st0);
            }
#pragma unroll
            for (uint32_t i = 0; i < HB; i += 1) {
                if (st0 + i < pc.hc) {
                    const float v = inj[(size_t)r * pc.inj_stride + pc.inj_off + st0 + i];
                    const float g = sigmoidf(v / (float)pc.hc);
#pragma unroll
                    for (int u = 0; u < 4; u += 1) {
                        hv[i][u] += acc[u] * 2.0f * g;
                    }
                    __builtin_nontemporal_store(hv[i], stream(st0 + i));
                }
            }
        }
    }
}

// One 16-byte slice of an expert row, read past the caches' normal retention:
// every expert row is read by exactly one token's workgroup, once.
typedef unsigned int rmda_u32x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint4 rmda_stream_load16(const uint4 *p) {
    const rmda_u32x4_t v = __builtin_nontemporal_load(reinterpret_cast<const rmda_u32x4_t *>(p));
    return make_uint4(v.x, v.y, v.z, v.w);
}

// One wave sums one token's 512 consecutive columns.  HC: the hyper-connection
// epilogue of shader/moe_combine.comp:36-38 in place of (or besides) the fp16
// output: h[r][s][c] += acc * 2 * sigmoid(inj / hc).
//
// What bounds it: HBM for many tokens, the chain slot -> row -> sum for few.
// The slots and weights are scalar loads, and the shared row and up to KB
// expert rows are all in flight before the first sum.  AHEAD: so are the
// streams' old values, for calls of few waves; with many the streams follow
// the sum one after another, which keeps the reads and writes of a stream
// together and 30 VGPRs free (four streams, read ahead against after: 2692
// tokens of hidden 2048, top-2 38.7 -> 36.5 us, 1309 of hidden 1792, top-6 23.7
// -> 23.0, 2692 of hidden 1024, top-3 23.8 -> 22.0, with the streams in the
// Infinity Cache; 44.5 -> 43.2, 28.4 -> 26.7 and 28.8 -> 27.4 without).
// A workgroup per token that read its slots through LDS and its rows one
// after another took (MI355X, by events, net of the empty interval): 16
// tokens of hidden 2560, top-10, four streams 10.7 -> 3.3 us; 128 tokens of
// hidden 2048, top-8 2.5 -> 1.2 us; 2048 tokens with the streams 49 -> 43 us
// (283 MB); 2048 tokens of hidden 2048 11.5 -> 11.0 us.  Single-wave workgroups
// spread few waves over the chip, groups of four spare the dispatcher many
// (4000 tokens of hidden 1024, top-1: 3.9 -> 3.0 us).
template <bool HC, uint32_t KB, bool AHEAD>
__global__ __launch_bounds__(256) void combine16_kernel(const float *__restrict__ wt,
                                                        const uint32_t *__restrict__ slot,
                                                        const uint16_t *__restrict__ y,
                                                        const float *__restrict__ proj,
                                                        uint32_t pstride, uint32_t sg_off,
                                                        uint32_t shared_row0, int has_shared,
                                                        uint16_t *__restrict__ out, uint32_t waves, uint32_t d,
                                                        uint32_t topk, rmda_hc_t hcp,
                                                        const uint32_t *__restrict__ run_if,
                                                        const uint32_t *__restrict__ yscale,
                                                        const uint32_t *__restrict__ ybound) {
    if (run_if != nullptr && *run_if == 0) {
        return;  // the down GEMM folded the combine in
    }
    const uint32_t d8 = d / 8;
    const uint32_t cw = (d8 + RMDA_WAVE - 1) / RMDA_WAVE;  // waves per token
    const uint32_t wid =
        blockIdx.x * (blockDim.x / RMDA_WAVE) + __builtin_amdgcn_readfirstlane(threadIdx.x / RMDA_WAVE);
    const uint32_t r = wid / cw;
    const uint32_t c = (wid - r * cw) * RMDA_WAVE + threadIdx.x % RMDA_WAVE;
    if (wid >= waves || c >= d8) {
        return;
    }
    constexpr uint32_t HB = AHEAD ? 4u : 1u;  // streams at a time
    float4 hv[HB][2];
    auto load_streams = [&](uint32_t st0) __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t i = 0; i < HB; i += 1) {
            if (st0 + i < hcp.hc) {
                const float4 *h = reinterpret_cast<const float4 *>(hcp.h + ((size_t)r * hcp.hc + st0 + i) * d) + 2 * c;
                hv[i][0] = h[0];
                hv[i][1] = h[1];
            }
        }
    };
    if (HC && AHEAD) {
        load_streams(0);
    }
    // the slot-scaled mode's rows stand for y * f, f a power of two: taken
    // into the weights, which gives the same products bit for bit
    const float f = ybound != nullptr ? rmda_slot_inv(yscale) / rmda_ye_mul(ybound) : 1.0f;
    const uint4 *const yc = reinterpret_cast<const uint4 *>(y) + c;
    uint4 sh = make_uint4(0u, 0u, 0u, 0u);
    float sw = 0.0f;
    if (has_shared) {
        sh = rmda_stream_load16(yc + (size_t)(shared_row0 + r) * d8);
        sw = sigmoidf(proj[(size_t)r * pstride + sg_off]) * f;
    }
    float acc[8];
#pragma unroll
    for (int v = 0; v < 8; v += 1) {
        acc[v] = 0.0f;
    }
    for (uint32_t j0 = 0; j0 < topk; j0 += KB) {
        uint4 q[KB];
        uint32_t s[KB];
        float w[KB];
#pragma unroll
        for (uint32_t j = 0; j < KB; j += 1) {
            const size_t i = (size_t)r * topk + min(j0 + j, topk - 1u);
            s[j] = slot[i];
            w[j] = wt[i];
        }
#pragma unroll
        for (uint32_t j = 0; j < KB; j += 1) {
            if (j0 + j < topk) {
                q[j] = rmda_stream_load16(yc + (size_t)(s[j] != RMDA_NONE ? s[j] : 0u) * d8);
            }
        }
#pragma unroll
        for (uint32_t j = 0; j < KB; j += 1) {
            if (j0 + j < topk && s[j] != RMDA_NONE) {
                rmda_comb_acc8(acc, w[j] * f, q[j]);
            }
        }
    }
    if (has_shared) {
        rmda_comb_acc8(acc, sw, sh);
    }
    if (out != nullptr) {
        reinterpret_cast<uint4 *>(out + (size_t)r * d)[c] = rmda_pack8_f16(acc);
    }
    if (HC) {
        for (uint32_t st0 = 0; st0 < hcp.hc; st0 += HB) {
            if (!AHEAD) {
                asm volatile("" ::: "memory");  // keeps the loads of all streams from moving up together
            }
            if (!AHEAD || st0 > 0) {
                load_streams(st0);
            }
#pragma unroll
            for (uint32_t i = 0; i < HB; i += 1) {
                const uint32_t st = st0 + i;
                if (st < hcp.hc) {
                    const float v = hcp.inj[(size_t)r * hcp.inj_stride + hcp.inj_off + st];
                    rmda_hc_fma8(hv[i], acc, 2.0f * sigmoidf(v / (float)hcp.hc));
                    float4 *h = reinterpret_cast<float4 *>(hcp.h + ((size_t)r * hcp.hc + st) * d) + 2 * c;
                    h[0] = hv[i][0];
                    h[1] = hv[i][1];
                }
            }
        }
    }
}

}  // namespace

hipError_t rmda_launch_combine(hipStream_t s, const rmda_pc_moe_combine_t *pc, const float *wt,
                               const uint32_t *slot, const float *y, const float *proj,
                               const float *sh, const float *inj, float *h, uint16_t *out) {
    const uint64_t n = (uint64_t)pc->rows * pc->d;
    if (n == 0) {
        return hipSuccess;
    }
    // the vector kernel reads y, sh and h as float4 and writes out as 8-byte
    // words; other alignments take the per-element kernel
    const auto al = [](const void *q, uintptr_t a) { return (reinterpret_cast<uintptr_t>(q) & (a - 1)) == 0; };
    const bool vec_ok = al(y, 16) && al(sh, 16) && al(h, 16) && al(out, 8);
    if (pc->d % 4 == 0 && pc->topk <= RMDA_MAX_TOPK && pc->hc <= RMDA_MAX_HC && vec_ok) {
        // the streams when h is given, the fp16 output when out is (both
        // for the fused layer's slot-scaled mode)
        const bool streams = h != nullptr && pc->hc > 0;
        const auto kernel = streams ? (pc->topk <= 2 ? combine32_kernel<true, 2> : combine32_kernel<true, 8>)
                                    : (pc->topk <= 2 ? combine32_kernel<false, 2> : combine32_kernel<false, 8>);
        const uint32_t cw = (pc->d / 4 + RMDA_WAVE - 1) / RMDA_WAVE;
        // one launch, unless its threads would not fit 32 bits
        const uint32_t most = std::max(1u, (1u << 25) / cw);
        for (uint32_t r0 = 0; r0 < pc->rows; r0 += most) {
            const uint32_t waves = cw * std::min(most, pc->rows - r0);
            const uint32_t wpb = waves <= 1024 ? 1u : 4u;
            hipLaunchKernelGGL(kernel, dim3((waves + wpb - 1) / wpb), dim3(wpb * RMDA_WAVE), 0, s, *pc, waves,
                               wt + (size_t)r0 * pc->topk, slot + (size_t)r0 * pc->topk, y,
                               sh != nullptr ? proj + (size_t)r0 * pc->pstride : nullptr,
                               sh != nullptr ? sh + (size_t)r0 * pc->d : nullptr,
                               streams ? inj + (size_t)r0 * pc->inj_stride : nullptr,
                               streams ? h + (size_t)r0 * pc->hc * pc->d : nullptr,
                               out != nullptr ? out + (size_t)r0 * pc->d : nullptr);
        }
        return hipGetLastError();
    }
    hipLaunchKernelGGL(combine_ref_kernel, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, s, *pc, wt, slot,
                       y, proj, sh, inj, h, out);
    return hipGetLastError();
}

hipError_t rmda_launch_combine16(hipStream_t s, const float *wt, const uint32_t *slot,
                                 const uint16_t *y, const float *proj, uint32_t pstride,
                                 uint32_t sg_off, uint32_t shared_row0, int has_shared,
                                 uint16_t *out, uint32_t rows, uint32_t d, uint32_t topk,
                                 const rmda_hc_t *hc, const uint32_t *run_if, const uint32_t *yscale,
                                 const uint32_t *ybound) {
    if (rows == 0) {
        return hipSuccess;
    }
    const bool streams = hc != nullptr && hc->h != nullptr;
    const uint32_t cw = (d / 8 + RMDA_WAVE - 1) / RMDA_WAVE;
    // one launch, unless its threads would not fit 32 bits
    const uint32_t most = std::max(1u, (1u << 25) / cw);
    for (uint32_t r0 = 0; r0 < rows; r0 += most) {
        const uint32_t waves = cw * std::min(most, rows - r0);
        const bool few = waves <= 1024;
        const uint32_t wpb = few ? 1u : 4u;
        const auto kernel = !streams ? (topk <= 2 ? combine16_kernel<false, 2, false> : combine16_kernel<false, 8, false>)
                            : few    ? (topk <= 2 ? combine16_kernel<true, 2, true> : combine16_kernel<true, 8, true>)
                                     : (topk <= 2 ? combine16_kernel<true, 2, false> : combine16_kernel<true, 8, false>);
        rmda_hc_t h{};
        if (streams) {
            h = *hc;
            h.h += (size_t)r0 * h.hc * d;
            h.inj += (size_t)r0 * h.inj_stride;
        }
        hipLaunchKernelGGL(kernel, dim3((waves + wpb - 1) / wpb), dim3(wpb * RMDA_WAVE), 0, s, wt + (size_t)r0 * topk,
                           slot + (size_t)r0 * topk, y, proj + (size_t)r0 * pstride, pstride, sg_off,
                           shared_row0 + r0, has_shared, out != nullptr ? out + (size_t)r0 * d : nullptr, waves, d,
                           topk, h, run_if, yscale, ybound);
    }
    return hipGetLastError();
}
