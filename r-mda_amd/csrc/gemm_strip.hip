// Grouped expert GEMM of the fused layer for calls of few rows per expert or
// few experts (gfx950, packed weights).
//
// What bounds it.  Such a call is a weight stream: the streaming tile
// (gemm2.hip) hands out (item, 256 weight rows) tasks of a whole workgroup
// each, so one token of 8 selected experts is 48 gate_up and 64 down tasks on
// 256 CUs, each waiting on its own chain of five 16 KiB stages, and a call
// whose tasks do not fill the last round of workgroups leaves CUs idle.  Here
// a task is one wave: a chunk of up to 64 rows of a work item times 32 weight
// rows (a strip), 8 times as many tasks of which none waits for another.
//   * A packed slab keeps 16 weight rows x 32 k (one MFMA operand) in one
//     contiguous KiB, so a wave loads it straight into registers, 16 bytes
//     per lane: no LDS and no barriers.  The weights carry the non-temporal
//     hint.
//   * 5 to 16 K steps (by live row groups and variant) are in flight per wave
//     in a register ring, within 256 VGPRs so that two waves share a SIMD: 32 MB
//     in flight over the chip against about 3 us of loaded HBM latency.  One
//     wave per workgroup: with 4 or 8 a finished wave's registers wait for the
//     others (one 16-token block, hidden 2048, 128 experts top-8, width 768:
//     gate_up 74 us, 77 and 80 us).
//   * Activation rows are read in the MFMA layout from L2, only the live
//     16-row groups of the chunk: the loop is specialised on their number.
//   * The strips and chunks of one slab run on one XCD, so a chunk re-reads
//     its weights from L2 (32 tokens of the shape above: gate_up 126 -> 102
//     us against strips dealt round the XCDs).
// Measured against the streaming tile on MI355X (gate_up + down, us): the
// shape above at 1 token 33.0 + 12.8 -> 7.2 + 3.9, 16 tokens 103 + 45 -> 76
// + 39 (6.7 TB/s), 32 tokens 116 + 60 -> 102 + 52; 256 tokens of 8 experts
// top-2, hidden 512, width 1024: 13.2 + 19.4 -> 8.4 + 4.8.
// Per output element the MFMA sequence and the epilogue are those of the
// other tiles (K steps of 32 in order from a zero accumulator), so the output
// is bitwise the same.
#include <algorithm>

#include "common.h"
#include "gemm_sched.h"

namespace {

using namespace rmda_gemm;

constexpr uint32_t SLAB = RMDA_SLAB;
constexpr uint32_t BK = 32;        // K step of a slab block
constexpr uint32_t STEP = SLAB * BK;
constexpr uint32_t STRIPS = 8;     // strips of 32 weight rows in a slab
constexpr uint32_t CHUNK = 64;     // rows of a chunk

typedef float float8_t __attribute__((ext_vector_type(8)));

// One MFMA operand of A as it is loaded: fp16, or (CAST) fp32 to be scaled
// and rounded as hp_cast_kernel does it.
template <bool CAST>
struct a_frag_t {
    half8_t v;
    __device__ __forceinline__ void load(const rmda_gemm_args_t &g, uint32_t i) {
        v = *reinterpret_cast<const half8_t *>(g.a + i);
    }
    __device__ __forceinline__ half8_t get(float) const { return v; }
};
template <>
struct a_frag_t<true> {
    float8_t v;
    __device__ __forceinline__ void load(const rmda_gemm_args_t &g, uint32_t i) {
        v = *reinterpret_cast<const float8_t *>(g.a32 + i);
    }
    __device__ __forceinline__ half8_t get(float scale) const {
        half8_t h;
#pragma unroll
        for (int j = 0; j < 8; j += 1) {
            h[j] = (_Float16)(v[j] * scale);
        }
        return h;
    }
};

// One chunk of MT live 16-row groups times one strip.
template <int MODE, int MT, int DEPTH, bool SC, bool CAST, bool MANY>
__device__ __forceinline__ void strip_chunk(const rmda_gemm_args_t &g, uint32_t row0, uint32_t rows, bool is_shared,
                                            const uint16_t *wb, uint32_t col0, float scale) {
    uint32_t lane = threadIdx.x;
    uint32_t steps = g.k / BK;
    if constexpr (MANY) {
        // opaque, so that the loop over tasks keeps nothing derived from them
        // in registers next to the ring (which would spill)
        asm volatile("" : "+v"(lane), "+s"(steps));
    }
    const uint32_t fr = lane % 16;
    const uint32_t fq = lane / 16;
    const uint16_t *const b0 = wb + fr * BK + (fq ^ swz<BK>(fr)) * 8;
    const uint16_t *const b1 = b0 + (MODE == RMDA_GEMM_SWIGLU ? 32u : 16u) * BK;
    constexpr uint32_t A_STEP = MODE == RMDA_GEMM_F16 ? RMDA_HP_ROWS * BK : BK;
    uint32_t a[MT];  // element offsets from g.a (the launch checks that they fit)
#pragma unroll
    for (int m = 0; m < MT; m += 1) {
        if (MODE == RMDA_GEMM_SWIGLU) {
            const uint32_t r = (uint32_t)m * 16u + fr;
            const uint32_t rr = r < rows ? r : 0u;
            uint32_t t = is_shared ? row0 + rr - g.shared_row0 : g.rowtok[row0 + rr];
            t = t < g.a_rows ? t : 0u;  // a bad index reads a valid row, never out of bounds
            a[m] = t * g.lda + fq * 8;
        } else {
            a[m] = (uint32_t)rmda_hp_index(row0 + (uint32_t)m * 16u, 0, g.lda) + fr * 32 + fq * 8;
        }
    }
    a_frag_t<CAST> ra[DEPTH][MT];
    half8_t rb[DEPTH][2];
    floatx4_t acc[MT][2];
#pragma unroll
    for (int m = 0; m < MT; m += 1) {
        acc[m][0] = floatx4_t{0.f, 0.f, 0.f, 0.f};
        acc[m][1] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    }
    auto load = [&](uint32_t s, int u) __attribute__((always_inline)) {
        rb[u][0] = __builtin_nontemporal_load(reinterpret_cast<const half8_t *>(b0 + (size_t)s * STEP));
        rb[u][1] = __builtin_nontemporal_load(reinterpret_cast<const half8_t *>(b1 + (size_t)s * STEP));
#pragma unroll
        for (int m = 0; m < MT; m += 1) {
            ra[u][m].load(g, s * A_STEP + a[m]);
        }
    };
    auto mma = [&](int u) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < MT; m += 1) {
            const half8_t av = ra[u][m].get(scale);
            acc[m][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, rb[u][0], acc[m][0], 0, 0, 0);
            acc[m][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, rb[u][1], acc[m][1], 0, 0, 0);
        }
    };
#pragma unroll
    for (int u = 0; u < DEPTH; u += 1) {
        load(min((uint32_t)u, steps - 1u), u);  // past the end: a valid step, never multiplied
    }
    uint32_t s = 0;
    // whole rounds whose loads all stay below `steps`
    for (; s + 2 * DEPTH <= steps; s += DEPTH) {
#pragma unroll
        for (int u = 0; u < DEPTH; u += 1) {
            mma(u);
            load(s + DEPTH + u, u);
            __builtin_amdgcn_sched_barrier(0);  // as written: a slot's loads leave right after its MFMAs
        }
    }
    // the last DEPTH steps, and up to DEPTH - 1 more that still need loading
    for (; s < steps; s += DEPTH) {
#pragma unroll
        for (int u = 0; u < DEPTH; u += 1) {
            if (s + u < steps) {
                mma(u);
                if (s + DEPTH + u < steps) {
                    load(s + DEPTH + u, u);
                }
            }
        }
    }
    // the slot-scaled mode's inverse scales (1 otherwise, which changes no bits)
    const float xinv = SC && MODE == RMDA_GEMM_SWIGLU ? rmda_slot_inv(g.xscale) : 1.0f;
    const float yinv = down_mul<SC, MODE>(g);
    uint16_t *const O = reinterpret_cast<uint16_t *>(g.out);
    float hmax = 0.0f;
#pragma unroll
    for (int m = 0; m < MT; m += 1) {
#pragma unroll
        for (int v = 0; v < 4; v += 1) {
            const uint32_t rr = (uint32_t)m * 16u + 4 * fq + v;
            if (rr < rows) {
                if (MODE == RMDA_GEMM_SWIGLU) {
                    const float h = rmda_swiglu_fast(acc[m][0][v] * xinv, acc[m][1][v] * xinv);
                    swiglu_store<SC, false>(g, O, rmda_hp_index(row0 + rr, col0 + fr, g.ldo), h, hmax);
                } else {
                    const size_t o = (size_t)(row0 + rr) * g.ldo + col0 + fr;
                    down_store<SC>(g, O, o, acc[m][0][v] * yinv);
                    down_store<SC>(g, O, o + 16, acc[m][1][v] * yinv);
                }
            }
        }
    }
    if (SC && MODE == RMDA_GEMM_SWIGLU) {
        const uint32_t r = rmda_wave_red_u32<true>(__builtin_bit_cast(uint32_t, hmax));
        if (lane == 0) {
            atomicMax(g.hp_amax + blockIdx.x % RMDA_AMAX_PARTS * RMDA_AMAX_STRIDE, r);
        }
    }
}

// DEEP: 16 steps in flight for one live row group, 12 for two, 8 and 7 for
// three and four, instead of 8, 8, 6 and 6.  It keeps HBM busy on long K
// loops (16 tokens of the shape above: layer 149 -> 145.5 us; 512 experts
// top-10, hidden 2560, width 640 at 512 tokens: 938 -> 915 us); a launch that
// the shallow ring covers at once only pays for its longer start (one token:
// 36.1 -> 37.3 us), and a K loop shorter than the ring reads its last step
// again (K = 256: down 15.7 -> 21.0 us).
template <int MODE, bool DEEP, bool SC, bool CAST, bool MANY>
__device__ __forceinline__ void strip_rows(const rmda_gemm_args_t &g, uint32_t row0, uint32_t rows, bool is_shared,
                                           const uint16_t *wb, uint32_t col0, float scale) {
    switch ((rows + 15u) / 16u) {
    case 1: strip_chunk<MODE, 1, DEEP ? 16 : 8, SC, CAST, MANY>(g, row0, rows, is_shared, wb, col0, scale); break;
    case 2: strip_chunk<MODE, 2, DEEP ? 12 : 8, SC, CAST, MANY>(g, row0, rows, is_shared, wb, col0, scale); break;
    case 3: strip_chunk<MODE, 3, DEEP ? 8 : 6, SC, CAST, MANY>(g, row0, rows, is_shared, wb, col0, scale); break;
    default: strip_chunk<MODE, 4, DEEP ? 7 : CAST ? 5 : 6, SC, CAST, MANY>(g, row0, rows, is_shared, wb, col0, scale); break;
    }
}

// MANY: a launch of several chunks per item whose bound on the tasks is above
// MANY_WAVES runs that many waves, each walking its share of the tasks that
// the work list holds.  The bound counts an item per expert and every chunk an
// item can have; under skewed routing, where few experts hold all rows, nine
// tasks in ten were empty, lay between the others and cost the dispatcher
// about 0.2 ns each (512 experts top-10, hidden 2560, width 640, 199 tokens
// with a Zipf-like bias: layer 176 -> 159 us; top-1, width 512, hidden 2048,
// 512 tokens 72 -> 57 us).  The chunks of an item are then one wave's, one
// after the other, unless the list has fewer than SPLIT_WAVES strips.  With one
// chunk per item the empty tasks are the last ones and cost nothing (51 tokens
// of the first shape 90 us either way, evenly routed 506 -> 515 us walking).
constexpr uint32_t MANY_WAVES = 16384;
constexpr uint32_t SPLIT_WAVES = 8192;

template <int MODE, bool DEEP, bool SC, bool CAST, bool MANY>
__global__ __launch_bounds__(RMDA_WAVE) __attribute__((amdgpu_waves_per_eu(2, 2))) void strip_kernel(
    rmda_gemm_args_t g, uint32_t chunks) {
    const const_u32p items = (const_u32p)g.items;
    float scale = 1.0f;
    if constexpr (CAST) {
        static_assert(RMDA_AMAX_PARTS == RMDA_WAVE, "one partial word per lane");
        const uint32_t m = rmda_wave_red_u32<true>(g.a_parts[threadIdx.x * RMDA_AMAX_STRIDE]);
        scale = rmda_amax_scale(m);
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            *g.a_slot = m;  // for the combine
        }
    }
    // task = (slab / 8, chunk, strip, slab % 8), slabs counted over the whole
    // work list: the strips and row chunks of a slab share an XCD's L2
    const uint32_t nslab = g.n_w / SLAB;
    uint32_t per = chunks;
    if constexpr (MANY) {
        per = *(const_u32p)g.n_items * nslab * STRIPS >= SPLIT_WAVES ? 1u : chunks;
    }
    for (uint32_t b = blockIdx.x;; b += gridDim.x) {
        const uint32_t j = b / 8u;
        const uint32_t jj = j / STRIPS;
        const uint32_t gs = jj / per * 8u + blockIdx.x % 8u;
        const uint32_t item = gs / nslab;
        const uint32_t slab = gs - item * nslab;
        const uint32_t strip = j % STRIPS;
        if (item >= *(const_u32p)g.n_items) {
            return;
        }
        const uint32_t grp = items[item * 4 + 0];
        const uint32_t item0 = items[item * 4 + 1];
        const uint32_t n = items[item * 4 + 2];
        const bool is_shared = grp == g.shared_group;
        const uint16_t *const wg = is_shared ? g.w_shared : g.w + (size_t)grp * g.n_w * g.k;
        // weight rows of the strip: two 16-row operands.  SWIGLU: 16 gate rows
        // and the matching up rows, 32 slab rows further; F16: 32 adjacent rows
        const uint32_t nb = MODE == RMDA_GEMM_SWIGLU ? strip / 2u * 64u + strip % 2u * 16u : strip * 32u;
        const uint32_t col0 = MODE == RMDA_GEMM_SWIGLU ? slab * (SLAB / 2) + strip * 16u : slab * SLAB + strip * 32u;
        const uint16_t *const wb = wg + (size_t)slab * (g.k / BK) * STEP + nb * BK;
        for (uint32_t r0 = jj % per * CHUNK; r0 < n; r0 += per * CHUNK) {
            strip_rows<MODE, DEEP, SC, CAST, MANY>(g, item0 + r0, min(n - r0, CHUNK), is_shared, wb, col0, scale);
            if constexpr (!MANY) {
                return;  // an item has at most `chunks` chunks
            }
        }
        if constexpr (!MANY) {
            return;
        }
    }
}

uint32_t strip_tasks(uint32_t items, uint32_t item_rows, uint32_t n_w) {
    return (items * (n_w / SLAB) + 7) / 8 * 8 * STRIPS * ((item_rows + CHUNK - 1) / CHUNK);
}

template <int MODE, bool DEEP, bool SC>
hipError_t launch_strip(hipStream_t s, const rmda_gemm_args_t *a, uint32_t items, uint32_t item_rows) {
    const uint32_t chunks = (item_rows + CHUNK - 1) / CHUNK;
    const uint32_t tasks = strip_tasks(items, item_rows, a->n_w);
    const uint32_t waves = rmda_gemm_strip_waves(items, item_rows, a->n_w);
    if constexpr (MODE == RMDA_GEMM_F16 && !DEEP && SC) {
        if (a->a32 != nullptr) {
            hipLaunchKernelGGL((strip_kernel<MODE, false, true, true, false>), dim3(tasks), dim3(RMDA_WAVE), 0, s, *a,
                               chunks);
            return hipGetLastError();
        }
    }
    if (tasks > waves) {
        hipLaunchKernelGGL((strip_kernel<MODE, DEEP, SC, false, true>), dim3(waves), dim3(RMDA_WAVE), 0, s, *a, chunks);
    } else {
        hipLaunchKernelGGL((strip_kernel<MODE, DEEP, SC, false, false>), dim3(tasks), dim3(RMDA_WAVE), 0, s, *a, chunks);
    }
    return hipGetLastError();
}

template <int MODE, bool DEEP>
hipError_t launch_strip(hipStream_t s, const rmda_gemm_args_t *a, uint32_t items, uint32_t item_rows) {
    return a->hp32 != nullptr || a->ye_bound != nullptr ? launch_strip<MODE, DEEP, true>(s, a, items, item_rows)
                                                        : launch_strip<MODE, DEEP, false>(s, a, items, item_rows);
}

// Whether strips hold up in both GEMMs where the rows may gather on few experts.
bool strip_spread(uint32_t rows, uint32_t topk, uint32_t inter, uint32_t d) {
    // The shape does not say how many rows the chosen experts get.  The bound
    // takes the worst load, all tokens on the same experts: the gate_up
    // weights that rows * topk / 64 full chunks and topk started ones read.
    // Layer in strips against the streaming tile under a Zipf-like bias and
    // under even routing, by these bytes.  Above 64 rows, where an expert's
    // chunks read its weights again: 71 MB (300 experts top-3, hidden 1280,
    // width 640, 400 tokens) 0.89 and 0.99; 101 MB (256 top-8, 2048, 768, 65)
    // 1.21 and 0.97; 104 MB (400 top-8, 2048, 384, 200) 0.97 and 1.00; 106 MB
    // (160 top-5, 2560, 1024, 65) 1.12 and 0.93; 126 MB (96 tokens of the
    // second) 1.18 and 1.04; 170 MB (512 top-10, 2560, 640, 102) 1.17 and 1.03.
    // Up to 64 rows, one chunk each: 118 MB (51 tokens of the last) 0.91 and
    // 0.97; 201 MB (256 top-16, 2048, 768, 64) 1.16 and 1.00; 210 MB (160
    // top-10, 2560, 1024, 64) 1.10 and 0.98.
    return 4ull * inter * d * topk * (rows + CHUNK) / CHUNK < (rows <= CHUNK ? 192ull << 20 : 96ull << 20);
}

// Whether strips beat the streaming tile in a GEMM of n_w weight rows of k for
// npairs rows over `groups` experts (shared one included).
bool strip_pays(uint32_t npairs, uint32_t groups, uint32_t items, uint32_t n_w, uint32_t k, bool spread) {
    const uint64_t tasks = (uint64_t)items * (n_w / SLAB);  // the streaming tile's
    // Experts average few rows: every strip is read once and the weights
    // decide.  Up to 4 rows where the streaming tile's tasks fill two rounds
    // of the 256 workgroups (128 experts of width 768: 4 rows, layer 210 ->
    // 204 us; 8 rows, 215 -> 213 us but 85 -> 91 us under skewed routing; 16
    // rows, 225 -> 244 us), and the more the emptier its rounds are (128
    // tasks: 16 rows, 82 -> 69 us; 32 rows, 94 -> 118 us).
    if (spread && (uint64_t)npairs * (tasks < 512 ? tasks : 512) <= 4ull * 512 * groups) {
        return true;
    }
    // Few weights for the streaming tile's workgroups: one round or less of
    // tasks, and with the 64-row chunks counted at most 64 MB moved from L2 (8
    // experts, hidden 512, width 1024: 64 rows per expert 51 -> 34 us, 128
    // rows 60 -> 42 us, 256 rows' gate_up, 75 MB, 18.9 -> 27.9 us), less where
    // the tasks nearly fill the round.  gate_up alone in strips, layer against
    // the streaming tile by tasks x MB: 45 x 62 0.78, 72 x 66 0.92, 116 x 50
    // 0.98, 128 x 59 1.02, 114 x 66 1.09, 148 x 50 1.06 (0.82 under a Zipf-like
    // bias), 138 x 67 1.09, 160 x 63 1.12 (0.89).
    const uint64_t moved = 2ull * groups * n_w * k * ((uint64_t)npairs + 32ull * groups) / (64ull * groups);
    return tasks <= 256 && moved <= (64ull << 20) && tasks * moved <= (8192ull << 20);
}

}  // namespace

uint32_t rmda_gemm_strip_waves(uint32_t items, uint32_t item_rows, uint32_t n_w) {
    const uint32_t tasks = strip_tasks(items, item_rows, n_w);
    return item_rows <= CHUNK ? tasks : std::min(tasks, MANY_WAVES);
}

uint32_t rmda_gemm_strip_items(uint32_t npairs, uint32_t experts, uint32_t sh_rows) {
    return std::min(npairs, experts) + npairs / RMDA_GEMM2_BM + (sh_rows + RMDA_GEMM2_BM - 1) / RMDA_GEMM2_BM;
}

uint32_t rmda_gemm_strip_choice(uint32_t rows, uint32_t topk, uint32_t experts, uint32_t sh_rows, uint32_t inter,
                                uint32_t d) {
    const uint32_t npairs = rows * topk;
    const uint32_t items = rmda_gemm_strip_items(npairs, experts, sh_rows);
    const uint32_t groups = experts + (sh_rows > 0 ? 1u : 0u);
    const bool spread = strip_spread(rows, topk, inter, d);
    const bool gu = strip_pays(npairs + sh_rows, groups, items, 2 * inter, d, spread);
    const bool dn = strip_pays(npairs + sh_rows, groups, items, d, inter, spread);
    // One GEMM in strips keeps the other off the compute tile, which large
    // experts want: from 192 rows on average, only where the strips replace at
    // most a quarter round of tasks.  down alone in strips, layer against the
    // tiles by its tasks: 36 (8 experts, hidden 512, width 1024, 256 rows each)
    // 0.78, 48 (384 rows) 0.88, 58 (512) 0.94; 76 (13 experts, 512 x 384, 384
    // rows) 0.95, 85 (8, 1280 x 512, 224) 0.94, 94 (13, 512 rows) 1.00, 106 (20,
    // 512 x 512, 320) 1.01, 112 (12, 1024 x 384, 256) 1.03, 120 (13, 700 rows)
    // 1.11, 144 (12, 384 rows) 1.13.
    if (gu != dn && npairs >= 192 * experts && (uint64_t)items * ((gu ? 2 * inter : d) / SLAB) > 64) {
        return 0;
    }
    return (gu ? 1u : 0u) | (dn ? 2u : 0u);
}

bool rmda_gemm_strip_casts(uint32_t items, uint32_t n_w) {
    // Casting in down spares a launch, but every strip converts the rows
    // again and reads twice the bytes: hp cast + down, 24 waves of hidden 768,
    // width 256 7.0 -> 4.2 us; 336 waves of hidden 512, width 384 10.9 -> 9.4;
    // 880 waves of hidden 2560, width 640 21.5 -> 21.9; 11000 waves 224 -> 239.
    return (uint64_t)items * (n_w / 32u) <= 512;
}

bool rmda_gemm_strip_deep(uint32_t items, uint32_t n_w, uint32_t k) {
    // more waves than the chip holds at once (two per SIMD), and a K loop that
    // fills the deep ring
    return (uint64_t)items * (n_w / 32u) > 2048 && k >= 16 * BK;
}

hipError_t rmda_launch_gemm_strip(hipStream_t s, const rmda_gemm_args_t *a, uint32_t items, uint32_t item_rows) {
    if (a->n_w % SLAB != 0 || a->k % BK != 0 || a->n_items == nullptr || a->fc.cnt != nullptr || a->ye32 != nullptr ||
        (a->a32 != nullptr && (a->mode != RMDA_GEMM_F16 || a->ye_bound == nullptr))) {
        return hipErrorInvalidValue;
    }
    if (items == 0 || item_rows == 0) {
        return hipSuccess;
    }
    const bool deep = a->a32 == nullptr && rmda_gemm_strip_deep(items, a->n_w, a->k);
    if (a->mode == RMDA_GEMM_SWIGLU) {
        return deep ? launch_strip<RMDA_GEMM_SWIGLU, true>(s, a, items, item_rows)
                    : launch_strip<RMDA_GEMM_SWIGLU, false>(s, a, items, item_rows);
    }
    return deep ? launch_strip<RMDA_GEMM_F16, true>(s, a, items, item_rows)
                : launch_strip<RMDA_GEMM_F16, false>(s, a, items, item_rows);
}
