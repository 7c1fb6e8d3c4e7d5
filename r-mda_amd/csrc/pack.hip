// Weight packing of the fused layer: HF-layout expert matrices (fp16, or bf16
// converted on the way) into the slab order the grouped GEMMs stream, the
// router rows into the router kernel's order, and the down weights' row-sum
// bound, in two launches.
//
// What bounds it: HBM, every weight read and written once.  Measured on
// MI355X, 512 experts of hidden 2560 and width 640 with a shared one, from
// bf16 (10.1 GB moved): 2.62 -> 1.63 ms, 6.2 TB/s (a device copy reaches
// 5.2); 12 experts of hidden 1280, width 384, also with a shared one: 43 ->
// 23 us.
//   * Whole 128-byte lines on both sides: a tile's row is 256 (down: 128)
//     columns, and 16 rows x 32 columns of a slab block are one contiguous
//     KiB.  With one K step of 32 per thread block, as before, each line of
//     the source was read by two blocks on different XCDs.
//   * Small tiles in address order, loads and stores non-temporal: gate_up in
//     tiles of 16 rows x 256 columns runs at 6.5 TB/s; 32 x 256 cost 5% more
//     over both launches, 256 x 128 8%, 256 x 64 16%; ordinary loads 3%,
//     ordinary stores 5%.  The price: the last 256 MB packed are no longer in
//     the Infinity Cache when the first layer runs, which then takes 12 us
//     (128 experts, 2048 x 768, 777 tokens) or 19 us (512 experts, 2048 x 512,
//     4096 tokens) longer, once; packing these is 0.2 to 1.0 ms shorter.
//   * The bound is summed from the tile in LDS while the next one loads, in
//     place of a second pass over the packed down weights (0.37 ms).
#include "common.h"
#include "gemm_sched.h"

namespace {

using namespace rmda_gemm;

constexpr uint32_t BK = 32;      // K step of a slab block
constexpr uint32_t CH = BK / 8;  // 16-byte units of a row in a block

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// ROWS x TK of a slab, moved by PT threads: thread t moves unit t % TU of
// rows t / TU, t / TU + PT / TU, ...
template <int MODE, uint32_t ROWS, uint32_t TK, uint32_t PT>
struct tile_t {
    static constexpr uint32_t TU = TK / 8;           // 16-byte units of a tile row
    static constexpr uint32_t UPT = ROWS * TU / PT;  // units per thread
    static_assert(UPT * PT == ROWS * TU && PT % TU == 0, "whole rows per pass");
    const uint16_t *src;  // the expert's matrix [n_w][k]
    uint32_t k, slab, inter, r0;
    u32x4_t v[UPT];

    __device__ __forceinline__ void load(uint32_t k0) {
#pragma unroll
        for (uint32_t i = 0; i < UPT; i += 1) {
            const uint32_t n = r0 + threadIdx.x / TU + i * (PT / TU);
            const uint16_t *p = src + (size_t)slab_row<MODE>(slab, n, inter) * k + k0 + threadIdx.x % TU * 8;
            v[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t *>(p));
        }
    }
    __device__ __forceinline__ void convert() {
#pragma unroll
        for (uint32_t i = 0; i < UPT; i += 1) {
#pragma unroll
            for (int q = 0; q < 4; q += 1) {
                const float lo = __builtin_bit_cast(float, v[i][q] << 16);
                const float hi = __builtin_bit_cast(float, v[i][q] & 0xffff0000u);
                v[i][q] = (uint32_t)rmda_f2h(lo) | ((uint32_t)rmda_f2h(hi) << 16);
            }
        }
    }
    // dst: the slab's first block; LROW > 0: a copy of the tile goes to lds,
    // tile row n's units in packed order from n * LROW
    template <uint32_t LROW>
    __device__ __forceinline__ void store(u32x4_t *dst, uint32_t k0, u32x4_t *lds) {
        const uint32_t c = threadIdx.x % TU;
#pragma unroll
        for (uint32_t i = 0; i < UPT; i += 1) {
            const uint32_t n = threadIdx.x / TU + i * (PT / TU);
            const uint32_t p = c % CH ^ swz<BK>(r0 + n);
            __builtin_nontemporal_store(v[i], dst + ((size_t)(k0 / BK + c / CH) * RMDA_SLAB + r0 + n) * CH + p);
            if constexpr (LROW > 0) {
                lds[n * LROW + c / CH * CH + p] = v[i];
            }
        }
    }
};

constexpr uint32_t GU_PT = 256, GU_ROWS = 16, GU_TK = 256;

// gate_up (routed, then shared), one tile per block, after the blocks that
// pack the router rows; block 0 also clears the bound word.
__global__ __launch_bounds__(GU_PT) void pack_gate_up_kernel(rmda_pack_args_t a, uint32_t router_blocks) {
    uint32_t b = blockIdx.x;
    if (b < router_blocks) {
        if (b == 0 && threadIdx.x < 64) {
            a.bound[threadIdx.x] = 0;
        }
        rmda_router_pack_share(a.w_router, a.router, a.router_cols, a.d, b, router_blocks);
        return;
    }
    b -= router_blocks;
    constexpr uint32_t RB = RMDA_SLAB / GU_ROWS;
    const uint32_t slabs = 2 * a.inter / RMDA_SLAB;        // per expert
    const uint32_t tiles = RB * (a.d / GU_TK);             // per slab
    const bool shared = b >= a.experts * slabs * tiles;
    const rmda_pack_mat_t &m = shared ? a.sh_gate_up : a.gate_up;
    b -= shared ? a.experts * slabs * tiles : 0u;
    const uint32_t ts = b / tiles;  // slab, counted over the experts
    const uint32_t e = ts / slabs;
    const uint32_t k0 = (b - ts * tiles) / RB * GU_TK;
    tile_t<RMDA_GEMM_SWIGLU, GU_ROWS, GU_TK, GU_PT> t{
        m.src + (size_t)e * 2 * a.inter * a.d, a.d, ts - e * slabs, a.inter, b % RB * GU_ROWS, {}};
    t.load(k0);
    if (m.bf16) {
        t.convert();
    }
    t.template store<0>(reinterpret_cast<u32x4_t *>(m.dst) + (size_t)ts * RMDA_SLAB * a.d / 8, k0, nullptr);
}

constexpr uint32_t DN_ROWS = 128, DN_TK = 128;  // one thread per row

// down (routed, then shared): 128 rows of a slab per block over all of K,
// with the largest row sum of |w| (see rmda_launch_pack).
__global__ __launch_bounds__(DN_ROWS) void pack_down_kernel(rmda_pack_args_t a) {
    constexpr uint32_t TU = DN_TK / 8;
    constexpr uint32_t LROW = TU + 1;  // one unit of padding: 8 rows' reads sit in distinct banks
    __shared__ u32x4_t lds[DN_ROWS * LROW];
    __shared__ uint32_t s_max[DN_ROWS / RMDA_WAVE];
    constexpr uint32_t RB = RMDA_SLAB / DN_ROWS;
    uint32_t b = blockIdx.x;
    const uint32_t slabs = a.d / RMDA_SLAB;
    const bool shared = b >= a.experts * slabs * RB;
    const rmda_pack_mat_t &m = shared ? a.sh_down : a.down;
    b -= shared ? a.experts * slabs * RB : 0u;
    const uint32_t ts = b / RB;  // slab, counted over the experts
    const uint32_t e = ts / slabs;
    tile_t<RMDA_GEMM_F16, DN_ROWS, DN_TK, DN_ROWS> t{
        m.src + (size_t)e * a.d * a.inter, a.inter, ts - e * slabs, 0, b % RB * DN_ROWS, {}};
    u32x4_t *const dst = reinterpret_cast<u32x4_t *>(m.dst) + (size_t)ts * RMDA_SLAB * a.inter / 8;
    float sum = 0.0f;  // of tile row threadIdx.x, in packed order
    t.load(0);
    for (uint32_t k0 = 0; k0 < a.inter; k0 += DN_TK) {
        if (m.bf16) {
            t.convert();
        }
        if (k0 > 0) {
            __syncthreads();  // the last tile's rows are summed
        }
        t.template store<LROW>(dst, k0, lds);
        if (k0 + DN_TK < a.inter) {
            t.load(k0 + DN_TK);
        }
        __syncthreads();
#pragma unroll
        for (uint32_t u = 0; u < TU; u += 1) {
            const u32x4_t v = lds[threadIdx.x * LROW + u];
#pragma unroll
            for (int i = 0; i < 4; i += 1) {
                sum += fabsf(rmda_h2f((uint16_t)(v[i] & 0xffffu))) + fabsf(rmda_h2f((uint16_t)(v[i] >> 16)));
            }
        }
    }
    const float mx = sum <= 3.4028235e38f ? sum : 0.0f;  // inf and NaN left out
    const uint32_t r = rmda_wave_red_u32<true>(__builtin_bit_cast(uint32_t, mx));
    if (threadIdx.x % RMDA_WAVE == 0) {
        s_max[threadIdx.x / RMDA_WAVE] = r;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t q = s_max[0];
        for (uint32_t w = 1; w < DN_ROWS / RMDA_WAVE; w += 1) {
            q = max(q, s_max[w]);
        }
        // the word only grows: a block whose maximum it already holds leaves it alone
        if (q > rmda_load_agent(a.bound)) {
            atomicMax(a.bound, q);
        }
    }
}

}  // namespace

hipError_t rmda_launch_pack(hipStream_t s, const rmda_pack_args_t *a) {
    if (a->d % GU_TK != 0 || a->inter % DN_TK != 0) {
        return hipErrorInvalidValue;
    }
    const uint64_t n = (uint64_t)a->d * rmda_router_cpad(a->router_cols);
    const uint32_t router_blocks = (uint32_t)(n / GU_PT < 2048 ? (n + GU_PT - 1) / GU_PT : 2048);
    const uint32_t groups = a->experts + (a->sh_gate_up.src != nullptr ? 1u : 0u);
    const uint64_t gu =
        (uint64_t)groups * (2 * a->inter / RMDA_SLAB) * (RMDA_SLAB / GU_ROWS) * (a->d / GU_TK) + router_blocks;
    const uint64_t dn = (uint64_t)groups * (a->d / DN_ROWS);
    if (gu > 0xffffffffu / GU_PT || dn > 0xffffffffu / DN_ROWS) {  // threads of a launch fit 32 bits
        return hipErrorInvalidValue;
    }
    hipLaunchKernelGGL(pack_gate_up_kernel, dim3((uint32_t)gu), dim3(GU_PT), 0, s, *a, router_blocks);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        return e;
    }
    hipLaunchKernelGGL(pack_down_kernel, dim3((uint32_t)dn), dim3(DN_ROWS), 0, s, *a);
    return hipGetLastError();
}
