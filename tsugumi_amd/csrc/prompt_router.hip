// prompt_router.hip — the BF16 router of a prompt chunk (more than
// kMaxRouterRows rows): logits of every (row, expert), top-8, softmax.
//
// Reference semantics: prefill.metal:555-794, PrefillRouter.swift:127-236.
//
// A row's logit is the decode router's, bit for bit (decode.hip
// router_chunks_dot): 64 partial sums, partial l over the 8-element chunks l,
// l + 64, ... element by element in order with acc = fma(w, x * es, acc), added
// as a binary tree. v_mfma_f32_16x16x4_f32 accumulates its four products with
// four fmas in the order of k, rounding after each (checked on the device over
// 51,200 sums), so partial l of 16 experts x 16 rows is a chain of two MFMAs a
// chunk and the tree is added from the accumulators.
//
// What bounds it: the fp32 matrix rate. 2 T E d flops at 157 TFLOP/s are 9.4 us
// for T = 2048, E = 128, d = 2816 and 27 us for T = 4096, E = 256, d = 2048.
// Both launches, back to back in a HIP graph over router weights in turn, take
// 25.1-25.7 and 63.0 us there, 13.0 for T = 67 and 14.0 for T = 509; of it the
// selection 4.5, 5.1 and 3.9 us (kernel trace: 22.1 + 4.5, 62.7 + 5.1, 10.3 +
// 3.9; in a prompt's layer, with other kernels between, 27.6 + 5.7 for T =
// 2048). One wave an expert on vector fmas, each converting every row's
// activations again, took 192 and 612 us, 29 for T = 64 and 44 for T = 300
// (13.2 and 13.6 here).
#include "router_select.hpp"
#include <type_traits>

namespace tsg {
namespace {

typedef float f4_t __attribute__((ext_vector_type(4)));

constexpr uint32_t kPromptWaves = 8;
constexpr uint32_t kPromptThreads = 64u * kPromptWaves;
constexpr uint32_t kHalf = 32;  // chunks of a row that a step holds

// LDS of a workgroup of ROWS = 16 (EA + RB) staged rows: two stages of a step's
// chunks (reused by the exchange of the waves' sums), then the effective scale.
template <int EA, int RB>
struct PromptLds {
    static constexpr uint32_t kRows = 16u * (EA + RB);
    static constexpr uint32_t kStage = kRows * kHalf * 16u;
    static constexpr uint32_t kEs = 2u * kStage;
    static constexpr uint32_t kExchange = 2u * kPromptWaves * EA * RB * 1024u;
    static_assert(kExchange <= kEs, "the exchange fits the stages");
    // the effective scale up to whole pairs of steps
    static constexpr uint32_t bytes(uint32_t d) { return kEs + (d + 511u) / 512u * 1024u; }
};

// The largest of the 16 lanes' (key, expert) pairs, ties to the lower expert;
// every lane of the 16 gets it.
template <int CTRL>
__device__ __forceinline__ void take_larger(uint32_t& key, uint32_t& inv) {
    const uint32_t k = dpp_u32<CTRL>(key), i = dpp_u32<CTRL>(inv);
    const bool other = k > key || (k == key && i > inv);
    key = other ? k : key;
    inv = other ? i : inv;
}

// Top-8 and softmax of one row on 16 lanes (four rows a wave): the selection
// rule of decode.hip's wave_topk_softmax_regs (descending, ties to the lower
// expert, -inf and NaN never enter, unfilled slots keep expert 0 and -inf) and
// the arithmetic of its slot_softmax_lane. Lane r < 8 of the 16 returns slot
// r. Lane l holds experts l + 16 j; 16 lanes a row keep every step inside the
// DPP row, where a whole wave a row would take four times the rounds.
template <int NJ>
__device__ __forceinline__ void row16_top8(const float* __restrict__ logits, uint32_t ne,
                                           const uint16_t* __restrict__ gains, uint32_t& id,
                                           uint16_t& weight) {
    const uint32_t l16 = threadIdx.x & 15u;
    uint32_t key[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const uint32_t e = l16 + 16u * j;
        const float s = e < ne ? logits[e] : -INFINITY;
        key[j] = (s == s && s != -INFINITY) ? order_key(s) : 0u;
    }
    uint32_t my_key = 0u, my_id = 0u;
#pragma unroll 1  // the code is run once a launch: its fetch counts
    for (uint32_t r = 0; r < kTopK; ++r) {
        uint32_t best = key[0], j_best = 0u;
#pragma unroll
        for (int j = 1; j < NJ; ++j) {
            const bool larger = key[j] > best;  // a tie keeps the lower expert
            best = larger ? key[j] : best;
            j_best = larger ? (uint32_t)j : j_best;
        }
        uint32_t inv = ~(l16 + 16u * j_best);
        take_larger<0xB1>(best, inv);   // quad_perm [1,0,3,2]
        take_larger<0x4E>(best, inv);   // quad_perm [2,3,0,1]
        take_larger<0x141>(best, inv);  // row_half_mirror
        take_larger<0x140>(best, inv);  // row_mirror
        const uint32_t e = best ? ~inv : 0u;
        if (l16 == r) {
            my_key = best;
            my_id = e;
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            if (l16 + 16u * j == e) key[j] = 0u;
    }
    const float my_s = my_key ? order_key_value(my_key) : -INFINITY;
    const float my_exp = expf(my_s - __shfl(my_s, 0, 16));
    float sum_exp = __shfl(my_exp, 0, 16);
#pragma unroll
    for (int r = 1; r < (int)kTopK; ++r) sum_exp += __shfl(my_exp, r, 16);
    id = my_id;
    weight = f32_to_f16(my_exp / sum_exp * bf16_to_f32(gains[my_id]));
}

// One chunk of a wave's partial sum as MFMA operands: lane (n, g) holds element
// g (half 0) and g + 4 (half 1) of row n. The bf16 values are read into the
// high halves of registers whose low halves stay zero, which makes them fp32
// without a VALU op; the fp16 ones are read as they are.
template <int EA, int RB>
struct ChunkOps {
    uint32_t e[2], w[2][EA];  // fp32 bit patterns
    uint32_t x[2][RB];        // fp16 in the low half
};

// The LDS reads of a chunk and the wait for them, in one block (no read is in
// flight outside it): `data` + XO the lane's address of its element 0 in row n
// of the first token rows, `scale` + EO of the same element of the effective
// scale; 16 rows are 8192 bytes apart.
template <uint32_t XO, uint32_t EO>
__device__ __forceinline__ void read_chunk(ChunkOps<1, 1>& o, uint32_t data, uint32_t scale) {
    asm volatile("ds_read_u16_d16_hi %0, %7 offset:%c9\n\t"
                 "ds_read_u16 %2, %6 offset:%c8\n\t"
                 "ds_read_u16_d16_hi %4, %6 offset:%c8+8192\n\t"
                 "ds_read_u16_d16_hi %1, %7 offset:%c9+8\n\t"
                 "ds_read_u16 %3, %6 offset:%c8+8\n\t"
                 "ds_read_u16_d16_hi %5, %6 offset:%c8+8200\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "+v"(o.e[0]), "+v"(o.e[1]), "=&v"(o.x[0][0]), "=&v"(o.x[1][0]),
                   "+v"(o.w[0][0]), "+v"(o.w[1][0])
                 : "v"(data), "v"(scale), "n"(XO), "n"(EO)
                 : "memory");
}
template <uint32_t XO, uint32_t EO>
__device__ __forceinline__ void read_chunk(ChunkOps<2, 2>& o, uint32_t data, uint32_t scale) {
    asm volatile("ds_read_u16_d16_hi %0, %11 offset:%c13\n\t"
                 "ds_read_u16 %2, %10 offset:%c12\n\t"
                 "ds_read_u16 %3, %10 offset:%c12+8192\n\t"
                 "ds_read_u16_d16_hi %6, %10 offset:%c12+16384\n\t"
                 "ds_read_u16_d16_hi %7, %10 offset:%c12+24576\n\t"
                 "ds_read_u16_d16_hi %1, %11 offset:%c13+8\n\t"
                 "ds_read_u16 %4, %10 offset:%c12+8\n\t"
                 "ds_read_u16 %5, %10 offset:%c12+8200\n\t"
                 "ds_read_u16_d16_hi %8, %10 offset:%c12+16392\n\t"
                 "ds_read_u16_d16_hi %9, %10 offset:%c12+24584\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "+v"(o.e[0]), "+v"(o.e[1]), "=&v"(o.x[0][0]), "=&v"(o.x[0][1]),
                   "=&v"(o.x[1][0]), "=&v"(o.x[1][1]), "+v"(o.w[0][0]), "+v"(o.w[0][1]),
                   "+v"(o.w[1][0]), "+v"(o.w[1][1])
                 : "v"(data), "v"(scale), "n"(XO), "n"(EO)
                 : "memory");
}

// fp32 product of the fp16 value in the low half of x and e: x * e is exact in
// fp32, so the fma with zero gives the product.
__device__ __forceinline__ float half_times(uint32_t x, uint32_t e) {
    return __builtin_fmaf((float)__builtin_bit_cast(_Float16, (uint16_t)x), __uint_as_float(e), 0.0f);
}

// grid (expert tiles of 16 EA, row tiles of 16 RB), 8 waves. Step k holds
// chunks 32 k .. 32 k + 31 of the tile's rows, staged in LDS while the step
// before runs (chunk c of row r in slot c ^ swz(r), so the reads of 16 rows
// meet no bank conflict). In steps of parity h wave q runs the partial sums
// 32 h + 4 q + (0..3) over the whole tile, so a quad of the tree is added in
// registers and the quads meet in LDS once, at the end.
// fp32 MFMAs and VALU instructions share their units here (each VALU
// instruction between two MFMAs adds its own issue time, the first one twice
// that), so the operands come out of LDS ready for use: only x * es is left to
// compute. prompt_top8_kernel selects from the logits.
template <int EA, int RB>
__global__ __launch_bounds__(kPromptThreads) void prompt_router_kernel(
    const uint16_t* __restrict__ w, const uint16_t* __restrict__ hidden,
    const uint16_t* __restrict__ es, uint32_t stride, uint32_t ne, uint32_t d, uint32_t rows,
    float* __restrict__ logits) {
    using L = PromptLds<EA, RB>;
    constexpr int kTiles = EA * RB;
    constexpr int kUnits = (int)(L::kRows * kHalf / kPromptThreads);  // 16-byte units a thread
    extern __shared__ __align__(128) uint8_t smem[];
    const uint32_t t = threadIdx.x, lane = t & 63u, n = lane & 15u, g = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t e0 = blockIdx.x * 16u * EA, r0 = blockIdx.y * 16u * RB;
    const uint32_t nchunks = d / 8u, nsteps = (nchunks + kHalf - 1u) / kHalf;

    // unit u of thread t: chunk t % 32 of staged row 16 u + t / 32; the rows
    // are the tile's token rows, then its expert rows (past the end: the last)
    const uint32_t piece = t & 31u;
    const uint16_t* src[kUnits];
    uint32_t dst[kUnits];
#pragma unroll
    for (int u = 0; u < kUnits; ++u) {
        const uint32_t r = (t >> 5) + 16u * u;
        src[u] = u < RB ? hidden + (uint64_t)min(r0 + r, rows - 1u) * stride
                        : w + (uint64_t)min(e0 + r - 16u * RB, ne - 1u) * d;
        dst[u] = (r * kHalf + (piece ^ (r & 7u) ^ ((r >> 3) & 1u))) * 16u;
    }
    // a step's units are requested two steps ahead, into the registers of its
    // parity: one step's sums (0.9 us) are over before they come back
    u32x4_t in[2][kUnits];
    auto load_step = [&](uint32_t h, uint32_t k) {
        const uint32_t at = min(kHalf * k + piece, nchunks - 1u) * 8u;
#pragma unroll
        for (int u = 0; u < kUnits; ++u) in[h][u] = *reinterpret_cast<const u32x4_t*>(src[u] + at);
        asm volatile("" ::: "memory");  // requested here, ahead of the step's sums
    };
    auto store_step = [&](uint32_t h) {
#pragma unroll
        for (int u = 0; u < kUnits; ++u)
            *reinterpret_cast<u32x4_t*>(smem + h * L::kStage + dst[u]) = in[h][u];
    };
    load_step(0u, 0u);
    load_step(1u, 1u);
    for (uint32_t c = t; c < (nsteps + 1u) / 2u * 64u; c += kPromptThreads)
        *reinterpret_cast<u32x4_t*>(smem + L::kEs + 16u * c) =
            *reinterpret_cast<const u32x4_t*>(es + 8u * min(c, nchunks - 1u));
    store_step(0u);
    lds_barrier();

    const uint32_t base = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t*)smem;
    uint32_t data[4];  // chunk 4 q + j of row n, stage 0
#pragma unroll
    for (uint32_t j = 0; j < 4u; ++j)
        data[j] = base + (n * kHalf + ((4u * wave + j) ^ (n & 7u) ^ (n >> 3))) * 16u + 2u * g;
    uint32_t scale = base + L::kEs + 64u * wave + 2u * g;
    ChunkOps<EA, RB> o;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        o.e[h] = 0u;
#pragma unroll
        for (int a = 0; a < EA; ++a) o.w[h][a] = 0u;
    }
    f4_t acc[2][4][kTiles];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int q = 0; q < kTiles; ++q) acc[h][j][q] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
    auto run_chunk = [&](auto h_c, auto j_c) {
        constexpr uint32_t h = decltype(h_c)::value, j = decltype(j_c)::value;
        read_chunk<h * L::kStage, h * 512u + j * 16u>(o, data[j], scale);
        float xe[2][RB];
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
            for (int b = 0; b < RB; ++b) xe[half][b] = half_times(o.x[half][b], o.e[half]);
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
            for (int a = 0; a < EA; ++a)
#pragma unroll
                for (int b = 0; b < RB; ++b)
                    acc[h][j][a * RB + b] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                        __uint_as_float(o.w[half][a]), xe[half][b], acc[h][j][a * RB + b], 0, 0, 0);
    };
    auto run_step = [&](auto h_c, uint32_t k) {
        constexpr uint32_t h = decltype(h_c)::value;
        if (k + 2u < nsteps) load_step(h, k + 2u);
        const uint32_t c = kHalf * k + 4u * wave;  // chunks past the row's end add nothing
        if (c + 3u < nchunks) {
            run_chunk(h_c, std::integral_constant<uint32_t, 0>{});
            run_chunk(h_c, std::integral_constant<uint32_t, 1>{});
            run_chunk(h_c, std::integral_constant<uint32_t, 2>{});
            run_chunk(h_c, std::integral_constant<uint32_t, 3>{});
        } else {
            if (c < nchunks) run_chunk(h_c, std::integral_constant<uint32_t, 0>{});
            if (c + 1u < nchunks) run_chunk(h_c, std::integral_constant<uint32_t, 1>{});
            if (c + 2u < nchunks) run_chunk(h_c, std::integral_constant<uint32_t, 2>{});
        }
        if (k + 1u < nsteps) store_step(h ^ 1u);
        lds_barrier();
    };
    for (uint32_t k = 0; k < nsteps; k += 2u) {
        run_step(std::integral_constant<uint32_t, 0>{}, k);
        if (k + 1u < nsteps) run_step(std::integral_constant<uint32_t, 1>{}, k + 1u);
        scale += 1024u;
    }

    // The tree: quads of partial sums in registers, the rest of it from LDS,
    // one tile a wave.
    f4_t* const ex = reinterpret_cast<f4_t*>(smem);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int q = 0; q < kTiles; ++q)
            ex[((h * kPromptWaves + wave) * kTiles + q) * 64u + lane] =
                (acc[h][0][q] + acc[h][1][q]) + (acc[h][2][q] + acc[h][3][q]);
    lds_barrier();
    if (wave < (uint32_t)kTiles) {
        f4_t r32[2];  // the 32 partial sums of a parity
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            f4_t v[kPromptWaves];
#pragma unroll
            for (uint32_t q = 0; q < kPromptWaves; ++q)
                v[q] = ex[((h * kPromptWaves + q) * kTiles + wave) * 64u + lane];
            r32[h] = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
        }
        const f4_t sum = r32[0] + r32[1];
        const uint32_t row = r0 + 16u * (wave % RB) + n, ex0 = e0 + 16u * (wave / RB) + 4u * g;
        if (row < rows) {
            float* out = logits + (uint64_t)row * kMaxExperts + ex0;
            if (ex0 + 3u < ne) *reinterpret_cast<f4_t*>(out) = sum;
            else
#pragma unroll
                for (uint32_t q = 0; q < 4u; ++q)
                    if (ex0 + q < ne) out[q] = sum[q];
        }
    }
}

// One row on 16 lanes, 16 rows a workgroup. A launch of its own: with the
// selection left to the last workgroup of each row tile, every workgroup waits
// for its stores and an atomic, and the tile's rows are ranked by one compute
// unit (T = 4096, E = 256: 81 us as one launch, 62 as two; T = 67, E = 128:
// 12.7 both ways).
__global__ __launch_bounds__(256) void prompt_top8_kernel(const float* __restrict__ logits,
                                                          const uint16_t* __restrict__ pes,
                                                          uint32_t* __restrict__ out_idx,
                                                          uint16_t* __restrict__ out_w,
                                                          uint32_t ne, uint32_t rows) {
    const uint32_t row = (blockIdx.x * 256u + threadIdx.x) >> 4, rr = min(row, rows - 1u);
    uint32_t id;
    uint16_t weight;
    if (ne <= 128u) row16_top8<8>(logits + (uint64_t)rr * kMaxExperts, ne, pes, id, weight);
    else row16_top8<16>(logits + (uint64_t)rr * kMaxExperts, ne, pes, id, weight);
    const uint32_t slot = threadIdx.x & 15u;
    if (row < rows && slot < kTopK) {
        out_idx[(uint64_t)row * kTopK + slot] = id;
        out_w[(uint64_t)row * kTopK + slot] = weight;
    }
}

template <int EA, int RB>
tsg_status launch(tsg_ctx* ctx, hipStream_t stream, const PromptRouterArgs& a) {
    const uint32_t lds = PromptLds<EA, RB>::bytes(a.d);
    auto kern = prompt_router_kernel<EA, RB>;
    if (lds > 64u * 1024u)
        TSG_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const dim3 grid((a.ne + 16u * EA - 1u) / (16u * EA), (a.rows + 16u * RB - 1u) / (16u * RB));
    hipLaunchKernelGGL(kern, grid, dim3(kPromptThreads), lds, stream, a.w, a.hidden, a.es, a.stride,
                       a.ne, a.d, a.rows, ctx->logits);
    return check_launch("prompt_router");
}

}  // namespace

tsg_status prompt_router_launch(tsg_ctx* ctx, hipStream_t stream, const PromptRouterArgs& a) {
    // 32 x 32 tiles halve the LDS reads of an MFMA and the rows a tile stages,
    // but take a compute unit each for 20-23 us however few they are. 16 x 16
    // against 32 x 32 tiles in us, E = 128, d = 2816: T = 1024 (128 of the
    // latter) 17.8 and 23.0, T = 1280 (160) 24.0 and 23.3, T = 2048 29.6 and
    // 24.4; E = 256, d = 2048: T = 512 (128) 14.7 and 19.8, T = 768 (192) 19.7
    // and 19.5, T = 1024 23.6 and 19.8.
    const uint64_t wide = (uint64_t)((a.ne + 31u) / 32u) * ((a.rows + 31u) / 32u);
    const bool fills = wide * 8u >= (uint64_t)ctx->num_cus * 5u;
    const tsg_status st = fills ? launch<2, 2>(ctx, stream, a) : launch<1, 1>(ctx, stream, a);
    if (st) return st;
    hipLaunchKernelGGL(prompt_top8_kernel, dim3((a.rows + 15u) / 16u), dim3(256), 0, stream, ctx->logits,
                       a.pes, a.out_idx, a.out_w, a.ne, a.rows);
    return check_launch("prompt_top8");
}

}  // namespace tsg
