// qmv.hip — dense int4 GEMV (DequantInt4GEMV.swift:6-364,
// dequant_int4.metal:135-358) and the bit-exact dequantisation check.
//
// One output row per 16 lanes, 16-byte weight chunks (one g32 group, half a
// g64 group) streamed with all loads in flight, nibbles -> fp16 by the 0x6400
// exponent trick, v_dot2_f32_f16 against x staged in LDS, fp32 scale fma.
// The rows form keeps T <= 8 accumulators per lane so a weight chunk is read
// once for all rows; each row's sum runs in exactly the one-row order.
//
// What bounds it: latency (a launch is 2-2.5 us, the rest the round trip of
// staging and weights and, for several rows, a lane's dot2 chains and LDS
// reads at one wave a SIMD). Back to back in a HIP graph over weights that no
// cache holds, us before and now, group 32 sym: 704 x 2816 3.90 -> 3.26, 2816 x
// 4096 6.12 -> 4.23, 4096 x 2816 3.95 -> 3.82; five rows of them 9.25 -> 5.98,
// 15.95 -> 7.75, 7.23 -> 6.42; group 64 affine 2816 x 4096 6.35 -> 4.86, five
// rows 17.5 -> 9.1, eight 68 -> 12.4.
#include "gemv_lane.hpp"

namespace tsg {
namespace {

constexpr uint32_t kMaxRows = 8;

// compute_batch for T token rows, the rows' dot2 chains side by side (one
// after the other, a wave waits for each dot2 of a 16-long chain: eight rows of
// 8192 x 2816 12.1 us against 10.9, of 2816 x 4096 14.7 against 10.4). Each row
// takes compute_batch's steps.
// Affine, several rows: the chunk sums are read ahead and the empty asm keeps
// each row's value out of a branch on c < nchunks. Left alone, the compiler
// makes that branch, a row and chunk at a time, and moves the row's dot2 chain
// and its chunk sum's read behind it. Chunk slots that no lane has are passed
// over instead (the branch's one use). us, one chain after the other with
// batches of six, that branch, and now: five rows of 2816 x 4096 18.4, 10.3,
// 9.1; eight of 8192 x 1024 8.0, 9.7, 7.3, of 8192 x 512 6.9, 8.7, 5.9. Sym
// keeps its selects (five rows of 2816 x 4096 7.8; passing over slots 8.1),
// and so does one row.
template <int G, bool SYM, int KB, int T>
__device__ __forceinline__ void compute_rows(const ChunkBatch<KB>& bt, uint32_t base, uint32_t j,
                                             uint32_t nchunks, const uint16_t* xs, uint32_t row_h,
                                             const float* xsum, float (&acc)[T]) {
    constexpr bool kAffineRows = !SYM && T > 1;
    const h2_t bias = SYM ? h2_t{(_Float16)1032.0f, (_Float16)1032.0f}
                          : h2_t{(_Float16)1024.0f, (_Float16)1024.0f};
#pragma unroll
    for (int i = 0; i < KB; ++i) {
        if (kAffineRows && base + kGULanes * i >= nchunks) break;
        const uint32_t c = base + j + kGULanes * i;
        const uint32_t cc = min(c, nchunks - 1u);
        const uint32_t w[4] = {bt.w[i].x, bt.w[i].y, bt.w[i].z, bt.w[i].w};
        float dot[T], sums[T];
#pragma unroll
        for (int r = 0; r < T; ++r) {
            dot[r] = 0.0f;
            sums[r] = kAffineRows ? xsum[r * nchunks + cc] : 0.0f;
        }
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            h2_t q[4];
            nib8_to_pairs(w[b], bias, q);
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int r = 0; r < T; ++r)
                    dot[r] = dot2(q[k], staged_chunk(xs + (size_t)r * row_h, cc)[4 * b + k], dot[r]);
        }
        const float s = bf16_to_f32((uint16_t)bt.s[i]);
        float bi = 0.0f;
        if constexpr (!SYM) bi = bf16_to_f32((uint16_t)bt.b[i]);
#pragma unroll
        for (int r = 0; r < T; ++r) {
            float v = __builtin_fmaf(s, dot[r], acc[r]);
            if constexpr (!SYM) v = __builtin_fmaf(bi, kAffineRows ? sums[r] : xsum[r * nchunks + cc], v);
            if constexpr (kAffineRows) asm volatile("" : "+v"(v));
            acc[r] = c < nchunks ? v : acc[r];  // a chunk past the row end leaves acc as it is
        }
    }
}

constexpr uint32_t kRowsPerBlock = 16;  // weight rows a block, 16 lanes each
constexpr uint32_t kQmvThreads = 16u * kRowsPerBlock;
constexpr int kOneBatch = 6;  // chunks a lane loads when they are the whole row (n <= 3072)

// A weight row's lane sums over its T token rows; `bt` holds the first batch.
template <int G, bool SYM, int KB, int T, int WA>
__device__ __forceinline__ void row_sums(const uint8_t* w, const uint16_t* s, const uint16_t* b,
                                         uint32_t j, uint32_t nchunks, ChunkBatch<KB>& bt,
                                         const uint16_t* xs, uint32_t row_h, const float* xsum,
                                         float (&acc)[T]) {
    uint32_t base = 0u;
    if constexpr (KB > kOneBatch) {
        constexpr uint32_t kStep = kGULanes * KB;
        for (; base + kStep < nchunks; base += kStep) {
            ChunkBatch<KB> next;
            load_batch<G, SYM, KB, kGULanes, WA>(w, s, b, base + kStep, j, nchunks, next);
            compute_rows<G, SYM, KB, T>(bt, base, j, nchunks, xs, row_h, xsum, acc);
            bt = next;
        }
    }
    compute_rows<G, SYM, KB, T>(bt, base, j, nchunks, xs, row_h, xsum, acc);
}

// T token rows. WA: the weights' alignment, 16 or 2 (a weights pointer bound
// at a 2-byte offset, DequantInt4GEMV.swift:93-96: every row starts at the
// same offset modulo 16, since a row is a multiple of 16 bytes). KB: chunks a
// lane loads at once: kOneBatch, or 8 with the batch after requested before
// this one's sums.
// The parameters the first loads need fill the first 14 dwords, which the
// dispatch preloads into SGPRs: no kernel-argument load comes before them.
// Every block stages the token rows: with 4 weight rows a block (one wave) the
// staging took up to ten round trips to memory, and its LDS left three waves
// to a compute unit (five rows of 2816 x 4096: 15.7 us against 11.4 with 16).
template <int G, bool SYM, int T, int WA, int KB>
__global__ __launch_bounds__(kQmvThreads) void qmv_kernel(const uint8_t* __restrict__ w,
                                                          const uint16_t* __restrict__ scales,
                                                          const uint16_t* __restrict__ biases,
                                                          const uint16_t* __restrict__ x,
                                                          uint16_t* __restrict__ y, uint32_t n,
                                                          uint32_t m, uint32_t x_stride,
                                                          uint32_t y_stride) {
    extern __shared__ __align__(16) uint8_t smem[];
    const uint32_t row_h = lds_chunks_halves(n);
    uint16_t* xs = reinterpret_cast<uint16_t*>(smem);                        // T rows
    float* xsum = reinterpret_cast<float*>(smem + (size_t)T * row_h * 2u);  // T * n / 32

    const uint32_t row = blockIdx.x * kRowsPerBlock + (threadIdx.x >> 4);
    const uint32_t j = threadIdx.x & 15u;
    const bool live = row < m;
    const uint32_t rr = live ? row : 0u;
    const uint32_t ngroups = n / G, nchunks = n / 32u;
    const uint8_t* wr = w + (uint64_t)rr * (n / 2u);
    const uint16_t* sr = scales + (uint64_t)rr * ngroups;
    const uint16_t* br = biases + (uint64_t)rr * ngroups;
    ChunkBatch<KB> bt;
    auto issue_weights = [&] { load_batch<G, SYM, KB, kGULanes, WA>(wr, sr, br, 0u, j, nchunks, bt); };
    constexpr int kPer = T == 1 ? 4 : T <= 4 ? 8 : 12;
    stage_act_rows_around<SYM, decltype(issue_weights)&, kPer, kQmvThreads>(
        x, x_stride, T, n, xs, row_h, xsum, nullptr, issue_weights);
    __syncthreads();
    float acc[T];
#pragma unroll
    for (int r = 0; r < T; ++r) acc[r] = 0.0f;
    row_sums<G, SYM, KB, T, WA>(wr, sr, br, j, nchunks, bt, xs, row_h, xsum, acc);
#pragma unroll
    for (int r = 0; r < T; ++r) {
        acc[r] = group16_sum(acc[r]);
    }
    if (live && j == 0) {
#pragma unroll
        for (int r = 0; r < T; ++r) y[(uint64_t)r * y_stride + row] = f32_to_f16(acc[r]);
    }
}

// The dense MLP's gate and up rows and its activation in one launch: lanes
// 0..15 of each 32 sum a gate row, lanes 16..31 the up row beside it, each as
// qmv_kernel does, and act = half(gelu(half(gate)) * half(up)) is gelu_mul's
// (shared.hip). The halves are left in the caller's scratch too, as the
// separate launches leave them (the three stores by one lane in their order:
// the activation may share a buffer with either half). One launch for three,
// and one staging of x: 2112 x 2816 in a 30-layer pass 3.9 + 3.9 + 2.0 us
// against 5.1.
template <int G, bool SYM, int WA, int KB>
__global__ __launch_bounds__(kQmvThreads) void mlp_gate_up_kernel(
    const uint8_t* __restrict__ gate_w, const uint8_t* __restrict__ up_w,
    const uint16_t* __restrict__ gate_s, const uint16_t* __restrict__ up_s,
    const uint16_t* __restrict__ x, uint32_t n, uint32_t m, const uint16_t* __restrict__ gate_b,
    const uint16_t* __restrict__ up_b, uint16_t* gate, uint16_t* up, uint16_t* act) {
    extern __shared__ __align__(16) uint8_t smem[];
    uint16_t* xs = reinterpret_cast<uint16_t*>(smem);
    float* xsum = reinterpret_cast<float*>(smem + lds_chunks_halves(n) * 2u);
    const uint32_t row = blockIdx.x * (kRowsPerBlock / 2u) + (threadIdx.x >> 5);
    const uint32_t j = threadIdx.x & 15u;
    const bool is_up = (threadIdx.x >> 4) & 1u, live = row < m;
    const uint32_t rr = live ? row : 0u;
    const uint32_t ngroups = n / G, nchunks = n / 32u;
    const uint8_t* wr = (is_up ? up_w : gate_w) + (uint64_t)rr * (n / 2u);
    const uint16_t* sr = (is_up ? up_s : gate_s) + (uint64_t)rr * ngroups;
    const uint16_t* br = (is_up ? up_b : gate_b) + (uint64_t)rr * ngroups;
    ChunkBatch<KB> bt;
    auto issue_weights = [&] { load_batch<G, SYM, KB, kGULanes, WA>(wr, sr, br, 0u, j, nchunks, bt); };
    stage_act_rows_around<SYM, decltype(issue_weights)&, 4, kQmvThreads>(x, n, 1u, n, xs, 0u, xsum,
                                                                         nullptr, issue_weights);
    __syncthreads();
    float acc[1] = {0.0f};
    row_sums<G, SYM, KB, 1, WA>(wr, sr, br, j, nchunks, bt, xs, 0u, xsum, acc);
    const uint16_t v = f32_to_f16(group16_sum(acc[0]));
    const uint32_t other = shfl_xor((uint32_t)v, 16);  // gate lanes receive the up row's
    if (live && !is_up && j == 0) {
        gate[row] = v;
        up[row] = (uint16_t)other;
        act[row] = f32_to_f16(gate_activation<TSG_ACT_GELU_TANH>(f16_to_f32(v)) *
                              f16_to_f32((uint16_t)other));
    }
}

// out[r, k] = half(fma(q, s, b)), b = -8 s under sym (prefill.metal:1021-1026).
template <int G, bool SYM>
__global__ void dequant_f16_kernel(const uint8_t* __restrict__ w,
                                   const uint16_t* __restrict__ scales,
                                   const uint16_t* __restrict__ biases,
                                   uint16_t* __restrict__ out, uint32_t rows, uint32_t n) {
    const uint64_t total = (uint64_t)rows * n;
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < total;
         i += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t r = i / n;
        const uint32_t k = (uint32_t)(i - r * n);
        const uint8_t byte = w[r * (n / 2u) + k / 2u];
        const uint32_t q = (k & 1u) ? (byte >> 4) : (byte & 0xFu);
        const uint32_t g = k / G;
        const float s = bf16_to_f32(scales[r * (n / G) + g]);
        const float b = SYM ? -8.0f * s : bf16_to_f32(biases[r * (n / G) + g]);
        out[i] = f32_to_f16(__builtin_fmaf((float)q, s, b));
    }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

template <int G, bool SYM, int WA>
tsg_status launch_qmv(hipStream_t s, const uint8_t* w, const uint16_t* sc, const uint16_t* bi,
                      const uint16_t* x, uint32_t xs, uint16_t* y, uint32_t ys, uint32_t t,
                      uint32_t m, uint32_t n) {
    const dim3 grid((m + kRowsPerBlock - 1u) / kRowsPerBlock), block(kQmvThreads);
    const size_t lds = (size_t)t * (lds_chunks_halves(n) * 2u + (SYM ? 0u : (n / 32u) * 4u));
    const bool one = n <= 32u * kGULanes * (uint32_t)kOneBatch;
#define TSG_QMV_CASE(TT)                                                                          \
    case TT: {                                                                                    \
        auto kern = one ? qmv_kernel<G, SYM, TT, WA, kOneBatch> : qmv_kernel<G, SYM, TT, WA, 8>;  \
        hipLaunchKernelGGL(kern, grid, block, lds, s, w, sc, bi, x, y, n, m, xs, ys);             \
        break;                                                                                    \
    }
    switch (t) {
        TSG_QMV_CASE(1)
        TSG_QMV_CASE(2)
        TSG_QMV_CASE(3)
        TSG_QMV_CASE(4)
        TSG_QMV_CASE(5)
        TSG_QMV_CASE(6)
        TSG_QMV_CASE(7)
        TSG_QMV_CASE(8)
        default: return fail(TSG_ERR_INVALID_ARGUMENT, "t=%u not in 1..8", t);
    }
#undef TSG_QMV_CASE
    return check_launch("qmv_int4");
}

// LDS of one staged row with its affine sums.
size_t staged_row_bytes(uint32_t n) { return (size_t)lds_chunks_halves(n) * 2u + (n / 32u) * 4u; }

tsg_status check_qmv(const tsg_ctx* ctx, const uint8_t* w, const uint16_t* sc, const uint16_t* bi,
                     const uint16_t* x, uint32_t xs, const uint16_t* y, uint32_t m, uint32_t n) {
    TSG_REQUIRE(ctx, TSG_ERR_INVALID_ARGUMENT, "ctx is NULL");
    TSG_REQUIRE(w && sc && x && y, TSG_ERR_INVALID_ARGUMENT, "NULL operand");
    TSG_REQUIRE(ctx->scheme == TSG_SYM || bi, TSG_ERR_INVALID_ARGUMENT,
                "biases is NULL under the affine scheme");
    TSG_REQUIRE(n > 0 && n % ctx->group_size == 0, TSG_ERR_INVALID_ARGUMENT,
                "N must be a multiple of %u, got %u", ctx->group_size, n);
    TSG_REQUIRE(m > 0, TSG_ERR_INVALID_ARGUMENT, "m must be positive");
    // The reference reads weights through ushort* and needs a 2-aligned
    // weightsOffset (DequantInt4GEMV.swift:91-96). Rows are n / 2 bytes, a
    // multiple of 16 (n % 32 == 0), so every 16-byte chunk has the base's
    // alignment: 16-byte loads when the base is 16-byte aligned, else the
    // 2-byte-safe load (load16_a2).
    TSG_REQUIRE((reinterpret_cast<uintptr_t>(w) & 1u) == 0, TSG_ERR_ALIGNMENT,
                "weights need a 2-aligned offset (got %p)", (const void*)w);
    TSG_REQUIRE((reinterpret_cast<uintptr_t>(sc) & 1u) == 0 &&
                    (reinterpret_cast<uintptr_t>(bi ? bi : sc) & 1u) == 0,
                TSG_ERR_ALIGNMENT, "scales and biases must be 2-byte aligned");
    TSG_REQUIRE(aligned16(x) && xs % 8 == 0, TSG_ERR_ALIGNMENT,
                "x rows must be 16-byte aligned");
    TSG_REQUIRE(staged_row_bytes(n) <= 160u * 1024u, TSG_ERR_UNSUPPORTED,
                "a row of n=%u does not fit the LDS staging", n);
    return TSG_OK;
}

tsg_status qmv_dispatch(tsg_ctx* ctx, hipStream_t s, const uint8_t* w, const uint16_t* sc,
                        const uint16_t* bi, const uint16_t* x, uint32_t xs, uint16_t* y,
                        uint32_t ys, uint32_t t, uint32_t m, uint32_t n) {
    tsg_status st = check_qmv(ctx, w, sc, bi, x, xs, y, m, n);
    if (st) return st;
    const bool w16 = aligned16(w);
    // Rows are independent (each is summed exactly as on its own), so rows
    // that do not fit the LDS staging together run in several launches.
    const uint32_t fit = (uint32_t)std::min<size_t>(kMaxRows, (160u * 1024u) / staged_row_bytes(n));
    const bool sym = ctx->scheme == TSG_SYM;
    for (uint32_t r0 = 0; r0 < t; r0 += fit) {
        const uint32_t tt = std::min(fit, t - r0);
        const uint16_t* xr = x + (size_t)r0 * xs;
        uint16_t* yr = y + (size_t)r0 * ys;
#define TSG_QMV_WA(WA)                                                                 \
    if (ctx->group_size == 32)                                                         \
        st = sym ? launch_qmv<32, true, WA>(s, w, sc, sc, xr, xs, yr, ys, tt, m, n)    \
                 : launch_qmv<32, false, WA>(s, w, sc, bi, xr, xs, yr, ys, tt, m, n);  \
    else                                                                               \
        st = sym ? launch_qmv<64, true, WA>(s, w, sc, sc, xr, xs, yr, ys, tt, m, n)    \
                 : launch_qmv<64, false, WA>(s, w, sc, bi, xr, xs, yr, ys, tt, m, n);
        if (w16) {
            TSG_QMV_WA(16)
        } else {
            TSG_QMV_WA(2)
        }
#undef TSG_QMV_WA
        if (st) return st;
    }
    return TSG_OK;
}

template <int G, bool SYM, int WA>
tsg_status launch_mlp_gate_up(hipStream_t s, const tsg_int4_projection& g,
                              const tsg_int4_projection& u, const uint16_t* x, uint16_t* gate,
                              uint16_t* up, uint16_t* act) {
    const uint32_t m = g.rows, n = g.cols;
    const dim3 grid((m + kRowsPerBlock / 2u - 1u) / (kRowsPerBlock / 2u)), block(kQmvThreads);
    const size_t lds = (size_t)lds_chunks_halves(n) * 2u + (SYM ? 0u : (n / 32u) * 4u);
    const bool one = n <= 32u * kGULanes * (uint32_t)kOneBatch;
    auto kern = one ? mlp_gate_up_kernel<G, SYM, WA, kOneBatch> : mlp_gate_up_kernel<G, SYM, WA, 8>;
    hipLaunchKernelGGL(kern, grid, block, lds, s, g.weights, u.weights, g.scales, u.scales, x, n, m,
                       g.biases, u.biases, gate, up, act);
    return check_launch("mlp_gate_up");
}

template <int G, bool SYM>
tsg_status mlp_gate_up(hipStream_t s, const tsg_int4_projection& g, const tsg_int4_projection& u,
                       const uint16_t* x, uint16_t* gate, uint16_t* up, uint16_t* act) {
    return aligned16(g.weights) && aligned16(u.weights)
               ? launch_mlp_gate_up<G, SYM, 16>(s, g, u, x, gate, up, act)
               : launch_mlp_gate_up<G, SYM, 2>(s, g, u, x, gate, up, act);
}

}  // namespace
}  // namespace tsg

using namespace tsg;

extern "C" tsg_status tsg_qmv_int4(tsg_ctx* ctx, tsg_stream stream, const uint8_t* w,
                                   const uint16_t* scales, const uint16_t* biases,
                                   const uint16_t* x, uint16_t* y, uint32_t m, uint32_t n) {
    return qmv_dispatch(ctx, as_stream(stream), w, scales, biases, x, n, y, m, 1, m, n);
}

extern "C" tsg_status tsg_qmv_int4_rows(tsg_ctx* ctx, tsg_stream stream, const uint8_t* w,
                                        const uint16_t* scales, const uint16_t* biases,
                                        const uint16_t* x, uint32_t x_stride, uint16_t* y,
                                        uint32_t y_stride, uint32_t t, uint32_t m,
                                        uint32_t n) {
    TSG_REQUIRE(t >= 1 && t <= kMaxRows, TSG_ERR_INVALID_ARGUMENT, "t=%u not in 1..%u", t,
                kMaxRows);
    return qmv_dispatch(ctx, as_stream(stream), w, scales, biases, x, x_stride, y, y_stride, t,
                        m, n);
}

// SharedExpertInt4.encode (Kernels/MoE/SharedExpertInt4.swift:30-93): the
// dense int4 MLP y = down(gelu(gate x) * up x). The reference encodes QMV gate
// and up into fp16 scratch, gelu_mul_fp16 and QMV down; here the first three
// are one launch, with their bits.
extern "C" tsg_status tsg_shared_expert_int4(
    tsg_ctx* ctx, tsg_stream stream, const uint16_t* x, uint64_t x_bytes,
    const tsg_int4_projection* gate, const tsg_int4_projection* up,
    const tsg_int4_projection* down, uint16_t* y, uint64_t y_bytes, uint16_t* scratch_gate,
    uint64_t scratch_gate_bytes, uint16_t* scratch_up, uint64_t scratch_up_bytes,
    uint16_t* scratch_act, uint64_t scratch_act_bytes) {
    TSG_REQUIRE(ctx && gate && up && down, TSG_ERR_INVALID_ARGUMENT, "NULL ctx or projection");
    if (!(gate->rows == up->rows && gate->cols == up->cols && down->rows == gate->cols &&
          down->cols == gate->rows))
        return fail(TSG_ERR_INVALID_ARGUMENT,
                    "dimensionMismatch: gate=(%u,%u) up=(%u,%u) down=(%u,%u)", gate->rows,
                    gate->cols, up->rows, up->cols, down->rows, down->cols);
    const uint64_t required = (uint64_t)gate->rows * 2u;
    if (scratch_gate_bytes < required || scratch_up_bytes < required || scratch_act_bytes < required)
        return fail(TSG_ERR_INVALID_ARGUMENT,
                    "scratchTooSmall: need %llu bytes per intermediate buffer",
                    (unsigned long long)required);
    if (x_bytes < (uint64_t)gate->cols * 2u)
        return fail(TSG_ERR_INVALID_ARGUMENT, "scratchTooSmall: input range exceeds x buffer");
    if (y_bytes < (uint64_t)down->rows * 2u)
        return fail(TSG_ERR_INVALID_ARGUMENT, "scratchTooSmall: output range exceeds y buffer");
    tsg_status st;
    if ((st = check_qmv(ctx, gate->weights, gate->scales, gate->biases, x, gate->cols, scratch_gate,
                        gate->rows, gate->cols)))
        return st;
    if ((st = check_qmv(ctx, up->weights, up->scales, up->biases, x, up->cols, scratch_up, up->rows,
                        up->cols)))
        return st;
    TSG_REQUIRE(scratch_act, TSG_ERR_INVALID_ARGUMENT, "NULL operand");
    // One launch needs x and the halves apart, and the activation apart from x
    // and from each half or in its place. Where buffers share bytes otherwise
    // (the activation in x's buffer, both halves in one) the separate launches
    // keep their order of reads and writes.
    const uint64_t x_len = (uint64_t)gate->cols * 2u;
    auto apart = [](const uint16_t* a, uint64_t an, const uint16_t* b, uint64_t bn) {
        const uintptr_t a0 = reinterpret_cast<uintptr_t>(a), b0 = reinterpret_cast<uintptr_t>(b);
        return a0 + an <= b0 || b0 + bn <= a0;
    };
    auto in_place = [&](const uint16_t* half) {
        return scratch_act == half || apart(scratch_act, required, half, required);
    };
    const bool one_launch = apart(x, x_len, scratch_act, required) &&
                            apart(x, x_len, scratch_gate, required) &&
                            apart(x, x_len, scratch_up, required) &&
                            apart(scratch_gate, required, scratch_up, required) &&
                            in_place(scratch_gate) && in_place(scratch_up);
    if (!one_launch) {
        if ((st = tsg_qmv_int4(ctx, stream, gate->weights, gate->scales, gate->biases, x,
                               scratch_gate, gate->rows, gate->cols)) ||
            (st = tsg_qmv_int4(ctx, stream, up->weights, up->scales, up->biases, x, scratch_up,
                               up->rows, up->cols)) ||
            (st = tsg_gelu_mul_f16(ctx, stream, scratch_gate, scratch_up, scratch_act, gate->rows)))
            return st;
        return tsg_qmv_int4(ctx, stream, down->weights, down->scales, down->biases, scratch_act, y,
                            down->rows, down->cols);
    }
    hipStream_t s = as_stream(stream);
    tsg_int4_projection g = *gate, u = *up;
    const bool sym = ctx->scheme == TSG_SYM;
    if (sym) g.biases = g.scales, u.biases = u.scales;  // not read
    if (ctx->group_size == 32)
        st = sym ? mlp_gate_up<32, true>(s, g, u, x, scratch_gate, scratch_up, scratch_act)
                 : mlp_gate_up<32, false>(s, g, u, x, scratch_gate, scratch_up, scratch_act);
    else
        st = sym ? mlp_gate_up<64, true>(s, g, u, x, scratch_gate, scratch_up, scratch_act)
                 : mlp_gate_up<64, false>(s, g, u, x, scratch_gate, scratch_up, scratch_act);
    if (st) return st;
    return tsg_qmv_int4(ctx, stream, down->weights, down->scales, down->biases, scratch_act, y,
                        down->rows, down->cols);
}

extern "C" tsg_status tsg_debug_dequant_f16(tsg_ctx* ctx, tsg_stream stream, const uint8_t* w,
                                            const uint16_t* scales, const uint16_t* biases,
                                            uint16_t* out, uint32_t rows, uint32_t n) {
    TSG_REQUIRE(ctx && w && scales && out, TSG_ERR_INVALID_ARGUMENT, "NULL operand");
    TSG_REQUIRE(ctx->scheme == TSG_SYM || biases, TSG_ERR_INVALID_ARGUMENT,
                "biases is NULL under the affine scheme");
    TSG_REQUIRE(n > 0 && n % ctx->group_size == 0 && rows > 0, TSG_ERR_INVALID_ARGUMENT,
                "bad shape rows=%u n=%u", rows, n);
    const uint64_t total = (uint64_t)rows * n;
    uint64_t blocks = (total + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipStream_t s = as_stream(stream);
    const bool sym = ctx->scheme == TSG_SYM;
    if (ctx->group_size == 32) {
        if (sym) hipLaunchKernelGGL((dequant_f16_kernel<32, true>), dim3(blocks), dim3(256), 0, s, w, scales, scales, out, rows, n);
        else hipLaunchKernelGGL((dequant_f16_kernel<32, false>), dim3(blocks), dim3(256), 0, s, w, scales, biases, out, rows, n);
    } else {
        if (sym) hipLaunchKernelGGL((dequant_f16_kernel<64, true>), dim3(blocks), dim3(256), 0, s, w, scales, scales, out, rows, n);
        else hipLaunchKernelGGL((dequant_f16_kernel<64, false>), dim3(blocks), dim3(256), 0, s, w, scales, biases, out, rows, n);
    }
    return check_launch("debug_dequant_f16");
}
