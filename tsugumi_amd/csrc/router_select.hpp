// router_select.hpp — the ordering of router logits, shared by the top-8
// selections (decode.hip, prompt_router.hip).
#pragma once

#include "tsg_internal.hpp"

namespace tsg {
namespace {

// Scores as order-preserving 32-bit keys (0 marks "not eligible"; -0 is keyed
// as +0, the two compare equal).
__device__ __forceinline__ uint32_t order_key(float v) {
    const uint32_t u = __float_as_uint(v + 0.0f);  // -0 -> +0
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ float order_key_value(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t k) {
    return __builtin_amdgcn_update_dpp(0u, k, CTRL, 0xF, 0xF, false);
}

}  // namespace

// The prompt router (prompt_router.hip): routes `rows` hidden rows, the
// arguments already checked by the caller.
struct PromptRouterArgs {
    const uint16_t* w;       // bf16 [ne, d]
    const uint16_t* hidden;  // fp16 rows, `stride` elements apart
    const uint16_t* es;      // bf16 [d]
    const uint16_t* pes;     // bf16 [ne]
    uint32_t* out_idx;
    uint16_t* out_w;
    uint32_t stride, ne, d, rows;
};
tsg_status prompt_router_launch(tsg_ctx* ctx, hipStream_t stream, const PromptRouterArgs& a);

}  // namespace tsg
