// What the kernels that write fragment after fragment share (conv2d_i8_px.hip, conv2d_i8_pt*.hip): a fragment of 32 channels x 32
// positions from its accumulators to its stores.
#pragma once
#include "igemm_i8.hpp"

namespace tsx {

constexpr unsigned NOWHERE = 0xfffffff0u;      // beyond any buffer: loads 0, stores nothing
constexpr int STREAMING = 2;                   // a buffer instruction's non-temporal bit

// all of LDS written and read, no wait for global loads and stores
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// where position l % 32 of a fragment has its values: byte offsets of the lane's first channel in fp32 tensors, of its 16 channels
// in the consumer's staged one (or NOWHERE), and the consumer's scale
struct PxWhere { unsigned out, st; float scale; };

// RES: a residual joins.  F32, Q: fp32 values, requantized ones leave.  MISHX: the activation is the exact Mish.  STREAM: fp32 values in
// streaming stores.  terms: the 32 channels'
// scales and biases in LDS; row0, row: byte offset of the first channel in an fp32 image, and of one to the next.  next_residual() is called
// when res is free.  The loads and stores are the same in every call, without branches: the compiler counts how many are in flight
// and waits for those it needs only.
template <bool RES, bool F32, bool Q, bool MISHX, bool STREAM = false, class Next>
__device__ __forceinline__ void px_finish(const EpiParams &p, const v16i &acc, const float *terms, const float (&res)[16], const PxWhere &to, unsigned row0, unsigned row,
                                          __amdgpu_buffer_rsrc_t outr, __amdgpu_buffer_rsrc_t str, const MishTablesInLds &tables, Next &&next_residual) {
    float v[16];
    int at = 4 * (threadIdx.x % 64 / 32);
    asm volatile("" : "+v"(at));     // (read in every turn, not kept in 32 registers)
    const float *term = terms + at;
    static_for<0, 4>([&](auto gc) {
        constexpr int g4 = decltype(gc)::value;
        const v4f dq = *reinterpret_cast<const v4f *>(term + 8 * g4), bias = *reinterpret_cast<const v4f *>(term + 32 + 8 * g4);
        static_for<0, 4>([&](auto ic) { constexpr int i = decltype(ic)::value; v[4 * g4 + i] = __fadd_rn(__fmul_rn(float(acc[4 * g4 + i]), dq[i]), bias[i]); });
    });
    if (RES && !p.res_after) static_for<0, 16>([&](auto rc) { constexpr int r = decltype(rc)::value; v[r] = __fadd_rn(v[r], res[r]); });
    uint32_t word[4];
    if (MISHX) {
        if constexpr (Q && !F32) {
            if (RES && p.res_after) mish_words_for_rounding<true>(v, res, to.scale, p.n_qscales == 1, word, tables);
            else mish_words_for_rounding<false>(v, res, to.scale, p.n_qscales == 1, word, tables);
        } else {
            mish_fragment(v, tables);
        }
    } else {
        activate_results(v, p.act, p.slope);
    }
    if (RES && p.res_after && !(MISHX && Q && !F32)) static_for<0, 16>([&](auto rc) { constexpr int r = decltype(rc)::value; v[r] = __fadd_rn(v[r], res[r]); });
    next_residual();
    if (F32) static_for<0, 16>([&](auto rc) {
        constexpr int r = decltype(rc)::value;
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v[r]), outr, int(to.out), int(row0 + (8 * (r / 4) + r % 4) * row), STREAM ? STREAMING : 0);
    });
    if (Q) {
        if (!(MISHX && !F32)) quantize_words(v, to.scale, p.n_qscales == 1, word);
        const auto s02 = __builtin_amdgcn_permlane32_swap(word[0], word[2], false, false);
        const auto s13 = __builtin_amdgcn_permlane32_swap(word[1], word[3], false, false);
        typedef unsigned v4u __attribute__((ext_vector_type(4)));
        const v4u packed = {s02[0], s02[1], s13[0], s13[1]};
        __builtin_amdgcn_raw_buffer_store_b128(packed, str, int(to.st), 0, 0);
        if (p.st_up == 2) {
            const unsigned right = unsigned(p.st_cp), down = unsigned(p.st_ws) * unsigned(p.st_cp);
            const bool in = to.st != NOWHERE;
            __builtin_amdgcn_raw_buffer_store_b128(packed, str, int(in ? to.st + right : NOWHERE), 0, 0);
            __builtin_amdgcn_raw_buffer_store_b128(packed, str, int(in ? to.st + down : NOWHERE), 0, 0);
            __builtin_amdgcn_raw_buffer_store_b128(packed, str, int(in ? to.st + down + right : NOWHERE), 0, 0);
        }
    }
}

}  // namespace tsx
