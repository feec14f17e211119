// Shared device helpers for the attention kernels (gfx950 only).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "tri_attn.h"

namespace tri {

constexpr float kLog2e = 1.4426950408889634f;  // trident/language/constant.py:17-20

typedef _Float16 f16_t;
typedef __bf16 bf16_t;

// Kernel-side view of TriAttnArgs: batch/head/row strides only (innermost stride is 1),
// scale folded into the log2 domain, dropout threshold resolved.
struct KParams {
    const void* q;
    const void* k;
    const void* v;
    void* o;
    float* lse;
    const void* mask;
    const void* d_o;
    void* dq;
    void* dk;
    void* dv;
    void* dmask;
    float* delta;
    const uint8_t* mcls;   // classes of the mask's 64 x 64 blocks or nullptr
    int64_t qs[3], ks[3], vs[3], os[3], dos[3], dqs[3], dks[3], dvs[3], ms[3], dms[3];
    int64_t mcs[3];        // strides of mcls (bytes) over batch, head, row block; the column-block stride is 1
    int B, H, S, D;
    int causal;
    int mask_dtype;
    int mask_padded;   // mask rows may be read up to the next multiple of 64 entries (finite values there)
    int mask_binary;   // every mask value is 0 or -inf
    float scale;       // softmax_scale
    float scale_log2;  // softmax_scale * log2(e)
    float inv_scale;   // 1 / softmax_scale (0 where the scale is 0)
    uint32_t seed_lo, seed_hi, offset;
    int dmask_acc;     // dmask is summed over a broadcast dimension (stride 0): fp32 buffer, atomic adds
    int thr8;          // 0 = no dropout; keep iff u8 >= thr8
    float zscale;      // 256 / (256 - thr8), 0 when thr8 == 256
    // A launch whose items are split along the streamed dimension (split.hpp): 0 units = it is not.
    int part_units;    // workgroups per head
    int part_tiles;    // 64-row tiles of a part
    int part_group;    // causal: how many items in a row have the same number of parts; 0: all have the same
    float* partial;    // fp32 accumulators of the parts, then (forward) their row statistics
    void* workspace;   // what the caller has for them
    int64_t workspace_bytes;
};

template <typename T>
__device__ __forceinline__ float to_f32(T x) {
    return static_cast<float>(x);
}
template <typename T>
__device__ __forceinline__ T from_f32(float x) {
    return static_cast<T>(x);
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float fast_log2(float x) { return __builtin_amdgcn_logf(x); }

__device__ __forceinline__ float load_mask_elem(const void* base, int dtype, int64_t off) {
    if (dtype == TRI_ATTN_F32) return static_cast<const float*>(base)[off];
    if (dtype == TRI_ATTN_F16) return to_f32(static_cast<const f16_t*>(base)[off]);
    return to_f32(static_cast<const bf16_t*>(base)[off]);
}
__device__ __forceinline__ void store_mask_elem(void* base, int dtype, int64_t off, float x) {
    if (dtype == TRI_ATTN_F32) static_cast<float*>(base)[off] = x;
    else if (dtype == TRI_ATTN_F16) static_cast<f16_t*>(base)[off] = from_f32<f16_t>(x);
    else static_cast<bf16_t*>(base)[off] = from_f32<bf16_t>(x);
}

// Philox4x32-10 (Random123 constants; the generator behind tl.rand used at
// trident/kernel/attention.py:159).
struct Philox4 {
    uint32_t w[4];
};
constexpr uint32_t kPhiloxM0 = 0xD2511F53u, kPhiloxM1 = 0xCD9E8D57u;  // multipliers
constexpr uint32_t kPhiloxW0 = 0x9E3779B9u, kPhiloxW1 = 0xBB67AE85u;  // key increments
// One of the ten rounds (r = 0 .. 9), for callers that spread them over other work or have folded the first ones. (The exclusive or of
// three words is one instruction, which the compiler does not find by itself.)
__device__ __forceinline__ void philox_round(Philox4& s, int r, uint32_t k0, uint32_t k1) {
    const uint64_t p0 = static_cast<uint64_t>(kPhiloxM0) * s.w[0];
    const uint64_t p1 = static_cast<uint64_t>(kPhiloxM1) * s.w[2];
    s.w[0] = __builtin_amdgcn_bitop3_b32(static_cast<uint32_t>(p1 >> 32), s.w[1], k0 + r * kPhiloxW0, 0x96);
    s.w[2] = __builtin_amdgcn_bitop3_b32(static_cast<uint32_t>(p0 >> 32), s.w[3], k1 + r * kPhiloxW1, 0x96);
    s.w[1] = static_cast<uint32_t>(p1);
    s.w[3] = static_cast<uint32_t>(p0);
}
__device__ __forceinline__ Philox4 philox4x32_10(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3,
                                                 uint32_t k0, uint32_t k1) {
    Philox4 out = {{c0, c1, c2, c3}};
#pragma unroll
    for (int r = 0; r < 10; ++r) philox_round(out, r, k0, k1);
    return out;
}

// The 16 dropout bytes of the 4x4 block (rows 4*ib.., cols 4*jb..) of head bh:
// word r = row within the block, byte c = column within the block.
__device__ __forceinline__ Philox4 dropout_block(const KParams& p, uint32_t bh, uint32_t ib, uint32_t jb) {
    return philox4x32_10(jb, ib, bh, p.offset, p.seed_lo, p.seed_hi);
}
__device__ __forceinline__ bool dropout_keep(const KParams& p, uint32_t bh, uint32_t i, uint32_t j) {
    const Philox4 r = dropout_block(p, bh, i >> 2, j >> 2);
    const uint32_t s = i & 3;
    const uint32_t word = s == 0 ? r.w[0] : (s == 1 ? r.w[1] : (s == 2 ? r.w[2] : r.w[3]));
    const int u8 = static_cast<int>((word >> (8 * (j & 3))) & 0xffu);
    return u8 >= p.thr8;
}

}  // namespace tri
