// Launches of the forward kernel whose items are split along the keys (split.hpp).
#include "mfma_fwd.hpp"

namespace tri {
namespace {

// Few heads: items split along the keys, in workgroups with boundary handling. As many waves as launch_fwd_waves gives a ragged
// length, at D = 128 eight (four beside a mask and dropout, which need the whole register file).
template <typename T, int D, bool CAUSAL, int MASK>
int launch_fwd_split(const KParams& p, int waves, hipStream_t stream) {
    constexpr int NW = D == 128 ? 8 : 4;
    const dim3 grid = split_grid(p);
    if (waves != NW) {
        if constexpr (D == 128 && MASK != kNoMask) hipLaunchKernelGGL((mfma_fwd_kernel<T, D, 4, CAUSAL, MASK, true, true, true>), grid, dim3(256), 0, stream, p);
    } else if (p.thr8 > 0) {
        if constexpr (!(D == 128 && MASK != kNoMask)) hipLaunchKernelGGL((mfma_fwd_kernel<T, D, NW, CAUSAL, MASK, true, true, true>), grid, dim3(64 * NW), 0, stream, p);
    } else {
        hipLaunchKernelGGL((mfma_fwd_kernel<T, D, NW, CAUSAL, MASK, false, true, true>), grid, dim3(64 * NW), 0, stream, p);
    }
    return static_cast<int>(hipGetLastError());
}

template <typename T, int D>
int launch_fwd_split_variant(int dtype, const KParams& p, int waves, hipStream_t stream) {
    if (p.causal) return launch_fwd_split<T, D, true, kNoMask>(p, waves, stream);
    if (p.mask == nullptr) return launch_fwd_split<T, D, false, kNoMask>(p, waves, stream);
    if (p.mask_dtype == TRI_ATTN_F32) return launch_fwd_split<T, D, false, kMaskF32>(p, waves, stream);
    if (p.mask_dtype == dtype) return launch_fwd_split<T, D, false, kMaskT>(p, waves, stream);
    return TRI_ATTN_EDTYPE;
}

SplitShape fwd_split_shape(const KParams& p) {
    const bool f32_mask = p.mask != nullptr && p.mask_dtype == TRI_ATTN_F32;
    const int waves = p.D == 128 && !(p.mask != nullptr && p.thr8 > 0) ? 8 : 4;
    const int slots = p.D == 128 ? 1 : p.D == 64 ? 2 : p.mask == nullptr ? 4 : p.thr8 > 0 || (f32_mask && p.D == 32) ? 2 : 3;
    // (beside mask and dropout at D = 128 whole launches of multiples of 256 have eight waves, half the items: bf16 fp32 mask, 10 heads,
    // S=4096, whole 90 us, split 213)
    const int whole_rows = p.D == 128 && waves == 4 && p.S % 256 == 0 ? 256 : 32 * waves;
    const double us = split_work(p) * (p.D == 128 ? 1.4 : p.D == 64 ? 0.9 : 0.62);
    return SplitShape{32 * waves, slots, 1, true, 20, us, slots == 1 ? us : 0.6 * us, split_gain(p), split_unclassed(p), whole_rows};
}

template <typename T>
int launch_fwd_split_head(int dtype, const KParams& p, int waves, hipStream_t stream) {
    if (p.D == 128) return launch_fwd_split_variant<T, 128>(dtype, p, waves, stream);
    if (p.D == 64) return launch_fwd_split_variant<T, 64>(dtype, p, waves, stream);
    if (p.D == 32) return launch_fwd_split_variant<T, 32>(dtype, p, waves, stream);
    return launch_fwd_split_variant<T, 16>(dtype, p, waves, stream);
}

}  // namespace

int64_t mfma_fwd_workspace(const KParams& p) {
    KParams plan = p;
    return plan_split(fwd_split_shape(p), p.causal != 0, &plan);
}

int launch_mfma_fwd_split(int dtype, KParams p, hipStream_t stream) {
    const SplitShape shape = fwd_split_shape(p);
    if (!take_workspace(plan_split(shape, p.causal != 0, &p), &p)) return TRI_ATTN_ENOFUSE;
    const int rc = dtype == TRI_ATTN_BF16 ? launch_fwd_split_head<bf16_t>(dtype, p, shape.rows / 32, stream)
                                          : launch_fwd_split_head<f16_t>(dtype, p, shape.rows / 32, stream);
    return rc ? rc : launch_combine_forward(dtype, p, shape.rows, stream);
}

}  // namespace tri
