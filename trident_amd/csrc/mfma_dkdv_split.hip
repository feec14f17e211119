// Launches of the dK/dV kernels whose items are split along the rows (split.hpp).
#include "mfma_dkdv.hpp"

namespace tri {
namespace {

// Few heads: items split along the rows, in workgroups with boundary handling, chosen as for a ragged length.
bool dkdv_splits_phased(const KParams& p) {
    return p.D == 128 && (p.mask == nullptr || (p.ms[2] == 0 && (p.mask_binary || p.S % 128 == 0)));
}
SplitShape dkdv_split_shape(const KParams& p) {
    if (dkdv_splits_phased(p)) {
        const double us = split_work(p) * 1.35;
        return SplitShape{128, 1, 2, false, 20, us, us, split_gain(p)};
    }
    const int slots = p.D == 128 || (p.D == 64 && p.mask != nullptr && p.thr8 > 0) ? 1 : p.D == 64 || p.mask != nullptr ? 2 : 3;
    const double us = split_work(p) * (p.D >= 64 ? 1.65 : p.D == 32 ? 1.22 : 1.05);
    return SplitShape{128, slots, 2, false, 20, us, slots == 1 ? us : (p.D == 64 ? 0.58 : 0.52) * us, split_gain(p) - (p.D < 64 ? 0.04 : 0.0), split_unclassed(p)};
}

template <typename T, int D, bool CAUSAL, int MASK>
int launch_dkdv_split(const KParams& p, hipStream_t stream) {
    const dim3 grid = split_grid(p);
    if constexpr (D == 128) {
        if (dkdv_splits_phased(p)) {
            if (p.thr8 > 0) hipLaunchKernelGGL((mfma_dkdv_phased_kernel<T, D, CAUSAL, true, MASK, true, true>), grid, dim3(512), 0, stream, p);
            else hipLaunchKernelGGL((mfma_dkdv_phased_kernel<T, D, CAUSAL, false, MASK, true, true>), grid, dim3(512), 0, stream, p);
            return static_cast<int>(hipGetLastError());
        }
    }
    if constexpr (D < 128 || MASK != kNoMask) {
        if (p.thr8 > 0) hipLaunchKernelGGL((mfma_dkdv_wide_kernel<T, D, CAUSAL, MASK, true, true, true>), grid, dim3(256), 0, stream, p);
        else hipLaunchKernelGGL((mfma_dkdv_wide_kernel<T, D, CAUSAL, MASK, false, true, true>), grid, dim3(256), 0, stream, p);
    }
    return static_cast<int>(hipGetLastError());
}

template <typename T, int D>
int launch_dkdv_split_variant(int dtype, const KParams& p, hipStream_t stream) {
    if (p.causal) return launch_dkdv_split<T, D, true, kNoMask>(p, stream);
    if (p.mask == nullptr) return launch_dkdv_split<T, D, false, kNoMask>(p, stream);
    if (p.mask_dtype == TRI_ATTN_F32) return launch_dkdv_split<T, D, false, kMaskF32>(p, stream);
    if (p.mask_dtype == dtype) return launch_dkdv_split<T, D, false, kMaskT>(p, stream);
    return TRI_ATTN_EDTYPE;
}

template <typename T>
int launch_dkdv_split_head(int dtype, const KParams& p, hipStream_t stream) {
    if (p.D == 128) return launch_dkdv_split_variant<T, 128>(dtype, p, stream);
    if (p.D == 64) return launch_dkdv_split_variant<T, 64>(dtype, p, stream);
    if (p.D == 32) return launch_dkdv_split_variant<T, 32>(dtype, p, stream);
    return launch_dkdv_split_variant<T, 16>(dtype, p, stream);
}

}  // namespace

int64_t mfma_dkdv_workspace(const KParams& p) {
    KParams plan = p;
    return plan_split(dkdv_split_shape(p), p.causal != 0, &plan);
}

int launch_mfma_dkdv_split(int dtype, KParams p, hipStream_t stream) {
    const SplitShape shape = dkdv_split_shape(p);
    if (!take_workspace(plan_split(shape, p.causal != 0, &p), &p)) return TRI_ATTN_ENOFUSE;
    const int rc = dtype == TRI_ATTN_BF16 ? launch_dkdv_split_head<bf16_t>(dtype, p, stream)
                                          : launch_dkdv_split_head<f16_t>(dtype, p, stream);
    return rc ? rc : launch_combine_backward(dtype, p, shape.rows, true, stream);
}

}  // namespace tri
