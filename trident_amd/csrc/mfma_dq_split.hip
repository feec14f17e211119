// Launches of the dQ kernels whose items are split along the keys (split.hpp).
#include "mfma_dq.hpp"

namespace tri {
namespace {

// Few heads: items split along the keys, in workgroups with boundary handling: at D = 128 without mask and dropout the phased
// kernel, else the one above with as many waves as a ragged length has.
SplitShape dq_split_shape(const KParams& p) {
    const int waves = p.D == 128 && p.mask == nullptr && p.thr8 <= 0 ? 8 : 4;
    const int slots = p.D == 128 ? 1 : p.D == 64 || (p.D == 32 && p.mask != nullptr) ? 2 : p.mask != nullptr ? 3 : 4;
    // Beside a mask at D = 128 parts have four waves, one per SIMD, and take longer than they promise (bf16 key mask with dropout, 12
    // heads, S=1489, whole 45 us, split 59); whole launches of multiples of 256 have eight, half the items (8 heads, S=6400, 287 and 400).
    const int whole_rows = p.D == 128 && p.mask != nullptr && p.thr8 <= 0 && p.S % 256 == 0 ? 256 : 32 * waves;
    const double gain = split_gain(p) * (p.D == 128 && p.mask != nullptr ? 0.85 : 1.0);
    const double us = split_work(p) * (p.D == 128 ? 1.55 : p.D == 64 ? 0.96 : p.D == 32 ? 0.68 : 0.53);
    return SplitShape{32 * waves, slots, 1, false, 20, us, slots == 1 ? us : (p.D == 64 ? 0.65 : 0.59) * us, gain, split_unclassed(p), whole_rows};
}

template <typename T, int D, bool CAUSAL, int MASK>
int launch_dq_split(const KParams& p, hipStream_t stream, bool with_delta) {
    constexpr int NW = 4;
    const dim3 grid = split_grid(p);
    if (MASK == kNoMask && !with_delta) return TRI_ATTN_ESHAPE;  // (dq_splits)
    if constexpr (D == 128 && MASK == kNoMask) {
        if (p.thr8 <= 0) {
            hipLaunchKernelGGL((mfma_dq_phased_kernel<T, D, CAUSAL, false, true, true, true>), grid, dim3(512), 0, stream, p);
            return static_cast<int>(hipGetLastError());
        }
    }
    const auto launch = [&](auto delta) {
        constexpr bool kDelta = decltype(delta)::value;
        if (p.thr8 > 0) hipLaunchKernelGGL((mfma_dq_kernel<T, D, NW, CAUSAL, MASK, true, true, false, kDelta, true>), grid, dim3(64 * NW), 0, stream, p);
        else if constexpr (!(D == 128 && MASK == kNoMask))
            hipLaunchKernelGGL((mfma_dq_kernel<T, D, NW, CAUSAL, MASK, false, true, false, kDelta, true>), grid, dim3(64 * NW), 0, stream, p);
        return static_cast<int>(hipGetLastError());
    };
    if constexpr (MASK == kNoMask) return launch(std::true_type{});
    else if constexpr (D > 64) return launch(std::false_type{});
    else return with_delta ? launch(std::true_type{}) : launch(std::false_type{});
}

template <typename T, int D>
int launch_dq_split_variant(int dtype, const KParams& p, hipStream_t stream, bool with_delta) {
    if (p.causal) return launch_dq_split<T, D, true, kNoMask>(p, stream, with_delta);
    if (p.mask == nullptr) return launch_dq_split<T, D, false, kNoMask>(p, stream, with_delta);
    if (p.mask_dtype == TRI_ATTN_F32) return launch_dq_split<T, D, false, kMaskF32>(p, stream, with_delta);
    if (p.mask_dtype == dtype) return launch_dq_split<T, D, false, kMaskT>(p, stream, with_delta);
    return TRI_ATTN_EDTYPE;
}

// (a mask gradient is written by whole items only; without a mask the parts bring delta along, with one they may up to D = 64)
// Beside dropout at D = 128 a workgroup's start, with one wave per SIMD, costs more than the last round of a launch that fills the GPU
// saves (bf16 S=4352, 11 heads: 209 -> 286 us), except where parts are what makes use of a mask's classes (6 heads, S=5694: 530 -> 281).
bool dq_splits(const KParams& p, bool with_delta) {
    const int64_t items = static_cast<int64_t>(p.B) * p.H * ((p.S + 127) / 128);
    if (p.D == 128 && p.thr8 > 0 && !p.causal && items >= persistent_grid(1 << 20) && !(split_unclassed(p) > 1.0 && p.S > 64 * 64)) return false;
    return p.dmask == nullptr && (p.mask == nullptr ? with_delta : !with_delta || p.D <= 64);
}

template <typename T>
int launch_dq_split_head(int dtype, const KParams& p, hipStream_t stream, bool with_delta) {
    if (p.D == 128) return launch_dq_split_variant<T, 128>(dtype, p, stream, with_delta);
    if (p.D == 64) return launch_dq_split_variant<T, 64>(dtype, p, stream, with_delta);
    if (p.D == 32) return launch_dq_split_variant<T, 32>(dtype, p, stream, with_delta);
    return launch_dq_split_variant<T, 16>(dtype, p, stream, with_delta);
}

}  // namespace

int64_t mfma_dq_workspace(const KParams& p, bool with_delta) {
    KParams plan = p;
    return dq_splits(p, with_delta) ? plan_split(dq_split_shape(p), p.causal != 0, &plan) : 0;
}

int launch_mfma_dq_split(int dtype, KParams p, hipStream_t stream, bool with_delta) {
    const SplitShape shape = dq_split_shape(p);
    if (!dq_splits(p, with_delta) || !take_workspace(plan_split(shape, p.causal != 0, &p), &p)) return TRI_ATTN_ENOFUSE;
    const int rc = dtype == TRI_ATTN_BF16 ? launch_dq_split_head<bf16_t>(dtype, p, stream, with_delta)
                                          : launch_dq_split_head<f16_t>(dtype, p, stream, with_delta);
    return rc ? rc : launch_combine_backward(dtype, p, shape.rows, false, stream);
}

}  // namespace tri
