// Launches of the forward kernel (mfma_fwd.hpp); split ones: mfma_fwd_split.hip.
#include "launch.hpp"
#include "mfma_fwd.hpp"

namespace tri {
namespace {

template <typename T, bool CAUSAL, bool RAGGED, int MASK>
int launch_fwd_three(const KParams& p, hipStream_t stream) {
    const dim3 grid(p.B * p.H * ((p.S + 127) / 128)), block(256);
    if (p.thr8 > 0) hipLaunchKernelGGL((mfma_fwd_kernel<T, 64, 4, CAUSAL, MASK, true, RAGGED, false, true>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((mfma_fwd_kernel<T, 64, 4, CAUSAL, MASK, false, RAGGED, false, true>), grid, block, 0, stream, p);
    return static_cast<int>(hipGetLastError());
}

template <typename T, int D, int NW, bool CAUSAL, int MASK = kNoMask>
int launch_fwd_ragged(const KParams& p, hipStream_t stream) {
    if constexpr (D == 128 && NW == 8 && MASK != kNoMask && MASK != kMaskKeys) {
        // (mask, dropout and boundary handling together need the whole register file: four waves)
        if (p.thr8 > 0) return launch_fwd_ragged<T, D, 4, CAUSAL, MASK>(p, stream);
    }
    const int items = p.B * p.H * ((p.S + 32 * NW - 1) / (32 * NW));
    if constexpr (D == 64 && NW == 4 && (MASK == kNoMask || MASK == kMaskKeys)) {
        if (three_workgroups_per_cu(p)) return launch_fwd_three<T, CAUSAL, true, MASK>(p, stream);
    }
    if constexpr (D == 128 && NW == 4 && MASK == kNoMask) {
        if (p.S % 128 == 0) {  // (causal only with dropout: fwd_runs_four_waves)
            if (p.thr8 > 0) hipLaunchKernelGGL((mfma_fwd_kernel<T, D, NW, CAUSAL, MASK, true>), dim3(items), dim3(64 * NW), 0, stream, p);
            else if constexpr (!CAUSAL) hipLaunchKernelGGL((mfma_fwd_kernel<T, D, NW, CAUSAL, MASK, false>), dim3(items), dim3(64 * NW), 0, stream, p);
            return static_cast<int>(hipGetLastError());
        }
    }
    // (NW == 8: the kernel's kPersistent, one workgroup per CU walks the items)
    const dim3 grid(NW == 8 && MASK == kNoMask ? persistent_grid(items) : items), block(64 * NW);
    if (p.thr8 > 0) {
        if constexpr (!(D == 128 && NW == 8 && MASK != kNoMask))
            hipLaunchKernelGGL((mfma_fwd_kernel<T, D, NW, CAUSAL, MASK, true, true>), grid, block, 0, stream, p);
    } else if constexpr (!(D == 128 && NW == 4 && MASK != kNoMask)) {
        hipLaunchKernelGGL((mfma_fwd_kernel<T, D, NW, CAUSAL, MASK, false, true>), grid, block, 0, stream, p);
    }
    return static_cast<int>(hipGetLastError());
}

template <typename T, int D, int NW, bool CAUSAL, int MASK>
int launch_fwd_dropout(const KParams& p, hipStream_t stream) {
    if constexpr (D == 64 && NW == 4 && (MASK == kNoMask || MASK == kMaskKeys)) {
        if (three_workgroups_per_cu(p)) return launch_fwd_three<T, CAUSAL, false, MASK>(p, stream);
    }
    const int items = p.B * p.H * (p.S / (32 * NW));
    // (the kernel's kPersistent: one workgroup per CU walks the items)
    const dim3 grid(NW == 8 && MASK == kNoMask ? persistent_grid(items) : items), block(64 * NW);
    if (p.thr8 > 0) {
        if constexpr (!(D == 128 && MASK == kMaskKeys)) hipLaunchKernelGGL((mfma_fwd_kernel<T, D, NW, CAUSAL, MASK, true>), grid, block, 0, stream, p);
    } else {
        hipLaunchKernelGGL((mfma_fwd_kernel<T, D, NW, CAUSAL, MASK, false>), grid, block, 0, stream, p);
    }
    return static_cast<int>(hipGetLastError());
}

template <typename T, int D, int NW>
int launch_fwd_variant(int dtype, const KParams& p, hipStream_t stream) {
    if constexpr (!(D == 128 && NW == 4)) {  // (without a mask D = 128 never runs four waves: launch_fwd_waves)
        if (p.causal) return launch_fwd_dropout<T, D, NW, true, kNoMask>(p, stream);
        if (p.mask == nullptr) return launch_fwd_dropout<T, D, NW, false, kNoMask>(p, stream);
    }
    if (p.mask_dtype == TRI_ATTN_F32) return launch_fwd_dropout<T, D, NW, false, kMaskF32>(p, stream);
    if (p.mask_dtype == dtype) return launch_fwd_dropout<T, D, NW, false, kMaskT>(p, stream);
    return TRI_ATTN_EDTYPE;
}

// D = 128 without a mask, S no multiple of 256: 128-row workgroups of four waves where they are all on the chip at once, which
// then is a matter of one workgroup's time. bf16, time of the four waves over that of the eight: with dropout 0.78-0.98
// (causal 0.79-0.97, but 1.03 at S = 384, whose last 256 rows are half empty for the eight), without 0.92-0.98 at S = 129 .. 500
// and from 640 on 1.00-1.12 with boundary handling, 0.88-0.94 at multiples of 128, which need none; causal 0.86-1.00 up to
// S = 500, 1.02-1.19 beyond and at multiples of 128; S <= 128 without dropout 1.00-1.05.
bool fwd_runs_four_waves(const KParams& p) {
    if (!four_waves_fit_one_round(p)) return false;
    const bool whole = p.S % 128 == 0;
    if (p.thr8 > 0) return !p.causal || !whole || p.S >= 640;
    return p.S > 128 && (whole ? !p.causal : p.S <= 512);
}

template <typename T, int D>
int launch_fwd_waves(int dtype, const KParams& p, hipStream_t stream) {
    // 8 waves (256 query rows) at D = 128 when the sequence allows it: two waves per SIMD out of phase. Up to D = 64 four waves everywhere,
    // whose workgroups share a CU, so that starts and ends pass behind one another's tiles and less of the chip is idle in the last round. Time of
    // the four over that of the eight at multiples of 256: D = 32 0.78; D = 64 without a mask 0.82-0.86 at half as many items of 256 rows as CUs,
    // 0.93-0.99 at as many, 0.99-1.03 at twice as many (causal 0.77-0.86, 0.88-0.91 and 0.95-1.00), more than that: three_workgroups_per_cu; with
    // dropout 0.70-0.99; beside 16-bit masks 0.90-1.01; beside fp32 ones, whose ring of three lets two workgroups onto a CU, 0.88-0.96, length
    // masks 0.84-1.00 (dense ones in whole rounds of S = 2048 1.04-1.06).
    if constexpr (D == 128) {
        if (mask_is_key_bits(p))
            return p.S % 256 == 0 ? launch_fwd_dropout<T, D, 8, false, kMaskKeys>(p, stream) : launch_fwd_ragged<T, D, 8, false, kMaskKeys>(p, stream);
        if (p.S % 256 == 0) return launch_fwd_variant<T, D, 8>(dtype, p, stream);
    }
    // Without a mask D = 128 keeps the 8 waves at every other length too, with boundary handling: its ring leaves room for
    // one workgroup per CU, so that four waves are one per SIMD. bf16 causal, heads x S: 768 x 130 0.057 -> 0.034 ms,
    // 768 x 450 0.168 -> 0.110, 136 x 1531 0.170 -> 0.109, 32 x 3000 0.141 -> 0.084; 768 x 65 0.026 -> 0.022. Launches
    // that leave CUs idle either way are another matter (above).
    if constexpr (D == 128) {
        if (p.mask == nullptr) {
            if (fwd_runs_four_waves(p)) return p.causal ? launch_fwd_ragged<T, D, 4, true>(p, stream) : launch_fwd_ragged<T, D, 4, false>(p, stream);
            return p.causal ? launch_fwd_ragged<T, D, 8, true>(p, stream) : launch_fwd_ragged<T, D, 8, false>(p, stream);
        }
    }
    if constexpr (D < 128) {
        if (mask_is_key_bits(p))
            return p.S % 128 == 0 ? launch_fwd_dropout<T, D, 4, false, kMaskKeys>(p, stream) : launch_fwd_ragged<T, D, 4, false, kMaskKeys>(p, stream);
    }
    if (p.S % 128 == 0) return launch_fwd_variant<T, D, 4>(dtype, p, stream);
    if (p.mask != nullptr) {
        // A padded mask: at D = 64 two workgroups of 4 waves share a CU's LDS with the mask's staging regions (beside an fp32 mask one of 8
        // waves was 1-19 % slower)
        if (p.mask_dtype == TRI_ATTN_F32) return launch_fwd_ragged<T, D, D == 128 ? 8 : 4, false, kMaskF32>(p, stream);
        if (p.mask_dtype == dtype) return launch_fwd_ragged<T, D, D == 128 ? 8 : 4, false, kMaskT>(p, stream);
        return TRI_ATTN_EDTYPE;
    }
    // any other length (no mask: mfma_supported) at D <= 64: 128-row workgroups with boundary handling, two of which share
    // a CU (256-row ones measured 5-30 % slower at D = 64, S = 65 .. 6001)
    if constexpr (D < 128) return p.causal ? launch_fwd_ragged<T, D, 4, true>(p, stream) : launch_fwd_ragged<T, D, 4, false>(p, stream);
    return TRI_ATTN_ESHAPE;
}

template <typename T>
int launch_fwd_head(int dtype, const KParams& p, hipStream_t stream) {
    if (p.D == 128) return launch_fwd_waves<T, 128>(dtype, p, stream);
    if (p.D == 64) return launch_fwd_waves<T, 64>(dtype, p, stream);
    if (p.D == 32) return launch_fwd_waves<T, 32>(dtype, p, stream);
    return launch_fwd_waves<T, 16>(dtype, p, stream);
}

}  // namespace

int launch_mfma_fwd(int dtype, const KParams& p, hipStream_t stream) {
    if (p.workspace != nullptr && mfma_fwd_workspace(p) > 0) {
        const int rc = launch_mfma_fwd_split(dtype, p, stream);
        if (rc != TRI_ATTN_ENOFUSE) return rc;  // (a workspace too small for it)
    }
    return dtype == TRI_ATTN_BF16 ? launch_fwd_head<bf16_t>(dtype, p, stream) : launch_fwd_head<f16_t>(dtype, p, stream);
}

}  // namespace tri
