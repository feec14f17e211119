// Launches of the dK/dV kernels (mfma_dkdv.hpp); split ones: mfma_dkdv_split.hip.
#include "launch.hpp"
#include "mfma_dkdv.hpp"

namespace tri {
namespace {

// D = 128 without a mask, S no multiple of 128: 32 keys per wave instead of the phased pairs where the rows are one tile, which
// the pairs pad to four blocks: time over theirs 0.75-0.91, with dropout 0.68-0.81 (S = 65: 1.01-1.19).
bool dkdv_runs_four_waves(const KParams& p) { return p.S <= 64; }

template <typename T, int D, bool CAUSAL, int MASK>
int launch_dkdv_dropout(const KParams& p, hipStream_t stream) {
    if (p.S % 128 != 0) {
        // any length (no mask): 128-key workgroups with boundary handling
        if constexpr (MASK == kNoMask) {
            if (D < 128 || dkdv_runs_four_waves(p)) {
                const dim3 grid(p.B * p.H * ((p.S + 127) / 128)), block(256);
                if (p.thr8 > 0) hipLaunchKernelGGL((mfma_dkdv_wide_kernel<T, D, CAUSAL, kNoMask, true, true>), grid, block, 0, stream, p);
                else hipLaunchKernelGGL((mfma_dkdv_wide_kernel<T, D, CAUSAL, kNoMask, false, true>), grid, block, 0, stream, p);
                return static_cast<int>(hipGetLastError());
            }
            if constexpr (D == 128) {
                const dim3 grid(p.B * p.H * ((p.S + 127) / 128)), block(512);
                if (p.thr8 > 0) hipLaunchKernelGGL((mfma_dkdv_phased_kernel<T, D, CAUSAL, true, kNoMask, true>), grid, block, 0, stream, p);
                else hipLaunchKernelGGL((mfma_dkdv_phased_kernel<T, D, CAUSAL, false, kNoMask, true>), grid, block, 0, stream, p);
                return static_cast<int>(hipGetLastError());
            }
        }
        if constexpr (MASK != kNoMask && D == 128) {
            // A key-padding mask: as below. Only one of zeros and -inf: this kernel works with S - lse / c, and the lse of a row
            // whose keys all carry a large finite value would take the score's digits (or, in fp16, not fit at all).
            if (p.ms[2] == 0 && p.mask_binary) {
                const dim3 grid(p.B * p.H * ((p.S + 127) / 128)), block(512);
                if (p.thr8 > 0) hipLaunchKernelGGL((mfma_dkdv_phased_kernel<T, D, false, true, MASK, true>), grid, block, 0, stream, p);
                else hipLaunchKernelGGL((mfma_dkdv_phased_kernel<T, D, false, false, MASK, true>), grid, block, 0, stream, p);
                return static_cast<int>(hipGetLastError());
            }
        }
        // a padded mask: 4 waves, of which two workgroups share a CU at D = 64 (time over that of one of 8 waves: beside a 16-bit mask 0.88 of
        // a training step, beside an fp32 one 0.76-0.98), but for dropout, beside which it takes the whole register file, as at D = 128
        if constexpr (MASK != kNoMask) {
            const dim3 grid(p.B * p.H * ((p.S + 127) / 128)), block(256);
            if (p.thr8 > 0) hipLaunchKernelGGL((mfma_dkdv_wide_kernel<T, D, false, MASK, true, true>), grid, block, 0, stream, p);
            else hipLaunchKernelGGL((mfma_dkdv_wide_kernel<T, D, false, MASK, false, true>), grid, block, 0, stream, p);
            return static_cast<int>(hipGetLastError());
        }
        return TRI_ATTN_ESHAPE;
    }
    if constexpr (D <= 64) {
        // 128 keys to a workgroup of four waves; two and more share a CU. One of eight waves, which every wave of a SIMD's pair waits for at
        // its barriers and whose 256 keys leave more CUs idle in the last round, takes (time of the four over its): without a mask 0.74-0.77 at
        // half as many items of 256 keys as CUs, 0.82-1.07 at as many, 0.94-1.03 beyond; with dropout 0.68-1.00; beside masks 0.88-0.98, few items 0.73;
        // D = 32 0.85-0.95.
        const dim3 grid(p.B * p.H * (p.S / 128)), block(256);
        if (p.thr8 > 0) hipLaunchKernelGGL((mfma_dkdv_wide_kernel<T, D, CAUSAL, MASK, true>), grid, block, 0, stream, p);
        else hipLaunchKernelGGL((mfma_dkdv_wide_kernel<T, D, CAUSAL, MASK, false>), grid, block, 0, stream, p);
        return static_cast<int>(hipGetLastError());
    } else {
        // D = 128: K, V and both gradient accumulators of a 32-key block take 192 registers, too many
        // for two waves per SIMD, so two waves are paired on each key block of a 128-key workgroup
        const dim3 grid(p.B * p.H * (p.S / kBM)), block(512);
        if constexpr (MASK == kNoMask) {
            if (p.thr8 <= 0) hipLaunchKernelGGL((mfma_dkdv_phased_kernel<T, D, CAUSAL, false>), grid, block, 0, stream, p);
            else hipLaunchKernelGGL((mfma_dkdv_phased_kernel<T, D, CAUSAL, true>), grid, block, 0, stream, p);
            return static_cast<int>(hipGetLastError());
        }
        if constexpr (MASK != kNoMask && !CAUSAL) {
            // a mask that is the same for every query row (a key-padding mask) is one value per key: the phased kernel
            if (p.ms[2] == 0) {
                if (p.thr8 <= 0) hipLaunchKernelGGL((mfma_dkdv_phased_kernel<T, D, false, false, MASK>), grid, block, 0, stream, p);
                else hipLaunchKernelGGL((mfma_dkdv_phased_kernel<T, D, false, true, MASK>), grid, block, 0, stream, p);
                return static_cast<int>(hipGetLastError());
            }
        }
        if (p.thr8 > 0) hipLaunchKernelGGL((mfma_dkdv_pair_kernel<T, D, CAUSAL, MASK, true>), grid, block, 0, stream, p);
        else hipLaunchKernelGGL((mfma_dkdv_pair_kernel<T, D, CAUSAL, MASK, false>), grid, block, 0, stream, p);
        return static_cast<int>(hipGetLastError());
    }
}

template <typename T, int D>
int launch_dkdv_variant(int dtype, const KParams& p, hipStream_t stream) {
    if (p.causal) return launch_dkdv_dropout<T, D, true, kNoMask>(p, stream);
    if (p.mask == nullptr) return launch_dkdv_dropout<T, D, false, kNoMask>(p, stream);
    if constexpr (D < 128) {
        if (mask_is_key_bits(p)) return launch_dkdv_dropout<T, D, false, kMaskKeys>(p, stream);
    }
    if (p.mask_dtype == TRI_ATTN_F32) return launch_dkdv_dropout<T, D, false, kMaskF32>(p, stream);
    if (p.mask_dtype == dtype) return launch_dkdv_dropout<T, D, false, kMaskT>(p, stream);
    return TRI_ATTN_EDTYPE;
}

template <typename T>
int launch_dkdv_head(int dtype, const KParams& p, hipStream_t stream) {
    if (p.D == 128) return launch_dkdv_variant<T, 128>(dtype, p, stream);
    if (p.D == 64) return launch_dkdv_variant<T, 64>(dtype, p, stream);
    if (p.D == 32) return launch_dkdv_variant<T, 32>(dtype, p, stream);
    return launch_dkdv_variant<T, 16>(dtype, p, stream);
}

}  // namespace

int launch_mfma_dkdv(int dtype, const KParams& p, hipStream_t stream) {
    if (p.workspace != nullptr && mfma_dkdv_workspace(p) > 0) {
        const int rc = launch_mfma_dkdv_split(dtype, p, stream);
        if (rc != TRI_ATTN_ENOFUSE) return rc;  // (a workspace too small for it)
    }
    return dtype == TRI_ATTN_BF16 ? launch_dkdv_head<bf16_t>(dtype, p, stream)
                                  : launch_dkdv_head<f16_t>(dtype, p, stream);
}

}  // namespace tri
