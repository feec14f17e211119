// Launches of the dK/dV kernels (mfma_dkdv.hpp); split ones: mfma_dkdv_split.hip.
#include "launch.hpp"
#include "mfma_dkdv.hpp"

namespace tri {
namespace {

template <typename T, int D, int NW, bool CAUSAL, int MASK>
int launch_dkdv_waves(const KParams& p, hipStream_t stream) {
    const dim3 grid(p.B * p.H * (p.S / (32 * NW))), block(64 * NW);
    if (p.thr8 > 0) hipLaunchKernelGGL((mfma_dkdv_wide_kernel<T, D, NW, CAUSAL, MASK, true>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((mfma_dkdv_wide_kernel<T, D, NW, CAUSAL, MASK, false>), grid, block, 0, stream, p);
    return static_cast<int>(hipGetLastError());
}

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
                if (p.thr8 > 0) hipLaunchKernelGGL((mfma_dkdv_wide_kernel<T, D, 4, CAUSAL, kNoMask, true, true>), grid, block, 0, stream, p);
                else hipLaunchKernelGGL((mfma_dkdv_wide_kernel<T, D, 4, CAUSAL, kNoMask, false, true>), grid, block, 0, stream, p);
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
        // a padded mask: at D = 64 beside an fp32 one's regions one workgroup of 8 waves per CU; beside a 16-bit one's the LDS holds two
        // of 4 with a ring of three, whose 128 keys end closer to the sequence's end and wait at barriers of their own (fp16 B=16 H=12
        // S=777 with key padding, forward and backward, 248 -> 218 us). 4 waves with the whole register file at D = 128
        if constexpr (MASK != kNoMask) {
            // (dropout beside mask and boundary handling does not fit 256 registers: four waves)
            constexpr int NW = D == 64 && MASK == kMaskF32 ? 8 : 4;
            const int nw = p.thr8 > 0 ? 4 : NW;
            const dim3 grid(p.B * p.H * ((p.S + 32 * nw - 1) / (32 * nw))), block(64 * nw);
            if (p.thr8 > 0) hipLaunchKernelGGL((mfma_dkdv_wide_kernel<T, D, 4, false, MASK, true, true>), grid, block, 0, stream, p);
            else hipLaunchKernelGGL((mfma_dkdv_wide_kernel<T, D, NW, false, MASK, false, true>), grid, block, 0, stream, p);
            return static_cast<int>(hipGetLastError());
        }
        return TRI_ATTN_ESHAPE;
    }
    if constexpr (D <= 64) {
        // the two-waves-per-SIMD kernel fits its registers: 8 waves (256 keys) when the sequence
        // allows it, else 4 waves (128 keys)
        if constexpr (D > 16) {
            // (beside a 16-bit mask two workgroups of 4 fit a CU, as above, and are faster wherever those of 8 leave CUs idle in
            // their last round: bf16 training steps at D = 64, heads x S, 96 x 512 93.6 -> 91.9 us, 96 x 768 180 -> 167; in whole
            // rounds 64 x 1024 127.5 either way against 128.3. 192 x 640, one of 4 before, 199 -> 161)
            const int64_t items = static_cast<int64_t>(p.B) * p.H * (p.S / 256);
            const bool pairs = D == 64 && MASK == kMaskT && p.thr8 <= 0 && items % persistent_grid(1 << 20) != 0;
            if (p.S % 256 == 0 && !pairs) return launch_dkdv_waves<T, D, 8, CAUSAL, MASK>(p, stream);
        }
        return launch_dkdv_waves<T, D, 4, CAUSAL, MASK>(p, stream);
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
