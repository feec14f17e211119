// Launches of the dQ kernels (mfma_dq.hpp); split ones: mfma_dq_split.hip.
#include "launch.hpp"
#include "mfma_dq.hpp"

namespace tri {
namespace {

// ---------------------------------------------------------------------------------- launch
template <typename T, bool CAUSAL, bool RAGGED, int MASK>
int launch_dq_three(const KParams& p, hipStream_t stream) {  // (with delta)
    const dim3 grid(p.B * p.H * ((p.S + 127) / 128)), block(256);
    if (p.thr8 > 0) hipLaunchKernelGGL((mfma_dq_kernel<T, 64, 4, CAUSAL, MASK, true, RAGGED, false, true, false, true>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((mfma_dq_kernel<T, 64, 4, CAUSAL, MASK, false, RAGGED, false, true, false, true>), grid, block, 0, stream, p);
    return static_cast<int>(hipGetLastError());
}

template <typename T, int D, int NW, bool CAUSAL, int MASK>
int launch_dq_waves(const KParams& p, hipStream_t stream, bool with_delta = false) {
    if constexpr (D == 64 && NW == 4 && (MASK == kNoMask || MASK == kMaskKeys)) {
        if (with_delta && three_workgroups_per_cu(p)) return launch_dq_three<T, CAUSAL, false, MASK>(p, stream);
    }
    const dim3 grid(p.B * p.H * (p.S / (32 * NW))), block(64 * NW);
    if constexpr (NW == 8 && D == 128 && MASK != kNoMask) {
        // with a mask gradient or dropout on top of a mask the 8-wave kernel does not fit its registers at D = 128 and
        // would spill to scratch memory (whose reloads are vector-memory loads that drain the tile prefetch): those
        // problems take 128-row workgroups, which fit
        if (p.dmask != nullptr || p.thr8 > 0) return launch_dq_waves<T, D, 4, CAUSAL, MASK>(p, stream, with_delta);
        hipLaunchKernelGGL((mfma_dq_kernel<T, D, NW, CAUSAL, MASK, false>), grid, block, 0, stream, p);
    } else {
        if constexpr (MASK == kMaskF32 || MASK == kMaskT) {
            if (p.dmask != nullptr) {
                if (p.thr8 > 0) hipLaunchKernelGGL((mfma_dq_kernel<T, D, NW, CAUSAL, MASK, true, false, true>), grid, block, 0, stream, p);
                else hipLaunchKernelGGL((mfma_dq_kernel<T, D, NW, CAUSAL, MASK, false, false, true>), grid, block, 0, stream, p);
                return static_cast<int>(hipGetLastError());
            }
        }
        if constexpr (MASK == kNoMask && D == 128 && NW == 8) {  // (without dropout: the phased kernel)
            if (with_delta) hipLaunchKernelGGL((mfma_dq_kernel<T, D, NW, CAUSAL, MASK, true, false, false, true>), grid, block, 0, stream, p);
            else hipLaunchKernelGGL((mfma_dq_kernel<T, D, NW, CAUSAL, MASK, true>), grid, block, 0, stream, p);
        } else {
            if constexpr (MASK == kNoMask || D <= 64) {
                if (with_delta) {
                    if (p.thr8 > 0) hipLaunchKernelGGL((mfma_dq_kernel<T, D, NW, CAUSAL, MASK, true, false, false, true>), grid, block, 0, stream, p);
                    else hipLaunchKernelGGL((mfma_dq_kernel<T, D, NW, CAUSAL, MASK, false, false, false, true>), grid, block, 0, stream, p);
                    return static_cast<int>(hipGetLastError());
                }
            }
            if (p.thr8 > 0) hipLaunchKernelGGL((mfma_dq_kernel<T, D, NW, CAUSAL, MASK, true>), grid, block, 0, stream, p);
            else hipLaunchKernelGGL((mfma_dq_kernel<T, D, NW, CAUSAL, MASK, false>), grid, block, 0, stream, p);
        }
    }
    return static_cast<int>(hipGetLastError());
}

// whether the phased dQ kernel serves this problem (no mask, 256-row workgroups, D >= 64; with dropout at D = 128 it
// fits its registers only under the causal mask, without boundary handling and with a fragment ring of 4). At D = 32 the
// kernel above needs 112 registers, and four of its workgroups that share a CU measured 27 % faster than the phased pairs.
// At D = 64 with S a multiple of 256 only launches that fill the chip with 256-row workgroups, and not causal ones: time of
// unphased workgroups of four waves, two or three to a CU, over that of the phased one, at half as many items of 256 rows as CUs 0.80-0.90, at
// as many 1.03-1.09, beyond 0.90-1.06 (causal 0.78-0.84, 0.83-0.95 and 0.81-0.98); with dropout 0.69-0.98.
// Lengths that are no multiple of 256: at D = 128 the phased kernel with boundary handling (against 4 unphased waves, bf16
// causal, heads x S: 768 x 130 0.071 -> 0.044 ms, 768 x 450 0.216 -> 0.152, 136 x 1531 0.216 -> 0.145; 768 x 65 equal); at
// D = 64 two 128-row workgroups share a CU, which is 5-30 % faster than the phased kernel up to S = 3000.
template <int D, int MASK>
bool dq_is_phased(const KParams& p) {
    if (MASK == kMaskKeys) return D == 128 && p.thr8 <= 0;
    if (MASK != kNoMask) return false;
    if (D == 64) {
        const int64_t items = static_cast<int64_t>(p.B) * p.H * (p.S / 256), cus = persistent_grid(1 << 20);
        return p.S % 256 == 0 && p.thr8 <= 0 && !p.causal && 2 * items > cus;
    }
    return D == 128 && (p.thr8 <= 0 || (p.causal && p.S % 256 == 0));
}

// D = 128 without a mask: workgroups of four waves, two to a CU, instead of one of eight, whose pairs of waves are phased where their
// registers allow it. Four waves gain where 128 rows waste less than 256 (rows that do not exist, keys above the diagonal), where starts and
// ends are a large part of the time, and where 256-row items leave CUs idle in the last round; per tile the eight phased waves need less. Time of
// four waves over that of eight, bf16, 0.5 to 24 workgroups per CU (a half round: of workgroups of four waves; a round of the eight is two):
//   S <= 128                                  0.58-0.95
//   up to a workgroup per CU                  0.72-0.98 (causal 384 rows, whose second item is light, 0.92-1.01)
//   causal with dropout, up to 1024 rows      0.67-1.03; longer: up to 8/3 per CU 0.81-0.91, 4 to 16 up to 4096 rows 0.86-1.01; else 0.94-1.11
//   causal, up to 800 rows, up to 16 per CU   0.68-1.02, but one to two per CU at 257 to 384 rows 0.95-1.08, three to four
//                                             at more without a half-empty last item 0.96-1.09; beyond 16 1.01-1.12, out of the caches
//   causal, longer, up to 3/2 per CU          0.90-1.01; else 0.96-1.17
//   not causal with dropout                   fewer half rounds 0.58-0.98; up to 800 rows from two per CU on 0.62-0.97, up to 2048 from four on
//                                             0.89-1.00; else 0.95-1.09
//   not causal, up to 512 rows, above two per CU  0.69-0.97; one to two 1.00-1.07
//   not causal, up to 800 rows, half-empty last item, eight waves in more than a round  0.67-1.03
//   not causal, longer, three quarters of the half rounds  0.92-1.02; else 0.96-1.20
bool dq_runs_four_waves(const KParams& p) {
    const int64_t cus = persistent_grid(1 << 20), heads = static_cast<int64_t>(p.B) * p.H;
    const int64_t items = heads * ((p.S + 127) / 128), items256 = heads * ((p.S + 255) / 256);
    const int64_t halves = (items + cus - 1) / cus, rounds256 = (items256 + cus - 1) / cus;
    const bool half_empty = (p.S - 1) % 256 < 128;
    // (long rows with boundary handling, without dropout: 1.02-1.05 but where the eight need half as many half rounds more, 0.81)
    if (p.S > 1024 && p.S % 128 != 0 && p.thr8 <= 0) return !p.causal && items > cus && 3 * halves <= 4 * rounds256;
    if (p.S <= 128 || items <= cus) return true;
    if (p.causal && p.thr8 > 0) return p.S <= 1024 || 3 * items <= 8 * cus || (p.S <= 4096 && items > 4 * cus && items <= 16 * cus);
    if (p.causal) {
        if (p.S > 800) return 2 * items <= 3 * cus;
        if (p.S > 256 && items > (p.S <= 384 ? 1 : 3) * cus && items <= (p.S <= 384 ? 2 : 4) * cus) return p.S > 384 && half_empty;
        return items <= 16 * cus;
    }
    if (p.thr8 > 0) return halves < 2 * rounds256 || (p.S <= 800 && items > 2 * cus) || (p.S <= 2048 && items > 4 * cus);
    if (p.S <= 512) return items > 2 * cus;
    if (p.S <= 800 && half_empty) return items256 > cus;
    return 4 * halves <= 6 * rounds256;
}

// ... and whether those four run phases (mfma_dq_phased_kernel, whose rows come through LDS) or not (kPair): a few tiles are over before that
// pays. Time of the phased over the unphased ones: S <= 128 0.83-1.10; up to a workgroup per CU 0.84-1.06; else up to 384 rows 0.93-1.13, with
// dropout up to 800 rows 0.95-1.13, beyond 0.91-1.05.
bool dq_four_waves_phased(const KParams& p) {
    if (p.S <= 128) return false;
    const int64_t items = static_cast<int64_t>(p.B) * p.H * ((p.S + 127) / 128);
    return p.S > (p.thr8 > 0 ? 800 : 384) || items <= persistent_grid(1 << 20);
}

// any length (no mask, or a padded one), with boundary handling
template <typename T, int D, int NW, bool CAUSAL, int MASK = kNoMask>
int launch_dq_ragged(const KParams& p, hipStream_t stream, bool with_delta) {
    if constexpr (D == 64 && NW == 4 && (MASK == kNoMask || MASK == kMaskKeys)) {
        if (with_delta && three_workgroups_per_cu(p)) return launch_dq_three<T, CAUSAL, true, MASK>(p, stream);
    }
    const dim3 grid(p.B * p.H * ((p.S + 32 * NW - 1) / (32 * NW))), block(64 * NW);
    if constexpr (MASK != kNoMask) {
        if constexpr (D <= 64) {
            if (with_delta) {
                if (p.thr8 > 0) hipLaunchKernelGGL((mfma_dq_kernel<T, D, NW, CAUSAL, MASK, true, true, false, true>), grid, block, 0, stream, p);
                else hipLaunchKernelGGL((mfma_dq_kernel<T, D, NW, CAUSAL, MASK, false, true, false, true>), grid, block, 0, stream, p);
                return static_cast<int>(hipGetLastError());
            }
        }
        if (p.thr8 > 0) hipLaunchKernelGGL((mfma_dq_kernel<T, D, NW, CAUSAL, MASK, true, true>), grid, block, 0, stream, p);
        else hipLaunchKernelGGL((mfma_dq_kernel<T, D, NW, CAUSAL, MASK, false, true>), grid, block, 0, stream, p);
        return static_cast<int>(hipGetLastError());
    }
    constexpr bool kDropoutOnly = D == 128 && NW == 8;  // (eight waves without dropout: the phased kernel)
    if (kDropoutOnly || p.thr8 > 0) {
        if (with_delta) hipLaunchKernelGGL((mfma_dq_kernel<T, D, NW, CAUSAL, kNoMask, true, true, false, true>), grid, block, 0, stream, p);
        else hipLaunchKernelGGL((mfma_dq_kernel<T, D, NW, CAUSAL, kNoMask, true, true>), grid, block, 0, stream, p);
    } else if constexpr (!kDropoutOnly) {
        if (with_delta) hipLaunchKernelGGL((mfma_dq_kernel<T, D, NW, CAUSAL, kNoMask, false, true, false, true>), grid, block, 0, stream, p);
        else hipLaunchKernelGGL((mfma_dq_kernel<T, D, NW, CAUSAL, kNoMask, false, true>), grid, block, 0, stream, p);
    }
    return static_cast<int>(hipGetLastError());
}

template <typename T, int D, bool CAUSAL, bool RAGGED, int MASK, int NW = 8>
int launch_dq_phased(const KParams& p, hipStream_t stream, bool with_delta) {
    const dim3 grid(p.B * p.H * ((p.S + 32 * NW - 1) / (32 * NW))), block(64 * NW);
    constexpr bool kKeys = MASK == kMaskKeys;
    if constexpr (NW == 4 || (D == 128 && CAUSAL && !RAGGED)) {
        if (p.thr8 > 0) {
            if (with_delta) hipLaunchKernelGGL((mfma_dq_phased_kernel<T, D, CAUSAL, true, true, RAGGED, false, kKeys, NW>), grid, block, 0, stream, p);
            else hipLaunchKernelGGL((mfma_dq_phased_kernel<T, D, CAUSAL, true, false, RAGGED, false, kKeys, NW>), grid, block, 0, stream, p);
            return static_cast<int>(hipGetLastError());
        }
    }
    if (with_delta) hipLaunchKernelGGL((mfma_dq_phased_kernel<T, D, CAUSAL, false, true, RAGGED, false, kKeys, NW>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((mfma_dq_phased_kernel<T, D, CAUSAL, false, false, RAGGED, false, kKeys, NW>), grid, block, 0, stream, p);
    return static_cast<int>(hipGetLastError());
}

template <typename T, int D, bool CAUSAL, int MASK>
int launch_dq_dropout(const KParams& p, hipStream_t stream, bool with_delta) {
    if constexpr (D == 128 && MASK == kNoMask) {
        if (dq_runs_four_waves(p)) {
            if (dq_four_waves_phased(p))
                return p.S % 128 == 0 ? launch_dq_phased<T, D, CAUSAL, false, MASK, 4>(p, stream, with_delta) : launch_dq_phased<T, D, CAUSAL, true, MASK, 4>(p, stream, with_delta);
            return p.S % 128 == 0 ? launch_dq_waves<T, D, 4, CAUSAL, MASK>(p, stream, with_delta) : launch_dq_ragged<T, D, 4, CAUSAL>(p, stream, with_delta);
        }
    }
    if constexpr (D == 128 && MASK == kMaskKeys) {
        // Four phased waves, with dropout always (training step on a padded batch against the kernels that read the mask's values and had a CU
        // for four waves: 0.70-0.89, one item per CU 0.83-1.01); without it as without a mask (0.57-1.02), but not at 385 to 512 rows (1.05-1.07)
        if (p.thr8 > 0 || (dq_runs_four_waves(p) && (p.S <= 384 || p.S > 512)))
            return p.S % 128 == 0 ? launch_dq_phased<T, D, CAUSAL, false, MASK, 4>(p, stream, with_delta) : launch_dq_phased<T, D, CAUSAL, true, MASK, 4>(p, stream, with_delta);
    }
    if constexpr ((MASK == kNoMask || MASK == kMaskKeys) && (D == 128 || (D == 64 && !CAUSAL && MASK == kNoMask))) {
        if (dq_is_phased<D, MASK>(p)) {
            if constexpr (D == 128) {
                if (p.S % 256 != 0) return launch_dq_phased<T, D, CAUSAL, true, MASK>(p, stream, with_delta);
            }
            return launch_dq_phased<T, D, CAUSAL, false, MASK>(p, stream, with_delta);
        }
    }
    if constexpr (D == 128 && MASK == kMaskKeys) return TRI_ATTN_ESHAPE;  // (never: the two above take every such problem)
    else {
    if (with_delta && MASK != kNoMask && (D > 64 || p.dmask != nullptr)) return TRI_ATTN_ESHAPE;  // (callers ask mfma_dq_fuses_delta first)
    // D = 128: 8 waves (256 query rows) when the sequence allows it, else 4 waves (128 rows). Up to D = 64 always 4: several such workgroups
    // share a CU (time over that of 8 waves at multiples of 256: D = 32 0.92-1.00; D = 64 beside 16-bit masks 0.90-1.02, beside fp32 ones with a
    // ring of three 0.78-1.05, in most cases 0.95-0.98)
    if constexpr (D == 128 && !CAUSAL) {  // (causal: the phased kernel)
        if (p.S % 256 == 0) return launch_dq_waves<T, D, 8, CAUSAL, MASK>(p, stream, with_delta);
    }
    if constexpr (D == 128 && MASK == kNoMask) return launch_dq_ragged<T, D, 8, CAUSAL>(p, stream, with_delta);  // (dropout)
    if (p.S % 128 == 0) return launch_dq_waves<T, D, 4, CAUSAL, MASK>(p, stream, with_delta);
    if constexpr (MASK == kNoMask && D < 128) return launch_dq_ragged<T, D, 4, CAUSAL>(p, stream, with_delta);  // any other length
    // a padded mask: four waves; at D = 128 with the whole register file (in 256 registers the kernel spills)
    if constexpr (MASK != kNoMask) return launch_dq_ragged<T, D, 4, CAUSAL, MASK>(p, stream, with_delta);
    return TRI_ATTN_ESHAPE;
    }
}

template <typename T, int D>
int launch_dq_variant(int dtype, const KParams& p, hipStream_t stream, bool with_delta) {
    if (p.causal) return launch_dq_dropout<T, D, true, kNoMask>(p, stream, with_delta);
    if (p.mask == nullptr) return launch_dq_dropout<T, D, false, kNoMask>(p, stream, with_delta);
    if (mask_is_key_bits(p)) return launch_dq_dropout<T, D, false, kMaskKeys>(p, stream, with_delta);
    if (p.mask_dtype == TRI_ATTN_F32) return launch_dq_dropout<T, D, false, kMaskF32>(p, stream, with_delta);
    if (p.mask_dtype == dtype) return launch_dq_dropout<T, D, false, kMaskT>(p, stream, with_delta);
    return TRI_ATTN_EDTYPE;
}

template <typename T>
int launch_dq_head(int dtype, const KParams& p, hipStream_t stream, bool with_delta) {
    if (p.D == 128) return launch_dq_variant<T, 128>(dtype, p, stream, with_delta);
    if (p.D == 64) return launch_dq_variant<T, 64>(dtype, p, stream, with_delta);
    if (p.D == 32) return launch_dq_variant<T, 32>(dtype, p, stream, with_delta);
    return launch_dq_variant<T, 16>(dtype, p, stream, with_delta);
}

}  // namespace

int launch_mfma_dq(int dtype, const KParams& p, hipStream_t stream, bool with_delta) {
    if (p.workspace != nullptr && mfma_dq_workspace(p, with_delta) > 0) {
        const int rc = launch_mfma_dq_split(dtype, p, stream, with_delta);
        if (rc != TRI_ATTN_ENOFUSE) return rc;  // (a workspace too small for it)
    }
    return dtype == TRI_ATTN_BF16 ? launch_dq_head<bf16_t>(dtype, p, stream, with_delta)
                                  : launch_dq_head<f16_t>(dtype, p, stream, with_delta);
}

}  // namespace tri
