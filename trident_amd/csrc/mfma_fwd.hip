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
    if constexpr (D == 128 && NW == 4 && (MASK == kNoMask || MASK == kMaskKeys)) {
        if (p.S % 128 == 0) {
            if (p.thr8 > 0) hipLaunchKernelGGL((mfma_fwd_kernel<T, D, NW, CAUSAL, MASK, true>), dim3(items), dim3(64 * NW), 0, stream, p);
            else hipLaunchKernelGGL((mfma_fwd_kernel<T, D, NW, CAUSAL, MASK, false>), dim3(items), dim3(64 * NW), 0, stream, p);
            return static_cast<int>(hipGetLastError());
        }
    }
    // (NW == 8: the kernel's kPersistent, one workgroup per CU walks the items)
    const dim3 grid(NW == 8 && MASK == kNoMask ? persistent_grid(items) : items), block(64 * NW);
    if (p.thr8 > 0) {
        if constexpr (!(D == 128 && NW == 8 && MASK != kNoMask))
            hipLaunchKernelGGL((mfma_fwd_kernel<T, D, NW, CAUSAL, MASK, true, true>), grid, block, 0, stream, p);
    } else if constexpr (!(D == 128 && NW == 4 && MASK != kNoMask && MASK != kMaskKeys)) {
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
    if constexpr (!(D == 128 && NW == 4)) {  // (without a mask: launch_fwd_ragged)
        if (p.causal) return launch_fwd_dropout<T, D, NW, true, kNoMask>(p, stream);
        if (p.mask == nullptr) return launch_fwd_dropout<T, D, NW, false, kNoMask>(p, stream);
    }
    if (p.mask_dtype == TRI_ATTN_F32) return launch_fwd_dropout<T, D, NW, false, kMaskF32>(p, stream);
    if (p.mask_dtype == dtype) return launch_fwd_dropout<T, D, NW, false, kMaskT>(p, stream);
    return TRI_ATTN_EDTYPE;
}

// D = 128 without a mask: workgroups of four waves (kPair), two to a CU, instead of one of eight whose waves run in opposite phases. Per tile
// the eight need up to 9 % less time (not causal, without dropout); four waves gain where 128 rows waste less than 256 (rows that do not exist, keys
// above the diagonal), where starts and ends are a large part of the time, and where 256-row items leave CUs idle in the last round. Beside dropout
// two independent workgroups overlap the generator with the other one's MFMAs better than the phases do. Time of four waves over that of eight, bf16,
// 0.4 to 24 workgroups per CU (a half round: of workgroups of four waves; a round of the eight is two):
//   S <= 128                                      0.56-0.88
//   up to a workgroup per CU                      0.68-0.90
//   causal with dropout                           0.54-1.03 (from 4096 rows on, in whole rounds of the eight, 0.91-1.03; 16384 rows in such 0.98-1.02)
//   causal, up to 1024 rows                       0.64-1.02; 3 to 4 per CU without a half-empty last item 0.88-1.14; beyond 16 or 10 per CU, out of
//                                                 the caches, 0.91-1.14 (a head's items, heaviest first, read its keys far apart in time)
//   causal, longer                                up to 3 per CU 0.70-1.02; up to 5 where the eight's last round is not full 0.82-1.03, else 0.96-1.18
//   not causal with dropout, fewer half rounds    0.53-0.92; else up to 512 rows 0.78-1.00, up to 1024 and from 4 per CU on 0.77-0.99, others 0.93-1.09
//   not causal, up to 512 rows                    fewer half rounds 0.64-1.00; more than four per CU 0.75-0.99; else 0.89-1.15
//   not causal, longer, three quarters of the half rounds  0.61-1.08 (0.89-0.98 in most; 1000 rows of a number of heads the XCDs don't share evenly
//                                                 1.04-1.08, not taken); up to 800 rows from 8 per CU on, fewer half rounds 0.83-0.97; else 0.91-1.17
bool fwd_runs_four_waves(const KParams& p) {
    const int64_t cus = persistent_grid(1 << 20), heads = static_cast<int64_t>(p.B) * p.H;
    const int64_t items = heads * ((p.S + 127) / 128), items256 = heads * ((p.S + 255) / 256);
    const int64_t halves = (items + cus - 1) / cus, rounds256 = (items256 + cus - 1) / cus;
    const bool half_empty = (p.S - 1) % 256 < 128;
    if (p.S <= 128 || items <= cus) return true;
    if (p.causal && p.thr8 > 0) return p.S <= 8192 || items <= 3 * cus;
    if (p.causal) {
        if (p.S <= 1024) return items <= (p.S <= 800 ? 16 : 10) * cus && (half_empty || p.S < 256 || items <= 3 * cus || items > 4 * cus);
        return items <= 3 * cus || (items <= 5 * cus && 16 * items256 <= 15 * rounds256 * cus);
    }
    if (p.thr8 > 0) return p.S <= 512 || halves < 2 * rounds256 || (p.S <= 1024 && items > 4 * cus);
    if (p.S <= 512) return halves < 2 * rounds256 || items > 4 * cus;
    if (4 * halves <= 6 * rounds256) return half_empty || p.S > 1024 || heads % 8 == 0;
    return p.S <= 800 && items > 8 * cus && halves < 2 * rounds256;
}

template <typename T, int D>
int launch_fwd_waves(int dtype, const KParams& p, hipStream_t stream) {
    // 8 waves (256 query rows) at D = 128 where the sequence allows it (without a mask as above): two waves per SIMD out of phase. Up to D = 64 four waves everywhere,
    // whose workgroups share a CU, so that starts and ends pass behind one another's tiles and less of the chip is idle in the last round. Time of
    // the four over that of the eight at multiples of 256: D = 32 0.78; D = 64 without a mask 0.82-0.86 at half as many items of 256 rows as CUs,
    // 0.93-0.99 at as many, 0.99-1.03 at twice as many (causal 0.77-0.86, 0.88-0.91 and 0.95-1.00), more than that: three_workgroups_per_cu; with
    // dropout 0.70-0.99; beside 16-bit masks 0.90-1.01; beside fp32 ones, whose ring of three lets two workgroups onto a CU, 0.88-0.96, length
    // masks 0.84-1.00 (dense ones in whole rounds of S = 2048 1.04-1.06).
    if constexpr (D == 128) {
        if (mask_is_key_bits(p)) {  // (with dropout always four waves: two workgroups to a CU against one of four waves that read the mask's values)
            if (p.thr8 > 0 || fwd_runs_four_waves(p)) return launch_fwd_ragged<T, D, 4, false, kMaskKeys>(p, stream);
            return p.S % 256 == 0 ? launch_fwd_dropout<T, D, 8, false, kMaskKeys>(p, stream) : launch_fwd_ragged<T, D, 8, false, kMaskKeys>(p, stream);
        }
        if (p.mask == nullptr && fwd_runs_four_waves(p)) return p.causal ? launch_fwd_ragged<T, D, 4, true>(p, stream) : launch_fwd_ragged<T, D, 4, false>(p, stream);
        if (p.S % 256 == 0) return launch_fwd_variant<T, D, 8>(dtype, p, stream);
        if (p.mask == nullptr) return p.causal ? launch_fwd_ragged<T, D, 8, true>(p, stream) : launch_fwd_ragged<T, D, 8, false>(p, stream);
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
