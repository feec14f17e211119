// Host-side launch entry points shared between the translation units of libtrident_attn.so.
#pragma once
#include <hip/hip_runtime.h>

#include "common.hpp"

namespace tri {

enum GenericKernel { kGenericFwd = 0, kGenericDelta = 1, kGenericDkdv = 2, kGenericDq = 3 };

// generic.hip: any shape / dtype, vector-ALU fp32 arithmetic.
int launch_generic_any(int which, int dtype, const KParams& p, hipStream_t stream);

// mfma_*.hip: fp16/bf16, D in {16,32,64,128}, 16-byte aligned rows; any S without a mask or with a padded one, S a multiple
// of 128 with any other.
enum MfmaKernel { kMfmaFwd = 0, kMfmaDkdv = 1, kMfmaDq = 2 };
bool mfma_supported(int which, int dtype, const KParams& p);
int launch_mfma_fwd(int dtype, const KParams& p, hipStream_t stream);
// with_delta: the dQ pass also computes and stores delta (only where mfma_dq_fuses_delta() says so; the
// dK/dV pass must then follow it)
int launch_mfma_dq(int dtype, const KParams& p, hipStream_t stream, bool with_delta = false);
bool mfma_dq_fuses_delta(const KParams& p);
int launch_mfma_dkdv(int dtype, const KParams& p, hipStream_t stream);
// Bytes of workspace (KParams::workspace) with which these launches run split along the streamed dimension; 0: they never do.
int64_t mfma_fwd_workspace(const KParams& p);
int64_t mfma_dq_workspace(const KParams& p, bool with_delta);
int64_t mfma_dkdv_workspace(const KParams& p);
int launch_delta(int dtype, const KParams& p, hipStream_t stream);

// mfma_dmask.hip: gradient of a mask, summed over the batches or heads that share it.
bool mfma_dmask_supported(int dtype, const KParams& p);
int launch_mfma_dmask(int dtype, KParams p, hipStream_t stream);
int64_t mfma_dmask_workspace(const KParams& p);  // bytes with which it deals the pairs of a tile to several workgroups; 0: it never does

// mfma32.hip: the fp32 matrix instruction. fp32 / fp16 / bf16 storage, D in {16,32,64,128}, any S, any mask, rows
// aligned to four elements. `which` is a MfmaKernel.
bool mfma32_supported(int which, int dtype, const KParams& p);
int64_t mfma32_workspace(int which, int dtype, const KParams& p);  // as mfma_fwd_workspace below
int launch_mfma32(int which, int dtype, const KParams& p, hipStream_t stream, bool with_delta = false);
bool mfma32_dq_fuses_delta(int dtype, const KParams& p);  // (as mfma_dq_fuses_delta, where mfma32_supported)
// Classes of the mask's 64 x 64 blocks (0 all zero, 1 all -inf, 2 mixed) into `out`, laid out as p.mcs says.
int launch_classify_mask(const KParams& p, uint8_t* out, hipStream_t stream);
// Source mask (additive, or bytes: TRI_ATTN_BOOL) -> padded additive mask `out` laid out as p.ms says, and its block classes
// (unless nullptr) as p.mcs says.
int launch_prepare_mask(const KParams& p, void* out, uint8_t* classes, const void* source, int source_dtype, const int64_t* source_stride,
                        hipStream_t stream);
enum MaskClass { kMaskZero = 0, kMaskNegInf = 1, kMaskMixed = 2 };
// Number of workgroups for a kernel whose workgroups are persistent (one per CU, each walking several of
// the `items`): min(items, CUs of the current device).
int persistent_grid(int items);
// Whether forward and dQ at D = 64 without a mask run their 128-row workgroups three to a CU (in 168 registers, with a ring of three tiles)
// instead of two: launches of several rounds. Time of three over that of two, or of the eight-wave kernels that ran before, by the number
// of workgroups: up to two per CU forward 0.97-1.06, dQ 0.97-1.09; causal at 3.4 to 4 per CU forward 0.93-0.98 (16 heads of S = 8192: 1.03),
// dQ 0.81-0.98, at 5.5 to 16 forward 0.88-0.92, dQ 0.88-0.93; not causal at 3.4 to 4 forward 0.96-1.09, dQ 0.98-1.06, from 5.5 on forward
// 0.90-0.96, dQ 0.90-1.01.
bool three_workgroups_per_cu(const KParams& p);
// Whether the mask is one of keys (the same for every row) that is 0 or -inf, of the operand type and over few enough tiles for the kernels
// that keep it as bits (KeyBits).
bool mask_is_key_bits(const KParams& p);

}  // namespace tri
