// Gradient of an additive mask that is shared by batches or heads (or both) for fp16/bf16 problems, D in {16,32,64,128}, any S
// (trident/kernel/attention.py:332-335 stores dS per batch and head; autograd then sums it over the broadcast dimensions).
//
// A workgroup owns a tile of the mask and walks the (batch, head) pairs that share it, adding dS = P (dP - delta) in registers:
// no atomic, no zero fill, a fixed order of summation, and the tile of the mask itself is read once for all pairs. The price is
// S and dP once more (2 of the pass's 7 products), where the dQ pass, which has them, would send every dS to memory by itself:
// bf16 B=8 H=12 S=512 D=64, bias [1,H,S,S]: the dQ pass with atomic adds took 0.61 ms, bound by the 25 M adds; without them
// it takes 0.023 ms and this kernel 0.039.
//
// A wave takes 32 rows x 64 keys: the K and V rows are the A operands, the Q and dO rows the B operands, so that lane l32 owns
// a row with its lse and delta, and the accumulators (8 keys groups of 4) leave in row pieces. The rows of a (batch, head) are
// read by S / 32 workgroups of one XCD and sit in its L2.
// D = 64: a workgroup stages the rows of a pair in LDS, in whole lines and K and V once for its four waves, with the next pair's
// on their way in registers. Straight from memory, 16 bytes per lane, a load touches 32 cache lines and bounds the kernel: the
// case above 0.059 -> 0.039 ms, B=2 H=16 S=2048 0.346 -> 0.278 ms. The other head sizes keep the direct loads: at D = 128 the
// staged rows leave one workgroup per CU (0.511 -> 0.645 ms staged), at D = 32 the exponentials weigh more and the barriers cost
// what the loads save (0.203 -> 0.228 ms).
// SPLIT: too few tiles to fill the chip. The four waves of a workgroup then share one tile, take every fourth pair each, and
// their sums meet in LDS; otherwise they are four row blocks of one key tile.
#include "launch.hpp"
#include "mfma_common.hpp"

namespace tri {
namespace {

constexpr int kKeys = 64;

template <typename T, int D, bool DROPOUT, bool SPLIT>
__global__ __launch_bounds__(256, 2) void mfma_dmask_kernel(const KParams p, int units, int per_xcd, bool by_fours) {
    constexpr int KK = D / 16;
    // staged rows of a pair: 64 of K, 64 of V, 128 of Q, 128 of dO, each 16 bytes longer than its elements (a fragment read's
    // lanes then fall on different banks at every head size)
    constexpr int kPitch = 2 * D + 16, kStaged = 2 * kKeys + 2 * 128;
    constexpr bool kStage = !SPLIT && D == 64;
    __shared__ __attribute__((aligned(16))) char smem[SPLIT ? 3 * 32 * 64 * 4 : kStage ? kStaged * kPitch : 16];
    float* const sums = reinterpret_cast<float*>(smem);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63, l32 = lane & 31, h = lane >> 5;
    // consecutive tiles of one mask on one XCD
    const int unit = static_cast<int>(blockIdx.x & 7) * per_xcd + static_cast<int>(blockIdx.x >> 3);
    if (unit >= units) return;
    constexpr int kRows = SPLIT ? 32 : 128;
    const int key_tiles = (p.S + kKeys - 1) / kKeys, row_tiles = (p.S + kRows - 1) / kRows;
    const int kt = unit % key_tiles, rt = unit / key_tiles % row_tiles, m = unit / key_tiles / row_tiles;
    // the mask's own batches and heads; the others are summed over
    const int mask_heads = p.dms[1] == 0 ? 1 : p.H;
    const int mask_b = m / mask_heads, mask_h = m % mask_heads;
    const int sum_b = p.dms[0] == 0 ? p.B : 1, sum_h = p.dms[1] == 0 ? p.H : 1;
    const int t0 = kt * kKeys;
    const int wrow0 = rt * kRows + (SPLIT ? 0 : 32 * wave);
    const int qrow = wrow0 + l32;
    const bool row_ok = qrow < p.S;
    const int qrow_ld = min(qrow, p.S - 1);
    if (!SPLIT && !kStage && wrow0 >= p.S) return;  // (a wave without a single row; no barrier in this variant)

    // mask values of this lane's row (log2 domain), the same for every pair; -inf for keys that do not exist
    float mk[32];
    {
        const int64_t at = mask_b * p.ms[0] + mask_h * p.ms[1] + static_cast<int64_t>(qrow_ld) * p.ms[2];
#pragma unroll
        for (int i = 0; i < 32; ++i) {
            const int key = t0 + 32 * (i >> 4) + c_row(i & 15, h);
            mk[i] = key < p.S ? load_mask_elem(p.mask, p.mask_dtype, at + key) * kLog2e : -INFINITY;
        }
    }
    const int key_ld0 = min(t0 + l32, p.S - 1), key_ld1 = min(t0 + 32 + l32, p.S - 1);
    float acc[32];
#pragma unroll
    for (int i = 0; i < 32; ++i) acc[i] = 0.f;

    // dS of 32 rows x 32 keys of one pair, added to the accumulators of key block kb
    const auto add = [&](int kb, int64_t bh, float lse, float dlt, const u32x4(&kf)[KK], const u32x4(&vf)[KK], const u32x4(&qf)[KK],
                         const u32x4(&gf)[KK]) {
        f32x16 s = zero16(), dp = zero16();
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            s = Mma<T>::run(kf[kk], qf[kk], s);
            dp = Mma<T>::run(vf[kk], gf[kk], dp);
        }
        if constexpr (DROPOUT) {
            const Philox4 mine = dropout_block(p, static_cast<uint32_t>(bh), qrow >> 2, (t0 + 32 * kb + 8 * (lane & 3) + 4 * h) >> 2);
            uint32_t w[4];
            quad_row_words(mine, lane, w);
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int bb = 0; bb < 4; ++bb) {
                    const bool keep = static_cast<int>((w[g] >> (8 * bb)) & 0xffu) >= p.thr8;
                    dp[4 * g + bb] = keep ? dp[4 * g + bb] * p.zscale : 0.f;
                }
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[16 * kb + i] += fast_exp2(fmaf(s[i], p.scale_log2, mk[16 * kb + i]) - lse) * (dp[i] - dlt);
    };

    const int pairs = sum_b * sum_h;
    if constexpr (!kStage) {
        for (int pair = SPLIT ? wave : 0; pair < pairs; pair += SPLIT ? 4 : 1) {
            const int b = mask_b + pair / sum_h, hd = mask_h + pair % sum_h;
            const int64_t bh = static_cast<int64_t>(b) * p.H + hd;
            const T* qp = static_cast<const T*>(p.q) + b * p.qs[0] + hd * p.qs[1] + qrow_ld * p.qs[2] + 8 * h;
            const T* gp = static_cast<const T*>(p.d_o) + b * p.dos[0] + hd * p.dos[1] + qrow_ld * p.dos[2] + 8 * h;
            const T* kp = static_cast<const T*>(p.k) + b * p.ks[0] + hd * p.ks[1] + 8 * h;
            const T* vp = static_cast<const T*>(p.v) + b * p.vs[0] + hd * p.vs[1] + 8 * h;
            const float lse = p.lse[bh * p.S + qrow_ld];
            const float dlt = p.delta[bh * p.S + qrow_ld];
            u32x4 qf[KK], gf[KK];
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) {
                qf[kk] = *reinterpret_cast<const u32x4*>(qp + 16 * kk);
                gf[kk] = *reinterpret_cast<const u32x4*>(gp + 16 * kk);
            }
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                const int64_t key = kb ? key_ld1 : key_ld0;
                u32x4 kf[KK], vf[KK];
#pragma unroll
                for (int kk = 0; kk < KK; ++kk) {
                    kf[kk] = *reinterpret_cast<const u32x4*>(kp + key * p.ks[2] + 16 * kk);
                    vf[kk] = *reinterpret_cast<const u32x4*>(vp + key * p.vs[2] + 16 * kk);
                }
                add(kb, bh, lse, dlt, kf, vf, qf, gf);
            }
        }
    } else {
        // Thread t moves the 16-byte pieces t, t + 256, ... of the pair's rows: consecutive lanes, consecutive addresses. The
        // next pair's pieces are on their way while this one is multiplied.
        constexpr int kPerRow = D / 8, kStep = 256 / kPerRow, kPieces = kStaged / kStep;
        const int piece_row = static_cast<int>(threadIdx.x) / kPerRow, piece_col = static_cast<int>(threadIdx.x) % kPerRow * 8;
        u32x4 piece[kPieces];
        float lse_next, dlt_next;
        const auto fetch = [&](int pair) {
            const int b = mask_b + pair / sum_h, hd = mask_h + pair % sum_h;
            const int64_t bh = static_cast<int64_t>(b) * p.H + hd;
            const T* qp = static_cast<const T*>(p.q) + b * p.qs[0] + hd * p.qs[1] + piece_col;
            const T* gp = static_cast<const T*>(p.d_o) + b * p.dos[0] + hd * p.dos[1] + piece_col;
            const T* kp = static_cast<const T*>(p.k) + b * p.ks[0] + hd * p.ks[1] + piece_col;
            const T* vp = static_cast<const T*>(p.v) + b * p.vs[0] + hd * p.vs[1] + piece_col;
            int row0 = piece_row;
            asm volatile("" : "+v"(row0));  // (row offsets are computed again for each pair: kept, they spill at D = 64)
#pragma unroll
            for (int i = 0; i < kPieces; ++i) {
                const int r = row0 + i * kStep;  // (rows beyond the sequence: its last one, masked or not stored)
                const T* from = r < kKeys           ? kp + min(t0 + r, p.S - 1) * p.ks[2]
                                : r < 2 * kKeys       ? vp + min(t0 + r - kKeys, p.S - 1) * p.vs[2]
                                : r < 2 * kKeys + 128 ? qp + min(rt * 128 + r - 2 * kKeys, p.S - 1) * p.qs[2]
                                                      : gp + min(rt * 128 + r - 2 * kKeys - 128, p.S - 1) * p.dos[2];
                piece[i] = *reinterpret_cast<const u32x4*>(from);
            }
            lse_next = p.lse[bh * p.S + qrow_ld];
            dlt_next = p.delta[bh * p.S + qrow_ld];
        };
        const auto fragment = [&](int row, int kk) {
            return *reinterpret_cast<const u32x4*>(smem + (row + l32) * kPitch + 32 * kk + 16 * h);
        };
        fetch(0);
        for (int pair = 0; pair < pairs; ++pair) {
            const int64_t bh = static_cast<int64_t>(mask_b + pair / sum_h) * p.H + mask_h + pair % sum_h;
            const float lse = lse_next, dlt = dlt_next;
            lds_barrier();  // (the fragments of the pair before have been read)
#pragma unroll
            for (int i = 0; i < kPieces; ++i) *reinterpret_cast<u32x4*>(smem + (piece_row + i * kStep) * kPitch + 2 * piece_col) = piece[i];
            lds_barrier();
            if (pair + 1 < pairs) fetch(pair + 1);
            u32x4 qf[KK], gf[KK];
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) {
                qf[kk] = fragment(2 * kKeys + 32 * wave, kk);
                gf[kk] = fragment(2 * kKeys + 128 + 32 * wave, kk);
            }
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                u32x4 kf[KK], vf[KK];
#pragma unroll
                for (int kk = 0; kk < KK; ++kk) {
                    kf[kk] = fragment(32 * kb, kk);
                    vf[kk] = fragment(kKeys + 32 * kb, kk);
                }
                add(kb, bh, lse, dlt, kf, vf, qf, gf);
                __builtin_amdgcn_sched_barrier(0);  // (one key block's fragments at a time)
            }
        }
    }
    if constexpr (SPLIT) {
        if (wave > 0) {
#pragma unroll
            for (int i = 0; i < 32; ++i) sums[((wave - 1) * 32 + i) * 64 + lane] = acc[i];
        }
        __syncthreads();
        if (wave > 0) return;
#pragma unroll
        for (int i = 0; i < 32; ++i) acc[i] += (sums[i * 64 + lane] + sums[(32 + i) * 64 + lane]) + sums[(64 + i) * 64 + lane];
    }
    if (!row_ok) return;
    const int64_t at = mask_b * p.dms[0] + mask_h * p.dms[1] + static_cast<int64_t>(qrow) * p.dms[2] + t0;
#pragma unroll
    for (int g = 0; g < 8; ++g) {
        const int key = 32 * (g >> 2) + 8 * (g & 3) + 4 * h;  // keys key .. key + 3 of the tile
        const float* v = &acc[4 * g];
        if (by_fours && t0 + key + 3 < p.S) {
            if (p.mask_dtype == TRI_ATTN_F32) *reinterpret_cast<f32x4*>(static_cast<float*>(p.dmask) + at + key) = f32x4{v[0], v[1], v[2], v[3]};
            else *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(p.dmask) + at + key) = p.mask_dtype == TRI_ATTN_F16
                ? u32x2{Mma<f16_t>::pack2(v[0], v[1]), Mma<f16_t>::pack2(v[2], v[3])} : u32x2{Mma<bf16_t>::pack2(v[0], v[1]), Mma<bf16_t>::pack2(v[2], v[3])};
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (t0 + key + e < p.S) store_mask_elem(p.dmask, p.mask_dtype, at + key + e, v[e]);
        }
    }
}

bool splits_pairs(const KParams& p, int64_t masks) { return masks * ((p.S + kKeys - 1) / kKeys) * ((p.S + 127) / 128) < 256; }

template <typename T, int D>
int launch_dmask_t(const KParams& p, hipStream_t stream) {
    const int64_t masks = (p.dms[0] == 0 ? int64_t{1} : p.B) * (p.dms[1] == 0 ? 1 : p.H);
    const int64_t key_tiles = (p.S + kKeys - 1) / kKeys;
    // one key tile x 128 rows per workgroup where that gives every compute unit one, else 32 rows with the pairs split (with
    // 384 such workgroups, the case above, split ones took 0.065 ms against 0.062 with direct loads in both, 0.039 staged)
    const bool split = splits_pairs(p, masks);
    const int64_t units = masks * key_tiles * (split ? (p.S + 31) / 32 : (p.S + 127) / 128);
    if (units > 2147483647LL / 8) return TRI_ATTN_ESHAPE;
    const int per_xcd = static_cast<int>((units + 7) / 8);
    const dim3 grid(8 * per_xcd), block(256);
    const int n = static_cast<int>(units);
    const bool fours = reinterpret_cast<uintptr_t>(p.dmask) % 16 == 0 && p.dms[0] % 4 == 0 && p.dms[1] % 4 == 0 && p.dms[2] % 4 == 0;
    if (p.thr8 > 0) {
        if (split) hipLaunchKernelGGL((mfma_dmask_kernel<T, D, true, true>), grid, block, 0, stream, p, n, per_xcd, fours);
        else hipLaunchKernelGGL((mfma_dmask_kernel<T, D, true, false>), grid, block, 0, stream, p, n, per_xcd, fours);
    } else {
        if (split) hipLaunchKernelGGL((mfma_dmask_kernel<T, D, false, true>), grid, block, 0, stream, p, n, per_xcd, fours);
        else hipLaunchKernelGGL((mfma_dmask_kernel<T, D, false, false>), grid, block, 0, stream, p, n, per_xcd, fours);
    }
    return static_cast<int>(hipGetLastError());
}

template <typename T>
int launch_dmask_d(const KParams& p, hipStream_t stream) {
    return p.D == 128 ? launch_dmask_t<T, 128>(p, stream) : p.D == 64 ? launch_dmask_t<T, 64>(p, stream)
         : p.D == 32 ? launch_dmask_t<T, 32>(p, stream) : launch_dmask_t<T, 16>(p, stream);
}

bool rows8(const void* ptr, const int64_t* s) {
    return reinterpret_cast<uintptr_t>(ptr) % 16 == 0 && s[0] % 8 == 0 && s[1] % 8 == 0 && s[2] % 8 == 0;
}

}  // namespace

bool mfma_dmask_supported(int dtype, const KParams& p) {
    if (dtype != TRI_ATTN_F16 && dtype != TRI_ATTN_BF16) return false;
    if (p.mask == nullptr || p.dmask == nullptr || p.causal) return false;
    const bool over_b = p.dms[0] == 0 && p.B > 1, over_h = p.dms[1] == 0 && p.H > 1;
    if (!over_b && !over_h && p.S % 128 == 0) return false;                      // (written in place by the dQ pass)
    if (p.dms[2] == 0 && p.S > 1) return false;                                  // (summed over the rows: atomics)
    if ((over_b && p.ms[0] != 0) || (over_h && p.ms[1] != 0)) return false;      // (one mask tile for all pairs)
    // A wave's pairs follow one another (about 0.75 us each per 16 columns of the head size: latency), while the atomic adds of
    // the dQ pass go through at 41 G/s: few tiles shared by very many pairs stay there (bf16 [1,1,S,S], B=32 H=8 S=128 D=128:
    // 0.40 ms here, 0.23 ms with atomics).
    const int64_t masks = (p.dms[0] == 0 ? 1 : p.B) * static_cast<int64_t>(p.dms[1] == 0 ? 1 : p.H);
    const int64_t heads = static_cast<int64_t>(p.B) * p.H, pairs = heads / masks;
    const double walk_us = static_cast<double>(splits_pairs(p, masks) ? (pairs + 3) / 4 : pairs) * 0.75 * (p.D / 16);
    if (walk_us > 20.0 + static_cast<double>(heads) * p.S * p.S / 41e3) return false;
    return rows8(p.q, p.qs) && rows8(p.k, p.ks) && rows8(p.v, p.vs) && rows8(p.d_o, p.dos);
}

int launch_mfma_dmask(int dtype, const KParams& p, hipStream_t stream) {
    return dtype == TRI_ATTN_BF16 ? launch_dmask_d<bf16_t>(p, stream) : launch_dmask_d<f16_t>(p, stream);
}

}  // namespace tri
