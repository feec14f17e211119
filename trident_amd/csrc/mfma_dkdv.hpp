// dK/dV pass of the backward on the matrix cores for fp16/bf16, D in {16,32,64,128} (the dQ pass: mfma_dq.hip;
// together they replace trident/kernel/attention.py:169-339):
//
//   dK/dV pass one workgroup per 256 (128) keys (a wave, or for D = 128 a pair of waves, owns 32),
//              streaming query tiles of 64: S = Q K^T, dP = dO V^T, dV^T += dO^T P, dK^T += Q^T dS
//
// The lane index is the key that owns the accumulators, the stationary operands (K, V) stay in registers as MFMA B
// operands, and P / dS go from the accumulators of one MFMA to the B operand of the next without leaving registers.
#pragma once
#include <type_traits>

#include "split.hpp"

namespace tri {
namespace {

constexpr int kBM = 128;  // stationary rows per workgroup
constexpr int kBN = 64;   // streamed rows per tile

enum MaskKind { kNoMask = 0, kMaskF32 = 1, kMaskT = 2, kMaskKeys = 3 };  // (kMaskKeys: of the operand type, see KeyBits)

template <typename T, int MASK>
__device__ __forceinline__ float mask_at(const void* mask, int64_t off) {
    if constexpr (MASK == kMaskF32) return static_cast<const float*>(mask)[off];
    else return static_cast<float>(static_cast<const T*>(mask)[off]);
}

// ------------------------------------------------------------------ dK, dV (4 waves)
// Same data flow as the dQ kernel with the roles of queries and keys exchanged: a workgroup of
// 4 waves owns 128 keys, one wave 32 of them with its K and V rows in registers (B operands)
// and dK^T, dV^T in fp32 accumulators; two workgroups and more per CU. Q and dO stream as 64-row swizzled LDS
// tiles (plus their lse and delta) in a ring of 4 filled by LDS-direct loads three tiles ahead.
// Per 32-row query block: S = Q K^T and dP = dO V^T from row fragments, P and dS on the vector
// ALU, dV^T += dO^T P and dK^T += Q^T dS with the transposed LDS reads of the same tiles.
// RAGGED (no mask, or a padded one): S is not a multiple of 128. Loads clamp their
// row index to S - 1, query rows >= S get probability 0 (they would otherwise add the last row once more), keys >= S
// are not stored.
// SPLIT (with RAGGED): a workgroup streams one part of its item's row tiles (split.hpp).
template <int D, int MASK, bool DROPOUT>
constexpr bool kThree = D == 64 && (MASK == kNoMask || MASK == kMaskKeys) && !DROPOUT;
template <typename T, int D, bool CAUSAL, int MASK, bool DROPOUT, bool RAGGED = false, bool SPLIT = false>
__global__ __launch_bounds__(256, (kThree<D, MASK, DROPOUT>) ? 3 : RAGGED && !((MASK == kMaskF32 || MASK == kMaskT) && D == 64 && !DROPOUT) ? 1 : 2) void mfma_dkdv_wide_kernel(const KParams p) {
    static_assert(RAGGED || !SPLIT, "parts have boundary handling");
    using Tile = SwzTile<D>;
    constexpr int NW = 4;
    constexpr int kKeys = 32 * NW;
    // (a ring of three, or two beside an fp32 mask, where it lets a second workgroup onto the CU beside the mask regions, whose tiles hide what
    // the shorter lead leaves of the loads' latency: launch_dkdv_dropout says what that gives)
    constexpr bool kMatrix = MASK == kMaskF32 || MASK == kMaskT;  // a mask whose values are read tile by tile
    constexpr int kStages = kMatrix && D == 64 && !(DROPOUT && RAGGED) ? (MASK == kMaskT ? 3 : 2) : kThree<D, MASK, DROPOUT> ? 3 : 4;
    constexpr int kAhead = kStages - 1;  // tile j + kAhead is requested in tile j, into the slot of tile j - 1
    constexpr int kStageBytes = 2 * Tile::kBytes + 2 * kBN * 4;  // Q tile, dO tile, lse, delta
    constexpr int KK = D / 16;
    constexpr int DB = D >= 32 ? D / 32 : 1;  // (D = 16: one block of gradient columns, the upper 16 are not stored)
    constexpr int kBlocksPerWave = 2 * Tile::kBlocks / NW;
    constexpr int kLoadsPerTile = kBlocksPerWave + 1;            // + lse or delta: exact for every wave
    static_assert(2 * Tile::kBlocks % NW == 0, "tile blocks must divide among the waves");
    // A mask block of a wave (64 rows x its 32 keys) goes through a private LDS region (8 KiB fp32, 4 KiB for a mask
    // of the operand type) when it fits (D = 64). Plain loads would be tracked by the compiler, whose waits for them
    // also drain the LDS-direct tile loads issued in between (the counter completes in order), which makes the
    // tile prefetch synchronous. Geometry of a 64-row SwzTile<64> / SwzTile<32> (128- or 64-byte rows = 32 keys).
    constexpr bool kMaskViaLds = kMatrix && D <= 64;
    constexpr int kMaskElt = MASK == kMaskF32 ? 4 : 2;
    using MaskTile = std::conditional_t<MASK == kMaskF32, SwzTile<64>, SwzTile<32>>;
    constexpr int kMaskLoads = MaskTile::kBlocks;
    __shared__ __attribute__((aligned(1024))) char smem[kStages * kStageBytes + (kMaskViaLds ? NW * MaskTile::kBytes : 0)];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, l32 = lane & 31, h = lane >> 5;
    int bh, kt;
    [[maybe_unused]] Part part{};
    if constexpr (SPLIT) {
        if (!map_part(p, blockIdx.x, gridDim.x, (p.S + kKeys - 1) / kKeys, (p.S + kBN - 1) / kBN, CAUSAL, &part)) return;
        bh = part.bh;
        kt = part.tile;
    } else {
        map_block_for<MASK>(p, blockIdx.x, (p.S + kKeys - 1) / kKeys, CAUSAL ? kHeavyFirst : kUniformTiles, &bh, &kt);
    }
    const int b = bh / p.H, hd = bh % p.H;
    const int k0 = kt * kKeys;
    const int wkey0 = k0 + 32 * wave;
    const int key = wkey0 + l32;
    const int key_ld = RAGGED ? min(key, p.S - 1) : key;  // (a key that does not exist reads the last one)

    const char* kbase = static_cast<const char*>(p.k) + (b * p.ks[0] + hd * p.ks[1]) * 2;
    const char* vbase = static_cast<const char*>(p.v) + (b * p.vs[0] + hd * p.vs[1]) * 2;
    const char* qbase = static_cast<const char*>(p.q) + (b * p.qs[0] + hd * p.qs[1]) * 2;
    const char* gbase = static_cast<const char*>(p.d_o) + (b * p.dos[0] + hd * p.dos[1]) * 2;
    const int64_t qrow_bytes = p.qs[2] * 2, grow_bytes = p.dos[2] * 2;
    const float* lse_base = p.lse + static_cast<int64_t>(bh) * p.S;
    const float* delta_base = p.delta + static_cast<int64_t>(bh) * p.S;

    u32x4 kf[KK], vf[KK];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
        kf[kk] = *reinterpret_cast<const u32x4*>(kbase + static_cast<int64_t>(key_ld) * p.ks[2] * 2 + (2 * kk + h) * 16);
        vf[kk] = *reinterpret_cast<const u32x4*>(vbase + static_cast<int64_t>(key_ld) * p.vs[2] * 2 + (2 * kk + h) * 16);
    }
    const float c = p.scale_log2;
    [[maybe_unused]] const float inv_scale = p.inv_scale;  // (a mask value joins its score before the scale: s + mask / scale)
    // a mask of keys is one value per lane
    bool hidden = false, some_hidden = false;
    if constexpr (MASK == kMaskKeys) {
        hidden = mask_at<T, kMaskT>(p.mask, b * p.ms[0] + hd * p.ms[1] + key_ld) != 0.f;
        some_hidden = __builtin_amdgcn_ballot_w64(hidden) != 0;
    }
    // Without dropout the subtraction in dS = P (dP - delta) is left to the matrix pipe: the dP accumulators start from
    // the rows' delta values (as they come from the tile: the accumulator's layout) and take the product with the V
    // fragments negated, which gives delta - dP; dS then comes out negated and the sign goes into dK's final scale.
    constexpr bool kDeltaInAcc = !DROPOUT;

    f32x16 dk[DB], dv[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) {
        dk[db] = zero16();
        dv[db] = zero16();
    }

    int src_off[kBlocksPerWave];
#pragma unroll
    for (int i = 0; i < kBlocksPerWave; ++i) {
        const int blk = wave * kBlocksPerWave + i;
        const bool is_g = blk >= Tile::kBlocks;
        src_off[i] = static_cast<int>(Tile::src_off(is_g ? blk - Tile::kBlocks : blk, lane, is_g ? grow_bytes : qrow_bytes));
    }
    int t_begin = CAUSAL ? k0 / kBN : 0;                        // first tile with rows that see the workgroup's keys
    const int my_begin = CAUSAL ? wkey0 / kBN : 0;              // first tile with rows that see this wave's keys
    int n_tiles = (p.S + kBN - 1) / kBN;
    if constexpr (SPLIT) {
        t_begin += part.index * p.part_tiles;
        n_tiles = max(t_begin, min(n_tiles, t_begin + p.part_tiles));
    }
    const int t_first = SPLIT ? t_begin : 0;  // the tile the classes count from
    [[maybe_unused]] const int rows_end = min(n_tiles * kBN, p.S);
    // With the classes of the mask's blocks at hand: row tiles before the first and behind the last one that is not
    // masked out altogether over the workgroup's keys are not streamed (keys beyond every length: nothing at all, the
    // gradients are zero), and tiles whose mask is all zero over the workgroup's keys are not read.
    // A row without a single visible key (its lse is -inf) turns all of dK and dV to NaN, as softmax does. Where a padded mask
    // leaves row tiles out, such rows are looked for among theirs: left_out, a factor of the results, is NaN if there are
    // any. (Usual padding and length masks leave rows out only of workgroups whose keys nobody sees.)
    [[maybe_unused]] float left_out = 1.f;
    uint64_t zero_tiles = 0;
    if constexpr (MASK != kNoMask) {
        if (p.mcls != nullptr && n_tiles - t_first <= 64) {
            const uint8_t* const classes = p.mcls + b * p.mcs[0] + hd * p.mcs[1] + k0 / 64;
            const int all_tiles = (p.S + kBN - 1) / kBN, across = RAGGED ? min(kKeys / 64, all_tiles - k0 / 64) : kKeys / 64;
            const TileClasses tc = tile_classes(classes + t_first * p.mcs[2], p.mcs[2], n_tiles - t_first, across, 1, lane);
            zero_tiles = tc.zero;
            if constexpr (SPLIT) {
                const int2 on = active_range(classes, p.mcs[2], all_tiles, across, 1, lane);
                t_begin = max(t_first, min(on.x, n_tiles));
                n_tiles = max(t_begin, min(on.y, n_tiles));
            } else if (tc.active) {
                n_tiles = 64 - __builtin_clzll(tc.active);
                t_begin = __builtin_ctzll(tc.active);
            } else {
                n_tiles = t_begin = 0;
            }
            // (whole items at multiples of 128 with classes leave them out unlooked; those of the paired kernel, D = 128, leave out none)
            if (RAGGED && !(SPLIT && D < 128 && p.S % 128 == 0 && all_tiles <= 64)) {
                bool lost = false;
                for (int r = t_first * kBN + lane; r < t_begin * kBN; r += 64) lost |= !(lse_base[r] > -INFINITY);
                for (int r = n_tiles * kBN + lane; r < rows_end; r += 64) lost |= !(lse_base[r] > -INFINITY);
                if (__builtin_amdgcn_ballot_w64(lost) != 0) left_out = __builtin_nanf("");
            }
        }
    }
    auto mask_is_zero = [&](int t) { return MASK != kNoMask && ((zero_tiles >> (t - t_first)) & 1) != 0; };
    auto issue_tile = [&](int t) {
        char* stage = smem + (t % kStages) * kStageBytes;
        const bool partial = RAGGED && (t + 1) * kBN > p.S;  // the sequence ends inside this tile
        const int last = p.S - 1 - t * kBN;
#pragma unroll
        for (int i = 0; i < kBlocksPerWave; ++i) {
            const int blk = wave * kBlocksPerWave + i;
            const bool is_g = blk >= Tile::kBlocks;
            const char* tile_src = is_g ? gbase + static_cast<int64_t>(t) * kBN * grow_bytes
                                        : qbase + static_cast<int64_t>(t) * kBN * qrow_bytes;
            char* dst = stage + (is_g ? Tile::kBytes + (blk - Tile::kBlocks) * 1024 : blk * 1024);
            if (partial)
                lds_direct_load16(tile_src, Tile::src_off_clamped(is_g ? blk - Tile::kBlocks : blk, lane, is_g ? grow_bytes : qrow_bytes, last), dst);
            else
                lds_direct_load16(tile_src, src_off[i], dst);
        }
        // every wave issues exactly one more load, so that the vmcnt bookkeeping is the same in all of
        // them: even waves fetch the 64 lse values, odd waves the 64 delta values (duplicates land
        // on the same bytes)
        const int aux = (partial ? min(lane, last) : lane) * 4;
        if (wave & 1) lds_direct_load4(delta_base + t * kBN, aux, stage + 2 * Tile::kBytes + kBN * 4);
        else lds_direct_load4(lse_base + t * kBN, aux, stage + 2 * Tile::kBytes);
    };
    char* mask_lds = smem + kStages * kStageBytes + wave * MaskTile::kBytes;
    auto issue_mask = [&](int t) {  // rows of tile t x this wave's keys -> the wave's region, unless the tile is all zero
        if constexpr (kMaskViaLds) {
            if (mask_is_zero(t)) return;
            const int col0 = RAGGED && wkey0 >= p.S ? 0 : wkey0;  // (a wave without a single key reads some row's first ones)
            const char* src = static_cast<const char*>(p.mask) +
                              (b * p.ms[0] + hd * p.ms[1] + static_cast<int64_t>(t) * kBN * p.ms[2] + col0) * kMaskElt;
            int l = lane;
            asm volatile("" : "+v"(l));  // offsets recomputed per tile rather than kept in registers
#pragma unroll
            for (int blk = 0; blk < kMaskLoads; ++blk)
                lds_direct_load16(src, RAGGED ? MaskTile::src_off_clamped(blk, l, p.ms[2] * kMaskElt, p.S - 1 - t * kBN)
                                              : static_cast<uint32_t>(MaskTile::src_off(blk, l, p.ms[2] * kMaskElt)), mask_lds + blk * 1024);
        }
    };
    // issue order: mask block of the first tile, kAhead tiles, then per tile j: mask j+1, tile j+kAhead
    if (t_begin < n_tiles) {
        issue_mask(t_begin);
        issue_tile(t_begin);
    }
    if (kAhead > 1 && t_begin + 1 < n_tiles) issue_tile(t_begin + 1);
    if (kAhead > 2 && t_begin + 2 < n_tiles) issue_tile(t_begin + 2);
    // (the K and V fragments were requested before the tiles, so both latencies overlap)
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
        settle(kf[kk]);
        settle(vf[kk]);
        if constexpr (kDeltaInAcc) {
#pragma unroll
            for (int i = 0; i < 4; ++i) vf[kk][i] ^= 0x80008000u;
        }
    }

    [[maybe_unused]] DropoutKeys drop;
    if constexpr (DROPOUT) drop.init(p, bh, key >> 2);
    int row_off0 = Tile::off(l32, h);
    int tr_off0 = Tile::tr_off(0, 0, lane), tr_off1 = Tile::tr_off(0, 1, lane);

    for (int j = t_begin; j < n_tiles; ++j) {
        {
            // with a staged mask, block j must have landed too: only tile j + kAhead - 1 was issued after it
            // (the kAhead first tiles after the first block)
            // (a block that is all zero was never requested: then the kAhead - 1 youngest tiles are what may be in flight)
            // (kAhead == 1: tile j itself was issued after its mask block, nothing may be in flight)
            const int younger = kMaskViaLds && j > t_begin && !mask_is_zero(j) ? min(min(1, kAhead - 1), max(0, n_tiles - (kAhead - 1) - j)) : min(kAhead - 1, n_tiles - 1 - j);
            if (younger == 2) TRI_WAIT_VMCNT(2 * kLoadsPerTile);
            else if (younger == 1) TRI_WAIT_VMCNT(kLoadsPerTile);
            else TRI_WAIT_VMCNT(0);
        }
        lds_barrier();
        float mk2[kMaskViaLds ? 32 : 1];
        if constexpr (kMaskViaLds) {
            // (a mask excludes the causal variant, so every wave works on every tile)
            if (!mask_is_zero(j)) {  // (a tile whose mask is all zero takes the arithmetic of a tile without a mask)
#pragma unroll
                for (int i = 0; i < 32; ++i) {  // row 32 (i / 16) + c_row(i % 16, h), this lane's key
                    const int row = 32 * (i >> 4) + c_row(i & 15, h);
                    if constexpr (MASK == kMaskF32)
                        mk2[i] = *reinterpret_cast<const float*>(mask_lds + MaskTile::off(row, l32 >> 2) + (l32 & 3) * 4);
                    else
                        mk2[i] = to_f32(*reinterpret_cast<const T*>(mask_lds + MaskTile::off(row, l32 >> 3) + (l32 & 7) * 2));
                }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // region read before it is refilled
            }
            if (j + 1 < n_tiles) issue_mask(j + 1);
        }
        if (j + kAhead < n_tiles) issue_tile(j + kAhead);
        if (j < my_begin) continue;

        const char* sQ = smem + (j % kStages) * kStageBytes;
        const char* sG = sQ + Tile::kBytes;
        const float* sLse = reinterpret_cast<const float*>(sG + Tile::kBytes);
        const float* sDelta = sLse + kBN;
        const int r0 = j * kBN;
        // (the fragments' offsets of the column blocks are made from these here, not kept in registers across the loop)
        if constexpr (kThree<D, MASK, DROPOUT>) asm volatile("" : "+v"(row_off0), "+v"(tr_off0), "+v"(tr_off1));
        const bool diag = CAUSAL && r0 < wkey0 + 31;  // some row of the tile is above some key of the wave
#pragma unroll 1
        for (int qb = 0; qb < 2; ++qb) {
            const int rb = r0 + 32 * qb;
            if (CAUSAL && rb + 31 < wkey0) continue;  // whole block above the wave's keys
            float mk[kMatrix ? 16 : 1];
            const bool masked = kMatrix && !mask_is_zero(j);
            if constexpr (kMaskViaLds) {
                if (masked) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) mk[i] = qb ? mk2[16 + i] : mk2[i];  // static indices keep it in registers
                }
            } else if constexpr (kMatrix) {
                if (masked) {
                    const int64_t mbase = b * p.ms[0] + hd * p.ms[1] + key_ld;
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const int row = RAGGED ? min(rb + c_row(i, h), p.S - 1) : rb + c_row(i, h);
                        mk[i] = mask_at<T, MASK>(p.mask, mbase + static_cast<int64_t>(row) * p.ms[2]);
                    }
                }
            }
            const int qoff = 32 * qb * Tile::kRowBytes;
            u32x4 fr[KK];
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) fr[kk] = lds_read16(sQ, (row_off0 ^ (kk << 5)) + qoff);
            __builtin_amdgcn_sched_barrier(0);
            f32x16 s = zero16(), dp = zero16();
            if constexpr (kDeltaInAcc) {
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const f32x4 d4 = *reinterpret_cast<const f32x4*>(sDelta + 32 * qb + 8 * g + 4 * h);
                    dp[4 * g + 0] = d4.x; dp[4 * g + 1] = d4.y; dp[4 * g + 2] = d4.z; dp[4 * g + 3] = d4.w;
                }
            }
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) {
                s = Mma<T>::run(fr[kk], kf[kk], s);
                fr[kk] = lds_read16(sG, (row_off0 ^ (kk << 5)) + qoff);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) dp = Mma<T>::run(fr[kk], vf[kk], dp);
            __builtin_amdgcn_sched_barrier(0);
            if (diag && rb < wkey0 + 31) {  // a block that crosses the diagonal: scores above it drop out
                asm volatile("");           // (a real branch: the other blocks skip the comparisons)
#pragma unroll
                for (int i = 0; i < 16; ++i) s[i] = key <= rb + c_row(i, h) ? s[i] : -INFINITY;
            }
            if (MASK == kMaskKeys && some_hidden) {
                asm volatile("");
#pragma unroll
                for (int i = 0; i < 16; ++i) s[i] = hidden ? -INFINITY : s[i];
            }
            if (RAGGED && rb + 32 > p.S) {  // query rows that do not exist contribute nothing
#pragma unroll
                for (int i = 0; i < 16; ++i) s[i] = rb + c_row(i, h) < p.S ? s[i] : -INFINITY;
            }
            u32x4 pb[2], sb[2];
            {
                float pr[16], ds[16];
                // the probabilities first: with the mask's values, or as in a tile without a mask where they are all zero
                float pexp[16];
                if (masked) {
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const f32x4 l4 = *reinterpret_cast<const f32x4*>(sLse + 32 * qb + 8 * g + 4 * h);
#pragma unroll
                        for (int bb = 0; bb < 4; ++bb) {  // (a padded mask joins its score behind the scale, as in the forward)
                            const int i = 4 * g + bb;
                            pexp[i] = RAGGED ? fast_exp2(fmaf(s[i], c, mk[i] * kLog2e) - l4[bb]) : fast_exp2(fmaf(fmaf(mk[i], inv_scale, s[i]), c, -l4[bb]));
                        }
                    }
                } else {
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const f32x4 l4 = *reinterpret_cast<const f32x4*>(sLse + 32 * qb + 8 * g + 4 * h);
#pragma unroll
                        for (int bb = 0; bb < 4; ++bb) pexp[4 * g + bb] = fast_exp2(fmaf(s[4 * g + bb], c, -l4[bb]));
                    }
                }
                uint32_t w[4];  // (this lane's share of the quad's four blocks: rows rb + 8 (lane % 4) + 4 h .. +3)
                if constexpr (DROPOUT) DropoutKeys::words(drop.block(p, (rb + 8 * (lane & 3) + 4 * h) >> 2), w);
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    f32x4 d4 = {0.f, 0.f, 0.f, 0.f};
                    if constexpr (!kDeltaInAcc) d4 = *reinterpret_cast<const f32x4*>(sDelta + 32 * qb + 8 * g + 4 * h);
#pragma unroll
                    for (int bb = 0; bb < 4; ++bb) {
                        const int i = 4 * g + bb;
                        const float pv = pexp[i];
                        float dpv = dp[i];
                        if constexpr (DROPOUT) {
                            const bool keep = static_cast<int>((w[g] >> (8 * bb)) & 0xffu) >= p.thr8;
                            dpv = keep ? dpv : 0.f;
                            pr[i] = keep ? pv : 0.f;  // (the 1 / (1 - p) factor: at the end)
                        } else {
                            pr[i] = pv;
                        }
                        ds[i] = kDeltaInAcc ? pv * dpv : pv * fmaf(dpv, p.zscale, -d4[bb]);
                    }
                }
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    pb[g] = pack8<T>(&pr[8 * g]);
                    sb[g] = pack8<T>(&ds[8 * g]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            // dV^T += dO^T P, then dK^T += Q^T dS; DB transposed fragments in flight
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                u32x4 tf[DB];
#pragma unroll
                for (int db = 0; db < DB; ++db) tf[db] = Tile::tr_frag(sG, tr_off0 ^ (db << 6), tr_off1 ^ (db << 6), 2 * qb + g);
#pragma unroll
                for (int db = 0; db < DB; ++db) {
                    dv[db] = Mma<T>::run(tf[db], pb[g], dv[db]);
                    tf[db] = Tile::tr_frag(sQ, tr_off0 ^ (db << 6), tr_off1 ^ (db << 6), 2 * qb + g);
                }
#pragma unroll
                for (int db = 0; db < DB; ++db) dk[db] = Mma<T>::run(tf[db], sb[g], dk[db]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }

    constexpr bool kLeftOut = RAGGED && MASK != kNoMask;
    if constexpr (SPLIT) {
        if (part.count > 1) {
            float* const sums = p.partial + (static_cast<int64_t>(part.unit) * 2 * kKeys + 32 * wave) * D;
            store_partial<DB, D>(dk, sums, 0, lane, (kDeltaInAcc ? -1.f : 1.f) * (kLeftOut ? left_out : 1.f));
            store_partial<DB, D>(dv, sums + static_cast<int64_t>(kKeys) * D, 0, lane, (DROPOUT ? p.zscale : 1.f) * (kLeftOut ? left_out : 1.f));
            return;
        }
    }
    // every wave is out of the loop: the ring can serve as the waves' private transposition patches
    lds_barrier();
    {
        using Store = RowBlockStore<T, DB, D < 32 ? D : 32 * DB>;
        static_assert(NW * Store::kPatchBytes <= kStages * kStageBytes, "patches must fit into the ring");
        char* patch = smem + wave * Store::kPatchBytes;
        char* dk0 = static_cast<char*>(p.dk) + (b * p.dks[0] + hd * p.dks[1] + static_cast<int64_t>(wkey0) * p.dks[2]) * 2;
        char* dv0 = static_cast<char*>(p.dv) + (b * p.dvs[0] + hd * p.dvs[1] + static_cast<int64_t>(wkey0) * p.dvs[2]) * 2;
        const float sc = (kDeltaInAcc ? -p.scale : p.scale) * (kLeftOut ? left_out : 1.f);
        const int keys_here = RAGGED ? p.S - wkey0 : 32;
        Store::run(dk, [sc](float x) { return x * sc; }, patch, dk0, p.dks[2] * 2, lane, keys_here);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // patch read before it is rewritten
        const float dv_sc = (DROPOUT ? p.zscale : 1.f) * (kLeftOut ? left_out : 1.f);
        Store::run(dv, [dv_sc](float x) { return DROPOUT || kLeftOut ? x * dv_sc : x; }, patch, dv0, p.dvs[2] * 2, lane, keys_here);
    }
}

// ------------------------------------------------------------------ dK, dV (paired waves)
// For D = 128 the K and V rows plus both gradient accumulators of a 32-key block need 192
// registers, which rules out two waves per SIMD. Here two waves share a key block instead: a
// workgroup of 8 waves owns 128 keys; waves w and w+4 both hold the K and V rows of key block w%4.
// Per 64-row tile of Q and dO (swizzled LDS ring filled by LDS-direct loads, as in the dQ kernel)
//   score step:        member m of a pair computes S, dP, P and dS of query block m (16 MFMA +
//                      softmax) and leaves P and dS, already packed as B operands, in an LDS slot;
//   accumulation step: each member accumulates, for BOTH query blocks, the half of the head
//                      dimension it owns: dV^T[2m..2m+1] += dO^T P, dK^T[2m..2m+1] += Q^T dS (16 MFMA).
// No MFMA is executed twice, and a wave keeps only 128 persistent registers.
template <typename T, int D, bool CAUSAL, int MASK, bool DROPOUT>
__global__ __launch_bounds__(512, 2) void mfma_dkdv_pair_kernel(const KParams p) {
    using Tile = SwzTile<D>;
    constexpr int NW = 8;
    constexpr int kKeys = 128;
    constexpr int kStages = 3;
    constexpr int kStageBytes = 2 * Tile::kBytes + 2 * kBN * 4;  // Q tile, dO tile, lse, delta
    constexpr int kXchBytes = NW * 4 * 1024;                     // per wave: P[2], dS[2] fragments
    constexpr int KK = D / 16;
    constexpr int DB = D / 32;
    constexpr int DH = DB / 2;                                   // column blocks a pair member accumulates
    constexpr int kBlocksPerWave = 2 * Tile::kBlocks / NW;
    constexpr int kLoadsPerTile = kBlocksPerWave + 1;            // + lse or delta: exact for every wave
    __shared__ __attribute__((aligned(1024))) char smem[kStages * kStageBytes + kXchBytes];
    char* xch = smem + kStages * kStageBytes;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kb = wave & 3, member = wave >> 2;
    const int lane = tid & 63, l32 = lane & 31, h = lane >> 5;
    int bh, kt;
    map_block_for<MASK>(p, blockIdx.x, p.S / kKeys, CAUSAL ? kHeavyFirst : kUniformTiles, &bh, &kt);
    const int b = bh / p.H, hd = bh % p.H;
    const int k0 = kt * kKeys;
    const int wkey0 = k0 + 32 * kb;
    const int key = wkey0 + l32;

    const char* kbase = static_cast<const char*>(p.k) + (b * p.ks[0] + hd * p.ks[1]) * 2;
    const char* vbase = static_cast<const char*>(p.v) + (b * p.vs[0] + hd * p.vs[1]) * 2;
    const char* qbase = static_cast<const char*>(p.q) + (b * p.qs[0] + hd * p.qs[1]) * 2;
    const char* gbase = static_cast<const char*>(p.d_o) + (b * p.dos[0] + hd * p.dos[1]) * 2;
    const int64_t qrow_bytes = p.qs[2] * 2, grow_bytes = p.dos[2] * 2;
    const float* lse_base = p.lse + static_cast<int64_t>(bh) * p.S;
    const float* delta_base = p.delta + static_cast<int64_t>(bh) * p.S;

    const float c = p.scale_log2;
    [[maybe_unused]] const float inv_scale = p.inv_scale;  // (a mask value joins its score before the scale: s + mask / scale)

    f32x16 dk[DH], dv[DH];
#pragma unroll
    for (int d = 0; d < DH; ++d) {
        dk[d] = zero16();
        dv[d] = zero16();
    }

    int src_off[kBlocksPerWave];
#pragma unroll
    for (int i = 0; i < kBlocksPerWave; ++i) {
        const int blk = wave * kBlocksPerWave + i;
        const bool is_g = blk >= Tile::kBlocks;
        src_off[i] = static_cast<int>(Tile::src_off(is_g ? blk - Tile::kBlocks : blk, lane, is_g ? grow_bytes : qrow_bytes));
    }
    const int t_begin = CAUSAL ? k0 / kBN : 0;
    const int n_tiles = p.S / kBN;
    auto issue_tile = [&](int t) {
        char* stage = smem + ((t - t_begin) % kStages) * kStageBytes;  // slots count from the first tile
#pragma unroll
        for (int i = 0; i < kBlocksPerWave; ++i) {
            const int blk = wave * kBlocksPerWave + i;
            const bool is_g = blk >= Tile::kBlocks;
            const char* tile_src = is_g ? gbase + static_cast<int64_t>(t) * kBN * grow_bytes
                                        : qbase + static_cast<int64_t>(t) * kBN * qrow_bytes;
            char* dst = stage + (is_g ? Tile::kBytes + (blk - Tile::kBlocks) * 1024 : blk * 1024);
            lds_direct_load16(tile_src, src_off[i], dst);
        }
        // every wave issues exactly one more load, so that the vmcnt bookkeeping is the same in all of
        // them: even waves fetch the 64 lse values, odd waves the 64 delta values (duplicates land
        // on the same bytes)
        if (wave & 1) lds_direct_load4(delta_base + t * kBN, lane * 4, stage + 2 * Tile::kBytes + kBN * 4);
        else lds_direct_load4(lse_base + t * kBN, lane * 4, stage + 2 * Tile::kBytes);
    };
    // The K and V rows of the workgroup (128 keys = two 64-row tiles each) also arrive through LDS:
    // lanes own keys, so loading the fragments straight into registers would touch 32 cache lines
    // per instruction (measured: 4.5 us of a 95 us workgroup), while LDS-direct loads fetch whole rows.
    // They land in the third ring slot plus the exchange slots, which nobody uses before the loop.
    char* kv_lds = smem + 2 * kStageBytes;
    static_assert(kStageBytes + kXchBytes >= 4 * Tile::kBytes, "K and V must fit behind the first two ring slots");
    static_assert(4 * Tile::kBlocks % NW == 0, "K/V blocks must divide among the waves");
    constexpr int kKvLoads = 4 * Tile::kBlocks / NW;
    {
        const int64_t krow_bytes = p.ks[2] * 2, vrow_bytes = p.vs[2] * 2;
#pragma unroll
        for (int i = 0; i < kKvLoads; ++i) {
            const int blk = wave * kKvLoads + i;           // 0 .. 4*kBlocks-1: K tile 0, K tile 1, V tile 0, V tile 1
            const int tile = blk / Tile::kBlocks, b16 = blk % Tile::kBlocks;
            const bool is_v = tile >= 2;
            const int64_t rb = is_v ? vrow_bytes : krow_bytes;
            const char* src = (is_v ? vbase : kbase) + (k0 + 64 * (tile & 1)) * rb;
            lds_direct_load16(src, static_cast<uint32_t>(Tile::src_off(b16, lane, rb)), kv_lds + blk * 1024);
        }
    }
    issue_tile(t_begin);
    if (t_begin + 1 < n_tiles) issue_tile(t_begin + 1);

    const int row_off0 = Tile::off(l32, h);
    const int tr_off0 = Tile::tr_off(0, 0, lane), tr_off1 = Tile::tr_off(0, 1, lane);
    // K and V have landed (the Q/dO tiles issued after them may still be in flight)
    if (t_begin + 1 < n_tiles) TRI_WAIT_VMCNT(2 * kLoadsPerTile);
    else TRI_WAIT_VMCNT(kLoadsPerTile);
    lds_barrier();
    u32x4 kf[KK], vf[KK];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
        const int off = (row_off0 ^ (kk << 5)) + 32 * (kb & 1) * Tile::kRowBytes;
        kf[kk] = lds_read16(kv_lds + (kb >> 1) * Tile::kBytes, off);
        vf[kk] = lds_read16(kv_lds + (2 + (kb >> 1)) * Tile::kBytes, off);
    }
    lds_barrier();  // every wave has its fragments: the region is free for the exchange slots and tile 2
    char* my_xch = xch + wave * 4096 + lane * 16;
    const char* peer_xch = xch + (wave ^ 4) * 4096 + lane * 16;

    // The two members of a pair sit on the same SIMD and run half a tile apart, so that one is in
    // its score phase (softmax arithmetic) while the other is in its accumulation phase (MFMA only).
    // Half-step hs: member 0 scores tile hs/2 on even steps, member 1 on odd steps; a wave publishes
    // its P and dS at the start of its next accumulation step, so a slot is never rewritten before
    // the barrier after the partner's read. Member 1 accumulates tile t on step 2t+2, member 0 on
    // step 2t+3; by then it has scored tile t+1, so it takes its own P and dS of tile t back from
    // its slot just before it overwrites them.
    const int n_local = n_tiles - t_begin;
    [[maybe_unused]] DropoutKeys drop;
    if constexpr (DROPOUT) drop.init(p, bh, key >> 2);
    u32x4 cur_p[2], cur_s[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        cur_p[g] = cur_s[g] = u32x4{0, 0, 0, 0};
        *reinterpret_cast<u32x4*>(my_xch + g * 1024) = cur_p[g];
        *reinterpret_cast<u32x4*>(my_xch + (2 + g) * 1024) = cur_s[g];
    }

    // even half-step 2*lt: tile lt must have landed; tile lt+1 is the only other one that can be in
    // flight. After the barrier every wave is done with tile lt-2, whose slot tile lt+1 takes.
    auto open_even_step = [&](int lt) {
        if (lt == 0 && n_local > 1) TRI_WAIT_VMCNT(kLoadsPerTile);
        else TRI_WAIT_VMCNT(0);
        lds_barrier();
    };
    // (after the barrier every wave is done with tile lt-2, whose slot tile lt+1 takes; a member issues
    // its share of the loads at the start of its accumulation step, the part of a tile in which it
    // would otherwise only wait: a load instruction holds the wave until the memory pipeline takes it)
    auto issue_next = [&](int lt) {
        if (lt >= 1 && lt + 1 < n_local) issue_tile(t_begin + lt + 1);
    };
    // A step is split once more, so that the matrix pipe and the vector ALU of the SIMD are both busy:
    //   first part:  the scoring member runs its 16 MFMAs (S and dP); the accumulating member exchanges
    //                P and dS through the LDS slots and requests its first fragments;
    //   second part: the scoring member does the softmax arithmetic; the accumulating member runs its
    //                16 MFMAs.
    // (Both members issuing MFMAs at once, and the arithmetic afterwards with an idle matrix pipe, cost
    // more than twice the time.) part_barrier() separates the parts; it does not wait for LDS reads in
    // flight, which the second part consumes.
    auto part_barrier = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    // The state a step carries from its first part to its second. Every variable is assigned in every
    // first part (zeros on the idle paths), so that none of them stays live around the loop.
    f32x16 sc_s, sc_dp;                      // scores
    f32x4 sc_lse[4];                         // lse of this lane's 16 rows
    // (fetching delta ahead like lse, and deeper fragment rings, were measured: no gain)
    constexpr bool kRoomy = false;
    f32x4 sc_dlt[kRoomy ? 4 : 1];            // delta of the same rows
    float sc_mk[MASK != kNoMask ? 16 : 1];   // mask values of the same rows at this lane's key
    const uint32_t mask_lane_off = MASK == kMaskF32 ? static_cast<uint32_t>((4 * h * p.ms[2] + key) * 4) : 0u;
    u32x4 own_p[2], own_s[2], pp[2], ps[2];  // B operands of the accumulation
    constexpr int kAccSteps = 8 * DH, kAccRing = 4;
    u32x4 tf[kAccRing];                      // first transposed fragments of the accumulation
    // score step, first part: S and dP of query block `member` of local tile lt against this pair's keys
    auto score_mfma = [&](int lt) {
        const int j = t_begin + lt;
        const int rb = j * kBN + 32 * member;
        const char* sQ = smem + ((lt < n_local ? lt : 0) % kStages) * kStageBytes;
        const char* sG = sQ + Tile::kBytes;
        const float* sLse = reinterpret_cast<const float*>(sG + Tile::kBytes);
        if (lt < n_local && (!CAUSAL || rb + 31 >= wkey0)) {
            if constexpr (MASK != kNoMask) {
                // requested before anything else of the step and used in its second part: the loads' latency, which
                // used to stand in front of every block's arithmetic, passes behind the MFMAs and the barrier between
                // the parts (a row of the block is 128 contiguous bytes across the lanes of a half wave). Requesting
                // them a whole accumulation step earlier measured no better.
                if constexpr (MASK == kMaskF32) {
                    // (row rb + 8 g + 4 h + bb: a uniform 64-bit base per (g, bb), scalar arithmetic, plus one 32-bit
                    // offset per lane that does not change over the kernel: the row stride is below 2^24 elements.
                    // The 16-bit loads take the plain form: with this one they measured 2.4 times slower.)
                    const char* ubase = static_cast<const char*>(p.mask) + (b * p.ms[0] + hd * p.ms[1] + static_cast<int64_t>(rb) * p.ms[2]) * 4;
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        sc_mk[i] = *reinterpret_cast<const float*>(ubase + static_cast<int64_t>(8 * (i >> 2) + (i & 3)) * p.ms[2] * 4 + mask_lane_off);
                } else {
                    const int64_t mbase = b * p.ms[0] + hd * p.ms[1] + key;
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        sc_mk[i] = mask_at<T, MASK>(p.mask, mbase + static_cast<int64_t>(rb + c_row(i, h)) * p.ms[2]);
                }
            }
            const int qoff = 32 * member * Tile::kRowBytes;
            // row fragments of Q, then of dO, through a ring of kRing reads in flight
            constexpr int kRing = 4;
            auto row_frag = [&](int n) {
                return lds_read16(n < KK ? sQ : sG, (row_off0 ^ ((n % KK) << 5)) + qoff);
            };
            u32x4 fr[kRing];
#pragma unroll
            for (int n = 0; n < kRing; ++n) fr[n] = row_frag(n);
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(2);
            f32x16 s = zero16(), dp = zero16();
#pragma unroll
            for (int n = 0; n < 2 * KK; ++n) {
                if (n < KK) s = Mma<T>::run(fr[n % kRing], kf[n], s);
                else dp = Mma<T>::run(fr[n % kRing], vf[n - KK], dp);
                if (n + kRing < 2 * KK) fr[n % kRing] = row_frag(n + kRing);
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_s_setprio(0);
            sc_s = s;
            sc_dp = dp;
        } else {
            sc_s = zero16();
            sc_dp = zero16();
        }
        // requested now, used in the second part (harmless where the step is idle)
#pragma unroll
        for (int g = 0; g < 4; ++g) sc_lse[g] = *reinterpret_cast<const f32x4*>(sLse + 32 * member + 8 * g + 4 * h);
        if constexpr (kRoomy) {
#pragma unroll
            for (int g = 0; g < 4; ++g) sc_dlt[g] = *reinterpret_cast<const f32x4*>(sLse + kBN + 32 * member + 8 * g + 4 * h);
        }
    };
    // score step, second part: P and dS from the scores, packed as B operands
    auto score_valu = [&](int lt) {
        const int j = t_begin + lt;
        const int rb = j * kBN + 32 * member;
        if (lt < n_local && (!CAUSAL || rb + 31 >= wkey0)) {
            const char* sQ = smem + (lt % kStages) * kStageBytes;
            const char* sG = sQ + Tile::kBytes;
            const float* sDelta = reinterpret_cast<const float*>(sG + Tile::kBytes) + kBN;
            f32x16 s = sc_s;
            const f32x16 dp = sc_dp;
            if (CAUSAL && rb < wkey0 + 31) {  // a block that crosses the diagonal: scores above it drop out
                asm volatile("");             // (a real branch: the other blocks skip the comparisons)
#pragma unroll
                for (int i = 0; i < 16; ++i) s[i] = key <= rb + c_row(i, h) ? s[i] : -INFINITY;
            }
            float mk[MASK != kNoMask ? 16 : 1];
            if constexpr (MASK != kNoMask) {
#pragma unroll
                for (int i = 0; i < 16; ++i) mk[i] = sc_mk[i];
            }
            uint32_t w[4];  // (this lane's share of the quad's four blocks: rows rb + 8 (lane % 4) + 4 h .. +3)
            if constexpr (DROPOUT) DropoutKeys::words(drop.block(p, (rb + 8 * (lane & 3) + 4 * h) >> 2), w);
#pragma unroll
            for (int gg = 0; gg < 2; ++gg) {  // eight rows at a time, packed as soon as they are done
                float pr[8], ds[8];
                f32x4 dlt4[2];
#pragma unroll
                for (int g2 = 0; g2 < 2; ++g2) {
                    if constexpr (kRoomy) dlt4[g2] = sc_dlt[2 * gg + g2];
                    else dlt4[g2] = *reinterpret_cast<const f32x4*>(sDelta + 32 * member + 8 * (2 * gg + g2) + 4 * h);
                }
#pragma unroll
                for (int g2 = 0; g2 < 2; ++g2) {
                    const int g = 2 * gg + g2;
                    f32x4 l4 = sc_lse[g];
                    const f32x4 d4 = dlt4[g2];
#pragma unroll
                    for (int bb = 0; bb < 4; ++bb) {
                        const int i = 4 * g + bb;
                        float pv;
                        if constexpr (MASK != kNoMask) pv = fast_exp2(fmaf(fmaf(mk[i], inv_scale, s[i]), c, -l4[bb]));
                        else pv = fast_exp2(fmaf(s[i], c, -l4[bb]));
                        float dpv = dp[i];
                        if constexpr (DROPOUT) {
                            const bool keep = static_cast<int>((w[g] >> (8 * bb)) & 0xffu) >= p.thr8;
                            dpv = keep ? dpv : 0.f;
                            pr[4 * g2 + bb] = keep ? pv : 0.f;  // (the 1 / (1 - p) factor: at the end)
                        } else {
                            pr[4 * g2 + bb] = pv;
                        }
                        ds[4 * g2 + bb] = pv * (DROPOUT ? fmaf(dpv, p.zscale, -d4[bb]) : dpv - d4[bb]);
                    }
                }
                cur_p[gg] = pack8<T>(pr);
                cur_s[gg] = pack8<T>(ds);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
#pragma unroll
            for (int g = 0; g < 2; ++g) cur_p[g] = cur_s[g] = u32x4{0, 0, 0, 0};
        }
    };
    // accumulation step, first part: publish the latest scores, fetch the partner's and the first
    // transposed fragments. Second part: add local tile lt to this member's half of the head dimension
    // for both query blocks: 8 DH MFMAs in the order (query block, K-step, dV^T or dK^T, column block),
    // their A operands through one ring of fragments.
    auto acc_frag = [&](int lt, int n) {
        const char* sQ = smem + (lt % kStages) * kStageBytes;
        const char* sG = sQ + Tile::kBytes;
        const int d = n % DH, which = (n / DH) % 2, g = (n / (2 * DH)) % 2, qb = n / (4 * DH);
        const int db = DH * member + d;
        return Tile::tr_frag(which ? sQ : sG, tr_off0 ^ (db << 6), tr_off1 ^ (db << 6), 2 * qb + g);
    };
    auto acc_on = [&](int lt) {
        return lt >= 0 && lt < n_local && (!CAUSAL || (t_begin + lt) * kBN + kBN - 1 >= wkey0);
    };
    auto acc_prep = [&](int lt) {
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            if (member == 0) {  // LDS operations of one wave complete in order: read, then overwrite
                own_p[g] = *reinterpret_cast<const u32x4*>(my_xch + g * 1024);
                own_s[g] = *reinterpret_cast<const u32x4*>(my_xch + (2 + g) * 1024);
            } else {
                own_p[g] = cur_p[g];
                own_s[g] = cur_s[g];
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            *reinterpret_cast<u32x4*>(my_xch + g * 1024) = cur_p[g];
            *reinterpret_cast<u32x4*>(my_xch + (2 + g) * 1024) = cur_s[g];
        }
        // (unconditional reads: harmless where the step is idle)
#pragma unroll
        for (int g = 0; g < 2; ++g) {  // the partner's P and dS
            pp[g] = *reinterpret_cast<const u32x4*>(peer_xch + g * 1024);
            ps[g] = *reinterpret_cast<const u32x4*>(peer_xch + (2 + g) * 1024);
        }
        const int lt_safe = lt >= 0 && lt < n_local ? lt : 0;
#pragma unroll
        for (int n = 0; n < kAccRing; ++n) tf[n] = acc_frag(lt_safe, n);
    };
    auto acc_mfma = [&](int lt) {
        if (acc_on(lt)) {
            __builtin_amdgcn_s_setprio(2);
#pragma unroll
            for (int n = 0; n < kAccSteps; ++n) {
                const int d = n % DH, which = (n / DH) % 2, g = (n / (2 * DH)) % 2, qb = n / (4 * DH);
                if (which == 0) dv[d] = Mma<T>::run(tf[n % kAccRing], qb == member ? own_p[g] : pp[g], dv[d]);
                else dk[d] = Mma<T>::run(tf[n % kAccRing], qb == member ? own_s[g] : ps[g], dk[d]);
                if (n + kAccRing < kAccSteps) tf[n % kAccRing] = acc_frag(lt, n + kAccRing);
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_s_setprio(0);
        }
    };

    if (member == 0) {
#pragma unroll 1
        for (int lt = 0; lt <= n_local; ++lt) {
            open_even_step(lt);
            score_mfma(lt);
            part_barrier();
            score_valu(lt);
            lds_barrier();
            issue_next(lt);  // in the part where this member only waits for the partner's MFMAs
            acc_prep(lt - 1);
            part_barrier();
            acc_mfma(lt - 1);
        }
    } else {
#pragma unroll 1
        for (int lt = 0; lt <= n_local; ++lt) {
            open_even_step(lt);
            issue_next(lt);
            acc_prep(lt - 1);
            part_barrier();
            acc_mfma(lt - 1);
            lds_barrier();
            score_mfma(lt);
            part_barrier();
            score_valu(lt);
        }
    }

    // every wave is out of the loop: the ring can serve as the waves' private transposition patches
    lds_barrier();
    {
        using Store = RowBlockStore<T, DH>;
        static_assert(NW * Store::kPatchBytes <= kStages * kStageBytes, "patches must fit into the ring");
        char* patch = smem + wave * Store::kPatchBytes;
        const int64_t row = wkey0;  // first key of this pair; this member writes columns 32*DH*member ..
        char* dk0 = static_cast<char*>(p.dk) + (b * p.dks[0] + hd * p.dks[1] + row * p.dks[2] + 32 * DH * member) * 2;
        char* dv0 = static_cast<char*>(p.dv) + (b * p.dvs[0] + hd * p.dvs[1] + row * p.dvs[2] + 32 * DH * member) * 2;
        const float sc = p.scale;
        // (the lane index taken afresh: the epilogue's per-lane offsets are computed here, not kept across the loop)
        int elane = threadIdx.x & 63;
        asm volatile("" : "+v"(elane));
        Store::run(dk, [sc](float x) { return x * sc; }, patch, dk0, p.dks[2] * 2, elane);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // patch read before it is rewritten
        const float dv_sc = DROPOUT ? p.zscale : 1.f;
        Store::run(dv, [dv_sc](float x) { return DROPOUT ? x * dv_sc : x; }, patch, dv0, p.dvs[2] * 2, elane);
    }
}

// ------------------------------------------------------------------ dK, dV (paired waves, phased; no mask)
// The pairing of the kernel above (waves w and w+4 share key block w%4, each accumulates half of the
// head dimension) with the phase structure of the forward kernel. Q and dO stream as 32-row blocks
// (plus their lse and delta) through a ring of 7 slots; even blocks are scored by member 0, odd
// blocks by member 1, and both members accumulate every block. A member alternates
//   vector phase:  P and dS of its block from S' and dP' (softmax backward), published in its LDS slot;
//                  the partner's latest block is fetched from the partner's slot;
//   matrix phase:  dV^T, dK^T += the partner's latest block and its own (16 MFMAs), then S' = S - lse / c
//                  and dP' = dP - delta of its next block (18 MFMAs), through one ring of LDS fragments;
// with a workgroup barrier after each phase, member 1 one phase behind member 0: a SIMD always has one
// wave on the matrix pipe and one on the vector ALU. Block r is first read in phase r-1 and last in
// phase r+2; in phase ph every wave issues its share of block ph+4 and, before the barrier, waits for
// its share of block ph+2.
// With DROPOUT only -lse / c is folded into the accumulators: dS = P (Z dP - delta) needs delta beside the dropped dP,
// so the vector phase reads its 16 row values from the block's slot, and draws the keep decisions of its block (one
// Philox call per lane, shared inside the quad).
// With KEYMASK (kMaskF32 / kMaskT; never with the causal mask): an additive mask that is the same for every query row
// (row stride 0: a key-padding mask). Lanes own keys here, so the whole mask is one value per lane, read once, and goes
// into the exponent for free (the multiply by the scale becomes a fused multiply-add).
// RAGGED: S is not a multiple of 128. Loads clamp their row index to S - 1, rows at or beyond S get probability 0 (the
// number of blocks is rounded up to an even one, at least four, as the phases assume; blocks wholly beyond S hold the
// last row again and again), keys at or beyond S are not stored.
// SPLIT (with RAGGED): a workgroup streams one part of its item's rows (split.hpp), at least two 64-row tiles unless the sequence
// ends inside it (or before it: blocks of nothing but rows that do not exist).
template <typename T, int D, bool CAUSAL, bool DROPOUT = false, int KEYMASK = kNoMask, bool RAGGED = false, bool SPLIT = false>
__global__ __launch_bounds__(512, 2) void mfma_dkdv_phased_kernel(const KParams p) {
    static_assert(RAGGED || !SPLIT, "parts have boundary handling");
    static_assert(KEYMASK == kNoMask || !CAUSAL, "a mask excludes the causal variant");
    using Tile = SwzTile<D>;
    constexpr int NW = 8;
    constexpr int kKeys = 128;
    constexpr int kBR = 32;                                  // rows per streamed block
    constexpr int kSlots = 7;
    constexpr int kHalfBytes = kBR * Tile::kRowBytes;        // one operand of a block
    constexpr int kSlotBytes = 2 * kHalfBytes + 512;         // Q rows, dO rows, lse, delta (256 B each)
    constexpr int kXchBytes = NW * 4096;                     // per wave: P[2], dS[2] fragments
    constexpr int KK = D / 16;
    constexpr int DB = D / 32;
    constexpr int DH = DB / 2;                               // column blocks a pair member accumulates
    constexpr int kLoads = 5;                                // loads per requesting wave and block
    static_assert(kHalfBytes == NW * 1024, "two Q loads and two dO loads per requesting wave and block");
    constexpr int kAccSteps = 4 * DH;                        // MFMAs that add one block
    constexpr int kSteps = 2 * kAccSteps + 2 * KK;           // matrix phase
    // (one fragment fewer in flight where boundary handling leaves no registers for four)
    constexpr int kRing = RAGGED && !CAUSAL && !DROPOUT && std::is_same<T, f16_t>::value ? 3 : 4;
    __shared__ __attribute__((aligned(1024))) char smem[kSlots * kSlotBytes + kXchBytes];
    char* xch = smem + kSlots * kSlotBytes;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kb = wave & 3, member = wave >> 2;
    const int lane = tid & 63, l32 = lane & 31, h = lane >> 5;
    int bh, kt;
    [[maybe_unused]] Part part{};
    if constexpr (SPLIT) {
        if (!map_part(p, blockIdx.x, gridDim.x, (p.S + kKeys - 1) / kKeys, (p.S + kBN - 1) / kBN, CAUSAL, &part)) return;
        bh = part.bh;
        kt = part.tile;
    } else {
        map_block(blockIdx.x, p.B * p.H, (p.S + kKeys - 1) / kKeys, CAUSAL ? kHeavyFirst : kUniformTiles, &bh, &kt);
    }
    const int b = bh / p.H, hd = bh % p.H;
    const int k0 = kt * kKeys;
    const int wkey0 = k0 + 32 * kb;
    const int key = wkey0 + l32;

    const char* kbase = static_cast<const char*>(p.k) + (b * p.ks[0] + hd * p.ks[1]) * 2;
    const char* vbase = static_cast<const char*>(p.v) + (b * p.vs[0] + hd * p.vs[1]) * 2;
    const char* qbase = static_cast<const char*>(p.q) + (b * p.qs[0] + hd * p.qs[1]) * 2;
    const char* gbase = static_cast<const char*>(p.d_o) + (b * p.dos[0] + hd * p.dos[1]) * 2;
    const int64_t qrow_bytes = p.qs[2] * 2, grow_bytes = p.dos[2] * 2;
    const float* lse_base = p.lse + static_cast<int64_t>(bh) * p.S;
    const float* delta_base = p.delta + static_cast<int64_t>(bh) * p.S;
    const float c = p.scale_log2;
    [[maybe_unused]] const float inv_scale = p.inv_scale;  // (a mask value joins its score before the scale: s + mask / scale)
    float key_bias = 0.f;  // mask value of this lane's key, log2 domain
    if constexpr (KEYMASK != kNoMask) key_bias = mask_at<T, KEYMASK>(p.mask, b * p.ms[0] + hd * p.ms[1] + (RAGGED ? min(key, p.S - 1) : key)) * kLog2e;

    f32x16 dk[DH], dv[DH];
#pragma unroll
    for (int d = 0; d < DH; ++d) {
        dk[d] = zero16();
        dv[d] = zero16();
    }

    const int row_first = (CAUSAL ? k0 : 0) + (SPLIT ? part.index * p.part_tiles * kBN : 0);          // first streamed row (block 0)
    const int rows_left = SPLIT ? min(p.S - row_first, p.part_tiles * kBN) : p.S - row_first;
    const int n_blocks = RAGGED ? max(4, (rows_left + 2 * kBR - 1) / (2 * kBR) * 2) : rows_left / kBR;   // >= 4, even
    const int first_on = SPLIT && part.index > 0 ? -1 : kb;  // causal: block on the diagonal, before which this pair has nothing (-1: none)
    // A block is requested by the four waves of ONE member, the one that is in its vector phase when the request is
    // due (member 0 the even blocks, member 1 the odd ones): a vector-memory instruction holds its wave until the
    // memory pipeline has taken it, which the matrix phase cannot afford. Wave kb of the member fetches the 1 KiB
    // pieces kb and kb + 4 of the Q rows and of the dO rows (rows 16 apart share the swizzle, so one per-lane offset
    // serves both) and the block's 32 lse (kb even) or delta (kb odd) values; lanes 32-63 repeat those. The source
    // pointers and the ring slot advance by two blocks per call.
    const uint32_t qoff = static_cast<uint32_t>(Tile::src_off(kb, lane, qrow_bytes));
    const uint32_t goff = static_cast<uint32_t>(Tile::src_off(kb, lane, grow_bytes));
    int next_block = member, next_slot = member;
    const char* next_q = qbase + (row_first + member * kBR) * qrow_bytes;
    const char* next_g = gbase + (row_first + member * kBR) * grow_bytes;
    const float* next_aux = ((kb & 1) ? delta_base : lse_base) + row_first + member * kBR;
    const int aux_lds = 2 * kHalfBytes + ((kb & 1) ? 256 : 0);
    auto issue_block = [&]() {  // this wave's share of its member's next block, if it exists
        if (next_block < n_blocks) {
            char* slot = smem + next_slot * kSlotBytes;
            const int row0 = row_first + next_block * kBR;
            if (RAGGED && row0 + kBR > p.S) {  // the sequence ends inside this block or before it
                const int from = min(row0, p.S - 1), last = p.S - 1 - from;
                int lane = threadIdx.x & 63;  // (offsets made here, not kept in registers across the loop)
                asm volatile("" : "+v"(lane));
                const char* q_from = qbase + from * qrow_bytes;
                const char* g_from = gbase + from * grow_bytes;
                lds_direct_load16(q_from, Tile::src_off_clamped(kb, lane, qrow_bytes, last), slot + kb * 1024);
                lds_direct_load16(g_from, Tile::src_off_clamped(kb, lane, grow_bytes, last), slot + kHalfBytes + kb * 1024);
                lds_direct_load16(q_from, Tile::src_off_clamped(kb + 4, lane, qrow_bytes, last), slot + (kb + 4) * 1024);
                lds_direct_load16(g_from, Tile::src_off_clamped(kb + 4, lane, grow_bytes, last), slot + kHalfBytes + (kb + 4) * 1024);
                lds_direct_load4(((kb & 1) ? delta_base : lse_base) + from, min(lane & 31, last) * 4, slot + aux_lds);
            } else {
                lds_direct_load16(next_q, qoff, slot + kb * 1024);
                lds_direct_load16(next_g, goff, slot + kHalfBytes + kb * 1024);
                lds_direct_load16(next_q + 16 * qrow_bytes, qoff, slot + (kb + 4) * 1024);
                lds_direct_load16(next_g + 16 * grow_bytes, goff, slot + kHalfBytes + (kb + 4) * 1024);
                int aux = threadIdx.x & 31;
                if constexpr (RAGGED) asm volatile("" : "+v"(aux));
                lds_direct_load4(next_aux, aux * 4, slot + aux_lds);
            }
        }
        next_block += 2;
        next_slot = next_slot >= kSlots - 2 ? next_slot + 2 - kSlots : next_slot + 2;
        next_q += 2 * kBR * qrow_bytes;
        next_g += 2 * kBR * grow_bytes;
        next_aux += 2 * kBR;
    };
    // before the barrier that ends vector phase ph of a member: its block ph+2 has landed, its block ph+4 may be in flight
    auto wait_blocks = [&](int ph) {
        if (ph + 4 < n_blocks) TRI_WAIT_VMCNT(kLoads);
        else TRI_WAIT_VMCNT(0);
    };

    // The K and V rows of the workgroup (128 keys = two 64-row tiles each) arrive through LDS too (lanes
    // own keys, so direct loads would touch 32 cache lines per instruction); they land behind the first
    // four ring slots, which take blocks 0-3 meanwhile.
    char* kv_lds = smem + 4 * kSlotBytes;
    static_assert(3 * kSlotBytes + kXchBytes >= 4 * Tile::kBytes, "K and V must fit behind the first four slots");
    constexpr int kKvLoads = 4 * Tile::kBlocks / NW;
    {
        const int64_t krow_bytes = p.ks[2] * 2, vrow_bytes = p.vs[2] * 2;
#pragma unroll
        for (int i = 0; i < kKvLoads; ++i) {
            const int blk = wave * kKvLoads + i;           // 0 .. 4*kBlocks-1: K tile 0, K tile 1, V tile 0, V tile 1
            const int tile = blk / Tile::kBlocks, b16 = blk % Tile::kBlocks;
            const bool is_v = tile >= 2;
            const int64_t rb = is_v ? vrow_bytes : krow_bytes;
            const int row0 = k0 + 64 * (tile & 1), from = RAGGED ? min(row0, p.S - 1) : row0;
            const char* src = (is_v ? vbase : kbase) + from * rb;
            lds_direct_load16(src, RAGGED ? Tile::src_off_clamped(b16, lane, rb, p.S - 1 - from) : static_cast<uint32_t>(Tile::src_off(b16, lane, rb)),
                              kv_lds + blk * 1024);
        }
    }
    issue_block();  // blocks 0 and 2 (member 0), 1 and 3 (member 1)
    issue_block();

    int row_off0 = Tile::off(l32, h);
    int tr_off0 = Tile::tr_off(0, 0, lane), tr_off1 = Tile::tr_off(0, 1, lane);
    // Taken afresh at the head of each member's loop: with every register in use, values computed once up here and
    // needed by only one of the two loops would otherwise be spilled around the other.
    auto refresh_lane_offsets = [&]() {
        int l = lane;
        asm volatile("" : "+v"(l));
        row_off0 = Tile::off(l & 31, l >> 5);
        tr_off0 = Tile::tr_off(0, 0, l);
        tr_off1 = Tile::tr_off(0, 1, l);
    };
    TRI_WAIT_VMCNT(2 * kLoads);  // K and V have landed
    lds_barrier();
    u32x4 kf[KK], vf[KK];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
        const int off = (row_off0 ^ (kk << 5)) + 32 * (kb & 1) * Tile::kRowBytes;
        kf[kk] = lds_read16(kv_lds + (kb >> 1) * Tile::kBytes, off);
        vf[kk] = lds_read16(kv_lds + (2 + (kb >> 1)) * Tile::kBytes, off);
    }
    lds_barrier();  // every wave has its fragments: the region is free for the exchange slots and later blocks
    char* my_xch = xch + wave * 4096 + lane * 16;
    const char* peer_xch = xch + (wave ^ 4) * 4096 + lane * 16;
    u32x4 cur_p[2], cur_s[2];   // P and dS of this member's current block
    u32x4 par_p[2], par_s[2];   // the partner's latest block
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        cur_p[g] = cur_s[g] = par_p[g] = par_s[g] = u32x4{0, 0, 0, 0};
        *reinterpret_cast<u32x4*>(my_xch + g * 1024) = cur_p[g];
        *reinterpret_cast<u32x4*>(my_xch + (2 + g) * 1024) = cur_s[g];
    }
    TRI_WAIT_VMCNT(kLoads);  // blocks 0 and 1 have landed
    lds_barrier();

    // whether this pair has anything in block r (under the causal mask: rows at or below its first key)
    auto block_on = [&](int r) { return r >= 0 && r < n_blocks && (!CAUSAL || r >= first_on); };

    [[maybe_unused]] DropoutKeys drop;
    if constexpr (DROPOUT) drop.init(p, bh, key >> 2);
    constexpr float kFoldUnit = 256.f;  // the constant the first of the split terms multiplies (keeps f16 terms in range)
    const float neg_inv_c = -1.f / c;
    f32x16 sc_s, sc_dp;  // S - lse / c and dP - delta of this member's next block
    u32x4 ring[kRing];
    // Ring slots are named by their byte offset in LDS and stepped from block to block (a slot index taken modulo 7
    // for every block a phase touches costs a dozen scalar instructions each time).
    constexpr int kRingBytes = kSlots * kSlotBytes;
    auto slot_step = [&](int so, int d) {
        int t = so + d * kSlotBytes;
        t = t >= kRingBytes ? t - kRingBytes : t;
        return t < 0 ? t + kRingBytes : t;
    };
    // fragment n of a matrix phase that adds the blocks in slots sa and sb and scores the block in slot ss
    auto frag = [&](int sa, int sb, int ss, int n) {
        if (n < 2 * kAccSteps) {
            const char* slot = smem + (n < kAccSteps ? sa : sb);
            const int m = n % kAccSteps;
            const int d = m % DH, which = (m / DH) % 2, g = m / (2 * DH);
            const int db = DH * member + d;
            return Tile::tr_frag(slot + (which ? 0 : kHalfBytes), tr_off0 ^ (db << 6), tr_off1 ^ (db << 6), g);
        }
        const int m = n - 2 * kAccSteps;
        return lds_read16(smem + ss + (m < KK ? 0 : kHalfBytes), row_off0 ^ ((m % KK) << 5));
    };
    auto matrix_phase = [&](auto with_acc, int sa, int sb, int ss, bool own_on = true, bool score_on = true) {
        constexpr int first = decltype(with_acc)::value ? 0 : 2 * kAccSteps;
        f32x16 s = zero16(), dp = zero16();
        // One more MFMA each puts -lse / c and -delta under S and dP (a row's value split into three 16-bit
        // terms against a column of constants), so that the vector phase needs neither value: P = exp2(c S'),
        // dS = P dP'. Each lane asks for its row's two values at the start of the phase.
        float row_lse = 0.f, row_delta = 0.f;
#pragma unroll
        for (int n = first; n < kSteps; ++n) {
            const int slot = (n - first) % kRing;
            if ((n == kAccSteps && !own_on && !score_on) || (n == 2 * kAccSteps && !score_on)) break;
            if (n == first) {
                const float* sLse = reinterpret_cast<const float*>(smem + ss + 2 * kHalfBytes);
                row_lse = sLse[l32];
                if constexpr (!DROPOUT) row_delta = sLse[64 + l32];
            }
            if (n == 2 * kAccSteps) {
                const u32x4 zero4 = {0, 0, 0, 0};
                const u32x4 al = Split3<T>::terms(row_lse * neg_inv_c * (1.f / kFoldUnit));
                const u32x4 ad = Split3<T>::terms(row_delta * (-1.f / kFoldUnit));
                const u32x4 units = h == 0 ? Split3<T>::units(kFoldUnit) : zero4;
                s = Mma<T>::run(h == 0 ? al : zero4, units, s);
                if constexpr (!DROPOUT) dp = Mma<T>::run(h == 0 ? ad : zero4, units, dp);
            }
            if (n < 2 * kAccSteps) {
                const int m = n % kAccSteps;
                const int d = m % DH, which = (m / DH) % 2, g = m / (2 * DH);
                const bool own = n >= kAccSteps;
                if (which == 0) dv[d] = Mma<T>::run(ring[slot], own ? cur_p[g] : par_p[g], dv[d]);
                else dk[d] = Mma<T>::run(ring[slot], own ? cur_s[g] : par_s[g], dk[d]);
            } else {
                const int m = n - 2 * kAccSteps;
                if (m < KK) s = Mma<T>::run(ring[slot], kf[m], s);
                else dp = Mma<T>::run(ring[slot], vf[m - KK], dp);
            }
            if (n + kRing < kSteps) ring[slot] = frag(sa, sb, ss, n + kRing);
            __builtin_amdgcn_sched_barrier(0);
        }
        sc_s = s;
        sc_dp = dp;
    };
    using Yes = std::integral_constant<bool, true>;
    using No = std::integral_constant<bool, false>;

    // P = exp2(c S') and dS = P dP' of the block whose first row is rb, eight rows at a time, packed as soon as
    // they are done; only the block on the diagonal pays for the causal comparison (scores above it become -inf)
    auto softmax_backward = [&](bool on_diagonal, int rb, int so) {
        if (on_diagonal) {
            // a real branch, taken for one block per workgroup; the row base goes through a scalar register the
            // compiler cannot see through, so that the 16 comparisons are made here and not kept as lane masks
            // across the whole loop
            int rbo = rb;
            asm volatile("" : "+s"(rbo));
#pragma unroll
            for (int i = 0; i < 16; ++i) sc_s[i] = key <= rbo + c_row(i, h) ? sc_s[i] : -INFINITY;
        }
        if (RAGGED && rb + kBR > p.S) {  // rows that do not exist (taken for the last blocks only, as above)
            int left = p.S - rb - 4 * h;
            asm volatile("" : "+v"(left));
#pragma unroll
            for (int i = 0; i < 16; ++i) sc_s[i] = c_row(i, 0) < left ? sc_s[i] : -INFINITY;
        }
        const f32x16 s = sc_s, dp = sc_dp;
        const float* sDelta = reinterpret_cast<const float*>(smem + so + 2 * kHalfBytes) + 64;
        uint32_t w[4];  // (this lane's share of the quad's four blocks: rows rb + 8 (lane % 4) + 4 h .. +3)
        if constexpr (DROPOUT) DropoutKeys::words(drop.block(p, (rb + 8 * (lane & 3) + 4 * h) >> 2), w);
#pragma unroll
        for (int gg = 0; gg < 2; ++gg) {
            float pr[8], ds[8];
#pragma unroll
            for (int g2 = 0; g2 < 2; ++g2) {
                const int g = 2 * gg + g2;
                f32x4 d4 = {0.f, 0.f, 0.f, 0.f};
                if constexpr (DROPOUT) d4 = *reinterpret_cast<const f32x4*>(sDelta + 8 * g + 4 * h);
#pragma unroll
                for (int bb = 0; bb < 4; ++bb) {
                    const int i = 4 * g + bb, j = 4 * g2 + bb;
                    const float pv = KEYMASK != kNoMask ? fast_exp2(fmaf(s[i], c, key_bias)) : fast_exp2(s[i] * c);
                    if constexpr (DROPOUT) {
                        const bool keep = static_cast<int>((w[g] >> (8 * bb)) & 0xffu) >= p.thr8;
                        pr[j] = keep ? pv : 0.f;  // (the 1 / (1 - p) factor: at the end)
                        ds[j] = pv * fmaf(keep ? dp[i] : 0.f, p.zscale, -d4[bb]);
                    } else {
                        pr[j] = pv;
                        ds[j] = pv * dp[i];
                    }
                }
            }
            cur_p[gg] = pack8<T>(pr);
            cur_s[gg] = pack8<T>(ds);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // vector phase for block r (this member's): P and dS from sc_s, sc_dp
    auto vector_phase = [&](int r, int so) {
        if (block_on(r)) {
            const int rb = row_first + r * kBR;
            softmax_backward(CAUSAL && r == first_on, rb, so);
        } else {
            // (the zeros are made inside this branch, where the compiler cannot lift them in front of the test above:
            // lifted, they are sixteen moves in every phase of the loop. The one variant that has no two registers to
            // spare for that keeps the plain assignment.)
            constexpr bool kPlainZeros = std::is_same<T, f16_t>::value && CAUSAL && !DROPOUT;
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                if constexpr (kPlainZeros) {
                    cur_p[g] = cur_s[g] = u32x4{0, 0, 0, 0};
                } else {
                    uint32_t z[8];
#pragma unroll
                    for (int i = 0; i < 8; ++i) asm volatile("v_mov_b32 %0, 0" : "=v"(z[i]));
                    cur_p[g] = u32x4{z[0], z[1], z[2], z[3]};
                    cur_s[g] = u32x4{z[4], z[5], z[6], z[7]};
                }
            }
        }
    };
    // the second half of a vector phase in global phase ph, for a member whose block is r: publish, fetch
    // the partner's block r-1, request the first fragments of the matrix phase, meet the barrier
    // (so: the slot of block r; block r - 1 sits one slot before it, block r + 2 two after; at the ends of the range the
    // neighbour that does not exist is replaced by one that does, its P and dS are zero)
    auto close_vector_phase = [&](int ph, int r, int so) {
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            *reinterpret_cast<u32x4*>(my_xch + g * 1024) = cur_p[g];
            *reinterpret_cast<u32x4*>(my_xch + (2 + g) * 1024) = cur_s[g];
        }
        issue_block();
        asm volatile("" ::: "memory");  // the reads below are issued after the writes above
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            par_p[g] = *reinterpret_cast<const u32x4*>(peer_xch + g * 1024);
            par_s[g] = *reinterpret_cast<const u32x4*>(peer_xch + (2 + g) * 1024);
        }
        const int before = slot_step(so, -1);
        const int sa = r > 0 ? before : so, sb = r < n_blocks ? so : before;
#pragma unroll
        for (int n = 0; n < kRing; ++n) ring[n] = frag(sa, sb, slot_step(so, 2), n);
        // LDS operations of a wave complete in order: once at most the 4 + 2 kRing reads above are
        // outstanding, the slot is published
        static_assert(4 + 2 * kRing <= 15, "lgkmcnt range");
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xC07F | ((4 + 2 * kRing) << 8));
        wait_blocks(ph);
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_barrier" ::: "memory");  // (the reads above stay in flight)
        __builtin_amdgcn_sched_barrier(0);
    };
    auto run_matrix_phase = [&](int r, int so) {
        // (the last rounds have no own block to add and no block r + 2 to score: those steps are left out, except
        // with dropout, where the shorter instruction stream would cost registers the variant does not have)
        __builtin_amdgcn_s_setprio(2);
        const int before = slot_step(so, -1);
        matrix_phase(Yes{}, r > 0 ? before : so, r < n_blocks ? so : before, slot_step(so, 2), DROPOUT || r < n_blocks,
                     DROPOUT || r + 2 < n_blocks);
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
        lds_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };

    // before phase 0: S and dP of each member's first block (member 0: block 0, member 1: block 1)
    {
#pragma unroll
        for (int n = 0; n < kRing; ++n) ring[n] = frag(0, 0, member * kSlotBytes, 2 * kAccSteps + n);
        __builtin_amdgcn_sched_barrier(0);
        matrix_phase(No{}, 0, 0, member * kSlotBytes);
        lds_barrier();
    }
    const int n_iter = n_blocks / 2;
    if (member == 0) {
        refresh_lane_offsets();
        int so = 0;  // slot of block r
#pragma unroll 1
        for (int t = 0; t <= n_iter; ++t) {   // the last round only adds member 1's last block
            const int r = 2 * t;
            vector_phase(r, so);
            close_vector_phase(2 * t, r, so);
            run_matrix_phase(r, so);
            so = slot_step(so, 2);
        }
    } else {
        refresh_lane_offsets();
        lds_barrier();  // (phase 0: member 0 alone)
        int so = kSlotBytes;  // slot of block r
#pragma unroll 1
        for (int t = 0; t < n_iter; ++t) {
            const int r = 2 * t + 1;
            vector_phase(r, so);
            close_vector_phase(2 * t + 1, r, so);
            run_matrix_phase(r, so);
            so = slot_step(so, 2);
        }
        lds_barrier();  // (the last phase: member 0 alone)
    }

    if constexpr (SPLIT) {
        if (part.count > 1) {
            int elane = threadIdx.x & 63;
            asm volatile("" : "+v"(elane));
            float* const sums = p.partial + (static_cast<int64_t>(part.unit) * 2 * kKeys + 32 * kb) * D;
            store_partial<DH, D>(dk, sums, DH * member, elane, 1.f);
            store_partial<DH, D>(dv, sums + static_cast<int64_t>(kKeys) * D, DH * member, elane, DROPOUT ? p.zscale : 1.f);
            return;
        }
    }
    // every wave is out of the loop: the ring can serve as the waves' private transposition patches
    lds_barrier();
    {
        using Store = RowBlockStore<T, DH>;
        static_assert(NW * Store::kPatchBytes <= kSlots * kSlotBytes, "patches must fit into the ring");
        char* patch = smem + wave * Store::kPatchBytes;
        const int64_t row = wkey0;  // first key of this pair; this member writes columns 32*DH*member ..
        char* dk0 = static_cast<char*>(p.dk) + (b * p.dks[0] + hd * p.dks[1] + row * p.dks[2] + 32 * DH * member) * 2;
        char* dv0 = static_cast<char*>(p.dv) + (b * p.dvs[0] + hd * p.dvs[1] + row * p.dvs[2] + 32 * DH * member) * 2;
        const float sc = p.scale;
        // (the lane index taken afresh: the epilogue's per-lane offsets are computed here, not kept across the loop)
        int elane = threadIdx.x & 63;
        asm volatile("" : "+v"(elane));
        Store::run(dk, [sc](float x) { return x * sc; }, patch, dk0, p.dks[2] * 2, elane, RAGGED ? p.S - wkey0 : 32);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // patch read before it is rewritten
        const float dv_sc = DROPOUT ? p.zscale : 1.f;
        Store::run(dv, [dv_sc](float x) { return DROPOUT ? x * dv_sc : x; }, patch, dv0, p.dvs[2] * 2, elane, RAGGED ? p.S - wkey0 : 32);
    }
}

}  // namespace
}  // namespace tri
