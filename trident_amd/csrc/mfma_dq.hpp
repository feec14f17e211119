// dQ pass of the backward on the matrix cores for fp16/bf16, D in {16,32,64,128} (the dK/dV pass: mfma_dkdv.hip;
// together they replace trident/kernel/attention.py:169-339, split in two so that no gradient tile is ever accumulated
// in global memory):
//
//   dQ pass    one workgroup per 256 (128) query rows (a wave owns 32), streaming key tiles of 64:
//              S^T = K Q^T, dP^T = V dO^T, dS^T = P^T * (dP^T - delta), dQ^T += K^T dS^T
//
// The lane index is the query row that owns the accumulators, the stationary operands (Q, dO) stay in registers as
// MFMA B operands, and dS goes from the accumulators of one MFMA to the B operand of the next without leaving registers.
#pragma once
#include <type_traits>

#include "split.hpp"

namespace tri {
namespace {

constexpr int kBN = 64;   // streamed rows per tile

enum MaskKind { kNoMask = 0, kMaskF32 = 1, kMaskT = 2, kMaskKeys = 3 };  // (kMaskKeys: of the operand type, see KeyBits)

template <typename T, int MASK>
__device__ __forceinline__ float mask_at(const void* mask, int64_t off) {
    if constexpr (MASK == kMaskF32) return static_cast<const float*>(mask)[off];
    else return static_cast<float>(static_cast<const T*>(mask)[off]);
}

// ------------------------------------------------------------------------------------ dQ
// A workgroup of NW waves owns 32*NW query rows, one wave 32 of them with its Q and dO rows in
// registers (B operands) and dQ^T in fp32 accumulators; two waves per SIMD. K and V stream as
// 64-key swizzled LDS tiles in a ring of 4 (3, 2: kStages), filled by LDS-direct loads three (two, one)
// tiles ahead (no staging registers, no ds_write). Per 32-key block: S^T = K Q^T and dP^T = V dO^T from row
// fragments, dS^T = P^T (dP^T - delta) on the vector ALU, dQ^T += K^T dS^T with K^T read through
// transposed LDS reads of the same K tile.
// RAGGED (no mask, or a padded one; no mask gradient): S is not a multiple of 32 NW. Rows and keys at or beyond S do not exist: loads clamp
// their row index to S - 1, keys >= S get probability 0, rows >= S are not stored.
// DMASK (with a mask): the kernel also writes the mask gradient dS (trident/kernel/attention.py:332-335), each lane four
// consecutive keys of its row at a time; where the mask is broadcast over a dimension (dmask stride 0) the values are
// added to the caller's zero-filled fp32 buffer with atomic adds instead.
// DELTA (no mask, or D <= 64 without a mask gradient): the kernel also computes delta = rowsum(dO * O) of its rows from the dO rows it loads anyway, instead
// of reading it, and stores it for the dK/dV pass, which then runs after this one (tri_attn_bwd_dq_delta).
// SPLIT (with RAGGED): a workgroup streams one part of its item's tiles (split.hpp). Tiles count from the part's first one, keys from
// key0; the first part stores delta. Parts beside a mask at D = 16 are held to 168 registers: at 169, with two workgroups per CU instead
// of three, they took a quarter longer (bf16 key mask, 4 heads, S=10368, with the second launch: 77 -> 96 us).
// THREE (D = 64, no mask, 4 waves): three workgroups to a CU instead of two (three_workgroups_per_cu).
template <typename T, int D, int NW, bool CAUSAL, int MASK, bool DROPOUT, bool RAGGED = false, bool DMASK = false, bool DELTA = false,
          bool SPLIT = false, bool THREE = false>
__global__ __launch_bounds__(NW * 64, D == 128 && NW == 4 && RAGGED && (MASK != kNoMask || SPLIT) ? 1 : THREE || D == 16 && SPLIT && MASK != kNoMask ? 3 : 2) void mfma_dq_kernel(const KParams p) {
    static_assert(RAGGED || !SPLIT, "parts have boundary handling");
    static_assert(!RAGGED || !DMASK, "ragged lengths: no mask gradient");
    static_assert(!DMASK || MASK != 0, "a mask gradient needs a mask");
    static_assert(!THREE || (D == 64 && NW == 4 && (MASK == kNoMask || MASK == kMaskKeys) && !SPLIT), "three workgroups per CU");
    constexpr bool kMatrix = MASK == kMaskF32 || MASK == kMaskT;  // a mask whose values are read tile by tile
    static_assert(!DELTA || MASK == 0 || (D <= 64 && !DMASK), "delta on the way: no mask, or a small head without a mask gradient");
    using Tile = SwzTile<D>;
    constexpr int kRows = 32 * NW;
    // Without a mask the workgroups of four waves at D = 128 run two to a CU: a ring of two tiles in half of the LDS, and half of the registers.
    // One alone, with a ring of four and all registers, leaves a wave per SIMD (time of the two over its: 0.72-0.78 at S <= 128; causal with
    // dropout 40 heads x 1000 48.7 -> 40.4 us).
    constexpr bool kPair = D == 128 && NW == 4 && MASK == kNoMask && !SPLIT;
    constexpr int kStages = kPair ? 2 : THREE || (MASK == kMaskF32 && D == 64 && NW == 4) ? 3 : 4;
    constexpr int kAhead = kStages - 1;  // tile j + kAhead is requested in tile j, into the slot of tile j - 1
    constexpr int kStageBytes = 2 * Tile::kBytes;  // K tile, V tile
    constexpr int KK = D / 16;
    constexpr int DB = D >= 32 ? D / 32 : 1;  // (D = 16: one block of gradient columns, the upper 16 are not stored)
    constexpr int kBlocksPerWave = 2 * Tile::kBlocks / NW;  // LDS-direct loads per wave and tile
    static_assert(2 * Tile::kBlocks % NW == 0, "tile blocks must divide among the waves");
    // A mask block of a wave (32 rows x 64 keys) goes through a private LDS region (8 KiB fp32, 4 KiB for a mask of
    // the operand type) when it fits (D = 64): lanes own rows, so direct loads would touch 32 cache lines per
    // instruction, while LDS-direct loads fetch whole rows. Geometry of a 32-row SwzTile<128> / SwzTile<64>.
    constexpr bool kMaskViaLds = kMatrix && D <= 64;  // (at D = 128 the 4 KiB regions of a 16-bit mask would fit, but the kernel then spills)
    constexpr int kMaskElt = MASK == kMaskF32 ? 4 : 2;
    using MaskTile = std::conditional_t<MASK == kMaskF32, SwzTile<128>, SwzTile<64>>;
    constexpr int kMaskBytes = 32 * MaskTile::kRowBytes;
    constexpr int kMaskLoads = kMaskBytes / 1024;
    __shared__ __attribute__((aligned(1024))) char smem[kStages * kStageBytes + (kMaskViaLds ? NW * kMaskBytes : 0)];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, l32 = lane & 31, h = lane >> 5;
    int bh, qt;
    const int num_key_tiles = (p.S + kBN - 1) / kBN;
    [[maybe_unused]] Part part{};
    int key0 = 0;  // first key of tile 0
    if constexpr (SPLIT) {
        if (!map_part(p, blockIdx.x, gridDim.x, (p.S + kRows - 1) / kRows, num_key_tiles, false, &part)) return;
        bh = part.bh;
        qt = part.tile;
        key0 = part.index * p.part_tiles * kBN;
    } else {
        map_block_for<MASK>(p, blockIdx.x, (p.S + kRows - 1) / kRows, CAUSAL ? kHeavyLast : kUniformTiles, &bh, &qt);
    }
    const int keys = SPLIT ? p.S - key0 : p.S;  // keys from tile 0 on
    const int b = bh / p.H, hd = bh % p.H;
    const int q0 = qt * kRows;
    const int wrow0 = q0 + 32 * wave;
    const int qrow = wrow0 + l32;
    const int qrow_ld = RAGGED ? min(qrow, p.S - 1) : qrow;  // (a row that does not exist reads the last one)

    const char* qrowp = static_cast<const char*>(p.q) + (b * p.qs[0] + hd * p.qs[1] + static_cast<int64_t>(qrow_ld) * p.qs[2]) * 2;
    const char* gorowp = static_cast<const char*>(p.d_o) + (b * p.dos[0] + hd * p.dos[1] + static_cast<int64_t>(qrow_ld) * p.dos[2]) * 2;
    const char* kbase = static_cast<const char*>(p.k) + (b * p.ks[0] + hd * p.ks[1] + (SPLIT ? key0 * p.ks[2] : 0)) * 2;
    const char* vbase = static_cast<const char*>(p.v) + (b * p.vs[0] + hd * p.vs[1] + (SPLIT ? key0 * p.vs[2] : 0)) * 2;
    const int64_t krow_bytes = p.ks[2] * 2, vrow_bytes = p.vs[2] * 2;

    u32x4 qf[KK], gf[KK];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
        qf[kk] = *reinterpret_cast<const u32x4*>(qrowp + (2 * kk + h) * 16);
        gf[kk] = *reinterpret_cast<const u32x4*>(gorowp + (2 * kk + h) * 16);
    }
    float lse = p.lse[static_cast<int64_t>(bh) * p.S + qrow_ld];
    float dlt = 0.f;
    u32x4 of[DELTA ? KK : 1];
    if constexpr (DELTA) {
        // this lane holds half of its dO row (the other half is in lane ^ 32) and fetches the same half of the O row
        const char* orowp = static_cast<const char*>(p.o) + (b * p.os[0] + hd * p.os[1] + static_cast<int64_t>(qrow_ld) * p.os[2]) * 2;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) of[kk] = *reinterpret_cast<const u32x4*>(orowp + (2 * kk + h) * 16);
    } else {
        dlt = p.delta[static_cast<int64_t>(bh) * p.S + qrow_ld];
    }
    const float c = p.scale_log2;
    [[maybe_unused]] const float inv_scale = p.inv_scale;  // (a mask value joins its score before the scale: s + mask / scale)
    // Without dropout (and where the registers allow) the subtraction in dS = P (dP - delta) is left to the matrix pipe:
    // the dP^T accumulators start from delta and take the product with the dO rows negated, which gives delta - dP^T;
    // dS^T then comes out negated and the sign goes into the scale of the final store.
    constexpr bool kDeltaInAcc = !DROPOUT && !DMASK && D <= 64;

    f32x16 acc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) acc[db] = zero16();

    int n_tiles = CAUSAL ? min((q0 + kRows) / kBN, num_key_tiles) : num_key_tiles;  // tiles the workgroup streams
    int my_tiles = CAUSAL ? min((wrow0 + 31) / kBN + 1, n_tiles) : n_tiles;         // tiles with keys visible to this wave
    if constexpr (SPLIT) {
        n_tiles = max(0, min(n_tiles - key0 / kBN, p.part_tiles));
        my_tiles = max(0, min(my_tiles - key0 / kBN, n_tiles));
    }
    if (RAGGED && wrow0 >= p.S) my_tiles = 0;                                       // (a wave without a single row)
    // With the classes of the mask's blocks at hand: key tiles behind the last one that is not masked out altogether
    // are not streamed, and tiles whose mask is all zero over the workgroup's rows are not read.
    uint64_t zero_tiles = 0;
    [[maybe_unused]] KeyBits key_bits;
    if constexpr (MASK == kMaskKeys) {  // (at most 64 tiles)
        key_bits.load(static_cast<const T*>(p.mask) + b * p.ms[0] + hd * p.ms[1], p.S, n_tiles, lane);
        zero_tiles = key_bits.tiles.zero;
        n_tiles = key_bits.tiles.active ? 64 - __builtin_clzll(key_bits.tiles.active) : 1;
        my_tiles = RAGGED && wrow0 >= p.S ? 0 : n_tiles;
    } else if constexpr (MASK != kNoMask) {
        if (p.mcls != nullptr && n_tiles <= 64) {
            const uint8_t* const classes = p.mcls + b * p.mcs[0] + hd * p.mcs[1] + (q0 / 64) * p.mcs[2] + key0 / kBN;
            const int across = RAGGED ? min(kRows / 64, num_key_tiles - q0 / 64) : kRows / 64;
            const TileClasses tc = tile_classes(classes, 1, n_tiles, across, p.mcs[2], lane);
            zero_tiles = tc.zero;
            // (a mask gradient written in place covers every tile: the tiles behind the last active one get their
            // zeros from the loop; an accumulated one adds into a buffer the caller has zero-filled)
            if (!DMASK || p.dmask_acc) {
                if (!(SPLIT && any_active(classes + n_tiles, 1, num_key_tiles - key0 / kBN - n_tiles, across, p.mcs[2], lane)))
                    n_tiles = tc.active ? 64 - __builtin_clzll(tc.active) : SPLIT && part.index > 0 ? 0 : 1;
                my_tiles = RAGGED && wrow0 >= p.S ? 0 : n_tiles;
            }
        }
    }
    auto mask_is_zero = [&](int t) { return MASK != kNoMask && ((zero_tiles >> t) & 1) != 0; };

    int src_off[kBlocksPerWave];
#pragma unroll
    for (int i = 0; i < kBlocksPerWave; ++i) {
        const int blk = wave * kBlocksPerWave + i;  // 0 .. 2*kBlocks-1 over the K tile then the V tile
        const bool is_v = blk >= Tile::kBlocks;
        src_off[i] = static_cast<int>(Tile::src_off(is_v ? blk - Tile::kBlocks : blk, lane, is_v ? vrow_bytes : krow_bytes));
    }
    auto issue_tile = [&](int t) {
        char* stage = smem + (t % kStages) * kStageBytes;
#pragma unroll
        for (int i = 0; i < kBlocksPerWave; ++i) {
            const int blk = wave * kBlocksPerWave + i;
            const bool is_v = blk >= Tile::kBlocks;
            const char* tile_src = is_v ? vbase + static_cast<int64_t>(t) * kBN * vrow_bytes
                                        : kbase + static_cast<int64_t>(t) * kBN * krow_bytes;
            // the sequence ends inside this tile (at D = 128 every tile takes the clamped form: no registers for kept offsets)
            if (RAGGED && ((D == 128 && !kPair) || (t + 1) * kBN > keys)) {
                int l = lane;
                asm volatile("" : "+v"(l));
                lds_direct_load16(tile_src, Tile::src_off_clamped(is_v ? blk - Tile::kBlocks : blk, l, is_v ? vrow_bytes : krow_bytes,
                                                                  keys - 1 - t * kBN), stage + blk * 1024);
            }
            else
                lds_direct_load16(tile_src, src_off[i], stage + blk * 1024);
        }
    };
    char* mask_lds = smem + kStages * kStageBytes + wave * kMaskBytes;
    auto issue_mask = [&](int t) {  // mask block of tile t -> this wave's region, unless it is all zero
        if constexpr (kMaskViaLds) {
            if (mask_is_zero(t)) return;
            const int row0 = RAGGED ? min(wrow0, p.S - 1) : wrow0;
            const char* src = static_cast<const char*>(p.mask) +
                              (b * p.ms[0] + hd * p.ms[1] + static_cast<int64_t>(row0) * p.ms[2] + key0 + t * kBN) * kMaskElt;
            int l = lane;
            asm volatile("" : "+v"(l));  // offsets recomputed per tile rather than kept in registers
#pragma unroll
            for (int blk = 0; blk < kMaskLoads; ++blk)
                lds_direct_load16(src, RAGGED ? MaskTile::src_off_clamped(blk, l, p.ms[2] * kMaskElt, p.S - 1 - row0)
                                              : static_cast<uint32_t>(MaskTile::src_off(blk, l, p.ms[2] * kMaskElt)), mask_lds + blk * 1024);
        }
    };
    // issue order: mask 0, kAhead tiles, then per tile j: mask j+1, tile j+kAhead
    if (!SPLIT || n_tiles > 0) {
        issue_mask(0);
        issue_tile(0);
    }
    if (kAhead > 1 && 1 < n_tiles) issue_tile(1);
    if (kAhead > 2 && 2 < n_tiles) issue_tile(2);
    // (the row fragments were requested before the tiles, so both latencies overlap)
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
        settle(qf[kk]);
        settle(gf[kk]);
    }
    settle(lse);
    if constexpr (DELTA) {
        float sum = 0.f;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            settle(of[kk]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                sum = fmaf(Mma<T>::lo(of[kk][i]), Mma<T>::lo(gf[kk][i]), sum);
                sum = fmaf(Mma<T>::hi(of[kk][i]), Mma<T>::hi(gf[kk][i]), sum);
            }
        }
        dlt = sum_xor32(sum);
        if (h == 0 && (!RAGGED || qrow < p.S) && (!SPLIT || part.index == 0)) p.delta[static_cast<int64_t>(bh) * p.S + qrow] = dlt;
    } else {
        settle(dlt);
    }
    f32x16 dlt16;
    if constexpr (kDeltaInAcc) {
#pragma unroll
        for (int kk = 0; kk < KK; ++kk)
#pragma unroll
            for (int i = 0; i < 4; ++i) gf[kk][i] ^= 0x80008000u;
#pragma unroll
        for (int i = 0; i < 16; ++i) dlt16[i] = dlt;
        asm volatile("" : "+v"(dlt16));  // (kept in registers: as a splat it would be made anew for every block)
    }

    [[maybe_unused]] DropoutRows drop;
    if constexpr (DROPOUT) drop.init(p, bh, qrow >> 2);
    int row_off0 = Tile::off(l32, h);
    int tr_off0 = Tile::tr_off(0, 0, lane), tr_off1 = Tile::tr_off(0, 1, lane);

    for (int j = 0; j < n_tiles; ++j) {
        // (the fragments' offsets of the column blocks are made from these here, not kept in registers across the loop)
        if constexpr (THREE || kPair) asm volatile("" : "+v"(row_off0), "+v"(tr_off0), "+v"(tr_off1));
        // tile j has landed (up to kAhead - 1 younger tiles may still be in flight) and is visible to all
        // waves; every wave is done with tile j-1, whose slot takes the load of tile j + kAhead
        {
            // with a staged mask, block j must have landed too: only tile j + kAhead - 1 was issued after it
            // (the kAhead first tiles after the first block)
            // (a block that is all zero was never requested: then the kAhead - 1 youngest tiles are what may be in flight)
            const int younger = kMaskViaLds && j > 0 && !mask_is_zero(j) ? min(1, max(0, n_tiles - (kAhead - 1) - j)) : min(kAhead - 1, n_tiles - 1 - j);
            if (younger == 2) TRI_WAIT_VMCNT(2 * kBlocksPerWave);
            else if (younger == 1) TRI_WAIT_VMCNT(kBlocksPerWave);
            else TRI_WAIT_VMCNT(0);
        }
        lds_barrier();
        float mk2[kMaskViaLds ? 32 : 1];
        if constexpr (kMaskViaLds) {
            // (a mask excludes the causal variant, so every wave works on every tile)
            if (!mask_is_zero(j)) {  // (a tile whose mask is all zero takes the arithmetic of a tile without a mask)
#pragma unroll
                for (int g = 0; g < 8; ++g) {  // keys 8 g + 4 h .. + 3 of this lane's row
                    if constexpr (MASK == kMaskF32) {
                        const f32x4 v = *reinterpret_cast<const f32x4*>(mask_lds + MaskTile::off(l32, 2 * g + h));
                        mk2[4 * g + 0] = v.x; mk2[4 * g + 1] = v.y; mk2[4 * g + 2] = v.z; mk2[4 * g + 3] = v.w;
                    } else {
                        const u32x2 v = *reinterpret_cast<const u32x2*>(mask_lds + MaskTile::off(l32, g) + 8 * h);
                        mk2[4 * g + 0] = Mma<T>::lo(v.x); mk2[4 * g + 1] = Mma<T>::hi(v.x);
                        mk2[4 * g + 2] = Mma<T>::lo(v.y); mk2[4 * g + 3] = Mma<T>::hi(v.y);
                    }
                }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // region read before it is refilled
            }
            if (j + 1 < n_tiles) issue_mask(j + 1);
        }
        if (j + kAhead < n_tiles) issue_tile(j + kAhead);
        if (j >= my_tiles) continue;

        const char* sK = smem + (j % kStages) * kStageBytes;
        const char* sV = sK + Tile::kBytes;
        const int t0 = key0 + j * kBN;
        const bool diag = CAUSAL && t0 + kBN - 1 > wrow0;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            float mk[kMatrix ? 16 : 1];
            // (at D = 128 the registers do not hold a second form of the arithmetic: a tile whose mask is all zero adds zeros)
            const bool masked = kMatrix && (D == 128 || !mask_is_zero(j));
            if constexpr (kMaskViaLds) {
                if (masked) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) mk[i] = mk2[16 * kb + i];
                }
            } else if constexpr (kMatrix) {
                if (mask_is_zero(j)) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) mk[i] = 0.f;
                } else {
                    const int64_t mrow = b * p.ms[0] + hd * p.ms[1] + static_cast<int64_t>(qrow_ld) * p.ms[2] + t0 + 32 * kb;
#pragma unroll
                    for (int i = 0; i < 16; ++i) mk[i] = mask_at<T, MASK>(p.mask, mrow + c_row(i, h));
                }
            }
            u32x4 fr[KK];
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) fr[kk] = lds_read16(sK, (row_off0 ^ (kk << 5)) + 32 * kb * Tile::kRowBytes);
            __builtin_amdgcn_sched_barrier(0);
            f32x16 st = zero16(), dpt = zero16();
            if constexpr (kDeltaInAcc) dpt = dlt16;
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) {
                st = Mma<T>::run(fr[kk], qf[kk], st);
                fr[kk] = lds_read16(sV, (row_off0 ^ (kk << 5)) + 32 * kb * Tile::kRowBytes);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) dpt = Mma<T>::run(fr[kk], gf[kk], dpt);
            // first transposed K fragments of this block: they arrive during the vector-ALU part
            u32x4 tf[2 * DB];
#pragma unroll
            for (int i = 0; i < 2 * DB; ++i)
                tf[i] = Tile::tr_frag(sK, tr_off0 ^ ((i % DB) << 6), tr_off1 ^ ((i % DB) << 6), 2 * kb + i / DB);
            __builtin_amdgcn_sched_barrier(0);
            if (diag && t0 + 32 * kb + 31 > wrow0) {  // a block that crosses the diagonal: scores above it drop out
                asm volatile("");                     // (a real branch: the other blocks skip the comparisons)
#pragma unroll
                for (int i = 0; i < 16; ++i) st[i] = t0 + 32 * kb + c_row(i, h) <= qrow ? st[i] : -INFINITY;
            }
            if constexpr (MASK == kMaskKeys) {
                if (!mask_is_zero(j)) {
                    const uint32_t visible = key_bits.block(j, kb, h);
#pragma unroll
                    for (int i = 0; i < 16; ++i) st[i] = (visible >> c_row(i, 0) & 1) != 0 ? st[i] : -INFINITY;
                }
            }
            if (RAGGED && !CAUSAL && t0 + 32 * kb + 32 > p.S) {  // keys that do not exist
                int left = p.S - t0 - 32 * kb - 4 * h;
                asm volatile("" : "+v"(left));
#pragma unroll
                for (int i = 0; i < 16; ++i) st[i] = c_row(i, 0) < left ? st[i] : -INFINITY;
            }
            float ds[16];
            if (masked) {
#pragma unroll
                for (int i = 0; i < 16; ++i)  // (s + mask / scale, then the scale; a padded mask behind the scale, as in the forward)
                    ds[i] = RAGGED ? fast_exp2(fmaf(st[i], c, mk[i] * kLog2e) - lse) : fast_exp2(fmaf(fmaf(mk[i], inv_scale, st[i]), c, -lse));
            } else {
#pragma unroll
                for (int i = 0; i < 16; ++i) ds[i] = fast_exp2(fmaf(st[i], c, -lse));
            }
            if constexpr (DROPOUT) {
                uint32_t w[4];
                DropoutRows::words(drop.block(p, (t0 + 32 * kb + 8 * (lane & 3) + 4 * h) >> 2), w);
#pragma unroll
                for (int g = 0; g < 4; ++g)
#pragma unroll
                    for (int bb = 0; bb < 4; ++bb) {
                        const bool keep = static_cast<int>((w[g] >> (8 * bb)) & 0xffu) >= p.thr8;
                        dpt[4 * g + bb] = keep ? dpt[4 * g + bb] : 0.f;
                    }
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) ds[i] *= kDeltaInAcc ? dpt[i] : DROPOUT ? fmaf(dpt[i], p.zscale, -dlt) : dpt[i] - dlt;
            if constexpr (DMASK) {
                const int64_t at = b * p.dms[0] + hd * p.dms[1] + static_cast<int64_t>(qrow) * p.dms[2] + t0 + 32 * kb + 4 * h;
                if (p.dmask_acc) {
                    float* dst = static_cast<float*>(p.dmask) + at;
#pragma unroll
                    for (int i = 0; i < 16; ++i) unsafeAtomicAdd(dst + 8 * (i >> 2) + (i & 3), ds[i]);
                } else if constexpr (MASK == kMaskF32) {
#pragma unroll
                    for (int g = 0; g < 4; ++g)
                        *reinterpret_cast<f32x4*>(static_cast<float*>(p.dmask) + at + 8 * g) = f32x4{ds[4 * g], ds[4 * g + 1], ds[4 * g + 2], ds[4 * g + 3]};
                } else {
#pragma unroll
                    for (int g = 0; g < 4; ++g)
                        *reinterpret_cast<u32x2*>(static_cast<T*>(p.dmask) + at + 8 * g) =
                            u32x2{Mma<T>::pack2(ds[4 * g], ds[4 * g + 1]), Mma<T>::pack2(ds[4 * g + 2], ds[4 * g + 3])};
                }
            }
            u32x4 bop[2];
            bop[0] = pack8<T>(&ds[0]);
            bop[1] = pack8<T>(&ds[8]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 2 * DB; ++i) acc[i % DB] = Mma<T>::run(tf[i], bop[i / DB], acc[i % DB]);
        }
    }

    if constexpr (SPLIT) {
        if (part.count > 1) {
            store_partial<DB, D>(acc, p.partial + (static_cast<int64_t>(part.unit) * kRows + 32 * wave) * D, 0, lane, kDeltaInAcc ? -1.f : 1.f);
            return;
        }
    }
    // every wave is out of the loop: the ring can serve as the waves' private transposition patches
    lds_barrier();
    {
        using Store = RowBlockStore<T, DB, D < 32 ? D : 32 * DB>;
        static_assert(NW * Store::kPatchBytes <= kStages * kStageBytes, "patches must fit into the ring");
        char* out0 = static_cast<char*>(p.dq) + (b * p.dqs[0] + hd * p.dqs[1] + static_cast<int64_t>(wrow0) * p.dqs[2]) * 2;
        const float sc = kDeltaInAcc ? -p.scale : p.scale;
        Store::run(acc, [sc](float x) { return x * sc; }, smem + wave * Store::kPatchBytes, out0, p.dqs[2] * 2, lane,
                   RAGGED ? p.S - wrow0 : 32);
    }
}

// ------------------------------------------------------------------ dQ, phased (no mask, or one of keys)
// Same data flow and tile ring as above, restructured so that the two waves of a SIMD (w and w+4)
// never do the same kind of work at once. Per 64-key tile a wave runs a vector phase (P and dS of the
// tile from its S^T and dP^T, packed as B operands) and a matrix phase (dQ^T += K^T dS^T of this
// tile, then S^T and dP^T of the next one: 6 D / 16 MFMAs through one ring of LDS fragments), with a
// workgroup barrier after each; waves 4-7 run one phase behind waves 0-3. Tile loads are issued at
// the top of the vector phase (two tiles ahead in waves 0-3, three in waves 4-7, which start their
// phase later) and awaited before its barrier.
// With DELTA the kernel also computes delta = rowsum(dO * O) of its rows (instead of reading it) and stores
// it for the dK/dV pass, which then has to run after this one: the separate pre-pass over O and dO
// (trident/kernel/softmax.py:180-238) disappears into the prologue that loads the dO rows anyway.
// RAGGED: S is not a multiple of 256; rows and keys at or beyond S as in the kernel above (clamped loads, probability 0,
// not stored), a wave without a single row of its own only fetches and meets the barriers.
// KEYS: beside a mask of keys that is 0 or -inf (KeyBits).
// NW = 4 (D = 128): workgroups of 128 rows, two to a CU, whose waves share a SIMD without any order between them. 80 KiB of LDS hold three K
// tiles and two V tiles: a tile's matrix phase, behind a barrier that every wave meets once it is done with the phase before (K of tiles t - 1
// and t, V of tile t), requests K and V of tile t + 2 into the slots of K of tile t - 1 and V of tile t; the next tile's barrier awaits them.
// bf16, us, eight waves -> these, heads x S: 16 x 1024 31.4 -> 26.5, 640 x 256 60.6 -> 51.7 (unphased four), 72 x 777 61.3 -> 43.0, causal 104 x 640
// 37.4 -> 30.1; with dropout 16 x 2048 95.8 -> 65.6, 40 x 4096 588 -> 502, causal 64 x 4096 463 -> 425.
template <typename T, int D, bool CAUSAL, bool DROPOUT, bool DELTA, bool RAGGED = false, bool SPLIT = false, bool KEYS = false, int NW = 8>
__global__ __launch_bounds__(64 * NW, 2) void mfma_dq_phased_kernel(const KParams p) {
    static_assert(!RAGGED || D == 128, "boundary handling: D = 128 only");
    static_assert(!KEYS || !(CAUSAL || SPLIT), "a mask excludes the causal variant");
    static_assert(RAGGED || !SPLIT, "parts have boundary handling");
    static_assert(NW == 8 || (NW == 4 && D == 128 && !SPLIT), "eight waves, or four at D = 128");
    using Tile = SwzTile<D>;
    constexpr bool kPair = NW == 4;
    constexpr int kRows = 32 * NW;
    constexpr int kStages = 4;
    constexpr int kStageBytes = 2 * Tile::kBytes;  // K tile, V tile
    // byte offsets of K and V of tile t (-1 is never read)
    auto k_slot = [](int t) { return kPair ? static_cast<int>(static_cast<unsigned>(t + 3) % 3) * Tile::kBytes : ((t + kStages) % kStages) * kStageBytes; };
    auto v_slot = [](int t) { return kPair ? (3 + (t & 1)) * Tile::kBytes : ((t + kStages) % kStages) * kStageBytes + Tile::kBytes; };
    constexpr int KK = D / 16;
    constexpr int DB = D / 32;
    constexpr int kBlocksPerWave = 2 * Tile::kBlocks / NW;
    constexpr int kPerOperand = Tile::kBlocks / NW;
    constexpr int kRowStep = NW * Tile::kRowsPerBlock;
    static_assert(kRowStep % 16 == 0 && 2 * kPerOperand == kBlocksPerWave, "block assignment");
    constexpr int kDqSteps = 4 * DB;           // MFMAs of dQ^T per tile
    constexpr int kSteps = kDqSteps + 4 * KK;  // + S^T and dP^T of the next tile
    constexpr int kRing = D == 128 ? 4 : 6;  // (registers: with dropout the Philox state, without it the delta accumulators)
    static_assert(kRing <= kDqSteps, "the vector phase requests dQ fragments only");
    // The workgroup's Q and dO rows reach the registers through LDS as well: lanes own rows, so direct loads
    // touch 32 cache lines per instruction, while LDS-direct loads fetch whole rows. Each wave stages its
    // own 32 rows behind ring stage 0, which takes tile 0 meanwhile; tiles 1 and 2 follow once every wave
    // has its rows. The O rows (for delta) take the place of the Q rows in a second round (LDS has no room
    // for a third operand at once; fetching them by direct loads during the first round measured 1 %
    // slower). What remains of a workgroup's start is the latency of its first loads (about 6 000 cycles
    // for a single plain load).
    constexpr int kWaveRowBytes = 32 * Tile::kRowBytes;  // a wave's rows of one operand
    constexpr int kRowLoads = kWaveRowBytes / 1024;      // LDS-direct loads per wave and operand
    // (four waves: the Q rows in the place of K of tiles 1 and 2, the dO rows in that of the V tiles)
    constexpr int kStaging = kPair ? Tile::kBytes : kStageBytes;
    constexpr int kRingBytes = kPair ? 5 * Tile::kBytes : kStages * kStageBytes;
    __shared__ __attribute__((aligned(1024))) char smem[kStaging + 2 * NW * kWaveRowBytes];
    static_assert(kStaging + 2 * NW * kWaveRowBytes >= kRingBytes, "the ring lies inside");
    static_assert(!kPair || kStaging + NW * kWaveRowBytes == 3 * Tile::kBytes, "the V tiles take the place of the dO rows");

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, l32 = lane & 31, h = lane >> 5;
    int bh, qt;
    [[maybe_unused]] Part part{};
    int key0 = 0;  // first key of tile 0
    if constexpr (SPLIT) {
        if (!map_part(p, blockIdx.x, gridDim.x, (p.S + kRows - 1) / kRows, (p.S + kBN - 1) / kBN, false, &part)) return;
        bh = part.bh;
        qt = part.tile;
        key0 = part.index * p.part_tiles * kBN;
    } else {
        map_block(blockIdx.x, p.B * p.H, (p.S + kRows - 1) / kRows, CAUSAL ? kHeavyLast : kUniformTiles, &bh, &qt);
    }
    const int keys = SPLIT ? p.S - key0 : p.S;  // keys from tile 0 on
    const int b = bh / p.H, hd = bh % p.H;
    const int q0 = qt * kRows;
    const int wrow0 = q0 + 32 * wave;
    const int qrow = wrow0 + l32;
    const int wrow_ld = RAGGED ? min(wrow0, p.S - 1) : wrow0;  // (rows that do not exist read the last one)
    const int qrow_ld = RAGGED ? min(qrow, p.S - 1) : qrow;
    auto row_off = [&](int blk, int64_t stride_bytes) {  // of piece blk of this wave's rows, from row wrow_ld
        return RAGGED ? Tile::src_off_clamped(blk, lane, stride_bytes, p.S - 1 - wrow_ld) : static_cast<uint32_t>(Tile::src_off(blk, lane, stride_bytes));
    };

    const char* qrows = static_cast<const char*>(p.q) + (b * p.qs[0] + hd * p.qs[1] + static_cast<int64_t>(wrow_ld) * p.qs[2]) * 2;
    const char* gorows = static_cast<const char*>(p.d_o) + (b * p.dos[0] + hd * p.dos[1] + static_cast<int64_t>(wrow_ld) * p.dos[2]) * 2;
    const char* kbase = static_cast<const char*>(p.k) + (b * p.ks[0] + hd * p.ks[1] + (SPLIT ? key0 * p.ks[2] : 0)) * 2;
    const char* vbase = static_cast<const char*>(p.v) + (b * p.vs[0] + hd * p.vs[1] + (SPLIT ? key0 * p.vs[2] : 0)) * 2;
    const int64_t krow_bytes = p.ks[2] * 2, vrow_bytes = p.vs[2] * 2;

    float lse = p.lse[static_cast<int64_t>(bh) * p.S + qrow_ld];
    float dlt = 0.f;
    if constexpr (!DELTA) dlt = p.delta[static_cast<int64_t>(bh) * p.S + qrow_ld];
    char* q_stage = smem + kStaging + wave * kWaveRowBytes;
    char* g_stage = q_stage + NW * kWaveRowBytes;
#pragma unroll
    for (int blk = 0; blk < kRowLoads; ++blk)
        lds_direct_load16(qrows, row_off(blk, p.qs[2] * 2), q_stage + blk * 1024);
#pragma unroll
    for (int blk = 0; blk < kRowLoads; ++blk)
        lds_direct_load16(gorows, row_off(blk, p.dos[2] * 2), g_stage + blk * 1024);
    const float c = p.scale_log2;
    [[maybe_unused]] const float inv_scale = p.inv_scale;  // (a mask value joins its score before the scale: s + mask / scale)

    f32x16 acc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) acc[db] = zero16();

    int n_tiles = CAUSAL ? (q0 + kRows) / kBN : p.S / kBN;     // tiles the workgroup streams
    int my_tiles = CAUSAL ? (wrow0 + 31) / kBN + 1 : n_tiles;  // tiles with keys visible to this wave
    if constexpr (RAGGED) {
        const int num_key_tiles = (p.S + kBN - 1) / kBN;
        n_tiles = CAUSAL ? min(n_tiles, num_key_tiles) : num_key_tiles;
        my_tiles = wrow0 >= p.S ? 0 : (CAUSAL ? min(my_tiles, n_tiles) : n_tiles);
        if constexpr (SPLIT) {
            n_tiles = max(0, min(n_tiles - key0 / kBN, p.part_tiles));
            my_tiles = max(0, min(my_tiles - key0 / kBN, n_tiles));
        }
    }

    [[maybe_unused]] KeyBits key_bits;
    if constexpr (KEYS) {  // (at most 64 tiles; those behind the last one with a visible key are not streamed)
        key_bits.load(static_cast<const T*>(p.mask) + b * p.ms[0] + hd * p.ms[1], p.S, n_tiles, lane);
        n_tiles = key_bits.tiles.active ? 64 - __builtin_clzll(key_bits.tiles.active) : 1;
        my_tiles = RAGGED && wrow0 >= p.S ? 0 : n_tiles;
    }

    // A wave fetches blocks wave, wave + NW, ... of the K tile and of the V tile: their rows are a
    // multiple of 16 apart, so one per-lane source offset serves all of them.
    const uint32_t koff = static_cast<uint32_t>(Tile::src_off(wave, lane, krow_bytes));
    const uint32_t voff = static_cast<uint32_t>(Tile::src_off(wave, lane, vrow_bytes));
    auto issue_k = [&](int t) {  // (four waves)
        char* stage = smem + k_slot(t) + wave * 1024;
        const bool partial = RAGGED && (t + 1) * kBN > keys;
        int l = lane;
        if constexpr (kPair) asm volatile("" : "+v"(l));  // (offsets made here, not kept in registers across the loop)
#pragma unroll
        for (int i = 0; i < kPerOperand; ++i) {
            if (partial)
                lds_direct_load16(kbase + static_cast<int64_t>(t) * kBN * krow_bytes,
                                  Tile::src_off_clamped(wave + i * NW, l, krow_bytes, keys - 1 - t * kBN), stage + i * NW * 1024);
            else
                lds_direct_load16(kbase + (static_cast<int64_t>(t) * kBN + i * kRowStep) * krow_bytes, koff, stage + i * NW * 1024);
        }
    };
    auto issue_v = [&](int t) {
        char* stage = smem + v_slot(t) + wave * 1024;
        const bool partial = RAGGED && (t + 1) * kBN > keys;
        int l = lane;
        if constexpr (kPair) asm volatile("" : "+v"(l));  // (offsets made here, not kept in registers across the loop)
#pragma unroll
        for (int i = 0; i < kPerOperand; ++i) {
            if (partial)
                lds_direct_load16(vbase + static_cast<int64_t>(t) * kBN * vrow_bytes,
                                  Tile::src_off_clamped(wave + i * NW, l, vrow_bytes, keys - 1 - t * kBN), stage + i * NW * 1024);
            else
                lds_direct_load16(vbase + (static_cast<int64_t>(t) * kBN + i * kRowStep) * vrow_bytes, voff, stage + i * NW * 1024);
        }
    };
    auto issue_tile = [&](int t) {
        if constexpr (kPair) {
            issue_k(t);
            issue_v(t);
            return;
        }
        char* stage = smem + k_slot(t) + wave * 1024;
        if (RAGGED && (t + 1) * kBN > keys) {  // the sequence ends inside this tile
            const int last = keys - 1 - t * kBN;
#pragma unroll
            for (int i = 0; i < kPerOperand; ++i)
                lds_direct_load16(kbase + static_cast<int64_t>(t) * kBN * krow_bytes,
                                  Tile::src_off_clamped(wave + i * NW, lane, krow_bytes, last), stage + i * NW * 1024);
#pragma unroll
            for (int i = 0; i < kPerOperand; ++i)
                lds_direct_load16(vbase + static_cast<int64_t>(t) * kBN * vrow_bytes,
                                  Tile::src_off_clamped(wave + i * NW, lane, vrow_bytes, last), stage + Tile::kBytes + i * NW * 1024);
            return;
        }
#pragma unroll
        for (int i = 0; i < kPerOperand; ++i)
            lds_direct_load16(kbase + (static_cast<int64_t>(t) * kBN + i * kRowStep) * krow_bytes, koff, stage + i * NW * 1024);
#pragma unroll
        for (int i = 0; i < kPerOperand; ++i)
            lds_direct_load16(vbase + (static_cast<int64_t>(t) * kBN + i * kRowStep) * vrow_bytes, voff,
                              stage + Tile::kBytes + i * NW * 1024);
    };
    const int group = wave >> 2;
    const int dist = 2 + group;
    const int n_first = min(dist, n_tiles);
    if constexpr (SPLIT) {
        if (n_tiles == 0) {  // (the last part of an item that the sequence cuts short)
            store_partial<DB, D>(acc, p.partial + (static_cast<int64_t>(part.unit) * kRows + 32 * wave) * D, 0, lane, 1.f);
            TRI_WAIT_VMCNT(0);  // (the rows on their way to LDS land before the workgroup gives it back)
            return;
        }
    }
    if constexpr (kPair) issue_k(0);
    else issue_tile(0);

    int row_off0 = Tile::off(l32, h);
    TRI_WAIT_VMCNT(kPair ? kPerOperand : kBlocksPerWave);  // this wave's Q and dO rows have landed (tile 0 may be on its way)
    asm volatile("" ::: "memory");
    u32x4 qf[KK], gf[KK];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
        qf[kk] = lds_read16(q_stage, row_off0 ^ (kk << 5));
        gf[kk] = lds_read16(g_stage, row_off0 ^ (kk << 5));
    }
    if constexpr (kPair) {  // every wave has its rows in registers: the V tiles can follow
        lds_barrier();
        issue_v(0);
        if (n_tiles > 1) issue_v(1);
    }
    if constexpr (DELTA) {
        // the O rows follow into the place of the Q rows; this lane holds half of its row (the other half is
        // in lane ^ 32)
        const char* orows = static_cast<const char*>(p.o) + (b * p.os[0] + hd * p.os[1] + static_cast<int64_t>(wrow_ld) * p.os[2]) * 2;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the Q rows are in registers
#pragma unroll
        for (int blk = 0; blk < kRowLoads; ++blk)
            lds_direct_load16(orows, row_off(blk, p.os[2] * 2), q_stage + blk * 1024);
        TRI_WAIT_VMCNT(0);
        asm volatile("" ::: "memory");
        float sum = 0.f;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            const u32x4 of = lds_read16(q_stage, row_off0 ^ (kk << 5));
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                sum = fmaf(Mma<T>::lo(of[i]), Mma<T>::lo(gf[kk][i]), sum);
                sum = fmaf(Mma<T>::hi(of[i]), Mma<T>::hi(gf[kk][i]), sum);
            }
        }
        dlt = sum_xor32(sum);
        if (h == 0 && (!RAGGED || qrow < p.S) && (!SPLIT || part.index == 0)) p.delta[static_cast<int64_t>(bh) * p.S + qrow] = dlt;
    }

    // Without dropout the subtraction in dS = P (dP - delta) is left to the matrix pipe: the dP^T accumulators start from
    // delta and take the product with the dO rows negated (delta - dP^T); dS^T comes out negated and the sign goes into
    // the scale of the final store.
    constexpr bool kDeltaInAcc = !DROPOUT && !RAGGED && !KEYS;  // (boundary handling and a mask leave no registers for it)
    f32x16 dlt16;
    if constexpr (kDeltaInAcc) {
#pragma unroll
        for (int kk = 0; kk < KK; ++kk)
#pragma unroll
            for (int i = 0; i < 4; ++i) gf[kk][i] ^= 0x80008000u;
#pragma unroll
        for (int i = 0; i < 16; ++i) dlt16[i] = dlt;
        asm volatile("" : "+v"(dlt16));  // (kept in registers: as a splat it would be made anew for every tile)
    }
    [[maybe_unused]] DropoutRows drop;
    if constexpr (DROPOUT) drop.init(p, bh, qrow >> 2);
    int tr_off0 = Tile::tr_off(0, 0, lane), tr_off1 = Tile::tr_off(0, 1, lane);

    // fragment n of the matrix phase of tile t: n < kDqSteps: K^T of tile t (column block n % DB, K-step
    // n / DB); then the K rows (key block 0, 1) and the V rows (key block 0, 1) of tile t + 1
    auto frag = [&](int t, int n) {
        if (n < kDqSteps) {
            const char* sK = smem + k_slot(t);
            return Tile::tr_frag(sK, tr_off0 ^ ((n % DB) << 6), tr_off1 ^ ((n % DB) << 6), n / DB);
        }
        const int m = n - kDqSteps;
        const char* sT = smem + (m < 2 * KK ? k_slot(t + 1) : v_slot(t + 1));
        return lds_read16(sT, (row_off0 ^ ((m % KK) << 5)) + 32 * ((m / KK) & 1) * Tile::kRowBytes);
    };
    f32x16 st[2], dpt[2];  // S^T and dP^T of the current tile (two key blocks)
    u32x4 bop[4];          // dS^T of the current tile as B operands
    u32x4 ring[kRing];
    auto matrix_phase = [&](auto with_dq, int t, bool with_scores = true) {
        constexpr int first = decltype(with_dq)::value ? 0 : kDqSteps;
        f32x16 s_new[2] = {zero16(), zero16()}, dp_new[2] = {zero16(), zero16()};
        if constexpr (kDeltaInAcc) {
            dp_new[0] = dlt16;
            dp_new[1] = dlt16;
        }
#pragma unroll
        for (int n = first; n < kSteps; ++n) {
            if (n >= kDqSteps && !with_scores) break;
            const int slot = (n - first) % kRing;
            const int m = n - kDqSteps;
            if (n < kDqSteps) acc[n % DB] = Mma<T>::run(ring[slot], bop[n / DB], acc[n % DB]);
            else if (m < 2 * KK) s_new[m / KK] = Mma<T>::run(ring[slot], qf[m % KK], s_new[m / KK]);
            else dp_new[(m / KK) & 1] = Mma<T>::run(ring[slot], gf[m % KK], dp_new[(m / KK) & 1]);
            if (n + kRing < kSteps) ring[slot] = frag(t, n + kRing);
            __builtin_amdgcn_sched_barrier(0);
        }
        st[0] = s_new[0]; st[1] = s_new[1];
        dpt[0] = dp_new[0]; dpt[1] = dp_new[1];
    };
    using Yes = std::integral_constant<bool, true>;
    using No = std::integral_constant<bool, false>;
    auto wait_tile = [&](bool newest_in_flight) {
        if (newest_in_flight) TRI_WAIT_VMCNT(kBlocksPerWave);
        else TRI_WAIT_VMCNT(0);
    };

    // tile 0 has landed and is visible to all waves, and every wave has its rows in registers: the staging
    // area returns to the ring
    TRI_WAIT_VMCNT(0);
    settle(lse);
    if constexpr (!DELTA) settle(dlt);
    lds_barrier();
    if constexpr (kPair) {
        if (n_first > 1) issue_k(1);
    } else {
        if (n_first > 1) issue_tile(1);
        if (n_first > 2) issue_tile(2);
    }
    if (group == 1) {
        // group 1 starts one phase late; group 0 reads tile 1 in its first matrix phase
        if (n_first == 3) TRI_WAIT_VMCNT(kBlocksPerWave);
        else TRI_WAIT_VMCNT(0);
        lds_barrier();
    }
    {
#pragma unroll
        for (int r = 0; r < kRing; ++r) ring[r] = frag(-1, kDqSteps + r);
        __builtin_amdgcn_sched_barrier(0);
        matrix_phase(No{}, -1);
    }

    for (int t = 0; t < my_tiles; ++t) {
        const bool issued = t + dist < n_tiles;
        // (the fragments' offsets of the column blocks are made from these here, not kept in registers across the loop)
        if constexpr (kPair) asm volatile("" : "+v"(row_off0), "+v"(tr_off0), "+v"(tr_off1));
        if (!kPair && issued) issue_tile(t + dist);
        // ---- vector phase: P and dS of the tile (only 32-key blocks that cross the diagonal pay for the
        // causal comparison)
        auto softmax_backward = [&](auto on_diagonal, int kb) {
            const int first_key = key0 + t * kBN + 32 * kb;
            if constexpr (KEYS) {
                if (!((key_bits.tiles.zero >> t) & 1)) {
                    const uint32_t visible = key_bits.block(t, kb, h);
#pragma unroll
                    for (int i = 0; i < 16; ++i) st[kb][i] = (visible >> c_row(i, 0) & 1) != 0 ? st[kb][i] : -INFINITY;
                }
            }
            if (RAGGED && !CAUSAL && first_key + 32 > p.S) {  // keys that do not exist (under the causal mask no existing row sees them)
                asm volatile("");                        // (a real branch)
#pragma unroll
                for (int i = 0; i < 16; ++i) st[kb][i] = first_key + c_row(i, h) < p.S ? st[kb][i] : -INFINITY;
            }
            float ds[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                float pr = fast_exp2(fmaf(st[kb][i], c, -lse));
                if constexpr (decltype(on_diagonal)::value) pr = first_key + c_row(i, h) <= qrow ? pr : 0.f;
                ds[i] = pr;
            }
            f32x16 dpv = dpt[kb];
            if constexpr (DROPOUT) {
                uint32_t w[4];
                DropoutRows::words(drop.block(p, (first_key + 8 * (lane & 3) + 4 * h) >> 2), w);
#pragma unroll
                for (int g = 0; g < 4; ++g)
#pragma unroll
                    for (int bb = 0; bb < 4; ++bb) {
                        const bool keep = static_cast<int>((w[g] >> (8 * bb)) & 0xffu) >= p.thr8;
                        dpv[4 * g + bb] = keep ? dpv[4 * g + bb] : 0.f;
                    }
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) ds[i] *= kDeltaInAcc ? dpv[i] : DROPOUT ? fmaf(dpv[i], p.zscale, -dlt) : dpv[i] - dlt;
            bop[2 * kb + 0] = pack8<T>(&ds[0]);
            bop[2 * kb + 1] = pack8<T>(&ds[8]);
        };
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            if (CAUSAL && key0 + t * kBN + 32 * kb + 31 > wrow0) softmax_backward(Yes{}, kb);
            else softmax_backward(No{}, kb);
        }
        // the first fragments of the matrix phase (K^T of this tile, visible since the previous barrier)
#pragma unroll
        for (int r = 0; r < kRing; ++r) ring[r] = frag(t, r);
        // tile t + dist - 1 has landed (the newest one may still be in flight); after the barrier it is
        // visible to every wave, and the partner group changes phase
        wait_tile(!kPair && issued);
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if (kPair && issued) issue_tile(t + dist);
        // ---- matrix phase (a wave's last tile has no successor to score; the dropout variant runs the S^T /
        // dP^T steps all the same, on whatever the next slot holds: leaving them out costs it registers it does
        // not have, and the result is never used)
        __builtin_amdgcn_s_setprio(2);
        matrix_phase(Yes{}, t, DROPOUT || t + 1 < my_tiles);
        __builtin_amdgcn_s_setprio(0);
        if constexpr (!kPair) {
            __builtin_amdgcn_sched_barrier(0);
            lds_barrier();
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // afterwards a wave only keeps fetching its share of the remaining tiles and meeting the barriers
    for (int t = my_tiles; t < n_tiles; ++t) {
        const bool issued = t + dist < n_tiles;
        if (!kPair && issued) issue_tile(t + dist);
        wait_tile(!kPair && issued);
        lds_barrier();
        if constexpr (kPair) {
            if (issued) issue_tile(t + dist);
        } else {
            lds_barrier();
        }
    }
    if (!kPair && group == 0) lds_barrier();  // group 1 is still in its last matrix phase

    if constexpr (SPLIT) {
        if (part.count > 1) {
            int elane = threadIdx.x & 63;
            asm volatile("" : "+v"(elane));
            store_partial<DB, D>(acc, p.partial + (static_cast<int64_t>(part.unit) * kRows + 32 * wave) * D, 0, elane, kDeltaInAcc ? -1.f : 1.f);
            return;
        }
    }
    // every wave is out of the loop: the ring can serve as the waves' private transposition patches
    lds_barrier();
    {
        using Store = RowBlockStore<T, DB>;
        static_assert(NW * Store::kPatchBytes <= kRingBytes, "patches must fit into the ring");
        char* out0 = static_cast<char*>(p.dq) + (b * p.dqs[0] + hd * p.dqs[1] + static_cast<int64_t>(wrow0) * p.dqs[2]) * 2;
        const float sc = kDeltaInAcc ? -p.scale : p.scale;
        // the lane index taken afresh: the epilogue's per-lane offsets are then computed here instead of being
        // kept (or, with every register in use, spilled) across the loop
        int elane = threadIdx.x & 63;
        asm volatile("" : "+v"(elane));
        Store::run(acc, [sc](float x) { return x * sc; }, smem + wave * Store::kPatchBytes, out0, p.dqs[2] * 2, elane, RAGGED ? p.S - wrow0 : 32);
    }
}

}  // namespace
}  // namespace tri
