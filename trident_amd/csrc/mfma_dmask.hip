// Gradient of an additive mask for fp16/bf16 problems, D in {16,32,64,128}, any S: of one that is shared by batches or heads (or
// both), and of any mask with rows and keys of its own where the dQ pass does not write it
// (trident/kernel/attention.py:332-335 stores dS per batch and head; autograd then sums it over the broadcast dimensions).
//
// A workgroup owns a tile of the mask, 128 rows x 128 keys, and walks the (batch, head) pairs that share it, adding
// dS = P (dP - delta) in registers: no atomic, no zero fill, a fixed order of summation, and the tile of the mask itself is read
// once for all pairs. The price is S and dP once more (2 of the pass's 7 products), where the dQ pass, which has them, would send
// every dS to memory by itself: bf16 B=8 H=12 S=512 D=64, bias [1,H,S,S]: the dQ pass with atomic adds took 0.61 ms, bound by the
// 25 M adds.
//
// Eight waves, each 32 rows x 64 keys: the K and V rows are the A operands, the Q and dO rows the B operands, so that lane l32 owns
// a row with its lse and delta, and the accumulators (8 groups of 4 keys) leave in row pieces. What a pair needs, 128 rows of each
// operand, comes through LDS by LDS-direct loads (64 columns of the head size at a time: 64 KiB, two slots), the next pair's on
// their way while this one's products run. Before, four waves staged 64 keys x 128 rows through registers, or every wave read
// 16 bytes per lane straight from memory, and one workgroup walked all pairs: MFMA 7 % busy, no unit was. Case above 41 -> 27 us;
// few tiles under many pairs: B=256 H=4 S=128 D=64 178 -> 28, B=64 H=16 S=64 D=128 93 -> 29, B=100 H=4 S=733 D=64 337 -> 197 (with the second launch).
//
// Too few tiles to fill the chip: the pairs of a tile are dealt to several workgroups, which leave their fp32 sums in the
// caller's workspace, and a second launch adds those up in their order.
#include <algorithm>

#include "launch.hpp"
#include "mfma_common.hpp"

namespace tri {
namespace {

constexpr int kTile = 128;                       // rows and keys of a mask tile
constexpr int64_t kPartFloats = kTile * kTile;   // a part's sums in the workspace

struct Plan {
    int tiles;       // workgroups of one part: mask tiles over all masks
    int parts;       // workgroups per tile
    int pairs_each;  // pairs a workgroup walks
};

// Where a tile lies: mask m, row tile rt, key tile kt.
struct TileAt {
    int mask_b, mask_h, row0, key0;
};
__device__ __forceinline__ TileAt tile_at(const KParams& p, int tile) {
    const int n = (p.S + kTile - 1) / kTile, mask_heads = p.dms[1] == 0 ? 1 : p.H;
    const int m = tile / (n * n);
    return TileAt{m / mask_heads, m % mask_heads, tile / n % n * kTile, tile % n * kTile};
}

// One group of four keys of a row of dS, in the mask's type.
__device__ __forceinline__ void store_group(const KParams& p, int64_t at, int keys_left, bool by_fours, const float* v) {
    if (by_fours && keys_left >= 4) {
        if (p.mask_dtype == TRI_ATTN_F32) *reinterpret_cast<f32x4*>(static_cast<float*>(p.dmask) + at) = f32x4{v[0], v[1], v[2], v[3]};
        else *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(p.dmask) + at) = p.mask_dtype == TRI_ATTN_F16
            ? u32x2{Mma<f16_t>::pack2(v[0], v[1]), Mma<f16_t>::pack2(v[2], v[3])} : u32x2{Mma<bf16_t>::pack2(v[0], v[1]), Mma<bf16_t>::pack2(v[2], v[3])};
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (e < keys_left) store_mask_elem(p.dmask, p.mask_dtype, at + e, v[e]);
    }
}

template <typename T, int D, bool DROPOUT>
__global__ __launch_bounds__(512, 2) void mfma_dmask_kernel(const KParams p, const Plan plan, bool mask_by_fours, bool by_fours) {
    constexpr int CH = D < 64 ? D : 64;            // columns of the head size in a slot
    constexpr int kChunks = D / CH, KK = CH / 16;
    using Tile = SwzTile<CH>;                      // 64 rows
    constexpr int kSlotTiles = 8;                  // K, V, Q, dO: two tiles each
    constexpr int kSlotBytes = kSlotTiles * Tile::kBytes + 1024;  // + lse and delta of 128 rows
    constexpr int kSlots = CH == 64 ? 2 : 4;
    constexpr int kLoads = kSlotTiles * Tile::kBlocks / 8;        // LDS-direct loads per wave and slot (one more for lse / delta)
    __shared__ __attribute__((aligned(1024))) char smem[kSlots * kSlotBytes];

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63, l32 = lane & 31, h = lane >> 5;
    // an XCD takes workgroups in a row: the tiles of one mask under the same pairs, whose rows then sit in its L2
    const int unit = static_cast<int>(blockIdx.x & 7) * static_cast<int>(gridDim.x >> 3) + static_cast<int>(blockIdx.x >> 3);
    if (unit >= plan.tiles * plan.parts) return;
    const int per_mask = ((p.S + kTile - 1) / kTile) * ((p.S + kTile - 1) / kTile);
    const int mask = unit / (per_mask * plan.parts), part = unit / per_mask % plan.parts;
    const int tile = mask * per_mask + unit % per_mask;
    const TileAt at = tile_at(p, tile);
    const int sum_h = p.dms[1] == 0 ? p.H : 1, pairs = (p.dms[0] == 0 ? p.B : 1) * sum_h;
    const int first = part * plan.pairs_each, n_pairs = max(0, min(pairs - first, plan.pairs_each));
    const int rb = wave & 3, kh = wave >> 2;      // this wave's row block and half of the keys
    const int t0 = at.key0 + 64 * kh;
    const int qrow = at.row0 + 32 * rb + l32;

    // This wave's share of a slot's loads: block blk of 1 KiB of tile blk / kBlocks (K 0-1, V 2-3, Q 4-5, dO 6-7). The rows are the
    // same for every pair: a lane's offset from the first one is kept, and only the pair's base changes.
    uint32_t off[kLoads];
    int64_t row_start[kLoads];  // (wave-uniform)
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int blk = wave * kLoads + i, tl = blk / Tile::kBlocks, operand = tl >> 1;
        const int64_t stride = (operand == 0 ? p.ks[2] : operand == 1 ? p.vs[2] : operand == 2 ? p.qs[2] : p.dos[2]) * 2;
        const int row = (operand < 2 ? at.key0 : at.row0) + 64 * (tl & 1), from = min(row, p.S - 1);  // (rows beyond the sequence: its last one)
        off[i] = Tile::src_off_clamped(blk % Tile::kBlocks, lane, stride, p.S - 1 - from);
        row_start[i] = from * stride;
    }
    const int aux_row = min(at.row0 + 64 * (wave & 1), p.S - 1), aux_off = min(lane, p.S - 1 - aux_row) * 4;
    const auto issue = [&](int step) {
        const int pair = first + step / kChunks, chunk = step % kChunks;
        const int b = at.mask_b + pair / sum_h, hd = at.mask_h + pair % sum_h;
        char* slot = smem + (step % kSlots) * kSlotBytes;
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int blk = wave * kLoads + i, operand = blk / Tile::kBlocks >> 1;
            const char* base = operand == 0   ? static_cast<const char*>(p.k) + (b * p.ks[0] + hd * p.ks[1]) * 2
                               : operand == 1 ? static_cast<const char*>(p.v) + (b * p.vs[0] + hd * p.vs[1]) * 2
                               : operand == 2 ? static_cast<const char*>(p.q) + (b * p.qs[0] + hd * p.qs[1]) * 2
                                              : static_cast<const char*>(p.d_o) + (b * p.dos[0] + hd * p.dos[1]) * 2;
            lds_direct_load16(base + row_start[i] + chunk * CH * 2, off[i], slot + blk * 1024);
        }
        // every wave issues exactly one more load: lse (even quarters of the waves) or delta of 64 of the rows (duplicates land on the
        // same bytes)
        const float* aux = ((wave & 2) ? p.delta : p.lse) + (static_cast<int64_t>(b) * p.H + hd) * p.S + aux_row;
        lds_direct_load4(aux, aux_off, slot + kSlotTiles * Tile::kBytes + ((wave & 2) ? 512 : 0) + 256 * (wave & 1));
    };
    const int steps = n_pairs * kChunks;
#pragma unroll
    for (int s = 0; s < kSlots - 1; ++s)
        if (s < steps) issue(s);

    // mask values of this lane's row (log2 domain), the same for every pair; -inf for keys that do not exist
    float mk[32];
    {
        const int64_t from = at.mask_b * p.ms[0] + at.mask_h * p.ms[1] + static_cast<int64_t>(min(qrow, p.S - 1)) * p.ms[2];
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            const int key = t0 + 32 * (g >> 2) + 8 * (g & 3) + 4 * h;
            if (mask_by_fours && key + 4 <= p.S) {
                f32x4 v;
                if (p.mask_dtype == TRI_ATTN_F32) {
                    v = *reinterpret_cast<const f32x4*>(static_cast<const float*>(p.mask) + from + key);
                } else {
                    const u32x2 w = *reinterpret_cast<const u32x2*>(static_cast<const uint16_t*>(p.mask) + from + key);
                    if (p.mask_dtype == TRI_ATTN_F16) v = f32x4{Mma<f16_t>::lo(w.x), Mma<f16_t>::hi(w.x), Mma<f16_t>::lo(w.y), Mma<f16_t>::hi(w.y)};
                    else v = f32x4{Mma<bf16_t>::lo(w.x), Mma<bf16_t>::hi(w.x), Mma<bf16_t>::lo(w.y), Mma<bf16_t>::hi(w.y)};
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) mk[4 * g + e] = v[e] * kLog2e;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) mk[4 * g + e] = key + e < p.S ? load_mask_elem(p.mask, p.mask_dtype, from + key + e) * kLog2e : -INFINITY;
            }
        }
#pragma unroll
        for (int i = 0; i < 32; ++i) settle(mk[i]);
    }
    float acc[32];
#pragma unroll
    for (int i = 0; i < 32; ++i) acc[i] = 0.f;
    const bool live = at.row0 + 32 * rb < p.S && t0 < p.S;  // (else this wave only fetches and meets the barriers)
    const int row_off = Tile::off(l32, h);
    f32x16 s[2], dp[2];

    for (int step = 0; step < steps; ++step) {
        // this step's slot has landed (kSlots - 2 younger ones may be on their way) and is visible; every wave is done with the one before
        const int younger = min(kSlots - 2, steps - 1 - step);
        if (kSlots > 2 && younger == 2) TRI_WAIT_VMCNT(2 * (kLoads + 1));
        else if (kSlots > 2 && younger == 1) TRI_WAIT_VMCNT(kLoads + 1);
        else TRI_WAIT_VMCNT(0);
        lds_barrier();
        if (step + kSlots - 1 < steps) issue(step + kSlots - 1);
        if (!live) continue;
        const char* slot = smem + (step % kSlots) * kSlotBytes;
        const char* sK = slot + kh * Tile::kBytes;
        const char* sQ = slot + (4 + (rb >> 1)) * Tile::kBytes + 32 * (rb & 1) * Tile::kRowBytes;
        if (step % kChunks == 0) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) s[kb] = dp[kb] = zero16();
        }
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            const int o = row_off ^ (kk << 5);
            const u32x4 qf = lds_read16(sQ, o), gf = lds_read16(sQ + 2 * Tile::kBytes, o);
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                s[kb] = Mma<T>::run(lds_read16(sK, o + 32 * kb * Tile::kRowBytes), qf, s[kb]);
                dp[kb] = Mma<T>::run(lds_read16(sK + 2 * Tile::kBytes, o + 32 * kb * Tile::kRowBytes), gf, dp[kb]);
            }
        }
        if (step % kChunks != kChunks - 1) continue;
        const float* aux = reinterpret_cast<const float*>(slot + kSlotTiles * Tile::kBytes) + 32 * rb + l32;
        const float lse = aux[0], dlt = aux[128];
        if constexpr (DROPOUT) {
            const int pair = first + step / kChunks;
            const int64_t bh = static_cast<int64_t>(at.mask_b + pair / sum_h) * p.H + at.mask_h + pair % sum_h;
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                const Philox4 mine = dropout_block(p, static_cast<uint32_t>(bh), qrow >> 2, (t0 + 32 * kb + 8 * (lane & 3) + 4 * h) >> 2);
                uint32_t w[4];
                DropoutRows::words(mine, w);
#pragma unroll
                for (int g = 0; g < 4; ++g)
#pragma unroll
                    for (int bb = 0; bb < 4; ++bb) {
                        const bool keep = static_cast<int>((w[g] >> (8 * bb)) & 0xffu) >= p.thr8;
                        dp[kb][4 * g + bb] = keep ? dp[kb][4 * g + bb] * p.zscale : 0.f;
                    }
            }
        }
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[16 * kb + i] += fast_exp2(fmaf(s[kb][i], p.scale_log2, mk[16 * kb + i]) - lse) * (dp[kb][i] - dlt);
    }
    if (!live) return;
    if (plan.parts > 1) {
        f32x4* to = reinterpret_cast<f32x4*>(p.partial + (static_cast<int64_t>(tile) * plan.parts + part) * kPartFloats) + wave * 512 + lane;
#pragma unroll
        for (int g = 0; g < 8; ++g) to[g * 64] = f32x4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
        return;
    }
    if (qrow >= p.S) return;
    const int64_t out = at.mask_b * p.dms[0] + at.mask_h * p.dms[1] + static_cast<int64_t>(qrow) * p.dms[2] + t0;
#pragma unroll
    for (int g = 0; g < 8; ++g) {
        const int key = 32 * (g >> 2) + 8 * (g & 3) + 4 * h;  // keys key .. key + 3 of this wave's half
        store_group(p, out + key, p.S - t0 - key, by_fours, &acc[4 * g]);
    }
}

// The parts of a tile, added up in their order. A workgroup takes 32 rows x 64 keys, one wave two of the eight groups.
__global__ __launch_bounds__(256) void dmask_combine_kernel(const KParams p, const Plan plan, bool by_fours) {
    const int tile = static_cast<int>(blockIdx.x >> 3), block = static_cast<int>(blockIdx.x & 7), wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const TileAt at = tile_at(p, tile);
    const int t0 = at.key0 + 64 * (block >> 2), row = at.row0 + 32 * (block & 3) + (lane & 31);
    if (t0 >= p.S || row >= p.S) return;  // (blocks without a single row or key were not stored either)
    const f32x4* from = reinterpret_cast<const f32x4*>(p.partial + static_cast<int64_t>(tile) * plan.parts * kPartFloats) + block * 512 + 2 * wave * 64 + lane;
    f32x4 sum[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll 8
    for (int i = 0; i < plan.parts; ++i) {
        sum[0] += from[i * (kPartFloats / 4)];
        sum[1] += from[i * (kPartFloats / 4) + 64];
    }
    const int64_t out = at.mask_b * p.dms[0] + at.mask_h * p.dms[1] + static_cast<int64_t>(row) * p.dms[2] + t0;
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        const int g = 2 * wave + n, key = 32 * (g >> 2) + 8 * (g & 3) + 4 * (lane >> 5);
        const float v[4] = {sum[n].x, sum[n].y, sum[n].z, sum[n].w};
        store_group(p, out + key, p.S - t0 - key, by_fours, v);
    }
}

// One workgroup per CU (LDS). Microseconds of a workgroup's start and end, of a pair and of the second launch, as measured.
Plan plan_dmask(const KParams& p, bool may_split) {
    const int64_t masks = (p.dms[0] == 0 ? int64_t{1} : p.B) * (p.dms[1] == 0 ? 1 : p.H), n = (p.S + kTile - 1) / kTile;
    const int64_t pairs = static_cast<int64_t>(p.B) * p.H / masks, tiles = masks * n * n;
    Plan plan{static_cast<int>(std::min<int64_t>(tiles, 2147483647LL / 16)), 1, static_cast<int>(pairs)};
    if (!may_split || tiles > (1 << 20)) return plan;
    const int64_t slots = static_cast<int64_t>(persistent_grid(1 << 20));
    const double pair_us = p.D == 128 ? 2.5 : 1.5;
    const auto time = [&](int64_t parts) {
        return static_cast<double>((tiles * parts + slots - 1) / slots) * (6.0 + static_cast<double>((pairs + parts - 1) / parts) * pair_us) +
               (parts > 1 ? 5.0 + static_cast<double>(tiles * parts) * kPartFloats * 8 / 5e6 : 0.0);
    };
    double best = time(1);
    for (int64_t parts = 2; parts <= std::min<int64_t>(pairs, 256); ++parts) {
        const double t = time(parts);
        if (t < 0.95 * best) {
            best = t;
            plan.parts = static_cast<int>(parts);
            plan.pairs_each = static_cast<int>((pairs + parts - 1) / parts);
        }
    }
    return plan;
}

bool fours(const void* ptr, const int64_t* s) { return reinterpret_cast<uintptr_t>(ptr) % 16 == 0 && s[0] % 4 == 0 && s[1] % 4 == 0 && s[2] % 4 == 0; }

template <typename T, int D>
void launch_dmask_t(const KParams& p, const Plan& plan, hipStream_t stream) {
    const dim3 grid(static_cast<unsigned>((static_cast<int64_t>(plan.tiles) * plan.parts + 7) / 8 * 8)), block(512);
    const bool in = fours(p.mask, p.ms), out = fours(p.dmask, p.dms);
    if (p.thr8 > 0) hipLaunchKernelGGL((mfma_dmask_kernel<T, D, true>), grid, block, 0, stream, p, plan, in, out);
    else hipLaunchKernelGGL((mfma_dmask_kernel<T, D, false>), grid, block, 0, stream, p, plan, in, out);
}

template <typename T>
void launch_dmask_d(const KParams& p, const Plan& plan, hipStream_t stream) {
    if (p.D == 128) launch_dmask_t<T, 128>(p, plan, stream);
    else if (p.D == 64) launch_dmask_t<T, 64>(p, plan, stream);
    else if (p.D == 32) launch_dmask_t<T, 32>(p, plan, stream);
    else launch_dmask_t<T, 16>(p, plan, stream);
}

// (a tile's 64 rows are reached with an unsigned 32-bit byte offset)
bool rows8(const void* ptr, const int64_t* s) {
    return reinterpret_cast<uintptr_t>(ptr) % 16 == 0 && s[0] % 8 == 0 && s[1] % 8 == 0 && s[2] % 8 == 0 && s[2] < (int64_t{1} << 24);
}

}  // namespace

bool mfma_dmask_supported(int dtype, const KParams& p) {
    if (dtype != TRI_ATTN_F16 && dtype != TRI_ATTN_BF16) return false;
    if (p.mask == nullptr || p.dmask == nullptr || p.causal) return false;
    const bool over_b = p.dms[0] == 0 && p.B > 1, over_h = p.dms[1] == 0 && p.H > 1;
    if (!over_b && !over_h && p.S % 128 == 0) return false;                      // (written in place by the dQ pass)
    if (p.dms[2] == 0 && p.S > 1) return false;                                  // (summed over the rows: atomics)
    if ((over_b && p.ms[0] != 0) || (over_h && p.ms[1] != 0)) return false;      // (one mask tile for all pairs)
    const int64_t masks = (p.dms[0] == 0 ? int64_t{1} : p.B) * (p.dms[1] == 0 ? 1 : p.H), n = (p.S + kTile - 1) / kTile;
    if (masks * n * n > 2147483647LL / 16) return false;
    return rows8(p.q, p.qs) && rows8(p.k, p.ks) && rows8(p.v, p.vs) && rows8(p.d_o, p.dos);
}

int64_t mfma_dmask_workspace(const KParams& p) {
    const Plan plan = plan_dmask(p, true);
    return plan.parts > 1 ? static_cast<int64_t>(plan.tiles) * plan.parts * kPartFloats * 4 : 0;
}

int launch_mfma_dmask(int dtype, KParams p, hipStream_t stream) {
    const int64_t bytes = mfma_dmask_workspace(p);
    const bool split = bytes > 0 && p.workspace != nullptr && p.workspace_bytes >= bytes && reinterpret_cast<uintptr_t>(p.workspace) % 16 == 0;
    const Plan plan = plan_dmask(p, split);
    p.partial = static_cast<float*>(p.workspace);
    if (dtype == TRI_ATTN_BF16) launch_dmask_d<bf16_t>(p, plan, stream);
    else launch_dmask_d<f16_t>(p, plan, stream);
    const int rc = static_cast<int>(hipGetLastError());
    if (rc || plan.parts == 1) return rc;
    hipLaunchKernelGGL(dmask_combine_kernel, dim3(static_cast<unsigned>(plan.tiles) * 8), dim3(256), 0, stream, p, plan, fours(p.dmask, p.dms));
    return static_cast<int>(hipGetLastError());
}

}  // namespace tri
