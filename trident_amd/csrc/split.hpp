// Splitting a launch along the streamed dimension. A workgroup of the attention kernels owns 128 or 256 rows and streams all
// tiles of the other operand; a call of few heads has fewer such items than the GPU has room for (B=1 H=4 S=3200 D=128: 52 of
// 256), under the causal mask with one long one per head. Such a launch runs every item as several parts, workgroups that
// stream part_tiles tiles each and leave fp32 accumulators in the caller's workspace; a second launch (mfma_combine.hip) adds
// the parts of an item up in a fixed order and stores the result as the kernel itself would.
// Kernel times, whole and split with the second launch (microseconds, B=1 H=4; forward, dQ, dK/dV):
//   bf16 causal S=6016 D=128 forward   137 -> 51 + 8
//   bf16 causal S=2321 D=128           56, 60, 59 -> 21 + 7, 24 + 5, 26 + 7
//   fp16 causal S=4995 D=64            77, 80, 145 -> 27 + 8, 33 + 6, 50 + 7
//   bf16 key-padding mask S=8192 D=32  129, 199, 274 -> 71 + 7, 78 + 6, 136 + 8
#pragma once
#include "launch.hpp"
#include "mfma_common.hpp"

namespace tri {

// One part: item `tile` of head `bh`, part `index` of `count`; `unit` numbers the parts of a launch.
struct Part {
    int bh, tile, index, count, unit;
};

// Items of a causal launch come in groups of part_group with the same number of parts, one more from group to group.
__device__ __forceinline__ int parts_of(const KParams& p, int tile, int all_tiles) {
    return p.part_group > 0 ? tile / p.part_group + 1 : (all_tiles + p.part_tiles - 1) / p.part_tiles;
}
// First unit (within its head) of an item: the items with most parts come first.
__device__ __forceinline__ int first_unit(const KParams& p, int tile, int items, int all_tiles) {
    if (p.part_group == 0) return tile * parts_of(p, tile, all_tiles);
    const int g = tile / p.part_group;
    int unit = 0;
    for (int k = (items - 1) / p.part_group; k > g; --k) unit += min(p.part_group, items - k * p.part_group) * (k + 1);
    return unit + (tile - g * p.part_group) * (g + 1);
}
// The part of workgroup `bid`; false: there is none (the grid is rounded up to whole rounds of the XCDs). An XCD takes units
// in a row, so that one or two heads' tiles stay in its L2. `items` and `all_tiles` of a head; heavy_first: item 0 streams
// most tiles (dK/dV under the causal mask), so that groups count from the last one.
__device__ __forceinline__ bool map_part(const KParams& p, int bid, int grid, int items, int all_tiles, bool heavy_first, Part* part) {
    const int total = p.B * p.H * p.part_units;
    const int unit = (bid & 7) * (grid >> 3) + (bid >> 3);
    if (unit >= total) return false;
    part->unit = unit;
    part->bh = unit / p.part_units;
    int u = unit % p.part_units;
    if (p.part_group == 0) {
        const int count = parts_of(p, 0, all_tiles);
        part->count = count;
        part->tile = u / count;
        part->index = u % count;
        return true;
    }
    int k = (items - 1) / p.part_group;
    for (; k > 0; --k) {
        const int here = min(p.part_group, items - k * p.part_group) * (k + 1);
        if (u < here) break;
        u -= here;
    }
    part->count = k + 1;
    part->tile = k * p.part_group + u / (k + 1);
    part->index = u % (k + 1);
    if (heavy_first) part->tile = items - 1 - part->tile;
    return true;
}

// Whole items leave out only tiles before the first and behind the last one that is not masked out altogether: in between, probability 0
// times a NaN or an infinity of a hidden key or row reaches the result. So it does from parts, which ask for all of the item's `n` tiles
// (as tile_classes, any n): whether one of them is active, and the first and the end of those that are.
__device__ __forceinline__ bool any_active(const uint8_t* first, int64_t tile_step, int n, int across, int64_t step, int lane) {
    for (int t = 0; t < n; t += 64)
        if (tile_classes(first + t * tile_step, tile_step, min(64, n - t), across, step, lane).active != 0) return true;
    return false;
}
__device__ __forceinline__ int2 active_range(const uint8_t* first, int64_t tile_step, int n, int across, int64_t step, int lane) {
    int2 range = make_int2(0, 0);
    for (int t = 0; t < n; t += 64) {
        const uint64_t active = tile_classes(first + t * tile_step, tile_step, min(64, n - t), across, step, lane).active;
        if (active == 0) continue;
        if (range.y == 0) range.x = t + __builtin_ctzll(active);
        range.y = t + 64 - __builtin_clzll(active);
    }
    return range;
}

// Accumulators of a wave's NB blocks of 32 rows (this lane: row l32) x 32 columns as they are, whole lines per store. `base`: of
// the wave's 32 rows (all columns) in the workspace; first: the wave's first column block. D = 16 has half a block.
template <int NB, int D>
__device__ __forceinline__ void store_partial(const f32x16 (&acc)[NB], float* base, int first, int lane, float sign) {
    f32x4* dst = reinterpret_cast<f32x4*>(base) + first * 256 + lane;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int g = 0; g < (D < 32 ? 2 : 4); ++g)
            dst[(nb * 4 + g) * 64] = f32x4{acc[nb][4 * g] * sign, acc[nb][4 * g + 1] * sign, acc[nb][4 * g + 2] * sign, acc[nb][4 * g + 3] * sign};
}

// Host side. A launch of `items` workgroups of `rows` rows per head, `slots` of which the GPU holds at once, streaming
// ceil(S / 64) tiles (`causal`: as many as the diagonal leaves).
struct SplitShape {
    int rows;          // stationary rows of a workgroup
    int slots_per_cu;  // workgroups a CU holds (registers and LDS)
    int outputs;       // accumulators of D columns per row
    bool statistics;   // two more floats per row
    int min_tiles;     // below so many there is less to win than the second launch costs
    double tile_us;    // a workgroup's time for one tile, alone on its CU
    double cu_us;      // a full CU's time for one tile of one workgroup
    double gain;       // split where the plan's time is below this share of the whole launch's
    double unclassed = 1.0;  // what a tile of a workgroup that streams more than 64, and so does without the mask's classes, takes more
    int whole_rows = 0;      // rows of a whole launch's workgroup, where others than a part's
};
// What masks and dropout add to a tile's time (a mask of keys is read once, or not at all where it is zero).
inline double split_work(const KParams& p) { return (p.mask == nullptr ? 1.0 : p.ms[2] == 0 ? 1.3 : 1.6) * (p.thr8 > 0 ? 1.7 : 1.0); }
// A mask of keys is all zero or all -inf but for a block: kernels that look at classes (up to 64 tiles a workgroup) read next to nothing of
// it, others every tile (whole -> parts of up to 64 tiles, bf16: 4 heads S=11776 D=16 dQ 255 -> 123 us; 16 heads S=9108 D=32 with dropout,
// forward 827 -> 409, dK/dV 1275 -> 632). Of a matrix the host does not know.
inline double split_unclassed(const KParams& p) { return p.mask != nullptr && p.ms[2] == 0 && p.mcls != nullptr ? 1.5 : 1.0; }
// Lengths that are multiples of 128 have faster kernels than the parts, which have boundary handling, most of all beside a mask (a value
// joins its score before the scale, row sums on the matrix pipe). Causal plans turn out faster than they promise: what they cut
// are the long items.
inline double split_gain(const KParams& p) { return (p.S % 128 != 0 ? 0.98 : p.mask != nullptr ? 0.84 : 0.93) + (p.causal ? 0.08 : 0.0); }
// Fills p->part_* and returns the bytes of workspace the split launch needs; 0: the launch stays whole.
int64_t plan_split(const SplitShape& shape, bool causal, KParams* p);
// Whether the caller's workspace holds what plan_split asked for; sets p->partial.
bool take_workspace(int64_t bytes, KParams* p);
inline dim3 split_grid(const KParams& p) { return dim3(static_cast<unsigned>((static_cast<int64_t>(p.B) * p.H * p.part_units + 7) / 8 * 8)); }

// mfma_*_split.hip: TRI_ATTN_ENOFUSE and nothing launched where the workspace does not do
int launch_mfma_fwd_split(int dtype, KParams p, hipStream_t stream);
int launch_mfma_dq_split(int dtype, KParams p, hipStream_t stream, bool with_delta);
int launch_mfma_dkdv_split(int dtype, KParams p, hipStream_t stream);
// mfma_combine.hip
int launch_combine_forward(int dtype, const KParams& p, int rows, hipStream_t stream);
// dQ (dk == nullptr) or dK and dV
int launch_combine_backward(int dtype, const KParams& p, int rows, bool dkdv, hipStream_t stream);

}  // namespace tri
