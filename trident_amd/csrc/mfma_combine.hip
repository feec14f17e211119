// Second launch of a split attention pass (split.hpp): the parts of an item, left as fp32 accumulators in the workspace, become
// the rows of O and lse, of dQ, or of dK and dV. A wave takes 32 rows x 32 columns in the accumulators' own layout (lane = row), adds the
// parts up in their order and stores through the transposition patch of the kernels' epilogues. Bound by the workspace's
// bytes: each is read once, in whole lines, out of the L2 or the Infinity Cache that has just taken it.
#include <algorithm>

#include "split.hpp"

namespace tri {
namespace {

// The wave's place: rows row0 .. row0 + 31 and columns 32 column .. of head bh, block `block` of item `tile`. Waves of items
// that are one part have nothing to do: the kernel stored those itself. A wave takes one block of columns and has four parts
// in flight: with all columns of its rows (D = 128) it took 50 us for what takes 6 (bf16 B=1 H=4 S=1417, dK and dV), one load
// after the other in 180 waves.
struct Place {
    int bh, tile, block, row0, column;
    bool ok;
};
template <int D>
__device__ __forceinline__ Place place_of(const KParams& p, int rows) {
    constexpr int DB = D >= 32 ? D / 32 : 1;
    const int blocks = (p.S + 31) / 32;
    const int64_t w = static_cast<int64_t>(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    Place r;
    r.ok = w < static_cast<int64_t>(p.B) * p.H * blocks * DB;
    r.column = static_cast<int>(w % DB);
    r.bh = static_cast<int>(w / DB / blocks);
    r.row0 = 32 * static_cast<int>(w / DB % blocks);
    r.tile = r.row0 / rows;
    r.block = r.row0 % rows / 32;
    return r;
}

// Where a wave's block goes: 16-bit results through the epilogue's transposition patch, fp32 ones 16 bytes per lane and row.
template <typename T, int COLS>
struct BlockStore : RowBlockStore<T, 1, COLS> {};
template <int COLS>
struct BlockStore<float, COLS> {
    static constexpr int kPatchBytes = 16;
    template <typename Scale>
    static __device__ __forceinline__ void run(const f32x16 (&acc)[1], Scale scale, char*, char* row0, int64_t row_stride_bytes, int lane, int rows) {
        const int l32 = lane & 31, h = lane >> 5;
        if (l32 >= rows) return;
#pragma unroll
        for (int g = 0; g < COLS / 8; ++g)
            *reinterpret_cast<f32x4*>(row0 + l32 * row_stride_bytes + (8 * g + 4 * h) * 4) =
                f32x4{scale(acc[0][4 * g]), scale(acc[0][4 * g + 1]), scale(acc[0][4 * g + 2]), scale(acc[0][4 * g + 3])};
    }
};

template <typename T, int D>
__global__ __launch_bounds__(256) void combine_forward_kernel(const KParams p, int rows) {
    constexpr int G = D < 32 ? 2 : 4;
    using Store = BlockStore<T, D < 32 ? D : 32>;
    __shared__ __attribute__((aligned(1024))) char smem[4 * Store::kPatchBytes];
    const int lane = threadIdx.x & 63, l32 = lane & 31, h = lane >> 5;
    const Place at = place_of<D>(p, rows);
    if (!at.ok) return;
    const int all_tiles = (p.S + 63) / 64, items = (p.S + rows - 1) / rows;
    const int count = parts_of(p, at.tile, all_tiles);
    if (count == 1) return;
    const int64_t unit0 = static_cast<int64_t>(at.bh) * p.part_units + first_unit(p, at.tile, items, all_tiles);
    const int64_t units = static_cast<int64_t>(p.B) * p.H * p.part_units;
    const float2* stats = reinterpret_cast<const float2*>(p.partial + units * rows * D) + unit0 * rows + at.block * 32 + l32;
    float m = -INFINITY;
    bool nan = false;
#pragma unroll 8
    for (int i = 0; i < count; ++i) {
        const float x = stats[static_cast<int64_t>(i) * rows].x;
        nan |= x != x;
        m = fmaxf(m, x);
    }
    if (nan) m = __builtin_nanf("");
    const float ref = m == -INFINITY ? 0.f : m;  // (no score of any part has had a value: the sums are 0, or NaN where scores were)
    f32x16 acc[1] = {zero16()};
    float l = 0.f;
    const f32x4* src = reinterpret_cast<const f32x4*>(p.partial + (unit0 * rows + at.block * 32) * D) + at.column * 256 + lane;
    const int64_t step = static_cast<int64_t>(rows) * D / 4;
#pragma unroll 4
    for (int i = 0; i < count; ++i) {
        const float2 ml = stats[static_cast<int64_t>(i) * rows];
        // (a part without a tile has left nothing but that; every other one takes part, also with weight 0: what its keys' scores
        // and values have made NaN stays NaN)
        const bool none = ml.y < 0.f;
        const float w = fast_exp2(ml.x - ref);
        l += none ? 0.f : w * ml.y;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const f32x4 v = src[i * step + g * 64];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[0][4 * g + e] = fmaf(w, none ? 0.f : v[e], acc[0][4 * g + e]);
        }
    }
    const float inv = (sizeof(T) == 2 && p.thr8 > 0 ? p.zscale : 1.f) / l;  // (the fp32 kernels scale what they keep at once)
    const int b = at.bh / p.H, hd = at.bh % p.H, rows_here = p.S - at.row0;
    char* o0 = static_cast<char*>(p.o) + (b * p.os[0] + hd * p.os[1] + at.row0 * p.os[2] + 32 * at.column) * sizeof(T);
    Store::run(acc, [inv](float x) { return x * inv; }, smem + (threadIdx.x >> 6) * Store::kPatchBytes, o0, p.os[2] * sizeof(T), lane, rows_here);
    if (at.column == 0 && h == 0 && l32 < rows_here) p.lse[static_cast<int64_t>(at.bh) * p.S + at.row0 + l32] = m + fast_log2(l);
}

// OUTPUTS = 2: dK (blockIdx.y = 0) and dV (1); the accumulators of a unit's rows for the first come before those for the second.
template <typename T, int D, int OUTPUTS>
__global__ __launch_bounds__(256) void combine_backward_kernel(const KParams p, int rows) {
    constexpr int G = D < 32 ? 2 : 4;
    using Store = BlockStore<T, D < 32 ? D : 32>;
    __shared__ __attribute__((aligned(1024))) char smem[4 * Store::kPatchBytes];
    const int lane = threadIdx.x & 63;
    const Place at = place_of<D>(p, rows);
    if (!at.ok) return;
    const int all_tiles = (p.S + 63) / 64, items = (p.S + rows - 1) / rows;
    const int tile = OUTPUTS == 2 && p.part_group > 0 ? items - 1 - at.tile : at.tile;  // (causal dK/dV: item 0 streams most rows)
    const int count = parts_of(p, tile, all_tiles);
    if (count == 1) return;
    const int64_t unit0 = static_cast<int64_t>(at.bh) * p.part_units + first_unit(p, tile, items, all_tiles);
    const int b = at.bh / p.H, hd = at.bh % p.H, n = OUTPUTS == 2 ? static_cast<int>(blockIdx.y) : 0;
    f32x16 acc[1] = {zero16()};
    const f32x4* src = reinterpret_cast<const f32x4*>(p.partial + ((unit0 * OUTPUTS + n) * rows + at.block * 32) * D) + at.column * 256 + lane;
    const int64_t step = static_cast<int64_t>(rows) * D / 4 * OUTPUTS;
#pragma unroll 4
    for (int i = 0; i < count; ++i) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const f32x4 v = src[i * step + g * 64];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[0][4 * g + e] += v[e];
        }
    }
    char* to = static_cast<char*>(OUTPUTS == 1 ? p.dq : n == 0 ? p.dk : p.dv);
    const int64_t* s = OUTPUTS == 1 ? p.dqs : n == 0 ? p.dks : p.dvs;
    const float scale = n == 1 ? 1.f : p.scale;
    Store::run(acc, [scale](float x) { return x * scale; }, smem + (threadIdx.x >> 6) * Store::kPatchBytes,
               to + (b * s[0] + hd * s[1] + at.row0 * s[2] + 32 * at.column) * sizeof(T), s[2] * sizeof(T), lane, p.S - at.row0);
}

dim3 combine_grid(const KParams& p, int outputs) {
    const int64_t waves = static_cast<int64_t>(p.B) * p.H * ((p.S + 31) / 32) * (p.D >= 32 ? p.D / 32 : 1);
    return dim3(static_cast<unsigned>((waves + 3) / 4), outputs);
}

template <typename T>
int combine_forward(const KParams& p, int rows, hipStream_t st) {
    const dim3 g = combine_grid(p, 1), block(256);
    if (p.D == 128) hipLaunchKernelGGL((combine_forward_kernel<T, 128>), g, block, 0, st, p, rows);
    else if (p.D == 64) hipLaunchKernelGGL((combine_forward_kernel<T, 64>), g, block, 0, st, p, rows);
    else if (p.D == 32) hipLaunchKernelGGL((combine_forward_kernel<T, 32>), g, block, 0, st, p, rows);
    else hipLaunchKernelGGL((combine_forward_kernel<T, 16>), g, block, 0, st, p, rows);
    return static_cast<int>(hipGetLastError());
}

template <typename T, int OUTPUTS>
int combine_backward(const KParams& p, int rows, hipStream_t st) {
    const dim3 g = combine_grid(p, OUTPUTS), block(256);
    if (p.D == 128) hipLaunchKernelGGL((combine_backward_kernel<T, 128, OUTPUTS>), g, block, 0, st, p, rows);
    else if (p.D == 64) hipLaunchKernelGGL((combine_backward_kernel<T, 64, OUTPUTS>), g, block, 0, st, p, rows);
    else if (p.D == 32) hipLaunchKernelGGL((combine_backward_kernel<T, 32, OUTPUTS>), g, block, 0, st, p, rows);
    else hipLaunchKernelGGL((combine_backward_kernel<T, 16, OUTPUTS>), g, block, 0, st, p, rows);
    return static_cast<int>(hipGetLastError());
}

}  // namespace

int launch_combine_forward(int dtype, const KParams& p, int rows, hipStream_t stream) {
    if (dtype == TRI_ATTN_F32) return combine_forward<float>(p, rows, stream);
    return dtype == TRI_ATTN_BF16 ? combine_forward<bf16_t>(p, rows, stream) : combine_forward<f16_t>(p, rows, stream);
}

int launch_combine_backward(int dtype, const KParams& p, int rows, bool dkdv, hipStream_t stream) {
    if (dtype == TRI_ATTN_F32) return dkdv ? combine_backward<float, 2>(p, rows, stream) : combine_backward<float, 1>(p, rows, stream);
    if (dtype == TRI_ATTN_BF16) return dkdv ? combine_backward<bf16_t, 2>(p, rows, stream) : combine_backward<bf16_t, 1>(p, rows, stream);
    return dkdv ? combine_backward<f16_t, 2>(p, rows, stream) : combine_backward<f16_t, 1>(p, rows, stream);
}

int64_t plan_split(const SplitShape& shape, bool causal, KParams* p) {
    p->part_units = 0;
    const int64_t heads = static_cast<int64_t>(p->B) * p->H;
    const int tiles = (p->S + 63) / 64, items = (p->S + shape.rows - 1) / shape.rows, step = shape.rows / 64;
    const int64_t cus = static_cast<int64_t>(persistent_grid(1 << 20)), slots = cus * shape.slots_per_cu;
    // Microseconds, as measured over 9000 passes of 1 to 40 heads and 193 to 12000 rows: a workgroup's start and end, the second launch,
    // bytes of the workspace (mostly in the caches) that both launches move in one. A CU with several workgroups takes longer for a
    // tile of each than one workgroup alone on it, but less than for that many one after the other.
    constexpr double kFixed = 4, kCombine = 7, kBytesPerUs = 5e6;
    constexpr int64_t kMostBytes = int64_t{1} << 28;  // (what a call may ask its caller for; reached beyond 16384 rows)
    const auto time = [&](int64_t units, int each) {
        const int64_t on_cu = (units + cus - 1) / cus, rounds = (on_cu + shape.slots_per_cu - 1) / shape.slots_per_cu;
        return static_cast<double>(rounds) * kFixed +
               (each > 64 ? shape.unclassed : 1.0) * each * std::max(static_cast<double>(rounds) * shape.tile_us, static_cast<double>(on_cu) * shape.cu_us);
    };
    // A launch with a workgroup for every CU is worth it only where the workgroups are long. One of two full rounds has little to win, unless
    // its parts are what makes use of the mask's classes.
    const int64_t most = shape.unclassed > 1.0 && tiles > 64 ? cus * 256 / std::max(p->D, 32) : 2 * slots;
    if (tiles < shape.min_tiles || heads * items >= most || (tiles < 64 && heads * items >= cus)) return 0;
    // (causal: the longest item shares its CU with others that are half as long on average)
    const int64_t beside = std::min<int64_t>((heads * items + cus - 1) / cus, shape.slots_per_cu) - 1;
    const double whole = causal ? kFixed + std::max(tiles * std::max(shape.tile_us, shape.cu_us * (1.0 + 0.5 * static_cast<double>(beside))),
                                                    static_cast<double>(heads) * items * (tiles + step) / 2.0 * shape.cu_us / cus)
                                : time(heads * (shape.whole_rows > 0 ? (p->S + shape.whole_rows - 1) / shape.whole_rows : items), tiles);
    const int64_t unit_bytes = shape.rows * (static_cast<int64_t>(p->D) * shape.outputs + (shape.statistics ? 2 : 0)) * 4;
    double best = shape.gain * whole;
    for (int c = std::max(shape.min_tiles / 5, step); c < tiles; c += causal ? step : 1) {  // (parts of at least a fifth of min_tiles)
        int64_t units;
        if (causal) {
            const int64_t group = c / step, full = items / group, rest = items % group;
            units = group * full * (full + 1) / 2 + rest * (full + 1);
        } else {
            units = static_cast<int64_t>(items) * ((tiles + c - 1) / c);
        }
        if (heads * units * unit_bytes > kMostBytes) continue;
        const double t = time(heads * units, c) + kCombine + 2.0 * heads * units * unit_bytes / kBytesPerUs;
        if (t < best) {
            best = t;
            p->part_units = static_cast<int>(units);
            p->part_tiles = c;
            p->part_group = causal ? c / step : 0;
        }
    }
    return heads * p->part_units * unit_bytes;
}

bool take_workspace(int64_t bytes, KParams* p) {
    if (bytes > 0 && p->workspace != nullptr && p->workspace_bytes >= bytes && reinterpret_cast<uintptr_t>(p->workspace) % 16 == 0) {
        p->partial = static_cast<float*>(p->workspace);
        return true;
    }
    p->part_units = 0;
    return false;
}

}  // namespace tri
