// Row softmax, masked row softmax and dropout: the HBM-bound sibling operations of the attention path
// (C ABI in include/tri_rowops.h). Statistics are kept in fp32 in the log2 domain, as in the attention kernels.
#include <math.h>
#include <stddef.h>
#include <string.h>

#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "tri_rowops.h"

namespace tri {
namespace {

constexpr float kMaskEps = 2.220446049250313e-16f;  // trident/language/constant.py:17-20 (eps)
constexpr uint32_t kDropoutStream = 0x44524F50u;    // counter word 2 of the stand-alone dropout ("DROP")

struct RowParams {
    const void* input;
    void* output;
    const void* mask;
    const void* grad_output;
    void* grad_input;
    int64_t y_size, x_size, y_stride, x_stride;
    int mask_dtype;
    uint32_t seed_lo, seed_hi, offset;
    int thr8;
    float zscale;
    // columns split along their length: elements of a part and number of parts, and what the parts leave for each column
    int64_t part_size;
    int parts;
    void* part_stats;
    void* workspace;
    int64_t workspace_bytes;
};

// M = element type of the mask (void: no mask). A position is masked where its mask value exceeds eps
// (trident/kernel/masked_softmax.py:76), i.e. is positive for the integer types.
template <typename M>
__device__ __forceinline__ bool mask_hit(const void* base, int64_t off) {
    if constexpr (std::is_same<M, void>::value) return false;
    else if constexpr (std::is_integral<M>::value) return static_cast<const M*>(base)[off] > 0;
    else return to_f32(static_cast<const M*>(base)[off]) > kMaskEps;
}

// (max, sum) pairs of a softmax in the log2 domain and their merge (the reference's language.combine_softmax,
// trident/language/combine.py:30-33); a -inf maximum stands for "nothing seen yet".
struct Stat {
    float m, l;
};
// Exponents are fma(x, log2 e, -reference(m)) with m, the maximum times log2 e, rounded: a factor common to all exponentials,
// which the division by their sum takes out again. Half a unit in the last place of m is 64 at 1.6e9 and overflows beyond, so
// that the reference goes no lower (elements below it are 0 beside any that are not, also where a thread or a wave sees no
// other), and rows whose maximum is that far from 0 are computed once more with the maximum subtracted from their elements
// before the product (far_from_zero; a row of nothing but -1e10 would have the sum 0 or infinity).
__device__ __forceinline__ float reference(float m) { return fmaxf(m, -1.6e9f); }
__device__ __forceinline__ bool far_from_zero(float m) { return fabsf(m) > 1.5e9f && m > -INFINITY; }
__device__ __forceinline__ Stat merge(Stat a, Stat b) {
    const float m = fmaxf(a.m, b.m), ms = reference(m);
    return Stat{m, a.l * fast_exp2(a.m - ms) + b.l * fast_exp2(b.m - ms)};
}

template <typename T, int V>
struct alignas(sizeof(T) * V) Vec {
    T e[V];
};

// mask hits of V consecutive elements, bit e = element e
template <typename M, int V>
__device__ __forceinline__ uint32_t mask_bits(const void* base, int64_t off) {
    if constexpr (std::is_same<M, void>::value) {
        return 0u;
    } else {
        struct alignas(sizeof(M) * V > 16 ? 16 : sizeof(M) * V) Pack {
            M e[V];
        };
        const Pack v = *reinterpret_cast<const Pack*>(static_cast<const M*>(base) + off);
        uint32_t bits = 0;
#pragma unroll
        for (int e = 0; e < V; ++e) bits |= mask_hit<M>(v.e, e) ? 1u << e : 0u;
        return bits;
    }
}

// V elements of a row as they lie in memory, in whole registers: 16-bit elements held one by one take a register each.
template <typename T, int V>
struct Piece {
    static constexpr int kWords = V * sizeof(T) >= 4 ? V * sizeof(T) / 4 : 1;
    uint32_t w[kWords];
    __device__ __forceinline__ void load(const T* from) {
        if constexpr (V * sizeof(T) >= 4) {
            struct alignas(V * sizeof(T)) Words {
                uint32_t w[kWords];
            };
            const Words v = *reinterpret_cast<const Words*>(from);
#pragma unroll
            for (int i = 0; i < kWords; ++i) w[i] = v.w[i];
        } else {
            w[0] = *reinterpret_cast<const uint16_t*>(from);
        }
    }
    __device__ __forceinline__ void fill(float x) {
        const uint32_t b = bits(x);
#pragma unroll
        for (int i = 0; i < kWords; ++i) w[i] = b;
    }
    __device__ __forceinline__ float get(int e) const {
        if constexpr (sizeof(T) == 4) return __uint_as_float(w[e]);
        else return to_f32(__builtin_bit_cast(T, static_cast<uint16_t>(w[e >> 1] >> (16 * (e & 1)))));
    }
    __device__ __forceinline__ void set(int e, float x) {
        const uint32_t half = sizeof(T) == 4 ? 0xffffffffu : 0xffffu << (16 * (e & 1));
        uint32_t& word = w[sizeof(T) == 4 ? e : e >> 1];
        word = (word & ~half) | (bits(x) & half);
    }
    // elements outside [lo, hi): x
    __device__ __forceinline__ void trim(int lo, int hi, float x) {
        const uint32_t b = bits(x);
        constexpr int kPer = sizeof(T) == 4 ? 1 : 2;  // elements of a word
#pragma unroll
        for (int i = 0; i < kWords; ++i) {
            uint32_t keep = i * kPer >= lo && i * kPer < hi ? (kPer == 1 ? 0xffffffffu : 0xffffu) : 0u;
            if constexpr (kPer == 2) keep |= i * kPer + 1 >= lo && i * kPer + 1 < hi ? 0xffff0000u : 0u;
            w[i] = (w[i] & keep) | (b & ~keep);
        }
    }
    // element e (not known to the compiler) := the element whose bits() are b, as far as it lies in word i
    __device__ __forceinline__ void put(int i, int e, uint32_t b) {
        constexpr int kPer = sizeof(T) == 4 ? 1 : 2;
        const uint32_t half = kPer == 1 ? 0xffffffffu : 0xffffu << (16 * (e & 1));
        w[i] = e / kPer == i ? (w[i] & ~half) | (b & half) : w[i];
    }
    // converted anew by the next reader: values kept across would take twice the registers of the words
    __device__ __forceinline__ void hide() {
#pragma unroll
        for (int i = 0; i < kWords; ++i) asm volatile("" : "+v"(w[i]));
    }
    static __device__ __forceinline__ uint32_t bits(float x) {
        if constexpr (sizeof(T) == 4) return __float_as_uint(x);
        else return __builtin_bit_cast(uint16_t, from_f32<T>(x)) * 0x10001u;
    }
};

// ------------------------------------------------------------------ rows with unit stride along x
// Mask of V consecutive elements on its way from memory to a Piece: as it lies there where that is 16 bytes or less, so that a
// thread's mask loads are all in flight before the first is looked at, as bits where it is more. (Each piece's bits made, and its
// elements selected one by one, as it came: bf16 16384 x 1000 with a uint8 mask 0.0174 -> 0.0153 ms, fp32 1024 x 8192 0.0207 -> 0.0135,
// of which the order of the second sweep, below, is a part.)
template <typename M, int V>
struct MaskPiece {
    static constexpr bool kRaw = sizeof(M) * V <= 16;
    struct alignas(kRaw ? sizeof(M) * V : alignof(M)) Raw {
        M e[kRaw ? V : 1];
    };
    Raw raw;
    uint32_t bits;
    __device__ __forceinline__ void load(const void* base, int64_t off) {
        if constexpr (kRaw) raw = *reinterpret_cast<const Raw*>(static_cast<const M*>(base) + off);
        else bits = mask_bits<M, V>(base, off);
    }
    // elements [lo, hi) one by one, the others not masked
    __device__ __forceinline__ void load(const void* base, int64_t off, int lo, int hi) {
        bits = 0;
#pragma unroll
        for (int e = 0; e < V; ++e) {
            const bool live = e >= lo && e < hi;
            if constexpr (kRaw) raw.e[e] = live ? static_cast<const M*>(base)[off + e] : static_cast<M>(0);
            else if (live && mask_hit<M>(base, off + e)) bits |= 1u << e;
        }
    }
    __device__ __forceinline__ void clear() { load(nullptr, 0, 0, 0); }  // nothing masked
    // masked elements: -inf
    template <typename T>
    __device__ __forceinline__ void apply(Piece<T, V>& piece) const {
        if constexpr (kRaw && sizeof(M) == 1 && sizeof(T) == 2 && V % 4 == 0) {
            // bytes to halfwords: the top bit of a byte that is not 0, moved to the top of its halfword and spread over it
            typedef short Halves __attribute__((ext_vector_type(2)));
            const uint32_t inf = Piece<T, V>::bits(-INFINITY);
#pragma unroll
            for (int q = 0; q < V / 4; ++q) {
                const uint32_t w = __builtin_bit_cast(Words, raw).w[q];
                const uint32_t top = ((w & 0x7f7f7f7fu) + 0x7f7f7f7fu) | w;
                const uint32_t low = __builtin_bit_cast(uint32_t, __builtin_bit_cast(Halves, __builtin_amdgcn_perm(top, top, 0x010c000cu)) >> 15);
                const uint32_t high = __builtin_bit_cast(uint32_t, __builtin_bit_cast(Halves, __builtin_amdgcn_perm(top, top, 0x030c020cu)) >> 15);
                piece.w[2 * q] = (inf & low) | (piece.w[2 * q] & ~low);
                piece.w[2 * q + 1] = (inf & high) | (piece.w[2 * q + 1] & ~high);
            }
        } else {
#pragma unroll
            for (int e = 0; e < V; ++e)
                if (kRaw ? mask_hit<M>(raw.e, e) : (bits >> e & 1) != 0) piece.set(e, -INFINITY);
        }
    }

private:
    struct Words {
        uint32_t w[sizeof(Raw) >= 4 ? sizeof(Raw) / 4 : 1];
    };
};

// HBM-bound: one read and one write of every tensor. G threads share a row (16 or 64 of a wave for short rows, the whole
// workgroup for long ones); a row is worked through in pieces of V elements (16 bytes), kHeld of them per thread at a
// time, all loaded together. A row of up to G * V * kHeld elements stays in registers between the statistics and the
// output; a longer one takes two sweeps, the second of which finds the row in the L2 it was just read through.
// SHIFT: rows that do not start on 16-byte boundaries (an odd row length): the pieces are those of the tensor, not of the
// row. A row's first and last piece, which it shares with its neighbours, are read whole, too, and trimmed in registers, so that all
// of a thread's loads are in flight before the first is looked at; only what lies behind the tensor's last whole piece is read element by
// element, and the two pieces are written so. (Read element by element, a branch each, they held up the loads behind them and were
// most of the vector work. Launches in a row, us, bf16 12288 x 2047 with a uint8 mask: forward 37 -> 27 = 4.6 TB/s, backward 33 -> 26; fp16
// 17740 x 2589 with the mask 113 -> 73, backward 86 -> 62; bf16 65536 x 197 24 -> 18; fp32 23855 x 477, backward, 28 -> 24.) One element
// per load, which still serves short odd rows and tensors that are not 16-byte aligned themselves, 0.0545 and 0.0493 ms. Rows on 16-byte
// boundaries: bf16 65536 x 64 forward 0.0092 ms (a wave per row, most of it idle: 0.0265), fp32 8192 x 1536 backward 0.0226
// (two sweeps: 0.0362), bf16 16384 x 8192 forward 0.1027 (5.2 TB/s), with the mask 0.134 (one mask byte per load: 0.139).
constexpr int held_pieces(bool shift) { return shift ? 5 : 4; }  // (a shifted row has up to one piece more)

template <typename T, int V, int G, bool SHIFT>
struct RowPlace {
    int t;            // this thread's position in its row
    bool live;
    int64_t at0;      // element offset of the row's piece 0
    int shift;        // where in piece 0 the row starts
    int64_t pieces;   // number of pieces of the row
    int64_t readable; // pieces from the row's first on that end within the tensor
    int64_t x_size;
    __device__ __forceinline__ explicit RowPlace(const RowParams& p) : x_size(p.x_size) {
        t = threadIdx.x % G;
        // (a wave has one row from G == 64 on: what follows from its number stays in scalar registers)
        const int in_group = threadIdx.x / G;
        const int64_t row = static_cast<int64_t>(blockIdx.x) * (256 / G) + (G >= 64 ? __builtin_amdgcn_readfirstlane(in_group) : in_group);
        live = row < p.y_size;  // (G == 256: always)
        at0 = (live ? row : 0) * p.y_stride;
        shift = SHIFT ? static_cast<int>(at0 % V) : 0;
        at0 -= shift;
        pieces = live ? (x_size + shift + V - 1) / V : 0;
        readable = ((p.y_size - 1) * p.y_stride + x_size - at0) / V;
    }
    // G pieces of the row from piece `first` on, one per thread.
    struct Step {
        int64_t at;     // element offset of the first one
        bool head;      // it is the row's first piece
        int count, end; // how many pieces there are of the row, and the number of the row's elements from `at` on
        int readable;   // how many end within the tensor
    };
    static __device__ __forceinline__ int bounded(int64_t x) { return static_cast<int>(min(x, static_cast<int64_t>(1) << 20)); }
    __device__ __forceinline__ Step step(int64_t first) const {
        return Step{at0 + first * V, first == 0, bounded(pieces - first), bounded(live ? x_size + shift - first * V : 0), bounded(readable - first)};
    }
    // the row's elements [lo, hi) of this thread's piece (V > 1 without SHIFT: always the whole piece); hi < 1: it is not a piece of the row
    __device__ __forceinline__ void range(const Step& s, int* lo, int* hi) const {
        *lo = s.head && t == 0 ? shift : 0;
        *hi = min(s.end - t * V, V);
    }
    __device__ __forceinline__ bool whole(const Step& s) const { return !SHIFT || (!(s.head && t == 0 && shift != 0) && (t + 1) * V <= s.end); }
    // where this thread reads its piece: with SHIFT one that ends within the tensor, whatever it is
    __device__ __forceinline__ int read_at(const Step& s) const { return (SHIFT ? min(t, s.readable - 1) : t) * V; }
    // Pieces c0 + k * G + t of the row. All of them are requested before the first is looked at. With SHIFT a row's first and last
    // piece come whole, with their neighbours' elements, and are trimmed in registers (trim); only a piece behind the last one that ends
    // within the tensor is read element by element. (Pieces whose number is beyond every thread's share are skipped by a branch the
    // whole row takes.)
    __device__ __forceinline__ void load(const T* base, const Step& s, Piece<T, V>& held, float outside) const {
        if (SHIFT ? s.count > 0 : t < s.count) held.load(base + s.at + read_at(s));
        else held.fill(outside);
    }
    // (once all loads are on their way; element(offset): the value of one element)
    template <typename Element>
    __device__ __forceinline__ void trim(const Step& s, Piece<T, V>& held, float outside, Element element) const {
        if constexpr (SHIFT) {
            if (s.count <= 0 || whole(s)) return;
            int lo, hi;
            range(s, &lo, &hi);
            asm volatile("" : "+v"(lo), "+v"(hi));  // (comparisons made where they are needed, not kept as lane masks)
            held.trim(lo, hi, outside);
            if (t >= s.readable && t < s.count) {
#pragma unroll 1
                for (int e = lo; e < hi; ++e) {
                    const uint32_t b = Piece<T, V>::bits(element(s.at + t * V + e));
#pragma unroll
                    for (int w = 0; w < Piece<T, V>::kWords; ++w) held.put(w, e, b);
                }
            }
        }
    }
    // The mask's piece beside one. (What it says of elements that are not the row's does not matter: they are trimmed behind it.)
    template <typename M, bool PIECES>
    __device__ __forceinline__ void mask(const void* base, const Step& s, MaskPiece<M, V>& r) const {
        if constexpr (PIECES) {
            r.load(base, s.at + read_at(s));
        } else {
            int lo = 0, hi = V;
            if (!whole(s)) range(s, &lo, &hi);
            r.load(base, s.at + t * V, lo, hi);
        }
    }
    // Output of the held pieces c0 + k * G + t, value(k, e) each: whole pieces at once; a row's first and last, of which a thread has at most
    // one unless the last falls to thread 0, element by element in one pass behind the others.
    template <int N, typename Value>
    __device__ __forceinline__ void store(T* base, int64_t c0, Value value) const {
        [[maybe_unused]] Vec<T, V> rest;
        [[maybe_unused]] int lo = 0, hi = 0;
        [[maybe_unused]] T* rest_to = base;
        [[maybe_unused]] auto store_rest = [&]() {
            if (lo < hi) {
#pragma unroll
                for (int e = 0; e < V; ++e)
                    if (e >= lo && e < hi) rest_to[e] = rest.e[e];
                hi = 0;
            }
        };
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const Step s = step(c0 + k * G);
            if (t < s.count) {
                Vec<T, V> v;
#pragma unroll
                for (int e = 0; e < V; ++e) v.e[e] = from_f32<T>(value(k, e));
                T* to = base + s.at + t * V;
                if (whole(s)) {
                    *reinterpret_cast<Vec<T, V>*>(to) = v;
                } else if constexpr (SHIFT) {
                    range(s, &lo, &hi);
                    rest = v;
                    rest_to = to;
                }
            }
            if constexpr (SHIFT) {
                if (k == 0 && (pieces - 1) % G == 0) store_rest();
            }
        }
        if constexpr (SHIFT) store_rest();
    }
};

// Softmax of a row or column whose maximum is far from zero, element by element: one of the threads t, t + threads, ... that
// share it. maximum and sum reduce over them.
template <typename T, typename M, typename Maximum, typename Sum>
__device__ __forceinline__ void softmax_far(const RowParams& p, int64_t base, int64_t stride, int64_t size, int t, int threads, Maximum maximum, Sum sum) {
    const auto element = [&](int64_t i) {
        const int64_t at = base + i * stride;
        return mask_hit<M>(p.mask, at) ? -INFINITY : to_f32(static_cast<const T*>(p.input)[at]);
    };
    float m = -INFINITY, l = 0.f;
#pragma unroll 1
    for (int64_t i = t; i < size; i += threads) m = fmaxf(m, element(i));
    m = maximum(m);
    const float ms = m == -INFINITY ? 0.f : m;
#pragma unroll 1
    for (int64_t i = t; i < size; i += threads) l += fast_exp2((element(i) - ms) * kLog2e);
    const float inv = 1.f / sum(l);
#pragma unroll 1
    for (int64_t i = t; i < size; i += threads)
        static_cast<T*>(p.output)[base + i * stride] = from_f32<T>(fast_exp2((element(i) - ms) * kLog2e) * inv);
}

// Reduction over the lanes of a wave from distance `from` up to `to`, and over the waves of the workgroup through LDS if there are
// several.
template <typename Op>
__device__ __forceinline__ float reduce(float x, int from, int to, int waves, float* shared, Op op) {
    for (int d = from; d < to; d <<= 1) x = op(x, __shfl_xor(x, d));
    if (waves > 1) {
        __syncthreads();  // (what was there has been read)
        if ((threadIdx.x & 63) == 0) shared[threadIdx.x >> 6] = x;
        __syncthreads();
        x = shared[0];
        for (int w = 1; w < waves; ++w) x = op(x, shared[w]);
    }
    return x;
}
struct MaxOp {
    __device__ __forceinline__ float operator()(float a, float b) const { return fmaxf(a, b); }
};
struct SumOp {
    __device__ __forceinline__ float operator()(float a, float b) const { return a + b; }
};

// PIECES: the mask, too, starts on a 16-byte boundary; otherwise it alone is read element by element (bf16 4096 x 8192, uint8
// mask one byte off: 0.0305 ms, with everything read so 0.0750; 16384 x 1024 0.0180 and 0.0347).
template <typename T, int V, int G, bool SHIFT, typename M, bool PIECES = true>
__global__ __launch_bounds__(256) void softmax_fwd_rows_kernel(const RowParams p) {
    __shared__ Stat part[4];
    constexpr int kHeld = held_pieces(SHIFT);
    constexpr bool kOnce = V > 1 && G < 256;  // (launch_rows: the row fits)
    const RowPlace<T, V, G, SHIFT> row(p);
    const T* in = static_cast<const T*>(p.input);
    T* out = static_cast<T*>(p.output);
    Piece<T, V> held[kHeld];
    auto load = [&](int64_t c0) {  // masked elements and those that are not the row's: -inf
#pragma unroll
        for (int k = 0; k < kHeld; ++k) row.load(in, row.step(c0 + k * G), held[k], -INFINITY);
        if constexpr (!std::is_same<M, void>::value) {
            MaskPiece<M, V> masks[kHeld];
#pragma unroll
            for (int k = 0; k < kHeld; ++k) {
                const auto step = row.step(c0 + k * G);
                if (row.t < step.count) row.template mask<M, PIECES>(p.mask, step, masks[k]);
            }
#pragma unroll
            for (int k = 0; k < kHeld; ++k)
                if (row.t < row.step(c0 + k * G).count) masks[k].apply(held[k]);
        }
#pragma unroll
        for (int k = 0; k < kHeld; ++k)
            row.trim(row.step(c0 + k * G), held[k], -INFINITY, [&](int64_t at) { return mask_hit<M>(p.mask, at) ? -INFINITY : to_f32(in[at]); });
    };
    Stat s{-INFINITY, 0.f};
    int64_t last = 0;
    for (int64_t c0 = 0; c0 < (kOnce ? 1 : row.pieces); c0 += G * kHeld) {
        last = c0;
        load(c0);
        float mx = -INFINITY;
#pragma unroll
        for (int k = 0; k < kHeld; ++k)
            if (c0 + k * G < row.pieces) {
#pragma unroll
                for (int e = 0; e < V; ++e) mx = fmaxf(mx, held[k].get(e));
                held[k].hide();
            }
        const float m = fmaxf(s.m, mx * kLog2e), ms = reference(m);
        float l = s.l * fast_exp2(s.m - ms);
#pragma unroll
        for (int k = 0; k < kHeld; ++k)
            if (c0 + k * G < row.pieces) {
#pragma unroll
                for (int e = 0; e < V; ++e) l += fast_exp2(fmaf(held[k].get(e), kLog2e, -ms));
                held[k].hide();
            }
        s = Stat{m, l};
    }
#pragma unroll
    for (int d = 1; d < (G < 64 ? G : 64); d <<= 1) s = merge(s, Stat{__shfl_xor(s.m, d), __shfl_xor(s.l, d)});
    if constexpr (G == 256) {
        if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
        __syncthreads();
        s = merge(merge(part[0], part[1]), merge(part[2], part[3]));
    }
    if (__builtin_amdgcn_ballot_w64(far_from_zero(s.m)) != 0) {  // (G == 256: the same in all waves)
        constexpr int kLanes = G < 64 ? G : 64;
        float* const shared = &part[0].m;
        softmax_far<T, M>(p, row.at0 + row.shift, 1, row.live ? p.x_size : 0, row.t, G,
                          [&](float x) { return reduce(x, 1, kLanes, G / kLanes, shared, MaxOp{}); },
                          [&](float x) { return reduce(x, 1, kLanes, G / kLanes, shared, SumOp{}); });
        return;
    }
    const float ms = reference(s.m), inv = 1.f / s.l;  // a fully masked row: 0 * inf = NaN, as softmax gives
    // the other way round: what the first sweep read last is still here (bf16 500 x 16384 masked 0.0113 -> 0.0100 ms, one sweep
    // like the other 0.0130 before masks went as they do now; fp32 4096 x 8192 0.0575 -> 0.0488)
    for (int64_t c0 = kOnce ? 0 : last; c0 >= 0; c0 -= G * kHeld) {
        if (!kOnce && c0 != last) load(c0);
        row.template store<kHeld>(out, c0, [&](int k, int e) { return fast_exp2(fmaf(held[k].get(e), kLog2e, -ms)) * inv; });
    }
}

template <typename T, int V, int G, bool SHIFT>
__global__ __launch_bounds__(256) void softmax_bwd_rows_kernel(const RowParams p) {
    __shared__ float part[4];
    constexpr int kHeld = held_pieces(SHIFT);
    constexpr bool kOnce = V > 1 && G < 256;  // (launch_rows: the row fits)
    const RowPlace<T, V, G, SHIFT> row(p);
    const T* o = static_cast<const T*>(p.output);
    const T* g = static_cast<const T*>(p.grad_output);
    T* gi = static_cast<T*>(p.grad_input);
    Piece<T, V> held_o[kHeld], held_g[kHeld];
    auto load = [&](int64_t c0) {
#pragma unroll
        for (int k = 0; k < kHeld; ++k) {
            const auto step = row.step(c0 + k * G);
            if (SHIFT ? step.count > 0 : row.t < step.count) {  // (one branch for both)
                held_o[k].load(o + step.at + row.read_at(step));
                held_g[k].load(g + step.at + row.read_at(step));
            } else {
                held_o[k].fill(0.f);
                held_g[k].fill(0.f);
            }
        }
#pragma unroll
        for (int k = 0; k < kHeld; ++k) {
            row.trim(row.step(c0 + k * G), held_o[k], 0.f, [&](int64_t at) { return to_f32(o[at]); });
            row.trim(row.step(c0 + k * G), held_g[k], 0.f, [&](int64_t at) { return to_f32(g[at]); });
        }
    };
    float delta = 0.f;
    int64_t last = 0;
    for (int64_t c0 = 0; c0 < (kOnce ? 1 : row.pieces); c0 += G * kHeld) {
        last = c0;
        load(c0);
#pragma unroll
        for (int k = 0; k < kHeld; ++k)
            if (c0 + k * G < row.pieces) {
#pragma unroll
                for (int e = 0; e < V; ++e) delta = fmaf(held_o[k].get(e), held_g[k].get(e), delta);
                held_o[k].hide();
                held_g[k].hide();
            }
    }
#pragma unroll
    for (int d = 1; d < (G < 64 ? G : 64); d <<= 1) delta += __shfl_xor(delta, d);
    if constexpr (G == 256) {
        if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = delta;
        __syncthreads();
        delta = (part[0] + part[1]) + (part[2] + part[3]);
    }
    // the other way round, as in the forward (fp32 4096 x 8192 0.0964 -> 0.0774 ms, bf16 1024 x 12288 0.0186 -> 0.0154)
    for (int64_t c0 = kOnce ? 0 : last; c0 >= 0; c0 -= G * kHeld) {
        if (!kOnce && c0 != last) load(c0);
        row.template store<kHeld>(gi, c0, [&](int k, int e) { return held_o[k].get(e) * (held_g[k].get(e) - delta); });
    }
}

// ------------------------------------------------------------------ columns: neighbouring lanes on neighbouring rows
// Softmax along dim 0 of a row-major matrix (y_stride == 1: the softmax "rows" are its columns), and every layout whose
// x_stride is not 1. HBM-bound like the row kernels, with the matrix cut into panels of a few columns: a workgroup owns a
// panel of L lanes x V elements (16 bytes per lane where the geometry allows it) and all of its length; the threads of a
// lane position take every RG-th element down the column. The first kColHeld pieces of a thread are loaded at once and
// stay in registers between statistics and output, so a panel of up to RG x kColHeld elements of length is read once;
// a longer one is swept twice (the second sweep finds it in L2 or the Infinity Cache as far as it fits). Neighbouring
// panels go to the same XCD: where a panel row is narrower than a 128-byte line, the other half is then still in its L2.
// The statistics' LDS is sized by the workgroup, so that single-wave ones fill a CU.
// fp32 4096 x 4096 along dim 0, launches in a row: forward 0.0254 ms = 5.3 TB/s (what a large copy reaches), backward 0.0435 ms =
// 4.6 TB/s (in a training step, whose four tensors fill the Infinity Cache, 0.031 and 0.059 ms). One
// thread per column, which this replaces, took 2.1 and 2.4 ms: 64 waves in flight on the whole chip, each waiting for one
// load at a time. (Its sums ran in plain order, too: at 65536 elements off by 7.5e-5, these by 1.8e-7.)
constexpr int kColHeld = 16;        // forward: pieces a thread keeps (64 registers)
constexpr int kColHeldBwd = 8;      // backward: of each of its two inputs

struct ColPlace {
    int lane, group, groups;  // lane position in the panel, row group of this thread and their number
    int64_t first;            // the panel's first column
    int64_t base;             // element offset of this thread's first column (in its part)
    int64_t x_size;           // length of the column (of the part)
    bool live;
};
// A column launch does all of a column's work in one workgroup (kWhole), or, where that leaves CUs idle and sweeps long columns
// twice, in two launches of parts (blockIdx.y): one leaves each column's statistics in the workspace (kStatistics), the next
// reads those of all parts and writes its own part (kOutput). Microseconds, forward and backward, one workgroup per panel ->
// split: bf16 38122 x 424 with a uint8 mask 399 and 327 -> 61 and 57, fp16 29960 x 156 186 and 251 -> 34 and 39, bf16 9485 x 232
// with mask 111 and 79 -> 25 and 15.
enum ColWork { kWhole = 0, kStatistics = 1, kOutput = 2 };
template <ColWork W>
__device__ __forceinline__ void place_in_part(const RowParams& p, ColPlace* c) {
    if constexpr (W != kWhole) {
        const int64_t row0 = blockIdx.y * p.part_size;
        c->x_size = min(p.part_size, p.x_size - row0);
        if (c->live) c->base += row0 * p.x_stride;
    }
}
template <ColWork W>
__device__ __forceinline__ int64_t length(const RowParams& p, const ColPlace& c) {
    return W == kWhole ? p.x_size : c.x_size;
}
// Columns of a panel's statistics over all parts, merged in their order by as many threads as there are: thread t takes column
// t % columns and every (threads / columns)-th part, and `shared` takes what these leave.
template <typename S, typename Merge>
__device__ __forceinline__ void merge_parts(const RowParams& p, const ColPlace& c, int columns, S none, S* shared, Merge merge) {
    const S* stats = static_cast<const S*>(p.part_stats);
    const int chunks = max(1, static_cast<int>(blockDim.x) / columns);
    for (int t = threadIdx.x; t < columns * chunks; t += blockDim.x) {
        const int64_t col = c.first + t % columns;
        S x = none;
        if (col < p.y_size)
            for (int i = t / columns; i < p.parts; i += chunks) x = merge(x, stats[i * p.y_size + col]);
        shared[t] = x;
    }
    __syncthreads();
    for (int t = threadIdx.x; t < columns; t += blockDim.x) {
        S x = shared[t];
        for (int i = 1; i < chunks; ++i) x = merge(x, shared[i * columns + t]);
        shared[t] = x;
    }
    __syncthreads();
}
__device__ __forceinline__ bool place_in_panel(const RowParams& p, int v, int lanes_log2, int64_t panels, ColPlace* c, bool narrow = false) {
    const int64_t per_xcd = (panels + 7) / 8;
    int64_t i = blockIdx.x >> 3;
    // Panels of 32 bytes, one workgroup per CU, run in up to four rounds of an XCD's 32 CUs. In order, a round covers every other KiB of
    // the matrix's rows, which the HBM channels take badly; so the first half takes the even 128-byte lines and the second the odd ones
    // (fp32 4096 x 4096, forward and backward, 102 -> 93.6 us; pieces of 64 bytes 100.7, of 256 bytes 94.8, the lines dealt to the XCDs
    // in turn 95.5). Forward and backward, in order -> dealt, us: two rounds, fp32 2304 x 4096 58.6 -> 56.6, 4096 x 3072 93.0 -> 90.6,
    // bf16 4096 x 8192 106 -> 97.5; three, fp32 4096 x 5120 146 -> 142.6, 4096 x 6144 153 -> 151, 4096 x 4608 138.5 -> 138.2; four, 4096 x
    // 7680 206 -> 200. One round (4096 x 2048) and numbers of panels that do not divide (2304 columns) are as they were. The backward
    // alone gains up to 16 % in two and four full rounds; in between it is from 1.5 % faster to 3 % slower (2304 x 6144 58.6 -> 60.3).
    if (narrow && per_xcd % 8 == 0) {
        const int64_t half = per_xcd / 8, u = i >> 2;
        i = ((u < half ? 2 * u : 2 * (u - half) + 1) << 2) + (i & 3);
    }
    const int64_t panel = (blockIdx.x & 7) * per_xcd + i;
    if (panel >= panels) return false;  // (the whole workgroup)
    c->lane = threadIdx.x & ((1 << lanes_log2) - 1);
    c->group = threadIdx.x >> lanes_log2;
    c->groups = blockDim.x >> lanes_log2;
    c->first = (panel << lanes_log2) * v;
    const int64_t col = c->first + c->lane * v;
    c->live = col < p.y_size;
    c->base = c->live ? col * p.y_stride : 0;
    return true;
}

// Element offset of piece k of a sweep step that starts at r0, and whether it exists, walked from k = 0 on. The offset is
// hidden from the compiler at every step: left to itself it keeps all addresses of a step from the loads to the stores
// (two registers each, which the held pieces need).
struct ColWalk {
    int64_t at, step;
    int left, groups;  // elements from this one to the column's end
    __device__ __forceinline__ ColWalk(const RowParams& p, const ColPlace& c, int64_t length, int64_t r0)
        : at((r0 + c.group) * p.x_stride), step(c.groups * p.x_stride), left(0), groups(c.groups) {
        const int64_t rest = length - r0 - c.group;
        left = !c.live || rest < 0 ? 0 : (rest > 0x3fffffff ? 0x3fffffff : static_cast<int>(rest));
        asm volatile("" : "+v"(at), "+v"(left));
    }
    __device__ __forceinline__ bool exists() const { return left > 0; }
    __device__ __forceinline__ void next() {
        at += step;
        left -= groups;
        asm volatile("" : "+v"(at), "+v"(left));
    }
};

template <typename T, int V, typename M, ColWork W = kWhole>
__global__ __launch_bounds__(1024) void softmax_fwd_cols_kernel(const RowParams p, int lanes_log2, int64_t panels) {
    extern __shared__ Stat part[];  // one per wave and column of the panel
    ColPlace c;
    if (!place_in_panel(p, V, lanes_log2, panels, &c)) return;
    place_in_part<W>(p, &c);
    using VT = Vec<T, V>;
    const T* in = static_cast<const T*>(p.input) + c.base;
    T* out = static_cast<T*>(p.output) + c.base;
    const int64_t sweep = static_cast<int64_t>(kColHeld) * c.groups;  // elements of a column a sweep step covers
    Piece<T, V> held[kColHeld];
    auto load = [&](int64_t r0) {  // masked elements and those beyond the column's end: -inf
        ColWalk w(p, c, length<W>(p, c), r0);
#pragma unroll
        for (int k = 0; k < kColHeld; ++k, w.next()) {
            if (w.exists()) {
                held[k].load(in + w.at);
            } else {
                held[k].fill(-INFINITY);
            }
        }
        if constexpr (!std::is_same<M, void>::value) {
            ColWalk m(p, c, length<W>(p, c), r0);
            if constexpr (V == 8 || sizeof(M) * V > 16) {  // (bits, one piece at a time: there are no registers left for more)
#pragma unroll
                for (int k = 0; k < kColHeld; ++k, m.next()) {
                    const uint32_t hit = m.exists() ? mask_bits<M, V>(p.mask, c.base + m.at) : 0u;
#pragma unroll
                    for (int e = 0; e < V; ++e)
                        if (hit >> e & 1) held[k].set(e, -INFINITY);
                }
            } else {
                constexpr int kGroup = 4;
                MaskPiece<M, V> masks[kGroup];
#pragma unroll
                for (int k = 0; k < kColHeld; k += kGroup) {
#pragma unroll
                    for (int i = 0; i < kGroup; ++i, m.next()) {
                        if (m.exists()) masks[i].load(p.mask, c.base + m.at);
                        else masks[i].clear();
                    }
#pragma unroll
                    for (int i = 0; i < kGroup; ++i) masks[i].apply(held[k + i]);
                }
            }
        }
    };
    Stat s[V];
#pragma unroll
    for (int e = 0; e < V; ++e) s[e] = Stat{-INFINITY, 0.f};
    for (int64_t r0 = 0; W != kOutput && r0 < length<W>(p, c); r0 += sweep) {
        load(r0);
#pragma unroll
        for (int e = 0; e < V; ++e) {
            float mx = held[0].get(e);
#pragma unroll
            for (int k = 1; k < kColHeld; ++k) mx = fmaxf(mx, held[k].get(e));
            const float m = fmaxf(s[e].m, mx * kLog2e), ms = reference(m);
            float l = s[e].l * fast_exp2(s[e].m - ms);
#pragma unroll
            for (int k = 0; k < kColHeld; ++k) l += fast_exp2(fmaf(held[k].get(e), kLog2e, -ms));
            s[e] = Stat{m, l};
            if constexpr (V > 1) __builtin_amdgcn_sched_barrier(0);  // (one column at a time: interleaved, the pieces' conversions to fp32 fill the registers)
        }
    }
    // the row groups of a wave, then the waves: one thread per column
    if constexpr (W != kOutput) {
        for (int d = 1 << lanes_log2; d < 64; d <<= 1) {
#pragma unroll
            for (int e = 0; e < V; ++e) s[e] = merge(s[e], Stat{__shfl_xor(s[e].m, d), __shfl_xor(s[e].l, d)});
        }
    }
    const int columns = V << lanes_log2, waves = blockDim.x / 64;
    if constexpr (W == kOutput) {
        merge_parts(p, c, columns, Stat{-INFINITY, 0.f}, part, [](Stat x, Stat y) { return merge(x, y); });
    } else {
        if ((threadIdx.x & 63) < (1 << lanes_log2)) {
#pragma unroll
            for (int e = 0; e < V; ++e) part[(threadIdx.x / 64) * columns + c.lane * V + e] = s[e];
        }
        __syncthreads();
    }
    for (int i = threadIdx.x; i < columns; i += blockDim.x) {
        Stat t = part[i];
        for (int w = 1; W != kOutput && w < waves; ++w) t = merge(t, part[w * columns + i]);
        if constexpr (W == kStatistics) {
            if (c.first + i < p.y_size) static_cast<Stat*>(p.part_stats)[blockIdx.y * p.y_size + c.first + i] = t;
        }
        part[i] = Stat{t.m, 1.f / t.l};  // a fully masked column: 0 * inf = NaN, as softmax gives
    }
    if constexpr (W == kStatistics) return;
    __syncthreads();
    bool far = false;
#pragma unroll
    for (int e = 0; e < V; ++e) {
        s[e] = part[c.lane * V + e];
        far |= far_from_zero(s[e].m);
        s[e].m = reference(s[e].m);
    }
    if (__builtin_amdgcn_ballot_w64(far) != 0) {  // (a wave has all columns of the panel: the same in all waves, and in all parts)
        if (W == kOutput && blockIdx.y > 0) return;
        float* const shared = &part[0].m;
        for (int i = 0; i < columns && c.first + i < p.y_size; ++i)
            softmax_far<T, M>(p, (c.first + i) * p.y_stride, p.x_stride, p.x_size, threadIdx.x, blockDim.x,
                              [&](float x) { return reduce(x, 1, 64, waves, shared, MaxOp{}); },
                              [&](float x) { return reduce(x, 1, 64, waves, shared, SumOp{}); });
        return;
    }
    if (!c.live) return;
    for (int64_t r0 = 0; r0 < length<W>(p, c); r0 += sweep) {
        if (W == kOutput || length<W>(p, c) > sweep) load(r0);
        ColWalk w(p, c, length<W>(p, c), r0);
#pragma unroll
        for (int k = 0; k < kColHeld; ++k, w.next()) {
            if (w.exists()) {
                VT o;
#pragma unroll
                for (int e = 0; e < V; ++e) o.e[e] = from_f32<T>(fast_exp2(fmaf(held[k].get(e), kLog2e, -s[e].m)) * s[e].l);
                *reinterpret_cast<VT*>(out + w.at) = o;
            }
        }
    }
}

template <typename T, int V, ColWork W = kWhole>
__global__ __launch_bounds__(1024) void softmax_bwd_cols_kernel(const RowParams p, int lanes_log2, int64_t panels) {
    extern __shared__ float part_sums[];  // one per wave and column of the panel
    ColPlace c;
    if (!place_in_panel(p, V, lanes_log2, panels, &c, (sizeof(T) * V << lanes_log2) == 32)) return;
    place_in_part<W>(p, &c);
    using VT = Vec<T, V>;
    const T* o = static_cast<const T*>(p.output) + c.base;
    const T* g = static_cast<const T*>(p.grad_output) + c.base;
    T* gi = static_cast<T*>(p.grad_input) + c.base;
    const int64_t sweep = static_cast<int64_t>(kColHeldBwd) * c.groups;
    Piece<T, V> held_o[kColHeldBwd], held_g[kColHeldBwd];
    auto load = [&](int64_t r0) {
        ColWalk w(p, c, length<W>(p, c), r0);
#pragma unroll
        for (int k = 0; k < kColHeldBwd; ++k, w.next()) {
            if (w.exists()) {
                held_o[k].load(o + w.at);
                held_g[k].load(g + w.at);
            } else {
                held_o[k].fill(0.f);
                held_g[k].fill(0.f);
            }
        }
    };
    float delta[V];
#pragma unroll
    for (int e = 0; e < V; ++e) delta[e] = 0.f;
    for (int64_t r0 = 0; W != kOutput && r0 < length<W>(p, c); r0 += sweep) {
        load(r0);
#pragma unroll
        for (int k = 0; k < kColHeldBwd; ++k)
#pragma unroll
            for (int e = 0; e < V; ++e) delta[e] = fmaf(held_o[k].get(e), held_g[k].get(e), delta[e]);
    }
    if constexpr (W != kOutput) {
        for (int d = 1 << lanes_log2; d < 64; d <<= 1) {
#pragma unroll
            for (int e = 0; e < V; ++e) delta[e] += __shfl_xor(delta[e], d);
        }
    }
    const int columns = V << lanes_log2, waves = blockDim.x / 64;
    if constexpr (W == kOutput) {
        merge_parts(p, c, columns, 0.f, part_sums, [](float x, float y) { return x + y; });
    } else {
        if ((threadIdx.x & 63) < (1 << lanes_log2)) {
#pragma unroll
            for (int e = 0; e < V; ++e) part_sums[(threadIdx.x / 64) * columns + c.lane * V + e] = delta[e];
        }
        __syncthreads();
        for (int i = threadIdx.x; i < columns; i += blockDim.x) {
            float t = part_sums[i];
            for (int w = 1; w < waves; ++w) t += part_sums[w * columns + i];
            if constexpr (W == kStatistics) {
                if (c.first + i < p.y_size) static_cast<float*>(p.part_stats)[blockIdx.y * p.y_size + c.first + i] = t;
            }
            part_sums[i] = t;
        }
        if constexpr (W == kStatistics) return;
        __syncthreads();
    }
    if (!c.live) return;
#pragma unroll
    for (int e = 0; e < V; ++e) delta[e] = part_sums[c.lane * V + e];
    for (int64_t r0 = 0; r0 < length<W>(p, c); r0 += sweep) {
        if (W == kOutput || length<W>(p, c) > sweep) load(r0);
        ColWalk w(p, c, length<W>(p, c), r0);
#pragma unroll
        for (int k = 0; k < kColHeldBwd; ++k, w.next()) {
            if (w.exists()) {
                VT x;
#pragma unroll
                for (int e = 0; e < V; ++e) x.e[e] = from_f32<T>(held_o[k].get(e) * (held_g[k].get(e) - delta[e]));
                *reinterpret_cast<VT*>(gi + w.at) = x;
            }
        }
    }
}

// Columns of a few elements (a few rows of a wide matrix): HBM-bound still, but in panels most of a thread's pieces would not
// exist, and their exponentials would bound it. Here a thread holds its V columns whole and nothing is exchanged; pieces
// beyond the last row are skipped by branches the whole launch takes. 2 x 4194304, bf16: forward 0.0835 ms in panels ->
// 0.0093, backward 0.0231 -> 0.0106; fp32 0.0515 -> 0.0134 and 0.0181 -> 0.0158 (a thread per column, as before the panels,
// 0.0162 and 0.0192). 16 x 1048576, bf16: forward 0.0296 -> 0.0173; backward at 9 rows the same either way (0.0133).
constexpr int kFewRows = 16;    // (64 registers; 16-bit columns one per thread: 32 rows)
template <typename T>
constexpr int kFewRowsBwd = sizeof(T) == 2 ? 8 : 4;  // (of each of its two inputs; fp32 8 x 1048576 0.0178 ms so, in panels 0.0165)

template <typename T, int V, typename M, int ROWS = kFewRows>
__global__ __launch_bounds__(256) void softmax_fwd_few_rows_kernel(const RowParams p) {
    const int64_t col = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * V;
    if (col >= p.y_size) return;
    const int64_t base = col * p.y_stride;
    const T* in = static_cast<const T*>(p.input) + base;
    T* out = static_cast<T*>(p.output) + base;
    const int rows = static_cast<int>(p.x_size);
    Piece<T, V> held[ROWS];
#pragma unroll
    for (int k = 0; k < ROWS; ++k)
        if (k < rows) held[k].load(in + k * p.x_stride);
    if constexpr (!std::is_same<M, void>::value) {
        MaskPiece<M, V> masks[8];
#pragma unroll
        for (int k = 0; k < ROWS; k += 8) {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (k + i < rows) masks[i].load(p.mask, base + (k + i) * p.x_stride);
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (k + i < rows) masks[i].apply(held[k + i]);
        }
    }
    float ms[V], l[V];
    bool far = false;
#pragma unroll
    for (int e = 0; e < V; ++e) {
        ms[e] = -INFINITY;
        l[e] = 0.f;
    }
#pragma unroll
    for (int k = 0; k < ROWS; ++k)
        if (k < rows) {
#pragma unroll
            for (int e = 0; e < V; ++e) ms[e] = fmaxf(ms[e], held[k].get(e));
            held[k].hide();
        }
#pragma unroll
    for (int e = 0; e < V; ++e) {
        far |= far_from_zero(ms[e] * kLog2e);
        ms[e] = reference(ms[e] * kLog2e);
    }
    if (__builtin_amdgcn_ballot_w64(far) != 0) {
        const auto own = [](float x) { return x; };
        for (int e = 0; e < V; ++e) softmax_far<T, M>(p, base + e * p.y_stride, p.x_stride, p.x_size, 0, 1, own, own);
        return;
    }
#pragma unroll
    for (int k = 0; k < ROWS; ++k)
        if (k < rows) {
#pragma unroll
            for (int e = 0; e < V; ++e) l[e] += fast_exp2(fmaf(held[k].get(e), kLog2e, -ms[e]));
            held[k].hide();
        }
#pragma unroll
    for (int e = 0; e < V; ++e) l[e] = 1.f / l[e];  // a fully masked column: 0 * inf = NaN, as softmax gives
#pragma unroll
    for (int k = 0; k < ROWS; ++k)
        if (k < rows) {
            Vec<T, V> o;
#pragma unroll
            for (int e = 0; e < V; ++e) o.e[e] = from_f32<T>(fast_exp2(fmaf(held[k].get(e), kLog2e, -ms[e])) * l[e]);
            *reinterpret_cast<Vec<T, V>*>(out + k * p.x_stride) = o;
        }
}

template <typename T, int V>
__global__ __launch_bounds__(256) void softmax_bwd_few_rows_kernel(const RowParams p) {
    const int64_t col = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * V;
    if (col >= p.y_size) return;
    const int64_t base = col * p.y_stride;
    const T* o = static_cast<const T*>(p.output) + base;
    const T* g = static_cast<const T*>(p.grad_output) + base;
    T* gi = static_cast<T*>(p.grad_input) + base;
    const int rows = static_cast<int>(p.x_size);
    constexpr int kRows = kFewRowsBwd<T>;
    Piece<T, V> held_o[kRows], held_g[kRows];
#pragma unroll
    for (int k = 0; k < kRows; ++k)
        if (k < rows) {
            held_o[k].load(o + k * p.x_stride);
            held_g[k].load(g + k * p.x_stride);
        }
    float delta[V];
#pragma unroll
    for (int e = 0; e < V; ++e) delta[e] = 0.f;
#pragma unroll
    for (int k = 0; k < kRows; ++k)
        if (k < rows) {
#pragma unroll
            for (int e = 0; e < V; ++e) delta[e] = fmaf(held_o[k].get(e), held_g[k].get(e), delta[e]);
        }
#pragma unroll
    for (int k = 0; k < kRows; ++k)
        if (k < rows) {
            Vec<T, V> x;
#pragma unroll
            for (int e = 0; e < V; ++e) x.e[e] = from_f32<T>(held_o[k].get(e) * (held_g[k].get(e) - delta[e]));
            *reinterpret_cast<Vec<T, V>*>(gi + k * p.x_stride) = x;
        }
}

// ------------------------------------------------------------------ dropout
// A thread makes one Philox call = the 16 decisions of elements 16 t .. 16 t + 15; BACKWARD reads grad_output instead
// of input. A wave's 1024 elements are read and written 16 bytes per lane with consecutive lanes on consecutive
// addresses (whole cache lines per instruction), so a lane's piece belongs to another lane's Philox block: every lane
// leaves its four words in LDS and picks up the words of its pieces from there. Blocks that are ragged or unaligned
// fall back to a thread working through its own 16 elements.
__device__ __forceinline__ uint32_t drop_byte(const Philox4& r, int e) { return (r.w[e >> 2] >> (8 * (e & 3))) & 0xffu; }

template <typename T>
__global__ __launch_bounds__(256) void dropout_kernel(const RowParams p, const T* __restrict__ src, T* __restrict__ dst, int64_t n) {
    __shared__ __attribute__((aligned(16))) uint32_t words[256 * 4];
    const int64_t blk = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const int lane = threadIdx.x & 63;
    uint32_t* wave_words = words + (threadIdx.x - lane) * 4;
    const int64_t wave_i0 = (blk - lane) * 16;  // first element of this wave's 1024
    const Philox4 r = philox4x32_10(static_cast<uint32_t>(blk), static_cast<uint32_t>(blk >> 32), kDropoutStream, p.offset,
                                    p.seed_lo, p.seed_hi);
    *reinterpret_cast<uint4*>(wave_words + lane * 4) = uint4{r.w[0], r.w[1], r.w[2], r.w[3]};
    __syncthreads();
    if (wave_i0 >= n) return;
    constexpr int V = 16 / sizeof(T);  // elements of a 16-byte piece
    constexpr int W = V / 4;           // Philox words of a piece
    constexpr int PPB = 16 / V;        // pieces per Philox block
    using VT = Vec<T, V>;
    const bool whole = wave_i0 + 1024 <= n && (reinterpret_cast<uintptr_t>(src) & 15) == 0 && (reinterpret_cast<uintptr_t>(dst) & 15) == 0;
    if (whole) {  // (the same for every lane of the wave)
#pragma unroll
        for (int c = 0; c < PPB; ++c) {
            const int piece = c * 64 + lane;  // of the wave's 64 PPB pieces: words piece * W .. + W - 1 of the wave
            uint32_t w[W];
#pragma unroll
            for (int k = 0; k < W; ++k) w[k] = wave_words[piece * W + k];
            const VT v = *reinterpret_cast<const VT*>(src + wave_i0 + static_cast<int64_t>(piece) * V);
            VT o;
#pragma unroll
            for (int e = 0; e < V; ++e) {
                const bool keep = static_cast<int>((w[e >> 2] >> (8 * (e & 3))) & 0xffu) >= p.thr8;
                o.e[e] = from_f32<T>(keep ? to_f32(v.e[e]) * p.zscale : 0.f);
            }
            *reinterpret_cast<VT*>(dst + wave_i0 + static_cast<int64_t>(piece) * V) = o;
        }
    } else {
        const int64_t i0 = blk * 16;
        for (int e = 0; e < 16 && i0 + e < n; ++e) {
            const bool keep = static_cast<int>(drop_byte(r, e)) >= p.thr8;
            dst[i0 + e] = from_f32<T>(keep ? to_f32(src[i0 + e]) * p.zscale : 0.f);
        }
    }
}

// ------------------------------------------------------------------ host side
int make_row_params(const TriRowArgs* a, bool backward, bool dropout, RowParams* p) {
    if (a == nullptr) return TRI_ATTN_ENULL;
    // (structures of callers built before the workspace fields were added end there)
    if (a->struct_size != sizeof(TriRowArgs) && a->struct_size != offsetof(TriRowArgs, workspace)) return TRI_ATTN_ESIZE;
    if (a->dtype < TRI_ATTN_F32 || a->dtype > TRI_ATTN_BF16) return TRI_ATTN_EDTYPE;
    if (a->y_size <= 0 || a->x_size <= 0) return TRI_ATTN_ESHAPE;
    if (!dropout && (a->y_stride < 0 || a->x_stride < 0)) return TRI_ATTN_ESTRIDE;
    if (a->mask != nullptr && (a->mask_dtype < TRI_ATTN_F32 || a->mask_dtype > TRI_ROW_MASK_U8)) return TRI_ATTN_EDTYPE;
    if (dropout && !(a->p >= 0.f && a->p <= 1.f)) return TRI_ATTN_EDROPOUT;
    if (backward) {
        if (!a->grad_output || !a->grad_input || (!dropout && !a->output)) return TRI_ATTN_ENULL;
    } else if (!a->input || !a->output) {
        return TRI_ATTN_ENULL;
    }
    memset(p, 0, sizeof(*p));
    if (a->struct_size == sizeof(TriRowArgs)) {
        p->workspace = a->workspace;
        p->workspace_bytes = a->workspace_size;
    }
    p->input = a->input;
    p->output = a->output;
    p->mask = a->mask;
    p->grad_output = a->grad_output;
    p->grad_input = a->grad_input;
    p->y_size = a->y_size;
    p->x_size = a->x_size;
    p->y_stride = a->y_stride;
    p->x_stride = a->x_stride;
    p->mask_dtype = a->mask_dtype;
    p->seed_lo = static_cast<uint32_t>(a->seed);
    p->seed_hi = static_cast<uint32_t>(a->seed >> 32);
    p->offset = static_cast<uint32_t>(a->offset);
    int thr = static_cast<int>(rintf(a->p * 256.f));
    thr = thr < 0 ? 0 : (thr > 256 ? 256 : thr);
    p->thr8 = thr;
    p->zscale = thr >= 256 ? 0.f : 256.f / static_cast<float>(256 - thr);
    return TRI_ATTN_OK;
}

bool aligned16(const void* ptr) { return ptr == nullptr || (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; }

// Geometry of a column launch: panels as wide as leaves one for every CU, but no narrower than the 64 bytes HBM moves at
// a time (16 lanes without vector accesses), and as many threads as give each kColHeld (kColHeldBwd) pieces of its column.
// A matrix narrower than 256 such panels leaves CUs idle; column_split is for the long ones among them.
struct ColLaunch {
    int lanes_log2;
    int64_t panels;
    dim3 grid, block;
    unsigned stats;  // waves x columns of a panel
};
ColLaunch column_launch(const RowParams& p, int v, int held) {
    ColLaunch c;
    const int widest = v == 1 ? 6 : (v == 4 ? 5 : 4), narrowest = v == 1 ? 4 : 2;
    c.lanes_log2 = widest;
    auto panels = [&]() { return (p.y_size + (static_cast<int64_t>(v) << c.lanes_log2) - 1) / (static_cast<int64_t>(v) << c.lanes_log2); };
    while (c.lanes_log2 > narrowest && panels() < 256) --c.lanes_log2;
    // (half as wide where that lets the column stay in registers: backward at 4096 x 4096 fp32 0.0447 ms, in two sweeps 0.0602)
    if (v > 1 && c.lanes_log2 == narrowest && static_cast<int64_t>(1024 >> narrowest) * held < p.x_size && p.x_size <= static_cast<int64_t>(2048 >> narrowest) * held)
        --c.lanes_log2;
    c.panels = panels();
    int threads = 64;
    while (threads < 1024 && static_cast<int64_t>(threads >> c.lanes_log2) * held < p.x_size) threads <<= 1;
    c.grid = dim3(static_cast<unsigned>((c.panels + 7) / 8 * 8));
    c.block = dim3(threads);
    c.stats = static_cast<unsigned>(threads / 64 * (v << c.lanes_log2));
    return c;
}

// Geometry of the split launches: workgroups of 256 threads, panels of 64 bytes, and as many parts as give two workgroups per CU,
// each at least four pieces per thread and at most the forward's sixteen, kMaxParts of them at most, whose statistics every
// workgroup of the second launch reads. (Panels of 256 bytes in workgroups of 1024 threads: 38122 x 424 bf16 with mask 107 and 76
// us, so 61 and 57.) Returns the bytes of workspace, 0: the launch stays whole. That is where half the CUs and more have a panel, or
// a panel's columns stay in its registers, which are then read once and not twice.
constexpr int kMaxParts = 128;
int64_t column_split(const RowParams& p, int v, int elem_bytes, int held, int stat_bytes, RowParams* split, ColLaunch* c) {
    const ColLaunch whole = column_launch(p, v, held);
    if (whole.panels > 128 || p.x_size <= static_cast<int64_t>(whole.block.x >> whole.lanes_log2) * held) return 0;
    *c = whole;
    c->lanes_log2 = v > 1 ? 2 : (elem_bytes == 4 ? 4 : 5);
    const int64_t columns = static_cast<int64_t>(v) << c->lanes_log2, groups = 256 >> c->lanes_log2;
    c->panels = (p.y_size + columns - 1) / columns;
    c->block = dim3(256);
    const auto parts_of = [&](int64_t rows) { return (p.x_size + rows - 1) / rows; };
    const int64_t parts = std::min<int64_t>(kMaxParts, std::max(parts_of(groups * 16), std::min((512 + c->panels - 1) / c->panels, parts_of(groups * 4))));
    *split = p;
    split->part_size = parts_of(parts);
    split->parts = static_cast<int>(parts_of(split->part_size));
    c->grid = dim3(static_cast<unsigned>((c->panels + 7) / 8 * 8), static_cast<unsigned>(split->parts));
    c->stats = static_cast<unsigned>(std::max<int64_t>(4 * columns, 256));  // (statistics of four waves, or of 256 threads' columns)
    return split->parts * p.y_size * stat_bytes;
}
bool take_workspace(int64_t bytes, RowParams* split) {
    if (bytes <= 0 || split->workspace == nullptr || split->workspace_bytes < bytes || reinterpret_cast<uintptr_t>(split->workspace) % 16 != 0) return false;
    split->part_stats = split->workspace;
    return true;
}

// whether a column launch takes whole vectors of neighbouring columns: every element row starts on a 16-byte boundary and holds
// whole vectors
bool columns_vec(const RowParams& p, int v, bool aligned) { return p.y_stride == 1 && p.y_size % v == 0 && p.x_stride % v == 0 && aligned; }

dim3 few_rows_grid(const RowParams& p, int v) { return dim3(static_cast<unsigned>((p.y_size + 256 * v - 1) / (256 * v))); }

// Calls launch(V, G, SHIFT) with the variant for rows of this geometry.
template <typename T, typename Launch>
int launch_rows(const RowParams& p, bool base16, bool backward, Launch launch) {
    constexpr int kV = 16 / sizeof(T);
    using std::integral_constant;
    using One = integral_constant<int, 1>;
    using Full = integral_constant<int, kV>;
    using Yes = integral_constant<bool, true>;
    using No = integral_constant<bool, false>;
    // a row goes to the fewest threads whose registers hold it: 16 (up to 512 16-bit elements), a wave (2048), a workgroup
    // (element by element a wave also takes rows that it sweeps twice: bf16 32768 x 512 forward 0.0530 -> 0.0256 ms, 16384 x 1024
    // 0.0320 -> 0.0245; fp32 8192 x 2048 0.0279 -> 0.0314)
    auto with_group = [&](auto v, auto shift) {
        constexpr int held = held_pieces(decltype(shift)::value) * decltype(v)::value;
        const int64_t worst = p.x_size + (decltype(shift)::value ? kV - 1 : 0);
        if (worst <= 16 * held) launch(v, integral_constant<int, 16>{}, shift);
        else if (worst <= (decltype(v)::value == 1 ? 1024 : 64 * held)) launch(v, integral_constant<int, 64>{}, shift);
        else launch(v, integral_constant<int, 256>{}, shift);
    };
    // 16-byte accesses when the tensors start on 16-byte boundaries; shifted ones when the rows do not, but for short rows, of which
    // one element per load is less work (16.7 M elements, us, shifted and by elements: forward bf16 33 per row 72 and 43, 49 49 and 32, 65
    // 38 and 76, 255 20 and 25; fp32 49 43 and 34, 65 42 and 76. Backward bf16 49 42 and 23, 65 34 and 51, 197 19.6 and 20.8, 255 20.5 and 19.3;
    // fp32 49 38 and 39, 65 40 and 59, 110 34 and 39, 150 36 and 33, 197 37 and 32, 255 37 and 33, 301 36 and 42).
    const bool by_element = p.x_size <= 64 || (backward && sizeof(T) == 4 && p.x_size > 128 && p.x_size <= 256);
    if (!base16) with_group(One{}, No{});
    else if (p.x_size % kV == 0 && p.y_stride % kV == 0) with_group(Full{}, No{});
    else if (by_element) with_group(One{}, No{});
    else with_group(Full{}, Yes{});
    return static_cast<int>(hipGetLastError());
}

template <typename T, typename M>
int launch_softmax_fwd(const RowParams& p, hipStream_t st) {
    constexpr int kV = 16 / sizeof(T);
    const dim3 block(256);
    if (p.x_stride != 1 && p.x_size != 1) {
        const bool vec = columns_vec(p, kV, aligned16(p.input) && aligned16(p.output) && aligned16(p.mask));
        // Whole vectors where they leave two workgroups and more per CU: below, one column per thread is faster (forward, bf16 16 x
        // 16384 0.0094 -> 0.0057 ms, 262144 columns 0.0110 -> 0.0079; from 524288 columns on the vectors, 16 x 1048576 0.0180 to 0.0207).
        // 16-bit columns of up to 32 elements go one per thread, too, with a mask, which the panels work through piece by piece
        // (bf16 17 x 16384 0.0093 -> 0.0064 ms, 17 x 1048576 0.0363 -> 0.0259), or up to 262144 of them (24 x 1048576 0.0265 in panels).
        if (p.x_size <= kFewRows) {
            if (vec && p.y_size >= 1 << 19) hipLaunchKernelGGL((softmax_fwd_few_rows_kernel<T, kV, M>), few_rows_grid(p, kV), block, 0, st, p);
            else hipLaunchKernelGGL((softmax_fwd_few_rows_kernel<T, 1, M>), few_rows_grid(p, 1), block, 0, st, p);
            return static_cast<int>(hipGetLastError());
        }
        if constexpr (sizeof(T) == 2) {
            if (p.x_size <= 32 && (!std::is_same<M, void>::value || p.y_size <= 1 << 18)) {
                hipLaunchKernelGGL((softmax_fwd_few_rows_kernel<T, 1, M, 32>), few_rows_grid(p, 1), block, 0, st, p);
                return static_cast<int>(hipGetLastError());
            }
        }
        {
            RowParams split;
            ColLaunch c;
            if (p.workspace != nullptr && take_workspace(column_split(p, vec ? kV : 1, sizeof(T), kColHeld, sizeof(Stat), &split, &c), &split)) {
                const unsigned lds = c.stats * sizeof(Stat);
                if (vec) {
                    hipLaunchKernelGGL((softmax_fwd_cols_kernel<T, kV, M, kStatistics>), c.grid, c.block, lds, st, split, c.lanes_log2, c.panels);
                    hipLaunchKernelGGL((softmax_fwd_cols_kernel<T, kV, M, kOutput>), c.grid, c.block, lds, st, split, c.lanes_log2, c.panels);
                } else {
                    hipLaunchKernelGGL((softmax_fwd_cols_kernel<T, 1, M, kStatistics>), c.grid, c.block, lds, st, split, c.lanes_log2, c.panels);
                    hipLaunchKernelGGL((softmax_fwd_cols_kernel<T, 1, M, kOutput>), c.grid, c.block, lds, st, split, c.lanes_log2, c.panels);
                }
                return static_cast<int>(hipGetLastError());
            }
        }
        const ColLaunch c = column_launch(p, vec ? kV : 1, kColHeld);
        const unsigned lds = c.stats * sizeof(Stat);
        if (vec) hipLaunchKernelGGL((softmax_fwd_cols_kernel<T, kV, M>), c.grid, c.block, lds, st, p, c.lanes_log2, c.panels);
        else hipLaunchKernelGGL((softmax_fwd_cols_kernel<T, 1, M>), c.grid, c.block, lds, st, p, c.lanes_log2, c.panels);
        return static_cast<int>(hipGetLastError());
    }
    const bool base16 = aligned16(p.input) && aligned16(p.output);
    const bool mask16 = aligned16(p.mask);
    return launch_rows<T>(p, base16, false, [&](auto v, auto g, auto shift) {
        constexpr int V = decltype(v)::value, G = decltype(g)::value;
        constexpr bool kShift = decltype(shift)::value;
        const dim3 grid(static_cast<unsigned>((p.y_size * G + 255) / 256));
        if constexpr (V > 1 && !std::is_same<M, void>::value) {
            if (!mask16) {
                hipLaunchKernelGGL((softmax_fwd_rows_kernel<T, V, G, kShift, M, false>), grid, block, 0, st, p);
                return;
            }
        }
        hipLaunchKernelGGL((softmax_fwd_rows_kernel<T, V, G, kShift, M>), grid, block, 0, st, p);
    });
}

template <typename T>
int launch_softmax_bwd(const RowParams& p, hipStream_t st) {
    constexpr int kV = 16 / sizeof(T);
    const dim3 block(256);
    if (p.x_stride != 1 && p.x_size != 1) {
        const bool vec = columns_vec(p, kV, aligned16(p.output) && aligned16(p.grad_output) && aligned16(p.grad_input));
        if (p.x_size <= kFewRowsBwd<T>) {
            if (vec) hipLaunchKernelGGL((softmax_bwd_few_rows_kernel<T, kV>), few_rows_grid(p, kV), block, 0, st, p);
            else hipLaunchKernelGGL((softmax_bwd_few_rows_kernel<T, 1>), few_rows_grid(p, 1), block, 0, st, p);
            return static_cast<int>(hipGetLastError());
        }
        {
            RowParams split;
            ColLaunch c;
            if (p.workspace != nullptr && take_workspace(column_split(p, vec ? kV : 1, sizeof(T), kColHeldBwd, sizeof(float), &split, &c), &split)) {
                const unsigned lds = c.stats * sizeof(float);
                if (vec) {
                    hipLaunchKernelGGL((softmax_bwd_cols_kernel<T, kV, kStatistics>), c.grid, c.block, lds, st, split, c.lanes_log2, c.panels);
                    hipLaunchKernelGGL((softmax_bwd_cols_kernel<T, kV, kOutput>), c.grid, c.block, lds, st, split, c.lanes_log2, c.panels);
                } else {
                    hipLaunchKernelGGL((softmax_bwd_cols_kernel<T, 1, kStatistics>), c.grid, c.block, lds, st, split, c.lanes_log2, c.panels);
                    hipLaunchKernelGGL((softmax_bwd_cols_kernel<T, 1, kOutput>), c.grid, c.block, lds, st, split, c.lanes_log2, c.panels);
                }
                return static_cast<int>(hipGetLastError());
            }
        }
        const ColLaunch c = column_launch(p, vec ? kV : 1, kColHeldBwd);
        const unsigned lds = c.stats * sizeof(float);
        if (vec) hipLaunchKernelGGL((softmax_bwd_cols_kernel<T, kV>), c.grid, c.block, lds, st, p, c.lanes_log2, c.panels);
        else hipLaunchKernelGGL((softmax_bwd_cols_kernel<T, 1>), c.grid, c.block, lds, st, p, c.lanes_log2, c.panels);
        return static_cast<int>(hipGetLastError());
    }
    const bool base16 = aligned16(p.output) && aligned16(p.grad_output) && aligned16(p.grad_input);
    return launch_rows<T>(p, base16, true, [&](auto v, auto g, auto shift) {
        hipLaunchKernelGGL((softmax_bwd_rows_kernel<T, decltype(v)::value, decltype(g)::value, decltype(shift)::value>),
                           dim3(static_cast<unsigned>((p.y_size * decltype(g)::value + 255) / 256)), block, 0, st, p);
    });
}

template <typename T>
int launch_softmax(const RowParams& p, bool backward, hipStream_t st) {
    if (p.y_size > 2147483647LL) return TRI_ATTN_ESHAPE;
    if (backward) return launch_softmax_bwd<T>(p, st);
    if (p.mask == nullptr) return launch_softmax_fwd<T, void>(p, st);
    switch (p.mask_dtype) {
        case TRI_ATTN_F32: return launch_softmax_fwd<T, float>(p, st);
        case TRI_ATTN_F16: return launch_softmax_fwd<T, f16_t>(p, st);
        case TRI_ATTN_BF16: return launch_softmax_fwd<T, bf16_t>(p, st);
        case TRI_ROW_MASK_I64: return launch_softmax_fwd<T, int64_t>(p, st);
        case TRI_ROW_MASK_I32: return launch_softmax_fwd<T, int32_t>(p, st);
        default: return launch_softmax_fwd<T, uint8_t>(p, st);
    }
}

int launch_softmax_any(int dtype, const RowParams& p, bool backward, hipStream_t st) {
    switch (dtype) {
        case TRI_ATTN_F32: return launch_softmax<float>(p, backward, st);
        case TRI_ATTN_F16: return launch_softmax<f16_t>(p, backward, st);
        default: return launch_softmax<bf16_t>(p, backward, st);
    }
}

template <typename T>
int launch_dropout(const RowParams& p, bool backward, hipStream_t st) {
    const int64_t n = p.y_size * p.x_size;
    const int64_t threads = (n + 15) / 16, groups = (threads + 255) / 256;
    if (groups > 2147483647LL) return TRI_ATTN_ESHAPE;
    const T* src = static_cast<const T*>(backward ? p.grad_output : p.input);
    T* dst = static_cast<T*>(backward ? p.grad_input : p.output);
    hipLaunchKernelGGL((dropout_kernel<T>), dim3(static_cast<unsigned>(groups)), dim3(256), 0, st, p, src, dst, n);
    return static_cast<int>(hipGetLastError());
}

int launch_dropout_any(int dtype, const RowParams& p, bool backward, hipStream_t st) {
    switch (dtype) {
        case TRI_ATTN_F32: return launch_dropout<float>(p, backward, st);
        case TRI_ATTN_F16: return launch_dropout<f16_t>(p, backward, st);
        default: return launch_dropout<bf16_t>(p, backward, st);
    }
}

}  // namespace
}  // namespace tri

using namespace tri;

extern "C" {

int tri_softmax_fwd(const TriRowArgs* args) {
    RowParams p;
    const int rc = make_row_params(args, false, false, &p);
    if (rc) return rc;
    return launch_softmax_any(args->dtype, p, false, static_cast<hipStream_t>(args->stream));
}

int tri_softmax_bwd(const TriRowArgs* args) {
    RowParams p;
    const int rc = make_row_params(args, true, false, &p);
    if (rc) return rc;
    p.mask = nullptr;  // masked positions have output 0: the gradient needs no mask
    return launch_softmax_any(args->dtype, p, true, static_cast<hipStream_t>(args->stream));
}

int64_t tri_softmax_workspace_size(const TriRowArgs* args, int backward) {
    RowParams p, split;
    const int rc = make_row_params(args, backward != 0, false, &p);
    if (rc) return rc;
    const int v = args->dtype == TRI_ATTN_F32 ? 4 : 8;
    if (p.x_stride == 1 || p.x_size <= 32) return 0;
    ColLaunch c;
    if (backward) {
        const bool vec = columns_vec(p, v, aligned16(p.output) && aligned16(p.grad_output) && aligned16(p.grad_input));
        return column_split(p, vec ? v : 1, 16 / v, kColHeldBwd, sizeof(float), &split, &c);
    }
    const bool vec = columns_vec(p, v, aligned16(p.input) && aligned16(p.output) && aligned16(p.mask));
    return column_split(p, vec ? v : 1, 16 / v, kColHeld, sizeof(Stat), &split, &c);
}

int tri_dropout_fwd(const TriRowArgs* args) {
    RowParams p;
    const int rc = make_row_params(args, false, true, &p);
    if (rc) return rc;
    return launch_dropout_any(args->dtype, p, false, static_cast<hipStream_t>(args->stream));
}

int tri_dropout_bwd(const TriRowArgs* args) {
    RowParams p;
    const int rc = make_row_params(args, true, true, &p);
    if (rc) return rc;
    return launch_dropout_any(args->dtype, p, true, static_cast<hipStream_t>(args->stream));
}

}  // extern "C"
