// Shared by the kernels that put several rows of at most 128 columns side by side in a wave
// (narrow_rows.hip, narrow_forward.hip).
#pragma once

#include "box_sampling_common.hpp"

namespace boxconv {

namespace {

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
template <class V>
__device__ __forceinline__ void finish_here(V& v) { asm volatile("" : "+v"(v)); }

// Row r confined to [0, last], and the byte offset of a row: one instruction each (the compiler makes two
// of the first, and a product of four times the cost of the second; rows and their bytes are below 2^24).
__device__ __forceinline__ int confine(int r, int last) {
    int v;
    asm("v_med3_i32 %0, %1, 0, %2" : "=v"(v) : "v"(r), "s"(last));
    return v;
}
__device__ __forceinline__ unsigned row_offset(int r, unsigned row_bytes, unsigned first) {
    return __umul24(static_cast<unsigned>(r), row_bytes) + first;
}

// LDS serves a wave's accesses in order; only the compiler has to be kept from moving them.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Four elements in flight, as they are in memory.
template <class TG>
struct RawQuad {
    Quad<TG> q;
    template <bool ALIGNED>
    __device__ __forceinline__ void load(const TG* p) {
        if constexpr (ALIGNED) {
            typedef unsigned Words __attribute__((ext_vector_type(sizeof(Quad<TG>) / 4)));
            q = __builtin_bit_cast(Quad<TG>, *reinterpret_cast<const Words*>(p));
        } else if constexpr (sizeof(TG) == 4) {
            q = __builtin_bit_cast(Quad<TG>, *reinterpret_cast<const w4_dword_aligned*>(p));
        } else {
            q = __builtin_bit_cast(Quad<TG>, *reinterpret_cast<const w2_half_aligned*>(p));
        }
    }
    __device__ __forceinline__ float get(int k) const { return widen(q.v[k]); }
};

// Lane `l` of the L that share a row, and the LDS layout of 64 / L row pairs side by side: column c of
// row s is element s * (L + 4) + c / 4 + 2 of plane c % 4, with two zeros in front of every row and
// behind it (see tap_run). Rows that are no multiple of four columns: see RowLane.
template <int L>
struct NarrowLane {
    static constexpr int S = 64 / L, ROW = L + 2 * kQuadPad, PLANE = S * ROW + 2;
    int seg, l, c0, quads, twice;
    unsigned cl;
    bool in;
    __device__ __forceinline__ NarrowLane(int lane, int w)
        : seg(lane / L), l(lane & (L - 1)), c0(min(4 * l, w - 4)), quads((w + 3) / 4), in(4 * l < w) {
        cl = in ? static_cast<unsigned>(c0) : 0u;
        twice = in ? 4 * l - c0 : 0;
    }
    __device__ __forceinline__ bool shares(int k) const { return k < 3 && k < twice; }
    __device__ __forceinline__ bool owns(int k) const { return in && !shares(k); }
    // element of column c0 + k, for an idle lane one that nobody reads
    __device__ __forceinline__ unsigned place(int k) const {
        const int c = c0 + k;
        return static_cast<unsigned>(in ? (c & 3) * PLANE + seg * ROW + (c >> 2) + kQuadPad : k * PLANE + S * ROW) *
               static_cast<unsigned>(sizeof(RowPair<float>));
    }
    __device__ __forceinline__ TapRun taps(int first) const {
        TapRun t = tap_run<PLANE>(c0, first, quads);
#pragma unroll
        for (int m = 0; m < 4; ++m)
            t.at[m] = (in ? t.at[m] : 0u) + static_cast<unsigned>(seg * ROW) * static_cast<unsigned>(sizeof(RowPair<float>));
        return t;
    }
};

}  // namespace

}  // namespace boxconv
