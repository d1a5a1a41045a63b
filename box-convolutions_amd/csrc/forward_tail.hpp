// Shared by the forward kernels (box_forward.hip, narrow_forward.hip): the fused tail, and quads of four
// output elements as one access.
#pragma once

#include "box_sampling_common.hpp"

namespace boxconv {

// TO: element type of the output (T, or a 16-bit type when T is float). TAIL: what happens to a
// box sum S on its way out, fused into the store (inference only, there is no backward for it):
//   y = S * channel_scale[c*F+f] + channel_shift[c*F+f]  (+ residual[same pixel])  (max(y, 0))
// which is the tail of a block such as BoxConv -> BatchNorm (eval) -> residual add -> ReLU.
// Absent pieces are neutral: a null scale/shift reads as 1/0, a null residual as zeros (its row
// descriptors get size 0, so the loads return 0 without a branch).
template <class TO>
struct ForwardTail {
    TO* dst;
    const TO* residual;
    const float* channel_scale;
    const float* channel_shift;
    int relu;
};

// narrow_forward.hip: `a` holds the source, the boxes and the store policy; the rest is set there.
template <class TO>
hipError_t narrow_forward_launch(SampleArgs<float> a, ForwardTail<TO> tail, Dims d, bool has_tail, bool exact, hipStream_t stream);

namespace {

template <class TO, bool ALIGNED> struct QuadWords;
template <class TO> struct QuadWords<TO, true> { typedef unsigned Type __attribute__((ext_vector_type(sizeof(Quad<TO>) / 4))); };
template <> struct QuadWords<float, false> { typedef w4_dword_aligned Type; };
template <> struct QuadWords<f16_t, false> { typedef w2_half_aligned Type; };
template <> struct QuadWords<bf16_t, false> { typedef w2_half_aligned Type; };
template <bool STREAM, bool ALIGNED, class TO>
__device__ __forceinline__ Quad<TO> load_quad(const TO* p) {
    typedef typename QuadWords<TO, ALIGNED>::Type Words;
    if constexpr (STREAM) return __builtin_bit_cast(Quad<TO>, __builtin_nontemporal_load(reinterpret_cast<const Words*>(p)));
    else return __builtin_bit_cast(Quad<TO>, *reinterpret_cast<const Words*>(p));   // (one expression for both would drop the policy)
}
template <bool ALIGNED, class TO>
__device__ __forceinline__ void store_quad(TO* p, const Quad<TO>& q, bool stream) {
    typedef typename QuadWords<TO, ALIGNED>::Type Words;
    const Words v = __builtin_bit_cast(Words, q);
    if (stream) __builtin_nontemporal_store(v, reinterpret_cast<Words*>(p));
    else *reinterpret_cast<Words*>(p) = v;
}

}  // namespace

}  // namespace boxconv
