// Forward box sampling of rows of at most 128 columns (float integral image; replaces
// cpu::boxConvUpdateOutput, src/box_convolution.cpp:100-261, as forward_rows_kernel does, which has the
// math). Compiled once per element type of the output (BOXCONV_INST_TO). A wave takes 64 / L bands of one (plane, filter)
// side by side, L = 8, 16 or 32 lanes of four consecutive columns each (narrow_rows.hpp), where the kernels
// with one row per wave leave half and more of their lanes idle and store one element per lane.

#include <cmath>

#include "forward_tail.hpp"
#include "narrow_rows.hpp"

namespace boxconv {

namespace {

template <class TO, int L, bool EXACT, bool QUADS, bool TAIL, bool RESIDUAL>
__global__ void __launch_bounds__(64)
narrow_forward_kernel(SampleArgs<float> a, ForwardTail<TO> tl) {
    using T = float;
    using Lane = NarrowLane<L>;
    constexpr int K = 4, S = Lane::S, PLANE = Lane::PLANE;
    __shared__ __align__(16) RowPair<T> vrow[2][K * PLANE];
    const unsigned vid = xcd_contiguous_id(a.per_xcd);
    if (vid >= a.total) return;
    const unsigned slots = a.acc_slots, nfilt = a.F;     // waves per (plane, filter)
    const int slot = static_cast<int>(vid % slots);
    const unsigned pf32 = vid / slots;
    const int f = static_cast<int>(pf32 % nfilt);
    const int64_t pf = pf32, p = pf32 / nfilt;
    const int k_par = static_cast<int>(static_cast<unsigned>(a.plane0 + p) % static_cast<unsigned>(a.C)) * a.F + f;
    const int h = a.h, w = a.w, R = a.R;
    const Lane ln(threadIdx.x, w);
    const int i0 = (slot * S + ln.seg) * R, i1 = min(h, i0 + R);   // (a band past the plane: no rows)
    const int rows = uniform(min(R, h - slot * S * R));            // of the wave's first band: the most that any has

    const BoxOfWorkgroup<T> bx = load_box(a.prm, k_par);
    BoxSplit<T> s = split_forward(bx.xmin, bx.xmax, bx.ymin, bx.ymax);
    s.xlo = uniform(s.xlo); s.xhi = uniform(s.xhi); s.ylo = uniform(s.ylo); s.yhi = uniform(s.yhi);
    const T scale = a.normalize
        ? inverse_extent(bx.xmin, bx.xmax, bx.ymin, bx.ymax, EXACT, true, true) : T(1);

    const T* iplane = a.src + p * static_cast<int64_t>(h + 1) * (w + 1) + 1;
    const unsigned i_bytes = 4u * static_cast<unsigned>(w + 1);
    auto load_i = [&](int r, T (&dst)[K]) {
        load4_dword_aligned(at_bytes(iplane, row_offset(confine(r, h), i_bytes, 4u * ln.cl)), dst);
    };
    const unsigned o_bytes = static_cast<unsigned>(sizeof(TO)) * static_cast<unsigned>(w), o_first = static_cast<unsigned>(sizeof(TO)) * ln.cl;
    TO* const oplane = tl.dst + pf * static_cast<int64_t>(h) * w;
    const TO* const rplane = RESIDUAL ? tl.residual + pf * static_cast<int64_t>(h) * w : nullptr;
    T ch_scale = T(1), ch_shift = T(0);
    if (TAIL) {
        if (tl.channel_scale != nullptr) ch_scale = tl.channel_scale[k_par];
        if (tl.channel_shift != nullptr) ch_shift = tl.channel_shift[k_par];
    }
    const bool relu = TAIL && tl.relu != 0;

    T ta[K], bc[K];                       // I[t(i-1)], I[b(i)]
    T t0[K], t1[K], b1[K], b2[K];         // I[t(i)], I[t(i+1)], I[b(i+1)], I[b(i+2)]
    load_i(i0 + s.xlo - 1, ta);
    load_i(i0 + s.xhi, bc);
    load_i(i0 + s.xlo, t0);
    load_i(i0 + 1 + s.xlo, t1);
    load_i(i0 + 1 + s.xhi, b1);
    load_i(i0 + 2 + s.xhi, b2);
    auto load_residual = [&](int i, RawQuad<TO>& q) {
        if constexpr (RESIDUAL) q.template load<QUADS>(at_bytes(rplane, row_offset(confine(i, h - 1), o_bytes, o_first)));
    };
    RawQuad<TO> res0{}, res1{};
    load_residual(i0, res0);
    load_residual(i0 + 1, res1);

    // V[1..w] by column; V[0] and what clamps to it is a zero in front of the row, what lies behind it V[w]
    for (int e = threadIdx.x; e < 2 * S; e += 64) vrow[e / S][(e % S) * Lane::ROW] = RowPair<T>{T(0), T(0)};
    unsigned place[QUADS ? 1 : K], right[K + 1], left[K + 1];
#pragma unroll
    for (int k = 0; k < (QUADS ? 1 : K); ++k) place[k] = ln.place(k);
    auto own = [&](RowPair<T>* row, int k) {
        return QUADS ? at_bytes(row + k * PLANE, place[0]) : at_bytes(row, place[QUADS ? 0 : k]);
    };
    auto tap = [&](int c) {
        c = min(c, w - 1);
        return static_cast<unsigned>(ln.seg * Lane::ROW + (c < 0 ? 0 : (c & (K - 1)) * PLANE + c / K + kQuadPad)) *
               static_cast<unsigned>(sizeof(RowPair<T>));
    };
#pragma unroll
    for (int m = 0; m < K + 1; ++m) {
        right[m] = tap(ln.c0 + s.yhi - 1 + m);
        left[m] = tap(ln.c0 + s.ylo - 2 + m);
    }
    wave_lds_order();

    auto row_pair = [&](int lr, auto prefetch_tag, auto flip_tag) {
        constexpr bool PREFETCH = decltype(prefetch_tag)::value;
        constexpr int FLIP = decltype(flip_tag)::value;
        const int i = i0 + lr;
        T n0[K] = {}, n1[K] = {}, n2[K] = {}, n3[K] = {};
        RawQuad<TO> m0{}, m1{};
        if (PREFETCH) {
            load_residual(i + 2, m0);
            load_residual(i + 3, m1);
            load_i(i + 2 + s.xlo, n0);
            load_i(i + 3 + s.xlo, n1);
            load_i(i + 3 + s.xhi, n2);
            load_i(i + 4 + s.xhi, n3);
        }
#pragma unroll
        for (int k = 0; k < K; ++k)
            *own(vrow[FLIP], k) = RowPair<T>{blend<T, EXACT>(ta[k], t0[k], bc[k], b1[k], s.fxlo, s.fxhi),
                                             blend<T, EXACT>(t0[k], t1[k], b1[k], b2[k], s.fxlo, s.fxhi)};
        wave_lds_order();
        RowPair<T> Rt[K + 1], Lt[K + 1];
#pragma unroll
        for (int m = 0; m < K + 1; ++m) {
            if (EXACT || m < K) Rt[m] = *at_bytes(vrow[FLIP], right[m]);
            if (EXACT || m > 0) Lt[m] = *at_bytes(vrow[FLIP], left[m]);
        }
        Quad<TO> z0, z1;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            T y0 = blend<T, EXACT>(Lt[k].r0, Lt[k + 1].r0, Rt[k].r0, Rt[k + 1].r0, s.fylo, s.fyhi) * scale;
            T y1 = blend<T, EXACT>(Lt[k].r1, Lt[k + 1].r1, Rt[k].r1, Rt[k + 1].r1, s.fylo, s.fyhi) * scale;
            if (TAIL) {
                y0 = y0 * ch_scale + ch_shift + (RESIDUAL ? res0.get(k) : T(0));
                y1 = y1 * ch_scale + ch_shift + (RESIDUAL ? res1.get(k) : T(0));
                if (relu) { y0 = y0 < T(0) ? T(0) : y0; y1 = y1 < T(0) ? T(0) : y1; }
            }
            narrow(y0, z0.v[k]);
            narrow(y1, z1.v[k]);
        }
        if (ln.in && i < i1) {
            store_quad<QUADS>(at_bytes(oplane, row_offset(i, o_bytes, o_first)), z0, a.stream_out != 0);
            if (i + 1 < i1) store_quad<QUADS>(at_bytes(oplane, row_offset(i + 1, o_bytes, o_first)), z1, a.stream_out != 0);
        }
        if (PREFETCH) {
#pragma unroll
            for (int k = 0; k < K; ++k) {
                ta[k] = t1[k]; bc[k] = b2[k];
                t0[k] = n0[k]; t1[k] = n1[k]; b1[k] = n2[k]; b2[k] = n3[k];
            }
            if (RESIDUAL) { res0 = m0; res1 = m1; }
        }
        wave_lds_order();
    };
    int lr = 0;
    for (; lr + 4 < rows; lr += 4) {
        row_pair(lr, std::true_type{}, Flip0{});
        row_pair(lr + 2, std::true_type{}, Flip1{});
    }
    if (lr + 2 < rows) {
        row_pair(lr, std::true_type{}, Flip0{});
        row_pair(lr + 2, std::false_type{}, Flip1{});
    } else {
        row_pair(lr, std::false_type{}, Flip0{});
    }
}

}  // namespace

template <class TO>
hipError_t narrow_forward_launch(SampleArgs<float> a, ForwardTail<TO> tail, Dims d, bool has_tail, bool exact, hipStream_t stream) {
    const int lanes = d.w <= 32 ? 8 : d.w <= 64 ? 16 : 32, side = 64 / lanes;
    const int64_t planes_f = d.planes * d.F;
    // rows per band for the least rounds of waves (five per SIMD) times row pairs and about two to begin with
    double best = 0.0;
    for (int R = 4; R <= 32; R *= 2) {
        const int slots = ((d.h + R - 1) / R + side - 1) / side;
        const double rounds = static_cast<double>(planes_f) * slots / (1024 * 5);
        const double cost = (rounds < 4 ? std::ceil(rounds) : rounds) * (std::min(R, d.h) / 2 + 2);
        if (R == 4 || cost <= best) { best = cost; a.R = R; a.acc_slots = slots; }
    }
    finish_args(a, planes_f * a.acc_slots);
    const dim3 grid(static_cast<unsigned>(a.per_xcd * kXcds));
    // whole quads only from addresses that are aligned to them; else loads and stores that need elements to be (the same for odd rows)
    const bool quads = d.w % 4 == 0 && quads_aligned(tail.dst, sizeof(TO), d.w) && quads_aligned(tail.residual, sizeof(TO), d.w);
    const char* const name = d.w % 4 == 0 && !quads ? "forward_narrow_unaligned" : "forward_narrow";
#define LAUNCH_NF_TAIL(L, EX, QUADS)                                                                                    \
    do {                                                                                                                \
        if (!has_tail) BOXCONV_LAUNCH(name, (narrow_forward_kernel<TO, L, EX, QUADS, false, false>), grid, dim3(64), 0, stream, a, tail); \
        else if (tail.residual == nullptr) BOXCONV_LAUNCH(name, (narrow_forward_kernel<TO, L, EX, QUADS, true, false>), grid, dim3(64), 0, stream, a, tail); \
        else BOXCONV_LAUNCH(name, (narrow_forward_kernel<TO, L, EX, QUADS, true, true>), grid, dim3(64), 0, stream, a, tail); \
    } while (0)
#define LAUNCH_NF(L)                                                                                                    \
    if (quads) { if (exact) LAUNCH_NF_TAIL(L, true, true); else LAUNCH_NF_TAIL(L, false, true); }                       \
    else       { if (exact) LAUNCH_NF_TAIL(L, true, false); else LAUNCH_NF_TAIL(L, false, false); }
    if (lanes == 8)       { LAUNCH_NF(8) }
    else if (lanes == 16) { LAUNCH_NF(16) }
    else                  { LAUNCH_NF(32) }
#undef LAUNCH_NF
#undef LAUNCH_NF_TAIL
    return hipGetLastError();
}

template hipError_t narrow_forward_launch<BOXCONV_INST_TO>(SampleArgs<float>, ForwardTail<BOXCONV_INST_TO>, Dims, bool, bool, hipStream_t);

}  // namespace boxconv
