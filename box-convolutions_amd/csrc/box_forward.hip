// Forward box sampling for gfx950: output[p][f] = box sums of integral plane p for box (c, f).
// Replaces cpu::boxConvUpdateOutput, src/box_convolution.cpp:100-261 (CUDA:
// box_convolution_cuda_forward.cu:28-251). The math and the row-streaming scheme are described at
// the top of box_sampling.hip.

#include "forward_tail.hpp"

namespace boxconv {

namespace {

// ---------------------------------------------------------------------------------------------
// Forward. Work item = (plane p, filter f, band). blockDim = NT, K >= ceil(w / NT).
// LDS: [2 buffers][w+3] RowPair<T>.
//
template <class T, class TO, int NT, int K, bool EXACT, bool FULL, bool TAIL>
__global__ void __launch_bounds__(NT) forward_rows_kernel(SampleArgs<T> a, ForwardTail<TO> tl) {
    const unsigned vid = xcd_contiguous_id(a.per_xcd);
    if (vid >= a.total) return;
    const unsigned nbands = a.nb, nfilt = a.F;
    // (plane, filter, band) order, or (plane, band, filter): see forward_launch_any
    const unsigned inner = a.band_major ? nfilt : nbands, outer = a.band_major ? nbands : nfilt;
    const unsigned v_in = vid % inner, v_rest = vid / inner;
    const unsigned v_out = v_rest % outer, p32 = v_rest / outer;
    const int band = static_cast<int>(a.band_major ? v_out : v_in);
    const int f = static_cast<int>(a.band_major ? v_in : v_out);
    const int64_t p = p32, pf = p * nfilt + f;
    const int k_par = static_cast<int>(static_cast<unsigned>(a.plane0 + p) % static_cast<unsigned>(a.C)) * a.F + f;
    const int h = a.h, w = a.w;
    const unsigned row_bytes = static_cast<unsigned>(w) * sizeof(T);

    const BoxOfWorkgroup<T> bx = load_box(a.prm, k_par);
    const BoxSplit<T> s = split_forward(bx.xmin, bx.xmax, bx.ymin, bx.ymax);
    const T scale = a.normalize
        ? inverse_extent(bx.xmin, bx.xmax, bx.ymin, bx.ymax, EXACT, true, true) : T(1);

    const int64_t pitch = w + 1;
    const T* plane = a.src + p * static_cast<int64_t>(h + 1) * pitch;
    // output rows start one element early so that column slot q = j + 1 lands on pixel j
    const LoadRows<T> irows(plane, pitch, w + 1, h + 1);
    const Rows<TO, FULL> orows(tl.dst + pf * static_cast<int64_t>(h) * w - 1, w, w + 1, h);
    const Rows<const TO, false> rrows((tl.residual != nullptr ? tl.residual : tl.dst) +
                                          pf * static_cast<int64_t>(h) * w - 1,
                                      w, tl.residual != nullptr ? w + 1 : 0, h);
    T ch_scale = T(1), ch_shift = T(0);
    if (TAIL) {
        if (tl.channel_scale != nullptr) ch_scale = static_cast<T>(tl.channel_scale[k_par]);
        if (tl.channel_shift != nullptr) ch_shift = static_cast<T>(tl.channel_shift[k_par]);
    }
    const bool relu = TAIL && tl.relu != 0;
    RowPair<T>* vbuf = reinterpret_cast<RowPair<T>*>(smem_raw);
    const int vlen = w + 3;
    clear_row_pads(vbuf, vlen);

    const int i0 = band * a.R;
    const int i1 = min(h, i0 + a.R);

    const int q1 = lane_q1<T>();
    const int qo = lane_q1<TO>();         // the same column slots in a row of TO
    unsigned lo[K], hi[K];
    column_taps<T, NT, K>(lo, hi, s.ylo, s.yhi, w);

    T ta[K], bc[K];                       // I[t(i-1)], I[b(i)]
    T t0[K], t1[K], b1[K], b2[K];         // I[t(i)], I[t(i+1)], I[b(i+1)], I[b(i+2)]
    load_row<T, NT, K>(irows.row(clampi(i0 + s.xlo - 1, 0, h)), q1, ta);
    load_row<T, NT, K>(irows.row(clampi(i0 + s.xhi, 0, h)), q1, bc);
    load_pair<T, NT, K, FULL>(irows, i0, s.xlo, s.xhi, h, q1, t0, t1, b1, b2);

    // One row pair. PREFETCH and the LDS buffer are compile-time tags: the loop body always
    // issues the next pair's loads and the last pair is peeled, so no branch joins a path with
    // loads in flight to one without (the wait-count insertion would have to drain the prefetch
    // at such a join); the loop is unrolled over both buffers so that LDS addresses are lane
    // constants plus immediates and the sliding rows rotate by renaming instead of moves.
    auto row_pair = [&](int i, auto prefetch_tag, auto flip_tag) {
        constexpr bool PREFETCH = decltype(prefetch_tag)::value;
        constexpr int FLIP = decltype(flip_tag)::value;
        T n0[K] = {}, n1[K] = {}, n2[K] = {}, n3[K] = {};
        if (PREFETCH)
            load_pair<T, NT, K, FULL>(irows, i + 2, s.xlo, s.xhi, h, q1, n0, n1, n2, n3);

        // residual of the two output rows: issued with the row loads, used after the barrier
        TO res0[K] = {}, res1[K] = {};
        if (TAIL) {
            const RowRef rb0 = rrows.row(i);
            const RowRef rb1 = rrows.row(min(i + 1, h - 1), i + 1 < i1);
#pragma unroll
            for (int k = 0; k < K; ++k) {
                res0[k] = load_slot<TO, NT, kCacheStream>(rb0, qo, k);
                res1[k] = load_slot<TO, NT, kCacheStream>(rb1, qo, k);
            }
        }

        RowPair<T>* V = vbuf + (FLIP ? vlen : 0);
        T v0[K], v1[K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            v0[k] = blend<T, EXACT>(ta[k], t0[k], bc[k], b1[k], s.fxlo, s.fxhi);
            v1[k] = blend<T, EXACT>(t0[k], t1[k], b1[k], b2[k], s.fxlo, s.fxhi);
        }
        publish_rows<T, NT, K, FULL>(V, v0, v1, w, row_bytes, q1);
        __syncthreads();

        const RowRef ob0 = orows.row(i);
        const RowRef ob1 = orows.row(min(i + 1, h - 1), i + 1 < i1);   // may lie past the band
#pragma unroll
        for (int k = 0; k < K; ++k) {
            if (slot_valid<T, NT, FULL>(q1, k, row_bytes)) {
                const RowPair<T> o = sample_columns<T, EXACT>(V, lo[k], hi[k], s.fylo, s.fyhi);
                T y0 = o.r0 * scale, y1 = o.r1 * scale;
                if (TAIL) {
                    y0 = y0 * ch_scale + ch_shift + static_cast<T>(widen(res0[k]));
                    y1 = y1 * ch_scale + ch_shift + static_cast<T>(widen(res1[k]));
                    if (relu) { y0 = y0 < T(0) ? T(0) : y0; y1 = y1 < T(0) ? T(0) : y1; }
                }
                TO z0, z1;
                narrow(y0, z0);
                narrow(y1, z1);
                if (a.stream_out) {                      // (workgroup-uniform)
                    store_slot<TO, NT, kCacheStream>(z0, ob0, qo, k);
                    store_slot<TO, NT, kCacheStream>(z1, ob1, qo, k);
                } else {
                    store_slot<TO, NT, kCacheDefault>(z0, ob0, qo, k);
                    store_slot<TO, NT, kCacheDefault>(z1, ob1, qo, k);
                }
            }
        }
        if (PREFETCH) {
#pragma unroll
            for (int k = 0; k < K; ++k) {
                ta[k] = t1[k]; bc[k] = b2[k];
                t0[k] = n0[k]; t1[k] = n1[k]; b1[k] = n2[k]; b2[k] = n3[k];
            }
        }
    };
    int i = i0;
    for (; i + 4 < i1; i += 4) {
        row_pair(i, std::true_type{}, Flip0{});
        row_pair(i + 2, std::true_type{}, Flip1{});
    }
    if (i + 2 < i1) {
        row_pair(i, std::true_type{}, Flip0{});
        row_pair(i + 2, std::false_type{}, Flip1{});
    } else {
        row_pair(i, std::false_type{}, Flip0{});
    }
}

// The same for float rows of up to 2048 columns: a lane owns 4 CONSECUTIVE columns, for the integral rows
// (one 16-byte load per row) as for the output (one 16- or 8-byte store per row), and V sits in LDS by
// column modulo four (tap_run). The planes hold V[1..w]; the places in front of them stay zero (V[0] =
// 0 and what clamps to it), those behind hold V[w]. Rows that are no multiple of four columns (FIT): the last
// lane takes the row's last four columns (RowLane) and stores those it shares with its neighbour, too: the
// same values. Not where the residual is the output itself: the neighbour may be in another wave, and what
// this lane stored early would be added a second time there.
// The tail's residual: none, or loaded with the ordinary or the streaming cache policy.
enum ResidualLoads { kNoResidual, kResidualCached, kResidualStreamed };
// Without a residual nothing is loaded for it (loads of the output in its place, dropped, cost a read as
// large as the output: 16 x 8 planes of 512 x 1024 in float16 153 -> 91 us, 256 x 4 of 128 x 256 in
// bfloat16, output not in any cache, 42 -> 26). With one, the rows of the next pair are requested
// with its integral rows: workgroups of few waves otherwise wait for memory right before the barrier
// (residual not in any cache, 46 planes of 398 x 140 in float32 12.1 -> 10.0 us, 128 x 4 of 135 x 240
// in bfloat16 27.7 -> 26.3); with two waves, and from five on, the registers cost more than that brings. From five on they have to
// fit six waves per SIMD: at five, which three registers more are enough for, 46 x 18 planes of 64 x 1164 in bfloat16 take 73.8 us instead
// of 67.4, 1 x 20 of 326 x 1608 17.1 instead of 14.4. Its cache policy: see forward_launch_any.
template <class TO, int NT, bool EXACT, int FIT, bool TAIL, int RESIDUAL>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(RESIDUAL != kNoResidual && NT > 256 && FIT != kRowAny ? 6 : 1))) forward_quads_kernel(SampleArgs<float> a, ForwardTail<TO> tl) {
    using T = float;
    constexpr int K = 4, PLANE = quad_plane(NT), WAVES = NT / 64;
    constexpr bool EARLY = RESIDUAL != kNoResidual && WAVES <= 4 && WAVES != 2;   // residual rows a pair ahead
    __shared__ __align__(16) RowPair<T> vrow[2][K][PLANE];
    const unsigned vid = xcd_contiguous_id(a.per_xcd);
    if (vid >= a.total) return;                      // whole workgroup leaves together
    const unsigned nbands = a.nb, nfilt = a.F;
    const unsigned inner = a.band_major ? nfilt : nbands, outer = a.band_major ? nbands : nfilt;
    const unsigned v_in = vid % inner, v_rest = vid / inner;
    const unsigned v_out = v_rest % outer, p32 = v_rest / outer;
    const int band = static_cast<int>(a.band_major ? v_out : v_in);
    const int f = static_cast<int>(a.band_major ? v_in : v_out);
    const int64_t p = p32, pf = p * nfilt + f;
    const int k_par = static_cast<int>(static_cast<unsigned>(a.plane0 + p) % static_cast<unsigned>(a.C)) * a.F + f;
    const int h = a.h, w = a.w, tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr bool ALIGNED = FIT != kRowAny;
    const RowLane<NT, FIT> ln(tid, w);
    const int quads = ln.quads;
    const bool lane_in = ln.in;
    const unsigned cl = static_cast<unsigned>(ln.cl);

    const BoxOfWorkgroup<T> bx = load_box(a.prm, k_par);
    BoxSplit<T> s = split_forward(bx.xmin, bx.xmax, bx.ymin, bx.ymax);
    s.xlo = __builtin_amdgcn_readfirstlane(s.xlo); s.xhi = __builtin_amdgcn_readfirstlane(s.xhi);
    s.ylo = __builtin_amdgcn_readfirstlane(s.ylo); s.yhi = __builtin_amdgcn_readfirstlane(s.yhi);
    const T scale = a.normalize
        ? inverse_extent(bx.xmin, bx.xmax, bx.ymin, bx.ymax, EXACT, true, true) : T(1);

    const int64_t pitch = w + 1;
    const T* plane = a.src + p * static_cast<int64_t>(h + 1) * pitch + 1;
    auto load_i = [&](int r, T (&dst)[K]) {
        load4_dword_aligned(at_bytes(plane + clampi(r, 0, h) * pitch, 4u * cl), dst);
    };
    const int64_t out0 = pf * static_cast<int64_t>(h) * w;
    T ch_scale = T(1), ch_shift = T(0);
    if (TAIL) {
        if (tl.channel_scale != nullptr) ch_scale = tl.channel_scale[k_par];
        if (tl.channel_shift != nullptr) ch_shift = tl.channel_shift[k_par];
    }
    const bool relu = TAIL && tl.relu != 0;
    const bool in_place = RESIDUAL != kNoResidual && FIT == kRowAny && tl.residual == tl.dst;

    if (tid < 2 * K * kQuadPad)
        vrow[tid / (K * kQuadPad)][tid / kQuadPad % K][tid % kQuadPad] = RowPair<T>{T(0), T(0)};
    const TapRun er = tap_run<PLANE>(ln.c0, s.yhi - 1, quads), el = tap_run<PLANE>(ln.c0, s.ylo - 2, quads);
    const QuadPlace<PLANE, FIT> place(ln);
    const int last = (quads - 1) & 63;               // lane of the last wave that owns column w

    const int i0 = band * a.R;
    const int i1 = min(h, i0 + a.R);
    T ta[K], bc[K];                       // I[t(i-1)], I[b(i)]
    T t0[K], t1[K], b1[K], b2[K];         // I[t(i)], I[t(i+1)], I[b(i+1)], I[b(i+2)]
    auto load_residual = [&](int i, Quad<TO>& q0, Quad<TO>& q1) {
        const int64_t row = out0 + static_cast<int64_t>(i) * w;
        q0 = load_quad<RESIDUAL == kResidualStreamed, ALIGNED>(tl.residual + row + cl);
        q1 = load_quad<RESIDUAL == kResidualStreamed, ALIGNED>(tl.residual + (i + 1 < i1 ? row + w : row) + cl);
    };
    Quad<TO> res0{}, res1{};
    if (EARLY) {                          // in front of the integral rows: they mostly come from the L2, the residual from memory
        load_residual(i0, res0, res1);    // (behind them 256 x 4 planes of 128 x 256 in bfloat16 41.2 -> 41.6 us)
        __builtin_amdgcn_sched_barrier(0);
    }
    load_i(i0 + s.xlo - 1, ta);
    load_i(i0 + s.xhi, bc);
    load_i(i0 + s.xlo, t0);
    load_i(i0 + 1 + s.xlo, t1);
    load_i(i0 + 1 + s.xhi, b1);
    load_i(i0 + 2 + s.xhi, b2);

    auto row_pair = [&](int i, auto prefetch_tag, auto flip_tag) {
        constexpr bool PREFETCH = decltype(prefetch_tag)::value;
        constexpr int FLIP = decltype(flip_tag)::value;
        T n0[K] = {}, n1[K] = {}, n2[K] = {}, n3[K] = {};
        Quad<TO> m0{}, m1{};
        if (PREFETCH) {
            if (EARLY) load_residual(i + 2, m0, m1);
            load_i(i + 2 + s.xlo, n0);
            load_i(i + 3 + s.xlo, n1);
            load_i(i + 3 + s.xhi, n2);
            load_i(i + 4 + s.xhi, n3);
        }
        const bool second = i + 1 < i1;
        const int64_t row0 = out0 + static_cast<int64_t>(i) * w, row1 = second ? row0 + w : row0;
        if (RESIDUAL != kNoResidual && !EARLY) load_residual(i, res0, res1);
        T v0[K], v1[K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            v0[k] = blend<T, EXACT>(ta[k], t0[k], bc[k], b1[k], s.fxlo, s.fxhi);
            v1[k] = blend<T, EXACT>(t0[k], t1[k], b1[k], b2[k], s.fxlo, s.fxhi);
        }
#pragma unroll
        for (int k = 0; k < K; ++k) *place.at(vrow[FLIP][0], k) = RowPair<T>{v0[k], v1[k]};
        if (wave == WAVES - 1) {                     // (scalar)
            const RowPair<T> end{read_lane(v0[K - 1], last), read_lane(v1[K - 1], last)};
            const int e = tid & 63;
            if (e < K * kQuadPad) vrow[FLIP][e / kQuadPad][kQuadPad + quads + e % kQuadPad] = end;
            else if (FIT == kRowAny && e - K * kQuadPad < K && e - K * kQuadPad >= w % K)   // (the rest of the last quad)
                vrow[FLIP][e - K * kQuadPad][kQuadPad + quads - 1] = end;
        }
        __syncthreads();

        RowPair<T> R[K + 1], L[K + 1];
        read_taps(vrow[FLIP][0], er, R);
        read_taps(vrow[FLIP][0], el, L);
        Quad<TO> z0, z1;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            T y0 = blend<T, EXACT>(L[k].r0, L[k + 1].r0, R[k].r0, R[k + 1].r0, s.fylo, s.fyhi) * scale;
            T y1 = blend<T, EXACT>(L[k].r1, L[k + 1].r1, R[k].r1, R[k + 1].r1, s.fylo, s.fyhi) * scale;
            if (TAIL) {
                y0 = y0 * ch_scale + ch_shift + (RESIDUAL != kNoResidual ? widen(res0.v[k]) : T(0));
                y1 = y1 * ch_scale + ch_shift + (RESIDUAL != kNoResidual ? widen(res1.v[k]) : T(0));
                if (relu) { y0 = y0 < T(0) ? T(0) : y0; y1 = y1 < T(0) ? T(0) : y1; }
            }
            narrow(y0, z0.v[k]);
            narrow(y1, z1.v[k]);
        }
        if (in_place) {                              // (scalar)
#pragma unroll
            for (int k = 0; k < K; ++k)
                if (ln.owns(k)) {
                    tl.dst[row0 + cl + k] = z0.v[k];
                    if (second) tl.dst[row1 + cl + k] = z1.v[k];
                }
        } else if (FIT == kRowFull || lane_in) {
            store_quad<ALIGNED>(tl.dst + row0 + cl, z0, a.stream_out != 0);
            if (second) store_quad<ALIGNED>(tl.dst + row1 + cl, z1, a.stream_out != 0);
        }
        if (PREFETCH) {
#pragma unroll
            for (int k = 0; k < K; ++k) {
                ta[k] = t1[k]; bc[k] = b2[k];
                t0[k] = n0[k]; t1[k] = n1[k]; b1[k] = n2[k]; b2[k] = n3[k];
            }
            if (EARLY) { res0 = m0; res1 = m1; }
        }
    };
    int i = i0;
    for (; i + 4 < i1; i += 4) {
        row_pair(i, std::true_type{}, Flip0{});
        row_pair(i + 2, std::true_type{}, Flip1{});
    }
    if (i + 2 < i1) {
        row_pair(i, std::true_type{}, Flip0{});
        row_pair(i + 2, std::false_type{}, Flip1{});
    } else {
        row_pair(i, std::false_type{}, Flip0{});
    }
}

template <class T, class TO, bool EXACT, bool TAIL>
__global__ void __launch_bounds__(256) forward_gather_kernel(SampleArgs<T> a, ForwardTail<TO> tl) {
    const int64_t hw = static_cast<int64_t>(a.h) * a.w;
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (idx >= a.total) return;
    const int64_t pf = idx / hw;
    const int pix = static_cast<int>(idx % hw);
    const int i = pix / a.w, j = pix % a.w;
    const int64_t p = pf / a.F;
    const int k_par = static_cast<int>(static_cast<unsigned>(a.plane0 + p) % static_cast<unsigned>(a.C)) * a.F + static_cast<int>(pf % a.F);
    const BoxOfWorkgroup<T> bx = load_box(a.prm, k_par);
    const BoxSplit<T> s = split_forward(bx.xmin, bx.xmax, bx.ymin, bx.ymax);
    const T scale = a.normalize
        ? inverse_extent(bx.xmin, bx.xmax, bx.ymin, bx.ymax, EXACT, true, true) : T(1);
    const T* plane = a.src + p * static_cast<int64_t>(a.h + 1) * (a.w + 1);
    T y = gather_box<T, EXACT>(plane, s, i, j, a.h, a.w) * scale;
    if (TAIL) {
        const T ch_scale = tl.channel_scale != nullptr ? static_cast<T>(tl.channel_scale[k_par]) : T(1);
        const T ch_shift = tl.channel_shift != nullptr ? static_cast<T>(tl.channel_shift[k_par]) : T(0);
        const T res = tl.residual != nullptr ? static_cast<T>(widen(tl.residual[idx])) : T(0);
        y = y * ch_scale + ch_shift + res;
        if (tl.relu != 0 && y < T(0)) y = T(0);
    }
    narrow(y, tl.dst[idx]);
}

}  // namespace

namespace {

// Rows that one wave covers: where four consecutive columns per lane (forward_quads_kernel) are
// faster than columns 64 apart (forward_rows_kernel), by columns, output pixels and element size.
// Both were timed on 8000 shapes, output buffers reused and in no cache; time of the first over the
// second:
//  * fewer than 96 columns leave too many lanes idle; exactly 128 fill the other kernel's two waves
//    (0.96 to 1.25);
//  * 96 to 127 are two waves at one column per lane there, a shorter chain: 1.1 to 1.3 below 2^21
//    pixels, 0.85 to 0.93 above;
//  * 129 to 192 are three columns per lane there and leave fewer lanes idle: 0.87 to 0.97 below 2^22
//    pixels, 1.0 to 1.25 above; with a residual 0.8 and 1.0 (in no cache) there too;
//  * 193 to 256: 0.70 to 0.97. But float32 rows that start on 64-byte boundaries, which the other
//    kernel stores best: no tail 1.0 to 1.17 from 2^22 pixels (208 to 240 columns), and 256 columns
//    0.92 to 1.02 below 2^25 pixels, 1.0 to 1.1 above;
//  * output and integral images that do not fit the memory-side cache together: 1.2 to 1.9 (408 x 4
//    planes of 330 x 160 70 against 130 us, 308 x 2 of 794 x 112 62 against 101), except with a residual
//    and for 129 columns and more that do not start on 64-byte boundaries (0.8 to 0.9).
bool one_wave_quads_pay(int w, uint64_t pixels, uint64_t integral_bytes, size_t elem_size, bool tail, bool residual) {
    if (w < 96) return false;
    if (switches().quads_any_size) return true;
    if (w == 128) return false;
    const bool whole_sectors = static_cast<size_t>(w) * elem_size % 64 == 0;
    if (!residual && pixels * elem_size + integral_bytes >= (256ull << 20)) return w > 128 && !whole_sectors;
    if (w < 128) return pixels >= (1ull << 21);
    if (w <= 192) return residual || pixels < (1ull << 22);
    if (elem_size == 4 && whole_sectors) return w == 256 ? pixels < (1ull << 25) : tail || pixels < (1ull << 22);
    return true;
}

}  // namespace

// TAIL selects the kernels with the fused tail; without it only tail.dst is used.
template <class T, class TO, bool TAIL>
hipError_t forward_launch_any(const T* integ, BoxParams<T> prm, ForwardTail<TO> tail, Dims d,
                              bool normalize, bool exact, hipStream_t stream) {
    const int64_t planes_f = d.planes * d.F;
    if (planes_f == 0 || d.hw() == 0) return hipSuccess;
    SampleArgs<T> a = base_args(prm, d);
    a.src = integ; a.normalize = normalize ? 1 : 0;

    // (the row kernel keeps two row pairs of w + 3 columns in LDS, up to 64 KiB + 48 bytes for the
    // widest rows it takes; a device that grants a workgroup less goes to the gather kernel)
    if (!row_kernels_apply(d.h, d.w, sizeof(T)) ||
        4 * static_cast<size_t>(d.w + 3) * sizeof(T) > std::min(kMaxDynamicLds, device_lds_limit())) {
        finish_args(a, planes_f * d.hw());
        const dim3 grid(static_cast<unsigned>((a.total + 255) / 256));
        if (exact) BOXCONV_LAUNCH("forward_gather", (forward_gather_kernel<T, TO, true, TAIL>), grid, dim3(256), 0, stream, a, tail);
        else       BOXCONV_LAUNCH("forward_gather", (forward_gather_kernel<T, TO, false, TAIL>), grid, dim3(256), 0, stream, a, tail);
        return hipGetLastError();
    }

    const RowConfig rc = row_config(d.w, switches().fwd_threads);
    // Many short-lived workgroups (bands of 8 rows at the headline size): the kernel then ends
    // with a short tail. Measured per step: 16 workgroup-waves' worth of bands 0.501 ms, 8 0.508 ms,
    // 4 0.517 ms, 32 (bands of 4 rows, too much halo) 0.523 ms.
    a.nb = bands_for(planes_f, d.h, 8, 16384);
    a.R = (d.h + a.nb - 1) / a.nb;
    a.R += a.R & 1;                                   // rows are handled in pairs
    a.nb = (d.h + a.R - 1) / a.R;
    finish_args(a, planes_f * a.nb);
    // An integral plane that does not fit an XCD's 4 MB L2 is streamed from memory once per filter
    // when the bands of one filter run one after the other; with the filters of a band side by
    // side their rows (a box height apart at most) are fetched together (1024 x 2048 with two
    // filters: 737 -> 703 us). Planes that fit are faster in filter order (512 x 1024: 97 vs 100 us).
    a.band_major = (static_cast<uint64_t>(d.h + 1) * (d.w + 1) * sizeof(T) > (4u << 20)) ? 1 : 0;
    // The output is written once and not read again by this pass: non-temporal stores keep it out
    // of the way of the integral rows in the caches (512 x 1024, 16 x 8 planes: 97 against 130 us,
    // and the grad-input pass that follows 121 against 132). A lane stores one element per
    // instruction, though, and where rows do not start on 64-byte boundaries such stores reach
    // memory as partly covered 32-byte sectors that nothing merges any more: 256 x 132, 16 x 64
    // planes, 61 against 37 us; 256 x 300 51 against 38. Such rows keep the ordinary policy while
    // the output fits the memory-side cache; beyond that the streaming policy wins even so
    // (500 x 1000, 512 MB: 128 against 142 us, and the next pass 122 against 138).
    const uint64_t out_bytes = static_cast<uint64_t>(planes_f) * d.hw() * sizeof(TO);
    a.stream_out = ((static_cast<uint64_t>(d.w) * sizeof(TO)) % 64 == 0 || out_bytes > (256ull << 20)) ? 1 : 0;
    const dim3 grid(static_cast<unsigned>(a.per_xcd * kXcds));
    if constexpr (std::is_same<T, float>::value) {
        if (narrow_forward_pays(d.planes, d.F, d.h, d.w, sizeof(TO), TAIL))
            return narrow_forward_launch<TO>(a, tail, d, TAIL, exact, stream);
        // Four consecutive columns per lane: rows of one wave where one_wave_quads_pay says so, and
        // 16-bit outputs of wider rows, where the other kernel stores 2 bytes per lane. Measured, us, other
        // kernel -> this one: bfloat16 16 x 8 planes of 300 x 768 with the tail 74 -> 50, 1080 x 1920 380 -> 321;
        // without it 512 x 1024 118 -> 90, 720 x 1280 97 -> 76. Not for wider float32 rows (256 x 512 54 -> 72,
        // 720 x 1280 105 -> 111, 1080 x 1920 229 -> 373: stores of 16 bytes per lane reach the memory no
        // better, and the loads start at odd addresses), nor without a tail beyond 1280 columns
        // (1080 x 1920 213 -> 237) or where an eighth of the lanes idles (200 x 384 27 -> 31).
        const int lanes = d.w / 4, cnt = consecutive_threads(d.w);
        const uint64_t integral_bytes = static_cast<uint64_t>(d.planes) * (d.h + 1) * (d.w + 1) * sizeof(T);
        const bool one_wave = cnt == 64 && one_wave_quads_pay(d.w, static_cast<uint64_t>(planes_f) * d.hw(), integral_bytes,
                                                              sizeof(TO), TAIL, tail.residual != nullptr);
        const bool wide_half = sizeof(TO) == 2 && cnt > 64 && (TAIL || (d.w <= 1280 && lanes * 8 >= cnt * 7));
        const size_t align = 4 * sizeof(TO);
        const bool quads = d.w % 4 == 0 && (one_wave || wide_half) && reinterpret_cast<uintptr_t>(tail.dst) % align == 0 &&
                           reinterpret_cast<uintptr_t>(tail.residual) % align == 0;
        const bool odd = odd_forward_quads_pay(d.planes, d.F, d.h, d.w, sizeof(TO), TAIL);
        if (switches().forward_quads && d.w <= 2048 && (quads || odd)) {
            // A residual that an earlier layer has just left in the memory-side cache is worth reading from
            // there (256 x 4 planes of 128 x 256 in bfloat16 30 us, 40 with the streaming policy); one that
            // does not fit it beside the output would only push that out (16-bit outputs, 16 x 8 planes of
            // 512 x 1024 153 -> 150 us, of 720 x 1280 158 -> 149, of 1080 x 1920 335 -> 321; float32 of 128 MB
            // and more 0.9 of the time).
            const bool stream_residual = out_bytes > (128ull << 20);
#define LAUNCH_FQ_TAIL(NT, EX, FU)                                                                                     \
    do {                                                                                                               \
        if constexpr (TAIL)                                                                                            \
            if (tail.residual != nullptr) {                                                                            \
                if (stream_residual)                                                                                   \
                    BOXCONV_LAUNCH("forward_quads", (forward_quads_kernel<TO, NT, EX, FU, true, kResidualStreamed>), grid, dim3(NT), 0, stream, a, tail); \
                else                                                                                                   \
                    BOXCONV_LAUNCH("forward_quads", (forward_quads_kernel<TO, NT, EX, FU, true, kResidualCached>), grid, dim3(NT), 0, stream, a, tail); \
                break;                                                                                                 \
            }                                                                                                          \
        BOXCONV_LAUNCH("forward_quads", (forward_quads_kernel<TO, NT, EX, FU, TAIL, kNoResidual>), grid, dim3(NT), 0, stream, a, tail); \
    } while (0)
#define LAUNCH_FQ(NT)                                                                                                  \
    case NT:                                                                                                           \
        if (odd) { if (exact) LAUNCH_FQ_TAIL(NT, true, kRowAny); else LAUNCH_FQ_TAIL(NT, false, kRowAny); }            \
        else if (lanes == NT) { if (exact) LAUNCH_FQ_TAIL(NT, true, kRowFull); else LAUNCH_FQ_TAIL(NT, false, kRowFull); } \
        else     { if (exact) LAUNCH_FQ_TAIL(NT, true, kRowQuads); else LAUNCH_FQ_TAIL(NT, false, kRowQuads); }        \
        break;
            switch (cnt) {
                LAUNCH_FQ(64) LAUNCH_FQ(128) LAUNCH_FQ(192) LAUNCH_FQ(256)
                LAUNCH_FQ(320) LAUNCH_FQ(384) LAUNCH_FQ(448) LAUNCH_FQ(512)
                default: return hipErrorInvalidValue;
            }
#undef LAUNCH_FQ
#undef LAUNCH_FQ_TAIL
            return hipGetLastError();
        }
    }
    const size_t lds = 4 * static_cast<size_t>(d.w + 3) * sizeof(T);
#define LAUNCH_FWD(NT, KK, EX, FU) \
    BOXCONV_LAUNCH("forward_rows", (forward_rows_kernel<T, TO, NT, KK, EX, FU, TAIL>), grid, dim3(NT), lds, stream, a, tail)
    BOXCONV_DISPATCH_SHAPE_EXACT_FULL(LAUNCH_FWD, rc, exact)
#undef LAUNCH_FWD
    return hipGetLastError();
}

template <class T>
hipError_t forward_launch(const T* integ, BoxParams<T> prm, T* out, Dims d, bool normalize,
                          bool exact, hipStream_t stream) {
    return forward_launch_any<T, T, false>(integ, prm, ForwardTail<T>{out, nullptr, nullptr, nullptr, 0},
                                           d, normalize, exact, stream);
}

template <class TO>
hipError_t forward_fused_launch(const float* integ, BoxParams<float> prm, TO* out, const TO* residual,
                                const float* channel_scale, const float* channel_shift, bool relu,
                                Dims d, bool normalize, bool exact, hipStream_t stream) {
    const ForwardTail<TO> tail{out, residual, channel_scale, channel_shift, relu ? 1 : 0};
    if (residual == nullptr && channel_scale == nullptr && channel_shift == nullptr && !relu)
        return forward_launch_any<float, TO, false>(integ, prm, tail, d, normalize, exact, stream);
    return forward_launch_any<float, TO, true>(integ, prm, tail, d, normalize, exact, stream);
}

// Compiled once per element type of the output (BOXCONV_INST_TO).
#ifdef BOXCONV_INST_DOUBLE
template hipError_t forward_launch<double>(const double*, BoxParams<double>, double*, Dims, bool, bool, hipStream_t);
#else
template hipError_t forward_fused_launch<BOXCONV_INST_TO>(const float*, BoxParams<float>, BOXCONV_INST_TO*, const BOXCONV_INST_TO*,
                                                          const float*, const float*, bool, Dims, bool, bool, hipStream_t);
#ifdef BOXCONV_INST_SAME_TYPE
template hipError_t forward_launch<float>(const float*, BoxParams<float>, float*, Dims, bool, bool, hipStream_t);
#endif
#endif

}  // namespace boxconv
