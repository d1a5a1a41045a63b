// Both backward kernels for rows of at most 128 columns, which would leave half and more of the lanes
// of grad_output_stream_consec_kernel and grad_input_taps_kernel idle (they replace the same reference
// code: src/box_convolution.cpp:480-715 and :286-456). Compiled once per element type of grad_output
// (BOXCONV_INST_TG). The math and the snapshots that connect the two are those of these kernels; the
// difference is how a wave is filled: 64 / L rows side by side, L = 8, 16 or 32 lanes of four
// consecutive columns each, every lane walking down its own rows:
//  * narrow_sums_kernel: a wave takes 64 / L neighbouring bands of one (plane, filter). Its box is the
//    same in all lanes, so only row addresses are per lane; rows per band are a multiple of the
//    snapshots' group, so that a row whose sum is kept is kept by all bands at the same step.
//  * narrow_input_kernel: a wave takes 64 / L neighbouring groups of 8 output rows of one plane. Waves
//    of a workgroup share the filters of their groups and add their sums up through LDS at the end:
//    a wave that walks through all filters alone is one chain of their memory round trips.
// Waves do not wait for each other inside a row pair: what a wave reads from LDS it wrote itself.
// Both kernels are bound by instruction issue (64 planes of 64 x 128 with 4 filters, batch 8: the vector ALU
// issues for 15 of 20 us of the sums), so what a row costs beside its arithmetic counts: its address
// is two instructions per lane, and a branch that mostly no lane takes guards what only some rows need.
// Against the kernels for wider rows, both gradients, float32: 64 x 128, 512 x 4 planes 61 -> 42 us; 64 x 64 48 -> 29;
// 928 x 32, 78 x 19 planes 287 -> 108; 72 x 107, 671 x 37 planes 807 -> 519; 833 x 23, 578 planes 139 -> 60.

#include "box_sampling_impl.hpp"
#include "narrow_rows.hpp"

namespace boxconv {

namespace {

// Snapshots of these kernels: per (plane, filter) a row of zeros, the rows for the upper and the lower edge of
// the mirrored box (one per group of output rows each), the sum of every band.
__device__ __forceinline__ int narrow_snapshot_rows(const SampleArgs<float>& a) { return 1 + snapshot_rows(a); }

// Running sums within the L lanes that share a row.
template <int L, class A>
__device__ __forceinline__ A row_scan(A x, int l) {
    if (L == 8) {
        A y = dpp_move<0x111, 0xf>(x, x);
        x += l >= 1 ? y : A(0);
        y = dpp_move<0x112, 0xf>(x, x);
        x += l >= 2 ? y : A(0);
        y = dpp_move<0x114, 0xf>(x, x);
        x += l >= 4 ? y : A(0);
        return x;
    }
    x += dpp_move<0x111, 0xf>(x, x);
    x += dpp_move<0x112, 0xf>(x, x);
    x += dpp_move<0x114, 0xf>(x, x);
    x += dpp_move<0x118, 0xf>(x, x);
    if (L == 32) x += dpp_move<0x142, 0xa>(A(0), x);
    return x;
}

// ---------------------------------------------------------------------------------------------
// SNAP: snapshots for narrow_input_kernel, else the parameter sums alone. QUADS: rows of a multiple of
// four columns, aligned to four elements.
template <class TG, int L, bool EXACT, bool QUADS, bool SNAP>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(SNAP ? 3 : 4, 4)))
narrow_sums_kernel(SampleArgs<float> a) {
    using T = float;
    using Lane = NarrowLane<L>;
    constexpr int K = 4, S = Lane::S, PLANE = Lane::PLANE;
    struct alignas(16) LastColumn { T v, dt, db, unused; };
    __shared__ __align__(16) RowPair<T> grow[2][K * PLANE];
    __shared__ LastColumn xw[2][64];                 // of every lane: its row's last one is read
    __shared__ double red[5];

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
    const int band = slot * S + ln.seg;
    const int i0 = band * R, i1 = min(h, i0 + R);         // (a band past the plane: no rows)
    const int rows = uniform(min(R, h - slot * S * R));   // of the wave's first band: the most that any has
    const int whole = uniform(max(0, min(R, h - (slot * S + S - 1) * R)));   // rows that every band has

    const BoxOfWorkgroup<T> bx = load_box(a.prm, k_par);
    BoxSplit<T> s = split_grad_params(bx.xmin, bx.xmax, bx.ymin, bx.ymax);
    s.xlo = uniform(s.xlo); s.xhi = uniform(s.xhi); s.ylo = uniform(s.ylo); s.yhi = uniform(s.yhi);
    const BoxSplit<T> sm = split_grad_input(bx.xmin, bx.xmax, bx.ymin, bx.ymax);
    const int snap_lo = uniform(sm.xlo), snap_hi = uniform(sm.xhi);

    const int64_t mpitch = a.mpitch;
    const T* iplane = a.src + p * static_cast<int64_t>(h + 1) * (w + 1) + 1;
    const TG* gplane = reinterpret_cast<const TG*>(a.grad_out) + pf * static_cast<int64_t>(h) * w;
    const unsigned i_bytes = 4u * static_cast<unsigned>(w + 1), g_bytes = static_cast<unsigned>(sizeof(TG)) * static_cast<unsigned>(w);
    // The upper rows end at those of the plane's last output row, and so do the lower ones: a row behind it, of
    // which bands past the plane have many, adds V times zero, and what only it would read may be infinite.
    const int top_last = uniform(min(max(h - 1 + s.xlo, 0), h)), bottom_last = uniform(min(max(h + s.xhi, 0), h));
    auto load_i = [&](int r, int last, T (&dst)[K]) {
        load4_dword_aligned(at_bytes(iplane, row_offset(confine(r, last), i_bytes, 4u * ln.cl)), dst);
    };
    auto load_g = [&](int i, RawQuad<TG>& q) {
        q.template load<QUADS>(at_bytes(gplane, row_offset(min(i, h - 1), g_bytes, static_cast<unsigned>(sizeof(TG)) * ln.cl)));
    };
    auto load_window = [&](int i, T (&t0)[K], T (&t1)[K], T (&b1)[K], T (&b2)[K]) {
        load_i(i + s.xlo, top_last, t0);
        load_i(i + 1 + s.xlo, top_last, t1);
        load_i(i + 1 + s.xhi, bottom_last, b1);
        load_i(i + 2 + s.xhi, bottom_last, b2);
    };
    RawQuad<TG> r0, r1;
    load_g(i0, r0);
    load_g(i0 + 1, r1);

    // zeros around the rows (and behind them: nobody writes there)
    for (int e = threadIdx.x; e < 2 * K * PLANE; e += 64) (&grow[0][0])[e] = RowPair<T>{T(0), T(0)};
    T* const snap = a.dst + (pf * narrow_snapshot_rows(a) + 1) * mpitch;
    if (SNAP && slot == 0 && threadIdx.x < L && ln.in) store_row_quad<QUADS>(snap - mpitch + ln.cl, Quad<T>{});

    T delta[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int j = ln.c0 + k;
        const T d = (EXACT ? (T(1) - s.fyhi) : T(1)) * T(j > w - s.yhi) + (EXACT ? s.fyhi : T(0)) * T(j > w - s.yhi - 1)
                  - (EXACT ? (T(1) - s.fylo) : T(1)) * T(j > w - s.ylo) - (EXACT ? s.fylo : T(0)) * T(j > w - s.ylo + 1);
        delta[k] = ln.owns(k) ? d : T(0);
    }
    const TapRun er = ln.taps(-s.yhi), el = ln.taps(1 - s.ylo);
    unsigned place[QUADS ? 1 : K];
#pragma unroll
    for (int k = 0; k < (QUADS ? 1 : K); ++k) place[k] = ln.place(k);
    auto own = [&](RowPair<T>* row, int k) {
        return QUADS ? at_bytes(row + k * PLANE, place[0]) : at_bytes(row, place[QUADS ? 0 : k]);
    };
    // the two single taps of column w, for the row's first lane (all others: a zero)
    auto place_of = [&](int j) {
        return ln.seg * Lane::ROW + (ln.l == 0 && j >= 0 && j < w ? (j & (K - 1)) * PLANE + j / K + kQuadPad : 0);
    };
    const int at_ymax = place_of(w - s.yhi), at_ymin = place_of(w - s.ylo + 1);
    const int owner = ln.seg * L + ln.quads - 1;     // the lane whose last column is column w

    double total[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    T colacc[K] = {T(0), T(0), T(0), T(0)};
    T ta[K], bc[K], t0[K], t1[K], b1[K], b2[K];
    load_i(i0 + s.xlo - 1, top_last, ta);
    load_i(i0 + s.xhi, bottom_last, bc);
    load_window(i0, t0, t1, b1, b2);

    const int mask = (1 << a.snap_shift) - 1;
    // the sums of the bands' first `r` rows, where narrow_input_kernel will want them (the same step for
    // all bands: they start on multiples of the group's rows)
    auto keep_snapshots = [&](int r) {
        const Quad<T> q{{colacc[0], colacc[1], colacc[2], colacc[3]}};
        const bool lane_row = ln.in && i0 + r <= i1;
        auto keep = [&](int edge, int first) {
            if (((r - edge) & mask) != 0) return;
            const int u = i0 + r - edge, group = u >> a.snap_shift;
            if (lane_row && u >= 0 && group < a.snap_groups)
                store_row_quad<QUADS>(snap + (first + group) * mpitch + ln.cl, q);
        };
        keep(snap_lo, 0);
        keep(snap_hi, a.snap_groups);
    };

    // Rows i, i+1 into LDS buffer FL, the lane's share of their tails, and the column sums. A macro for the
    // reason given at BOXCONV_PUBLISH_PAIR.
#define BOXCONV_PUBLISH_NARROW(FL, LR, RA, RB_, TL0, TL1)                                           \
    {                                                                                               \
        T ga[K], gb[K];                                                                             \
        _Pragma("unroll")                                                                           \
        for (int k = 0; k < K; ++k) { ga[k] = RA.get(k); gb[k] = RB_.get(k); }                      \
        if ((LR) + 1 >= whole) {                     /* (scalar, and kept a branch) */              \
            _Pragma("unroll")                                                                       \
            for (int k = 0; k < K; ++k) {                                                           \
                ga[k] = i0 + (LR) < i1 ? ga[k] : T(0);                                              \
                gb[k] = i0 + (LR) + 1 < i1 ? gb[k] : T(0);                                          \
                finish_here(ga[k]); finish_here(gb[k]);                                             \
            }                                                                                       \
        }                                                                                           \
        _Pragma("unroll")                                                                           \
        for (int k = 0; k < K; ++k) *own(grow[FL], k) = RowPair<T>{ga[k], gb[k]};                   \
        TL0 = T(0); TL1 = T(0);                                                                     \
        _Pragma("unroll")                                                                           \
        for (int k = 0; k < K; ++k) { TL0 += delta[k] * ga[k]; TL1 += delta[k] * gb[k]; }           \
        if (SNAP) {                                                                                 \
            _Pragma("unroll")                                                                       \
            for (int k = 0; k < K; ++k) colacc[k] += ga[k];                                         \
            keep_snapshots((LR) + 1);                                                               \
            _Pragma("unroll")                                                                       \
            for (int k = 0; k < K; ++k) colacc[k] += gb[k];                                         \
            keep_snapshots((LR) + 2);                                                               \
        }                                                                                           \
    }

    T tl0, tl1;
    wave_lds_order();                                // (the zeros above come first)
    BOXCONV_PUBLISH_NARROW(0, 0, r0, r1, tl0, tl1)
    wave_lds_order();

    auto row_pair = [&](int lr, auto prefetch_tag, auto flip_tag) {
        constexpr bool PREFETCH = decltype(prefetch_tag)::value;
        constexpr int FLIP = decltype(flip_tag)::value;
        T n0[K] = {}, n1[K] = {}, n2[K] = {}, n3[K] = {};
        RawQuad<TG> m0{}, m1{};
        if (PREFETCH) {
            load_window(i0 + lr + 2, n0, n1, n2, n3);
            load_g(i0 + lr + 2, m0);
            load_g(i0 + lr + 3, m1);
        }
        const RowPair<T>* G = grow[FLIP];
        {
            T v0[K], v1[K];
#pragma unroll
            for (int k = 0; k < K; ++k) {
                v0[k] = bc[k] - t0[k]; v1[k] = b1[k] - t1[k];
                if (EXACT) {
                    v0[k] += s.fxhi * (b1[k] - bc[k]); v0[k] += s.fxlo * (t0[k] - ta[k]);
                    v1[k] += s.fxhi * (b2[k] - b1[k]); v1[k] += s.fxlo * (t1[k] - t0[k]);
                }
            }
            xw[0][threadIdx.x] = LastColumn{v0[K - 1], t0[K - 1] - ta[K - 1], b1[K - 1] - bc[K - 1], T(0)};
            xw[1][threadIdx.x] = LastColumn{v1[K - 1], t1[K - 1] - t0[K - 1], b2[K - 1] - b1[K - 1], T(0)};
            wave_lds_order();
            // The row pair's share of a column goes to double at once (two products, as in the kernel for wider rows
            // at one column per lane). finish_here: left alone the compiler holds all the sums back and spills.
            auto add = [&](const T (&sum)[5]) {
#pragma unroll
                for (int n = 0; n < 5; ++n) {
                    T part = sum[n];
                    finish_here(part);
                    total[n] += static_cast<double>(part);
                    finish_here(total[n]);
                }
            };
            {
                const LastColumn x0 = xw[0][owner], x1 = xw[1][owner];
                const RowPair<T> gmax = G[at_ymax], gmin = G[at_ymin];
                const T sum[5] = {-(x0.dt * tl0 + x1.dt * tl1), x0.db * tl0 + x1.db * tl1, -(x0.v * gmin.r0 + x1.v * gmin.r1),
                                  x0.v * gmax.r0 + x1.v * gmax.r1, x0.v * tl0 + x1.v * tl1};
                add(sum);
            }
            RowPair<T> R[K + 1], Lt[K + 1];
            read_taps(G, er, R);
            read_taps(G, el, Lt);
#pragma unroll
            for (int k = 0; k < K; ++k) {
                T sum[5] = {T(0), T(0), T(0), T(0), T(0)};
                const RowPair<T> grA = R[k], gr = R[k + 1], gl = Lt[k], glA = Lt[k + 1];
                const T dr0 = grA.r0 - gr.r0, dl0 = gl.r0 - glA.r0;
                const T dr1 = grA.r1 - gr.r1, dl1 = gl.r1 - glA.r1;
                T w0 = gr.r0 - gl.r0, w1 = gr.r1 - gl.r1;
                if (EXACT) {
                    w0 += s.fyhi * dr0; w0 += s.fylo * dl0;
                    w1 += s.fyhi * dr1; w1 += s.fylo * dl1;
                }
                if (!QUADS && ln.shares(k)) { w0 = w1 = v0[k] = v1[k] = T(0); }
                sum[4] += v0[k] * w0;
                sum[1] += (b1[k] - bc[k]) * w0;
                sum[0] -= (t0[k] - ta[k]) * w0;
                sum[3] += v0[k] * dr0;
                sum[2] -= v0[k] * dl0;
                sum[4] += v1[k] * w1;
                sum[1] += (b2[k] - b1[k]) * w1;
                sum[0] -= (t1[k] - t0[k]) * w1;
                sum[3] += v1[k] * dr1;
                sum[2] -= v1[k] * dl1;
                add(sum);
            }
        }
        if (PREFETCH) {
            BOXCONV_PUBLISH_NARROW(FLIP ^ 1, lr + 2, m0, m1, tl0, tl1)
#pragma unroll
            for (int k = 0; k < K; ++k) {
                ta[k] = t1[k]; bc[k] = b2[k];
                t0[k] = n0[k]; t1[k] = n1[k]; b1[k] = n2[k]; b2[k] = n3[k];
            }
        }
        wave_lds_order();
        __builtin_amdgcn_sched_barrier(0);
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
#undef BOXCONV_PUBLISH_NARROW

    if (SNAP && ln.in && i0 < h)                     // the sum of the band
        store_row_quad<QUADS>(snap + (2 * a.snap_groups + band) * mpitch + ln.cl, Quad<T>{{colacc[0], colacc[1], colacc[2], colacc[3]}});
    block_accumulate5(total, a.acc + ((static_cast<int64_t>(a.plane0 + p) * a.F + f) * slots + slot) * 5, red, false);
}

// ---------------------------------------------------------------------------------------------
// FS waves share the filters: wave n takes n, n + FS, ...; their sums are added in that order.
template <class TG, int L, int FS, bool EXACT, bool QUADS>
__global__ void __launch_bounds__(64 * FS) __attribute__((amdgpu_waves_per_eu(2, 3)))
narrow_input_kernel(SampleArgs<float> a, FinalizeArgs<float> fin) {
    using Lane = NarrowLane<L>;
    constexpr int K = 4, S = Lane::S, PLANE = Lane::PLANE, RB = 8, RC = 4, PAIRS = RC / 2, STAGES = RB / RC, MORE = 6;
    constexpr int ROWS = 4 * K * PLANE;                      // elements of a wave's rows
    constexpr int SUMS = (RB * K + RB) * 64 / 2;             // the same memory holds a wave's sums at the end
    __shared__ __align__(16) RowPair<float> lds[FS][FS > 1 && SUMS > ROWS ? SUMS : ROWS];

    // rides along, a box or a few per wave: see grad_input_cols_kernel
    if (fin.acc != nullptr)
        for (int k = uniform(blockIdx.x * FS + (threadIdx.x >> 6)); k < fin.n; k += gridDim.x * FS)
            finalize_box(fin, a.prm, k, static_cast<int>(threadIdx.x & 63));
    unsigned vid = xcd_contiguous_id(a.per_xcd);
    if (vid >= a.total) return;                      // whole workgroup leaves together
    if (a.reverse) vid = static_cast<unsigned>(a.total) - 1u - vid;
    const unsigned items = a.nb;                     // workgroups per plane
    const int64_t p = vid / items;
    const int c_in = static_cast<int>(static_cast<unsigned>(a.plane0 + p) % static_cast<unsigned>(a.C));
    const int h = a.h, w = a.w;
    const Lane ln(threadIdx.x & 63, w);
    const int set = FS > 1 ? uniform(threadIdx.x >> 6) : 0;
    const int group = static_cast<int>(vid % items) * S + ln.seg;
    const int i0 = group * RB;
    const int64_t spitch = a.mpitch;
    const unsigned s_bytes = 4u * static_cast<unsigned>(a.mpitch);
    RowPair<float>(*rows)[PAIRS][K * PLANE] = reinterpret_cast<RowPair<float>(*)[PAIRS][K * PLANE]>(lds[set]);
    for (int e = threadIdx.x & 63; e < ROWS; e += 64) lds[set][e] = RowPair<float>{0.0f, 0.0f};
    unsigned place[QUADS ? 1 : K];
#pragma unroll
    for (int k = 0; k < (QUADS ? 1 : K); ++k) place[k] = ln.place(k);
    auto own = [&](RowPair<float>* row, int k) {
        return QUADS ? at_bytes(row + k * PLANE, place[0]) : at_bytes(row, place[QUADS ? 0 : k]);
    };

    const int srows = narrow_snapshot_rows(a);
    float E[RB][K], tail[RB];
#pragma unroll
    for (int r = 0; r < RB; ++r) {
        tail[r] = 0.0f;
#pragma unroll
        for (int k = 0; k < K; ++k) E[r][k] = 0.0f;
    }

    RawQuad<TG> top[RC], bot[RC];
    RawQuad<float> snap_t, snap_b, between[2];
    auto split_of = [&](int f, float& scale) {
        const BoxOfWorkgroup<float> bx = load_box(a.prm, c_in * a.F + f);
        BoxSplit<float> s = split_grad_input(bx.xmin, bx.xmax, bx.ymin, bx.ymax);
        s.xlo = uniform(s.xlo); s.xhi = uniform(s.xhi); s.ylo = uniform(s.ylo); s.yhi = uniform(s.yhi);
        scale = a.normalize ? inverse_extent(bx.xmin, bx.xmax, bx.ymin, bx.ymax, EXACT, true, true) : 1.0f;
        return s;
    };
    auto band_of = [&](int edge) { return max(clampi(i0 + edge, 0, h) - 1, 0) >> a.m_shift; };
    const unsigned g_bytes = static_cast<unsigned>(sizeof(TG)) * static_cast<unsigned>(w);
    auto request = [&](int f, const BoxSplit<float>& s, int chunk) {
        const TG* g = reinterpret_cast<const TG*>(a.grad_out) + (p * a.F + f) * static_cast<int64_t>(h) * w;
        // (rows outside the image: the nearest one, cleared when it is used)
        auto row = [&](int i) {
            return at_bytes(g, row_offset(confine(i, h - 1), g_bytes, static_cast<unsigned>(sizeof(TG)) * ln.cl));
        };
        if (chunk == 0) {
            const float* snaps = a.src + (p * a.F + f) * static_cast<int64_t>(srows) * spitch;
            auto snapshot = [&](int row) { return at_bytes(snaps, row_offset(row, s_bytes, 4u * ln.cl)); };
            auto at_edge = [&](int edge, int first) {
                const int r = i0 + edge;
                return snapshot(r <= 0 ? 0 : r >= h ? srows - 1 : first + min(group, a.snap_groups - 1));
            };
            snap_t.load<QUADS>(at_edge(s.xlo, 1));
            snap_b.load<QUADS>(at_edge(s.xhi, 1 + a.snap_groups));
            const int bt = band_of(s.xlo), bb = band_of(s.xhi), lo = min(bt, bb), hi = max(bt, bb);
#pragma unroll
            for (int n = 0; n < 2; ++n)
                between[n].load<QUADS>(snapshot(lo + n < hi ? 1 + 2 * a.snap_groups + lo + n : 0));
        }
#pragma unroll
        for (int r = 0; r < RC; ++r) {
            top[r].template load<QUADS>(row(i0 + chunk * RC + r + s.xlo - 1));
            bot[r].template load<QUADS>(row(i0 + chunk * RC + r + s.xhi));
        }
    };

    // what was loaded for a row outside the image becomes zeros (a branch: mostly no lane has one)
    auto outside = [&](int i, float (&v)[K]) {
        const bool in_image = static_cast<unsigned>(i) < static_cast<unsigned>(h);
        if (!__all(in_image)) {
#pragma unroll
            for (int k = 0; k < K; ++k) { v[k] = in_image ? v[k] : 0.0f; finish_here(v[k]); }
        }
    };

    float scale = 0.0f;
    BoxSplit<float> s{};
    if (set < a.F) {
        s = split_of(set, scale);
        request(set, s, 0);
    }
    wave_lds_order();

#pragma unroll 1
    for (int f = set; f < a.F; f += FS) {
        // the box's sum at the group's first row: snapshots, and the bands between them in double
        float core[K];
        {
            const int bt = band_of(s.xlo), bb = band_of(s.xhi), lo = min(bt, bb), hi = max(bt, bb);
            const float* snaps = a.src + (p * a.F + f) * static_cast<int64_t>(srows) * spitch;
            double sum[K];
#pragma unroll
            for (int k = 0; k < K; ++k) {
                sum[k] = 0.0;
#pragma unroll
                for (int n = 0; n < 2; ++n) sum[k] += static_cast<double>(between[n].get(k));
            }
#pragma unroll 1
            for (int b = lo + 2; b < hi; b += MORE) {        // (tall boxes; so many loads in flight together)
                RawQuad<float> q[MORE];
#pragma unroll
                for (int n = 0; n < MORE; ++n)
                    q[n].load<QUADS>(at_bytes(snaps, row_offset(b + n < hi ? 1 + 2 * a.snap_groups + b + n : 0, s_bytes, 4u * ln.cl)));
#pragma unroll
                for (int n = 0; n < MORE; ++n)
#pragma unroll
                    for (int k = 0; k < K; ++k) sum[k] += static_cast<double>(q[n].get(k));
            }
#pragma unroll
            for (int k = 0; k < K; ++k)
                core[k] = (snap_b.get(k) - snap_t.get(k)) + static_cast<float>(bb > bt ? sum[k] : -sum[k]);
        }
        const float wr = EXACT ? scale * (1.0f - s.fyhi) : scale, wra = scale * s.fyhi;
        const float wl = EXACT ? scale * (1.0f - s.fylo) : scale, wla = scale * s.fylo;
        // tail(q) as two ramps confined to [0, 1]: 1 up to the column in front of an edge, the border weight in it
        float tw[K];
        bool has_tail = false;
        const float upper = static_cast<float>(s.yhi - 1 - ln.c0), lower = static_cast<float>(s.ylo - 2 - ln.c0);
        const float in_upper = EXACT ? s.fyhi : 0.0f, in_lower = EXACT ? 1.0f - s.fylo : 1.0f;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const float t = __builtin_amdgcn_fmed3f((upper - k) + in_upper, 0.0f, 1.0f) -
                            __builtin_amdgcn_fmed3f((lower - k) + in_lower, 0.0f, 1.0f);
            tw[k] = ln.owns(k) ? t * scale : 0.0f;
            has_tail = has_tail || tw[k] != 0.0f;
        }
        has_tail = __any(has_tail) != 0;             // wave-uniform
        const TapRun er = ln.taps(s.yhi - 1), el = ln.taps(s.ylo - 2);
        const float fxhi = s.fxhi, fxlo = s.fxlo;
#pragma unroll
        for (int stage = 0; stage < STAGES; ++stage) {
            const int buf = stage & 1;
#pragma unroll
            for (int q = 0; q < PAIRS; ++q) {
                float v[2][K];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const int rc = 2 * q + e, r = stage * RC + rc;   // row of the chunk, of the group
                    float t[K], b[K];
#pragma unroll
                    for (int k = 0; k < K; ++k) { t[k] = top[rc].get(k); b[k] = bot[rc].get(k); }
                    outside(i0 + r + s.xlo - 1, t);
                    outside(i0 + r + s.xhi, b);
#pragma unroll
                    for (int k = 0; k < K; ++k) {
                        if (r > 0) core[k] -= t[k];
                        v[e][k] = core[k];
                        if (EXACT) {
                            v[e][k] += fxhi * b[k];
                            v[e][k] += fxlo * t[k];
                        }
                        core[k] += b[k];
                    }
                    if (has_tail) {
#pragma unroll
                        for (int k = 0; k < K; ++k) tail[r] += tw[k] * v[e][k];
                    }
                    finish_here(tail[r]);
                }
#pragma unroll
                for (int k = 0; k < K; ++k) *own(rows[buf][q], k) = RowPair<float>{v[0][k], v[1][k]};
            }
            __builtin_amdgcn_sched_barrier(0);
            if (stage < STAGES - 1) {
                request(f, s, stage + 1);
            } else if (f + FS < a.F) {
                s = split_of(f + FS, scale);
                request(f + FS, s, 0);
            }
            wave_lds_order();
#pragma unroll
            for (int q = 0; q < PAIRS; ++q) {
                RowPair<float> R[K + 1], Lt[K + 1];
                read_taps(rows[buf][q], er, R);
                read_taps(rows[buf][q], el, Lt);
                const int r = stage * RC + 2 * q;
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    E[r][k] += wr * R[k].r0;
                    E[r + 1][k] += wr * R[k].r1;
                    E[r][k] -= wl * Lt[k + 1].r0;
                    E[r + 1][k] -= wl * Lt[k + 1].r1;
                    if (EXACT) {
                        E[r][k] += wra * R[k + 1].r0;
                        E[r + 1][k] += wra * R[k + 1].r1;
                        E[r][k] -= wla * Lt[k].r0;
                        E[r + 1][k] -= wla * Lt[k].r1;
                    }
                    finish_here(E[r][k]);
                    finish_here(E[r + 1][k]);
                }
            }
        }
    }

    if constexpr (FS > 1) {
        wave_lds_order();
        float* mine = reinterpret_cast<float*>(lds[set]) + (threadIdx.x & 63);
        if (set > 0) {
#pragma unroll
            for (int r = 0; r < RB; ++r) {
#pragma unroll
                for (int k = 0; k < K; ++k) mine[(r * K + k) * 64] = E[r][k];
                mine[(RB * K + r) * 64] = tail[r];
            }
        }
        __syncthreads();
        if (set > 0) return;
#pragma unroll 1
        for (int n = 1; n < FS; ++n) {
            const float* part = reinterpret_cast<const float*>(lds[n]) + threadIdx.x;
#pragma unroll
            for (int r = 0; r < RB; ++r) {
#pragma unroll
                for (int k = 0; k < K; ++k) E[r][k] += part[(r * K + k) * 64];
                tail[r] += part[(RB * K + r) * 64];
            }
        }
    }

    TG* out = reinterpret_cast<TG*>(a.dst) + p * static_cast<int64_t>(h) * w + ln.c0;
    const int last = (threadIdx.x & 63) | (L - 1);   // the last lane of the row
#pragma unroll
    for (int r = 0; r < RB; ++r) {
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (!ln.owns(k)) E[r][k] = 0.0f;         // (the neighbour's columns count once, an idle lane's not at all)
#pragma unroll
        for (int k = 1; k < K; ++k) E[r][k] += E[r][k - 1];
        const float left = row_scan<L>(E[r][K - 1], ln.l) - E[r][K - 1];
        const float base = left + __shfl(row_scan<L>(tail[r], ln.l), last);
        const int i = i0 + r;
        if (ln.in && i < h) {
            Quad<TG> q;
#pragma unroll
            for (int k = 0; k < K; ++k) narrow(base + E[r][k], q.v[k]);
            TG* orow = out + static_cast<int64_t>(i) * w;
            if (a.vec_out && ln.twice == 0) {
                store_row_quad<QUADS>(orow, q);
            } else {
#pragma unroll
                for (int k = 0; k < K; ++k)
                    if (ln.owns(k)) orow[k] = q.v[k];
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

}  // namespace

template <class TG>
hipError_t narrow_sums_launch(const float* integ, const TG* grad_out, BoxParams<float> prm, double* acc, int slots,
                              float* snapshots, const StreamPlan& sp, const SnapshotPlan* plan, Dims d, bool exact,
                              hipStream_t stream) {
    SampleArgs<float> a = base_args(prm, d);
    a.src = integ; a.grad_out = reinterpret_cast<const float*>(grad_out); a.acc = acc; a.acc_slots = slots;
    a.dst = snapshots;
    a.mpitch = column_workspace_pitch(d.w);
    a.nb = sp.nb; a.R = sp.R;
    if (plan != nullptr) { a.snap_shift = plan->shift; a.snap_groups = plan->groups; a.snap_bands = sp.nb; }
    if (slots != sp.slots() || (plan == nullptr) != (snapshots == nullptr) || (plan != nullptr && sp.R % (1 << plan->shift) != 0)) return hipErrorInvalidValue;
    finish_args(a, d.planes * d.F * slots);
    const dim3 grid(static_cast<unsigned>(a.per_xcd * kXcds));
    const bool quads = d.w % 4 == 0;
#define LAUNCH_NS_SNAP(L, QUADS, SNAP)                                                                                  \
    if (exact) BOXCONV_LAUNCH("grad_output_stream", (narrow_sums_kernel<TG, L, true, QUADS, SNAP>), grid, dim3(64), 0, stream, a);   \
    else       BOXCONV_LAUNCH("grad_output_stream", (narrow_sums_kernel<TG, L, false, QUADS, SNAP>), grid, dim3(64), 0, stream, a)
#define LAUNCH_NS_QUADS(L, QUADS)                                                                                       \
    if (plan != nullptr) { LAUNCH_NS_SNAP(L, QUADS, true); } else { LAUNCH_NS_SNAP(L, QUADS, false); }
#define LAUNCH_NS(L)                                                                                                    \
    if (quads) { LAUNCH_NS_QUADS(L, true) } else { LAUNCH_NS_QUADS(L, false) }
    if (sp.lanes == 8)       { LAUNCH_NS(8) }
    else if (sp.lanes == 16) { LAUNCH_NS(16) }
    else if (sp.lanes == 32) { LAUNCH_NS(32) }
    else return hipErrorInvalidValue;
#undef LAUNCH_NS
#undef LAUNCH_NS_QUADS
#undef LAUNCH_NS_SNAP
    return hipGetLastError();
}

template <class TG>
hipError_t narrow_input_launch(const TG* grad_out, const float* snapshots, const SnapshotPlan& plan, const StreamPlan& sp,
                               BoxParams<float> prm, TG* grad_in, Dims d, bool normalize, bool exact, hipStream_t stream,
                               const ParamFinish<float>* finish, bool* finish_done) {
    if (finish_done != nullptr) *finish_done = false;
    SampleArgs<float> a = base_args(prm, d);
    a.src = snapshots; a.grad_out = reinterpret_cast<const float*>(grad_out);
    a.dst = reinterpret_cast<float*>(grad_in);
    a.normalize = normalize ? 1 : 0;
    a.reverse = switches().gi_reverse ? 1 : 0;
    a.vec_out = quads_aligned(grad_in, sizeof(TG), d.w) ? 1 : 0;
    a.mpitch = column_workspace_pitch(d.w);
    a.snap_shift = plan.shift; a.snap_groups = plan.groups; a.snap_bands = sp.nb;
    while ((1 << a.m_shift) < sp.R) ++a.m_shift;
    if (plan.shift != 3 || (1 << a.m_shift) != sp.R) return hipErrorInvalidValue;
    const int side = 64 / sp.lanes;
    a.nb = (plan.groups + side - 1) / side;
    finish_args(a, d.planes * a.nb);
    const dim3 grid(static_cast<unsigned>(a.per_xcd * kXcds));
    FinalizeArgs<float> fin{};
    const bool quads = d.w % 4 == 0;
    const int fs = narrow_filter_sets(a.total, d.F);
    if (finish != nullptr && finish->acc != nullptr && 4 * static_cast<int64_t>(grid.x) * fs >= finish->n_boxes) {
        fin = finalize_args(*finish);
        if (finish_done != nullptr) *finish_done = true;
    }
#define LAUNCH_NI_QUADS(L, FS, QUADS)                                                                                   \
    if (exact) BOXCONV_LAUNCH("grad_input_taps", (narrow_input_kernel<TG, L, FS, true, QUADS>), grid, dim3(64 * FS), 0, stream, a, fin);   \
    else       BOXCONV_LAUNCH("grad_input_taps", (narrow_input_kernel<TG, L, FS, false, QUADS>), grid, dim3(64 * FS), 0, stream, a, fin)
#define LAUNCH_NI_FS(L, FS)                                                                                             \
    if (quads) { LAUNCH_NI_QUADS(L, FS, true); } else { LAUNCH_NI_QUADS(L, FS, false); }
#define LAUNCH_NI(L)                                                                                                    \
    if (fs == 8)      { LAUNCH_NI_FS(L, 8) }                                                                            \
    else if (fs == 4) { LAUNCH_NI_FS(L, 4) }                                                                            \
    else if (fs == 2) { LAUNCH_NI_FS(L, 2) }                                                                            \
    else              { LAUNCH_NI_FS(L, 1) }
    if (sp.lanes == 8)       { LAUNCH_NI(8) }
    else if (sp.lanes == 16) { LAUNCH_NI(16) }
    else if (sp.lanes == 32) { LAUNCH_NI(32) }
    else return hipErrorInvalidValue;
#undef LAUNCH_NI
#undef LAUNCH_NI_FS
#undef LAUNCH_NI_QUADS
    return hipGetLastError();
}

template hipError_t narrow_sums_launch<BOXCONV_INST_TG>(const float*, const BOXCONV_INST_TG*, BoxParams<float>, double*, int,
                                                        float*, const StreamPlan&, const SnapshotPlan*, Dims, bool, hipStream_t);
template hipError_t narrow_input_launch<BOXCONV_INST_TG>(const BOXCONV_INST_TG*, const float*, const SnapshotPlan&,
                                                         const StreamPlan&, BoxParams<float>, BOXCONV_INST_TG*, Dims, bool,
                                                         bool, hipStream_t, const ParamFinish<float>*, bool*);

}  // namespace boxconv
