// Gradient w.r.t. the input formed from grad_output itself, for the rows that
// grad_output_stream_consec_kernel covers (replaces the same reference code as
// grad_input_cols_kernel: src/box_convolution.cpp:286-456 and tmpArray.sum(2),
// src/box_convolution_interface.cpp:274). Compiled once per element type of grad_output
// (BOXCONV_INST_TG).
//
// Per filter grad_input is grad_output box-filtered with the mirrored box. With s the split of that
// box, g(i) row i of one filter's grad_output (0 outside the image) and P(r) the sum of the rows
// above row r (r clamped to [0, h]):
//   vertical    VB(i) = core(i) + fxhi*g(i+xhi) + fxlo*g(i+xlo-1),
//               core(i) = P(i+xhi) - P(i+xlo),  core(i+1) = core(i) + g(i+xhi) - g(i+xlo);
//   horizontal  T(c)  = (1-fyhi)*VB[c+yhi-1] + fyhi*VB[c+yhi] - (1-fylo)*VB[c+ylo-1] - fylo*VB[c+ylo-2],
//               H(c)  = H(-1) + T(0) + ... + T(c),   H(-1) = sum_q VB[q]*tail(q),
//               tail(q) = [q < yhi-1] - [q < ylo-1] + fyhi*[q == yhi-1] + fylo*[q == ylo-2].
// Both T and H(-1) are linear in VB, so the filters are added up before the prefix sum along the
// row: one prefix sum per row of grad_input instead of one per row and filter.
//
// A workgroup owns RB output rows at full width, a lane 4 consecutive columns. Per filter a lane
// loads RB rows at either edge of the box, slides core down them, leaves VB in LDS (two rows side by
// side per column, as the other row kernels do) and adds its columns' taps to the sums in registers;
// the next filter's rows are requested before the barrier in the middle. core of the group's first
// row comes from the preceding pass over grad_output (StreamMode kStreamSnapshots), which leaves
// P at exactly the rows i0+xlo and i0+xhi of every group's first row i0, relative to its band, and
// the sum of each band.
//
// It replaces the column workspace, which is written whole and read twice (grad_input_cols_kernel),
// by a second read of grad_output and snapshots of 1/4 or 1/8 of that size (two rows per group of 8 or 16
// output rows) and one row per band. Both backward kernels together, 16 x 8 planes: 512 x 1024 x 2 346 ->
// 266 us, 720 x 1280 357 -> 304 us (270 with its sums in one round of workgroups); 32 x 4 planes of 128 x 256 x 4 44 -> 41 us (x 8 in bfloat16 79 -> 57); 128 x 2
// planes of 1024 x 2048 1632 -> 1520 us. Not every launch gains: snapshots_pay (box_sampling.hip).
// Bound (512 x 1024, 131 us): latency and issue at 6.6 resident waves per CU; the vector ALU issues a third
// of the time, the LDS pipe is busy for 15 % of it with no bank conflicts; 578 MB are fetched for 537 MB of
// grad_output and 54 of snapshots, so its second read hits the L2 for the most part (at 1024 x 2048, with
// planes of 8 MB, 2.5 GB for 2.1).
// Groups of 16 rows where that leaves two waves per SIMD, else of 8: against 8 rows, 16 take 132 against
// 137 us at 512 x 1024, 159 against 191 at 720 x 1280, 687 against 774 at 1024 x 2048 (half the
// snapshots), but 25 against 19 us at 128 planes of 128 x 256, where they leave half of the SIMDs idle.

#include "box_sampling_impl.hpp"

namespace boxconv {

namespace {

// Rows are read through a base that is the same for the whole wave.
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// A sum that is next needed in another basic block is computed there if the compiler may choose,
// and its operands (here: what was read from LDS) stay in registers until then. This keeps it where
// it is written; no instruction.
__device__ __forceinline__ void finish_here(float& v) { asm volatile("" : "+v"(v)); }

template <class TG, bool ALIGNED>
struct GradQuad;
template <bool ALIGNED>
struct GradQuad<float, ALIGNED> {
    typedef float f4 __attribute__((ext_vector_type(4)));
    f4 q;
    __device__ __forceinline__ void load(const float* p) {
        if constexpr (ALIGNED) q = *reinterpret_cast<const f4*>(p);
        else q = *reinterpret_cast<const f4_dword_aligned*>(p);
    }
    __device__ __forceinline__ float get(int v) const { return q[v]; }
};
template <class H, bool ALIGNED>
struct GradQuadHalf {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    typedef unsigned u2_at_any_half __attribute__((ext_vector_type(2), aligned(2)));
    u2 q;
    __device__ __forceinline__ void load(const H* p) {
        if constexpr (ALIGNED) q = *reinterpret_cast<const u2*>(p);
        else q = *reinterpret_cast<const u2_at_any_half*>(p);
    }
    __device__ __forceinline__ float get(int v) const {
        const unsigned word = v < 2 ? q.x : q.y;
        return widen(H{static_cast<unsigned short>((v & 1) ? word >> 16 : word & 0xffffu)});
    }
};
template <bool ALIGNED> struct GradQuad<f16_t, ALIGNED> : GradQuadHalf<f16_t, ALIGNED> {};
template <bool ALIGNED> struct GradQuad<bf16_t, ALIGNED> : GradQuadHalf<bf16_t, ALIGNED> {};

template <class TG, int NT, int RB, bool EXACT, int FIT>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2, RB == 8 ? 3 : 2)))
grad_input_taps_kernel(SampleArgs<float> a, FinalizeArgs<float> fin) {
    constexpr int K = 4, PLANE = quad_plane(NT), WAVES = NT / 64;
    constexpr int RC = 4, PAIRS = RC / 2;                    // rows (row pairs) in flight and in LDS at a time
    constexpr int STAGES = RB / RC;
    static_assert(STAGES % 2 == 0, "two LDS buffers in turn");
    struct alignas(8) WaveSums { float tot, tail; };
    __shared__ __align__(16) RowPair<float> rows[2][PAIRS][K][PLANE];
    __shared__ WaveSums wsum[WAVES][RB];

    if (fin.acc != nullptr && blockIdx.x < static_cast<unsigned>(fin.n) && threadIdx.x < 64)
        finalize_box(fin, a.prm, static_cast<int>(blockIdx.x), static_cast<int>(threadIdx.x));
    unsigned vid = xcd_contiguous_id(a.per_xcd);
    if (vid >= a.total) return;                      // whole workgroup leaves together
    if (a.reverse) vid = static_cast<unsigned>(a.total) - 1u - vid;
    const unsigned groups = a.snap_groups;
    const int group = static_cast<int>(vid % groups);
    const int64_t p = vid / groups;
    const int c_in = static_cast<int>(static_cast<unsigned>(a.plane0 + p) % static_cast<unsigned>(a.C));
    const int h = a.h, w = a.w, tid = threadIdx.x, lane = tid & 63;
    const int wave = uniform(tid >> 6);
    const int i0 = group * RB;
    const RowLane<NT, FIT> ln(tid, w);
    const int c0 = ln.c0, cl = ln.cl;
    const bool lane_in = ln.in;
    const int64_t spitch = a.mpitch;                 // of the snapshots

    for (int e = tid; e < 2 * PAIRS * K * 2 * kQuadPad; e += NT) {
        const int plane = e / (2 * kQuadPad), n = e % (2 * kQuadPad);
        (&rows[0][0][0][0])[plane * PLANE + (n < kQuadPad ? n : NT + n)] = RowPair<float>{0.0f, 0.0f};
    }
    ln.template clear_behind<PLANE, 2 * PAIRS>(&rows[0][0][0][0], w);
    const QuadPlace<PLANE, FIT> place(ln);

    const float* zeros = a.src;
    const int srows = snapshot_rows(a);
    float E[RB][K], tail[RB];
#pragma unroll
    for (int r = 0; r < RB; ++r) {
        tail[r] = 0.0f;
#pragma unroll
        for (int k = 0; k < K; ++k) E[r][k] = 0.0f;
    }
    bool wave_any_tail = false;

    // what is in flight for the coming filter
    GradQuad<TG, FIT != kRowAny> top[RC], bot[RC];
    GradQuad<float, FIT != kRowAny> snap_t, snap_b, between[2];
    auto split_of = [&](int f, float& scale) {
        const BoxOfWorkgroup<float> bx = load_box(a.prm, c_in * a.F + f);
        BoxSplit<float> s = split_grad_input(bx.xmin, bx.xmax, bx.ymin, bx.ymax);
        s.xlo = uniform(s.xlo); s.xhi = uniform(s.xhi); s.ylo = uniform(s.ylo); s.yhi = uniform(s.yhi);
        scale = a.normalize ? inverse_extent(bx.xmin, bx.xmax, bx.ymin, bx.ymax, EXACT, true, true) : 1.0f;
        return s;
    };
    auto band_of = [&](int edge) { return max(clampi(i0 + edge, 0, h) - 1, 0) / a.off_R; };
    auto request = [&](int f, const BoxSplit<float>& s, int chunk) {
        const TG* g = reinterpret_cast<const TG*>(a.grad_out) + (p * a.F + f) * static_cast<int64_t>(h) * w;
        const unsigned row_bytes = static_cast<unsigned>(w) * static_cast<unsigned>(sizeof(TG));
        auto row = [&](int i) {                      // (both addresses are formed: a select, no branch)
            const uintptr_t at = reinterpret_cast<uintptr_t>(at_bytes(g, static_cast<unsigned>(clampi(i, 0, h - 1)) * row_bytes));
            const uintptr_t none = reinterpret_cast<uintptr_t>(zeros);
            return reinterpret_cast<const TG*>(static_cast<unsigned>(i) < static_cast<unsigned>(h) ? at : none);
        };
        if (chunk == 0) {
            const float* snaps = a.src + spitch + (p * a.F + f) * static_cast<int64_t>(srows) * spitch;
            auto snapshot = [&](int edge, int first) {
                const int r = i0 + edge;
                const uintptr_t at = reinterpret_cast<uintptr_t>(snaps + static_cast<int64_t>(r >= h ? srows - 1 : first + group) * spitch);
                const uintptr_t none = reinterpret_cast<uintptr_t>(zeros);
                return reinterpret_cast<const float*>(r <= 0 ? none : at);
            };
            snap_t.load(snapshot(s.xlo, 0) + cl);
            snap_b.load(snapshot(s.xhi, a.snap_groups) + cl);
            const int bt = band_of(s.xlo), bb = band_of(s.xhi), lo = min(bt, bb), hi = max(bt, bb);
            const float* first = snaps + static_cast<int64_t>(2 * a.snap_groups + lo) * spitch;
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                const uintptr_t at = reinterpret_cast<uintptr_t>(first + n * spitch), none = reinterpret_cast<uintptr_t>(zeros);
                between[n].load(reinterpret_cast<const float*>(lo + n < hi ? at : none) + cl);
            }
        }
#pragma unroll
        for (int r = 0; r < RC; ++r) {
            top[r].load(row(i0 + chunk * RC + r + s.xlo - 1) + cl);
            bot[r].load(row(i0 + chunk * RC + r + s.xhi) + cl);
        }
    };

    float scale;
    BoxSplit<float> s = split_of(0, scale);
    request(0, s, 0);
    __syncthreads();                                 // pads are in place

#pragma unroll 1
    for (int f = 0; f < a.F; ++f) {
        // the box's sum at the group's first row: snapshots, and the bands between them in double
        float core[K];
        {
            const int bt = band_of(s.xlo), bb = band_of(s.xhi), lo = min(bt, bb), hi = max(bt, bb);
            const float* bands = a.src + spitch + ((p * a.F + f) * static_cast<int64_t>(srows) + 2 * a.snap_groups) * spitch + cl;
            double sum[K];
#pragma unroll
            for (int k = 0; k < K; ++k) {
                sum[k] = 0.0;
#pragma unroll
                for (int n = 0; n < 2; ++n) sum[k] += static_cast<double>(between[n].get(k));
            }
            for (int b = lo + 2; b < hi; ++b) {
                GradQuad<float, FIT != kRowAny> q;
                q.load(bands + static_cast<int64_t>(b) * spitch);
#pragma unroll
                for (int k = 0; k < K; ++k) sum[k] += static_cast<double>(q.get(k));
            }
#pragma unroll
            for (int k = 0; k < K; ++k)
                core[k] = (snap_b.get(k) - snap_t.get(k)) + static_cast<float>(bb > bt ? sum[k] : -sum[k]);
        }
        // weights of this filter: taps, and what H(-1) takes from the lane's columns
        const float wr = EXACT ? scale * (1.0f - s.fyhi) : scale, wra = scale * s.fyhi;
        const float wl = EXACT ? scale * (1.0f - s.fylo) : scale, wla = scale * s.fylo;
        float tw[K];
        bool has_tail = false;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int q = c0 + k;
            float t = static_cast<float>(q < s.yhi - 1) - static_cast<float>(q < s.ylo - 1);
            if (EXACT) {
                t += q == s.yhi - 1 ? s.fyhi : 0.0f;
                t += q == s.ylo - 2 ? s.fylo : 0.0f;
            }
            tw[k] = ln.owns(k) ? t * scale : 0.0f;
            has_tail = has_tail || tw[k] != 0.0f;
        }
        has_tail = __any(has_tail) != 0;             // wave-uniform
        wave_any_tail = wave_any_tail || has_tail;
        const TapRun er = lane_taps<PLANE>(ln, s.yhi - 1), el = lane_taps<PLANE>(ln, s.ylo - 2);
        const float fxhi = s.fxhi, fxlo = s.fxlo;
#pragma unroll
        for (int stage = 0; stage < STAGES; ++stage) {
            const int buf = stage & 1;
            if (lane_in) {
#pragma unroll
                for (int q = 0; q < PAIRS; ++q) {
                    float v[2][K];
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const int rc = 2 * q + e, r = stage * RC + rc;   // row of the chunk, of the group
#pragma unroll
                        for (int k = 0; k < K; ++k) {
                            if (r > 0) core[k] -= top[rc].get(k);
                            v[e][k] = core[k];
                            if (EXACT) {
                                v[e][k] += fxhi * bot[rc].get(k);
                                v[e][k] += fxlo * top[rc].get(k);
                            }
                            core[k] += bot[rc].get(k);
                        }
                        if (has_tail) {
#pragma unroll
                            for (int k = 0; k < K; ++k) tail[r] += tw[k] * v[e][k];
                        }
                        finish_here(tail[r]);
                    }
#pragma unroll
                    for (int k = 0; k < K; ++k) *place.at(rows[buf][q][0], k) = RowPair<float>{v[0][k], v[1][k]};
                }
            }
            __builtin_amdgcn_sched_barrier(0);       // (loads moved up past the stores above would spill)
            if (stage < STAGES - 1) {                // the registers of this chunk are free again
                request(f, s, stage + 1);
            } else if (f + 1 < a.F) {
                s = split_of(f + 1, scale);
                request(f + 1, s, 0);
            }
            __syncthreads();
#pragma unroll
            for (int q = 0; q < PAIRS; ++q) {
                RowPair<float> R[K + 1], L[K + 1];
                read_taps(rows[buf][q][0], er, R);
                read_taps(rows[buf][q][0], el, L);
                const int r = stage * RC + 2 * q;
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    E[r][k] += wr * R[k].r0;
                    E[r + 1][k] += wr * R[k].r1;
                    E[r][k] -= wl * L[k + 1].r0;
                    E[r + 1][k] -= wl * L[k + 1].r1;
                    if (EXACT) {
                        E[r][k] += wra * R[k + 1].r0;
                        E[r + 1][k] += wra * R[k + 1].r1;
                        E[r][k] -= wla * L[k].r0;
                        E[r + 1][k] -= wla * L[k].r1;
                    }
                    finish_here(E[r][k]);
                    finish_here(E[r + 1][k]);
                }
            }
        }
    }

    // prefix sums along the row: inside the lane, over the lanes to the left, over the waves
    float left[RB];
#pragma unroll
    for (int r = 0; r < RB; ++r) {
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (ln.shares(k)) E[r][k] = 0.0f;        // (the neighbour's columns count once)
#pragma unroll
        for (int k = 1; k < K; ++k) E[r][k] += E[r][k - 1];
        const float inc = wave_inclusive_scan(E[r][K - 1]);
        left[r] = inc - E[r][K - 1];
        const float t = wave_any_tail ? wave_sum_to_last(tail[r]) : 0.0f;
        if (lane == 63) wsum[wave][r] = WaveSums{inc, t};
        __builtin_amdgcn_sched_barrier(0);           // (all rows' scans at once would spill)
    }
    __syncthreads();
    if (!lane_in) return;
    TG* out = reinterpret_cast<TG*>(a.dst) + p * static_cast<int64_t>(h) * w + c0;
#pragma unroll
    for (int r = 0; r < RB; ++r) {
        const int i = i0 + r;
        if (i >= h) break;
        float base = 0.0f;
#pragma unroll
        for (int wv = 0; wv < WAVES; ++wv) {
            const WaveSums ws = wsum[wv][r];
            base += ws.tail;
            if (wv < wave) base += ws.tot;           // `wave` is scalar
        }
        base += left[r];
        Quad<TG> q;
#pragma unroll
        for (int k = 0; k < K; ++k) narrow(base + E[r][k], q.v[k]);
        TG* orow = out + static_cast<int64_t>(i) * w;
        if (a.vec_out && (FIT != kRowAny || ln.twice == 0)) {
            store_row_quad<FIT != kRowAny>(orow, q);
        } else {
#pragma unroll
            for (int k = 0; k < K; ++k)
                if (ln.owns(k)) orow[k] = q.v[k];
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

}  // namespace

template <class TG>
SnapshotPlan plan_snapshots(const TG* grad_out, const StreamPlan& sp, Dims d) {
    SnapshotPlan plan{};
    // 16 rows per group where that still makes two waves per SIMD (measured above)
    const int64_t waves16 = d.planes * ((d.h + 15) / 16) * (consecutive_threads(d.w) / 64);
    plan.shift = waves16 >= 2048 && sp.lanes == 0 ? 4 : 3;
    plan.groups = (d.h + (1 << plan.shift) - 1) >> plan.shift;
    // (the last condition: the snapshots fit where the column workspace would be)
    plan.use = snapshots_pay(d.planes, d.F, d.h, d.w) && sp.usable && sp.parts == 1 &&
               quads_aligned(grad_out, sizeof(TG), d.w) && 2 * plan.groups + sp.nb + 1 <= d.h + 1;
    return plan;
}

template <class TG>
hipError_t grad_input_taps_launch(const TG* grad_out, const float* snapshots, const SnapshotPlan& plan,
                                  const StreamPlan& sp, BoxParams<float> prm, TG* grad_in, Dims d,
                                  bool normalize, bool exact, hipStream_t stream,
                                  const ParamFinish<float>* finish, bool* finish_done) {
    if (finish_done != nullptr) *finish_done = false;
    if (d.planes == 0 || d.hw() == 0) return hipSuccess;
    if (sp.lanes > 0)
        return narrow_input_launch<TG>(grad_out, snapshots, plan, sp, prm, grad_in, d, normalize, exact, stream, finish, finish_done);
    SampleArgs<float> a = base_args(prm, d);
    a.src = snapshots; a.grad_out = reinterpret_cast<const float*>(grad_out);
    a.dst = reinterpret_cast<float*>(grad_in);
    a.normalize = normalize ? 1 : 0;
    a.off_R = sp.R;
    a.reverse = switches().gi_reverse ? 1 : 0;
    a.vec_out = quads_aligned(grad_in, sizeof(TG), d.w) ? 1 : 0;
    a.mpitch = column_workspace_pitch(d.w);
    a.snap_shift = plan.shift; a.snap_groups = plan.groups; a.snap_bands = sp.nb;
    finish_args(a, d.planes * plan.groups);
    const dim3 grid(static_cast<unsigned>(a.per_xcd * kXcds));
    FinalizeArgs<float> fin{};
    if (finish != nullptr && finish->acc != nullptr && grid.x >= static_cast<unsigned>(finish->n_boxes)) {
        fin = finalize_args(*finish);
        if (finish_done != nullptr) *finish_done = true;
    }
#define LAUNCH_GT_FIT(NT, RB, FIT)                                                                                    \
    if (exact) BOXCONV_LAUNCH("grad_input_taps", (grad_input_taps_kernel<TG, NT, RB, true, FIT>), grid, dim3(NT), 0, stream, a, fin);   \
    else       BOXCONV_LAUNCH("grad_input_taps", (grad_input_taps_kernel<TG, NT, RB, false, FIT>), grid, dim3(NT), 0, stream, a, fin)
#define LAUNCH_GT_RB(NT, RB)                                                                                          \
    if (d.w % 4 == 0) { LAUNCH_GT_FIT(NT, RB, kRowQuads); }                                                            \
    else              { LAUNCH_GT_FIT(NT, RB, kRowAny); }
#define LAUNCH_GT(NT)                                                                                               \
    case NT:                                                                                                        \
        if (plan.shift == 4) { LAUNCH_GT_RB(NT, 16) } else { LAUNCH_GT_RB(NT, 8) }                                   \
        break;
    switch (consecutive_threads(d.w)) {
        LAUNCH_GT(64)
        LAUNCH_GT(128)
        LAUNCH_GT(192)
        LAUNCH_GT(256)
        LAUNCH_GT(320)
        LAUNCH_GT(384)
        LAUNCH_GT(448)
        LAUNCH_GT(512)
        default: return hipErrorInvalidValue;
    }
#undef LAUNCH_GT
#undef LAUNCH_GT_RB
#undef LAUNCH_GT_FIT
    return hipGetLastError();
}

template SnapshotPlan plan_snapshots<BOXCONV_INST_TG>(const BOXCONV_INST_TG*, const StreamPlan&, Dims);
template hipError_t grad_input_taps_launch<BOXCONV_INST_TG>(const BOXCONV_INST_TG*, const float*, const SnapshotPlan&,
                                                            const StreamPlan&, BoxParams<float>, BOXCONV_INST_TG*,
                                                            Dims, bool, bool, hipStream_t, const ParamFinish<float>*,
                                                            bool*);

}  // namespace boxconv
