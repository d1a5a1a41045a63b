// Host-side pieces of the box-sampling kernels that do not depend on the element type; the
// kernels themselves are templates in box_sampling_impl.hpp, instantiated by box_sampling_inst.hip.

#include <atomic>
#include <cmath>
#include <mutex>

#include "box_sampling_impl.hpp"   // stream_lds_bytes; the templates in it are not instantiated here

namespace boxconv {

namespace {

Switches read_switches() {
    auto text = [](const char* name) { return std::getenv(name); };
    auto flag_unless_zero = [&](const char* name) { const char* e = text(name); return e == nullptr || e[0] != '0'; };
    auto threads = [&](const char* name, int fallback) {
        const char* e = text(name);
        const int n = e ? std::atoi(e) : fallback;
        return (n == 256 || n == 512) ? n : fallback;
    };
    Switches s{};
    const char* e = text("BOXCONV_FORCE_GATHER");
    s.force_gather = e != nullptr && e[0] == '1';
    s.gi_reverse = flag_unless_zero("BOXCONV_GI_REVERSE");
    s.bwd_reverse = flag_unless_zero("BOXCONV_BWD_REVERSE");
    e = text("BOXCONV_GI_SPLIT_FILTERS");
    s.gi_split_filters = e == nullptr || std::atoi(e) != 0;
    e = text("BOXCONV_INTEGRAL_LOOKBACK");
    s.lookback = e == nullptr || std::atoi(e) != 0;
    s.lookback_any_shape = e != nullptr && std::atoi(e) == 2;
    e = text("BOXCONV_NARROW");
    s.narrow_rows = e == nullptr || e[0] != '0';
    s.narrow_any_size = e != nullptr && std::atoi(e) == 2;
    s.plane_integral = flag_unless_zero("BOXCONV_INTEGRAL_PLANE");
    e = text("BOXCONV_INTEGRAL_PLANE");
    s.plane_integral_tall = e == nullptr || (e[0] != '0' && e[0] != '1');
    s.stream_consecutive = flag_unless_zero("BOXCONV_STREAM_CONSEC");
    {
        const char* e = text("BOXCONV_STREAM_CONSEC");
        s.stream_consecutive_partial = e == nullptr || (e[0] != '0' && e[0] != '1');
        s.odd_rows_any_size = e != nullptr && e[0] == '3';
        s.stream_ragged = e == nullptr || s.odd_rows_any_size;
    }
    s.stream_narrow_double = flag_unless_zero("BOXCONV_STREAM_F64_NARROW");
    s.interleave_workspace = flag_unless_zero("BOXCONV_M_INTERLEAVE");
    s.forward_quads = flag_unless_zero("BOXCONV_FWD_QUADS");
    e = text("BOXCONV_FWD_QUADS");
    s.odd_forward_quads = e == nullptr || std::atoi(e) != 1;
    s.quads_any_size = e != nullptr && std::atoi(e) == 2;
    s.input_from_snapshots = flag_unless_zero("BOXCONV_GI_SNAPSHOTS");
    e = text("BOXCONV_GI_SNAPSHOTS");
    s.snapshots_any_shape = e != nullptr && std::atoi(e) == 2;
    e = text("BOXCONV_STREAM_WGS");
    s.stream_workgroups = e != nullptr ? std::max(1, std::atoi(e)) : 2048;
    e = text("BOXCONV_INTEGRAL_SPIN");
    s.spin_limit = e != nullptr ? std::max(0, std::atoi(e)) : 64;
    s.fwd_threads = threads("BOXCONV_FWD_THREADS", 512);
    s.stream_threads = threads("BOXCONV_STREAM_THREADS", 256);
    e = text("BOXCONV_L_KEEP_MB");
    s.keep_tail_bytes = static_cast<int64_t>(e != nullptr ? std::max(0, std::atoi(e)) : 192) << 20;
    return s;
}

std::mutex g_switch_mutex;
std::atomic<bool> g_switches_read{false};
Switches g_switches;

constexpr int kLdsDevices = 64;
std::atomic<int64_t> g_lds_limit[kLdsDevices];     // 0 = not looked up yet, -1 = query failed

}  // namespace

const Switches& switches() {
    if (!g_switches_read.load(std::memory_order_acquire)) {
        std::lock_guard<std::mutex> lock(g_switch_mutex);
        if (!g_switches_read.load(std::memory_order_relaxed)) {
            g_switches = read_switches();
            g_switches_read.store(true, std::memory_order_release);
        }
    }
    return g_switches;
}

void reload_switches() {
    std::lock_guard<std::mutex> lock(g_switch_mutex);
    g_switches = read_switches();
    g_switches_read.store(true, std::memory_order_release);
}

size_t device_lds_limit() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kLdsDevices) return 0;
    int64_t v = g_lds_limit[dev].load(std::memory_order_relaxed);
    if (v == 0) {
        int bytes = 0;
        v = hipDeviceGetAttribute(&bytes, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) == hipSuccess && bytes > 0
                ? bytes : -1;
        g_lds_limit[dev].store(v, std::memory_order_relaxed);
    }
    return v > 0 ? static_cast<size_t>(v) : 0;
}

namespace {

__global__ void fill_zero_kernel(double* __restrict__ p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0;
}

}  // namespace

hipError_t grad_params_begin(double* acc, int n_boxes, hipStream_t stream) {
    if (n_boxes == 0) return hipSuccess;
    BOXCONV_LAUNCH("fill_zero", fill_zero_kernel, dim3((n_boxes * 5 + 255) / 256), dim3(256), 0,
                   stream, acc, n_boxes * 5);
    return hipGetLastError();
}

namespace {

// Several bands side by side in a wave: rows per band (a power of two of at least a group, so that groups
// of rows start with bands) for the least rounds of waves times row pairs of a band and what it takes to
// start and end one, about three pairs. A launch is short of waves or, with bands that end
// in the middle of a wave, wastes them: 671 x 37 planes of 72 x 107, the sums, bands of 16, 32 and 64
// rows 247, 298 and 295 us; 512 x 4 of 64 x 128 22, 19 and 29. No more bands than a box's column
// sums are quickly added up from (78 x 19 of 928 x 32, both kernels 156, 124 and 107).
struct NarrowBands {
    int lanes, R, nb;       // lanes == 0: none
    double used;            // how much of what the waves hold are the plane's rows
};
NarrowBands narrow_bands(int64_t planes_f, int h, int w) {
    NarrowBands b{};
    const int lanes = w <= 32 ? 8 : w <= 64 ? 16 : 32, side = 64 / lanes;
    double best = 0.0;
    for (int R = 128; R >= 8; R /= 2) {
        const int nb = (h + R - 1) / R, slots = (nb + side - 1) / side;
        const double waves = static_cast<double>(planes_f) * slots, rounds = waves / (256 * 12);
        const double cost = (rounds < 4 ? std::ceil(rounds) : rounds) * (std::min(R, h) / 2 + 3);
        // (rows that the kernel with one row per wave takes, too: no more waves than that one may launch)
        if (consecutive_rows(w) && planes_f * slots > std::max<int64_t>(2 * switches().stream_workgroups, planes_f)) break;
        if (b.lanes > 0 && (cost >= best || nb > 40)) continue;
        best = cost;
        b = {lanes, R, nb, static_cast<double>(h) / (static_cast<double>(slots) * side * R)};
    }
    return b;
}

}  // namespace

StreamPlan plan_grad_output_stream(int64_t planes, int F, int h, int w, size_t elem_size, bool sums_only) {
    const int64_t planes_f = planes * F;
    StreamPlan sp{};
    const RowConfig rc = stream_row_config(std::max(w, 1), elem_size);
    sp.usable = row_kernels_apply(h, w, elem_size) &&
                stream_lds_bytes(rc.K, rc.nt, elem_size) <= kMaxDynamicLds;
    int nb = bands_for(std::max<int64_t>(planes_f, 1), h, 32, switches().stream_workgroups);
    // Parameter sums of rows that one wave covers at four columns per lane: four such workgroups
    // fit every SIMD and the band's chain of row pairs is what they wait for, so up to twice as many,
    // but no more than fit (256 x 4 planes of 128 x 256 in bfloat16, bands of 64 -> 32 rows: 40 -> 30 us,
    // and 28 -> 29 in the grad-input pass, which adds up more bands; but 416 planes of 661 x 204,
    // parameter sums alone, 77 us with 5 bands, 80 with 9, 91 with 10, which are 4160 workgroups). Wider
    // rows lose there what they gain (512 x 1024: 136 -> 133 and 129 -> 138 us), and so does the pass
    // that also leaves the column workspace (64 x 8 planes of 200 x 252, both kernels: 70 -> 82 us).
    if (sums_only && elem_size == 4 && consecutive_rows(w) && consecutive_threads(w) == 64)
        nb = std::max(nb, static_cast<int>(std::min<int64_t>(2 * switches().stream_workgroups / std::max<int64_t>(planes_f, 1),
                                                             std::max(1, h / 32))));
    // Rows of five, six and seven waves: a CU holds two such workgroups, a third would need its SIMDs to be
    // shared more evenly than they are, so as many bands as make one round of two per CU, where that
    // many come to 7/8 of it at least. Both backward kernels with snapshots / the sums alone: 16 x 8 planes of
    // 720 x 1280 313 -> 270 / 151 -> 118 us, 8 x 8 of 900 x 1792 260 -> 223 / 114 -> 100, 32 x 4 of 400 x 1200
    // 195 -> 172 / 89 -> 68; at 0.78 of it 0.94 to 1.02 of the time, and one band per plane, which cannot be cut
    // to fit, 1.0 to 1.24. Four waves are worse off (16 x 8 of 512 x 1024 265 -> 287), as are eight
    // (1024 x 2048 1455 -> 1615). Bands get up to h / 2 rows long by this; what the snapshots' float column sums would lose over
    // so many rows, kSumRows (box_sampling_impl.hpp) keeps.
    const int waves = consecutive_threads(w) / 64;
    if (sums_only && elem_size == 4 && consecutive_rows(w) && waves >= 5 && waves <= 7) {
        const int64_t one_round = switches().stream_workgroups / 4;
        const int64_t bands = std::min<int64_t>(one_round / std::max<int64_t>(planes_f, 1), h / 32);
        if (bands >= 2 && bands * planes_f * 8 >= one_round * 7) nb = static_cast<int>(bands);
    }
    int R = (h + nb - 1) / nb;
    R += R & 1;                                        // rows are handled in pairs
    sp.R = std::max(R, 2);
    sp.nb = (h + sp.R - 1) / sp.R;
    sp.parts = (rc.nt == 1024 || stream_double_wide_split(w, elem_size)) ? 2 : 1;
    if (sp.usable && sums_only && elem_size == 4 && narrow_rows_pay(planes, F, h, w)) {
        const NarrowBands b = narrow_bands(planes_f, h, w);
        sp.lanes = b.lanes; sp.R = b.R; sp.nb = b.nb;
    }
    return sp;
}

namespace {

// grad_input_taps_kernel walks through a plane's filters one after the other, 1.5 to 2.5 us each
// however few the planes are, where grad_input_cols_kernel spreads filters and rows over more waves.
// Both backward kernels together were timed against the column workspace on 5600 shapes (1 to 512
// planes, 1 to 40 filters, 16 to 1100 rows, 96 to 2048 columns, float32 and bfloat16):
//  * input pixels over filters (eight at most): below 2^17.5 the chain is all there is (8 planes of
//    17 x 100 with 40 filters 22 us by the workspace, 104 by snapshots; 1 of 96 x 256 with 8, 23
//    against 35; 16 of 200 x 252 with 8, 36 against 44), above it the workspace's bytes count
//    (8 of 300 x 700 with 16 filters, 101 against 83);
//  * fewer than 24 rows leave too much of a group's 8 rows empty (86 of 17 x 1212 with 8: 62 against 83);
//  * a last round of workgroups that is nearly empty costs what the workspace does while rounds times
//    filters is small (15 of 552 x 1124 with one filter 46 against 63, 479 of 69 x 100 with two 37
//    against 46, 99 of 186 x 96 with four 40 against 50): one round, or four over all filters.
// By this rule 2.5 % of the shapes are more than 3 % slower than by the workspace; without it 44 % were.
// Rows that are no multiple of four columns were timed on 2300 shapes against the workspace of
// grad_output_stream_kernel (0.70 to 0.85 of its time from 2^24 output pixels on, 0.88 to 1.0 below); in addition
//  * fewer than 40 rows (487 x 4 planes of 33 x 151 47 against 56 us, 90 x 8 of 34 x 506 46 against 54), or
//    up to 192 columns and fewer than 2^24 output pixels (5 x 4 of 1055 x 171 45 against 51), are up to 1.2;
//  * three waves whose last one has a single lane in use (513 to 515 columns, 1754 shapes) against the workspace, written
//    by the same kernel: 0.95 of the time below 2^22 output pixels, 0.97 (up to 1.13, one shape in four more than 3 %
//    slower: 53 x 10 planes of 55 x 514 68 against 77 us) from there to 2^25, 0.90 above (16 x 8 of 512 x 514 130 -> 114 us).
//    Of more waves the lane costs less than the workspace does (16 x 8 planes of 512 x 1025 321 -> 183 us, of
//    720 x 1281 466 -> 291).
bool wide_snapshots_pay(int64_t planes, int F, int h, int w) {
    if (!consecutive_rows(w)) return false;
    if (switches().snapshots_any_shape) return true;
    const int64_t pixels = planes * h * w;
    if (h < 24 || pixels < 180000 * static_cast<int64_t>(std::min(F, 8))) return false;
    // resident: three waves per SIMD, ten workgroups of one wave by their LDS. Of two workgroups of five or
    // six waves on a CU the second slows the first by as much as it brings: they count as two rounds
    const int waves = consecutive_threads(w) / 64;
    if (w % 4 != 0 && (h < 40 || (w <= 192 && pixels * F < (1 << 24)) ||
                       (waves == 3 && (w + 3) / 4 % 64 == 1 && pixels * F >= (1 << 22) && pixels * F < (1 << 25)))) return false;
    const int64_t workgroups = planes * ((h + 7) / 8), resident = 256 * (waves == 1 ? 10 : 12 / waves);
    return workgroups <= (waves > 4 ? 256 : resident) || workgroups * F >= 4 * resident;
}

}  // namespace

// Rows of at most 128 columns: the kernels that put several of them side by side in a wave (narrow_rows.hip)
// against those for wider rows (column workspace, or snapshots where wide_snapshots_pay), timed on 31000 shapes (1 to 2048
// planes, 1 to 40 filters, 16 to 1100 rows; float32 and bfloat16 with both gradients, float32 with the parameter sums
// alone): by this rule 0.66, 0.68 and 0.63 of the time in the geometric mean, 44 of the 11800 shapes it takes (and none
// of the 6500 with 96 to 124 columns in a multiple of four) more than 3 % slower, up to 1.14 (293 x 27 planes of
// 37 x 45 77 -> 87 us). Left to the others:
//  * fewer than 28 rows (nine shapes in ten of 16 to 23 rows 0.73 to 1.30 of the time, of 24 to 27 rows 0.64 to 1.12;
//    51 x 23 planes of 20 x 36 20.7 against 26.8 us);
//  * bands that leave nearly half of the waves' lanes without rows (0.61 to 1.09; 185 x 12 planes of 33 x 110, the
//    sums, 22.7 against 27.7 us); for 96 to 124 columns in a multiple of four, of which the kernels for wider rows
//    leave few lanes idle, a quarter (0.65 to 1.08; 554 x 3 of 135 x 96, the sums, 48.7 against 58.9);
//  * fewer than 2^17 output pixels, where a step is bound by its launches, and few input pixels for the filters, which
//    waves visit one after the other (25 planes of 24 x 16 with 40 filters 22 against 32 us; 32 of 28 x 28 26 against 30);
//  * tall planes that give too few waves: their bands are cut short, and a box spans many of them (15 x 4
//    planes of 1086 x 23 30 against 37 us; the sums alone of 4 x 8 of 754 x 90 13.3 against 17.0).
bool narrow_rows_pay(int64_t planes, int F, int h, int w) {
    const Switches& sw = switches();
    if (!sw.narrow_rows || !sw.input_from_snapshots || F < 1 || w < 16 || w > 128 || h < 8 || h >= (1 << 22)) return false;
    if (sw.narrow_any_size) return true;
    if (sw.snapshots_any_shape) return false;
    const int64_t pixels = planes * h * w;
    return h >= 28 && pixels >= 3000 * static_cast<int64_t>(F) && pixels * F >= (h <= 400 ? 1 << 17 : 1 << 22) &&
           narrow_bands(planes * F, h, w).used >= (w % 4 == 0 && w >= 96 && w < 128 ? 0.75 : 0.55);
}

// Output and integral images together; the memory-side cache holds 256 MB.
static int64_t forward_bytes(int64_t planes, int F, int h, int w, size_t elem_size) {
    return planes * (static_cast<int64_t>(F) * h * w * static_cast<int64_t>(elem_size) + static_cast<int64_t>(h + 1) * (w + 1) * 4);
}
static bool beyond_memory_side_cache(int64_t planes, int F, int h, int w, size_t elem_size) {
    return forward_bytes(planes, F, h, w, elem_size) >= (256ll << 20);
}

// Forward of rows of at most 128 columns with several of them side by side in a wave (narrow_forward.hip)
// against forward_rows_kernel, timed on 7400 shapes (float32; bfloat16 with and without the tail and a residual): 0.71,
// 0.68 and 0.70 of the time in the geometric mean, 3 shapes more than 3 % slower. Not for float32 rows of more
// than 32 columns without a tail that the memory-side cache does not hold (0.9 to 1.8).
// 96 to 124 columns in a multiple of four, against whichever of forward_rows_kernel and forward_quads_kernel
// one_wave_quads_pay has them, on 13000 shapes: 16-bit outputs 0.75 to 0.79 (4 of 6800 more than 3 % slower);
// float32 without a tail 0.78 (2 of 2044) up to 256 MB, 0.73 to 1.7 beyond; with a tail 0.80, with a residual,
// too, 0.83 (24 of 1856, up to 1.15) up to 128 MB, 0.57 to 1.5 beyond.
bool narrow_forward_pays(int64_t planes, int F, int h, int w, size_t elem_size, bool tail) {
    const Switches& sw = switches();
    if (!sw.forward_quads || !sw.narrow_rows || w < 16 || w > 128 || h >= (1 << 22)) return false;
    if (sw.narrow_any_size) return true;
    if (sw.quads_any_size) return false;
    if (w <= 32 || elem_size == 2) return true;
    if (w >= 96 && w < 128 && w % 4 == 0 && tail) return forward_bytes(planes, F, h, w, elem_size) < (128ll << 20);
    return tail || !beyond_memory_side_cache(planes, F, h, w, elem_size);
}

// forward_quads_kernel on rows that are no multiple of four columns, against forward_rows_kernel, timed on 9900
// shapes: with a tail 0.83 of the time (0.56 to 1.09); without one, by this rule, 0.95 in float32 and 0.92 in bfloat16
// (0.68 to 1.09). Left out: three or four columns per lane of one or two waves, which idle less in the other kernel
// (129 to 191 columns 1.06 to 1.11 from 2^20 output pixels on, 257 to 384 columns 1.01 to 1.06 from 2^22), 769 to
// 1024 columns below 2^20 (1.03), and float32 rows of more than 256 columns that the memory-side cache does not hold:
// 6500 of these 0.55 to 1.6, without a bound that parts them but the filters, which share a plane's integral rows; from
// 16 of them and 100 rows on 0.78 (5 of 844 shapes more than 3 % slower, up to 1.11; 64 planes of 270 x 481 with 16
// filters 189 -> 136 us), below that 1.04.
bool odd_forward_quads_pay(int64_t planes, int F, int h, int w, size_t elem_size, bool tail) {
    const Switches& sw = switches();
    if (!sw.forward_quads || !sw.odd_forward_quads || w % 4 == 0 || w <= 128 || w > 2048) return false;
    if (sw.quads_any_size || tail) return true;
    const int64_t pixels = planes * F * h * w;
    if (elem_size == 4 && beyond_memory_side_cache(planes, F, h, w, elem_size)) return w <= 256 || (F >= 16 && h >= 100);
    if (w < 192) return pixels < (1 << 20);
    if (w > 256 && w <= 384) return pixels < (1 << 22);
    return w <= 768 || w > 1024 || pixels >= (1 << 20);
}

int narrow_filter_sets(int64_t workgroups, int F) {
    int sets = 1;
    while (sets < 8 && 2 * sets <= F && workgroups * sets < 2048) sets *= 2;
    return sets;
}

bool snapshots_pay(int64_t planes, int F, int h, int w) {
    if (narrow_rows_pay(planes, F, h, w)) return true;
    return switches().input_from_snapshots && F >= 1 && wide_snapshots_pay(planes, F, h, w);
}

}  // namespace boxconv
