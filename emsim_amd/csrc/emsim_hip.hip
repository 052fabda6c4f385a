// C ABI of the gfx950 multislice backend (declarations: include/emsim_hip.h).
//
// Host side only: argument checks, float32 constants computed in the
// reference's operation order, constant-table uploads, and launches of the
// kernels in kernels_wave.hpp / kernels_slice.hpp on the caller's stream.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <exception>
#include <mutex>
#include <new>
#include <string>
#include <thread>
#include <vector>

#include "../../include/emsim_hip.h"
#include "host_common.hpp"
#include "fft_lds.hpp"
#include "kernels_slice.hpp"
#include "kernels_wave.hpp"
#include "kernels_fused.hpp"
#include "kernels_prep.hpp"
#include "kernels_dft.hpp"

#include <complex>

using namespace emsim;

namespace emsim_host {

thread_local std::string g_last_error;

int fail(int code, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_last_error = buf;
    return code;
}

// --------------------------------------------------------------------------
// launches: error check plus optional per-kernel event timing
// (emsim_hip_timing_enable / emsim_hip_timing_collect).  Events are recorded
// on the launch stream, immediately before and after the kernel.
// --------------------------------------------------------------------------
struct TimingRecord {
    const char* name;
    int n;
    hipEvent_t start, stop;
};
std::mutex g_timing_mutex;
bool g_timing_on = false;
std::vector<TimingRecord> g_timing_records;
std::vector<hipEvent_t> g_event_pool;

hipEvent_t pooled_event() {
    if (!g_event_pool.empty()) {
        hipEvent_t e = g_event_pool.back();
        g_event_pool.pop_back();
        return e;
    }
    hipEvent_t e = nullptr;
    if (hipEventCreate(&e) != hipSuccess) return nullptr;
    return e;
}

hipEvent_t timing_begin(hipStream_t s) {
    std::lock_guard<std::mutex> lock(g_timing_mutex);
    if (!g_timing_on) return nullptr;
    hipEvent_t e = pooled_event();
    if (e && hipEventRecord(e, s) != hipSuccess) {
        g_event_pool.push_back(e);
        return nullptr;
    }
    return e;
}

void timing_end(hipEvent_t start, const char* name, int n, hipStream_t s) {
    if (!start) return;
    std::lock_guard<std::mutex> lock(g_timing_mutex);
    hipEvent_t e = pooled_event();
    if (!e || hipEventRecord(e, s) != hipSuccess) {
        g_event_pool.push_back(start);
        if (e) g_event_pool.push_back(e);
        return;
    }
    g_timing_records.push_back({name, n, start, e});
}

}  // namespace emsim_host

using namespace emsim_host;

namespace {

// The reference's PI literal (WavePropagator.cpp:10) as float32.
constexpr float kPi32 = 3.14159265358979324f;

bool pow2_supported(int n) { return n >= 8 && n <= kTwN && (n & (n - 1)) == 0; }
// Lengths the chirp-z path takes: any n with a power-of-two convolution
// length 2n - 1 <= M <= kTwN.
constexpr int kChirpMaxN = kTwN / 2;
bool chirp_supported(int n) { return n >= 8 && n <= kChirpMaxN; }
bool size_supported(int n) { return pow2_supported(n) || chirp_supported(n); }

// --------------------------------------------------------------------------
// chirp-z plans (kernels_dft.hpp): c_m = exp(-i pi m^2 / n) and the transform
// of the circular chirp b, both computed in float64 on the host
// --------------------------------------------------------------------------
struct ChirpPlan {
    int n = 0, M = 0;
    float2* c = nullptr;   // (n) exp(-i pi m^2 / n)
    float2* b = nullptr;   // (M) FFT_M of conj(c) placed at m and M - m, / M
    ChirpTab tab() const { return ChirpTab{c, b, n}; }
};

// In-place iterative radix-2 FFT in float64, forward sign exp(-2 pi i j k / M).
void host_fft(std::vector<std::complex<double>>& a) {
    const size_t m = a.size();
    for (size_t i = 1, j = 0; i < m; ++i) {
        size_t bit = m >> 1;
        for (; j & bit; bit >>= 1) j ^= bit;
        j ^= bit;
        if (i < j) std::swap(a[i], a[j]);
    }
    const double two_pi = 6.283185307179586476925286766559;
    for (size_t len = 2; len <= m; len <<= 1) {
        for (size_t i = 0; i < m; i += len) {
            for (size_t k = 0; k < len / 2; ++k) {
                const double ang = -two_pi * (double)k / (double)len;
                const std::complex<double> w(std::cos(ang), std::sin(ang));
                const std::complex<double> u = a[i + k], v = a[i + k + len / 2] * w;
                a[i + k] = u + v;
                a[i + k + len / 2] = u - v;
            }
        }
    }
}

void chirp_plan_free(ChirpPlan& p) {
    for (float2** q : {&p.c, &p.b}) {
        if (*q) (void)hipFree(*q);
        *q = nullptr;
    }
}

int chirp_plan_create(int n, ChirpPlan& p) {
    int M = 1;
    while (M < 2 * n - 1) M <<= 1;
    if (M < 8) M = 8;
    if (M > kTwN) return fail(EMSIM_HIP_EUNSUPPORTED, "chirp-z length %d needs M = %d > %d", n, M, kTwN);
    p.n = n;
    p.M = M;
    const double pi = 3.14159265358979323846264338327950288;
    std::vector<std::complex<double>> c(n);
    for (int m = 0; m < n; ++m) {
        const long long q = ((long long)m * m) % (2LL * n);   // m^2 mod 2n: exact angle
        c[m] = std::polar(1.0, -pi * (double)q / (double)n);
    }
    std::vector<float2> hc(n), hb(M);
    for (int m = 0; m < n; ++m) hc[m] = make_float2((float)c[m].real(), (float)c[m].imag());
    // the convolution kernel: conj of the transform's chirp, circular
    std::vector<std::complex<double>> b(M, 0.0);
    for (int m = 0; m < n; ++m) {
        b[m] = std::conj(c[m]);
        if (m > 0) b[M - m] = b[m];
    }
    host_fft(b);
    const double inv_m = 1.0 / (double)M;   // exact: M is a power of two
    for (int k = 0; k < M; ++k)
        hb[k] = make_float2((float)(b[k].real() * inv_m), (float)(b[k].imag() * inv_m));
    hipError_t err = hipSuccess;
    const std::vector<float2>* src[2] = {&hc, &hb};
    float2** dst[2] = {&p.c, &p.b};
    for (int i = 0; i < 2 && err == hipSuccess; ++i) {
        err = hipMalloc(dst[i], src[i]->size() * sizeof(float2));
        if (err == hipSuccess)
            err = hipMemcpy(*dst[i], src[i]->data(), src[i]->size() * sizeof(float2),
                            hipMemcpyHostToDevice);
    }
    if (err != hipSuccess) {
        chirp_plan_free(p);
        return fail(EMSIM_HIP_EDEVICE, "chirp plan: %s", hipGetErrorString(err));
    }
    return EMSIM_HIP_OK;
}

// --------------------------------------------------------------------------
// per-device twiddle table w[m] = exp(-2 pi i m / 4096), float64 -> float32
// --------------------------------------------------------------------------
std::mutex g_tw_mutex;
std::vector<float2*> g_twiddles;

int get_twiddles(const float2** out) {
    int dev = 0;
    EMSIM_HIP_CHECK(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(g_tw_mutex);
    if ((int)g_twiddles.size() <= dev) g_twiddles.resize(dev + 1, nullptr);
    if (!g_twiddles[dev]) {
        std::vector<float2> host(kTwN);
        const double two_pi = 6.283185307179586476925286766559;
        for (int m = 0; m < kTwN; ++m) {
            const double a = -two_pi * (double)m / (double)kTwN;
            host[m] = make_float2((float)std::cos(a), (float)std::sin(a));
        }
        float2* d = nullptr;
        EMSIM_HIP_CHECK(hipMalloc(&d, kTwN * sizeof(float2)));
        hipError_t err = hipMemcpy(d, host.data(), kTwN * sizeof(float2), hipMemcpyHostToDevice);
        if (err != hipSuccess) {
            (void)hipFree(d);
            return fail(EMSIM_HIP_EDEVICE, "twiddle upload failed: %s", hipGetErrorString(err));
        }
        g_twiddles[dev] = d;
    }
    *out = g_twiddles[dev];
    return EMSIM_HIP_OK;
}

// --------------------------------------------------------------------------
// numpy.arange(start, stop, step) for float64, as the reference's binning
// calls it (slice_builder_base.py:183-186): length ceil((stop-start)/step),
// element 0 = start, element 1 = start + step, element i >= 2 =
// start + i * ((start + step) - start).
// --------------------------------------------------------------------------
void numpy_arange(double start, double stop, double step, std::vector<double>& out) {
    out.clear();
    const double len_f = std::ceil((stop - start) / step);
    if (!(len_f > 0)) return;
    const long len = (long)len_f;
    out.resize(len);
    out[0] = start;
    if (len == 1) return;
    const double next = start + step;
    out[1] = next;
    const double delta = next - start;
    for (long i = 2; i < len; ++i) out[i] = start + (double)i * delta;
}

void reference_edges(int n, double d, std::vector<double>& e64) {
    const double start = -d * (double)(n / 2);
    const double end = start + (double)n * d;
    numpy_arange(start, end + d, d, e64);
}

// Smallest float32 >= x.
float round_up_f32(double x) {
    float f = (float)x;
    if ((double)f < x) f = std::nextafter(f, INFINITY);
    return f;
}

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Row stride of the half-spectrum workspace: H = n2/2+1 rounded up to a
// multiple of 16 complex, so that column tiles start on 64-byte boundaries.
int half_ld(int H) { return (H + 15) & ~15; }

int grid_for(int64_t n, int block) {
    int64_t g = ceil_div(n, block);
    if (g < 1) g = 1;
    if (g > 65536) g = 65536;
    return (int)g;
}

}  // namespace

// ==========================================================================
// handles
// ==========================================================================
struct emsim_hip_slice_builder {
    int n_elems = 0, n_slices = 0, n1 = 0, n2 = 0, H = 0;
    double dz = 0, d1 = 0, d2 = 0;
    int one_slice = 0;
    float* sf = nullptr;        // (n_elems, n1, H)
    // the same, tile-major for the fused spectrum pass: (n_elems, tiles, n1,
    // C) with C = spec_tile_cols(n1) columns per tile, zeros beyond H
    float* sf_tiles = nullptr;
    float* edges = nullptr;     // axis0 (n0+1) | axis1 (n1+1) | axis2 (n2+1)
    int last_exact[3] = {0, 0, 0};
    float inv_d[3] = {0, 0, 0};
    int tile_rows = 1, tiles_per_plane = 1;
    const float2* tw = nullptr;
    // a lateral size that is not a power of two: chirp-z plans of both axes
    bool chirp = false;
    ChirpPlan p1, p2;
};

namespace {
// Rows of the fused path's Y also hold the spectrum kernel's per-element
// column-0 transforms in padding columns H .. H + n_elems - 1.
int fused_ld(const emsim_hip_slice_builder* b) { return half_ld(b->H + b->n_elems); }
}  // namespace

struct emsim_hip_wave_propagator {
    int n1 = 0, n2 = 0;
    float d1 = 0, d2 = 0, lam = 0, gamma = 0;
    float dfx = 0, dfy = 0, filter2 = 0, factor = 0;
    const float2* tw = nullptr;
    // a wave shape that is not a power of two: chirp-z plans of both axes
    bool chirp = false;
    ChirpPlan p1, p2;
};

// ==========================================================================
// size dispatch
// ==========================================================================
#define EMSIM_DISPATCH(n, FN, ...)                                                  \
    switch (n) {                                                                    \
        case 8: return FN<8>(__VA_ARGS__);                                          \
        case 16: return FN<16>(__VA_ARGS__);                                        \
        case 32: return FN<32>(__VA_ARGS__);                                        \
        case 64: return FN<64>(__VA_ARGS__);                                        \
        case 128: return FN<128>(__VA_ARGS__);                                      \
        case 256: return FN<256>(__VA_ARGS__);                                      \
        case 512: return FN<512>(__VA_ARGS__);                                      \
        case 1024: return FN<1024>(__VA_ARGS__);                                    \
        case 2048: return FN<2048>(__VA_ARGS__);                                    \
        case 4096: return FN<4096>(__VA_ARGS__);                                    \
        default: return fail(EMSIM_HIP_EUNSUPPORTED, "unsupported FFT length %d", n); \
    }

namespace {

// Launch-shape knobs (emsim_hip_tuning_set); 0 selects the built-in rule.
// They change how work is split over blocks, never the arithmetic.
int g_row_items_per_block = 0;   // row groups per row-worker block
int g_col_tiles_per_block = 0;   // column tiles per column-kernel block
int g_col_shape = 0;             // column-tile shape (ColCfg SHAPE) of the propagator pass

// Grid of the row worker for n_items rows (or row pairs) of length N.  With
// resident > 0 (blocks of this kernel the device holds at once), the fewest
// rows per block that still fit the grid in one round of resident blocks, so
// no partial second round trails the first; otherwise rows_per_block.
template <int N>
void row_grid(int64_t n_items, int& rpw, dim3& grid, int64_t resident = 0) {
    using Cfg = RowCfg<N>;
    const int64_t groups = ceil_div(n_items, Cfg::G);
    if (g_row_items_per_block > 0) {
        rpw = g_row_items_per_block;
    } else if (resident > 0) {
        const int64_t r = ceil_div(groups, resident);
        rpw = (int)(r < 1 ? 1 : (r > 16 ? 16 : r));
    } else {
        rpw = rows_per_block(groups);
    }
    grid = dim3((unsigned)ceil_div(groups, rpw));
}

// Blocks of kernel k (block size bs, no dynamic LDS) resident on the current
// device at once, from its occupancy and CU count; 0 if unknown.  Cached per
// device (a race between threads stores the same value).
template <class K>
int64_t resident_blocks(K k, int bs, int (&cache)[64]) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
    if (cache[dev] == 0) {
        int per_cu = 0, cus = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k, bs, 0) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return 0;
        cache[dev] = per_cu > 0 && cus > 0 ? per_cu * cus : -1;
    }
    return cache[dev] > 0 ? cache[dev] : 0;
}

template <int N>
int launch_row_fft(bool inv, const float2* in, float2* out, int64_t rows, const float2* tw,
                   hipStream_t s) {
    int rpw;
    dim3 grid;
    row_grid<N>(rows, rpw, grid);
    const dim3 block(RowCfg<N>::BLOCK);
    if (inv) EMSIM_LAUNCH(N, (k_row_fft<N, true>), grid, block, 0, s, OpFFT<N, true>{in, out}, rows, rpw, tw);
    else EMSIM_LAUNCH(N, (k_row_fft<N, false>), grid, block, 0, s, OpFFT<N, false>{in, out}, rows, rpw, tw);
    return EMSIM_HIP_OK;
}

// Wave columns [lo, hi] that the multiplier zeroes whole (none by default):
// pass B loads none of them, and with skip_tiles leaves out the column
// tiles that hold only such columns (their contents are then left as they
// are, for callers that never read them).
struct ColDead {
    int lo = 1 << 30, hi = -1;
    bool skip_tiles = false;
    // the mean's rounding rests, one per image, or null; first: none yet
    float2* carry = nullptr;
    bool carry_first = true;
};

template <int N>
int launch_row_transmit_fft(bool first, const float2* in, const float* V, float2* out,
                            int64_t rows, int rows_per_img, int64_t v_img_stride, float factor,
                            ColDead cd, const float2* tw, hipStream_t s) {
    static int resident_cache[64];
    const int64_t resident =
        resident_blocks(k_row_transmit_fft<N, false>, RowCfg<N>::BLOCK, resident_cache);
    int rpw;
    dim3 grid;
    row_grid<N>(rows, rpw, grid, resident);
    const dim3 block(RowCfg<N>::BLOCK);
    if (first)
        EMSIM_LAUNCH(N, (k_row_transmit_fft<N, true>), grid, block, 0, s,
                     (OpTransmit<N, true>{in, V, out, rows_per_img, v_img_stride, factor, cd.lo,
                                            cd.hi}), rows,
                     rpw, tw);
    else
        EMSIM_LAUNCH(N, (k_row_transmit_fft<N, false>), grid, block, 0, s,
                     (OpTransmit<N, false>{in, V, out, rows_per_img, v_img_stride, factor, cd.lo,
                                            cd.hi}), rows,
                     rpw, tw);
    return EMSIM_HIP_OK;
}

template <int N>
int launch_row_ifft_intensity(const float2* in, float* out, int64_t rows, const float2* tw,
                              hipStream_t s) {
    static int resident_cache[64];
    const int64_t resident =
        resident_blocks(k_row_ifft_intensity<N>, RowCfg<N>::BLOCK, resident_cache);
    int rpw;
    dim3 grid;
    row_grid<N>(rows, rpw, grid, resident);
    EMSIM_LAUNCH(N, (k_row_ifft_intensity<N>), grid, dim3(RowCfg<N>::BLOCK), 0, s,
                 (OpIfftIntensity<N>{in, out}), rows, rpw, tw);
    return EMSIM_HIP_OK;
}

template <int N, class Mul, int SHAPE = 0>
int launch_col_mul_shape(float2* data, int ld, int ncols, int64_t img_stride, int n_img, Mul mul,
                         const float2* tw, hipStream_t s, ColDead cd) {
    using Cfg = ColCfg<N, SHAPE>;
    const int tiles_per_img = (int)ceil_div(ncols, Cfg::C);
    DeadCols dc;
    dc.lo = cd.lo;
    dc.hi = cd.hi;
    dc.live_per_img = tiles_per_img;
    dc.skip_lo = tiles_per_img;
    dc.skip_n = 0;
    if (cd.skip_tiles && cd.lo <= cd.hi) {
        // tiles [first, end) lie inside [lo, hi]
        const int first = (int)ceil_div(cd.lo, Cfg::C), end = (cd.hi + 1) / Cfg::C;
        if (end > first) {
            dc.skip_lo = first;
            dc.skip_n = end - first;
            dc.live_per_img = tiles_per_img - dc.skip_n;
        }
    }
    const int64_t n_tiles = (int64_t)dc.live_per_img * n_img;
    if (n_tiles <= 0) return EMSIM_HIP_OK;   // nothing to transform
    if (n_tiles >= ((int64_t)1 << 31))
        return fail(EMSIM_HIP_EINVAL, "column pass: %lld column tiles, at most 2^31 - 1",
                    (long long)n_tiles);
    // Blocks pair up on an XCD over strips of two tiles (see
    // k_col_fft_mul_ifft).  By default one round of resident blocks (two
    // per CU) with the strips dealt out evenly, or one strip per pair when
    // there are fewer strips than that; the tiles-per-block knob instead
    // sets the strips per pair.  Pairs come in eights (a grid of whole
    // multiples of 16).
    static int resident_cache[64];
    const int64_t strips = ceil_div(n_tiles, 2);
    int64_t pairs;
    if (g_col_tiles_per_block > 0) {
        pairs = ceil_div(strips, g_col_tiles_per_block);
    } else {
        const int64_t resident =
            resident_blocks(k_col_fft_mul_ifft<N, Mul, SHAPE>, Cfg::BLOCK, resident_cache);
        const int64_t max_pairs = resident >= 16 ? resident / 16 * 8 : 256;
        pairs = strips < max_pairs ? strips : max_pairs;
    }
    pairs = ceil_div(pairs, 8) * 8;
    const RunSched sched{(int)(strips / pairs), (int)(strips % pairs)};
    const dim3 grid((unsigned)(2 * pairs));
    EMSIM_LAUNCH(N, (k_col_fft_mul_ifft<N, Mul, SHAPE>), grid, dim3(Cfg::BLOCK), 0, s, data, ld,
                 ncols, dc, img_stride, n_tiles, sched, mul, cd.carry, cd.carry_first, tw);
    return EMSIM_HIP_OK;
}

// Full-width column tiles a launch over n_img images has (ColDead's skipped
// tiles left out).
template <int N>
int64_t full_col_tiles(int ncols, int n_img, const ColDead& cd) {
    constexpr int C = ColCfg<N>::C;
    int64_t per = ceil_div(ncols, C);
    if (cd.skip_tiles && cd.lo <= cd.hi)
        per -= std::max<int64_t>((cd.hi + 1) / C - ceil_div(cd.lo, C), 0);
    return per * n_img;
}

// The propagator and last-slice passes take the tuned tile shape
// (emsim_hip_tuning_set("col_shape")) at the lengths that have one; otherwise
// col_shape_for decides.  The shapes give the same values: each transform's
// butterflies are the same whichever threads run them.
template <int N, class Mul>
int launch_col_mul_impl(float2* data, int ld, int ncols, int64_t img_stride, int n_img, Mul mul,
                        const float2* tw, hipStream_t s, ColDead cd = ColDead{},
                        bool tuned = false) {
    constexpr bool kTunable = col_shapes(N);
    const int shape = kTunable && tuned && g_col_shape > 0
                          ? g_col_shape
                          : col_shape_for<N>(full_col_tiles<N>(ncols, n_img, cd));
    if constexpr (kTunable || N == 128) {
        if (shape == 1)
            return launch_col_mul_shape<N, Mul, 1>(data, ld, ncols, img_stride, n_img, mul, tw, s,
                                                   cd);
    }
    if constexpr (kTunable) {
        if (shape == 2)
            return launch_col_mul_shape<N, Mul, 2>(data, ld, ncols, img_stride, n_img, mul, tw, s,
                                                   cd);
    }
    if constexpr (N == 128 || N == 256) {
        if (shape == 3)
            return launch_col_mul_shape<N, Mul, 3>(data, ld, ncols, img_stride, n_img, mul, tw, s,
                                                   cd);
    }
    return launch_col_mul_shape<N, Mul, 0>(data, ld, ncols, img_stride, n_img, mul, tw, s, cd);
}

template <int N>
int launch_col_prop(float2* data, int ld, int ncols, int64_t img_stride, int n_img,
                    PropagatorMul mul, const float2* tw, hipStream_t s, ColDead cd) {
    return launch_col_mul_impl<N>(data, ld, ncols, img_stride, n_img, mul, tw, s, cd, true);
}

template <int N>
int launch_col_lens(float2* data, int ld, int ncols, int64_t img_stride, int n_img, LensMul mul,
                    const float2* tw, hipStream_t s) {
    return launch_col_mul_impl<N>(data, ld, ncols, img_stride, n_img, mul, tw, s);
}

template <int N>
int launch_r2c_pairs(const float* in, float2* out, int64_t n_pairs, int rows_per_plane,
                     int planes_per_group, int64_t in_group_stride, int64_t in_plane0, int ldh,
                     const float2* tw, hipStream_t s) {
    int rpw;
    dim3 grid;
    row_grid<N>(n_pairs, rpw, grid);
    OpR2CPairs<N> op;
    op.in = in;
    op.out = out;
    op.rows_per_plane = rows_per_plane;
    op.planes_per_group = planes_per_group;
    op.ldh = ldh;
    op.in_group_stride = in_group_stride;
    op.in_plane0 = in_plane0;
    EMSIM_LAUNCH(N, (k_row_r2c_pairs<N>), grid, dim3(RowCfg<N>::BLOCK), 0, s, op, n_pairs, rpw,
                 tw);
    return EMSIM_HIP_OK;
}

template <int N>
int launch_c2r_pairs(const float2* in, float* out, int64_t n_pairs, float clip_lo, int ldh,
                     const float2* tw, hipStream_t s) {
    int rpw;
    dim3 grid;
    row_grid<N>(n_pairs, rpw, grid);
    EMSIM_LAUNCH(N, (k_row_c2r_pairs<N>), grid, dim3(RowCfg<N>::BLOCK), 0, s,
                 (OpC2RPairs<N>{in, out, clip_lo, ldh}), n_pairs, rpw, tw);
    return EMSIM_HIP_OK;
}

template <int N>
int launch_col_spectrum(float2* X, const float* sf, int n_elems, int n_sc, int H, int ldh,
                        int n2, int bandlimit, int band_r2, float inv_npix, const float2* tw,
                        hipStream_t s) {
    using Cfg = SpecCfg<N>;
    const dim3 grid((unsigned)ceil_div(H, Cfg::C), (unsigned)n_sc);
    EMSIM_LAUNCH(N, (k_col_spectrum<N>), grid, dim3(Cfg::BLOCK), 0, s, X, sf, n_elems, n_sc, H,
                       ldh, n2, bandlimit, band_r2, inv_npix, tw);
    return EMSIM_HIP_OK;
}

int row_fft(int n, bool inv, const float2* in, float2* out, int64_t rows, const float2* tw,
            hipStream_t s) {
    EMSIM_DISPATCH(n, launch_row_fft, inv, in, out, rows, tw, s);
}
int row_transmit_fft(int n, bool first, const float2* in, const float* V, float2* out,
                     int64_t rows, int rows_per_img, int64_t v_img_stride, float factor,
                     ColDead cd, const float2* tw, hipStream_t s) {
    EMSIM_DISPATCH(n, launch_row_transmit_fft, first, in, V, out, rows, rows_per_img,
                   v_img_stride, factor, cd, tw, s);
}
int row_ifft_intensity(int n, const float2* in, float* out, int64_t rows, const float2* tw,
                       hipStream_t s) {
    EMSIM_DISPATCH(n, launch_row_ifft_intensity, in, out, rows, tw, s);
}
int col_prop(int n, float2* data, int ld, int ncols, int64_t img_stride, int n_img,
             PropagatorMul mul, const float2* tw, hipStream_t s, ColDead cd = ColDead{}) {
    EMSIM_DISPATCH(n, launch_col_prop, data, ld, ncols, img_stride, n_img, mul, tw, s, cd);
}
int col_lens(int n, float2* data, int ld, int ncols, int64_t img_stride, int n_img, LensMul mul,
             const float2* tw, hipStream_t s) {
    EMSIM_DISPATCH(n, launch_col_lens, data, ld, ncols, img_stride, n_img, mul, tw, s);
}
int r2c_pairs(int n, const float* in, float2* out, int64_t n_pairs, int rows_per_plane,
              int planes_per_group, int64_t in_group_stride, int64_t in_plane0, int ldh,
              const float2* tw, hipStream_t s) {
    EMSIM_DISPATCH(n, launch_r2c_pairs, in, out, n_pairs, rows_per_plane, planes_per_group,
                   in_group_stride, in_plane0, ldh, tw, s);
}
int c2r_pairs(int n, const float2* in, float* out, int64_t n_pairs, float clip_lo, int ldh,
              const float2* tw, hipStream_t s) {
    EMSIM_DISPATCH(n, launch_c2r_pairs, in, out, n_pairs, clip_lo, ldh, tw, s);
}
int col_spectrum(int n, float2* X, const float* sf, int n_elems, int n_sc, int H, int ldh,
                 int n2, int bandlimit, int band_r2, float inv_npix, const float2* tw,
                 hipStream_t s) {
    EMSIM_DISPATCH(n, launch_col_spectrum, X, sf, n_elems, n_sc, H, ldh, n2, bandlimit, band_r2,
                   inv_npix, tw, s);
}

// Float32 constants of the propagators, in the reference's operation order
// (WavePropagator.cpp:19-23,62-85,108-130).
PropagatorMul make_propagator(const emsim_hip_wave_propagator* w, float dz) {
    PropagatorMul p;
    p.n1 = w->n1;
    p.n2 = w->n2;
    p.dfx = w->dfx;
    p.dfy = w->dfy;
    p.filter2 = w->filter2;
    const float lp = w->lam * kPi32;
    p.lpd = lp * dz;
    p.inv_npix = 1.0f / (float)(w->n1 * w->n2);
    return p;
}

// The wave columns the propagator zeroes whole.  Its mask keeps
// f^2 = fx^2 + fy^2 <= filter^2 (PropagatorMul::apply), and in float32
// round-to-nearest f^2 >= fy^2, so every column with fy^2 > filter^2 is
// zero; fy^2 is formed by the same float32 operations as on the device.
// Reported only as one contiguous run of column indices (else none).
ColDead dead_columns(const PropagatorMul& p) {
    ColDead d;
    int lo = -1, hi = -1;
    for (int j = 0; j < p.n2; ++j) {
        const float fy = (float)freq_int(j, p.n2) * p.dfy;
        const float fy2 = fy * fy;
        if (fy2 <= p.filter2) continue;
        if (lo < 0) lo = j;
        else if (hi != j - 1) return ColDead{};
        hi = j;
    }
    if (lo >= 0) {
        d.lo = lo;
        d.hi = hi;
    }
    return d;
}

LensMul make_lens(const emsim_hip_wave_propagator* w, float cs_mm, float defocus, float aperture) {
    LensMul l;
    l.n1 = w->n1;
    l.n2 = w->n2;
    l.dfx = w->dfx;
    l.dfy = w->dfy;
    float c1 = 0.5f * kPi32;
    c1 = c1 * cs_mm;
    c1 = c1 * 1e7f;
    c1 = c1 * w->lam;
    c1 = c1 * w->lam;
    c1 = c1 * w->lam;
    float c2 = kPi32 * defocus;
    c2 = c2 * w->lam;
    const float f_aper = aperture / w->lam;
    l.c1 = c1;
    l.c2 = c2;
    l.faper2 = f_aper * f_aper;
    l.inv_npix = 1.0f / (float)(w->n1 * w->n2);
    return l;
}

// --------------------------------------------------------------------------
// chirp-z launches (sizes that are not powers of two), dispatched on the
// convolution length M
// --------------------------------------------------------------------------
template <int M, int MODE>
int launch_chirp_rows_mode(ChirpRows a, const float2* tw, hipStream_t s) {
    static int resident_cache[64];
    dim3 grid;
    row_grid<M>(a.rows, a.rpb, grid,
                resident_blocks(k_chirp_rows<M, MODE>, RowCfg<M>::BLOCK, resident_cache));
    EMSIM_LAUNCH(M, (k_chirp_rows<M, MODE>), grid, dim3(RowCfg<M>::BLOCK), 0, s, a, tw);
    return EMSIM_HIP_OK;
}
template <int M>
int launch_chirp_rows(int mode, const ChirpRows& a, const float2* tw, hipStream_t s) {
    if (mode == kChirpFwd) return launch_chirp_rows_mode<M, kChirpFwd>(a, tw, s);
    if (mode == kChirpMid) return launch_chirp_rows_mode<M, kChirpMid>(a, tw, s);
    if (mode == kChirpInv) return launch_chirp_rows_mode<M, kChirpInv>(a, tw, s);
    return launch_chirp_rows_mode<M, kChirpInt>(a, tw, s);
}

// Narrow column tiles while the wide ones would not give every CU a block (one
// 75^2 image of 20 slices: 222 us against 255; past it both measure the same).
bool chirp_narrow(int64_t wide_tiles) { return wide_tiles < 256; }

// Runs of n_tiles column tiles over at most one round of resident blocks.
template <class K>
int chirp_sched(K k, int block, int64_t n_tiles, int (&cache)[64], RunSched& sched, dim3& grid) {
    if (n_tiles >= ((int64_t)1 << 31))
        return fail(EMSIM_HIP_EINVAL, "chirp-z columns: %lld tiles, at most 2^31 - 1",
                    (long long)n_tiles);
    const int64_t resident = resident_blocks(k, block, cache);
    const int64_t blocks = resident > 0 && resident < n_tiles ? resident : n_tiles;
    sched = RunSched{(int)(n_tiles / blocks), (int)(n_tiles % blocks)};
    grid = dim3((unsigned)blocks);
    return EMSIM_HIP_OK;
}

template <int M, class Mul, bool NARROW>
int launch_chirp_cols_cfg(float2* data, int n_img, int n2, const ChirpTab& col, const Mul& mul,
                          const float2* tw, hipStream_t s) {
    using Cfg = ChirpColCfg<M, NARROW>;
    static int resident_cache[64];
    const int tiles = (int)ceil_div(n2, Cfg::C);
    const int64_t n_tiles = (int64_t)tiles * n_img;
    RunSched sched;
    dim3 grid;
    const int rc = chirp_sched(k_chirp_cols<M, Mul, NARROW>, Cfg::BLOCK, n_tiles, resident_cache,
                               sched, grid);
    if (rc) return rc;
    EMSIM_LAUNCH(M, (k_chirp_cols<M, Mul, NARROW>), grid, dim3(Cfg::BLOCK), 0, s, data, n2, tiles,
                 n_tiles, sched, col, mul, tw);
    return EMSIM_HIP_OK;
}
template <int M, class Mul>
int launch_chirp_cols(float2* data, int n_img, int n2, const ChirpTab& col, const Mul& mul,
                      const float2* tw, hipStream_t s) {
    if (chirp_narrow(ceil_div(n2, ChirpColCfg<M, false>::C) * n_img))
        return launch_chirp_cols_cfg<M, Mul, true>(data, n_img, n2, col, mul, tw, s);
    return launch_chirp_cols_cfg<M, Mul, false>(data, n_img, n2, col, mul, tw, s);
}

template <int M>
int launch_chirp_r2c(const float* hist, float2* X, int n_elems, int n_slices, int s0, int sc,
                     int n1, int ldh, const ChirpTab& row, const float2* c1, const float2* tw,
                     hipStream_t s) {
    static int resident_cache[64];
    const int64_t pairs = (int64_t)n_elems * sc * ((n1 + 1) / 2);
    int rpb;
    dim3 grid;
    row_grid<M>(pairs, rpb, grid,
                resident_blocks(k_chirp_r2c<M>, RowCfg<M>::BLOCK, resident_cache));
    EMSIM_LAUNCH(M, (k_chirp_r2c<M>), grid, dim3(RowCfg<M>::BLOCK), 0, s, hist, X, n_elems,
                 n_slices, s0, sc, n1, ldh, rpb, row, c1, tw);
    return EMSIM_HIP_OK;
}

template <int M, bool NARROW>
int launch_chirp_spectrum_cfg(float2* X, const float* sf, int n_elems, int sc, int H, int ldh,
                              int n2, int bandlimit, int band_r2, float inv_npix,
                              const ChirpTab& col, const float2* tw, hipStream_t s) {
    using Cfg = ChirpColCfg<M, NARROW>;
    static int resident_cache[64];
    const int tiles = (int)ceil_div(H, Cfg::C);
    RunSched sched;
    dim3 grid;
    const int rc = chirp_sched(k_chirp_spectrum<M, NARROW>, Cfg::BLOCK, (int64_t)tiles * sc,
                               resident_cache, sched, grid);
    if (rc) return rc;
    EMSIM_LAUNCH(M, (k_chirp_spectrum<M, NARROW>), grid, dim3(Cfg::BLOCK), 0, s, X, sf, n_elems,
                 sc, tiles, sched, H, ldh, n2, bandlimit, band_r2, inv_npix, col, tw);
    return EMSIM_HIP_OK;
}
template <int M>
int launch_chirp_spectrum(float2* X, const float* sf, int n_elems, int sc, int H, int ldh, int n2,
                          int bandlimit, int band_r2, float inv_npix, const ChirpTab& col,
                          const float2* tw, hipStream_t s) {
    if (chirp_narrow(ceil_div(H, ChirpColCfg<M, false>::C) * sc))
        return launch_chirp_spectrum_cfg<M, true>(X, sf, n_elems, sc, H, ldh, n2, bandlimit,
                                                  band_r2, inv_npix, col, tw, s);
    return launch_chirp_spectrum_cfg<M, false>(X, sf, n_elems, sc, H, ldh, n2, bandlimit, band_r2,
                                               inv_npix, col, tw, s);
}

template <int M>
int launch_chirp_c2r(const float2* X, float* out, int sc, int n1, int ldh, float clip_lo,
                     const ChirpTab& row, const float2* tw, hipStream_t s) {
    static int resident_cache[64];
    int rpb;
    dim3 grid;
    row_grid<M>((int64_t)sc * ((n1 + 1) / 2), rpb, grid,
                resident_blocks(k_chirp_c2r<M>, RowCfg<M>::BLOCK, resident_cache));
    EMSIM_LAUNCH(M, (k_chirp_c2r<M>), grid, dim3(RowCfg<M>::BLOCK), 0, s, X, out, sc, n1, ldh, rpb,
                 clip_lo, row, tw);
    return EMSIM_HIP_OK;
}

#define EMSIM_CHIRP_DISPATCH(M, FN, ...)                                             \
    switch (M) {                                                                     \
        case 16: return FN<16>(__VA_ARGS__);                                         \
        case 32: return FN<32>(__VA_ARGS__);                                         \
        case 64: return FN<64>(__VA_ARGS__);                                         \
        case 128: return FN<128>(__VA_ARGS__);                                       \
        case 256: return FN<256>(__VA_ARGS__);                                       \
        case 512: return FN<512>(__VA_ARGS__);                                       \
        case 1024: return FN<1024>(__VA_ARGS__);                                     \
        case 2048: return FN<2048>(__VA_ARGS__);                                     \
        case 4096: return FN<4096>(__VA_ARGS__);                                     \
        default: return fail(EMSIM_HIP_EUNSUPPORTED, "unsupported chirp-z length %d", M); \
    }

int chirp_rows(int M, int mode, const ChirpRows& a, const float2* tw, hipStream_t s) {
    EMSIM_CHIRP_DISPATCH(M, launch_chirp_rows, mode, a, tw, s);
}
int chirp_cols(int M, float2* data, int n_img, int n2, const ChirpTab& col, const PropagatorMul& mul,
               const float2* tw, hipStream_t s) {
    EMSIM_CHIRP_DISPATCH(M, launch_chirp_cols, data, n_img, n2, col, mul, tw, s);
}
int chirp_cols(int M, float2* data, int n_img, int n2, const ChirpTab& col, const LensMul& mul,
               const float2* tw, hipStream_t s) {
    EMSIM_CHIRP_DISPATCH(M, launch_chirp_cols, data, n_img, n2, col, mul, tw, s);
}
int chirp_r2c(int M, const float* hist, float2* X, int n_elems, int n_slices, int s0, int sc, int n1,
              int ldh, const ChirpTab& row, const float2* c1, const float2* tw, hipStream_t s) {
    EMSIM_CHIRP_DISPATCH(M, launch_chirp_r2c, hist, X, n_elems, n_slices, s0, sc, n1, ldh, row, c1,
                         tw, s);
}
int chirp_spectrum(int M, float2* X, const float* sf, int n_elems, int sc, int H, int ldh, int n2,
                   int bandlimit, int band_r2, float inv_npix, const ChirpTab& col,
                   const float2* tw, hipStream_t s) {
    EMSIM_CHIRP_DISPATCH(M, launch_chirp_spectrum, X, sf, n_elems, sc, H, ldh, n2, bandlimit,
                         band_r2, inv_npix, col, tw, s);
}
int chirp_c2r(int M, const float2* X, float* out, int sc, int n1, int ldh, float clip_lo,
              const ChirpTab& row, const float2* tw, hipStream_t s) {
    EMSIM_CHIRP_DISPATCH(M, launch_chirp_c2r, X, out, sc, n1, ldh, clip_lo, row, tw, s);
}

// Row-pass arguments of a batch of waves (V: one slice's potentials, or null).
ChirpRows chirp_row_args(const emsim_hip_wave_propagator* w, const float2* in, float2* out,
                         int batch, const float* V, int64_t v_img_stride) {
    ChirpRows a;
    a.in = in;
    a.out = out;
    a.image = nullptr;
    a.V = V;
    a.v_img_stride = v_img_stride;
    a.factor = w->factor;
    a.rows = (int64_t)batch * w->n1;
    a.rows_per_img = w->n1;
    a.row = w->p2.tab();
    a.c1 = w->p1.c;
    a.rpb = 1;
    return a;
}

// FFT -> Fourier-space multiplier -> IFFT of every image of a batch (out: the
// wave, or with image set its intensity, out being scratch).
template <class Mul>
int chirp_filter(const emsim_hip_wave_propagator* w, const float2* in, float2* out, float* image,
                 int batch, const Mul& mul, hipStream_t s) {
    ChirpRows a = chirp_row_args(w, in, out, batch, nullptr, 0);
    int rc = chirp_rows(w->p2.M, kChirpFwd, a, w->tw, s);
    if (rc) return rc;
    rc = chirp_cols(w->p1.M, out, batch, w->n2, w->p1.tab(), mul, w->tw, s);
    if (rc) return rc;
    a.in = out;
    a.image = image;
    return chirp_rows(w->p2.M, image ? kChirpInt : kChirpInv, a, w->tw, s);
}

}  // namespace

// ==========================================================================
// library
// ==========================================================================
extern "C" int emsim_hip_abi_version(void) { return EMSIM_HIP_ABI_VERSION; }

extern "C" const char* emsim_hip_last_error(void) { return g_last_error.c_str(); }

extern "C" int emsim_hip_fft_size_supported(int n) {
    return pow2_supported(n) ? 1 : (chirp_supported(n) ? 2 : 0);
}

extern "C" int emsim_hip_bin_edges(int n, double d, double* edges64_host, float* edges32_host,
                                   int cap, int* len_out) {
    if (n < 1 || !(d > 0) || !len_out) return fail(EMSIM_HIP_EINVAL, "bin_edges: bad arguments");
    std::vector<double> e;
    reference_edges(n, d, e);
    *len_out = (int)e.size();
    for (int i = 0; i < (int)e.size() && i < cap; ++i) {
        if (edges64_host) edges64_host[i] = e[i];
        if (edges32_host) edges32_host[i] = round_up_f32(e[i]);
    }
    return EMSIM_HIP_OK;
}

// ==========================================================================
// slice builder
// ==========================================================================
extern "C" int emsim_hip_slice_builder_create(emsim_hip_slice_builder** out,
                                              const float* sf_host, int n_elems, int n_slices,
                                              int n1, int n2, double dz, double d1, double d2,
                                              int one_slice) {
    if (!out) return fail(EMSIM_HIP_EINVAL, "slice_builder_create: null output handle");
    *out = nullptr;
    if (!sf_host || n_elems < 1 || n_slices < 1)
        return fail(EMSIM_HIP_EINVAL, "slice_builder_create: need n_elems >= 1, n_slices >= 1 "
                                      "and a scattering-factor table");
    if (n_elems > kMaxElems)
        return fail(EMSIM_HIP_EUNSUPPORTED, "slice_builder_create: at most %d elements", kMaxElems);
    if (!size_supported(n1) || !size_supported(n2))
        return fail(EMSIM_HIP_EUNSUPPORTED,
                    "slice_builder_create: lateral size %dx%d; the hip backend implements "
                    "sizes from 8 to %d (powers of two up to %d)", n1, n2, kChirpMaxN, kTwN);
    if (one_slice && n_slices != 1)
        return fail(EMSIM_HIP_EINVAL, "slice_builder_create: one-slice builder needs n_slices == 1");
    if (!(d1 > 0) || !(d2 > 0) || (!one_slice && !(dz > 0)))
        return fail(EMSIM_HIP_EINVAL, "slice_builder_create: voxel sizes must be positive");

    // Edge tables (float64 numpy.arange semantics, then rounded up to float32).
    const int ns[3] = {one_slice ? 1 : n_slices, n1, n2};
    const double ds[3] = {one_slice ? 1.0 : dz, d1, d2};
    std::vector<float> edges32;
    int last_exact[3];
    float inv_d[3];
    for (int a = 0; a < 3; ++a) {
        std::vector<double> e;
        reference_edges(ns[a], ds[a], e);
        if ((int)e.size() != ns[a] + 1) {
            if (a == 0 && one_slice) {
                e.resize(2);  // axis 0 is ignored by the one-slice builder
                e[0] = -1.0;
                e[1] = 1.0;
            } else {
                return fail(EMSIM_HIP_EUNSUPPORTED,
                            "binning axis %d: numpy.arange makes %d edges for %d bins of %.17g "
                            "(the reference would return a %d-bin histogram on this axis and "
                            "misalign its slices); choose a pixel size that divides evenly",
                            a, (int)e.size(), ns[a], ds[a], (int)e.size() - 1);
            }
        }
        for (double x : e) edges32.push_back(round_up_f32(x));
        last_exact[a] = ((double)(float)e.back() == e.back()) ? 1 : 0;
        inv_d[a] = (float)(1.0 / ds[a]);
    }

    emsim_hip_slice_builder* b = new (std::nothrow) emsim_hip_slice_builder();
    if (!b) return fail(EMSIM_HIP_ENOMEM, "slice_builder_create: out of host memory");
    b->n_elems = n_elems;
    b->n_slices = n_slices;
    b->n1 = n1;
    b->n2 = n2;
    b->H = n2 / 2 + 1;
    b->dz = dz;
    b->d1 = d1;
    b->d2 = d2;
    b->one_slice = one_slice ? 1 : 0;
    for (int a = 0; a < 3; ++a) {
        b->last_exact[a] = last_exact[a];
        b->inv_d[a] = inv_d[a];
    }
    int rows = kBinTileWords / n2;
    if (rows < 1) rows = 1;
    if (rows > n1) rows = n1;
    b->tile_rows = rows;
    b->tiles_per_plane = (int)ceil_div(n1, rows);

    int rc = get_twiddles(&b->tw);
    if (!rc && !(pow2_supported(n1) && pow2_supported(n2))) {
        b->chirp = true;
        rc = chirp_plan_create(n1, b->p1);
        if (!rc) rc = chirp_plan_create(n2, b->p2);
    }
    if (rc) {
        emsim_hip_slice_builder_destroy(b);
        return rc;
    }
    const size_t sf_bytes = (size_t)n_elems * n1 * b->H * sizeof(float);
    hipError_t err = hipMalloc(&b->sf, sf_bytes);
    if (err == hipSuccess) err = hipMemcpy(b->sf, sf_host, sf_bytes, hipMemcpyHostToDevice);
    if (err == hipSuccess && pow2_supported(n1)) {
        const int C = spec_tile_cols(n1), tiles = (int)ceil_div(b->H, C);
        std::vector<float> t((size_t)n_elems * tiles * n1 * C, 0.f);
        for (int e = 0; e < n_elems; ++e)
            for (int x = 0; x < n1; ++x)
                for (int j = 0; j < b->H; ++j)
                    t[(((size_t)e * tiles + j / C) * n1 + x) * C + j % C] =
                        sf_host[((size_t)e * n1 + x) * b->H + j];
        err = hipMalloc(&b->sf_tiles, t.size() * sizeof(float));
        if (err == hipSuccess)
            err = hipMemcpy(b->sf_tiles, t.data(), t.size() * sizeof(float), hipMemcpyHostToDevice);
    }
    if (err == hipSuccess) err = hipMalloc(&b->edges, edges32.size() * sizeof(float));
    if (err == hipSuccess)
        err = hipMemcpy(b->edges, edges32.data(), edges32.size() * sizeof(float),
                        hipMemcpyHostToDevice);
    if (err != hipSuccess) {
        emsim_hip_slice_builder_destroy(b);
        return fail(EMSIM_HIP_EDEVICE, "slice_builder_create: %s", hipGetErrorString(err));
    }
    *out = b;
    return EMSIM_HIP_OK;
}

extern "C" int emsim_hip_slice_builder_destroy(emsim_hip_slice_builder* b) {
    if (!b) return EMSIM_HIP_OK;
    chirp_plan_free(b->p1);
    chirp_plan_free(b->p2);
    if (b->sf) (void)hipFree(b->sf);
    if (b->sf_tiles) (void)hipFree(b->sf_tiles);
    if (b->edges) (void)hipFree(b->edges);
    delete b;
    return EMSIM_HIP_OK;
}

namespace {
struct BinWorkspace {
    int32_t* atom_tile;
    uint32_t* atom_local;
    uint32_t* bucket;
    uint32_t* tile_count;
    uint32_t* tile_start;
    uint32_t* block_sums;
    size_t bytes;
};

size_t align_up(size_t x) { return (x + 255) & ~(size_t)255; }

BinWorkspace bin_layout(const emsim_hip_slice_builder* b, int64_t n_atoms, char* base) {
    const int64_t n0 = b->one_slice ? 1 : b->n_slices;
    const int64_t n_tiles = (int64_t)b->n_elems * n0 * b->tiles_per_plane;
    const int64_t n_scan = n_tiles + 1;
    const int64_t n_blocks = ceil_div(n_scan, kScanTile);
    BinWorkspace w;
    size_t off = 0;
    w.atom_tile = (int32_t*)(base + off);  off += align_up(sizeof(int32_t) * (size_t)n_atoms);
    w.atom_local = (uint32_t*)(base + off); off += align_up(sizeof(uint32_t) * (size_t)n_atoms);
    w.bucket = (uint32_t*)(base + off);     off += align_up(sizeof(uint32_t) * (size_t)n_atoms);
    w.tile_count = (uint32_t*)(base + off); off += align_up(sizeof(uint32_t) * (size_t)n_scan);
    w.tile_start = (uint32_t*)(base + off); off += align_up(sizeof(uint32_t) * (size_t)n_scan);
    w.block_sums = (uint32_t*)(base + off); off += align_up(sizeof(uint32_t) * (size_t)n_blocks);
    w.bytes = off;
    return w;
}
}  // namespace

extern "C" size_t emsim_hip_bin_workspace_size(const emsim_hip_slice_builder* b, int64_t n_atoms) {
    if (!b || n_atoms < 0) return 0;
    return bin_layout(b, n_atoms, nullptr).bytes;
}

extern "C" int emsim_hip_bin_atoms(const emsim_hip_slice_builder* b, const float* coords,
                                   const int64_t* counts_host, int64_t n_atoms, float* hist,
                                   void* workspace, size_t workspace_bytes,
                                   emsim_stream_t stream_) {
    hipStream_t s = (hipStream_t)stream_;
    if (!b || !hist || !counts_host || n_atoms < 0 || (n_atoms > 0 && !coords))
        return fail(EMSIM_HIP_EINVAL, "bin_atoms: bad arguments");
    if (n_atoms >= (int64_t)0x7fffffff)
        return fail(EMSIM_HIP_EUNSUPPORTED, "bin_atoms: at most 2^31-1 atoms per call");
    ElemOffsets eo;
    eo.n_elems = b->n_elems;
    eo.off[0] = 0;
    for (int e = 0; e < b->n_elems; ++e) {
        if (counts_host[e] < 0) return fail(EMSIM_HIP_EINVAL, "bin_atoms: negative count");
        eo.off[e + 1] = eo.off[e] + counts_host[e];
    }
    if (eo.off[b->n_elems] > n_atoms)
        return fail(EMSIM_HIP_EINVAL, "bin_atoms: counts sum to %lld but only %lld atoms given",
                    (long long)eo.off[b->n_elems], (long long)n_atoms);
    BinWorkspace w = bin_layout(b, n_atoms, (char*)workspace);
    if (!workspace || workspace_bytes < w.bytes)
        return fail(EMSIM_HIP_EWORKSPACE, "bin_atoms: workspace needs %zu bytes", w.bytes);

    const int64_t n0 = b->one_slice ? 1 : b->n_slices;
    BinGeom g;
    g.e0 = b->edges;
    g.e1 = b->edges + (n0 + 1);
    g.e2 = g.e1 + (b->n1 + 1);
    g.n0 = (int)n0;
    g.n1 = b->n1;
    g.n2 = b->n2;
    g.last0 = b->last_exact[0];
    g.last1 = b->last_exact[1];
    g.last2 = b->last_exact[2];
    g.inv0 = b->inv_d[0];
    g.inv1 = b->inv_d[1];
    g.inv2 = b->inv_d[2];
    g.one_slice = b->one_slice;
    g.tile_rows = b->tile_rows;
    g.tiles_per_plane = b->tiles_per_plane;

    const int64_t n_tiles = (int64_t)b->n_elems * n0 * b->tiles_per_plane;
    const int64_t n_scan = n_tiles + 1;
    const int64_t n_blocks = ceil_div(n_scan, kScanTile);

    EMSIM_LAUNCH(0, k_fill_u32, dim3(grid_for(n_scan, 256)), dim3(256), 0, s, w.tile_count,
                       n_scan, 0u);
    if (n_atoms > 0) {
        EMSIM_LAUNCH(0, k_bin_classify, dim3(grid_for(n_atoms, 256)), dim3(256), 0, s, coords,
                           n_atoms, eo, g, w.atom_tile, w.atom_local, w.tile_count);
    }
    EMSIM_LAUNCH(0, k_scan_tiles, dim3((unsigned)n_blocks), dim3(kScanBlock), 0, s,
                       w.tile_count, w.tile_start, n_scan, w.block_sums);
    EMSIM_LAUNCH(0, k_scan_sums, dim3(1), dim3(kScanBlock), 0, s, w.block_sums, n_blocks);
    EMSIM_LAUNCH(0, k_scan_add, dim3((unsigned)n_blocks), dim3(kScanBlock), 0, s, w.tile_start,
                       n_scan, w.block_sums);
    if (n_atoms > 0) {
        EMSIM_LAUNCH(0, k_bin_scatter, dim3(grid_for(n_atoms, 256)), dim3(256), 0, s, n_atoms,
                           w.atom_tile, w.atom_local, w.tile_start, w.tile_count, w.bucket);
    }
    EMSIM_LAUNCH(0, k_bin_tiles, dim3((unsigned)n_tiles), dim3(kBinBlock), 0, s, w.bucket,
                       w.tile_start, g, hist);
    return EMSIM_HIP_OK;
}

extern "C" int emsim_hip_add_water(const emsim_hip_slice_builder* b, float* hist, int idx_h,
                                   int idx_o, double voxel_water, uint64_t seed,
                                   emsim_stream_t stream_) {
    if (!b || !hist || idx_h < 0 || idx_o < 0 || idx_h >= b->n_elems || idx_o >= b->n_elems ||
        idx_h == idx_o || !(voxel_water >= 0))
        return fail(EMSIM_HIP_EINVAL, "add_water: bad arguments");
    const int64_t n0 = b->one_slice ? 1 : b->n_slices;
    const int64_t vox = n0 * b->n1 * b->n2;
    const float lam_o = (float)voxel_water, lam_h = (float)(2.0 * voxel_water);
    const float exp_o = (float)std::exp(-voxel_water), exp_h = (float)std::exp(-2.0 * voxel_water);
    EMSIM_LAUNCH(0, k_add_water, dim3(grid_for(vox, 256)), dim3(256), 0, (hipStream_t)stream_,
                       hist, b->n_elems, vox, idx_h, idx_o, lam_o, exp_o, lam_h, exp_h, seed);
    return EMSIM_HIP_OK;
}

namespace {
// Workspace of make_slices per slice of a chunk: the half spectra of every
// element.
size_t slices_bytes_per_slice(const emsim_hip_slice_builder* b) {
    return (size_t)b->n_elems * b->n1 * half_ld(b->H) * sizeof(float2);
}
}  // namespace

extern "C" size_t emsim_hip_slices_workspace_size(const emsim_hip_slice_builder* b,
                                                  int max_chunk) {
    if (!b) return 0;
    int chunk = (max_chunk <= 0 || max_chunk > b->n_slices) ? b->n_slices : max_chunk;
    return slices_bytes_per_slice(b) * (size_t)chunk;
}

extern "C" int emsim_hip_make_slices(const emsim_hip_slice_builder* b, const float* hist,
                                     float* out, int symmetric_bandlimit, void* workspace,
                                     size_t workspace_bytes, emsim_stream_t stream_) {
    hipStream_t s = (hipStream_t)stream_;
    if (!b || !hist || !out) return fail(EMSIM_HIP_EINVAL, "make_slices: bad arguments");
    if (symmetric_bandlimit && b->n1 != b->n2)
        return fail(EMSIM_HIP_EINVAL,
                    "make_slices: the symmetric band-limit needs a square grid (the reference's "
                    "mask does not broadcast for %dx%d)", b->n1, b->n2);
    const int ldh = half_ld(b->H);
    const size_t per_slice = slices_bytes_per_slice(b);
    if (!workspace || workspace_bytes < per_slice)
        return fail(EMSIM_HIP_EWORKSPACE, "make_slices: workspace needs at least %zu bytes",
                    per_slice);
    int chunk = (int)(workspace_bytes / per_slice);
    if (chunk > b->n_slices) chunk = b->n_slices;
    if (chunk > 65535) chunk = 65535;
    float2* X = (float2*)workspace;
    const int r = (b->n1 < b->n2 ? b->n1 : b->n2) / 2;
    const float inv_npix = 1.0f / (float)((int64_t)b->n1 * b->n2);
    if (b->chirp) {
        // the same passes through chirp-z transforms
        for (int s0 = 0; s0 < b->n_slices; s0 += chunk) {
            const int sc = (b->n_slices - s0) < chunk ? (b->n_slices - s0) : chunk;
            int rc = chirp_r2c(b->p2.M, hist, X, b->n_elems, b->n_slices, s0, sc, b->n1, ldh,
                               b->p2.tab(), b->p1.c, b->tw, s);
            if (rc) return rc;
            rc = chirp_spectrum(b->p1.M, X, b->sf, b->n_elems, sc, b->H, ldh, b->n2,
                                symmetric_bandlimit ? 1 : 0, r * r, inv_npix, b->p1.tab(), b->tw,
                                s);
            if (rc) return rc;
            rc = chirp_c2r(b->p2.M, X, out + (int64_t)s0 * b->n1 * b->n2, sc, b->n1, ldh, 1e-13f,
                           b->p2.tab(), b->tw, s);
            if (rc) return rc;
        }
        return EMSIM_HIP_OK;
    }
    for (int s0 = 0; s0 < b->n_slices; s0 += chunk) {
        const int sc = (b->n_slices - s0) < chunk ? (b->n_slices - s0) : chunk;
        int rc = r2c_pairs(b->n2, hist, X, (int64_t)b->n_elems * sc * (b->n1 / 2), b->n1, sc,
                           b->n_slices, s0, ldh, b->tw, s);
        if (rc) return rc;
        rc = col_spectrum(b->n1, X, b->sf, b->n_elems, sc, b->H, ldh, b->n2,
                          symmetric_bandlimit ? 1 : 0, r * r, inv_npix, b->tw, s);
        if (rc) return rc;
        rc = c2r_pairs(b->n2, X, out + (int64_t)s0 * b->n1 * b->n2, (int64_t)sc * (b->n1 / 2),
                       1e-13f, ldh, b->tw, s);
        if (rc) return rc;
    }
    return EMSIM_HIP_OK;
}

// ==========================================================================
// wave propagator
// ==========================================================================
extern "C" int emsim_hip_wave_propagator_create(emsim_hip_wave_propagator** out, int n1, int n2,
                                                float d1, float d2, float wave_length,
                                                float relativity_gamma) {
    if (!out) return fail(EMSIM_HIP_EINVAL, "wave_propagator_create: null output handle");
    *out = nullptr;
    if (!size_supported(n1) || !size_supported(n2))
        return fail(EMSIM_HIP_EUNSUPPORTED,
                    "wave_propagator_create: wave shape %dx%d; the hip backend implements "
                    "sizes from 8 to %d (powers of two up to %d)", n1, n2, kChirpMaxN, kTwN);
    if (!(d1 > 0) || !(d2 > 0) || !(wave_length > 0))
        return fail(EMSIM_HIP_EINVAL, "wave_propagator_create: sizes must be positive");
    emsim_hip_wave_propagator* w = new (std::nothrow) emsim_hip_wave_propagator();
    if (!w) return fail(EMSIM_HIP_ENOMEM, "wave_propagator_create: out of host memory");
    w->n1 = n1;
    w->n2 = n2;
    w->d1 = d1;
    w->d2 = d2;
    w->lam = wave_length;
    w->gamma = relativity_gamma;
    // WavePropagator.cpp:19-23
    float dfx = 1.0f / d1;
    w->dfx = dfx / (float)n1;
    float dfy = 1.0f / d2;
    w->dfy = dfy / (float)n2;
    const float fmax = 0.5f / (d1 >= d2 ? d1 : d2);
    const float filt = 0.6667f * fmax;
    w->filter2 = filt * filt;
    w->factor = wave_length * relativity_gamma;   // WavePropagator.cpp:42
    int rc = get_twiddles(&w->tw);
    if (!rc && !(pow2_supported(n1) && pow2_supported(n2))) {
        w->chirp = true;
        rc = chirp_plan_create(n1, w->p1);
        if (!rc) rc = chirp_plan_create(n2, w->p2);
    }
    if (rc) {
        emsim_hip_wave_propagator_destroy(w);
        return rc;
    }
    *out = w;
    return EMSIM_HIP_OK;
}

extern "C" int emsim_hip_wave_propagator_destroy(emsim_hip_wave_propagator* w) {
    if (!w) return EMSIM_HIP_OK;
    chirp_plan_free(w->p1);
    chirp_plan_free(w->p2);
    delete w;
    return EMSIM_HIP_OK;
}

extern "C" int emsim_hip_init_wave(const emsim_hip_wave_propagator* w, float value, float* wave,
                                   int batch, emsim_stream_t stream_) {
    if (!w || !wave || batch < 1) return fail(EMSIM_HIP_EINVAL, "init_wave: bad arguments");
    const int64_t n = (int64_t)batch * w->n1 * w->n2;
    EMSIM_LAUNCH(0, k_fill_complex, dim3(grid_for(n, 256)), dim3(256), 0,
                       (hipStream_t)stream_, (float2*)wave, n, value);
    return EMSIM_HIP_OK;
}

extern "C" int emsim_hip_slice_transmit(const emsim_hip_wave_propagator* w, const float* wave,
                                        const float* slice, int64_t slice_batch_stride,
                                        float* out, int batch, emsim_stream_t stream_) {
    if (!w || !wave || !slice || !out || batch < 1 || slice_batch_stride < 0)
        return fail(EMSIM_HIP_EINVAL, "slice_transmit: bad arguments");
    const int64_t npix = (int64_t)w->n1 * w->n2;
    const int64_t n = npix * batch;
    EMSIM_LAUNCH(0, k_transmit, dim3(grid_for(n, 256)), dim3(256), 0, (hipStream_t)stream_,
                       (const float2*)wave, slice, (float2*)out, npix, n, slice_batch_stride,
                       w->factor);
    return EMSIM_HIP_OK;
}

extern "C" int emsim_hip_space_propagate(const emsim_hip_wave_propagator* w, const float* wave,
                                         float dz, float* out, int batch,
                                         emsim_stream_t stream_) {
    hipStream_t s = (hipStream_t)stream_;
    if (!w || !wave || !out || batch < 1) return fail(EMSIM_HIP_EINVAL, "space_propagate: bad arguments");
    if (batch > 65535) return fail(EMSIM_HIP_EUNSUPPORTED, "space_propagate: batch <= 65535");
    if (w->chirp)
        return chirp_filter(w, (const float2*)wave, (float2*)out, nullptr, batch,
                            make_propagator(w, dz), s);
    const int64_t rows = (int64_t)batch * w->n1;
    const int64_t npix = (int64_t)w->n1 * w->n2;
    float2* o = (float2*)out;
    int rc = row_fft(w->n2, false, (const float2*)wave, o, rows, w->tw, s);
    if (!rc) rc = col_prop(w->n1, o, w->n2, w->n2, npix, batch, make_propagator(w, dz), w->tw, s);
    if (!rc) rc = row_fft(w->n2, true, o, o, rows, w->tw, s);
    return rc;
}

extern "C" int emsim_hip_multislice_propagate(const emsim_hip_wave_propagator* w,
                                              const float* wave, const float* slices,
                                              int n_slices, int64_t slices_batch_stride,
                                              float dz, float* out, int batch,
                                              emsim_stream_t stream_) {
    hipStream_t s = (hipStream_t)stream_;
    if (!w || !wave || !slices || !out || batch < 1 || n_slices < 1 || slices_batch_stride < 0)
        return fail(EMSIM_HIP_EINVAL, "multislice_propagate: bad arguments");
    if (batch > 65535) return fail(EMSIM_HIP_EUNSUPPORTED, "multislice_propagate: batch <= 65535");
    const int64_t rows = (int64_t)batch * w->n1;
    const int64_t npix = (int64_t)w->n1 * w->n2;
    const PropagatorMul prop = make_propagator(w, dz);
    float2* o = (float2*)out;
    if (w->chirp) {
        // WavePropagator.cpp:90-103; the wave stays chirped between the passes
        ChirpRows a = chirp_row_args(w, (const float2*)wave, o, batch, slices, slices_batch_stride);
        for (int sl = 0; sl < n_slices; ++sl) {
            a.V = slices + (int64_t)sl * npix;
            int rc = chirp_rows(w->p2.M, sl == 0 ? kChirpFwd : kChirpMid, a, w->tw, s);
            if (rc) return rc;
            a.in = o;
            rc = chirp_cols(w->p1.M, o, batch, w->n2, w->p1.tab(), prop, w->tw, s);
            if (rc) return rc;
        }
        return chirp_rows(w->p2.M, kChirpInv, a, w->tw, s);
    }
    // The columns that the propagator zeroes whole are written as zeros by the
    // first row pass and left alone from there on: a third of the column
    // pass's tiles and of the row pass's traffic (16 waves of 512^2 through 50
    // slices: 26.3 + 19.1 -> 21.4 + 15.5 us per slice).
    ColDead dead = dead_columns(prop);
    dead.skip_tiles = true;
    for (int sl = 0; sl < n_slices; ++sl) {
        const float2* src = sl == 0 ? (const float2*)wave : o;
        int rc = row_transmit_fft(w->n2, sl == 0, src, slices + (int64_t)sl * npix, o, rows,
                                  w->n1, slices_batch_stride, w->factor, dead, w->tw, s);
        if (rc) return rc;
        rc = col_prop(w->n1, o, w->n2, w->n2, npix, batch, prop, w->tw, s, dead);
        if (rc) return rc;
    }
    return row_fft(w->n2, true, o, o, rows, w->tw, s);
}

extern "C" int emsim_hip_lens_propagate(const emsim_hip_wave_propagator* w, const float* wave,
                                        float cs_mm, float defocus, float aperture, float* out,
                                        int batch, emsim_stream_t stream_) {
    hipStream_t s = (hipStream_t)stream_;
    if (!w || !wave || !out || batch < 1) return fail(EMSIM_HIP_EINVAL, "lens_propagate: bad arguments");
    if (batch > 65535) return fail(EMSIM_HIP_EUNSUPPORTED, "lens_propagate: batch <= 65535");
    if (w->chirp)
        return chirp_filter(w, (const float2*)wave, (float2*)out, nullptr, batch,
                            make_lens(w, cs_mm, defocus, aperture), s);
    const int64_t rows = (int64_t)batch * w->n1;
    const int64_t npix = (int64_t)w->n1 * w->n2;
    float2* o = (float2*)out;
    int rc = row_fft(w->n2, false, (const float2*)wave, o, rows, w->tw, s);
    if (!rc)
        rc = col_lens(w->n1, o, w->n2, w->n2, npix, batch, make_lens(w, cs_mm, defocus, aperture),
                      w->tw, s);
    if (!rc) rc = row_fft(w->n2, true, o, o, rows, w->tw, s);
    return rc;
}

extern "C" int emsim_hip_lens_intensity(const emsim_hip_wave_propagator* w, const float* wave,
                                        float cs_mm, float defocus, float aperture,
                                        float* scratch, float* image, int batch,
                                        emsim_stream_t stream_) {
    hipStream_t s = (hipStream_t)stream_;
    if (!w || !wave || !scratch || !image || batch < 1)
        return fail(EMSIM_HIP_EINVAL, "lens_intensity: bad arguments");
    if (batch > 65535) return fail(EMSIM_HIP_EUNSUPPORTED, "lens_intensity: batch <= 65535");
    const int64_t rows = (int64_t)batch * w->n1;
    const int64_t npix = (int64_t)w->n1 * w->n2;
    float2* o = (float2*)scratch;
    if (w->chirp)
        return chirp_filter(w, (const float2*)wave, o, image, batch,
                            make_lens(w, cs_mm, defocus, aperture), s);
    int rc = row_fft(w->n2, false, (const float2*)wave, o, rows, w->tw, s);
    if (!rc)
        rc = col_lens(w->n1, o, w->n2, w->n2, npix, batch, make_lens(w, cs_mm, defocus, aperture),
                      w->tw, s);
    if (!rc) rc = row_ifft_intensity(w->n2, o, image, rows, w->tw, s);
    return rc;
}

extern "C" int emsim_hip_intensity(const float* wave, float* out, int64_t n,
                                   emsim_stream_t stream_) {
    if (!wave || !out || n < 0) return fail(EMSIM_HIP_EINVAL, "intensity: bad arguments");
    if (n == 0) return EMSIM_HIP_OK;
    EMSIM_LAUNCH(0, k_intensity, dim3(grid_for(n, 256)), dim3(256), 0, (hipStream_t)stream_,
                       (const float2*)wave, out, n);
    return EMSIM_HIP_OK;
}

// ==========================================================================
// per-kernel timing
// ==========================================================================
extern "C" int emsim_hip_timing_enable(int on) {
    std::lock_guard<std::mutex> lock(g_timing_mutex);
    g_timing_on = on != 0;
    return EMSIM_HIP_OK;
}

// ==========================================================================
// one molecule in many orientations, on the device
// ==========================================================================
extern "C" size_t emsim_hip_orient_workspace_size(int batch) {
    return batch < 1 ? 0 : align_up(sizeof(uint32_t) * 6 * (size_t)batch);
}

namespace {
// The three launches of an orientation batch; bbox holds 6 keys per instance
// (device memory, cleared here by a fill kernel before use).
int orient_launch(const float* base, int64_t n_atoms, const float* rot, float c0x, float c0y,
                  float c0z, int batch, float* out, uint32_t* bbox, hipStream_t s) {
    EMSIM_LAUNCH(0, k_bbox_init, dim3((unsigned)ceil_div(6 * (int64_t)batch, 256)), dim3(256), 0,
                 s, bbox, batch);
    EMSIM_LAUNCH(0, k_orient, dim3((unsigned)ceil_div(n_atoms, 256), (unsigned)batch), dim3(256),
                 0, s, base, n_atoms, rot, c0x, c0y, c0z, out, bbox);
    const int64_t total = (int64_t)batch * n_atoms * 3;
    EMSIM_LAUNCH(0, k_recenter, dim3(grid_for(total, 256)), dim3(256), 0, s, out, n_atoms, batch,
                 (const uint32_t*)bbox);
    return EMSIM_HIP_OK;
}
}  // namespace

extern "C" int emsim_hip_orient_batch(const float* base, int64_t n_atoms, const float* rot,
                                      float c0x, float c0y, float c0z, int batch, float* out,
                                      void* workspace, size_t workspace_bytes,
                                      emsim_stream_t stream_) {
    if (!base || !rot || !out || !workspace || n_atoms < 1 || batch < 1)
        return fail(EMSIM_HIP_EINVAL, "orient_batch: bad arguments");
    if (batch > 65535) return fail(EMSIM_HIP_EUNSUPPORTED, "orient_batch: batch <= 65535");
    if (workspace_bytes < emsim_hip_orient_workspace_size(batch))
        return fail(EMSIM_HIP_EWORKSPACE, "orient_batch: workspace too small");
    return orient_launch(base, n_atoms, rot, c0x, c0y, c0z, batch, out, (uint32_t*)workspace,
                         (hipStream_t)stream_);
}

// --------------------------------------------------------------------------
// the same without a workspace argument, for callers that cannot allocate
// --------------------------------------------------------------------------
// The bounding-box keys live in a library-owned device array.  In host code
// `scratch` only names the symbol; its device address (one copy per GPU) comes
// from hipGetSymbolAddress, taken once per device with that device current.
static __device__ __align__(256) uint32_t scratch[6 * EMSIM_HIP_ORIENT_NOALLOC_MAX_BATCH];

namespace {
std::mutex g_scratch_mutex;
std::vector<uint32_t*> g_scratch_ptr;   // per device; null until first use

int scratch_address(uint32_t** out) {
    int dev = 0;
    EMSIM_HIP_CHECK(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if ((int)g_scratch_ptr.size() <= dev) g_scratch_ptr.resize(dev + 1, nullptr);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        const hipError_t err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (err != hipSuccess || !p)
            return fail(EMSIM_HIP_EDEVICE, "orient_batch_noalloc: hipGetSymbolAddress failed: %s",
                        hipGetErrorString(err));
        g_scratch_ptr[dev] = (uint32_t*)p;
    }
    *out = g_scratch_ptr[dev];
    return EMSIM_HIP_OK;
}
}  // namespace

extern "C" int emsim_hip_orient_batch_noalloc(const float* base, int64_t n_atoms,
                                              const float* rot, float c0x, float c0y, float c0z,
                                              int batch, float* out, emsim_stream_t stream_) {
    if (!base || !rot || !out || n_atoms < 1 || batch < 1)
        return fail(EMSIM_HIP_EINVAL, "orient_batch_noalloc: bad arguments");
    if (batch > EMSIM_HIP_ORIENT_NOALLOC_MAX_BATCH)
        return fail(EMSIM_HIP_EUNSUPPORTED,
                    "orient_batch_noalloc: batch %d exceeds the library's scratch (at most %d "
                    "orientations per call; use emsim_hip_orient_batch with a workspace)",
                    batch, EMSIM_HIP_ORIENT_NOALLOC_MAX_BATCH);
    uint32_t* bbox = nullptr;
    const int rc = scratch_address(&bbox);
    if (rc) return rc;
    return orient_launch(base, n_atoms, rot, c0x, c0y, c0z, batch, out, bbox,
                         (hipStream_t)stream_);
}

// ==========================================================================
// launch-shape knobs
// ==========================================================================
extern "C" int emsim_hip_tuning_set(const char* key, int value) {
    if (!key) return fail(EMSIM_HIP_EINVAL, "tuning_set: null key");
    if (std::strcmp(key, "row_items_per_block") == 0) {
        if (value < 0 || value > 64) return fail(EMSIM_HIP_EINVAL, "row_items_per_block in [0, 64]");
        g_row_items_per_block = value;
    } else if (std::strcmp(key, "col_tiles_per_block") == 0) {
        if (value < 0 || value > 32) return fail(EMSIM_HIP_EINVAL, "col_tiles_per_block in [0, 32]");
        g_col_tiles_per_block = value;
    } else if (std::strcmp(key, "col_shape") == 0) {
        if (value < 0 || value > 2) return fail(EMSIM_HIP_EINVAL, "col_shape in [0, 2]");
        g_col_shape = value;
    } else {
        return fail(EMSIM_HIP_EINVAL, "tuning_set: unknown key '%s'", key);
    }
    return EMSIM_HIP_OK;
}

extern "C" int emsim_hip_tuning_get(const char* key) {
    if (key && std::strcmp(key, "row_items_per_block") == 0) return g_row_items_per_block;
    if (key && std::strcmp(key, "col_tiles_per_block") == 0) return g_col_tiles_per_block;
    if (key && std::strcmp(key, "col_shape") == 0) return g_col_shape;
    return fail(EMSIM_HIP_EINVAL, "tuning_get: unknown key");
}

extern "C" int emsim_hip_timing_collect(char* buf, size_t cap, size_t* needed) {
    struct Agg {
        std::string name;
        int n;
        long count;
        double total, lo, hi;
    };
    std::vector<Agg> aggs;
    std::vector<TimingRecord> recs;
    {
        std::lock_guard<std::mutex> lock(g_timing_mutex);
        recs.swap(g_timing_records);
    }
    int rc = EMSIM_HIP_OK;
    for (const TimingRecord& r : recs) {
        float ms = 0.f;
        hipError_t err = hipEventSynchronize(r.stop);
        if (err == hipSuccess) err = hipEventElapsedTime(&ms, r.start, r.stop);
        if (err != hipSuccess) {
            rc = fail(EMSIM_HIP_EDEVICE, "timing_collect: %s", hipGetErrorString(err));
            continue;
        }
        Agg* a = nullptr;
        for (Agg& x : aggs)
            if (x.n == r.n && x.name == r.name) a = &x;
        if (!a) {
            aggs.push_back({r.name, r.n, 0, 0.0, 1e30, 0.0});
            a = &aggs.back();
        }
        a->count += 1;
        a->total += ms;
        a->lo = ms < a->lo ? ms : a->lo;
        a->hi = ms > a->hi ? ms : a->hi;
    }
    {
        std::lock_guard<std::mutex> lock(g_timing_mutex);
        for (const TimingRecord& r : recs) {
            g_event_pool.push_back(r.start);
            g_event_pool.push_back(r.stop);
        }
    }
    std::string text;
    char line[256];
    for (const Agg& a : aggs) {
        snprintf(line, sizeof(line), "%s\t%d\t%ld\t%.6f\t%.6f\t%.6f\n", a.name.c_str(), a.n,
                 a.count, a.total, a.lo, a.hi);
        text += line;
    }
    if (needed) *needed = text.size() + 1;
    if (buf && cap > 0) {
        const size_t m = text.size() < cap - 1 ? text.size() : cap - 1;
        memcpy(buf, text.data(), m);
        buf[m] = '\0';
    }
    return rc;
}

// ==========================================================================
// fused batched path (kernels_fused.hpp)
// ==========================================================================
namespace {

template <int N>
int launch_spec_sparse(const uint32_t* row_start, const uint16_t* bucket, const float* sf,
                       const float* sft, float2* Y, int slice0, int n_sc, int n_slices,
                       int n_elems, int H, int ldh, int n2, int bandlimit, int band_r2,
                       float inv_npix, int batch, const int* order, const WaterPlanes& wp,
                       const float2* tw, hipStream_t s) {
    using Cfg = SpecCfg<N>;
    if (H != n2 / 2 + 1 || n2 < 2 || ldh < H + n_elems)
        return fail(EMSIM_HIP_EINVAL, "spectrum: needs H = n2/2 + 1, n2 >= 2, ldh >= H + n_elems");
    // with spec_pack(N), column n2/2 is carried by column 0
    const int cols = spec_pack(N) ? n2 / 2 : H;
    const int64_t blocks = ceil_div(cols, Cfg::C) * (int64_t)batch * n_sc;
    if (blocks >= ((int64_t)1 << 31))
        return fail(EMSIM_HIP_EINVAL, "spectrum: %lld blocks, at most 2^31 - 1", (long long)blocks);
    if (!sft) return fail(EMSIM_HIP_EINVAL, "spectrum: no tile-major form-factor table");
    if (wp.X)
        EMSIM_LAUNCH(N, (k_spec_sparse<N, true>), dim3((unsigned)blocks), dim3(Cfg::BLOCK), 0, s,
                     row_start, bucket, sf, sft, Y, slice0, n_sc, n_slices, n_elems, H, ldh, n2,
                     batch, bandlimit, band_r2, inv_npix, order, wp, tw);
    else
        EMSIM_LAUNCH(N, (k_spec_sparse<N, false>), dim3((unsigned)blocks), dim3(Cfg::BLOCK), 0, s,
                     row_start, bucket, sf, sft, Y, slice0, n_sc, n_slices, n_elems, H, ldh, n2,
                     batch, bandlimit, band_r2, inv_npix, order, wp, tw);
    return EMSIM_HIP_OK;
}

// Rows dealt out evenly over one round of resident blocks, as in pass A.
template <int N>
int launch_water_rows(const WaterRows& a, int n_sc, const float2* tw, hipStream_t s) {
    static int resident_cache[64];
    const int64_t resident =
        resident_blocks(k_water_rows<N>, RowCfg<N>::BLOCK, resident_cache);
    const int64_t n_rows = (int64_t)n_sc * a.batch * a.n1, groups = ceil_div(n_rows, RowCfg<N>::G);
    if (groups <= 0) return EMSIM_HIP_OK;
    int64_t blocks = resident > 0 ? resident : 2048;
    if (blocks > groups) blocks = groups;
    const RunSched sched{(int)(groups / blocks), (int)(groups % blocks)};
    EMSIM_LAUNCH(N, (k_water_rows<N>), dim3((unsigned)blocks), dim3(RowCfg<N>::BLOCK), 0, s, a,
                 n_rows, sched, tw);
    return EMSIM_HIP_OK;
}

// vout (nullable) receives the slice's potential, (B, n_slices, n1, N)
template <int N>
int launch_slice_pass_a(bool first, const float2* Y, float2* wave, int64_t n_pairs, int ldh,
                        float psi0, float factor, float* vout, int slice, int n_slices, int n1,
                        ColDead cd, const float2* tw, hipStream_t s) {
    // one round of resident blocks: pass A is latency-bound, and a partial
    // second round (or a grid below the resident count) leaves SIMDs idle
    // The row-pair groups are dealt out evenly over one round of resident
    // waves (RunSched), so every SIMD ends up with about the same number of
    // pairs; the rows-per-block knob instead fixes the blocks' count.
    static int resident_cache[64];
    const int64_t resident =
        resident_blocks(k_slice_pass_a<N, false>, RowCfg<N>::BLOCK, resident_cache);
    const int64_t groups = ceil_div(n_pairs, RowCfg<N>::G);
    if (groups <= 0) return EMSIM_HIP_OK;
    int64_t blocks;
    if (g_row_items_per_block > 0) blocks = ceil_div(groups, g_row_items_per_block);
    else if (resident > 0) blocks = groups < resident ? groups : resident;
    else blocks = ceil_div(groups, rows_per_block(groups));
    const RunSched sched{(int)(groups / blocks), (int)(groups % blocks)};
    const dim3 grid((unsigned)blocks);
    const dim3 block(RowCfg<N>::BLOCK);
    const int64_t plane = (int64_t)n1 * N;
    if (first)
        EMSIM_LAUNCH(N, (k_slice_pass_a<N, true>), grid, block, 0, s,
                     (OpSlicePassA<N, true>{Y, wave, ldh, psi0, factor, vout, n_slices * plane,
                                            slice * plane, n1, cd.lo, cd.hi}),
                     n_pairs, sched, tw);
    else
        EMSIM_LAUNCH(N, (k_slice_pass_a<N, false>), grid, block, 0, s,
                     (OpSlicePassA<N, false>{Y, wave, ldh, psi0, factor, vout, n_slices * plane,
                                             slice * plane, n1, cd.lo, cd.hi}),
                     n_pairs, sched, tw);
    return EMSIM_HIP_OK;
}

// The transmission functions of n_sc slices, and one slice's wave rows through
// them (pass A in two kernels).
template <int N>
int launch_phase_rows(const float2* Y, float2* phase, int n_sc, int batch, int n1, int ldh,
                      float factor, float* vout, int slice0, int n_slices, const float2* tw,
                      hipStream_t s) {
    static int resident_cache[64];
    const int64_t n_pairs = (int64_t)n_sc * batch * (n1 / 2), plane = (int64_t)n1 * N;
    int rpw;
    dim3 grid;
    row_grid<N>(n_pairs, rpw, grid,
                resident_blocks(k_phase_rows<N>, RowCfg<N>::BLOCK, resident_cache));
    EMSIM_LAUNCH(N, (k_phase_rows<N>), grid, dim3(RowCfg<N>::BLOCK), 0, s,
                 (OpPhaseRows<N>{Y, phase, ldh, factor, vout, n_slices * plane, slice0 * plane, n1,
                                 batch}),
                 n_pairs, rpw, tw);
    return EMSIM_HIP_OK;
}
template <int N>
int launch_phase_apply(bool first, const float2* phase, float2* wave, int64_t rows, float psi0,
                       ColDead cd, const float2* tw, hipStream_t s) {
    static int resident_cache[64];
    int rpw;
    dim3 grid;
    row_grid<N>(rows, rpw, grid,
                resident_blocks(k_phase_apply<N, false>, RowCfg<N>::BLOCK, resident_cache));
    const dim3 block(RowCfg<N>::BLOCK);
    if (first)
        EMSIM_LAUNCH(N, (k_phase_apply<N, true>), grid, block, 0, s,
                     (OpPhaseApply<N, true>{phase, wave, psi0, cd.lo, cd.hi}), rows, rpw, tw);
    else
        EMSIM_LAUNCH(N, (k_phase_apply<N, false>), grid, block, 0, s,
                     (OpPhaseApply<N, false>{phase, wave, psi0, cd.lo, cd.hi}), rows, rpw, tw);
    return EMSIM_HIP_OK;
}

template <int N>
int launch_col_lensprop(float2* data, int ld, int ncols, int64_t img_stride, int n_img,
                        LensPropMul mul, const float2* tw, hipStream_t s, ColDead cd) {
    return launch_col_mul_impl<N>(data, ld, ncols, img_stride, n_img, mul, tw, s, cd, true);
}

int spec_sparse(int n, const uint32_t* row_start, const uint16_t* bucket, const float* sf,
                const float* sft, float2* Y, int slice0, int n_sc, int n_slices, int n_elems,
                int H, int ldh, int n2, int bandlimit, int band_r2, float inv_npix, int batch,
                const int* order, const WaterPlanes& wp, const float2* tw, hipStream_t s) {
    EMSIM_DISPATCH(n, launch_spec_sparse, row_start, bucket, sf, sft, Y, slice0, n_sc, n_slices,
                   n_elems, H, ldh, n2, bandlimit, band_r2, inv_npix, batch, order, wp, tw, s);
}
int water_rows(int n, const WaterRows& a, int n_sc, const float2* tw, hipStream_t s) {
    EMSIM_DISPATCH(n, launch_water_rows, a, n_sc, tw, s);
}
int phase_rows(int n, const float2* Y, float2* phase, int n_sc, int batch, int n1, int ldh,
               float factor, float* vout, int slice0, int n_slices, const float2* tw,
               hipStream_t s) {
    EMSIM_DISPATCH(n, launch_phase_rows, Y, phase, n_sc, batch, n1, ldh, factor, vout, slice0,
                   n_slices, tw, s);
}
int phase_apply(int n, bool first, const float2* phase, float2* wave, int64_t rows, float psi0,
                ColDead cd, const float2* tw, hipStream_t s) {
    EMSIM_DISPATCH(n, launch_phase_apply, first, phase, wave, rows, psi0, cd, tw, s);
}
int slice_pass_a(int n, bool first, const float2* Y, float2* wave, int64_t n_pairs, int ldh,
                 float psi0, float factor, float* vout, int slice, int n_slices, int n1,
                 ColDead cd, const float2* tw, hipStream_t s) {
    EMSIM_DISPATCH(n, launch_slice_pass_a, first, Y, wave, n_pairs, ldh, psi0, factor, vout,
                   slice, n_slices, n1, cd, tw, s);
}
int col_lensprop(int n, float2* data, int ld, int ncols, int64_t img_stride, int n_img,
                 LensPropMul mul, const float2* tw, hipStream_t s, ColDead cd) {
    EMSIM_DISPATCH(n, launch_col_lensprop, data, ld, ncols, img_stride, n_img, mul, tw, s, cd);
}

// Pass A in two kernels (transmission functions of a chunk of slices, then
// per slice only the wave's transforms) for batches of at most this many
// pixels: below it the per-slice pass is one short round of waves and its
// chain of dependent transforms is the time (one 256^2 image of 45 slices
// 740 -> 580 us, eight 128^2 images of 50 slices 797 -> 625 us, two 512^2
// images 1,083 -> 1,020 us); above it the extra traffic costs more than the
// shorter chain saves (four 512^2 images 1,433 -> 1,500 us, 64 of 256^2
// 3,440 -> 4,190 us).
constexpr int64_t kSplitPixels = (int64_t)2 * 512 * 512;
bool fused_split(const emsim_hip_slice_builder* b, int batch) {
    return (int64_t)batch * b->n1 * b->n2 <= kSplitPixels;
}
// Slices whose half spectra (and, split, transmission functions) one launch
// builds.  The spectrum pass does not depend on the wave, so a small batch
// takes as many slices at once as fit kChunkBytes of planes -- most of the
// 256 MB cache behind the L2s, from which they are read back -- instead of
// one part-filled round of blocks per slice (one 256^2 image, 45 slices:
// 1,526 -> 740 us; 64 of 256^2 4,124 -> 3,440 us; 64 / 128 / 192 / 256 MB
// measured 6,145 / 5,478 / 5,352 / 5,424 us for 32 of 512^2 x 50).
// Planes that don't fit come back from HBM, but one launch of many rounds has
// one tail instead of one per slice, so larger batches take kMinChunk: 256
// images of 512^2 x 30 26.4 ms at one slice, 25.2 at eight.  From 512 to 2048
// rows the tail is worth it where not even two slices fit, or where blocks run
// long because a slice has kDenseRow atoms and more per row (64 of 512^2 x 4,
// 20 a row, at two slices 1.87 ms, four 1.83; x 8, 49 a row, 6.13 and at eight
// 5.97).  Otherwise the planes stay in the cache: 64 of 512^2 x 100, 0.8 a row,
// at two slices 17.35 ms, three 17.95, eight 17.65; with atoms in half those
// slices 13.17 and 14.03; x 20, 4 a row, 4.49 and 4.55; x 8, 10 a row, 2.38 and
// 2.39; four of 2048^2 x 40, 4 a row, at three slices 22.1, eight 22.4; x 12, 12
// a row, 8.09 and 8.06.  256 images of 256^2 x 40 measured 9.39 at two, 9.20 at
// eight, and one of 4096^2 x 20 13.42 and 13.12.
// A run of up to four slices whose planes all together take at most half as much
// again goes in one launch, which mostly still finds them in the cache (64 of
// 512^2 x 4, 11 a row, 1.63 ms in two launches, 1.59 in one; four of 2048^2 x 3
// 1.78 and 1.75).
// The minimum ends at kMaxChunkBytes: a batch whose single slice is as large
// takes one slice at a time and no more workspace than that (64 of 2048^2 x 8
// 68.7 ms, 76.1 at eight slices).
constexpr int64_t kChunkBytes = (int64_t)192 << 20;
constexpr int64_t kMinChunk = 8;
constexpr int64_t kMaxChunkBytes = (int64_t)2 << 30;
constexpr int64_t kDenseRow = 12;
int fused_chunk(const emsim_hip_slice_builder* b, int batch, int64_t n_atoms, bool water) {
    const int64_t rows = (int64_t)batch * b->n1;
    const int64_t per = rows * (fused_ld(b) + (fused_split(b, batch) ? b->n2 : 0) +
                                (water ? 2 * half_ld(b->H) : 0)) *
                        (int64_t)sizeof(float2);
    if (b->n_slices <= 4 && b->n_slices * per <= kChunkBytes / 2 * 3) return b->n_slices;
    int64_t c = std::max<int64_t>(kChunkBytes / per, 1);
    const bool dense = n_atoms / b->n_slices >= kDenseRow * rows;
    if (c < 2 || dense || b->n1 < 512 || b->n1 > 2048)
        c = std::max(c, std::min(kMinChunk, kMaxChunkBytes / per));
    return (int)std::min(c, (int64_t)b->n_slices);
}

struct FusedWorkspace {
    int chunk;        // slices per launch of the spectrum pass
    float2* phase;    // transmission functions (chunk, batch, n1, n2), or null
    int32_t* order;   // spectrum-pass molecule slots per slice, or null (identity)
    int64_t* mol_off;
    int64_t* elem_off;
    int32_t* atom_row;
    uint16_t* atom_y;
    uint16_t* bucket;
    uint32_t* row_count;
    uint32_t* row_start;
    uint32_t* block_sums;
    float2* Y;
    float2* wave;
    float2* carry;    // (batch): rounding rests of the waves' means (pass B)
    // water fill (emsim_hip_simulate_water): half spectra of the hydrogen and
    // oxygen rows (chunk, batch, 2, n1, half_ld(H)), per-molecule seeds
    float2* X;
    uint64_t* seeds;
    // molecules given as they come (emsim_hip_simulate_raw): per-atom element
    // indices and bounding-box keys (batch, 6)
    const uint8_t* atom_elem;
    uint32_t* bbox;
    int64_t max_mol_atoms;
    int64_t n_rows;
    size_t bytes;
};

// Water-fill parameters of a fused run (emsim_hip_simulate_water).
struct WaterFill {
    bool on = false;
    int idx_h = 0, idx_o = 0;
    float lam_o = 0.f, exp_o = 1.f, lam_h = 0.f, exp_h = 1.f;
};

FusedWorkspace fused_layout(const emsim_hip_slice_builder* b, int batch, int64_t n_atoms,
                            bool own_wave, char* base, bool water = false, bool raw = false) {
    FusedWorkspace w;
    w.chunk = fused_chunk(b, batch, n_atoms, water);
    w.n_rows = (int64_t)batch * b->n_slices * b->n_elems * b->n1;
    const int64_t n_scan = w.n_rows + 1;
    const int64_t n_blocks = ceil_div(n_scan, kScanTile);
    const int ldh = fused_ld(b);
    size_t off = 0;
    w.order = (int32_t*)(base + off);
    off += align_up(sizeof(int32_t) * (size_t)batch * b->n_slices);
    w.mol_off = (int64_t*)(base + off);    off += align_up(sizeof(int64_t) * (size_t)(batch + 1));
    w.elem_off = (int64_t*)(base + off);
    off += align_up(sizeof(int64_t) * (size_t)batch * (b->n_elems + 1));
    w.atom_row = (int32_t*)(base + off);   off += align_up(sizeof(int32_t) * (size_t)n_atoms);
    w.atom_y = (uint16_t*)(base + off);    off += align_up(sizeof(uint16_t) * (size_t)n_atoms);
    w.bucket = (uint16_t*)(base + off);    off += align_up(sizeof(uint16_t) * (size_t)n_atoms);
    w.row_count = (uint32_t*)(base + off); off += align_up(sizeof(uint32_t) * (size_t)n_scan);
    w.row_start = (uint32_t*)(base + off); off += align_up(sizeof(uint32_t) * (size_t)n_scan);
    w.block_sums = (uint32_t*)(base + off); off += align_up(sizeof(uint32_t) * (size_t)n_blocks);
    w.Y = (float2*)(base + off);
    off += align_up(sizeof(float2) * (size_t)w.chunk * batch * b->n1 * ldh);
    w.phase = nullptr;
    if (fused_split(b, batch)) {
        w.phase = (float2*)(base + off);
        off += align_up(sizeof(float2) * (size_t)w.chunk * batch * b->n1 * b->n2);
    }
    w.wave = nullptr;
    if (own_wave) {
        w.wave = (float2*)(base + off);
        off += align_up(sizeof(float2) * (size_t)batch * b->n1 * b->n2);
    }
    w.carry = (float2*)(base + off);
    off += align_up(sizeof(float2) * (size_t)batch);
    w.X = nullptr;
    w.seeds = nullptr;
    if (water) {
        w.X = (float2*)(base + off);
        off += align_up(sizeof(float2) * 2 * (size_t)w.chunk * batch * b->n1 * half_ld(b->H));
        w.seeds = (uint64_t*)(base + off); off += align_up(sizeof(uint64_t) * (size_t)batch);
    }
    w.atom_elem = nullptr;
    w.bbox = nullptr;
    w.max_mol_atoms = 0;
    if (raw) {
        w.bbox = (uint32_t*)(base + off);
        off += align_up(sizeof(uint32_t) * 6 * (size_t)batch);
    }
    w.bytes = off;
    return w;
}

int check_simulate(const emsim_hip_slice_builder* b, const emsim_hip_wave_propagator* w,
                   const float* coords, int64_t n_atoms, int batch, int symmetric_bandlimit,
                   const float* out, int mode) {
    if (!b || !w || !out || batch < 1 || n_atoms < 0 || (n_atoms > 0 && !coords) ||
        (mode != 0 && mode != 1))
        return fail(EMSIM_HIP_EINVAL, "simulate: bad arguments");
    if (w->n1 != b->n1 || w->n2 != b->n2)
        return fail(EMSIM_HIP_EINVAL, "simulate: builder grid %dx%d != propagator grid %dx%d",
                    b->n1, b->n2, w->n1, w->n2);
    if (b->chirp || w->chirp)
        return fail(EMSIM_HIP_EUNSUPPORTED,
                    "simulate: the batched fused path needs power-of-two lateral sizes (%dx%d); "
                    "other sizes run through the per-call API", b->n1, b->n2);
    if (symmetric_bandlimit && b->n1 != b->n2)
        return fail(EMSIM_HIP_EINVAL, "simulate: the symmetric band-limit needs a square grid");
    if (batch > 65535) return fail(EMSIM_HIP_EUNSUPPORTED, "simulate: batch <= 65535");
    if (n_atoms >= (int64_t)0x7fffffff)
        return fail(EMSIM_HIP_EUNSUPPORTED, "simulate: at most 2^31-1 atoms per call");
    const int64_t n_rows_total = (int64_t)batch * b->n_slices * b->n_elems * b->n1;
    if (n_rows_total >= (int64_t)0x7fffffff)
        return fail(EMSIM_HIP_EUNSUPPORTED, "simulate: batch * slices * elements * n1 too large");
    return EMSIM_HIP_OK;
}

int simulate_core(const emsim_hip_slice_builder* b, const emsim_hip_wave_propagator* w,
                  const float* coords, int64_t n_atoms, const FusedWorkspace& ws, int batch,
                  float psi0, float cs_mm, float defocus, float aperture, int symmetric_bandlimit,
                  float* out, float* slices_out, int mode, hipStream_t s,
                  const WaterFill& water = WaterFill{});

// Host-side offsets of emsim_hip_simulate: elem_off (batch, n_elems + 1).
int host_offsets(const emsim_hip_slice_builder* b, const int64_t* mol_off_host,
                 const int64_t* elem_counts_host, int batch, int64_t n_atoms,
                 std::vector<int64_t>& elem_off) {
    if (mol_off_host[0] != 0 || mol_off_host[batch] != n_atoms)
        return fail(EMSIM_HIP_EINVAL, "simulate: molecule offsets must run from 0 to n_atoms");
    elem_off.assign((size_t)batch * (b->n_elems + 1), 0);
    for (int m = 0; m < batch; ++m) {
        if (mol_off_host[m + 1] < mol_off_host[m])
            return fail(EMSIM_HIP_EINVAL, "simulate: molecule offsets must not decrease");
        int64_t o = mol_off_host[m];
        elem_off[(size_t)m * (b->n_elems + 1)] = o;
        for (int e = 0; e < b->n_elems; ++e) {
            const int64_t c = elem_counts_host[(size_t)m * b->n_elems + e];
            if (c < 0) return fail(EMSIM_HIP_EINVAL, "simulate: negative element count");
            o += c;
            elem_off[(size_t)m * (b->n_elems + 1) + e + 1] = o;
        }
        if (o > mol_off_host[m + 1])
            return fail(EMSIM_HIP_EINVAL, "simulate: molecule %d's element counts exceed its atoms",
                        m);
    }
    return EMSIM_HIP_OK;
}

}  // namespace

extern "C" size_t emsim_hip_simulate_workspace_size(const emsim_hip_slice_builder* b, int batch,
                                                    int64_t n_atoms, int mode) {
    if (!b || batch < 1 || n_atoms < 0) return 0;
    return fused_layout(b, batch, n_atoms, mode == 0, nullptr).bytes;
}

extern "C" int emsim_hip_simulate(const emsim_hip_slice_builder* b,
                                  const emsim_hip_wave_propagator* w, const float* coords,
                                  int64_t n_atoms, const int64_t* mol_off_host,
                                  const int64_t* elem_counts_host, int batch, float psi0,
                                  float cs_mm, float defocus, float aperture,
                                  int symmetric_bandlimit, float* out, float* slices_out,
                                  int mode, void* workspace, size_t workspace_bytes,
                                  emsim_stream_t stream_) {
    hipStream_t s = (hipStream_t)stream_;
    if (!mol_off_host || !elem_counts_host) return fail(EMSIM_HIP_EINVAL, "simulate: null offsets");
    const int check = check_simulate(b, w, coords, n_atoms, batch, symmetric_bandlimit, out, mode);
    if (check) return check;
    std::vector<int64_t> elem_off;
    const int rc = host_offsets(b, mol_off_host, elem_counts_host, batch, n_atoms, elem_off);
    if (rc) return rc;
    FusedWorkspace ws = fused_layout(b, batch, n_atoms, mode == 0, (char*)workspace);
    if (!workspace || workspace_bytes < ws.bytes)
        return fail(EMSIM_HIP_EWORKSPACE, "simulate: workspace needs %zu bytes", ws.bytes);
    EMSIM_HIP_CHECK(hipMemcpyAsync(ws.mol_off, mol_off_host, sizeof(int64_t) * (batch + 1),
                                   hipMemcpyHostToDevice, s));
    EMSIM_HIP_CHECK(hipMemcpyAsync(ws.elem_off, elem_off.data(), sizeof(int64_t) * elem_off.size(),
                                   hipMemcpyHostToDevice, s));
    return simulate_core(b, w, coords, n_atoms, ws, batch, psi0, cs_mm, defocus, aperture,
                         symmetric_bandlimit, out, slices_out, mode, s);
}

extern "C" int emsim_hip_simulate_dev(const emsim_hip_slice_builder* b,
                                      const emsim_hip_wave_propagator* w, const float* coords,
                                      int64_t n_atoms, const int64_t* mol_off_dev,
                                      const int64_t* elem_off_dev, int batch, float psi0,
                                      float cs_mm, float defocus, float aperture,
                                      int symmetric_bandlimit, float* out, float* slices_out,
                                      int mode, void* workspace, size_t workspace_bytes,
                                      emsim_stream_t stream_) {
    if (!mol_off_dev || !elem_off_dev) return fail(EMSIM_HIP_EINVAL, "simulate_dev: null offsets");
    int rc = check_simulate(b, w, coords, n_atoms, batch, symmetric_bandlimit, out, mode);
    if (rc) return rc;
    FusedWorkspace ws = fused_layout(b, batch, n_atoms, mode == 0, (char*)workspace);
    if (!workspace || workspace_bytes < ws.bytes)
        return fail(EMSIM_HIP_EWORKSPACE, "simulate: workspace needs %zu bytes", ws.bytes);
    ws.mol_off = const_cast<int64_t*>(mol_off_dev);
    ws.elem_off = const_cast<int64_t*>(elem_off_dev);
    return simulate_core(b, w, coords, n_atoms, ws, batch, psi0, cs_mm, defocus, aperture,
                         symmetric_bandlimit, out, slices_out, mode, (hipStream_t)stream_);
}

extern "C" size_t emsim_hip_simulate_water_workspace_size(const emsim_hip_slice_builder* b,
                                                          int batch, int64_t n_atoms, int mode) {
    if (!b || batch < 1 || n_atoms < 0) return 0;
    return fused_layout(b, batch, n_atoms, mode == 0, nullptr, true).bytes;
}

extern "C" int emsim_hip_simulate_water(const emsim_hip_slice_builder* b,
                                        const emsim_hip_wave_propagator* w, const float* coords,
                                        int64_t n_atoms, const int64_t* mol_off_host,
                                        const int64_t* elem_counts_host, int batch, float psi0,
                                        float cs_mm, float defocus, float aperture,
                                        int symmetric_bandlimit, int idx_h, int idx_o,
                                        double voxel_water, const uint64_t* seeds_host,
                                        float* out, float* slices_out, int mode, void* workspace,
                                        size_t workspace_bytes, emsim_stream_t stream_) {
    hipStream_t s = (hipStream_t)stream_;
    if (!mol_off_host || !elem_counts_host || !seeds_host)
        return fail(EMSIM_HIP_EINVAL, "simulate_water: null offsets or seeds");
    int rc = check_simulate(b, w, coords, n_atoms, batch, symmetric_bandlimit, out, mode);
    if (rc) return rc;
    if (b->one_slice)
        return fail(EMSIM_HIP_EINVAL, "simulate_water: needs a multi-slice builder (the "
                    "one-slice path adds no water)");
    if (idx_h < 0 || idx_o < 0 || idx_h >= b->n_elems || idx_o >= b->n_elems || idx_h == idx_o ||
        !(voxel_water >= 0))
        return fail(EMSIM_HIP_EINVAL, "simulate_water: bad water arguments");
    // the range this entry point has always taken (and is tested over); no kernel
    // of the path needs it any more
    if ((size_t)b->n_elems * b->n2 * sizeof(float) > 64 * 1024)
        return fail(EMSIM_HIP_EUNSUPPORTED, "simulate_water: n_elems * n2 <= 16384");
    std::vector<int64_t> elem_off;
    rc = host_offsets(b, mol_off_host, elem_counts_host, batch, n_atoms, elem_off);
    if (rc) return rc;
    FusedWorkspace ws = fused_layout(b, batch, n_atoms, mode == 0, (char*)workspace, true);
    if (!workspace || workspace_bytes < ws.bytes)
        return fail(EMSIM_HIP_EWORKSPACE, "simulate_water: workspace needs %zu bytes", ws.bytes);
    EMSIM_HIP_CHECK(hipMemcpyAsync(ws.mol_off, mol_off_host, sizeof(int64_t) * (batch + 1),
                                   hipMemcpyHostToDevice, s));
    EMSIM_HIP_CHECK(hipMemcpyAsync(ws.elem_off, elem_off.data(), sizeof(int64_t) * elem_off.size(),
                                   hipMemcpyHostToDevice, s));
    EMSIM_HIP_CHECK(hipMemcpyAsync(ws.seeds, seeds_host, sizeof(uint64_t) * batch,
                                   hipMemcpyHostToDevice, s));
    WaterFill wf;
    wf.on = true;
    wf.idx_h = idx_h;
    wf.idx_o = idx_o;
    // the same float32 constants as emsim_hip_add_water
    wf.lam_o = (float)voxel_water;
    wf.lam_h = (float)(2.0 * voxel_water);
    wf.exp_o = (float)std::exp(-voxel_water);
    wf.exp_h = (float)std::exp(-2.0 * voxel_water);
    return simulate_core(b, w, coords, n_atoms, ws, batch, psi0, cs_mm, defocus, aperture,
                         symmetric_bandlimit, out, slices_out, mode, s, wf);
}

extern "C" size_t emsim_hip_simulate_raw_workspace_size(const emsim_hip_slice_builder* b,
                                                        int batch, int64_t n_atoms, int mode) {
    if (!b || batch < 1 || n_atoms < 0) return 0;
    return fused_layout(b, batch, n_atoms, mode == 0, nullptr, false, true).bytes;
}

extern "C" int emsim_hip_simulate_raw(const emsim_hip_slice_builder* b,
                                      const emsim_hip_wave_propagator* w, const float* coords,
                                      const uint8_t* elem, int64_t n_atoms,
                                      const int64_t* mol_off_host, int batch, float psi0,
                                      float cs_mm, float defocus, float aperture,
                                      int symmetric_bandlimit, float* out, float* slices_out,
                                      int mode, void* workspace, size_t workspace_bytes,
                                      emsim_stream_t stream_) {
    hipStream_t s = (hipStream_t)stream_;
    if (!mol_off_host || (n_atoms > 0 && !elem))
        return fail(EMSIM_HIP_EINVAL, "simulate_raw: null offsets or element indices");
    int rc = check_simulate(b, w, coords, n_atoms, batch, symmetric_bandlimit, out, mode);
    if (rc) return rc;
    if (mol_off_host[0] != 0 || mol_off_host[batch] != n_atoms)
        return fail(EMSIM_HIP_EINVAL, "simulate_raw: molecule offsets must run from 0 to n_atoms");
    int64_t max_atoms = 0;
    for (int m = 0; m < batch; ++m) {
        const int64_t len = mol_off_host[m + 1] - mol_off_host[m];
        if (len < 0) return fail(EMSIM_HIP_EINVAL, "simulate_raw: offsets must not decrease");
        if (len > max_atoms) max_atoms = len;
    }
    FusedWorkspace ws = fused_layout(b, batch, n_atoms, mode == 0, (char*)workspace, false, true);
    if (!workspace || workspace_bytes < ws.bytes)
        return fail(EMSIM_HIP_EWORKSPACE, "simulate_raw: workspace needs %zu bytes", ws.bytes);
    ws.atom_elem = elem;
    ws.max_mol_atoms = max_atoms;
    EMSIM_HIP_CHECK(hipMemcpyAsync(ws.mol_off, mol_off_host, sizeof(int64_t) * (batch + 1),
                                   hipMemcpyHostToDevice, s));
    return simulate_core(b, w, coords, n_atoms, ws, batch, psi0, cs_mm, defocus, aperture,
                         symmetric_bandlimit, out, slices_out, mode, s);
}

namespace {

// One molecule of emsim_hip_pack_raw; false if an element is outside the list.
bool pack_molecule(const float* c, const int64_t* z, int64_t n, const uint8_t* lut,
                   int64_t lut_size, float* c_out, uint8_t* e_out, float* extent) {
    std::memcpy(c_out, c, sizeof(float) * 3 * (size_t)n);
    bool ok = true;
    for (int64_t i = 0; i < n; ++i) {
        const uint8_t e = (uint64_t)z[i] < (uint64_t)lut_size ? lut[z[i]] : 255;
        ok = ok && e != 255;
        e_out[i] = e;
    }
    if (!extent) return ok;
    *extent = 0.f;
    if (n == 0) return ok;
    float lo = c[0], hi = c[0];
    bool nan = false;
    for (int64_t i = 0; i < n; ++i) {
        const float v = c[3 * i];
        nan = nan || v != v;
        lo = v < lo ? v : lo;
        hi = v > hi ? v : hi;
    }
    // adding the shift is monotonic, so the centred extremes are the shifted ones
    const float span = hi - lo, half = span / 2.0f;
    const float shift = -lo - half;
    const float zhi = hi + shift, zlo = lo + shift;
    *extent = nan ? NAN : zhi - zlo;
    return ok;
}

}  // namespace

extern "C" int emsim_hip_pack_raw(int n_mols, const float* const* coords, const int64_t* const* z,
                                  const int64_t* mol_off, const uint8_t* lut, int64_t lut_size,
                                  float* coords_out, uint8_t* elem_out, float* extent,
                                  int max_threads, int* bad) {
    if (n_mols < 1 || !coords || !z || !mol_off || !lut || lut_size < 1 || !bad)
        return fail(EMSIM_HIP_EINVAL, "pack_raw: bad arguments");
    for (int m = 0; m < n_mols; ++m) {
        const int64_t n = mol_off[m + 1] - mol_off[m];
        if (n < 0 || (n > 0 && (!coords[m] || !z[m] || !coords_out || !elem_out)))
            return fail(EMSIM_HIP_EINVAL, "pack_raw: molecule %d has no data", m);
    }
    std::atomic<int> next{0}, first_bad{n_mols};
    auto work = [&]() {
        for (int m; (m = next.fetch_add(1)) < n_mols;) {
            const int64_t o = mol_off[m];
            if (pack_molecule(coords[m], z[m], mol_off[m + 1] - o, lut, lut_size,
                              coords_out + 3 * o, elem_out + o, extent ? extent + m : nullptr))
                continue;
            int seen = first_bad.load();
            while (m < seen && !first_bad.compare_exchange_weak(seen, m)) {
            }
        }
    };
    // a thread per 100,000 atoms (about 150 us of work against 20 us to start one)
    const int64_t want = (mol_off[n_mols] - mol_off[0]) / 100000;
    const int extra = (int)std::min<int64_t>({want, (int64_t)max_threads - 1, (int64_t)n_mols - 1, 63});
    std::thread pool[63];
    int started = 0;
    try {
        for (; started < extra; ++started) pool[started] = std::thread(work);
    } catch (const std::exception&) {   // no thread or no memory for one: the caller's own does the rest
    }
    work();
    for (int t = 0; t < started; ++t) pool[t].join();
    *bad = first_bad.load() < n_mols ? first_bad.load() : -1;
    return EMSIM_HIP_OK;
}

namespace {

int simulate_core(const emsim_hip_slice_builder* b, const emsim_hip_wave_propagator* w,
                  const float* coords, int64_t n_atoms, const FusedWorkspace& ws, int batch,
                  float psi0, float cs_mm, float defocus, float aperture, int symmetric_bandlimit,
                  float* out, float* slices_out, int mode, hipStream_t s, const WaterFill& water) {
    int rc = EMSIM_HIP_OK;
    BatchGeom bg;
    bg.g.e0 = b->edges;
    bg.g.e1 = b->edges + (b->n_slices + 1);
    bg.g.e2 = bg.g.e1 + (b->n1 + 1);
    bg.g.n0 = b->n_slices;
    bg.g.n1 = b->n1;
    bg.g.n2 = b->n2;
    bg.g.last0 = b->last_exact[0];
    bg.g.last1 = b->last_exact[1];
    bg.g.last2 = b->last_exact[2];
    bg.g.inv0 = b->inv_d[0];
    bg.g.inv1 = b->inv_d[1];
    bg.g.inv2 = b->inv_d[2];
    bg.g.one_slice = b->one_slice;
    bg.g.tile_rows = 1;
    bg.g.tiles_per_plane = b->n1;
    bg.n_elems = b->n_elems;
    bg.batch = batch;

    // 1. bucket the atoms by (molecule, slice, element, row)
    const int64_t n_scan = ws.n_rows + 1;
    const int64_t n_blocks = ceil_div(n_scan, kScanTile);
    EMSIM_LAUNCH(0, k_fill_u32, dim3(grid_for(n_scan, 256)), dim3(256), 0, s, ws.row_count,
                 n_scan, 0u);
    if (ws.atom_elem && n_atoms > 0) {
        // molecules as they come: their bounding boxes, for centring on the fly
        EMSIM_LAUNCH(0, k_bbox_init, dim3((unsigned)ceil_div(6 * (int64_t)batch, 256)), dim3(256),
                     0, s, ws.bbox, batch);
        const int64_t chunks = ceil_div(ws.max_mol_atoms > 0 ? ws.max_mol_atoms : 1,
                                        256 * kBoxPerThread);
        EMSIM_LAUNCH(0, k_mol_bbox, dim3((unsigned)chunks, (unsigned)batch), dim3(256), 0, s,
                     coords, (const int64_t*)ws.mol_off, ws.atom_elem, b->n_elems, ws.bbox);
    }
    if (n_atoms > 0)
        EMSIM_LAUNCH(0, k_csr_classify, dim3(grid_for(n_atoms, 256)), dim3(256), 0, s, coords,
                     n_atoms, ws.mol_off, ws.elem_off, bg, ws.atom_row, ws.atom_y, ws.row_count,
                     ws.atom_elem, (const uint32_t*)ws.bbox);
    EMSIM_LAUNCH(0, k_scan_tiles, dim3((unsigned)n_blocks), dim3(kScanBlock), 0, s, ws.row_count,
                 ws.row_start, n_scan, ws.block_sums);
    EMSIM_LAUNCH(0, k_scan_sums, dim3(1), dim3(kScanBlock), 0, s, ws.block_sums, n_blocks);
    EMSIM_LAUNCH(0, k_scan_add, dim3((unsigned)n_blocks), dim3(kScanBlock), 0, s, ws.row_start,
                 n_scan, ws.block_sums);
    if (n_atoms > 0) {
        EMSIM_LAUNCH(0, k_csr_scatter, dim3(grid_for(n_atoms, 256)), dim3(256), 0, s, n_atoms,
                     ws.atom_row, ws.atom_y, ws.row_start, ws.row_count, ws.bucket);
        // a fixed order of every row's atoms for the float row sums
        EMSIM_LAUNCH(0, k_csr_sort_rows, dim3((unsigned)ceil_div(ws.n_rows, kSortRows)),
                     dim3(kSortRows), sizeof(uint16_t) * (size_t)sort_waves(b->n2) * b->n2, s, ws.n_rows,
                     b->n2, ws.row_start, ws.bucket);
    }
    // per-slice molecule order of the spectrum pass (identity beyond one
    // block's worth of molecules)
    const int32_t* order = nullptr;
    if (batch > 1 && batch <= 1024) {
        EMSIM_LAUNCH(0, k_slice_order, dim3((unsigned)b->n_slices), dim3((unsigned)batch), 0, s,
                     ws.row_start, b->n_slices, b->n_elems, b->n1, batch, ws.order);
        order = ws.order;
    }

    // 2. the slices
    float2* wave = mode == 0 ? ws.wave : (float2*)out;
    const int ldh = fused_ld(b);
    const int r = (b->n1 < b->n2 ? b->n1 : b->n2) / 2;
    const float inv_npix = 1.0f / (float)((int64_t)b->n1 * b->n2);
    const int64_t npix = (int64_t)b->n1 * b->n2;
    const int64_t rows = (int64_t)batch * b->n1;
    // a one-slice builder is the weak-phase-object path (emsim/pipe.py:57-64):
    // its slice is followed by singleslice_propagate(dz = 0), the mask alone
    const PropagatorMul prop = make_propagator(w, b->one_slice ? 0.f : (float)b->dz);
    // Columns the propagator zeroes whole are left out between the passes:
    // the wave buffer starts as zeros, pass A never stores into them and
    // pass B skips the tiles that hold only such columns (zeros from the
    // others).  The last pass B runs every tile.
    ColDead dead = dead_columns(prop);
    dead.skip_tiles = true;
    dead.carry = ws.carry;
    ColDead dead_last = dead;
    dead_last.skip_tiles = false;
    if (dead.lo <= dead.hi) {
        const int64_t n_wave = (int64_t)batch * npix;
        EMSIM_LAUNCH(0, k_fill_complex, dim3(grid_for(n_wave, 256)), dim3(256), 0, s, wave,
                     n_wave, 0.f);
    }
    for (int sl = 0; sl < b->n_slices; ++sl) {
        const bool last = sl == b->n_slices - 1;
        dead.carry_first = dead_last.carry_first = sl == 0;
        const int sc = sl % ws.chunk;   // plane of this slice in its chunk
        if (sc == 0) {
            const int n_sc = std::min(ws.chunk, b->n_slices - sl);
            WaterPlanes wp{nullptr, 0, 0, 0};
            if (water.on) {
                wp = WaterPlanes{ws.X, water.idx_h, water.idx_o, half_ld(b->H)};
                rc = water_rows(b->n2,
                                WaterRows{ws.row_start, ws.bucket, ws.seeds, ws.X, sl, b->n_slices,
                                          b->n_elems, b->n1, batch, wp.ldx, water.idx_h,
                                          water.idx_o, water.lam_o, water.exp_o, water.lam_h,
                                          water.exp_h},
                                n_sc, b->tw, s);
                if (rc) return rc;
            }
            rc = spec_sparse(b->n1, ws.row_start, ws.bucket, b->sf, b->sf_tiles, ws.Y, sl, n_sc,
                             b->n_slices, b->n_elems, b->H, ldh, b->n2, symmetric_bandlimit ? 1 : 0,
                             r * r, inv_npix, batch, order, wp, b->tw, s);
            if (!rc && ws.phase)
                rc = phase_rows(b->n2, ws.Y, ws.phase, n_sc, batch, b->n1, ldh, w->factor,
                                slices_out, sl, b->n_slices, b->tw, s);
            if (rc) return rc;
        }
        if (ws.phase)
            rc = phase_apply(b->n2, sl == 0, ws.phase + sc * batch * npix, wave, rows, psi0, dead,
                             b->tw, s);
        else
            rc = slice_pass_a(b->n2, sl == 0, ws.Y + (int64_t)sc * rows * ldh, wave, rows / 2, ldh,
                              psi0, w->factor, slices_out, sl, b->n_slices, b->n1, dead, b->tw, s);
        if (rc) return rc;
        if (mode == 0 && last) {
            LensPropMul lp;
            lp.p = prop;
            lp.l = make_lens(w, cs_mm, defocus, aperture);
            rc = col_lensprop(b->n1, wave, b->n2, b->n2, npix, batch, lp, b->tw, s, dead_last);
        } else {
            rc = col_prop(b->n1, wave, b->n2, b->n2, npix, batch, prop, b->tw, s,
                          last ? dead_last : dead);
        }
        if (rc) return rc;
    }
    // 3. back to real space: |psi|^2 of the image wave, or the exit wave
    if (mode == 0) return row_ifft_intensity(b->n2, wave, out, rows, b->tw, s);
    return row_fft(b->n2, true, wave, wave, rows, b->tw, s);
}

}  // namespace
