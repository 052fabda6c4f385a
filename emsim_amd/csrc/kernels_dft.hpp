// DFTs of any length n (8 <= n <= 2048) by Bluestein's chirp-z algorithm on
// the power-of-two FFT core, for the reference-shaped API calls at lateral
// sizes that are not powers of two (the reference's FFTW plans take any n,
// emsim/backend/fftw_ext/src/WavePropagator.cpp:25-33, SliceBuilder.cpp:41-55).
//
// With w = exp(-2 pi i / n), j k = (j^2 + k^2 - (k - j)^2) / 2 gives
//   X_k = sum_j x_j w^(j k) = c_k sum_j (x_j c_j) conj(c_(k-j)),
//   c_m = exp(-i pi m^2 / n),
// a convolution, done circularly at a power-of-two length M >= 2n - 1:
//   X = c . IFFT_M(FFT_M(x . c, zero-padded) . B),   B = FFT_M(b) / M,
// b_m = conj(c_m) at m and at M - m (0 <= m < n).  The inverse transform uses
// conj(c) in place of c; b is even, so its B is the conjugate.  c and B are
// computed on the host in float64 (m^2 reduced modulo 2n first) and rounded
// once (the 1/M is exact).
//
// A transform pair F^-1 (pointwise) F of the multislice recurrence is one
// kernel: both convolutions of a row (or column) run in registers and LDS, and
// the chirp factors between them are c conj(c) = 1, so they are left out.  The
// same holds across kernels: the factor c2[j] that ends a forward row transform
// meets the conj(c2[j]) that begins the next inverse one with only column
// operations between them, and c1[i] meets conj(c1[i]) with only row operations
// and the pointwise transmission between.  A wave therefore stays "chirped"
// from the first row pass to the last, which alone apply c1 c2 and its
// conjugate.
//
// Bound by the latency of a line's four dependent transforms for one image (a
// 150^2 slice: rows 5.5 us, columns 6.2 us, against 22 launches of 3-4 us when
// each line transform was five kernels through a line buffer), and by VALU and
// LDS exchanges for batches (24 waves of 400^2 through 20 slices: 49.6 ms
// before, 3.0 ms; a column tile per block without the runs and the prefetch
// 4.7 ms).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fft_lds.hpp"
#include "kernels_wave.hpp"

namespace emsim {

// One axis's tables: c (n), and the transformed convolution kernel B (M).
struct ChirpTab {
    const float2* c;
    const float2* b;
    int n;
};

// This thread's values t + m T of a length-M table.
template <int M, int EPT>
__device__ __forceinline__ void chirp_load_b(const float2* __restrict__ b, int t,
                                             float2 (&r)[EPT]) {
#pragma unroll
    for (int m = 0; m < EPT; ++m) r[m] = b[t + m * (M / EPT)];
}

// v <- IFFT_M(FFT_M(v) . b) (INV: conj(b), the inverse transform's) for the
// M/EPT threads of one line (every thread of the block calls it).  Inputs past n must be zero; n <= M/2, so the upper half
// of every thread's values always is.
template <int M, int EPT, bool INV, class TW>
__device__ __forceinline__ void chirp_conv(float2 (&v)[EPT], const float2 (&b)[EPT], float* re,
                                           float* im, int t, const TW& tw) {
    fft_n<M, EPT, false>(v, re, im, t, tw);
#pragma unroll
    for (int m = 0; m < EPT; ++m) v[m] = mul_tw<INV>(v[m], b[m]);
    fft_n<M, EPT, true>(v, re, im, t, tw);
}

// ---------------------------------------------------------------------------
// Row kernels: one row per group of M/8 threads, G rows side by side.  The
// rows of a wave (n long, n apart) belong to images of rows_per_img rows.
//   kChirpFwd:  real space in: [* exp(i factor V)] * c2[y] c1[x], forward
//   kChirpMid:  inverse, * exp(i factor V), forward (one slice's pass A)
//   kChirpInv:  inverse, * conj(c2[y] c1[x]): real space out
//   kChirpInt:  inverse, |.|^2 out (unit-modulus factors drop out)
// ---------------------------------------------------------------------------
enum ChirpRowMode { kChirpFwd = 0, kChirpMid = 1, kChirpInv = 2, kChirpInt = 3 };

struct ChirpRows {
    const float2* in;
    float2* out;
    float* image;           // kChirpInt
    const float* V;         // null: no transmission (kChirpFwd)
    int64_t v_img_stride;
    float factor;
    int64_t rows;
    int rows_per_img;
    ChirpTab row;           // along the row (length n)
    const float2* c1;       // the other axis's chirp, by row of the image
    int rpb;                // row groups per block
};

template <int M, int MODE>
__global__ __launch_bounds__(RowCfg<M>::BLOCK) void k_chirp_rows(ChirpRows a,
                                                                 const float2* __restrict__ tw) {
    using Cfg = RowCfg<M>;
    constexpr int EPT = Cfg::EPT, HALF = EPT / 2, T = Cfg::T;
    __shared__ float lds_re[Cfg::G * Cfg::WORDS];
    __shared__ float lds_im[Cfg::G * Cfg::WORDS];
    const int gi = row_in_block<T>();
    const int t = threadIdx.x % T;
    float* re = lds_re + gi * Cfg::WORDS;
    float* im = lds_im + gi * Cfg::WORDS;
    const int n = a.row.n;
    constexpr bool HAS_C = MODE == kChirpFwd || MODE == kChirpInv;
    constexpr bool HAS_V = MODE == kChirpFwd || MODE == kChirpMid;

    // the tables of this thread's positions, loaded once for the block's rows
    float2 b[EPT], c[HALF];
    chirp_load_b<M, EPT>(a.row.b, t, b);
    if constexpr (HAS_C) {
#pragma unroll
        for (int m = 0; m < HALF; ++m) c[m] = a.row.c[t + m * T < n ? t + m * T : n - 1];
    }
    TwCache<M, EPT> twc;
    twc.load(tw, t);

    // Rows first + r G of this block's run; the next row's values are loaded
    // before this one is transformed, from indices clamped into range (ok
    // guards the stores), so no load waits behind a branch.
    const int64_t first = (int64_t)blockIdx.x * a.rpb * Cfg::G + gi;
    struct Regs {
        float2 v[HALF];
        float pot[HALF];
        float2 cx;
    } cur, nxt;
    auto load = [&](int64_t row0, Regs& g) __attribute__((always_inline)) {
        const int64_t row = row0 < a.rows ? row0 : a.rows - 1;
        const int64_t img = row / a.rows_per_img;
        const int x = (int)(row - img * a.rows_per_img);
        const float2* src = a.in + row * n;
        const float* vrow = HAS_V && a.V ? a.V + img * a.v_img_stride + (int64_t)x * n : nullptr;
#pragma unroll
        for (int m = 0; m < HALF; ++m) {
            const int k = t + m * T, kc = k < n ? k : n - 1;
            g.v[m] = src[kc];
            g.pot[m] = vrow ? vrow[kc] : 0.f;
        }
        if constexpr (HAS_C) g.cx = a.c1[x];
    };
    load(first, cur);
    for (int r = 0; r < a.rpb; ++r) {
        const int64_t row = first + (int64_t)r * Cfg::G;
        if (r + 1 < a.rpb) load(row + Cfg::G, nxt);
        float2 v[EPT];
#pragma unroll
        for (int m = 0; m < HALF; ++m) {
            v[m] = t + m * T < n ? cur.v[m] : make_float2(0.f, 0.f);
            v[m + HALF] = make_float2(0.f, 0.f);
        }
        if constexpr (MODE != kChirpFwd) chirp_conv<M, EPT, true>(v, b, re, im, t, twc);
        if constexpr (HAS_V) {
#pragma unroll
            for (int m = 0; m < HALF; ++m) {
                if (MODE == kChirpMid || a.V) {
                    float s, co;
                    fast_sincos(__fmul_rn(cur.pot[m], a.factor), &s, &co);
                    v[m] = cmul(v[m], make_float2(co, s));
                }
                if constexpr (MODE == kChirpFwd) v[m] = cmul(v[m], cmul(c[m], cur.cx));
                if (t + m * T >= n) v[m] = make_float2(0.f, 0.f);
                v[m + HALF] = make_float2(0.f, 0.f);
            }
            chirp_conv<M, EPT, false>(v, b, re, im, t, twc);
        }
        if (row < a.rows) {
#pragma unroll
            for (int m = 0; m < HALF; ++m) {
                const int k = t + m * T;
                if (k >= n) continue;
                if constexpr (MODE == kChirpInt) a.image[row * n + k] = norm2(v[m]);
                else if constexpr (MODE == kChirpInv)
                    a.out[row * n + k] = mul_tw<true>(v[m], cmul(c[m], cur.cx));
                else a.out[row * n + k] = v[m];
            }
        }
        cur = nxt;
    }
}

// ---------------------------------------------------------------------------
// Column tiles: C adjacent columns per block, EPT values per thread.  Narrow
// tiles (a quarter of the columns) spread one image over more CUs.
// ---------------------------------------------------------------------------
template <int M, bool NARROW>
struct ChirpColCfg {
    static constexpr int EPT = M > 2048 ? 16 : 8;
    static constexpr int T = M / EPT;
    // four-wave blocks leave three to a CU at the 150 VGPRs of a thread's tables
    // (24 x 400^2 x 20 slices: 3.02 ms; eight-wave blocks 4.02 ms, held to 128
    // VGPRs 4.14 ms); at M >= 2048 they would hold one column, and two adjacent
    // ones per block are worth more (4 x 1000^2 x 5: 1.04 against 1.33 ms)
    static constexpr int THREADS = M >= 2048 ? 512 : 256;
    static constexpr int C0 = THREADS / T < 1 ? 1 : (THREADS / T < 16 ? THREADS / T : 16);
    static constexpr int C = NARROW ? (C0 >= 4 ? C0 / 4 : 1) : C0;
    static constexpr int BLOCK = T * C;
    static constexpr int STRIDE = LdsLayout<M>::kStride;
};

// Tiles of n_img images, in place: forward column transform, * mul, inverse.
// Each block runs a contiguous run of tiles (adjacent tiles share cache lines
// of every row), its tables loaded once and the next tile's columns loaded
// while the current one is transformed.
template <int M, class Mul, bool NARROW>
__global__ __launch_bounds__((ChirpColCfg<M, NARROW>::BLOCK)) void k_chirp_cols(
    float2* data, int n2, int tiles, int64_t n_tiles, RunSched sched, ChirpTab col, Mul mul,
    const float2* __restrict__ tw) {
    using Cfg = ChirpColCfg<M, NARROW>;
    constexpr int EPT = Cfg::EPT, HALF = EPT / 2;
    __shared__ float lds_re[Cfg::C * Cfg::STRIDE];
    __shared__ float lds_im[Cfg::C * Cfg::STRIDE];
    __shared__ float2 lds_px[Mul::kTable ? M / 2 : 1];
    const int c = threadIdx.x % Cfg::C, t = threadIdx.x / Cfg::C;
    float* re = lds_re + c * Cfg::STRIDE;
    float* im = lds_im + c * Cfg::STRIDE;
    const int n = col.n;
    int start, count;
    sched.run((int)blockIdx.x, start, count);
    auto load = [&](int64_t g, float2 (&v)[HALF], int& j, bool& ok) __attribute__((always_inline)) -> float2* {
        const int64_t img = g / tiles;
        const int j0 = (int)(g - img * tiles) * Cfg::C + c;
        ok = j0 < n2;
        j = ok ? j0 : n2 - 1;
        float2* base = data + img * n * n2 + j;
#pragma unroll
        for (int m = 0; m < HALF; ++m) {
            const int i = t + m * Cfg::T;
            v[m] = base[(int64_t)(i < n ? i : n - 1) * n2];
        }
        return base;
    };
    float2 cur[HALF], nxt[HALF], b[EPT];
    int j;
    bool ok;
    float2* base = load(start, cur, j, ok);
    chirp_load_b<M, EPT>(col.b, t, b);
    TwCache<M, EPT> twc;
    twc.load(tw, t);
    mul.prepare(lds_px, threadIdx.x, Cfg::BLOCK);   // n1 <= M / 2 entries
    if constexpr (Mul::kTable) __syncthreads();
    for (int r = 0; r < count; ++r) {
        int j_n;
        bool ok_n;
        float2* base_n = load(start + (r + 1 < count ? r + 1 : r), nxt, j_n, ok_n);
        const float2 py = mul.column(j);
        float2 v[EPT];
#pragma unroll
        for (int m = 0; m < HALF; ++m) {
            v[m] = t + m * Cfg::T < n ? cur[m] : make_float2(0.f, 0.f);
            v[m + HALF] = make_float2(0.f, 0.f);
        }
        chirp_conv<M, EPT, false>(v, b, re, im, t, twc);
#pragma unroll
        for (int m = 0; m < HALF; ++m) {
            const int i = t + m * Cfg::T;
            v[m] = i < n ? mul.apply(v[m], i, j, lds_px, py) : make_float2(0.f, 0.f);
            v[m + HALF] = make_float2(0.f, 0.f);
        }
        chirp_conv<M, EPT, true>(v, b, re, im, t, twc);
        if (ok) {
#pragma unroll
            for (int m = 0; m < HALF; ++m) {
                const int i = t + m * Cfg::T;
                if (i < n) base[(int64_t)i * n2] = v[m];
            }
        }
#pragma unroll
        for (int m = 0; m < HALF; ++m) cur[m] = nxt[m];
        base = base_n;
        j = j_n;
        ok = ok_n;
    }
}

// ---------------------------------------------------------------------------
// Potential slices.  k_chirp_r2c: half spectra of real rows, two rows (2q,
// 2q + 1) of one plane per transform as z = a + i b, split as
// A[k] = (Z[k] + conj Z[n-k]) / 2, B[k] = (Z[k] - conj Z[n-k]) / 2i, and
// multiplied by c1[x] for the column transform.  k_chirp_spectrum: per column
// of one slice, the forward transform of every element's half spectrum, * F_e,
// the sum in element order, the reference's disk, 1 / (n1 n2), the inverse
// transform and conj(c1[x]).  k_chirp_c2r: the Hermitian extension of two rows
// as a + i b, one inverse transform, clip.
// Planes: hist (n_elems, n_slices, n1, n2), X (n_elems, sc, n1, ldh).
// ---------------------------------------------------------------------------
template <int M>
__global__ __launch_bounds__(RowCfg<M>::BLOCK) void k_chirp_r2c(
    const float* __restrict__ hist, float2* __restrict__ X, int n_elems, int n_slices, int s0,
    int sc, int n1, int ldh, int rpb, ChirpTab row, const float2* __restrict__ c1,
    const float2* __restrict__ tw) {
    using Cfg = RowCfg<M>;
    constexpr int EPT = Cfg::EPT, HALF = EPT / 2, T = Cfg::T;
    using L = LdsLayout<M>;
    __shared__ float lds_re[Cfg::G * Cfg::WORDS];
    __shared__ float lds_im[Cfg::G * Cfg::WORDS];
    const int gi = row_in_block<T>();
    const int t = threadIdx.x % T;
    float* re = lds_re + gi * Cfg::WORDS;
    float* im = lds_im + gi * Cfg::WORDS;
    const int n = row.n, H = n / 2 + 1, ppp = (n1 + 1) / 2;   // pairs per plane
    const int64_t pairs = (int64_t)n_elems * sc * ppp;
    float2 b[EPT], c[HALF];
    chirp_load_b<M, EPT>(row.b, t, b);
#pragma unroll
    for (int m = 0; m < HALF; ++m) c[m] = row.c[t + m * T < n ? t + m * T : n - 1];
    TwCache<M, EPT> twc;
    twc.load(tw, t);
    struct Regs {
        float2 v[HALF], ca, cb;
    } cur, nxt;
    auto locate = [&](int64_t p0, int64_t& plane, int& xa) __attribute__((always_inline)) {
        const int64_t p = p0 < pairs ? p0 : pairs - 1;
        plane = p / ppp;                            // e sc + slice of the chunk
        xa = 2 * (int)(p - plane * ppp);
    };
    auto load = [&](int64_t p0, Regs& g) __attribute__((always_inline)) {
        int64_t plane;
        int xa;
        locate(p0, plane, xa);
        const int64_t e = plane / sc, s = plane - e * sc;
        const float* ra = hist + ((e * n_slices + s0 + s) * n1 + xa) * (int64_t)n;
        const int two = xa + 1 < n1 ? 1 : 0;
        const float* rb = ra + two * n;
#pragma unroll
        for (int m = 0; m < HALF; ++m) {
            const int k = t + m * T, kc = k < n ? k : n - 1;
            g.v[m] = make_float2(ra[kc], two ? rb[kc] : 0.f);
        }
        g.ca = c1[xa];
        g.cb = c1[xa + two];
    };
    const int64_t first = (int64_t)blockIdx.x * rpb * Cfg::G + gi;
    load(first, cur);
    for (int r = 0; r < rpb; ++r) {
        const int64_t p = first + (int64_t)r * Cfg::G;
        if (r + 1 < rpb) load(p + Cfg::G, nxt);
        float2 v[EPT];
#pragma unroll
        for (int m = 0; m < HALF; ++m) {
            v[m] = t + m * T < n ? cmul(cur.v[m], c[m]) : make_float2(0.f, 0.f);
            v[m + HALF] = make_float2(0.f, 0.f);
        }
        chirp_conv<M, EPT, false>(v, b, re, im, t, twc);
#pragma unroll
        for (int m = 0; m < HALF; ++m) {
            const int k = t + m * T;
            const float2 z = cmul(v[m], c[m]);
            if (k < n) {
                re[L::at(k)] = z.x;
                im[L::at(k)] = z.y;
            }
        }
        __syncthreads();
        if (p < pairs) {
            int64_t plane;
            int xa;
            locate(p, plane, xa);
            float2* oa = X + (plane * n1 + xa) * (int64_t)ldh;
            const bool two = xa + 1 < n1;
            for (int k = t; k < H; k += T) {
                const int ik = L::at(k), ir = L::at(k == 0 ? 0 : n - k);
                const float zr = re[ik], zi = im[ik], wr = re[ir], wi = -im[ir];   // conj Z[n-k]
                oa[k] = cmul(make_float2(0.5f * (zr + wr), 0.5f * (zi + wi)), cur.ca);
                if (two)
                    oa[ldh + k] = cmul(make_float2(0.5f * (zi - wi), -0.5f * (zr - wr)), cur.cb);
            }
        }
        __syncthreads();   // the planes are rewritten by the next pair
        cur = nxt;
    }
}

// The reference's band-limit disk index of row/column i (slice_builder_base.py
// :166-175): the entry of ifftshift(arange(-n//2, -n//2 + n)) at i, which for
// odd n is the FFT frequency minus one.
__host__ __device__ __forceinline__ int bandlimit_freq(int i, int n) {
    return (i + n / 2) % n - (n + 1) / 2;
}

// Runs of the sc * tiles column tiles; the result overwrites element 0's plane
// (each tile reads its element-0 columns before it writes them).  The next
// element's columns (of this tile, or the next one's first) load behind the
// current element's transforms.
template <int M, bool NARROW>
__global__ __launch_bounds__((ChirpColCfg<M, NARROW>::BLOCK)) void k_chirp_spectrum(
    float2* X, const float* __restrict__ sf, int n_elems, int sc, int tiles, RunSched sched, int H,
    int ldh, int n2, int bandlimit, int band_r2, float inv_npix, ChirpTab col,
    const float2* __restrict__ tw) {
    using Cfg = ChirpColCfg<M, NARROW>;
    constexpr int EPT = Cfg::EPT, HALF = EPT / 2;
    __shared__ float lds_re[Cfg::C * Cfg::STRIDE];
    __shared__ float lds_im[Cfg::C * Cfg::STRIDE];
    const int c = threadIdx.x % Cfg::C, t = threadIdx.x / Cfg::C;
    float* re = lds_re + c * Cfg::STRIDE;
    float* im = lds_im + c * Cfg::STRIDE;
    const int n = col.n;
    const int64_t plane = (int64_t)n * ldh;
    int start, count;
    sched.run((int)blockIdx.x, start, count);
    float2 b[EPT];
    chirp_load_b<M, EPT>(col.b, t, b);
    TwCache<M, EPT> twc;
    twc.load(tw, t);
    auto column = [&](int g, int& s, bool& ok) __attribute__((always_inline)) {
        s = g / tiles;
        const int j0 = (g - s * tiles) * Cfg::C + c;
        ok = j0 < H;
        return ok ? j0 : H - 1;
    };
    struct Regs {
        float2 v[HALF];
        float f[HALF];
    } cur, nxt;
    auto load = [&](int g, int e, Regs& q) __attribute__((always_inline)) {
        int s;
        bool ok;
        const int j = column(g, s, ok);
        const float2* src = X + ((int64_t)e * sc + s) * plane + j;
#pragma unroll
        for (int m = 0; m < HALF; ++m) {
            const int i = t + m * Cfg::T, ic = i < n ? i : n - 1;
            q.v[m] = src[(int64_t)ic * ldh];
            q.f[m] = sf[((int64_t)e * n + ic) * H + j];
        }
    };
    load(start, 0, cur);
    for (int r = 0; r < count; ++r) {
        const int g = start + r;
        int s;
        bool ok;
        const int j = column(g, s, ok);
        float2 acc[EPT];
#pragma unroll
        for (int m = 0; m < EPT; ++m) acc[m] = make_float2(0.f, 0.f);
        for (int e = 0; e < n_elems; ++e) {
            const bool more = e + 1 < n_elems;
            load(more || r + 1 >= count ? g : g + 1, more ? e + 1 : 0, nxt);
            float2 v[EPT];
#pragma unroll
            for (int m = 0; m < HALF; ++m) {
                v[m] = t + m * Cfg::T < n ? cur.v[m] : make_float2(0.f, 0.f);
                v[m + HALF] = make_float2(0.f, 0.f);
            }
            chirp_conv<M, EPT, false>(v, b, re, im, t, twc);
#pragma unroll
            for (int m = 0; m < HALF; ++m) {
                acc[m].x = fmaf(v[m].x, cur.f[m], acc[m].x);
                acc[m].y = fmaf(v[m].y, cur.f[m], acc[m].y);
            }
            cur = nxt;
        }
        const int kj = bandlimit_freq(j, n2);
#pragma unroll
        for (int m = 0; m < HALF; ++m) {
            const int i = t + m * Cfg::T;
            const int ki = bandlimit_freq(i < n ? i : 0, n);
            // past n acc holds the convolution's tail
            const bool keep = i < n && !(bandlimit && ki * ki + kj * kj > band_r2);
            acc[m] = keep ? make_float2(acc[m].x * inv_npix, acc[m].y * inv_npix)
                          : make_float2(0.f, 0.f);
        }
        chirp_conv<M, EPT, true>(acc, b, re, im, t, twc);
        if (!ok) continue;
        float2* dst = X + (int64_t)s * plane + j;
#pragma unroll
        for (int m = 0; m < HALF; ++m) {
            const int i = t + m * Cfg::T;
            if (i < n) dst[(int64_t)i * ldh] = mul_tw<true>(acc[m], col.c[i]);
        }
    }
}

// planes of n1 half rows in (ldh apart), pairs (2q, 2q + 1) within each plane, so
// that no slice's values (an infinity's NaN, a rounding) reach another one's rows
// where n1 is odd; real rows out, n apart.
template <int M>
__global__ __launch_bounds__(RowCfg<M>::BLOCK) void k_chirp_c2r(
    const float2* __restrict__ X, float* __restrict__ out, int planes, int n1, int ldh, int rpb,
    float clip_lo, ChirpTab row, const float2* __restrict__ tw) {
    using Cfg = RowCfg<M>;
    constexpr int EPT = Cfg::EPT, HALF = EPT / 2, T = Cfg::T;
    __shared__ float lds_re[Cfg::G * Cfg::WORDS];
    __shared__ float lds_im[Cfg::G * Cfg::WORDS];
    const int gi = row_in_block<T>();
    const int t = threadIdx.x % T;
    float* re = lds_re + gi * Cfg::WORDS;
    float* im = lds_im + gi * Cfg::WORDS;
    const int n = row.n, ppp = (n1 + 1) / 2;   // pairs per plane
    const int64_t pairs = (int64_t)planes * ppp;
    float2 b[EPT], c[HALF];
    chirp_load_b<M, EPT>(row.b, t, b);
#pragma unroll
    for (int m = 0; m < HALF; ++m) c[m] = row.c[t + m * T < n ? t + m * T : n - 1];
    TwCache<M, EPT> twc;
    twc.load(tw, t);
    struct Regs {
        float2 a[HALF], b[HALF];
    } cur, nxt;
    // the pair's first row (of all planes'), and whether it has a second one
    auto locate = [&](int64_t p0, bool& two) __attribute__((always_inline)) {
        const int64_t p = p0 < pairs ? p0 : pairs - 1;
        const int64_t plane = p / ppp;
        const int x = 2 * (int)(p - plane * ppp);
        two = x + 1 < n1;
        return plane * n1 + x;
    };
    auto load = [&](int64_t p0, Regs& g) __attribute__((always_inline)) {
        bool two;
        const float2* ia = X + locate(p0, two) * ldh;
        const float2* ib = two ? ia + ldh : ia;
#pragma unroll
        for (int m = 0; m < HALF; ++m) {
            const int k = t + m * T, kc = k < n ? k : n - 1;
            const int kk = 2 * kc <= n ? kc : n - kc;
            g.a[m] = ia[kk];
            g.b[m] = ib[kk];
        }
    };
    const int64_t first = (int64_t)blockIdx.x * rpb * Cfg::G + gi;
    load(first, cur);
    for (int r = 0; r < rpb; ++r) {
        const int64_t p = first + (int64_t)r * Cfg::G;
        if (r + 1 < rpb) load(p + Cfg::G, nxt);
        bool two;
        const int64_t ra = locate(p, two);
        float2 v[EPT];
#pragma unroll
        for (int m = 0; m < HALF; ++m) {
            const int k = t + m * T;
            float2 ya = cur.a[m], yb = cur.b[m];
            // a C2R transform ignores the imaginary parts of bin 0 and (even n) n/2
            if (k == 0 || 2 * k == n) { ya.y = 0.f; yb.y = 0.f; }
            if (2 * k > n) { ya.y = -ya.y; yb.y = -yb.y; }
            if (!two) yb = make_float2(0.f, 0.f);
            v[m] = k < n ? mul_tw<true>(make_float2(ya.x - yb.y, ya.y + yb.x), c[m])
                         : make_float2(0.f, 0.f);
            v[m + HALF] = make_float2(0.f, 0.f);
        }
        chirp_conv<M, EPT, true>(v, b, re, im, t, twc);
        if (p < pairs) {
#pragma unroll
            for (int m = 0; m < HALF; ++m) {
                const int k = t + m * T;
                if (k >= n) continue;
                const float2 z = mul_tw<true>(v[m], c[m]);
                out[ra * n + k] = fmaxf(z.x, clip_lo);
                if (two) out[(ra + 1) * n + k] = fmaxf(z.y, clip_lo);
            }
        }
        cur = nxt;
    }
}

}  // namespace emsim
