// FFT correlator: numerator from power spectra along the time axis.
//
// Reference: FFTWCorrelator._correlate_fft (correlator/dense.py:347-369) and
// CUFFTCorrelator (cuda.py:185-219): per bin, a float32 FFT of every pixel series
// zero-padded to Nf >= 2N (dense.py:289), times the FFT of the reversed series, one
// inverse FFT per pixel, a sum over pixels; the denominator is np.correlate of the
// integer frame sums (dense.py:365-366).
//
// Here, per bin:
//   Num(tau) = IFFT_Nf( sum_p |X_p(f)|^2 )[tau],   X_p = FFT_Nf(x_p zero-padded),
// (the product with the reversed series is the same autocorrelation; the inverse is
// linear, so one inverse per bin replaces one per pixel).  Nf = 2L with L >= N from a
// set of mixed-radix lengths (2^a 5^b), so a linear autocorrelation needs no more.
//
// A series is never transformed whole.  Nf = G H, and the bins f = G k + c of one class c
// are a transform of length H of the folded and modulated series
//   z_c[n] = exp(-2 pi i n c / Nf) sum_{m < G/2} x[n + H m] exp(-2 pi i m c / G),  n < H
// (the terms m >= G/2 are the zero padding).  |X(f)| = |X(Nf - f)| leaves the classes
// c = 0 .. G/2.  For 0 < c < G/2 one transform serves one series, and its H points are all
// of class c (and of class G - c by symmetry).  For c = 0 and G/2 z_c is a real sequence
// times a modulation, so two series share a transform as its real and imaginary parts:
// |Z(f)|^2 + |Z(-f)|^2 = 2 (|X_1|^2 + |X_2|^2), which the symmetric sum at the end undoes.
// No transform is unpacked, none is longer than LDS holds, and nothing goes through HBM
// between passes, up to N = 131,072.
//  * gather_pm_kernel<E>: frames -> series in pairs, D[pair][n][series][m] of the frame
//    element type E (n < H, m < G/2; zero past the last frame), so one load gives a thread
//    what a point of every class needs; 64 pixels x 256 frames per workgroup through an LDS
//    transpose; the same workgroup adds its 64 pixels per frame from the LDS tile and sends
//    each frame's total to the exact S_b(t) with one 64-bit atomic.
//  * fft_spectra_kernel<E, Plan, G>: one workgroup per (k-block of 64 series, class); an
//    FP32 mixed-radix Stockham FFT (Govindaraju et al., "High performance discrete Fourier
//    transforms on graphics processors", SC 2008) with register DFTs; |Z|^2 of the last
//    pass's outputs is accumulated in FP64 registers straight from the DFT.
//  * fft_inverse_*_kernel: Num(tau) = (P_0 + (-1)^tau P_L + 2 sum_{k=1}^{L-1} P_k
//    cos(2 pi k tau / Nf)) / Nf in FP64, in two steps.
// Twiddle tables are computed on the host in FP64 and rounded to FP32.
#include "dxg2_internal.h"

namespace dxg2 {

struct c32 {
    float x, y;
};
__device__ __forceinline__ c32 cmul(c32 a, c32 b) {
    return c32{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
__device__ __forceinline__ c32 cadd(c32 a, c32 b) { return c32{a.x + b.x, a.y + b.y}; }
__device__ __forceinline__ c32 csub(c32 a, c32 b) { return c32{a.x - b.x, a.y - b.y}; }
__device__ __forceinline__ c32 negi(c32 a) { return c32{a.y, -a.x}; }   // -i a
__device__ __forceinline__ c32 cscale(c32 a, float s) { return c32{a.x * s, a.y * s}; }
__device__ __forceinline__ c32 c_of(float2 t) { return c32{t.x, t.y}; }

// ------------------------------------------------------------- register DFTs
// Dft<R>::run(a): in place, natural order, a[k] = sum_n a[n] exp(-2 pi i n k / R).
template <int R>
struct Dft;

template <>
struct Dft<2> {
    __device__ __forceinline__ static void run(c32* a) {
        const c32 s = cadd(a[0], a[1]), d = csub(a[0], a[1]);
        a[0] = s;
        a[1] = d;
    }
};

template <>
struct Dft<4> {
    __device__ __forceinline__ static void run(c32* a) {
        const c32 s02 = cadd(a[0], a[2]), d02 = csub(a[0], a[2]);
        const c32 s13 = cadd(a[1], a[3]), d13 = negi(csub(a[1], a[3]));
        a[0] = cadd(s02, s13);
        a[1] = cadd(d02, d13);
        a[2] = csub(s02, s13);
        a[3] = csub(d02, d13);
    }
};

template <>
struct Dft<5> {
    __device__ __forceinline__ static void run(c32* a) {
        // cos(2 pi/5), cos(4 pi/5), sin(2 pi/5), sin(4 pi/5)
        constexpr float C1 = 0.30901699437494745f, C2 = -0.80901699437494734f;
        constexpr float S1 = 0.95105651629515353f, S2 = 0.58778525229247325f;
        const c32 t1 = cadd(a[1], a[4]), t2 = cadd(a[2], a[3]);
        const c32 t3 = csub(a[1], a[4]), t4 = csub(a[2], a[3]);
        const c32 b1 = c32{a[0].x + C1 * t1.x + C2 * t2.x, a[0].y + C1 * t1.y + C2 * t2.y};
        const c32 b2 = c32{a[0].x + C2 * t1.x + C1 * t2.x, a[0].y + C2 * t1.y + C1 * t2.y};
        const c32 d1 = c32{S1 * t3.x + S2 * t4.x, S1 * t3.y + S2 * t4.y};
        const c32 d2 = c32{S2 * t3.x - S1 * t4.x, S2 * t3.y - S1 * t4.y};
        a[0] = cadd(a[0], cadd(t1, t2));
        a[1] = cadd(b1, negi(d1));
        a[4] = csub(b1, negi(d1));
        a[2] = cadd(b2, negi(d2));
        a[3] = csub(b2, negi(d2));
    }
};

// exp(-2 pi i m / 10) for m < 5
__device__ __forceinline__ c32 w10(int m) {
    constexpr float C1 = 0.80901699437494742f, S1 = 0.58778525229247314f;
    constexpr float C2 = 0.30901699437494745f, S2 = 0.95105651629515353f;
    switch (m) {
        case 1: return c32{C1, -S1};
        case 2: return c32{C2, -S2};
        case 3: return c32{-C2, -S2};
        case 4: return c32{-C1, -S1};
        default: return c32{1.f, 0.f};
    }
}

template <>
struct Dft<10> {
    // n = 2 m + p: E_p = DFT5 over m of a[2m + p]; a[k] = E0[k] + w10^k E1[k],
    // a[k + 5] = E0[k] - w10^k E1[k]
    __device__ __forceinline__ static void run(c32* a) {
        c32 e0[5] = {a[0], a[2], a[4], a[6], a[8]};
        c32 e1[5] = {a[1], a[3], a[5], a[7], a[9]};
        Dft<5>::run(e0);
        Dft<5>::run(e1);
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            const c32 t = k ? cmul(w10(k), e1[k]) : e1[k];
            a[k] = cadd(e0[k], t);
            a[k + 5] = csub(e0[k], t);
        }
    }
};

// exp(-2 pi i m / 8) for m < 4
__device__ __forceinline__ c32 w8(int m) {
    constexpr float H = 0.70710678118654752f;
    switch (m) {
        case 1: return c32{H, -H};
        case 2: return c32{0.f, -1.f};
        case 3: return c32{-H, -H};
        default: return c32{1.f, 0.f};
    }
}

template <>
struct Dft<8> {
    // n = 2 m + p: E_p = DFT4 over m of a[2m + p]; a[k] = E0[k] + w8^k E1[k],
    // a[k + 4] = E0[k] - w8^k E1[k]
    __device__ __forceinline__ static void run(c32* a) {
        c32 e0[4] = {a[0], a[2], a[4], a[6]};
        c32 e1[4] = {a[1], a[3], a[5], a[7]};
        Dft<4>::run(e0);
        Dft<4>::run(e1);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const c32 t = k ? cmul(w8(k), e1[k]) : e1[k];
            a[k] = cadd(e0[k], t);
            a[k + 4] = csub(e0[k], t);
        }
    }
};

// exp(-2 pi i m / 16) for m = p k in {0, 1, 2, 3, 4, 6, 9}
__device__ __forceinline__ c32 w16(int m) {
    constexpr float C1 = 0.92387953251128674f, S1 = 0.38268343236508978f;
    constexpr float H = 0.70710678118654752f;
    switch (m) {
        case 1: return c32{C1, -S1};
        case 2: return c32{H, -H};
        case 3: return c32{S1, -C1};
        case 4: return c32{0.f, -1.f};
        case 6: return c32{-H, -H};
        case 9: return c32{-C1, S1};
        default: return c32{1.f, 0.f};
    }
}

template <>
struct Dft<16> {
    // n = 4 m + p: E_p = DFT4 over m of a[4m + p]; a[k + 4q] = DFT4 over p of
    // (w16^(p k) E_p[k]), output q
    __device__ __forceinline__ static void run(c32* a) {
        c32 e[4][4];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
#pragma unroll
            for (int m = 0; m < 4; ++m) e[p][m] = a[4 * m + p];
            Dft<4>::run(e[p]);
        }
        twist(e, a);
    }
    // second stage: a[k + 4q] = DFT4 over p of (w16^(p k) E_p[k]), output q
    __device__ __forceinline__ static void twist(c32 (&e)[4][4], c32* a) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            c32 v[4];
#pragma unroll
            for (int p = 0; p < 4; ++p) v[p] = (p && k) ? cmul(w16(p * k), e[p][k]) : e[p][k];
            Dft<4>::run(v);
#pragma unroll
            for (int q = 0; q < 4; ++q) a[k + 4 * q] = v[q];
        }
    }
};

// LDS index of point i: the low 4 bits are xor-ed with the next 4, so the stride-16
// accesses of a pass hit 16 different 8-byte slots and the array needs no padding.
__device__ __forceinline__ int sw(int i) { return i ^ ((i >> 4) & 15); }
// sw(base + r S) with r known at compile time (r may be negative): for S a multiple of
// 256, r S leaves bits 0..7 of base + r S as they are in base, so the swizzle is
// sw(base) + r S; for S an odd multiple of 128 it leaves bits 0..6 and flips bit 7 when
// r is odd, which flips bit 3 of the xor term: (sw(base) ^ 8) + r S.  Either way one
// address per butterfly and constant offsets.
template <int S>
__device__ __forceinline__ int sw_step(int base, int r) {
    if constexpr (S % 256 == 0) return sw(base) + r * S;
    else if constexpr (S % 128 == 0) return (sw(base) ^ ((r & 1) << 3)) + r * S;
    else return sw(base + r * S);
}

// ----------------------------------------------------------- series layout
// One point n of a pair of series: G elements (series p, fold m) at index p G/2 + m.
template <typename E, int G>
struct RawPoint {
    static constexpr int NW = G * (int)sizeof(E) / 4;
    uint32_t w[NW];
    __device__ __forceinline__ void load(const uint8_t* row, int n) {
        const uint8_t* src = row + (int64_t)n * (4 * NW);
        if constexpr (NW == 1) {
            w[0] = *reinterpret_cast<const uint32_t*>(src);
        } else if constexpr (NW == 2) {
            const uint2 v = *reinterpret_cast<const uint2*>(src);
            w[0] = v.x;
            w[1] = v.y;
        } else {
#pragma unroll
            for (int i = 0; i < NW; i += 4) {
                const uint4 v = *reinterpret_cast<const uint4*>(src + 4 * i);
                w[i] = v.x;
                w[i + 1] = v.y;
                w[i + 2] = v.z;
                w[i + 3] = v.w;
            }
        }
    }
    __device__ __forceinline__ int value(int e) const {
        if constexpr (sizeof(E) == 1)
            return (int)(E)((w[e >> 2] >> (8 * (e & 3))) & 0xFFu);
        else
            return (int)(E)((w[e >> 1] >> (16 * (e & 1))) & 0xFFFFu);
    }
    // Series p's elements in the first half: one shift or mask a word, p known at run time.
    __device__ __forceinline__ RawPoint series(int p) const {
        RawPoint r;
        if constexpr (NW == 1) {
            r.w[0] = w[0] >> (p * 16);
        } else {
#pragma unroll
            for (int i = 0; i < NW / 2; ++i) {
                const uint32_t m = 0u - (uint32_t)p;
                r.w[i] = (w[NW / 2 + i] & m) | (w[i] & ~m);
                r.w[NW / 2 + i] = 0u;
            }
        }
        return r;
    }
};

// --------------------------------------------------------------- pixel-major gather
// grid (k-blocks in gather order, frame tiles of 256).  Lane = pixel of the k-block: each
// load instruction reads one frame of the 64 pixels (the k-block's stretch of detector
// row).  A lane packs 4 / sizeof(E) consecutive frames into one 32-bit word and writes
// it to its pixel's row of an LDS tile whose row stride is an odd number of words, so
// the 64 lanes' column writes fall in distinct banks.  Loads past the last frame repeat it and
// are masked afterwards: a condition on each load keeps them from being in flight together
// (4.23 -> 3.95 ms at 479,980 pixels x 10,000 frames; 515 x 1031 x 1,000, where every
// load is a byte, 1.27 -> 1.06 ms a call).  The tile's frames are G / 2 runs,
// run m at frames H m + n0 .., so it holds every element of SEG points of the pairs: a
// thread reads the G words (series, run) of a few points of one pair, transposes them in
// registers and stores 4 G contiguous bytes.  The frame sums S_b(t) (zeroed by the caller)
// come from the same tile: a thread adds one word (4 frames of 8-bit values in 16-bit
// halves, or 2 of 16-bit values in 32-bit registers) down 16 or 32 pixel rows, the row
// groups meet in LDS, and each frame's total over the 64 pixels (below 2^31) goes to
// sums with one 64-bit atomic (the row groups' partials reuse the tile's LDS once every
// thread has read it).  SGN (int8 frames): bytes are added as v ^ 0x80 = v + 128
// and 64 x 128 is taken off the total (padded pixels and frames hold 0, so they add 128
// each and are taken off with the rest).
// quad_kb (8-bit frames, 4 | hw, frames 4-aligned; else null): per bin, the leading
// k-blocks whose list entries are 16 aligned quads of detector pixels 4a .. 4a + 3.  In
// those, lane (g, kk) = (lane % 16, lane / 16) reads quad g of frame 4k + f (f < 4) of word
// k = 4 (wave + 4 i) + kk as one aligned 4-byte load (a quarter of the load instructions),
// and a 4 x 4 byte transpose in registers turns the four frames' quads into the four
// pixels' words of the tile.
// A workgroup takes KPB k-blocks that are neighbours in detector order (work item
// blockIdx.x; kb -1: none) over 256 / KPB frames, so that the workgroups in flight read
// a larger share of each frame row, and still stores whole 128-byte lines of each pair.
template <typename E, bool SGN, int KPB, int G>
__global__ __launch_bounds__(256) void gather_pm_kernel(const uint8_t* __restrict__ frames,
                                                        int64_t hw, int nframes, int H,
                                                        const int32_t* __restrict__ pix_idx,
                                                        const int32_t* __restrict__ quad_kb,
                                                        const BinDev* __restrict__ bins,
                                                        const KbWork* __restrict__ work,
                                                        uint8_t* __restrict__ xs,
                                                        int64_t* __restrict__ sums) {
    constexpr int FT = 256 / KPB;      // frames per workgroup
    constexpr int ES = sizeof(E);
    constexpr int FPW = 4 / ES;        // frames per word
    constexpr int WPR = FT / FPW;      // words per pixel row of the tile
    constexpr int STRIDE = WPR + 1;    // odd
    constexpr int ROWS = KPB * KB;     // pixel rows of the tile
    constexpr int RG = 256 / WPR;      // row groups of the sums (threads = WPR x RG)
    constexpr int RPG = ROWS / RG;     // rows per group: within one k-block
    constexpr int SEG = FT / (G / 2);  // frames per run
    static_assert(SEG % 4 == 0 && SEG % FPW == 0, "a word lies in one run");
    static_assert(KB % RPG == 0 && FT * KPB == 256 && WPR % 16 == 0, "gather shape");
    __shared__ __attribute__((aligned(16))) uint32_t tile[ROWS * STRIDE];
    static_assert(RG * FT <= ROWS * STRIDE, "partials fit the tile");
    const KbWork* item = work + (int64_t)blockIdx.x * KPB;
    if (item[0].kb < 0) return;  // padding of the gather order (the first slot is filled first)
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int n0 = blockIdx.y * SEG;
    auto frame_of = [&](int f) { return (f / SEG) * H + n0 + f % SEG; };  // of tile column f
    constexpr uint32_t MASK = ES == 1 ? 0xFFu : 0xFFFFu;
#pragma unroll
    for (int j = 0; j < KPB; ++j) {
        const KbWork w = item[j];
        if (w.kb < 0) continue;  // the same for the whole workgroup
        const BinDev bd = bins[w.bin];
        uint32_t* rows = tile + j * KB * STRIDE;
        if (ES == 1 && quad_kb && w.kb < quad_kb[w.bin]) {
            const int g = lane & 15, kk = lane >> 4;
            const int q0 = pix_idx[bd.idx_off + (int64_t)w.kb * KB + 4 * g];  // 4 | q0
            uint32_t vs[WPR / 16][4];
#pragma unroll
            for (int i = 0; i < WPR / 16; ++i)
#pragma unroll
                for (int f4 = 0; f4 < 4; ++f4) {
                    const int t = frame_of(4 * (4 * (wave + 4 * i) + kk)) + f4;
                    vs[i][f4] = *reinterpret_cast<const uint32_t*>(
                        frames + (int64_t)min(t, nframes - 1) * hw + q0);
                }
#pragma unroll
            for (int i = 0; i < WPR / 16; ++i) {
                const int k = 4 * (wave + 4 * i) + kk;
                uint32_t v[4];
#pragma unroll
                for (int f4 = 0; f4 < 4; ++f4)
                    v[f4] = frame_of(4 * k) + f4 < nframes ? vs[i][f4] : 0u;
                // v[f] byte b = pixel 4g + b at frame 4k + f  ->  word k of pixel 4g + b
                const uint32_t l01 = __builtin_amdgcn_perm(v[1], v[0], 0x05010400u);
                const uint32_t h01 = __builtin_amdgcn_perm(v[1], v[0], 0x07030602u);
                const uint32_t l23 = __builtin_amdgcn_perm(v[3], v[2], 0x05010400u);
                const uint32_t h23 = __builtin_amdgcn_perm(v[3], v[2], 0x07030602u);
                uint32_t* row = rows + (4 * g) * STRIDE + k;
                row[0] = __builtin_amdgcn_perm(l23, l01, 0x05040100u);
                row[STRIDE] = __builtin_amdgcn_perm(l23, l01, 0x07060302u);
                row[2 * STRIDE] = __builtin_amdgcn_perm(h23, h01, 0x05040100u);
                row[3 * STRIDE] = __builtin_amdgcn_perm(h23, h01, 0x07060302u);
            }
        } else {
            const int p = pix_idx[bd.idx_off + (int64_t)w.kb * KB + lane];
            const E* fr = reinterpret_cast<const E*>(frames) + (p >= 0 ? p : 0);
            const int nt = p >= 0 ? nframes : 0;
            // 16 loads at a time
            constexpr int AT = 16 / FPW;
            static_assert(WPR / 4 % AT == 0, "whole steps");
#pragma unroll
            for (int i0 = 0; i0 < WPR / 4; i0 += AT) {
                E vs[AT][FPW];
#pragma unroll
                for (int i = 0; i < AT; ++i)
#pragma unroll
                    for (int q = 0; q < FPW; ++q)
                        vs[i][q] = fr[(int64_t)min(frame_of(FPW * (wave + 4 * (i0 + i))) + q,
                                                   nframes - 1) * hw];
#pragma unroll
                for (int i = 0; i < AT; ++i) {
                    const int k = wave + 4 * (i0 + i);  // word k: tile columns FPW k ..
                    const int tk = frame_of(FPW * k);
                    uint32_t word = 0u;
#pragma unroll
                    for (int q = 0; q < FPW; ++q)
                        word |= tk + q < nt ? ((uint32_t)vs[i][q] & MASK) << (8 * ES * q) : 0u;
                    rows[lane * STRIDE + k] = word;
                }
            }
        }
    }
    __syncthreads();
    // pair r of the tile (rows 2r, 2r + 1), word k of every run: FPW points, 4 G bytes
    constexpr int WPS = SEG / FPW;  // words per run
    for (int c = threadIdx.x; c < ROWS / 2 * WPS; c += 256) {
        const int r = c / WPS, k = c % WPS;
        const KbWork w = item[2 * r / KB];
        if (w.kb < 0) continue;
        uint32_t v[G], o[G];  // v[p G/2 + m]: series p, run m
#pragma unroll
        for (int i = 0; i < G; ++i)
            v[i] = tile[(2 * r + i / (G / 2)) * STRIDE + (i % (G / 2)) * WPS + k];
        if constexpr (ES == 1) {
#pragma unroll
            for (int i = 0; i < G; i += 4) {  // 4 x 4 bytes: element i + j of point q
                const uint32_t l01 = __builtin_amdgcn_perm(v[i + 1], v[i], 0x05010400u);
                const uint32_t h01 = __builtin_amdgcn_perm(v[i + 1], v[i], 0x07030602u);
                const uint32_t l23 = __builtin_amdgcn_perm(v[i + 3], v[i + 2], 0x05010400u);
                const uint32_t h23 = __builtin_amdgcn_perm(v[i + 3], v[i + 2], 0x07030602u);
                o[i / 4] = __builtin_amdgcn_perm(l23, l01, 0x05040100u);
                o[G / 4 + i / 4] = __builtin_amdgcn_perm(l23, l01, 0x07060302u);
                o[G / 2 + i / 4] = __builtin_amdgcn_perm(h23, h01, 0x05040100u);
                o[3 * G / 4 + i / 4] = __builtin_amdgcn_perm(h23, h01, 0x07060302u);
            }
        } else {
#pragma unroll
            for (int i = 0; i < G; i += 2) {  // 2 x 2 halves
                o[i / 2] = __builtin_amdgcn_perm(v[i + 1], v[i], 0x05040100u);
                o[G / 2 + i / 2] = __builtin_amdgcn_perm(v[i + 1], v[i], 0x07060302u);
            }
        }
        const int64_t pair = (bins[w.bin].idx_off + (int64_t)w.kb * KB) / 2 + r % (KB / 2);
        uint8_t* dst = xs + (pair * H + n0 + FPW * k) * (G * ES);
#pragma unroll
        for (int i = 0; i < G; i += 4)
            *reinterpret_cast<uint4*>(dst + 4 * i) =
                make_uint4(o[i], o[i + 1], o[i + 2], o[i + 3]);
    }
    const int k = threadIdx.x % WPR, g = threadIdx.x / WPR;  // word k, rows RPG g ..
    const uint32_t* col = tile + RPG * g * STRIDE + k;
    uint32_t s0 = 0u, s1 = 0u;
    if constexpr (ES == 1) {
        // s0: frames 4k, 4k + 2 and s1: 4k + 1, 4k + 3 in 16-bit halves (16 rows x 255)
#pragma unroll
        for (int j = 0; j < RPG; ++j) {
            const uint32_t x = col[j * STRIDE] ^ (SGN ? 0x80808080u : 0u);
            s0 += x & 0x00FF00FFu;
            s1 += (x >> 8) & 0x00FF00FFu;
        }
    } else {
        // s0: frame 2k, s1: 2k + 1 (32 rows x 65535)
#pragma unroll 8
        for (int j = 0; j < RPG; ++j) {
            const uint32_t x = col[j * STRIDE];
            s0 += x & 0xFFFFu;
            s1 += x >> 16;
        }
    }
    static_assert(ES != 1 || RPG <= 256, "16-bit halves");
    __syncthreads();  // every thread has read the tile: its words now hold the partials
    int32_t* part = reinterpret_cast<int32_t*>(tile);  // [RG][FT]
    if constexpr (ES == 1)
        *reinterpret_cast<int4*>(part + FT * g + 4 * k) =
            make_int4((int)(s0 & 0xFFFFu), (int)(s1 & 0xFFFFu), (int)(s0 >> 16),
                      (int)(s1 >> 16));
    else
        *reinterpret_cast<int2*>(part + FT * g + 2 * k) = make_int2((int)s0, (int)s1);
    __syncthreads();
    // thread (j, f): column f of k-block j, from the RG / KPB row groups of that k-block
    const int jb = threadIdx.x / FT, f = threadIdx.x % FT;
    const KbWork w = item[jb];
    const int t = frame_of(f);
    if (w.kb >= 0 && t < nframes) {
        constexpr int GPK = RG / KPB;  // row groups per k-block
        int64_t tot = SGN ? -(int64_t)KB * 128 : 0;
#pragma unroll
        for (int q = 0; q < GPK; ++q) tot += part[FT * (GPK * jb + q) + f];
        if (tot)
            atomicAdd(reinterpret_cast<unsigned long long*>(sums + (int64_t)w.bin * nframes + t),
                      (unsigned long long)tot);
    }
}

// ------------------------------------------------------------------- spectra
// A plan: L complex points (the H of a series length G H / 2), T threads, radices R1..R4
// (R4 = 1 when there are three passes).  The middle passes' twiddles are in LDS tables
// (pass p's table holds exp(-2 pi i m / P_p), m < P_p = R1 ... R_p).
template <int L_, int T_, int R1_, int R2_, int R3_, int R4_>
struct FftPlan {
    static constexpr int L = L_, T = T_, R1 = R1_, R2 = R2_, R3 = R3_, R4 = R4_;
    static constexpr int NP = R4 > 1 ? 4 : 3;
    static constexpr int RL = NP == 4 ? R4 : R3;        // radix of the last pass
    static constexpr int P2 = R1 * R2;                   // table of pass 2
    static constexpr int P3 = NP == 4 ? R1 * R2 * R3 : 1;  // table of pass 3 (4 passes)
    static_assert(R1 * R2 * R3 * R4 == L, "radices must multiply to L");
};

template <typename Plan, int R, int NS, int PT>
__device__ __forceinline__ void mid_pass(c32* z, const c32* tab, int tid) {
    constexpr int L = Plan::L, T = Plan::T;
    constexpr int NB = L / R;
    constexpr int M = (NB + T - 1) / T;
    c32 v[M][R];
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const int b = tid + m * T;
        if (NB % T == 0 || b < NB) {
            const int k = b % NS;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                c32 a = z[sw_step<NB>(b, r)];
                if (r) a = cmul(a, tab[r * k]);      // exp(-2 pi i r k / (R NS)), PT = R NS
                v[m][r] = a;
            }
            Dft<R>::run(v[m]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const int b = tid + m * T;
        if (NB % T == 0 || b < NB) {
            const int k = b % NS;
            const int o = (b - k) * R + k;
#pragma unroll
            for (int q = 0; q < R; ++q) z[sw_step<NS>(o, q)] = v[m][q];
        }
    }
    __syncthreads();
}

// What a class's transforms are made of.
enum FftClass {
    PAIR_PLAIN,  // class 0: two series as real and imaginary parts
    PAIR_MOD,    // class G/2: the same, modulated
    SINGLE       // classes between: one series each
};

// The transforms of nser series (pairs from `rows`) and one class; the sums of |Z[k]|^2
// over them are added to prow[k], k < H.
template <typename E, typename Plan, int G, FftClass MODE>
__device__ __forceinline__ void spectra_class(const uint8_t* __restrict__ rows, int nser, int cls,
                                              const float2* __restrict__ twl,
                                              const float2* __restrict__ uw,
                                              double* __restrict__ prow, c32* z, const c32* tab2,
                                              const c32* tab3) {
    constexpr int H = Plan::L, T = Plan::T;
    constexpr int R1 = Plan::R1, R2 = Plan::R2, R3 = Plan::R3, RL = Plan::RL;
    constexpr int NB1 = H / R1, M1 = (NB1 + T - 1) / T;  // first pass
    constexpr int NBL = H / RL, ML = (NBL + T - 1) / T;  // last pass
    using Raw = RawPoint<E, G>;
    const int tid = threadIdx.x;
    const int npair = (nser + 1) / 2;
    double acc[ML][RL];
#pragma unroll
    for (int m = 0; m < ML; ++m)
#pragma unroll
        for (int q = 0; q < RL; ++q) acc[m][q] = 0.0;
    c32 fold[G / 2];  // exp(-2 pi i m cls / G)
#pragma unroll
    for (int m = 0; m < G / 2; ++m) sincospif(-2.0f * (m * cls) / G, &fold[m].y, &fold[m].x);
    auto modn = [&](int b, int r) { return c_of(uw[(b + r * NB1) * cls]); };
    const int64_t row_bytes = (int64_t)H * G * sizeof(E);
    // A pair's points are loaded while the transform before it runs, where the registers
    // allow it.
    constexpr bool AHEAD = M1 * R1 * Raw::NW <= (T > 768 ? 8 : 32);
    Raw raw[AHEAD ? M1 : 1][R1];
    auto load = [&](const uint8_t* row, int t) {
#pragma unroll
        for (int m = 0; m < (AHEAD ? M1 : 0); ++m)
#pragma unroll
            for (int r = 0; r < R1; ++r) {
                const int b = t + m * T;
                if (NB1 % T == 0 || b < NB1) raw[m][r].load(row, b + r * NB1);
            }
    };
    load(rows, tid);
    __syncthreads();  // tables

    const int count = MODE == SINGLE ? nser : npair;
    for (int j = 0; j < count; ++j) {
        // Every address and twiddle below depends on the thread only; an opaque copy of
        // the thread index per transform keeps the compiler from holding them all in
        // registers across the loop (which spills).
        int t = tid;
        asm volatile("" : "+v"(t));
        // first pass (stride 1) from the registers loaded during the previous transform:
        // point b + r NB1 -> outputs q at b R1 + q
#pragma unroll
        for (int m = 0; m < M1; ++m) {
            const int b = t + m * T;
            if (NB1 % T == 0 || b < NB1) {
                c32 v[R1];
#pragma unroll
                for (int r = 0; r < R1; ++r) {
                    Raw& x0 = raw[AHEAD ? m : 0][r];
                    if (!AHEAD) x0.load(rows + (MODE == SINGLE ? j / 2 : j) * row_bytes, b + r * NB1);
                    if (MODE == SINGLE) {
                        const Raw x = x0.series(j & 1);
                        if (G == 4) {  // fold[1] = -i
                            const float a0 = x.value(0), a1 = x.value(1);
                            const c32 w = modn(b, r);
                            v[r] = c32{a0 * w.x + a1 * w.y, a0 * w.y - a1 * w.x};
                        } else {
                            c32 a{0.f, 0.f};
#pragma unroll
                            for (int i = 0; i < G / 2; ++i) {
                                const float xi = x.value(i);
                                a.x += xi * fold[i].x;
                                a.y += xi * fold[i].y;
                            }
                            v[r] = cmul(a, modn(b, r));
                        }
                    } else {  // integer sums, alternating in class G/2
                            const Raw& x = x0;
                        int s0 = 0, s1 = 0;
#pragma unroll
                        for (int i = 0; i < G / 2; ++i) {
                            const bool neg = MODE == PAIR_MOD && (i & 1);
                            s0 += neg ? -x.value(i) : x.value(i);
                            s1 += neg ? -x.value(G / 2 + i) : x.value(G / 2 + i);
                        }
                        v[r] = c32{(float)s0, (float)s1};
                        if (MODE == PAIR_MOD) v[r] = cmul(v[r], modn(b, r));
                    }
                }
                Dft<R1>::run(v);
#pragma unroll
                for (int q = 0; q < R1; ++q) z[sw(b * R1 + q)] = v[q];
            }
        }
        // the next pair's inputs, in flight during this transform's passes
        const int next = MODE == SINGLE ? (j + 1) / 2 : j + 1;
        if ((MODE != SINGLE || (j & 1)) && next < npair) load(rows + next * row_bytes, t);
        __syncthreads();
        mid_pass<Plan, R2, R1, Plan::P2>(z, tab2, t);
        if (Plan::NP == 4) mid_pass<Plan, R3, R1 * R2, Plan::P3>(z, tab3, t);
        // last pass: butterfly b reads z[b + r NBL], twiddles exp(-2 pi i r b / H) (its
        // table is r-major), and its outputs q are the bins k = b + q NBL
#pragma unroll
        for (int m = 0; m < ML; ++m) {
            const int b = t + m * T;
            if (NBL % T == 0 || b < NBL) {
                c32 v[RL];
#pragma unroll
                for (int r = 0; r < RL; ++r) {
                    const c32 a = z[sw_step<NBL>(b, r)];
                    v[r] = r ? cmul(a, c_of(twl[r * NBL + b])) : a;
                }
                Dft<RL>::run(v);
#pragma unroll
                for (int q = 0; q < RL; ++q) {
                    const double xr = v[q].x, xi = v[q].y;
                    acc[m][q] = fma(xi, xi, fma(xr, xr, acc[m][q]));
                }
            }
        }
        __syncthreads();  // z is rewritten by the next transform
    }
#pragma unroll
    for (int m = 0; m < ML; ++m) {
        const int b = tid + m * T;
        if (NBL % T != 0 && b >= NBL) continue;
#pragma unroll
        for (int q = 0; q < RL; ++q)
            if (acc[m][q] != 0.0) atomicAdd(prow + b + q * NBL, acc[m][q]);
    }
}

// G / 2 + 1 workgroups (classes) per k-block, the classes of a k-block 8 apart so that they
// share an XCD's L2 (items of 2, 4 and 8 k-blocks, which flush fewer sums, were 1, 4 and 9 %
// slower).  What bounds the kernel is VALU issue and, with two barriers a pass, the waves a
// CU holds: at H = L / 2 twice the workgroups fit that a transform of L points allows, and
// plans of 8 to 10 points a thread leave 20 waves a CU where radix-16 passes of 16 points
// left 15 (10.6 against 13.7 ms at 479,980 series of 10,000 frames; 14.2 for whole
// transforms with an unpacking step).  262,144 series of 20,000 frames: 14.0 ms, against
// 55 for whole transforms through a scratch in HBM; folding those once more (G = 8, H =
// 5,120) 16.  Error of g2 against 64 bits: 7e-6 -> 8e-7 and 4e-6 -> 1.3e-6.
template <typename E, typename Plan, int G>
__global__ __launch_bounds__(Plan::T, Plan::T == 640 ? 5 : 4) void fft_spectra_kernel(
    const uint8_t* __restrict__ xs, const BinDev* __restrict__ bins,
    const KbWork* __restrict__ work, int n_work, const float2* __restrict__ tw,
    double* __restrict__ power) {
    constexpr int H = Plan::L, T = Plan::T, NC = G / 2 + 1;
    __shared__ c32 z[H];
    __shared__ c32 tab2[Plan::P2];
    __shared__ c32 tab3[Plan::P3];
    const int bx = blockIdx.x;
    const int i = bx / (8 * NC) * 8 + (bx & 7);
    const int cls = NC - 1 - (bx >> 3) % NC;
    if (i >= n_work) return;
    const KbWork w = work[i];
    const BinDev bd = bins[w.bin];
    const int nser = min(KB, bd.npix - w.kb * KB);
    const int64_t kb = (bd.idx_off + (int64_t)w.kb * KB) / KB;
    const uint8_t* rows = xs + kb * (KB / 2) * ((int64_t)H * G * sizeof(E));
    const float2* twl = tw + H;
    const float2* uw = tw + 2 * H;
    double* prow = power + ((int64_t)w.bin * NC + cls) * H;
    for (int m = threadIdx.x; m < Plan::P2; m += T) tab2[m] = c_of(tw[m * (H / Plan::P2)]);
    if (Plan::NP == 4)
        for (int m = threadIdx.x; m < Plan::P3; m += T) tab3[m] = c_of(tw[m * (H / Plan::P3)]);
    if (cls == 0)
        spectra_class<E, Plan, G, PAIR_PLAIN>(rows, nser, 0, twl, uw, prow, z, tab2, tab3);
    else if (cls == G / 2)
        spectra_class<E, Plan, G, PAIR_MOD>(rows, nser, cls, twl, uw, prow, z, tab2, tab3);
    else
        spectra_class<E, Plan, G, SINGLE>(rows, nser, cls, twl, uw, prow, z, tab2, tab3);
}

// Num(tau) = sum_f P_f cos(2 pi f tau / Nf) / Nf over f < Nf in FP64, in two steps of A and B
// terms, A B = Nf (one of Nf / 2 terms a lag was 0.41 ms at 20 bins x 10,000 frames and 0.83 at 10
// x 20,000, against 0.04 and 0.05).  With f = A k1 + k0 and tau0 = tau mod B
//   U[k0][tau0] = sum_{k1 < B} P_{A k1 + k0} exp(2 pi i k1 tau0 / B),
//   Num(tau) = Re sum_{k0 < A} U[k0][tau0] exp(2 pi i k0 tau / Nf) / Nf.
// P is even, so the terms k0 and A - k0 are equal: k0 = 0 .. A / 2 are enough.
// The rows of `power` are the classes' sums [class c <= G/2][k < H]: bin f = G k + c, and
// f = Nf - G k - c for the classes past G/2.  The pair classes hold every bin twice, as f
// and Nf - f (but f = 0 and L once), each time the same |X_1|^2 + |X_2|^2 plus a term that
// changes sign: P_f is their mean.
__device__ __forceinline__ double power_of(const double* __restrict__ row, int G, int H, int f) {
    int c = f % G, k = f / G;
    if (2 * c > G) {  // the mirror of a class below G/2: Nf - f = G (H - 1 - k) + G - c
        c = G - c;
        k = H - 1 - k;
    }
    const double p = row[c * H + k];
    if (c != 0 && 2 * c != G) return p;
    const int m = c ? H - 1 - k : (k ? H - k : 0);
    return 0.5 * (p + row[c * H + m]);
}
// The B of a length: a divisor with A = Nf / B even, near where the steps' terms, B for each of
// Nf / 2 sums and A / 2 for each of up to Nf / 2 lags, are fewest.
constexpr int INV_B = 512;
int fft_inverse_b(const FftShape& f) {
    const int nf = f.G * f.H;
    int best = 1;
    for (int b = 1; b <= INV_B; ++b)
        if (nf % (2 * b) == 0 && b + nf / b / 2 < best + nf / best / 2) best = b;
    return best;
}

// Step 1, grid (A / 2 + 1, bins): the twiddles and the P of one k0 in LDS, a thread a tau0.
__global__ __launch_bounds__(256) void fft_inverse_cols_kernel(const double* __restrict__ power,
                                                               int G, int H, int B,
                                                               double2* __restrict__ u) {
    __shared__ double2 tw[INV_B];
    __shared__ double pk[INV_B];
    const int nf = G * H, A = nf / B, k0 = blockIdx.x;
    const double* row = power + (int64_t)blockIdx.y * (G / 2 + 1) * H;
    for (int i = threadIdx.x; i < B; i += 256) {
        double s, c;
        sincospi(2.0 * i / B, &s, &c);
        tw[i] = make_double2(c, s);
        const int f = A * i + k0;
        pk[i] = power_of(row, G, H, 2 * f > nf ? nf - f : f);
    }
    __syncthreads();
    double2* out = u + ((int64_t)blockIdx.y * (A / 2 + 1) + k0) * B;
    for (int t0 = threadIdx.x; t0 < B; t0 += 256) {
        double x = 0.0, y = 0.0;
        int j = 0;  // k1 t0 mod B
        for (int k1 = 0; k1 < B; ++k1) {
            x = fma(pk[k1], tw[j].x, x);
            y = fma(pk[k1], tw[j].y, y);
            j += t0;
            j -= j >= B ? B : 0;
        }
        out[t0] = make_double2(x, y);
    }
}

// Step 2, grid (ceil(N / 256), bins), a thread a lag: the cosines of k0 = 4 m + r by four
// rotations (each turning by 4 theta, theta = 2 pi tau / Nf), so four dependent chains overlap;
// the partial sums are joined in a fixed order.
__global__ __launch_bounds__(256) void fft_inverse_rows_kernel(const double2* __restrict__ u,
                                                               int nf, int B, int nframes,
                                                               double* __restrict__ num) {
    const int tau = blockIdx.x * 256 + threadIdx.x;
    if (tau >= nframes) return;
    const int half = nf / B / 2;
    const double2* col = u + (int64_t)blockIdx.y * (half + 1) * B + tau % B;
    double c[4], s[4], acc[4] = {};
#pragma unroll
    for (int r = 0; r < 4; ++r)
        sincospi(2.0 * (double)((int64_t)r * tau % nf) / nf, &s[r], &c[r]);
    double c4, s4;
    sincospi(2.0 * (double)((int64_t)4 * tau % nf) / nf, &s4, &c4);
    auto term = [&](int k0, int r) {
        const double2 x = col[(int64_t)k0 * B];
        return x.x * c[r] - x.y * s[r];
    };
    const double first = col[0].x;
    int k0 = 0;
    for (; k0 + 4 <= half; k0 += 4)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            acc[r] += term(k0 + r, r);
            const double cn = c[r] * c4 - s[r] * s4;
            s[r] = s[r] * c4 + c[r] * s4;
            c[r] = cn;
        }
    double last = 0.0;  // k0 = half, counted once
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (k0 + r < half) acc[r] += term(k0 + r, r);
        if (k0 + r == half) last = term(half, r);
    }
    num[(int64_t)blockIdx.y * nframes + tau] =
        (last - first + 2.0 * ((acc[0] + acc[1]) + (acc[2] + acc[3]))) / nf;
}

// ------------------------------------------------------------------ launchers
// Plans: H points, threads, radices.
using Plan256 = FftPlan<256, 64, 4, 4, 4, 4>;
using Plan320 = FftPlan<320, 64, 5, 8, 8, 1>;
using Plan512 = FftPlan<512, 64, 8, 8, 8, 1>;
using Plan640 = FftPlan<640, 64, 10, 8, 8, 1>;
using Plan1024 = FftPlan<1024, 128, 16, 8, 8, 1>;
using Plan1280 = FftPlan<1280, 128, 16, 8, 10, 1>;
using Plan1600 = FftPlan<1600, 192, 10, 16, 10, 1>;
using Plan2048 = FftPlan<2048, 256, 8, 8, 8, 4>;
using Plan2560 = FftPlan<2560, 256, 16, 4, 8, 5>;
using Plan3200 = FftPlan<3200, 448, 8, 8, 5, 10>;
using Plan4096 = FftPlan<4096, 256, 16, 16, 16, 1>;
using Plan5120 = FftPlan<5120, 640, 8, 8, 8, 10>;
using Plan6400 = FftPlan<6400, 832, 8, 8, 10, 10>;
using Plan8192 = FftPlan<8192, 1024, 8, 8, 8, 16>;
using Plan10240 = FftPlan<10240, 1024, 16, 10, 8, 8>;
using Plan12800 = FftPlan<12800, 1024, 16, 10, 10, 8>;
using Plan16384 = FftPlan<16384, 1024, 16, 8, 8, 16>;

// Series lengths L = G H / 2 with their plan.  Each L is one of the lengths a series of N
// frames may be padded to (the smallest with L >= N); H is a multiple of 64 (gather_pm_kernel).
// A finer set than the powers of two and five quarters of them: 490 x 694 x 229 0.74 -> 0.38 ms
// a call (1,024 -> 512), 333 x 335 x 6,000 2.8 -> 2.5 (8,192 -> 6,400), 201 x 203 x 12,000
// 3.2 -> 2.9 (16,384 -> 12,800).
// A call of 8-bit frames at N = L, 256 x 256 pixels in 5 bins, ms, whole transforms at their finest
// length -> these: 512 0.38 -> 0.15, 640 0.38 -> 0.19, 1,024 0.39 -> 0.22, 1,280 0.51 -> 0.33, 2,048 0.53 ->
// 0.38, 2,560 0.79 -> 0.54, 3,200 0.93 -> 0.72, 4,096 0.99 -> 0.72, 5,120 2.20 -> 1.04, 6,400 2.52 -> 1.36,
// 8,192 2.61 -> 1.59, 10,240 3.25 -> 2.13, 12,800 4.73 -> 3.32, 16,384 4.92 -> 3.62, 20,480 16.0 -> 4.65,
// 25,600 18.4 -> 5.92; 160 x 160: 32,768 11.7 -> 3.37, 40,960 14.8 -> 4.22, 65,536 26.0 -> 7.03, 81,920
// 33.9 -> 9.22, 131,072 64.9 -> 19.8.
#define DXG2_FFT_SHAPES(X)                                                               \
    X(256, 4) X(320, 4) X(512, 4) X(640, 4) X(1024, 4) X(1280, 4) X(1600, 4) X(2048, 4)  \
    X(2560, 4) X(3200, 4) X(4096, 4) X(5120, 4) X(6400, 4) X(8192, 4) X(10240, 4)        \
    X(12800, 4) X(16384, 4) X(10240, 8) X(16384, 8) X(10240, 16) X(16384, 16)

#define DXG2_FFT_CHECK(HH, GG) \
    static_assert(HH % (256 / PM_KPB / (GG / 2)) == 0, "a gather workgroup's points divide H");
DXG2_FFT_SHAPES(DXG2_FFT_CHECK)
#undef DXG2_FFT_CHECK

bool fft_shape(int n, FftShape* out) {
    int best = 0;
#define DXG2_FFT_SHAPE(HH, GG)                                     \
    if (HH * GG / 2 >= n && (!best || HH * GG / 2 < best)) {       \
        best = HH * GG / 2;                                        \
        *out = FftShape{best, HH, GG, Plan##HH::RL};               \
    }
    DXG2_FFT_SHAPES(DXG2_FFT_SHAPE)
#undef DXG2_FFT_SHAPE
    return best > 0;
}

template <typename E, bool SGN, int G>
static void gather_pm_typed(const uint8_t* frames, int64_t hw, int nframes, int H,
                            const int32_t* pix_idx, const int32_t* quad_kb, const BinDev* bins,
                            const KbWork* work, int n_work, uint8_t* xs, int64_t* sums,
                            hipStream_t s) {
    constexpr int SEG = 256 / PM_KPB / (G / 2);  // divides every H (checked above)
    gather_pm_kernel<E, SGN, PM_KPB, G>
        <<<dim3((unsigned)n_work, (unsigned)(H / SEG)), 256, 0, s>>>(
            frames, hw, nframes, H, pix_idx, quad_kb, bins, work, xs, sums);
}

template <int G>
static void gather_pm_fold(const uint8_t* frames, int dtype, int64_t hw, int nframes, int H,
                           const int32_t* pix_idx, const int32_t* quad_kb, const BinDev* bins,
                           const KbWork* work, int n_work, uint8_t* xs, int64_t* sums,
                           hipStream_t s) {
    if (dtype == DXG2_U16)
        gather_pm_typed<uint16_t, false, G>(frames, hw, nframes, H, pix_idx, nullptr, bins, work,
                                            n_work, xs, sums, s);
    else if (dtype == DXG2_I8)
        gather_pm_typed<uint8_t, true, G>(frames, hw, nframes, H, pix_idx, quad_kb, bins, work,
                                          n_work, xs, sums, s);
    else
        gather_pm_typed<uint8_t, false, G>(frames, hw, nframes, H, pix_idx, quad_kb, bins, work,
                                           n_work, xs, sums, s);
}

void launch_gather_pm(const uint8_t* frames, int dtype, int64_t hw, int nframes,
                      const FftShape& shape, const int32_t* pix_idx, const int32_t* quad_kb,
                      const BinDev* bins, int n_bins, const KbWork* work, int n_work,
                      uint8_t* xs, int64_t* sums, hipStream_t s) {
    if (n_bins <= 0 || n_work <= 0) return;
    // aligned quad loads need 4 | hw and a 4-aligned frame pointer
    if (hw % 4 != 0 || reinterpret_cast<uintptr_t>(frames) % 4 != 0) quad_kb = nullptr;
    if (shape.G == 4)
        gather_pm_fold<4>(frames, dtype, hw, nframes, shape.H, pix_idx, quad_kb, bins, work,
                          n_work, xs, sums, s);
    else if (shape.G == 8)
        gather_pm_fold<8>(frames, dtype, hw, nframes, shape.H, pix_idx, quad_kb, bins, work,
                          n_work, xs, sums, s);
    else
        gather_pm_fold<16>(frames, dtype, hw, nframes, shape.H, pix_idx, quad_kb, bins, work,
                           n_work, xs, sums, s);
}

template <typename Plan, int G>
static void spectra_dtype(int dtype, const uint8_t* xs, const BinDev* bins, const KbWork* work,
                          int n_work, const float2* tw, double* power, hipStream_t s) {
    const dim3 grid((unsigned)((n_work + 7) / 8 * 8 * (G / 2 + 1)));
    if (dtype == DXG2_U16)
        fft_spectra_kernel<uint16_t, Plan, G>
            <<<grid, Plan::T, 0, s>>>(xs, bins, work, n_work, tw, power);
    else if (dtype == DXG2_I8)
        fft_spectra_kernel<int8_t, Plan, G>
            <<<grid, Plan::T, 0, s>>>(xs, bins, work, n_work, tw, power);
    else
        fft_spectra_kernel<uint8_t, Plan, G>
            <<<grid, Plan::T, 0, s>>>(xs, bins, work, n_work, tw, power);
}

int launch_fft_power(const FftShape& shape, int dtype, const uint8_t* xs, const BinDev* bins,
                     const KbWork* work, int n_work, const float2* tw, double* power,
                     hipStream_t s) {
    if (n_work <= 0) return 0;
#define DXG2_FFT_CASE(HH, GG)                                                        \
    if (shape.H == HH && shape.G == GG) {                                            \
        spectra_dtype<Plan##HH, GG>(dtype, xs, bins, work, n_work, tw, power, s);    \
        return 0;                                                                    \
    }
    DXG2_FFT_SHAPES(DXG2_FFT_CASE)
#undef DXG2_FFT_CASE
    return -1;
}

size_t fft_inverse_elems(const FftShape& f) {
    const int b = fft_inverse_b(f);
    return ((size_t)(f.G * f.H / b / 2) + 1) * b;
}

void launch_fft_inverse(const double* power, const FftShape& shape, int n_bins, int nframes,
                        double2* work, double* num, hipStream_t s) {
    if (n_bins <= 0) return;
    const int nf = shape.G * shape.H, b = fft_inverse_b(shape);
    fft_inverse_cols_kernel<<<dim3((unsigned)(nf / b / 2 + 1), (unsigned)n_bins), 256, 0, s>>>(
        power, shape.G, shape.H, b, work);
    fft_inverse_rows_kernel<<<dim3((unsigned)((nframes + 255) / 256), (unsigned)n_bins), 256, 0,
                              s>>>(work, nf, b, nframes, num);
}

}  // namespace dxg2
