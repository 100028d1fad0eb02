// Narrow pixels: the counts of photon-counting movies are mostly 0 and 1, and a pixel whose
// counts never exceed NARROW_MAX = 4 in magnitude can be correlated in FP4: the matrix cores
// multiply FP4 at twice the rate of i8 and a frame takes half the bytes.  The codes are exact
// (counts in units of 1/2) and so are the products' sums (multiples of 1/4 below 2^22, in
// FP32), so numerators and frame sums are the same integers as those of the i8 path.
//
// A dense call on a plan with a narrow slab (uint8 / int8, see narrow_applies() in capi.hip)
// goes, all decided on the device:
//  * narrow_sample_kernel looks at NARROW_SAMPLES frames spread over the stack and sets
//    route[0]: NARROW_F4 when few pixels are expected to be wide (a count above NARROW_MAX in
//    some frame), else NARROW_OFF;
//  * NARROW_F4: gather_band_f4_kernel writes every pixel's codes to the narrow slab and flags
//    the wide pixels; wide_compact_kernel lists them per bin, narrow_mask_kernel clears their
//    codes, wide_gather_kernel writes them to the first k-blocks of the bin's i8 slab, and
//    the numerators are the narrow slab's Gram (gram_f4_queue_kernel) plus the i8 Gram of
//    those k-blocks;
//  * NARROW_OFF: gather_band_kernel fills the i8 slab and its Gram covers every k-block.
// Kernels of the other route return at once.  nwkb[b] is the number of k-blocks of bin b the
// i8 Gram reads, nwkb[n_bins] the largest, nwkb[n_bins + 1 + b] the wide pixels.
#include "dxg2_internal.h"

namespace dxg2 {

constexpr int NARROW_SAMPLES = 64;           // frames
constexpr int NARROW_SAMPLE_KB = 1024;       // k-blocks (at the line of 30 % of 65,536 pixels
                                             // about 20,000 turn wide over the stack)

// One thread per list entry of every `stride`-th k-block: wide in the first half of the sampled
// frames (ctl[1]), in any of them (ctl[2]), of ctl[4] pixels; the last block decides (ctl[0] is
// the route, ctl[3] counts blocks; all zeroed beforehand).  Pixels that turn wide go on
// appearing at the rate of the second half at most (hot pixels are all seen in the first
// frames, and the rest saturate), so
//   wide <= ctl[2] + (ctl[2] - ctl[1]) (N - n) / (n / 2).
// The line is at 30 % of the pixels: a wide pixel costs its share of the i8 Gram, of the time
// of which the FP4 Gram of every pixel takes about half.
template <bool SGN>
__global__ __launch_bounds__(256) void narrow_sample_kernel(
    const uint8_t* __restrict__ frames, int64_t hw, int nframes,
    const int32_t* __restrict__ pix, int64_t n_entries, int stride, int* __restrict__ ctl) {
    const int n = min(nframes, NARROW_SAMPLES);
    const int64_t i0 = blockIdx.x * 256 + (int64_t)threadIdx.x;
    const int64_t k = i0 / KB * stride * KB + i0 % KB;
    const int p = k < n_entries ? pix[k] : -1;
    bool first = false, any = false;
    if (p >= 0) {
#pragma unroll 8
        for (int i = 0; i < n; ++i) {
            const int t = (int)(((2 * (int64_t)i + 1) * nframes) / (2 * n));
            const uint8_t x = frames[(int64_t)t * hw + p];
            const int v = SGN ? (int)(int8_t)x : (int)x;
            const bool wide = v > NARROW_MAX || v < -NARROW_MAX;
            any |= wide;
            first |= wide && 2 * i < n;
        }
    }
    const int nf = __popcll(__ballot(first)), na = __popcll(__ballot(any));
    const int np = __popcll(__ballot(p >= 0));
    if ((threadIdx.x & 63) == 0) {
        if (nf) atomicAdd(ctl + 1, nf);
        if (na) atomicAdd(ctl + 2, na);
        if (np) atomicAdd(ctl + 4, np);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        __threadfence();
        if (atomicAdd(ctl + 3, 1) == (int)gridDim.x - 1) {
            const double f = atomicAdd(ctl + 1, 0), a = atomicAdd(ctl + 2, 0);
            const double half = (n + 1) / 2;  // frames with 2 i < n
            const double grow = n > 1 ? (a - f) / (n - half) : 0.0;
            const double wide = a + grow * (double)(nframes - n);
            ctl[0] = wide <= 0.3 * (double)atomicAdd(ctl + 4, 0) ? NARROW_F4 : NARROW_OFF;
        }
    }
}

// nwkb from the wide pixels' counts (nwkb + n_bins + 1) and the route.
__global__ __launch_bounds__(256) void narrow_clip_kernel(const BinDev* __restrict__ bins,
                                                          int n_bins, const int* __restrict__ route,
                                                          int* __restrict__ nwkb) {
    const int* count = nwkb + n_bins + 1;
    for (int b = threadIdx.x; b < n_bins; b += 256) {
        const int clip = route[0] == NARROW_F4 ? (count[b] + KB - 1) / KB : bins[b].nkb;
        nwkb[b] = clip;
        atomicMax(nwkb + n_bins, clip);
    }
}

// Clear the codes of the wide pixels in the narrow slab.  Grid (k-blocks of the longest bin,
// bins, frame chunks); a k-block without wide pixels costs one load of its list and flags.
constexpr int MASK_GROUPS = 16;  // 32-frame groups per wave
__global__ __launch_bounds__(256) void narrow_mask_kernel(const int32_t* __restrict__ pix,
                                                          const BinDev* __restrict__ bins,
                                                          const uint8_t* __restrict__ flag,
                                                          const int* __restrict__ route,
                                                          int n_bins, int nrows,
                                                          const int* __restrict__ nwkb,
                                                          int8_t* __restrict__ slab4) {
    if (route[0] != NARROW_F4 || nwkb[n_bins] == 0) return;
    const int b = blockIdx.y, kb = blockIdx.x;
    const BinDev bd = bins[b];
    if (kb >= bd.nkb || nwkb[b] == 0) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int p = pix[bd.idx_off + (int64_t)kb * KB + lane];
    const uint64_t wide = __ballot(p >= 0 && flag[p]);
    if (wide == 0) return;
    const uint32_t half = (uint32_t)(lane < 32 ? wide : wide >> 32);  // pixels of this lane's half
    uint32_t keep[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        keep[w] = 0u;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (!(half >> (8 * w + e) & 1)) keep[w] |= 0xFu << (8 * e);
            if (!(half >> (8 * w + 4 + e) & 1)) keep[w] |= 0xF0u << (8 * e);
        }
    }
    const int ng = nrows >> 5;
    const int g0 = (blockIdx.z * 4 + wave) * MASK_GROUPS;
    int8_t* base = slab4 + bd.slab_off / 2 + (int64_t)kb * ng * 1024 + lane * 16;
#pragma unroll 4
    for (int g = g0; g < min(ng, g0 + MASK_GROUPS); ++g) {
        uint4* x = reinterpret_cast<uint4*>(base + (int64_t)g * 1024);
        uint4 v = *x;
        v.x &= keep[0];
        v.y &= keep[1];
        v.z &= keep[2];
        v.w &= keep[3];
        *x = v;
    }
}

void launch_narrow_sample(const uint8_t* frames, int dtype, int64_t hw, int nframes,
                          const int32_t* pix, int64_t n_entries, int* ctl, hipStream_t s) {
    const int64_t nkb = n_entries / KB;  // the lists are padded to whole k-blocks
    const int stride = (int)((nkb + NARROW_SAMPLE_KB - 1) / NARROW_SAMPLE_KB);
    const dim3 grid((unsigned)((nkb + stride - 1) / stride * KB + 255) / 256);
    if (dtype == DXG2_I8)
        narrow_sample_kernel<true><<<grid, 256, 0, s>>>(frames, hw, nframes, pix, n_entries, stride,
                                                        ctl);
    else
        narrow_sample_kernel<false><<<grid, 256, 0, s>>>(frames, hw, nframes, pix, n_entries,
                                                         stride, ctl);
}

void launch_narrow_clip(const BinDev* bins, int n_bins, const int* route, int* nwkb,
                        hipStream_t s) {
    narrow_clip_kernel<<<1, 256, 0, s>>>(bins, n_bins, route, nwkb);
}

void launch_narrow_mask(const int32_t* pix, const BinDev* bins, int n_bins, int max_nkb,
                        const uint8_t* flag, const int* route, int nrows, const int* nwkb,
                        int8_t* slab4, hipStream_t s) {
    if (n_bins <= 0 || max_nkb <= 0) return;
    const int chunks = ((nrows >> 5) + 4 * MASK_GROUPS - 1) / (4 * MASK_GROUPS);
    narrow_mask_kernel<<<dim3((unsigned)max_nkb, (unsigned)n_bins, (unsigned)chunks), 256, 0, s>>>(
        pix, bins, flag, route, n_bins, nrows, nwkb, slab4);
}

}  // namespace dxg2
