// Dense frames -> per-pixel event lists, on the GPU: the FramesCompressor layout of the
// event correlator's input (correlator/event.py:207-321).
//
// For every pixel p in raster order, its samples with value > 0 (signed for int8, as
// `frames > 0` in event.py:276,293) are listed in frame order: data[offsets[p] ..
// offsets[p+1]) and the matching frame indices times[...].
//
// Whole stack (compress_all_stack, event.py:267-284): a count pass, a scan over the frame
// chunks and one over the pixels into offsets, and a fill pass that re-reads the frames and
// writes each pixel's events from its offset on.  Loads are wide whatever their alignment:
// frames of odd sizes start at any byte, and one byte a thread and load took 1.80 + 3.36 ms
// where these take 0.40 + 0.53 ms (1030 x 1065 x 2,000, 44 million events).
//
// Streaming (process_frame / get_compacted_events, event.py:287-321): each pushed frame
// appends its events to per-pixel slots of max_nnz entries; compaction scans the
// per-pixel counters and copies the slots into the same 1-D layout.
#include <algorithm>
#include <type_traits>

#include "dxg2_internal.h"

namespace dxg2 {

template <typename T>
__device__ __forceinline__ bool positive(T v) {
    return v > T(0);
}

template <typename T>
struct Words {
    static constexpr int PIXELS = 4 / sizeof(T);
    static constexpr int FRAMES = 32 / PIXELS;  // 8 or 16: the bits of a sample
    static constexpr uint32_t FIELD = FRAMES == 8 ? 0xFFu : 0xFFFFu;  // a pixel's bits of a mask
    static constexpr uint32_t SAMPLE = sizeof(T) == 1 ? 0xFFu : 0xFFFFu;
    static constexpr uint32_t HIGH = sizeof(T) == 1 ? 0x80808080u : 0x80008000u;
    // The high bit of every positive sample of w.
    __device__ __forceinline__ static uint32_t flags(uint32_t w) {
        const uint32_t low = (w & ~HIGH) + ~HIGH;  // high bit: low bits not all zero
        return (std::is_signed<T>::value ? low & ~w : low | w) & HIGH;
    }
};

// A thread's word of every frame: pixels PIXELS v .. of which `have` lie in the frame, by one
// load at any byte alignment (frames of odd sizes start anywhere).  The frame's last word is
// loaded from its last 4 bytes and shifted, without a branch beside the loads of a wave, which
// would keep them from being in flight together.  TINY: frames below 4 bytes, byte by byte.
template <typename T, bool TINY>
struct WordReader {
    static constexpr int P = Words<T>::PIXELS;
    const T* row;
    int64_t hw;
    int64_t at;
    int have, shift;
    __device__ __forceinline__ WordReader(const T* frames, int64_t hw_, int64_t v)
        : row(frames), hw(hw_) {
        have = (int)max((int64_t)0, min((int64_t)P, hw - v * P));
        at = TINY ? v * P : max((int64_t)0, min(v * P, hw - P));
        shift = have > 0 ? 8 * (int)sizeof(T) * (int)(v * P - at) : 0;
    }
    __device__ __forceinline__ uint32_t word(int t) const {
        const T* p = row + (int64_t)t * hw + at;
        uint32_t w = 0u;
        if (TINY) {
            for (int k = 0; k < have; ++k)
                w |= ((uint32_t)p[k] & Words<T>::SAMPLE) << (8 * (int)sizeof(T) * k);
        } else {
            __builtin_memcpy(&w, p, 4);
        }
        return w >> shift;
    }
    // FRAMES words from frame t on, zero from t1 on (loads past t1 repeat frame t1 - 1); a lane
    // past the frame's end gets zeros.
    __device__ __forceinline__ void words(uint32_t (&w)[Words<T>::FRAMES], int t, int t1) const {
#pragma unroll
        for (int i = 0; i < Words<T>::FRAMES; ++i) w[i] = word(min(t + i, t1 - 1));
#pragma unroll
        for (int i = 0; i < Words<T>::FRAMES; ++i) w[i] = t + i < t1 && have > 0 ? w[i] : 0u;
    }
};

// The frame axis is cut into C chunks of F frames: per-chunk counts cnt[c][p] -> per-pixel
// bases within the pixel's list (cnt becomes base in place, total into offsets[p]) ->
// exclusive scan over pixels -> fill.  C is what fills the chip: about a million words in
// flight, chunks of at least 32 frames (each chunk costs four passes over 4 bytes a pixel).
int compress_chunks(int nframes, int64_t hw) {
    const int64_t c = std::min<int64_t>(((int64_t)1 << 20) / std::max<int64_t>(hw / 4, 1),
                                        nframes / 32);
    return (int)std::max<int64_t>(1, std::min<int64_t>(c, 64));
}

// Counts: the flags of a thread's words are added to a word of 8-bit (16-bit) counters, emptied
// every 255 frames.  Bound by HBM.
template <typename T, bool TINY>
__global__ __launch_bounds__(256) void compress_count_kernel(const T* __restrict__ frames,
                                                             int nframes, int64_t hw, int F,
                                                             uint32_t* __restrict__ cnt) {
    using W = Words<T>;
    constexpr int P = W::PIXELS, BITS = 8 * sizeof(T);
    const int64_t v = blockIdx.x * 256 + (int64_t)threadIdx.x;
    if (v * P >= hw) return;
    const WordReader<T, TINY> in(frames, hw, v);
    const int t0 = blockIdx.y * F, t1 = min(nframes, t0 + F);
    uint32_t n[P] = {};
    for (int ta = t0; ta < t1; ta += 255) {
        const int tb = min(t1, ta + 255);
        uint32_t acc = 0u;
#pragma unroll 8
        for (int t = ta; t < tb; ++t) acc += W::flags(in.word(t)) >> (BITS - 1);
#pragma unroll
        for (int k = 0; k < P; ++k) n[k] += (acc >> (BITS * k)) & ((1u << BITS) - 1u);
    }
#pragma unroll
    for (int k = 0; k < P; ++k)
        if (k < in.have) cnt[blockIdx.y * hw + v * P + k] = n[k];
}

// cnt[c][p] -> exclusive base over c (in place); offsets[p] = the pixel's total.
__global__ void compress_chunk_scan_kernel(uint32_t* __restrict__ cnt, int64_t hw, int C,
                                           uint32_t* __restrict__ total) {
    for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < hw;
         p += (int64_t)gridDim.x * blockDim.x) {
        uint32_t run = 0;
        for (int c = 0; c < C; ++c) {
            const uint32_t n = cnt[(int64_t)c * hw + p];
            cnt[(int64_t)c * hw + p] = run;
            run += n;
        }
        total[p] = run;
    }
}

// FRAMES frames' words of a thread as one 32-bit mask of positive samples, bit FRAMES k + i for
// pixel k of frame i: the fill passes loop over a lane's events (a few a wave and mask) and not
// over samples.
template <typename T>
__device__ __forceinline__ uint32_t events_mask(const uint32_t (&w)[Words<T>::FRAMES]) {
    uint32_t mask = 0u;
#pragma unroll
    for (int i = 0; i < Words<T>::FRAMES; ++i)
        mask |= Words<T>::flags(w[i]) >> (Words<T>::FRAMES - 1 - i);
    return mask;
}

// Fill of small detectors: each (word, chunk) thread writes from offsets[p] + base[c][p].
template <typename T, bool TINY>
__global__ __launch_bounds__(256) void compress_fill_kernel(const T* __restrict__ frames,
                                                            int nframes, int64_t hw, int F,
                                                            const uint32_t* __restrict__ base,
                                                            const uint32_t* __restrict__ offsets,
                                                            int32_t* __restrict__ times,
                                                            T* __restrict__ data) {
    using W = Words<T>;
    constexpr int P = W::PIXELS, G = W::FRAMES;
    __shared__ uint32_t held[G][256];  // a thread's words, for its events' values
    const int64_t v = blockIdx.x * 256 + (int64_t)threadIdx.x;
    if (v * P >= hw) return;
    const WordReader<T, TINY> in(frames, hw, v);
    const int c = blockIdx.y;
    const int t0 = c * F, t1 = min(nframes, t0 + F);
    uint32_t cur[P];
#pragma unroll
    for (int k = 0; k < P; ++k)
        cur[k] = k < in.have ? offsets[v * P + k] + base[(int64_t)c * hw + v * P + k] : 0u;
    uint32_t w[G];
    in.words(w, t0, t1);
    for (int t = t0; t < t1; t += G) {
        const uint32_t mask = events_mask<T>(w);
#pragma unroll
        for (int i = 0; i < G; ++i) held[i][threadIdx.x] = w[i];
        in.words(w, t + G, t1);
#pragma unroll
        for (int k = 0; k < P; ++k)
            for (uint32_t m = (mask >> (k * G)) & W::FIELD; m; m &= m - 1) {
                const int i = __builtin_ctz(m);
                times[cur[k]] = t + i;
                data[cur[k]] = (T)(held[i][threadIdx.x] >> (k * 8 * (int)sizeof(T)));
                ++cur[k];
            }
    }
}

// Fill of large detectors: a workgroup takes 64 words of pixels, whose lists are one run of the
// output, over all frames, and assembles the run in LDS.  Written event by event, a stack's
// lists are more open lines than the caches hold, and every 4-byte and 1-byte store goes to
// memory by itself (2.0 ms at the size above).  Wave g has the frames FRAMES g .. of each
// 8 FRAMES, so the ranks of its events follow from the masks' counts of the waves before it,
// byte k of a word for pixel k.  Places in the run (below 65,536) are four 16-bit fields of one
// word, so a lane's loop over its events picks a pixel's by a shift.  A longer run goes out
// event by event.
constexpr int COMPRESS_RUN = 11264;  // events
template <typename T, bool TINY>
__global__ __launch_bounds__(512) void compress_tile_kernel(const T* __restrict__ frames,
                                                            int nframes, int64_t hw,
                                                            const uint32_t* __restrict__ offsets,
                                                            int32_t* __restrict__ times,
                                                            T* __restrict__ data, int n_tiles) {
    using W = Words<T>;
    constexpr int P = W::PIXELS, G = W::FRAMES, TP = 64 * P;
    constexpr int RUN = sizeof(T) == 1 ? COMPRESS_RUN : COMPRESS_RUN / 2;
    __shared__ int32_t run_t[RUN];
    __shared__ T run_d[RUN];
    __shared__ uint32_t held[G][512];
    __shared__ uint32_t counts[2][8][64];
    // neighbouring tiles share lines of the frames: a stretch of them to each XCD
    const int per = (n_tiles + 7) / 8;
    const int tile = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    if (tile >= n_tiles) return;
    const int lane = threadIdx.x & 63;
    const int g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t p0 = (int64_t)tile * TP, p = p0 + lane * P;
    const WordReader<T, TINY> in(frames, hw, (int64_t)tile * 64 + lane);
    const uint32_t e0 = offsets[p0];
    const uint32_t n_events = offsets[min(hw, p0 + TP)] - e0;
    const bool staged = n_events <= (uint32_t)RUN;
    uint32_t cur[P];
    uint64_t place = 0;
#pragma unroll
    for (int k = 0; k < P; ++k) {
        cur[k] = k < in.have ? offsets[p + k] : e0;
        place |= (uint64_t)(staged ? cur[k] - e0 : 0u) << (16 * k);
    }
    // byte k of x to 16-bit field k
    auto fields = [](uint32_t x) {
        return (uint64_t)__builtin_amdgcn_perm(0u, x, 0x0c010c00u) |
               (uint64_t)__builtin_amdgcn_perm(0u, x, 0x0c030c02u) << 32;
    };
    uint32_t w[G];
    in.words(w, g * G, nframes);
    int buf = 0;
    for (int t0 = 0; t0 < nframes; t0 += 8 * G, buf ^= 1) {
        const int t = t0 + g * G;
        const uint32_t mask = events_mask<T>(w);
        uint32_t mine = 0u;
#pragma unroll
        for (int k = 0; k < P; ++k)
            mine |= (uint32_t)__popc((mask >> (k * G)) & W::FIELD) << (8 * k);
        counts[buf][g][lane] = mine;
#pragma unroll
        for (int i = 0; i < G; ++i) held[i][threadIdx.x] = w[i];
        in.words(w, t + 8 * G, nframes);
        __syncthreads();
        uint32_t before = 0u, all = 0u;  // at most 8 FRAMES a byte
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const uint32_t x = counts[buf][q][lane];
            all += x;
            before += q < g ? x : 0u;
        }
        if (staged) {
            const uint64_t first = place + fields(before);
            const T* mine_d = reinterpret_cast<const T*>(&held[0][threadIdx.x]);
            for (uint32_t m = mask; m; m &= m - 1) {
                const int b = __builtin_ctz(m);
                const int k = b / G, i = b % G;
                // events of the pixel in earlier frames of the mask
                const uint32_t rank = __popc(mask & ((1u << b) - 1u) & (~0u << (k * G)));
                const uint32_t at = ((uint32_t)(first >> (16 * k)) & 0xFFFFu) + rank;
                run_t[at] = t + i;
                run_d[at] = mine_d[i * 512 * P + k];
            }
            place += fields(all);
        } else {
#pragma unroll
            for (int k = 0; k < P; ++k) {
                uint32_t at = cur[k] + ((before >> (8 * k)) & 0xFFu);
                for (uint32_t m = (mask >> (k * G)) & W::FIELD; m; m &= m - 1, ++at) {
                    const int i = __builtin_ctz(m);
                    times[at] = t + i;
                    data[at] = (T)(held[i][threadIdx.x] >> (k * 8 * (int)sizeof(T)));
                }
                cur[k] += (all >> (8 * k)) & 0xFFu;
            }
        }
    }
    if (!staged) return;
    __syncthreads();
    for (uint32_t x = threadIdx.x; x < n_events; x += 512) {
        times[e0 + x] = run_t[x];
        data[e0 + x] = run_d[x];
    }
}

static unsigned compress_grid(int64_t n) {
    int64_t g = (n + 255) / 256;
    if (g < 1) g = 1;
    if (g > 65536) g = 65536;
    return (unsigned)g;
}

template <typename T, bool TINY>
static void compress_launch(bool fill, const T* frames, int nframes, int64_t hw, uint32_t* cnt,
                            const uint32_t* offsets, int32_t* times, T* data, hipStream_t s) {
    const int C = compress_chunks(nframes, hw);
    const int F = (nframes + C - 1) / C;
    const int64_t words = (hw + Words<T>::PIXELS - 1) / Words<T>::PIXELS;
    const dim3 grid((unsigned)((words + 255) / 256), (unsigned)C);
    const unsigned tiles = (unsigned)((words + 63) / 64);
    if (!fill)
        compress_count_kernel<T, TINY><<<grid, 256, 0, s>>>(frames, nframes, hw, F, cnt);
    else if (tiles >= 512)  // two workgroups a CU
        compress_tile_kernel<T, TINY><<<(tiles + 7) / 8 * 8, 512, 0, s>>>(
            frames, nframes, hw, offsets, times, data, (int)tiles);
    else
        compress_fill_kernel<T, TINY><<<grid, 256, 0, s>>>(frames, nframes, hw, F, cnt, offsets,
                                                              times, data);
}
template <typename T>
static void compress_dispatch(bool fill, const T* frames, int nframes, int64_t hw, uint32_t* cnt,
                              const uint32_t* offsets, int32_t* times, T* data, hipStream_t s) {
    if (hw >= Words<T>::PIXELS)
        compress_launch<T, false>(fill, frames, nframes, hw, cnt, offsets, times, data, s);
    else
        compress_launch<T, true>(fill, frames, nframes, hw, cnt, offsets, times, data, s);
}

size_t compress_scratch_bytes(int nframes, int64_t hw) {
    return ((size_t)compress_chunks(nframes, hw) * hw + (hw + 1023) / 1024 + 2) * sizeof(uint32_t);
}

void launch_compress_count(int dtype, const void* frames, int nframes, int64_t hw,
                           uint32_t* scratch, uint32_t* offsets, hipStream_t s) {
    if (hw <= 0) return;
    const int C = compress_chunks(nframes, hw);
    uint32_t* cnt = scratch;
    uint32_t* tot = scratch + (size_t)C * hw;
    if (dtype == DXG2_U16)
        compress_dispatch<uint16_t>(false, (const uint16_t*)frames, nframes, hw, cnt, nullptr,
                                    nullptr, nullptr, s);
    else if (dtype == DXG2_I8)
        compress_dispatch<int8_t>(false, (const int8_t*)frames, nframes, hw, cnt, nullptr, nullptr,
                                  nullptr, s);
    else
        compress_dispatch<uint8_t>(false, (const uint8_t*)frames, nframes, hw, cnt, nullptr,
                                   nullptr, nullptr, s);
    compress_chunk_scan_kernel<<<compress_grid(hw), 256, 0, s>>>(cnt, hw, C, offsets);
    launch_excl_scan(offsets, hw, tot, offsets, s);  // offsets[hw] = total
}

void launch_compress_fill(int dtype, const void* frames, int nframes, int64_t hw,
                          const uint32_t* scratch, const uint32_t* offsets, int32_t* times,
                          void* data, hipStream_t s) {
    if (hw <= 0) return;
    uint32_t* base = const_cast<uint32_t*>(scratch);
    if (dtype == DXG2_U16)
        compress_dispatch<uint16_t>(true, (const uint16_t*)frames, nframes, hw, base, offsets,
                                    times, (uint16_t*)data, s);
    else if (dtype == DXG2_I8)
        compress_dispatch<int8_t>(true, (const int8_t*)frames, nframes, hw, base, offsets, times,
                                  (int8_t*)data, s);
    else
        compress_dispatch<uint8_t>(true, (const uint8_t*)frames, nframes, hw, base, offsets, times,
                                   (uint8_t*)data, s);
}

// Streaming: append frame t's events to the per-pixel slots (pixel p owns entries
// [p * max_nnz, (p + 1) * max_nnz)).  A pixel whose slots are full sets *err and keeps
// its count at max_nnz + 1 (so compaction can refuse).
template <typename T>
__global__ void compress_push_kernel(const T* __restrict__ frame, int64_t hw, int t, int max_nnz,
                                     uint32_t* __restrict__ counter, T* __restrict__ events,
                                     int32_t* __restrict__ times, int* __restrict__ err) {
    for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < hw;
         p += (int64_t)gridDim.x * blockDim.x) {
        const T x = frame[p];
        if (!positive(x)) continue;
        const uint32_t c = counter[p];
        if (c < (uint32_t)max_nnz) {
            events[p * max_nnz + c] = x;
            times[p * max_nnz + c] = t;
            counter[p] = c + 1;
        } else {
            counter[p] = (uint32_t)max_nnz + 1;
            *err = 1;
        }
    }
}

template <typename T>
__global__ void compress_compact_kernel(const uint32_t* __restrict__ counter,
                                        const T* __restrict__ events,
                                        const int32_t* __restrict__ times, int64_t hw,
                                        int max_nnz, const uint32_t* __restrict__ offsets,
                                        T* __restrict__ out_data, int32_t* __restrict__ out_times) {
    for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < hw;
         p += (int64_t)gridDim.x * blockDim.x) {
        const uint32_t n = min(counter[p], (uint32_t)max_nnz);
        const uint32_t o = offsets[p];
        for (uint32_t k = 0; k < n; ++k) {
            out_data[o + k] = events[p * max_nnz + k];
            out_times[o + k] = times[p * max_nnz + k];
        }
    }
}

void launch_compress_push(int dtype, const void* frame, int64_t hw, int t, int max_nnz,
                          uint32_t* counter, void* events, int32_t* times, int* err,
                          hipStream_t s) {
    if (hw <= 0) return;
    const unsigned g = compress_grid(hw);
    if (dtype == DXG2_U16)
        compress_push_kernel<uint16_t><<<g, 256, 0, s>>>((const uint16_t*)frame, hw, t, max_nnz,
                                                         counter, (uint16_t*)events, times, err);
    else if (dtype == DXG2_I8)
        compress_push_kernel<int8_t><<<g, 256, 0, s>>>((const int8_t*)frame, hw, t, max_nnz,
                                                       counter, (int8_t*)events, times, err);
    else
        compress_push_kernel<uint8_t><<<g, 256, 0, s>>>((const uint8_t*)frame, hw, t, max_nnz,
                                                        counter, (uint8_t*)events, times, err);
}

void launch_compress_compact(int dtype, const uint32_t* counter, const void* events,
                             const int32_t* times, int64_t hw, int max_nnz, uint32_t* scratch,
                             uint32_t* offsets, void* out_data, int32_t* out_times,
                             hipStream_t s) {
    if (hw <= 0) return;
    launch_copy_u32(counter, offsets, hw, s);
    launch_clamp_u32(offsets, hw, (uint32_t)max_nnz, s);
    launch_excl_scan(offsets, hw, scratch, offsets, s);
    const unsigned g = compress_grid(hw);
    if (dtype == DXG2_U16)
        compress_compact_kernel<uint16_t><<<g, 256, 0, s>>>(counter, (const uint16_t*)events, times,
                                                            hw, max_nnz, offsets,
                                                            (uint16_t*)out_data, out_times);
    else if (dtype == DXG2_I8)
        compress_compact_kernel<int8_t><<<g, 256, 0, s>>>(counter, (const int8_t*)events, times, hw,
                                                          max_nnz, offsets, (int8_t*)out_data,
                                                          out_times);
    else
        compress_compact_kernel<uint8_t><<<g, 256, 0, s>>>(counter, (const uint8_t*)events, times,
                                                           hw, max_nnz, offsets,
                                                           (uint8_t*)out_data, out_times);
}

__global__ void clamp_u32_kernel(uint32_t* __restrict__ p, int64_t n, uint32_t hi) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = min(p[i], hi);
}

void launch_clamp_u32(uint32_t* p, int64_t n, uint32_t hi, hipStream_t s) {
    if (n > 0) clamp_u32_kernel<<<compress_grid(n), 256, 0, s>>>(p, n, hi);
}

}  // namespace dxg2
