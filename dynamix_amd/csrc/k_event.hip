// Event (sparse) correlator kernels.
//
// Reference: EventCorrelator (correlator/event.py:162-204) with event_correlator
// (resources/opencl/evtcorrelator.cl:3-46): one work-item per pixel walks every ordered
// pair j <= i of that pixel's frame-sorted events and does a global atomic
// res[bin][t_i - t_j] += d_i d_j, plus sums[bin][t_i] += d_i.
//
// Here:
//  * work items are (bin, range of the bin's pixel list) x (lag window), and pairs go to an LDS
//    lag histogram (EvHist below) flushed once per work item with one global 64-bit atomic per
//    non-zero lag;
//  * 8-bit counts: a wave stages the events of several pixels in LDS and a lane takes an event
//    (event_flat_item);
//  * 16-bit counts and the longest series: a wave takes one pixel at a time (the next pixel's
//    events load into registers meanwhile), stages its events in LDS, and each lane takes
//    events i = lane + 128 r and i + 64 together; a binary search finds the first partner j > i
//    whose lag t_j - t_i reaches the window (event_pairs_item);
//  * the self pairs (lag 0, d_i^2) are added in the first window; S_b(t) comes from a launch of
//    its own (event_sums_item), or from the first window's launch where events are few;
//  * the input is validated on the device (frames in [0, N), strictly increasing per
//    pixel, as compress_all_stack produces, event.py:267-284); a violation sets a
//    flag the host turns into an error instead of reading out of bounds.
// Frame-sorted COO input (pixel, frame, count) is first turned into this pixel-major
// layout on the device: the (frame, count) pairs, packed into one word, are ordered by
// pixel with this file's stable LSD radix sort (8-bit digits over the bits a pixel
// index needs), so each pixel's events keep the input's frame order; the offsets are
// the lower bounds of every pixel in the sorted keys, and the packed words are split
// into times and counts.
#include <algorithm>

#include "dxg2_internal.h"

namespace dxg2 {

constexpr int ECAP = 256;       // staging entries of one wave in LDS
constexpr int EMAX = ECAP - 4;  // events of a staged pixel: its 4 sentinels always fit
constexpr int EPF = ECAP / 64;  // event rounds of the next pixel prefetched in registers

// LDS lag histogram of one work item, shared by the NW waves of its workgroup: 8 KiB of
// counters per wave, so that with NW = 4 four workgroups (16 waves, enough to cover the
// dependent LDS reads of the searches) share a CU with their staging, and with NW = 8
// two workgroups of twice the lag window do.
//  * 8-bit counts: 2048 NW lags of 32-bit counters.  A pixel adds at most sum_k d_k^2 to
//    any one lag (Cauchy-Schwarz: at a fixed lag each event pairs with at most one
//    partner), so each wave adds to the histogram only while its pixels' sum of d^2
//    stays below budget(NW) = 2^32 / NW (uint8) or 2^31 / NW (int8), and sends the pairs
//    of a pixel beyond it straight to the global 64-bit numerators.  The NW waves then
//    bound every counter below 2^32 (uint8) or its magnitude below 2^31 (int8, two's
//    complement), so it is exact.
//  * uint16 counts: 1024 NW lags of 64-bit counters, exact for any data.
template <typename T> struct EvHist {
    using type = uint32_t;
    static constexpr int lags_per_wave = 2048;
    // lags of one window: the last 64 counters stay outside every window, so the staged
    // partner loop can send each rejected partner's product to its own lane's counter there
    static constexpr int window(int nw) { return lags_per_wave * nw - 64; }
    static constexpr long long budget(int nw) {
        return (std::is_signed<T>::value ? (1ll << 31) : (1ll << 32)) / nw;
    }
    static __device__ __forceinline__ unsigned long long widen(uint32_t v) {
        return std::is_signed<T>::value ? (unsigned long long)(long long)(int32_t)v
                                        : (unsigned long long)v;
    }
};
template <> struct EvHist<uint16_t> {
    using type = unsigned long long;
    static constexpr int lags_per_wave = 1024;
    static constexpr int window(int nw) { return lags_per_wave * nw; }
    static constexpr long long budget(int) { return 0; }  // no bound needed
    static __device__ __forceinline__ unsigned long long widen(unsigned long long v) { return v; }
};

template <typename T>
__device__ __forceinline__ long long as_count(T v) { return (long long)v; }

__device__ __forceinline__ long long wave_sum64(long long v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Per-pixel bookkeeping of one wave: pixel index and event range, valid or not.
struct EvPixel {
    int p;
    uint32_t beg, end;
    int n;  // events to correlate: 0 for an empty, unbinned or invalid range
};

// One event's count to its frame's sum (few events: see event_sums_item()).
__device__ __forceinline__ void add_sum(int64_t* sum, long long d) {
    if (d) atomicAdd(reinterpret_cast<unsigned long long*>(sum), (unsigned long long)d);
}

// One pixel's pairs by a wave, lags [w0, w1), its n > 0 events at `beg`: staged by the wave (S; pt,
// pd: frames and counts, sq: this lane's share of the sum of d^2) or read from memory.  used: see
// EvHist.  srow: the bin's frame sums where this launch forms them, else null.
template <typename T, int NW, bool S>
__device__ __forceinline__ void event_pixel(const int32_t* __restrict__ times,
                                            const T* __restrict__ data, uint32_t beg, int n,
                                            int lane, int w0, int w1, int nframes, const int* pt,
                                            const int* pd,
                                            typename EvHist<T>::type* __restrict__ hist,
                                            unsigned long long* __restrict__ nwin, long long& used,
                                            long long sq, int64_t* __restrict__ srow,
                                            int* __restrict__ err) {
    using H = typename EvHist<T>::type;
    constexpr bool BOUNDED = sizeof(H) == 4;
    auto time_of = [&](int k) -> int {
        if constexpr (S) return pt[k];
        else return times[beg + k];
    };
    // 8-bit counts multiply in 32 bits (|d_i d_j| <= 255^2), 16-bit in 64
    using C = typename std::conditional<sizeof(T) == 1, int, long long>::type;
    auto count_of = [&](int k) -> C {
        if constexpr (S) return (C)pd[k];
        else return (C)as_count<T>(data[beg + k]);
    };
    // Validation, in the first lag window: frames in [0, N) and strictly increasing.  An invalid pixel is
    // skipped there and flagged, and the call reports the error; the other
    // windows do not repeat the check, and their lag test below keeps every
    // write inside the window whatever the input.
    if (w0 == 0) {
        int bad = 0;
        for (int k = lane; k < n; k += 64) {
            const int t = time_of(k);
            if (t < 0 || t >= nframes) bad = 1;
            else if (srow) add_sum(srow + t, (long long)count_of(k));
            if (k + 1 < n && time_of(k + 1) <= t) bad = 1;
        }
        if (bad) atomicOr(err, 1);
        if (__any(bad)) return;
    }
    long long sq_lane = sq;
    if constexpr (!S)
        for (int k = lane; k < n; k += 64) {
            const long long d = count_of(k);
            sq_lane += d * d;
        }
    const long long sqw = wave_sum64(sq_lane);  // sum of d^2: the lag-0 term
    bool to_lds = true;
    if constexpr (BOUNDED) {
        to_lds = used + sqw < EvHist<T>::budget(NW);
        if (to_lds) used += sqw;
    }
    if (w0 == 0 && lane == 0 && sqw != 0) {  // lag 0
        if (to_lds)
            atomicAdd(&hist[0], (H)sqw);
        else
            atomicAdd(nwin, (unsigned long long)sqw);
    }
    const unsigned span = (unsigned)(w1 - w0);
    // the rest in one of two instantiations: LDS counters, or (past the budget)
    // the global 64-bit numerators, so the pair loop carries no branch on it
    auto events = [&](auto lds_tag) {
    constexpr bool LDS = decltype(lds_tag)::value;
    auto add = [&](int lag, C prod) {  // lag in [0, w1 - w0)
        if constexpr (LDS)
            atomicAdd(&hist[lag], (H)prod);
        else
            atomicAdd(nwin + lag, (unsigned long long)(long long)prod);
    };
    // pairs (i, j), j > i, with lag t_j - t_i in [max(w0, 1), w1): partners from
    // the first j with t_j >= t_i + max(w0, 1) while t_j < t_i + w1, four per
    // step so that their reads and atomics overlap.  The lag test is one unsigned
    // compare, which also rejects a negative lag.
    auto partners = [&](int ti, C di, int j) {
        const int base = ti + w0;
        for (; j < n; j += 4) {
            int tj[4];
            C dj[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const bool in = j + u < n;
                const int jj = in ? j + u : n - 1;
                const int t = time_of(jj);
                const C d = count_of(jj);
                tj[u] = in ? t : base + (int)span;
                dj[u] = in ? d : (C)0;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const unsigned lag = (unsigned)(tj[u] - base);
                const C prod = di * dj[u];
                if (lag < span && prod != 0) add((int)lag, prod);
            }
            if (tj[3] - base >= (int)span) break;  // times increase: the rest are later
        }
    };
    // wave-uniform steps of the first-partner search: powers of two from the
    // largest not above n
    const int top = 1 << (31 - __builtin_clz(n));
    // Each lane takes events i and i + 64 together, so that their two searches
    // for the first partner overlap.
    for (int i0 = lane; i0 < n; i0 += 128) {
        const int i1 = i0 + 64;
        const bool has1 = i1 < n;
        const int ti0 = time_of(i0);
        const int ti1 = has1 ? time_of(i1) : 0;
        const C d0 = count_of(i0);
        const C d1 = has1 ? count_of(i1) : (C)0;
        // first partner: i + 1 in the first window (times strictly increase),
        // else one past the last p >= i with t_p < t_i + w0, by a descent over
        // power-of-two steps (a monotone test; reads clamped inside the list)
        int p0 = i0, p1 = has1 ? i1 : n - 1;
        if (w0 > 0) {
            const int g0 = ti0 + w0, g1 = ti1 + w0;
            for (int step = top; step > 0; step >>= 1) {
                const int q0 = p0 + step, q1 = p1 + step;
                const int t0 = time_of(min(q0, n - 1));
                const int t1 = time_of(min(q1, n - 1));
                if (q0 < n && t0 < g0) p0 = q0;
                if (q1 < n && t1 < g1) p1 = q1;
            }
        }
        partners(ti0, d0, p0 + 1);
        if (has1) partners(ti1, d1, p1 + 1);
    }
    };
    if (to_lds)
        events(std::true_type{});
    else
        events(std::false_type{});
}

// The pairs of one work item (a run of one bin's pixels) in lag window blockIdx.y, with
// the workgroup's LDS: the lag histogram and each wave's staged events (uint8, int8 and
// uint16 counts fit 32 bits), times and counts in one array st[2][NW][ECAP] so that the
// two reads of a step share one address.
template <typename T, int NW>
__device__ __forceinline__ void event_pairs_item(
    const int32_t* __restrict__ times, const T* __restrict__ data,
    const uint32_t* __restrict__ offsets, const int32_t* __restrict__ pix_idx,
    const BinDev* __restrict__ bins, const EventWork w, int nframes, int64_t nnz,
    int64_t* __restrict__ num, int64_t* __restrict__ sums, int* __restrict__ err,
    typename EvHist<T>::type* __restrict__ hist, int (*__restrict__ st)[NW][ECAP]) {
    int (*const st_t)[ECAP] = st[0];
    int (*const st_d)[ECAP] = st[1];
    using H = typename EvHist<T>::type;
    constexpr int EW = EvHist<T>::lags_per_wave * NW;  // counters
    constexpr int WS = EvHist<T>::window(NW);          // lags of a window
    constexpr int NT = 64 * NW;
    const BinDev bd = bins[w.bin];
    const int w0 = blockIdx.y * WS;
    if (w0 >= nframes) return;
    const int w1 = min(nframes, w0 + WS);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int k = threadIdx.x; k < EW; k += NT) hist[k] = 0;
    __syncthreads();
    unsigned long long* nwin = reinterpret_cast<unsigned long long*>(num + (int64_t)w.bin * nframes + w0);
    int64_t* srow = sums ? sums + (int64_t)w.bin * nframes : nullptr;
    long long used = 0;  // this wave's sum of d^2 added to the histogram (BOUNDED)

    // The wave takes pixels w.k0 + wave + NW r, r < nr.  Their list entries and offsets are
    // loaded 64 at a time (lane r % 64 holds pixel r), and while the pairs of pixel r are
    // counted, the first ECAP events of pixel r + 1 are already loading into registers,
    // so the chain list entry -> offsets -> events is not waited for once per pixel.
    const int npx = w.k1 - w.k0 - wave;
    const int nr = npx > 0 ? (npx + NW - 1) / NW : 0;
    int mp = -1;
    uint32_t mb = 0u, me = 0u;
    auto load_meta = [&](int r0) {
        const int r = r0 + lane;
        mp = -1;
        mb = me = 0u;
        if (r < nr) {
            mp = pix_idx[bd.idx_off + w.k0 + wave + NW * r];
            if (mp >= 0) {
                mb = offsets[mp];
                me = offsets[mp + 1];
            }
        }
    };
    auto meta = [&](int r) {
        EvPixel x;
        x.p = __builtin_amdgcn_readlane(mp, r & 63);
        x.beg = (uint32_t)__builtin_amdgcn_readlane((int)mb, r & 63);
        x.end = (uint32_t)__builtin_amdgcn_readlane((int)me, r & 63);
        const bool bad = x.p >= 0 && (x.end < x.beg || x.end > (uint64_t)nnz);
        x.n = (x.p < 0 || bad || x.end <= x.beg) ? 0 : (int)(x.end - x.beg);
        if (bad && lane == 0) atomicOr(err, 2);
        return x;
    };
    int ct[EPF];
    int cd[EPF];
    auto prefetch = [&](const EvPixel& x) {
#pragma unroll
        for (int q = 0; q < EPF; ++q) {
            const int k = lane + 64 * q;
            if (k < x.n && x.n <= EMAX) {
                ct[q] = times[x.beg + k];
                cd[q] = (int)data[x.beg + k];
            }
        }
    };

    EvPixel cur = {-1, 0u, 0u, 0};
    if (nr > 0) {
        load_meta(0);
        cur = meta(0);
        prefetch(cur);
    }
    for (int r = 0; r < nr; ++r) {
        // wave-uniform (the compiler keeps them, and the loops they bound, scalar)
        const int n = __builtin_amdgcn_readfirstlane(cur.n);
        const uint32_t beg = (uint32_t)__builtin_amdgcn_readfirstlane((int)cur.beg);
        const bool staged = n <= EMAX;
        long long sq = 0;  // this lane's share of the pixel's sum of d^2
        if (n > 0 && staged) {
#pragma unroll
            for (int q = 0; q < EPF; ++q) {
                const int k = lane + 64 * q;
                if (k < n) {
                    st_t[wave][k] = ct[q];
                    st_d[wave][k] = cd[q];
                    sq += (long long)cd[q] * cd[q];
                } else if (k < n + 4) {
                    st_t[wave][k] = 0x7fffffff;  // sentinel time: no partner lies there
                    st_d[wave][k] = 0;
                }
            }
        }
        // the next pixel's range, and its events into the registers just staged
        if (r + 1 < nr) {
            if (((r + 1) & 63) == 0) load_meta(r + 1);
            cur = meta(r + 1);
            prefetch(cur);
        }
        if (n == 0) continue;
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): staged values visible to the wave
        __builtin_amdgcn_wave_barrier();
        if (staged)
            event_pixel<T, NW, true>(times, data, beg, n, lane, w0, w1, nframes, st_t[wave],
                                     st_d[wave], hist, nwin, used, sq, srow, err);
        else
            event_pixel<T, NW, false>(times, data, beg, n, lane, w0, w1, nframes, nullptr, nullptr,
                                      hist, nwin, used, 0, srow, err);
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    for (int k = threadIdx.x; k < w1 - w0; k += NT) {
        const H v = hist[k];
        if (v != 0) atomicAdd(nwin + k, EvHist<T>::widen(v));
    }
}

template <typename T, int NW>
__global__ __launch_bounds__(64 * NW) void event_pairs_kernel(
    const int32_t* __restrict__ times, const T* __restrict__ data,
    const uint32_t* __restrict__ offsets, const int32_t* __restrict__ pix_idx,
    const BinDev* __restrict__ bins, const EventWork* __restrict__ work, int nframes,
    int64_t nnz, int64_t* __restrict__ num, int64_t* __restrict__ sums, int* __restrict__ err) {
    __shared__ typename EvHist<T>::type hist[EvHist<T>::lags_per_wave * NW];
    __shared__ __attribute__((aligned(16))) int st[2][NW][ECAP];
    event_pairs_item<T, NW>(times, data, offsets, pix_idx, bins, work[blockIdx.x], nframes, nnz,
                            num, sums, err, hist, st);
}

// A pointer read from a job table, marked as global memory (a generic pointer would
// turn every access into a flat one).
template <typename P>
__device__ __forceinline__ P* global_ptr(P* p) {
    using G = __attribute__((address_space(1))) P*;
    return (P*)reinterpret_cast<G>(reinterpret_cast<uintptr_t>(p));
}

// Several jobs in one launch: work item w belongs to job w.pad (padding items: bin < 0);
// lag windows past a job's frame count return at once.
template <typename T, int NW>
__global__ __launch_bounds__(64 * NW) void event_pairs_jobs_kernel(
    const EventJob* __restrict__ jobs, const EventWork* __restrict__ work, bool with_sums) {
    __shared__ typename EvHist<T>::type hist[EvHist<T>::lags_per_wave * NW];
    __shared__ __attribute__((aligned(16))) int st[2][NW][ECAP];
    const EventWork w = work[blockIdx.x];
    if (w.bin < 0) return;
    const EventJob j = jobs[w.pad];
    event_pairs_item<T, NW>(global_ptr(j.times), global_ptr(reinterpret_cast<const T*>(j.data)),
                            global_ptr(j.offsets), global_ptr(j.pix), global_ptr(j.bins), w,
                            j.nframes, j.nnz, global_ptr(j.num),
                            with_sums ? global_ptr(j.sums) : nullptr, global_ptr(j.err), hist, st);
}

// Frame sums S_b(t) of a work item's pixels (densecorrelator.cl:65-150 has them dense,
// evtcorrelator.cl:40 adds each event to global memory), in LDS counters of the frames [t0, t0 +
// window) and from there to `sums`.  One 64-bit global atomic an event holds a call at 17-23e9
// events/s whatever its pairs, and is left to calls of few events (sums_with_pairs()).  A wave
// loads the ranges of 64 pixels and streams each stretch of them that is one run of the event
// list (neighbours in a row are).  32-bit counters: an item has at most EVENT_ITEM_MAX pixels,
// each with one event a frame.  Ranges and frames that the pair kernel reports as invalid are
// left out.
constexpr int SUMS_WINDOW = 40000;  // frames: 160,000 bytes
template <typename T>
__device__ __forceinline__ void event_sums_item(const int32_t* __restrict__ times,
                                                const T* __restrict__ data,
                                                const uint32_t* __restrict__ offsets,
                                                const int32_t* __restrict__ pix_idx,
                                                const BinDev* __restrict__ bins, const EventWork w,
                                                int nframes, int64_t nnz, int window,
                                                int64_t* __restrict__ sums, uint32_t* hist) {
    const int t0 = blockIdx.y * window;
    if (t0 >= nframes) return;
    const unsigned len = (unsigned)min(window, nframes - t0);
    for (unsigned i = threadIdx.x; i < len; i += blockDim.x) hist[i] = 0u;
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int32_t* list = pix_idx + bins[w.bin].idx_off;
    const int step = (int)blockDim.x;
    for (int r = w.k0 + (int)(threadIdx.x - lane); r < w.k1; r += step) {
        const int p = r + lane < w.k1 ? list[r + lane] : -1;
        uint32_t b = 0u, e = 0u;
        if (p >= 0) {
            b = offsets[p];
            e = offsets[p + 1];
            if (e < b || (int64_t)e > nnz) e = b = 0u;
        }
        const uint32_t before = (uint32_t)__shfl_up((int)e, 1);
        uint64_t runs = __ballot(lane == 0 || b != before);
        while (runs) {
            const int first = __builtin_ctzll(runs);
            runs &= runs - 1;
            const int last = (runs ? __builtin_ctzll(runs) : 64) - 1;
            const uint32_t x1 = (uint32_t)__builtin_amdgcn_readlane((int)e, last);
            for (uint32_t x = (uint32_t)__builtin_amdgcn_readlane((int)b, first) + lane;
                 x - lane < x1; x += 512) {
                int t[8], d[8];
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const bool in = x + 64 * q < x1 && x + 64 * q >= x;
                    t[q] = in ? times[x + 64 * q] : -1;
                    d[q] = in ? (int)data[x + 64 * q] : 0;
                }
#pragma unroll
                for (int q = 0; q < 8; ++q)
                    if ((unsigned)(t[q] - t0) < len && t[q] >= 0)
                        atomicAdd(&hist[t[q] - t0], (uint32_t)d[q]);
                if (x1 - (x - lane) <= 512u) break;  // (no wrap at 2^32)
            }
        }
    }
    __syncthreads();
    int64_t* row = sums + (int64_t)w.bin * nframes + t0;
    for (unsigned i = threadIdx.x; i < len; i += blockDim.x) {
        const uint32_t v = hist[i];
        if (v)
            atomicAdd(reinterpret_cast<unsigned long long*>(row + i),
                      std::is_signed<T>::value ? (unsigned long long)(long long)(int32_t)v
                                               : (unsigned long long)v);
    }
}

template <typename T>
__global__ __launch_bounds__(1024) void event_sums_kernel(
    const int32_t* __restrict__ times, const T* __restrict__ data,
    const uint32_t* __restrict__ offsets, const int32_t* __restrict__ pix_idx,
    const BinDev* __restrict__ bins, const EventWork* __restrict__ work, int nframes, int64_t nnz,
    int window, int64_t* __restrict__ sums) {
    extern __shared__ uint32_t sums_hist[];
    event_sums_item<T>(times, data, offsets, pix_idx, bins, work[blockIdx.x], nframes, nnz, window,
                       sums, sums_hist);
}
template <typename T>
__global__ __launch_bounds__(1024) void event_sums_jobs_kernel(const EventJob* __restrict__ jobs,
                                                               const EventWork* __restrict__ work,
                                                               int window) {
    extern __shared__ uint32_t sums_hist[];
    const EventWork w = work[blockIdx.x];
    if (w.bin < 0) return;
    const EventJob j = jobs[w.pad];
    event_sums_item<T>(global_ptr(j.times), global_ptr(reinterpret_cast<const T*>(j.data)),
                       global_ptr(j.offsets), global_ptr(j.pix), global_ptr(j.bins), w, j.nframes,
                       j.nnz, window, global_ptr(j.sums), sums_hist);
}
// Frames per window: as even as SUMS_WINDOW allows.
static int sums_window(int nframes) {
    const int n = (nframes + SUMS_WINDOW - 1) / SUMS_WINDOW;
    return (nframes + n - 1) / n;
}
// Whether the pair kernel adds each event to its frame's sum by a global atomic (add_sum) and
// event_sums_item()'s launch is left out.  So few events that their atomics, at about 21e9/s
// beside the pairs, take less than that launch, and that LDS counters (`counters`: frames of every
// item) would join none of them.  Both costs beside the atomics, the pairs that hide them and the
// launch's repeated reads, grow with the lag windows.  Pairs and sums with the launch -> without:
// 8-bit, 128 x 128 x 400,000 (1.6e6 events, 13 windows) 264 -> 233 us, 514 x 1030 x 40,000 (2.1e6,
// 2 windows) 167 -> 166, 300 x 300 x 40,000 (3.6e6, 2) 165 -> 191, 512 x 512 x 100,000 (5.2e6, 4)
// 295 -> 324, x 200,000 (7) 455 -> 432, 1030 x 1065 x 250,000 (2.7e7, 8) 1,899 -> 2,376; 16-bit,
// whose pairs take longer, 512 x 512 x 100,000 (5.2e6) 1,327 -> 1,234, 514 x 1030 x 5,000 (1.3e7, 1)
// 692 -> 720, 1030 x 1065 x 50,000 (5.5e7, 4) 4,397 -> 5,317.
template <typename T>
static bool sums_with_pairs(int64_t counters, int64_t nnz, int windows) {
    const int64_t most = sizeof(T) == 1 ? std::max<int64_t>(2000000, 1200000ll * windows)
                                        : 7000000ll * std::max(1, windows / 4);
    return nnz <= std::min(counters, most);
}
// Threads: two workgroups share a CU's threads where their counters leave room for it.
static int sums_threads(int window) { return window > SUMS_WINDOW / 2 ? 1024 : 512; }

// ---------------------------------------------------------------- 8-bit counts
//
// The pair kernel of 8-bit counts, N <= FLAT_FRAMES (others: event_pairs_item()).  A wave takes up to 64 neighbouring pixels
// of a bin at a time and their events in batches of up to FLAT_EVENTS, end to end in LDS as
// (frame << 10 | count), and a lane takes an event, whatever its pixel: few events a pixel (0.3
// to 120 in use) leave no lane idle, and no pixel costs a wave's steps for itself.
//  * ONE (one lag window, N <= 32,704): event i of a pixel's n pairs with the (n - 1) / 2 events
//    after it in the circle of the pixel's events, and for even n the first half with the one
//    opposite too: each pair once, the same number of steps for every lane of a pixel.  The
//    first n / 2 events are staged again behind the last, so a lane's partners lie in a row.
//  * otherwise event i's partners run from the first with a lag in the window, found by a
//    search, to the first past it, and what lies outside goes to one of 64 counters behind it.
// Partners go four a step; the last step adds zeros for those past the lane's count, so every
// atomic falls on a counter whatever the input.  A step is 16 VALU instructions, four LDS atomics
// and two LDS reads.  Events out of range are staged as frame 0, and out of order can only
// misplace counts: both are flagged.  Pixels of more events than a batch go through
// event_pixel().  Bound by VALU issue and LDS atomics.
// Pairs, against a wave a pixel: 1030 x 1065 x 2,000 (4.4e7 events, 8.8e8 pairs) 1.31 -> 0.45 ms;
// 514 x 1030 x 20,000 (1.1e7) 0.36 -> 0.15; x 100,000 (1.1e8, 5.6e9 pairs, four windows) 5.36 ->
// 4.43; 60 x 80 x 1,000 0.110 -> 0.005.
constexpr int FLAT_EVENTS = 256;
constexpr int FLAT_STAGE = 512;  // words a wave: 3 / 2 FLAT_EVENTS, 4 past them, 64 of marks
constexpr int FLAT_WAVES = 16;
constexpr int FLAT_WINDOW = 32704;       // lags; 64 more counters take what lies outside
constexpr int FLAT_FRAMES = 1 << 21;     // frame + lag below 2^22

// Inclusive scans over a wave (0 is the identity).
template <typename Op>
__device__ __forceinline__ int wave_scan(int v, Op op) {
    v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false));  // row_shr:1
    v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false));
    v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false));
    v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false));
    v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false));  // row_bcast:15
    v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false));  // row_bcast:31
    return v;
}

// LDS written by this wave's lanes is read by its others after this.
__device__ __forceinline__ void wave_lds() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
}

template <typename T, bool ONE>
__device__ __forceinline__ void event_flat_item(
    const int32_t* __restrict__ times, const T* __restrict__ data,
    const uint32_t* __restrict__ offsets, const int32_t* __restrict__ pix_idx,
    const BinDev* __restrict__ bins, const EventWork w, int nframes, int64_t nnz,
    int64_t* __restrict__ num, int64_t* __restrict__ sums, int* __restrict__ err,
    uint32_t* __restrict__ hist, uint32_t* __restrict__ stages) {
    constexpr int R = FLAT_EVENTS / 64;
    const int w0 = ONE ? 0 : (int)blockIdx.y * FLAT_WINDOW;
    if (w0 >= nframes) return;
    const int span = min(FLAT_WINDOW, nframes - w0);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int k = threadIdx.x; k < span + 64; k += 64 * FLAT_WAVES) hist[k] = 0u;
    __syncthreads();
    const int32_t* list = pix_idx + bins[w.bin].idx_off;
    unsigned long long* nwin =
        reinterpret_cast<unsigned long long*>(num + (int64_t)w.bin * nframes + w0);
    int64_t* srow = sums && w0 == 0 ? sums + (int64_t)w.bin * nframes : nullptr;
    uint32_t* st = stages + wave * FLAT_STAGE;
    uint8_t* marks = reinterpret_cast<uint8_t*>(st + FLAT_STAGE - FLAT_EVENTS / 4);
    long long used = 0;  // this wave's sum of d^2 in the histogram (EvHist)
    const auto sum = [](int a, int b) { return a + b; };
    const auto most = [](int a, int b) { return a > b ? a : b; };
    const auto from = [](int v, int l) { return __builtin_amdgcn_ds_bpermute(4 * l, v); };
    const auto count = [](uint32_t word) -> int {
        return std::is_signed<T>::value ? (int)(int8_t)word : (int)(word & 0xFFu);
    };

    // a short item is spread over its waves
    const int chunk = min(64, (w.k1 - w.k0 + FLAT_WAVES - 1) / FLAT_WAVES);
    for (int r0 = w.k0 + wave * chunk; r0 < w.k1; r0 += FLAT_WAVES * chunk) {
        const int p = lane < chunk && r0 + lane < w.k1 ? list[r0 + lane] : -1;
        uint32_t beg = 0u;
        int n = 0;
        if (p >= 0) {
            beg = offsets[p];
            const uint32_t end = offsets[p + 1];
            if (end < beg || (int64_t)end > nnz)
                atomicOr(err, 2);
            else
                n = (int)min(end - beg, 0x7fffffffu);
        }
        for (uint64_t longs = __ballot(n > FLAT_EVENTS); longs; longs &= longs - 1) {
            const int l = __builtin_ctzll(longs);
            event_pixel<T, FLAT_WAVES, false>(times, data,
                                              (uint32_t)__builtin_amdgcn_readlane((int)beg, l),
                                              __builtin_amdgcn_readlane(n, l), lane, w0, w0 + span,
                                              nframes, nullptr, nullptr, hist, nwin, used, 0, srow,
                                              err);
        }
        if (n > FLAT_EVENTS) n = 0;
        // events and staged words of the lanes up to and with this one
        const int own = n | (ONE ? n + n / 2 : n) << 16;
        const int upto = wave_scan(own, sum);
        const int total = __builtin_amdgcn_readlane(upto, 63) & 0xFFFF;
        int done = 0, first = 0;  // events and lanes of earlier batches (done: as upto)
        while ((done & 0xFFFF) < total) {
            const int end = __popcll(__ballot((upto & 0xFFFF) - (done & 0xFFFF) <= FLAT_EVENTS));
            const int all = __builtin_amdgcn_readlane(upto, end - 1) - done;
            const int E = all & 0xFFFF;
            const int at = upto - own - done;  // this pixel's first event and staged word
            // each event's pixel: its first event is marked, the largest mark so far is its own
            reinterpret_cast<uint32_t*>(marks)[lane] = 0u;
            wave_lds();
            if (lane >= first && lane < end && n > 0) marks[at & 0xFFFF] = (uint8_t)(lane + 1);
            wave_lds();
            int carry = 0, i_[R], n_[R], s_[R];
            uint32_t x_[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int x = lane + 64 * r;
                const int m = most(wave_scan((int)marks[x], most), carry);
                carry = __builtin_amdgcn_readlane(m, 63);
                const int l = m > 0 ? m - 1 : 0;
                const int a = from(at, l), size = from(n, l);  // (by all lanes, for all lanes)
                n_[r] = x < E ? size : 0;
                i_[r] = x - (a & 0xFFFF);
                s_[r] = a >> 16;
                x_[r] = (uint32_t)from((int)beg, l) + (uint32_t)i_[r];
            }
            int t_[R], d_[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                t_[r] = n_[r] ? times[x_[r]] : 0;
                d_[r] = n_[r] ? (int)data[x_[r]] : 0;
            }
            int bad = 0;
            uint32_t sq = 0u;  // below 2^24 over the batch
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if ((unsigned)t_[r] >= (unsigned)nframes) {
                    bad = 1;
                    t_[r] = 0;
                } else if (srow) {
                    add_sum(srow + t_[r], d_[r]);
                }
                const uint32_t word = (uint32_t)t_[r] << 10 | ((uint32_t)d_[r] & 0xFFu);
                if (n_[r]) {
                    st[s_[r] + i_[r]] = word;
                    if (ONE && i_[r] < n_[r] / 2) st[s_[r] + n_[r] + i_[r]] = word;
                }
                sq += (uint32_t)(d_[r] * d_[r]);
            }
            if (lane < 4) st[(all >> 16) + lane] = 0u;  // read by last steps, counted as zeros
            wave_lds();
            if (w0 == 0) {
#pragma unroll
                for (int r = 0; r < R; ++r)
                    if (i_[r] + 1 < n_[r] && (int)(st[s_[r] + i_[r] + 1] >> 10) <= t_[r]) bad = 1;
                if (bad) atomicOr(err, 1);
            }
            const int sqw = __builtin_amdgcn_readlane(wave_scan((int)sq, sum), 63);
            const bool to_lds = used + sqw < EvHist<T>::budget(FLAT_WAVES);
            if (to_lds) used += sqw;
            if (w0 == 0 && lane == 0 && sqw) {  // lag 0
                if (to_lds)
                    atomicAdd(&hist[0], (uint32_t)sqw);
                else
                    atomicAdd(nwin, (unsigned long long)sqw);
            }
            // partners of each event: `m` staged words from `a` on (with several windows, those
            // of them up to the window's end), lags from t0
            auto pairs = [&](auto lds_tag) {
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    int a = s_[r] + i_[r] + 1, m;
                    if (ONE) {
                        m = n_[r] ? (n_[r] - 1) / 2 + (n_[r] % 2 == 0 && i_[r] < n_[r] / 2) : 0;
                    } else {
                        const int end = s_[r] + n_[r];
                        if (w0 > 0) {  // past the events below the window's first lag
                            const uint32_t k0 = (uint32_t)(t_[r] + w0) << 10;
                            int at = a - 1;
#pragma unroll
                            for (int step = FLAT_EVENTS / 2; step > 0; step >>= 1) {
                                const int q = at + step;
                                if (st[min(q, FLAT_EVENTS)] < k0 && q < end) at = q;
                            }
                            a = at + 1;
                        }
                        m = n_[r] ? end - a : 0;
                    }
                    const uint32_t t0 = (uint32_t)(t_[r] + w0) << 10;
                    // a word is frame << 10 | count: a difference >> 8 is the counter's byte
                    auto add = [&](uint32_t word, int d) {
                        uint32_t at;
                        if (ONE) {
                            uint32_t diff;
                            asm("v_sad_u32 %0, %1, %2, 0" : "=v"(diff) : "v"(word & ~0x3FFu), "v"(t0));
                            at = diff >> 8;
                        } else {
                            at = min((word - t0) >> 8, 4u * (uint32_t)(span + lane));
                        }
                        const int prod = std::is_signed<T>::value
                                             ? __mul24(d, count(word))
                                             : (int)__umul24((unsigned)d, (unsigned)count(word));
                        if constexpr (decltype(lds_tag)::value) {
                            atomicAdd(reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(hist) +
                                                                  at),
                                      (uint32_t)prod);
                        } else {
                            if (prod && (at >> 2) < (uint32_t)span)
                                atomicAdd(nwin + (at >> 2), (unsigned long long)(long long)prod);
                        }
                    };
                    const uint32_t* q = st + a;
                    bool more = true;
                    for (; m >= 4 && more; m -= 4, q += 4) {
                        const uint32_t y[4] = {q[0], q[1], q[2], q[3]};
#pragma unroll
                        for (int u = 0; u < 4; ++u) add(y[u], d_[r]);
                        if (!ONE) more = (int)(y[3] - t0) < span << 10;
                    }
                    if (m > 0 && more) {
                        const uint32_t y[3] = {q[0], q[1], q[2]};
#pragma unroll
                        for (int u = 0; u < 3; ++u) add(y[u], u < m ? d_[r] : 0);
                    }
                }
            };
            if (to_lds)
                pairs(std::true_type{});
            else
                pairs(std::false_type{});
            wave_lds();  // the next batch overwrites the stage
            done += all;
            first = end;
        }
    }
    __syncthreads();
    for (int k = threadIdx.x; k < span; k += 64 * FLAT_WAVES) {
        const uint32_t v = hist[k];
        if (v != 0) atomicAdd(nwin + k, EvHist<T>::widen(v));
    }
}

template <typename T, bool ONE>
__global__ __launch_bounds__(64 * FLAT_WAVES) void event_flat_kernel(
    const int32_t* __restrict__ times, const T* __restrict__ data,
    const uint32_t* __restrict__ offsets, const int32_t* __restrict__ pix_idx,
    const BinDev* __restrict__ bins, const EventWork* __restrict__ work, int nframes, int64_t nnz,
    int64_t* __restrict__ num, int64_t* __restrict__ sums, int* __restrict__ err) {
    extern __shared__ uint32_t flat_lds[];
    event_flat_item<T, ONE>(times, data, offsets, pix_idx, bins, work[blockIdx.x], nframes, nnz, num,
                            sums, err, flat_lds + FLAT_WAVES * FLAT_STAGE, flat_lds);
}
template <typename T, bool ONE>
__global__ __launch_bounds__(64 * FLAT_WAVES) void event_flat_jobs_kernel(
    const EventJob* __restrict__ jobs, const EventWork* __restrict__ work, bool with_sums) {
    extern __shared__ uint32_t flat_lds[];
    const EventWork w = work[blockIdx.x];
    if (w.bin < 0) return;
    const EventJob j = jobs[w.pad];
    event_flat_item<T, ONE>(global_ptr(j.times), global_ptr(reinterpret_cast<const T*>(j.data)),
                            global_ptr(j.offsets), global_ptr(j.pix), global_ptr(j.bins), w,
                            j.nframes, j.nnz, global_ptr(j.num),
                            with_sums ? global_ptr(j.sums) : nullptr, global_ptr(j.err),
                            flat_lds + FLAT_WAVES * FLAT_STAGE, flat_lds);
}
static size_t flat_lds_bytes(int nframes) {
    return 4 * ((size_t)FLAT_WAVES * FLAT_STAGE + std::min(nframes, FLAT_WINDOW) + 64);
}

// Waves per workgroup of event_pairs_kernel: 16 (one workgroup per CU, the most counters, so the
// fewest windows and the least per-window work per pixel), or DXG2_EVENT_WAVES = 8 (two per CU)
// or 4 (four per CU).
int event_waves() {
    static const int nw = [] {
        const char* v = getenv("DXG2_EVENT_WAVES");
        const int x = v ? atoi(v) : 16;
        return (x == 4 || x == 8) ? x : 16;
    }();
    return nw;
}

int event_lag_window(int dtype, int nframes) {
    if (dtype == DXG2_U16) return EvHist<uint16_t>::window(event_waves());
    return nframes <= FLAT_FRAMES ? FLAT_WINDOW : EvHist<uint8_t>::window(event_waves());
}

template <typename T, int NW>
void pairs_jobs_launch(const EventJob* jobs, const EventWork* work, int n_work, int max_frames,
                       int64_t counters, int64_t nnz, hipStream_t s) {
    constexpr int WS = EvHist<T>::window(NW);
    const bool with_sums = sums_with_pairs<T>(counters, nnz, (max_frames + WS - 1) / WS);
    const int win = sums_window(max_frames);
    if (!with_sums)
        event_sums_jobs_kernel<T><<<dim3((unsigned)n_work, (unsigned)((max_frames + win - 1) / win)),
                                    sums_threads(win), 4 * win, s>>>(jobs, work, win);
    if constexpr (sizeof(T) == 1) {
        if (max_frames <= FLAT_FRAMES) {
            const dim3 grid((unsigned)n_work, (unsigned)((max_frames + FLAT_WINDOW - 1) / FLAT_WINDOW));
            const size_t lds = flat_lds_bytes(max_frames);
            if (grid.y == 1)
                event_flat_jobs_kernel<T, true><<<grid, 64 * FLAT_WAVES, lds, s>>>(jobs, work,
                                                                                   with_sums);
            else
                event_flat_jobs_kernel<T, false><<<grid, 64 * FLAT_WAVES, lds, s>>>(jobs, work,
                                                                                    with_sums);
            return;
        }
    }
    event_pairs_jobs_kernel<T, NW><<<dim3((unsigned)n_work, (unsigned)((max_frames + WS - 1) / WS)),
                                     64 * NW, 0, s>>>(jobs, work, with_sums);
}

template <typename T>
void pairs_jobs_typed(const EventJob* jobs, const EventWork* work, int n_work, int max_frames,
                      int64_t counters, int64_t nnz, hipStream_t s) {
    if (event_waves() == 4)
        pairs_jobs_launch<T, 4>(jobs, work, n_work, max_frames, counters, nnz, s);
    else if (event_waves() == 16)
        pairs_jobs_launch<T, 16>(jobs, work, n_work, max_frames, counters, nnz, s);
    else
        pairs_jobs_launch<T, 8>(jobs, work, n_work, max_frames, counters, nnz, s);
}

void launch_event_pairs_jobs(int dtype, const EventJob* jobs, const EventWork* work, int n_work,
                             int max_frames, int64_t counters, int64_t nnz, hipStream_t s) {
    if (n_work <= 0 || max_frames <= 0) return;
    if (dtype == DXG2_U16)
        pairs_jobs_typed<uint16_t>(jobs, work, n_work, max_frames, counters, nnz, s);
    else if (dtype == DXG2_I8)
        pairs_jobs_typed<int8_t>(jobs, work, n_work, max_frames, counters, nnz, s);
    else
        pairs_jobs_typed<uint8_t>(jobs, work, n_work, max_frames, counters, nnz, s);
}

template <typename T, int NW>
void pairs_launch(const int32_t* times, const void* data, const uint32_t* offsets,
                  const int32_t* pix_idx, const BinDev* bins, const EventWork* work, int n_work,
                  int nframes, int64_t nnz, int64_t* num, int64_t* sums, int* err, hipStream_t s) {
    constexpr int WS = EvHist<T>::window(NW);
    int64_t* psums = nullptr;  // frame sums of the pair kernel
    if (sums_with_pairs<T>((int64_t)n_work * nframes, nnz, (nframes + WS - 1) / WS)) {
        psums = sums;
    } else {
        const int win = sums_window(nframes);
        event_sums_kernel<T><<<dim3((unsigned)n_work, (unsigned)((nframes + win - 1) / win)),
                               sums_threads(win), 4 * win, s>>>(
            times, (const T*)data, offsets, pix_idx, bins, work, nframes, nnz, win, sums);
    }
    if constexpr (sizeof(T) == 1) {
        if (nframes <= FLAT_FRAMES) {
            const dim3 grid((unsigned)n_work, (unsigned)((nframes + FLAT_WINDOW - 1) / FLAT_WINDOW));
            const size_t lds = flat_lds_bytes(nframes);
            if (grid.y == 1)
                event_flat_kernel<T, true><<<grid, 64 * FLAT_WAVES, lds, s>>>(
                    times, (const T*)data, offsets, pix_idx, bins, work, nframes, nnz, num, psums,
                    err);
            else
                event_flat_kernel<T, false><<<grid, 64 * FLAT_WAVES, lds, s>>>(
                    times, (const T*)data, offsets, pix_idx, bins, work, nframes, nnz, num, psums,
                    err);
            return;
        }
    }
    event_pairs_kernel<T, NW><<<dim3((unsigned)n_work, (unsigned)((nframes + WS - 1) / WS)),
                                64 * NW, 0, s>>>(times, (const T*)data, offsets, pix_idx, bins,
                                                 work, nframes, nnz, num, psums, err);
}

template <typename T>
void pairs_typed(const int32_t* times, const void* data, const uint32_t* offsets,
                 const int32_t* pix_idx, const BinDev* bins, const EventWork* work, int n_work,
                 int nframes, int64_t nnz, int64_t* num, int64_t* sums, int* err, hipStream_t s) {
    if (event_waves() == 4)
        pairs_launch<T, 4>(times, data, offsets, pix_idx, bins, work, n_work, nframes, nnz, num,
                           sums, err, s);
    else if (event_waves() == 16)
        pairs_launch<T, 16>(times, data, offsets, pix_idx, bins, work, n_work, nframes, nnz, num,
                            sums, err, s);
    else
        pairs_launch<T, 8>(times, data, offsets, pix_idx, bins, work, n_work, nframes, nnz, num,
                           sums, err, s);
}

void launch_event_pairs(int dtype, const int32_t* times, const void* data,
                        const uint32_t* offsets, const int32_t* pix_idx, const BinDev* bins,
                        const EventWork* work, int n_work, int nframes, int64_t nnz,
                        int64_t* num, int64_t* sums, int* err, hipStream_t s) {
    if (n_work <= 0 || nframes <= 0) return;
    if (dtype == DXG2_U16)
        pairs_typed<uint16_t>(times, data, offsets, pix_idx, bins, work, n_work, nframes, nnz,
                              num, sums, err, s);
    else if (dtype == DXG2_I8)
        pairs_typed<int8_t>(times, data, offsets, pix_idx, bins, work, n_work, nframes, nnz, num,
                            sums, err, s);
    else
        pairs_typed<uint8_t>(times, data, offsets, pix_idx, bins, work, n_work, nframes, nnz,
                             num, sums, err, s);
}

// LDS atomic-add throughput, the ceiling the pair kernel's histogram updates are measured
// against: workgroups of 256 threads with that kernel's LDS footprint (8192 32-bit
// counters and 8 KiB of staging, four workgroups per CU), each lane adding 1 `iters`
// times at pseudo-random counters (mode 0; a linear congruential sequence per lane) or
// at lane-consecutive ones (mode 1).
template <int MODE>
__global__ __launch_bounds__(256) void lds_atomic_rate_kernel(uint32_t* __restrict__ out,
                                                              int iters) {
    __shared__ uint32_t h[(EvHist<uint8_t>::lags_per_wave * 4)];
    __shared__ int stage_share[2 * 4 * ECAP];  // the staging arrays of four waves
    for (int i = threadIdx.x; i < (EvHist<uint8_t>::lags_per_wave * 4); i += 256) h[i] = 0;
    if (threadIdx.x < 8) stage_share[threadIdx.x] = 0;
    __syncthreads();
    uint32_t x = blockIdx.x * 2654435761u + threadIdx.x * 40503u + 1u;
    for (int i = 0; i < iters; ++i) {
        uint32_t a;
        if (MODE == 0) {
            x = x * 1664525u + 1013904223u;
            a = x >> 19;  // 0 .. 8191
        } else {
            a = (threadIdx.x + 64u * (uint32_t)i) & ((EvHist<uint8_t>::lags_per_wave * 4) - 1);
        }
        atomicAdd(&h[a], 1u);
    }
    __syncthreads();
    if (threadIdx.x == 0)
        out[blockIdx.x] = h[blockIdx.x & ((EvHist<uint8_t>::lags_per_wave * 4) - 1)] + (uint32_t)stage_share[0];
}

void launch_lds_atomic_rate(int mode, int blocks, int iters, uint32_t* out, hipStream_t s) {
    if (mode == 0)
        lds_atomic_rate_kernel<0><<<blocks, 256, 0, s>>>(out, iters);
    else
        lds_atomic_rate_kernel<1><<<blocks, 256, 0, s>>>(out, iters);
}

// ----------------------------------------------------------------- COO -> CSR
__global__ void fill_u32_kernel(uint32_t* __restrict__ p, int64_t n, uint32_t v) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

__global__ void coo_count_kernel(const uint32_t* __restrict__ pix, int64_t nnz, uint32_t npix,
                                 uint32_t* __restrict__ count, int* __restrict__ err) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < nnz;
         e += (int64_t)gridDim.x * blockDim.x) {
        const uint32_t p = pix[e];
        if (p >= npix) {
            atomicOr(err, 4);
            continue;
        }
        atomicAdd(&count[p], 1u);
    }
}

// Exclusive scan of n counts into out[0..n] (out[n] = total), three passes over
// blocks of 1024: per-block totals, a scan of the totals, then the block scans.
constexpr int SCAN_B = 1024;

__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t* sh, uint32_t* total) {
    // 256 threads x 4 values handled by the caller; here one value per thread
    const int tid = threadIdx.x;
    sh[tid] = v;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        const uint32_t x = tid >= off ? sh[tid - off] : 0u;
        __syncthreads();
        sh[tid] += x;
        __syncthreads();
    }
    const uint32_t incl = sh[tid];
    *total = sh[255];
    __syncthreads();
    return incl - v;
}

__global__ __launch_bounds__(256) void scan_block_totals(const uint32_t* __restrict__ in,
                                                         int64_t n, uint32_t* __restrict__ tot) {
    __shared__ uint32_t sh[256];
    const int64_t base = (int64_t)blockIdx.x * SCAN_B + threadIdx.x * 4;
    uint32_t s = 0;
    for (int k = 0; k < 4; ++k)
        if (base + k < n) s += in[base + k];
    uint32_t total;
    block_excl_scan(s, sh, &total);
    if (threadIdx.x == 0) tot[blockIdx.x] = total;
}

__global__ __launch_bounds__(256) void scan_totals(uint32_t* __restrict__ tot, int nb) {
    __shared__ uint32_t sh[256];
    uint32_t carry = 0;
    for (int b0 = 0; b0 < nb; b0 += 256) {
        const int b = b0 + threadIdx.x;
        const uint32_t v = b < nb ? tot[b] : 0u;
        uint32_t total;
        const uint32_t ex = block_excl_scan(v, sh, &total);
        if (b < nb) tot[b] = carry + ex;
        carry += total;
    }
}

__global__ __launch_bounds__(256) void scan_apply(const uint32_t* __restrict__ in, int64_t n,
                                                  const uint32_t* __restrict__ tot,
                                                  uint32_t* __restrict__ out) {
    __shared__ uint32_t sh[256];
    const int64_t base = (int64_t)blockIdx.x * SCAN_B + threadIdx.x * 4;
    uint32_t v[4], s = 0;
    for (int k = 0; k < 4; ++k) {
        v[k] = base + k < n ? in[base + k] : 0u;
        s += v[k];
    }
    uint32_t total;
    uint32_t ex = block_excl_scan(s, sh, &total) + tot[blockIdx.x];
    for (int k = 0; k < 4; ++k) {
        if (base + k < n) out[base + k] = ex;
        ex += v[k];
    }
    if (base <= n - 1 && n - 1 < base + 4) out[n] = ex;  // grand total
}

__global__ void copy_u32_kernel(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst,
                                int64_t n) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

// (frame, count) of event e packed as frame << CB | count; a frame past the series sets
// flag bit 0 (the packing keeps CB bits of count and the rest for the frame).
template <typename V, typename T, int CB>
__global__ void coo_pack_kernel(const uint32_t* __restrict__ pix, const uint32_t* __restrict__ frame,
                                const T* __restrict__ cnt, int64_t nnz, uint32_t npix, int nframes,
                                V* __restrict__ out, int* __restrict__ err) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < nnz;
         e += (int64_t)gridDim.x * blockDim.x) {
        const uint32_t f = frame[e];
        if (f >= (uint32_t)nframes) atomicOr(err, 1);
        if (pix[e] >= npix) atomicOr(err, 4);
        out[e] = ((V)f << CB) | (V)cnt[e];
    }
}

template <typename V, typename T, int CB>
__global__ void coo_unpack_kernel(const V* __restrict__ in, int64_t nnz,
                                  int32_t* __restrict__ times, T* __restrict__ data) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < nnz;
         e += (int64_t)gridDim.x * blockDim.x) {
        const V v = in[e];
        times[e] = (int32_t)(uint32_t)(v >> CB);
        data[e] = (T)(v & (((V)1 << CB) - 1));
    }
}

// Key bits of pixel indices below npix.
static int pixel_key_bits(uint32_t npix) {
    int b = 1;
    while (b < 32 && ((uint64_t)1 << b) < npix) ++b;
    return b;
}

static unsigned grid_for(int64_t n, int64_t cap = 65536);

// First index in times[b, e) (ascending) whose frame is >= t.
__device__ __forceinline__ uint32_t lower_frame(const int32_t* __restrict__ times, uint32_t b,
                                                uint32_t e, int t) {
    while (b < e) {
        const uint32_t m = b + (e - b) / 2;
        if (times[m] < t)
            b = m + 1;
        else
            e = m;
    }
    return b;
}

// Frame window [t0, t1) of a pixel-major event list: per-pixel counts, then (after a scan
// of the counts into new offsets) the copy with frames re-based to t - t0.
__global__ void window_count_kernel(const uint32_t* __restrict__ offsets,
                                    const int32_t* __restrict__ times, int64_t npix, int t0,
                                    int t1, uint32_t* __restrict__ count) {
    for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < npix;
         p += (int64_t)gridDim.x * blockDim.x) {
        const uint32_t b = offsets[p], e = offsets[p + 1];
        count[p] = lower_frame(times, b, e, t1) - lower_frame(times, b, e, t0);
    }
}

template <typename T>
__global__ void window_copy_kernel(const uint32_t* __restrict__ offsets,
                                   const int32_t* __restrict__ times, const T* __restrict__ data,
                                   int64_t npix, int t0, const uint32_t* __restrict__ out_off,
                                   int32_t* __restrict__ out_times, T* __restrict__ out_data) {
    for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < npix;
         p += (int64_t)gridDim.x * blockDim.x) {
        const uint32_t lo = lower_frame(times, offsets[p], offsets[p + 1], t0);
        const uint32_t o = out_off[p], n = out_off[p + 1] - o;
        for (uint32_t i = 0; i < n; ++i) {
            out_times[o + i] = times[lo + i] - t0;
            out_data[o + i] = data[lo + i];
        }
    }
}

void launch_events_window(int dtype, const uint32_t* offsets, const int32_t* times,
                          const void* data, int64_t npix, int t0, int t1, uint32_t* scratch,
                          uint32_t* out_offsets, int32_t* out_times, void* out_data,
                          hipStream_t s) {
    if (npix <= 0) return;
    window_count_kernel<<<grid_for(npix), 256, 0, s>>>(offsets, times, npix, t0, t1, out_offsets);
    launch_excl_scan(out_offsets, npix, scratch, out_offsets, s);  // in place
    if (dtype == DXG2_U16)
        window_copy_kernel<uint16_t><<<grid_for(npix), 256, 0, s>>>(
            offsets, times, (const uint16_t*)data, npix, t0, out_offsets, out_times,
            (uint16_t*)out_data);
    else
        window_copy_kernel<uint8_t><<<grid_for(npix), 256, 0, s>>>(
            offsets, times, (const uint8_t*)data, npix, t0, out_offsets, out_times,
            (uint8_t*)out_data);
}

// Events of listed pixels -> dense columns: out[t * n_cols + k] = the count of pixel
// cols[k] at frame t (zero where it has no event).  One thread per listed pixel walks its
// events; a frame outside [0, nframes) sets bit 0 of *err and is skipped, a listed pixel
// outside [0, npix) sets bit 1.  The caller's buffer is cleared first by fill_bytes_kernel.
__global__ void fill_bytes_kernel(uint32_t* __restrict__ p, int64_t words) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < words;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = 0u;
}

__global__ void fill_tail_kernel(uint8_t* __restrict__ p, int64_t from, int64_t to) {
    const int64_t i = from + threadIdx.x;
    if (i < to) p[i] = 0;
}

template <typename T>
__global__ void events_to_columns_kernel(const uint32_t* __restrict__ offsets,
                                         const int32_t* __restrict__ times,
                                         const T* __restrict__ data, int64_t npix,
                                         const int32_t* __restrict__ cols, int64_t n_cols,
                                         int nframes, T* __restrict__ out, int* __restrict__ err) {
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < n_cols;
         k += (int64_t)gridDim.x * blockDim.x) {
        const int32_t p = cols[k];
        if (p < 0 || p >= npix) {
            if (err) atomicOr(err, 2);
            continue;
        }
        const uint32_t e1 = offsets[p + 1];
        for (uint32_t i = offsets[p]; i < e1; ++i) {
            const int32_t t = times[i];
            if (t < 0 || t >= nframes) {
                if (err) atomicOr(err, 1);
                continue;
            }
            out[(int64_t)t * n_cols + k] = data[i];
        }
    }
}

void launch_events_to_columns(int dtype, const uint32_t* offsets, const int32_t* times,
                              const void* data, int64_t npix, const int32_t* cols,
                              int64_t n_cols, int nframes, void* out, int* err, hipStream_t s) {
    const int64_t bytes = n_cols * nframes * (dtype == DXG2_U16 ? 2 : 1);
    const int64_t words = bytes / 4;
    if (words > 0) fill_bytes_kernel<<<grid_for(words), 256, 0, s>>>((uint32_t*)out, words);
    if (bytes > words * 4)
        fill_tail_kernel<<<1, 64, 0, s>>>((uint8_t*)out, words * 4, bytes);
    if (n_cols <= 0) return;
    if (dtype == DXG2_U16)
        events_to_columns_kernel<uint16_t><<<grid_for(n_cols), 256, 0, s>>>(
            offsets, times, (const uint16_t*)data, npix, cols, n_cols, nframes, (uint16_t*)out,
            err);
    else
        events_to_columns_kernel<uint8_t><<<grid_for(n_cols), 256, 0, s>>>(
            offsets, times, (const uint8_t*)data, npix, cols, n_cols, nframes, (uint8_t*)out,
            err);
}

void launch_excl_scan(const uint32_t* in, int64_t n, uint32_t* tot, uint32_t* out, hipStream_t s) {
    if (n <= 0) return;
    const int nb = (int)((n + SCAN_B - 1) / SCAN_B);
    scan_block_totals<<<nb, 256, 0, s>>>(in, n, tot);
    scan_totals<<<1, 256, 0, s>>>(tot, nb);
    scan_apply<<<nb, 256, 0, s>>>(in, n, tot, out);
}

void launch_copy_u32(const uint32_t* src, uint32_t* dst, int64_t n, hipStream_t s) {
    if (n > 0) copy_u32_kernel<<<grid_for(n), 256, 0, s>>>(src, dst, n);
}

void launch_fill_u32(uint32_t* p, int64_t n, hipStream_t s) {
    if (n > 0) fill_u32_kernel<<<grid_for(n), 256, 0, s>>>(p, n, 0u);
}

static unsigned grid_for(int64_t n, int64_t cap) {
    int64_t g = (n + 255) / 256;
    if (g < 1) g = 1;
    if (g > cap) g = cap;
    return (unsigned)g;
}

bool coo_narrow_values(int dtype, int nframes) {
    return dtype != DXG2_U16 && nframes <= (1 << 24);
}

// ------------------------------------------------------- stable LSD radix sort
// Sorts (key, value) pairs by the key bits [0, 8 * passes), 8 bits per pass, stably.
// Per pass over tiles of RS_TILE = 4096 pairs (4 waves x 16 rounds x 64 lanes, element
// index = wave * 1024 + round * 64 + lane):
//   radix_hist_kernel     digit histogram of each tile -> hist[digit * n_tiles + tile];
//   exclusive scan of hist (digit-major): the output position of each tile's first
//                         element of each digit;
//   radix_scatter_kernel  each wave ranks its 16 rounds in order: the lanes holding one
//                         digit find each other with 8 ballots (one per digit bit), the
//                         rank is the wave's running count of that digit plus the lanes
//                         below with it; the waves' counts give the cross-wave base; the
//                         tile is then reordered by digit in LDS and written out in runs.
constexpr int RS_TILE = 4096;
constexpr int RS_ROUNDS = 16;   // per wave

__global__ __launch_bounds__(256) void radix_hist_kernel(const uint32_t* __restrict__ keys,
                                                         int64_t n, int shift,
                                                         uint32_t* __restrict__ hist,
                                                         int n_tiles) {
    __shared__ uint32_t cnt[256];
    cnt[threadIdx.x] = 0u;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * RS_TILE;
    for (int i = threadIdx.x; i < RS_TILE; i += 256) {
        const int64_t e = base + i;
        if (e < n) atomicAdd(&cnt[(keys[e] >> shift) & 255u], 1u);
    }
    __syncthreads();
    hist[(int64_t)threadIdx.x * n_tiles + blockIdx.x] = cnt[threadIdx.x];
}

template <typename V>
__global__ __launch_bounds__(256) void radix_scatter_kernel(
    const uint32_t* __restrict__ keys_in, const V* __restrict__ vals_in, int64_t n, int shift,
    const uint32_t* __restrict__ pos, int n_tiles, uint32_t* __restrict__ keys_out,
    V* __restrict__ vals_out) {
    __shared__ uint32_t wave_cnt[4][256];     // per wave: count of each digit so far
    __shared__ uint32_t local_off[256];       // the tile's exclusive digit offsets
    __shared__ uint32_t tot;
    __shared__ uint32_t s_keys[RS_TILE];
    __shared__ V s_vals[RS_TILE];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    for (int w = 0; w < 4; ++w) wave_cnt[w][tid] = 0u;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * RS_TILE + wave * (RS_TILE / 4);
    const uint64_t below = (1ull << lane) - 1ull;
    uint32_t key[RS_ROUNDS];
    V val[RS_ROUNDS];
    uint32_t rank[RS_ROUNDS];
#pragma unroll
    for (int r = 0; r < RS_ROUNDS; ++r) {
        const int64_t e = base + r * 64 + lane;
        const bool valid = e < n;
        key[r] = valid ? keys_in[e] : 0u;
        val[r] = valid ? vals_in[e] : (V)0;
    }
#pragma unroll
    for (int r = 0; r < RS_ROUNDS; ++r) {
        const int64_t e = base + r * 64 + lane;
        const bool valid = e < n;
        const uint32_t d = (key[r] >> shift) & 255u;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const uint64_t m = __ballot((d >> b) & 1u);
            peers &= ((d >> b) & 1u) ? m : ~m;
        }
        const uint32_t before = wave_cnt[wave][d];      // same value for every peer
        rank[r] = before + (uint32_t)__popcll(peers & below);
        if (valid && (peers & below) == 0ull)           // the lowest peer updates
            wave_cnt[wave][d] = before + (uint32_t)__popcll(peers);
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    // per digit (thread = digit): the waves' counts, their prefix, the tile's total
    const uint32_t c0 = wave_cnt[0][tid], c1 = wave_cnt[1][tid], c2 = wave_cnt[2][tid],
                   c3 = wave_cnt[3][tid];
    const uint32_t total = c0 + c1 + c2 + c3;
    __syncthreads();
    wave_cnt[0][tid] = 0u;
    wave_cnt[1][tid] = c0;
    wave_cnt[2][tid] = c0 + c1;
    wave_cnt[3][tid] = c0 + c1 + c2;
    // exclusive scan of the 256 totals into local_off (Hillis-Steele in LDS)
    local_off[tid] = total;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        const uint32_t x = tid >= off ? local_off[tid - off] : 0u;
        __syncthreads();
        local_off[tid] += x;
        __syncthreads();
    }
    const uint32_t incl = local_off[tid];
    __syncthreads();
    local_off[tid] = incl - total;
    if (tid == 255) tot = incl;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RS_ROUNDS; ++r) {
        const int64_t e = base + r * 64 + lane;
        if (e < n) {
            const uint32_t d = (key[r] >> shift) & 255u;
            const uint32_t p = local_off[d] + wave_cnt[wave][d] + rank[r];
            s_keys[p] = key[r];
            s_vals[p] = val[r];
        }
    }
    __syncthreads();
    const uint32_t count = tot;
    for (uint32_t i = tid; i < count; i += 256) {
        const uint32_t k = s_keys[i];
        const uint32_t d = (k >> shift) & 255u;
        const int64_t o = (int64_t)pos[(int64_t)d * n_tiles + blockIdx.x] + (i - local_off[d]);
        keys_out[o] = k;
        vals_out[o] = s_vals[i];
    }
}

static int radix_passes(uint32_t npix) { return (pixel_key_bits(npix) + 7) / 8; }

static int64_t radix_tiles(int64_t n) { return (n + RS_TILE - 1) / RS_TILE; }

// Workspace of the sort beyond the caller's keys / value buffers: a second key buffer,
// the histogram and its scan totals.
size_t coo_sort_bytes(int dtype, int nframes, int64_t cap, uint32_t npix) {
    (void)dtype;
    (void)nframes;
    (void)npix;
    const int64_t nt = radix_tiles(std::max<int64_t>(cap, 1));
    const int64_t hist = 256 * nt;
    // second key buffer (64-aligned), histogram + the scan's grand total, scan totals
    return (size_t)((cap + 63) / 64 * 64) * 4 + (size_t)(hist + 1) * 4 +
           (size_t)((hist + 1023) / 1024 + 1) * 4 + 256;
}

// Sorts (pix, v0) by pixel; returns the buffers holding the sorted keys and values.
template <typename V>
static void radix_sort_by_pixel(const uint32_t* pix, V* v0, V* v1, int64_t n, uint32_t npix,
                                const CooSortBufs& b, const uint32_t** keys_sorted,
                                const V** vals_sorted, hipStream_t s) {
    const int64_t nt = radix_tiles(n);
    uint32_t* keys2 = reinterpret_cast<uint32_t*>(b.tmp);
    uint32_t* hist = keys2 + ((n + 63) / 64) * 64;
    uint32_t* tot = hist + 256 * nt + 1;   // the in-place scan writes hist[256 nt]
    const uint32_t* kin = pix;
    const V* vin = v0;
    uint32_t* kbuf[2] = {b.keys, keys2};
    V* vbuf[2] = {v1, v0};
    const int passes = radix_passes(npix);
    for (int p = 0; p < passes; ++p) {
        uint32_t* kout = kbuf[p & 1];
        V* vout = vbuf[p & 1];
        radix_hist_kernel<<<(unsigned)nt, 256, 0, s>>>(kin, n, 8 * p, hist, (int)nt);
        launch_excl_scan(hist, 256 * nt, tot, hist, s);
        radix_scatter_kernel<V><<<(unsigned)nt, 256, 0, s>>>(kin, vin, n, 8 * p, hist, (int)nt,
                                                             kout, vout);
        kin = kout;
        vin = vout;
    }
    *keys_sorted = kin;
    *vals_sorted = vin;
}

// offsets[p] = the first position of a key >= p in the sorted keys, p = 0 .. npix.
__global__ void offsets_from_keys_kernel(const uint32_t* __restrict__ keys, int64_t n,
                                         uint32_t npix, uint32_t* __restrict__ offsets) {
    for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p <= (int64_t)npix;
         p += (int64_t)gridDim.x * blockDim.x) {
        int64_t lo = 0, hi = n;
        while (lo < hi) {
            const int64_t m = lo + (hi - lo) / 2;
            if (keys[m] < (uint32_t)p)
                lo = m + 1;
            else
                hi = m;
        }
        offsets[p] = (uint32_t)lo;
    }
}

template <typename V, typename T, int CB>
static void coo_sort_split(const uint32_t* pix, const uint32_t* frame, const T* cnt, int64_t nnz,
                           uint32_t npix, int nframes, const CooSortBufs& b, uint32_t* offsets,
                           int32_t* times, T* data, int* err, hipStream_t s) {
    V* v0 = reinterpret_cast<V*>(b.vals0);
    V* v1 = reinterpret_cast<V*>(b.vals1);
    coo_pack_kernel<V, T, CB><<<grid_for(nnz), 256, 0, s>>>(pix, frame, cnt, nnz, npix, nframes,
                                                           v0, err);
    const uint32_t* keys = nullptr;
    const V* vals = nullptr;
    radix_sort_by_pixel<V>(pix, v0, v1, nnz, npix, b, &keys, &vals, s);
    offsets_from_keys_kernel<<<grid_for((int64_t)npix + 1), 256, 0, s>>>(keys, nnz, npix,
                                                                        offsets);
    coo_unpack_kernel<V, T, CB><<<grid_for(nnz), 256, 0, s>>>(vals, nnz, times, data);
}

hipError_t launch_coo_to_csr(int dtype, const uint32_t* pix, const uint32_t* frame,
                             const void* cnt, int64_t nnz, uint32_t npix, int nframes,
                             uint32_t* offsets, const CooSortBufs& sort, int32_t* times,
                             void* data, int* err, hipStream_t s) {
    if (nnz <= 0) {
        fill_u32_kernel<<<grid_for((int64_t)npix + 1), 256, 0, s>>>(offsets, (int64_t)npix + 1, 0u);
        return hipGetLastError();
    }
    if (dtype == DXG2_U16)
        coo_sort_split<uint64_t, uint16_t, 16>(pix, frame, (const uint16_t*)cnt, nnz, npix,
                                               nframes, sort, offsets, times, (uint16_t*)data,
                                               err, s);
    else if (coo_narrow_values(dtype, nframes))
        coo_sort_split<uint32_t, uint8_t, 8>(pix, frame, (const uint8_t*)cnt, nnz, npix, nframes,
                                             sort, offsets, times, (uint8_t*)data, err, s);
    else
        coo_sort_split<uint64_t, uint8_t, 16>(pix, frame, (const uint8_t*)cnt, nnz, npix,
                                              nframes, sort, offsets, times, (uint8_t*)data, err,
                                              s);
    return hipGetLastError();
}

}  // namespace dxg2
