// Grouped i8-MFMA Gram over every q-bin with the diagonal (tau) reduction fused.
//
// Reference numerator: per bin, a float32 sgemm of the gathered (N, n_b) matrix with
// itself followed by a host loop over the N diagonals (correlator/dense.py:54,61-64),
// or the OpenCL loop of densecorrelator.cl:6-57.  Here one launch covers every bin:
// a work item is one T x T output tile (rows ti, columns tj >= ti) of one bin's Gram
// G = A A^T over a range of k-blocks.  v_mfma_i32_32x32x32_i8 accumulates exact int32
// dot products (the work list caps a range at 2047 k-blocks so |sum| < 2^31), and the
// epilogue folds the tile into its 2T-1 diagonals tau = (tj-ti)*T + c - r in LDS
// before one 64-bit global atomic per diagonal.  Nothing of size N x N is stored
// (except by the calc_std variant, which also writes its tile to a scratch slot).
//
// Data movement: the slab is stored fragment-contiguous (slab_offset()): the 32 frames
// x 32 bytes an MFMA operand takes from one k-block are one 1 KiB run in lane order.
//
// T = 256 (PanelLoop): 2 x 2 waves of 4 x 4 blocks.  The runs of a tile's row and column
// panels go to LDS by global->LDS DMA and each wave reads its eight fragments of a unit
// (one K = 32 step) from there, so a run crosses the CU's vector-memory path once instead of
// once for each of the two waves that use it (64 B/clk a CU, which the 128 x 128 blocks of
// four waves would need in full at the MFMA rate).  Three buffers of GRAM_UNITS units form a
// ring; everything is spread over the unit's 16 MFMAs, four at a time: two or three fragment
// reads of the next unit and one DMA of the unit two stages ahead (DMAs issued in a burst
// hold back the wave's MFMAs behind them, a quarter of the time; 480,000 pixels x 10,000 frames
// 14.9 ms, 15.6 for fragments loaded straight into registers).  One barrier a
// stage, ahead of its last unit: by then that unit's fragments are in registers, so the
// buffer is free, and the next stage has landed (the wait leaves this stage's DMAs in
// flight), so its first fragments are read under the last unit's MFMAs and no latency is
// seen.  Two compiler behaviours shape the code:
//   * sched_barrier fences pin the order, which the machine scheduler would undo;
//   * the waitcnt pass waits for every DMA before an LDS read that may alias it: the buffers
//     are separate __shared__ arrays and each stage names its own, with the loop unrolled
//     over the ring and no branch inside (a merge of paths brings the wait back).
// Units past the item's end read zeros for A, so a stage is always whole.
//
// T = 128 (GramTile): each wave loads its operand fragments straight from global memory into
// VGPRs with one global_load_dwordx4 per fragment, two register slots deep: the loads of
// k-block kb + 2 are issued right after the MFMAs of kb have consumed the slot.  Every path
// issues the same loads (the k-block index is clamped to the item's last k-block near the
// end), as the waitcnt pass takes the minimum over paths.
//
// Diagonal tiles (ti == tj): the wave below the diagonal has nothing to compute and
// skips the loop; the other waves compute whole 32 x 32 blocks and the epilogue drops
// lags below the diagonal.  The two waves on the diagonal also sum the bytes of their
// A fragments (v_dot4), which gives the per-frame bin sums S_b(t) (densecorrelator.cl:
// 65-150) with no extra pass over the data.
//
// uint16 frames arrive as two biased digit planes H, L (k-blocks [0, nkb) and
// [nkb, 2 nkb) of the bin).  Work items then come in three kinds, each adding into its
// own output row: H H^T over [0, nkb), L L^T over [nkb, 2 nkb) (both in the plain
// kernel), and the cross product [H|L] [L|H]^T = H L^T + L H^T over [0, 2 nkb) in the
// CROSS kernel, whose B operand reads k-block kb +- nkb.  The cross Gram is symmetric,
// so the same upper-triangle tiles cover it; its diagonal tiles run as full tiles.
//
// LDS diagonal sums stay in 32-bit words: every int32 value v is split as
// v = hi * 2^16 + lo with lo in [0, 2^16) and hi in [-2^15, 2^15); a diagonal of a
// T <= 256 tile collects at most 256 values, so sum(lo) < 2^24 and |sum(hi)| < 2^23
// are exact, and the 64-bit total hi_sum * 2^16 + lo_sum is formed once per slot.  Values
// below 2^23 (short k-ranges, FP4) are added whole.
#include <algorithm>
#include <type_traits>

#include "dxg2_internal.h"

namespace dxg2 {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(1))) const v4i global_v4i;

// 16-byte load through a global-address-space pointer: a generic pointer (one read from
// a job descriptor) would give flat loads, which the waitcnt pass also counts as LDS
// traffic and drains before every MFMA group.
__device__ __forceinline__ v4i gload16(const int8_t* p) {
    return *reinterpret_cast<global_v4i*>(reinterpret_cast<uintptr_t>(p));
}

// 64-bit atomic add through a global-address-space pointer (see gload16).
__device__ __forceinline__ void gatomic_add(int64_t* p, int64_t v) {
    __hip_atomic_fetch_add(reinterpret_cast<__attribute__((address_space(1))) unsigned long long*>(
                               reinterpret_cast<uintptr_t>(p)),
                           (unsigned long long)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A bin descriptor read through a global-address-space pointer (two 16-byte loads).
static_assert(sizeof(BinDev) == 32, "BinDev is loaded as two 16-byte words");
__device__ __forceinline__ BinDev gload_bin(const BinDev* p) {
    union {
        v4i v[2];
        BinDev b;
    } u;
    u.v[0] = gload16(reinterpret_cast<const int8_t*>(p));
    u.v[1] = gload16(reinterpret_cast<const int8_t*>(p) + 16);
    return u.b;
}

template <int WM, int WN>
struct GramShape {
    static constexpr int TM = 2 * WM * 32;  // 2 x 2 waves of WM x WN MFMA blocks
    static constexpr int TN = 2 * WN * 32;
    static constexpr int NDIAG = TM + TN - 1;
};

// Frame sums of a diagonal tile's wave: rs[m] = this lane's share of row row + 32 m +
// lane % 32 (lanes l and l + 32 hold the two 32-byte halves of the frame row).
template <int WM>
__device__ __forceinline__ void frame_sums(const int (&rs)[WM], int row, int lane, int nframes,
                                           int64_t bias, int64_t* __restrict__ sums) {
#pragma unroll
    for (int m = 0; m < WM; ++m) {
        const int v = rs[m] + __shfl_xor(rs[m], 32);
        const int t = row + m * 32 + lane;
        const int64_t s64 = (int64_t)v + bias;
        if (lane < 32 && t < nframes && s64 != 0) gatomic_add(sums + t, s64);
    }
}

// (FP4 accumulators hold quarters.)
__device__ __forceinline__ int exact_value(int v) { return v; }
__device__ __forceinline__ int exact_value(float v) { return (int)(4.f * v); }

// A wave's accumulators added to the tile's diagonal sums in LDS, and with STORE written to
// `tile` (row-major).  32x32 accumulator layout: lane holds column (lane & 31) and rows
// 8*(v/4) + 4*(lane/32) + (v%4), v = 0..15.  Diagonal slot c - r + TM - 1: the blocks of one
// n - m fall on the same slots and are added in registers first, since the LDS takes about
// 11 atomics a clock (a tile's 512 a lane were 5 us).
// small: every |value| < 2^23, so a diagonal's up to 256 values need no splitting.
template <int WM, int WN, bool STORE, typename Acc>
__device__ __forceinline__ void fold_tile(const Acc (&acc)[WM][WN], int wr, int wc, int lane,
                                          bool small, unsigned int* sDiag,
                                          int* __restrict__ tile) {
    using S = GramShape<WM, WN>;
    // slot = lane part + (n - m) 32 - 8 (v / 4) - v % 4; the second part is a
    // compile-time constant >= MINOFF, so every atomic is one base VGPR plus an
    // immediate offset (no per-element address registers).
    constexpr int MINOFF = -(WM - 1) * 32 - 15;
    unsigned int* sd = sDiag + (wc * WN * 32 + (lane & 31)) - (wr * WM * 32 + 4 * (lane >> 5)) +
                       S::TM - 1 + MINOFF;
    auto fold = [&](auto split) {
#pragma unroll
        for (int d = -(WM - 1); d < WN; ++d) {  // d = n - m
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int k = d * 32 - 8 * (v >> 2) - (v & 3) - MINOFF;
                unsigned lo = 0u, hi = 0u;
#pragma unroll
                for (int m = 0; m < WM; ++m) {
                    if (m + d < 0 || m + d >= WN) continue;
                    const int val = exact_value(acc[m][m + d][v]);
                    lo += decltype(split)::value ? (unsigned)(val & 0xFFFF) : (unsigned)val;
                    hi += (unsigned)(val >> 16);
                }
                atomicAdd(sd + k, lo);
                if (decltype(split)::value) atomicAdd(sd + S::NDIAG + k, hi);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    if (small)
        fold(std::false_type{});
    else
        fold(std::true_type{});
    if (STORE) {
        // Lanes 0-31 and 32-63 of one store write two 128-byte row segments.
#pragma unroll
        for (int m = 0; m < WM; ++m)
#pragma unroll
            for (int n = 0; n < WN; ++n) {
                const int c = wc * WN * 32 + n * 32 + (lane & 31);
                const int rbase = wr * WM * 32 + m * 32 + 4 * (lane >> 5);
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    tile[(rbase + 8 * (v >> 2) + (v & 3)) * S::TN + c] = exact_value(acc[m][n][v]);
            }
    }
}

// The tile's diagonal sums to the numerators: lag = shift + slot - (TM - 1).
template <typename S>
__device__ __forceinline__ void flush_diagonals(const unsigned int* sDiag, bool small, int tid,
                                                int shift, int nframes,
                                                int64_t* __restrict__ out) {
    for (int i = tid; i < S::NDIAG; i += 256) {
        const long long v = small ? (long long)(int)sDiag[i]
                                  : (long long)(int)sDiag[S::NDIAG + i] * 65536 +
                                        (long long)sDiag[i];
        const int tau = shift + i - (S::TM - 1);
        if (v != 0 && tau >= 0 && tau < nframes) gatomic_add(out + tau, v);
    }
}

template <int WM, int WN, bool DIAG, bool CROSS, bool STORE = false>
struct GramTile {
    using S = GramShape<WM, WN>;
    const int8_t* __restrict__ slab_bin;
    int kb0, kb1, row0, col0, nframes, nrows;
    int tid, lane, wr, wc;
    int nkbp;  // CROSS: k-blocks per digit plane (B reads kb + nkbp or kb - nkbp)
    unsigned int* sDiag;

    v16i acc[WM][WN];
    v4i fa[2][2][WM];  // [slot][ks][block]
    v4i fb[2][2][WN];
    int rs[WM];        // DIAG: partial frame sums of this lane's A rows

    __device__ __forceinline__ void load(int s, int kb, const int8_t* pa, const int8_t* pb,
                                         int64_t kstride) {
        const int8_t* a = pa + kb * kstride;
        const int kbb = CROSS ? (kb < nkbp ? kb + nkbp : kb - nkbp) : kb;
        const int8_t* b = pb + kbb * kstride;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
            for (int m = 0; m < WM; ++m) fa[s][ks][m] = gload16(a + m * 2048 + ks * 1024);
#pragma unroll
            for (int n = 0; n < WN; ++n) fb[s][ks][n] = gload16(b + n * 2048 + ks * 1024);
        }
    }

    __device__ __forceinline__ void mma(int s) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int m = 0; m < WM; ++m) {
#pragma unroll
                for (int n = 0; n < WN; ++n)
                    acc[m][n] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[s][ks][m], fb[s][ks][n],
                                                                      acc[m][n], 0, 0, 0);
                if (DIAG) {
                    const v4i x = fa[s][ks][m];
                    rs[m] = __builtin_amdgcn_sdot4(x.x, 0x01010101, rs[m], false);
                    rs[m] = __builtin_amdgcn_sdot4(x.y, 0x01010101, rs[m], false);
                    rs[m] = __builtin_amdgcn_sdot4(x.z, 0x01010101, rs[m], false);
                    rs[m] = __builtin_amdgcn_sdot4(x.w, 0x01010101, rs[m], false);
                }
            }
    }

    // STORE: also write the int32 tile to `tile` (row-major T x T).  Frame sums only when
    // `sums` is not null.
    __device__ __forceinline__ void run(int biased, int64_t* __restrict__ out,
                                        int64_t* __restrict__ sums,
                                        int* __restrict__ tile = nullptr) {
        for (int i = tid; i < 2 * S::NDIAG; i += 256) sDiag[i] = 0u;
#pragma unroll
        for (int m = 0; m < WM; ++m) {
            rs[m] = 0;
#pragma unroll
            for (int n = 0; n < WN; ++n)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[m][n][v] = 0;
        }

        // Fragment (k-block kb, 32-frame group g, half ks) starts at
        // slab_bin + (kb * ngroups + g) * 2048 + ks * 1024; lane l reads 16 bytes at +16 l.
        const int64_t kstride = (int64_t)(nrows >> 5) * 2048;
        const int8_t* pa = slab_bin + (int64_t)((row0 >> 5) + wr * WM) * 2048 + lane * 16;
        const int8_t* pb = slab_bin + (int64_t)((col0 >> 5) + wc * WN) * 2048 + lane * 16;
        // idle: every block of this wave is below the diagonal, or lies wholly in the
        // padding frames past the last one (a STORE tile's readers skip both parts)
        const bool idle = (DIAG && wr > wc) || row0 + wr * WM * 32 >= nframes ||
                          col0 + wc * WN * 32 >= nframes;
        if (!idle && kb0 < kb1) {
            const int last = kb1 - 1;
            load(0, kb0, pa, pb, kstride);
            load(1, min(kb0 + 1, last), pa, pb, kstride);
            for (int kb = kb0; kb < kb1; kb += 2) {
                mma(0);
                __builtin_amdgcn_sched_barrier(0);
                load(0, min(kb + 2, last), pa, pb, kstride);
                __builtin_amdgcn_sched_barrier(0);
                // An odd count ends with slot 1 holding a repeat of the last k-block:
                // its A fragments are zeroed so those MFMAs add nothing (no tail code
                // after the loop, whose live fragments would spill).
                const bool repeat = kb + 1 > last;
#pragma unroll
                for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                    for (int m = 0; m < WM; ++m) {
                        const v4i x = fa[1][ks][m];
                        fa[1][ks][m] = v4i{repeat ? 0 : x.x, repeat ? 0 : x.y, repeat ? 0 : x.z,
                                           repeat ? 0 : x.w};
                    }
                mma(1);
                __builtin_amdgcn_sched_barrier(0);
                load(1, min(kb + 3, last), pa, pb, kstride);
                __builtin_amdgcn_sched_barrier(0);
            }
        }

        if (DIAG && wr == wc && sums)
            frame_sums<WM>(rs, row0 + wr * WM * 32, lane, nframes,
                           biased ? (int64_t)128 * (kb1 - kb0) * KB : 0, sums);
        __syncthreads();
        if (!idle) fold_tile<WM, WN, STORE>(acc, wr, wc, lane, false, sDiag, tile);
        __syncthreads();
        flush_diagonals<S>(sDiag, false, tid, col0 - row0, nframes, out);
    }
};

// One 256 x 256 tile through an LDS ring (see above).
constexpr int GRAM_UNITS = 3;                      // units per stage
constexpr int GRAM_PANEL = 8 * 1024;               // one unit of a panel: 8 runs
constexpr int GRAM_STAGE = GRAM_UNITS * 2 * GRAM_PANEL;
typedef __attribute__((address_space(3))) void lds_void;
typedef float v16f __attribute__((ext_vector_type(16)));
typedef int v8i __attribute__((ext_vector_type(8)));

__device__ const int8_t gram_zeros[4 * 2048] __attribute__((aligned(1024))) = {};

// s_waitcnt immediates (vmcnt in bits 3:0 and 15:14, expcnt and lgkmcnt not waited for unless
// said).
constexpr int wait_vm(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }
constexpr int wait_vm_lgkm0(int n) { return 0x0070 | (n & 15) | ((n >> 4) << 14); }

// Operand formats.  I8: a unit is half a k-block (K = 32), one run is 32 frames x 32 bytes.
// F4 (narrow pixels, see k_narrow.hip): a unit is a whole k-block (K = 64) of FP4 codes, one
// run is 32 frames x 64 codes; a code c is the FP4 value c / 2, so sums of products come out
// in quarters, exactly (multiples of 1/4 below 2^22).
enum GramFormat { I8, F4 };
template <GramFormat FMT>
struct GramOps;
template <>
struct GramOps<I8> {
    typedef v16i Acc;
    static constexpr int PER_KB = 2;       // units per k-block
    static constexpr int RUN_STRIDE = 2048;  // bytes between neighbouring frame groups
    __device__ __forceinline__ static v16i mma(v4i a, v4i b, v16i c) {
        return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
    }
    __device__ __forceinline__ static int sum(v4i x, int s) {  // + the 16 bytes
#pragma unroll
        for (int i = 0; i < 4; ++i) s = __builtin_amdgcn_sdot4(x[i], 0x01010101, s, false);
        return s;
    }
};
template <>
struct GramOps<F4> {
    typedef v16f Acc;
    static constexpr int PER_KB = 1;
    static constexpr int RUN_STRIDE = 1024;
    __device__ __forceinline__ static v16f mma(v4i a, v4i b, v16f c) {
        const v8i x = __builtin_shufflevector(a, a, 0, 1, 2, 3, -1, -1, -1, -1);
        const v8i y = __builtin_shufflevector(b, b, 0, 1, 2, 3, -1, -1, -1, -1);
        return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(x, y, c, 4, 4, 0, 0, 0, 0);
    }
    __device__ __forceinline__ static int sum(v4i x, int s) {  // + the 32 codes' counts
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t mag = (uint32_t)x[i] & 0x77777777u;
            const uint32_t neg = ((uint32_t)x[i] >> 3) & 0x11111111u;
            s = (int)__builtin_amdgcn_udot8(mag, 0x11111111u, (uint32_t)s, false);
            s -= 2 * (int)__builtin_amdgcn_udot8(mag, neg, 0u, false);
        }
        return s;
    }
};

// One k-range of a tile in one format: acc += panel x panel^T.
template <GramFormat FMT, bool DIAG, bool CROSS>
struct PanelLoop {
    using Ops = GramOps<FMT>;
    static constexpr int U = GRAM_UNITS;
    const int8_t* __restrict__ slab_bin;
    int kb0, kb1, row0, col0, nrows;
    int lane, wr, wc;
    int nkbp;  // CROSS: k-blocks per digit plane (B reads kb + nkbp or kb - nkbp)

    typename Ops::Acc acc[4][4];
    v4i fa[U][4], fb[U][4];
    int rs[4];     // DIAG: partial frame sums of this lane's A rows

    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            rs[m] = 0;
#pragma unroll
            for (int n = 0; n < 4; ++n)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[m][n][v] = 0;
        }
    }
    // This wave's source of unit u (its four runs are RUN_STRIDE bytes apart): waves 0 and 1
    // copy the row panel, 2 and 3 the column panel.
    __device__ __forceinline__ const int8_t* source(int u) const {
        int kb = u / Ops::PER_KB;
        const bool past = kb >= kb1;
        kb = min(kb, kb1 - 1);
        if (CROSS && wr) kb = kb < nkbp ? kb + nkbp : kb - nkbp;
        const int group = ((wr ? col0 : row0) >> 5) + wc * 4;
        const int8_t* p = slab_bin + ((int64_t)kb * (nrows >> 5) + group) * Ops::RUN_STRIDE +
                          (u % Ops::PER_KB) * 1024;
        return past && !wr ? gram_zeros : p;
    }
    __device__ __forceinline__ void dma(int8_t* buf, int un, const int8_t* src, int o) const {
        __builtin_amdgcn_global_load_lds(
            (const void*)(src + o * Ops::RUN_STRIDE + lane * 16),
            (lds_void*)(buf + (un * 2 + wr) * GRAM_PANEL + (wc * 4 + o) * 1024), 16, 0, 0);
    }
    __device__ __forceinline__ v4i frag_a(const int8_t* unit, int m) const {
        return *reinterpret_cast<const v4i*>(unit + (wr * 4 + m) * 1024 + lane * 16);
    }
    __device__ __forceinline__ v4i frag_b(const int8_t* unit, int n) const {
        return *reinterpret_cast<const v4i*>(unit + GRAM_PANEL + (wc * 4 + n) * 1024 + lane * 16);
    }

    // The units of stage `cur` (unit 0's fragments are in slot 0), with the first fragments of
    // `next` and the copies of units u .. u + U - 1 into `rel`, the buffer of the stage before.
    __device__ __forceinline__ void stage(const int8_t* cur, const int8_t* next, int8_t* rel,
                                          int u) {
#pragma unroll
        for (int un = 0; un < U; ++un) {
            if (un == U - 1) {
                __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0((U - 1) * 4));
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");  // the reads below stay below
                __builtin_amdgcn_sched_barrier(0);
            }
            const int8_t* src = source(u + un);
            const int8_t* from = un + 1 < U ? cur + (un + 1) * 2 * GRAM_PANEL : next;
            const int sl = (un + 1) % U;
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                if (m == 0) {
                    fa[sl][0] = frag_a(from, 0);
                    fb[sl][0] = frag_b(from, 0);
                    fb[sl][1] = frag_b(from, 1);
                } else if (m == 1) {
                    fb[sl][2] = frag_b(from, 2);
                    fb[sl][3] = frag_b(from, 3);
                    fa[sl][1] = frag_a(from, 1);
                } else if (m == 2) {
                    fa[sl][2] = frag_a(from, 2);
                    fa[sl][3] = frag_a(from, 3);
                }
                dma(rel, un, src, m);
                const v4i x = fa[un][m];
#pragma unroll
                for (int n = 0; n < 4; ++n) acc[m][n] = Ops::mma(x, fb[un][n], acc[m][n]);
                if (DIAG) rs[m] = Ops::sum(x, rs[m]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    // The same for a wave with nothing to compute: its copies and the barrier.
    __device__ __forceinline__ void idle_stage(int8_t* rel, int u) const {
#pragma unroll
        for (int un = 0; un < U; ++un) {
            if (un == U - 1) {
                __builtin_amdgcn_s_waitcnt(wait_vm((U - 1) * 4));
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
            }
            const int8_t* src = source(u + un);
#pragma unroll
            for (int o = 0; o < 4; ++o) dma(rel, un, src, o);
        }
    }
    // kb0 < kb1.  Ends with no copy in flight and no wave of the workgroup past its reads.
    __device__ __forceinline__ void run(bool idle, int8_t* buf0, int8_t* buf1, int8_t* buf2) {
        const int u0 = Ops::PER_KB * kb0;
        const int n_stage = (Ops::PER_KB * (kb1 - kb0) + U - 1) / U;
#pragma unroll
        for (int un = 0; un < 2 * U; ++un) {
            const int8_t* src = source(u0 + un);
#pragma unroll
            for (int o = 0; o < 4; ++o) dma(un < U ? buf0 : buf1, un % U, src, o);
        }
        __builtin_amdgcn_s_waitcnt(wait_vm(U * 4));
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        int st = 0, u = u0 + 2 * U;  // u: first unit copied by stage st
        if (idle) {
            for (; st + 3 <= n_stage; st += 3, u += 3 * U) {
                idle_stage(buf2, u);
                idle_stage(buf0, u + U);
                idle_stage(buf1, u + 2 * U);
            }
            if (st < n_stage) {
                idle_stage(buf2, u);
                if (st + 1 < n_stage) idle_stage(buf0, u + U);
            }
        } else {
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                fa[0][m] = frag_a(buf0, m);
                fb[0][m] = frag_b(buf0, m);
            }
            for (; st + 3 <= n_stage; st += 3, u += 3 * U) {
                stage(buf0, buf1, buf2, u);
                stage(buf1, buf2, buf0, u + U);
                stage(buf2, buf0, buf1, u + 2 * U);
            }
            if (st < n_stage) {
                stage(buf0, buf1, buf2, u);
                if (st + 1 < n_stage) stage(buf1, buf2, buf0, u + U);
            }
        }
        __builtin_amdgcn_s_waitcnt(wait_vm(0));
        __syncthreads();
    }
};

// A tile over k-blocks [kb0, kb1) of a slab in format FMT.  Its frame sums go to sums and to
// wsums, each when not null (wsums only beside sums).
template <GramFormat FMT, bool DIAG, bool CROSS, bool STORE>
__device__ __forceinline__ void panel_tile(const int8_t* __restrict__ slab_bin, int kb0, int kb1,
                                           int row0, int col0, int nframes, int nrows, int tid,
                                           int wr, int wc, int nkbp, int biased,
                                           int64_t* __restrict__ out, int64_t* __restrict__ sums,
                                           int64_t* __restrict__ wsums, int* __restrict__ tile,
                                           unsigned int* sDiag, int8_t* buf0, int8_t* buf1,
                                           int8_t* buf2) {
    using S = GramShape<4, 4>;
    const int lane = tid & 63;
    for (int i = tid; i < 2 * S::NDIAG; i += 256) sDiag[i] = 0u;
    // idle: every block of this wave is below the diagonal, or lies wholly in the padding
    // frames past the last one (a STORE tile's readers skip both parts)
    const bool idle = (DIAG && wr > wc) || row0 + wr * 128 >= nframes || col0 + wc * 128 >= nframes;
    PanelLoop<FMT, DIAG, CROSS> t{slab_bin, kb0, kb1, row0, col0, nrows, lane, wr, wc, nkbp};
    t.clear();
    t.run(idle, buf0, buf1, buf2);
    if (DIAG && wr == wc && sums) {
        const int64_t bias = biased ? (int64_t)128 * (kb1 - kb0) * KB : 0;
        frame_sums<4>(t.rs, row0 + wr * 128, lane, nframes, bias, sums);
        if (wsums) frame_sums<4>(t.rs, row0 + wr * 128, lane, nframes, bias, wsums);
    }
    // |value| <= 64 x 16384 a k-block (i8), 64 x 16 (FP4, at most 2047 k-blocks)
    const bool small = FMT == F4 || kb1 - kb0 < 8;
    if (!idle) fold_tile<4, 4, STORE>(t.acc, wr, wc, lane, small, sDiag, tile);
    __syncthreads();
    flush_diagonals<S>(sDiag, small, tid, col0 - row0, nframes, out);
}

// K-range of item `w` and the CROSS kernel's plane distance.  nwkb (uint16 plans whose
// wide pixels -- those with a count above 255 -- have k-blocks of their own; null: every
// item whole, distance nkb): per bin, `clip` k-blocks at the start of the high plane
// hold the wide pixels' high bytes, and
//  * HH items (plain, k-blocks below nkb) stop at clip; LL items are whole;
//  * cross items: the first half [0, nkb) stops at clip and reads its B operand `off`
//    k-blocks further; the second half [nkb, 2 nkb) moves to [off, off + clip) and reads
//    B `off` k-blocks back.  off = clip when the wide pixels' low bytes follow their high
//    bytes in the high plane (2 clip <= nkb), else nkb (clip = nkb: every pixel, the high
//    and low planes in list order).
struct ItemRange {
    int kb0, kb1, nkbp;
};
template <bool CROSS>
__device__ __forceinline__ ItemRange item_range(const GramWork& w, int nkb, const int* nwkb) {
    if (!nwkb) return ItemRange{w.kb0, w.kb1, nkb};
    const int clip = nwkb[w.bin];
    const int off = 2 * clip <= nkb ? clip : nkb;
    if (w.kb0 < nkb) return ItemRange{w.kb0, min(w.kb1, clip), off};
    if (!CROSS) return ItemRange{w.kb0, w.kb1, nkb};
    return ItemRange{off + (w.kb0 - nkb), off + min(w.kb1 - nkb, clip), off};
}

// One work item: the tile of `w` in a bin whose slab starts at slab_bin, over k-blocks
// [r.kb0, r.kb1) (a CROSS item's B operand r.nkbp k-blocks away).
// LDS of one workgroup: the diagonal sums, and for T = 256 the ring's buffers, which stay
// separate __shared__ arrays of the kernel (see the top of the file).
#define DXG2_GRAM_LDS(WM)                                                                     \
    constexpr int ring_bytes = WM == 4 ? GRAM_STAGE : 16;                                     \
    __shared__ __attribute__((aligned(1024))) int8_t buf0[ring_bytes];                        \
    __shared__ __attribute__((aligned(1024))) int8_t buf1[ring_bytes];                        \
    __shared__ __attribute__((aligned(1024))) int8_t buf2[ring_bytes];                        \
    __shared__ unsigned int sDiag[2 * GramShape<WM, WM>::NDIAG]

template <int WM, int WN, bool CROSS, bool STORE>
__device__ __forceinline__ void gram_item(const GramWork& w, ItemRange r, const int8_t* slab_bin,
                                          int nframes, int nrows, int biased,
                                          int64_t* __restrict__ out, int64_t* __restrict__ sums,
                                          int* __restrict__ tile, unsigned int* sDiag,
                                          int8_t* buf0, int8_t* buf1, int8_t* buf2,
                                          int64_t* __restrict__ wsums = nullptr) {
    using S = GramShape<WM, WN>;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    auto go = [&](auto diag) {
        constexpr bool DIAG = decltype(diag)::value;
        if constexpr (WM == 4) {
            panel_tile<I8, DIAG, CROSS, STORE>(slab_bin, r.kb0, r.kb1, w.ti * S::TM,
                                               w.tj * S::TN, nframes, nrows, tid, wave >> 1,
                                               wave & 1, r.nkbp, biased, out, sums, wsums, tile,
                                               sDiag, buf0, buf1, buf2);
        } else {
            GramTile<WM, WN, DIAG, CROSS, STORE> t{slab_bin, r.kb0, r.kb1, w.ti * S::TM,
                                                   w.tj * S::TN, nframes, nrows, tid, tid & 63,
                                                   wave >> 1, wave & 1, r.nkbp, sDiag};
            t.run(biased, out, sums, tile);
        }
    };
    if (!CROSS && w.ti == w.tj)
        go(std::true_type{});
    else
        go(std::false_type{});
}

template <int WM, int WN, bool CROSS>
__global__ __launch_bounds__(256) void gram_i8_kernel(const int8_t* __restrict__ slab,
                                                      const BinDev* __restrict__ bins,
                                                      const GramWork* __restrict__ work,
                                                      int nframes, int nrows, int biased,
                                                      const int* __restrict__ nwkb,
                                                      int64_t* __restrict__ ugram,
                                                      int64_t* __restrict__ sums) {
    using S = GramShape<WM, WN>;
    static_assert(S::TM == S::TN, "square tiles");
    DXG2_GRAM_LDS(WM);
    const GramWork w = work[blockIdx.x];
    if (w.bin < 0) return;  // padding item
    const BinDev bd = bins[w.bin];
    const ItemRange r = item_range<CROSS>(w, bd.nkb, nwkb);
    if (r.kb1 <= r.kb0) return;  // nothing of this item is left
    gram_item<WM, WN, CROSS, false>(w, r, slab + bd.slab_off, nframes, nrows, biased,
                                    ugram + (int64_t)w.out * nframes,
                                    sums + (int64_t)w.out * nframes, nullptr, sDiag, buf0, buf1, buf2);
}

// XCD (accelerator complex die) this wave runs on: HW_REG_XCC_ID bits [3:0].
__device__ __forceinline__ int xcc_id() {
    return (int)(__builtin_amdgcn_s_getreg((20) | (0 << 6) | (15 << 11)) & 0xF);
}

// Next work item for a workgroup on XCD `home`: the head of its own XCD's queue, then
// (once that is drained) the other XCDs' queues in turn.  Queue x holds items
// [qoff[x], qoff[x+1]) of the work list; heads[x] counts the items taken from it.
__device__ __forceinline__ int next_item(int home, const int* __restrict__ qoff, int* heads) {
    auto pop = [&](int x) {
        const int n = qoff[x + 1] - qoff[x];
        const int i = atomicAdd(heads + x, 1);
        return i < n ? qoff[x] + i : -1;
    };
    const int n0 = qoff[home + 1] - qoff[home];
    if (__hip_atomic_load(heads + home, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < n0) {
        const int i = pop(home);
        if (i >= 0) return i;
    }
    // the other heads are read together: one after the other, the last look at the drained
    // queues alone was several microseconds of every launch
    int seen[8];
#pragma unroll
    for (int k = 1; k < 8; ++k)
        seen[k] = __hip_atomic_load(heads + ((home + k) & 7), __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int k = 1; k < 8; ++k) {
        const int x = (home + k) & 7;
        if (seen[k] >= qoff[x + 1] - qoff[x]) continue;
        const int i = pop(x);
        if (i >= 0) return i;
    }
    return -1;
}

// Persistent grouped launch: one workgroup per resident slot, each taking tiles from
// the device work queues until all are empty.  Tiles of one queue share frame panels
// in their XCD's L2; stealing evens out the XCDs' finishing times.  heads[] must be
// zero at launch.
template <int WM, int WN, bool CROSS>
__global__ __launch_bounds__(256) void gram_i8_queue_kernel(
    const int8_t* __restrict__ slab, const BinDev* __restrict__ bins,
    const GramWork* __restrict__ work, const int* __restrict__ qoff, int* heads, int nframes,
    int nrows, int biased, const int* __restrict__ nwkb, int n_bins, int64_t* __restrict__ ugram,
    int64_t* __restrict__ sums, int64_t* __restrict__ wsums) {
    using S = GramShape<WM, WN>;
    static_assert(S::TM == S::TN, "square tiles");
    DXG2_GRAM_LDS(WM);
    __shared__ int s_item;
    if (wsums && nwkb[n_bins] == 0) return;  // no wide pixel in any bin
    const int home = xcc_id() & 7;
    for (;;) {
        if (threadIdx.x == 0) s_item = next_item(home, qoff, heads);
        __syncthreads();
        const int it = s_item;
        if (it < 0) break;
        const GramWork w = work[it];
        const BinDev bd = bins[w.bin];
        const ItemRange r = item_range<CROSS>(w, bd.nkb, nwkb);
        if (r.kb1 > r.kb0)  // the same for every thread of the workgroup
            gram_item<WM, WN, CROSS, false>(w, r, slab + bd.slab_off, nframes, nrows, biased,
                                            ugram + (int64_t)w.out * nframes,
                                            sums + (int64_t)w.out * nframes, nullptr, sDiag, buf0,
                                            buf1, buf2,
                                            wsums ? wsums + (int64_t)w.out * nframes : nullptr);
        __syncthreads();  // s_item and sDiag are reused by the next item
    }
}

// The narrow pixels' Gram of a plan with an FP4 slab (k_narrow.hip), when the call took that
// route.  The wide pixels' follows through gram_i8_queue_kernel, with nwkb and wsums.
__global__ __launch_bounds__(256) void gram_f4_queue_kernel(
    const int8_t* __restrict__ slab4, const BinDev* __restrict__ bins,
    const GramWork* __restrict__ work, const int* __restrict__ qoff, int* heads, int nframes,
    int nrows, const int* __restrict__ route, int64_t* __restrict__ ugram,
    int64_t* __restrict__ sums) {
    DXG2_GRAM_LDS(4);
    __shared__ int s_item;
    if (route[0] != NARROW_F4) return;
    const int home = xcc_id() & 7;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    for (;;) {
        if (tid == 0) s_item = next_item(home, qoff, heads);
        __syncthreads();
        const int it = s_item;
        if (it < 0) break;
        const GramWork w = work[it];
        const int8_t* s4 = slab4 + bins[w.bin].slab_off / 2;
        const int64_t o = (int64_t)w.bin * nframes;
        if (w.ti == w.tj)
            panel_tile<F4, true, false, false>(s4, w.kb0, w.kb1, w.ti * 256, w.tj * 256, nframes,
                                               nrows, tid, wave >> 1, wave & 1, 0, 0, ugram + o,
                                               sums + o, nullptr, nullptr, sDiag, buf0, buf1,
                                               buf2);
        else
            panel_tile<F4, false, false, false>(s4, w.kb0, w.kb1, w.ti * 256, w.tj * 256, nframes,
                                                nrows, tid, wave >> 1, wave & 1, 0, 0, ugram + o,
                                                sums + o, nullptr, nullptr, sDiag, buf0, buf1,
                                                buf2);
        __syncthreads();  // s_item and sDiag are reused by the next item
    }
}

template <int WM, int WN, bool CROSS>
int queue_grid() {
    static int grid[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (!grid[dev]) {
        int cus = 0, per = 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            cus = 256;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &per, reinterpret_cast<const void*>(gram_i8_queue_kernel<WM, WN, CROSS>), 256, 0) !=
                hipSuccess ||
            per < 1)
            per = 1;
        grid[dev] = cus * per;
    }
    return grid[dev];
}

void launch_gram_f4_queue(const int8_t* slab4, const BinDev* bins, const GramWork* work,
                          int n_work, const int* qoff, int* heads, int nframes, int nrows,
                          const int* route, int64_t* ugram, int64_t* sums, hipStream_t s) {
    if (n_work <= 0) return;
    gram_f4_queue_kernel<<<dim3((unsigned)std::min(n_work, queue_grid<4, 4, false>())), 256, 0,
                           s>>>(slab4, bins, work, qoff, heads, nframes, nrows, route, ugram,
                                sums);
}

void gram_queue_prepare(int tile) {
    if (tile == 128) {
        (void)queue_grid<2, 2, false>();
        (void)queue_grid<2, 2, true>();
    } else {
        (void)queue_grid<4, 4, false>();
        (void)queue_grid<4, 4, true>();
    }
}

void launch_gram_i8_queue(int tile, bool cross, const int8_t* slab, const BinDev* bins,
                          const GramWork* work, int n_work, const int* qoff, int* heads,
                          int nframes, int nrows, int biased, const int* nwkb, int64_t* ugram,
                          int64_t* sums, hipStream_t s, int n_bins, int64_t* wsums) {
    if (n_work <= 0) return;
    const dim3 block(256);
#define DXG2_QUEUE_LAUNCH(WM, CR)                                                             \
    gram_i8_queue_kernel<WM, WM, CR><<<dim3((unsigned)std::min(n_work, queue_grid<WM, WM, CR>())), \
                                       block, 0, s>>>(slab, bins, work, qoff, heads, nframes,    \
                                                      nrows, biased, nwkb, n_bins, ugram, sums,  \
                                                      wsums)
    if (tile == 128) {
        if (cross)
            DXG2_QUEUE_LAUNCH(2, true);
        else
            DXG2_QUEUE_LAUNCH(2, false);
    } else {
        if (cross)
            DXG2_QUEUE_LAUNCH(4, true);
        else
            DXG2_QUEUE_LAUNCH(4, false);
    }
#undef DXG2_QUEUE_LAUNCH
}

// calc_std variant: the same tiles (work items carry a scratch slot), which also write
// their int32 tile to tiles + slot * T * T for the per-element ratio pass.  Where one launch
// covers every tile its diagonal tiles give the frame sums as in the plain launch (a pass over
// the slab for them took 0.21 of 1.89 ms at 480,000 pixels x 2,000 frames); a chunk of the
// tiles cannot be reduced before all its frames' sums are known, so with several chunks they
// come from that pass (sums is null here).
template <int WM, int WN, bool CROSS>
__global__ __launch_bounds__(256) void gram_i8_store_kernel(
    const int8_t* __restrict__ slab, const BinDev* __restrict__ bins,
    const GramWork* __restrict__ work, int nframes, int nrows, int biased,
    int64_t* __restrict__ ugram, int64_t* __restrict__ sums, int* __restrict__ tiles) {
    using S = GramShape<WM, WN>;
    static_assert(S::TM == S::TN, "square tiles");
    DXG2_GRAM_LDS(WM);
    const GramWork w = work[blockIdx.x];
    if (w.bin < 0) return;  // padding item
    const BinDev bd = bins[w.bin];
    gram_item<WM, WN, CROSS, true>(w, ItemRange{w.kb0, w.kb1, bd.nkb}, slab + bd.slab_off,
                                   nframes, nrows, biased, ugram + (int64_t)w.out * nframes,
                                   sums ? sums + (int64_t)w.out * nframes : nullptr,
                                   tiles + (int64_t)w.slot * S::TM * S::TN, sDiag,
                                   buf0, buf1, buf2);
}

// Grouped launch over several plans (continuous batching of dense jobs): the same tile
// code, with the slab, bins, frame counts and outputs of each item's job.
template <int WM, int WN, bool CROSS>
__global__ __launch_bounds__(256) void gram_i8_jobs_kernel(const GramJob* __restrict__ jobs,
                                                           const GramWork* __restrict__ work) {
    using S = GramShape<WM, WN>;
    static_assert(S::TM == S::TN, "square tiles");
    DXG2_GRAM_LDS(WM);
    const GramWork w = work[blockIdx.x];
    if (w.bin < 0) return;  // padding item
    const GramJob j = jobs[w.job];
    const BinDev bd = gload_bin(j.bins + w.bin);
    gram_item<WM, WN, CROSS, false>(w, ItemRange{w.kb0, w.kb1, bd.nkb}, j.slab + bd.slab_off,
                                    j.nframes, j.nrows, j.biased,
                                    j.ugram + (int64_t)w.out * j.nframes,
                                    j.sums + (int64_t)w.out * j.nframes, nullptr, sDiag, buf0, buf1, buf2);
}

void launch_gram_i8_jobs(int tile, bool cross, const GramJob* jobs, const GramWork* work,
                         int n_work, hipStream_t s) {
    if (n_work <= 0) return;
    const dim3 grid((unsigned)n_work), block(256);
    if (tile == 128) {
        if (cross)
            gram_i8_jobs_kernel<2, 2, true><<<grid, block, 0, s>>>(jobs, work);
        else
            gram_i8_jobs_kernel<2, 2, false><<<grid, block, 0, s>>>(jobs, work);
    } else {
        if (cross)
            gram_i8_jobs_kernel<4, 4, true><<<grid, block, 0, s>>>(jobs, work);
        else
            gram_i8_jobs_kernel<4, 4, false><<<grid, block, 0, s>>>(jobs, work);
    }
}

int gram_tile_size(int variant) { return variant == 1 ? 128 : 256; }

void launch_gram_i8_store(int tile, bool cross, const int8_t* slab, const BinDev* bins,
                          const GramWork* work, int n_work, int nframes, int nrows, int biased,
                          int64_t* ugram, int64_t* sums, int* tiles, hipStream_t s) {
    if (n_work <= 0) return;
    const dim3 grid((unsigned)n_work), block(256);
    if (tile == 128) {
        if (cross)
            gram_i8_store_kernel<2, 2, true><<<grid, block, 0, s>>>(slab, bins, work, nframes,
                                                                    nrows, biased, ugram, sums, tiles);
        else
            gram_i8_store_kernel<2, 2, false><<<grid, block, 0, s>>>(slab, bins, work, nframes,
                                                                     nrows, biased, ugram, sums, tiles);
    } else {
        if (cross)
            gram_i8_store_kernel<4, 4, true><<<grid, block, 0, s>>>(slab, bins, work, nframes,
                                                                    nrows, biased, ugram, sums, tiles);
        else
            gram_i8_store_kernel<4, 4, false><<<grid, block, 0, s>>>(slab, bins, work, nframes,
                                                                     nrows, biased, ugram, sums, tiles);
    }
}

void launch_gram_i8(int tile, bool cross, const int8_t* slab, const BinDev* bins,
                    const GramWork* work, int n_work, int nframes, int nrows, int biased,
                    const int* nwkb, int64_t* ugram, int64_t* sums, hipStream_t s) {
    if (n_work <= 0) return;
    const dim3 grid((unsigned)n_work), block(256);
    if (tile == 128) {
        if (cross)
            gram_i8_kernel<2, 2, true><<<grid, block, 0, s>>>(slab, bins, work, nframes, nrows,
                                                              biased, nwkb, ugram, sums);
        else
            gram_i8_kernel<2, 2, false><<<grid, block, 0, s>>>(slab, bins, work, nframes, nrows,
                                                               biased, nwkb, ugram, sums);
    } else {
        if (cross)
            gram_i8_kernel<4, 4, true><<<grid, block, 0, s>>>(slab, bins, work, nframes, nrows,
                                                              biased, nwkb, ugram, sums);
        else
            gram_i8_kernel<4, 4, false><<<grid, block, 0, s>>>(slab, bins, work, nframes, nrows,
                                                               biased, nwkb, ugram, sums);
    }
}

}  // namespace dxg2
