// half_tile.h -- matrix-core tiles over operands that are already fp16 in
// memory (packed by the caller): LDS-DMA loads, no register staging.
//
// A K slice of an operand tile goes from memory to LDS by
// `buffer_load_dwordx4 ... lds`: each lane names the 16 bytes it wants, and
// the wave's 64 pieces land at consecutive LDS addresses in lane order. The
// bank swizzle is therefore applied on the source side: the lane that fills
// slot s of a row asks for the chunk that belongs there. Two layouts:
//   K-contiguous  (rows of BK halves, one per M / N index), read as fragments
//                 by one ds_read_b128;
//   MN-contiguous (rows of R halves, one per k), read as fragments by two
//                 ds_read_b64_tr_b16, which transpose 4 k x 16 columns.
// Loads past the buffer's end (an offset of kBufOOB) put zeros into LDS.
#pragma once

#include <type_traits>

#include "mfma_core.h"

namespace seera {

typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef __fp16 fp16x4 __attribute__((ext_vector_type(4)));

template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt holds 6 bits");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// Every wave's LDS reads are done and every wave is here; no wait for loads in
// flight (a __syncthreads() would wait for the whole DMA pipeline).
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

typedef int dma_rsrc_t __attribute__((ext_vector_type(4)));

// 16 bytes per lane from resource r at voff + soff to LDS, lane after lane from
// `lds` (wave-uniform). Written in asm, which has no register result: through
// the builtin the compiler sees LDS written and waits for every load in flight
// before each transposed read (dW of 64 images, 256 -> 256 channels at 14 x 14:
// 43.6 against 27.2 us). The callers wait (wait_vm) before a barrier that precedes the reads.
__device__ __forceinline__ void dma16(dma_rsrc_t r, half_t* lds, uint32_t voff, uint32_t soff) {
    const uint32_t at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) half_t*)lds;
    // M0 holds the LDS address. The compiler never allocates it, and warns that a
    // clobber of it will not be preserved, which is what is meant: an M0 that it
    // set up itself before this statement has to be set up again after it.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(at), "v"(voff), "s"(r), "s"(soff)
                 : "memory", "m0");
#pragma clang diagnostic pop
}

// The words of a buffer resource over `bytes` bytes at `base` (wave-uniform; at
// most kMaxTileSpanBytes): raw 32-bit format as in make_rsrc.
__device__ __forceinline__ dma_rsrc_t make_dma_rsrc(const void* base, uint32_t bytes) {
    const uint64_t a = (uint64_t)base;
    return dma_rsrc_t{(int)(uint32_t)a, (int)((uint32_t)(a >> 32) & 0xFFFF), (int)bytes, 0x00020000};
}

// ---- K-contiguous tile: R rows x BK halves ----
template <int R, int BK, int NT>
struct KcTile {
    static constexpr int HALVES = R * BK;
    static constexpr int ITEMS = R * BK / 8;
    static constexpr int PASSES = ITEMS / NT;
    static_assert(ITEMS % NT == 0, "every thread moves the same number of pieces");
    // The row and the chunk (8 halves) of it that item `i` fills: the inverse
    // of lds_off.
    static __device__ __forceinline__ void item(int i, int& row, int& chunk) {
        const int j = i >> 3, s = i & 7;
        if constexpr (BK == 64) {
            row = j;
            chunk = s ^ (((j ^ (j >> 3)) & 3) | (j & 4));
        } else {
            static_assert(BK == 32, "BK must be 32 or 64");
            const int x = s ^ (((j ^ (j >> 2)) & 1) | (j & 2) | ((j >> 1) & 4));
            row = 2 * j + (x >> 2);
            chunk = x & 3;
        }
    }
    static __device__ __forceinline__ half8 frag(const half_t* tile, int m0, int kk, int lane) {
        return lds_read8<BK>(tile, m0 + (lane & 31), kk * 2 + (lane >> 5));
    }
};

// ---- MN-contiguous tile: BK rows (k) x R halves ----
template <int R, int BK, int NT>
struct McTile {
    static_assert(R == 64 || R == 128 || R == 256, "rows of 128, 256 or 512 bytes");
    static constexpr int HALVES = R * BK;
    static constexpr int ITEMS = R * BK / 8;
    static constexpr int PASSES = ITEMS / NT;
    static constexpr int CPR = R / 8;
    static_assert(ITEMS % NT == 0, "every thread moves the same number of pieces");
    // A transposed read takes 4 consecutive k x 64 bytes per half wave: the
    // 64-byte groups of 4 consecutive rows go to different places modulo the
    // 256 bytes that one access covers.
    static __device__ __forceinline__ int swz(int k) {
        return R >= 128 ? (k & 3) << 2 : ((k >> 1) & 1) << 2;
    }
    static __device__ __forceinline__ void item(int i, int& k, int& chunk) {
        k = i / CPR;
        chunk = (i % CPR) ^ swz(k);
    }
    static __device__ __forceinline__ half4 tr4(const half_t* tile, int k, int col) {
        const half_t* p = tile + k * R + ((((col >> 3) ^ swz(k)) << 3) | (col & 7));
        typedef __attribute__((address_space(3))) fp16x4 lds_fp16x4;
        return __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_fp16x4*)(p)));
    }
    static __device__ __forceinline__ half8 frag(const half_t* tile, int m0, int kk, int lane) {
        // lane 16 g + 4 e + c reads k = e, columns 4c .. 4c + 3 of its group's
        // 4 x 16 block; it receives column 4 (its own l % 16) of the four k.
        const int g = lane >> 4, e = (lane >> 2) & 3, c = lane & 3;
        const int k = kk * 16 + 8 * (g >> 1) + e, col = m0 + 16 * (g & 1) + 4 * c;
        const half4 lo = tr4(tile, k, col), hi = tr4(tile, k + 4, col);
        return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    }
};

// acc[i][j] += sum over `n` slices of A rows (m0 + 32 i ..) x B rows (n0 + 32 j
// ..), KK 16-deep steps of each from step kk0 on. Stage t of `smem` (`stage`
// halves each, NS of them) holds slice s with s % NS == t: A at 0, B at b_off.
//   load(l, dst)   issues load l (of LOADS) of the next slice into the stage
//                  at dst; called for the slices in order
//   done(s)        after the products of slice s
// One barrier per slice, in front of the slice's last step: there every wave
// has read all of slice s, so the stage is free for slice s + NS, and slice
// s + 1 has landed, so its first fragments are read behind the products of the
// last step. The matrix cores have work queued across the barrier, and every
// fragment is read one step ahead of its products (left to itself the
// scheduler sinks each read to just before its use). The DMA instructions are
// dealt out among the products: issued in one go they hold the wave for as
// long as the loads take to enter the memory pipe, about as long as a slice's
// products.
template <class TA, class TB, int KK, int NS, int LOADS, int TM, int TN, class Load, class Done>
__device__ __forceinline__ void half_pipeline(half_t* smem, int stage, int b_off, int m0, int n0,
                                              int kk0, int lane, int n, floatx16 (&acc)[TM][TN],
                                              Load load, Done done) {
    static_assert(KK % 2 == 0 && NS >= 3, "fragment sets alternate by step; two slices in flight");
    constexpr int NM = (KK - 1) * TM * TN;  // products that loads are dealt among
    half8 a[2][TM], b[2][TN];
    auto read = [&](const half_t* t, int kk) {
#pragma unroll
        for (int i = 0; i < TM; ++i) a[kk & 1][i] = TA::frag(t, m0 + 32 * i, kk0 + kk, lane);
#pragma unroll
        for (int j = 0; j < TN; ++j) b[kk & 1][j] = TB::frag(t + b_off, n0 + 32 * j, kk0 + kk, lane);
    };
    auto products = [&](int kk, auto between) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                acc[i][j] = mfma32x32x16(a[kk & 1][i], b[kk & 1][j], acc[i][j]);
                between((kk * TM + i) * TN + j);
            }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto nothing = [](int) {};
    if (n <= 0) return;
#pragma unroll
    for (int s = 0; s < NS - 1; ++s)
        if (s < n) {
#pragma unroll
            for (int l = 0; l < LOADS; ++l) load(l, smem + s * stage);
        }
    if (n >= NS - 1)
        wait_vm<LOADS * (NS - 2)>();
    else
        wait_vm<0>();
    lds_barrier();
    read(smem, 0);
    const half_t* cur = smem;
    half_t* prev = smem + (NS - 1) * stage;  // the stage that slice s - 1 left
    const half_t* const last = smem + (NS - 1) * stage;
    int s = 0;
    for (; s + NS - 1 < n; ++s) {
        const half_t* nxt = cur == last ? smem : cur + stage;
#pragma unroll
        for (int kk = 0; kk + 1 < KK; ++kk) {
            read(cur, kk + 1);
            products(kk, [&](int m) {
#pragma unroll
                for (int l = m * LOADS / NM; l < (m + 1) * LOADS / NM; ++l) {
                    __builtin_amdgcn_sched_barrier(0);
                    load(l, prev);
                    __builtin_amdgcn_sched_barrier(0);
                }
            });
        }
        wait_vm<LOADS * (NS - 2)>();
        lds_barrier();
        read(nxt, 0);
        products(KK - 1, nothing);
        done(s);
        prev = const_cast<half_t*>(cur);
        cur = nxt;
    }
    for (; s < n; ++s) {
        const half_t* nxt = cur == last ? smem : cur + stage;
#pragma unroll
        for (int kk = 0; kk + 1 < KK; ++kk) {
            read(cur, kk + 1);
            products(kk, nothing);
        }
        if (s + 1 < n) {
            wait_vm<0>();
            lds_barrier();
            read(nxt, 0);
        }
        products(KK - 1, nothing);
        done(s);
        cur = nxt;
    }
}

// The sums of at most PARTS slices at a time: after every PARTS-th slice the
// accumulators are added to `sum` and begun anew. A chain of fp32 additions
// rounds in proportion to its length, so the parts keep the error of one long
// contraction at that of the kernels which split it.
template <int PARTS, int TM, int TN>
__device__ __forceinline__ void add_part(int s, floatx16 (&acc)[TM][TN], floatx16 (&sum)[TM][TN]) {
    if (s % PARTS != PARTS - 1) return;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                sum[i][j][r] += acc[i][j][r];
                acc[i][j][r] = 0.f;
            }
}

// Wave groups that split K hand their sums to group 0 through LDS: wave w of
// group g > 0 adds into wave w of group 0, group after group in order. `lds`
// holds 16 * TM * TN floats per thread of one group. Called by every wave.
template <int KG, int GW, int TM, int TN>
__device__ __forceinline__ void sum_groups(float* lds, int wave, int lane, floatx16 (&acc)[TM][TN]) {
    if constexpr (KG > 1) {
        const int g = wave / GW, t = (wave % GW) * 64 + lane;
#pragma unroll
        for (int k = 1; k < KG; ++k) {
            __syncthreads();
            if (g == k) {
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                            lds[((i * TN + j) * 16 + r) * (GW * 64) + t] = acc[i][j][r];
            }
            __syncthreads();
            if (g == 0) {
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                            acc[i][j][r] += lds[((i * TN + j) * 16 + r) * (GW * 64) + t];
            }
        }
    }
}

// n / d for 0 <= n < 2^31 by a multiplication (Granlund and Montgomery 1994):
// three instructions where a division takes about thirty. Built on the host.
struct FastDiv {
    uint32_t mul, shift;
    FastDiv() = default;
    explicit FastDiv(uint32_t d) {
        shift = 0;
        while ((1ull << shift) < d) ++shift;
        mul = (uint32_t)((((1ull << shift) - d) << 32) / d + 1);
    }
    __device__ __forceinline__ int div(int n) const {
        return (int)((__umulhi((uint32_t)n, mul) + (uint32_t)n) >> shift);
    }
};

// The workgroup's place in an order in which the blocks that one XCD receives
// (the dispatcher deals ids round-robin over the 8 XCDs) are consecutive:
// neighbours share operand rows in that XCD's L2. A bijection on [0, n).
__device__ __forceinline__ int xcd_order(int bid, int n) {
    const int x = bid & 7, i = bid >> 3, q = n >> 3, r = n & 7;
    return x * q + min(x, r) + i;
}

}  // namespace seera
