// FP8 GEMM for gfx950: D[N][M] = (B[N][K] . A[M][K]^T) * a_scale_inv * b_scale_inv (+bias) (+D).
//
// Both operands are K-contiguous, which is the layout the 32x32x64 FP8 MFMA wants: a lane holds
// 32 consecutive K bytes of one row.  Inside the kernel the operand that supplies D's rows is X
// (= B of the API, N rows) and the one that supplies D's columns is Y (= A of the API, M rows).
//
// Block tile BR x BC over K slices of 128 bytes, four wavefronts in a 2 x 2 arrangement, LDS
// double-buffered with a 16-byte-chunk XOR swizzle that keeps both the 128-bit tile writes and
// the 128-bit fragment reads off shared banks.  Tiles are handed to workgroups so that the
// workgroups of one XCD (one L2) work on neighbouring tiles.
#pragma once
#include "common.cuh"
#include "gemm_call.h"

#include <atomic>

#include <type_traits>

namespace msamp {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kGemmThreads = 256;

__device__ __forceinline__ int swz(int row, int chunk) { return chunk ^ ((row & 7) ^ ((row >> 3) & 1)); }

template <int ROWS, bool KGUARD>
struct TileLoader {
    static constexpr int kIters = ROWS * 8 / kGemmThreads;
    uint4 regs[kIters];

    // rows beyond `nrows` are clamped (their products land in output rows that are never stored);
    // with KGUARD, K chunks beyond `K` read as zero (without it K is a multiple of the stage).
    __device__ __forceinline__ void gload(const uint8_t* __restrict__ base, int row0, int nrows, int K, int k0) {
        const int t = threadIdx.x;
#pragma unroll
        for (int i = 0; i < kIters; ++i) {
            const int idx = t + kGemmThreads * i;
            const int r = idx >> 3, c = idx & 7;
            int gr = row0 + r;
            gr = gr < nrows ? gr : nrows - 1;
            const int kk = k0 + c * 16;
            if (!KGUARD || kk < K) {
                regs[i] = *reinterpret_cast<const uint4*>(base + static_cast<size_t>(gr) * K + kk);
            } else {
                regs[i] = make_uint4(0, 0, 0, 0);
            }
        }
    }
    __device__ __forceinline__ void lstore(uint8_t* lds) const {
        const int t = threadIdx.x;
#pragma unroll
        for (int i = 0; i < kIters; ++i) {
            const int idx = t + kGemmThreads * i;
            const int r = idx >> 3, c = idx & 7;
            *reinterpret_cast<uint4*>(lds + r * kBK + (swz(r, c) << 4)) = regs[i];
        }
    }
};

// 32 K-bytes of one tile row for this lane: chunks 2*kc, 2*kc+1 of the 128-byte row
__device__ __forceinline__ v8i read_frag(const uint8_t* lds, int row, int kc) {
    const v4i lo = *reinterpret_cast<const v4i*>(lds + row * kBK + (swz(row, 2 * kc) << 4));
    const v4i hi = *reinterpret_cast<const v4i*>(lds + row * kBK + (swz(row, 2 * kc + 1) << 4));
    v8i f;
    f[0] = lo[0], f[1] = lo[1], f[2] = lo[2], f[3] = lo[3];
    f[4] = hi[0], f[5] = hi[1], f[6] = hi[2], f[7] = hi[3];
    return f;
}

typedef float v4f __attribute__((ext_vector_type(4)));

// 16 x 16 x 128 FP8 MFMA (the non-scaled form: block scales 0).  On this part it sustains about a tenth more
// throughput under the power limit than the 32 x 32 x 64 form on the same data.
template <int XF, int YF>
__device__ __forceinline__ v4f mfma16(const v8i& x, const v8i& y, const v4f& c) {
    constexpr int cb = (XF == MSAMP_DT_E4M3) ? 0 : 1;
    constexpr int bl = (YF == MSAMP_DT_E4M3) ? 0 : 1;
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(x, y, c, cb, bl, 0, 0, 0, 0);
}

template <typename OT>
__device__ __forceinline__ void store_out(OT* p, float v, bool accumulate) {
    if (accumulate) v += Elem<OT>::load(p);
    Elem<OT>::store(p, v);
}

__device__ __forceinline__ float load_bias(const void* bias, int dt, int i) {
    if (dt == MSAMP_DT_F32) return static_cast<const float*>(bias)[i];
    if (dt == MSAMP_DT_F16) return f16_bits_to_float(static_cast<const uint16_t*>(bias)[i]);
    return bf16_bits_to_float(static_cast<const uint16_t*>(bias)[i]);
}

// workgroup id -> tile, keeping the workgroups of one XCD on adjacent tiles and walking groups of `kGroup` tile rows
// column by column (or, with `by_columns`, groups of tile columns row by row): the 32 CUs of an XCD then work on an
// 8 x 4 patch of tiles and share its 12 operand panels through that L2.
__device__ __forceinline__ void tile_of_id(int id, int tiles_r, int tiles_c, bool by_columns, bool wide, int& tr, int& tc) {
    constexpr int kXcd = 8, kGroup = 8;
    const int n_a = by_columns ? tiles_c : tiles_r, n_b = by_columns ? tiles_r : tiles_c;    // a: grouped, b: walked
    const int nt = tiles_r * tiles_c;
    // XCD x runs the workgroups x, x + 8, ...: they get the contiguous ids that start where those of XCDs 0 .. x-1 end
    // (the first nt % 8 XCDs run one workgroup more than the others)
    const int x = id % kXcd, extra = nt % kXcd;
    id = x * (nt / kXcd) + (x < extra ? x : extra) + id / kXcd;
    const int per_group = kGroup * n_b;
    const int g = id / per_group;
    const int first_a = g * kGroup;
    const int here = (n_a - first_a) < kGroup ? (n_a - first_a) : kGroup;
    const int in_g = id - g * per_group;
    int a = first_a + in_g % here, b = in_g / here;
    if (wide && here == kGroup) {
        // the patch of an XCD the other way round: 32 consecutive ids are 4 of the grouped dimension x 8 of the walked one
        const int blk = in_g / (8 * kGroup), r = in_g % (8 * kGroup);
        if ((blk + 1) * 8 <= n_b) {
            a = first_a + (r / 32) * 4 + (r % 4);
            b = blk * 8 + (r % 32) / 4;
        }
    }
    tr = by_columns ? b : a;
    tc = by_columns ? a : b;
}
__device__ __forceinline__ void tile_of_block(int tiles_r, int tiles_c, int& tr, int& tc) {
    tile_of_id(blockIdx.x, tiles_r, tiles_c, false, false, tr, tc);
}

// Which operand the walk of 256 x 256 tiles groups.  The panels of the grouped operand (eight per group, one group per
// XCD at a time) are read again for every few tiles of the walk, out of the memory-side cache if they are still
// there; the other operand streams past and is swept once per group.  Between two sweeps the cache has to hold the
// grouped panels in flight plus all of the other operand.  When that fits, grouping the larger operand is better (each
// of its panels comes from HBM once, in a burst at the start of a group; a streamed large operand puts HBM latency into
// every tile); when it does not, the grouped panels of a large operand are evicted between two reads, and grouping the
// smaller one loses less.  Measured on 64 shapes (4096 .. 32768 squared, K 4096 .. 28672): up to 16 % between the two
// walks, and this rule picks the faster one wherever they differ by more than 3 %.
__device__ __forceinline__ bool walk_by_columns(int tiles_r, int tiles_c, int K) {
    constexpr long long kCacheBudget = 288ll << 20;    // a little above the 256 MiB: eviction is not strictly LRU
    const long long panel = static_cast<long long>(kDmaTile) * K;
    const bool tall = tiles_r > tiles_c;
    const long long big = (tall ? tiles_r : tiles_c) * panel, small = (tall ? tiles_c : tiles_r) * panel;
    const long long in_flight = 64 * panel;
    const bool fits = (big < in_flight ? big : in_flight) + small <= kCacheBudget;
    return fits ? !tall : tall;
}

template <int BR, int BC, int XF, int YF, typename OT, bool KGUARD>
__global__ __launch_bounds__(kGemmThreads) void fp8_gemm_kernel(const uint8_t* __restrict__ X,
                                                                 const uint8_t* __restrict__ Y, OT* __restrict__ D,
                                                                 int NR, int NC, int K,
                                                                 const float* __restrict__ x_scale_inv,
                                                                 const float* __restrict__ y_scale_inv, int accumulate,
                                                                 const void* __restrict__ bias, int bias_dt) {
    constexpr int WR = BR / 2, WC = BC / 2;    // wave tile
    constexpr int TR = WR / 16, TC = WC / 16;  // MFMA tiles per wave
    constexpr int kStage = (BR + BC) * kBK;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];

    int tr, tc;
    tile_of_block((NR + BR - 1) / BR, (NC + BC - 1) / BC, tr, tc);
    const int row0 = tr * BR, col0 = tc * BC;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wr = wave >> 1, wc = wave & 1;
    const int l16 = lane & 15, g4 = lane >> 4;

    v4f acc[TR][TC];
#pragma unroll
    for (int i = 0; i < TR; ++i)
#pragma unroll
        for (int j = 0; j < TC; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.0f;

    TileLoader<BR, KGUARD> lx;
    TileLoader<BC, KGUARD> ly;
    const int nk = (K + kBK - 1) / kBK;
    // The K slices are walked in ascending order, 128 bytes of K per MFMA, exactly as the direct-to-LDS kernel below
    // walks them: the two kernels add up the same blocks in the same order and agree to the bit.  (Walking them in
    // an order rotated per workgroup, to spread the memory channels, was measured slower: 2-4 % at 2048 x 2048 x 4096,
    // 10-14 % at 4096 x 4096 x 4112.)
    auto slice = [&](int kt) { return kt * kBK; };
    lx.gload(X, row0, NR, K, slice(0));
    ly.gload(Y, col0, NC, K, slice(0));
    lx.lstore(smem);
    ly.lstore(smem + BR * kBK);
    __syncthreads();

    for (int kt = 0; kt < nk; ++kt) {
        const uint8_t* sx = smem + (kt & 1) * kStage;
        const uint8_t* sy = sx + BR * kBK;
        if (kt + 1 < nk) {
            lx.gload(X, row0, NR, K, slice(kt + 1));
            ly.gload(Y, col0, NC, K, slice(kt + 1));
        }
        {
            // a lane holds, for row lane % 16 of a 16-row block, the 32 K-bytes (lane / 16) * 32 .. + 31 of the slice
            v8i fx[TR], fy[TC];
#pragma unroll
            for (int i = 0; i < TR; ++i) fx[i] = read_frag(sx, wr * WR + i * 16 + l16, g4);
#pragma unroll
            for (int j = 0; j < TC; ++j) fy[j] = read_frag(sy, wc * WC + j * 16 + l16, g4);
#pragma unroll
            for (int i = 0; i < TR; ++i)
#pragma unroll
                for (int j = 0; j < TC; ++j) acc[i][j] = mfma16<XF, YF>(fx[i], fy[j], acc[i][j]);
        }
        if (kt + 1 < nk) {
            uint8_t* nx = smem + ((kt + 1) & 1) * kStage;
            lx.lstore(nx);
            ly.lstore(nx + BR * kBK);
        }
        __syncthreads();
    }

    // srcA = X rows: a lane holds D column (Y row) lane % 16 of a block and the four D rows (lane / 16) * 4 .. + 3
    const float alpha = (*x_scale_inv) * (*y_scale_inv);
#pragma unroll
    for (int j = 0; j < TC; ++j) {
        const int col = col0 + wc * WC + j * 16 + l16;
        if (col >= NC) continue;
        const float bv = bias != nullptr ? load_bias(bias, bias_dt, col) : 0.0f;
#pragma unroll
        for (int i = 0; i < TR; ++i) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = row0 + wr * WR + i * 16 + g4 * 4 + r;
                if (row < NR) {
                    store_out<OT>(D + static_cast<size_t>(row) * NC + col, fmaf(acc[i][j][r], alpha, bv), accumulate != 0);
                }
            }
        }
    }
}



// two floats -> packed 16-bit pair with the hardware's round-to-nearest-even converters
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    const f32x2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
__device__ __forceinline__ uint32_t pack_f16(float a, float b) {
    const f32x2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2));
}

template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (N > 0) {
        static_for<N - 1>(f);
        f(std::integral_constant<int, N - 1>{});
    }
}

// four consecutive elements of an output row straight from the accumulators, one by one: ragged edges,
// bias and accumulation, all in float32 with a single rounding to the output type
template <typename OT>
__device__ __noinline__ void store_quad_slow(OT* D, int row, int col, int NR, int NC, float alpha, float v0, float v1,
                                             float v2, float v3, int accumulate, const void* bias, int bias_dt) {
    if (row >= NR) return;
    const float v[4] = {v0, v1, v2, v3};
    for (int e = 0; e < 4; ++e) {
        if (col + e >= NC) break;
        const float bv = bias != nullptr ? load_bias(bias, bias_dt, col + e) : 0.0f;
        store_out<OT>(D + static_cast<size_t>(row) * NC + col + e, fmaf(v[e], alpha, bv), accumulate != 0);
    }
}


// 16 bytes of output, stored past the caches (non-temporal).  A round of tiles writes 128 KiB per CU, 4 MiB per XCD: as
// ordinary stores that is the whole L2, and the operand panels that the next tiles are about to read get evicted for
// data nobody reads again soon.  Measured on the Llama-7B shapes: 3 to 9 % off the whole GEMM.
__device__ __forceinline__ void store_out16(void* p, const uint4& v) {
    typedef uint32_t v4u_t __attribute__((ext_vector_type(4)));
    const v4u_t vv = {v.x, v.y, v.z, v.w};
    __builtin_nontemporal_store(vv, static_cast<v4u_t*>(p));
}

// the old output of an accumulating GEMM is read once: past the caches as well
__device__ __forceinline__ uint4 load_out16(const void* p) {
    typedef uint32_t v4u_t __attribute__((ext_vector_type(4)));
    const v4u_t v = __builtin_nontemporal_load(static_cast<const v4u_t*>(p));
    return make_uint4(v[0], v[1], v[2], v[3]);
}

// ---------------------------------------------------------------------------------------------
// Main kernel: 256 x 256 output tile over 128-byte K slices, four wavefronts each owning a 128 x 128
// quadrant (8 x 8 accumulators of the 16x16x128 FP8 MFMA = 256 accumulation registers per lane).
//  * Tiles travel global -> LDS with the direct-to-LDS load: no staging registers, no LDS stores.  A
//    lane group of 8 fetches one whole 128-byte line (full-line requests are what the L2 serves best).
//  * The LDS is a ring of five blocks of 32 KiB, one operand's part of a slice each.  A slice is computed in four quarters of
//    16 MFMAs (X half x Y half); the fragment half the next quarters need is read while the current one executes.
//  * One workgroup barrier per slice, in the third quarter: by then every wave holds the whole slice in registers, so its two
//    blocks are refilled with Y of the slice after next and X of the one behind it, spread evenly over a slice's time.
//  * LDS reads and tile loads are interleaved with the MFMAs one at a time, so that neither the LDS nor
//    the vector-memory queue backs up and stalls the MFMA stream.
typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef const __attribute__((address_space(1))) void* gbl_ptr_t;

constexpr int kDmaBlock = kDmaTile * kBK;    // one operand's part of a slice: 32 KiB
constexpr int kDmaBlocks = 5;                // all 160 KiB of the LDS

// s_waitcnt vmcnt(N), leaving the other counters unconstrained (gfx9 encoding: vmcnt = [3:0] and [15:14])
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

//  * XT / YT: that operand is handed over K-major, T[K][rows] with the rows contiguous (the transpose of
//    what the product needs), so that callers need not materialize transposed copies.  Its slice sits in
//    LDS as 128 k-rows of 256 bytes (same 32 KiB block), filled by the same eight 1 KiB loads, and its
//    fragments come from the transposing LDS read: a 16-lane group reads eight k-rows of 16 bytes and
//    lane i receives byte i of each, i.e. eight consecutive k for its row -- four such reads make the
//    32-byte operand of the MFMA.  The 16-byte position inside a k-row is XOR-ed with k % 8 (on the global
//    side again) so that the eight k-rows of one read fall into different banks.  Needs that operand's
//    row count to be a multiple of 256.
typedef int v2i __attribute__((ext_vector_type(2)));

//  * QF (an FP8 format, or 0): the output is not stored in OT but cast on to FP8 with in-time scaling in the same
//    launch, the way cast_to_fp8 of the stored output would: D is rounded to OT in registers, max |D| is taken over
//    the whole matrix, the scale follows from it, and the codes of D * scale are what reaches memory -- bit for
//    bit what the two steps give, without D's trip through memory.  Every workgroup holds its tile in registers
//    while the maxima meet (slots in the workspace, as in the one-pass in-time cast), so the launch must have all
//    its workgroups on the chip at once: the host only takes this path for at most one tile per CU.
//  * QSPEC: the cast to FP8 rides along on speculation instead, for any number of tiles.  The output is stored in OT as
//    usual and, next to it, the codes of the rounded output times the scale the meta holds before the call; every
//    workgroup folds the maximum of its rounded outputs into one word of the workspace, and the workgroup that
//    finishes last (a ticket counter tells) applies the scale rule, rewrites the meta and leaves a flag that says
//    whether the rule arrived at another scale than the one used.  Only then does the caller's next kernel read the
//    stored output again and cast it with the new scale; otherwise the codes stand, bit for bit what the two steps
//    give, and the stored output is never read back.  No workgroup waits for another.
// QuantArgs (the meta pointers, meeting slots and workspace words of the fused casts) is declared in gemm_call.h

// a * b rounded to OT (as the plain epilogue stores it) and widened again
template <typename OT>
__device__ __forceinline__ void round_pair(float a, float b, float& ra, float& rb) {
    if constexpr (sizeof(OT) == 4) {
        ra = a, rb = b;
    } else if constexpr (__is_same(OT, bf16_t)) {
        const uint32_t p = pack_bf16(a, b);
        ra = __uint_as_float(p << 16), rb = __uint_as_float(p & 0xffff0000u);
    } else {
        const f32x2 v = {a, b};
        const f16x2 h = __builtin_convertvector(v, f16x2);
        ra = static_cast<float>(h[0]), rb = static_cast<float>(h[1]);
    }
}

// element-wise unsigned maximum of two packed 16-bit pairs
__device__ __forceinline__ uint32_t pk_umax16(uint32_t a, uint32_t b) {
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
}

// ---- the accumulators of the DMA kernel live in fixed AGPRs: block (i, j) of the wave's 8 x 8 in a[4n .. 4n+3], n = i * 8 + j.
// The register allocator never sees them.  Left to it, they are renumbered between the K loop, its straight-line tail
// and the epilogue, which costs copies between the MFMAs or spills once all 256 are taken.
#define MSAMP_A10(p) "a" #p "0", "a" #p "1", "a" #p "2", "a" #p "3", "a" #p "4", "a" #p "5", "a" #p "6", "a" #p "7", "a" #p "8", "a" #p "9"
#define MSAMP_ALL_AGPRS                                                                                                \
    "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", MSAMP_A10(1), MSAMP_A10(2), MSAMP_A10(3), MSAMP_A10(4),  \
        MSAMP_A10(5), MSAMP_A10(6), MSAMP_A10(7), MSAMP_A10(8), MSAMP_A10(9), MSAMP_A10(10), MSAMP_A10(11), MSAMP_A10(12), \
        MSAMP_A10(13), MSAMP_A10(14), MSAMP_A10(15), MSAMP_A10(16), MSAMP_A10(17), MSAMP_A10(18), MSAMP_A10(19),          \
        MSAMP_A10(20), MSAMP_A10(21), MSAMP_A10(22), MSAMP_A10(23), MSAMP_A10(24), "a250", "a251", "a252", "a253", "a254", \
        "a255"

// a[4N .. 4N+3] += srcA x srcB.  No clobber list: the compiler follows a clobbered register with a wait state, one per
// MFMA.  It learns of the AGPRs from acc_clear() and acc_fence(), which name them all.
template <int N, int CB, int BL>
__device__ __forceinline__ void mfma_fixed(const v8i& a, const v8i& b) {
    asm volatile("v_mfma_f32_16x16x128_f8f6f4 a[%2:%3], %0, %1, a[%2:%3] cbsz:%4 blgp:%5"
                 :
                 : "v"(a), "v"(b), "n"(N * 4), "n"(N * 4 + 3), "n"(CB), "n"(BL));
}
// A wave's load of 1 KiB, 16 bytes a lane, from `src` (scalar: operand + slice) + `off` (the lane's, 32 bits: no vector instruction is
// spent on addresses) to LDS at `dst`.  Written as assembly so that the compiler does not see an LDS write it cannot tell apart from
// the fragment reads: it would otherwise make every LDS read wait for all loads in flight.  Completion is tracked by hand with
// wait_vmcnt<>() before the barriers of the kernels.
struct LdsLoad {
    uint32_t dst, off;
    const uint8_t* src;
};
// The destination goes through M0, and between its write and the load there has to be another instruction, which the compiler sees to
// only for loads of its own.  In front of the K loop that is an s_nop, in it the MFMA that the load goes with.  us with nothing between
// them | an s_nop | the MFMA: 16384 x 8192 x 28672 row-major 2348 | 2357 | 2340, both K-major 2373 | 2391 | 2358, 16384 x 16384 x 16384 2783 | 2797 |
// 2769; 128 x 128 tiles, 1024 x 1024 x 8192 both K-major 32.1 | 32.2 | 31.4, the others level.
__device__ __forceinline__ void load_to_lds(const LdsLoad& l) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(l.dst), "v"(l.off), "s"(l.src) : "memory", "m0");
}
template <int N, int CB, int BL>
__device__ __forceinline__ void mfma_fixed_and_load(const v8i& a, const v8i& b, const LdsLoad& l) {
    asm volatile("s_mov_b32 m0, %6\n\tv_mfma_f32_16x16x128_f8f6f4 a[%2:%3], %0, %1, a[%2:%3] cbsz:%4 blgp:%5\n\tglobal_load_lds_dwordx4 %7, %8"
                 :
                 : "v"(a), "v"(b), "n"(N * 4), "n"(N * 4 + 3), "n"(CB), "n"(BL), "s"(l.dst), "v"(l.off), "s"(l.src)
                 : "memory", "m0");
}
__device__ __forceinline__ void acc_clear() {
    static_for<64>([&](auto nc) {
        constexpr int n = decltype(nc)::value;
        asm volatile("v_accvgpr_write_b32 a[%0], 0\n\tv_accvgpr_write_b32 a[%1], 0\n\tv_accvgpr_write_b32 a[%2], 0\n\t"
                     "v_accvgpr_write_b32 a[%3], 0"
                     :
                     : "n"(n * 4), "n"(n * 4 + 1), "n"(n * 4 + 2), "n"(n * 4 + 3));
    });
    asm volatile("s_nop 4" : : : MSAMP_ALL_AGPRS);
}
// Fragment registers that vector instructions have just written: an MFMA may read them two wait states later, which the
// compiler cannot know of an MFMA in assembly.
__device__ __forceinline__ void settle16(int* f) {
    asm volatile("s_nop 1"
                 : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4]), "+v"(f[5]), "+v"(f[6]), "+v"(f[7]), "+v"(f[8]), "+v"(f[9]),
                   "+v"(f[10]), "+v"(f[11]), "+v"(f[12]), "+v"(f[13]), "+v"(f[14]), "+v"(f[15]));
}
// 32 fragment registers (four blocks of eight dwords) of the last, ragged K slice: the bytes past its `rem` K bytes become
// zero.  Dword w of a block holds the four K bytes from (lane / 16) * 32 + 4w.
__device__ __forceinline__ void mask_fragments(int* f, int g4, int rem) {
#pragma unroll
    for (int w = 0; w < 8; ++w) {
        const int bytes = rem - (g4 * 32 + w * 4);
        const int m = bytes >= 4 ? -1 : bytes <= 0 ? 0 : (1 << (bytes * 8)) - 1;
#pragma unroll
        for (int b = 0; b < 4; ++b) f[b * 8 + w] &= m;
    }
    settle16(f);
    settle16(f + 16);
}
// After the last MFMA: waits out the MFMA pipe (a 16-pass MFMA's result may be read 18 wait states later) and hands out
// the token that ties the reads below to this point of the program.
__device__ __forceinline__ uint32_t acc_fence() {
    uint32_t token;
    asm volatile("s_nop 15\n\ts_nop 7\n\tv_mov_b32 %0, 0" : "=v"(token) : : MSAMP_ALL_AGPRS);
    return token;
}
__device__ __forceinline__ uint32_t acc_refence(uint32_t token) {
    asm volatile("" : "+v"(token));
    return token;
}
// Not volatile: the compiler may place the read where it likes after the fence that made the token.
template <int N>
__device__ __forceinline__ v4f acc_quad(uint32_t token) {
    v4f r;
    float x, y, z, w;
    asm("v_accvgpr_read_b32 %0, a[%1]" : "=v"(x) : "n"(N * 4), "v"(token));
    asm("v_accvgpr_read_b32 %0, a[%1]" : "=v"(y) : "n"(N * 4 + 1), "v"(token));
    asm("v_accvgpr_read_b32 %0, a[%1]" : "=v"(z) : "n"(N * 4 + 2), "v"(token));
    asm("v_accvgpr_read_b32 %0, a[%1]" : "=v"(w) : "n"(N * 4 + 3), "v"(token));
    r[0] = x, r[1] = y, r[2] = z, r[3] = w;
    return r;
}

// A product in gridDim.y parts of K: this workgroup's part, which is another pointer and another K (the rows of a row-major operand
// stay as far apart as they are).  Its unscaled float32 sum goes to the y-th of gridDim.y arrays of NR x NC; ksplit_finish_kernel adds
// them up.  Every part but the last is whole slices.
// (large tiles; the 128 x 128 tiles take any operands)
template <typename OT, bool XT, bool YT>
constexpr bool kTakesKParts = XT && YT && std::is_same<OT, float>::value;
template <bool XT, bool YT, typename In, typename Out>
__device__ __forceinline__ void k_part(In& X, In& Y, Out& D, int NR, int NC, int& K) {
    if (gridDim.y == 1) return;
    const int nk = (K + kBK - 1) / kBK, parts = gridDim.y, y = blockIdx.y;
    const int first = static_cast<int>(static_cast<long long>(nk) * y / parts) * kBK;
    const int end = y + 1 == parts ? K : static_cast<int>(static_cast<long long>(nk) * (y + 1) / parts) * kBK;
    X += XT ? static_cast<size_t>(first) * kmajor_pitch(NR) : first;
    Y += YT ? static_cast<size_t>(first) * kmajor_pitch(NC) : first;
    D += static_cast<size_t>(y) * NR * NC;
    K = end - first;
}

template <int XF, int YF, typename OT, bool XT = false, bool YT = false, int QF = 0, bool QSPEC = false, bool KTAIL = false>
__global__ __launch_bounds__(kGemmThreads) void fp8_gemm_dma_kernel(const uint8_t* __restrict__ X,
                                                                     const uint8_t* __restrict__ Y, OT* __restrict__ D,
                                                                     int NR, int NC, int K,
                                                                     const float* __restrict__ x_scale_inv,
                                                                     const float* __restrict__ y_scale_inv, int accumulate,
                                                                     const void* __restrict__ bias, int bias_dt,
                                                                     QuantArgs qa) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    if constexpr (KTAIL && kTakesKParts<OT, XT, YT>) k_part<XT, YT>(X, Y, D, NR, NC, K);
    const int tiles_r = (NR + kDmaTile - 1) / kDmaTile, tiles_c = (NC + kDmaTile - 1) / kDmaTile;
    bool by_columns = walk_by_columns(tiles_r, tiles_c, K);
    int tr, tc;
    // Which way round the 32 tiles of an XCD lie.  A K-major operand with a long leading dimension that is a multiple
    // of 4 KiB is hard on that XCD's L2: the 128 k-rows of a tile's 256-byte strip lie a multiple of 4 KiB apart, L2
    // misses double (TCC_MISS, FETCH_SIZE x 2.4 on 8192 x 28672 x 16384 with Y as [K, 28672]) and the CUs that share
    // the strip all wait.  Eight such strips shared by four CUs each then beat four shared by eight: the patch is turned
    // so that this operand gets the eight (that shape: 2.82 -> 3.07 PFLOP/s; with X K-major as well 2.73 -> 3.09;
    // 28672 x 8192 x 16384, both K-major: 2.88 -> 3.02).  Measured only where it is applied: K of 16384 and more, one
    // such operand (with two, or at K = 8192, turning the patch lost 1 to 7 %).
    auto strips = [](int n) { return n % 4096 == 0 && n >= 12288; };
    const bool strips_x = XT && strips(NR), strips_y = YT && strips(NC);
    bool wide = K >= 16384 && strips_x != strips_y && (strips_y ? !by_columns : by_columns);
    // Weight gradients (both operands K-major) over 16384 .. 24576 tokens: the longer operand gets the eight whenever its
    // leading dimension is 10240 or more and a multiple of 256, whichever walk the cache rule above prefers.  Measured
    // at K = 16384 on 41 shapes (long side 5120 .. 28672, short side 4096 / 5120 / 8192, either way round) against
    // the three other walks: 10240 x 8192 +7 %, 8192 x 10240 +11 %, 14336 x 4096 +13 %, 4096 x 14336 +14 %,
    // 8192 x 14336 +11 %, 8192 x 22016 +8 %, 13824 x 4096 +6 %, 11008 x 4096 +3 %, the multiples of 4096 that the rule above already turned
    // unchanged, nothing below -2 % (5120 x 13824); +2 to 5 % at K = 20480, +1 to 3 % at 24576; nothing at K = 12288, and
    // at K = 32768 the turned patch loses 3 to 6 %.
    // Input gradients (only Y K-major) with 12288 or more columns and K of 8192 or more: Y gets the eight, walking
    // groups of tile rows.  Measured on 35 shapes (8192 .. 32768 rows, 12288 .. 28672 columns, K 8192 .. 28672) against
    // the three other walks: up to +9 % (8192 x 14336 x 12288 and x 16384), 16384 x 28672 x 8192 +4 %, nothing below -0.7 %;
    // with 8192 columns (x 28672) it loses 3 %, at K = 4096 nothing moves.
    if (!XT && YT && NC >= 12288 && K >= 8192) by_columns = false, wide = true;
    if (XT && YT && K >= 16384 && K <= 24576 && NR != NC) {
        const bool x_long = NR > NC;
        const int long_n = x_long ? NR : NC, short_n = x_long ? NC : NR;
        if (long_n >= 10240 && long_n % 256 == 0 && short_n <= 8192) by_columns = x_long, wide = true;
    }
    static_assert(!KTAIL || QF == 0, "a ragged last slice: plain and speculative forms only");
    // a walk registered for this problem (timed on this machine) overrides the rules
    if (qa.walk_plus_one > 0) by_columns = (qa.walk_plus_one - 1) & 1, wide = ((qa.walk_plus_one - 1) >> 1) & 1;
    tile_of_id(blockIdx.x, tiles_r, tiles_c, by_columns, wide, tr, tc);
    const int row0 = tr * kDmaTile, col0 = tc * kDmaTile;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wr = wave >> 1, wc = wave & 1;
    // the output factor is fetched now: left to the epilogue, the two scalar loads sit on its critical path
    float alpha_early = (*x_scale_inv) * (*y_scale_inv);
    if constexpr (KTAIL && kTakesKParts<OT, XT, YT>) alpha_early = gridDim.y > 1 ? 1.0f : alpha_early;
    // and so are the bias values of two of this wave's 128 columns per lane (-0 without a bias: fma(x, y, -0) is x * y to
    // the bit, signed zeros included)
    float bias_early[2] = {-0.0f, -0.0f};
    if constexpr (QF == 0 && !QSPEC) {
        if (bias != nullptr) {
            const int c = col0 + wc * 128 + lane * 2;
            bias_early[0] = c < NC ? load_bias(bias, bias_dt, c) : 0.0f;
            bias_early[1] = c + 1 < NC ? load_bias(bias, bias_dt, c + 1) : 0.0f;
        }
        asm volatile("" : "+v"(bias_early[0]), "+v"(bias_early[1]));
    }
    asm volatile("" : "+v"(alpha_early));
    // QSPEC: the scale the codes are written with, as the meta holds it now (the last workgroup rewrites the meta)
    float guess = 1.0f;
    if constexpr (QSPEC) {
        guess = *qa.scale;
        asm volatile("" : "+v"(guess));
    }

    // ---- global -> LDS.  A block of the ring holds 256 X rows or 256 Y rows, 128 bytes per row.  One wave
    // instruction fills 8 rows (1 KiB, lane-contiguous): lane l lands in row l/8, 16-byte position l%8,
    // and therefore fetches the logical chunk position ^ swizzle(row).  Rows past the end of the matrix
    // are clamped to its last row (their results are never stored).
    const int chunk = (lane & 7) ^ (lane >> 3) ^ (wave & 1);
    const uint32_t lds_base = __builtin_amdgcn_readfirstlane(
        static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)smem)));
    // K-major operand: one wave instruction fills 4 k-rows of 256 bytes; lane l lands in k-row l/16,
    // position l%16, and fetches the logical chunk position ^ (k-row % 8)
    const int chunk_t = (lane & 15) ^ ((wave & 1) * 4 + (lane >> 4));
    // K-major operand, last tile: 16-byte chunks past the end of a k-row are fetched from the tile's first chunk instead
    // (rows of D that do not exist; a k-row's pitch is a multiple of 16, so a chunk is inside it or not as a whole)
    const int xcol = row0 + chunk_t * 16 < NR ? row0 + chunk_t * 16 : row0;
    const int ycol = col0 + chunk_t * 16 < NC ? col0 + chunk_t * 16 : col0;
    const int ldx = kmajor_pitch(NR), ldy = kmajor_pitch(NC);
    uint32_t xoff[8], yoff[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int r = (i * 4 + wave) * 8 + (lane >> 3);
        int gx = row0 + r, gy = col0 + r;
        gx = gx < NR ? gx : NR - 1;
        gy = gy < NC ? gy : NC - 1;
        const int krow = (i * 4 + wave) * 4 + (lane >> 4);
        xoff[i] = XT ? static_cast<uint32_t>(krow) * static_cast<uint32_t>(ldx) + xcol
                     : static_cast<uint32_t>(gx) * static_cast<uint32_t>(K) + chunk * 16;
        yoff[i] = YT ? static_cast<uint32_t>(krow) * static_cast<uint32_t>(ldy) + ycol
                     : static_cast<uint32_t>(gy) * static_cast<uint32_t>(K) + chunk * 16;
    }
    // KTAIL: K is no multiple of 128 and the last slice holds `rem` bytes of K only.  Its loads stay inside the operand (a
    // lane whose chunk or k-row lies past the end fetches the slice's first one instead) and its fragments are masked
    // byte by byte between LDS and MFMA, in both operands (what lies past the end may hold NaN codes): zeros, as
    // the generic kernel has them there, and the same bits out.  The last slice is straight-line code at the end, so
    // the K loop is the one of the plain form.
    const int nk = KTAIL ? (K + kBK - 1) / kBK : K / kBK;
    const int rem = K - (nk - 1) * kBK;
    const uint32_t tail_back = KTAIL && chunk * 16 >= rem ? chunk * 16 : 0;
    // The ring: X and Y of a slice side by side, slice after slice.  Where the block lies that is that many on from the one at s0.
    // (s0, X of the present slice, is handed around as a value: captured by reference it ended up in scratch memory in some forms.)
    constexpr int kX = 0, kY = 1, kPerSlice = 2;
    auto place = [](int s0, int blocks_on) __attribute__((always_inline)) {
        const int p = s0 + blocks_on % kDmaBlocks * kDmaBlock;
        return p >= kDmaBlocks * kDmaBlock ? p - kDmaBlocks * kDmaBlock : p;
    };
    // one of this wave's eight loads for a block of slice kt, which is `ahead` slices on from the present one
    auto load_of = [&](int s0, int block, int kt, int ahead, int w, bool last) __attribute__((always_inline)) {
        const bool is_x = block == kX;
        const size_t slice = static_cast<size_t>(kt) * kBK;
        const uint8_t* src = is_x ? X + (XT ? slice * ldx : slice) : Y + (YT ? slice * ldy : slice);
        uint32_t off = is_x ? xoff[w] : yoff[w];
        if (KTAIL && last) {
            if (is_x ? XT : YT) {
                if ((w * 4 + wave) * 4 + (lane >> 4) >= rem) off = is_x ? xcol : ycol;
            } else {
                off -= tail_back;
            }
        }
        // (wave-uniform by construction; the readfirstlane keeps it in a scalar register whatever the compiler makes of it)
        const uint32_t dst = __builtin_amdgcn_readfirstlane(lds_base + place(s0, ahead * kPerSlice + block) + (w * 4 + wave) * 1024);
        return LdsLoad{dst, off, src};
    };

    // ---- LDS -> fragments of the 16x16x128 MFMA: a lane holds, for row lane % 16 of a 16-row block, the 32 K-bytes
    // (lane / 16) * 32 .. + 31 of the 128-byte slice.  Row-major operand: two 16-byte reads at the swizzled chunks
    // 2 * (lane / 16) and + 1.  K-major operand: four transposing reads, each handing a 16-lane group eight
    // consecutive k of 16 rows.
    const int fsw = (lane & 7) ^ ((lane >> 3) & 1);
    const int l16 = lane & 15, g4 = lane >> 4;
    const int off_lo = ((2 * g4) ^ fsw) << 4;    // low 16 bytes of this lane's 32; the high ones are at ^ 16
    const int tj = l16 >> 1;
    const int t_lane = (g4 * 32 + tj) * 256 + (l16 & 1) * 8;    // k-row and 8-byte half of this lane's address
    // this lane's first read of half 0 in a block; the 16-row blocks of a row-major operand follow 2 KiB apart, of a K-major one
    // at ^ 16 (its half 1 at ^ 64)
    const int xlane = XT ? t_lane + wr * 128 + (tj << 4) : (wr * 128 + l16) * kBK + off_lo;
    const int ylane = YT ? t_lane + wc * 128 + (tj << 4) : (wc * 128 + l16) * kBK + off_lo;
    // The wave's 128 x 128 quadrant is 8 x 8 blocks of 16 x 16.  Fragments are kept by halves: fx[h] / fy[h] hold the
    // four 16-row blocks 4h .. 4h+3 of X / Y (8 registers each).  A half arrives in pieces: two 16-byte reads per
    // block of a row-major operand, four 8-byte transposing reads otherwise.
    constexpr int kPX = XT ? 16 : 8, kPY = YT ? 16 : 8;
    auto read_piece = [&](int* dst, int at, bool is_x, int half, int p) __attribute__((always_inline)) {
        if ((is_x && !XT) || (!is_x && !YT)) {
            const int b = p >> 1, hf = p & 1;
            const v4i val = *reinterpret_cast<const v4i*>(smem + (at ^ (hf * 16)) + (half * 4 + b) * 16 * kBK);
            int* d = dst + b * 8 + hf * 4;
            d[0] = val[0], d[1] = val[1], d[2] = val[2], d[3] = val[3];
        } else {
            const int b = p >> 2, qq = p & 3;
            const v2i val = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                (__attribute__((address_space(3))) v2i*)(smem + (at ^ ((half * 4 + b) * 16)) + qq * 8 * 256));
            int* d = dst + b * 8 + qq * 2;
            d[0] = val[0], d[1] = val[1];
        }
    };

    // accumulator block (i, j): D rows i * 16 + lane % 16, D columns j * 16 + (lane / 16) * 4 .. + 3 of the quadrant
    acc_clear();

    int fx[2][32], fy[2][32];

    // One quarter of a slice: the 16 MFMAs of X half hx against Y half hy, with the reads of a fragment half (X or Y half rd_half out
    // of the block that many on, into rd_dst, if do_read) spread between them, and four loads of slice ld_kt (X, then Y; if do_load),
    // one every four MFMAs.  With VM >= 0 the waves meet after the second MFMA (by then the fragments read last have come back): what
    // the quarters before have read nobody needs in the LDS any more, and all but the last VM loads of each wave have landed.
    // srcA = Y rows (columns of D), srcB = X rows (rows of D): a lane then holds, for D row lane % 16 of a block, four
    // consecutive D columns -- the layout the epilogue wants.
    auto quarter = [&](auto hxc, auto hyc, auto vmc, int s0, int* rd_dst, bool rd_x, int rd_lane, int rd_blocks_on, int rd_half, bool do_read,
                       int ld_kt, int ld_block, int ld_first, bool do_load, bool ld_last) __attribute__((always_inline)) {
        constexpr int cb = (YF == MSAMP_DT_E4M3) ? 0 : 1;
        constexpr int bl = (XF == MSAMP_DT_E4M3) ? 0 : 1;
        const int np = rd_x ? kPX : kPY;
        constexpr int hx = decltype(hxc)::value, hy = decltype(hyc)::value, vm = decltype(vmc)::value;
        int block = place(s0, rd_blocks_on);
        asm volatile("" : "+s"(block));
        const int at = rd_lane + block;
        static_for<4>([&](auto jc) {    // the Y fragment stays for four MFMAs in a row
            static_for<4>([&](auto ic) {
                constexpr int i = decltype(ic)::value, j = decltype(jc)::value;
                constexpr int n = j * 4 + i;
                const int* cx = fx[hx] + i * 8;
                const int* cy = fy[hy] + j * 8;
                const v8i vx = {cx[0], cx[1], cx[2], cx[3], cx[4], cx[5], cx[6], cx[7]};
                const v8i vy = {cy[0], cy[1], cy[2], cy[3], cy[4], cy[5], cy[6], cy[7]};
                if (do_load && (n & 3) == 3)
                    mfma_fixed_and_load<(hx * 4 + i) * 8 + hy * 4 + j, cb, bl>(vy, vx, load_of(s0, ld_block, ld_kt, 2, ld_first + (n >> 2), ld_last));
                else
                    mfma_fixed<(hx * 4 + i) * 8 + hy * 4 + j, cb, bl>(vy, vx);
                if constexpr (vm >= 0 && n == 1) {
                    wait_vmcnt<(vm < 0 ? 0 : vm)>();
                    __syncthreads();
                }
                if (do_read && n >= 2 && n < 14) {
#pragma unroll
                    for (int p = (n - 2) * np / 12; p < (n - 1) * np / 12; ++p) read_piece(rd_dst, at, rd_x, rd_half, p);
                }
                // Nothing moves across: one MFMA, with it the load and then the reads that go with it, so that the LDS reads and
                // the tile loads stay spread evenly between the MFMAs as written.
                __builtin_amdgcn_sched_barrier(0);
            });
        });
    };
    // A step: slice kt, whose X half 0 and Y half 0 are in registers and whose blocks are in the ring, with those of slice kt + 1
    // there or on their way and the place of X of slice kt + 2 free.  X0 x Y0 while Y half 1 is read, X0 x Y1 while X half 1 is -- all
    // of slice kt is in registers now -- X1 x Y0 while X half 0 of slice kt + 1 is and X1 x Y1 while its Y half 0 is.  X of slice kt + 2 is
    // sent for in the first two quarters; the waves meet in the third (slice kt + 1 has landed, and the eight loads of that X may
    // still be on their way; nobody needs the LDS copy of slice kt); Y of slice kt + 2 follows in the place of X of slice kt.  So
    // a load has three quarters of a step to one and a half to land, and one goes out every four MFMAs.
    // What bounds the loop is the way of its loads.  With two stages of a slice each all sixteen went out in the second half of a
    // step, one every other MFMA, to land by the middle of the next: too late wherever they missed the L2.  us in a loop / each among
    // other kernels, two stages -> ring, bfloat16:
    //   row-major      8192 x 2048 x 8192  100 / 109 -> 97 / 101   8192 x 4096 x 4096  103 / 114 -> 103 / 107   8192 x 8192 x 2048  114 / 121 -> 113 / 117
    //                  12605 x 4304 x 1200  96 / 103 -> 92 / 98    16384 x 11008 x 4096  564 / 567 -> 544 / 541  16384 x 4096 x 11008  528 / 528 -> 495 / 487
    //   Y K-major      8192 x 2048 x 8192  99 / 105 -> 96 / 99     16384 x 4096 x 11008  541 / 538 -> 497 / 489  16384 x 28672 x 8192  2662 / 2658 -> 2600 / 2595
    //   both           2048 x 8192 x 8192  95 / 105 -> 92 / 94     11008 x 4096 x 16384  519 / 521 -> 493 / 498  8192 x 28672 x 16384  2602 / 2595 -> 2426 / 2425
    //   level          8192 x 8192 x 512  51 / 54 -> 50 / 56       4096 x 4096 x 8192, both  91 / 103 -> 91 / 94   8192 x 8192 x 4096, both  190 / 208 -> 192 / 194
    // (Row-major with K of 12288 and more had a form of its own before, its loads in the order of need over a whole step and two meetings
    // in it.  16384 x 8192 x K with that form | here: K = 12288 1007 / 1011 | 1005 / 1004, 16384 1335 / 1329 | 1330 / 1321, 20480 1660 / 1657 |
    // 1659 / 1652, 28672 2349 / 2345 | 2346 / 2344.  Four slices behind kernels that have passed other data
    // through the caches: with the two stages | here 8192 x 8192 x 512 50 | 49, 4096 x 8192 x 512 29 | 28; on one card of four either form varied, by
    // a quarter, and this one was more often at the slow end, 49 to 64 and 28 to 36, medians 52 | 61 and 29 to 35 | 35.)
    // (The ring in units of 16 KiB with two meetings a step, every load two steps to land, was no faster, and slower with both K-major, whose k-rows it took in pieces of 128 bytes: 8192 x 28672 x 16384 2500.)
    // `to_go`: slices behind this one, 2 standing for two or more; the last two load nothing.  KTAIL: `last`, the slice that this step
    // loads is the last one.
    auto step = [&](auto to_go_c, int s0, int kt, bool last) __attribute__((always_inline)) {
        constexpr std::integral_constant<int, 0> c0{};
        constexpr std::integral_constant<int, 1> c1{};
        constexpr std::integral_constant<int, -1> none{};
        constexpr int to_go = decltype(to_go_c)::value;
        constexpr bool masked = KTAIL && to_go == 0, loads = to_go >= 2, next = to_go >= 1;
        constexpr std::integral_constant<int, loads ? 8 : 0> meet{};
        if (masked) mask_fragments(fx[0], g4, rem), mask_fragments(fy[0], g4, rem);
        quarter(c0, c0, none, s0, fy[1], false, ylane, kY, 1, true, kt + 2, kX, 0, loads, last);
        if (masked) mask_fragments(fy[1], g4, rem);
        quarter(c0, c1, none, s0, fx[1], true, xlane, kX, 1, true, kt + 2, kX, 4, loads, last);
        if (masked) mask_fragments(fx[1], g4, rem);
        quarter(c1, c0, meet, s0, fx[0], true, xlane, kPerSlice + kX, 0, next, kt + 2, kY, 0, loads, last);
        quarter(c1, c1, none, s0, fy[0], false, ylane, kPerSlice + kY, 0, next, kt + 2, kY, 4, loads, last);
        return place(s0, kPerSlice);
    };

    // prologue: slices 0 and 1 (the host sends no problem with fewer than two slices here); wait for slice 0; read
    // its first fragment halves
#pragma unroll
    for (int w = 0; w < 16; ++w) load_to_lds(load_of(0, w < 8 ? kX : kY, 0, 0, w & 7, false));
#pragma unroll
    for (int w = 0; w < 16; ++w) load_to_lds(load_of(0, w < 8 ? kX : kY, 1, 1, w & 7, nk == 2));
    wait_vmcnt<16>();
    __syncthreads();
#pragma unroll
    for (int p = 0; p < kPX; ++p) read_piece(fx[0], xlane + place(0, kX), true, 0, p);
#pragma unroll
    for (int p = 0; p < kPY; ++p) read_piece(fy[0], ylane + place(0, kY), false, 0, p);
    // The last two steps follow the loop as straight-line code (KTAIL: the last three, so that the loop loads whole slices only): they
    // load nothing and the last one reads no fragments for a successor, which the compiler then knows.
    constexpr std::integral_constant<int, 2> go2{};
    constexpr std::integral_constant<int, 1> go1{};
    constexpr std::integral_constant<int, 0> go0{};
    int kt = 0, s0 = 0;
    for (; kt + (KTAIL ? 3 : 2) < nk; ++kt) s0 = step(go2, s0, kt, false);
    if (KTAIL && kt + 3 == nk) s0 = step(go2, s0, kt, true), ++kt;
    s0 = step(go1, s0, kt, false);
    step(go0, s0, kt + 1, false);
    // The workgroup that follows this one on the CU is, as a rule, the one 256 ids on (same XCD).  Touch the first two K
    // slices of its tile now -- one 4-byte load per 128-byte line, dropped into an LDS corner that nothing reads -- so that
    // its prologue finds them in this XCD's L2 instead of waiting for HBM with the MFMA pipe idle.  The loads have no
    // register destination, so nothing has to wait for them; the hardware drains them before the wave ends.
    {
        const int nid = blockIdx.x + 256;
        if (nid < tiles_r * tiles_c) {
            int ntr, ntc;
            tile_of_id(nid, tiles_r, tiles_c, by_columns, wide, ntr, ntc);
            const int nr0 = ntr * kDmaTile, nc0 = ntc * kDmaTile;
            // line L of an operand's 512: row-major, half L % 2 of row L / 2; K-major, half L % 2 of the tile's 256 bytes in
            // k-row L / 2; clamped like the tile loads (K > 128 here)
            auto line = [&](int L, bool is_x) __attribute__((always_inline)) -> const uint8_t* {
                const int r = L >> 1, hf = (L & 1) * 128;
                const uint8_t* base = is_x ? X : Y;
                const int n = is_x ? NR : NC, first = is_x ? nr0 : nc0;
                if (is_x ? XT : YT)
                    return base + static_cast<size_t>(!KTAIL || r < K ? r : K - 1) * (is_x ? ldx : ldy) + (first + hf < n ? first + hf : first);
                const int row = first + r < n ? first + r : n - 1;
                return base + static_cast<size_t>(row) * K + hf;
            };
            const int t = threadIdx.x;
            const uint32_t dump = __builtin_amdgcn_readfirstlane(lds_base + kDmaBlocks * kDmaBlock - 256);
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off\n\tglobal_load_lds_dword %2, off\n\t"
                         "global_load_lds_dword %3, off\n\tglobal_load_lds_dword %4, off"
                         : : "s"(dump), "v"(line(t, true)), "v"(line(t + 256, true)), "v"(line(t, false)), "v"(line(t + 256, false))
                         : "memory", "m0");
        }
    }
    const uint32_t acc_token = acc_fence();
    // No barrier here: the last LDS reads of every wave were issued (and awaited) before the barrier of the last
    // slice, and no load is in flight but the touches, so each wave may start on its patch as soon as its own MFMAs are done.
    uint32_t* const red = reinterpret_cast<uint32_t*>(smem + kDmaBlocks * kDmaBlock - 512);    // a few words behind all patches

    // The epilogues below handle the quadrant in four units of 32 rows (two 16-row blocks): unit u, half h, column
    // block j -> acc[2u + h][j], patch row h * 16 + lane % 16, patch columns j * 16 + (lane / 16) * 4 .. + 3.
    if constexpr (QF != 0) {
        // ---- fused in-time cast (whole tiles only, no bias, no accumulation: the host sees to that)
        uint32_t* const q_red = red;
        uint32_t &q_scale = red[kGemmThreads / kWave], &q_amax = red[kGemmThreads / kWave + 1];
        const float alpha = alpha_early;
        // max |acc| as an ordered bit pattern: NaN above Inf above everything finite, so a NaN reaches the amax
        // as it does through abs().max()
        uint32_t m = 0;
        static_for<64>([&](auto nc) {
            const v4f a = acc_quad<decltype(nc)::value>(acc_token);
#pragma unroll
            for (int r = 0; r < 4; ++r) m = umax(m, __float_as_uint(a[r]) & 0x7fffffffu);
        });
        m = block_max_u32(m, q_red);    // valid in lane 0 of wave 0
        const int tid = threadIdx.x;
        if (tid == 0) {
            // Scaling by |alpha| and rounding to OT never reorder magnitudes, so the maximum of the rounded outputs
            // is the rounded, scaled maximum.
            float am, unused;
            round_pair<OT>(__uint_as_float(m) * fabsf(alpha), 0.0f, am, unused);
            m = __float_as_uint(am) & 0x7fffffffu;
            __hip_atomic_store(qa.slots + blockIdx.x, (static_cast<uint64_t>(qa.token) << 32) | m, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        }
        // Workgroup 0 collects the slots (its first wave), derives amax and scale and posts
        // both, tagged with the token, in the two words behind the slots; the other workgroups poll only those.
        // Every wait is bounded.  Workgroup 0 posts even when it gives up (NaN amax, old scale), and the others wait
        // longer for the post than it waits for them; whoever gives up sets the sticky error word of the workspace.
        uint64_t* post = qa.slots + kMaxSlots;
        if (blockIdx.x == 0) {
            if (tid < kWave) {
                uint32_t mm = 0;
                bool all_in = false;
                for (uint32_t spins = 0; !all_in && spins < qa.spin_limit; ++spins) {
                    uint64_t sv[kMaxSlots / kWave];
#pragma unroll
                    for (int j = 0; j < kMaxSlots / kWave; ++j)
                        sv[j] = __hip_atomic_load(qa.slots + tid + j * kWave, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    bool ok = true;
                    mm = 0;
#pragma unroll
                    for (int j = 0; j < kMaxSlots / kWave; ++j) {
                        const bool live = static_cast<uint32_t>(tid + j * kWave) < gridDim.x;
                        ok = ok && (!live || static_cast<uint32_t>(sv[j] >> 32) == qa.token);
                        mm = umax(mm, live ? static_cast<uint32_t>(sv[j]) : 0u);
                    }
                    all_in = __all(ok);
                }
                mm = wave_max_u32(mm);
                if (tid == 0) {
                    float am = __uint_as_float(mm);
                    if (!all_in) {    // gave up: NaN amax, old scale, both still posted, sticky error word set
                        am = __uint_as_float(0x7fc00000u);
                        report_wait_expired(qa.error_word, kErrCollectorGaveUp);
                    } else if ((qa.flags & MSAMP_FLAG_NAN_TO_INF) && !(am < __uint_as_float(0x7f800000u))) {
                        am = __uint_as_float(0x7f800000u);
                    }
                    const float sc = scale_rule(am, *qa.scale, qa.fp_max, qa.margin);
                    const uint64_t tag = static_cast<uint64_t>(qa.token) << 32;
                    __hip_atomic_store(post, tag | __float_as_uint(am), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    __hip_atomic_store(post + 1, tag | __float_as_uint(sc), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    q_scale = __float_as_uint(sc);
                    q_amax = __float_as_uint(am);
                    *qa.amax = am;
                    *qa.scale = sc;
                    *qa.scale_inv = 1.0f / sc;
                }
            }
        } else {
            if (tid == 0) {
                uint64_t pa = 0, ps = 0;
                bool posted = false;
                const uint64_t follower_limit = static_cast<uint64_t>(qa.spin_limit) * kFollowerSpinFactor;
                for (uint64_t spins = 0; !posted && spins < follower_limit; ++spins) {
                    pa = __hip_atomic_load(post, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    ps = __hip_atomic_load(post + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    posted = static_cast<uint32_t>(pa >> 32) == qa.token && static_cast<uint32_t>(ps >> 32) == qa.token;
                }
                if (!posted) report_wait_expired(qa.error_word, kErrFollowerGaveUp);
                q_amax = posted ? static_cast<uint32_t>(pa) : 0x7fc00000u;
                q_scale = posted ? static_cast<uint32_t>(ps) : 0x7fc00000u;
            }
        }
        __syncthreads();    // also: every wave is through with the ring, which the patches below reuse
        const float sc = __uint_as_float(q_scale);
        const uint32_t acc_token2 = acc_refence(acc_token);    // a second round of reads, not the first one kept alive
        // with a positive finite amax and the scale derived from it nothing leaves the format and nothing is NaN:
        // the clamp and the NaN patch of the general conversion can go
        const bool in_range = __uint_as_float(q_amax) * sc <= qa.fp_max && __uint_as_float(q_amax) > 0.0f;
        constexpr int kQPitch = 128 + 16;    // bytes per patch row: 128 codes and padding that staggers the banks
        uint8_t* qpatch = smem + wave * (32 * kQPitch);
        auto emit = [&](auto checked) {
            constexpr bool kChecked = decltype(checked)::value;
            static_for<4>([&](auto uc) {
                constexpr int u = decltype(uc)::value;
                static_for<2>([&](auto hc) {
                    constexpr int h = decltype(hc)::value;
                    static_for<8>([&](auto jc) {
                        constexpr int j = decltype(jc)::value;
                        // the outputs as OT would hold them, then scaled
                        const v4f a = acc_quad<(2 * u + h) * 8 + j>(acc_token2);
                        float r0, r1, r2, r3;
                        round_pair<OT>(a[0] * alpha, a[1] * alpha, r0, r1);
                        round_pair<OT>(a[2] * alpha, a[3] * alpha, r2, r3);
                        uint32_t w;
                        if constexpr (kChecked) w = quant4<QF>(r0 * sc, r1 * sc, r2 * sc, r3 * sc);
                        else w = quant4_in_range<QF>(r0 * sc, r1 * sc, r2 * sc, r3 * sc);
                        *reinterpret_cast<uint32_t*>(qpatch + (h * 16 + l16) * kQPitch + j * 16 + g4 * 4) = w;
                    });
                });
                // the patch is private to this wave and the LDS serves one wave's requests in order: no waits here
                auto rd = [&](int t) {
                    return *reinterpret_cast<const uint4*>(qpatch + (t * 8 + (lane >> 3)) * kQPitch + (lane & 7) * 16);
                };
                const uint4 val0 = rd(0), val1 = rd(1), val2 = rd(2), val3 = rd(3);
                auto st = [&](int t, const uint4& v) {
                    const int grow = row0 + wr * 128 + u * 32 + t * 8 + (lane >> 3);
                    const int gcol = col0 + wc * 128 + (lane & 7) * 16;
                    store_out16(qa.q + static_cast<size_t>(grow) * NC + gcol, v);
                };
                st(0, val0), st(1, val1), st(2, val2), st(3, val3);
            });
        };
        if (in_range) emit(std::false_type{}); else emit(std::true_type{});
        return;
    }

    // ---- epilogue: per 32-row unit, accumulators -> this wave's LDS patch -> 16-byte row stores
    constexpr int kEsz = static_cast<int>(sizeof(OT));
    constexpr int kPitch = 128 * kEsz + 16;    // bytes per patch row (padding staggers the banks)
    uint8_t* patch = smem + wave * (32 * kPitch);
    const float alpha = alpha_early;
    const bool vec_ok = (NC % (16 / kEsz) == 0) && ((reinterpret_cast<uintptr_t>(D) & 15) == 0);
    const bool pairs_ok = (NC % 2 == 0) && ((reinterpret_cast<uintptr_t>(D) & 3) == 0);
    constexpr int kChunksPerRow = 128 * kEsz / 16;      // 16 (2-byte) or 32 (float)
    constexpr int kRowsPerPass = 64 / kChunksPerRow;    // 4 or 2
    constexpr int kElemsPerChunk = 16 / kEsz;           // 8 or 4
    // QSPEC: the codes of a unit leave through a second per-wave patch, behind the room of the four largest (float32)
    // output patches; spec_max is the running maximum of the rounded outputs' magnitudes, as float32 bit patterns or
    // as two packed 16-bit patterns (NaN patterns compare above Inf, so a NaN reaches the amax as through abs().max())
    constexpr int kCPitch = 128 + 16;
    uint8_t* cpatch = smem + 4 * (32 * (128 * 4 + 16)) + wave * (32 * kCPitch);
    uint32_t spec_max = 0;
    // the values a packed pair of 16-bit outputs stands for
    auto widen_pair = [&](uint32_t pk, float& lo, float& hi) __attribute__((always_inline)) {
        if constexpr (__is_same(OT, bf16_t)) {
            lo = __uint_as_float(pk << 16), hi = __uint_as_float(pk & 0xffff0000u);
        } else {
            lo = f16_bits_to_float(pk & 0xffffu), hi = f16_bits_to_float(pk >> 16);
        }
    };
    auto emit_fused_rows = [&]() __attribute__((always_inline)) {
        // ---- accumulation (and bias) with 16-byte row accesses: the raw float32 accumulators of a 32-row unit go
        // through a per-wave float32 patch, each lane picks up one 16-byte segment of an output row, reads the old
        // output there if it is to be added, and stores fma(acc, alpha, bias) (+ old) rounded once -- the expression of
        // the element-wise path below and of the generic kernel.  A lane's columns are the same in every pass, so
        // its bias values are fetched once.
        constexpr int kFPitch = 128 * 4 + 16;    // bytes per float32 patch row
        uint8_t* fpatch = smem + wave * (32 * kFPitch);
        const int pc = lane % kChunksPerRow, prl = lane / kChunksPerRow;
        const int gcol = col0 + wc * 128 + pc * kElemsPerChunk;
        const bool col_ok = gcol < NC;
        float bv[kElemsPerChunk];
#pragma unroll
        for (int e = 0; e < kElemsPerChunk; ++e) bv[e] = (bias != nullptr && col_ok) ? load_bias(bias, bias_dt, gcol + e) : 0.0f;
        constexpr int kPasses = 32 / kRowsPerPass;    // 8 or 16
        constexpr int kGroup = 4;                     // passes whose old outputs are in flight together
        static_for<4>([&](auto uc) {
            constexpr int u = decltype(uc)::value;
            static_for<2>([&](auto hc) {
                constexpr int h = decltype(hc)::value;
                static_for<8>([&](auto jc) {
                    constexpr int j = decltype(jc)::value;
                    const v4f a = acc_quad<(2 * u + h) * 8 + j>(acc_token);
                    *reinterpret_cast<float4*>(fpatch + (h * 16 + l16) * kFPitch + (j * 16 + g4 * 4) * 4) =
                        make_float4(a[0], a[1], a[2], a[3]);
                });
            });
            // the patch is private to this wave and the LDS serves one wave's requests in order: no waits needed
            static_for<kPasses / kGroup>([&](auto gc) {
                constexpr int p0 = decltype(gc)::value * kGroup;
                uint4 old[kGroup];
                bool ok[kGroup];
#pragma unroll
                for (int t = 0; t < kGroup; ++t) {
                    const int grow = row0 + wr * 128 + u * 32 + (p0 + t) * kRowsPerPass + prl;
                    ok[t] = col_ok && grow < NR;
                    old[t] = make_uint4(0, 0, 0, 0);
                    if (accumulate && ok[t]) old[t] = load_out16(D + static_cast<size_t>(grow) * NC + gcol);
                }
#pragma unroll
                for (int t = 0; t < kGroup; ++t) {
                    const int pr = (p0 + t) * kRowsPerPass + prl;
                    const int grow = row0 + wr * 128 + u * 32 + pr;
                    const float* src = reinterpret_cast<const float*>(fpatch + pr * kFPitch + pc * kElemsPerChunk * 4);
                    float r[kElemsPerChunk], o[kElemsPerChunk];
                    const float4 a0 = *reinterpret_cast<const float4*>(src);
                    r[0] = a0.x, r[1] = a0.y, r[2] = a0.z, r[3] = a0.w;
                    if constexpr (kElemsPerChunk == 8) {
                        const float4 a1 = *reinterpret_cast<const float4*>(src + 4);
                        r[4] = a1.x, r[5] = a1.y, r[6] = a1.z, r[7] = a1.w;
                    }
                    if constexpr (kEsz == 4) {
                        o[0] = __uint_as_float(old[t].x), o[1] = __uint_as_float(old[t].y);
                        o[2] = __uint_as_float(old[t].z), o[3] = __uint_as_float(old[t].w);
                    } else {
                        In16<OT>::decode(old[t], o);
                    }
#pragma unroll
                    for (int e = 0; e < kElemsPerChunk; ++e) {
                        r[e] = fmaf(r[e], alpha, bv[e]);
                        if (accumulate) r[e] += o[e];
                    }
                    uint4 v;
                    if constexpr (kEsz == 4) {
                        v = make_uint4(__float_as_uint(r[0]), __float_as_uint(r[1]), __float_as_uint(r[2]), __float_as_uint(r[3]));
                    } else if constexpr (__is_same(OT, bf16_t)) {
                        v = make_uint4(pack_bf16(r[0], r[1]), pack_bf16(r[2], r[3]), pack_bf16(r[4], r[5]), pack_bf16(r[6], r[7]));
                    } else {
                        v = make_uint4(pack_f16(r[0], r[1]), pack_f16(r[2], r[3]), pack_f16(r[4], r[5]), pack_f16(r[6], r[7]));
                    }
                    if (ok[t]) store_out16(D + static_cast<size_t>(grow) * NC + gcol, v);
                    if constexpr (QSPEC) {
                        // the codes of the eight (four) outputs just rounded: 8 (4) bytes of a row of q per lane
                        float rr[kElemsPerChunk];
                        if constexpr (kEsz == 4) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) rr[e] = r[e], spec_max = umax(spec_max, __float_as_uint(r[e]) & 0x7fffffffu);
                        } else {
                            const uint32_t pk[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                spec_max = pk_umax16(spec_max, pk[e] & 0x7fff7fffu);
                                widen_pair(pk[e], rr[2 * e], rr[2 * e + 1]);
                            }
                        }
                        uint8_t* qo = qa.q + static_cast<size_t>(grow) * NC + gcol;
                        const uint32_t c0 = quant4_in_range<MSAMP_DT_E4M3>(rr[0] * guess, rr[1] * guess, rr[2] * guess, rr[3] * guess);
                        if constexpr (kEsz == 4) {
                            if (ok[t]) __builtin_nontemporal_store(c0, reinterpret_cast<uint32_t*>(qo));
                        } else {
                            const uint32_t c1 = quant4_in_range<MSAMP_DT_E4M3>(rr[4] * guess, rr[5] * guess, rr[6] * guess, rr[7] * guess);
                            typedef uint32_t v2u_t __attribute__((ext_vector_type(2)));
                            const v2u_t cc = {c0, c1};
                            if (ok[t]) __builtin_nontemporal_store(cc, reinterpret_cast<v2u_t*>(qo));
                        }
                    }
                }
            });
        });
    };
    if (!QSPEC && accumulate && vec_ok) {
        emit_fused_rows();
        return;
    }
    if (!QSPEC && accumulate) {
        static_for<8>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            static_for<8>([&](auto jc) {
                constexpr int j = decltype(jc)::value;
                const v4f a = acc_quad<i * 8 + j>(acc_token);
                store_quad_slow<OT>(D, row0 + wr * 128 + i * 16 + l16, col0 + wc * 128 + j * 16 + g4 * 4, NR, NC, alpha, a[0], a[1],
                                    a[2], a[3], accumulate, bias, bias_dt);
            });
        });
        return;
    }
    // Three copies of the plain epilogue, chosen once per workgroup so that the one that runs is straight-line code:
    // whole tile with 16-byte row stores (no bounds checks; the address is a scalar row base plus one per-lane offset),
    // 16-byte row stores with bounds checks (tiles on the right or bottom edge), and rows that 16-byte stores do not fit.
    // (With the choice made per store, every store dragged three variants and their branches along.)
    // A bias is added here as well, as fma(acc, alpha, bias): a lane's accumulators lie in 32 columns, whose values it
    // takes from the wave's patch, where the lanes put the two each of them fetched at the start.  (Through the float32
    // patch of the accumulating form, with the bias fetched after the K loop, a tile took about 8 us longer: 8192 x 8192
    // x 2048 with a bias 142 us, now 114; 12605 x 4304 x 1200 into float16 116 us, now 93.)
    auto emit_plain = [&](auto vec_c, auto inside_c) __attribute__((always_inline)) {
        constexpr bool kVec = decltype(vec_c)::value, kInside = decltype(inside_c)::value;
        const int pc = lane % kChunksPerRow, prl = lane / kChunksPerRow;
        const int gcol = col0 + wc * 128 + pc * kElemsPerChunk;
        // whole tile: byte offset of this lane's segment from the first element of its pass's first row
        const uint32_t lane_off = (static_cast<uint32_t>(prl) * static_cast<uint32_t>(NC) + static_cast<uint32_t>(pc * kElemsPerChunk)) * kEsz;
        float bq[32];
        if constexpr (!QSPEC) {
            *reinterpret_cast<uint2*>(patch + lane * 8) = make_uint2(__float_as_uint(bias_early[0]), __float_as_uint(bias_early[1]));
            asm volatile("" : : : "memory");
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const uint4 b = *reinterpret_cast<const uint4*>(patch + (j * 16 + g4 * 4) * 4);
                bq[4 * j] = __uint_as_float(b.x), bq[4 * j + 1] = __uint_as_float(b.y);
                bq[4 * j + 2] = __uint_as_float(b.z), bq[4 * j + 3] = __uint_as_float(b.w);
            }
            asm volatile("" : : : "memory");
        }
        auto scaled = [&](float x, int c) __attribute__((always_inline)) { return QSPEC ? x * alpha : fmaf(x, alpha, bq[c]); };
        static_for<4>([&](auto uc) {
            constexpr int u = decltype(uc)::value;
            static_for<2>([&](auto hc) {
                constexpr int h = decltype(hc)::value;
                static_for<8>([&](auto jc) {
                    constexpr int j = decltype(jc)::value;
                    const v4f a = acc_quad<(2 * u + h) * 8 + j>(acc_token);
                    // 8-byte writes of 16 rows at a time: rows r and r + 8 are 8 * (pitch mod 128 bytes) = 128 bytes apart in
                    // bank terms, the same 8-byte slot; the upper eight rows swap each pair of slots (undone when read back)
                    uint8_t* dst = patch + (h * 16 + l16) * kPitch + (((j * 16 + g4 * 4) * kEsz) ^ (kEsz == 2 ? ((l16 >> 3) & 1) << 3 : 0));
                    const float v0 = scaled(a[0], 4 * j), v1 = scaled(a[1], 4 * j + 1), v2 = scaled(a[2], 4 * j + 2),
                                v3 = scaled(a[3], 4 * j + 3);
                    float r0 = v0, r1 = v1, r2 = v2, r3 = v3;    // QSPEC: the outputs as OT holds them
                    if constexpr (kEsz == 4) {
                        *reinterpret_cast<float4*>(dst) = make_float4(v0, v1, v2, v3);
                        if constexpr (QSPEC)
                            spec_max = umax(umax(spec_max, __float_as_uint(v0) & 0x7fffffffu),
                                            umax(umax(__float_as_uint(v1) & 0x7fffffffu, __float_as_uint(v2) & 0x7fffffffu),
                                                 __float_as_uint(v3) & 0x7fffffffu));
                    } else {
                        uint32_t p01, p23;
                        if constexpr (__is_same(OT, bf16_t)) p01 = pack_bf16(v0, v1), p23 = pack_bf16(v2, v3);
                        else p01 = pack_f16(v0, v1), p23 = pack_f16(v2, v3);
                        *reinterpret_cast<uint2*>(dst) = make_uint2(p01, p23);
                        if constexpr (QSPEC) {
                            spec_max = pk_umax16(spec_max, pk_umax16(p01 & 0x7fff7fffu, p23 & 0x7fff7fffu));
                            widen_pair(p01, r0, r1);
                            widen_pair(p23, r2, r3);
                        }
                    }
                    if constexpr (QSPEC)
                        *reinterpret_cast<uint32_t*>(cpatch + (h * 16 + l16) * kCPitch + j * 16 + g4 * 4) =
                            quant4_in_range<MSAMP_DT_E4M3>(r0 * guess, r1 * guess, r2 * guess, r3 * guess);
                });
            });
            // no wait between the writes above and the reads below, nor before the next unit's writes: the patch is
            // private to this wave and the LDS serves one wave's requests in order
            constexpr int kPasses = 32 / kRowsPerPass;    // 8 or 16
            static_for<kPasses / 8>([&](auto gc) {
                constexpr int p0 = decltype(gc)::value * 8;
                // eight reads in flight together, then the eight stores (named values: an array here ends up in scratch)
                auto rd = [&](int t) {
                    const int pr = (p0 + t) * kRowsPerPass + prl;
                    const uint4 v = *reinterpret_cast<const uint4*>(patch + pr * kPitch + pc * 16);
                    const bool swapped = kEsz == 2 && (((p0 + t) * kRowsPerPass) >> 3) & 1;    // the same for all lanes of a pass
                    return swapped ? make_uint4(v.z, v.w, v.x, v.y) : v;
                };
                const uint4 val0 = rd(0), val1 = rd(1), val2 = rd(2), val3 = rd(3), val4 = rd(4), val5 = rd(5), val6 = rd(6),
                            val7 = rd(7);
                auto st = [&](int t, const uint4& v) {
                    const int first_row = row0 + wr * 128 + u * 32 + (p0 + t) * kRowsPerPass;    // wave-uniform
                    if constexpr (kVec && kInside) {
                        uint8_t* row_base = reinterpret_cast<uint8_t*>(D + static_cast<size_t>(first_row) * NC + (col0 + wc * 128));
                        store_out16(row_base + lane_off, v);
                    } else if constexpr (kVec) {
                        const int grow = first_row + prl;
                        if (grow < NR && gcol < NC) store_out16(D + static_cast<size_t>(grow) * NC + gcol, v);
                    } else {
                        // an output whose rows are not 16-byte aligned, or end inside a segment: the lane's segment one
                        // element at a time (still whole rows side by side: the 64 stores of a wave instruction touch few lines)
                        const int grow = first_row + prl;
                        if (grow < NR) {
                            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
                            OT* out = D + static_cast<size_t>(grow) * NC + gcol;
                            if (kEsz == 4 || pairs_ok) {    // 4-byte stores: float32, or 2-byte elements in aligned pairs
#pragma unroll
                                for (int e = 0; e < 4; ++e)
                                    if (gcol + e * (4 / kEsz) < NC) reinterpret_cast<uint32_t*>(out)[e] = w[e];
                            } else {
#pragma unroll
                                for (int e = 0; e < kElemsPerChunk; ++e)
                                    if (gcol + e < NC) reinterpret_cast<uint16_t*>(out)[e] = static_cast<uint16_t>(w[e >> 1] >> ((e & 1) * 16));
                            }
                        }
                    }
                };
                st(0, val0), st(1, val1), st(2, val2), st(3, val3), st(4, val4), st(5, val5), st(6, val6), st(7, val7);
            });
            if constexpr (QSPEC) {
                // the unit's codes: 32 rows of 128 bytes, eight rows per pass, 16 bytes per lane (whole tiles only)
                auto crd = [&](int t) {
                    return *reinterpret_cast<const uint4*>(cpatch + (t * 8 + (lane >> 3)) * kCPitch + (lane & 7) * 16);
                };
                const uint4 c0 = crd(0), c1 = crd(1), c2 = crd(2), c3 = crd(3);
                auto cst = [&](int t, const uint4& v) {
                    const int grow = row0 + wr * 128 + u * 32 + t * 8 + (lane >> 3);
                    const int gcol = col0 + wc * 128 + (lane & 7) * 16;
                    store_out16(qa.q + static_cast<size_t>(grow) * NC + gcol, v);
                };
                cst(0, c0), cst(1, c1), cst(2, c2), cst(3, c3);
            }
        });
    };
    if constexpr (QSPEC) {
        // whole tiles and 16-byte rows only, no bias (the host sees to that): the output in OT and its codes side by side
        if (accumulate) emit_fused_rows();
        else emit_plain(std::true_type{}, std::true_type{});
        uint32_t m = spec_max;
        if constexpr (kEsz == 2) {
            m = umax(m & 0xffffu, m >> 16);
            if constexpr (__is_same(OT, bf16_t)) m <<= 16;
            else m = __float_as_uint(f16_bits_to_float(m));
        }
        m = block_max_u32(m, red);    // valid in lane 0 of wave 0
        if (threadIdx.x == 0) {
            // Fold into the call's one word, then draw a ticket.  Both are atomics of agent scope on neighbouring words,
            // carried out where all XCDs meet; the maximum's old value has come back before the ticket is asked for, so
            // whoever draws the last ticket finds every workgroup's maximum in the word.  No fence: at agent scope a
            // fence writes this XCD's L2 back, outputs of the other compute units included, once per workgroup.
            uint32_t* w = qa.spec_words;
            uint32_t before = 0;
            if (m > __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                before = __hip_atomic_fetch_max(w, m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            asm volatile("s_waitcnt vmcnt(0)" : "+v"(before) : : "memory");
            const uint32_t ticket = __hip_atomic_fetch_add(w + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (ticket == gridDim.x - 1) {
                const uint32_t mm = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(w, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);    // ready for the next call
                __hip_atomic_store(w + 1, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                float am = __uint_as_float(mm);
                if ((qa.flags & MSAMP_FLAG_NAN_TO_INF) && !(am < __uint_as_float(0x7f800000u))) am = __uint_as_float(0x7f800000u);
                const float sc = scale_rule(am, guess, qa.fp_max, qa.margin);
                *qa.amax = am;
                *qa.scale = sc;
                *qa.scale_inv = 1.0f / sc;
                // The codes stand if the rule confirms the scale they were written with and every output times that scale
                // is finite and inside the format (they were converted without clamp or NaN patch); otherwise the
                // caller's next kernel writes them again from the stored output.
                const bool stand = __float_as_uint(sc) == __float_as_uint(guess) && am * guess <= qa.fp_max;
                w[2] = stand ? 0u : 1u;
            }
        }
        return;
    }
    const bool inside = row0 + kDmaTile <= NR && col0 + kDmaTile <= NC;
    // (the per-lane offset of the whole-tile form is 32 bits: four rows of the output)
    if (vec_ok && inside && static_cast<unsigned long long>(NC) * kEsz * 4 < (1ull << 31)) emit_plain(std::true_type{}, std::true_type{});
    else if (vec_ok) emit_plain(std::true_type{}, std::false_type{});
    else emit_plain(std::false_type{}, std::false_type{});
}

template <int XF, int YF, typename OT, bool XT, bool YT, bool KTAIL>
static int launch_gemm_dma_tail(const uint8_t* X, const uint8_t* Y, void* D, int NR, int NC, int K, const float* xs,
                                const float* ys, int accumulate, const void* bias, int bias_dt, hipStream_t st, int parts = 1) {
    constexpr int smem = kDmaBlocks * kDmaBlock;
    static std::atomic<bool> configured{false};    // setting the attribute twice is harmless
    auto kern = fp8_gemm_dma_kernel<XF, YF, OT, XT, YT, 0, false, KTAIL>;
    if (!configured.load(std::memory_order_acquire)) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
        if (e != hipSuccess) return hip_fail(e, "hipFuncSetAttribute(fp8_gemm_dma_kernel)");
        configured.store(true, std::memory_order_release);
    }
    const int tiles = ((NR + kDmaTile - 1) / kDmaTile) * ((NC + kDmaTile - 1) / kDmaTile);
    QuantArgs qa = {};
    qa.walk_plus_one = registered_walk(NR, NC, K, XT, YT) + 1;
    hipLaunchKernelGGL(kern, dim3(tiles, parts), dim3(kGemmThreads), smem, st, X, Y, static_cast<OT*>(D), NR, NC, K, xs, ys,
                       accumulate, bias, bias_dt, qa);
    MSAMP_CHECK_LAUNCH("fp8_gemm_dma_kernel");
    return MSAMP_OK;
}

template <int XF, int YF, typename OT, bool XT = false, bool YT = false>
static int launch_gemm_dma(const uint8_t* X, const uint8_t* Y, void* D, int NR, int NC, int K, const float* xs,
                           const float* ys, int accumulate, const void* bias, int bias_dt, hipStream_t st) {
    return launch_gemm_dma_tail<XF, YF, OT, XT, YT, false>(X, Y, D, NR, NC, K, xs, ys, accumulate, bias, bias_dt, st);
}

// the same kernel with the in-time cast to FP8 fused in (see QF above); the caller has checked the shape
template <int XF, int YF, typename OT, bool XT, bool YT, int QF>
static int launch_gemm_dma_quant(const uint8_t* X, const uint8_t* Y, int NR, int NC, int K, const float* xs,
                                        const float* ys, const QuantArgs& qa, hipStream_t st) {
    constexpr int smem = kDmaBlocks * kDmaBlock;
    static std::atomic<bool> configured{false};    // setting the attribute twice is harmless
    auto kern = fp8_gemm_dma_kernel<XF, YF, OT, XT, YT, QF>;
    if (!configured.load(std::memory_order_acquire)) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
        if (e != hipSuccess) return hip_fail(e, "hipFuncSetAttribute(fp8_gemm_dma_kernel, fused cast)");
        configured.store(true, std::memory_order_release);
    }
    // its workgroups wait for each other, one per CU: the runtime must confirm that one fits (asked once per instantiation)
    static std::atomic<int> resident{-1};
    int fits = resident.load(std::memory_order_acquire);
    if (fits < 0) {
        int blocks = 0;
        fits = hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, reinterpret_cast<const void*>(kern), kGemmThreads, smem) == hipSuccess &&
               blocks >= 1;
        resident.store(fits, std::memory_order_release);
    }
    if (!fits) return MSAMP_NOT_FUSED;
    const int tiles = (NR / kDmaTile) * (NC / kDmaTile);
    QuantArgs qw = qa;
    qw.walk_plus_one = registered_walk(NR, NC, K, XT, YT) + 1;
    hipLaunchKernelGGL(kern, dim3(tiles), dim3(kGemmThreads), smem, st, X, Y, static_cast<OT*>(nullptr), NR, NC, K, xs, ys, 0,
                       static_cast<const void*>(nullptr), 0, qw);
    MSAMP_CHECK_LAUNCH("fp8_gemm_dma_kernel (fused cast)");
    return MSAMP_OK;
}

// the same kernel with the cast to FP8 riding along on speculation (see QSPEC above); the caller has checked the shape
template <int XF, int YF, typename OT, bool XT, bool YT>
static int launch_gemm_dma_spec(const uint8_t* X, const uint8_t* Y, void* D, int NR, int NC, int K, const float* xs,
                                       const float* ys, int accumulate, const QuantArgs& qa, hipStream_t st) {
    constexpr int smem = kDmaBlocks * kDmaBlock;
    static std::atomic<bool> configured{false};    // setting the attribute twice is harmless
    auto kern = fp8_gemm_dma_kernel<XF, YF, OT, XT, YT, 0, true>;
    if (!configured.load(std::memory_order_acquire)) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
        if (e != hipSuccess) return hip_fail(e, "hipFuncSetAttribute(fp8_gemm_dma_kernel, speculative cast)");
        configured.store(true, std::memory_order_release);
    }
    const int tiles = (NR / kDmaTile) * (NC / kDmaTile);
    QuantArgs qw = qa;
    qw.walk_plus_one = registered_walk(NR, NC, K, XT, YT) + 1;
    hipLaunchKernelGGL(kern, dim3(tiles), dim3(kGemmThreads), smem, st, X, Y, static_cast<OT*>(D), NR, NC, K, xs, ys, accumulate,
                       static_cast<const void*>(nullptr), 0, qw);
    MSAMP_CHECK_LAUNCH("fp8_gemm_dma_kernel (speculative cast)");
    return MSAMP_OK;
}

template <int BR, int BC, int XF, int YF, typename OT, bool KGUARD>
static int launch_gemm_k(const uint8_t* X, const uint8_t* Y, void* D, int NR, int NC, int K, const float* xs,
                       const float* ys, int accumulate, const void* bias, int bias_dt, hipStream_t st) {
    constexpr int smem = 2 * (BR + BC) * kBK;
    static std::atomic<bool> configured{false};    // setting the attribute twice is harmless
    auto kern = fp8_gemm_kernel<BR, BC, XF, YF, OT, KGUARD>;
    if (!configured.load(std::memory_order_acquire)) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
        if (e != hipSuccess) return hip_fail(e, "hipFuncSetAttribute(fp8_gemm_kernel)");
        configured.store(true, std::memory_order_release);
    }
    const int tiles = ((NR + BR - 1) / BR) * ((NC + BC - 1) / BC);
    hipLaunchKernelGGL(kern, dim3(tiles), dim3(kGemmThreads), smem, st, X, Y, static_cast<OT*>(D), NR, NC, K, xs, ys,
                       accumulate, bias, bias_dt);
    MSAMP_CHECK_LAUNCH("fp8_gemm_kernel");
    return MSAMP_OK;
}

template <int BR, int BC, int XF, int YF, typename OT>
static int launch_gemm(const uint8_t* X, const uint8_t* Y, void* D, int NR, int NC, int K, const float* xs,
                       const float* ys, int accumulate, const void* bias, int bias_dt, hipStream_t st) {
    if (K % kBK == 0) return launch_gemm_k<BR, BC, XF, YF, OT, false>(X, Y, D, NR, NC, K, xs, ys, accumulate, bias, bias_dt, st);
    return launch_gemm_k<BR, BC, XF, YF, OT, true>(X, Y, D, NR, NC, K, xs, ys, accumulate, bias, bias_dt, st);
}

}    // namespace msamp
#include "gemm_small_tile.cuh"
namespace msamp {

// (problems for the 128 x 128 tiles and those with a ragged last slice of K have gone their way in run_gemm_pair)
template <int XF, int YF, typename OT>
static int pick_tile(const uint8_t* X, const uint8_t* Y, void* D, int NR, int NC, int K, const float* xs,
                     const float* ys, int accumulate, const void* bias, int bias_dt, hipStream_t st) {
    if (K % kBK == 0 && K >= 2 * kBK && fits_offsets(NR, NC, K) && small_tile_limit() >= 0)
        return launch_gemm_dma<XF, YF, OT>(X, Y, D, NR, NC, K, xs, ys, accumulate, bias, bias_dt, st);
    return launch_gemm<128, 128, XF, YF, OT>(X, Y, D, NR, NC, K, xs, ys, accumulate, bias, bias_dt, st);
}

template <int XF, int YF>
static int pick_out(const uint8_t* X, const uint8_t* Y, void* D, int d_dtype, int NR, int NC, int K, const float* xs,
                    const float* ys, int accumulate, const void* bias, int bias_dt, hipStream_t st) {
    switch (d_dtype) {
        case MSAMP_DT_F32:
            return pick_tile<XF, YF, float>(X, Y, D, NR, NC, K, xs, ys, accumulate, bias, bias_dt, st);
        case MSAMP_DT_F16:
            return pick_tile<XF, YF, f16_t>(X, Y, D, NR, NC, K, xs, ys, accumulate, bias, bias_dt, st);
        default:
            return pick_tile<XF, YF, bf16_t>(X, Y, D, NR, NC, K, xs, ys, accumulate, bias, bias_dt, st);
    }
}

template <int XF, int YF, bool XT, bool YT>
static int pick_out_kmajor(const uint8_t* X, const uint8_t* Y, void* D, int d_dtype, int NR, int NC, int K, const float* xs,
                           const float* ys, int accumulate, const void* bias, int bias_dt, hipStream_t st) {
    switch (d_dtype) {
        case MSAMP_DT_F32:
            return launch_gemm_dma<XF, YF, float, XT, YT>(X, Y, D, NR, NC, K, xs, ys, accumulate, bias, bias_dt, st);
        case MSAMP_DT_F16:
            return launch_gemm_dma<XF, YF, f16_t, XT, YT>(X, Y, D, NR, NC, K, xs, ys, accumulate, bias, bias_dt, st);
        default:
            return launch_gemm_dma<XF, YF, bf16_t, XT, YT>(X, Y, D, NR, NC, K, xs, ys, accumulate, bias, bias_dt, st);
    }
}

template <int XF, int YF, bool T>
static int pick_out_quant(const uint8_t* X, const uint8_t* Y, int d_dtype, int NR, int NC, int K, const float* xs, const float* ys,
                          const QuantArgs& qa, hipStream_t st) {
    switch (d_dtype) {
        case MSAMP_DT_F32:
            return launch_gemm_dma_quant<XF, YF, float, T, T, MSAMP_DT_E4M3>(X, Y, NR, NC, K, xs, ys, qa, st);
        case MSAMP_DT_F16:
            return launch_gemm_dma_quant<XF, YF, f16_t, T, T, MSAMP_DT_E4M3>(X, Y, NR, NC, K, xs, ys, qa, st);
        default:
            return launch_gemm_dma_quant<XF, YF, bf16_t, T, T, MSAMP_DT_E4M3>(X, Y, NR, NC, K, xs, ys, qa, st);
    }
}

template <int XF, int YF, bool T>
static int pick_out_spec(const uint8_t* X, const uint8_t* Y, void* D, int d_dtype, int NR, int NC, int K, const float* xs,
                         const float* ys, int accumulate, const QuantArgs& qa, hipStream_t st) {
    switch (d_dtype) {
        case MSAMP_DT_F32:
            // a float32 product takes the two steps: with four-byte outputs the epilogue that also emits codes does not
            // fit the vector registers left beside the accumulators
            return MSAMP_NOT_FUSED;
        case MSAMP_DT_F16:
            return launch_gemm_dma_spec<XF, YF, f16_t, T, T>(X, Y, D, NR, NC, K, xs, ys, accumulate, qa, st);
        default:
            return launch_gemm_dma_spec<XF, YF, bf16_t, T, T>(X, Y, D, NR, NC, K, xs, ys, accumulate, qa, st);
    }
}

#ifdef MSAMP_GEMM_SECOND_UNIT
// output type and operand layout of a call -> one instantiation of LAUNCH<XF, YF, output type, XT, YT>
#define MSAMP_LAYOUT_LAUNCH(LAUNCH, OT)                                                                                              \
    do {                                                                                                                             \
        if (c.xt && c.yt) return LAUNCH<XF, YF, OT, true, true>(MSAMP_CALL_ARGS);                                                     \
        if (c.yt) return LAUNCH<XF, YF, OT, false, true>(MSAMP_CALL_ARGS);                                                            \
        return LAUNCH<XF, YF, OT, false, false>(MSAMP_CALL_ARGS);                                                                     \
    } while (0)
#define MSAMP_CALL_ARGS c.X, c.Y, c.D, c.NR, c.NC, c.K, c.xs, c.ys, c.accumulate, c.bias, c.bias_dt, c.st
#define MSAMP_TYPE_LAUNCH(LAUNCH)                                   \
    switch (c.d_dtype) {                                            \
        case MSAMP_DT_F32: MSAMP_LAYOUT_LAUNCH(LAUNCH, float);      \
        case MSAMP_DT_F16: MSAMP_LAYOUT_LAUNCH(LAUNCH, f16_t);      \
        default: MSAMP_LAYOUT_LAUNCH(LAUNCH, bf16_t);               \
    }

template <int XF, int YF, typename OT, bool XT, bool YT>
static int launch_gemm_ragged(const uint8_t* X, const uint8_t* Y, void* D, int NR, int NC, int K, const float* xs,
                              const float* ys, int accumulate, const void* bias, int bias_dt, hipStream_t st) {
    return launch_gemm_dma_tail<XF, YF, OT, XT, YT, true>(X, Y, D, NR, NC, K, xs, ys, accumulate, bias, bias_dt, st);
}
template <int XF, int YF>
int run_gemm_ragged(const GemmCall& c) {
    MSAMP_TYPE_LAUNCH(launch_gemm_ragged)
}
template <int XF, int YF>
int run_gemm_small(const GemmCall& c) {
    MSAMP_TYPE_LAUNCH(launch_gemm_dma128)
}
template <int XF, int YF>
int run_gemm_pair128(const GemmCall& c) {
    MSAMP_TYPE_LAUNCH(launch_gemm_pair128)
}
template <int XF, int YF>
int run_gemm_parts(const GemmCall& c, const KSplit& split) {
#define MSAMP_PARTS_LAUNCH(XT, YT) \
    return launch_gemm_dma128_tail<XF, YF, float, XT, YT, true>(c.X, c.Y, c.D, c.NR, c.NC, c.K, c.xs, c.ys, 0, nullptr, 0, c.st, split.parts)
    if (!c.yt) MSAMP_PARTS_LAUNCH(false, false);
    if (!c.xt) MSAMP_PARTS_LAUNCH(false, true);
    if (split.small_tiles) MSAMP_PARTS_LAUNCH(true, true);
#undef MSAMP_PARTS_LAUNCH
    return launch_gemm_dma_tail<XF, YF, float, true, true, true>(c.X, c.Y, c.D, c.NR, c.NC, c.K, c.xs, c.ys, 0, nullptr, 0, c.st, split.parts);
}
#endif

// Everything behind the C entry points for one pair of operand formats.  gemm_inst.hip instantiates it once per
// pair (four translation units, so that they compile side by side).
//
// Which kernel: few 256 x 256 tiles leave most compute units idle and take 128 x 128 tiles, two workgroups to a compute unit
// (takes_paired_tiles()) or one (takes_small_tiles()).  The direct-to-LDS kernels need 32-bit row offsets and, but for the paired
// form, more than one 128-byte slice of K; where they can run they are the faster ones at every size (256 x 256 x 4096: 14 against
// 80 us with the generic kernel, 8192 x 4096 x 4096: 100 against 555), also with a ragged last slice (12605 x 4304 x 1200 into
// float16: 94 against 153, 8192 x 4096 x 4080: 121 against 195).  Everything else takes the generic register-staged kernel.  So does
// a float32 output of at most 16 columns over less than a slice of K, with a bias or of a few rows, which is a launch and little else
// (K of 16 to 64, generic against paired, us: with a bias 48 x 16 4.6, 5.2, 2048 x 16 5.2, 6.1; without 16 x 16 3.8, 4.1, 48 x 16 4.5, 4.6,
// 112 x 16 5.0, 5.0; in bfloat16 it is the paired form that is ahead, 512 x 16 5.7 to 4.7, and with 24 columns everywhere).
template <int XF, int YF>
int run_gemm_pair(const GemmCall& c) {
    if (c.qa == nullptr && fits_offsets(c.NR, c.NC, c.K)) {
        const bool sliver = !c.yt && c.K < kBK && c.NC <= 16 && c.d_dtype == MSAMP_DT_F32 && (c.bias != nullptr || c.NR <= 64);
        if (!sliver && (takes_paired_tiles(c.NR, c.NC, c.K) || (c.yt && c.K <= kBK))) return run_gemm_pair128<XF, YF>(c);
        if (takes_small_tiles(c.NR, c.NC, c.K)) return run_gemm_small<XF, YF>(c);
        if (c.K > kBK && c.K % kBK && (c.yt || small_tile_limit() >= 0)) return run_gemm_ragged<XF, YF>(c);
    }
    if (c.qa != nullptr && c.qspec) {
        if (c.xt) return pick_out_spec<XF, YF, true>(c.X, c.Y, c.D, c.d_dtype, c.NR, c.NC, c.K, c.xs, c.ys, c.accumulate, *c.qa, c.st);
        return pick_out_spec<XF, YF, false>(c.X, c.Y, c.D, c.d_dtype, c.NR, c.NC, c.K, c.xs, c.ys, c.accumulate, *c.qa, c.st);
    }
    if (c.qa != nullptr) {
        if (c.xt) return pick_out_quant<XF, YF, true>(c.X, c.Y, c.d_dtype, c.NR, c.NC, c.K, c.xs, c.ys, *c.qa, c.st);
        return pick_out_quant<XF, YF, false>(c.X, c.Y, c.d_dtype, c.NR, c.NC, c.K, c.xs, c.ys, *c.qa, c.st);
    }
    if (c.xt && c.yt)
        return pick_out_kmajor<XF, YF, true, true>(c.X, c.Y, c.D, c.d_dtype, c.NR, c.NC, c.K, c.xs, c.ys, c.accumulate, c.bias, c.bias_dt, c.st);
    if (c.yt)
        return pick_out_kmajor<XF, YF, false, true>(c.X, c.Y, c.D, c.d_dtype, c.NR, c.NC, c.K, c.xs, c.ys, c.accumulate, c.bias, c.bias_dt, c.st);
    return pick_out<XF, YF>(c.X, c.Y, c.D, c.d_dtype, c.NR, c.NC, c.K, c.xs, c.ys, c.accumulate, c.bias, c.bias_dt, c.st);
}

}    // namespace msamp
