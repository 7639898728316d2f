// The direct-to-LDS FP8 GEMM with 128 x 128 output tiles, for problems that leave most compute units idle with
// 256 x 256 tiles (a 2048 x 2048 output is 64 of those, a quarter of the chip, and 256 of these).  At least four
// 128-byte slices of K (the last one may be ragged: KTAIL); operands row-major (K-contiguous) or, with XT / YT, K-major ([K][rows], kmajor_pitch() apart):
// the slice then lies in LDS as 128 k-rows of 128 bytes, the 16-byte position XOR-ed with k % 8, and the fragments
// come from the transposing LDS read, as in the large tile.
//
// Four wavefronts, each owning a 64 x 64 quadrant as 4 x 4 accumulators of the 16x16x128 FP8 MFMA, in fixed AGPRs like
// those of the large tile (block (i, j) in a[16i + 4j .. + 3]; left to the register allocator they were renumbered
// from slice to slice, with copies and wait states between the MFMAs).  A K slice is 128 X rows
// and 128 Y rows of 128 bytes, 32 KiB, brought in by eight direct-to-LDS loads per wavefront with the same swizzle
// as the large tile; five stages -- the whole LDS -- so that three slices are on their way while one is being read and
// another worked on (a slice is only 16 MFMAs per wavefront, a fifth of a microsecond, and the way to L2 is close to
// a microsecond).  The fragments of slice kt + 1 are read from LDS between the first eight MFMAs of slice kt, and the
// eight loads of slice kt + 4 go out one every other MFMA (issued in one go after the barrier they held the wave, and
// its MFMAs, while the memory pipe accepted them: 0.54 against 0.43 us per slice); one barrier per slice.
//
// Per flop this tile needs twice the L2 -> LDS bytes of the large one (32 KiB per 16 MFMAs per wavefront against
// 64 KiB per 64), which is what bounds it once every compute unit runs one: 2048 x 2048 x 4096 takes 16.7 us with the
// MFMAs and 15.5 us without them (an ablation), 95 GB/s per compute unit where a bare loop of such loads reaches 121.
// It is the faster kernel only while the large tile leaves compute units idle, and the host picks it only then.
//
// PAIR: two workgroups to a compute unit, so that one's launch, prologue and epilogue run under the other's products, and up to
// two tiles a unit go side by side instead of one after the other (which products: takes_paired_tiles()).  80 KiB of LDS each:
// a ring of five units of 16 KiB, one operand's part of a slice, with a slice being read and one and a half on their way; any
// number of slices.  Two waves to a SIMD leave each 256 registers: the X fragments are not doubled (a block of the next slice is
// read behind the last product of the present one), and the accumulators are v192 .. v255, which the compiler is kept from by
// amdgpu_num_vgpr (half of 192: the unit of the attribute is a pair here).  With AGPRs in use it would halve the 256 instead, and
// 128 do not hold the fragments.  Bound by the LDS: 96 KiB through it per slice and tile, 768 of its cycles beside 512 of the
// matrix pipes; hence the larger tiles where there are enough of them.
//
// Every output element is accumulated over the 128-byte blocks of K in ascending order, one MFMA per block, and
// scaled, biased, summed and rounded with the expressions of the large tile: the kernels agree to the bit.
#pragma once

namespace msamp {

constexpr int kSmallTile = 128;
constexpr int kSmallStage = 2 * kSmallTile * kBK;    // 32 KiB
constexpr int kSmallStages = 5;    // all 160 KiB of the LDS
constexpr int kPairUnit = kSmallTile * kBK;    // PAIR: one operand's part of a slice, 16 KiB
constexpr int kPairUnits = 5;                  // 80 KiB, half of the LDS

// The accumulators of the PAIR form, block n in v[192 + 4n .. 195 + 4n], handled as those in AGPRs are (gemm_kernels.cuh).
#define MSAMP_VACC                                                                                                      \
    "v192", "v193", "v194", "v195", "v196", "v197", "v198", "v199", "v200", "v201", "v202", "v203", "v204", "v205", "v206", \
        "v207", "v208", "v209", "v210", "v211", "v212", "v213", "v214", "v215", "v216", "v217", "v218", "v219", "v220",     \
        "v221", "v222", "v223", "v224", "v225", "v226", "v227", "v228", "v229", "v230", "v231", "v232", "v233", "v234",     \
        "v235", "v236", "v237", "v238", "v239", "v240", "v241", "v242", "v243", "v244", "v245", "v246", "v247", "v248",     \
        "v249", "v250", "v251", "v252", "v253", "v254", "v255"
constexpr int kVacc = 192;
template <int N, int CB, int BL>
__device__ __forceinline__ void vmfma_fixed(const v8i& a, const v8i& b) {
    asm volatile("v_mfma_f32_16x16x128_f8f6f4 v[%2:%3], %0, %1, v[%2:%3] cbsz:%4 blgp:%5"
                 :
                 : "v"(a), "v"(b), "n"(kVacc + N * 4), "n"(kVacc + N * 4 + 3), "n"(CB), "n"(BL));
}
template <int N, int CB, int BL>
__device__ __forceinline__ void vmfma_fixed_and_load(const v8i& a, const v8i& b, const LdsLoad& l) {
    asm volatile("s_mov_b32 m0, %6\n\tv_mfma_f32_16x16x128_f8f6f4 v[%2:%3], %0, %1, v[%2:%3] cbsz:%4 blgp:%5\n\tglobal_load_lds_dwordx4 %7, %8"
                 :
                 : "v"(a), "v"(b), "n"(kVacc + N * 4), "n"(kVacc + N * 4 + 3), "n"(CB), "n"(BL), "s"(l.dst), "v"(l.off), "s"(l.src)
                 : "memory", "m0");
}
__device__ __forceinline__ void vacc_clear() {
    static_for<16>([&](auto nc) {
        constexpr int n = decltype(nc)::value;
        asm volatile("v_mov_b32 v[%0], 0\n\tv_mov_b32 v[%1], 0\n\tv_mov_b32 v[%2], 0\n\tv_mov_b32 v[%3], 0"
                     :
                     : "n"(kVacc + n * 4), "n"(kVacc + n * 4 + 1), "n"(kVacc + n * 4 + 2), "n"(kVacc + n * 4 + 3));
    });
    asm volatile("s_nop 4" : : : MSAMP_VACC);
}
__device__ __forceinline__ uint32_t vacc_fence() {
    uint32_t token;
    asm volatile("s_nop 15\n\ts_nop 7\n\tv_mov_b32 %0, 0" : "=v"(token) : : MSAMP_VACC);
    return token;
}
template <int N>
__device__ __forceinline__ v4f vacc_quad(uint32_t token) {
    v4f r;
    float x, y, z, w;
    asm("v_mov_b32 %0, v[%1]" : "=v"(x) : "n"(kVacc + N * 4), "v"(token));
    asm("v_mov_b32 %0, v[%1]" : "=v"(y) : "n"(kVacc + N * 4 + 1), "v"(token));
    asm("v_mov_b32 %0, v[%1]" : "=v"(z) : "n"(kVacc + N * 4 + 2), "v"(token));
    asm("v_mov_b32 %0, v[%1]" : "=v"(w) : "n"(kVacc + N * 4 + 3), "v"(token));
    r[0] = x, r[1] = y, r[2] = z, r[3] = w;
    return r;
}

template <int XF, int YF, typename OT, bool XT, bool YT, bool KTAIL, bool PAIR = false>
__device__ __forceinline__ void gemm_dma128(const uint8_t* __restrict__ X, const uint8_t* __restrict__ Y, OT* __restrict__ D, int NR,
                                            int NC, int K, const float* __restrict__ x_scale_inv,
                                            const float* __restrict__ y_scale_inv, int accumulate, const void* __restrict__ bias,
                                            int bias_dt) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    constexpr bool kParts = KTAIL && !PAIR && std::is_same<OT, float>::value;
    const int ldk = K;    // from one row of a row-major operand to the next
    if constexpr (kParts) k_part<XT, YT>(X, Y, D, NR, NC, K);
    const int tiles_r = (NR + kSmallTile - 1) / kSmallTile, tiles_c = (NC + kSmallTile - 1) / kSmallTile;
    int tr, tc;
    tile_of_id(blockIdx.x, tiles_r, tiles_c, false, false, tr, tc);
    const int row0 = tr * kSmallTile, col0 = tc * kSmallTile;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wr = wave >> 1, wc = wave & 1;
    // the output factor and the bias are fetched now: in the epilogue they would sit on its critical path
    constexpr int kEsz = static_cast<int>(sizeof(OT));
    constexpr int kElems = 16 / kEsz;              // outputs per 16-byte segment: 8 or 4
    constexpr int kSegs = 64 / kElems;             // segments per 64-column row: 8 or 16
    const int seg = lane % kSegs;
    const int gcol = col0 + wc * 64 + seg * kElems;
    float alpha = (*x_scale_inv) * (*y_scale_inv);
    if constexpr (kParts) alpha = gridDim.y > 1 ? 1.0f : alpha;
    // (one column of the wave's 64 a lane, handed out in the epilogue: a load for each of a lane's columns, one behind the other, took
    // up to 3 us of a tile's time: 4608 x 4096 x 512 with two workgroups to a compute unit 20.5 -> 17.9 us, 8192 x 4096 x 512 29.5 -> 25.4)
    // (PAIR: as it lies in memory, and made a float in the epilogue, so that nothing waits for it; fetched behind the products it was
    // waited for.  Both changes, bfloat16 with a bias, us: 2048 x 2048 x 528 7.7 -> 7.6, x 912 both K-major 9.0 -> 8.2, 256 x 256 x
    // 400 6.5 -> 5.9, 512 x 16 x 64 5.7 -> 5.3)
    float bias_lane = 0.0f;
    uint32_t bias_bits = 0;
    if (const int c = col0 + wc * 64 + lane; bias != nullptr && c < NC) {
        if constexpr (!PAIR) bias_lane = load_bias(bias, bias_dt, c);
        else if (bias_dt == MSAMP_DT_F32) bias_bits = static_cast<const uint32_t*>(bias)[c];
        else bias_bits = static_cast<const uint16_t*>(bias)[c];
    }
    if constexpr (!PAIR) asm volatile("" : "+v"(bias_lane));
    asm volatile("" : "+v"(alpha));

    // ---- global -> LDS: one wave instruction fills 8 rows of 128 bytes (lane l: row l / 8, 16-byte position l % 8,
    // fetching the logical chunk position ^ swizzle(row)); rows past the end of the matrix are clamped to its last row
    // K-major operand: one wave instruction fills 8 k-rows of 128 bytes (lane l: k-row l / 8, position l % 8, fetching
    // the logical chunk position ^ (k-row % 8))
    const int chunk = (lane & 7) ^ (lane >> 3) ^ (wave & 1);
    const int chunk_t = (lane & 7) ^ (lane >> 3);
    const uint32_t lds_base = __builtin_amdgcn_readfirstlane(
        static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)smem)));
    // K-major operand, last tile: chunks past the end of a k-row are fetched from the tile's first chunk instead
    const int xcol = row0 + chunk_t * 16 < NR ? row0 + chunk_t * 16 : row0;
    const int ycol = col0 + chunk_t * 16 < NC ? col0 + chunk_t * 16 : col0;
    const int ldx = kmajor_pitch(NR), ldy = kmajor_pitch(NC);
    uint32_t xoff[4], yoff[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = (i * 4 + wave) * 8 + (lane >> 3);
        int gx = row0 + r, gy = col0 + r;
        gx = gx < NR ? gx : NR - 1;
        gy = gy < NC ? gy : NC - 1;
        const int krow = (i * 4 + wave) * 8 + (lane >> 3);
        xoff[i] = XT ? static_cast<uint32_t>(krow) * static_cast<uint32_t>(ldx) + xcol
                     : static_cast<uint32_t>(gx) * static_cast<uint32_t>(ldk) + chunk * 16;
        yoff[i] = YT ? static_cast<uint32_t>(krow) * static_cast<uint32_t>(ldy) + ycol
                     : static_cast<uint32_t>(gy) * static_cast<uint32_t>(ldk) + chunk * 16;
    }
    // KTAIL: a ragged last slice of `rem` K bytes, handled as in the large tile (loads kept inside the operand, fragments
    // masked)
    const int nk = KTAIL ? (K + kBK - 1) / kBK : K / kBK;    // at least 4, PAIR: 1 (the host sees to that)
    const int rem = K - (nk - 1) * kBK;
    const uint32_t tail_back = KTAIL && chunk * 16 >= rem ? chunk * 16 : 0;
    // where the X or Y half of slice kt lies in the LDS
    auto place = [&](int kt, bool is_x) __attribute__((always_inline)) {
        return PAIR ? (2 * kt + (is_x ? 0 : 1)) % kPairUnits * kPairUnit
                    : kt % kSmallStages * kSmallStage + (is_x ? 0 : kSmallTile * kBK);
    };
    // one of the 8 loads of a slice (0..3: X rows, 4..7: Y rows); where it comes from and goes to
    auto load_of = [&](int kt, int which, bool last = false) __attribute__((always_inline)) {
        const bool is_x = which < 4;
        const size_t slice = static_cast<size_t>(kt) * kBK;
        const uint8_t* src = is_x ? X + (XT ? slice * ldx : slice) : Y + (YT ? slice * ldy : slice);
        uint32_t off = is_x ? xoff[which] : yoff[which - 4];
        if (KTAIL && last) {
            if (is_x ? XT : YT) {
                if (((which & 3) * 4 + wave) * 8 + (lane >> 3) >= rem) off = is_x ? xcol : ycol;
            } else {
                off -= tail_back;
            }
        }
        const uint32_t dst = __builtin_amdgcn_readfirstlane(lds_base + place(kt, is_x) + ((which & 3) * 4 + wave) * 1024);
        return LdsLoad{dst, off, src};
    };
    auto dma = [&](int kt, int which, bool last = false) __attribute__((always_inline)) { load_to_lds(load_of(kt, which, last)); };
    auto dma_slice = [&](int kt, bool last = false) __attribute__((always_inline)) {
#pragma unroll
        for (int w = 0; w < 8; ++w) dma(kt, w, last);
    };

    // ---- LDS -> fragments: for row lane % 16 of a 16-row block a lane holds the K-bytes (lane / 16) * 32 .. + 31 of the
    // slice, two 16-byte reads at the swizzled chunks
    const int l16 = lane & 15, g4 = lane >> 4;
    const int fsw = (lane & 7) ^ ((lane >> 3) & 1);
    const int off_lo = ((2 * g4) ^ fsw) << 4;
    const int xrow = (wr * 64 + l16) * kBK;
    const int yrow = (wc * 64 + l16) * kBK;
    const int tj = l16 >> 1;
    const int t_lane = (g4 * 32 + tj) * kBK + (l16 & 1) * 8;    // k-row and 8-byte half of this lane's transposing reads
    // A slice's fragments arrive in pieces: two 16-byte reads per 16-row block of a row-major operand (block p / 2, half
    // p % 2), four 8-byte transposing reads per block of a K-major one (block p / 4, eight k each); X pieces first.
    constexpr int kPX = XT ? 16 : 8, kPY = YT ? 16 : 8, kPieces = kPX + kPY;
    auto read_piece = [&](int* fxd, int* fyd, int px, int py, int p) __attribute__((always_inline)) {
        const bool is_x = p < kPX;
        const uint8_t* base = smem + (is_x ? px : py);
        const int q = is_x ? p : p - kPX;
        if ((is_x && !XT) || (!is_x && !YT)) {
            const int b = q >> 1, hf = q & 1;
            const v4i val = *reinterpret_cast<const v4i*>(base + (is_x ? xrow : yrow) + b * 16 * kBK + (off_lo ^ (hf * 16)));
            int* d = (is_x ? fxd : fyd) + b * 8 + hf * 4;
            d[0] = val[0], d[1] = val[1], d[2] = val[2], d[3] = val[3];
        } else {
            const int b = q >> 2, qq = q & 3;
            const int wq = is_x ? wr : wc;
            const int addr = t_lane + (qq * 8) * kBK + (((wq * 4 + b) ^ tj) << 4);
            const v2i val = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i*)(base + addr));
            int* d = (is_x ? fxd : fyd) + b * 8 + qq * 2;
            d[0] = val[0], d[1] = val[1];
        }
    };

    if constexpr (PAIR) vacc_clear();
    else acc_clear();
    int fx[PAIR ? 1 : 2][32], fy[2][32];

    // the 16 MFMAs of the slice held in fragment set `cur`, with the 16 fragment reads of slice rd_kt (into the other
    // set) between them.  srcA = Y rows, srcB = X rows: a lane then holds, for D row lane % 16 of a block, four
    // consecutive D columns.
    // PAIR: `do_load` stands for the Y half of slice ld_kt, `next_x` for the X half of the slice behind it, and `ld_last`
    // for the last slice of K being the one (if next_x) or the other.
    auto step = [&](auto curc, int rd_kt, bool do_read, int ld_kt, bool do_load, bool ld_last = false, bool masked = false,
                    bool next_x = false) __attribute__((always_inline)) {
        constexpr int cur = decltype(curc)::value;
        if (KTAIL && masked) mask_fragments(fx[PAIR ? 0 : cur], g4, rem), mask_fragments(fy[cur], g4, rem);
        constexpr int cb = (YF == MSAMP_DT_E4M3) ? 0 : 1;
        constexpr int bl = (XF == MSAMP_DT_E4M3) ? 0 : 1;
        int px = place(rd_kt, true), py = place(rd_kt, false);
        // (opaque: otherwise every read's address is worked out for both turns in front of the loop, in registers that PAIR
        // does not have)
        if constexpr (PAIR) asm volatile("" : "+s"(px), "+s"(py));
        static_for<16>([&](auto nc) {
            constexpr int n = decltype(nc)::value;
            constexpr int i = PAIR ? n >> 2 : n & 3, j = PAIR ? n & 3 : n >> 2;
            const int* cx = fx[PAIR ? 0 : cur] + i * 8;
            const int* cy = fy[cur] + j * 8;
            const v8i vx = {cx[0], cx[1], cx[2], cx[3], cx[4], cx[5], cx[6], cx[7]};
            const v8i vy = {cy[0], cy[1], cy[2], cy[3], cy[4], cy[5], cy[6], cy[7]};
            if constexpr (PAIR) {
                const bool load_y = do_load && (n & 1) && n < 8, load_x = next_x && (n & 1) && n >= 8, tail = KTAIL && ld_last;
                auto load = [&]() __attribute__((always_inline)) {
                    return load_y ? load_of(ld_kt, 4 + (n >> 1), ld_last && !next_x) : load_of(ld_kt + 1, (n >> 1) - 4, ld_last);
                };
                // (the loads of a ragged last slice have offsets of their own, for which there is no register beside the operands)
                if ((load_y || load_x) && !tail) vmfma_fixed_and_load<i * 4 + j, cb, bl>(vy, vx, load());
                else vmfma_fixed<i * 4 + j, cb, bl>(vy, vx);
                if ((load_y || load_x) && tail) load_to_lds(load());
                // the Y fragments of the next slice with the first eight MFMAs, an X block in place of this slice's behind
                // its last MFMA
                if (do_read && n < 8) {
#pragma unroll
                    for (int p = n * kPY / 8; p < (n + 1) * kPY / 8; ++p) read_piece(fx[0], fy[cur ^ 1], px, py, kPX + p);
                }
                if (do_read && (n & 3) == 3) {
#pragma unroll
                    for (int p = i * kPX / 4; p < (i + 1) * kPX / 4; ++p) read_piece(fx[0], fy[cur ^ 1], px, py, p);
                }
            } else {
                // the eight tile loads of slice ld_kt, one every other MFMA: issued in one go they hold the wave, and with
                // it its MFMAs, for as long as the memory pipe takes to accept them
                if (do_load && (n & 1)) mfma_fixed_and_load<i * 4 + j, cb, bl>(vy, vx, load_of(ld_kt, n >> 1, ld_last));
                else mfma_fixed<i * 4 + j, cb, bl>(vy, vx);
                // the fragment reads go with the first eight MFMAs (two to four each) and have come back by the barrier that
                // follows the last one; nothing moves across, so they stay spread as written
                if (do_read && n < 8) {
#pragma unroll
                    for (int p = n * kPieces / 8; p < (n + 1) * kPieces / 8; ++p) read_piece(fx[cur ^ 1], fy[cur ^ 1], px, py, p);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    constexpr std::integral_constant<int, 0> c0{};
    constexpr std::integral_constant<int, 1> c1{};

    if constexpr (PAIR) {
        auto half = [&](int kt, int first, bool last = false) __attribute__((always_inline)) {
#pragma unroll
            for (int w = 0; w < 4; ++w) dma(kt, first + w, last);
        };
        dma_slice(0, nk == 1);
        if (nk > 1) dma_slice(1, nk == 2);
        if (nk > 2) {
            half(2, 0, nk == 3);
            wait_vmcnt<12>();
        } else if (nk == 2) {
            wait_vmcnt<8>();
        } else {
            wait_vmcnt<0>();
        }
        __syncthreads();
#pragma unroll
        for (int p = 0; p < kPieces; ++p) read_piece(fx[0], fy[0], place(0, true), place(0, false), p);

        // Before the step of slice kt: slice kt is in registers, slice kt + 1 and the X half of kt + 2 are on their way.  Wait
        // for slice kt + 1, meet (it has landed, and the two units of slice kt are free), compute slice kt while reading
        // kt + 1 and sending for the Y half of kt + 2 and the X half of kt + 3.
        auto turn = [&](auto curc, int kt, bool ld_last = false) __attribute__((always_inline)) {
            wait_vmcnt<4>();
            __syncthreads();
            step(curc, kt + 1, true, kt + 2, true, ld_last, false, true);
        };
        auto tail2 = [&](auto ac, auto bc, int k0) __attribute__((always_inline)) {
            wait_vmcnt<0>();
            __syncthreads();
            step(ac, k0 + 1, true, 0, false);
            step(bc, 0, false, 0, false, false, true);
        };
        auto tail3 = [&](auto ac, auto bc, int k0) __attribute__((always_inline)) {
            wait_vmcnt<4>();
            __syncthreads();
            step(ac, k0 + 1, true, k0 + 2, true, true);
            tail2(bc, ac, k0 + 1);
        };
        int kt = 0;
        for (; kt + 5 < nk; kt += 2) {
            turn(c0, kt);
            turn(c1, kt + 1);
        }
        // four or five slices are left, or there are three or fewer in all
        if constexpr (KTAIL) {
            // These ways to the end come out one behind the other, each tested for, and what the others would start from stayed in
            // its registers through the way of four slices, where nine others spilled.  Here it is given up at the end of that one,
            // which comes first (at the end of each way the others took 1 to 2 % longer).  Row-major, one operand K-major, both, us:
            // 2048 x 2048 x 400 7.13, 6.40, 6.98 -> 6.6, 6.4, 6.5; 2048 x 2048 x 912 9.0, 7.7, 8.3 -> 8.4, 7.7, 7.7; five slices, which
            // spilled nothing, 2048 x 2048 x 528 6.96, 6.7, 6.65 and as before.  (Nor do whole slices, which have it the plain way.)
            int left = nk - kt;
            auto is = [&](int n) __attribute__((always_inline)) {
                asm volatile("" : "+s"(left));
                return left == n;
            };
            auto give_up = [&]() __attribute__((always_inline)) {
                left = 0;
#pragma unroll
                for (int i = 0; i < 32; ++i) asm volatile("" : "=v"(fx[0][i]), "=v"(fy[0][i]), "=v"(fy[1][i]));
            };
            if (is(4)) turn(c0, kt, true), tail3(c1, c0, kt + 1), give_up();
            if (is(5)) {
                turn(c0, kt), turn(c1, kt + 1, true), tail3(c0, c1, kt + 2);
            } else if (left == 3) {
                tail3(c0, c1, 0);
            } else if (left == 2) {
                tail2(c0, c1, 0);
            } else if (left == 1) {
                step(c0, 0, false, 0, false, false, true);
            }
        } else if (kt + 5 == nk) {
            turn(c0, kt);
            turn(c1, kt + 1, true);
            tail3(c0, c1, kt + 2);
        } else if (kt + 4 == nk) {
            turn(c0, kt, true);
            tail3(c1, c0, kt + 1);
        } else if (nk == 3) {
            tail3(c0, c1, 0);
        } else if (nk == 2) {
            tail2(c0, c1, 0);
        } else {
            step(c0, 0, false, 0, false, false, true);
        }
    } else {
        dma_slice(0);
        dma_slice(1);
        dma_slice(2);
        dma_slice(3, nk == 4);
        wait_vmcnt<24>();
        __syncthreads();
    #pragma unroll
        for (int p = 0; p < kPieces; ++p) read_piece(fx[0], fy[0], place(0, true), place(0, false), p);

        // Before the step of slice kt: slices kt + 1 .. kt + 3 are on their way (24 loads of this wave), slice kt is in
        // registers.  Wait for slice kt + 1, meet (it has landed in every wave's part of the stage, and nobody reads the
        // stage of slice kt - 1 any more), compute slice kt while reading kt + 1 and sending for slice kt + 4 into that stage.
        auto turn = [&](auto curc, int kt, bool ld_last = false) __attribute__((always_inline)) {
            wait_vmcnt<16>();
            __syncthreads();
            step(curc, kt + 1, true, kt + 4, true, ld_last);
        };
        int kt = 0;
        for (; kt + (KTAIL ? 6 : 5) < nk; kt += 2) {    // (KTAIL: the load of the last slice is not part of the loop)
            turn(c0, kt);
            turn(c1, kt + 1);
        }
        // four or five slices are left; the last four load nothing
        auto tail4 = [&](auto ac, auto bc, int k0) __attribute__((always_inline)) {
            wait_vmcnt<16>();
            __syncthreads();
            step(ac, k0 + 1, true, 0, false);
            wait_vmcnt<8>();
            __syncthreads();
            step(bc, k0 + 2, true, 0, false);
            wait_vmcnt<0>();
            __syncthreads();
            step(ac, k0 + 3, true, 0, false);
            step(bc, 0, false, 0, false, false, true);
        };
        if (kt + 5 == nk) {
            turn(c0, kt, true);
            tail4(c1, c0, kt + 1);
        } else {
            if (KTAIL && kt + 6 == nk) {
                turn(c0, kt);
                turn(c1, kt + 1, true);
                kt += 2;
            }
            tail4(c0, c1, kt);
        }
    }
    if constexpr (PAIR) {
        bias_lane = bias_dt == MSAMP_DT_F32   ? __uint_as_float(bias_bits)
                    : bias_dt == MSAMP_DT_F16 ? f16_bits_to_float(static_cast<uint16_t>(bias_bits))
                                              : bf16_bits_to_float(static_cast<uint16_t>(bias_bits));
    }
    const uint32_t acc_token = PAIR ? vacc_fence() : acc_fence();
    __syncthreads();    // every wave is through with the stages, which the patches below reuse

    // ---- epilogue: the raw accumulators of a 16-row block go through a per-wave float32 patch; each lane then picks up
    // one 16-byte segment of an output row and applies the factor (bias, old output) with one rounding
    constexpr int kRowsPerPass = 64 / kSegs;       // 8 or 4
    constexpr int kFPitch = 64 * 4 + 16;           // bytes per patch row
    uint8_t* patch = smem + wave * (16 * kFPitch);
    const bool vec_ok = (NC % kElems == 0) && ((reinterpret_cast<uintptr_t>(D) & 15) == 0);
    const bool plain = !accumulate && bias == nullptr;
    const int prl = lane / kSegs;
    // (behind one branch: a choice for each value came out as eight far jumps behind the last product of every tile, 0.2 us)
    float bv[kElems] = {};
    if (bias != nullptr) {
#pragma unroll
        for (int e = 0; e < kElems; ++e)
            bv[e] = __int_as_float(__builtin_amdgcn_ds_bpermute((seg * kElems + e) * 4, __float_as_int(bias_lane)));
    }
    static_for<4>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        static_for<4>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            const v4f a = PAIR ? vacc_quad<i * 4 + j>(acc_token) : acc_quad<i * 4 + j>(acc_token);
            *reinterpret_cast<float4*>(patch + l16 * kFPitch + (j * 16 + g4 * 4) * 4) = make_float4(a[0], a[1], a[2], a[3]);
        });
        // (the patch is private to this wave and the LDS serves one wave's requests in order: no waits needed)
#pragma unroll
        for (int pass = 0; pass < 16 / kRowsPerPass; ++pass) {
            const int pr = pass * kRowsPerPass + prl;
            const int grow = row0 + wr * 64 + i * 16 + pr;
            const float* src = reinterpret_cast<const float*>(patch + pr * kFPitch + seg * kElems * 4);
            float r[kElems];
            const float4 a0 = *reinterpret_cast<const float4*>(src);
            r[0] = a0.x, r[1] = a0.y, r[2] = a0.z, r[3] = a0.w;
            if constexpr (kElems == 8) {
                const float4 a1 = *reinterpret_cast<const float4*>(src + 4);
                r[4] = a1.x, r[5] = a1.y, r[6] = a1.z, r[7] = a1.w;
            }
            if (grow >= NR || gcol >= NC) continue;
            OT* out = D + static_cast<size_t>(grow) * NC + gcol;
            if (vec_ok && gcol + kElems <= NC) {
                if (plain) {
#pragma unroll
                    for (int e = 0; e < kElems; ++e) r[e] = r[e] * alpha;
                } else {
                    float o[kElems];
#pragma unroll
                    for (int e = 0; e < kElems; ++e) o[e] = 0.0f;
                    if (accumulate) {
                        const uint4 old = load_out16(out);
                        if constexpr (kEsz == 4) {
                            o[0] = __uint_as_float(old.x), o[1] = __uint_as_float(old.y);
                            o[2] = __uint_as_float(old.z), o[3] = __uint_as_float(old.w);
                        } else {
                            In16<OT>::decode(old, o);
                        }
                    }
#pragma unroll
                    for (int e = 0; e < kElems; ++e) {
                        r[e] = fmaf(r[e], alpha, bv[e]);
                        if (accumulate) r[e] += o[e];
                    }
                }
                uint4 v;
                if constexpr (kEsz == 4) {
                    v = make_uint4(__float_as_uint(r[0]), __float_as_uint(r[1]), __float_as_uint(r[2]), __float_as_uint(r[3]));
                } else if constexpr (__is_same(OT, bf16_t)) {
                    v = make_uint4(pack_bf16(r[0], r[1]), pack_bf16(r[2], r[3]), pack_bf16(r[4], r[5]), pack_bf16(r[6], r[7]));
                } else {
                    v = make_uint4(pack_f16(r[0], r[1]), pack_f16(r[2], r[3]), pack_f16(r[4], r[5]), pack_f16(r[6], r[7]));
                }
                store_out16(out, v);
            } else {
                // rows that 16-byte accesses do not fit, or a segment that ends past the last column: one by one
#pragma unroll
                for (int e = 0; e < kElems; ++e) {
                    if (gcol + e < NC) {
                        if (plain) Elem<OT>::store(out + e, r[e] * alpha);
                        else store_out<OT>(out + e, fmaf(r[e], alpha, bv[e]), accumulate != 0);
                    }
                }
            }
        }
    });
}

template <int XF, int YF, typename OT, bool XT = false, bool YT = false>
__global__ __launch_bounds__(kGemmThreads) void fp8_gemm_dma128_kernel(const uint8_t* __restrict__ X, const uint8_t* __restrict__ Y,
                                                                        OT* __restrict__ D, int NR, int NC, int K,
                                                                        const float* __restrict__ x_scale_inv,
                                                                        const float* __restrict__ y_scale_inv, int accumulate,
                                                                        const void* __restrict__ bias, int bias_dt) {
    gemm_dma128<XF, YF, OT, XT, YT, false>(X, Y, D, NR, NC, K, x_scale_inv, y_scale_inv, accumulate, bias, bias_dt);
}
// the same for a ragged last slice of K
template <int XF, int YF, typename OT, bool XT = false, bool YT = false>
__global__ __launch_bounds__(kGemmThreads) void fp8_gemm_ragged128_kernel(const uint8_t* __restrict__ X, const uint8_t* __restrict__ Y,
                                                                           OT* __restrict__ D, int NR, int NC, int K,
                                                                           const float* __restrict__ x_scale_inv,
                                                                           const float* __restrict__ y_scale_inv, int accumulate,
                                                                           const void* __restrict__ bias, int bias_dt) {
    gemm_dma128<XF, YF, OT, XT, YT, true>(X, Y, D, NR, NC, K, x_scale_inv, y_scale_inv, accumulate, bias, bias_dt);
}

template <int XF, int YF, typename OT, bool XT, bool YT, bool KTAIL>
__global__ __launch_bounds__(kGemmThreads) __attribute__((amdgpu_num_vgpr(96))) void fp8_gemm_pair128_kernel(const uint8_t* __restrict__ X, const uint8_t* __restrict__ Y,
                                                                            OT* __restrict__ D, int NR, int NC, int K,
                                                                            const float* __restrict__ x_scale_inv,
                                                                            const float* __restrict__ y_scale_inv, int accumulate,
                                                                            const void* __restrict__ bias, int bias_dt) {
    gemm_dma128<XF, YF, OT, XT, YT, KTAIL, true>(X, Y, D, NR, NC, K, x_scale_inv, y_scale_inv, accumulate, bias, bias_dt);
}

template <int XF, int YF, typename OT, bool XT, bool YT, bool KTAIL>
static int launch_gemm_pair128_tail(const uint8_t* X, const uint8_t* Y, void* D, int NR, int NC, int K, const float* xs, const float* ys,
                                    int accumulate, const void* bias, int bias_dt, hipStream_t st) {
    constexpr int smem = kPairUnits * kPairUnit;
    static std::atomic<bool> configured{false};    // setting the attribute twice is harmless
    auto kern = fp8_gemm_pair128_kernel<XF, YF, OT, XT, YT, KTAIL>;
    if (!configured.load(std::memory_order_acquire)) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
        if (e != hipSuccess) return hip_fail(e, "hipFuncSetAttribute(fp8_gemm_pair128_kernel)");
        configured.store(true, std::memory_order_release);
    }
    const int tiles = ((NR + kSmallTile - 1) / kSmallTile) * ((NC + kSmallTile - 1) / kSmallTile);
    hipLaunchKernelGGL(kern, dim3(tiles), dim3(kGemmThreads), smem, st, X, Y, static_cast<OT*>(D), NR, NC, K, xs, ys, accumulate, bias,
                       bias_dt);
    MSAMP_CHECK_LAUNCH("fp8_gemm_pair128_kernel");
    return MSAMP_OK;
}

template <int XF, int YF, typename OT, bool XT = false, bool YT = false>
static int launch_gemm_pair128(const uint8_t* X, const uint8_t* Y, void* D, int NR, int NC, int K, const float* xs, const float* ys,
                               int accumulate, const void* bias, int bias_dt, hipStream_t st) {
    if (K % kBK) return launch_gemm_pair128_tail<XF, YF, OT, XT, YT, true>(X, Y, D, NR, NC, K, xs, ys, accumulate, bias, bias_dt, st);
    return launch_gemm_pair128_tail<XF, YF, OT, XT, YT, false>(X, Y, D, NR, NC, K, xs, ys, accumulate, bias, bias_dt, st);
}

template <int XF, int YF, typename OT, bool XT, bool YT, bool KTAIL>
static int launch_gemm_dma128_tail(const uint8_t* X, const uint8_t* Y, void* D, int NR, int NC, int K, const float* xs, const float* ys,
                              int accumulate, const void* bias, int bias_dt, hipStream_t st, int parts = 1) {
    constexpr int smem = kSmallStages * kSmallStage;
    static std::atomic<bool> configured{false};    // setting the attribute twice is harmless
    auto kern = KTAIL ? fp8_gemm_ragged128_kernel<XF, YF, OT, XT, YT> : fp8_gemm_dma128_kernel<XF, YF, OT, XT, YT>;
    if (!configured.load(std::memory_order_acquire)) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
        if (e != hipSuccess) return hip_fail(e, "hipFuncSetAttribute(fp8_gemm_dma128_kernel)");
        configured.store(true, std::memory_order_release);
    }
    const int tiles = ((NR + kSmallTile - 1) / kSmallTile) * ((NC + kSmallTile - 1) / kSmallTile);
    hipLaunchKernelGGL(kern, dim3(tiles, parts), dim3(kGemmThreads), smem, st, X, Y, static_cast<OT*>(D), NR, NC, K, xs, ys, accumulate,
                       bias, bias_dt);
    MSAMP_CHECK_LAUNCH("fp8_gemm_dma128_kernel");
    return MSAMP_OK;
}

template <int XF, int YF, typename OT, bool XT = false, bool YT = false>
static int launch_gemm_dma128(const uint8_t* X, const uint8_t* Y, void* D, int NR, int NC, int K, const float* xs, const float* ys,
                              int accumulate, const void* bias, int bias_dt, hipStream_t st) {
    if (K % kBK) return launch_gemm_dma128_tail<XF, YF, OT, XT, YT, true>(X, Y, D, NR, NC, K, xs, ys, accumulate, bias, bias_dt, st);
    return launch_gemm_dma128_tail<XF, YF, OT, XT, YT, false>(X, Y, D, NR, NC, K, xs, ys, accumulate, bias, bias_dt, st);
}

}    // namespace msamp
