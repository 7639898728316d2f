// What the C entry points of the FP8 GEMM hand to the kernels' translation units.
#pragma once

#include "common.cuh"

namespace msamp {

constexpr int kBK = 128;         // K bytes per LDS stage
constexpr int kDmaTile = 256;    // output tile edge of the direct-to-LDS kernel

struct QuantArgs {
    uint8_t* q;          // [NR][NC] FP8 codes
    float* scale;        // in: the fallback of the scale rule; out: the scale used
    float* amax;         // out: max |D|
    float* scale_inv;    // out: 1 / scale
    uint64_t* slots;     // kMaxSlots meeting slots and two post words
    float fp_max;
    int margin;
    int flags;
    uint32_t token;
    uint32_t spin_limit;
    uint32_t* error_word;    // sticky: set when a bounded wait runs out
    uint32_t* spec_words;    // speculative form: [0] running maximum, [1] ticket counter (both zero between calls), [2] out: 1 = cast again
    int walk_plus_one;       // every form of the kernel: 0 = the tile walk the built-in rule picks, 1..4 = walk 0..3 (see registered_walk)
};

// From one k-row of a K-major operand to the next: its row count, which the entry points want to be a multiple of 16, or in the
// calls for a linear layer, whose casts write them so, the next one.
__host__ __device__ inline int kmajor_pitch(int rows) { return (rows + 15) & ~15; }

// One product D[NR][NC] = X[NR][K] . Y[NC][K]^T * *xs * *ys.  xt / yt: that operand is handed over K-major.
// qa != nullptr: the output is cast on to FP8 in the same launch; D is not written, unless `qspec` asks for the
// speculative form, which stores D as usual and the codes of D times the scale in force next to it.
struct GemmCall {
    const uint8_t* X;
    const uint8_t* Y;
    void* D;
    int d_dtype;
    int NR, NC, K;
    const float* xs;
    const float* ys;
    int accumulate;
    const void* bias;
    int bias_dt;
    bool xt, yt;
    const QuantArgs* qa;
    hipStream_t st;
    bool qspec = false;
};

template <int XF, int YF>
int run_gemm_pair(const GemmCall& c);
// The other half of a pair's instantiations lives in a translation unit of its own (gemm_inst.hip built with
// -DMSAMP_GEMM_SECOND_UNIT), so that they compile side by side: the 256 x 256-tile kernel for a ragged last slice of K and the
// 128 x 128-tile kernels (all layouts and output types).
template <int XF, int YF>
int run_gemm_ragged(const GemmCall& c);
template <int XF, int YF>
int run_gemm_small(const GemmCall& c);
template <int XF, int YF>
int run_gemm_pair128(const GemmCall& c);
// A product in parts of K: which tile, and how many parts (1: not split).
struct KSplit {
    bool small_tiles;
    int parts;
};
// (Large tiles: both operands K-major.)  c.D is the float32 scratch of `parts` arrays that receives the parts' unscaled sums.
template <int XF, int YF>
int run_gemm_parts(const GemmCall& c, const KSplit& split);
// The size up to which 128 x 128 tiles are looked at, in 256 x 256 tiles (msamp_set_small_tile_limit).  Any other value than the
// default serves to compare the kernels: the paired form is off then (but for K-major operands with a single slice of K), and a
// negative one sends every row-major product to the generic kernel.
constexpr int kSmallTileLimit = 128;
int small_tile_limit();
// The tile walk registered for this problem of the 256 x 256-tile kernel (msamp_fp8_gemm_set_walk / _tune), or -1: bit 0 =
// groups of tile columns walked row by row instead of groups of tile rows, bit 1 = the XCD's patch of 32 tiles turned (4 of
// the grouped dimension x 8 of the walked one).  Any walk gives the same output bits: it only decides which workgroup
// takes which tile.  (Bit 2 is taken and means nothing: it asked for what every product does now.)
int registered_walk(int NR, int NC, int K, bool XT, bool YT);
// 128 x 128 tiles with the whole LDS to a workgroup: at least four slices of K; up to half the limit always (one small tile per
// compute unit with the default limit), up to the limit where K is long enough for the second round of small tiles to
// pay (measured: 128 large tiles level at K = 2048, 15 % ahead at 4096).
inline bool takes_small_tiles(int NR, int NC, int K) {
    const long big_tiles = static_cast<long>((NR + kDmaTile - 1) / kDmaTile) * ((NC + kDmaTile - 1) / kDmaTile);
    const int limit = small_tile_limit();
    return K > 3 * kBK && (big_tiles <= limit / 2 || (big_tiles <= limit && K >= 3072));
}

// 128 x 128 tiles with two workgroups to a compute unit (the rule and its figures: gemm.hip).
bool takes_paired_tiles(int NR, int NC, int K);

// msamp_fp8_gemm_kmajor for any K (a single slice of it is left to the paired tiles) and any m and n, with the operands' k-rows
// kmajor_pitch() apart.
int gemm_kmajor(const uint8_t* a, int a_type, const float* a_scale_inv, const uint8_t* b, int b_type, const float* b_scale_inv,
                int b_kmajor, void* d, int d_dtype, int m, int n, int k, int accumulate, hipStream_t st);
// A product in parts of K: the floats of scratch that it takes (0: it is better off whole), and the product (all operands and
// c.D 16-byte aligned).
size_t gemm_parts_scratch(int NR, int NC, int K, bool xt, bool yt);
int gemm_parts(int x_type, int y_type, const GemmCall& c, float* scratch, size_t n_floats);

// row offsets of the direct-to-LDS kernels are 32 bits
inline bool fits_offsets(int NR, int NC, int K) {
    return static_cast<unsigned long long>(NR) * K < (1ull << 32) && static_cast<unsigned long long>(NC) * K < (1ull << 32);
}

// Implemented with the cast kernels: q = FP8(d * *scale) over n elements, unless *redo is zero (then nothing is done).
int cast_again_if_flagged(const void* d, int d_dtype, size_t n, const float* scale, uint8_t* q, int q_type, const uint32_t* redo,
                          hipStream_t st);

extern template int run_gemm_pair<MSAMP_DT_E4M3, MSAMP_DT_E4M3>(const GemmCall&);
extern template int run_gemm_pair<MSAMP_DT_E4M3, MSAMP_DT_E5M2>(const GemmCall&);
extern template int run_gemm_pair<MSAMP_DT_E5M2, MSAMP_DT_E4M3>(const GemmCall&);
extern template int run_gemm_pair<MSAMP_DT_E5M2, MSAMP_DT_E5M2>(const GemmCall&);
extern template int run_gemm_ragged<MSAMP_DT_E4M3, MSAMP_DT_E4M3>(const GemmCall&);
extern template int run_gemm_small<MSAMP_DT_E4M3, MSAMP_DT_E4M3>(const GemmCall&);
extern template int run_gemm_pair128<MSAMP_DT_E4M3, MSAMP_DT_E4M3>(const GemmCall&);
extern template int run_gemm_parts<MSAMP_DT_E4M3, MSAMP_DT_E4M3>(const GemmCall&, const KSplit&);
extern template int run_gemm_ragged<MSAMP_DT_E4M3, MSAMP_DT_E5M2>(const GemmCall&);
extern template int run_gemm_small<MSAMP_DT_E4M3, MSAMP_DT_E5M2>(const GemmCall&);
extern template int run_gemm_pair128<MSAMP_DT_E4M3, MSAMP_DT_E5M2>(const GemmCall&);
extern template int run_gemm_parts<MSAMP_DT_E4M3, MSAMP_DT_E5M2>(const GemmCall&, const KSplit&);
extern template int run_gemm_ragged<MSAMP_DT_E5M2, MSAMP_DT_E4M3>(const GemmCall&);
extern template int run_gemm_small<MSAMP_DT_E5M2, MSAMP_DT_E4M3>(const GemmCall&);
extern template int run_gemm_pair128<MSAMP_DT_E5M2, MSAMP_DT_E4M3>(const GemmCall&);
extern template int run_gemm_parts<MSAMP_DT_E5M2, MSAMP_DT_E4M3>(const GemmCall&, const KSplit&);
extern template int run_gemm_ragged<MSAMP_DT_E5M2, MSAMP_DT_E5M2>(const GemmCall&);
extern template int run_gemm_small<MSAMP_DT_E5M2, MSAMP_DT_E5M2>(const GemmCall&);
extern template int run_gemm_pair128<MSAMP_DT_E5M2, MSAMP_DT_E5M2>(const GemmCall&);
extern template int run_gemm_parts<MSAMP_DT_E5M2, MSAMP_DT_E5M2>(const GemmCall&, const KSplit&);

}    // namespace msamp
