// The two directions of an FP8Linear layer as one call each: the casts and products of the entry points below, enqueued from
// here.  A small layer is bound by the host, not by these kernels, and most of the host's time went into reaching them one
// library call at a time (allocation, pointers, stream and argument conversion of each).  Host time by single calls and by
// these, with the same launches: forward of 16 x 512 -> 512 61 -> 33 us, training step of two 1024-wide blocks over 2048 tokens
// 1522 -> 1137 us; by now some of the launches are one (the casts beside the gate, cast.hip), that forward 27 us.
// Widths that are no multiples of 16: the products read 16 bytes at a time, so the codes were copied into padded rows, and x, dy and
// the weight transposed (byte by byte where a length is odd) for products that could not read them in place.  The casts here leave
// their codes in rows a multiple of 16 apart, zeros behind them, which all three products read as they lie; what a product writes is
// dense.  Forward and backward, bfloat16, us: 145 x 16744 -> 12064 926 -> 595, 861 x 15616 -> 16935 with a bias 1644 -> 1132,
// 597 x 9654 -> 256 205 -> 91 (host), two of 8949 x 4480 -> 2157 1129 -> 773; forward alone 79 x 936 -> 840 70 -> 27.
#include "common.cuh"
#include "gemm_call.h"
#include "linear_call.h"

#include <algorithm>

namespace msamp {

// ---- a few tokens through a layer nobody differentiates ---------------------------------------------------------------
// y[tokens][d_out] = x . fp8(w)^T, the weight read in its scaled 16- or 32-bit form and quantized on its way to the matrix pipes,
// with the codes msamp_cast_scaled_to_fp8 gives: it is read once (2 bytes an element), where the cast and the product move 4.
// Bound by that read and by the codes of x, which every workgroup reads again out of the L2: 48 tokens through 4096 -> 12288 are
// 2.75 M requests of the L1s to it, 0.86 M of which miss (0.79 M are the weight's lines).  A workgroup takes 16 rows of w and all
// tokens; its wavefronts take the 128-wide slices of K in turn, and their float32 sums meet in LDS in a fixed order.
// A load of w covers whole rows of the slice (16-bit: four of 256 bytes): it is read as it would be for a matrix instruction, 16 rows
// to a load, at 0.85 of that speed (100 MB by nothing but such loads: 19.0 us, 16.2).  The codes go through 2 KiB of LDS that is the
// wavefront's own, where the operand's registers find them, and the loads of the next slice are on their way as soon as the codes
// are made: into the same registers, which leaves room for another workgroup.  Inside a slice the k of an MFMA's operand bytes are
// dealt out anew, alike for both operands: lane group g holds k = 16 g .. +15 and 64 + 16 g .. +15.  x comes in the order of the
// operand registers from its cast (few_cast_fragments): read row by row, 16 rows a long power of two apart, it cost as much as w
// (48 tokens 7 us more).  Both casts and the product together, replayed from a graph, us, with the weight cast to memory and the
// product after it | with the weight read in the operand's order and quantized one by one | now, for 4096 -> 12288: 16 tokens
// 47.1 | 29.4 | 23.0, 48 47.5 | 34.4 | 28.5, 64 48.3 | 37.8 | 31.8; 64 x 8192 -> 8192 64.0 | 48.5 | 40.3, 64 x 16384 -> 4096 82.1 | 52.3 | 43.8,
// 64 x 2048 -> 16384 33.1 | 25.9 | 21.5, 16 x 512 -> 512 14.3 | 6.9 | 6.7 (launches).  Where d_out gives a few workgroups and K is long,
// the product in parts of K that a forward with gradients takes was ahead by a little: 64 x 16384 -> 256 32.9 | 25.0, 23.1 in parts.
__device__ __forceinline__ float few_bias(const void* bias, int dt, int i) {
    if (dt == MSAMP_DT_F32) return static_cast<const float*>(bias)[i];
    if (dt == MSAMP_DT_F16) return f16_bits_to_float(static_cast<const uint16_t*>(bias)[i]);
    return bf16_bits_to_float(static_cast<const uint16_t*>(bias)[i]);
}
typedef int few_v8i __attribute__((ext_vector_type(8)));
typedef short few_v2s __attribute__((ext_vector_type(2)));
// Four 16-bit weights times a power of two to E4M3 codes, by one instruction a pair where quant4 takes ten with the widening: the same
// codes, but 0x7f (NaN) for whatever lies beyond the format, which quant4 saturates (all patterns of both types at 61 scales).  A slice
// with such a code is quantized again by quant4, and so is every slice whose factor is no power of two.  Alone it gave 1 us of 30.
template <typename WT>
__device__ __forceinline__ uint32_t few_codes4(uint32_t lo, uint32_t hi, float inv_scale) {
    few_v2s q = {0, 0};
    if constexpr (__is_same(WT, bf16_t)) {
        typedef __bf16 v2b __attribute__((ext_vector_type(2)));
        q = __builtin_amdgcn_cvt_scalef32_pk_fp8_bf16(q, __builtin_bit_cast(v2b, lo), inv_scale, false);
        q = __builtin_amdgcn_cvt_scalef32_pk_fp8_bf16(q, __builtin_bit_cast(v2b, hi), inv_scale, true);
    } else {
        typedef _Float16 v2h __attribute__((ext_vector_type(2)));
        q = __builtin_amdgcn_cvt_scalef32_pk_fp8_f16(q, __builtin_bit_cast(v2h, lo), inv_scale, false);
        q = __builtin_amdgcn_cvt_scalef32_pk_fp8_f16(q, __builtin_bit_cast(v2h, hi), inv_scale, true);
    }
    return __builtin_bit_cast(uint32_t, q);
}
typedef float few_v4f __attribute__((ext_vector_type(4)));

template <typename WT, typename OT, int MB, bool STREAM>
__global__ __launch_bounds__(512) void few_tokens_kernel(const WT* __restrict__ w, const uint8_t* __restrict__ x, OT* __restrict__ y,
                                                          int tokens, int d_out, int K, const float* __restrict__ w_amax,
                                                          const float* __restrict__ w_scale_inv, const float* __restrict__ x_scale_inv,
                                                          const void* __restrict__ bias, int bias_dt) {
    extern __shared__ __attribute__((aligned(16))) float4 few_part[];    // [wavefronts][MB][64]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    const int l16 = lane & 15, g4 = lane >> 4;
    const float s_new = scale_rule(*w_amax, 1.0f, 448.0f, 0);
    const float s = s_new * *w_scale_inv;
    const uint32_t s_exp = __float_as_uint(s) >> 23;
    const bool pow2 = sizeof(WT) == 2 && (__float_as_uint(s) & 0x7fffffu) == 0u && s_exp >= 127u - 30u && s_exp <= 127u + 30u;
    const float s_inv = 1.0f / s;
    const uint8_t* xp = x + lane * 16;
    const int slices = (K + 127) / 128;
    few_v4f acc[MB];
#pragma unroll
    for (int b = 0; b < MB; ++b) acc[b] = few_v4f{0.0f, 0.0f, 0.0f, 0.0f};

    constexpr int kPer = 16 / static_cast<int>(sizeof(WT));    // weights of a 16-byte load
    constexpr int kAcross = 128 / kPer;                        // lanes to a row of a slice
    constexpr int kRows = 64 / kAcross, kLoads = 16 / kRows;   // rows of a load, loads of a slice
    const int k_lane = lane % kAcross * kPer, r_lane = lane / kAcross;
    struct Weights { uint4 v[kLoads]; };
    // (rows past the end are clamped: their products land in outputs that are not stored)
    const WT* wp[kLoads];
#pragma unroll
    for (int j = 0; j < kLoads; ++j) wp[j] = w + static_cast<size_t>(min(static_cast<int>(blockIdx.x) * 16 + j * kRows + r_lane, d_out - 1)) * K;
    // (K is a multiple of 16: the k of a load lie inside together or not at all.  A load past the end reads the row's last 16 bytes
    // instead: loads that may or may not be made can't be counted, and the product then waits for the next slice's weights)
    auto fetch = [&](int kt, Weights& f) __attribute__((always_inline)) {
        const int k = min(kt * 128 + k_lane, K - kPer);
#pragma unroll
        for (int j = 0; j < kLoads; ++j) f.v[j] = ld16(wp[j] + k, STREAM);
    };
    uint8_t* const codes = reinterpret_cast<uint8_t*>(few_part + waves * MB * 64) + wave * 2048;    // of a slice, 128 bytes a row
    // where the codes of load j go: 16-byte chunk c of row r lies at c ^ (r % 8)
    auto code_at = [&](int j) __attribute__((always_inline)) {
        const int r = j * kRows + r_lane;
        return codes + r * 128 + (((k_lane >> 4) ^ (r & 7)) << 4) + (k_lane & 15);
    };
    Weights f = {};
    if (wave < slices) fetch(wave, f);
    for (int kt = wave; kt < slices; kt += waves) {
        uint4 xr[MB][2];
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int h = 0; h < 2; ++h) xr[b][h] = *reinterpret_cast<const uint4*>(xp + ((static_cast<size_t>(kt) * MB + b) * 2 + h) * 1024);
        const bool in = kt * 128 + k_lane < K;    // (the ragged last slice: what was not loaded is zero)
        bool done = false;
        if constexpr (sizeof(WT) == 2) {
            if (pow2) {
                uint2 c[kLoads];
                uint32_t odd = 0u;    // high bits: a code of all ones below its sign
#pragma unroll
                for (int j = 0; j < kLoads; ++j) {
                    c[j] = make_uint2(few_codes4<WT>(f.v[j].x, f.v[j].y, s_inv), few_codes4<WT>(f.v[j].z, f.v[j].w, s_inv));
                    if (!in) c[j] = make_uint2(0u, 0u);
                    odd |= ((c[j].x & 0x7f7f7f7fu) + 0x01010101u) | ((c[j].y & 0x7f7f7f7fu) + 0x01010101u);
                    *reinterpret_cast<uint2*>(code_at(j)) = c[j];
                }
                done = !__any((odd & 0x80808080u) != 0u);
            }
        }
        if (!done) {
#pragma unroll
            for (int j = 0; j < kLoads; ++j) {
                float v[kPer];
                In16<WT>::decode(f.v[j], v);
#pragma unroll
                for (int e = 0; e < kPer / 4; ++e) {
                    const uint32_t c = quant4<MSAMP_DT_E4M3>(v[4 * e] * s, v[4 * e + 1] * s, v[4 * e + 2] * s, v[4 * e + 3] * s);
                    *reinterpret_cast<uint32_t*>(code_at(j) + 4 * e) = in ? c : 0u;
                }
            }
        }
        fetch(kt + waves, f);
        // (the rows are this wavefront's own and the LDS serves its requests in order: only the compiler has to keep them so)
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
        few_v8i a;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint4 c = *reinterpret_cast<const uint4*>(codes + l16 * 128 + (((g4 + 4 * h) ^ (l16 & 7)) << 4));
            a[h * 4] = c.x, a[h * 4 + 1] = c.y, a[h * 4 + 2] = c.z, a[h * 4 + 3] = c.w;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");    // (and the next slice's codes behind these reads)
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int b = 0; b < MB; ++b) {
            few_v8i bx;
#pragma unroll
            for (int h = 0; h < 2; ++h) bx[h * 4] = xr[b][h].x, bx[h * 4 + 1] = xr[b][h].y, bx[h * 4 + 2] = xr[b][h].z, bx[h * 4 + 3] = xr[b][h].w;
            acc[b] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, bx, acc[b], 0, 0, 0, 0, 0, 0);
        }
    }
#pragma unroll
    for (int b = 0; b < MB; ++b) few_part[(wave * MB + b) * 64 + lane] = make_float4(acc[b][0], acc[b][1], acc[b][2], acc[b][3]);
    __syncthreads();

    // a lane of a block of tokens has four consecutive outputs of one token
    const float alpha = *x_scale_inv * (1.0f / s_new);
    const bool whole = d_out % 4 == 0;
    for (int i = threadIdx.x; i < MB * 64; i += blockDim.x) {
        float4 t = few_part[i];
        for (int v = 1; v < waves; ++v) {
            const float4 u = few_part[v * MB * 64 + i];
            t.x += u.x, t.y += u.y, t.z += u.z, t.w += u.w;
        }
        const int token = i / 64 * 16 + (i & 15), col = blockIdx.x * 16 + ((i & 63) >> 4) * 4;
        if (token >= tokens) continue;
        const float f[4] = {t.x, t.y, t.z, t.w};
        struct __attribute__((aligned(4 * sizeof(OT)))) Four { OT v[4]; };
        Four o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (bias != nullptr) Elem<OT>::store(&o.v[e], fmaf(f[e], alpha, col + e < d_out ? few_bias(bias, bias_dt, col + e) : 0.0f));
            else Elem<OT>::store(&o.v[e], f[e] * alpha);
        }
        OT* out = y + static_cast<size_t>(token) * d_out + col;
        if (whole) {
            if (col < d_out) *reinterpret_cast<Four*>(out) = o;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (col + e < d_out) out[e] = o.v[e];
        }
    }
}

template <typename WT, typename OT, int MB>
static int launch_few_tokens(const msamp_linear_forward_args& a, hipStream_t st) {
    const int tokens = static_cast<int>(a.tokens), d_out = static_cast<int>(a.d_out), K = static_cast<int>(a.d_in);
    // Up to two workgroups of eight wavefronts fit a CU, and what no longer fits at once begins a round of its own: beyond two a CU
    // (here 512) they are of four wavefronts, five a CU.  us with eight and four: 48 x 4096 -> 12288 33.3, 28.5, 64 x 4096 -> 11008 33.1, 28.0,
    // 64 x 2048 -> 16384 23.0, 21.5, 48 x 4096 -> 32000 66.4, 64.3; up to 512, 48 x 1040 -> 6000 11.1, 10.9, 64 x 4096 -> 8192 20.9, 21.0,
    // 16 x 8192 -> 8192 30.1, 32.6, 32 x 11008 -> 4096 24.9, 27.1.  Just beyond the line either is ahead somewhere: 16 x 4096 -> 8208 18.1, 16.7,
    // 48 tokens 19.5, 20.8, 16 x 8192 -> 8208 32.0, 34.9, 16 x 16384 -> 8208 67.6, 61.6.
    const int workgroups = (d_out + 15) / 16, waves = std::min(workgroups > 2 * cu_count() ? 4 : 8, (K + 127) / 128);
    const bool stream = static_cast<size_t>(d_out) * K * sizeof(WT) >= kStreamBytes;
    const auto kernel = stream ? few_tokens_kernel<WT, OT, MB, true> : few_tokens_kernel<WT, OT, MB, false>;
    hipLaunchKernelGGL(kernel, dim3(workgroups), dim3(64 * waves), waves * (MB * 1024 + 2048), st,
                       static_cast<const WT*>(a.w), a.x_codes, static_cast<OT*>(a.y), tokens, d_out, K, a.w_amax, a.w_scale_inv,
                       a.x_scale_inv, a.bias, static_cast<int>(a.bias_dtype));
    MSAMP_CHECK_LAUNCH("few_tokens_kernel");
    return MSAMP_OK;
}

template <typename WT, typename OT>
static int few_tokens_blocks(const msamp_linear_forward_args& a, hipStream_t st) {
    switch ((a.tokens + 15) / 16) {
        case 1: return launch_few_tokens<WT, OT, 1>(a, st);
        case 2: return launch_few_tokens<WT, OT, 2>(a, st);
        case 3: return launch_few_tokens<WT, OT, 3>(a, st);
        default: return launch_few_tokens<WT, OT, 4>(a, st);
    }
}

template <typename WT>
static int few_tokens_out(const msamp_linear_forward_args& a, hipStream_t st) {
    if (a.y_dtype == MSAMP_DT_F32) return few_tokens_blocks<WT, float>(a, st);
    if (a.y_dtype == MSAMP_DT_F16) return few_tokens_blocks<WT, f16_t>(a, st);
    return few_tokens_blocks<WT, bf16_t>(a, st);
}

static int few_tokens(const msamp_linear_forward_args& a, hipStream_t st) {
    if (a.w_dtype == MSAMP_DT_F32) return few_tokens_out<float>(a, st);
    if (a.w_dtype == MSAMP_DT_F16) return few_tokens_out<f16_t>(a, st);
    return few_tokens_out<bf16_t>(a, st);
}

static size_t round_up(size_t n) { return (n + 255) / 256 * 256; }

// where a backward call's parts of its scratch begin (the two products take the same room for parts of K one after the other)
struct BackwardScratch {
    size_t sums, parts, n_dx_parts, n_parts, end;
};

static int backward_scratch(int tokens, int d_in, int d_out, int dy_dtype, int out_dtype, bool dx, bool wgrad, bool bias, BackwardScratch* s) {
    s->sums = wgrad ? round_up(static_cast<size_t>(d_out) * d_in * hp_size(out_dtype)) : 0;    // (the product comes first)
    size_t words = 0;
    if (bias) {
        const int rc = msamp_cast_colsum_scratch(tokens, d_out, dy_dtype, &words);
        if (rc != MSAMP_OK) return rc;
    }
    s->parts = s->sums + round_up(words * sizeof(float));
    s->n_dx_parts = dx ? gemm_parts_scratch(tokens, d_in, kmajor_pitch(d_out), false, true) : 0;
    s->n_parts = wgrad ? gemm_parts_scratch(d_out, d_in, tokens, true, true) : 0;
    s->end = s->parts + std::max(s->n_dx_parts, s->n_parts) * sizeof(float);
    return MSAMP_OK;
}

static bool dims_ok(int64_t tokens, int64_t d_in, int64_t d_out) {
    constexpr int64_t kLimit = (1ll << 31) - 16;    // (rounded up to a multiple of 16 they are still an int)
    return tokens > 0 && d_in > 0 && d_out > 0 && tokens < kLimit && d_in < kLimit && d_out < kLimit;
}

}    // namespace msamp

using namespace msamp;

extern "C" int msamp_linear_forward(const msamp_linear_forward_args* a, msamp_stream_t stream) {
    MSAMP_REQUIRE(a != nullptr, MSAMP_ERR_NULL, "msamp_linear_forward: null arguments");
    MSAMP_REQUIRE(dims_ok(a->tokens, a->d_in, a->d_out), MSAMP_ERR_SHAPE, "msamp_linear_forward: %lld x %lld -> %lld",
                  static_cast<long long>(a->tokens), static_cast<long long>(a->d_in), static_cast<long long>(a->d_out));
    MSAMP_REQUIRE(a->w_codes == nullptr || a->w_meta, MSAMP_ERR_NULL, "msamp_linear_forward: null w_meta");
    const int x_dtype = static_cast<int>(a->x_dtype), w_dtype = static_cast<int>(a->w_dtype), y_dtype = static_cast<int>(a->y_dtype);
    if (a->w_codes == nullptr) {
        // (refused here and not behind the cast, which changes the input meta)
        MSAMP_REQUIRE(is_hp(w_dtype) && is_hp(y_dtype) && (a->bias == nullptr || is_hp(static_cast<int>(a->bias_dtype))), MSAMP_ERR_DTYPE,
                      "msamp_linear_forward: dtypes %d -> %d", w_dtype, y_dtype);
        MSAMP_REQUIRE(a->tokens <= MSAMP_FEW_TOKENS && a->d_in % 16 == 0, MSAMP_ERR_SHAPE,
                      "msamp_linear_forward: %lld x %lld without codes of w", static_cast<long long>(a->tokens), static_cast<long long>(a->d_in));
        MSAMP_REQUIRE(a->w && a->y && a->w_amax && a->w_scale_inv, MSAMP_ERR_NULL, "msamp_linear_forward: null pointer");
        MSAMP_REQUIRE(aligned(a->w, 16) && aligned(a->x_codes, 16) && aligned(a->y, 16), MSAMP_ERR_ALIGNMENT,
                      "msamp_linear_forward: w, x_codes and y must be 16-byte aligned");
    }
    if (a->w_codes == nullptr) {
        const int rc = few_cast_fragments(a->x, x_dtype, static_cast<int>(a->tokens), static_cast<int>(a->d_in), a->x_scale, a->x_amax,
                                          a->x_scale_inv, a->x_codes, static_cast<int>(a->flags), a->x_counter,
                                          static_cast<int>(a->x_window), a->workspace, static_cast<hipStream_t>(stream));
        return rc != MSAMP_OK ? rc : few_tokens(*a, static_cast<hipStream_t>(stream));
    }
    const int rc = cast_linear_inputs(*a, static_cast<hipStream_t>(stream));
    if (rc != MSAMP_OK) return rc;
    const int tokens = static_cast<int>(a->tokens), d_out = static_cast<int>(a->d_out), K = kmajor_pitch(static_cast<int>(a->d_in));
    const int bias_dtype = static_cast<int>(a->bias_dtype);
    const size_t n_parts = a->scratch_bytes > 0 ? gemm_parts_scratch(tokens, d_out, K, false, false) : 0;
    if (n_parts == 0 || static_cast<size_t>(a->scratch_bytes) < n_parts * sizeof(float) || !a->scratch || !is_hp(y_dtype) ||
        (a->bias && !is_hp(bias_dtype)) || !aligned(a->y, 16) || !aligned(a->w_codes, 16) || !aligned(a->x_codes, 16))
        return msamp_fp8_gemm(a->w_codes, MSAMP_DT_E4M3, a->w_meta + 1, a->x_codes, MSAMP_DT_E4M3, a->x_scale_inv, a->y, y_dtype, d_out,
                              tokens, K, 0, a->bias, bias_dtype, stream);
    MSAMP_REQUIRE(a->y, MSAMP_ERR_NULL, "msamp_linear_forward: null pointer");
    const GemmCall c = {a->x_codes, a->w_codes, a->y, y_dtype, tokens, d_out, K, a->x_scale_inv, a->w_meta + 1, 0, a->bias, bias_dtype,
                        false, false, nullptr, static_cast<hipStream_t>(stream)};
    return gemm_parts(MSAMP_DT_E4M3, MSAMP_DT_E4M3, c, static_cast<float*>(a->scratch), n_parts);
}

extern "C" int msamp_linear_forward_scratch(int tokens, int d_in, int d_out, size_t* bytes) {
    MSAMP_REQUIRE(dims_ok(tokens, d_in, d_out), MSAMP_ERR_SHAPE, "msamp_linear_forward_scratch: %d x %d -> %d", tokens, d_in, d_out);
    MSAMP_REQUIRE(bytes != nullptr, MSAMP_ERR_NULL, "msamp_linear_forward_scratch: null pointer");
    *bytes = gemm_parts_scratch(tokens, d_out, kmajor_pitch(d_in), false, false) * sizeof(float);
    return MSAMP_OK;
}

extern "C" int msamp_linear_backward_scratch(int tokens, int d_in, int d_out, int dy_dtype, int out_dtype, int want_dx, int want_wgrad,
                                             int want_bias, size_t* bytes, size_t* least) {
    MSAMP_REQUIRE(dims_ok(tokens, d_in, d_out), MSAMP_ERR_SHAPE, "msamp_linear_backward_scratch: %d x %d -> %d", tokens, d_in, d_out);
    MSAMP_REQUIRE(is_hp(dy_dtype) && is_hp(out_dtype), MSAMP_ERR_DTYPE, "msamp_linear_backward_scratch: dtypes %d, %d", dy_dtype, out_dtype);
    MSAMP_REQUIRE(bytes && least, MSAMP_ERR_NULL, "msamp_linear_backward_scratch: null pointer");
    BackwardScratch s;
    const int rc = backward_scratch(tokens, d_in, d_out, dy_dtype, out_dtype, want_dx != 0, want_wgrad != 0, want_bias != 0, &s);
    if (rc != MSAMP_OK) return rc;
    *bytes = s.end, *least = s.parts;
    return MSAMP_OK;
}

extern "C" int msamp_linear_backward(const msamp_linear_backward_args* a, msamp_stream_t stream) {
    MSAMP_REQUIRE(a != nullptr, MSAMP_ERR_NULL, "msamp_linear_backward: null arguments");
    MSAMP_REQUIRE(dims_ok(a->tokens, a->d_in, a->d_out), MSAMP_ERR_SHAPE, "msamp_linear_backward: %lld x %lld -> %lld",
                  static_cast<long long>(a->tokens), static_cast<long long>(a->d_in), static_cast<long long>(a->d_out));
    const int tokens = static_cast<int>(a->tokens), d_in = static_cast<int>(a->d_in), d_out = static_cast<int>(a->d_out);
    const int dy_dtype = static_cast<int>(a->dy_dtype), out_dtype = static_cast<int>(a->out_dtype), flags = static_cast<int>(a->flags);
    MSAMP_REQUIRE(is_hp(dy_dtype) && is_hp(out_dtype), MSAMP_ERR_DTYPE, "msamp_linear_backward: dtypes %d, %d", dy_dtype, out_dtype);
    const bool wgrad = a->wq != nullptr, bias = a->bias_sum != nullptr, accumulate = a->old_codes != nullptr;
    BackwardScratch s;
    int rc = backward_scratch(tokens, d_in, d_out, dy_dtype, out_dtype, a->dx != nullptr, wgrad, bias, &s);
    if (rc != MSAMP_OK) return rc;
    MSAMP_REQUIRE(s.parts == 0 || (a->scratch && aligned(a->scratch, 16) && a->scratch_bytes >= static_cast<int64_t>(s.parts)),
                  MSAMP_ERR_WORKSPACE, "msamp_linear_backward: scratch of %lld bytes", static_cast<long long>(a->scratch_bytes));
    hipStream_t st = static_cast<hipStream_t>(stream);
    uint8_t* codes = a->dy_codes;
    uint8_t* product = static_cast<uint8_t*>(a->scratch);
    rc = cast_output_gradient(*a, product, reinterpret_cast<float*>(product + s.sums), st);
    if (rc != MSAMP_OK) return rc;
    // (the scratch may be without the room for parts of K)
    const bool room = a->scratch != nullptr && a->scratch_bytes >= static_cast<int64_t>(s.end);
    float* parts = reinterpret_cast<float*>(product + s.parts);
    if (a->dx != nullptr) {
        const int K = kmajor_pitch(d_out);
        if (s.n_dx_parts != 0 && room && a->w_codes && a->w_scale_inv && aligned(a->dx, 16)) {
            const GemmCall c = {codes, a->w_codes, a->dx, out_dtype, tokens, d_in, K, a->g_scale_inv, a->w_scale_inv, 0, nullptr, MSAMP_DT_F32,
                                false, true, nullptr, st};
            rc = gemm_parts(MSAMP_DT_E5M2, MSAMP_DT_E4M3, c, parts, s.n_dx_parts);
        } else {
            rc = gemm_kmajor(a->w_codes, MSAMP_DT_E4M3, a->w_scale_inv, codes, MSAMP_DT_E5M2, a->g_scale_inv, 0, a->dx, out_dtype, d_in,
                             tokens, K, 0, st);
        }
        if (rc != MSAMP_OK) return rc;
    }
    if (!wgrad) return MSAMP_OK;
    const size_t n = static_cast<size_t>(d_out) * d_in;
    if (s.n_parts != 0 && room && a->x_codes && a->x_scale_inv) {
        const GemmCall c = {codes, a->x_codes, product, out_dtype, d_out, d_in, tokens, a->g_scale_inv, a->x_scale_inv, accumulate, nullptr,
                            MSAMP_DT_F32, true, true, nullptr, st};
        rc = gemm_parts(MSAMP_DT_E5M2, MSAMP_DT_E4M3, c, parts, s.n_parts);
    } else {
        rc = gemm_kmajor(a->x_codes, MSAMP_DT_E4M3, a->x_scale_inv, codes, MSAMP_DT_E5M2, a->g_scale_inv, 1, product, out_dtype, d_in, d_out,
                         tokens, accumulate, st);
    }
    if (rc != MSAMP_OK) return rc;
    return msamp_cast_to_fp8_intime(product, out_dtype, n, a->q_scale, a->q_amax, a->q_scale_inv, a->wq, MSAMP_DT_E4M3, 0,
                                    flags | MSAMP_FLAG_NAN_TO_INF, a->workspace, stream);
}
