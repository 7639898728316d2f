// The two directions of an FP8Linear layer as one call each: the casts and products of the entry points below, enqueued from
// here.  A small layer is bound by the host, not by these kernels, and most of the host's time went into reaching them one
// library call at a time (allocation, pointers, stream and argument conversion of each).  Host time by single calls and by
// these, the same launches: forward of 16 x 512 -> 512 61 -> 33 us, training step of two 1024-wide blocks over 2048 tokens
// 1522 -> 1137 us.
#include "common.cuh"
#include "gemm_call.h"


namespace msamp {

static size_t round_up(size_t n) { return (n + 255) / 256 * 256; }

// where a backward call's parts of its scratch begin
struct BackwardScratch {
    size_t sums, parts, n_parts, end;
};

static int backward_scratch(int tokens, int d_in, int d_out, int dy_dtype, int out_dtype, bool wgrad, bool bias, BackwardScratch* s) {
    s->sums = wgrad ? round_up(static_cast<size_t>(d_out) * d_in * hp_size(out_dtype)) : 0;    // (the product comes first)
    size_t words = 0;
    if (bias) {
        const int rc = msamp_cast_colsum_scratch(tokens, d_out, dy_dtype, &words);
        if (rc != MSAMP_OK) return rc;
    }
    s->parts = s->sums + round_up(words * sizeof(float));
    s->n_parts = 0;
    if (wgrad) {
        const int rc = msamp_fp8_gemm_ksplit_scratch(d_in, d_out, tokens, &s->n_parts);
        if (rc != MSAMP_OK) return rc;
    }
    s->end = s->parts + s->n_parts * sizeof(float);
    return MSAMP_OK;
}

static bool dims_ok(int64_t tokens, int64_t d_in, int64_t d_out) {
    return tokens > 0 && d_in > 0 && d_out > 0 && tokens < (1ll << 31) && d_in < (1ll << 31) && d_out < (1ll << 31);
}

}    // namespace msamp

using namespace msamp;

extern "C" int msamp_linear_forward(const msamp_linear_forward_args* a, msamp_stream_t stream) {
    MSAMP_REQUIRE(a != nullptr, MSAMP_ERR_NULL, "msamp_linear_forward: null arguments");
    MSAMP_REQUIRE(dims_ok(a->tokens, a->d_in, a->d_out), MSAMP_ERR_SHAPE, "msamp_linear_forward: %lld x %lld -> %lld",
                  static_cast<long long>(a->tokens), static_cast<long long>(a->d_in), static_cast<long long>(a->d_out));
    MSAMP_REQUIRE(a->w_meta, MSAMP_ERR_NULL, "msamp_linear_forward: null w_meta");
    const size_t nx = static_cast<size_t>(a->tokens) * a->d_in, nw = static_cast<size_t>(a->d_out) * a->d_in;
    const int x_dtype = static_cast<int>(a->x_dtype), w_dtype = static_cast<int>(a->w_dtype), y_dtype = static_cast<int>(a->y_dtype);
    int rc = msamp_cast_to_fp8_gated(a->x, x_dtype, nx, a->x_scale, a->x_amax, a->x_scale_inv, a->x_codes, MSAMP_DT_E4M3, 0,
                                     static_cast<int>(a->flags), a->x_counter, static_cast<int>(a->x_window), a->workspace, stream);
    if (rc != MSAMP_OK) return rc;
    float* meta = a->w_meta;
    rc = msamp_cast_scaled_to_fp8(a->w, w_dtype, nw, a->w_amax, a->w_scale_inv, meta, meta + 1, meta + 3, static_cast<int>(a->w_window),
                                  reinterpret_cast<int32_t*>(meta + 2), a->w_codes, MSAMP_DT_E4M3, 0, stream);
    if (rc != MSAMP_OK) return rc;
    return msamp_fp8_gemm(a->w_codes, MSAMP_DT_E4M3, meta + 1, a->x_codes, MSAMP_DT_E4M3, a->x_scale_inv, a->y, y_dtype,
                          static_cast<int>(a->d_out), static_cast<int>(a->tokens), static_cast<int>(a->d_in), 0, a->bias,
                          static_cast<int>(a->bias_dtype), stream);
}

extern "C" int msamp_linear_backward_scratch(int tokens, int d_in, int d_out, int dy_dtype, int out_dtype, int want_wgrad, int want_bias,
                                             size_t* bytes, size_t* least) {
    MSAMP_REQUIRE(dims_ok(tokens, d_in, d_out), MSAMP_ERR_SHAPE, "msamp_linear_backward_scratch: %d x %d -> %d", tokens, d_in, d_out);
    MSAMP_REQUIRE(is_hp(dy_dtype) && is_hp(out_dtype), MSAMP_ERR_DTYPE, "msamp_linear_backward_scratch: dtypes %d, %d", dy_dtype, out_dtype);
    MSAMP_REQUIRE(bytes && least, MSAMP_ERR_NULL, "msamp_linear_backward_scratch: null pointer");
    BackwardScratch s;
    const int rc = backward_scratch(tokens, d_in, d_out, dy_dtype, out_dtype, want_wgrad != 0, want_bias != 0, &s);
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
    int rc = backward_scratch(tokens, d_in, d_out, dy_dtype, out_dtype, wgrad, bias, &s);
    if (rc != MSAMP_OK) return rc;
    MSAMP_REQUIRE(s.parts == 0 || (a->scratch && aligned(a->scratch, 16) && a->scratch_bytes >= static_cast<int64_t>(s.parts)),
                  MSAMP_ERR_WORKSPACE, "msamp_linear_backward: scratch of %lld bytes", static_cast<long long>(a->scratch_bytes));
    hipStream_t st = static_cast<hipStream_t>(stream);
    uint8_t* codes = a->dy_codes;
    uint8_t* product = static_cast<uint8_t*>(a->scratch);
    if (bias) {
        rc = msamp_cast_to_fp8_colsum_gated(a->dy, dy_dtype, tokens, d_out, a->g_scale, a->g_amax, a->g_scale_inv, codes, MSAMP_DT_E5M2,
                                            a->bias_sum, static_cast<int>(a->bias_sum_dtype), reinterpret_cast<float*>(product + s.sums), 0,
                                            flags, a->g_counter, static_cast<int>(a->g_window), a->workspace, stream);
    } else {
        rc = msamp_cast_to_fp8_gated(a->dy, dy_dtype, static_cast<size_t>(tokens) * d_out, a->g_scale, a->g_amax, a->g_scale_inv, codes,
                                     MSAMP_DT_E5M2, 0, flags, a->g_counter, static_cast<int>(a->g_window), a->workspace, stream);
    }
    if (rc != MSAMP_OK) return rc;
    if (a->dx != nullptr) {
        rc = gemm_kmajor(a->w_codes, MSAMP_DT_E4M3, a->w_scale_inv, codes, MSAMP_DT_E5M2, a->g_scale_inv, 0, a->dx, out_dtype, d_in, tokens,
                         d_out, 0, st);
        if (rc != MSAMP_OK) return rc;
    }
    if (!wgrad) return MSAMP_OK;
    const size_t n = static_cast<size_t>(d_out) * d_in;
    if (accumulate) {
        rc = msamp_cast_from_fp8(a->old_codes, static_cast<int>(a->old_type), n, a->old_scale_inv, product, out_dtype, stream);
        if (rc != MSAMP_OK) return rc;
    }
    if (s.n_parts != 0 && a->scratch_bytes >= static_cast<int64_t>(s.end)) {
        rc = msamp_fp8_gemm_ksplit(a->x_codes, MSAMP_DT_E4M3, a->x_scale_inv, codes, MSAMP_DT_E5M2, a->g_scale_inv, product, out_dtype, d_in,
                                   d_out, tokens, accumulate, reinterpret_cast<float*>(product + s.parts), s.n_parts, stream);
    } else {
        rc = gemm_kmajor(a->x_codes, MSAMP_DT_E4M3, a->x_scale_inv, codes, MSAMP_DT_E5M2, a->g_scale_inv, 1, product, out_dtype, d_in, d_out,
                         tokens, accumulate, st);
    }
    if (rc != MSAMP_OK) return rc;
    return msamp_cast_to_fp8_intime(product, out_dtype, n, a->q_scale, a->q_amax, a->q_scale_inv, a->wq, MSAMP_DT_E4M3, 0,
                                    flags | MSAMP_FLAG_NAN_TO_INF, a->workspace, stream);
}
