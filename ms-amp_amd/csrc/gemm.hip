// C entry points of the FP8 GEMM: D[N][M] = (B[N][K] . A[M][K]^T) * a_scale_inv * b_scale_inv (+bias) (+D).
// The kernels live in gemm_kernels.cuh and are compiled once per pair of operand formats (gemm_inst.hip); this
// file checks the arguments and hands the call over.  Inside the kernels the operand that supplies D's rows is
// X (= B of the API, N rows) and the one that supplies D's columns is Y (= A of the API, M rows).
#include "gemm_call.h"

#include <algorithm>
#include <atomic>
#include <map>
#include <mutex>
#include <tuple>

namespace msamp {

static int dispatch_pair(int x_type, int y_type, const GemmCall& c) {
    if (x_type == MSAMP_DT_E4M3 && y_type == MSAMP_DT_E4M3) return run_gemm_pair<MSAMP_DT_E4M3, MSAMP_DT_E4M3>(c);
    if (x_type == MSAMP_DT_E4M3) return run_gemm_pair<MSAMP_DT_E4M3, MSAMP_DT_E5M2>(c);
    if (y_type == MSAMP_DT_E4M3) return run_gemm_pair<MSAMP_DT_E5M2, MSAMP_DT_E4M3>(c);
    return run_gemm_pair<MSAMP_DT_E5M2, MSAMP_DT_E5M2>(c);
}

// K-major operands: only the direct-to-LDS kernels read them, so the shape must suit them: two slices of K, rows that are
// read 16 bytes at a time (a K-major operand's row count and a row-major one's K are its leading dimension)
static bool kmajor_rows_ok(int NR, int NC, int K, bool xt, bool yt) {
    return fits_offsets(NR, NC, K) && (xt ? NR % 16 == 0 : K % 16 == 0) && (yt ? NC % 16 == 0 : K % 16 == 0);
}
static bool kmajor_shape_ok(int NR, int NC, int K, bool xt, bool yt) { return K > kBK && kmajor_rows_ok(NR, NC, K, xt, yt); }

static int dispatch_parts(int x_type, int y_type, const GemmCall& c, const KSplit& s) {
    if (x_type == MSAMP_DT_E4M3 && y_type == MSAMP_DT_E4M3) return run_gemm_parts<MSAMP_DT_E4M3, MSAMP_DT_E4M3>(c, s);
    if (x_type == MSAMP_DT_E4M3) return run_gemm_parts<MSAMP_DT_E4M3, MSAMP_DT_E5M2>(c, s);
    if (y_type == MSAMP_DT_E4M3) return run_gemm_parts<MSAMP_DT_E5M2, MSAMP_DT_E4M3>(c, s);
    return run_gemm_parts<MSAMP_DT_E5M2, MSAMP_DT_E5M2>(c, s);
}

// Weight gradients (both operands K-major, K = tokens) whose output is a few tiles leave compute units idle, or run a second
// round of 128 x 128 tiles that is nearly empty; K is long there, so the chip is filled with parts of K.  What a form takes is
// estimated, in microseconds, as rounds of tiles times what a tile costs (a 128-byte slice 0.6 with small and 1.65 with large
// tiles, both with every compute unit busy; 5 and 9 around the K loop) plus, if split, the second launch and the way of the
// partial sums to memory and back.  The split must promise 15 % less, so that it is not taken where the estimate
// is near even.  Only problems of the 128 x 128 tiles are looked at: the others have tiles enough.  Whole against split, m x n
// x k in us: 1200 x 4304 x 12605 128.9 -> 83.0 (three parts of large tiles; 340 small tiles, one to a compute unit, before; two to
// a unit 121.3), 128 x 512 x 16000 54.9 -> 15.2, 256 x 1024 x 8192 29.9 -> 15.6, 1024 x 1024 x 16384 57.6 -> 33.4,
// 16 x 8192 x 8192 30.3 -> 19.7, 2048 x 1024 x 8192 32.8 -> 27.4, 512 x 512 x 2500 12.7 -> 11.4.  FP8Linear 12605 x 1200 -> 4304,
// forward and backward: 335 -> 292.
// Other operands (a forward product, an input gradient) only where the whole product would run 128 x 128 tiles one to a compute unit
// with a longer K than two to a unit take, and in small tiles: their outputs as a rule are larger.  The layer call,
// us: forward 468 x 11840 -> 512 61 -> 32, forward and backward twice over 791 x 15583 -> 1024 453 -> 387.
// The whole product is estimated as small tiles one to a unit; two to a unit take less (takes_paired_tiles), so that the estimate is
// too high for them.  Over 119 random products that the rule splits (up to 480 small tiles, K from 512 to 40000) the split was the
// slower choice twice, by 0.7 and 0.9 us (704 x 144 x 2048 10.0 whole, 48 x 320 x 2016 9.4); 4096 x 2048 x 32768 253 -> 182.
static KSplit ksplit_rule(int NR, int NC, int K, bool xt, bool yt) {
    KSplit best = {true, 1};
    // (the parts are added up four outputs at a time)
    if (!takes_small_tiles(NR, NC, K) || !fits_offsets(NR, NC, K) || static_cast<size_t>(NR) * NC % 4) return best;
    const bool both = xt && yt;
    if (!both && (K <= 2048 || takes_paired_tiles(NR, NC, K))) return best;
    const int nk = (K + kBK - 1) / kBK, cus = cu_count();
    auto tiles = [&](int edge) { return ((NR + edge - 1) / edge) * ((NC + edge - 1) / edge); };
    const int small = tiles(kDmaTile / 2), large = tiles(kDmaTile);
    const double out = static_cast<double>(NR) * NC;
    auto estimate = [&](int n, int parts, double slice, double around) {
        const double rounds = (n * parts + cus - 1) / cus;
        return rounds * ((nk + parts - 1) / parts * slice + around) + (parts > 1 ? 4.0 + out * (8.0 * parts + 2.0) / 5e6 : 0.0);
    };
    double least = 0.85 * estimate(small, 1, 0.6, 5.0);
    // (at least four slices to a part, which is also what the small tile needs)
    for (int parts = 2; parts <= 32 && nk / parts >= 4; ++parts) {
        if (static_cast<long>(small) * parts <= 4L * cus) {
            const double t = estimate(small, parts, 0.6, 5.0);
            if (t < least) least = t, best = {true, parts};
        }
        if (both && static_cast<long>(large) * parts <= 4L * cus) {
            const double t = estimate(large, parts, 1.65, 9.0);
            if (t < least) least = t, best = {false, parts};
        }
    }
    return best;
}

// D = (sum of the parts, in their order) * alpha (+ bias) (+ D), the expressions of the GEMM's own epilogue, one rounding.  Bound by
// the read of the parts; four elements a lane.
template <typename OT>
__global__ __launch_bounds__(256) void ksplit_finish_kernel(const float* __restrict__ part, OT* __restrict__ D, size_t n, int parts,
                                                            const float* __restrict__ xs, const float* __restrict__ ys, int accumulate,
                                                            const void* __restrict__ bias, int bias_dt, unsigned cols) {
    const size_t i = (static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
    if (i >= n) return;    // (n is a multiple of 4)
    const float alpha = (*xs) * (*ys);
    float4 s = *reinterpret_cast<const float4*>(part + i);
#pragma unroll 4
    for (int p = 1; p < parts; ++p) {
        const float4 v = *reinterpret_cast<const float4*>(part + static_cast<size_t>(p) * n + i);
        s.x += v.x, s.y += v.y, s.z += v.z, s.w += v.w;
    }
    const float r[4] = {s.x, s.y, s.z, s.w};
    struct __attribute__((aligned(4 * sizeof(OT)))) Four { OT v[4]; };
    Four o;
    if (bias != nullptr) {    // (never with an old output: the callers see to that)
        unsigned c = static_cast<unsigned>(i) % cols;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float b = bias_dt == MSAMP_DT_F32   ? static_cast<const float*>(bias)[c]
                            : bias_dt == MSAMP_DT_F16 ? Elem<f16_t>::load(static_cast<const f16_t*>(bias) + c)
                                                      : Elem<bf16_t>::load(static_cast<const bf16_t*>(bias) + c);
            Elem<OT>::store(&o.v[e], fmaf(r[e], alpha, b));
            c = c + 1 == cols ? 0 : c + 1;
        }
    } else if (accumulate) {
        const Four old = *reinterpret_cast<const Four*>(D + i);
#pragma unroll
        for (int e = 0; e < 4; ++e) Elem<OT>::store(&o.v[e], fmaf(r[e], alpha, 0.0f) + Elem<OT>::load(&old.v[e]));
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) Elem<OT>::store(&o.v[e], r[e] * alpha);
    }
    *reinterpret_cast<Four*>(D + i) = o;
}

// tile walks registered per problem (kernel-side naming: NR x NC output, K, which operands are K-major)
static std::mutex g_walk_mutex;
static std::map<std::tuple<int, int, int, int>, int> g_walks;
static thread_local int t_forced_walk = -2;    // -2: none; msamp_fp8_gemm_tune times its candidates through this
int registered_walk(int NR, int NC, int K, bool XT, bool YT) {
    if (t_forced_walk != -2) return t_forced_walk;
    std::lock_guard<std::mutex> lock(g_walk_mutex);
    if (g_walks.empty()) return -1;
    const auto it = g_walks.find(std::make_tuple(NR, NC, K, (XT ? 1 : 0) | (YT ? 2 : 0)));
    return it == g_walks.end() ? -1 : it->second;
}

static std::atomic<int> g_small_tile_limit{kSmallTileLimit};
int small_tile_limit() { return g_small_tile_limit.load(std::memory_order_relaxed); }

// 128 x 128 tiles with two workgroups to a compute unit, us against the kernel that would take the product otherwise (row-major,
// both K-major):
//   K <= 128 (the generic kernel)                        1024 x 1024  13.8 -> 4.6     8192 x 4096  58.5 -> 17.9
//   one tile a unit or fewer, K = 256 (large tiles)      2048 x 2048   8.4 -> 5.4,     8.7 -> 5.6
//     K = 1024 (small tiles, one workgroup a unit)       2048 x 2048   7.5 -> 7.0,     8.3 -> 7.3
//     K = 2048                                           2048 x 2048   9.9 -> 9.5,    11.4 -> 10.2    K = 4096: 18.1 -> 20.8, 20.1 -> 20.6
//   up to two tiles a unit, K = 1024 (large tiles)       4096 x 2048  13.9 -> 10.4,   14.2 -> 10.9
//     K = 4096 (small tiles)                             4096 x 2048  35.5 -> 30.4,   41.0 -> 31.9    K = 12288: 89.0 -> 83.2, 104.5 -> 87.6
//   more (large tiles)                                   3072 x 4096 x 1024  14.8 -> 13.9, 15.1 -> 15.1;   4096 x 4096 x 1024  16.9 -> 17.7, 17.3 -> 18.8
// Large tiles of which a few begin another round cost a whole one, where paired tiles, of half a round's time each, take what is
// there.  us, row-major with a bias, without, one operand K-major, both:
//   1 to 1.25 rounds, K <= 2048    5120 x 4096 x 512   22.9 -> 19.3, 22.1 -> 17.5, 22.0 -> 16.9, 21.9 -> 16.8   K = 2048  48.4 -> 45.0, 46.9 -> 41.8, 46.8 -> 42.9, 47.8 -> 43.8
//   1.25 to 1.5, K <= 1024         6144 x 4096 x 512   22.3 -> 19.8, 21.9 -> 18.5, 22.2 -> 19.1, 22.2 -> 19.7   K = 1024  31.0 -> 31.0, 29.9 -> 29.4, 30.3 -> 29.7, 30.2 -> 30.7
//   2 to 2.25, K <= 1536           9216 x 4096 x 512   34.3 -> 30.4, 32.9 -> 29.1, 33.1 -> 27.4, 33.4 -> 29.8   K = 1536  61.1 -> 59.2, 59.8 -> 58.1, 60.1 -> 58.3, 60.2 -> 59.4
//   elsewhere                      6144 x 4096 x 2048  47.4 -> 48.9, 46.8 -> 46.9, 47.0 -> 48.9, 47.1 -> 50.0   K = 1536  39.4 -> 40.4, 38.6 -> 39.0, 38.9 -> 39.3, 38.8 -> 40.1
//                                  9216 x 4096 x 2048  73.4 -> 73.7, 72.3 -> 71.1, 72.8 -> 72.5, 73.4 -> 75.5
//                                  7168 x 4096 x 512   23.1 -> 24.6, 22.6 -> 21.8, 23.0 -> 22.1                 K = 2048  47.5 -> 54.2, 48.0 -> 54.7, 49.1 -> 55.2 (of these three no row without)
//                                  6144 x 4096 x 4096  78.7 -> 80.7, 78.0 -> 81.0   5120 x 4096 x 8192  143.7 -> 131.8, 142.9 -> 140.7, 150.1 -> 172.0
bool takes_paired_tiles(int NR, int NC, int K) {
    if (small_tile_limit() != kSmallTileLimit) return false;
    const long tiles = static_cast<long>((NR + kDmaTile / 2 - 1) / (kDmaTile / 2)) * ((NC + kDmaTile / 2 - 1) / (kDmaTile / 2));
    const long large = static_cast<long>((NR + kDmaTile - 1) / kDmaTile) * ((NC + kDmaTile - 1) / kDmaTile), cus = cu_count();
    if (large > cus && ((tiles <= 5 * cus && K <= 2048) || (tiles <= 6 * cus && K <= 1024))) return true;
    if (large > 2 * cus && tiles <= 9 * cus && K <= 1536) return true;
    return K <= kBK || (tiles <= 2 * cus && (tiles > cus || K <= 2048));
}

}    // namespace msamp

using namespace msamp;

extern "C" void msamp_set_small_tile_limit(int big_tiles) {
    msamp::g_small_tile_limit.store(big_tiles, std::memory_order_relaxed);
}

extern "C" int msamp_fp8_gemm_set_walk(int m, int n, int k, int a_kmajor, int b_kmajor, int walk) {
    MSAMP_REQUIRE(walk >= -1 && walk <= 7, MSAMP_ERR_SHAPE, "msamp_fp8_gemm_set_walk: walk=%d", walk);
    // X = b (n rows of D), Y = a (m columns of D)
    const auto key = std::make_tuple(n, m, k, (b_kmajor ? 1 : 0) | (a_kmajor ? 2 : 0));
    std::lock_guard<std::mutex> lock(msamp::g_walk_mutex);
    if (walk < 0) msamp::g_walks.erase(key);
    else msamp::g_walks[key] = walk;
    return MSAMP_OK;
}

extern "C" int msamp_fp8_gemm_get_walk(int m, int n, int k, int a_kmajor, int b_kmajor) {
    std::lock_guard<std::mutex> lock(msamp::g_walk_mutex);
    const auto it = msamp::g_walks.find(std::make_tuple(n, m, k, (b_kmajor ? 1 : 0) | (a_kmajor ? 2 : 0)));
    return it == msamp::g_walks.end() ? -1 : it->second;
}

extern "C" int msamp_fp8_gemm_tune(const uint8_t* a, int a_type, const float* a_scale_inv, int a_kmajor, const uint8_t* b,
                                   int b_type, const float* b_scale_inv, int b_kmajor, void* d, int d_dtype, int m, int n,
                                   int k, const void* bias, int bias_dtype, int* chosen, msamp_stream_t stream) {
    hipStream_t st = static_cast<hipStream_t>(stream);
    auto run = [&]() {
        return msamp_fp8_gemm_kmajor(a, a_type, a_scale_inv, a_kmajor, b, b_type, b_scale_inv, b_kmajor, d, d_dtype, m, n, k, 0, bias,
                                     bias_dtype, stream);
    };
    if (chosen) *chosen = -1;
    // Only problems of the 256 x 256-tile kernel with at least two rounds of tiles have a walk worth timing, and timing
    // needs a stream that is not being captured; everything else is the plain product.
    const long tiles = (static_cast<long>(n) + kDmaTile - 1) / kDmaTile * ((static_cast<long>(m) + kDmaTile - 1) / kDmaTile);
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &capturing) != hipSuccess) capturing = hipStreamCaptureStatusActive, (void)hipGetLastError();
    const bool candidate = m > 0 && n > 0 && k >= 4 * kBK && k % kBK == 0 && tiles >= 2L * cu_count() && !takes_small_tiles(n, m, k) && !takes_paired_tiles(n, m, k) &&
                           capturing == hipStreamCaptureStatusNone;
    if (!candidate) return run();
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
        if (e0) (void)hipEventDestroy(e0);
        (void)hipGetLastError();
        return run();
    }
    // the rule's walk first and last, the four explicit ones between: two untimed launches, then as many as fill about four
    // milliseconds (at least four) between one pair of events
    float best_ms = 0.0f, rule_ms = 0.0f;
    int best = -1, rc = MSAMP_OK;
    const int turns = 6;
    for (int turn = 0; turn < turns && rc == MSAMP_OK; ++turn) {
        int walk = turn - 1;
        if (turn == turns - 1) walk = -1;    // (the rule's walk once more at the end: a cold start must not cost it the comparison)
        msamp::t_forced_walk = walk;
        for (int i = 0; i < 2 && rc == MSAMP_OK; ++i) rc = run();
        int reps = 4;
        if (walk >= 0 && rule_ms > 0.0f) reps = std::max(4, std::min(64, static_cast<int>(4.0f / rule_ms)));
        if (rc == MSAMP_OK && hipEventRecord(e0, st) != hipSuccess) rc = MSAMP_ERR_HIP;
        for (int i = 0; i < reps && rc == MSAMP_OK; ++i) rc = run();
        float ms = 0.0f;
        if (rc == MSAMP_OK && (hipEventRecord(e1, st) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
                               hipEventElapsedTime(&ms, e0, e1) != hipSuccess))
            rc = MSAMP_ERR_HIP;
        ms /= reps;
        if (turn == 0) rule_ms = best_ms = ms;
        else if (walk < 0) rule_ms = std::min(rule_ms, ms);
        else if (ms < best_ms) best_ms = ms, best = walk;
    }
    msamp::t_forced_walk = -2;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc != MSAMP_OK) {
        (void)hipGetLastError();
        return run();
    }
    // an explicit walk is kept only where it beats the rule's by more than the timing's noise
    if (best >= 0 && best_ms > 0.95f * rule_ms) best = -1;
    msamp_fp8_gemm_set_walk(m, n, k, a_kmajor, b_kmajor, best);
    if (chosen) *chosen = best;
    return MSAMP_OK;    // (d holds the product: every timed launch wrote it)
}

// words of the workspace that the speculative form of msamp_fp8_gemm_cast uses: running maximum, ticket counter (both
// left at zero by every call) and the flag its second launch reads
constexpr int kWsGemmSpec = 10;

extern "C" int msamp_fp8_gemm_cast(const uint8_t* a, int a_type, const float* a_scale_inv, int a_kmajor, const uint8_t* b,
                                   int b_type, const float* b_scale_inv, int b_kmajor, void* d, int d_dtype, int accumulate,
                                   uint8_t* q, int q_type, float* scale, float* amax, float* scale_inv, int m, int n, int k,
                                   int margin, int flags, void* workspace, msamp_stream_t stream) {
    MSAMP_REQUIRE(is_fp8(a_type) && is_fp8(b_type) && is_fp8(q_type), MSAMP_ERR_DTYPE, "msamp_fp8_gemm_cast: types %d, %d -> %d",
                  a_type, b_type, q_type);
    MSAMP_REQUIRE(is_hp(d_dtype), MSAMP_ERR_DTYPE, "msamp_fp8_gemm_cast: intermediate dtype %d", d_dtype);
    MSAMP_REQUIRE(m > 0 && n > 0 && k > 0, MSAMP_ERR_SHAPE, "msamp_fp8_gemm_cast: m=%d n=%d k=%d", m, n, k);
    MSAMP_REQUIRE(a && b && q && a_scale_inv && b_scale_inv && scale && amax && scale_inv, MSAMP_ERR_NULL,
                  "msamp_fp8_gemm_cast: null pointer");
    MSAMP_REQUIRE(!accumulate || d != nullptr, MSAMP_ERR_NULL, "msamp_fp8_gemm_cast: accumulate needs d");
    MSAMP_REQUIRE(aligned(a, 16) && aligned(b, 16) && aligned(q, 16) && aligned(d, 16), MSAMP_ERR_ALIGNMENT,
                  "msamp_fp8_gemm_cast: operands and outputs must be 16-byte aligned");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const bool both = a_kmajor && b_kmajor, neither = !a_kmajor && !b_kmajor;
    const long tiles = static_cast<long>(n / kDmaTile) * (m / kDmaTile);
    const bool fits32 = static_cast<unsigned long long>(n) * k < (1ull << 32) && static_cast<unsigned long long>(m) * k < (1ull << 32);
    if (q_type != MSAMP_DT_E4M3 || !(both || neither) || m % kDmaTile || n % kDmaTile || k % kBK || k < 2 * kBK || !fits32 ||
        workspace == nullptr)
        return MSAMP_NOT_FUSED;
    // A problem small enough for the 128 x 128 tiles is better off with the two steps: both forms below run 256 x 256
    // tiles, a few of them on a few compute units, where the small-tile GEMM and the one-pass cast of its (small) output
    // take less (1024 x 1024 x 8192: 38 against 70 us; 2048 x 2048 x 2048: 22 against 27).
    if (takes_small_tiles(n, m, k)) return MSAMP_NOT_FUSED;
    QuantArgs qa = {};
    qa.q = q, qa.scale = scale, qa.amax = amax, qa.scale_inv = scale_inv;
    qa.slots = reinterpret_cast<uint64_t*>(static_cast<char*>(workspace) + kWsSlotBytes);
    qa.fp_max = fp8_max(q_type), qa.margin = margin, qa.flags = flags;
    qa.error_word = static_cast<uint32_t*>(workspace) + kWsErrorWord;
    qa.spec_words = static_cast<uint32_t*>(workspace) + kWsGemmSpec;
    // one launch, D never stored: at most one tile per compute unit, on a stream that may run waiting kernels
    if (!accumulate && tiles <= cu_count() && tiles <= kMaxSlots && !(flags & MSAMP_FLAG_TWO_PASS) && waiting_kernels_allowed(st)) {
        qa.token = next_tokens(1);
        qa.spin_limit = collector_spin_limit();
        // X = b (rows of D), Y = a (columns of D)
        const GemmCall c = {b, a, nullptr, d_dtype, n, m, k, b_scale_inv, a_scale_inv, 0, nullptr, 0, both, both, &qa, st};
        const int rc = dispatch_pair(b_type, a_type, c);
        if (rc != MSAMP_NOT_FUSED) return rc;
    }
    if (d == nullptr || (flags & MSAMP_FLAG_NO_SPECULATION)) return MSAMP_NOT_FUSED;
    // on speculation: D and the codes for the scale in force side by side, then (only if the rule arrives at another
    // scale) the cast of D again
    GemmCall c = {b, a, d, d_dtype, n, m, k, b_scale_inv, a_scale_inv, accumulate, nullptr, 0, both, both, &qa, st};
    c.qspec = true;
    const int rc = dispatch_pair(b_type, a_type, c);
    if (rc != MSAMP_OK) return rc;
    return cast_again_if_flagged(d, d_dtype, static_cast<size_t>(n) * m, scale, q, q_type, qa.spec_words + 2, st);
}

extern "C" int msamp_fp8_gemm_kmajor(const uint8_t* a, int a_type, const float* a_scale_inv, int a_kmajor, const uint8_t* b,
                                     int b_type, const float* b_scale_inv, int b_kmajor, void* d, int d_dtype, int m, int n,
                                     int k, int accumulate, const void* bias, int bias_dtype, msamp_stream_t stream) {
    if (!a_kmajor && !b_kmajor)
        return msamp_fp8_gemm(a, a_type, a_scale_inv, b, b_type, b_scale_inv, d, d_dtype, m, n, k, accumulate, bias, bias_dtype, stream);
    MSAMP_REQUIRE(is_fp8(a_type) && is_fp8(b_type), MSAMP_ERR_DTYPE, "msamp_fp8_gemm_kmajor: operand types %d, %d", a_type, b_type);
    MSAMP_REQUIRE(is_hp(d_dtype), MSAMP_ERR_DTYPE, "msamp_fp8_gemm_kmajor: output dtype %d", d_dtype);
    MSAMP_REQUIRE(bias == nullptr || is_hp(bias_dtype), MSAMP_ERR_DTYPE, "msamp_fp8_gemm_kmajor: bias dtype %d", bias_dtype);
    MSAMP_REQUIRE(a_kmajor, MSAMP_ERR_SHAPE, "msamp_fp8_gemm_kmajor: b may be K-major only together with a");
    MSAMP_REQUIRE(m > 0 && n > 0 && k > 0 && kmajor_shape_ok(n, m, k, b_kmajor != 0, true), MSAMP_ERR_SHAPE,
                  "msamp_fp8_gemm_kmajor: m=%d n=%d k=%d (k must be more than 128, leading dimensions multiples of 16)", m, n, k);
    MSAMP_REQUIRE(a && b && d && a_scale_inv && b_scale_inv, MSAMP_ERR_NULL, "msamp_fp8_gemm_kmajor: null pointer");
    MSAMP_REQUIRE(aligned(a, 16) && aligned(b, 16), MSAMP_ERR_ALIGNMENT, "msamp_fp8_gemm_kmajor: operands must be 16-byte aligned");
    hipStream_t st = static_cast<hipStream_t>(stream);
    // X = b (rows of D), Y = a (columns of D)
    const GemmCall c = {b, a, d, d_dtype, n, m, k, b_scale_inv, a_scale_inv, accumulate, bias, bias_dtype, b_kmajor != 0, true, nullptr, st};
    return dispatch_pair(b_type, a_type, c);
}

int msamp::gemm_kmajor(const uint8_t* a, int a_type, const float* a_scale_inv, const uint8_t* b, int b_type, const float* b_scale_inv,
                       int b_kmajor, void* d, int d_dtype, int m, int n, int k, int accumulate, hipStream_t st) {
    MSAMP_REQUIRE(is_fp8(a_type) && is_fp8(b_type) && is_hp(d_dtype), MSAMP_ERR_DTYPE, "gemm_kmajor: types %d, %d -> %d", a_type, b_type,
                  d_dtype);
    MSAMP_REQUIRE(m > 0 && n > 0 && k > 0 && kmajor_rows_ok(kmajor_pitch(n), kmajor_pitch(m), k, b_kmajor != 0, true), MSAMP_ERR_SHAPE,
                  "gemm_kmajor: m=%d n=%d k=%d (K of a row-major operand must be a multiple of 16)", m, n, k);
    MSAMP_REQUIRE(a && b && d && a_scale_inv && b_scale_inv, MSAMP_ERR_NULL, "gemm_kmajor: null pointer");
    MSAMP_REQUIRE(aligned(a, 16) && aligned(b, 16), MSAMP_ERR_ALIGNMENT, "gemm_kmajor: operands must be 16-byte aligned");
    const GemmCall c = {b, a, d, d_dtype, n, m, k, b_scale_inv, a_scale_inv, accumulate, nullptr, MSAMP_DT_F32, b_kmajor != 0, true, nullptr, st};
    return dispatch_pair(b_type, a_type, c);
}

size_t msamp::gemm_parts_scratch(int NR, int NC, int K, bool xt, bool yt) {
    const KSplit split = ksplit_rule(NR, NC, K, xt, yt);
    return split.parts > 1 ? static_cast<size_t>(split.parts) * NR * NC : 0;
}

int msamp::gemm_parts(int x_type, int y_type, const GemmCall& c, float* scratch, size_t n_floats) {
    const KSplit split = ksplit_rule(c.NR, c.NC, c.K, c.xt, c.yt);
    const size_t count = static_cast<size_t>(c.NR) * c.NC;
    MSAMP_REQUIRE(split.parts > 1 && n_floats >= split.parts * count, MSAMP_ERR_SHAPE,
                  "gemm_parts: m=%d n=%d k=%d is not split, or needs more scratch than %zu floats", c.NC, c.NR, c.K, n_floats);
    MSAMP_REQUIRE(aligned(c.X, 16) && aligned(c.Y, 16) && aligned(c.D, 16) && aligned(scratch, 16), MSAMP_ERR_ALIGNMENT,
                  "gemm_parts: operands, output and scratch must be 16-byte aligned");
    GemmCall part = c;
    part.D = scratch, part.d_dtype = MSAMP_DT_F32;
    const int rc = dispatch_parts(x_type, y_type, part, split);
    if (rc != MSAMP_OK) return rc;
    const dim3 grid(static_cast<unsigned>((count / 4 + 255) / 256));
#define FINISH(OT) \
    hipLaunchKernelGGL((ksplit_finish_kernel<OT>), grid, dim3(256), 0, c.st, static_cast<const float*>(scratch), static_cast<OT*>(c.D), count, split.parts, c.xs, c.ys, c.accumulate, c.bias, c.bias_dt, static_cast<unsigned>(c.NC))
    if (c.d_dtype == MSAMP_DT_F32) FINISH(float);
    else if (c.d_dtype == MSAMP_DT_F16) FINISH(f16_t);
    else FINISH(bf16_t);
#undef FINISH
    MSAMP_CHECK_LAUNCH("ksplit_finish_kernel");
    return MSAMP_OK;
}

extern "C" int msamp_fp8_gemm_ksplit_scratch(int m, int n, int k, size_t* n_floats) {
    MSAMP_REQUIRE(m > 0 && n > 0 && k > 0, MSAMP_ERR_SHAPE, "msamp_fp8_gemm_ksplit_scratch: m=%d n=%d k=%d", m, n, k);
    MSAMP_REQUIRE(n_floats != nullptr, MSAMP_ERR_NULL, "msamp_fp8_gemm_ksplit_scratch: null pointer");
    *n_floats = kmajor_shape_ok(n, m, k, true, true) ? gemm_parts_scratch(n, m, k, true, true) : 0;
    return MSAMP_OK;
}

extern "C" int msamp_fp8_gemm_ksplit(const uint8_t* a, int a_type, const float* a_scale_inv, const uint8_t* b, int b_type,
                                     const float* b_scale_inv, void* d, int d_dtype, int m, int n, int k, int accumulate,
                                     float* scratch, size_t n_floats, msamp_stream_t stream) {
    MSAMP_REQUIRE(is_fp8(a_type) && is_fp8(b_type), MSAMP_ERR_DTYPE, "msamp_fp8_gemm_ksplit: operand types %d, %d", a_type, b_type);
    MSAMP_REQUIRE(is_hp(d_dtype), MSAMP_ERR_DTYPE, "msamp_fp8_gemm_ksplit: output dtype %d", d_dtype);
    MSAMP_REQUIRE(m > 0 && n > 0 && k > 0 && kmajor_shape_ok(n, m, k, true, true), MSAMP_ERR_SHAPE,
                  "msamp_fp8_gemm_ksplit: m=%d n=%d k=%d", m, n, k);
    MSAMP_REQUIRE(a && b && d && a_scale_inv && b_scale_inv && scratch, MSAMP_ERR_NULL, "msamp_fp8_gemm_ksplit: null pointer");
    // X = b (rows of D), Y = a (columns of D)
    const GemmCall c = {b, a, d, d_dtype, n, m, k, b_scale_inv, a_scale_inv, accumulate, nullptr, 0, true, true, nullptr, static_cast<hipStream_t>(stream)};
    return gemm_parts(b_type, a_type, c, scratch, n_floats);
}

extern "C" int msamp_fp8_gemm(const uint8_t* a, int a_type, const float* a_scale_inv, const uint8_t* b, int b_type,
                              const float* b_scale_inv, void* d, int d_dtype, int m, int n, int k, int accumulate,
                              const void* bias, int bias_dtype, msamp_stream_t stream) {
    MSAMP_REQUIRE(is_fp8(a_type) && is_fp8(b_type), MSAMP_ERR_DTYPE, "msamp_fp8_gemm: operand types %d, %d", a_type, b_type);
    MSAMP_REQUIRE(is_hp(d_dtype), MSAMP_ERR_DTYPE, "msamp_fp8_gemm: output dtype %d", d_dtype);
    MSAMP_REQUIRE(bias == nullptr || is_hp(bias_dtype), MSAMP_ERR_DTYPE, "msamp_fp8_gemm: bias dtype %d", bias_dtype);
    MSAMP_REQUIRE(m >= 0 && n >= 0 && k >= 0, MSAMP_ERR_SHAPE, "msamp_fp8_gemm: m=%d n=%d k=%d", m, n, k);
    if (m == 0 || n == 0) return MSAMP_OK;
    MSAMP_REQUIRE(k > 0 && k % 16 == 0, MSAMP_ERR_SHAPE, "msamp_fp8_gemm: k=%d must be a positive multiple of 16", k);
    MSAMP_REQUIRE(a && b && d && a_scale_inv && b_scale_inv, MSAMP_ERR_NULL, "msamp_fp8_gemm: null pointer");
    MSAMP_REQUIRE(aligned(a, 16) && aligned(b, 16), MSAMP_ERR_ALIGNMENT, "msamp_fp8_gemm: operands must be 16-byte aligned");
    hipStream_t st = static_cast<hipStream_t>(stream);
    // X = b (rows of D), Y = a (columns of D)
    const GemmCall c = {b, a, d, d_dtype, n, m, k, b_scale_inv, a_scale_inv, accumulate, bias, bias_dtype, false, false, nullptr, st};
    return dispatch_pair(b_type, a_type, c);
}

// Calibration aid: what the matrix pipes of this device sustain when nothing else moves.  Every wavefront issues
// 16x16x128 FP8 MFMAs on registers it loaded once; the sum is stored only if it equals a value it cannot take, so
// the loop is not optimised away and nothing is written.  FRAGS = 1: the same two operands for every MFMA (the
// operand buses never toggle); FRAGS = 8: eight X and eight Y fragments, every pair once per turn as in a K slice of
// the GEMM, so that consecutive MFMAs see different operands.
namespace msamp {
typedef int mfma_probe_v8i __attribute__((ext_vector_type(8)));
typedef float mfma_probe_v4f __attribute__((ext_vector_type(4)));
template <int FRAGS>
__global__ __launch_bounds__(256) void mfma_probe_kernel(const int* __restrict__ seed, float* __restrict__ sink, int iters) {
    mfma_probe_v8i a[FRAGS], b[FRAGS];
    for (int f = 0; f < FRAGS; ++f)
        for (int i = 0; i < 8; ++i) {
            a[f][i] = seed[(threadIdx.x * 8 + i + f * 37) & 1023];
            b[f][i] = seed[(threadIdx.x * 8 + i + 512 + f * 53) & 1023];
        }
    mfma_probe_v4f acc[16];
    for (int i = 0; i < 16; ++i) acc[i] = mfma_probe_v4f{0, 0, 0, 0};
    constexpr int kTurns = FRAGS == 1 ? 1 : 4;    // 16 or 64 MFMAs per turn of the loop
    for (int it = 0; it < iters; it += kTurns) {
#pragma unroll
        for (int n = 0; n < 16 * kTurns; ++n) {
            const int i = (n / FRAGS) % FRAGS, j = n % FRAGS;
            acc[n % 16] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a[i], b[j], acc[n % 16], 0, 0, 0, 0, 0, 0);
        }
    }
    float s = 0;
    for (int i = 0; i < 16; ++i) s += acc[i][0] + acc[i][1] + acc[i][2] + acc[i][3];
    if (s == 12345.678f) sink[0] = s;
}
}    // namespace msamp

extern "C" int msamp_mfma_probe(const void* seed, float* sink, int iters, int workgroups, int distinct_operands, double* flop,
                                msamp_stream_t stream) {
    MSAMP_REQUIRE(seed && sink, MSAMP_ERR_NULL, "msamp_mfma_probe: null pointer");
    MSAMP_REQUIRE(iters > 0 && iters % 4 == 0 && workgroups > 0 && workgroups <= 65536, MSAMP_ERR_SHAPE,
                  "msamp_mfma_probe: iters=%d (a positive multiple of 4) workgroups=%d", iters, workgroups);
    if (distinct_operands)
        hipLaunchKernelGGL(mfma_probe_kernel<8>, dim3(workgroups), dim3(256), 0, static_cast<hipStream_t>(stream),
                           static_cast<const int*>(seed), sink, iters);
    else
        hipLaunchKernelGGL(mfma_probe_kernel<1>, dim3(workgroups), dim3(256), 0, static_cast<hipStream_t>(stream),
                           static_cast<const int*>(seed), sink, iters);
    if (flop) *flop = 4.0 * workgroups * iters * 16.0 * 2.0 * 16 * 16 * 128;
    MSAMP_CHECK_LAUNCH("msamp_mfma_probe");
    return MSAMP_OK;
}
