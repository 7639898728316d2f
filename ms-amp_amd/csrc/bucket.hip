// Quantizing a bucket of high-precision gradients into one flat FP8 buffer, many tensors per launch: the
// compute steps of the FP8 gradient reducer (msamp/nn/distributed.py:143-184) either side of its amax
// all-reduce.  One workgroup handles one 16384-element chunk of one tensor; a device table describes the
// tensors and a block map assigns the chunks, as in the fused AdamW step.
#include "common.cuh"
#include "raise_max.cuh"

#include <algorithm>

namespace msamp {

constexpr int kBucketThreads = 256;

// max |x| of one chunk, as the bit pattern of the float (a NaN pattern compares above every number, so it wins)
// FMT != 0: the chunk is also quantized, with the scale the item has now, into its place in the flat buffer.  That
// scale is what the previous round's msamp_bucket_cast left there, and it is a power of two times a constant, so it is
// as a rule the scale this round will arrive at; msamp_bucket_cast then finds its work done (see bucket_scale_kernel).
template <typename IT, int FMT>
__global__ __launch_bounds__(kBucketThreads) void bucket_amax_kernel(msamp_bucket_item* __restrict__ items,
                                                                     const int32_t* __restrict__ block_map, int stream) {
    constexpr int EPT = In16<IT>::EPT;
    constexpr int kVecs = MSAMP_BUCKET_CHUNK / (kBucketThreads * EPT);    // 16 (fp32) or 8 (16-bit)
    __shared__ uint32_t red[kBucketThreads / kWave];
    const int t = block_map[2 * blockIdx.x], chunk = block_map[2 * blockIdx.x + 1];
    msamp_bucket_item& d = items[t];
    const IT* x = static_cast<const IT*>(d.src);
    const size_t n = d.numel, base = static_cast<size_t>(chunk) * MSAMP_BUCKET_CHUNK;
    uint32_t m = 0;
    uint8_t* out = d.dst;
    const float s = FMT != 0 ? *d.scale : 1.0f;
    const bool vec_out = FMT == 0 || (reinterpret_cast<uintptr_t>(out) & (EPT - 1)) == 0;
    if (base + MSAMP_BUCKET_CHUNK <= n && (reinterpret_cast<uintptr_t>(x) & 15) == 0 && vec_out) {
        float v[kVecs][EPT];
#pragma unroll
        for (int u = 0; u < kVecs; ++u)
            In16<IT>::load(x + base + (static_cast<size_t>(u) * kBucketThreads + threadIdx.x) * EPT, v[u], stream != 0);
#pragma unroll
        for (int u = 0; u < kVecs; ++u) {
#pragma unroll
            for (int j = 0; j < EPT; ++j) {
                const uint32_t a = __float_as_uint(v[u][j]) & 0x7fffffffu;
                m = a > m ? a : m;
            }
            if constexpr (FMT != 0) {
                uint32_t w[EPT / 4];
#pragma unroll
                for (int j = 0; j < EPT / 4; ++j)
                    w[j] = quant4<FMT>(v[u][4 * j] * s, v[u][4 * j + 1] * s, v[u][4 * j + 2] * s, v[u][4 * j + 3] * s);
                uint8_t* o = out + base + (static_cast<size_t>(u) * kBucketThreads + threadIdx.x) * EPT;
                if constexpr (EPT == 4) {
                    *reinterpret_cast<uint32_t*>(o) = w[0];
                } else {
                    *reinterpret_cast<uint2*>(o) = make_uint2(w[0], w[1]);
                }
            }
        }
    } else {
        for (size_t i = base + threadIdx.x; i < n && i < base + MSAMP_BUCKET_CHUNK; i += kBucketThreads) {
            const float xi = Elem<IT>::load(x + i);
            const uint32_t a = __float_as_uint(xi) & 0x7fffffffu;
            m = a > m ? a : m;
            if constexpr (FMT != 0) out[i] = static_cast<uint8_t>(quant1<FMT>(xi * s));
        }
    }
    m = block_max_u32(m, red);
    if (threadIdx.x == 0) raise_max(&d.acc, m);
}

// amax[0] of every tensor from the accumulated pattern (NaN and +Inf become +Inf when asked: the all-reduce that
// follows in the reducer ignores NaN); the accumulator goes back to zero
constexpr uint32_t kBucketDone = 0xffffffffu;    // item.reserved: the buffer already holds this round's codes

__global__ void bucket_amax_finish_kernel(msamp_bucket_item* items, int n_items, int flags, int speculative) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n_items) return;
    msamp_bucket_item& d = items[t];
    float a = __uint_as_float(d.acc);
    d.acc = 0u;
    // the scale the codes were written with, if they were (a positive finite one: anything else is no guess)
    const float guess = *d.scale;
    d.reserved = (speculative && guess > 0.0f && guess < __uint_as_float(0x7f800000u)) ? __float_as_uint(guess) : 0u;
    if ((flags & MSAMP_FLAG_NAN_TO_INF) && !(a < __uint_as_float(0x7f800000u))) a = __uint_as_float(0x7f800000u);
    *d.amax = a;
}

// scale = rule(amax[0], fallback = the scale in force) * pre_scale, scale_inv = (1 / scale) / inv_div (the reducer
// divides the finished ScalingTensor by the world size, which is a division of scale_inv: two roundings, kept)
__global__ void bucket_scale_kernel(msamp_bucket_item* items, int n_items, float fp_max, int margin, float pre_scale,
                                    float inv_div) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n_items) return;
    msamp_bucket_item& d = items[t];
    const float sf = scale_rule(*d.amax, *d.scale, fp_max, margin) * pre_scale;
    // after msamp_bucket_amax_speculative: did the codes go out with this very scale?  (A mark left by an earlier cast
    // of the same round is no guess: a second cast without a new amax pass writes the codes again.)
    if (d.reserved != 0u) d.reserved = (d.reserved != kBucketDone && __float_as_uint(sf) == d.reserved) ? kBucketDone : 0u;
    *d.scale = sf;
    const float inv = 1.0f / sf;
    *d.scale_inv = inv / inv_div;
}

template <typename IT, int FMT>
__global__ __launch_bounds__(kBucketThreads) void bucket_cast_kernel(const msamp_bucket_item* __restrict__ items,
                                                                     const int32_t* __restrict__ block_map, int stream) {
    constexpr int EPT = In16<IT>::EPT;
    constexpr int kVecs = MSAMP_BUCKET_CHUNK / (kBucketThreads * EPT);
    const int t = block_map[2 * blockIdx.x], chunk = block_map[2 * blockIdx.x + 1];
    const msamp_bucket_item& d = items[t];
    if (d.reserved == kBucketDone) return;    // written by the speculative first pass with the scale that came out
    const IT* x = static_cast<const IT*>(d.src);
    uint8_t* out = d.dst;
    const float s = *d.scale;
    const size_t n = d.numel, base = static_cast<size_t>(chunk) * MSAMP_BUCKET_CHUNK;
    // a tensor's place in the flat buffer follows from the sizes before it: vector stores only where it allows
    const bool vec = (reinterpret_cast<uintptr_t>(x) & 15) == 0 && (reinterpret_cast<uintptr_t>(out) & (EPT - 1)) == 0;
    if (base + MSAMP_BUCKET_CHUNK <= n && vec) {
        float v[kVecs][EPT];
#pragma unroll
        for (int u = 0; u < kVecs; ++u)
            In16<IT>::load(x + base + (static_cast<size_t>(u) * kBucketThreads + threadIdx.x) * EPT, v[u], stream != 0);
#pragma unroll
        for (int u = 0; u < kVecs; ++u) {
            uint32_t w[EPT / 4];
#pragma unroll
            for (int j = 0; j < EPT / 4; ++j)
                w[j] = quant4<FMT>(v[u][4 * j] * s, v[u][4 * j + 1] * s, v[u][4 * j + 2] * s, v[u][4 * j + 3] * s);
            uint8_t* o = out + base + (static_cast<size_t>(u) * kBucketThreads + threadIdx.x) * EPT;
            if constexpr (EPT == 4) {
                *reinterpret_cast<uint32_t*>(o) = w[0];
            } else {
                *reinterpret_cast<uint2*>(o) = make_uint2(w[0], w[1]);
            }
        }
    } else {
        for (size_t i = base + threadIdx.x; i < n && i < base + MSAMP_BUCKET_CHUNK; i += kBucketThreads)
            out[i] = static_cast<uint8_t>(quant1<FMT>(Elem<IT>::load(x + i) * s));
    }
}

// ---- norms of FP8 gradients (clip_grad_norm_) ----------------------------------------------------------------
// sum |q|^p (p = 1, 2) or max |q| over the codes of each tensor, accumulated in double (four elements at a time are
// summed in float32 first): the dequantization factor
// is constant per tensor and is applied once at the end, so a tensor is read at one byte per element and never
// expanded to float32 in memory.
// (one chunk, into `acc`)
template <int FMT, int KIND>    // KIND: 1, 2, or 0 for the maximum
__device__ __forceinline__ void fp8_norm_chunk(const uint8_t* q, size_t base, size_t n, double& acc) {
    auto take = [&](float v) {
        const double a = fabs(static_cast<double>(v));
        if constexpr (KIND == 0) {
            acc = (a != a || acc != acc) ? (a != a ? a : acc) : (a > acc ? a : acc);    // NaN wins
        } else if constexpr (KIND == 1) {
            acc += a;
        } else {
            acc = fma(a, a, acc);
        }
    };
    if (base + MSAMP_BUCKET_CHUNK <= n && (reinterpret_cast<uintptr_t>(q) & 15) == 0) {
        constexpr int kVecs = MSAMP_BUCKET_CHUNK / (kBucketThreads * 16);    // 4
        uint4 w[kVecs];
#pragma unroll
        for (int u = 0; u < kVecs; ++u)
            w[u] = *reinterpret_cast<const uint4*>(q + base + (static_cast<size_t>(u) * kBucketThreads + threadIdx.x) * 16);
#pragma unroll
        for (int u = 0; u < kVecs; ++u) {
            const uint32_t words[4] = {w[u].x, w[u].y, w[u].z, w[u].w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float a, b, c, f;
                dequant4<FMT>(words[j], a, b, c, f);
                if constexpr (KIND == 0) {
                    take(a), take(b), take(c), take(f);
                } else if constexpr (KIND == 1) {
                    // four values at a time in float32 (three roundings of 2^-24 each), then into the double sum: a
                    // double conversion and addition per element kept the vector units busier than the memory
                    acc += static_cast<double>((fabsf(a) + fabsf(b)) + (fabsf(c) + fabsf(f)));
                } else {
                    // the square of an FP8 value is exact in float32
                    acc += static_cast<double>(fmaf(a, a, b * b) + fmaf(c, c, f * f));
                }
            }
        }
    } else {
        for (size_t i = base + threadIdx.x; i < n && i < base + MSAMP_BUCKET_CHUNK; i += kBucketThreads) take(dequant1<FMT>(q[i]));
    }
}

// ---- clipping a list of gradients (clip_grad_norm_) ----------------------------------------------------------------
// The norms of all gradients of a model, whatever their types (FP8 codes with a scale_inv, or plain float32 / 16-bit
// tensors), their total and the clipping factor in two launches per 64 tensors, and the clipping itself in one, which
// looks at the factor on the device.  Per tensor this was a conversion to float32 with torch.norm or a multiplication
// (two to four launches of 1.3 to 4 us and 6 to 9 us of host time each), and the host waited for the factor.
// The descriptors travel as kernel arguments: no table in memory, no copy, nothing kept between calls.
// 32 FP8 gradients of 4 M codes, quantized as a bucket and clipped: 365 us in all with the calls per tensor, of which the
// GPU worked 150; 110 us now (norms 24 us, finish 5, clipping 4).  A small model's 13 parameters: 0.2 ms a step less.
constexpr int kGradTable = 64;         // 64 descriptors are 1.9 KB of the 4 KB that kernel arguments may take
constexpr int kGradBlocks = MSAMP_GRAD_BLOCKS;    // eight workgroups per compute unit; beyond that each takes a run of chunks
struct GradTable {
    const void* data[kGradTable];
    const float* scale_inv[kGradTable];    // nullptr: a plain tensor
    uint64_t numel[kGradTable];
    int32_t first[kGradTable + 1];         // tensor t has the workgroups first[t] .. first[t + 1] - 1
    uint8_t dtype[kGradTable];
    int32_t n;
};

__device__ __forceinline__ int tensor_of_block(const GradTable& g, int block) {
    int lo = 0, hi = g.n;    // first[lo] <= block < first[hi]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (g.first[mid] <= block) lo = mid; else hi = mid;
    }
    return lo;
}

template <int KIND>
__device__ __forceinline__ double norm_join(double a, double b) {
    if constexpr (KIND == 0) return a != a ? a : (b != b || b > a ? b : a);    // (NaN wins)
    else return a + b;
}

// elements base .. base + MSAMP_BUCKET_CHUNK - 1 of a plain tensor, in double: no square or sum is rounded to float32
template <typename IT, int KIND>
__device__ __forceinline__ void norm_chunk(const IT* x, size_t base, size_t n, double& acc) {
    constexpr int EPT = In16<IT>::EPT;
    auto take = [&](float v) {
        const double a = fabs(static_cast<double>(v));
        if constexpr (KIND == 2) acc = fma(a, a, acc);
        else acc = norm_join<KIND>(acc, a);
    };
    if (base + MSAMP_BUCKET_CHUNK <= n && (reinterpret_cast<uintptr_t>(x) & 15) == 0) {
        constexpr int kVecs = MSAMP_BUCKET_CHUNK / (kBucketThreads * EPT);    // 16 (float32) or 8
#pragma unroll 2
        for (int v = 0; v < kVecs; v += 4) {
            uint4 w[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                w[u] = *reinterpret_cast<const uint4*>(x + base + (static_cast<size_t>(v + u) * kBucketThreads + threadIdx.x) * EPT);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                float f[EPT];
                In16<IT>::decode(w[u], f);
#pragma unroll
                for (int e = 0; e < EPT; ++e) take(f[e]);
            }
        }
    } else {
        for (size_t i = base + threadIdx.x; i < n && i < base + MSAMP_BUCKET_CHUNK; i += kBucketThreads) take(Elem<IT>::load(x + i));
    }
}

// partial[block]: sum of |x|^p (maximum for KIND 0) over the workgroup's run of chunks of its tensor
template <int KIND>
__global__ __launch_bounds__(kBucketThreads) void grad_norm_kernel(GradTable g, double* __restrict__ partial) {
    __shared__ double red[kBucketThreads / kWave];
    const int t = tensor_of_block(g, blockIdx.x);
    const size_t n = g.numel[t], chunks = (n + MSAMP_BUCKET_CHUNK - 1) / MSAMP_BUCKET_CHUNK;
    const size_t blocks = g.first[t + 1] - g.first[t], run = (chunks + blocks - 1) / blocks;
    const size_t from = (blockIdx.x - g.first[t]) * run, to = from + run < chunks ? from + run : chunks;
    const void* x = g.data[t];
    const int dt = g.dtype[t];
    double acc = 0.0;
    for (size_t c = from; c < to; ++c) {
        const size_t base = c * MSAMP_BUCKET_CHUNK;
        if (dt == MSAMP_DT_E4M3) fp8_norm_chunk<MSAMP_DT_E4M3, KIND>(static_cast<const uint8_t*>(x), base, n, acc);
        else if (dt == MSAMP_DT_E5M2) fp8_norm_chunk<MSAMP_DT_E5M2, KIND>(static_cast<const uint8_t*>(x), base, n, acc);
        else if (dt == MSAMP_DT_F32) norm_chunk<float, KIND>(static_cast<const float*>(x), base, n, acc);
        else if (dt == MSAMP_DT_F16) norm_chunk<f16_t, KIND>(static_cast<const f16_t*>(x), base, n, acc);
        else norm_chunk<bf16_t, KIND>(static_cast<const bf16_t*>(x), base, n, acc);
    }
#pragma unroll
    for (int o = 32; o; o >>= 1) acc = norm_join<KIND>(acc, __shfl_xor(acc, o));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kBucketThreads / kWave; ++w) acc = norm_join<KIND>(acc, red[w]);
        partial[blockIdx.x] = acc;
    }
}

// One workgroup: norms[base + t] of the table's tensors, a wavefront each; with `total` also the norm of all norms[0 ..
// base + g.n - 1] and min(1, max_norm / (total + 1e-6)), evaluated as torch does (a reciprocal and a product).
constexpr int kNormFinishThreads = 1024;
template <int KIND>
__global__ __launch_bounds__(kNormFinishThreads) void grad_norm_finish_kernel(GradTable g, const double* __restrict__ partial,
                                                                              float* norms, int base, float* total, float* coef,
                                                                              float max_norm) {
    __shared__ double red[kNormFinishThreads / kWave];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int t = wave; t < g.n; t += kNormFinishThreads / kWave) {
        double acc = 0.0;
        for (int b = g.first[t] + lane; b < g.first[t + 1]; b += 64) acc = norm_join<KIND>(acc, partial[b]);
#pragma unroll
        for (int o = 32; o; o >>= 1) acc = norm_join<KIND>(acc, __shfl_xor(acc, o));
        if (lane == 0) {
            const double root = KIND == 2 ? sqrt(acc) : acc;
            const double si = g.scale_inv[t] != nullptr ? fabs(static_cast<double>(*g.scale_inv[t])) : 1.0;
            norms[base + t] = static_cast<float>(si * root);
        }
    }
    if (total == nullptr) return;
    __syncthreads();
    double acc = 0.0;
    for (int i = threadIdx.x; i < base + g.n; i += kNormFinishThreads) {
        const double v = norms[i];
        acc = KIND == 2 ? fma(v, v, acc) : norm_join<KIND>(acc, v);
    }
#pragma unroll
    for (int o = 32; o; o >>= 1) acc = norm_join<KIND>(acc, __shfl_xor(acc, o));
    if (lane == 0) red[wave] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kNormFinishThreads / kWave; ++w) acc = norm_join<KIND>(acc, red[w]);
        const float norm = static_cast<float>(KIND == 2 ? sqrt(acc) : acc);
        const float recip = 1.0f / (norm + 1e-6f);
        const float c = recip * max_norm;
        *total = norm;
        *coef = c > 1.0f ? 1.0f : c;    // (NaN stays)
    }
}

template <typename IT>
__device__ __forceinline__ void scale_run(IT* x, size_t from, size_t to, float factor) {
    constexpr int EPT = In16<IT>::EPT;
    size_t i = from + static_cast<size_t>(threadIdx.x) * EPT;
    if ((reinterpret_cast<uintptr_t>(x) & 15) == 0) {    // (`from` is a multiple of the chunk)
        for (; i + EPT <= to; i += kBucketThreads * EPT) {
            float f[EPT];
            In16<IT>::load(x + i, f);
            IT o[EPT];
#pragma unroll
            for (int e = 0; e < EPT; ++e) Elem<IT>::store(o + e, f[e] * factor);
            uint4 w;
            __builtin_memcpy(&w, o, 16);
            *reinterpret_cast<uint4*>(x + i) = w;
        }
        if (i < to)
            for (size_t j = i; j < to; ++j) Elem<IT>::store(x + j, Elem<IT>::load(x + j) * factor);
    } else {
        for (size_t j = from + threadIdx.x; j < to; j += kBucketThreads) Elem<IT>::store(x + j, Elem<IT>::load(x + j) * factor);
    }
}

// x *= coef where coef < 1; of an FP8 tensor only its scale_inv.  A 16-bit tensor takes the factor in its own type, as
// torch's product with a zero-dimensional float32 tensor does.
__global__ __launch_bounds__(kBucketThreads) void grad_clip_kernel(GradTable g, const float* __restrict__ coef) {
    const float c = *coef;
    if (!(c < 1.0f)) return;
    const int t = tensor_of_block(g, blockIdx.x);
    if (g.scale_inv[t] != nullptr) {
        if (threadIdx.x == 0) {
            float* si = const_cast<float*>(g.scale_inv[t]);
            *si *= c;
        }
        return;
    }
    const size_t n = g.numel[t], chunks = (n + MSAMP_BUCKET_CHUNK - 1) / MSAMP_BUCKET_CHUNK;
    const size_t blocks = g.first[t + 1] - g.first[t], run = (chunks + blocks - 1) / blocks * MSAMP_BUCKET_CHUNK;
    const size_t from = (blockIdx.x - g.first[t]) * run, to = from + run < n ? from + run : n;
    void* x = const_cast<void*>(g.data[t]);
    const int dt = g.dtype[t];
    if (dt == MSAMP_DT_F32) scale_run(static_cast<float*>(x), from, to, c);
    else if (dt == MSAMP_DT_F16) scale_run(static_cast<f16_t*>(x), from, to, f16_bits_to_float(float_to_f16_bits(c)));
    else scale_run(static_cast<bf16_t*>(x), from, to, bf16_bits_to_float(float_to_bf16_bits(c)));
}

static int check_grads(const char* who, const msamp_grad* grads, int n) {
    MSAMP_REQUIRE(n >= 0, MSAMP_ERR_SHAPE, "%s: n=%d", who, n);
    MSAMP_REQUIRE(n == 0 || grads != nullptr, MSAMP_ERR_NULL, "%s: null table", who);
    for (int i = 0; i < n; ++i) {
        MSAMP_REQUIRE(is_hp(grads[i].dtype) || is_fp8(grads[i].dtype), MSAMP_ERR_DTYPE, "%s: tensor %d: dtype %d", who, i, grads[i].dtype);
        MSAMP_REQUIRE(grads[i].data != nullptr || grads[i].numel == 0, MSAMP_ERR_NULL, "%s: tensor %d: null data", who, i);
        MSAMP_REQUIRE((grads[i].scale_inv != nullptr) == is_fp8(grads[i].dtype), MSAMP_ERR_NULL,
                      "%s: tensor %d: FP8 codes come with a scale_inv, plain tensors without", who, i);
        MSAMP_REQUIRE(aligned(grads[i].data, is_fp8(grads[i].dtype) ? 1 : hp_size(grads[i].dtype)), MSAMP_ERR_SHAPE, "%s: tensor %d: misaligned", who, i);
    }
    return MSAMP_OK;
}
// tensors from .. from + (at most) kGradTable - 1; `run`: chunks per workgroup; scales_only: one workgroup per FP8 tensor
static GradTable grad_table(const msamp_grad* grads, int from, int n, size_t run, bool scales_only) {
    GradTable g = {};
    g.n = std::min(kGradTable, n - from);
    for (int i = 0; i < g.n; ++i) {
        const msamp_grad& e = grads[from + i];
        const size_t chunks = (e.numel + MSAMP_BUCKET_CHUNK - 1) / MSAMP_BUCKET_CHUNK;
        const size_t blocks = scales_only && e.scale_inv != nullptr ? 1 : std::max<size_t>(1, (chunks + run - 1) / run);
        g.data[i] = e.data, g.scale_inv[i] = e.scale_inv, g.numel[i] = e.numel, g.dtype[i] = static_cast<uint8_t>(e.dtype);
        g.first[i + 1] = g.first[i] + static_cast<int32_t>(blocks);
    }
    return g;
}
static size_t grad_run(const msamp_grad* grads, int n) {
    size_t chunks = 0;
    for (int i = 0; i < n; ++i) chunks += (grads[i].numel + MSAMP_BUCKET_CHUNK - 1) / MSAMP_BUCKET_CHUNK;
    return std::max<size_t>(1, (chunks + kGradBlocks - 1) / kGradBlocks);
}

static int check_bucket_args(const char* who, const msamp_bucket_item* items, int n_items, const int32_t* block_map,
                             int n_blocks, int in_dtype) {
    MSAMP_REQUIRE(n_items >= 0 && n_blocks >= 0, MSAMP_ERR_SHAPE, "%s: n_items=%d n_blocks=%d", who, n_items, n_blocks);
    MSAMP_REQUIRE(is_hp(in_dtype), MSAMP_ERR_DTYPE, "%s: in_dtype %d", who, in_dtype);
    MSAMP_REQUIRE(n_items == 0 || items != nullptr, MSAMP_ERR_NULL, "%s: null descriptor table", who);
    MSAMP_REQUIRE(n_blocks == 0 || block_map != nullptr, MSAMP_ERR_NULL, "%s: null block map", who);
    return MSAMP_OK;
}

}    // namespace msamp

using namespace msamp;

extern "C" {

static int bucket_amax_launch(const char* who, msamp_bucket_item* items, int n_items, const int32_t* block_map, int n_blocks,
                              int in_dtype, int fp8_type, int flags, msamp_stream_t stream) {
    const int rc = check_bucket_args(who, items, n_items, block_map, n_blocks, in_dtype);
    if (rc != MSAMP_OK || n_items == 0) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    // more bytes than the caches keep: read them as a stream
    const int in_size = in_dtype == MSAMP_DT_F32 ? 4 : 2;
    const int streams = static_cast<size_t>(n_blocks) * MSAMP_BUCKET_CHUNK * in_size >= kStreamBytes ? 1 : 0;
    if (n_blocks > 0) {
#define BUCKET_AMAX(IT)                                                                                                 \
    do {                                                                                                              \
        if (fp8_type == MSAMP_DT_E4M3)                                                                                \
            hipLaunchKernelGGL((bucket_amax_kernel<IT, MSAMP_DT_E4M3>), dim3(n_blocks), dim3(kBucketThreads), 0, st, items, block_map, streams); \
        else if (fp8_type == MSAMP_DT_E5M2)                                                                           \
            hipLaunchKernelGGL((bucket_amax_kernel<IT, MSAMP_DT_E5M2>), dim3(n_blocks), dim3(kBucketThreads), 0, st, items, block_map, streams); \
        else                                                                                                          \
            hipLaunchKernelGGL((bucket_amax_kernel<IT, 0>), dim3(n_blocks), dim3(kBucketThreads), 0, st, items, block_map, streams); \
    } while (0)
        if (in_dtype == MSAMP_DT_F32) BUCKET_AMAX(float);
        else if (in_dtype == MSAMP_DT_F16) BUCKET_AMAX(f16_t);
        else BUCKET_AMAX(bf16_t);
#undef BUCKET_AMAX
        MSAMP_CHECK_LAUNCH("bucket_amax_kernel");
    }
    hipLaunchKernelGGL(bucket_amax_finish_kernel, dim3((n_items + 63) / 64), dim3(64), 0, st, items, n_items, flags,
                       fp8_type != 0 ? 1 : 0);
    MSAMP_CHECK_LAUNCH("bucket_amax_finish_kernel");
    return MSAMP_OK;
}

int msamp_bucket_amax(msamp_bucket_item* items, int n_items, const int32_t* block_map, int n_blocks, int in_dtype, int flags,
                      msamp_stream_t stream) {
    return bucket_amax_launch("msamp_bucket_amax", items, n_items, block_map, n_blocks, in_dtype, 0, flags, stream);
}

int msamp_bucket_amax_speculative(msamp_bucket_item* items, int n_items, const int32_t* block_map, int n_blocks, int in_dtype,
                                  int fp8_type, int flags, msamp_stream_t stream) {
    MSAMP_REQUIRE(is_fp8(fp8_type), MSAMP_ERR_DTYPE, "msamp_bucket_amax_speculative: fp8_type %d", fp8_type);
    return bucket_amax_launch("msamp_bucket_amax_speculative", items, n_items, block_map, n_blocks, in_dtype, fp8_type, flags,
                              stream);
}

int msamp_bucket_cast(msamp_bucket_item* items, int n_items, const int32_t* block_map, int n_blocks, int in_dtype,
                      int fp8_type, float pre_scale, float scale_inv_div, int margin, msamp_stream_t stream) {
    const int rc = check_bucket_args("msamp_bucket_cast", items, n_items, block_map, n_blocks, in_dtype);
    if (rc != MSAMP_OK) return rc;
    MSAMP_REQUIRE(is_fp8(fp8_type), MSAMP_ERR_DTYPE, "msamp_bucket_cast: fp8_type %d", fp8_type);
    if (n_items == 0) return MSAMP_OK;
    hipStream_t st = static_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(bucket_scale_kernel, dim3((n_items + 63) / 64), dim3(64), 0, st, items, n_items, fp8_max(fp8_type),
                       margin, pre_scale, scale_inv_div);
    MSAMP_CHECK_LAUNCH("bucket_scale_kernel");
    if (n_blocks == 0) return MSAMP_OK;
    const int in_size = in_dtype == MSAMP_DT_F32 ? 4 : 2;
    const int streams = static_cast<size_t>(n_blocks) * MSAMP_BUCKET_CHUNK * in_size >= kStreamBytes ? 1 : 0;
#define BUCKET_CAST(IT)                                                                                                  \
    do {                                                                                                               \
        if (fp8_type == MSAMP_DT_E4M3)                                                                                 \
            hipLaunchKernelGGL((bucket_cast_kernel<IT, MSAMP_DT_E4M3>), dim3(n_blocks), dim3(kBucketThreads), 0, st, items, block_map, streams); \
        else                                                                                                           \
            hipLaunchKernelGGL((bucket_cast_kernel<IT, MSAMP_DT_E5M2>), dim3(n_blocks), dim3(kBucketThreads), 0, st, items, block_map, streams); \
    } while (0)
    if (in_dtype == MSAMP_DT_F32) BUCKET_CAST(float);
    else if (in_dtype == MSAMP_DT_F16) BUCKET_CAST(f16_t);
    else BUCKET_CAST(bf16_t);
#undef BUCKET_CAST
    MSAMP_CHECK_LAUNCH("bucket_cast_kernel");
    return MSAMP_OK;
}

int msamp_grad_norms(const msamp_grad* grads, int n, int norm_kind, float max_norm, double* partials, float* norms, float* total,
                     float* coef, msamp_stream_t stream) {
    const int rc = check_grads("msamp_grad_norms", grads, n);
    if (rc != MSAMP_OK) return rc;
    MSAMP_REQUIRE(norm_kind >= 0 && norm_kind <= 2, MSAMP_ERR_SHAPE, "msamp_grad_norms: norm_kind %d (1, 2, or 0 for the maximum)",
                  norm_kind);
    MSAMP_REQUIRE(n > 0 && partials && norms && total && coef, MSAMP_ERR_NULL, "msamp_grad_norms: nothing to do or null pointer");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const size_t run = grad_run(grads, n);
    for (int from = 0; from < n; from += kGradTable) {
        const GradTable g = grad_table(grads, from, n, run, false);
        const bool last = from + g.n == n;
        float* total_out = last ? total : nullptr;
#define NORM_LAUNCH(KIND)                                                                                                 \
    do {                                                                                                                \
        hipLaunchKernelGGL((grad_norm_kernel<KIND>), dim3(g.first[g.n]), dim3(kBucketThreads), 0, st, g, partials);        \
        MSAMP_CHECK_LAUNCH("grad_norm_kernel");                                                                         \
        hipLaunchKernelGGL((grad_norm_finish_kernel<KIND>), dim3(1), dim3(kNormFinishThreads), 0, st, g, partials, norms, from, total_out, coef, max_norm); \
        MSAMP_CHECK_LAUNCH("grad_norm_finish_kernel");                                                                  \
    } while (0)
        if (norm_kind == 0) NORM_LAUNCH(0); else if (norm_kind == 1) NORM_LAUNCH(1); else NORM_LAUNCH(2);
#undef NORM_LAUNCH
    }
    return MSAMP_OK;
}

int msamp_grad_clip(const msamp_grad* grads, int n, const float* coef, msamp_stream_t stream) {
    const int rc = check_grads("msamp_grad_clip", grads, n);
    if (rc != MSAMP_OK || n == 0) return rc;
    MSAMP_REQUIRE(coef != nullptr, MSAMP_ERR_NULL, "msamp_grad_clip: null factor");
    const size_t run = grad_run(grads, n);
    for (int from = 0; from < n; from += kGradTable) {
        const GradTable g = grad_table(grads, from, n, run, true);
        hipLaunchKernelGGL(grad_clip_kernel, dim3(g.first[g.n]), dim3(kBucketThreads), 0, static_cast<hipStream_t>(stream), g, coef);
        MSAMP_CHECK_LAUNCH("grad_clip_kernel");
    }
    return MSAMP_OK;
}

}    // extern "C"
