// Stage 2: Base-Offset PE centroid-residual quantizer (peco/quantization.py:97-150),
// plus the fused "pack" kernel that applies it while gathering Q/K/V into cluster order
// and appending the unsorted text rows (peco/processor.py:141-149).
//
// The per-token arithmetic (base_offset.hpp) is one IEEE operation per step, in the torch
// reference's order.
//
// Layout: a token row of D elements is handled by G = D/8 lanes (8 elements per lane,
// 16-byte loads for 16-bit inputs), so one wavefront covers 64/G rows and min/max are
// reduced with log2(G) xor-shuffles inside the lane group. HBM-bound streaming kernel.
#include "base_offset.hpp"
#include "common.hpp"

#include <algorithm>

namespace peco {
namespace {

// Standalone quantizer and decoder. A workgroup takes kQuantPasses passes of 256 / G consecutive rows
// of one batch entry: the labels of every pass are requested first, then the rows, then the
// centres the labels select, so one group of lanes has four rows in flight and no thread divides a
// 64-bit row index. With a batch divisible by the XCD count entry b runs on XCD b % kXcdCount, whose
// L2 then fetches only its own entries' centres. 24 x 6750 x 128 bf16 rows, 4 bits: 18
// us to encode (62 MB) or fake-quantize (83 MB, 4.6 TB/s), 14.5 to decode (4.3 TB/s); one row per
// group and step took 20.5, 20.5 and 16.3.
constexpr int kQuantPasses = 4;

struct QuantArgs {
    const void* x;            // encode: [batch, tokens, D]
    const void* labels;       // [batch, tokens]
    const float* centroids;   // [batch, clusters, D]
    uint8_t* codes;           // encode: nullable output; decode: input
    float* low;
    float* scale;
    void* xhat;               // encode: nullable
    int batch, tokens, clusters, per_batch;
    float levels;
};

template <typename L, int G> struct QuantRows {
    static constexpr int R = 256 / G;
    int b, t0, sub;
    int64_t row0;
    const float* cent;
    int label[kQuantPasses];
    __device__ __forceinline__ QuantRows(const QuantArgs& a) {
        int chunk;
        const int block = blockIdx.x;
        if (a.batch % kXcdCount == 0) {
            const int slot = block / kXcdCount;
            b = block % kXcdCount + kXcdCount * (slot / a.per_batch);
            chunk = slot % a.per_batch;
        } else {
            b = block / a.per_batch;
            chunk = block % a.per_batch;
        }
        t0 = chunk * R * kQuantPasses + static_cast<int>(threadIdx.x) / G;
        sub = threadIdx.x % G;
        row0 = static_cast<int64_t>(b) * a.tokens;
        cent = a.centroids + static_cast<int64_t>(b) * a.clusters * (G * 8) + sub * 8;
#pragma unroll
        for (int u = 0; u < kQuantPasses; ++u) {  // clamped: every load is unconditional
            const L v = static_cast<const L*>(a.labels)[row0 + min(t0 + u * R, a.tokens - 1)];
            // Out-of-range labels (never valid input) read the last centre instead of past the end.
            label[u] = static_cast<int>(min(static_cast<uint64_t>(static_cast<int64_t>(v)),
                                            static_cast<uint64_t>(a.clusters - 1)));
        }
    }
    __device__ __forceinline__ int64_t at(const QuantArgs& a, int u) const { return row0 + min(t0 + u * R, a.tokens - 1); }
    __device__ __forceinline__ bool valid(const QuantArgs& a, int u) const { return t0 + u * R < a.tokens; }
};

template <int DT, int G, typename L>
__global__ __launch_bounds__(256) void base_offset_kernel(QuantArgs a) {
    constexpr int D = G * 8;
    const QuantRows<L, G> q(a);
    float x[kQuantPasses][8], c[kQuantPasses][8];
#pragma unroll
    for (int u = 0; u < kQuantPasses; ++u) Row8<DT>::load(a.x, q.at(a, u) * D + q.sub * 8, x[u]);
#pragma unroll
    for (int u = 0; u < kQuantPasses; ++u) load_centroid8(q.cent + static_cast<int64_t>(q.label[u]) * D, c[u]);
#pragma unroll
    for (int u = 0; u < kQuantPasses; ++u) {
        float out[8], lo, sc;
        uint8_t k[8];
        base_offset_lane<G>(x[u], c[u], a.levels, out, k, lo, sc);
        if (!q.valid(a, u)) continue;
        const int64_t row = q.at(a, u);
        if (a.codes) {
            u32x2 packed;
            packed[0] = k[0] | (k[1] << 8) | (k[2] << 16) | (static_cast<uint32_t>(k[3]) << 24);
            packed[1] = k[4] | (k[5] << 8) | (k[6] << 16) | (static_cast<uint32_t>(k[7]) << 24);
            *reinterpret_cast<u32x2*>(a.codes + row * D + q.sub * 8) = packed;
        }
        if (q.sub == 0) {
            if (a.low) a.low[row] = lo;
            if (a.scale) a.scale[row] = sc;
        }
        if (a.xhat) Row8<DT>::store(a.xhat, row * D + q.sub * 8, out);
    }
}

template <int DT, int G, typename L>
__global__ __launch_bounds__(256) void base_offset_decode_kernel(QuantArgs a) {
    constexpr int D = G * 8;
    const QuantRows<L, G> q(a);
    u32x2 packed[kQuantPasses];
    float lo[kQuantPasses], sc[kQuantPasses], c[kQuantPasses][8];
#pragma unroll
    for (int u = 0; u < kQuantPasses; ++u) {
        packed[u] = *reinterpret_cast<const u32x2*>(a.codes + q.at(a, u) * D + q.sub * 8);
        lo[u] = a.low[q.at(a, u)];
        sc[u] = a.scale[q.at(a, u)];
    }
#pragma unroll
    for (int u = 0; u < kQuantPasses; ++u) load_centroid8(q.cent + static_cast<int64_t>(q.label[u]) * D, c[u]);
#pragma unroll
    for (int u = 0; u < kQuantPasses; ++u) {
        if (!q.valid(a, u)) continue;
        float out[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t code = (packed[u][i / 4] >> (8 * (i % 4))) & 0xffu;
            const float step = sc[u] * static_cast<float>(code);
            const float resid = lo[u] + step;
            out[i] = c[u][i] + resid;
        }
        Row8<DT>::store(a.xhat, q.at(a, u) * D + q.sub * 8, out);
    }
}

}  // namespace

struct PackTensor {
    const void* input;        // [batch, length, dims]
    void* output;             // [batch, length, dims]
    const int32_t* indices;   // [batch, video]: original video token at each packed position
    const int32_t* labels;    // [batch, video] (read only when bits != 0)
    const float* centroids;   // [batch, clusters, dims] (read only when bits != 0)
    int clusters;
    int bits;                 // 0 = plain gather, 4 or 8 = fake-quantize while gathering
};

struct PackArgs {
    PackTensor t[3];
    int num, batch, length, video;
};

namespace {

template <int DT, int G>
// Grid (row tiles, batch, tensor): 16-lane groups (G lanes) own one output row each, so no
// thread divides a linear index.
__global__ __launch_bounds__(256) void pack_kernel(PackArgs a) {
    constexpr int D = G * 8;
    const int sub = threadIdx.x % G;
    const int j = static_cast<int>(blockIdx.x) * (256 / G) + static_cast<int>(threadIdx.x) / G;
    if (j >= a.length) return;
    const int64_t b = blockIdx.y;
    const PackTensor& T = a.t[blockIdx.z];
    const int64_t row = b * a.length + j;
    const int64_t dst = row * D + sub * 8;
    if (j >= a.video) {
        Row8<DT>::copy(T.input, dst, T.output, dst);
        return;
    }
    const int tok = T.indices[b * a.video + j];
    const int64_t src = (b * a.length + tok) * D + sub * 8;
    if (T.bits == 0) {
        Row8<DT>::copy(T.input, src, T.output, dst);
        return;
    }
    const int lab = T.labels[b * a.video + tok];
    float xv[8], cv[8], out[8], lo, sc;
    uint8_t q[8];
    Row8<DT>::load(T.input, src, xv);
    load_centroid8(T.centroids + (b * T.clusters + lab) * D + sub * 8, cv);
    base_offset_lane<G>(xv, cv, static_cast<float>((1 << T.bits) - 1), out, q, lo, sc);
    Row8<DT>::store(T.output, dst, out);
}

template <bool kDecode, typename L>
int launch_quant(QuantArgs a, int dtype, int dims, hipStream_t s) {
    const int G = dims / 8;
    a.per_batch = static_cast<int>(ceil_div(a.tokens, 256 / G * kQuantPasses));
    const int64_t blocks = static_cast<int64_t>(a.batch) * a.per_batch;
    if (blocks > 0x7fffffff) return kUnsupportedShape;
#define PECO_LAUNCH(DT_, G_)                                                                                        \
    do {                                                                                                            \
        if constexpr (kDecode)                                                                                      \
            hipLaunchKernelGGL((base_offset_decode_kernel<DT_, G_, L>), dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s, a); \
        else                                                                                                        \
            hipLaunchKernelGGL((base_offset_kernel<DT_, G_, L>), dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s, a); \
        return hipGetLastError();                                                                                   \
    } while (0)
    if (dtype == kBF16) {
        if (G == 16) PECO_LAUNCH(kBF16, 16);
        PECO_LAUNCH(kBF16, 8);
    } else if (dtype == kF16) {
        if (G == 16) PECO_LAUNCH(kF16, 16);
        PECO_LAUNCH(kF16, 8);
    } else if (dtype == kF32) {
        if (G == 16) PECO_LAUNCH(kF32, 16);
        PECO_LAUNCH(kF32, 8);
    }
#undef PECO_LAUNCH
    return kUnsupportedDtype;
}

bool valid_quant_args(int batch, int tokens, int clusters, int dims, int label_bytes) {
    return batch >= 1 && tokens >= 1 && clusters >= 1 && (dims == 64 || dims == 128) &&
           (label_bytes == 4 || label_bytes == 8);
}

}  // namespace
}  // namespace peco

using namespace peco;

PECO_API int peco_base_offset_apply(const void* x, int dtype, const void* labels, int label_bytes, const float* centroids,
                                    int batch, int tokens, int clusters, int dims, int bits, uint8_t* codes, float* low,
                                    float* scale, void* xhat, void* stream) {
    if (!x || !labels || !centroids || !valid_quant_args(batch, tokens, clusters, dims, label_bytes) ||
        (bits != 4 && bits != 8))
        return kInvalidValue;
    const QuantArgs a{x, labels, centroids, codes, low, scale, xhat, batch, tokens, clusters, 0,
                      static_cast<float>((1 << bits) - 1)};
    const auto s = static_cast<hipStream_t>(stream);
    return label_bytes == 4 ? launch_quant<false, int32_t>(a, dtype, dims, s)
                            : launch_quant<false, int64_t>(a, dtype, dims, s);
}

PECO_API int peco_base_offset_reconstruct(const uint8_t* codes, const float* low, const float* scale, const void* labels,
                                          int label_bytes, const float* centroids, int batch, int tokens, int clusters,
                                          int dims, int dtype, void* out, void* stream) {
    if (!codes || !low || !scale || !labels || !centroids || !out ||
        !valid_quant_args(batch, tokens, clusters, dims, label_bytes))
        return kInvalidValue;
    const QuantArgs a{nullptr, labels, centroids, const_cast<uint8_t*>(codes), const_cast<float*>(low),
                      const_cast<float*>(scale), out, batch, tokens, clusters, 0, 0.0f};
    const auto s = static_cast<hipStream_t>(stream);
    return label_bytes == 4 ? launch_quant<true, int32_t>(a, dtype, dims, s)
                            : launch_quant<true, int64_t>(a, dtype, dims, s);
}

PECO_API int peco_base_offset_encode(const void* x, int dtype, const int32_t* labels, const float* centroids,
                                     int batch, int tokens, int clusters, int dims, int bits, uint8_t* codes,
                                     float* low, float* scale, void* stream) {
    return peco_base_offset_apply(x, dtype, labels, 4, centroids, batch, tokens, clusters, dims, bits, codes, low, scale,
                                  nullptr, stream);
}

PECO_API int peco_base_offset_decode(const uint8_t* codes, const float* low, const float* scale,
                                     const int32_t* labels, const float* centroids, int batch, int tokens,
                                     int clusters, int dims, int dtype, void* out, void* stream) {
    return peco_base_offset_reconstruct(codes, low, scale, labels, 4, centroids, batch, tokens, clusters, dims, dtype,
                                        out, stream);
}

PECO_API int peco_base_offset_fake_quant(const void* x, int dtype, const int32_t* labels, const float* centroids,
                                         int batch, int tokens, int clusters, int dims, int bits, void* out,
                                         void* stream) {
    if (!out) return kInvalidValue;
    return peco_base_offset_apply(x, dtype, labels, 4, centroids, batch, tokens, clusters, dims, bits, nullptr, nullptr,
                                  nullptr, out, stream);
}

// One launch packs up to three tensors (Q, K, V) of shape [batch, length, dims]:
// rows [0, video) are gathered in cluster order (optionally fake-quantized),
// rows [video, length) (text) are copied in place.
PECO_API int peco_pack_clustered(const void* const* inputs, void* const* outputs, const int32_t* const* indices,
                                 const int32_t* const* labels, const float* const* centroids, const int* clusters,
                                 const int* bits, int num_tensors, int batch, int length, int video, int dims,
                                 int dtype, void* stream) {
    if (num_tensors < 1 || num_tensors > 3 || batch < 1 || length < 1 || video < 0 || video > length ||
        (dims != 64 && dims != 128))
        return kInvalidValue;
    PackArgs a{};
    a.num = num_tensors;
    a.batch = batch;
    a.length = length;
    a.video = video;
    for (int i = 0; i < num_tensors; ++i) {
        if (!inputs[i] || !outputs[i] || (video > 0 && !indices[i])) return kInvalidValue;
        if (bits[i] != 0 && bits[i] != 4 && bits[i] != 8) return kInvalidValue;
        if (bits[i] != 0 && (!labels[i] || !centroids[i] || clusters[i] < 1)) return kInvalidValue;
        a.t[i] = PackTensor{inputs[i], outputs[i], indices[i], labels[i], centroids[i], clusters[i], bits[i]};
    }
    if (batch > 65535) return kUnsupportedShape;
    const int G = dims / 8;
    const dim3 grid(static_cast<unsigned>(ceil_div(length, 256 / G)), static_cast<unsigned>(batch),
                    static_cast<unsigned>(num_tensors));
    const hipStream_t s = static_cast<hipStream_t>(stream);
#define PECO_PACK(DT_)                                                                   \
    do {                                                                                 \
        if (G == 16) hipLaunchKernelGGL((pack_kernel<DT_, 16>), grid, dim3(256), 0, s, a); \
        else hipLaunchKernelGGL((pack_kernel<DT_, 8>), grid, dim3(256), 0, s, a);          \
    } while (0)
    if (dtype == kBF16) PECO_PACK(kBF16);
    else if (dtype == kF16) PECO_PACK(kF16);
    else if (dtype == kF32) PECO_PACK(kF32);
    else return kUnsupportedDtype;
#undef PECO_PACK
    return hipGetLastError();
}
