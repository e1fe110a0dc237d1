// Prologue of the attention processor: projected rows into the head-major Q/K/V buffer
// (peco/processor.py:159-190), the per-channel RMS norm and the rotary embedding of the video rows
// applied on the way.
//
// A tensor [batch, heads, rows, D] (any strides, channels adjacent) goes to rows
// [first, first + rows) of a head-major buffer [batch, heads, length, D]. With tables cos/sin
// (fp32 [rows, D]) its rows are rotated over interleaved channel pairs, each step one fp32
// operation and one rounding to the dtype at the end, as the torch expression
//   (x.float() * cos + rotated.float() * sin).to(x.dtype), rotated = (-x1, x0) per pair
// computes it, so the results are the same bits. With a norm the rows are divided by their root mean
// square and multiplied by the channel weights first, in fp32 with one rounding to the dtype: the
// bits the block's torch.nn.RMSNorm would have stored.
//
// HBM-bound: a row of a head is G = D / 8 lanes of 16 bytes; a lane takes the same row of
// kPlaceHeads heads with all loads in flight, so the row's table values are read once per that many
// heads. 24 heads x 6750 rows x 128 channels: 20 us per tensor (83 MB, 4.2 TB/s of the 5.2 a plain
// copy reaches), about 60 us for Q, K and V; the torch operations it replaces (copies that split the
// heads, a dozen passes for the rotary embedding, most in fp32) took about 0.6 ms of the call. The
// norm costs a reduction over the row's lanes by DPP moves and no memory pass; as a module of its own
// it took 118 us per tensor of that shape (0.7 TB/s), the launch with it takes 22 us; the whole
// double-stream call 1870 -> 1550 us.
#include "common.hpp"

namespace peco {
namespace {

constexpr int kPlaceHeads = 8;

struct PlaceArgs {
    const uint16_t* in;
    uint16_t* out;        // first destination row of batch entry 0, head 0
    int64_t sb, sh, sr;   // input strides (elements) of batch, head, row
    const float* cos;     // nullable: no rotation
    const float* sin;
    const uint16_t* weight;  // nullable: RMS norm without channel weights
    float eps;
    int norm;
    int heads, rows;
    int64_t out_head;     // elements between heads of the output (length * D)
};

// Sums of squares over a row of G = 8 or 16 adjacent lanes, 8 channels each, in the order torch's RMS
// norm takes on this GPU (found from the inverse root it returns, aten::_fused_rms_norm): groups of
// four channels in turn, then groups half the row apart, a quarter, ..., adjacent ones.
template <int kCtrl> __device__ __forceinline__ float dpp_add(float v) {
    return v + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), kCtrl, 0xf, 0xf, false));
}
template <int G> __device__ __forceinline__ float row_squares(const float (&v)[8]) {
    float s[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        s[h] = v[4 * h] * v[4 * h];  // (products of 16-bit values are exact)
#pragma unroll
        for (int k = 1; k < 4; ++k) s[h] += v[4 * h + k] * v[4 * h + k];
        if constexpr (G == 16) {
            s[h] = dpp_add<0x128>(s[h]);  // row_ror:8, the lane 8 away
            s[h] = dpp_add<0x124>(s[h]);  // row_ror:4, the lane 4 away (sums repeat every 8 lanes)
        } else {
            const int bits = __float_as_int(s[h]);  // the lane 4 away: row_shl:4 and row_shr:4, each for half the quads
            const int low = __builtin_amdgcn_update_dpp(0, bits, 0x104, 0xf, 0x5, false);
            s[h] += __int_as_float(__builtin_amdgcn_update_dpp(low, bits, 0x114, 0xf, 0xa, false));
        }
        s[h] = dpp_add<0x4e>(s[h]);  // quad_perm [2, 3, 0, 1]
        s[h] = dpp_add<0xb1>(s[h]);  // quad_perm [1, 0, 3, 2]
    }
    return s[0] + s[1];
}

template <int DT, int D>
__global__ __launch_bounds__(256) void place_heads_kernel(PlaceArgs a) {
    constexpr int G = D / 8;
    const int b = blockIdx.z;
    const int row = blockIdx.x * (256 / G) + threadIdx.x / G;
    if (row >= a.rows) return;
    const int c0 = (threadIdx.x % G) * 8;
    const int h0 = blockIdx.y * kPlaceHeads;
    const uint16_t* src = a.in + b * a.sb + static_cast<int64_t>(row) * a.sr + c0;
    u16x8 x[kPlaceHeads];
#pragma unroll
    for (int i = 0; i < kPlaceHeads; ++i)  // clamped, unconditional: all loads in flight
        x[i] = *reinterpret_cast<const u16x8*>(src + static_cast<int64_t>(min(h0 + i, a.heads - 1)) * a.sh);
    if (a.norm) {
        float w[8];
        if (a.weight) {
            const u16x8 wv = *reinterpret_cast<const u16x8*>(a.weight + c0);
#pragma unroll
            for (int k = 0; k < 8; ++k) w[k] = half_to_f32<DT>(wv[k]);
        } else {
#pragma unroll
            for (int k = 0; k < 8; ++k) w[k] = 1.0f;
        }
#pragma unroll
        for (int i = 0; i < kPlaceHeads; ++i) {
            float v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = half_to_f32<DT>(x[i][k]);
            const float inverse = __builtin_amdgcn_rsqf(row_squares<G>(v) * (1.0f / D) + a.eps);  // as torch's
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                float y = v[k] * inverse * w[k];
                asm("" : "+v"(y));  // rounded to fp32 before the dtype (a mixed-precision product would round once)
                x[i][k] = f32_to_half<DT>(y);
            }
        }
    }
    if (a.cos) {
        float c[8], s[8];
        const int64_t e = static_cast<int64_t>(row) * D + c0;
#pragma unroll
        for (int k = 0; k < 8; k += 4) {
            const f32x4 cv = *reinterpret_cast<const f32x4*>(a.cos + e + k);
            const f32x4 sv = *reinterpret_cast<const f32x4*>(a.sin + e + k);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                c[k + i] = cv[i];
                s[k + i] = sv[i];
            }
        }
#pragma unroll
        for (int i = 0; i < kPlaceHeads; ++i)
#pragma unroll
            for (int k = 0; k < 8; k += 2) {
                const float re = half_to_f32<DT>(x[i][k]), im = half_to_f32<DT>(x[i][k + 1]);
                const float re_c = re * c[k], im_s = -im * s[k];
                const float im_c = im * c[k + 1], re_s = re * s[k + 1];
                x[i][k] = f32_to_half<DT>(re_c + im_s);
                x[i][k + 1] = f32_to_half<DT>(im_c + re_s);
            }
    }
    uint16_t* dst = a.out + (static_cast<int64_t>(b) * a.heads + h0) * a.out_head + static_cast<int64_t>(row) * D + c0;
#pragma unroll
    for (int i = 0; i < kPlaceHeads; ++i)
        if (h0 + i < a.heads) *reinterpret_cast<u16x8*>(dst + i * a.out_head) = x[i];
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

}  // namespace
}  // namespace peco

using namespace peco;

PECO_API int peco_place_heads(const void* input, int64_t stride_batch, int64_t stride_head, int64_t stride_row,
                              void* output, const float* cos, const float* sin, int norm, const void* weight, float eps,
                              int batch, int heads, int rows, int first, int length, int dims, int dtype,
                              void* stream) {
    if (!input || !output || !cos != !sin || (weight && !norm) || batch < 1 || heads < 1 || rows < 1 || first < 0 || length < rows ||
        first > length - rows)
        return kInvalidValue;
    if (dims != 64 && dims != 128) return kUnsupportedShape;
    if (dtype != kBF16 && dtype != kF16) return kUnsupportedDtype;
    if (batch > 65535 || ceil_div(heads, kPlaceHeads) > 65535) return kUnsupportedShape;
    // 16-byte loads and stores: every row of every head must start on one.
    if (!aligned16(input) || !aligned16(output) || !aligned16(cos) || !aligned16(sin) || !aligned16(weight) ||
        stride_batch % 8 || stride_head % 8 || stride_row % 8)
        return kInvalidValue;
    PlaceArgs a{};
    a.in = static_cast<const uint16_t*>(input);
    a.out = static_cast<uint16_t*>(output) + static_cast<int64_t>(first) * dims;
    a.sb = stride_batch;
    a.sh = stride_head;
    a.sr = stride_row;
    a.cos = cos;
    a.sin = sin;
    a.weight = static_cast<const uint16_t*>(weight);
    a.eps = eps;
    a.norm = norm;
    a.heads = heads;
    a.rows = rows;
    a.out_head = static_cast<int64_t>(length) * dims;
    const dim3 grid(static_cast<unsigned>(ceil_div(rows, 256 / (dims / 8))),
                    static_cast<unsigned>(ceil_div(heads, kPlaceHeads)), static_cast<unsigned>(batch));
    const auto s = static_cast<hipStream_t>(stream);
#define PECO_PLACE(DT_, D_) hipLaunchKernelGGL((place_heads_kernel<DT_, D_>), grid, dim3(256), 0, s, a)
    if (dtype == kBF16) {
        if (dims == 128) PECO_PLACE(kBF16, 128);
        else PECO_PLACE(kBF16, 64);
    } else {
        if (dims == 128) PECO_PLACE(kF16, 128);
        else PECO_PLACE(kF16, 64);
    }
#undef PECO_PLACE
    return hipGetLastError();
}
