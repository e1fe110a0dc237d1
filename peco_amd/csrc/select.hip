// Cluster-pair selection (peco/clustering.py:140-186) and the text partition
// (peco/processor.py:68-84) in one launch.
//
// One wavefront per (batch*head, query cluster) row:
//   score_j = (Cq . Ck_j) * fl(D^-0.5)                (fma chain over d ascending)
//   logit_j = score_j + log(count_j), or -inf for an empty key cluster
//   prob_j  = exp(logit_j - rowmax) / max(sum, FLT_MIN) (rowmax = 0 when no key is non-empty)
//   order   = probabilities descending, ties by ascending index (torch's stable sort)
//   keep_k  = (cumsum_k - prob_k) < p over that order, cumsum accumulated in double and
//             rounded per element (torch's CPU cumsum); p == 1 keeps all; the first
//             max(1, minimum) entries are always kept
//   map[c, j] = keep && count_j > 0 && qcount_c > 0
// With `extend`, the map gains the valid-text and padding groups: the valid-text row and
// column pair with everything but padding, padding pairs only with itself, and the size
// vectors gain (valid_text, text - valid_text).
//
// Layout: a workgroup of kSelWaves waves owns kSelWaves query rows of one batch entry.
// Scores: the key centroids stream through LDS in chunks of (up to 512 keys) x (C channels), so a
// key value is read from LDS once per workgroup row group instead of once per row: a wave holds two
// keys per lane and up to four query rows (8 independent fma chains). The finished dots go through
// LDS to the row layout: wave = row, lane l holds keys l, l + 64, ...
//
// The kept set is a prefix of the sorted order: with probabilities descending and the
// running sum nondecreasing, cum_{k+1} - prob_{k+1} >= cum_k - prob_k exactly, so the
// rounded `before` values are nondecreasing too. So the row is not sorted: a binary search over
// the probability bits finds the value v at which the prefix ends (every lane holds its keys, a
// step is a count by ballots and one wave sum), and the decision at the boundary is then made on
// the reference's own quantities. The cumulative sum enters only as fl32(cum): with D the double
// sum (in any order) of the prefix, |D - cum| < kCumEps, so when D - kCumEps and D + kCumEps
// decide alike, the sequential sum decides so too. Checked are the last entry above v (must be
// kept), every entry equal to v (in index order) and, when all of those are kept, the first
// entry below (must not be). A boundary the float sums of the search placed one value off is moved;
// a decision that stays open, or a row with non-finite mass, takes the sequential walk itself.
// Bound by latency: a few dependent phases of one to two workgroups per CU. Launch times (work-list
// form, 128 channels; before: one wave per row reading every key row from LDS for itself, a sort of
// 64-bit keys, the sequential walk, 196 VGPRs and so one workgroup per CU): 24 heads x 64 rows x
// 256 keys 27 us (37 before), 100 x 500 43 us (102), 128 x 512 52 us (113), 256 x 1024 147 us (366).
#include "common.hpp"
#include "work.hpp"

#include <algorithm>
#include <cmath>

namespace peco {
namespace {

constexpr int kSelWaves = 8;
constexpr int kSelThreads = kSelWaves * kWave;
constexpr int kSelBlock = 64;
constexpr int kSelMaxDims = 256;
constexpr int kSelStage = 16;  // staged floats per thread and chunk

// Shapes of the score phase for KPL keys per lane of a row.
template <int KPL> struct SelTiles {
    static constexpr int kBlocks = KPL < 8 ? KPL : 8;              // 64-key blocks per pass
    static constexpr int kPasses = KPL / kBlocks;
    static constexpr int kKeys = kSelBlock * kBlocks;              // keys per pass
    static constexpr int kChan = kSelStage * kSelThreads / kKeys;  // channels per chunk
    static constexpr int kStride = kChan + 1;                      // LDS row (odd: lanes on distinct banks)
    static constexpr int KW = KPL < 2 ? 1 : 2;                     // keys per lane of the score phase
    static constexpr int kGroups = kBlocks / KW;                   // key groups, one wave each per row set
    static constexpr int kRows = kGroups;                          // query rows per wave
    static constexpr size_t kLdsFloats = static_cast<size_t>(kKeys) * kStride + static_cast<size_t>(kSelWaves) * kKeys;
};

// Bound of |double sum of at most 2048 probabilities in any order - the sequential one| (each at
// most 2048 * 2^-53 of a sum near 1).
constexpr double kCumEps = 9.094947017729282e-13;  // 2^-40

__device__ __forceinline__ uint64_t shfl_xor_u64(uint64_t v, int mask) {
    const int lo = __shfl_xor(static_cast<int>(static_cast<uint32_t>(v)), mask, kWave);
    const int hi = __shfl_xor(static_cast<int>(static_cast<uint32_t>(v >> 32)), mask, kWave);
    return (static_cast<uint64_t>(static_cast<uint32_t>(hi)) << 32) | static_cast<uint32_t>(lo);
}

// Inverse of the key's high word (~orderable(prob)).
__device__ __forceinline__ float key_prob(uint32_t high) {
    const uint32_t ord = ~high;
    return __uint_as_float((ord & 0x80000000u) ? (ord & 0x7fffffffu) : ~ord);
}

// Lane exchange inside a 16-lane row. The four levels pair each lane with a lane of the other half
// of its group of 2, 4, 8 and 16; every lane of a half holds the half's result, so a reduction by
// these levels equals the xor-shuffle tree.
template <int kLevel> __device__ __forceinline__ int row_pair(int v) {
    constexpr int kCtrl = kLevel == 0 ? 0xb1 : kLevel == 1 ? 0x4e : kLevel == 2 ? 0x141 : 0x140;
    return __builtin_amdgcn_update_dpp(v, v, kCtrl, 0xf, 0xf, false);
}

template <typename Op> __device__ __forceinline__ float wave_reduce_f32(float v, Op op) {
    auto pair = [](int x) { return __int_as_float(x); };
    v = op(v, pair(row_pair<0>(__float_as_int(v))));
    v = op(v, pair(row_pair<1>(__float_as_int(v))));
    v = op(v, pair(row_pair<2>(__float_as_int(v))));
    v = op(v, pair(row_pair<3>(__float_as_int(v))));
    v = op(v, __shfl_xor(v, 16, kWave));
    return op(v, __shfl_xor(v, 32, kWave));
}

// The same for values whose order of combination does not matter (all lanes of a row hold the row's
// result after the four levels; the rows are then read as scalars).
template <typename Op> __device__ __forceinline__ int wave_reduce_i32(int v, Op op) {
    v = op(v, row_pair<0>(v));
    v = op(v, row_pair<1>(v));
    v = op(v, row_pair<2>(v));
    v = op(v, row_pair<3>(v));
    const int a = op(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16));
    return op(a, op(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

__device__ __forceinline__ float lane_f32(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

__device__ __forceinline__ float wave_sum_any(float v) {
    v += __int_as_float(row_pair<0>(__float_as_int(v)));
    v += __int_as_float(row_pair<1>(__float_as_int(v)));
    v += __int_as_float(row_pair<2>(__float_as_int(v)));
    v += __int_as_float(row_pair<3>(__float_as_int(v)));
    return (lane_f32(v, 0) + lane_f32(v, 16)) + (lane_f32(v, 32) + lane_f32(v, 48));
}

__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
    for (int m = 1; m < kWave; m <<= 1) v += __longlong_as_double(shfl_xor_u64(__double_as_longlong(v), m));
    return v;
}

// Whether entry k of the descending order (probability prob, cumulative sum cum up to and with it)
// is kept: 1 or 0, or -1 when the two ends of the cumulative sum's error band decide differently.
__device__ __forceinline__ int keep_decision(int k, int floor_keep, double cum, float prob, float p) {
    if (k < floor_keep) return 1;
    const bool lo = static_cast<float>(cum - kCumEps) - prob < p;
    const bool hi = static_cast<float>(cum + kCumEps) - prob < p;
    return lo == hi ? (lo ? 1 : 0) : -1;
}

// The kept prefix of one row by the sequential definition: entries in descending order (ties by
// index) until one past the minimum fails. Slot e of lane l is key 64 e + l; bit e of the result: slot
// e kept. Taken by rows with non-finite mass and by decisions the search leaves open.
template <int KPL>
__device__ __forceinline__ uint32_t keep_sequential(const float (&prob)[KPL], int ck, int floor_keep, float p) {
    const int lane = lane_id();
    uint32_t keep = 0;
    uint64_t last = 0;
    double run = 0.0;
    for (int k = 0; k < ck; ++k) {
        // Smallest sort key (~orderable(prob), index) past the last one.
        uint64_t best = ~0ull;
#pragma unroll
        for (int e = 0; e < KPL; ++e) {
            const int j = e * kSelBlock + lane;
            const uint64_t key = (static_cast<uint64_t>(~orderable(prob[e])) << 32) | static_cast<uint32_t>(j);
            if (j < ck && (k == 0 || key > last) && key < best) best = key;
        }
#pragma unroll
        for (int m = 1; m < kWave; m <<= 1) {
            const uint64_t other = shfl_xor_u64(best, m);
            best = other < best ? other : best;
        }
        const float pr = key_prob(static_cast<uint32_t>(best >> 32));
        run += static_cast<double>(pr);
        if (k >= floor_keep && !(static_cast<float>(run) - pr < p)) break;
        last = best;
        const int j = static_cast<int>(best & 0xffffffffu);
        if (lane == j % kSelBlock) keep |= 1u << (j / kSelBlock);
    }
    return keep;
}

// The same by search (see the head of the file); bit e of the result: slot e kept. False when a
// decision at the boundary stays open.
template <int KPL>
__device__ __forceinline__ bool keep_search(const float (&prob)[KPL], int ck, int floor_keep, float p, uint32_t& result) {
    const int lane = lane_id();
    int u[KPL];  // probability bits, ordered as integers; below 0 for an absent key (probability -1)
#pragma unroll
    for (int e = 0; e < KPL; ++e) u[e] = __float_as_int(prob[e]);
    // Entries with bits above v: their count and mass.
    auto above = [&](int v, int& n, float& mass) __attribute__((always_inline)) {
        float part = 0.0f;
        n = 0;
#pragma unroll
        for (int e = 0; e < KPL; ++e) {
            const bool g = u[e] > v;
            n += __popcll(__ballot(g));
            part += g ? prob[e] : 0.0f;
        }
        mass = wave_sum_any(part);
    };
    auto imax = [](int a, int b) { return max(a, b); };
    auto imin = [](int a, int b) { return min(a, b); };
    // The entry after those above v is kept when it is within the minimum or their mass is below p;
    // v: the smallest bits for which that holds (lo: a value it does not hold for).
    int v = u[0];
#pragma unroll
    for (int e = 1; e < KPL; ++e) v = max(v, u[e]);
    v = wave_reduce_i32(v, imax);
    int lo = -1, n_lo = ck, n_hi = 0;
    {
        int n;
        float mass;
        above(lo, n, mass);
        if (mass < p) v = lo;  // (all ck entries are past the minimum)
    }
    while (v - lo > 1) {
        const int mid = lo + ((v - lo) >> 1);
        int n;
        float mass;
        above(mid, n, mass);
        if (n < floor_keep || mass < p) {
            v = mid;
            n_hi = n;
        } else {
            lo = mid;
            n_lo = n;
        }
        if (n_lo - n_hi == 1) {  // one entry in (lo, v]: the value sought is its own
            int best = -1;
#pragma unroll
            for (int e = 0; e < KPL; ++e) best = u[e] <= v ? max(best, u[e]) : best;
            v = wave_reduce_i32(best, imax);
            break;
        }
    }
    for (int moves = 0; moves < 4; ++moves) {
        double part = 0.0;
        int n = 0, least = 0x7fffffff, below = -1;
        uint32_t keep = 0;
#pragma unroll
        for (int e = 0; e < KPL; ++e) {
            const bool g = u[e] > v;
            n += __popcll(__ballot(g));
            part += g ? static_cast<double>(prob[e]) : 0.0;
            least = g ? min(least, u[e]) : least;
            below = u[e] < v ? max(below, u[e]) : below;
            keep |= g ? 1u << e : 0u;
        }
        const double cum = wave_sum_f64(part);
        least = wave_reduce_i32(least, imin);
        below = wave_reduce_i32(below, imax);
        if (n > 0) {
            const int d = keep_decision(n - 1, floor_keep, cum, __int_as_float(least), p);
            if (d < 0) return false;
            if (d == 0) {
                v = least;
                continue;
            }
        }
        // Entries equal to v, in index order.
        const float value = __int_as_float(max(v, 0));
        int ties = 0;
        bool open = false, failed = false;
#pragma unroll
        for (int e = 0; e < KPL; ++e) {
            const bool q = u[e] == v && v >= 0;
            const uint64_t m = __ballot(q);
            if (m == 0) continue;
            const int rank = ties + static_cast<int>(__builtin_amdgcn_mbcnt_hi(
                                        static_cast<uint32_t>(m >> 32),
                                        __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0)));
            const int d = keep_decision(n + rank, floor_keep,
                                        cum + static_cast<double>(rank + 1) * static_cast<double>(value), value, p);
            open = open || (q && d < 0);
            failed = failed || (q && d == 0);
            keep |= q && d > 0 ? 1u << e : 0u;
            ties += __popcll(m);
        }
        if (__any(open)) return false;
        if (!__any(failed) && below >= 0) {
            const float next = __int_as_float(below);
            const int d = keep_decision(
                n + ties, floor_keep,
                cum + static_cast<double>(ties) * static_cast<double>(value) + static_cast<double>(next), next, p);
            if (d < 0) return false;
            if (d > 0) {
                v = below;
                continue;
            }
        }
        result = keep;
        return true;
    }
    return false;
}

template <int KPL>
__device__ __forceinline__ uint32_t keep_prefix(const float (&prob)[KPL], int ck, int floor_keep, float p, bool finite) {
    const int lane = lane_id();
    uint32_t keep = 0;
#pragma unroll
    for (int e = 0; e < KPL; ++e)
        if (e * kSelBlock + lane < ck) keep |= 1u << e;
    if (p >= 1.0f || ck <= floor_keep) return keep;
    if (!finite || !keep_search<KPL>(prob, ck, floor_keep, p, keep))
        keep = keep_sequential<KPL>(prob, ck, floor_keep, p);
    return keep;
}

// Kept-segment list of one map row, written by one wavefront: lane l takes clusters l,
// l + 64, ... of the extended cluster order, whose rows are [min(sk, prefix), min(sk, prefix +
// size)) of the key stream. A kept cluster with rows extends the current segment when the
// previous cluster with rows was kept too (their rows are adjacent), else it opens one.
// Returns the row's stream length L.
// kcnt[i] holds the size of key cluster 64 i + lane (0 past ck).
template <int KPL, typename Kept>
__device__ int write_segments(int2* __restrict__ srow, const int (&kcnt)[KPL], int ck, int ce, int valid_text,
                              int text, int sk, Kept kept) {
    const int lane = lane_id();
    const uint64_t below = (1ull << lane) - 1ull;
    int pre = 0, run = 0, nseg = 0;
    bool prev_on = false;
#pragma unroll
    for (int ch = 0; ch <= KPL; ++ch) {
        const int j0 = ch * kWave;
        if (j0 >= ce) break;
        const int j = j0 + lane;
        int size = ch < KPL ? kcnt[ch < KPL ? ch : 0] : 0;
        if (j >= ck && j < ce) size = j == ck ? valid_text : text - valid_text;
        const int incl = wave_incl_scan(size);
        const int a = min(sk, pre + incl - size), e = min(sk, pre + incl);
        const bool has_rows = e > a;
        const bool on = has_rows && kept(j, ch);
        const uint64_t with_rows = __ballot(has_rows), on_mask = __ballot(on);
        const uint64_t lower = with_rows & below;
        const bool prev = lower ? ((on_mask >> (63 - __builtin_clzll(lower))) & 1ull) != 0 : prev_on;
        const bool start = on && !prev;
        const uint64_t starts = __ballot(start);
        const int orows = on ? e - a : 0;
        const int oincl = wave_incl_scan(orows);
        const int off = run + oincl - orows;  // stream offset of cluster j
        if (start) srow[1 + nseg + __popcll(starts & below)] = int2{a - off, off};
        nseg += __popcll(starts);
        run += __builtin_amdgcn_readlane(oincl, kWave - 1);
        pre += __builtin_amdgcn_readlane(incl, kWave - 1);
        if (with_rows) prev_on = ((on_mask >> (63 - __builtin_clzll(with_rows))) & 1ull) != 0;
    }
    if (lane == 0) {
        srow[0] = int2{nseg, run};
        srow[1 + nseg] = int2{0, 0x7fffffff};
    }
    return run;
}

// kWork: besides (or instead of) the map, write every map row's kept-segment list and stream
// length into `work`; the last workgroup of each batch entry to finish (arrival counter) then
// orders that entry's attention items.
template <int KPL, bool kWork>
__global__ __launch_bounds__(kSelThreads, KPL > 16 ? 2 : 4) void select_kernel(
    const float* __restrict__ qc, const float* __restrict__ kc, const int32_t* __restrict__ qn,
    const int32_t* __restrict__ kn, int bh, int cq, int ck, int dims, float scale, float p, int minimum, int extend,
    int valid_text, int text, uint8_t* __restrict__ map, int32_t* __restrict__ ext_q, int32_t* __restrict__ ext_k,
    int32_t* __restrict__ kept_keys, int sq, int sk, SelWork work) {
    extern __shared__ __align__(16) unsigned char smem[];
    using T = SelTiles<KPL>;
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int groups = static_cast<int>(ceil_div(cq, kSelWaves));
    const int b = blockIdx.x / groups;
    const int c0 = (blockIdx.x % groups) * kSelWaves;
    const int c = c0 + wave;
    const bool active = c < cq;
    const int ce = extend ? ck + 2 : ck;
    const int re = extend ? cq + 2 : cq;
    const int qstride = (dims + 3) & ~3;             // keeps float4 reads of a row aligned
    float* qrows = reinterpret_cast<float*>(smem);   // [kSelWaves][qstride]
    float* kblk = qrows + kSelWaves * qstride;        // [kKeys][kStride] one chunk of the keys
    float* dots = kblk + T::kKeys * T::kStride;       // [kSelWaves][kKeys] a pass's scores, by row

    // Text partition rows and extended sizes (once per batch entry).
    if (extend && c0 == 0 && wave == 0) {
        if (map) {
            uint8_t* m = map + static_cast<int64_t>(b) * re * ce;
            for (int j = lane; j < ce; j += kWave) {
                m[static_cast<int64_t>(cq) * ce + j] = j < ck + 1;        // valid-text row: all but padding
                m[static_cast<int64_t>(cq + 1) * ce + j] = j == ck + 1;   // padding row: padding only
            }
        }
        if (ext_q)
            for (int i = lane; i < cq; i += kWave) ext_q[static_cast<int64_t>(b) * re + i] = qn[static_cast<int64_t>(b) * cq + i];
        if (ext_k)
            for (int j = lane; j < ck; j += kWave) ext_k[static_cast<int64_t>(b) * ce + j] = kn[static_cast<int64_t>(b) * ck + j];
        if (lane == 0 && ext_q && ext_k) {
            ext_q[static_cast<int64_t>(b) * re + cq] = valid_text;
            ext_q[static_cast<int64_t>(b) * re + cq + 1] = text - valid_text;
            ext_k[static_cast<int64_t>(b) * ce + ck] = valid_text;
            ext_k[static_cast<int64_t>(b) * ce + ck + 1] = text - valid_text;
        }
        if (kept_keys) {
            // The valid-text row sees every video key and the valid text; the padding row only
            // the padding.
            int all = 0;
            for (int j = lane; j < ck; j += kWave) all += max(0, kn[static_cast<int64_t>(b) * ck + j]);
#pragma unroll
            for (int m = 1; m < kWave; m <<= 1) all += __shfl_xor(all, m, kWave);
            if (lane == 0) {
                kept_keys[static_cast<int64_t>(b) * re + cq] = all + valid_text;
                kept_keys[static_cast<int64_t>(b) * re + cq + 1] = text - valid_text;
            }
        }
    }
    for (int t = threadIdx.x; t < kSelWaves * dims; t += blockDim.x) {
        const int r = c0 + t / dims;
        qrows[(t / dims) * qstride + t % dims] = r < cq ? qc[(static_cast<int64_t>(b) * cq + r) * dims + t % dims] : 0.0f;
    }
    const int32_t* kcount = kn + static_cast<int64_t>(b) * ck;

    // A chunk goes through registers: kSelStage floats per thread, all loads in flight (clamped, so
    // unconditional), requested while the chunk before is used.
    float staged[kSelStage];
    const int chunks = static_cast<int>(ceil_div(dims, T::kChan));
    const char* keys_bytes = reinterpret_cast<const char*>(kc + static_cast<int64_t>(b) * ck * dims);
    const int srow = threadIdx.x / T::kChan, scol = threadIdx.x % T::kChan;
    constexpr int kRowStep = kSelThreads / T::kChan;
    auto fetch = [&](int pass, int chunk) {
        const int col = min(chunk * T::kChan + scol, dims - 1);
#pragma unroll
        for (int i = 0; i < kSelStage; ++i) {
            const int row = min(pass * T::kKeys + srow + i * kRowStep, ck - 1);
            // 32-bit byte offsets from the uniform base: ck <= 2048 rows of at most 256 channels.
            staged[i] = *reinterpret_cast<const float*>(keys_bytes + static_cast<uint32_t>(row * dims + col) * 4u);
        }
    };
    // Score phase: this wave's key group and first query row.
    const int kg = wave % T::kGroups, r0 = (wave / T::kGroups) * T::kRows;
    int kcnt[KPL];      // counts of keys 64 e + lane (0 past ck)
    float prob[KPL];    // dot products, then logits, masses and probabilities
    fetch(0, 0);
#pragma unroll
    for (int pass = 0; pass < T::kPasses; ++pass) {
        if (pass > 0 && pass * T::kKeys >= ck) break;
        float acc[T::kRows][T::KW];
#pragma unroll
        for (int r = 0; r < T::kRows; ++r)
#pragma unroll
            for (int w = 0; w < T::KW; ++w) acc[r][w] = 0.0f;
        const bool has_keys = pass * T::kKeys + kg * T::KW * kSelBlock < ck;
        for (int chunk = 0; chunk < chunks; ++chunk) {
            __syncthreads();  // the previous chunk is consumed (and the query rows are staged)
#pragma unroll
            for (int i = 0; i < kSelStage; ++i) kblk[(srow + i * kRowStep) * T::kStride + scol] = staged[i];
            __syncthreads();
            if (chunk + 1 < chunks) fetch(pass, chunk + 1);
            else if ((pass + 1) * T::kKeys < ck) fetch(pass + 1, 0);
            if (!has_keys) continue;
            const float* kr = kblk + (kg * T::KW * kSelBlock + lane) * T::kStride;
            const float* qr = qrows + r0 * qstride + chunk * T::kChan;
            const int lim = min(T::kChan, dims - chunk * T::kChan);
            auto quad = [&](int d) {
                float kv[T::KW][4];
#pragma unroll
                for (int w = 0; w < T::KW; ++w)
#pragma unroll
                    for (int i = 0; i < 4; ++i) kv[w][i] = kr[w * kSelBlock * T::kStride + d + i];
#pragma unroll
                for (int r = 0; r < T::kRows; ++r) {
                    const float4 q4 = *reinterpret_cast<const float4*>(qr + r * qstride + d);
#pragma unroll
                    for (int w = 0; w < T::KW; ++w) {
                        acc[r][w] = fmaf(q4.x, kv[w][0], acc[r][w]);
                        acc[r][w] = fmaf(q4.y, kv[w][1], acc[r][w]);
                        acc[r][w] = fmaf(q4.z, kv[w][2], acc[r][w]);
                        acc[r][w] = fmaf(q4.w, kv[w][3], acc[r][w]);
                    }
                }
            };
            int d = 0;
            for (; d + 8 <= lim; d += 8) {
                quad(d);
                quad(d + 4);
            }
            for (; d + 4 <= lim; d += 4) quad(d);
            for (; d < lim; ++d)
#pragma unroll
                for (int r = 0; r < T::kRows; ++r)
#pragma unroll
                    for (int w = 0; w < T::KW; ++w)
                        acc[r][w] = fmaf(qr[r * qstride + d], kr[w * kSelBlock * T::kStride + d], acc[r][w]);
        }
        if (pass + 1 == T::kPasses || (pass + 1) * T::kKeys >= ck) {
            // The counts are requested only now: their latency overlaps the exchange, and the score
            // phase keeps their registers.
#pragma unroll
            for (int e = 0; e < KPL; ++e) {
                const int j = e * kSelBlock + lane;
                const int w = kcount[min(j, ck - 1)];
                kcnt[e] = j < ck ? max(0, w) : 0;
            }
        }
        // To the row layout (the previous pass's dots are read before its first chunk barrier).
        if (has_keys) {
#pragma unroll
            for (int r = 0; r < T::kRows; ++r)
#pragma unroll
                for (int w = 0; w < T::KW; ++w)
                    dots[(r0 + r) * T::kKeys + (kg * T::KW + w) * kSelBlock + lane] = acc[r][w];
        }
        __syncthreads();
#pragma unroll
        for (int e = 0; e < T::kBlocks; ++e) prob[pass * T::kBlocks + e] = dots[wave * T::kKeys + e * kSelBlock + lane];
    }
    if (active) {
        float lmax = -INFINITY;
#pragma unroll
        for (int e = 0; e < KPL; ++e) {
            prob[e] = kcnt[e] > 0 ? prob[e] * scale + logf(static_cast<float>(kcnt[e])) : -INFINITY;
            lmax = fmaxf(lmax, prob[e]);
        }
        lmax = wave_reduce_f32(lmax, [](float x, float y) { return fmaxf(x, y); });
        if (!(lmax > -INFINITY && lmax < INFINITY)) lmax = 0.0f;
        // Masses and their sum (lane partials in index order, then a fixed xor tree).
        float part = 0.0f;
#pragma unroll
        for (int e = 0; e < KPL; ++e) {
            if (e * kSelBlock + lane < ck) {
                prob[e] = expf(prob[e] - lmax);
                part += prob[e];
            }
        }
        part = wave_reduce_f32(part, [](float x, float y) { return x + y; });
        const float denom = fmaxf(part, 1.17549435e-38f);
#pragma unroll
        for (int e = 0; e < KPL; ++e) prob[e] = e * kSelBlock + lane < ck ? prob[e] / denom : -1.0f;
        uint32_t keep = keep_prefix<KPL>(prob, ck, max(1, minimum), p, part < INFINITY);
        const bool qnonempty = qn[static_cast<int64_t>(b) * cq + c] > 0;
        int kept_rows = 0;  // key rows behind this row's kept clusters
#pragma unroll
        for (int e = 0; e < KPL; ++e) {
            if (!qnonempty || kcnt[e] == 0) keep &= ~(1u << e);
            kept_rows += keep & (1u << e) ? kcnt[e] : 0;
        }
        if (kept_keys) {
            kept_rows = wave_reduce_i32(kept_rows, [](int x, int y) { return x + y; });
            if (lane == 0)
                kept_keys[static_cast<int64_t>(b) * re + c] = kept_rows + (extend ? valid_text : 0);  // as the map row
        }
        if (map) {
            uint8_t* mrow = map + (static_cast<int64_t>(b) * re + c) * ce;
#pragma unroll
            for (int e = 0; e < KPL; ++e) {
                const int j = e * kSelBlock + lane;
                if (j < ck) mrow[j] = (keep >> e) & 1u;
            }
            if (extend && lane < 2) mrow[ck + lane] = lane == 0;  // video rows see valid text, never padding
        }
        if constexpr (kWork) {
            // Video rows keep their selected clusters and the valid text, never the padding.
            int2* segs = work.segs + (static_cast<int64_t>(b) * re + c) * (ce + 2);
            const int rk = write_segments<KPL>(segs, kcnt, ck, ce, valid_text, text, sk,
                                               [&](int j, int e) { return j < ck ? ((keep >> e) & 1u) != 0 : j == ck; });
            if (lane == 0)
                __hip_atomic_store(work.row_keys + static_cast<int64_t>(b) * re + c, rk, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    if constexpr (kWork) {
        __shared__ int tmp[kSelWaves];
        __shared__ int last;
        if (extend && c0 == 0 && wave < 2) {
            // The text rows: valid text sees every video key and the valid text, padding only
            // itself.
            const int r = cq + wave;
            int2* segs = work.segs + (static_cast<int64_t>(b) * re + r) * (ce + 2);
            const int rk = write_segments<KPL>(segs, kcnt, ck, ce, valid_text, text, sk,
                                               [&](int j, int) { return wave == 0 ? j < ck + 1 : j == ck + 1; });
            if (lane == 0)
                __hip_atomic_store(work.row_keys + static_cast<int64_t>(b) * re + r, rk, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
        // Arrival. The row lengths are the only data the last workgroup reads from the others
        // (device-coherent stores and loads); the segment lists and items reach the attention
        // through the kernel boundary. The barrier orders every wavefront's stores before the
        // counter increment, a release at agent scope, and the last workgroup acquires before
        // it reads, so the hand-over holds under the memory model, not only on the hardware's
        // in-order completion of the stores.
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (threadIdx.x == 0)
            last = __hip_atomic_fetch_add(work.tickets + b, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT) ==
                   groups - 1;
        __syncthreads();
        if (!last) return;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        // Last workgroup of entry b: clamped query offsets of the extended partition and the
        // stream length of every row, then the entry's items in cost order.
        int* qoff = reinterpret_cast<int*>(smem);  // [re + 1]
        int* kept = qoff + re + 1;                 // [re]
        uint64_t* keys = reinterpret_cast<uint64_t*>(smem) + (2 * re + 2) / 2;  // [kSortCap]
        const int nt = kSelWaves * kWave;
        const int per = static_cast<int>(ceil_div(re, nt));
        const int r0 = min(re, static_cast<int>(threadIdx.x) * per), r1 = min(re, r0 + per);
        int local = 0;
        for (int r = r0; r < r1; ++r) {
            const int n = r < cq ? max(0, qn[static_cast<int64_t>(b) * cq + r])
                                 : (r == cq ? valid_text : text - valid_text);
            qoff[r] = n;
            local += n;
        }
        int total;
        int run = block_scan<kSelWaves>(local, tmp, &total);
        for (int r = r0; r < r1; ++r) {
            const int n = qoff[r];
            qoff[r] = min(sq, run);
            run += n;
        }
        if (threadIdx.x == 0) qoff[re] = min(sq, total);
        for (int r = threadIdx.x; r < re; r += nt)
            kept[r] = max(0, __hip_atomic_load(work.row_keys + static_cast<int64_t>(b) * re + r, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT));
        __syncthreads();
        order_head_items<kSelWaves>(qoff, kept, re, attention_item_rows(sq),
                                    work.items + static_cast<int64_t>(b) * work.cap * 3, work.counts + b, keys, tmp);
        if (threadIdx.x == 0) work.tickets[b] = 0;  // ready for the next call
    }
}

template <int KPL>
void launch_select(int blocks, size_t lds, hipStream_t stream, const float* qc, const float* kc, const int32_t* qn,
                   const int32_t* kn, int bh, int cq, int ck, int dims, float scale, float p, int minimum, int extend,
                   int valid_text, int text, uint8_t* map, int32_t* ext_q, int32_t* ext_k, int32_t* kept_keys,
                   int sq, int sk, const SelWork* work) {
    const size_t qstride = (static_cast<size_t>(dims) + 3) & ~static_cast<size_t>(3);
    lds = std::max(lds, sizeof(float) * (kSelWaves * qstride + SelTiles<KPL>::kLdsFloats));
    if (work)
        hipLaunchKernelGGL((select_kernel<KPL, true>), dim3(static_cast<unsigned>(blocks)), dim3(kSelThreads), lds, stream,
                           qc, kc, qn, kn, bh, cq, ck, dims, scale, p, minimum, extend, valid_text, text, map, ext_q,
                           ext_k, kept_keys, sq, sk, *work);
    else
        hipLaunchKernelGGL((select_kernel<KPL, false>), dim3(static_cast<unsigned>(blocks)), dim3(kSelThreads), lds, stream,
                           qc, kc, qn, kn, bh, cq, ck, dims, scale, p, minimum, extend, valid_text, text, map, ext_q,
                           ext_k, kept_keys, sq, sk, SelWork{});
}

// Shared host entry: validation, LDS size and the launch over the per-lane key count.
int select_launch(const float* qc, const float* kc, const int32_t* q_counts, const int32_t* k_counts, int bh, int cq,
                  int ck, int dims, float p, int minimum, int extend, int valid_text, int text, uint8_t* map,
                  int32_t* ext_q, int32_t* ext_k, int32_t* kept_keys, int sq, int sk, const SelWork* work,
                  void* stream) {
    if (!qc || !kc || !q_counts || !k_counts || bh < 1 || cq < 1 || ck < 1 || dims < 1 || dims > kSelMaxDims ||
        !(p >= 0.0f && p <= 1.0f) || minimum < 0 || (extend && (valid_text < 0 || valid_text > text)))
        return kInvalidValue;
    if (ck > kWave * 32) return kUnsupportedShape;
    const size_t qstride = (static_cast<size_t>(dims) + 3) & ~static_cast<size_t>(3);
    // Shapes this entry has always refused stay refused (a key block of 64 rows and a flag byte per
    // row and key beside the query rows); the kernel itself needs at most 60 KB for those it takes.
    if (sizeof(float) * (kSelWaves * qstride + static_cast<size_t>(kSelBlock) * (dims + 1)) +
            static_cast<size_t>(kSelWaves) * ck > 64 * 1024)
        return kUnsupportedShape;
    size_t lds = 0;
    if (work) {
        // The last workgroup of an entry reuses the LDS for its query offsets, row lengths and sort keys.
        const size_t re = static_cast<size_t>(extend ? cq + 2 : cq);
        lds = sizeof(int) * (2 * re + 2) + sizeof(uint64_t) * kSortCap;
        if (lds > 64 * 1024) return kUnsupportedShape;
    }
    const int blocks = bh * static_cast<int>(ceil_div(cq, kSelWaves));
    const float scale = static_cast<float>(std::pow(static_cast<double>(dims), -0.5));
    auto* s = static_cast<hipStream_t>(stream);
    const int per_lane = static_cast<int>(ceil_div(ck, kWave));
#define PECO_SELECT(K)                                                                                             \
    launch_select<K>(blocks, lds, s, qc, kc, q_counts, k_counts, bh, cq, ck, dims, scale, p, minimum, extend, valid_text, \
                     text, map, ext_q, ext_k, kept_keys, sq, sk, work)
    if (per_lane <= 1) PECO_SELECT(1);
    else if (per_lane <= 2) PECO_SELECT(2);
    else if (per_lane <= 4) PECO_SELECT(4);
    else if (per_lane <= 8) PECO_SELECT(8);
    else if (per_lane <= 16) PECO_SELECT(16);
    else PECO_SELECT(32);
#undef PECO_SELECT
    return hipGetLastError();
}

}  // namespace
}  // namespace peco

using namespace peco;

// Selection of cluster pairs, optionally extended with the text partition.
// qc [bh, cq, dims], kc [bh, ck, dims] fp32; q_counts [bh, cq], k_counts [bh, ck] int32.
// map: bool [bh, cq(+2), ck(+2)]; ext_q/ext_k (extend only): int32 [bh, cq+2] / [bh, ck+2].
// kept_keys (nullable): int32 [bh, cq(+2)], the number of key rows each map row keeps.
// minimum = ceil(min_kc_ratio * ck) computed by the caller. ck <= 2048, dims <= 256; the LDS use
// (8 query rows, a 64-row key block and 8 rows of ck flag bytes) must fit in 64 KiB.
PECO_API int peco_select_cluster_connections(const float* qc, const float* kc, const int32_t* q_counts,
                                             const int32_t* k_counts, int bh, int cq, int ck, int dims, float p,
                                             int minimum, int extend, int valid_text, int text, uint8_t* map,
                                             int32_t* ext_q, int32_t* ext_k, int32_t* kept_keys, void* stream) {
    if (!map || (extend && (!ext_q || !ext_k))) return kInvalidValue;
    return select_launch(qc, kc, q_counts, k_counts, bh, cq, ck, dims, p, minimum, extend, valid_text, text, map,
                         ext_q, ext_k, kept_keys, 0, 0, nullptr, stream);
}

// int32 elements of the work buffer of peco_select_work for bh entries, sq query rows and a
// (cq(+2)) x (ck(+2)) map.
PECO_API size_t peco_select_work_size(int bh, int sq, int cq, int ck, int extend) {
    if (bh < 1 || sq < 0 || cq < 1 || ck < 1) return 0;
    return sel_work_ints(bh, sq, extend ? cq + 2 : cq, extend ? ck + 2 : ck);
}

// Selection plus the attention's work list in one launch. Same selection as
// peco_select_cluster_connections (map, ext_q and ext_k optional here), and in `work`
// (peco_select_work_size int32, 8-byte aligned; the first bh of them zero before the first
// call, and every call leaves them zero) the kept-segment list and stream length of every map row and the items
// of every entry in cost order, which peco_sparse_attention_work consumes. sq and sk are the
// query and key lengths of the attention (video + text); key cluster rows are clamped to sk
// and query cluster rows to sq as the attention's own builder does.
PECO_API int peco_select_work(const float* qc, const float* kc, const int32_t* q_counts, const int32_t* k_counts,
                              int bh, int cq, int ck, int dims, float p, int minimum, int extend, int valid_text,
                              int text, int sq, int sk, uint8_t* map, int32_t* ext_q, int32_t* ext_k, int32_t* work,
                              size_t work_ints, void* stream) {
    if (!work || sq < 0 || sk < 0 || bh < 1 || cq < 1 || ck < 1) return kInvalidValue;
    const int re = extend ? cq + 2 : cq, ce = extend ? ck + 2 : ck;
    if (work_ints < sel_work_ints(bh, sq, re, ce)) return kWorkspaceTooSmall;
    const SelWork w = sel_work_layout(work, bh, sq, re, ce);
    return select_launch(qc, kc, q_counts, k_counts, bh, cq, ck, dims, p, minimum, extend, valid_text, text, map,
                         ext_q, ext_k, nullptr, sq, sk, &w, stream);
}
