// Attention of several tokens (prefill, or a chunk behind cached keys) on the
// bf16 matrix cores, with f32 accuracy.
//
// Every f32 operand is the sum of three bf16 values (split8, split_bf16.h),
// exact from 2^-110 up, and a product of two of them six MFMA products (those
// left out are at most 2^-24 of it together), summed in f32: 2.7 times the rate of the f32
// matrix instruction, whose head-64 kernel this replaces, and any head
// dimension up to 128.
//
// Rows.  The query heads of a KV head share its keys, so a block takes 128 rows
// of one KV head (64 beyond head dims of 64), numbered token-major (row = token *
// group + head): a short key range for causal rows, K and V split once for all of
// them.  Wave (wq, ws)
// owns 16 or 32 rows and every second 32-key slice (ws), each with its own
// online softmax; the slices merge at the end.
//
// Products.  S^T = K Q^T with v_mfma_f32_16x16x32_bf16 leaves lane l with row
// l % 16 and, over two 16-key tiles, keys 4 (l / 16) + r and 16 + 4 (l / 16) +
// r, r < 4.  O^T += V^T P^T takes its 32 keys in just that order, so P never
// leaves registers; V is stored transposed in LDS with its keys dealt alike.
// Scores are (q.k * scale) * scale and masked keys -inf (transformer.cpp:112-143).
//
// A row whose result is not finite (infinities, NaN, values past bf16's
// range) is computed again with plain f32 arithmetic.
//
// What bounds it: vector instructions (softmax, splitting P, K and V), which
// issue for 60% of a busy CU's time at heads of 64 and 53% at heads of 128, then
// MFMAs (34% and 31%), which the barriers of a step keep from overlapping much.
// 2048 tokens of 14 heads of 64 over 2 KV heads take 83 us and 10 for the merge
// (124 with f32 MFMAs), 256 tokens of 32 heads of 128 behind 1000 keys 48 and 5
// (905 in a kernel without MFMAs).
#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "device_common.h"
#include "kernels.h"
#include "split_bf16.h"

namespace leafhip {
namespace {

constexpr int kSlice = 32;        // keys per slice and step
constexpr int kSlices = 2;
constexpr int kStepKeys = kSlice * kSlices;
constexpr int kRowWaves = 4;
constexpr int kThreads = 64 * kRowWaves * kSlices;
// Rows per wave: two MFMA tiles up to 64 values (each K and V operand read
// from LDS then serves both, and fewer blocks split the same keys), one beyond
// (the split queries and outputs of two would not fit the registers).
constexpr int row_tiles_of(int dp) { return dp <= 64 ? 2 : 1; }
constexpr int block_rows(int dp) { return 16 * row_tiles_of(dp) * kRowWaves; }

// A call's work items per KV head, longest first: a tile of rows and a part of
// its keys.  An empty list is every tile whole, the last (longest) first.
constexpr int kMaxItems = 768;
struct RowItems {
    int count = 0, max_parts = 1, steps_per_part = 0;
    uint32_t item[kMaxItems];                                  // tile | part << 16
};
__host__ __device__ inline int parts_of(int steps, int steps_per_part) {
    return steps_per_part ? (steps + steps_per_part - 1) / steps_per_part : 1;
}

// The keys that a block's rows see: [begin, end) with begin a whole step.
__device__ __forceinline__ void block_keys(const AttentionCall& p, int group, int r0, int rows_per_block, int& begin,
                                           int& end) {
    const int rows = p.tokens * group;
    begin = p.window ? max(0, p.position + r0 / group + 1 - p.window) : 0;
    begin &= ~(kStepKeys - 1);
    end = p.position + min(r0 + rows_per_block - 1, rows - 1) / group + 1;
}

// exp(x) for x <= 0 to about an ulp: 2^t with t = x log2(e) rounded, corrected
// by its rounding error (below -200 the result is 0 anyway; NaN stays NaN, so
// that its row is found and computed again).
__device__ __forceinline__ float exp_negative(float x) {
    constexpr float kLog2e = 1.4426950408889634f;
    constexpr float kRest = (float)(1.4426950408889634 - (double)kLog2e), kLn2 = 0.6931471805599453f;
    x = x < -200.0f ? -200.0f : x;
    const float t = x * kLog2e;
    const float rest = fmaf(x, kRest, fmaf(x, kLog2e, -t));
    const float r = __builtin_amdgcn_exp2f(t);
    return fmaf(r, rest * kLn2, r);
}

__device__ __forceinline__ bool finite(float v) { return __builtin_fabsf(v) < INFINITY; }

__device__ __forceinline__ float visible_score(const AttentionCall& p, const float* q, const float* k) {
    float sum = 0.0f;
    for (int d = 0; d < p.dim; d += 4) {
        const v4f a = *(const v4f*)(q + d), b = *(const v4f*)(k + d);
#pragma unroll
        for (int e = 0; e < 4; ++e) sum = sum + a[e] * b[e];
    }
    return sum * p.scale * p.scale;
}

// One row's output by one wave, two passes over its keys [begin, end).  With
// part, the unnormalized output, sum and maximum instead: a maximum of NaN
// where a score is NaN, and of minus infinity with a sum of 0 where every score
// is (other parts may hold a finite one).  A NaN score ends the first pass, and
// it or one of infinity the row.  300 tokens of 14 heads of 64 with one NaN query
// take 19 us, with all 113 (18 without; 52 and 1,630 in two whole passes).
__device__ __forceinline__ void plain_row(const AttentionCall& p, int h, int t, int begin, int end, float* part) {
    const int lane = threadIdx.x & 63;
    const int kvh = h / (p.heads / p.kv_heads), qpos = p.position + t;
    end = min(end, qpos + 1);
    if (p.window) begin = max(begin, qpos + 1 - p.window);
    const float* q = p.q_heads + ((size_t)h * p.tokens + t) * p.dim;
    const float* K = p.keys + (size_t)kvh * p.capacity * p.dim;
    const float* V = p.values + (size_t)kvh * p.capacity * p.dim;
    float m = -INFINITY;
    bool nan = false;
    for (int k0 = begin; k0 < end && !nan; k0 += 64) {
        const float s = k0 + lane < end ? visible_score(p, q, K + (size_t)(k0 + lane) * p.dim) : -INFINITY;
        nan = __any(s != s);
        m = fmaxf(m, s);
    }
    m = wave_max_f32(m);
    nan = nan || m == INFINITY;               // (infinity less itself)
    if (nan) m = NAN;
    const float base = m == -INFINITY ? 0.0f : m;
    float l = 0.0f, o[2] = {0.0f, 0.0f};      // dims lane and lane + 64
    if (nan) l = o[0] = o[1] = NAN;
    for (int k0 = begin; k0 < end && !nan; k0 += 64) {
        const int k = k0 + lane;
        const float e = k < end ? expf(visible_score(p, q, K + (size_t)k * p.dim) - base) : 0.0f;
        l += e;
        for (int j = 0; j < min(64, end - k0); ++j) {
            const float pj = __shfl(e, j, 64);
#pragma unroll
            for (int c = 0; c < 2; ++c)
                if (lane + 64 * c < p.dim) o[c] = fmaf(pj, V[(size_t)(k0 + j) * p.dim + lane + 64 * c], o[c]);
        }
    }
    l = wave_sum_f32(l);
    if (part && lane == 0) {
        part[0] = m;
        part[1] = l;
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const int d = lane + 64 * c;
        if (d >= p.dim) continue;
        if (part) part[2 + d] = o[c];
        else p.out[((size_t)t * p.heads + h) * p.dim + d] = o[c] / l;   // a row sees a key: 0 / 0 where none has a weight
    }
}

// DP: the head dimension rounded up to whole steps of 32 (zeros past it).
template <int DP>
__global__ __launch_bounds__(kThreads) void attention_rows_kernel(AttentionCall p, int row_tiles, RowItems items) {
    constexpr int kDimSteps = DP / 32, kDimTiles = DP / 16;
    constexpr int kKRow = 2 * DP;                              // bytes of a key's row in one plane
    constexpr int kKPlane = kSlice * kKRow, kVPlane = DP * 2 * kSlice;
    constexpr int kSliceBytes = 3 * (kKPlane + kVPlane);
    constexpr int kKUnits = kStepKeys * DP / 8;                // 8 values of a key
    constexpr int kVUnits = kStepKeys / 4 * DP / 2;            // 4 keys x 2 values
    constexpr int kKLoads = (kKUnits + kThreads - 1) / kThreads, kVLoads = (kVUnits + kThreads - 1) / kThreads;
    __shared__ __align__(1024) uint8_t lds[kSlices * kSliceBytes];

    constexpr int QT = row_tiles_of(DP), kRows = block_rows(DP);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wq = wave % kRowWaves, ws = wave / kRowWaves;
    const int li = lane & 15, lq = lane >> 4;
    const int kvh = blockIdx.x % p.kv_heads;
    const int index = blockIdx.x / p.kv_heads;
    const int tile = items.count ? items.item[index] & 0xFFFF : row_tiles - 1 - index;
    const int part_index = items.count ? items.item[index] >> 16 : 0;
    const int group = p.heads / p.kv_heads, rows = p.tokens * group, dim = p.dim;
    const int r0 = tile * kRows, w0 = r0 + 16 * QT * wq;       // the block's and the wave's first row
    int begin, end;
    block_keys(p, group, r0, kRows, begin, end);
    const int all_steps = (end - begin + kStepKeys - 1) / kStepKeys;
    const int parts = items.count ? parts_of(all_steps, items.steps_per_part) : 1;
    const bool partial = parts > 1;
    if (partial) {
        const int first = begin;
        begin = first + int((long long)part_index * all_steps / parts) * kStepKeys;
        end = min(end, first + int((long long)(part_index + 1) * all_steps / parts) * kStepKeys);
    }
    int t[QT], h[QT], qpos[QT];
#pragma unroll
    for (int i = 0; i < QT; ++i) {
        const int row = min(w0 + 16 * i + li, rows - 1);
        t[i] = row / group;
        h[i] = kvh * group + row % group;
        qpos[i] = p.position + t[i];
    }
    const int wave_end = w0 < rows ? min(end, p.position + min(w0 + 16 * QT - 1, rows - 1) / group + 1) : 0;
    const int wave_safe = p.position + min(w0, rows - 1) / group + 1;   // every row sees the keys before
    const float* K = p.keys + (size_t)kvh * p.capacity * dim;
    const float* V = p.values + (size_t)kvh * p.capacity * dim;
    const float scale2 = p.scale * p.scale;

    // Q^T operand planes: row l % 16, values 8 (l / 16) + 0..7 of each 32
    v8bf qf[QT][kDimSteps][3];
#pragma unroll
    for (int i = 0; i < QT; ++i)
#pragma unroll
        for (int c = 0; c < kDimSteps; ++c) {
            float f[8];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int d = 32 * c + 8 * lq + 4 * e;
                const v4f v = d < dim ? *(const v4f*)(p.q_heads + ((size_t)h[i] * p.tokens + t[i]) * dim + d)
                                      : v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int j = 0; j < 4; ++j) f[4 * e + j] = v[j];
            }
            split8(f, qf[i][c][0], qf[i][c][1], qf[i][c][2]);
        }

    // ---- staging: a thread's K and V units of a step, held in registers until
    // the step before is done.  Keys at or past `end` were perhaps never
    // written: key 0 is loaded and zeros stored.
    v4f kr[kKLoads][2];
    v2f vr[kVLoads][4];
    auto load = [&](int k0) {
#pragma unroll
        for (int j = 0; j < kKLoads; ++j) {
            const int u = threadIdx.x + j * kThreads, key = k0 + u / (DP / 8), d = u % (DP / 8) * 8;
            const float* src = K + (size_t)(key < end && u < kKUnits ? key : 0) * dim;
#pragma unroll
            for (int e = 0; e < 2; ++e) kr[j][e] = *(const v4f*)(src + (d + 4 * e < dim ? d + 4 * e : 0));
        }
#pragma unroll
        for (int j = 0; j < kVLoads; ++j) {
            const int u = threadIdx.x + j * kThreads, key = k0 + u / (DP / 2) * 4, d = u % (DP / 2) * 2;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                vr[j][e] = *(const v2f*)(V + (size_t)(key + e < end && u < kVUnits ? key + e : 0) * dim + (d < dim ? d : 0));
        }
    };
    auto store = [&](int k0, auto whole_step) {                // whole: every key is below `end`
        constexpr bool kWhole = decltype(whole_step)::value;
#pragma unroll
        for (int j = 0; j < kKLoads; ++j) {
            const int u = threadIdx.x + j * kThreads, at = u / (DP / 8), seg = u % (DP / 8);
            if (kKUnits % kThreads && u >= kKUnits) continue;
            float f[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] = (kWhole || k0 + at < end) && 8 * seg + (e & 4) < dim ? kr[j][e / 4][e & 3] : 0.0f;
            v8bf planes[3];
            split8(f, planes[0], planes[1], planes[2]);
            const int key = at % kSlice;
            const int slot = DP % 64 == 0 ? seg ^ (key & 7) : seg ^ ((key >> 1) & 3);
#pragma unroll
            for (int q = 0; q < 3; ++q)
                *(v8bf*)(lds + at / kSlice * kSliceBytes + q * kKPlane + key * kKRow + slot * 16) = planes[q];
        }
#pragma unroll
        for (int j = 0; j < kVLoads; ++j) {
            const int u = threadIdx.x + j * kThreads, at = u / (DP / 2) * 4, d = u % (DP / 2) * 2;
            if (kVUnits % kThreads && u >= kVUnits) continue;
            float f[8];                                        // [value][key]
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] = (kWhole || k0 + at + (e & 3) < end) && d < dim ? vr[j][e & 3][e / 4] : 0.0f;
            v8bf planes[3];
            split8(f, planes[0], planes[1], planes[2]);
            const int quad = at % kSlice / 4;                  // keys 4 quad.. of the slice: half quad / 4 of segment quad % 4
#pragma unroll
            for (int q = 0; q < 3; ++q)
#pragma unroll
                for (int c = 0; c < 2; ++c)
                    *(v2u*)(lds + at / kSlice * kSliceBytes + 3 * kKPlane + q * kVPlane + (d + c) * 64 +
                            (((quad & 3) ^ (((d + c) >> 1) & 3)) * 16) + (quad >> 2) * 8) = ((const v2u*)&planes[q])[c];
        }
    };

    v4f o[QT][kDimTiles];                                      // O^T: values 16 dt + 4 lq + r of row li
    float m[QT], l[QT];                                        // m: of q.k; l: this lane's keys only
#pragma unroll
    for (int i = 0; i < QT; ++i) {
#pragma unroll
        for (int dt = 0; dt < kDimTiles; ++dt) o[i][dt] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
        m[i] = -INFINITY;
        l[i] = 0.0f;
    }
    constexpr int kOfK[6] = {2, 1, 0, 1, 0, 0}, kOfQ[6] = {0, 1, 2, 0, 1, 0};   // small products first
    load(begin);
    for (int k0 = begin; k0 < end; k0 += kStepKeys) {
        lds_barrier();                                         // the last step's operands are no longer read
        if (k0 + kStepKeys <= end) store(k0, std::true_type());
        else store(k0, std::false_type());
        if (k0 + kStepKeys < end) load(k0 + kStepKeys);
        lds_barrier();
        const int ks = k0 + kSlice * ws;
        const uint8_t* kb = lds + ws * kSliceBytes;
        const uint8_t* vb = kb + 3 * kKPlane;
        if (ks >= wave_end) continue;                          // the whole wave
        v4f sc[QT][2];
#pragma unroll
        for (int i = 0; i < QT; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) sc[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int c = 0; c < kDimSteps; ++c) {
            v8bf kf[2][3];
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    const int key = 16 * j + li, seg = 4 * c + lq;
                    const int slot = DP % 64 == 0 ? seg ^ (key & 7) : seg ^ ((key >> 1) & 3);
                    kf[j][q] = *(const v8bf*)(kb + q * kKPlane + key * kKRow + slot * 16);
                }
#pragma unroll
            for (int q = 0; q < 6; ++q)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int i = 0; i < QT; ++i)
                        sc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[j][kOfK[q]], qf[i][c][kOfQ[q]], sc[i][j], 0, 0, 0);
        }
        const bool masked = ks + kSlice > min(wave_safe, end) || p.window;
        v8bf pf[QT][3];
#pragma unroll
        for (int i = 0; i < QT; ++i) {
            float e[8], top = -INFINITY;
#pragma unroll
            for (int j = 0; j < 8; ++j) e[j] = sc[i][j / 4][j & 3];
            if (masked) {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int key = ks + 16 * (j / 4) + 4 * lq + (j & 3);
                    if (key > qpos[i] || key >= end || (p.window && key <= qpos[i] - p.window)) e[j] = -INFINITY;
                }
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) top = fmaxf(top, e[j]);
            top = max_xor32(max_xor16(top));
            const float m_new = fmaxf(m[i], top);
            const float base = m_new == -INFINITY ? 0.0f : m_new;   // nothing visible yet: every weight is 0
            if (__any(m_new != m[i])) {
                const float alpha = exp_negative((m[i] - base) * scale2);
                l[i] *= alpha;
#pragma unroll
                for (int dt = 0; dt < kDimTiles; ++dt) o[i][dt] = o[i][dt] * alpha;
                m[i] = m_new;
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) e[j] = exp_negative((e[j] - base) * scale2);
            l[i] += ((e[0] + e[1]) + (e[2] + e[3])) + ((e[4] + e[5]) + (e[6] + e[7]));
            split8(e, pf[i][0], pf[i][1], pf[i][2]);
        }
#pragma unroll
        for (int d0 = 0; d0 < kDimTiles; d0 += 2) {
            v8bf vf[2][3];
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    const int d = 16 * (d0 + j) + li;
                    vf[j][q] = *(const v8bf*)(vb + q * kVPlane + d * 64 + ((lq ^ ((d >> 1) & 3)) * 16));
                }
#pragma unroll
            for (int q = 0; q < 6; ++q)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int i = 0; i < QT; ++i)
                        o[i][d0 + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[j][kOfK[q]], pf[i][kOfQ[q]], o[i][d0 + j], 0, 0, 0);
        }
    }

    // ---- merge the second slice's state into the first's wave of the same rows
    __syncthreads();                                           // the last operands are no longer read
    constexpr int kRecord = QT * (4 * kDimTiles + 2);
    float* record = (float*)lds + (wq * 64 + lane) * kRecord;
    static_assert(kRowWaves * 64 * kRecord * 4 <= kSlices * kSliceBytes, "merge records fit");
#pragma unroll
    for (int i = 0; i < QT; ++i) l[i] = add_xor32(add_xor16(l[i]));
    if (ws == 1) {
#pragma unroll
        for (int i = 0; i < QT; ++i) {
            float* rec = record + i * (kRecord / QT);
#pragma unroll
            for (int dt = 0; dt < kDimTiles; ++dt)
#pragma unroll
                for (int r = 0; r < 4; ++r) rec[4 * dt + r] = o[i][dt][r];
            rec[4 * kDimTiles] = m[i];
            rec[4 * kDimTiles + 1] = l[i];
        }
    }
    __syncthreads();
    if (ws == 1) return;
    uint32_t redo = 0;
#pragma unroll
    for (int i = 0; i < QT; ++i) {
        const float* rec = record + i * (kRecord / QT);
        const float m1 = rec[4 * kDimTiles], mt = fmaxf(m[i], m1), base = mt == -INFINITY ? 0.0f : mt;
        const float a0 = exp_negative((m[i] - base) * scale2), a1 = exp_negative((m1 - base) * scale2);
        const float sum = l[i] * a0 + rec[4 * kDimTiles + 1] * a1;
        // (minus infinity: only where every score of the row's keys is)
        const int first = p.window ? max(begin, qpos[i] + 1 - p.window) : begin;
        bool bad = !finite(sum) || (mt == -INFINITY && first < min(end, qpos[i] + 1));
#pragma unroll
        for (int dt = 0; dt < kDimTiles; ++dt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                o[i][dt][r] = o[i][dt][r] * a0 + rec[4 * dt + r] * a1;
                bad = bad || !finite(o[i][dt][r]);
            }
        const bool live = w0 + 16 * i + li < rows;
        float* part = partial ? p.partial + (((size_t)t[i] * p.heads + h[i]) * items.max_parts + part_index) * (dim + 2) : nullptr;
        if (live) {
            if (part && lq == 0) {
                part[0] = mt * scale2;
                part[1] = sum;
            }
#pragma unroll
            for (int dt = 0; dt < kDimTiles; ++dt) {
                const int d = 16 * dt + 4 * lq;
                if (d >= dim) continue;
                if (part) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) part[2 + d + r] = o[i][dt][r];
                } else {
                    v4f v = v4f{0.0f, 0.0f, 0.0f, 0.0f};
                    if (sum > 0.0f) v = v4f{o[i][dt][0] / sum, o[i][dt][1] / sum, o[i][dt][2] / sum, o[i][dt][3] / sum};
                    *(v4f*)(p.out + ((size_t)t[i] * p.heads + h[i]) * dim + d) = v;
                }
            }
        }
        const uint64_t lanes = __ballot(bad && live);          // any value of a row spoils it
        redo |= (uint32_t)((lanes | lanes >> 16 | lanes >> 32 | lanes >> 48) & 0xFFFFu) << (16 * i);
    }
#pragma unroll 1
    while (redo) {
        const int row = w0 + __builtin_ctz(redo);
        redo &= redo - 1;
        const int tt = row / group, hh = kvh * group + row % group;
        plain_row(p, hh, tt, begin, end,
                  partial ? p.partial + (((size_t)tt * p.heads + hh) * items.max_parts + part_index) * (dim + 2) : nullptr);
    }
}

// Rows whose keys took several splits: their states merged, one wave a row.  A
// part's NaN (maximum, sum or value) reaches the row, and a weight of 0 times
// an infinite value is NaN, as unsplit; a row sees at least its own key, so a
// sum of 0 means that no key has a weight, and 0 / 0 is what such a row gives.
__global__ __launch_bounds__(256) void attention_rows_merge_kernel(AttentionCall p, int rows_per_block, int max_parts,
                                                                   int steps_per_part) {
    const int lane = threadIdx.x & 63, group = p.heads / p.kv_heads;
    const int item = blockIdx.x * 4 + (threadIdx.x >> 6);      // token * heads + head
    if (item >= p.tokens * p.heads) return;
    const int t = item / p.heads, h = item % p.heads, row = t * group + h % group;
    int begin, end;
    block_keys(p, group, row / rows_per_block * rows_per_block, rows_per_block, begin, end);
    const int count = parts_of((end - begin + kStepKeys - 1) / kStepKeys, steps_per_part);
    if (count <= 1) return;
    const float* part = p.partial + (size_t)item * max_parts * (p.dim + 2);
    const size_t stride = p.dim + 2;
    if (count <= 4) {
        // the usual few parts: every load at once
        float mk[4], lk[4], v[4][2], m = -INFINITY;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const float* q = part + min(s, count - 1) * stride;
            mk[s] = s < count ? q[0] : -INFINITY;
            lk[s] = q[1];
#pragma unroll
            for (int c = 0; c < 2; ++c) v[s][c] = q[2 + min(lane + 64 * c, p.dim - 1)];
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) m = fmaxf(m, mk[s]);
        float l = 0.0f, o[2] = {0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            if (s >= count) break;
            const float w = mk[s] == -INFINITY ? 0.0f : expf(mk[s] - m);
            l = fmaf(lk[s], w, l);
#pragma unroll
            for (int c = 0; c < 2; ++c) o[c] = fmaf(v[s][c], w, o[c]);
        }
#pragma unroll
        for (int c = 0; c < 2; ++c)
            if (lane + 64 * c < p.dim) p.out[(size_t)item * p.dim + lane + 64 * c] = o[c] / l;
        return;
    }
    float m = -INFINITY;
    for (int s = lane; s < count; s += 64) m = fmaxf(m, part[s * stride]);
    m = wave_max_f32(m);
    float l = 0.0f, o[2] = {0.0f, 0.0f};
    for (int s0 = 0; s0 < count; s0 += 64) {
        // a lane weighs one split, then lends its weight to the lanes of the values
        float a = 0.0f;
        if (s0 + lane < count) {
            const float ms = part[(s0 + lane) * stride];
            a = ms == -INFINITY ? 0.0f : expf(ms - m);
            l = fmaf(part[(s0 + lane) * stride + 1], a, l);
        }
        const int n = min(64, count - s0);
#pragma unroll 4
        for (int s = 0; s < n; ++s) {
            const float w = __shfl(a, s, 64);
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const float v = lane + 64 * c < p.dim ? part[(s0 + s) * stride + 2 + lane + 64 * c] : 0.0f;
                o[c] = fmaf(v, w, o[c]);
            }
        }
    }
    l = wave_sum_f32(l);
#pragma unroll
    for (int c = 0; c < 2; ++c)
        if (lane + 64 * c < p.dim) p.out[(size_t)item * p.dim + lane + 64 * c] = o[c] / l;
}

// How a call's keys are shared out: parts of at most a CU's share of the steps
// (and at least two steps), as many to a tile as it needs, equal within it.
// Half that size costs more in blocks and partial results than it evens out
// (512 tokens, 32 heads of 64: 47 instead of 37 us).  Parts grow until their
// results fit in max_floats.
struct RowsPlan {
    int row_tiles = 0;
    RowItems items;
};

size_t partial_floats(const AttentionCall& call, int max_parts) {
    return (size_t)max_parts * call.tokens * call.heads * (call.dim + 2);
}

void plan_rows(const AttentionCall& call, size_t max_floats, RowsPlan& plan) {
    const int group = call.heads / call.kv_heads, rows = call.tokens * group;
    const int per_block = block_rows((call.dim + 31) / 32 * 32);
    plan.row_tiles = (rows + per_block - 1) / per_block;
    RowItems& items = plan.items;
    if (plan.row_tiles > kMaxItems) return;                    // tiles enough
    int steps[kMaxItems], longest = 0;
    long total = 0;
    for (int tile = 0; tile < plan.row_tiles; ++tile) {
        const long end = (long)call.position + std::min((tile + 1) * per_block - 1, rows - 1) / group + 1;
        const long begin = call.window ? std::max(0L, (long)call.position + tile * per_block / group + 1 - call.window) : 0;
        steps[tile] = int((end - begin / kStepKeys * kStepKeys + kStepKeys - 1) / kStepKeys);
        total += steps[tile];
        longest = std::max(longest, steps[tile]);
    }
    int per = (int)std::max<long>(2, (total * call.kv_heads + 255) / 256);
    while (parts_of(longest, per) > 1 && partial_floats(call, parts_of(longest, per)) > max_floats) per += (per + 3) / 4;
    if (parts_of(longest, per) == 1) return;
    int count = 0;
    for (int tile = 0; tile < plan.row_tiles; ++tile) {
        const int parts = parts_of(steps[tile], per);
        if (count + parts > kMaxItems) return;
        for (int part = 0; part < parts; ++part) items.item[count++] = tile | part << 16;
    }
    std::sort(items.item, items.item + count, [&](uint32_t a, uint32_t b) {
        const int sa = steps[a & 0xFFFF], sb = steps[b & 0xFFFF];
        const long la = (long)sa * parts_of(sb, per), lb = (long)sb * parts_of(sa, per);   // sa / parts against sb / parts
        return la != lb ? la > lb : a > b;
    });
    items.count = count;
    items.max_parts = parts_of(longest, per);
    items.steps_per_part = per;
}

template <int DP>
void launch_rows(const AttentionCall& call, hipStream_t stream) {
    RowsPlan plan;
    plan_rows(call, call.partial ? (size_t)call.partial_capacity : 0, plan);
    const int items = plan.items.count ? plan.items.count : plan.row_tiles;
    attention_rows_kernel<DP><<<items * call.kv_heads, kThreads, 0, stream>>>(call, plan.row_tiles, plan.items);
    if (plan.items.count)
        attention_rows_merge_kernel<<<(call.tokens * call.heads + 3) / 4, 256, 0, stream>>>(
            call, block_rows(DP), plan.items.max_parts, plan.items.steps_per_part);
}

}  // namespace

bool attention_rows_supported(const AttentionCall& call) {
    auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    return call.tokens > 1 && call.dim > 0 && call.dim <= 128 && call.dim % 4 == 0 && aligned(call.q_heads) &&
           aligned(call.keys) && aligned(call.values) && aligned(call.out);
}

size_t attention_rows_scratch_floats(const AttentionCall& call) {
    RowsPlan plan;
    plan_rows(call, SIZE_MAX, plan);
    return plan.items.count ? partial_floats(call, plan.items.max_parts) : 0;
}

// The longest tile's steps are at most 2 / (tiles + 1) of a KV head's, so it has
// at most 512 / (kv_heads (tiles + 1)) + 1 parts, and one where kv_heads tiles
// reach 512; each holds a row of dim + 2 floats for all tiles * rows of them.
size_t attention_rows_scratch_limit(int tokens, int heads, int kv_heads, int dim) {
    const size_t per_block = block_rows((dim + 31) / 32 * 32);
    const size_t tiles = ((size_t)tokens * (heads / kv_heads) + per_block - 1) / per_block * kv_heads;
    return (512 + std::min<size_t>(tiles, 512)) * per_block * (dim + 2);
}

void launch_attention_rows(const AttentionCall& call, hipStream_t stream) {
    switch ((call.dim + 31) / 32) {
    case 1: launch_rows<32>(call, stream); break;
    case 2: launch_rows<64>(call, stream); break;
    case 3: launch_rows<96>(call, stream); break;
    default: launch_rows<128>(call, stream); break;
    }
}

}  // namespace leafhip
