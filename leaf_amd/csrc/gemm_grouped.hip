// Integer-activation GEMM with scale groups, on int8 MFMA.
//
//   Y[t, n] = sum over groups g of ((float)sum_{k in g} Xq[t, k] W[n, k] * s_x[t]) * s_w[n, g]  (+ b[n])
//
// for int8 or int4 weights whose groups are whole multiples of 32 values, one
// group per row included (decoder.cpp:571-627, 661-702).  A group's integer sum
// is exact; its term enters with the CPU path's roundings, groups in ascending
// order, so every output is bit-identical to it.  One wave forms an output's sums
// and adds its terms as they come: K is not split.
//
// v_mfma_i32_16x16x32_i8: the tokens are the A operand and the weight rows the
// B operand, so a lane holds four tokens of one weight row (one weight scale
// per group and tile).
// Int4: of the eight nibbles of a word, those of the odd columns are already
// the high halves of their bytes (16 times the value) and a shift brings the
// others there.  The operand so holds the even columns of a word, then the
// odd ones, and the tokens' bytes are permuted alike; the sums are 16 times
// the true ones, which (float)sum * (s_x / 16) undoes exactly.
//
// Tiles and scales go from global memory straight into LDS (global_load_lds),
// 128 values a stage, three or four stages ahead; rows of 128 (int4 weights 64) bytes hold segment
// c in slot c ^ (r % 8) (c ^ (r / 2 % 4)), as in gemm_w8a8.hip.
//
// What bounds it.  Groups of 32 (201 tokens x 4864 INT4 rows x 896, 17 us, 3,440
// as one thread per output): vector instructions issue for 75% of a busy CU's
// time, MFMAs run for 8%.  They are ten for 64 outputs and a group, three of them
// the term's (convert, multiply, multiply-add), the rest clearing the sums, int4
// operands and addresses; and of 1064 blocks 1024 are resident at once (35 KB of
// LDS each).  Long groups over few blocks (96 tokens x 2048 x 2048 INT8 in groups
// of 128, 12 us, 56 with operands loaded where they were used): the latency of a
// block's 16 stages, vector instructions at 22%, waits for half the time.  About 4
// us of either are the quantization.
#include <type_traits>

#include "device_common.h"
#include "kernels.h"

namespace leafhip {
namespace {

typedef __attribute__((address_space(3))) void* lds_ptr_t;

constexpr int kStageK = 128;

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N < 64, "vmcnt holds at most 63");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// FLUSH: groups end after every 1 or 2 steps of 32 values or at a stage's end
// (4: groups of whole stages), fused terms, no accumulator output; or (0)
// groups end anywhere, terms fused or not, accumulators stored on request.
// The first three have no branch inside a stage, so its four steps overlap
// (with those branches 20 instead of 17 us for 201 tokens x 4864 x 896).
// ALIGNED false: the tokens' rows start anywhere, and come through registers,
// which a load into LDS may not do; every stage then waits for its loads
// (512 x 11264 x 2048, groups of 64: 104 us, 59 copied to aligned memory first).
template <int BITS, int FLUSH, int T, bool ALIGNED = true>
__global__ __launch_bounds__(256) void gemm_grouped_kernel(WeightView w, const int8_t* __restrict__ xq,
                                                           const float* __restrict__ xs, int tokens,
                                                           float* __restrict__ y, int epilogue,
                                                           int32_t* __restrict__ acc_out, int unfused, int m_tiles) {
    constexpr int kWaves = 4, BM = 32 * T, BN = 32 * T;       // 2 x 2 waves of 16 T x 16 T
    constexpr int kWBytes = kStageK * BITS / 8;               // of a weight row per stage
    constexpr int kWLanes = kWBytes / 16;                     // lanes per weight row
    constexpr int kChunksX = BM * kStageK / 1024, kChunksW = BN * kWBytes / 1024;
    constexpr int kChunks = kChunksX + kChunksW, kLoads = (kChunks + kWaves - 1) / kWaves;
    constexpr int kStages = T == 1 ? 5 : 4;
    constexpr int kStageBytes = kChunks * 1024 + 1024;        // operands, then 256 floats of scales
    __shared__ __align__(1024) int8_t lds[kStages * kStageBytes];

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int K = w.cols, N = w.rows;
    const int m0 = (blockIdx.x % m_tiles) * BM, n0 = (blockIdx.x / m_tiles) * BN;
    const int steps = K / 32, stages = (K + kStageK - 1) / kStageK;
    const int groups = K / w.group, group_steps = w.group / 32;

    // ---- this wave's loads: 1 KiB chunks of whole row slices (where they do
    // not divide among the waves, the last chunk is loaded more than once)
    const int8_t* src[kLoads];
    int chunk[kLoads], at0[kLoads], step[kLoads], last[kLoads];
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
        const int c = min(j * kWaves + wave, kChunks - 1);
        chunk[j] = c * 1024;
        if (c < kChunksX) {
            const int row = c * 8 + (lane >> 3);
            src[j] = xq + (size_t)min(m0 + row, tokens - 1) * K;
            at0[j] = ((lane & 7) ^ (lane >> 3)) * 16;
            step[j] = kStageK;
            last[j] = K - 16;
        } else {
            const int row = (c - kChunksX) * (64 / kWLanes) + lane / kWLanes, slot = lane % kWLanes;
            src[j] = (const int8_t*)w.data + (size_t)min(n0 + row, N - 1) * K * BITS / 8;
            at0[j] = (BITS == 8 ? slot ^ (row & 7) : slot ^ ((row >> 1) & 3)) * 16;
            step[j] = kWBytes;
            last[j] = K * BITS / 8 - 16;
        }
    }
    // the scales of the groups that end in a stage (FLUSH 0: of each step's
    // group), [end][row]; one load of 64 a wave
    constexpr int kFlushes = FLUSH == 1 || FLUSH == 0 ? 4 : FLUSH == 2 ? 2 : 1;
    static_assert(kFlushes * BN <= 256, "a stage's scales are one load per wave");
    auto group_of = [&](int stage, int f) {
        return min(FLUSH == 1 ? 4 * stage + f : FLUSH == 2 ? 2 * stage + f : (4 * stage + f) / group_steps, groups - 1);
    };
    const int scale_end = min((int)threadIdx.x / BN, kFlushes - 1);
    const float* scale_row = w.scales + (size_t)min(n0 + (int)threadIdx.x % BN, N - 1) * groups;
    // Past the row's end (the last stage's tail, stages that do not exist) the
    // row's last 16 bytes (and last scale) are loaded; no group contains them.
    // Every stage is kLoads + 1 loads of each wave, so a wait names how many
    // younger ones stay in flight.
    auto load = [&](int stage, int buffer) {
        int8_t* base = lds + buffer * kStageBytes;
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const int8_t* from = src[j] + min(at0[j] + stage * step[j], last[j]);
            if (!ALIGNED && chunk[j] < kChunksX * 1024) {
                v4i v;
                __builtin_memcpy(&v, from, 16);
                *(v4i*)(base + chunk[j] + lane * 16) = v;
            } else {
                __builtin_amdgcn_global_load_lds((void*)from, (lds_ptr_t)(base + chunk[j] + lane * 16), 16, 0, 0);
            }
        }
        __builtin_amdgcn_global_load_lds((void*)(scale_row + group_of(stage, scale_end)),
                                         (lds_ptr_t)(base + kChunks * 1024 + wave * 256 + lane * 4), 4, 0, 0);
    };

    const int wm = (wave >> 1) * 16 * T, wn = (wave & 1) * 16 * T;
    const int li = lane & 15, lq = lane >> 4;
    float sx[T][4], res[T][T][4];
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float v = xs[min(m0 + wm + 16 * i + 4 * lq + r, tokens - 1)];
            sx[i][r] = BITS == 4 ? v * 0.0625f : v;
#pragma unroll
            for (int j = 0; j < T; ++j) res[i][j][r] = 0.0f;
        }
    v4i acc[T][T];
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j) acc[i][j] = v4i{0, 0, 0, 0};
    auto flush = [&](int g, const float (&sw)[T]) {
#pragma unroll
        for (int i = 0; i < T; ++i)
#pragma unroll
            for (int j = 0; j < T; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float term = (float)acc[i][j][r] * sx[i][r];
                    float& v = res[i][j][r];
                    if (FLUSH == 0 && unfused) v = __fadd_rn(v, __fmul_rn(term, sw[j]));
                    else v = fmaf(term, sw[j], v);
                }
        if (FLUSH == 0 && acc_out) {
#pragma unroll
            for (int i = 0; i < T; ++i)
#pragma unroll
                for (int j = 0; j < T; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int t = m0 + wm + 16 * i + 4 * lq + r, n = n0 + wn + 16 * j + li;
                        if (t < tokens && n < N)
                            acc_out[((size_t)t * N + n) * groups + g] = BITS == 4 ? acc[i][j][r] >> 4 : acc[i][j][r];
                    }
        }
#pragma unroll
        for (int i = 0; i < T; ++i)
#pragma unroll
            for (int j = 0; j < T; ++j) acc[i][j] = v4i{0, 0, 0, 0};
    };
#pragma unroll
    for (int s = 0; s < kStages - 1; ++s) load(s, s);
    int left = group_steps;                                   // steps until the group ends (FLUSH 0 and 4)
    auto run_stage = [&](int s, auto tail) {                  // tail: fewer than four steps
        constexpr bool kTail = decltype(tail)::value;
        wait_vmcnt<ALIGNED ? (kStages - 2) * (kLoads + 1) : 0>();
        lds_barrier();                                        // stage s landed; stage s - 1 is no longer read
        load(s + kStages - 1, (s + kStages - 1) % kStages);
        const int8_t* base = lds + (s % kStages) * kStageBytes;
        float sw[kFlushes][T];
#pragma unroll
        for (int f = 0; f < kFlushes; ++f)
#pragma unroll
            for (int j = 0; j < T; ++j) sw[f][j] = ((const float*)(base + kChunks * 1024))[f * BN + wn + 16 * j + li];
        // operands of all four steps: lane l supplies row l % 16, values 8 (l / 16) + 0..7 of 32
        int64_t a[4][T], b[4][T];
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int i = 0; i < T; ++i) {
                const int seg = 2 * q + (lq >> 1), row = 16 * i + li;
                a[q][i] = *(const int64_t*)(base + (wm + row) * kStageK + ((seg ^ (row & 7)) * 16) + 8 * (lq & 1));
                const int8_t* wrow = base + kChunksX * 1024 + (wn + row) * kWBytes;
                if constexpr (BITS == 8) {
                    b[q][i] = *(const int64_t*)(wrow + ((seg ^ (row & 7)) * 16) + 8 * (lq & 1));
                } else {
                    const uint32_t p = *(const uint32_t*)(wrow + ((q ^ ((row >> 1) & 3)) * 16) + 4 * lq);
                    const v2u n = v2u{(p << 4) & 0xF0F0F0F0u, p & 0xF0F0F0F0u};
                    b[q][i] = *(const int64_t*)&n;
                    const v2u x = *(const v2u*)&a[q][i];
                    const v2u dealt = v2u{__builtin_amdgcn_perm(x.y, x.x, 0x06040200u),
                                          __builtin_amdgcn_perm(x.y, x.x, 0x07050301u)};
                    a[q][i] = *(const int64_t*)&dealt;
                }
            }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (kTail && 4 * s + q >= steps) break;
#pragma unroll
            for (int i = 0; i < T; ++i)
#pragma unroll
                for (int j = 0; j < T; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x32_i8(a[q][i], b[q][j], acc[i][j], 0, 0, 0);
            if constexpr (FLUSH == 1) {
                flush(0, sw[q]);
            } else if constexpr (FLUSH == 2) {
                if (q & 1) flush(0, sw[q / 2]);
            } else if constexpr (FLUSH == 0) {
                if (--left == 0) {
                    flush(group_of(s, q), sw[q]);
                    left = group_steps;
                }
            }
        }
        if constexpr (FLUSH == 4) {
            left -= 4;
            if (left == 0) {
                flush(0, sw[0]);
                left = group_steps;
            }
        }
    };
    for (int s = 0; s < steps / 4; ++s) run_stage(s, std::false_type());
    if (steps % 4) run_stage(steps / 4, std::true_type());
    wait_vmcnt<0>();                                          // no load into LDS outlives the loop
#pragma unroll
    for (int j = 0; j < T; ++j) {
        const int n = n0 + wn + 16 * j + li;
        if (n >= N) continue;
        const float bias = w.bias ? w.bias[n] : 0.0f;
#pragma unroll
        for (int i = 0; i < T; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int t = m0 + wm + 16 * i + 4 * lq + r;
                if (t >= tokens) continue;
                float* out = y + (size_t)t * N + n;
                const float v = res[i][j][r] + bias;
                *out = epilogue == kAccumulate ? *out + v : v;
            }
    }
}

template <int BITS, int FLUSH, int T, bool ALIGNED = true>
void launch_tiles(const WeightView& w, const int8_t* xq, const float* xs, int tokens, float* y, int epilogue,
                  int32_t* acc_out, int unfused, hipStream_t stream) {
    const int m_tiles = (tokens + 32 * T - 1) / (32 * T), n_tiles = (w.rows + 32 * T - 1) / (32 * T);
    gemm_grouped_kernel<BITS, FLUSH, T, ALIGNED><<<m_tiles * n_tiles, 256, 0, stream>>>(w, xq, xs, tokens, y, epilogue, acc_out,
                                                                              unfused, m_tiles);
}

template <int BITS, int T>
void launch_flush(const WeightView& w, const int8_t* xq, const float* xs, int tokens, float* y, int epilogue,
                  int32_t* acc_out, int unfused, hipStream_t stream) {
    if (reinterpret_cast<uintptr_t>(xq) & 15)
        launch_tiles<BITS, 0, T, false>(w, xq, xs, tokens, y, epilogue, acc_out, unfused, stream);
    else if (unfused || acc_out) launch_tiles<BITS, 0, T>(w, xq, xs, tokens, y, epilogue, acc_out, unfused, stream);
    else if (w.group == 32) launch_tiles<BITS, 1, T>(w, xq, xs, tokens, y, epilogue, acc_out, unfused, stream);
    else if (w.group == 64) launch_tiles<BITS, 2, T>(w, xq, xs, tokens, y, epilogue, acc_out, unfused, stream);
    else if (w.group % kStageK == 0) launch_tiles<BITS, 4, T>(w, xq, xs, tokens, y, epilogue, acc_out, unfused, stream);
    else launch_tiles<BITS, 0, T>(w, xq, xs, tokens, y, epilogue, acc_out, unfused, stream);
}

}  // namespace

bool gemm_grouped_supported(const WeightView& w) {
    return (w.bits == 8 || w.bits == 4) && w.cols > 0 && w.group > 0 && w.group % 32 == 0 && w.cols % w.group == 0 &&
           (reinterpret_cast<uintptr_t>(w.data) & 15) == 0;
}

void launch_gemm_grouped(const WeightView& w, const int8_t* xq, const float* xs, int tokens, float* y, int epilogue,
                         int32_t* acc_out, bool unfused, hipStream_t stream) {
    // 32 x 32 blocks keep a short input's chain of groups on four times the
    // waves (96 x 2048 x 2048 in groups of 128: 13 against 18 us); 64 x 64 read
    // their operands half as often once either fills the CUs (512 x 11264 x
    // 2048, groups of 64: 63 against 90 us).  In between they are level.
    const long blocks = (long)((tokens + 63) / 64) * ((w.rows + 63) / 64);
    const bool small = tokens >= 256 ? blocks < 256 : blocks < 512;
    if (w.bits == 8) {
        if (small) launch_flush<8, 1>(w, xq, xs, tokens, y, epilogue, acc_out, unfused, stream);
        else launch_flush<8, 2>(w, xq, xs, tokens, y, epilogue, acc_out, unfused, stream);
    } else {
        if (small) launch_flush<4, 1>(w, xq, xs, tokens, y, epilogue, acc_out, unfused, stream);
        else launch_flush<4, 2>(w, xq, xs, tokens, y, epilogue, acc_out, unfused, stream);
    }
}

}  // namespace leafhip
