// FP32-math GEMM on the bf16 matrix cores, with exact products.
//
//   Y[t, n] = sum_k X[t, k] W[n, k] (+ bias[n], or added to Y)
//
// for weights stored as f32, BF16, or int8 / int4 with group scales
// (decoder.cpp:236-251's storage).
//
// Why bf16.  The f32 matrix instruction runs at 1/15 of the bf16 one's rate
// (156 against 2255 TFLOP/s measured on this card), and an f32 value from 2^-110
// up is the sum of three bf16 values: hi = rn(x), mid = rn(x - hi),
// lo = x - hi - mid (split_bf16.h).  A product of two bf16 values is exact in f32, so
//   BF16 weights:  x w = hi w + mid w + lo w                3 MFMA products;
//   int8 / int4:   the integer is a bf16 value, the products are summed per
//                  scale group and the group's sum enters with one fused
//                  multiply-add of its scale                3 products;
//   f32 weights:   w is split as well; mid lo, lo mid and lo lo are left out
//                  (at most 2^-24 of x w together, 1e-8 rms)   6 products.
// The matrix core rounds once per product of 32 K values, so the sums lose
// less than a chain of f32 multiply-adds does (over 960 columns 1.0e-7 of the
// result for BF16 weights and 1.2e-7 for f32 ones, against 5.6e-7 with the f32
// matrix instruction).  A value whose pieces are not
// finite (infinity, NaN, or a magnitude that rounds past bf16's largest) gives
// a non-finite sum; such outputs are recomputed in plain f32.
//
// Fragments.  v_mfma_f32_16x16x32_bf16: the weight rows are its A operand and
// the tokens its B operand, lane l supplying row (token) l % 16 and the K
// values 8 (l / 16) + 0..7 of each 32.  A lane then holds one token and four
// consecutive weight rows: 16-byte stores.
#include <cstdlib>
#include <cstring>

#include "device_common.h"
#include "kernels.h"
#include "split_bf16.h"

namespace leafhip {
namespace {

constexpr int kStageK = 32;    // K values per stage: one MFMA's

// How a stored weight becomes MFMA operands.
enum WeightMode : int {
    kExactRow = 0,      // one bf16 plane; no scale, or one scale per row at the end
    kExactGroup = 1,    // one plane of integers, a scale per group of whole stages
    kSplit = 2,         // f32, or any other grouping dequantized to f32: three planes
};

// Eight consecutive values of a weight row as stored.
template <int BITS>
struct RawUnit {
    uint32_t r[BITS / 4];
};

// Values k..k+7 of a weight row.  TAIL: the row ends (K % 4 == 0) within or before the eight
// values, those past it are zero; only 4-value alignment is assumed.
template <int BITS, bool TAIL>
__device__ __forceinline__ RawUnit<BITS> load_unit(const uint8_t* row, int k, int K) {
    RawUnit<BITS> u;
    const uint8_t* p = row + (size_t)k * BITS / 8;
    if constexpr (!TAIL) {
        if constexpr (BITS == 32) {
            *(uint4*)u.r = *(const uint4*)p;
            *(uint4*)(u.r + 4) = *(const uint4*)(p + 16);
        } else if constexpr (BITS == 16) {
            *(uint4*)u.r = *(const uint4*)p;
        } else if constexpr (BITS == 8) {
            *(uint2*)u.r = *(const uint2*)p;
        } else {
            u.r[0] = *(const uint32_t*)p;
        }
    } else {
#pragma unroll
        for (int i = 0; i < BITS / 4; ++i) u.r[i] = 0;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (k + 4 * h >= K) continue;
            if constexpr (BITS == 32) *(uint4*)(u.r + 4 * h) = *(const uint4*)(p + 16 * h);
            else if constexpr (BITS == 16) *(uint2*)(u.r + 2 * h) = *(const uint2*)(p + 8 * h);
            else if constexpr (BITS == 8) u.r[h] = *(const uint32_t*)(p + 4 * h);
            else u.r[0] |= (uint32_t)*(const uint16_t*)(p + 2 * h) << (16 * h);
        }
    }
    return u;
}

// One wave's 16 MT tokens x 32 values of x, moved through LDS into operand
// order.  Global memory is read eight lanes to a token's 128 bytes: an operand
// load (one token per lane) keeps the address unit busy for each lane's 16 bytes
// by itself (four times the cycles: 12.6 instead of 8.3 us for 16 tokens x 768
// f32 rows x 3072).  Segment c of row r
// sits in slot c ^ (r % 8).  The region belongs to the wave: LDS operations
// of a wave are in order, so no barrier is needed.
template <bool TAIL, int MT>
struct TokenTile {
    const float* rows[2 * MT];   // lane / 8-th of each group of eight tokens
    float* lds;                  // 16 MT x 32 floats
    int lane, K;
    v4f raw[2 * MT];

    __device__ __forceinline__ void init(const float* x, int m0, int tokens, int k, float* region, int l) {
        lane = l;
        K = k;
        lds = region;
#pragma unroll
        for (int j = 0; j < 2 * MT; ++j) rows[j] = x + (size_t)min(m0 + 8 * j + (lane >> 3), tokens - 1) * K;
    }
    // values past K are zero with TAIL (K % 4 == 0)
    __device__ __forceinline__ void load(int s) {
        const int k = s * kStageK + 4 * (lane & 7);
#pragma unroll
        for (int j = 0; j < 2 * MT; ++j) {
            raw[j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
            if (!TAIL || k < K) raw[j] = *(const v4f*)(rows[j] + k);
        }
    }
    __device__ __forceinline__ void store() {
#pragma unroll
        for (int j = 0; j < 2 * MT; ++j)
            *(v4f*)(lds + (8 * j + (lane >> 3)) * 32 + (((lane & 7) ^ (lane >> 3)) * 4)) = raw[j];
        asm volatile("" ::: "memory");
        __builtin_amdgcn_wave_barrier();
    }
    // lane l: token l % 16 of each 16, values 8 (l / 16) + 0..7
    __device__ __forceinline__ void read(float (&f)[MT][8]) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const v4f v = *(const v4f*)(lds + (16 * i + (lane & 15)) * 32 + (((2 * (lane >> 4) + h) ^ (lane & 7)) * 4));
#pragma unroll
                for (int e = 0; e < 4; ++e) f[i][4 * h + e] = v[e];
            }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_wave_barrier();
    }
};

// One wave's 16 NT weight rows x 32 values: f32 and BF16 rows through LDS as
// TokenTile does (8 or 4 lanes to a row), int8 / int4 rows straight to operand
// order (8 or 4 bytes a lane).
template <int BITS, bool TAIL, int NT>
struct WeightTile {
    static constexpr bool kStaged = BITS >= 16;
    static constexpr int kLanes = BITS == 32 ? 8 : 4;        // lanes per row
    static constexpr int kLoads = kStaged ? NT * kLanes / 4 : NT;
    const uint8_t* rows[kLoads];
    uint8_t* lds;
    int lane, K;
    v4u raw[kStaged ? kLoads : 1];
    RawUnit<BITS> direct[kStaged ? 1 : NT];

    __device__ __forceinline__ void init(const WeightView& w, int n0, float* region, int l) {
        lane = l;
        K = w.cols;
        lds = (uint8_t*)region;
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const int row = kStaged ? j * (64 / kLanes) + lane / kLanes : 16 * j + (lane & 15);
            rows[j] = (const uint8_t*)w.data + (size_t)min(n0 + row, w.rows - 1) * K * BITS / 8;
        }
    }
    __device__ __forceinline__ void load(const WeightView& w, int s) {
        if constexpr (BITS == 32) {
            const int k = s * kStageK + 4 * (lane & 7);
#pragma unroll
            for (int j = 0; j < kLoads; ++j) {
                raw[j] = v4u{0, 0, 0, 0};
                if (!TAIL || k < K) raw[j] = *(const v4u*)(rows[j] + 4 * k);
            }
        } else {
            const int k = s * kStageK + 8 * (kStaged ? lane & 3 : lane >> 4);
#pragma unroll
            for (int j = 0; j < kLoads; ++j) {
                const RawUnit<BITS> u = load_unit<BITS, TAIL>(rows[j], k, K);
                if constexpr (kStaged) raw[j] = *(const v4u*)u.r;
                else direct[j] = u;
            }
        }
    }
    __device__ __forceinline__ void store() {
        if constexpr (kStaged) {
#pragma unroll
            for (int j = 0; j < kLoads; ++j) {
                const int row = j * (64 / kLanes) + lane / kLanes, seg = lane % kLanes;
                const int slot = BITS == 32 ? seg ^ (row & 7) : seg ^ ((row >> 1) & 3);
                *(v4u*)(lds + row * (16 * kLanes) + slot * 16) = raw[j];
            }
            asm volatile("" ::: "memory");
            __builtin_amdgcn_wave_barrier();
        }
    }
    __device__ __forceinline__ void read(RawUnit<BITS> (&u)[NT]) {
        const int li = lane & 15, lq = lane >> 4;
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            if constexpr (BITS == 32) {
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    *(v4u*)(u[n].r + 4 * h) = *(const v4u*)(lds + (16 * n + li) * 128 + (((2 * lq + h) ^ (li & 7)) * 16));
            } else if constexpr (BITS == 16) {
                *(v4u*)u[n].r = *(const v4u*)(lds + (16 * n + li) * 64 + ((lq ^ ((li >> 1) & 3)) * 16));
            } else {
                u[n] = direct[n];
            }
        }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_wave_barrier();
    }
};

// Two exact f32 -> bf16 (the values have at most eight significant bits).
__device__ __forceinline__ uint32_t pack_bf16_exact(float a, float b) {
    return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}

// The stored integers as f32: int8 values, or int4 values / 16.
template <int BITS>
__device__ __forceinline__ void integers(const RawUnit<BITS>& u, float (&f)[8]) {
    if constexpr (BITS == 8) {
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = (float)(int)(int8_t)((u.r[e / 4] >> (8 * (e & 3))) & 0xFFu);
    } else {
        int4_sixteenths(u.r[0], f);
    }
}

// What a stored scale multiplies: int4 values enter as value / 16.
template <int BITS>
constexpr float kScaleFactor = BITS == 4 ? 16.0f : 1.0f;

// Operand planes of eight weights: out[0] (exact modes) or out[0..2] (split).
// The two scales are those of the unit's halves (kSplit of int8 / int4 only).
template <int BITS, int MODE>
__device__ __forceinline__ void unit_planes(const RawUnit<BITS>& u, float scale0, float scale1,
                                            v8bf (&out)[MODE == kSplit ? 3 : 1]) {
    if constexpr (MODE == kSplit) {
        float f[8];
        if constexpr (BITS == 32) {
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] = __uint_as_float(u.r[e]);
        } else {
            integers<BITS>(u, f);   // value / 16 times 16 scale: the dequantized value's single rounding
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] = f[e] * (e < 4 ? scale0 : scale1);
        }
        split8(f, out[0], out[1], out[2]);
    } else if constexpr (BITS == 16) {
        out[0] = *(const v8bf*)u.r;
    } else {
        float f[8];
        integers<BITS>(u, f);
        uint32_t packed[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) packed[p] = pack_bf16_exact(f[2 * p], f[2 * p + 1]);
        out[0] = *(const v8bf*)packed;
    }
}

__device__ __forceinline__ bool finite(float v) { return __builtin_fabsf(v) < INFINITY; }

// The lane's number, from no register that would stay live for it (one or two
// more and some of the kernels below lose a wave per SIMD).
__device__ __forceinline__ int this_lane() { return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0)); }

// Where the split sum is not finite: outputs t, row..row + 3 in f32, by the whole
// wave (rows past the last give the last one's).  One infinite activation
// spoils its token's every output: 300 tokens x 5120 BF16 rows x 960 with one
// such token take 62 us, with 300 735 (19 without; 2,612 and 3,558 as one
// chain per lane).
template <int BITS>
__device__ __forceinline__ void plain_quad(const WeightView& w, const float* x, int t, int row, float (&sum)[4]) {
    const int K = w.cols, groups = BITS <= 8 ? K / w.group : 1;
#pragma unroll
    for (int r = 0; r < 4; ++r) sum[r] = 0.0f;
#pragma unroll 1
    for (int k = 4 * this_lane(); k < K; k += 256) {
        const v4f xv = *(const v4f*)(x + (size_t)t * K + k);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int n = min(row + r, w.rows - 1);
            const uint8_t* p = (const uint8_t*)w.data + ((size_t)n * K + k) * BITS / 8;
            float v[4];
            if constexpr (BITS == 32) {
                const v4f u = *(const v4f*)p;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = u[e];
            } else if constexpr (BITS == 16) {
                const v2u u = *(const v2u*)p;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = bf16_to_f32((u[e / 2] >> (16 * (e & 1))) & 0xFFFFu);
            } else {
                const float scale = w.scales[(size_t)n * groups + k / w.group];   // groups are whole quads
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[e] = (float)(BITS == 8 ? (int)(int8_t)p[e] : nibble(p[e / 2], e & 1)) * scale;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) sum[r] = fmaf(xv[e], v[e], sum[r]);
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) sum[r] = wave_sum_f32(sum[r]);
}

// The operand planes of product q of a 16 x 16 x 32 step, small products first.
template <int PLANES>
constexpr int kProducts = PLANES == 3 ? 6 : 3;
template <int PLANES>
constexpr int w_plane(int q) {
    constexpr int of3[6] = {2, 1, 0, 1, 0, 0};
    return PLANES == 3 ? of3[q] : 0;
}
template <int PLANES>
constexpr int x_plane(int q) {
    constexpr int of3[6] = {0, 1, 2, 0, 1, 0};
    return PLANES == 3 ? of3[q] : 2 - q;
}

// Tiled kernel.  A block of WM waves owns 16 MT WM tokens x 16 NT weight rows,
// each wave MT x NT MFMA tiles of its own tokens, so x is split once per block
// and wave; the weight tile is shared by the block: widened on its way into
// LDS (two buffers, one barrier a stage), rows of 64 bytes with segment c of
// row r in slot c ^ (r / 2 % 4), which spreads any eight consecutive rows of an
// operand read over all banks.  Loads run a stage ahead, and every stage issues
// the same ones, so that a wait names a fixed number of loads still in flight
// (conditional loads made every wait a full one: 100 instead of 66 us for 777
// tokens x 896 rows x 4864).
//
// What bounds it: 2048 tokens x 5120 BF16 rows x 960 takes 67 us (was 221 with
// f32 MFMAs): 30 us of MFMAs at the rate the card holds on such data (2.0
// PFLOP/s at 2.06 GHz), 8 us to write the 42 MB result, the rest the staging of
// a stage and the last, partly filled round of blocks.  While a CU is busy its
// matrix cores are for 50% of the time and vector instructions issue for 49%.
// Where the tiles are few (the same block's down projection, 960 rows x 2560:
// 256 blocks, one wave a SIMD) 30% and 27%: loads are waited for.  Splitting x
// in a pass of its own measured the same (68 us, 5 of them the pass).
template <int BITS, int MODE, bool TAIL, int MT, int NT, int WM>
__global__ __launch_bounds__(64 * WM, 2) void gemm_f32_tiled_kernel(WeightView w, const float* __restrict__ x, int tokens,
                                                                float* __restrict__ y, int epilogue, int m_tiles,
                                                                int n_tiles, bool vec) {
    constexpr int kThreads = 64 * WM, BM = 16 * MT * WM, BN = 16 * NT;
    constexpr int kPlanes = MODE == kSplit ? 3 : 1;
    constexpr int kUnits = BN * 4 / kThreads;                // 8-value units per thread per stage
    static_assert(kUnits * kThreads == BN * 4 && BN <= kThreads, "units divide among the threads");
    constexpr int kPlaneBytes = BN * 64, kBuffer = kPlanes * kPlaneBytes;
    __shared__ __align__(1024) uint8_t lds[2 * kBuffer];
    __shared__ __align__(16) float scale_lds[MODE == kExactGroup ? 2 * BN : 4];
    __shared__ __align__(128) float x_lds[WM][MT * 512];

    // Blocks go to the eight XCDs round robin: each XCD takes a contiguous run
    // of tiles, token tiles fastest, so its L2 holds few weight tiles at a time.
    const int per = (m_tiles * n_tiles + 7) / 8;
    const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (tile >= m_tiles * n_tiles) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int li = lane & 15, lq = lane >> 4;
    const int K = w.cols, N = w.rows;
    const int n0 = (tile / m_tiles) * BN, m0 = (tile % m_tiles) * BM + wave * 16 * MT;
    const int ns = (K + kStageK - 1) / kStageK;
    const int groups = BITS <= 8 ? K / w.group : 1;

    TokenTile<TAIL, MT> xt;
    xt.init(x, m0, tokens, K, x_lds[wave], lane);
    RawUnit<BITS> raw[kUnits];
    float raw_scale[kUnits][2];
    float group_scale = 0.0f;
    auto load_w = [&](int s) {
#pragma unroll
        for (int j = 0; j < kUnits; ++j) {
            const int u = threadIdx.x + j * kThreads;
            const int row = min(n0 + (u >> 2), N - 1), k = s * kStageK + (u & 3) * 8;
            raw[j] = load_unit<BITS, TAIL>((const uint8_t*)w.data + (size_t)row * K * BITS / 8, k, K);
            if constexpr (MODE == kSplit && BITS <= 8) {
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    raw_scale[j][h] = w.scales[(size_t)row * groups + min(k + 4 * h, K - 1) / w.group];
            }
        }
        if constexpr (MODE == kExactGroup)
            if (threadIdx.x < BN)
                group_scale = w.scales[(size_t)min(n0 + (int)threadIdx.x, N - 1) * groups + s * kStageK / w.group];
    };
    auto store_w = [&](int buffer) {
#pragma unroll
        for (int j = 0; j < kUnits; ++j) {
            const int u = threadIdx.x + j * kThreads, row = u >> 2, seg = u & 3;
            v8bf planes[kPlanes];
            unit_planes<BITS, MODE>(raw[j], raw_scale[j][0] * kScaleFactor<BITS>, raw_scale[j][1] * kScaleFactor<BITS>,
                                    planes);
#pragma unroll
            for (int p = 0; p < kPlanes; ++p)
                *(v8bf*)(lds + buffer * kBuffer + p * kPlaneBytes + row * 64 + ((seg ^ ((row >> 1) & 3)) * 16)) =
                    planes[p];
        }
        if constexpr (MODE == kExactGroup)
            if (threadIdx.x < BN) scale_lds[buffer * BN + threadIdx.x] = group_scale * kScaleFactor<BITS>;
    };

    v4f acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[i][n] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    constexpr int NG = kPlanes == 1 && MT == 1 ? 4 : 2;      // weight tiles whose operands are read together
    const int frag = li * 64 + ((lq ^ ((li >> 1) & 3)) * 16);   // within a 16-row operand
    v8bf wf[2][NG][kPlanes];
    v4f sc[2][NG];
    auto read_w = [&](int s, int g) {
        const uint8_t* base = lds + (s & 1) * kBuffer + frag;
#pragma unroll
        for (int n = 0; n < NG; ++n) {
#pragma unroll
            for (int p = 0; p < kPlanes; ++p)
                wf[g & 1][n][p] = *(const v8bf*)(base + p * kPlaneBytes + (g * NG + n) * 1024);
            if constexpr (MODE == kExactGroup)
                sc[g & 1][n] = *(const v4f*)(scale_lds + (s & 1) * BN + 16 * (g * NG + n) + 4 * lq);
        }
    };
    // Every stage issues the same loads (the last stages load the last one
    // again), so that a wait names a fixed number of loads still in flight.
    float xf[MT][8];
    auto stage = [&](int s) {
        read_w(s, 0);
        v8bf xs[MT][3];
#pragma unroll
        for (int i = 0; i < MT; ++i) split8(xf[i], xs[i][0], xs[i][1], xs[i][2]);
        xt.store();                                          // stage s + 1, loaded a stage ago
        xt.load(min(s + 2, ns - 1));
        xt.read(xf);
#pragma unroll
        for (int g = 0; g < NT / NG; ++g) {
            if (g + 1 < NT / NG) read_w(s, g + 1);
            v4f c[MT][NG];
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int n = 0; n < NG; ++n)
                    c[i][n] = MODE == kExactGroup ? v4f{0.0f, 0.0f, 0.0f, 0.0f} : acc[i][g * NG + n];
            // small products first; consecutive MFMAs are independent
#pragma unroll
            for (int q = 0; q < kProducts<kPlanes>; ++q)
#pragma unroll
                for (int n = 0; n < NG; ++n)
#pragma unroll
                    for (int i = 0; i < MT; ++i)
                        c[i][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            wf[g & 1][n][w_plane<kPlanes>(q)], xs[i][x_plane<kPlanes>(q)], c[i][n], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int n = 0; n < NG; ++n) {
                    v4f& a = acc[i][g * NG + n];
                    if constexpr (MODE == kExactGroup) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) a[r] = fmaf(c[i][n][r], sc[g & 1][n][r], a[r]);
                    } else {
                        a = c[i][n];
                    }
                }
        }
        store_w((s + 1) & 1);         // last read in stage s - 1, before the barrier that ended it
        load_w(min(s + 2, ns - 1));
        lds_barrier();
    };
    load_w(0);
    xt.load(0);
    store_w(0);
    load_w(min(1, ns - 1));
    xt.store();
    xt.load(min(1, ns - 1));
    xt.read(xf);
    lds_barrier();
    for (int s = 0; s < ns; ++s) stage(s);

    // ---- epilogue: lane holds token m0 + 16 i + li and rows n0 + 16 n + 4 lq + r
    // (rows past N read the last row's scale and bias and are not stored)
    uint32_t bad = 0;                                        // quads to recompute
    static_assert(MT * NT <= 32, "one bit per quad");
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int row = n0 + 16 * n + 4 * lq;
        v4f sc4 = v4f{1.0f, 1.0f, 1.0f, 1.0f}, bias = v4f{0.0f, 0.0f, 0.0f, 0.0f};
        if constexpr (MODE == kExactRow && BITS <= 8)
#pragma unroll
            for (int r = 0; r < 4; ++r) sc4[r] = w.scales[min(row + r, N - 1)] * kScaleFactor<BITS>;
        if (w.bias)
#pragma unroll
            for (int r = 0; r < 4; ++r) bias[r] = w.bias[min(row + r, N - 1)];
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const int t = m0 + 16 * i + li;
            if (t >= tokens || row >= N) continue;
            v4f v = acc[i][n];
            if constexpr (MODE == kExactRow && BITS <= 8) v *= sc4;
            if (!(finite(v[0]) && finite(v[1]) && finite(v[2]) && finite(v[3]))) {
                bad |= 1u << (i * NT + n);
                continue;
            }
            v += bias;
            float* out = y + (size_t)t * N + row;
            if (vec) {
                if (epilogue == kAccumulate) v = *(const v4f*)out + v;
                *(v4f*)out = v;
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (row + r < N) out[r] = epilogue == kAccumulate ? out[r] + v[r] : v[r];
            }
        }
    }
    // the wave's lanes bring their quads up one after the other
    while (const uint64_t lanes = __ballot(bad != 0)) {
        const int from = __builtin_ctzll(lanes), b = __builtin_ctz((uint32_t)__shfl((int)bad, from, 64));
        const int lane = this_lane();
        if (lane == from) bad &= bad - 1;
        const int t = m0 + 16 * (b / NT) + (from & 15), row = n0 + 16 * (b % NT) + 4 * (from >> 4);
        float sum[4];
        plain_quad<BITS>(w, x, t, row, sum);
        if (lane < 4 && row + lane < N) {
            float* out = y + (size_t)t * N + row + lane;
            const float v = (lane & 2 ? lane & 1 ? sum[3] : sum[2] : lane & 1 ? sum[1] : sum[0]) +
                            (w.bias ? w.bias[row + lane] : 0.0f);
            *out = epilogue == kAccumulate ? *out + v : v;
        }
    }
}

// Few tokens (or few tiles): the whole block shares 16 MT tokens x 16 NT weight
// rows, and its WK waves take every WK-th stage of K, so that a short input
// still keeps enough loads in flight on enough CUs.  Each wave moves both
// operands through LDS of its own (each weight is used by one wave only); the
// waves' sums are added in wave order.  Bound by the latency of ns / WK stages:
// 16 tokens x 768 f32 rows x 3072 take 7.8 us (was 64 as 12 blocks of 64 x 64);
// where blocks are many by splitting x, once for every 32 weight rows (777
// tokens x 896 INT4 rows x 4864, 67 us: vector instructions issue for 69% of a
// CU's time, MFMAs run for 21%).
template <int BITS, int MODE, bool TAIL, int MT, int NT, int WK>
__global__ __launch_bounds__(64 * WK) void gemm_f32_few_kernel(WeightView w, const float* __restrict__ x, int tokens,
                                                                 float* __restrict__ y, int epilogue) {
    constexpr int kPlanes = MODE == kSplit ? 3 : 1;
    // each wave's x (and f32 / BF16 weight) tiles; afterwards every wave's sums
    constexpr int kTileFloats = MT * 512 + (BITS == 32 ? NT * 512 : BITS == 16 ? NT * 256 : 0);
    constexpr int kWaveFloats = kTileFloats > MT * NT * 256 ? kTileFloats : MT * NT * 256;
    __shared__ __align__(128) float red[WK * kWaveFloats];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int li = lane & 15, lq = lane >> 4;
    const int K = w.cols, N = w.rows;
    const int n0 = blockIdx.x * 16 * NT, m0 = blockIdx.y * 16 * MT;
    const int ns = (K + kStageK - 1) / kStageK;
    const int groups = BITS <= 8 ? K / w.group : 1;
    float* region = red + wave * kWaveFloats;
    TokenTile<TAIL, MT> xt;
    xt.init(x, m0, tokens, K, region, lane);
    WeightTile<BITS, TAIL, NT> wt;
    wt.init(w, n0, region + MT * 512, lane);
    float scale[NT][2];
    auto load = [&](int s) {
        wt.load(w, s);
        const int k = s * kStageK + 8 * lq;
        if constexpr (BITS <= 8 && MODE != kExactRow)
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                const float* row = w.scales + (size_t)min(n0 + 16 * n + li, N - 1) * groups;
                scale[n][0] = row[min(k, K - 1) / w.group] * kScaleFactor<BITS>;
                if constexpr (MODE == kSplit) scale[n][1] = row[min(k + 4, K - 1) / w.group] * kScaleFactor<BITS>;
            }
        xt.load(s);
    };
    // tokens are the A operand here: a lane's outputs share one weight row (one scale)
    v4f acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[i][n] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    auto use = [&](int next) {
        RawUnit<BITS> raw[NT];
        float sc[NT][2], xf[MT][8];
        xt.store();
        wt.store();
        xt.read(xf);
        wt.read(raw);
#pragma unroll
        for (int n = 0; n < NT; ++n) sc[n][0] = scale[n][0], sc[n][1] = scale[n][1];
        load(min(next, ns - 1));
        v8bf wf[NT][kPlanes];
#pragma unroll
        for (int n = 0; n < NT; ++n) unit_planes<BITS, MODE>(raw[n], sc[n][0], sc[n][1], wf[n]);
        v8bf xs[MT][3];
#pragma unroll
        for (int i = 0; i < MT; ++i) split8(xf[i], xs[i][0], xs[i][1], xs[i][2]);
        v4f c[MT][NT];
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int n = 0; n < NT; ++n) c[i][n] = MODE == kExactGroup ? v4f{0.0f, 0.0f, 0.0f, 0.0f} : acc[i][n];
#pragma unroll
        for (int q = 0; q < kProducts<kPlanes>; ++q)
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int i = 0; i < MT; ++i)
                    c[i][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xs[i][x_plane<kPlanes>(q)],
                                                                      wf[n][w_plane<kPlanes>(q)], c[i][n], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                if constexpr (MODE == kExactGroup) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[i][n][r] = fmaf(c[i][n][r], sc[n][0], acc[i][n][r]);
                } else {
                    acc[i][n] = c[i][n];
                }
            }
    };
    if (wave < ns) {
        load(wave);
        for (int s = wave; s < ns; s += WK) use(s + WK);
    }
    __syncthreads();       // the tiles are no longer read
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int n = 0; n < NT; ++n) *(v4f*)(red + wave * kWaveFloats + (i * NT + n) * 256 + 4 * lane) = acc[i][n];
    __syncthreads();
    for (int e = threadIdx.x; e < MT * NT * 256; e += 64 * WK) {
        // outputs of a token consecutive over the weight rows
        const int tok = e / (16 * NT), col = e % (16 * NT);
        const int i = tok / 16, n = col / 16;
        const int at = (i * NT + n) * 256 + 4 * (16 * ((tok & 15) >> 2) + (col & 15)) + (tok & 3);
        const int t = m0 + tok, row = n0 + col;
        const bool live = t < tokens && row < N;
        float v = 0.0f;
#pragma unroll
        for (int q = 0; q < WK; ++q) v += red[q * kWaveFloats + at];
        if constexpr (MODE == kExactRow && BITS <= 8) v *= w.scales[min(row, N - 1)] * kScaleFactor<BITS>;
        // (four lanes in a row have one token and four rows of weights)
        for (uint64_t lanes = __ballot(live && !finite(v)); lanes;) {
            const int from = __builtin_ctzll(lanes) & ~3;
            lanes &= ~((uint64_t)15 << from);
            float sum[4];
            plain_quad<BITS>(w, x, __shfl(t, from, 64), __shfl(row, from, 64), sum);
            if ((lane & ~3) == from && !finite(v))
                v = lane & 2 ? lane & 1 ? sum[3] : sum[2] : lane & 1 ? sum[1] : sum[0];
        }
        if (!live) continue;
        v += w.bias ? w.bias[row] : 0.0f;
        float* out = y + (size_t)t * N + row;
        *out = epilogue == kAccumulate ? *out + v : v;
    }
}

template <int BITS, int MODE, bool TAIL, int MT, int NT, int WM>
void launch_tiles(const WeightView& w, const float* x, int tokens, float* y, int epilogue, hipStream_t stream) {
    const int m_tiles = (tokens + 16 * MT * WM - 1) / (16 * MT * WM), n_tiles = (w.rows + 16 * NT - 1) / (16 * NT);
    const bool vec = w.rows % 4 == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0;
    gemm_f32_tiled_kernel<BITS, MODE, TAIL, MT, NT, WM><<<(m_tiles * n_tiles + 7) / 8 * 8, 64 * WM, 0, stream>>>(
        w, x, tokens, y, epilogue, m_tiles, n_tiles, vec);
}

template <int BITS, int MODE, bool TAIL, int MT, int NT, int WK>
void launch_few(const WeightView& w, const float* x, int tokens, float* y, int epilogue, hipStream_t stream) {
    const dim3 grid((w.rows + 16 * NT - 1) / (16 * NT), (tokens + 16 * MT - 1) / (16 * MT));
    gemm_f32_few_kernel<BITS, MODE, TAIL, MT, NT, WK><<<grid, 64 * WK, 0, stream>>>(w, x, tokens, y, epilogue);
}

// The blocks a product may run as: tiles of gemm_f32_tiled_kernel (tokens x rows),
// then those of gemm_f32_few_kernel.
enum Shape { k128x64, k64x128, k128x128, k64x64, kFew16x16, kFew32x16, kFew16x32, kFew32x32, kFew64x32, kShapes };
constexpr int kShapeTokens[kShapes] = {128, 64, 128, 64, 16, 32, 16, 32, 64};
constexpr int kShapeRows[kShapes] = {64, 128, 128, 64, 16, 16, 32, 32, 32};

// Microseconds of a product as t0 + t1 K + t2 K rounds + t3 blocks / 256, with
// rounds = ceil(blocks / 256 CUs): least-squares fits to 1,460 products timed
// on an MI355X (14 token counts from 5 to 2048 over 11 weight shapes from
// 256 x 1024 to 11264 x 2048, every shape of block that suits them).  Choosing
// by them costs 1-3% on average over the best shape of each product.
constexpr double kCost[3][kShapes][4] = {
    // one plane, no scale groups (BF16, per-row int8)
    {{3.4, 0.00379, 0.0143, 0}, {3.92, 0.00287, 0.0124, 0}, {6.56, 0, 0.0237, 0}, {2.36, 0.00447, 0.00738, 0},
     {2.94, 0, 0.00121, 0.242}, {2.56, 0.000499, 0.00221, 0.0235}, {2.98, 0, 0.00188, 0.00484},
     {2.78, 0.000202, 0.00286, 0.541}, {2.97, 0, 0.00541, 1.91}},
    // scale groups (int4)
    {{4.49, 0.00947, 0.0149, 0}, {4.95, 0.00608, 0.0147, 0}, {6.17, 0.00455, 0.0301, 0}, {4.08, 0.00608, 0.00831, 0},
     {2.38, 0.00025, 0.00212, 0}, {2.49, 0.000234, 0.00273, 0}, {2.0, 0.000846, 0.00339, 0},
     {2.69, 0.000485, 0.00415, 0}, {3.11, 0, 0.00577, 2.85}},
    // three planes (f32)
    {{5.1, 0.00155, 0.0236, 0}, {5.26, 0, 0.0275, 0}, {6.91, 0, 0.0409, 0}, {2.93, 0.00727, 0.0134, 0},
     {2.72, 0, 0.00197, 0.154}, {2.4, 0.000155, 0.00318, 0}, {2.39, 0.000136, 0.00342, 0},
     {2.61, 0.000128, 0.00473, 0.595}, {2.05, 0, 0.00751, 3.79}}};

// LEAF_F32_GEMM_TILE=128x64|64x128|128x128|64x64|few16x16|few32x16|few16x32|
// few32x32|few64x32 (tokens x rows) forces a block (tests compare them); any
// other value, or none, lets the cost decide.
Shape choose_shape(int mode, int tokens, int rows, int K) {
    if (const char* v = getenv("LEAF_F32_GEMM_TILE")) {
        const char* names[kShapes] = {"128x64",   "64x128",   "128x128",  "64x64",   "few16x16",
                                      "few32x16", "few16x32", "few32x32", "few64x32"};
        for (int i = 0; i < kShapes; ++i)
            if (strcmp(v, names[i]) == 0) return Shape(i);
    }
    Shape best = k128x64;
    double best_cost = 0.0;
    for (int i = 0; i < kShapes; ++i) {
        const long blocks = (long)((tokens + kShapeTokens[i] - 1) / kShapeTokens[i]) *
                            ((rows + kShapeRows[i] - 1) / kShapeRows[i]);
        const double* c = kCost[mode][i];
        const double cost = c[0] + K * (c[1] + c[2] * (double)((blocks + 255) / 256)) + c[3] * (double)blocks / 256;
        if (i == 0 || cost < best_cost) {
            best = Shape(i);
            best_cost = cost;
        }
    }
    return best;
}

template <int BITS, int MODE, bool TAIL>
void launch_mode(const WeightView& w, const float* x, int tokens, float* y, int epilogue, hipStream_t stream) {
    const Shape shape = choose_shape(MODE, tokens, w.rows, w.cols);
#define LEAF_TILE(MT, NT) launch_tiles<BITS, MODE, TAIL, MT, NT, 4>(w, x, tokens, y, epilogue, stream)
#define LEAF_FEW(MT, NT, WK) launch_few<BITS, MODE, TAIL, MT, NT, WK>(w, x, tokens, y, epilogue, stream)
    if constexpr (MODE == kSplit && BITS <= 8) {
        // groups that are not whole stages: any size, two shapes
        if (shape <= k64x64) LEAF_TILE(1, 4);
        else LEAF_FEW(2, 2, 8);
    } else {
        switch (shape) {
        case k128x64: LEAF_TILE(2, 4); break;
        case k64x128: LEAF_TILE(1, 8); break;
        case k128x128: LEAF_TILE(2, 8); break;
        case k64x64: LEAF_TILE(1, 4); break;
        case kFew16x16: LEAF_FEW(1, 1, 16); break;
        case kFew32x16: LEAF_FEW(2, 1, 8); break;
        case kFew16x32: LEAF_FEW(1, 2, 8); break;
        case kFew32x32: LEAF_FEW(2, 2, 8); break;
        default: LEAF_FEW(4, 2, 8); break;
        }
    }
#undef LEAF_TILE
#undef LEAF_FEW
}

template <int BITS>
void launch_bits(const WeightView& w, const float* x, int tokens, float* y, int epilogue, hipStream_t stream) {
    const bool tail = w.cols % kStageK != 0;
    if constexpr (BITS >= 16) {
        constexpr int mode = BITS == 32 ? kSplit : kExactRow;
        if (tail) launch_mode<BITS, mode, true>(w, x, tokens, y, epilogue, stream);
        else launch_mode<BITS, mode, false>(w, x, tokens, y, epilogue, stream);
    } else {
        if (!tail && w.group == w.cols) launch_mode<BITS, kExactRow, false>(w, x, tokens, y, epilogue, stream);
        else if (!tail && w.group % kStageK == 0) launch_mode<BITS, kExactGroup, false>(w, x, tokens, y, epilogue, stream);
        else launch_mode<BITS, kSplit, true>(w, x, tokens, y, epilogue, stream);
    }
}

}  // namespace

bool gemm_f32_supported(const WeightView& w, const float* x) {
    auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    if (w.cols <= 0 || w.cols % 4 != 0 || !aligned(x) || !aligned(w.data)) return false;
    if ((w.bits == 8 || w.bits == 4) && (w.group <= 0 || w.group % 4 != 0 || w.cols % w.group != 0)) return false;
    return w.bits == 32 || w.bits == 16 || w.bits == 8 || w.bits == 4;
}

void launch_gemm_f32(const WeightView& w, const float* x, int tokens, float* y, int epilogue, hipStream_t stream) {
    switch (w.bits) {
    case 32: launch_bits<32>(w, x, tokens, y, epilogue, stream); break;
    case 16: launch_bits<16>(w, x, tokens, y, epilogue, stream); break;
    case 8: launch_bits<8>(w, x, tokens, y, epilogue, stream); break;
    default: launch_bits<4>(w, x, tokens, y, epilogue, stream); break;
    }
}

}  // namespace leafhip
