// Projections of a long block of tokens (a prompt, a large host batch) on
// the matrix cores: the weights of a row tile decoded once for all of a
// workgroup's tokens.
//
// The sixteen-token GEMMs (qwn_gemv.hip) give each 16-row x 16-token tile a
// workgroup of its own, so every sixteen tokens load and decode the weights
// again and fetch their own activations: 64 tokens through one Qwen2-1.5B
// Q4_0 layer take 34 us of GEMMs, 1003 tokens 545 us in sixteen such blocks.
// Here a workgroup takes 64 or 128 rows x 64 tokens (fewer tokens where that
// leaves CUs without one), its activations staged through LDS once for its
// four waves: the 1003 tokens take 201 us in four launches, and the whole
// prompt through two layers 0.62 ms instead of 2.57.
// The gate/up launch (55 GFLOP, 97 us, 0.57 PFLOP/s) keeps the vector ALU
// busy half of the time and the matrix cores a quarter: waits for a unit's
// loads and the last, half-filled round of workgroups take the rest.
//
// Numerics are the sixteen-token GEMM's: exact products per weight block,
// one fp32 multiply-add per block and output with the row's scale(s), the
// per-token activation scale at the end.
//   HyperVSQ-2: int8 weights s_oct (q - 1) from a byte permute, four
//     v_mfma_i32_16x16x64_i8 per 256-weight block.
//   Q4_0: n - 8 and the int8 activations as f16 (both exact), one
//     v_mfma_f32_16x16x32_f16 per 32-weight block: every product and sum is
//     an integer below 2^15, so the fp32 result is the exact block dot that
//     the int8 instruction gives, at the same rate, without the
//     int-to-float conversion of every output and block.  (The kernel is
//     bound by the vector ALU: per block and output one multiply-add here,
//     a conversion more there.)
#include "qwn_device.h"
#include "qwn_internal.h"

#include <algorithm>

namespace qwn {
namespace {

typedef int wide_v4i __attribute__((ext_vector_type(4)));
typedef float wide_v4f __attribute__((ext_vector_type(4)));
typedef _Float16 wide_v2h __attribute__((ext_vector_type(2)));
typedef _Float16 wide_v8h __attribute__((ext_vector_type(8)));

constexpr int kWideWaves = 4;           // waves of a set: 16 RT rows each
constexpr int kTokenGroups = 4;         // 16-token groups of a workgroup (two where few tiles exist)
constexpr uint32_t kUnitImage = 4096;   // image bytes of one unit of a 16-token group (without the sums)

struct WideArgs {
    const uint8_t *payload[kMaxGroup];
    const uint8_t *meta[kMaxGroup];
    float *output[kMaxGroup];
    const float *bias[kMaxGroup];
    uint32_t rows[kMaxGroup];
    uint32_t stride[kMaxGroup];
    uint32_t job_block[kMaxGroup + 1];
    uint32_t units;
    const uint8_t *image;   // one image per 16-token group
    uint32_t group_bytes;
    const float *scales;
    uint32_t ntok, accumulate;
};

// The four operand words of one weight block for each of a unit's four
// matrix instructions, from a lane's 16 payload bytes.
// HyperVSQ-2: 64 code bytes quarter sl of chunk g (the lane's octants 2g,
// 2g + 1) through the table [-s, 0, s, 2s].
__device__ __forceinline__ void decode_hv(const uint4 &p, uint32_t subs, wide_v4i (&w)[4]) {
    const uint32_t cw[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
    for (int sl = 0; sl < 4; ++sl) {
        const uint32_t sub = (subs >> (4 * (sl >> 1))) & 15u;
        const uint32_t lut = ((0u - sub) & 0xffu) | (sub << 16) | ((2u * sub) << 24);
        const uint32_t c = cw[sl];
        w[sl].x = static_cast<int>(__builtin_amdgcn_perm(0u, lut, c & 0x03030303u));
        w[sl].y = static_cast<int>(__builtin_amdgcn_perm(0u, lut, (c >> 2) & 0x03030303u));
        w[sl].z = static_cast<int>(__builtin_amdgcn_perm(0u, lut, (c >> 4) & 0x03030303u));
        w[sl].w = static_cast<int>(__builtin_amdgcn_perm(0u, lut, (c >> 6) & 0x03030303u));
    }
}

// Q4_0: nibbles n placed in the low mantissa bits of 1024.0 (low nibbles) or
// 16 n in those of 1024.0 (high nibbles) give 1024 + n and 1024 + 16 n; one
// packed f16 operation leaves n - 8, exactly.  Word order of the image:
// elements {0, 4}, {1, 5}, {2, 6}, {3, 7} of the lane's eight.
// The constants in registers let the mask and the or be one instruction
// (v_and_or_b32 takes no literal).
__device__ __forceinline__ wide_v8h decode_q4(uint32_t c, uint32_t mlow, uint32_t mhigh, uint32_t k1024) {
    const uint32_t c8 = c >> 8;
    auto low = [&](uint32_t v) {
        const wide_v2h h = __builtin_bit_cast(wide_v2h, (v & mlow) | k1024);
        return h - wide_v2h{static_cast<_Float16>(1032.0f), static_cast<_Float16>(1032.0f)};
    };
    auto high = [&](uint32_t v) {
        const wide_v2h h = __builtin_bit_cast(wide_v2h, (v & mhigh) | k1024);
        return __builtin_elementwise_fma(h, wide_v2h{static_cast<_Float16>(0.0625f), static_cast<_Float16>(0.0625f)},
                                         wide_v2h{static_cast<_Float16>(-72.0f), static_cast<_Float16>(-72.0f)});
    };
    const wide_v2h a = low(c), b = high(c), d = low(c8), e = high(c8);
    return wide_v8h{a.x, a.y, b.x, b.y, d.x, d.y, e.x, e.y};
}

// A token group's step in the unit: its products, the operand reads of the
// next group and the multiply-adds of the group before it (one matrix
// instruction, then the vector instructions that run beside it).  Left to
// itself the compiler waits out every product before its multiply-adds.
template <int N, int V>
__device__ __forceinline__ void interleave_steps() {
#pragma unroll
    for (int k = 0; k < N; ++k) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);    // matrix
        __builtin_amdgcn_sched_group_barrier(0x2, V, 0);    // vector
    }
    __builtin_amdgcn_sched_barrier(0);
}

// grid (row tiles of the jobs, token tiles).  A workgroup computes
// 64 RT rows (PAIR: 32 RT rows of gate and of up) x 16 TT tokens, wave w its
// rows 16 RT w ..: the unit's image of the workgroup's token groups is
// staged in LDS (two buffers, the next unit's loads in flight through the
// products, one barrier a unit), each wave's weights come straight from the
// MFMA-order copy into registers a unit ahead.
// KW > 1: KW such sets of four waves split the units, each with its own image
// buffers; their sums meet in LDS at the end, in the sets' order.
template <int KIND, int RT, int TT, int KW, bool PAIR>
__global__ __launch_bounds__(64 * kWideWaves * KW, KW < 4 ? 2 : 4) void wide_gemm_kernel(WideArgs a) {
    static_assert(!PAIR || RT % 2 == 0, "gate/up pairs: half of a wave's row groups each");
    constexpr int RO = PAIR ? RT / 2 : RT;   // row groups of output per wave
    constexpr uint32_t kStage = TT * kUnitImage;
    constexpr bool HV = KIND == kHvsq2;
    constexpr uint32_t kSet = 2 * TT * (kUnitImage + (HV ? 64u : 0u));   // LDS bytes of a set's buffers
    extern __shared__ __align__(16) uint8_t smem_all[];   // per set [2][TT][4096], HV: [2][TT][64] sums
    const uint32_t tid = threadIdx.x % (64 * kWideWaves), lane = tid % 64;
    const uint32_t set = __builtin_amdgcn_readfirstlane(threadIdx.x / (64 * kWideWaves));
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / 64);
    uint8_t *smem = smem_all + set * kSet;
    const uint32_t g = lane >> 4, m = lane & 15;
    const uint32_t b1 = a.job_block[1], b2 = a.job_block[2], b3 = a.job_block[3];
    const uint32_t bx = blockIdx.x;
    const uint32_t job =
        PAIR ? 0u
             : __builtin_amdgcn_readfirstlane((bx >= b1 ? 1u : 0u) + (bx >= b2 ? 1u : 0u) + (bx >= b3 ? 1u : 0u));
    const uint32_t first = job == 0 ? 0u : job == 1 ? b1 : job == 2 ? b2 : b3;
    const uint32_t rows = a.rows[job], stride = a.stride[job], units = a.units;
    const uint32_t rg0 = ((bx - first) * kWideWaves + wave) * RO, last_rg = (rows - 1) / 16;
    const uint32_t tok0 = blockIdx.y * 16 * TT, last_grp = (a.ntok - 1) / 16;
    // the set's units; every set runs the same number of barriers
    const uint32_t per = (units + KW - 1) / KW;
    const uint32_t u0 = min(units, set * per), u1 = min(units, u0 + per);

    // row groups past the matrix re-read the last one and store nothing
    const uint8_t *pb[RT], *mb[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) {
        const uint32_t j = PAIR ? (i < RO ? 0u : 1u) : job;
        const size_t rg = min(rg0 + (PAIR ? i % RO : i), last_rg);
        pb[i] = a.payload[j] + rg * units * 1024 + lane * 16;
        mb[i] = a.meta[j] + rg * units * 128 + m * 8;
    }
    const uint8_t *img[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t)
        img[t] = a.image + static_cast<size_t>(min(tok0 / 16 + t, last_grp)) * a.group_bytes;
    // HV: the activation sums of a unit, 64 bytes per group: threads t * 4 + i
    const uint8_t *sums = nullptr;
    if constexpr (HV)
        sums = a.image + static_cast<size_t>(min(tok0 / 16 + min(tid / 4, TT - 1u), last_grp)) * a.group_bytes +
               static_cast<size_t>(units) * kUnitImage + (tid % 4) * 16;

    wide_v4i stage[TT], ssum = {0, 0, 0, 0};
    auto load_stage = [&](uint32_t u) {
#pragma unroll
        for (int t = 0; t < TT; ++t) stage[t] = *reinterpret_cast<const wide_v4i *>(img[t] + u * kUnitImage + tid * 16);
        if constexpr (HV)
            if (tid < 4 * TT) ssum = *reinterpret_cast<const wide_v4i *>(sums + u * 64);
    };
    auto store_stage = [&](uint32_t buf) {
#pragma unroll
        for (int t = 0; t < TT; ++t)
            *reinterpret_cast<wide_v4i *>(smem + buf * kStage + t * kUnitImage + tid * 16) = stage[t];
        if constexpr (HV)
            if (tid < 4 * TT) *reinterpret_cast<wide_v4i *>(smem + 2 * kStage + buf * TT * 64 + tid * 16) = ssum;
    };
    uint4 wn[RT];
    uint2 mn[RT];
    auto load_weights = [&](uint32_t u) {
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            wn[i] = *reinterpret_cast<const uint4 *>(pb[i] + static_cast<size_t>(u) * 1024);
            mn[i] = *reinterpret_cast<const uint2 *>(mb[i] + static_cast<size_t>(u) * 128);
        }
    };

    uint32_t mlow = 0x000f000fu, mhigh = 0x00f000f0u, k1024 = 0x64006400u;
    asm("" : "+s"(mlow), "+s"(mhigh), "+v"(k1024));
    wide_v4f acc[RT][TT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int t = 0; t < TT; ++t) acc[i][t] = wide_v4f{0.0f, 0.0f, 0.0f, 0.0f};

    if (u0 < u1) {
        load_stage(u0);
        load_weights(u0);
        store_stage(0);
    }
    lds_barrier();
    for (uint32_t it = 0; it < per; ++it) {
        const uint32_t u = u0 + it, buf = it & 1u;
        if (KW > 1 && u >= u1) {
            lds_barrier();
            continue;
        }
        const uint8_t *tile = smem + buf * kStage + lane * 16;
        const uint32_t next = min(u + 1, u1 - 1);   // the last unit re-reads itself: no branch in the loop
        if constexpr (HV) {
            wide_v4i w[RT][4];
            float dsc[RT], msc[RT];
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                decode_hv(wn[i], (mn[i].y >> (8 * g)) & 0xffu, w[i]);
                dsc[i] = half_to_float(mn[i].x & 0xffffu) * 0.125f;
                msc[i] = half_to_float(mn[i].x >> 16);
                asm volatile("" : "+v"(msc[i]));   // fp32 once, not in every multiply-add
            }
            load_stage(next);
            load_weights(next);
            wide_v4i x[2][4], ci[2][RT];
            wide_v4f sa[2];
            auto scale = [&](int t) {
#pragma unroll
                for (int i = 0; i < RT; ++i) {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        acc[i][t][r] =
                            fmaf(static_cast<float>(ci[t & 1][i][r]), dsc[i], fmaf(msc[i], sa[t & 1][r], acc[i][t][r]));
                    asm volatile("" : "+v"(acc[i][t]));
                }
            };
#pragma unroll
            for (int q = 0; q < 4; ++q) x[0][q] = *reinterpret_cast<const wide_v4i *>(tile + q * 1024);
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                if (t + 1 < TT)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        x[(t + 1) & 1][q] = *reinterpret_cast<const wide_v4i *>(tile + (t + 1) * kUnitImage + q * 1024);
                sa[t & 1] = *reinterpret_cast<const wide_v4f *>(smem + 2 * kStage + (buf * TT + t) * 64 + g * 16);
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int i = 0; i < RT; ++i)
                        ci[t & 1][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                            x[t & 1][q], w[i][q], q ? ci[t & 1][i] : wide_v4i{0, 0, 0, 0}, 0, 0, 0);
                if (t > 0) scale(t - 1);
                interleave_steps<4 * RT, 3>();
            }
            scale(TT - 1);
        } else {
            wide_v8h w[RT][4];
            float d[RT][4];
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const uint32_t cw[4] = {wn[i].x, wn[i].y, wn[i].z, wn[i].w}, dw[2] = {mn[i].x, mn[i].y};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    w[i][q] = decode_q4(cw[q], mlow, mhigh, k1024);
                    d[i][q] = half_to_float((dw[q >> 1] >> (16 * (q & 1))) & 0xffffu);
                    asm volatile("" : "+v"(d[i][q]));   // fp32 once, not in every multiply-add
                }
            }
            load_stage(next);
            load_weights(next);
            wide_v8h x[2][4];
            wide_v4f ci[2][4][RT];
            auto scale = [&](int t) {
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int i = 0; i < RT; ++i)
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[i][t][r] = fmaf(ci[t & 1][q][i][r], d[i][q], acc[i][t][r]);
#pragma unroll
                for (int i = 0; i < RT; ++i) asm volatile("" : "+v"(acc[i][t]));
            };
#pragma unroll
            for (int q = 0; q < 4; ++q) x[0][q] = *reinterpret_cast<const wide_v8h *>(tile + q * 1024);
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                if (t + 1 < TT)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        x[(t + 1) & 1][q] = *reinterpret_cast<const wide_v8h *>(tile + (t + 1) * kUnitImage + q * 1024);
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int i = 0; i < RT; ++i)
                        ci[t & 1][q][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            x[t & 1][q], w[i][q], wide_v4f{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                if (t > 0) scale(t - 1);
                interleave_steps<4 * RT, 4>();
            }
            scale(TT - 1);
        }
        // the other buffer was read a unit ago, before the last barrier
        store_stage(buf ^ 1u);
        lds_barrier();
    }

    if constexpr (KW > 1) {
        // the last barrier is behind every set's reads: the buffers are free
        wide_v4f *part = reinterpret_cast<wide_v4f *>(smem_all) + static_cast<size_t>(wave * RT * TT) * 64 + lane;
        constexpr uint32_t kPart = kWideWaves * RT * TT * 64;
        if (set > 0)
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int t = 0; t < TT; ++t) part[(set - 1) * kPart + (i * TT + t) * 64] = acc[i][t];
        lds_barrier();
        if (set > 0) return;
#pragma unroll
        for (int k = 0; k < KW - 1; ++k)
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int t = 0; t < TT; ++t) acc[i][t] += part[k * kPart + (i * TT + t) * 64];
    }

    // lane (g, m) holds tokens 4g .. 4g + 3 of row m of each tile
    float *out = a.output[job] + static_cast<size_t>(tok0 + 4 * g) * stride + rg0 * 16 + m;
    const float *bias = PAIR ? nullptr : a.bias[job];
    const uint32_t row0 = rg0 * 16 + m, left = a.ntok - tok0 - min(4 * g, a.ntok - tok0);
    float bv[RO];
#pragma unroll
    for (int i = 0; i < RO; ++i) bv[i] = bias && row0 + 16 * i < rows ? bias[row0 + 16 * i] : 0.0f;
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        float xs[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) xs[r] = a.scales[min(tok0 + 16 * t + 4 * g + r, a.ntok - 1)];
#pragma unroll
        for (int i = 0; i < RO; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float *dst = out + static_cast<size_t>(16 * t + r) * stride + 16 * i;
                float v = mul_rounded(acc[i][t][r], xs[r]);
                if constexpr (PAIR) {
                    // silu(gate) * up, the arithmetic of the SwiGLU input transform
                    const float uv = mul_rounded(acc[RO + i][t][r], xs[r]);
                    v = mul_rounded(v / (1.0f + expf(-v)), uv);
                } else {
                    if (bias) v = add_rounded(v, bv[i]);
                }
                if (16u * t + r < left && row0 + 16 * i < rows) *dst = !PAIR && a.accumulate ? add_rounded(*dst, v) : v;
            }
    }
}

struct WidePlan {
    uint32_t rt = 0, kw = 1;      // row groups per wave, sets of waves splitting K
    uint32_t tt = kTokenGroups;   // 16-token groups per workgroup
};

template <int KIND, int RT, int TT, int KW, bool PAIR>
hipError_t launch_wide_one(const WideArgs &a, dim3 grid, hipStream_t stream) {
    constexpr size_t stage = KW * 2 * TT * (kUnitImage + (KIND == kHvsq2 ? 64u : 0u));
    constexpr size_t part = (KW - 1) * kWideWaves * RT * TT * 64 * sizeof(wide_v4f);
    constexpr size_t lds = stage > part ? stage : part;
    static_assert(lds <= kMfmaLdsLimit, "LDS of one workgroup");
    hipLaunchKernelGGL((wide_gemm_kernel<KIND, RT, TT, KW, PAIR>), grid, dim3(64 * kWideWaves * KW), lds, stream, a);
    return hipGetLastError();
}

template <int KIND>
hipError_t launch_wide_kind(const WideArgs &a, const WidePlan &p, bool pair, dim3 grid, hipStream_t stream) {
    if (pair) return launch_wide_one<KIND, 2, kTokenGroups, 1, true>(a, grid, stream);
    if (p.rt == 2) return launch_wide_one<KIND, 2, kTokenGroups, 1, false>(a, grid, stream);
    switch (p.kw) {
    case 1: return launch_wide_one<KIND, 1, kTokenGroups, 1, false>(a, grid, stream);
    case 2: return launch_wide_one<KIND, 1, kTokenGroups, 2, false>(a, grid, stream);
    default:
        if (p.tt == 1) return launch_wide_one<KIND, 1, 1, 4, false>(a, grid, stream);
        if (p.tt == 2) return launch_wide_one<KIND, 1, 2, 4, false>(a, grid, stream);
        return launch_wide_one<KIND, 1, kTokenGroups, 4, false>(a, grid, stream);
    }
}

// Two row groups a wave (each operand read feeds two products) where that
// leaves four workgroups a CU, and for the pairs; else one, and with fewer
// than four (than one) workgroups a CU two (four) sets splitting K.  1003
// tokens x 1536 x 8960 Q4_0 in us, groups x sets: 2x1 78, 2x2 67, 1x1 75,
// 1x2 67, 1x4 77; 333 x 2560 x 9728 HyperVSQ-2: 47, 41, 38, 31, 30 (four K
// splits added with float atomics: 55 and 37).  128-token tiles: 131 and 78,
// and no faster for the pairs (1003 tokens x 2 x 8960 x 1536: 99 against 97).
// Four sets in a half (a quarter) of the CUs or fewer: each unit is a round of
// vector instructions of all its waves, so tiles of 32 (16) tokens on twice
// (four times) the workgroups.  65 tokens x 1536 x 8960 Q4_0 as a host call's
// kernels, 64-, 32-, 16-token tiles: 38.6, 30.1, 26.0 us; 65 x 2560 x 9728:
// 41.2 and 31.4; a 65-token prompt of the 1.5B-shaped decoder 3.40, 2.94 and
// 2.71 ms (3.17 as a narrow block of 64 and one of 1).
WidePlan wide_plan(const DeviceTensor *const *tensors, uint32_t count, uint32_t batch, bool pair) {
    const uint32_t token_tiles = (batch + 16 * kTokenGroups - 1) / (16 * kTokenGroups);
    auto tiles = [&](uint32_t rt) {
        uint32_t n = 0;
        for (uint32_t i = 0; i < count; ++i) n += (tensors[i]->rows + 16 * rt * kWideWaves - 1) / (16 * rt * kWideWaves);
        return n * token_tiles;
    };
    WidePlan p;
    if (pair || tiles(2) >= 4 * kChipCus) {
        p.rt = 2;
        return p;
    }
    p.rt = 1;
    const uint32_t sets = tiles(1) <= kChipCus ? 4 : tiles(1) < 4 * kChipCus ? 2 : 1;
    while (p.kw < sets && tensors[0]->units >= 4 * p.kw) p.kw *= 2;
    if (p.kw == 4 && 2 * tiles(1) <= kChipCus) p.tt = 4 * tiles(1) <= kChipCus ? 1 : 2;
    return p;
}

}  // namespace

size_t wide_image_bytes(const DeviceTensor &t) {
    if (t.kind == kQ4_0) return static_cast<size_t>(t.units) * kUnitImage;
    return t.kind == kHvsq2 ? mfma_image_bytes(t) : 0;
}

bool wide_gemm_supported(const DeviceTensor &t) {
    return (t.kind == kHvsq2 || t.kind == kQ4_0) && t.mfma_payload && t.mfma_meta && t.rows > 0;
}

hipError_t launch_wide_gemm(const DeviceTensor *const *tensors, float *const *outputs, uint32_t count,
                            const uint8_t *image, const float *scales, uint32_t batch, const uint32_t *output_strides,
                            hipStream_t stream, bool accumulate, const float *const *biases, bool swiglu) {
    // a launch holds 65535 token tiles (grid y)
    if (count == 0 || count > static_cast<uint32_t>(kMaxGroup) || !image || !scales || batch == 0 ||
        batch > 65535u * 16 * kTokenGroups)
        return hipErrorInvalidValue;
    const DeviceTensor &t0 = *tensors[0];
    for (uint32_t i = 0; i < count; ++i) {
        const DeviceTensor &t = *tensors[i];
        if (!wide_gemm_supported(t) || t.kind != t0.kind || t.units != t0.units || t.cols != t0.cols || !outputs[i])
            return hipErrorInvalidValue;
    }
    if (swiglu && (count != 2 || accumulate || tensors[1]->rows != t0.rows || (biases && (biases[0] || biases[1]))))
        return hipErrorInvalidValue;
    const WidePlan p = wide_plan(tensors, count, batch, swiglu);
    WideArgs a{};
    uint32_t grid = 0;
    const uint32_t tile_rows = 16 * kWideWaves * (swiglu ? p.rt / 2 : p.rt);
    for (uint32_t i = 0; i < static_cast<uint32_t>(kMaxGroup); ++i) {
        a.job_block[i] = grid;
        if (i >= count) continue;
        const DeviceTensor &t = *tensors[i];
        a.payload[i] = t.mfma_payload;
        a.meta[i] = t.mfma_meta;
        a.output[i] = outputs[i];
        a.bias[i] = biases ? biases[i] : nullptr;
        a.rows[i] = t.rows;
        a.stride[i] = output_strides && output_strides[i] ? output_strides[i] : t.rows;
        if (!swiglu || i == 0) grid += (t.rows + tile_rows - 1) / tile_rows;
    }
    a.job_block[kMaxGroup] = grid;
    a.units = t0.units;
    a.image = image;
    a.group_bytes = static_cast<uint32_t>(wide_image_bytes(t0));
    a.scales = scales;
    a.ntok = batch;
    a.accumulate = accumulate ? 1u : 0u;
    const dim3 dims(grid, (batch + 16 * p.tt - 1) / (16 * p.tt));
    return t0.kind == kHvsq2 ? launch_wide_kind<kHvsq2>(a, p, swiglu, dims, stream)
                             : launch_wide_kind<kQ4_0>(a, p, swiglu, dims, stream);
}

}  // namespace qwn
