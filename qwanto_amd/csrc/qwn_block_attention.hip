// Causal attention of a block of query tokens (prefill, verify, draft trees)
// over the Q8 KV cache, on the int8 matrix cores.
//
// Numerics are the decode attention's (c/qwanto_turboquant.c:555-702 per
// query head): scores and P.V as exact int8 products of three-piece splits
// of the fp32 query and probabilities (|x - sum| <= amax * 6e-8), softmax in
// fp32.  What differs is the shape of the work: the rows of a matrix tile
// are sixteen (token, query head) pairs of one KV head, so a tile's keys and
// values are read once for all of them, and each piece is an MFMA of its own
// with all sixteen rows used (the one-token kernel gives a head four rows,
// three of them pieces).
#include "qwn_device.h"
#include "qwn_internal.h"
#include "qwn_kv.h"

#include <algorithm>

namespace qwn {
namespace {

constexpr int kWaves = 4;       // waves per workgroup, each taking every fourth 64-token block
constexpr int kRows = 16;       // (token, head) rows per workgroup
constexpr float kTinyMax = 0x1p-100f, kLift = 0x1p80f;   // maxima below are lifted before their split
constexpr int kPieceRow = 80;   // LDS bytes between the rows of a piece tile: 64 tokens + 16 (bank spread)

struct BlockAttnArgs {
    KvCache c;
    const float *query;           // [count][heads][D]
    float *output;                // [count][heads][D] (nsplit == 1)
    float *partials;              // [count * heads][nsplit][D + 2] (nsplit > 1)
    const int32_t *position_ptr;  // [count] cache slot of each query token
    uint32_t heads, group, count, nsplit;
    float scale;
    const uint64_t *tree_mask;    // optional [count] ancestor masks over slots *tree_base + a
    const int32_t *tree_base;
};

// x as the byte 0 of 1.5 * 2^23 + rint(x inv): the rounded value is exact in
// fp32 (|x inv| <= 127.5), and subtracting the constant gives it back.
__device__ __forceinline__ float round_magic(float x, float inv) { return fmaf(x, inv, 12582912.0f); }

// The three int8 pieces of x (scale s1 = amax / 127, inv1 = 1 / s1), each in
// the low byte of its word: x ~= s1 (p0 + p1 / 254 + p2 / 64516), every
// residual exact by fma, so no piece passes +-127 and nothing is clamped.
// amax >= kTinyMax (64516 / s1 stays finite); smaller ones are lifted first.
__device__ __forceinline__ void split_pieces(float x, float s1, float inv1, uint32_t (&p)[3]) {
    const float y0 = round_magic(x, inv1);
    const float r0 = fmaf(-(y0 - 12582912.0f), s1, x);
    const float y1 = round_magic(r0, inv1 * 254.0f);
    const float r1 = fmaf(-(y1 - 12582912.0f), s1 * (1.0f / 254.0f), r0);
    const float y2 = round_magic(r1, inv1 * 64516.0f);
    p[0] = __builtin_bit_cast(uint32_t, y0);
    p[1] = __builtin_bit_cast(uint32_t, y1);
    p[2] = __builtin_bit_cast(uint32_t, y2);
}

// p0 + p1 / 254 + p2 / 64516 of three int32 dots: the two low ones meet in
// the integers (|254 c1 + c2| < 2^28), one conversion less
__device__ __forceinline__ float pieces_value(int c0, int c1, int c2) {
    return fmaf(static_cast<float>(__mul24(c1, 254) + c2), 1.0f / 64516.0f, static_cast<float>(c0));
}

// grid (row tiles, kv heads, nsplit).  A workgroup takes sixteen rows of one
// KV head over its split of their context; its waves take 64-token blocks in
// turn, each with its own online softmax, and merge through LDS.  A block's
// values are loaded once its scores are formed and the next block's keys
// then take the keys' registers: both are in flight through the softmax (at
// head_dim 256 a block does not fit the registers beside the outputs: its
// keys are loaded tile by tile and its values group by group at their use).
// Bound by the vector ALU (about a thousand instructions per 16 rows x 64
// tokens, most of them the probabilities' pieces) and, where a wave has one
// block only, by its latency.  64 tokens of 12 heads over up to 1003 tokens
// (head_dim 128, 2 KV heads): 12.4 us a launch.
template <int D, bool TREE>
__global__ __launch_bounds__(64 * kWaves, D <= 128 ? 2 : 1) void block_attention_kernel(BlockAttnArgs a) {
    constexpr int NG = D / 64;   // scale groups per head = MFMA k-steps of the scores
    constexpr int NT = 4;        // 16-token tiles per block
    constexpr bool kAhead = D <= 128;   // keys and values of the next block loaded ahead
    constexpr int kPieces = NG * 3 * kRows * kPieceRow;   // a wave's piece tiles
    // the waves' piece tiles, later their partial outputs [wave][row][D]
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ float ml_s[kWaves][kRows][2];
    __shared__ uint32_t lim_s[kRows];
    const KvCache &c = a.c;
    const uint32_t tid = threadIdx.x, lane = tid % 64;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const uint32_t col = lane % 16, kq = lane / 16;
    const uint32_t kvh = blockIdx.y, G = a.group, rows = a.count * G;
    // the last tiles attend to the most tokens: they go first
    const uint32_t row0 = (gridDim.x - 1 - blockIdx.x) * kRows;

    // 1. This lane's query row (row col of the tile, the A operand) and how
    //    many tokens it attends to (0: no such row, or a slot past the cache).
    const uint32_t arow = row0 + col < rows ? row0 + col : 0u;
    const uint32_t atok = arow / G, ahead = kvh * G + arow % G;
    const uint32_t apos = static_cast<uint32_t>(a.position_ptr[atok]);
    const float *qrow = a.query + (static_cast<size_t>(atok) * a.heads + ahead) * D + 16 * kq;
    float4 qv[NG][4];
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int i = 0; i < 4; ++i) qv[g][i] = *reinterpret_cast<const float4 *>(qrow + 64 * g + 4 * i);
    uint32_t tm_lo = 0, tm_hi = 0, tbase = 0;
    if constexpr (TREE) {
        const uint64_t m = a.tree_mask[atok];
        tm_lo = static_cast<uint32_t>(m);
        tm_hi = static_cast<uint32_t>(m >> 32);
        tbase = static_cast<uint32_t>(*a.tree_base);
    }
    const uint32_t alim = row0 + col < rows && apos < c.max_tokens ? apos + 1u : 0u;
    uint32_t most = alim;
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) most = max(most, static_cast<uint32_t>(__shfl_xor(static_cast<int>(most), off)));
    const uint32_t tokens = __builtin_amdgcn_readfirstlane(most);
    // the split's tokens [t0, t1): whole 64-token blocks, at least one per wave
    const uint32_t per = a.nsplit == 1 ? tokens
                                       : max(64u * kWaves, ((tokens + a.nsplit - 1) / a.nsplit + 63u) & ~63u);
    const uint32_t t0 = min(tokens, blockIdx.z * per), t1 = min(tokens, t0 + per);

    // 2. Loads of a block: keys (B of the scores) of token b0 + 16i + col,
    //    channels 64g + 16kq: page b0/16 + i, a wave-uniform address plus a
    //    fixed lane offset; values (B of P.V) of page b0/16 + kq, channel
    //    64g + 16n + col.  Pages past the cache's last one re-read that one;
    //    the tokens past a row's last are masked.
    constexpr uint32_t kPage = D * kKvPageTokens;   // bytes of a page of one head (keys, and values)
    const int8_t *kbase = c.keys + static_cast<size_t>(kvh) * c.pages * kPage;
    const int8_t *vbase = c.values + static_cast<size_t>(kvh) * c.pages * kPage;
    const float *ksbase = c.key_scales + static_cast<size_t>(kvh) * NG * c.quads * 64;
    const float *vsbase = c.value_scales + static_cast<size_t>(kvh) * NG * c.quads * 64;
    const uint32_t koff = kq * 256 + col * 16;
    att_v4i kb[NG][NT], vb[NG][4];
    float4 ks[NG], vs[NG];
    auto load_key_tile = [&](uint32_t b0, int i) {
        const int8_t *pg = kbase + static_cast<size_t>(min(b0 / kKvPageTokens + i, c.pages - 1)) * kPage;
#pragma unroll
        for (int g = 0; g < NG; ++g) kb[g][i] = *reinterpret_cast<const att_v4i *>(pg + koff + g * 1024);
    };
    auto load_keys = [&](uint32_t b0) {
        if constexpr (kAhead)
#pragma unroll
            for (int i = 0; i < NT; ++i) load_key_tile(b0, i);
        const float *sc = ksbase + b0 + 4 * col;   // b0 tokens start quad b0 / 64, 64 floats each
#pragma unroll
        for (int g = 0; g < NG; ++g) ks[g] = *reinterpret_cast<const float4 *>(sc + static_cast<size_t>(g) * c.quads * 64);
    };
    auto load_value_group = [&](uint32_t b0, int g) {
        // 64-bit to the block's first page: a head's values pass 2^32 bytes at 16 M tokens of head_dim 256
        const uint32_t page = b0 / kKvPageTokens;
        const int8_t *pg = vbase + static_cast<size_t>(page) * kPage;
        const uint32_t off = min(kq, c.pages - 1 - page) * kPage + col * 16;
#pragma unroll
        for (int n = 0; n < 4; ++n) vb[g][n] = *reinterpret_cast<const att_v4i *>(pg + (off + g * 1024 + n * 256));
    };
    auto load_values = [&](uint32_t b0) {
        const float *sc = vsbase + b0 + 4 * col;
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            vs[g] = *reinterpret_cast<const float4 *>(sc + static_cast<size_t>(g) * c.quads * 64);
            if constexpr (kAhead) load_value_group(b0, g);
        }
    };
    constexpr uint32_t step = 64 * kWaves;
    uint32_t b0 = t0 + 64 * wave;
    if (b0 < t1) load_keys(b0);

    // 3. The query pieces, per 64-channel group; a non-finite query gives a
    //    NaN scale, and so NaN scores, for its row.
    att_v4i qa[3][NG];
    float qs[NG][4];   // scale of row 4kq + r (the C layout's rows of this lane)
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        float amax = 0.0f, bad = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float x = fabsf(f4_at(qv[g][i], e));
                bad = x < INFINITY ? bad : 1.0f;
                amax = fmaxf(amax, x);
            }
        amax = fmaxf(amax, __shfl_xor(amax, 16));
        amax = fmaxf(amax, __shfl_xor(amax, 32));
        bad = fmaxf(bad, __shfl_xor(bad, 16));
        bad = fmaxf(bad, __shfl_xor(bad, 32));
        // a maximum below 2^-100 would overflow its reciprocal's multiples:
        // such a row is split after an exact lift
        const float lift = amax < kTinyMax ? kLift : 1.0f;
        amax *= lift;
        const bool live = amax > 0.0f && bad == 0.0f;
        const float s1 = live ? amax * (1.0f / 127.0f) : 0.0f, inv1 = live ? 127.0f / amax : 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t p[4][3];
#pragma unroll
            for (int e = 0; e < 4; ++e) split_pieces(live ? f4_at(qv[g][i], e) * lift : 0.0f, s1, inv1, p[e]);
#pragma unroll
            for (int j = 0; j < 3; ++j)
                qa[j][g][i] = static_cast<int>(pack_low_bytes(p[0][j], p[1][j], p[2][j], p[3][j]));
            __builtin_amdgcn_sched_barrier(0);
        }
        const float sq = bad > 0.0f ? __builtin_nanf("") : lift == 1.0f ? s1 : s1 * (1.0f / kLift);
#pragma unroll
        for (int r = 0; r < 4; ++r) qs[g][r] = __shfl(sq, 4 * kq + r);
    }
    uint32_t lim[4], mlo[4], mhi[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        lim[r] = static_cast<uint32_t>(__shfl(static_cast<int>(alim), 4 * kq + r));
        if constexpr (TREE) {
            mlo[r] = static_cast<uint32_t>(__shfl(static_cast<int>(tm_lo), 4 * kq + r));
            mhi[r] = static_cast<uint32_t>(__shfl(static_cast<int>(tm_hi), 4 * kq + r));
        }
    }
    if (wave == 0 && kq == 0) lim_s[col] = alim;

    float m_run[4], l_run[4], o_acc[NG][4][4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        m_run[r] = -INFINITY;
        l_run[r] = 0.0f;
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int n = 0; n < 4; ++n) o_acc[g][n][r] = 0.0f;
    }
    uint8_t *pp = smem + wave * kPieces;

    for (; b0 < t1; b0 += step) {
        // 4. Scores of rows 4kq + r for token b0 + 16i + col.
        float sc[NT][4];
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            if constexpr (!kAhead) load_key_tile(b0, i);
            float dot[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                att_v4i cp[3];
#pragma unroll
                for (int j = 0; j < 3; ++j)
                    cp[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(qa[j][g], kb[g][i], att_v4i{0, 0, 0, 0}, 0, 0, 0);
                const float kt = f4_at(ks[g], i);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    dot[r] = fmaf(pieces_value(cp[0][r], cp[1][r], cp[2][r]), qs[g][r] * kt, dot[r]);
            }
            const uint32_t t = b0 + 16 * i + col;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                bool valid = t < lim[r];
                if constexpr (TREE)
                    valid = valid && tree_attends(t, tbase, (static_cast<uint64_t>(mhi[r]) << 32) | mlo[r]);
                sc[i][r] = valid ? dot[r] * a.scale : -INFINITY;
                asm volatile("" : "+v"(sc[i][r]));   // formed here: one tile's products live at a time
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        load_values(b0);
        const uint32_t nb = b0 + step;
        if (nb < t1) load_keys(nb);
        __builtin_amdgcn_sched_barrier(0);
        // 5. Online softmax per row (a row's tokens lie in 16 lanes); p' = p
        //    times the value scale of each group, split into pieces -> LDS.
        float alpha[4], ps1[NG][4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float cm = row16_max(fmaxf(fmaxf(sc[0][r], sc[1][r]), fmaxf(sc[2][r], sc[3][r])));
            const float mn = fmaxf(m_run[r], cm);
            alpha[r] = m_run[r] == -INFINITY ? 0.0f : expf(m_run[r] - mn);
            m_run[r] = mn;
            float p[NT], sum = 0.0f;
#pragma unroll
            for (int i = 0; i < NT; ++i) {
                p[i] = sc[i][r] == -INFINITY ? 0.0f : expf(sc[i][r] - mn);
                sum += p[i];
            }
            l_run[r] = fmaf(l_run[r], alpha[r], row16_sum(sum));
            float pv[NG][NT], am[NG];
            uint32_t least = 0xffffffffu;   // of the maxima above 0, as bits less one
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                am[g] = 0.0f;
#pragma unroll
                for (int i = 0; i < NT; ++i) {
                    // masked tokens' scales may be any bits
                    pv[g][i] = p[i] == 0.0f ? 0.0f : p[i] * f4_at(vs[g], i);
                    am[g] = fmaxf(am[g], pv[g][i]);
                }
                am[g] = row16_max(am[g]);
                least = min(least, __builtin_bit_cast(uint32_t, am[g]) - 1u);
                ps1[g][r] = 1.0f / 127.0f;
            }
            // rare (a block far below its row's maximum, or values that
            // small): one test for the wave
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(least < __builtin_bit_cast(uint32_t, kTinyMax) - 1u) != 0, 0)) {
#pragma unroll
                for (int g = 0; g < NG; ++g) {
                    const float lift = am[g] < kTinyMax ? kLift : 1.0f;
                    ps1[g][r] *= 1.0f / lift;
                    am[g] *= lift;
#pragma unroll
                    for (int i = 0; i < NT; ++i) pv[g][i] *= lift;
                }
            }
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                const float s1 = am[g] * (1.0f / 127.0f), inv1 = am[g] > 0.0f ? 127.0f / am[g] : 0.0f;
                ps1[g][r] *= am[g];
#pragma unroll
                for (int i = 0; i < NT; ++i) {
                    uint32_t q[3];
                    split_pieces(pv[g][i], s1, inv1, q);
                    uint8_t *dst = pp + (g * 3 * kRows + 4 * kq + r) * kPieceRow + 16 * i + col;
#pragma unroll
                    for (int j = 0; j < 3; ++j) dst[j * kRows * kPieceRow] = static_cast<uint8_t>(q[j]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        lds_wave_sync();
        // 6. P.V: A lane = row col, tokens 16kq .. +15; C rows 4kq + r,
        //    channel 64g + 16n + col.
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            if constexpr (!kAhead) load_value_group(b0, g);
            att_v4i pa[3];
#pragma unroll
            for (int j = 0; j < 3; ++j)
                pa[j] = *reinterpret_cast<const att_v4i *>(pp + ((g * 3 + j) * kRows + col) * kPieceRow + 16 * kq);
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                att_v4i cp[3];
#pragma unroll
                for (int j = 0; j < 3; ++j)
                    cp[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(pa[j], vb[g][n], att_v4i{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    o_acc[g][n][r] = fmaf(pieces_value(cp[0][r], cp[1][r], cp[2][r]), ps1[g][r], o_acc[g][n][r] * alpha[r]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        lds_wave_sync();   // the piece tiles are read: the next block overwrites them
    }

    // 7. Merge the waves: their partial outputs take the piece tiles' place.
    __syncthreads();
    float *o_s = reinterpret_cast<float *>(smem);   // [kWaves][kRows][D]
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (col == 0) {
            ml_s[wave][4 * kq + r][0] = m_run[r];
            ml_s[wave][4 * kq + r][1] = l_run[r];
        }
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int n = 0; n < 4; ++n) o_s[(wave * kRows + 4 * kq + r) * D + 64 * g + 16 * n + col] = o_acc[g][n][r];
    }
    __syncthreads();
    for (uint32_t i = tid; i < kRows * D; i += blockDim.x) {
        const uint32_t row = i / D, d = i % D;
        if (lim_s[row] == 0) continue;
        float mx = -INFINITY;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) mx = fmaxf(mx, ml_s[w][row][0]);
        float l = 0.0f, o = 0.0f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const float m = ml_s[w][row][0], f = m == -INFINITY ? 0.0f : expf(m - mx);
            l = fmaf(ml_s[w][row][1], f, l);
            o = fmaf(o_s[(w * kRows + row) * D + d], f, o);
        }
        const uint32_t grow = row0 + row;
        const size_t out = static_cast<size_t>(grow / G) * a.heads + kvh * G + grow % G;   // [token][head]
        if (a.nsplit == 1) {
            a.output[out * D + d] = o / l;
        } else {
            float *dst = a.partials + (out * a.nsplit + blockIdx.z) * (D + 2);
            dst[2 + d] = o;
            if (d == 0) {
                dst[0] = mx;
                dst[1] = l;
            }
        }
    }
}

template <int D>
hipError_t launch_block(const BlockAttnArgs &a, dim3 grid, hipStream_t stream) {
    constexpr size_t pieces = kWaves * (D / 64) * 3 * kRows * kPieceRow, outs = kWaves * kRows * D * sizeof(float);
    constexpr size_t lds = pieces > outs ? pieces : outs;
    if (a.tree_mask)
        hipLaunchKernelGGL((block_attention_kernel<D, true>), grid, dim3(64 * kWaves), lds, stream, a);
    else
        hipLaunchKernelGGL((block_attention_kernel<D, false>), grid, dim3(64 * kWaves), lds, stream, a);
    return hipGetLastError();
}

// Splits of the context: one where the row tiles fill the chip, else enough
// for a workgroup per CU while each split keeps 512 tokens or more (two
// blocks per wave: a shorter split costs more in the merge than it saves).
uint32_t block_splits(const KvCache &c, uint32_t query_heads, uint32_t count, uint32_t span) {
    const uint32_t tiles = (count * (query_heads / c.kv_heads) + kRows - 1) / kRows * c.kv_heads;
    return std::max(1u, std::min(kChipCus / tiles, span / 512u));
}

}  // namespace

bool block_attention_supported(const KvCache &c, uint32_t query_heads) {
    return (c.head_dim == 64 || c.head_dim == 128 || c.head_dim == 256) && query_heads >= c.kv_heads &&
           query_heads % c.kv_heads == 0;
}

size_t block_attention_workspace_floats(const KvCache &c, uint32_t query_heads, uint32_t count, uint32_t span) {
    const uint32_t n = block_splits(c, query_heads, count, span);
    return n > 1 ? static_cast<size_t>(count) * query_heads * n * (c.head_dim + 2) : 0;
}

hipError_t launch_block_attention(const BlockAttentionLaunch &l, hipStream_t stream) {
    const KvCache &c = *l.cache;
    if (!block_attention_supported(c, l.query_heads) || l.count == 0 || !l.position_ptr || l.span == 0 ||
        l.span > c.max_tokens || (!l.tree_mask) != (!l.tree_base))
        return hipErrorInvalidValue;
    BlockAttnArgs a{};
    a.c = c;
    a.query = l.query;
    a.output = l.output;
    a.partials = l.partials;
    a.position_ptr = l.position_ptr;
    a.heads = l.query_heads;
    a.group = l.query_heads / c.kv_heads;
    a.count = l.count;
    a.nsplit = block_splits(c, l.query_heads, l.count, l.span);
    a.scale = l.scale;
    a.tree_mask = l.tree_mask;
    a.tree_base = l.tree_base;
    if (a.nsplit > 1 && !l.partials) return hipErrorInvalidValue;
    const dim3 grid((l.count * a.group + kRows - 1) / kRows, c.kv_heads, a.nsplit);
    hipError_t e;
    switch (c.head_dim) {
    case 64: e = launch_block<64>(a, grid, stream); break;
    case 128: e = launch_block<128>(a, grid, stream); break;
    default: e = launch_block<256>(a, grid, stream); break;
    }
    if (e != hipSuccess || a.nsplit == 1) return e;
    return launch_attention_merge(l.partials, l.output, l.count * l.query_heads, a.nsplit, c.head_dim, stream);
}

}  // namespace qwn
