// The matrix-core products of libtensomite_hip.so: many activation rows
// against block-format weights, with the host's bits (Quant.matmul,
// quant.cr:155-491).
#include "tmh_device.h"
#include "tmh_internal.h"

namespace tmh {

namespace {

// x · wᵀ for many activation rows on the int8 matrix cores, for k a multiple
// of 256 and 16-byte aligned weights and activation parts. A wave computes
// tiles of 32 activation rows x 32 outputs over the whole of k: per block, one
// v_mfma_i32_32x32x32_i8 gives a tile's 1024 integer dot products of that block
// alone, exact (a lane holds 16 outputs: column lane % 32, rows 8 (i / 4) + 4
// (lane / 32) + i % 4), and every output adds the block's contribution, in the
// host's expression, to its running f32 sum in block order (the expressions of
// k_matmul_mfma). The factors those expressions take per output come from f16
// MFMAs over operands whose k slots other than one hold zeros: d·sx and m·mx
// (products of two halves, exact in f32 -- the host's products) for Q8_0 and
// Q4_1, and sx (times 1) for Q4_0, whose weights go in as 16 (q - 8): a nibble
// less 8 in a byte's upper half, so that the dot product is 16 t, and 16 t ·
// (d / 16) rounds as t · d does.
//
// What bounds it: per tile and block two or three MFMAs (36 cycles each) and a
// conversion, one or two multiplies and one or two adds per output, each
// rounded by itself. Measured on this machine, a SIMD issues such an
// instruction every 2.4 cycles with two waves or more to choose from and every
// 4.8 with one, and its matrix and vector instructions take turns: 185 cycles a
// Q8_0 tile and block at best. So every wave folds, four of them a SIMD (128 x 128)
// or two (64 x 128), and unpacks its own weights from the raw blocks in LDS (8 to 24
// instructions a block). The 32 x 32 tiles are for products that would leave the
// chip idle otherwise: their four waves, one a SIMD and so at half that rate,
// share a tile's fold and each repeat its MFMAs and unpacking. k_matmul_mx, whose
// compute units hold one folding wave a SIMD and one that repacks weights for it,
// remains for the sizes between.
//
// The k axis goes in stages of 8 blocks through a ring of LDS buffers, one
// workgroup barrier a stage, every byte brought by direct loads (16 bytes a
// lane): the weight rows' 8 blocks as they lie in memory, the activation rows'
// 256 int8 values and their scales (and Q4_1 sums), rows an odd number of
// 16-byte pieces apart, so that 16 rows' reads fall on distinct banks. A
// workgroup's tile comes from its id so that the activation tiles of one
// weight tile run on one XCD (ids go round-robin over the 8 XCDs): the weight
// tile comes from HBM once, into that XCD's L2.
//
// Measured (a call, quantise pass included): Q8_0 512 x 2048 -> 8192 60.0 ->
// 35.5 us, Q4_0 67.0 -> 39.2, Q4_0 100 x 2048 -> 16384 35.0 -> 24.7, 100 x 8192
// -> 2048 53.6 -> 34.7.
constexpr uint32_t MX_STAGE = 8;
constexpr uint32_t MX_ROW = 272;  // LDS bytes per activation row (256 + a 16-byte pad)

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));

template <int KIND>
constexpr uint32_t BLOCK_BYTES = KIND == 0 ? 34u : KIND == 1 ? 18u : 20u;

// WN x WM groups of FS waves, each group 32 outputs x 32·MS activation rows.
template <int KIND, int MS, int WN, int WM, int FS>
struct Mx {
    static constexpr uint32_t WAVES = WN * WM * FS, THREADS = 64u * WAVES;
    static constexpr uint32_t TN = 32u * WN, TM = 32u * MS * WM;  // the workgroup's outputs and rows
    // a weight row's bytes in a stage, and their distance in LDS: an odd number
    // of 16-byte pieces, so that 16 rows' reads of a piece fall on distinct banks
    static constexpr uint32_t RB = MX_STAGE * BLOCK_BYTES<KIND>, WROW = RB / 16u % 2u ? RB : RB + 16u;
    // a stage's buffer: weights [TN][WROW], activations [TM][MX_ROW], scales
    // [TM][8] f32, Q4_1 sums [TM][8] f32; each in whole loads of a kilobyte
    static constexpr uint32_t kilobytes(uint32_t bytes) { return (bytes + 1023u) / 1024u * 1024u; }
    static constexpr uint32_t AT_A = kilobytes(TN * WROW), AT_S = AT_A + kilobytes(TM * MX_ROW);
    static constexpr uint32_t AT_E = AT_S + TM * 32u, BYTES = AT_E + (KIND == 2 ? TM * 32u : 0u);
    static constexpr uint32_t LOADS = BYTES / 1024u;
    static constexpr uint32_t ROOM = 159u * 1024u / BYTES;
    static constexpr uint32_t BUFS = ROOM < 4u ? ROOM : 4u;
    static constexpr uint32_t ZERO = BUFS * BYTES;  // 32 zero bytes
    static constexpr uint32_t LDS = ZERO + 32u;
    static_assert(AT_A % 1024u == 0 && AT_S % 1024u == 0 && AT_E % 1024u == 0 && BYTES % 1024u == 0, "whole loads");
    static_assert(BUFS >= 2u && LDS <= 160u * 1024u, "one workgroup's LDS");
};

// An f16 MFMA operand with `half` (a half's bits, or 0) in its first k slot.
__device__ __forceinline__ v4h mx_op(uint32_t half) {
    const v2u v = {half, 0u};
    return __builtin_bit_cast(v4h, v);
}

// Whether f16 MFMAs form the contributions' factors: where a wave folds whole
// tiles (one MFMA, 36 cycles, for 16 multiplies, 38); a wave that folds a part
// of a tile reads and multiplies for that part alone.
template <int FS>
constexpr bool mx_factors = FS == 1;

__device__ __forceinline__ uint32_t mx_half_bits(float x) { return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)x); }

__device__ __forceinline__ void mx_eight(float (&v)[8], const float* p) {
    const float4 a = ((const float4*)p)[0], b = ((const float4*)p)[1];
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
}

// A weight operand: the lane's 16 values of a block (k slots 16·(lane / 32) ...),
// and its scale and minimum as f16 bits, zero in lanes 32-63 (whose slots of
// the f16 MFMAs must be); Q4_0's scale is no MFMA operand and stays in every
// lane.
struct MxWeight {
    v4i q;
    uint32_t d, m;
};

// A pair of blocks' raw bytes in 16-byte pieces, read aligned (a dword at a
// time, the 32 rows' reads would meet on a quarter of the banks): blocks 2p and
// 2p + 1 of a stage's row lie from dword 17p (Q8_0), 9p (Q4_0) or 10p (Q4_1)
// on. A Q8_0 lane takes the four pieces from 4p + lane / 32 on, which hold its
// halves of both blocks from dword p and p + 9 on (and, in lanes 0-31, the
// scales); a Q4 lane the pieces that hold the pair.
template <int KIND>
struct MxRaw {
    static constexpr uint32_t DW = 2u * BLOCK_BYTES<KIND> / 4u;  // dwords of a pair
    static constexpr uint32_t PIECES = 4u;
    uint32_t e[4u * PIECES];
    uint32_t d0, d1;  // Q8_0: the dwords that hold the pair's scales
};

template <int KIND>
__device__ __forceinline__ void mx_read(MxRaw<KIND>& o, const uint8_t* row, uint32_t p, uint32_t half) {
    using R = MxRaw<KIND>;
    const uint4* pieces = (const uint4*)row + (KIND == 0 ? 4u * p + half : R::DW * p / 4u);
    const uint32_t count = KIND == 0 ? 4u : (R::DW * (p + 1u) + 3u) / 4u - R::DW * p / 4u;
#pragma unroll
    for (uint32_t i = 0; i < R::PIECES; ++i) {
        if (i >= count) break;
        const uint4 v = pieces[i];
        o.e[4 * i] = v.x, o.e[4 * i + 1] = v.y, o.e[4 * i + 2] = v.z, o.e[4 * i + 3] = v.w;
    }
    if constexpr (KIND == 0) {
        const uint32_t* pair = (const uint32_t*)row + 17u * p;
        o.d0 = pair[0], o.d1 = pair[8];
    }
}

// The operands of blocks 2p and 2p + 1 from their raw bytes; `width` 16 in
// lanes 0-31, 0 in the others.
template <int KIND, bool FACTORS>
__device__ __forceinline__ void mx_weights(const MxRaw<KIND>& raw, uint32_t p, uint32_t half, uint32_t width,
                                           MxWeight& w0, MxWeight& w1) {
    using R = MxRaw<KIND>;
    const uint32_t* e = raw.e + (KIND == 0 ? p : R::DW * p % 4u);  // dword 0 of the pair (Q8_0: of the lane's half)
    if constexpr (KIND == 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            w0.q[i] = (int)__builtin_amdgcn_alignbit(e[i + 1], e[i], 16);
            w1.q[i] = (int)e[9 + i];
        }
        w0.d = __builtin_amdgcn_ubfe(e[0], 0, width);
        w1.d = __builtin_amdgcn_ubfe(e[8], 16, width);
        if constexpr (!FACTORS) w0.d = raw.d0 & 0xffffu, w1.d = raw.d1 >> 16;
    } else if constexpr (KIND == 1) {
        // lanes 0-31 the low nibbles, moved up, lanes 32-63 the high ones
        const uint32_t right = half ? 16u : 12u, left = half ? 0u : 4u;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            w0.q[i] = (int)((__builtin_amdgcn_alignbit(e[i + 1], e[i], right) & 0xf0f0f0f0u) ^ 0x80808080u);
            w1.q[i] = (int)(((e[5 + i] << left) & 0xf0f0f0f0u) ^ 0x80808080u);
        }
        w0.d = e[0] & 0xffffu;
        w1.d = e[4] >> 16;
    } else {
        const uint32_t right = half ? 4u : 0u;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            w0.q[i] = (int)((e[1 + i] >> right) & 0x0f0f0f0fu);
            w1.q[i] = (int)((e[6 + i] >> right) & 0x0f0f0f0fu);
        }
        const uint32_t bits = FACTORS ? width : 16u;
        w0.d = __builtin_amdgcn_ubfe(e[0], 0, bits);
        w0.m = __builtin_amdgcn_ubfe(e[0], 16, bits);
        w1.d = __builtin_amdgcn_ubfe(e[5], 0, bits);
        w1.m = __builtin_amdgcn_ubfe(e[5], 16, bits);
    }
}

// One block's dot products (Q4_0: 16 times them) and, where MFMAs give them,
// the factors of its contributions (f: d·sx, or Q4_0 sx; g: Q4_1 m·mx), exact.
struct MxBlock {
    v16i t;
    v16f f, g;
};

// `a`: the lane's 16 activation values; FACTORS: sx, mx its row's scale and sum
// of the block, one: 1 (f16 bits, zero in lanes 32-63).
template <int KIND, bool FACTORS>
__device__ __forceinline__ void mx_block(MxBlock& o, const v4i& a, const MxWeight& w, uint32_t sx, uint32_t mx,
                                         uint32_t one) {
    const v16i zi = {};
    const v16f zf = {};
    o.t = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, w.q, zi, 0, 0, 0);
    if constexpr (FACTORS) {
        o.f = __builtin_amdgcn_mfma_f32_32x32x8f16(mx_op(sx), mx_op(KIND == 1 ? one : w.d), zf, 0, 0, 0);
        if constexpr (KIND == 2) o.g = __builtin_amdgcn_mfma_f32_32x32x8f16(mx_op(mx), mx_op(w.m), zf, 0, 0, 0);
    }
}

// Adds one block's contributions to the E sums of results FIRST ..., from the
// column's scale d (Q4_0: a sixteenth of it) and, without FACTORS, its minimum m
// and the results' rows' scales sx and sums mx.
template <int KIND, bool FACTORS, int E, int FIRST>
__device__ __forceinline__ void mx_add(float (&acc)[E], const MxBlock& o, float d, float m, const float (&sx)[E],
                                       const float (&mx)[E]) {
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int i = FIRST + e;
        const float ft = (float)o.t[i];
        if constexpr (KIND == 1) {
            const float p = ft * d;
            acc[e] += p * (FACTORS ? o.f[i] : sx[e]);
        } else {
            const float f = FACTORS ? o.f[i] : d * sx[e];
            if constexpr (KIND == 0) {
                acc[e] += ft * f;
            } else {
                const float g = FACTORS ? o.g[i] : m * mx[e];
                const float c = f * ft;
                acc[e] += c + g;
            }
        }
    }
}

template <int KIND, int MS, int WN, int WM, int FS, int PART>
__device__ __forceinline__ void mx_product(uint8_t* lds, const uint8_t* __restrict__ w, const Activations& act,
                                           float* __restrict__ dst, const float* __restrict__ bias,
                                           uint32_t bias_ld, uint32_t m, uint32_t n, uint32_t k, uint32_t tiles_m, uint32_t tiles) {
    using M = Mx<KIND, MS, WN, WM, FS>;
    constexpr bool PIPE = M::WAVES < 16;  // four waves a SIMD hide an MFMA's latency by themselves
    constexpr bool FACTORS = mx_factors<FS>;
    constexpr int E = 16 / FS;  // results of a tile this wave folds, from FIRST on
    constexpr int FIRST = PART * E;
    const uint32_t t = threadIdx.x, lane = t & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t l32 = lane & 31u, half = lane >> 5;
    const uint32_t nb = k >> 5, stages = nb / MX_STAGE;
    uint32_t g = blockIdx.x;
    if (tiles % 8u == 0) g = (g & 7u) * (tiles >> 3) + (g >> 3);
    const uint32_t n0 = (g / tiles_m) * M::TN, m0 = (g % tiles_m) * M::TM;
    const uint32_t wn = wave % WN, wm = wave / WN % WM;
    const uint32_t row_bytes = nb * BLOCK_BYTES<KIND>;
    if (t < 8u) ((uint32_t*)(lds + M::ZERO))[t] = 0;

    // The wave's direct loads of a stage: of each array the kilobytes wave,
    // wave + WAVES, ...; lane l fills 16 bytes, from an offset of its own from
    // the tile's first row, which moves along the row with the stage. (A pad
    // piece of a row brings the row's last piece again.)
    constexpr uint32_t WK = M::AT_A / 1024u, AK = (M::AT_S - M::AT_A) / 1024u, SK = (M::AT_E - M::AT_S) / 1024u;
    constexpr uint32_t WJ = (WK + M::WAVES - 1u) / M::WAVES, AJ = (AK + M::WAVES - 1u) / M::WAVES;
    constexpr uint32_t SJ = (SK + M::WAVES - 1u) / M::WAVES;
    uint32_t woff[WJ], aoff[AJ], soff[SJ], mine = 0;
#pragma unroll
    for (uint32_t j = 0; j < WJ; ++j) {
        const uint32_t at = 1024u * (wave + M::WAVES * j) + 16u * lane, row = at / M::WROW;
        woff[j] = (min(n0 + row, n - 1u) - n0) * row_bytes + min(at % M::WROW, M::RB - 16u);
        mine += wave + M::WAVES * j < WK ? 1u : 0u;
    }
#pragma unroll
    for (uint32_t j = 0; j < AJ; ++j) {
        const uint32_t at = 1024u * (wave + M::WAVES * j) + 16u * lane, row = at / MX_ROW;
        aoff[j] = (min(m0 + row, m - 1u) - m0) * k + min(at % MX_ROW, 240u);
        mine += wave + M::WAVES * j < AK ? 1u : 0u;
    }
#pragma unroll
    for (uint32_t j = 0; j < SJ; ++j) {
        const uint32_t at = 1024u * (wave + M::WAVES * j) + 16u * lane, row = at / 32u;
        soff[j] = (min(m0 + row, m - 1u) - m0) * nb * 4u + (at & 16u);
        mine += wave + M::WAVES * j < SK ? (KIND == 2 ? 2u : 1u) : 0u;
    }
    const uint8_t* wb = w + (size_t)n0 * row_bytes;
    const uint8_t* ab = (const uint8_t*)act.qs + (size_t)m0 * k;
    const uint8_t* sb = (const uint8_t*)(act.scales + (size_t)m0 * nb);
    const uint8_t* eb = KIND == 2 ? (const uint8_t*)(act.sums + (size_t)m0 * nb) : sb;
    const uint32_t lds0 = lds_address(lds) + wave * 1024u;
    // the next stage's loads, into `buffer`
    auto issue = [&](uint32_t buffer) {
        const uint32_t to = lds0 + buffer * M::BYTES;
#pragma unroll
        for (uint32_t j = 0; j < WJ; ++j)
            if (wave + M::WAVES * j < WK) lds_load16_at(wb, woff[j], to + j * (M::WAVES * 1024u));
#pragma unroll
        for (uint32_t j = 0; j < AJ; ++j)
            if (wave + M::WAVES * j < AK) lds_load16_at(ab, aoff[j], to + M::AT_A + j * (M::WAVES * 1024u));
#pragma unroll
        for (uint32_t j = 0; j < SJ; ++j)
            if (wave + M::WAVES * j < SK) {
                lds_load16_at(sb, soff[j], to + M::AT_S + j * (M::WAVES * 1024u));
                if constexpr (KIND == 2) lds_load16_at(eb, soff[j], to + M::AT_E + j * (M::WAVES * 1024u));
            }
        wb += M::RB, ab += 256u, sb += 32u, eb += 32u;
    };

    float acc[MS][E];
#pragma unroll
    for (int i = 0; i < MS; ++i)
#pragma unroll
        for (int e = 0; e < E; ++e) acc[i][e] = 0.0f;
    constexpr uint32_t AHEAD = M::BUFS - 1u;
#pragma unroll
    for (uint32_t s = 0; s < AHEAD; ++s)
        if (s < stages) issue(s);

    const uint32_t width = half ? 0u : 16u, one = half ? 0u : 0x3c00u;  // f16 1 in lanes 0-31
    uint32_t buffer = 0;
    for (uint32_t s = 0; s < stages; ++s) {
        // This stage's loads have landed (those of the stages after it stay
        // in flight) in every wave, and every wave is done with the buffer
        // that the next loads fill.
        const uint32_t later = min(AHEAD - 1u, stages - 1u - s);
        asm volatile("" ::: "memory");
        wait_vm_lds_in<0u, 31u>(later * mine);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (s + AHEAD < stages) issue(buffer == 0 ? AHEAD : buffer - 1u);

        const uint8_t* b0 = lds + buffer * M::BYTES;
        const uint8_t* wrow = b0 + (32u * wn + l32) * M::WROW;
        const uint8_t* arow[MS];
        float sx[MS][8], mx[MS][8];  // FACTORS: the lane's row's
#pragma unroll
        for (int i = 0; i < MS; ++i) {
            const uint32_t row = (wm * MS + i) * 32u + l32;
            arow[i] = b0 + M::AT_A + row * MX_ROW + 16u * half;
            if constexpr (FACTORS) {
                mx_eight(sx[i], (const float*)(half ? lds + M::ZERO : b0 + M::AT_S + row * 32u));
                if constexpr (KIND == 2) mx_eight(mx[i], (const float*)(half ? lds + M::ZERO : b0 + M::AT_E + row * 32u));
            }
        }
        // Tile after tile of block after block; a block's MFMAs go out before
        // the additions of the one before it, its operands are read a pair of
        // blocks ahead.
        MxBlock cur, next;
        MxWeight wt[2];
        MxRaw<KIND> raw, raw_next;
        v4i a[MS][2], a_next[MS][2];
        float rs[MS][2][E], rm[MS][2][E], rs_next[MS][2][E], rm_next[MS][2][E];  // the results' rows' scales, sums
        float cd = 0.0f, cm = 0.0f, cs[E], ce[E];
        auto read = [&](uint32_t p, MxRaw<KIND>& to, v4i (&ta)[MS][2], float (&ts)[MS][2][E], float (&tm)[MS][2][E]) {
            mx_read<KIND>(to, wrow, p, half);
#pragma unroll
            for (int i = 0; i < MS; ++i) {
                ta[i][0] = *(const v4i*)(arow[i] + 64u * p);
                ta[i][1] = *(const v4i*)(arow[i] + 64u * p + 32u);
                if constexpr (!FACTORS) {
#pragma unroll
                    for (int e = 0; e < E; ++e) {
                        const int o = FIRST + e;
                        const uint32_t row = (wm * MS + i) * 32u + 8u * (o / 4) + 4u * half + (o % 4);
                        const float2 v = *(const float2*)(b0 + M::AT_S + row * 32u + 8u * p);
                        ts[i][0][e] = v.x, ts[i][1][e] = v.y;
                        if constexpr (KIND == 2) {
                            const float2 u = *(const float2*)(b0 + M::AT_E + row * 32u + 8u * p);
                            tm[i][0][e] = u.x, tm[i][1][e] = u.y;
                        }
                    }
                }
            }
        };
        auto add = [&](float (&to)[E]) { mx_add<KIND, FACTORS, E, FIRST>(to, cur, cd, cm, cs, ce); };
        if constexpr (PIPE) read(0, raw_next, a_next, rs_next, rm_next);
#pragma unroll
        for (uint32_t b = 0; b < MX_STAGE; ++b) {
            if (b % 2u == 0) {
                if constexpr (PIPE) {
                    raw = raw_next;
#pragma unroll
                    for (int i = 0; i < MS; ++i)
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            a[i][h] = a_next[i][h];
                            if constexpr (!FACTORS) {
#pragma unroll
                                for (int e = 0; e < E; ++e)
                                    rs[i][h][e] = rs_next[i][h][e], rm[i][h][e] = KIND == 2 ? rm_next[i][h][e] : 0.0f;
                            }
                        }
                    if (b + 2u < MX_STAGE) read(b / 2u + 1u, raw_next, a_next, rs_next, rm_next);
                } else {
                    read(b / 2u, raw, a, rs, rm);
                }
                mx_weights<KIND, FACTORS>(raw, b / 2u, half, width, wt[0], wt[1]);
            }
#pragma unroll
            for (int i = 0; i < MS; ++i) {
                const MxWeight& now = wt[b % 2u];
                mx_block<KIND, FACTORS>(next, a[i][b % 2u], now, FACTORS ? mx_half_bits(sx[i][b]) : 0u,
                                        FACTORS && KIND == 2 ? mx_half_bits(mx[i][b]) : 0u, one);
                if (PIPE && (b > 0 || i > 0)) add(acc[(i + MS - 1) % MS]);
                cur = next;
                if (KIND == 1) cd = half_value(now.d) * 0.0625f;
                if constexpr (!FACTORS) {
                    if (KIND != 1) cd = half_value(now.d);
                    cm = KIND == 2 ? half_value(now.m) : 0.0f;
#pragma unroll
                    for (int e = 0; e < E; ++e) cs[e] = rs[i][b % 2u][e], ce[e] = KIND == 2 ? rm[i][b % 2u][e] : 0.0f;
                }
                if (!PIPE) add(acc[i]);
            }
        }
        if (PIPE) add(acc[MS - 1]);
        // The stage's sums are complete before the barrier: the compiler
        // would otherwise move the additions after it.
#pragma unroll
        for (int i = 0; i < MS; ++i)
#pragma unroll
            for (int e = 0; e < E; ++e) asm volatile("" : "+v"(acc[i][e]));
        buffer = buffer + 1u == M::BUFS ? 0u : buffer + 1u;
    }

    const uint32_t col = n0 + 32u * wn + l32;
    if (col >= n) return;
#pragma unroll
    for (int i = 0; i < MS; ++i)
#pragma unroll
        for (int e = 0; e < E; e += 4)
            add_bias<4>(acc[i] + e, bias, bias_ld, m0 + (wm * MS + i) * 32u + 2u * (FIRST + e) + 4u * half, col, m, n);
#pragma unroll
    for (int i = 0; i < MS; ++i)
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int o = FIRST + e;
            const uint32_t row = m0 + (wm * MS + i) * 32u + 8u * (o / 4) + 4u * half + (o % 4);
            if (row < m) dst[(size_t)row * n + col] = acc[i][e];
        }
}

}  // namespace

// FS waves share a group's tiles: each issues all the MFMAs and folds its part
// of every tile's results (the parts as separate code: a wave's results are
// registers known at compile time).
#define TMH_MX_KERNEL(NAME, MS, WN, WM, FS)                                                                        \
    template <int KIND>                                                                                            \
    __global__ __launch_bounds__(64 * WN * WM * FS)                                                                \
        __attribute__((amdgpu_waves_per_eu(WN * WM * FS / 4, WN * WM * FS / 4))) void NAME(                        \
            const uint8_t* __restrict__ w, Activations act, float* __restrict__ dst,                               \
            const float* __restrict__ bias, uint32_t m, uint32_t n, uint32_t k, uint32_t tiles_m, uint32_t tiles,  \
            uint32_t bias_ld) {                                                                                    \
        __shared__ __attribute__((aligned(16))) uint8_t lds[Mx<KIND, MS, WN, WM, FS>::LDS];                        \
        const uint32_t part = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) / (WN * WM);                        \
        if (FS == 1 || part == 0)                                                                                  \
            mx_product<KIND, MS, WN, WM, FS, 0>(lds, w, act, dst, bias, bias_ld, m, n, k, tiles_m, tiles);                  \
        else if (part == 1)                                                                                        \
            mx_product<KIND, MS, WN, WM, FS, 1 % FS>(lds, w, act, dst, bias, bias_ld, m, n, k, tiles_m, tiles);             \
        else if (part == 2)                                                                                        \
            mx_product<KIND, MS, WN, WM, FS, 2 % FS>(lds, w, act, dst, bias, bias_ld, m, n, k, tiles_m, tiles);             \
        else                                                                                                       \
            mx_product<KIND, MS, WN, WM, FS, 3 % FS>(lds, w, act, dst, bias, bias_ld, m, n, k, tiles_m, tiles);             \
    }
TMH_MX_KERNEL(k_matmul_128x128, 1, 4, 4, 1)  // rows x outputs of a workgroup
TMH_MX_KERNEL(k_matmul_64x128, 1, 4, 2, 1)
TMH_MX_KERNEL(k_matmul_32x32, 1, 1, 1, 4)
#undef TMH_MX_KERNEL

// Which kernel: the one whose rounds of workgroups (one a compute unit) take
// least, by the time of a round of each as measured at k = 2048 (us: 31 of
// 128 x 128, 19.5 of 64 x 128, 13 of k_matmul_mx's 64 x 64, 7.5 of 32 x 32; in
// proportion to k). The 64 x 64 tiles win where they fill at most one round that
// the 32 x 32 ones overflow: Q8_0 512 x 2048 -> 2048 18.2 us against 24.8 in
// tiles of 64 x 128 and 41.7 in tiles of 32 x 32.
MxTile mx_tile(uint32_t rows, uint32_t n, int compute_units) {
    struct {
        uint32_t tm, tn, cost;
        MxTile tile;
    } const choices[] = {{32, 32, 15, MX_32X32}, {64, 64, 26, MX_64X64}, {64, 128, 39, MX_64X128}, {128, 128, 62, MX_128X128}};
    MxTile best = MX_64X64;
    uint64_t least = ~0ull;
    for (const auto& c : choices) {
        const uint64_t tiles = (uint64_t)((rows + c.tm - 1u) / c.tm) * ((n + c.tn - 1u) / c.tn);
        const uint64_t cost = (tiles + compute_units - 1u) / compute_units * c.cost;
        if (cost < least) least = cost, best = c.tile;
    }
    return best;
}

template <int KIND>
static hipError_t launch_tiles(MxTile tile, const uint8_t* w, Activations act, float* dst, const float* bias,
                               uint32_t bias_ld, uint32_t rows, uint32_t n, uint32_t k, hipStream_t stream) {
    const uint32_t tm = tile == MX_128X128 ? 128u : tile == MX_64X128 ? 64u : 32u, tn = tile == MX_32X32 ? 32u : 128u;
    const uint32_t tiles_m = (rows + tm - 1u) / tm, tiles = tiles_m * ((n + tn - 1u) / tn);
    if (tile == MX_128X128)
        TMH_LAUNCH(k_matmul_128x128<KIND>, dim3(tiles), dim3(1024), 0, stream, w, act, dst, bias, rows, n, k, tiles_m,
                   tiles, bias_ld);
    else if (tile == MX_64X128)
        TMH_LAUNCH(k_matmul_64x128<KIND>, dim3(tiles), dim3(512), 0, stream, w, act, dst, bias, rows, n, k, tiles_m,
                   tiles, bias_ld);
    else
        TMH_LAUNCH(k_matmul_32x32<KIND>, dim3(tiles), dim3(256), 0, stream, w, act, dst, bias, rows, n, k, tiles_m,
                   tiles, bias_ld);
    return hipGetLastError();
}

hipError_t launch_matmul_tiles(uint32_t kind, MxTile tile, const uint8_t* w, Activations act, float* dst,
                               const float* bias, uint32_t bias_ld, uint32_t rows, uint32_t n, uint32_t k,
                               hipStream_t stream) {
    switch (kind) {
    case 0: return launch_tiles<0>(tile, w, act, dst, bias, bias_ld, rows, n, k, stream);
    case 1: return launch_tiles<1>(tile, w, act, dst, bias, bias_ld, rows, n, k, stream);
    default: return launch_tiles<2>(tile, w, act, dst, bias, bias_ld, rows, n, k, stream);
    }
}

}  // namespace tmh
