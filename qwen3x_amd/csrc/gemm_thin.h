// gemm_thin.h -- FP32 GEMM for a few A rows: Y[m, n] as gemm_x3.h forms it
// (exact bf16 products of the three-way split activations, FP32 sums, the
// block scale by FMA), for tiles of at most 32 A rows.
#pragma once

#include "gemm_x3.h"
#include "matvec.h"

namespace q3x {

// A unit of weights: 16 consecutive rows of one K segment of BLOCKS blocks,
// held as 144 bytes a row (Q8_0: 4 blocks are 136 bytes and the load takes 8
// more; Q4_0: 8 blocks).  2304 bytes: two 16-byte loads a lane and one of 4.
template <uint32_t QT>
struct SegUnit {
    static constexpr bool kQ4 = QT == Q3X_HIP_MATRIX_Q4_0;
    static constexpr int BB = kQ4 ? kQ4Bytes : kQ8Bytes;
    static constexpr int BLOCKS = kQ4 ? 8 : 4;
    static constexpr int STEP = BLOCKS * BB;  // bytes from a segment to the row's next
    static constexpr int PITCH = 144;
    static constexpr int BYTES = 16 * PITCH;
    static constexpr int WIDE = BYTES / 1024;
    static_assert(BYTES == WIDE * 1024 + 256 && STEP <= PITCH, "two 16-byte loads a lane and one of 4 bytes");
};

struct SegRegs {
    u32x4 wide[2];
    uint32_t rest;
};

// This lane's bf16 operand of block kb of a unit in LDS -- weight row l16,
// the eight values of chunk g16 -- and the row's block scale.  Q8_0: elements
// 8 g16 + [0, 8).  Q4_0: elements 4 g16 + [0, 4) and 16 + 4 g16 + [0, 4), as
// 16 (n - 8) with the scale d / 16 (BlockPart::values).
template <uint32_t QT>
__device__ __forceinline__ bf16x8 seg_operand(const uint8_t* unit, int l16, int g16, int kb, float& d) {
    using U = SegUnit<QT>;
    const uint8_t* blk = unit + l16 * U::PITCH + kb * U::BB;
    const uint32_t half = *reinterpret_cast<const uint16_t*>(blk);
    d = U::kQ4 ? f16_fast(half) * 0.0625f : f16_fast(half);
    asm("" : "+v"(d));  // an FP32 value: v_fma_f32 issues at twice v_fma_mix_f32's rate
    float v[8];
    // A block's values start 2 bytes past a dword for even kb, on one for odd.
    if constexpr (U::kQ4) {
        uint32_t w;
        if (kb % 2) {
            w = *reinterpret_cast<const uint32_t*>(blk + 2 + 4 * g16);
        } else {
            const uint32_t* a = reinterpret_cast<const uint32_t*>(blk + 4 * g16);
            w = __builtin_amdgcn_alignbyte(a[1], a[0], 2);
        }
        const uint32_t lo = ((w << 4) ^ 0x80808080u) & 0xf0f0f0f0u;
        const uint32_t hi = (w ^ 0x80808080u) & 0xf0f0f0f0u;
        v[0] = sbyte<0>(lo); v[1] = sbyte<1>(lo); v[2] = sbyte<2>(lo); v[3] = sbyte<3>(lo);
        v[4] = sbyte<0>(hi); v[5] = sbyte<1>(hi); v[6] = sbyte<2>(hi); v[7] = sbyte<3>(hi);
    } else {
        uint32_t w0, w1;
        if (kb % 2) {
            const uint32_t* a = reinterpret_cast<const uint32_t*>(blk + 2 + 8 * g16);
            w0 = a[0];
            w1 = a[1];
        } else {
            const uint32_t* a = reinterpret_cast<const uint32_t*>(blk + 8 * g16);
            const uint32_t a0 = a[0], a1 = a[1], a2 = a[2];
            w0 = __builtin_amdgcn_alignbyte(a1, a0, 2);
            w1 = __builtin_amdgcn_alignbyte(a2, a1, 2);
        }
        v[0] = sbyte<0>(w0); v[1] = sbyte<1>(w0); v[2] = sbyte<2>(w0); v[3] = sbyte<3>(w0);
        v[4] = sbyte<0>(w1); v[5] = sbyte<1>(w1); v[6] = sbyte<2>(w1); v[7] = sbyte<3>(w1);
    }
    u32x4 w;
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = bf16_pair(__float_as_uint(v[2 * e]), __float_as_uint(v[2 * e + 1]));
    return __builtin_bit_cast(bf16x8, w);
}

// A workgroup takes one A tile and 16 N weight rows; its WK waves take the K
// units (SegUnit) in turn and add their sums at the end through LDS, in wave
// order.  Nothing is shared before that, so a wave never waits for another:
// per unit it moves its N x 16 row pieces and its A chunk from registers to
// its own LDS, requests the next ones, and forms the operands from there.
//
// What bounds it, and why this shape (MI355X, in-kernel cycle stamps and
// variants with parts left out): with few A rows the launch is the weight
// stream plus the A rows every workgroup reads again.  An address that 64
// lanes read in 64 separate 16-byte pieces costs the vector memory pipeline 64
// cycles (14-15 B/clk a CU), adjacent lanes on adjacent memory 16 (52-57
// B/clk), so both operands are loaded along their rows and turned into operand
// order in LDS; loading A in operand order (16 rows a load) instead took
// 19.6 us where this takes 16.2 (7 x 12288 x 4096, Q8_0).  After that the
// instructions: converting eight weights takes 12 half-rate ones a lane
// whatever the A rows, splitting eight activations 22, which N row tiles
// share.  K is split over the waves of a workgroup, not over workgroups: a
// second launch to add the parts costs more than it gives at these sizes.
//
// TB blocks share the operand registers of one 16-row A subtile where a tile
// has at most 16 / TB rows: row group j of the subtile (16 / TB rows) carries
// block b + j.  Each block's product is formed with the same operand, a lane
// keeps the one its output rows belong to, and the row groups are added at
// the end: the activations of TB blocks are split for the price of one.
template <uint32_t QT, int NT, int TB, int N, int WK, class Policy>
__global__ __launch_bounds__(WK * kWave) void gemm_thin_kernel(Policy pol, int rows, int cols) {
    using U = SegUnit<QT>;
    static_assert(NT == 1 || TB == 1, "blocks share one A subtile only");
    static_assert(!Policy::kPairedColumns || N % 2 == 0, "paired columns need row tiles in pairs");
    constexpr int TR = 16 / TB;  // A rows of a subtile per block
    constexpr int BM = NT == 1 ? TR : 16 * NT, BN = 16 * N;
    constexpr int CB = NT == 1 ? 4 : 2;            // blocks of an A chunk
    constexpr int G = CB / TB;                     // operand groups of a chunk
    constexpr int kChunks = U::BLOCKS / CB;        // A chunks per weight unit
    constexpr int kALoads = BM * CB / 8;           // 16-byte loads a lane per A chunk
    constexpr int A_PITCH = CB * 128 + 16;         // bytes of an A row in LDS
    constexpr int A_BYTES = BM * A_PITCH;
    constexpr int kWaveLds = N * U::BYTES + A_BYTES;
    static_assert(kChunks >= 1 && G >= 1 && kWaveLds >= N * NT * 1024, "the sums reuse a wave's LDS");
    __shared__ __attribute__((aligned(16))) uint8_t lds[WK * kWaveLds];

    const int total = LinearTotal<Policy>::get(pol, gridDim.x), L = blockIdx.x;
    if (L >= total) return;
    GemmTile tile;
    if (!pol.tile(L / pol.tiles_x, BM, tile)) return;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
    const int l16 = lane & 15, g16 = lane >> 4;
    const int n0 = (L % pol.tiles_x) * BN;
    const int nblk = cols / kBlock;
    const int row_bytes = nblk * U::BB;
    const int units = nblk / U::BLOCKS;
    uint8_t* const wl = lds + wave * kWaveLds;
    uint8_t* const al = wl + N * U::BYTES;

    // A chunk: load j of a lane is 16 bytes of row j * (8 / CB) + lane / (8 CB),
    // so adjacent lanes read adjacent memory (rows past the valid ones read
    // the last one; their outputs are not stored).
    const float* a_src[kALoads];
#pragma unroll
    for (int j = 0; j < kALoads; ++j)
        a_src[j] = pol.a_row(tile, min(j * (8 / CB) + lane / (8 * CB), tile.mcount - 1)) + 4 * (lane % (8 * CB));
    f32x4 a_reg[kALoads];
    auto load_a = [&](int kb) {
#pragma unroll
        for (int j = 0; j < kALoads; ++j) a_reg[j] = *reinterpret_cast<const f32x4*>(a_src[j] + kBlock * kb);
    };
    auto store_a = [&]() {
#pragma unroll
        for (int j = 0; j < kALoads; ++j)
            *reinterpret_cast<f32x4*>(al + (j * (8 / CB) + lane / (8 * CB)) * A_PITCH + 16 * (lane % (8 * CB))) = a_reg[j];
    };
    if (wave < units) load_a(wave * U::BLOCKS);

    int off[U::WIDE + 1];
#pragma unroll
    for (int j = 0; j <= U::WIDE; ++j) {
        const int pos = j < U::WIDE ? 16 * (j * kWave + lane) : U::WIDE * 1024 + 4 * lane;
        off[j] = pos / U::PITCH * row_bytes + pos % U::PITCH;
    }
    const uint8_t* first[N];  // row 0 of each 16-row unit (uniform)
    int bytes[N];             // bytes of its valid rows
#pragma unroll
    for (int t = 0; t < N; ++t) {
        const int n = n0 + 16 * t;
        const uintptr_t p = reinterpret_cast<uintptr_t>(pol.b_row(tile, min(n, rows - 1)));
        const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(p));
        const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(p >> 32));
        first[t] = reinterpret_cast<const uint8_t*>((static_cast<uintptr_t>(hi) << 32) | lo);
        bytes[t] = max(0, min(16, rows - n)) * row_bytes;
    }
    SegRegs reg[N];
    auto load_units = [&](int u) {  // past the last unit: zeros, no memory touched
        const bool live = u < units;
        const int at = live ? u * U::STEP : 0;
#pragma unroll
        for (int t = 0; t < N; ++t) {
            const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<uint8_t*>(first[t] + at), 0, live ? max(0, bytes[t] - at) : 0, kBufferFlags);
#pragma unroll
            for (int j = 0; j < U::WIDE; ++j)
                reg[t].wide[j] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off[j], 0, kNonTemporal);
            reg[t].rest = __builtin_amdgcn_raw_buffer_load_b32(rsrc, off[U::WIDE], 0, kNonTemporal);
        }
    };
    auto store_units = [&]() {
#pragma unroll
        for (int t = 0; t < N; ++t) {
#pragma unroll
            for (int j = 0; j < U::WIDE; ++j)
                *reinterpret_cast<u32x4*>(wl + t * U::BYTES + 1024 * j + 16 * lane) = reg[t].wide[j];
            *reinterpret_cast<uint32_t*>(wl + t * U::BYTES + 1024 * U::WIDE + 4 * lane) = reg[t].rest;
        }
    };
    // All ones where this lane's output rows belong to block b + j or later.
    uint32_t pick[TB];
#pragma unroll
    for (int j = 0; j < TB; ++j) pick[j] = 4 * g16 >= j * TR ? 0xffffffffu : 0u;

    f32x4 acc[N][NT];
#pragma unroll
    for (int t = 0; t < N; ++t)
#pragma unroll
        for (int i = 0; i < NT; ++i) acc[t][i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    load_units(wave);
    for (int u = wave; u < units; u += WK) {
#pragma unroll
        for (int c = 0; c < kChunks; ++c) {
            store_a();
            if (c == 0) store_units();
            wave_lds_sync();
            // Loads return in order: the next unit's weights are requested
            // after the A values that are waited for before them.
            if (c + 1 < kChunks) load_a(u * U::BLOCKS + (c + 1) * CB);
            else load_a(min(u + WK, units - 1) * U::BLOCKS);
            if (c + 1 == kChunks) load_units(u + WK);
            bf16x8 plane[NT][G][3];
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int b = 0; b < G; ++b) {
                    const uint8_t* at =
                        al + (16 * i + l16 % TR) * A_PITCH + 128 * (b * TB + l16 / TR) + (U::kQ4 ? 16 : 32) * g16;
                    const f32x4 lo = *reinterpret_cast<const f32x4*>(at);
                    const f32x4 hi = *reinterpret_cast<const f32x4*>(at + (U::kQ4 ? 64 : 16));
                    uint32_t p[3][8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) split3(e < 4 ? lo[e] : hi[e - 4], p[0][e], p[1][e], p[2][e]);
#pragma unroll
                    for (int q = 0; q < 3; ++q)
                        plane[i][b][q] = __builtin_bit_cast(
                            bf16x8, u32x4{bf16_pair(p[q][0], p[q][1]), bf16_pair(p[q][2], p[q][3]),
                                          bf16_pair(p[q][4], p[q][5]), bf16_pair(p[q][6], p[q][7])});
                }
#pragma unroll
            for (int b = 0; b < G; ++b) {
                const int kb = c * CB + b * TB;
#pragma unroll
                for (int t = 0; t < N; ++t) {
                    const uint8_t* unit = wl + t * U::BYTES;
                    bf16x8 w[TB];
                    float d[TB];
#pragma unroll
                    for (int j = 0; j < TB; ++j) w[j] = seg_operand<QT>(unit, l16, g16, kb + j, d[j]);
                    float scale = d[0];
                    if constexpr (TB > 1) {
                        // The block this lane's output rows belong to.
                        const uint32_t half = *reinterpret_cast<const uint16_t*>(unit + l16 * U::PITCH +
                                                                                 (kb + 4 * g16 / TR) * U::BB);
                        scale = U::kQ4 ? f16_fast(half) * 0.0625f : f16_fast(half);
                    }
                    asm("" : "+v"(scale));  // an FP32 value: v_fma_f32 issues at twice v_fma_mix_f32's rate
#pragma unroll
                    for (int i = 0; i < NT; ++i) {
                        f32x4 sum[TB];
#pragma unroll
                        for (int j = 0; j < TB; ++j) sum[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                        for (int q = 2; q >= 0; --q)
#pragma unroll
                            for (int j = 0; j < TB; ++j)
                                sum[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(plane[i][b][q], w[j], sum[j], 0, 0, 0);
                        f32x4 own = sum[0];
#pragma unroll
                        for (int j = 1; j < TB; ++j)
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                own[e] = __uint_as_float((__float_as_uint(sum[j][e]) & pick[j]) |
                                                         (__float_as_uint(own[e]) & ~pick[j]));
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[t][i][e] = fmaf(scale, own[e], acc[t][i][e]);
                    }
                }
            }
            wave_lds_sync();
        }
    }

    // The WK waves' sums of a row tile, added in wave order; a lane of row
    // group j holds the sums over its blocks b + j, added in group order.
    __syncthreads();
    f32x4* part = reinterpret_cast<f32x4*>(lds);
    auto slot = [&](int k, int t, int i) { return (k * N * NT + t * NT + i) * kWave; };
#pragma unroll
    for (int t = 0; t < N; ++t)
#pragma unroll
        for (int i = 0; i < NT; ++i) part[slot(wave, t, i) + lane] = acc[t][i];
    __syncthreads();
    constexpr int STEP = Policy::kPairedColumns ? 2 : 1;
    for (int q = wave; q < N * NT / STEP; q += WK) {
        const int t = q / NT * STEP, i = q % NT;
        f32x4 sum[STEP];
#pragma unroll
        for (int h = 0; h < STEP; ++h) {
#pragma unroll
            for (int k = 0; k < WK; ++k) {
                f32x4 v = part[slot(k, t + h, i) + lane];
#pragma unroll
                for (int j = 1; j < TB; ++j) v += part[slot(k, t + h, i) + ((lane + j * (kWave / TB)) & (kWave - 1))];
                sum[h] = k ? sum[h] + v : v;
            }
        }
        const int n = n0 + 16 * t + l16;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int m = 16 * i + 4 * g16 + e;
            if (m >= tile.mcount || n >= rows) continue;
            if constexpr (Policy::kPairedColumns) pol.store_pair(tile, m, n, sum[0][e], sum[STEP - 1][e]);
            else pol.store(tile, m, n, sum[0][e]);
        }
    }
}

// Waves of a workgroup: eight (two workgroups a CU where the registers
// allow); four and sixteen measured slower on the 9B's and 27B's matrices
// except the shortest.
constexpr int kThinWaves = 8;
constexpr int kThinMaxRows = 32;  // A rows of the largest tile

// The kernel reads whole units of weight rows 16 bytes at a time: row length
// a multiple of 256 columns, 16-byte aligned rows and activations.  Against
// gemm_x3.h's tiles (with a K-split workspace) on Q8_0 and Q4_0 matrices of
// 128 to 20000 rows and 1024 to 24576 columns it took 0.33-0.58 of the time
// at 2 and 8 tokens, 0.41-0.73 at 16 and 0.45-0.98 at 32 up to 16384 columns;
// there, past that length, a wave's K units in turn took 0.65 to 1.08 of
// it.  From 33 tokens on, gemm_x3.h's 64-row tiles read the weights fewer times.
inline bool thin_ok(int count, int cols, bool aligned16) {
    return aligned16 && cols % (8 * kBlock) == 0 && cols <= (1 << 22) && count <= kThinMaxRows &&
           (count <= 16 || cols <= 16384);
}

// Row tiles per workgroup for `rows` weight rows: as many as leave one
// workgroup a CU, at most three (more spill registers).  Taller matrices take
// several workgroups a CU in turn: two row tiles each where the A operand is
// cheap (at most 8 rows), else three.
inline int thin_row_tiles(int rows, int count) {
    const int per_cu = ((rows + 15) / 16 + kCUs - 1) / kCUs;
    return per_cu <= 3 ? per_cu : count <= 8 ? 2 : 3;
}

template <uint32_t QT, int NT, int TB, class P>
int launch_thin_shape(P pol, int rows, int count, int cols, hipStream_t stream) {
    constexpr int BM = NT == 1 ? 16 / TB : 16 * NT;
    const int tiles_y = (count + BM - 1) / BM;
    auto launch = [&](auto n) {
        constexpr int N = decltype(n)::value;
        pol.tiles_x = (rows + 16 * N - 1) / (16 * N);
        const long long tiles = static_cast<long long>(pol.tiles_x) * tiles_y;
        if (tiles > 0x7fffffLL) return static_cast<int>(Q3X_HIP_EINVAL);
        hipLaunchKernelGGL((gemm_thin_kernel<QT, NT, TB, N, kThinWaves, P>), dim3(static_cast<unsigned>(tiles)),
                           dim3(kThinWaves * kWave), 0, stream, pol, rows, cols);
        return launch_status();
    };
    if constexpr (P::kPairedColumns) {
        return launch(std::integral_constant<int, 2>{});
    } else {
        switch (thin_row_tiles(rows, count)) {
            case 1: return launch(std::integral_constant<int, 1>{});
            case 2: return launch(std::integral_constant<int, 2>{});
            default: return launch(std::integral_constant<int, 3>{});
        }
    }
}

// One launch over `count` A rows and `rows` weight rows (thin_ok).  7 x 12288
// x 4096 Q8_0 16 us (43 on gemm_x3.h's tiles; a matvec of it 12), 24 rows 24
// (45); 7 x 17408 x 5120 Q4_0 25 us (63); 7 x 1024 x 4096 8 us (16).  The A tile is the smallest that holds the rows.
template <uint32_t QT, class P>
int launch_thin(const P& pol, int rows, int count, int cols, hipStream_t stream) {
    if (count <= 4) return launch_thin_shape<QT, 1, 4>(pol, rows, count, cols, stream);
    if (count <= 8) return launch_thin_shape<QT, 1, 2>(pol, rows, count, cols, stream);
    if (count <= 16) return launch_thin_shape<QT, 1, 1>(pol, rows, count, cols, stream);
    return launch_thin_shape<QT, 2, 1>(pol, rows, count, cols, stream);
}

}  // namespace q3x
