// gemm_thin.h -- FP32 GEMM for a few A rows: Y[m, n] as gemm_x3.h forms it
// (exact bf16 products of the three-way split activations, FP32 sums, the
// block scale by FMA), for tiles of at most 32 A rows.
#pragma once

#include "gemm_x3.h"
#include "matvec.h"

namespace q3x {

// A unit of weights: 16 consecutive rows of one K segment of BLOCKS blocks,
// PITCH bytes a row in LDS, loaded as 16-byte words a lane and one last dword.
// ANY = false: rows of whole units, every row piece 16-byte aligned.  Q8_0: 4
// blocks are 136 bytes and the load takes 8 more; Q4_0: 8 blocks, 144 bytes.
// ANY = true: rows of any number of blocks (the last unit may be short), 2-byte
// aligned; a row piece is loaded from the dword at or before its start, so a
// row of odd number starts 2 bytes in where a row is not whole dwords.
template <uint32_t QT, bool ANY>
struct SegUnit {
    static constexpr bool kQ4 = QT == Q3X_HIP_MATRIX_Q4_0;
    static constexpr int BB = kQ4 ? kQ4Bytes : kQ8Bytes;
    static constexpr int BLOCKS = kQ4 && !ANY ? 8 : 4;
    static constexpr int STEP = BLOCKS * BB;  // bytes from a segment to the row's next: whole dwords
    static constexpr int PITCH = kQ4 && ANY ? 80 : 144;
    static constexpr int BYTES = 16 * PITCH;
    static constexpr int WIDE = BYTES / 1024;
    static_assert(BYTES == WIDE * 1024 + 256 && STEP + (ANY ? 2 : 0) <= PITCH && STEP % 4 == 0,
                  "16-byte words and one dword a lane hold the row pieces");
};

template <int WIDE>
struct SegRegs {
    u32x4 wide[WIDE];
    uint32_t rest;
};

// This lane's bf16 operand of block kb of a unit in LDS: weight row l16, the
// eight values of chunk g16.  Q8_0: elements 8 g16 + [0, 8).  Q4_0: elements
// 4 g16 + [0, 4) and 16 + 4 g16 + [0, 4), as 16 (n - 8) (BlockPart::values;
// the scale is then d / 16).  skew: bytes the row starts late by (ANY).
template <uint32_t QT, bool ANY>
__device__ __forceinline__ bf16x8 seg_operand(const uint8_t* unit, int l16, int g16, int kb, int skew) {
    using U = SegUnit<QT, ANY>;
    const uint8_t* values = unit + l16 * U::PITCH + kb * U::BB + 2 + (U::kQ4 ? 4 : 8) * g16;
    // Whole dwords around them; aligned rows start 2 bytes into one for even
    // kb, on one for odd.
    const int late = ANY ? (2 * (kb + 1) + skew) % 4 : 2 * ((kb + 1) % 2);
    const uint32_t* a = reinterpret_cast<const uint32_t*>(values + (ANY ? skew : 0) - late);
    float v[8];
    if constexpr (U::kQ4) {
        const uint32_t w = ANY || late ? __builtin_amdgcn_alignbyte(a[1], a[0], late) : a[0];
        const uint32_t lo = ((w << 4) ^ 0x80808080u) & 0xf0f0f0f0u;
        const uint32_t hi = (w ^ 0x80808080u) & 0xf0f0f0f0u;
        v[0] = sbyte<0>(lo); v[1] = sbyte<1>(lo); v[2] = sbyte<2>(lo); v[3] = sbyte<3>(lo);
        v[4] = sbyte<0>(hi); v[5] = sbyte<1>(hi); v[6] = sbyte<2>(hi); v[7] = sbyte<3>(hi);
    } else {
        const uint32_t a0 = a[0], a1 = a[1];
        uint32_t w0 = a0, w1 = a1;
        if (ANY || late) {
            const uint32_t a2 = a[2];
            w0 = __builtin_amdgcn_alignbyte(a1, a0, late);
            w1 = __builtin_amdgcn_alignbyte(a2, a1, late);
        }
        v[0] = sbyte<0>(w0); v[1] = sbyte<1>(w0); v[2] = sbyte<2>(w0); v[3] = sbyte<3>(w0);
        v[4] = sbyte<0>(w1); v[5] = sbyte<1>(w1); v[6] = sbyte<2>(w1); v[7] = sbyte<3>(w1);
    }
    u32x4 w;
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = bf16_pair(__float_as_uint(v[2 * e]), __float_as_uint(v[2 * e + 1]));
    return __builtin_bit_cast(bf16x8, w);
}

// The scale of block kb (may differ by lane) of weight row l16.
template <uint32_t QT, bool ANY>
__device__ __forceinline__ float seg_scale(const uint8_t* unit, int l16, int kb, int skew) {
    using U = SegUnit<QT, ANY>;
    const uint32_t half = *reinterpret_cast<const uint16_t*>(unit + l16 * U::PITCH + kb * U::BB + (ANY ? skew : 0));
    float d = U::kQ4 ? f16_fast(half) * 0.0625f : f16_fast(half);
    asm("" : "+v"(d));  // an FP32 value: v_fma_f32 issues at twice v_fma_mix_f32's rate
    return d;
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
template <uint32_t QT, bool ANY, int NT, int TB, int N, int WK, class Policy>
__global__ __launch_bounds__(WK * kWave) void gemm_thin_kernel(Policy pol, int rows, int cols) {
    using U = SegUnit<QT, ANY>;
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
    const int units = (nblk + U::BLOCKS - 1) / U::BLOCKS;
    const int skew = ANY ? 2 * (l16 & 1 & (row_bytes >> 1)) : 0;  // this lane's weight row starts late by
    uint8_t* const wl = lds + wave * kWaveLds;
    uint8_t* const al = wl + N * U::BYTES;

    // A chunk: load j of a lane is 16 bytes of row j * (8 / CB) + lane / (8 CB),
    // so adjacent lanes read adjacent memory (rows past the valid ones read
    // the last one; their outputs are not stored).
    const float* a_src[kALoads];
#pragma unroll
    for (int j = 0; j < kALoads; ++j)
        a_src[j] = pol.a_row(tile, min(j * (8 / CB) + lane / (8 * CB), tile.mcount - 1)) + 4 * (lane % 8);
    f32x4 a_reg[kALoads];
    auto load_a = [&](int kb) {  // blocks past the last read the last
        const int block = kb + lane % (8 * CB) / 8;
        const int k = kBlock * (ANY ? min(block, nblk - 1) : block);
#pragma unroll
        for (int j = 0; j < kALoads; ++j) a_reg[j] = *reinterpret_cast<const f32x4*>(a_src[j] + k);
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
        const int start = pos / U::PITCH * row_bytes;
        off[j] = (ANY ? start & ~3 : start) + pos % U::PITCH;
    }
    const uint8_t* first[N];  // row 0 of each 16-row unit (uniform)
    // Bytes of its valid rows, in whole dwords (the buffer range drops a
    // dword that is not whole; the matrix starts on one).
    int bytes[N];
#pragma unroll
    for (int t = 0; t < N; ++t) {
        const int n = n0 + 16 * t;
        const uintptr_t p = reinterpret_cast<uintptr_t>(pol.b_row(tile, min(n, rows - 1)));
        const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(p));
        const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(p >> 32));
        first[t] = reinterpret_cast<const uint8_t*>((static_cast<uintptr_t>(hi) << 32) | lo);
        bytes[t] = (max(0, min(16, rows - n)) * row_bytes + 3) & ~3;
    }
    // Weights pass the caches by, but for a grouped launch's Q8_0 ones on one or
    // two waves (many tiles): a segment of 136 bytes shares lines with the
    // next, which a wave there reads long after (on more waves another one reads
    // it at the same time), and an expert's tiles read its rows one after the
    // other.  19 tokens x top 8 of 256 experts (H 2048, I 512) 125 -> 100 us,
    // 300 321 -> 271, all 300 tokens on the same eight 150 -> 143; 300 drawn
    // layers, their weights in turn from memory, 0.98 (0.78 to 0.9 where the
    // experts hold some 500 MB, 1.03 for 101 tokens top 4 of 256, H 1280, I
    // 128).  Q4_0 (144 bytes) up to 3% slower cached, Q8_0 on four waves up to 4%
    // (20 tokens top 2 of 32, H 1792, I 736), on eight 9% (2 tokens top 1 of 16,
    // H 16128), one matrix 2 x 16 x 65536 51 us for 44.
    constexpr int kPolicy = Policy::kPartialTiles && !U::kQ4 && WK <= 2 ? 0 : kNonTemporal;
    SegRegs<U::WIDE> reg[N];
    auto load_units = [&](int u) {  // past the last unit: zeros, no memory touched
        const bool live = u < units;
        const int at = live ? u * U::STEP : 0;
#pragma unroll
        for (int t = 0; t < N; ++t) {
            const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<uint8_t*>(first[t] + at), 0, live ? max(0, bytes[t] - at) : 0, kBufferFlags);
#pragma unroll
            for (int j = 0; j < U::WIDE; ++j)
                reg[t].wide[j] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off[j], 0, kPolicy);
            reg[t].rest = __builtin_amdgcn_raw_buffer_load_b32(rsrc, off[U::WIDE], 0, kPolicy);
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
                if (ANY && u * U::BLOCKS + kb >= nblk) break;  // a short last unit: whole groups (thin_ok)
#pragma unroll
                for (int t = 0; t < N; ++t) {
                    const uint8_t* unit = wl + t * U::BYTES;
                    bf16x8 w[TB];
#pragma unroll
                    for (int j = 0; j < TB; ++j) w[j] = seg_operand<QT, ANY>(unit, l16, g16, kb + j, skew);
                    // The scale of the block this lane's output rows belong to.
                    const float scale = seg_scale<QT, ANY>(unit, l16, kb + 4 * g16 / TR, skew);
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
// allow); four and sixteen measured slower on the 9B's and 27B's matrices but
// for sixteen on the shortest (1024 rows), where eight are taken too.
constexpr int kThinWaves = 8;
constexpr int kThinMaxRows = 32;  // A rows of the largest tile

// Dword-aligned weights (every 16-row unit then starts on a dword, whatever the
// row length) and 16-byte aligned activations.  Against gemm_x3.h's tiles
// (with a K-split workspace) on Q8_0 and Q4_0 matrices of 128 to 20000 rows
// and 1024 to 24576 columns it took 0.33-0.58 of the time at 2 and 8 tokens,
// 0.41-0.73 at 16 and 0.45-0.98 at 32 up to 16384 columns; there, past that
// length, a wave's K units in turn took 0.65 to 1.08 of it.  (1 to 300 rows of
// 256 to 65536 columns: 0.53 on average, none slower.)  From 33 tokens on,
// gemm_x3.h's 64-row tiles read the weights fewer times.
inline bool thin_ok(int count, int rows, int cols, bool aligned_ok) {
    return aligned_ok && cols <= (1 << 22) && rows <= (1 << 26) && count <= kThinMaxRows && (count <= 16 || cols <= 16384);
}

// Row tiles per workgroup for `rows` weight rows: as many as leave one
// workgroup a CU, at most three.  Taller matrices take several workgroups a CU
// in turn: two row tiles each where the A operand is cheap (at most 8 rows),
// else three.  Registers set the limit: Q8_0 takes 256 for three row tiles of
// 32 A rows, 246 for 16; Q4_0 on whole units, eight blocks each, is past it
// from 9 A rows on (16 A rows x 2 and 3 row tiles keep 16 and 92 bytes a lane
// in scratch, 32 x 3 12), on rows of any length, four blocks a unit, at most 156.
inline int thin_row_tiles(int rows, int count) {
    const int per_cu = ((rows + 15) / 16 + kCUs - 1) / kCUs;
    return per_cu <= 3 ? per_cu : count <= 8 ? 2 : 3;
}

// `tiles_y` A tiles of the shape's height (for a grouped launch: at most).
template <uint32_t QT, bool ANY, int NT, int TB, int WK, class P>
int launch_thin_shape(P pol, int rows, int count, int cols, int tiles_y, hipStream_t stream) {
    auto launch = [&](auto n) {
        constexpr int N = decltype(n)::value;
        pol.tiles_x = (rows + 16 * N - 1) / (16 * N);
        const long long tiles = static_cast<long long>(pol.tiles_x) * tiles_y;
        if (tiles > 0x7fffffLL) return static_cast<int>(Q3X_HIP_EINVAL);
        hipLaunchKernelGGL((gemm_thin_kernel<QT, ANY, NT, TB, N, WK, P>), dim3(static_cast<unsigned>(tiles)),
                           dim3(WK * kWave), 0, stream, pol, rows, cols);
        return launch_status();
    };
    if constexpr (P::kPairedColumns || P::kPartialTiles) {
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
// (45); 7 x 17408 x 5120 Q4_0 25 us (63); 7 x 1024 x 4096 8 us (16).  The A
// tile is the smallest that holds the rows.
template <uint32_t QT, bool ANY, class P>
int launch_thin_rows(const P& pol, int rows, int count, int cols, hipStream_t stream) {
    // A group of TB blocks must not straddle the row's end.
    const int nblk = cols / kBlock;
    if (count <= 4 && (!ANY || nblk % 4 == 0)) return launch_thin_shape<QT, ANY, 1, 4, kThinWaves>(pol, rows, count, cols, 1, stream);
    if (count <= 8 && (!ANY || nblk % 2 == 0)) return launch_thin_shape<QT, ANY, 1, 2, kThinWaves>(pol, rows, count, cols, 1, stream);
    if (count <= 16) return launch_thin_shape<QT, ANY, 1, 1, kThinWaves>(pol, rows, count, cols, 1, stream);
    return launch_thin_shape<QT, ANY, 2, 1, kThinWaves>(pol, rows, count, cols, 1, stream);
}

// Rows of whole units, 16-byte aligned?
inline bool thin_whole(int cols, bool aligned16) { return aligned16 && cols % (8 * kBlock) == 0; }

template <uint32_t QT, class P>
int launch_thin(const P& pol, int rows, int count, int cols, bool aligned16, hipStream_t stream) {
    return thin_whole(cols, aligned16) ? launch_thin_rows<QT, false>(pol, rows, count, cols, stream)
                                       : launch_thin_rows<QT, true>(pol, rows, count, cols, stream);
}

// A grouped launch (a tile table on the device, at most `tiles_y` tiles of
// `height` rows, about `tiles` of them live): two row tiles a workgroup.  K is
// split over about 16 waves a CU, no more: a wave waits some microseconds for
// its first unit whatever follows.  The 4- and 8-row shapes hold 16 at once (12
// on eight waves in some), the 16- and 32-row ones 8 to 12, but a split for 8
// there gained nothing (geometric mean 1.00 over 220 calls of 2 to 400 tokens,
// 0.90 to 1.09).  Two and four waves besides one and eight: 5 tokens x top 4 of
// 128 experts (H 2048, I 768) Q4_0 34 us for 47, 0.97 over the same calls.
template <uint32_t QT, bool ANY, class P>
int launch_thin_grouped(const P& pol, int height, int rows, int cols, int tiles_y, double tiles, hipStream_t stream) {
    using U = SegUnit<QT, ANY>;
    const int units = (cols / kBlock + U::BLOCKS - 1) / U::BLOCKS;
    const double split = std::min<double>(units, 16.0 * kCUs / (tiles * ((rows + 31) / 32)));
    auto waves = [&](auto nt, auto tb) {
        constexpr int NT = decltype(nt)::value, TB = decltype(tb)::value;
        if (split >= 6.0) return launch_thin_shape<QT, ANY, NT, TB, 8>(pol, rows, height, cols, tiles_y, stream);
        if (split >= 3.0) return launch_thin_shape<QT, ANY, NT, TB, 4>(pol, rows, height, cols, tiles_y, stream);
        if (split >= 1.5) return launch_thin_shape<QT, ANY, NT, TB, 2>(pol, rows, height, cols, tiles_y, stream);
        return launch_thin_shape<QT, ANY, NT, TB, 1>(pol, rows, height, cols, tiles_y, stream);
    };
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I4 = std::integral_constant<int, 4>;
    // Blocks share operand registers only where they do not straddle the row's
    // end; a taller tile shape takes a shorter tile too.
    const int nblk = cols / kBlock;
    if (height <= 4 && (!ANY || nblk % 4 == 0)) return waves(I1{}, I4{});
    if (height <= 8 && (!ANY || nblk % 2 == 0)) return waves(I1{}, I2{});
    if (height <= 16) return waves(I1{}, I1{});
    return waves(I2{}, I1{});
}

}  // namespace q3x
