// misc.hip -- sizes, error strings, dequantisation and the device quantizer.
#include <math.h>

#include "common.h"

namespace q3x {

// out[i] = f16(d) * q (Q8_0) or f16(d) * (nibble - 8) (Q4_0) for the values
// of `blocks` consecutive blocks: the reference's embed (arch/cpu.cpp:55-63,
// 81-90), bit for bit.  The scale is decoded with the reference's own bit
// manipulation, and the product of an 11-bit significand with an integer of
// at most 8 bits is exact in FP32.
//
// Bound by HBM: 4 bytes written per value for 0.56 or 1.06 read.  Rows follow
// each other without padding, so a value's block is its index / 32 and no
// thread divides by the row length.  A thread forms four consecutive values
// (one 16-byte store where `out` allows it) of kDequantQuads quads a
// workgroup apart, all of whose loads are requested before any is used; a
// wave's store is 1 KB contiguous and its loads the eight blocks behind it.
// Packing 17408 x 5120 BF16 values to Q4_0 and dequantising them (634 MB in
// all) takes 142 us against 368 us with one value per thread here and one
// block per thread in the quantizer (246 and 140 us of it), 4.5 TB/s, where a
// large device copy reaches 4.9.
constexpr int kDequantThreads = 256;
constexpr int kDequantQuads = 4;

template <uint32_t QT, bool WIDE>
__global__ __launch_bounds__(kDequantThreads) void dequant_kernel(const uint8_t* __restrict__ w, size_t quads,
                                                                  float* __restrict__ out) {
    constexpr int BB = QT == Q3X_HIP_MATRIX_Q8_0 ? kQ8Bytes : kQ4Bytes;
    const size_t first = static_cast<size_t>(blockIdx.x) * (kDequantThreads * kDequantQuads) + threadIdx.x;
    uint32_t scale[kDequantQuads], raw[kDequantQuads];
#pragma unroll
    for (int u = 0; u < kDequantQuads; ++u) {
        const size_t quad = min(first + static_cast<size_t>(u) * kDequantThreads, quads - 1);
        const uint8_t* blk = w + quad / 8 * BB;
        const int part = static_cast<int>(quad % 8);
        __builtin_memcpy(&scale[u], blk, 2);
        scale[u] &= 0xffffu;
        __builtin_memcpy(&raw[u], blk + 2 + 4 * (QT == Q3X_HIP_MATRIX_Q8_0 ? part : part % 4), 4);
    }
#pragma unroll
    for (int u = 0; u < kDequantQuads; ++u) {
        const size_t quad = first + static_cast<size_t>(u) * kDequantThreads;
        if (quad >= quads) break;
        const float d = f16_exact(scale[u]);
        const int high = static_cast<int>(quad % 8) / 4;  // Q4_0: elements 16..31 are high nibbles
        f32x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            int q;
            if (QT == Q3X_HIP_MATRIX_Q8_0) q = static_cast<int8_t>(raw[u] >> (8 * j));
            else q = static_cast<int>((raw[u] >> (8 * j + 4 * high)) & 15u) - 8;
            v[j] = d * static_cast<float>(q);
        }
        if constexpr (WIDE) {
            reinterpret_cast<f32x4*>(out)[quad] = v;
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) out[4 * quad + j] = v[j];
        }
    }
}

// IEEE binary32 -> binary16, round to nearest even (numpy's astype("<f2")),
// in integer arithmetic so the sign of zero and every rounding are explicit
// (the compiler may otherwise fold the conversion into a mixed-precision FMA
// with a +0 addend, which turns -0 into +0).
__device__ __forceinline__ uint16_t f32_to_f16_rne(float value) {
    const uint32_t bits = __float_as_uint(value);
    const uint32_t sign = (bits >> 16) & 0x8000u;
    const uint32_t exponent = (bits >> 23) & 0xffu;
    uint32_t mantissa = bits & 0x7fffffu;
    if (exponent == 0xffu)  // inf / nan (quiet the nan, keep its top payload bits)
        return static_cast<uint16_t>(sign | 0x7c00u | (mantissa ? 0x200u | (mantissa >> 13) : 0u));
    const int e = static_cast<int>(exponent) - 127 + 15;
    if (e >= 31) return static_cast<uint16_t>(sign | 0x7c00u);
    if (e <= 0) {  // half subnormal or zero
        if (e < -10) return static_cast<uint16_t>(sign);
        mantissa |= 0x800000u;
        const int shift = 14 - e;
        uint32_t half = mantissa >> shift;
        const uint32_t rest = mantissa & ((1u << shift) - 1u);
        const uint32_t halfway = 1u << (shift - 1);
        if (rest > halfway || (rest == halfway && (half & 1u))) ++half;
        return static_cast<uint16_t>(sign | half);
    }
    uint32_t half = (static_cast<uint32_t>(e) << 10) | (mantissa >> 13);
    const uint32_t rest = mantissa & 0x1fffu;
    if (rest > 0x1000u || (rest == 0x1000u && (half & 1u))) ++half;  // may carry into inf
    return static_cast<uint16_t>(sign | half);
}

// Eight consecutive values as FP32: FP32 input as is, BF16 input widened
// exactly (bits << 16), as the packer widens its BF16 rows
// (scripts/pack_weights.py:303-305).
__device__ __forceinline__ void load_eight(const float* __restrict__ src, size_t e, float (&v)[8]) {
    const f32x4* s4 = reinterpret_cast<const f32x4*>(src + e * 8);
    const f32x4 a = s4[0], b = s4[1];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[i] = a[i];
        v[4 + i] = b[i];
    }
}
__device__ __forceinline__ void load_eight(const uint16_t* __restrict__ src, size_t e, float (&v)[8]) {
    const u32x4 t = *reinterpret_cast<const u32x4*>(src + e * 8);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[2 * i] = __uint_as_float(t[i] << 16);
        v[2 * i + 1] = __uint_as_float(t[i] & 0xffff0000u);
    }
}

// The quantizers of scripts/pack_weights.py:299-343 on FP32 values.  Q8_0:
// d = max|v| / 127 (FP32), inverse = 1/d (0 when d == 0), q =
// clip(copysign(floor(|v * inverse| + 0.5), v * inverse), -127, 127).  Q4_0:
// m = the first value of largest magnitude, d = m / -8, inverse as above,
// nibble = min(15, trunc(v * inverse + 8.5)); low nibbles hold elements
// 0..15.  Both store d as fp16.  (A NaN is never larger; the first value of a
// Q4_0 block stays the choice where it is NaN itself.)
//
// Bound by HBM: 2 or 4 bytes read per value, 0.56 or 1.06 written.  Four
// lanes of a quad share a block, eight values each, so a wave reads 1 KB (BF16)
// contiguous per load; the block's maximum and, for Q4_0, the other half's
// nibbles are exchanged by DPP inside the quad.  A workgroup packs
// kQuantBlocks blocks into LDS and writes them out as one contiguous run of
// 16-byte words (kQuantBlocks blocks are a multiple of 16 bytes in either
// format); where dst is not 16-byte aligned, the words inside the run, put
// together from LDS dwords, and single bytes around them (all in single bytes
// 5001 x 2080 BF16 values to Q8_0 took 9.5 us, 8.6 so).  One thread
// per block, with 64- or 128-byte strided loads and 18 or 34 byte stores of
// its own, took 140 us for 17408 x 5120 BF16 values (1.6 TB/s); the figures of
// this form are beside dequant_kernel.
constexpr int kQuantThreads = 256;
constexpr int kQuantBlocks = 256;  // per workgroup: four rounds of 64 blocks

template <uint32_t QT, typename Src>
__global__ __launch_bounds__(kQuantThreads) void quantize_kernel(const Src* __restrict__ src, size_t blocks,
                                                                 uint8_t* __restrict__ dst, bool wide) {
    // The packer rounds every operation separately (numpy): no FMA contraction.
#pragma clang fp contract(off)
    constexpr int BB = QT == Q3X_HIP_MATRIX_Q8_0 ? kQ8Bytes : kQ4Bytes;
    constexpr int kRounds = kQuantBlocks * 4 / kQuantThreads;
    static_assert(kQuantBlocks * BB % 16 == 0, "a workgroup's run is whole 16-byte words");
    __shared__ __attribute__((aligned(16))) uint8_t packed[kQuantBlocks * BB + 16];  // and a dword past the last word
    const size_t block0 = static_cast<size_t>(blockIdx.x) * kQuantBlocks;
    const int part = threadIdx.x & 3;  // eighth values 8 * part .. + 7 of the block
    float v[kRounds][8];
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        const size_t e = block0 * 4 + r * kQuantThreads + threadIdx.x;
        load_eight(src, min(e, blocks * 4 - 1), v[r]);
    }
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        uint16_t* out = reinterpret_cast<uint16_t*>(packed + (r * kQuantThreads + threadIdx.x) / 4 * BB);
        if (QT == Q3X_HIP_MATRIX_Q8_0) {
            float maximum = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; ++i) maximum = fabsf(v[r][i]) > maximum ? fabsf(v[r][i]) : maximum;
            float other = dpp_f32<0xB1>(maximum);
            maximum = other > maximum ? other : maximum;
            other = dpp_f32<0x4E>(maximum);
            maximum = other > maximum ? other : maximum;
            const float scale = maximum / 127.0f;
            const float inverse = scale != 0.0f ? 1.0f / scale : 0.0f;
            if (part == 0) out[0] = f32_to_f16_rne(scale);
            uint32_t q[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float normalized = v[r][i] * inverse;
                float rounded = copysignf(floorf(fabsf(normalized) + 0.5f), normalized);
                rounded = fminf(fmaxf(rounded, -127.0f), 127.0f);
                q[i] = static_cast<uint32_t>(static_cast<int>(rounded)) & 0xffu;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) out[1 + 4 * part + i] = static_cast<uint16_t>(q[2 * i] | (q[2 * i + 1] << 8));
        } else {
            // Magnitudes order like their bits; a NaN ranks as zero, and as
            // the largest where it is the block's first value.
            uint32_t key = 0;
            float maximum = v[r][0];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t bits = __float_as_uint(v[r][i]) & 0x7fffffffu;
                uint32_t k = bits > 0x7f800000u ? 0u : bits;
                if (i == 0) {
                    key = bits > 0x7f800000u && part == 0 ? 0xffffffffu : k;
                } else if (k > key) {
                    key = k;
                    maximum = v[r][i];
                }
            }
            // Across the quad the lower lane's value wins a tie.
            auto merge = [&](uint32_t other_key, float other, bool other_first) {
                if (other_key > key || (other_key == key && other_first)) {
                    key = other_key;
                    maximum = other;
                }
            };
            merge(dpp_u32<0xB1>(key), dpp_f32<0xB1>(maximum), part & 1);
            merge(dpp_u32<0x4E>(key), dpp_f32<0x4E>(maximum), part & 2);
            const float scale = maximum / -8.0f;
            const float inverse = scale != 0.0f ? 1.0f / scale : 0.0f;
            if (part == 0) out[0] = f32_to_f16_rne(scale);
            uint32_t word[2] = {0u, 0u};
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float normalized = v[r][i] * inverse;
                const float t = truncf(normalized + 8.5f);
                word[i / 4] |= (static_cast<uint32_t>(static_cast<int>(fminf(t, 15.0f))) & 0xffu) << (8 * (i % 4));
            }
            // Lanes 2 and 3 hold the high nibbles of lanes 0 and 1.
            const uint32_t high0 = dpp_u32<0x4E>(word[0]) & 0x0f0f0f0fu, high1 = dpp_u32<0x4E>(word[1]) & 0x0f0f0f0fu;
            if (part < 2) {
                const uint32_t w0 = word[0] | (high0 << 4), w1 = word[1] | (high1 << 4);
                out[1 + 4 * part + 0] = static_cast<uint16_t>(w0);
                out[1 + 4 * part + 1] = static_cast<uint16_t>(w0 >> 16);
                out[1 + 4 * part + 2] = static_cast<uint16_t>(w1);
                out[1 + 4 * part + 3] = static_cast<uint16_t>(w1 >> 16);
            }
        }
    }
    __syncthreads();
    const int bytes = static_cast<int>(min(static_cast<size_t>(kQuantBlocks), blocks - block0)) * BB;
    uint8_t* run = dst + block0 * BB;
    // Bytes before the first 16-byte boundary of dst, and words after them.
    const int head = wide ? 0 : min(bytes, static_cast<int>(-reinterpret_cast<uintptr_t>(run) & 15));
    const int words = (bytes - head) / 16;
    if (wide) {
        for (int i = threadIdx.x; i < words; i += kQuantThreads)
            reinterpret_cast<u32x4*>(run)[i] = reinterpret_cast<const u32x4*>(packed)[i];
    } else {
        const uint32_t* dwords = reinterpret_cast<const uint32_t*>(packed) + head / 4;
        for (int i = threadIdx.x; i < words; i += kQuantThreads) {
            uint32_t w[5];
#pragma unroll
            for (int j = 0; j < 5; ++j) w[j] = dwords[4 * i + j];
            u32x4 v;
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = __builtin_amdgcn_alignbyte(w[j + 1], w[j], head & 3);
            reinterpret_cast<u32x4*>(run + head)[i] = v;
        }
        if (threadIdx.x < head) run[threadIdx.x] = packed[threadIdx.x];
    }
    for (int i = head + 16 * words + threadIdx.x; i < bytes; i += kQuantThreads) run[i] = packed[i];
}

}  // namespace q3x

using namespace q3x;

namespace q3x {

// A plain streaming read: every 16-byte chunk of the buffer once, with
// non-temporal loads, grid-stride over 512 workgroups of 1024 threads (two
// per CU).  The XOR of all words goes to *sink only if it equals a fixed
// pattern, so the loads stay live and the kernel practically never writes.
__global__ __launch_bounds__(1024) void read_probe_kernel(const u32x4* __restrict__ p, size_t n16,
                                                          uint32_t* __restrict__ sink) {
    uint32_t a = 0;
    for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < n16;
         i += static_cast<size_t>(gridDim.x) * blockDim.x) {
        const u32x4 v = __builtin_nontemporal_load(p + i);
        a ^= v.x ^ v.y ^ v.z ^ v.w;
    }
    if (a == 0x9e3779b9u) *sink = a;
}

}  // namespace q3x

extern "C" const char* q3x_hip_strerror(int code) {
    switch (code) {
    case Q3X_HIP_OK: return "ok";
    case Q3X_HIP_EINVAL: return "invalid argument";
    case Q3X_HIP_ERUNTIME: return "HIP runtime error";
    case Q3X_HIP_ENOTSUP: return "matrix type not handled by this backend";
    case Q3X_HIP_EMODEL: return "model.bin rejected";
    case Q3X_HIP_ESCRATCH: return "request needs more workspace than the library's static scratch";
    case Q3X_HIP_ESTATE: return "engine failed in an earlier forward; reset or restore it";
    default: return "unknown error";
    }
}

extern "C" int q3x_hip_quantized_bytes(uint32_t type, int rows, int cols, size_t* bytes) {
    size_t value;
    if (!bytes || !quantized_size(type, rows, cols, &value)) return Q3X_HIP_EINVAL;
    *bytes = value;
    return Q3X_HIP_OK;
}

extern "C" int q3x_hip_dequant(const void* w, uint32_t type, int cols, int row0, int nrows, float* out,
                               hipStream_t stream) {
    if (type == Q3X_HIP_MATRIX_BF16) return Q3X_HIP_ENOTSUP;
    size_t bytes;
    if (!w || !out || row0 < 0 || !quantized_size(type, nrows, cols, &bytes)) return Q3X_HIP_EINVAL;
    if (static_cast<long long>(row0) + nrows > 0x7fffffffLL) return Q3X_HIP_EINVAL;
    const size_t quads = static_cast<size_t>(nrows) * cols / 4;
    constexpr size_t kPerGroup = kDequantThreads * kDequantQuads;
    const size_t groups = (quads + kPerGroup - 1) / kPerGroup;
    if (groups > 0xffffffu) return Q3X_HIP_EINVAL;
    const size_t row_bytes = static_cast<size_t>(cols / kBlock) * block_bytes(type);
    const uint8_t* src = static_cast<const uint8_t*>(w) + row0 * row_bytes;
    const bool q8 = type == Q3X_HIP_MATRIX_Q8_0;
    auto kernel = aligned(out, 16) ? (q8 ? dequant_kernel<Q3X_HIP_MATRIX_Q8_0, true> : dequant_kernel<Q3X_HIP_MATRIX_Q4_0, true>)
                                   : (q8 ? dequant_kernel<Q3X_HIP_MATRIX_Q8_0, false> : dequant_kernel<Q3X_HIP_MATRIX_Q4_0, false>);
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(groups)), dim3(kDequantThreads), 0, stream, src, quads, out);
    return launch_status();
}

namespace {

template <typename Src>
int quantize_rows(uint32_t type, const Src* src, int rows, int cols, void* dst, hipStream_t stream) {
    if (type == Q3X_HIP_MATRIX_BF16) return Q3X_HIP_ENOTSUP;
    size_t bytes;
    if (!src || !dst || !quantized_size(type, rows, cols, &bytes) || !aligned(src, 16))
        return Q3X_HIP_EINVAL;
    const size_t blocks = static_cast<size_t>(rows) * (cols / kBlock);
    const size_t groups = (blocks + kQuantBlocks - 1) / kQuantBlocks;
    if (groups > 0xffffffu) return Q3X_HIP_EINVAL;
    auto kernel = type == Q3X_HIP_MATRIX_Q8_0 ? quantize_kernel<Q3X_HIP_MATRIX_Q8_0, Src>
                                              : quantize_kernel<Q3X_HIP_MATRIX_Q4_0, Src>;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(groups)), dim3(kQuantThreads), 0, stream, src, blocks,
                       static_cast<uint8_t*>(dst), aligned(dst, 16));
    return launch_status();
}

}  // namespace

extern "C" int q3x_hip_quantize(uint32_t type, const float* src, int rows, int cols, void* dst,
                                hipStream_t stream) {
    return quantize_rows(type, src, rows, cols, dst, stream);
}

extern "C" int q3x_hip_quantize_bf16(uint32_t type, const uint16_t* src, int rows, int cols, void* dst,
                                     hipStream_t stream) {
    return quantize_rows(type, src, rows, cols, dst, stream);
}

extern "C" int q3x_hip_read_probe(const void* buffer, size_t bytes, uint32_t* sink, hipStream_t stream) {
    if (!buffer || !sink || bytes == 0 || bytes % 16 != 0 || !aligned(buffer, 16)) return Q3X_HIP_EINVAL;
    hipLaunchKernelGGL(read_probe_kernel, dim3(2 * kCUs), dim3(1024), 0, stream,
                       static_cast<const u32x4*>(buffer), bytes / 16, sink);
    return launch_status();
}
