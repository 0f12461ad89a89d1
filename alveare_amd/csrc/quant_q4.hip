// GPU quantizer: float32 weights -> Q4 combined layout (alv_quantize_q4), or
// straight into a registered weight (alv_weight_quantize).
//
// The reference quantizes on the host in numpy (tools/convert/gemv_q_convert.py:
// quantize_to_q4_0 :5-51, pack_to_combined :53-85), after zero-padding the
// matrix to the kernel shape (tools/quantize_gemma4.py:26-41). Per 32-weight
// block of a row:
//   scale = max|w| / 7 in float32 (a NaN anywhere in the block makes it NaN,
//           as np.max does); a zero scale becomes 1.0;
//   q     = clip(round_half_even(w / scale), -8, 7), where a NaN quotient (a
//           NaN block, or inf / inf) becomes -8 -- numpy's astype(int32) gives
//           INT32_MIN for NaN on x86-64, which the clip takes to -8;
//   bytes = 16 nibble pairs (even column low), the bf16 scale (round to
//           nearest even, NaN -> 0x7FC0) little-endian, two zero bytes.
// The quotient is a correctly rounded float32 division (__fdiv_rn) and the
// rounding is v_rndne_f32, so the codes match numpy's bit for bit.
//
// Eight lanes share a block: lane p holds columns 4p..4p+3 of kQuantRows rows,
// all loaded (16 bytes each) before the first is needed; a wave covers 8 blocks,
// of one row where rows are that long, so its reads are 1 KiB lines and its
// writes contiguous. Blocks follow each other across rows, so that no lane idles
// at the end of a row (256 columns of one row per wave: 65536 x 64 13.2 us
// against 7.5, x 544 36.4 against 29.0, 16256 x 4128 68 against 55.5, no
// difference at multiples of 256). Bound by memory:
// 3840 x 15360 float32 weights quantized as 4096 x 16384 read and write 278 MB,
// which a copy at this card's 4.9 TB/s moves in 57 us; they take 54. (A block
// per 8 lanes by a 64-bit division of its number, four 4-byte loads and four
// IEEE divisions per lane took 82.)
#include <algorithm>

#include "q4_device.h"
#include "q4_host.h"

namespace alv {

namespace {

__device__ __forceinline__ uint32_t bf16_bits_rne(float v) {
    if (v != v) return 0x7FC0u;
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}

constexpr int kQuantRows = 4;

// max over the 8 lanes of a block (an aligned group, all active): pairs,
// quads, then the mirrored half row holds the other quad.
__device__ __forceinline__ uint32_t max8(uint32_t v) {
    v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, false));
    v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, false));
    return max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x141, 0xF, 0xF, false));
}

// kQuantRows rows from r0 on of the block that columns c0 .. c0 + 3 belong to;
// orow: bytes of an output row.
__device__ __forceinline__ void quant_rows(const float* W, int n_src, int k_src, int ldw, uint8_t* out, int N,
                                           size_t orow, int64_t r0, int c0, int part) {
    float v[kQuantRows][4];
#pragma unroll
    for (int t = 0; t < kQuantRows; ++t) {
        const float* src = W + (size_t)(r0 + t) * ldw + c0;
        if (r0 + t < n_src && c0 + 3 < k_src) {
            __builtin_memcpy(v[t], src, sizeof(v[t]));
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[t][e] = r0 + t < n_src && c0 + e < k_src ? src[e] : 0.0f;
        }
    }
#pragma unroll
    for (int t = 0; t < kQuantRows; ++t) {
        if (r0 + t >= N) break;
        // The largest magnitude by its bits: a NaN's are above infinity's.
        uint32_t mb = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) mb = max(mb, __builtin_bit_cast(uint32_t, v[t][e]) & 0x7FFFFFFFu);
        mb = max8(mb);
        float s = mb > 0x7F800000u ? __builtin_nanf("") : __fdiv_rn(__builtin_bit_cast(float, mb), 7.0f);
        if (s == 0.0f) s = 1.0f;
        // v / s rounded to an integer: v times the hardware reciprocal is
        // within 8 * 2^-22 of the quotient (|v / s| < 7.01), so it settles the
        // integer unless it lies within 2^-18 of a half; then, and for scales
        // outside the normal range (and NaN), the correctly rounded division.
        const float rs = __builtin_amdgcn_rcpf(s);
        float qf[4];
        bool near = !(s > 1e-30f && s < 1e30f);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float y = v[t][e] * rs;
            qf[e] = rintf(y);
            near |= fabsf(y - qf[e]) > 0.5f - 0x1p-18f;
        }
        if (near) {
#pragma unroll
            for (int e = 0; e < 4; ++e) qf[e] = rintf(__fdiv_rn(v[t][e], s));
        }
        uint32_t packed = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            int q = qf[e] != qf[e] ? -8 : (int)qf[e];
            q = q < -8 ? -8 : (q > 7 ? 7 : q);
            packed |= (uint32_t)(q & 0xF) << (4 * e);
        }
        // Even lanes write a dword of two lanes' codes, lane 1 the scale.
        const uint32_t next = (uint32_t)__builtin_amdgcn_mov_dpp((int)packed, 0xB1, 0xF, 0xF, false);
        const uint32_t word = part == 1 ? bf16_bits_rne(s) : packed | next << 16;
        if (part == 1 || !(part & 1))
            *reinterpret_cast<uint32_t*>(out + (size_t)(r0 + t) * orow + (size_t)(c0 >> 5) * kBlockBytes +
                                         (part == 1 ? 16 : 2 * part)) = word;
    }
}

// Row groups [0, groups) of the rows from row0 on: (group, block) pairs in one
// sequence, blocks fastest, eight lanes each.
__global__ void __launch_bounds__(256) quant_kernel(const float* W, int n_src, int k_src, int ldw, uint8_t* out,
                                                    int N, int K, int64_t row0, uint32_t groups) {
    const uint32_t nb = (uint32_t)K / 32, total = groups * nb;
    const int part = threadIdx.x & 7;
    const size_t orow = (size_t)nb * kBlockBytes;
    for (uint32_t i = blockIdx.x * 32 + (threadIdx.x >> 3); i < total; i += gridDim.x * 32) {
        const uint32_t rg = i / nb, b = i - rg * nb;
        quant_rows(W, n_src, k_src, ldw, out, N, orow, row0 + (int64_t)rg * kQuantRows, (int)(b * 32) + 4 * part, part);
    }
}

int check_quant(const float* W, int n_src, int k_src, int ldw, const void* out, int N, int K) {
    if (!W || !out) return fail(ALV_ERR_ARG, "null pointer");
    if (N < 1 || K < 32 || K % 32) return fail(ALV_ERR_ARG, "bad shape N=%d K=%d (K must be a positive multiple of 32)", N, K);
    if (n_src < 0 || k_src < 0 || n_src > N || k_src > K || ldw < k_src)
        return fail(ALV_ERR_ARG, "source %d x %d (row stride %d) does not fit the %d x %d output", n_src, k_src, ldw, N, K);
    if (reinterpret_cast<uintptr_t>(W) % 4) return fail(ALV_ERR_ALIGN, "W needs 4-byte alignment");
    if ((uint64_t)N * (uint64_t)(K / 32) * kBlockBytes >= (1ull << 40))
        return fail(ALV_ERR_RANGE, "output of %d x %d exceeds 1 TiB", N, K);
    return ALV_OK;
}

int launch_quant(const float* W, int n_src, int k_src, int ldw, uint8_t* out, int N, int K, hipStream_t s) {
    // One launch, unless its sequence would pass 2^30 pairs (K / 32 < 2^26 of them per group).
    const int64_t groups = ((int64_t)N + kQuantRows - 1) / kQuantRows, nb = K / 32, most = (1 << 30) / nb;
    for (int64_t g0 = 0; g0 < groups; g0 += most) {
        const int64_t n = std::min(most, groups - g0);
        const int grid = (int)std::min<int64_t>((n * nb + 31) / 32, 1 << 20);
        hipLaunchKernelGGL(quant_kernel, dim3(grid), dim3(256), 0, s, W, n_src, k_src, ldw, out, N, K, g0 * kQuantRows,
                           (uint32_t)n);
        if (int rc = hip_check(hipGetLastError(), "quant_kernel launch")) return rc;
    }
    return ALV_OK;
}

}  // namespace

}  // namespace alv

using namespace alv;

extern "C" int alv_quantize_q4(const float* W, int n_src, int k_src, int ldw, uint8_t* out, int N, int K,
                               void* stream) {
    if (int rc = check_quant(W, n_src, k_src, ldw, out, N, K)) return rc;
    if (reinterpret_cast<uintptr_t>(out) % 4) return fail(ALV_ERR_ALIGN, "out needs 4-byte alignment");
    return launch_quant(W, n_src, k_src, ldw, out, N, K, (hipStream_t)stream);
}

extern "C" int alv_weight_quantize(const float* W, int n_src, int k_src, int ldw, int N, int K, alv_weight_t* out,
                                   void* stream) {
    if (!out) return fail(ALV_ERR_ARG, "null output handle pointer");
    *out = nullptr;
    if (int rc = check_quant(W, n_src, k_src, ldw, W, N, K)) return rc;
    hipStream_t s = (hipStream_t)stream;
    uint8_t* tmp = nullptr;
    int rc = hip_check(hipMalloc(&tmp, (size_t)N * (K / 32) * kBlockBytes), "hipMalloc(quantized weights)");
    if (!rc) rc = launch_quant(W, n_src, k_src, ldw, tmp, N, K, s);
    // Registration tiles the combined bytes and waits for the stream, after
    // which the temporary can go.
    if (!rc) rc = alv_weight_register(tmp, N, K, out, stream);
    if (tmp) {
        const int rs = hip_check(hipStreamSynchronize(s), "hipStreamSynchronize");
        (void)hipFree(tmp);
        if (!rc) rc = rs;
    }
    if (rc && *out) {
        alv_weight_release(*out);
        *out = nullptr;
    }
    return rc;
}
