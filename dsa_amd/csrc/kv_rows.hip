// fp8 cache rows (656 bytes: 512 e4m3 latent values, four fp32 block scales,
// 64 bf16 rope values).  No reference counterpart: the reference takes a
// contiguous bf16 cache only (dsa/api.py:30-33).
//
// quantize_rows writes them from bf16 kv and k_rope.  It is bound by HBM
// (1,152 bytes read, 656 written a row) and, for the few rows of a decode
// step, by its launch: one pass, a wave per pair of rows, every load of the
// pair issued before the first use.  Lane l holds values 8 l .. 8 l + 7 of a
// row, so a 128-wide block is one 16-lane DPP row and its maximum four
// v_max_u32 row rotations; the rope dwords of both rows are one load.  Measured
// for 8,192 rows (14.8 MB): kernel 4.3 us, the call 8.0 us, against 97 us as
// tensor code (17 launches, about 160 MB moved).
//
// expand_rows is the reverse, for calls that gather every cache row many times
// (prefill chunks): each row becomes the bf16 row the attention kernels would
// make of it, kv[d] = bf16(fp32(e4m3[d]) * scale[d / 128]), in the contiguous
// [B, L] layout of the kernels that read bf16 rows.  Bound by HBM (656 bytes
// read, 1,152 written a row): four rows per wave and iteration, every load of
// the four issued first.  With it a 2,048-query chunk of 128 heads over 32,768
// rows takes 986 us, against 1,780 us when every gathered slot is expanded in
// LDS by the narrow kernels.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "host_entry.h"
#include "kernels.h"

namespace dsa {
namespace {

constexpr int kThreads = 256;
constexpr int kRow = 656, kScaleOff = 512, kRopeOff = 528;
// 16 workgroups of four waves on each of 256 CUs: rows beyond 2 * 16384 are
// further iterations of the same waves.
constexpr int kMaxGrid = 4096;

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t max_u16x2(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t,
                              __builtin_elementwise_max(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
}

// max over the 16 lanes of this lane's DPP row.
__device__ __forceinline__ uint32_t row16_max(uint32_t v) {
    v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x128, 0xf, 0xf, true));  // row_ror:8
    v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x124, 0xf, 0xf, true));
    v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x122, 0xf, 0xf, true));
    return max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x121, 0xf, 0xf, true));
}

// e4m3 code of v clamped to +-448, NaN kept (0x7f with v's sign): the values
// of a block that holds an infinity or a NaN.
__device__ __forceinline__ uint32_t code_special(float v) {
    if (v != v) return 0x7fu | (__float_as_uint(v) >> 31 << 7);
    return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(fminf(fmaxf(v, -448.f), 448.f), 0.f, 0, false) & 0xffu;
}

// 2^k as tensor code computes it on the GPU, 2.0f to the power k: exact for
// |k| <= kExactPow2 (block maxima from about 0.01 to 10^7, any ordinary cache),
// beyond that off by some units in the last place for some k, where the rows
// hold what powf gives and the codes its quotients.
constexpr int kExactPow2 = 15;
__device__ __forceinline__ bool exact_pow2(int k) { return k >= -kExactPow2 && k <= kExactPow2; }
__device__ __forceinline__ float pow2_scale(int k) {
    return __builtin_expect(exact_pow2(k), 1) ? ldexpf(1.f, k) : powf(2.f, (float)k);
}

// Codes and scale of this lane's eight values; the 16 lanes of a block agree
// on the scale (the quotient by 448 is a product with its rounded reciprocal,
// as tensor code divides by a scalar).  |value / scale| stays at or below 448
// up to rounding, and e4m3 rounds everything below 464 to 448 or less, so a
// finite block needs no clamp.  Dividing by a power of two is an exponent
// shift, exact unless the result is far below the smallest e4m3 value (code 0
// either way).
template <bool POW2>
__device__ __forceinline__ uint2 encode8(const uint4& v, float& scale) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    uint32_t m = 0;  // |x| in bf16 orders like its 15 bits; a NaN's exceed infinity's
#pragma unroll
    for (int i = 0; i < 4; ++i) m = max_u16x2(m, w[i] & 0x7fff7fffu);
    m = row16_max(max(m & 0xffffu, m >> 16));
    const float amax = __uint_as_float(m << 16);
    scale = amax > 0.f ? amax * (1.f / 448.f) : 1.f;
    int k = 0;
    bool shift = POW2;  // the scale is exactly 2^k
    if constexpr (POW2) {
        const float mant = __builtin_amdgcn_frexp_mantf(scale);
        k = __builtin_amdgcn_frexp_expf(scale) - (mant == 0.5f ? 1 : 0);
        scale = pow2_scale(k);
        shift = exact_pow2(k);
    }
    float f[8], x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] = __uint_as_float(i & 1 ? w[i >> 1] & 0xffff0000u : w[i >> 1] << 16);
    if (__builtin_expect(shift, POW2)) {
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = ldexpf(f[i], -k);
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = f[i] / scale;
    }
    uint2 c;
    if (__builtin_expect(m >= 0x7f80u || !(scale > 0.f && scale < INFINITY), 0)) {
        c.x = code_special(x[0]) | code_special(x[1]) << 8 | code_special(x[2]) << 16 | code_special(x[3]) << 24;
        c.y = code_special(x[4]) | code_special(x[5]) << 8 | code_special(x[6]) << 16 | code_special(x[7]) << 24;
    } else {
        c.x = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(
            x[2], x[3], __builtin_amdgcn_cvt_pk_fp8_f32(x[0], x[1], 0, false), true);
        c.y = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(
            x[6], x[7], __builtin_amdgcn_cvt_pk_fp8_f32(x[4], x[5], 0, false), true);
    }
    return c;
}

template <bool POW2>
__global__ __launch_bounds__(kThreads) void quantize_rows_kernel(const uint16_t* __restrict__ kv,
                                                                 const uint16_t* __restrict__ k_rope,
                                                                 uint8_t* __restrict__ out, int64_t rows) {
    const int lane = threadIdx.x & 63;
    const int64_t wave = (int64_t)blockIdx.x * (kThreads / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t waves = (int64_t)gridDim.x * (kThreads / 64);
    const uint4* src = reinterpret_cast<const uint4*>(kv);
    const uint32_t* rope = reinterpret_cast<const uint32_t*>(k_rope);
    for (int64_t r = 2 * wave; r < rows; r += 2 * waves) {
        const bool two = r + 1 < rows;  // uniform
        const uint4 v0 = src[r * 64 + lane];
        const uint4 v1 = src[(two ? r + 1 : r) * 64 + lane];
        const bool has_rope = lane < 32 || two;
        const uint32_t rp = has_rope ? rope[r * 32 + lane] : 0u;
        float s0, s1;
        const uint2 c0 = encode8<POW2>(v0, s0), c1 = encode8<POW2>(v1, s1);
        uint8_t* o0 = out + r * kRow;
        *reinterpret_cast<uint2*>(o0 + 8 * lane) = c0;
        if ((lane & 15) == 0) *reinterpret_cast<float*>(o0 + kScaleOff + (lane >> 2)) = s0;
        if (has_rope) *reinterpret_cast<uint32_t*>(o0 + (lane >> 5) * kRow + kRopeOff + 4 * (lane & 31)) = rp;
        if (two) {
            uint8_t* o1 = o0 + kRow;
            *reinterpret_cast<uint2*>(o1 + 8 * lane) = c1;
            if ((lane & 15) == 0) *reinterpret_cast<float*>(o1 + kScaleOff + (lane >> 2)) = s1;
        }
    }
}

constexpr int kExpand = 4;  // rows per wave and iteration

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Rows [0, rows) of the logical [B, L] cache; with a block table, logical row
// s of batch b is pool row table[b * max_blocks + s / block_size] * block_size
// + s % block_size, and a row behind an entry outside [0, num_blocks) becomes
// zeros (its slots are masked; kernels gather row 0 of a batch for them).
__global__ __launch_bounds__(kThreads) void expand_rows_kernel(const uint8_t* __restrict__ in,
                                                               uint16_t* __restrict__ kv,
                                                               uint16_t* __restrict__ k_rope, int64_t rows, int L,
                                                               BlockTable bt) {
    const int lane = threadIdx.x & 63;
    const int64_t wave = (int64_t)blockIdx.x * (kThreads / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t waves = (int64_t)gridDim.x * (kThreads / 64);
    for (int64_t r0 = kExpand * wave; r0 < rows; r0 += kExpand * waves) {
        uint2 code[kExpand];
        float scale[kExpand];
        uint32_t rope[kExpand];
        bool live[kExpand];
#pragma unroll
        for (int i = 0; i < kExpand; ++i) {  // uniform per row
            const int64_t r = min(r0 + i, rows - 1);
            int64_t phys = r;
            live[i] = true;
            if (bt.table != nullptr) {
                const int64_t b = r / L;
                const int s = (int)(r - b * L);
                const int blk = bt.table[b * bt.max_blocks + s / bt.block_size];
                live[i] = (uint32_t)blk < (uint32_t)bt.num_blocks;
                phys = (int64_t)(live[i] ? blk : 0) * bt.block_size + s % bt.block_size;
            }
            const uint8_t* row = in + phys * kRow;
            code[i] = *reinterpret_cast<const uint2*>(row + 8 * lane);
            scale[i] = *reinterpret_cast<const float*>(row + kScaleOff + 4 * (lane >> 4));
            rope[i] = *reinterpret_cast<const uint32_t*>(row + kRopeOff + 4 * (lane & 31));
        }
#pragma unroll
        for (int i = 0; i < kExpand; ++i) {
            if (r0 + i >= rows) break;
            bf16x8 o;
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                const int w = (int)(d ? code[i].y : code[i].x);
                const auto lo = __builtin_amdgcn_cvt_pk_f32_fp8(w, false);
                const auto hi = __builtin_amdgcn_cvt_pk_f32_fp8(w, true);
                o[4 * d + 0] = (__bf16)(lo[0] * scale[i]);
                o[4 * d + 1] = (__bf16)(lo[1] * scale[i]);
                o[4 * d + 2] = (__bf16)(hi[0] * scale[i]);
                o[4 * d + 3] = (__bf16)(hi[1] * scale[i]);
            }
            uint4 v = __builtin_bit_cast(uint4, o);
            if (!live[i]) v = uint4{0, 0, 0, 0}, rope[i] = 0;
            reinterpret_cast<uint4*>(kv)[(r0 + i) * 64 + lane] = v;
            if (lane < 32) reinterpret_cast<uint32_t*>(k_rope)[(r0 + i) * 32 + lane] = rope[i];
        }
    }
}

int64_t grid_for(int64_t rows, int rows_per_wave) {
    const int64_t per = (int64_t)rows_per_wave * (kThreads / 64);
    const int64_t want = (rows + per - 1) / per;
    return want < kMaxGrid ? want : kMaxGrid;
}

}  // namespace
}  // namespace dsa

extern "C" int dsa_kv_expand_rows(const uint8_t* in, uint16_t* kv, uint16_t* k_rope, int B, int L,
                                  const int32_t* block_table, int max_blocks, int block_size, int num_blocks,
                                  void* stream_) {
    const hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (!in || !kv || !k_rope) return dsa::set_error(-1, "%s", "NULL pointer argument");
    if (B <= 0 || L <= 0) return dsa::set_error(-1, "%s", "B and L must be positive");
    if ((((uintptr_t)in | (uintptr_t)kv) & 15) || (((uintptr_t)k_rope | (uintptr_t)block_table) & 3))
        return dsa::set_error(-1, "%s", "rows and kv must be 16-byte, k_rope and block_table 4-byte aligned");
    if (block_table && (max_blocks <= 0 || block_size <= 0 || num_blocks <= 0 || (int64_t)max_blocks * block_size != L))
        return dsa::set_error(-1, "%s", "L must equal max_blocks * block_size, num_blocks be positive");
    const int64_t rows = (int64_t)B * L;
    const dsa::BlockTable bt{block_table, max_blocks, block_size, num_blocks, 1};
    hipLaunchKernelGGL(dsa::expand_rows_kernel, dim3((unsigned)dsa::grid_for(rows, dsa::kExpand)),
                       dim3(dsa::kThreads), 0, stream, in, kv, k_rope, rows, L, bt);
    const int rc = (int)hipGetLastError();
    if (rc) return dsa::set_error(rc, "expand launch: %s", hipGetErrorString((hipError_t)rc));
    return 0;
}

extern "C" int dsa_kv_quantize_rows(const uint16_t* kv, const uint16_t* k_rope, uint8_t* out, int64_t rows, int pow2,
                                    void* stream_) {
    const hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (!kv || !k_rope || !out) return dsa::set_error(-1, "%s", "NULL pointer argument");
    if (rows <= 0) return dsa::set_error(-1, "%s", "rows must be positive");
    if ((((uintptr_t)kv | (uintptr_t)out) & 15) || ((uintptr_t)k_rope & 3))
        return dsa::set_error(-1, "%s", "kv and out must be 16-byte, k_rope 4-byte aligned");
    const dim3 grid((unsigned)dsa::grid_for(rows, 2));
    if (pow2)
        hipLaunchKernelGGL((dsa::quantize_rows_kernel<true>), grid, dim3(dsa::kThreads), 0, stream, kv, k_rope, out,
                           rows);
    else
        hipLaunchKernelGGL((dsa::quantize_rows_kernel<false>), grid, dim3(dsa::kThreads), 0, stream, kv, k_rope, out,
                           rows);
    const int rc = (int)hipGetLastError();
    if (rc) return dsa::set_error(rc, "quantize launch: %s", hipGetErrorString((hipError_t)rc));
    return 0;
}
