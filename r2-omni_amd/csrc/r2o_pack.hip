// Quantise/pack, gather and Recent-FP append/shift kernels for gfx950.
//
// Bit-exactness with the reference's torch CPU quantisers (compact_int4_key.py:83-110,
// quantization.py:19-50, int2_reference.py:96-151): IEEE fp32 division (__fdiv_rn), round half
// to even (__builtin_rintf -> v_rndne_f32), no contraction (the file is built with
// -ffp-contract=off), fp32 step quantisation with fp16-RNE storage of the step.  Where many values share a
// divisor its reciprocal is kept and r2o_div_by gives the same correctly rounded quotients.
#include <initializer_list>

#include "r2o_common.hpp"

namespace {

constexpr float kEps = 1.0e-6f;

// --------------------------------------------------------------------------------- values
// INT4 (per-token symmetric) and INT2 (per-token-group affine) values.  A row is 16 lanes of 8 channels
// (one 16-byte load), so a wave takes 4 rows per load and kVRows loads in flight; the reductions over a
// row or group are in-lane maxima and at most 4 DPP exchanges, and a lane's codes leave as one 4- or
// 2-byte store (256 or 128 contiguous bytes a wave).  VALU issue and the stream bound it about equally.
// Measured, bf16: INT2 of 131k tokens x 8 heads, group 128, 264 -> 70 us (1.15 -> 4.3 TB/s); of 23k x 4,
// group 32, 28 -> 10.9 us; INT4 of 27k x 4, 19.3 -> 10.6 us.  Before, one wave took a row at 2 channels a
// lane: 6 LDS permutes per row, two ~12-instruction divisions per element and byte stores.
// The codes are integers after RN(x / s) (+ z): the quotient is r2o_div_by's, and adding 1.5 * 2^23
// rounds it half to even into the low mantissa bits, from which v_alignbit collects the codes.
// Rows whose range is near or past the top of fp32 (kWideRange; infinities) take plain divisions.
constexpr int kVRows = 4;                              // rows per lane
constexpr int kVBlockRows = 4 * 4 * kVRows;            // per 256-thread block
constexpr float kRoundMagic = 12582912.f;              // 1.5 * 2^23
constexpr float kWideRange = 1e30f;

struct ValuePack {
    const uint16_t* src;
    int64_t src_tokens;
    const int64_t* index;  // nullable: token i is source row i
    int64_t n, dst_start;
    uint8_t* packed;
    void* scale;    // INT4: f32; INT2: fp16
    uint8_t* zero;  // INT2 only
    int64_t capacity;
    int group;      // INT2 only
};

// The 8 codes of a lane, BITS bits each, from the 8 integers rounded into the low mantissa bits of u.
template <int BITS>
__device__ __forceinline__ uint32_t collect_codes(const float (&u)[8]) {
    uint32_t w = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) w = __builtin_amdgcn_alignbit(__float_as_uint(u[i]), w, BITS);
    return BITS == 4 ? w : w >> 16;
}

// max (or, negated, min) over the 2, 4, 8 or 16 lanes that share a group of `lanes` lanes.
template <int BITS>
__device__ __forceinline__ float lanes_max(float v, int lanes) {
    v = fmaxf(v, r2o_lane_xor<1>(v));
    v = fmaxf(v, r2o_lane_xor<2>(v));
    if (BITS == 4 || lanes >= 8) v = fmaxf(v, r2o_lane_xor<4>(v));
    if (BITS == 4 || lanes >= 16) v = fmaxf(v, r2o_lane_xor<8>(v));
    return v;
}

template <int BITS, bool WIDE>
__device__ __forceinline__ uint32_t value_codes(const float (&x)[8], float s, float y, float z) {
    float u[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float q = WIDE ? __fdiv_rn(x[i], s) : r2o_div_by(x[i], s, y);
        // v_med3 of a NaN is the smaller of the other two, as fminf(fmaxf(NaN, lo), hi)
        u[i] = (BITS == 4 ? __builtin_amdgcn_fmed3f(q, -7.f, 7.f) : __builtin_amdgcn_fmed3f(q + z, 0.f, 3.f)) + kRoundMagic;
    }
    return collect_codes<BITS>(u);
}

// Element j of v for a lane index j (three selects; an array would be indexed through memory).
__device__ __forceinline__ float of_lane(int j, r2o_f4 v) {
    const float lo = (j & 1) ? v.y : v.x, hi = (j & 1) ? v.w : v.z;
    return (j & 2) ? hi : lo;
}

// Steps, zero points and codes of a lane's rows.  Lane j of a quad forms the step, its reciprocal and the
// zero point of row j for the quad's group (a quad never crosses a group), and each row reads its lane's.
template <int BITS, int DT, bool VEC, bool WIDE>
__device__ __forceinline__ void store_values(const ValuePack& a, int64_t h, int64_t i0, int c8, int glanes,
                                             const r2o_u4 (&raw)[kVRows], r2o_f4 range, r2o_f4 mn) {
    static_assert(kVRows == 4, "one row per lane of a quad");
    constexpr float kSteps = BITS == 4 ? 7.f : 3.f;
    const int j = c8 & 3;
    const float my_range = of_lane(j, range);
    const float s = fmaxf(WIDE ? __fdiv_rn(my_range, kSteps) : r2o_div_by(my_range, kSteps, 1.f / kSteps), kEps);
    const float y = WIDE ? 0.f : __fdiv_rn(1.f, s);
    float z = 0.f;
    if constexpr (BITS == 2) {
        const float my_mn = of_lane(j, mn);
        z = fminf(fmaxf(__builtin_rintf(WIDE ? __fdiv_rn(-my_mn, s) : r2o_div_by(-my_mn, s, y)), 0.f), 3.f);
    }
    const int64_t dst0 = h * a.capacity + a.dst_start + i0;  // row k of the lane is dst0 + 4 k
    if ((c8 & (glanes - 1)) < 4 && i0 + 4 * j < a.n) {
        if constexpr (BITS == 4) {
            reinterpret_cast<float*>(a.scale)[dst0 + 4 * j] = s;
        } else {
            const int64_t e = (dst0 + 4 * j) * (16 / glanes) + c8 / glanes;
            reinterpret_cast<uint16_t*>(a.scale)[e] = (uint16_t)r2o_f32_to_f16(s);
            a.zero[e] = (uint8_t)z;
        }
    }
    uint32_t codes[kVRows];
    auto row = [&](int k, float sk, float yk, float zk) {
        float x[8];
        r2o_unpack8<DT>(raw[k], x);
        codes[k] = value_codes<BITS, WIDE>(x, sk, yk, zk);
    };
    row(0, r2o_dpp<0x00>(s), r2o_dpp<0x00>(y), r2o_dpp<0x00>(z));
    row(1, r2o_dpp<0x55>(s), r2o_dpp<0x55>(y), r2o_dpp<0x55>(z));
    row(2, r2o_dpp<0xAA>(s), r2o_dpp<0xAA>(y), r2o_dpp<0xAA>(z));
    row(3, r2o_dpp<0xFF>(s), r2o_dpp<0xFF>(y), r2o_dpp<0xFF>(z));
    uint8_t* p = a.packed + dst0 * (16 * BITS) + BITS * c8;
#pragma unroll
    for (int k = 0; k < kVRows; ++k, p += 4 * 16 * BITS) {
        if (i0 + 4 * k >= a.n) break;
        if constexpr (!VEC) {
#pragma unroll
            for (int b = 0; b < BITS; ++b) p[b] = (uint8_t)(codes[k] >> (8 * b));
        } else if constexpr (BITS == 4) {
            *reinterpret_cast<uint32_t*>(p) = codes[k];
        } else {
            *reinterpret_cast<uint16_t*>(p) = (uint16_t)codes[k];
        }
    }
}

template <int BITS, int DT, bool VEC>
__device__ __forceinline__ void pack_values(const ValuePack& a, int64_t block, int64_t h) {
    const int lane = threadIdx.x & 63, c8 = lane & 15;
    const int64_t i0 = (block * 4 + (threadIdx.x >> 6)) * (4 * kVRows) + (lane >> 4);
    // every load first: the rows' indices (clamped to the last row, branch-free), then the rows
    int64_t rows[kVRows];
#pragma unroll
    for (int k = 0; k < kVRows; ++k) {
        const int64_t i = min(i0 + 4 * k, a.n - 1);
        rows[k] = a.index ? r2o_ldg(a.index + i) : i;
    }
    r2o_u4 raw[kVRows];
#pragma unroll
    for (int k = 0; k < kVRows; ++k) raw[k] = r2o_load8<VEC>(a.src + (h * a.src_tokens + rows[k]) * 128 + 8 * c8);
    const int glanes = BITS == 4 ? 16 : a.group / 8;  // lanes per group
    r2o_f4 range, mn;
#pragma unroll
    for (int k = 0; k < kVRows; ++k) {
        float x[8];
        r2o_unpack8<DT>(raw[k], x);
        mn[k] = 0.f;
        if constexpr (BITS == 4) {
            float mx = fabsf(x[0]);
#pragma unroll
            for (int i = 1; i < 8; ++i) mx = fmaxf(mx, fabsf(x[i]));
            range[k] = lanes_max<4>(mx, 16);
        } else {
            float lo = -x[0], hi = x[0];
#pragma unroll
            for (int i = 1; i < 8; ++i) {
                lo = fmaxf(lo, -x[i]);
                hi = fmaxf(hi, x[i]);
            }
            lo = lanes_max<2>(lo, glanes);
            hi = lanes_max<2>(hi, glanes);
            mn[k] = fminf(-lo, 0.f);
            range[k] = fmaxf(hi, 0.f) - mn[k];
        }
    }
    float most = range[0];
#pragma unroll
    for (int k = 1; k < kVRows; ++k) most = fmaxf(most, range[k]);
    if (__any(most > kWideRange)) store_values<BITS, DT, VEC, true>(a, h, i0, c8, glanes, raw, range, mn);
    else store_values<BITS, DT, VEC, false>(a, h, i0, c8, glanes, raw, range, mn);
}

template <int BITS, int DT, bool VEC>
__global__ __launch_bounds__(256) void pack_values_kernel(ValuePack a) {
    pack_values<BITS, DT, VEC>(a, blockIdx.x, blockIdx.y);
}

template <int BITS>
void launch_pack_values(const ValuePack& a, int64_t dtype, int64_t hkv, hipStream_t stream) {
    const dim3 grid((unsigned)((a.n + kVBlockRows - 1) / kVBlockRows), (unsigned)hkv);
    const bool vec = reinterpret_cast<uintptr_t>(a.src) % 16 == 0 && reinterpret_cast<uintptr_t>(a.packed) % 4 == 0;
    if (dtype == 0) {
        if (vec) hipLaunchKernelGGL((pack_values_kernel<BITS, 0, true>), grid, dim3(256), 0, stream, a);
        else hipLaunchKernelGGL((pack_values_kernel<BITS, 0, false>), grid, dim3(256), 0, stream, a);
    } else {
        if (vec) hipLaunchKernelGGL((pack_values_kernel<BITS, 1, true>), grid, dim3(256), 0, stream, a);
        else hipLaunchKernelGGL((pack_values_kernel<BITS, 1, false>), grid, dim3(256), 0, stream, a);
    }
}

// ------------------------------------------------------------------------------------ keys
// INT4 (per-channel affine over min(min x, 0) .. max(max x, 0)) and INT2 (OScaR form, int2_reference.py:
// 159-214, clip ratio 1: block min / max without 0, scale = range / 3, inv = (1 / range) * 3 as torch's
// ``3.0 / t``, zero = rne(-min * inv), offset = -zero * scale; constant channels keep scale 0 and offset =
// min) keys over superblocks of SB tokens.
//
// A wave takes 32 tokens of a superblock: lane (r, c8) holds channels 8 c8 .. 8 c8 + 7 of tokens 4 k + r in
// registers from one 16-byte load each, all 8 in flight at once.  The channel ranges fold over the lane's
// tokens, then over r by permlane swaps that also scatter them, so that lane (r, c8) ends with channels
// 8 c8 + 2 r and + 1 and forms their step, zero point and reciprocal once; the waves of a larger
// superblock meet in LDS.  Every lane reads the 8 channels it needs back and the codes leave as one store
// per token (256 or 128 contiguous bytes a wave).  Each key row is read once, and the stream bounds it.
// Measured, bf16: INT2 of 131k tokens x 8 heads, SB 128, 218 -> 61 us (5.1 TB/s); INT4 of 59k x 4, SB 32,
// 35 -> 20 us (4.0 TB/s); INT4 of a flush (128 tokens and a partial superblock x 4 heads) 20.6 -> 6.0 us.
// Before, a wave took a superblock at 2 or 4 channels a lane, token after token, reading it twice.
struct KeyPack {
    const uint16_t* src;
    int64_t src_tokens;
    const int64_t* index;  // nullable: token i is source row i
    int64_t n, tail, dst_start;
    uint8_t* packed;
    uint16_t* scale;
    void* zero;            // INT4: u8 zero points; INT2: fp16 offsets
    uint32_t* operands;    // nullable
    int64_t capacity, superblocks;
};

constexpr int kKeyWaves = 4;
constexpr int kKeyBlockTokens = 32 * kKeyWaves;

struct KeyLds {  // per wave: one value per channel
    float step[kKeyWaves][128];  // INT4: step; INT2: scale
    float mul[kKeyWaves][128];   // INT4: RN(1 / step); INT2: inv
    float zero[kKeyWaves][128];  // zero point
    float off[kKeyWaves][128];   // INT2: offset
};

// (m over the 4 lanes that share c8, for channel pairs) from 8 per-lane channel values: lane (r, c8) gets
// channels 8 c8 + 2 r and + 1.
__device__ __forceinline__ void scatter_max(const float (&m)[8], float& a, float& b) {
    float h[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // lanes below 32 keep channels 0 .. 3, lanes above them 4 .. 7
        const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(m[i]), __float_as_uint(m[i + 4]), false, false);
        h[i] = fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1]));
    }
    const auto s0 = __builtin_amdgcn_permlane16_swap(__float_as_uint(h[0]), __float_as_uint(h[2]), false, false);
    const auto s1 = __builtin_amdgcn_permlane16_swap(__float_as_uint(h[1]), __float_as_uint(h[3]), false, false);
    a = fmaxf(__uint_as_float(s0[0]), __uint_as_float(s0[1]));
    b = fmaxf(__uint_as_float(s1[0]), __uint_as_float(s1[1]));
}

__device__ __forceinline__ void read8(const float* p, float (&x)[8]) {
    const r2o_f4 lo = reinterpret_cast<const r2o_f4*>(p)[0], hi = reinterpret_cast<const r2o_f4*>(p)[1];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        x[i] = lo[i];
        x[i + 4] = hi[i];
    }
}

// Old metadata of a partial tail superblock for channels 8 c8 ..: what its codes dequantise with.
template <int BITS>
__device__ __forceinline__ void tail_metadata(const KeyPack& a, int64_t meta_row, int c8, float (&s)[8], float (&z)[8]) {
    const int64_t m = meta_row * 128 + 8 * c8;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        s[i] = r2o_f16_to_f32(a.scale[m + i]);
        z[i] = BITS == 4 ? (float)reinterpret_cast<const uint8_t*>(a.zero)[m + i]
                         : r2o_f16_to_f32(reinterpret_cast<const uint16_t*>(a.zero)[m + i]);
    }
}

// The 8 channels of a tail position, dequantised and rounded to the row dtype (compact_int4_key.py:215-216,
// compact_int2_key.py:114-121).
template <int BITS, int DT, bool VEC>
__device__ __forceinline__ r2o_u4 tail_row(const uint8_t* code, const float (&s)[8], const float (&z)[8]) {
    uint32_t w = 0;
    if constexpr (!VEC) {
#pragma unroll
        for (int b = 0; b < BITS; ++b) w |= (uint32_t)code[b] << (8 * b);
    } else {
        w = BITS == 4 ? *reinterpret_cast<const uint32_t*>(code) : *reinterpret_cast<const uint16_t*>(code);
    }
    r2o_u4 out = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float c = (float)((w >> (i * BITS)) & ((1 << BITS) - 1));
        const float x = BITS == 4 ? __fmul_rn(__fsub_rn(c, z[i]), s[i]) : __fadd_rn(__fmul_rn(c, s[i]), z[i]);
        out[i >> 1] |= (DT == 0 ? r2o_f32_to_bf16(x) : r2o_f32_to_f16(x)) << (16 * (i & 1));
    }
    return out;
}

// Codes of the wave's tokens own + 4 k + r < count of its superblock, from the channels' values in LDS.
template <int BITS, int DT, bool VEC, bool WIDE>
__device__ __forceinline__ void store_key_codes(const KeyPack& a, const KeyLds& lds, int wave, int64_t row0, int own,
                                                int count, int r, int c8, const r2o_u4 (&raw)[8]) {
    float step[8], mul[8], zero[8];
    if constexpr (BITS == 4) read8(lds.step[wave] + 8 * c8, step);
    read8(lds.mul[wave] + 8 * c8, mul);
    read8(lds.zero[wave] + 8 * c8, zero);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        float x[8], u[8];
        r2o_unpack8<DT>(raw[k], x);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            float q;  // v_med3 of a NaN is the smaller of the other two, as fminf(fmaxf(NaN, lo), hi)
            if constexpr (BITS == 2) q = __fmul_rn(x[i], mul[i]);
            else q = WIDE ? __fdiv_rn(x[i], step[i]) : r2o_div_by(x[i], step[i], mul[i]);
            u[i] = __builtin_amdgcn_fmed3f(q + zero[i], 0.f, BITS == 4 ? 15.f : 3.f) + kRoundMagic;
        }
        const uint32_t codes = collect_codes<BITS>(u);
        if (own + 4 * k + r >= count) break;
        uint8_t* p = a.packed + (row0 + own + 4 * k + r) * (16 * BITS) + BITS * c8;
        if constexpr (!VEC) {
#pragma unroll
            for (int b = 0; b < BITS; ++b) p[b] = (uint8_t)(codes >> (8 * b));
        } else if constexpr (BITS == 4) {
            *reinterpret_cast<uint32_t*>(p) = codes;
        } else {
            *reinterpret_cast<uint16_t*>(p) = (uint16_t)codes;
        }
    }
}

// Superblock metadata and QK MFMA operands (layout in r2o_sspa.h), by one wave.
template <int BITS, bool VEC>
__device__ __forceinline__ void store_key_metadata(const KeyPack& a, const KeyLds& lds, int wave, int64_t meta_row) {
    const int lane = threadIdx.x & 63;
    const float* step = lds.step[wave];
    const float* zero = BITS == 4 ? lds.zero[wave] : lds.off[wave];
    const uint32_t h0 = r2o_f32_to_f16(step[2 * lane]), h1 = r2o_f32_to_f16(step[2 * lane + 1]);
    const float z0 = zero[2 * lane], z1 = zero[2 * lane + 1];
    uint16_t* srow = a.scale + meta_row * 128 + 2 * lane;
    if constexpr (VEC) {
        *reinterpret_cast<uint32_t*>(srow) = h0 | (h1 << 16);
    } else {
        srow[0] = (uint16_t)h0;
        srow[1] = (uint16_t)h1;
    }
    if constexpr (BITS == 4) {
        uint8_t* zrow = reinterpret_cast<uint8_t*>(a.zero) + meta_row * 128 + 2 * lane;
        zrow[0] = (uint8_t)z0;
        zrow[1] = (uint8_t)z1;
    } else {
        uint16_t* zrow = reinterpret_cast<uint16_t*>(a.zero) + meta_row * 128 + 2 * lane;
        zrow[0] = (uint16_t)r2o_f32_to_f16(z0);
        zrow[1] = (uint16_t)r2o_f32_to_f16(z1);
    }
    if (!a.operands) return;
    const int g = lane >> 4, j = (lane >> 2) & 3, u = lane & 3;
    uint32_t* orow = a.operands + meta_row * 128 + g * 32 + 4 * j + u;
    if constexpr (BITS == 4) {
        const int c = 32 * g + 8 * j + u;  // pair (c, c + 4); odd u: read in place 4 bits up, 1024 + 16 code
        const float k = (u & 1) ? 0.0625f : 1.f;
        const uint32_t s0 = r2o_f32_to_f16(step[c]), s1 = r2o_f32_to_f16(step[c + 4]);
        const uint32_t shift = (u & 1) ? 4 : 0;
        orow[0] = r2o_f32_to_f16(r2o_f16_to_f32(s0) * k) | (r2o_f32_to_f16(r2o_f16_to_f32(s1) * k) << 16);
        orow[16] = (0xE400u | ((uint32_t)zero[c] << shift)) | ((0xE400u | ((uint32_t)zero[c + 4] << shift)) << 16);
    } else {
        const int c = 32 * g + 16 * (j >> 1) + 4 * (j & 1) + u;  // pair (c, c + 8); crumb u enters x 4^u
        const float k = u == 0 ? 1.f : (u == 1 ? 0.25f : (u == 2 ? 0.0625f : 0.015625f));
        const uint32_t s0 = r2o_f32_to_f16(step[c]), s1 = r2o_f32_to_f16(step[c + 8]);
        orow[0] = r2o_f32_to_f16(r2o_f16_to_f32(s0) * k) | (r2o_f32_to_f16(r2o_f16_to_f32(s1) * k) << 16);
        orow[16] = r2o_f32_to_f16(zero[c]) | (r2o_f32_to_f16(zero[c + 8]) << 16);
    }
}

// Tokens [128 block, 128 block + 128) of the destination range, by a 256-thread block (every thread calls
// this: the waves of a superblock of 64 or 128 tokens meet at a barrier).  Every read of old codes and
// metadata precedes the first store of a superblock: a wave's own reads before its own stores, the other
// waves' before the barrier.
template <int BITS, int SB, int DT, bool VEC>
__device__ __forceinline__ void pack_keys(const KeyPack& a, int64_t block, int64_t h, KeyLds& lds) {
    constexpr int kSbWaves = SB / 32;  // waves of a superblock
    const int lane = threadIdx.x & 63, c8 = lane & 15, r = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lead = wave & ~(kSbWaves - 1);
    const int own = 32 * (wave - lead);                                      // the wave's first token in it
    const int64_t first = block * kKeyBlockTokens + 32 * lead;               // relative to dst_start
    const int count = (int)min((int64_t)SB, a.tail + a.n - first);           // tokens of the superblock
    const int64_t block_row = (a.dst_start + first) / SB;
    r2o_u4 raw[8];
    float a0 = 0.f, a1 = 0.f, b0 = 0.f, b1 = 0.f;  // -min and max of channels 8 c8 + 2 r, + 1
    if (count > 0) {
        // tokens past the end read the superblock's last one again, which no range notices
        if (first >= a.tail) {
            int64_t rows[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int64_t i = first + min(own + 4 * k + r, count - 1) - a.tail;
                rows[k] = a.index ? r2o_ldg(a.index + i) : i;
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) raw[k] = r2o_load8<VEC>(a.src + (h * a.src_tokens + rows[k]) * 128 + 8 * c8);
        } else {  // the one superblock that holds tail positions
            float ts[8], tz[8];
            tail_metadata<BITS>(a, h * a.superblocks + block_row, c8, ts, tz);
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int64_t pos = first + min(own + 4 * k + r, count - 1), i = pos - a.tail;
                const uint8_t* code = a.packed + (h * a.capacity + a.dst_start + pos) * (16 * BITS) + BITS * c8;
                r2o_u4 v;
                if (i < 0) v = tail_row<BITS, DT, VEC>(code, ts, tz);
                else v = r2o_load8<VEC>(a.src + (h * a.src_tokens + (a.index ? r2o_ldg(a.index + i) : i)) * 128 + 8 * c8);
                raw[k] = v;
            }
        }
        float lo[8], hi[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) lo[i] = hi[i] = BITS == 4 ? 0.f : -INFINITY;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            float x[8];
            r2o_unpack8<DT>(raw[k], x);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                lo[i] = fmaxf(lo[i], -x[i]);
                hi[i] = fmaxf(hi[i], x[i]);
            }
        }
        scatter_max(lo, a0, a1);
        scatter_max(hi, b0, b1);
    }
    const int ch = 8 * c8 + 2 * r;
    if constexpr (kSbWaves > 1) {
        if (count > 0) {
            *reinterpret_cast<float2*>(&lds.step[wave][ch]) = make_float2(a0, a1);
            *reinterpret_cast<float2*>(&lds.mul[wave][ch]) = make_float2(b0, b1);
        }
        __syncthreads();
        if (count > 0) {
#pragma unroll
            for (int w = 1; w < kSbWaves; ++w) {
                const int o = lead + ((wave + w) & (kSbWaves - 1));
                const float2 lo = *reinterpret_cast<const float2*>(&lds.step[o][ch]);
                const float2 hi = *reinterpret_cast<const float2*>(&lds.mul[o][ch]);
                a0 = fmaxf(a0, lo.x);
                a1 = fmaxf(a1, lo.y);
                b0 = fmaxf(b0, hi.x);
                b1 = fmaxf(b1, hi.y);
            }
        }
        __syncthreads();  // the ranges are read: the same LDS takes the metadata
    }
    if (count <= 0) return;
    float step[2], mul[2], zero[2], off[2];
    bool wide = false;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const float mn = -(e ? a1 : a0), mx = e ? b1 : b0;
        const float range = mx - mn;
        if constexpr (BITS == 4) {
            wide |= range > kWideRange;
            step[e] = fmaxf(__fdiv_rn(range, 15.f), kEps);
            mul[e] = __fdiv_rn(1.f, step[e]);
            zero[e] = fminf(fmaxf(__builtin_rintf(__fdiv_rn(-mn, step[e])), 0.f), 15.f);
            off[e] = 0.f;
        } else {
            const bool nonconst = range > 0.f;
            step[e] = nonconst ? __fdiv_rn(range, 3.f) : 0.f;
            mul[e] = nonconst ? __fmul_rn(__fdiv_rn(1.f, fmaxf(range, 1e-30f)), 3.f) : 0.f;
            zero[e] = nonconst ? __builtin_rintf(__fmul_rn(-mn, mul[e])) : 0.f;
            off[e] = nonconst ? __fmul_rn(-zero[e], step[e]) : mn;
        }
    }
    *reinterpret_cast<float2*>(&lds.step[wave][ch]) = make_float2(step[0], step[1]);
    *reinterpret_cast<float2*>(&lds.mul[wave][ch]) = make_float2(mul[0], mul[1]);
    *reinterpret_cast<float2*>(&lds.zero[wave][ch]) = make_float2(zero[0], zero[1]);
    if constexpr (BITS == 2) *reinterpret_cast<float2*>(&lds.off[wave][ch]) = make_float2(off[0], off[1]);
    __builtin_amdgcn_wave_barrier();  // a wave's LDS operations complete in order
    const int64_t row0 = h * a.capacity + a.dst_start + first;
    if (BITS == 4 && __any(wide)) store_key_codes<BITS, DT, VEC, true>(a, lds, wave, row0, own, count, r, c8, raw);
    else store_key_codes<BITS, DT, VEC, false>(a, lds, wave, row0, own, count, r, c8, raw);
    if (wave == lead) store_key_metadata<BITS, VEC>(a, lds, wave, h * a.superblocks + block_row);
}

template <int BITS, int SB, int DT, bool VEC>
__global__ __launch_bounds__(64 * kKeyWaves) void pack_keys_kernel(KeyPack a) {
    __shared__ __align__(16) KeyLds lds;
    pack_keys<BITS, SB, DT, VEC>(a, blockIdx.x, blockIdx.y, lds);
}

template <int BITS, int SB, int DT>
void launch_pack_keys_of(const KeyPack& a, int64_t hkv, hipStream_t stream) {
    const dim3 grid((unsigned)((a.tail + a.n + kKeyBlockTokens - 1) / kKeyBlockTokens), (unsigned)hkv);
    const bool vec = reinterpret_cast<uintptr_t>(a.src) % 16 == 0 && reinterpret_cast<uintptr_t>(a.packed) % 4 == 0 &&
                     reinterpret_cast<uintptr_t>(a.scale) % 4 == 0;
    if (vec) hipLaunchKernelGGL((pack_keys_kernel<BITS, SB, DT, true>), grid, dim3(64 * kKeyWaves), 0, stream, a);
    else hipLaunchKernelGGL((pack_keys_kernel<BITS, SB, DT, false>), grid, dim3(64 * kKeyWaves), 0, stream, a);
}

template <int BITS>
void launch_pack_keys(const KeyPack& a, int64_t superblock, int64_t dtype, int64_t hkv, hipStream_t stream) {
    if (superblock == 32) dtype == 0 ? launch_pack_keys_of<BITS, 32, 0>(a, hkv, stream) : launch_pack_keys_of<BITS, 32, 1>(a, hkv, stream);
    else if (superblock == 64) dtype == 0 ? launch_pack_keys_of<BITS, 64, 0>(a, hkv, stream) : launch_pack_keys_of<BITS, 64, 1>(a, hkv, stream);
    else dtype == 0 ? launch_pack_keys_of<BITS, 128, 0>(a, hkv, stream) : launch_pack_keys_of<BITS, 128, 1>(a, hkv, stream);
}

// ---------------------------------------------------------------------------- gather rows
// 64 rows per 256-thread block: thread t moves 16-byte chunk t % 16 of rows t / 16 + 16 k, all loads first.
// Rows that start off 16 bytes move element by element.
constexpr int kGatherRows = 64;

struct RowGather {
    const uint16_t* src;
    int64_t src_tokens;
    const int64_t* index;  // nullable: token i is source row i
    int64_t n;
    uint16_t* dst;
    int64_t dst_stride;    // rows per head
};

template <bool VEC>
__device__ __forceinline__ void gather_rows(const RowGather& a, int64_t block, int64_t h) {
    const int c = threadIdx.x & 15;
    const int64_t i0 = block * kGatherRows + (threadIdx.x >> 4);
    int64_t rows[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {  // indices first (clamped to the last row, branch-free), then the rows
        const int64_t i = min(i0 + 16 * k, a.n - 1);
        rows[k] = a.index ? r2o_ldg(a.index + i) : i;
    }
    r2o_u4 v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
        v[k] = r2o_load8<VEC>(a.src + (h * a.src_tokens + rows[k]) * 128 + 8 * c);
#pragma unroll
    for (int k = 0; k < 4; ++k)  // keeps the four loads together (not sunk into the guarded stores)
        asm volatile("" ::"v"(v[k].x), "v"(v[k].y), "v"(v[k].z), "v"(v[k].w));
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int64_t i = i0 + 16 * k;
        if (i < a.n) r2o_store8<VEC>(a.dst + (h * a.dst_stride + i) * 128 + 8 * c, v[k]);
    }
}

template <bool VEC>
__global__ __launch_bounds__(256) void gather_rows_kernel(RowGather a) { gather_rows<VEC>(a, blockIdx.x, blockIdx.y); }

// ------------------------------------------------------------------- a cache's payload in one launch
// The keys, both packed value tiers and the 16-bit rows of a cache build, or the keys and values of a
// flush and its token indices: jobs on consecutive block ranges of one grid, the largest first.  Together
// they fill the chip where each alone leaves most of it idle (a flush's jobs are 1 to 3 blocks per head),
// and a prompt pays one launch for up to five.  Measured: a flush of 4 heads' INT4 keys, INT2 values and
// indices 6.7 us, against 6.0 + 4.9 + 2 x ~3 us and their gaps.
struct CachePack {
    KeyPack key;
    ValuePack v4, v2;
    RowGather fp, rows;            // 16-bit value rows; 16-bit key rows (K_BF16)
    int key_blocks, v4_blocks, v2_blocks, fp_blocks, row_blocks;
    int index_copies;              // flush: the ring's oldest indices, by one more block
    const int64_t* index_src[2];
    int64_t* index_dst[2];
};

// KB: bits of the packed keys (0: none).
template <int KB, int SB, int DT>
__global__ __launch_bounds__(256) void pack_cache_kernel(CachePack a) {
    const int64_t h = blockIdx.y;
    int block = blockIdx.x;
    if constexpr (KB != 0) {
        __shared__ __align__(16) KeyLds lds;
        if (block < a.key_blocks) {
            pack_keys<KB, SB, DT, true>(a.key, block, h, lds);
            return;
        }
        block -= a.key_blocks;
    }
    if (block < a.v4_blocks) return pack_values<4, DT, true>(a.v4, block, h);
    block -= a.v4_blocks;
    if (block < a.v2_blocks) return pack_values<2, DT, true>(a.v2, block, h);
    block -= a.v2_blocks;
    if (block < a.fp_blocks) return gather_rows<true>(a.fp, block, h);
    block -= a.fp_blocks;
    if (block < a.row_blocks) return gather_rows<true>(a.rows, block, h);
    if (h != 0) return;
    for (int i = threadIdx.x; i < a.index_copies; i += blockDim.x) {
        a.index_dst[0][i] = a.index_src[0][i];
        a.index_dst[1][i] = a.index_src[1][i];
    }
}

int64_t blocks_of(int64_t n, int64_t per) { return (n + per - 1) / per; }

template <int DT>
void launch_pack_cache_of(const CachePack& a, int key_bits, int64_t superblock, dim3 grid, hipStream_t st) {
    const dim3 block(256);
    if (key_bits == 4) {
        if (superblock == 32) hipLaunchKernelGGL((pack_cache_kernel<4, 32, DT>), grid, block, 0, st, a);
        else if (superblock == 64) hipLaunchKernelGGL((pack_cache_kernel<4, 64, DT>), grid, block, 0, st, a);
        else hipLaunchKernelGGL((pack_cache_kernel<4, 128, DT>), grid, block, 0, st, a);
    } else if (key_bits == 2) {
        if (superblock == 32) hipLaunchKernelGGL((pack_cache_kernel<2, 32, DT>), grid, block, 0, st, a);
        else if (superblock == 64) hipLaunchKernelGGL((pack_cache_kernel<2, 64, DT>), grid, block, 0, st, a);
        else hipLaunchKernelGGL((pack_cache_kernel<2, 128, DT>), grid, block, 0, st, a);
    } else {
        hipLaunchKernelGGL((pack_cache_kernel<0, 32, DT>), grid, block, 0, st, a);
    }
}

// Every pointer of the jobs 16-byte aligned (checked by the callers).
void launch_pack_cache(CachePack& a, int key_bits, int64_t superblock, int64_t dtype, int64_t hkv, hipStream_t st) {
    a.key_blocks = key_bits ? (int)blocks_of(a.key.tail + a.key.n, kKeyBlockTokens) : 0;
    a.v4_blocks = (int)blocks_of(a.v4.n, kVBlockRows);
    a.v2_blocks = (int)blocks_of(a.v2.n, kVBlockRows);
    a.fp_blocks = (int)blocks_of(a.fp.n, kGatherRows);
    a.row_blocks = (int)blocks_of(a.rows.n, kGatherRows);
    const int64_t blocks = (int64_t)a.key_blocks + a.v4_blocks + a.v2_blocks + a.fp_blocks + a.row_blocks + (a.index_copies > 0);
    if (blocks == 0) return;
    const dim3 grid((unsigned)blocks, (unsigned)hkv);
    if (dtype == 0) launch_pack_cache_of<0>(a, key_bits, superblock, grid, st);
    else launch_pack_cache_of<1>(a, key_bits, superblock, grid, st);
}

// ------------------------------------------------------------------- a cache's indices in one launch
// Before the payload: one wave per page writes its tokens' plan index, global and logical index in tier
// order, and blocks of up to kFillBytes copy the page words and fill what no token reaches (-1 for unused
// indices, 0 for the arenas' spare capacity and the ring).  In place of ~20 library launches (scan, gathers,
// fills of whole arenas) that a build spent most of its time queueing.  Measured, with the payload's
// launch: 4k tokens x 2 heads 3.6 + 5.4 us (a build 361 -> 68 us, the host's), 65k x 4 6.8 + 32 us (399 -> 75,
// the host's), 131k x 8 5.5 + 129 us (572 -> 142, of which the packers' own changes 234).  Latency-bound: each
// block's loads go out together (a fill's search through the arguments and a copy of 16 loads one after
// another took 5.3, 10.5 and 9.8 us in place of 3.6, 6.8 and 5.5).
constexpr int64_t kFillBytes = 32768;
constexpr int kMaxFills = 20;

struct Fill {
    unsigned char* dst;         // of head 0
    const unsigned char* src;   // nullable: fill with `byte`
    int64_t head_stride, bytes;
    int heads, first_block;     // consecutive blocks: heads x chunks of kFillBytes
    uint32_t byte;              // 0 or 0xff
};

struct CacheIndex {
    const int64_t* start;       // [n_pages] first tokens, then lengths, then positions
    int64_t n_pages;
    const int64_t* plan_global;
    const int64_t* plan_logical;
    int64_t* index;
    int64_t* global;            // survivors' global indices (each tier followed by its reserve), then logical
    int64_t* logical;
    int64_t* evicted;
    int64_t int2_at, reserve4, survivors;  // positions from int2_at on come after the INT4 reserve
    int page_blocks, n_fills;
    Fill fills[kMaxFills];
};

__global__ __launch_bounds__(256) void cache_index_kernel(CacheIndex a) {
    const int lane = threadIdx.x & 63;
    int block = blockIdx.x;
    if (block < a.page_blocks) {
        const int64_t page = (int64_t)block * 4 + (threadIdx.x >> 6);
        if (page >= a.n_pages) return;
        const int64_t start = a.start[page], len = a.start[a.n_pages + page], position = a.start[2 * a.n_pages + page];
        for (int64_t j = lane; j < len; j += 64) {
            const int64_t token = start + j, p = position + j, g = a.plan_global[token], l = a.plan_logical[token];
            if (p >= a.survivors) {
                a.evicted[p - a.survivors] = g;
                continue;
            }
            const int64_t slot = p + (p >= a.int2_at ? a.reserve4 : 0);
            a.index[p] = token;
            a.global[slot] = g;
            a.logical[slot] = l;
        }
        return;
    }
    block -= a.page_blocks;
    // all first blocks in one load: a search from fill to fill waited on the launch arguments at every step
    const bool begun = lane < a.n_fills && block >= a.fills[min(lane, kMaxFills - 1)].first_block;
    const Fill& f = a.fills[__builtin_amdgcn_readfirstlane(__popcll(__ballot(begun)) - 1)];
    block -= f.first_block;
    const int64_t first = (int64_t)(block / f.heads) * kFillBytes, n = min(kFillBytes, f.bytes - first);
    unsigned char* dst = f.dst + (block % f.heads) * f.head_stride + first;
    if (f.src) {  // the page words: 8-byte aligned, one head; every load first
        const int64_t* src = reinterpret_cast<const int64_t*>(f.src + first);
        constexpr int kEach = kFillBytes / 8 / 256;
        int64_t w[kEach];
#pragma unroll
        for (int k = 0; k < kEach; ++k) w[k] = src[min((int64_t)threadIdx.x + 256 * k, n / 8 - 1)];
#pragma unroll
        for (int k = 0; k < kEach; ++k)
            if (threadIdx.x + 256 * k < n / 8) reinterpret_cast<int64_t*>(dst)[threadIdx.x + 256 * k] = w[k];
        return;
    }
    const int64_t head = min((int64_t)(-reinterpret_cast<uintptr_t>(dst) & 15), n), body = (n - head) / 16;
    const uint32_t word = f.byte * 0x01010101u;
    if (threadIdx.x < head) dst[threadIdx.x] = (unsigned char)f.byte;
    for (int64_t e = threadIdx.x; e < body; e += 256)
        reinterpret_cast<r2o_u4*>(dst + head)[e] = r2o_u4{word, word, word, word};
    const int64_t done = head + 16 * body;
    if (threadIdx.x < n - done) dst[done + threadIdx.x] = (unsigned char)f.byte;
}

// Adds the fill of bytes [from, to) of each head's `stride` bytes.
void add_fill(CacheIndex& a, int64_t& blocks, void* base, const void* src, int64_t heads, int64_t stride, int64_t from,
              int64_t to, uint32_t byte) {
    if (to <= from || heads <= 0) return;
    Fill& f = a.fills[a.n_fills++];
    f.dst = reinterpret_cast<unsigned char*>(base) + from;
    f.src = reinterpret_cast<const unsigned char*>(src);
    f.head_stride = stride;
    f.bytes = to - from;
    f.heads = (int)heads;
    f.first_block = (int)blocks;
    f.byte = byte;
    blocks += heads * blocks_of(to - from, kFillBytes);
}

// ------------------------------------------------------------------------ Recent-FP ring
__global__ __launch_bounds__(256) void recent_append_kernel(
    uint16_t* rk, uint16_t* rv, int64_t hkv, int64_t capacity, const uint16_t* __restrict__ nk,
    const uint16_t* __restrict__ nv, int64_t pos, int64_t gidx, int64_t lpos, int32_t* length,
    int64_t* gbuf, int64_t* lbuf, int64_t* page_lengths, int64_t page_size) {
    for (int64_t e = threadIdx.x; e < hkv * 128; e += blockDim.x) {
        const int64_t h = e / 128, d = e % 128;
        rk[(h * capacity + pos) * 128 + d] = nk[e];
        rv[(h * capacity + pos) * 128 + d] = nv[e];
    }
    if (threadIdx.x == 0) {
        gbuf[pos] = gidx;
        lbuf[pos] = lpos;
        *length = (int32_t)(pos + 1);
        page_lengths[pos / page_size] = pos % page_size + 1;
    }
}

// Moves slots [flush, active) down to [0, remaining), then, with new_k, appends one token at slot
// `remaining`.  A thread owns one piece (T) of the rows r0, r0 + flush, r0 + 2 flush .. of one head's K or V
// and moves them down in that order: the rows it reads are its own, so no thread waits for another, and the
// appended row is written by the thread whose last read was its slot.  grid (hkv * flush * pieces / 256, 2
// for K and V); block (0, 0) keeps the indices the same way and writes the lengths.
// Latency bounds it: 109 -> 2.4 us for 128 rows of 4 heads (one block with 2-byte moves before).
struct RingShift {
    uint16_t* rows[2];       // K, V [hkv, capacity, 128]
    const uint16_t* add[2];  // nullable: the appended token's rows [hkv, 128]
    int64_t hkv, capacity, flush, remaining;
    int64_t* index[2];       // global, logical [capacity]
    int64_t add_index[2];
    int32_t* length;
    int64_t* page_lengths;
    int64_t page_size;
};

template <typename T>
__global__ __launch_bounds__(256) void recent_shift_kernel(RingShift a) {
    constexpr int kPieces = 256 / (int)sizeof(T);
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t c = e % kPieces, r0 = e / kPieces % a.flush, h = e / kPieces / a.flush;
    const bool add = a.add[0] != nullptr;
    if (h < a.hkv) {
        T* rows = reinterpret_cast<T*>(a.rows[blockIdx.y]) + h * a.capacity * kPieces + c;
        for (int64_t r = r0; r < a.remaining; r += a.flush) rows[r * kPieces] = rows[(r + a.flush) * kPieces];
        if (add && r0 == a.remaining % a.flush)
            rows[a.remaining * kPieces] = reinterpret_cast<const T*>(a.add[blockIdx.y])[h * kPieces + c];
    }
    if (blockIdx.x != 0) return;
    int64_t* index = a.index[blockIdx.y];
    for (int64_t i = threadIdx.x; i < a.flush; i += 256) {
        for (int64_t r = i; r < a.remaining; r += a.flush) index[r] = index[r + a.flush];
        if (add && i == a.remaining % a.flush) index[a.remaining] = a.add_index[blockIdx.y];
    }
    if (blockIdx.y != 0) return;
    const int64_t active = a.remaining + (add ? 1 : 0);
    for (int64_t p = threadIdx.x; p < a.capacity / a.page_size; p += 256)
        a.page_lengths[p] = min(max(active - p * a.page_size, (int64_t)0), a.page_size);
    if (threadIdx.x == 0) *a.length = (int32_t)active;
}

void launch_recent_shift(const RingShift& a, hipStream_t st) {
    const bool vec = (reinterpret_cast<uintptr_t>(a.rows[0]) | reinterpret_cast<uintptr_t>(a.rows[1]) |
                      reinterpret_cast<uintptr_t>(a.add[0]) | reinterpret_cast<uintptr_t>(a.add[1])) % 16 == 0;
    const int64_t threads = a.hkv * a.flush * (vec ? 16 : 128);
    const dim3 grid((unsigned)blocks_of(threads, 256), 2);
    if (vec) hipLaunchKernelGGL(recent_shift_kernel<r2o_u4>, grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL(recent_shift_kernel<uint16_t>, grid, dim3(256), 0, st, a);
}

}  // namespace

extern "C" {

int r2o_pack_int4_k(const uint16_t* src, int64_t dtype, int64_t hkv, int64_t src_tokens, const int64_t* index,
                    int64_t n, int64_t tail, int64_t dst_start, uint8_t* packed, uint16_t* scale, uint8_t* zero,
                    uint32_t* operands, int64_t capacity, int64_t superblocks, int64_t superblock, void* stream) {
    if (!(superblock == 32 || superblock == 64 || superblock == 128) || (dtype != 0 && dtype != 1)) return R2O_EINVAL;
    if (hkv <= 0 || n < 0 || tail < 0 || tail >= superblock || dst_start < 0 || dst_start % superblock) return R2O_EINVAL;
    if (dst_start + tail + n > capacity || capacity % superblock || superblocks * superblock != capacity) return R2O_EINVAL;
    if (n > 0 && (!src || src_tokens <= 0 || (!index && n > src_tokens))) return R2O_EINVAL;
    if (tail + n == 0) return R2O_OK;
    launch_pack_keys<4>({src, src_tokens, index, n, tail, dst_start, packed, scale, zero, operands, capacity, superblocks},
                        superblock, dtype, hkv, (hipStream_t)stream);
    R2O_CHECK_LAUNCH();
    return R2O_OK;
}

int r2o_pack_int2_k(const uint16_t* src, int64_t dtype, int64_t hkv, int64_t src_tokens, const int64_t* index,
                    int64_t n, int64_t tail, int64_t dst_start, uint8_t* packed, uint16_t* scale, uint16_t* offset,
                    uint32_t* operands, int64_t capacity, int64_t superblocks, int64_t superblock, void* stream) {
    if (!(superblock == 32 || superblock == 64 || superblock == 128) || (dtype != 0 && dtype != 1)) return R2O_EINVAL;
    if (hkv <= 0 || n < 0 || tail < 0 || tail >= superblock || dst_start < 0 || dst_start % superblock) return R2O_EINVAL;
    if (dst_start + tail + n > capacity || capacity % superblock || superblocks * superblock != capacity) return R2O_EINVAL;
    if (n > 0 && (!src || src_tokens <= 0 || (!index && n > src_tokens))) return R2O_EINVAL;
    if (tail + n == 0) return R2O_OK;
    launch_pack_keys<2>({src, src_tokens, index, n, tail, dst_start, packed, scale, offset, operands, capacity, superblocks},
                        superblock, dtype, hkv, (hipStream_t)stream);
    R2O_CHECK_LAUNCH();
    return R2O_OK;
}

int r2o_pack_int4_v(const uint16_t* src, int64_t dtype, int64_t hkv, int64_t src_tokens, const int64_t* index,
                    int64_t n, int64_t dst_start, uint8_t* packed, float* scale, int64_t capacity, void* stream) {
    if ((dtype != 0 && dtype != 1) || hkv <= 0 || n < 0 || dst_start < 0 || dst_start + n > capacity) return R2O_EINVAL;
    if (n == 0) return R2O_OK;
    if (!src || src_tokens <= 0 || n > 0x7fffffff || (!index && n > src_tokens)) return R2O_EINVAL;
    launch_pack_values<4>({src, src_tokens, index, n, dst_start, packed, scale, nullptr, capacity, 128}, dtype, hkv,
                          (hipStream_t)stream);
    R2O_CHECK_LAUNCH();
    return R2O_OK;
}

int r2o_pack_int2_v(const uint16_t* src, int64_t dtype, int64_t hkv, int64_t src_tokens, const int64_t* index,
                    int64_t n, int64_t dst_start, int64_t group, uint8_t* packed, uint16_t* scale, uint8_t* zero,
                    int64_t capacity, void* stream) {
    if ((dtype != 0 && dtype != 1) || !(group == 32 || group == 64 || group == 128)) return R2O_EINVAL;
    if (hkv <= 0 || n < 0 || dst_start < 0 || dst_start + n > capacity) return R2O_EINVAL;
    if (n == 0) return R2O_OK;
    if (!src || src_tokens <= 0 || n > 0x7fffffff || (!index && n > src_tokens)) return R2O_EINVAL;
    launch_pack_values<2>({src, src_tokens, index, n, dst_start, packed, scale, zero, capacity, (int)group}, dtype, hkv,
                          (hipStream_t)stream);
    R2O_CHECK_LAUNCH();
    return R2O_OK;
}

int r2o_gather_rows(const uint16_t* src, int64_t hkv, int64_t src_tokens, const int64_t* index, int64_t n,
                    uint16_t* dst, int64_t dst_stride, void* stream) {
    if (hkv <= 0 || n < 0 || n > dst_stride || n > 0x7fffffff) return R2O_EINVAL;
    if (n == 0) return R2O_OK;
    if (!src || !dst || src_tokens <= 0 || (!index && n > src_tokens)) return R2O_EINVAL;
    const RowGather a{src, src_tokens, index, n, dst, dst_stride};
    const dim3 grid((unsigned)blocks_of(n, kGatherRows), (unsigned)hkv);
    const hipStream_t st = (hipStream_t)stream;
    if ((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) % 16 == 0)
        hipLaunchKernelGGL(gather_rows_kernel<true>, grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL(gather_rows_kernel<false>, grid, dim3(256), 0, st, a);
    R2O_CHECK_LAUNCH();
    return R2O_OK;
}

int r2o_recent_append(uint16_t* recent_k, uint16_t* recent_v, int64_t hkv, int64_t capacity, const uint16_t* new_k,
                      const uint16_t* new_v, int64_t position, int64_t global_index, int64_t logical_position,
                      int32_t* length, int64_t* global_buf, int64_t* logical_buf, int64_t* page_lengths,
                      int64_t page_size, void* stream) {
    if (hkv <= 0 || position < 0 || position >= capacity || page_size <= 0 || capacity % page_size) return R2O_EINVAL;
    if (!recent_k || !recent_v || !new_k || !new_v || !length || !global_buf || !logical_buf || !page_lengths)
        return R2O_EINVAL;
    hipLaunchKernelGGL(recent_append_kernel, dim3(1), dim3(256), 0, (hipStream_t)stream, recent_k, recent_v, hkv,
                       capacity, new_k, new_v, position, global_index, logical_position, length, global_buf,
                       logical_buf, page_lengths, page_size);
    R2O_CHECK_LAUNCH();
    return R2O_OK;
}

int r2o_recent_shift(uint16_t* recent_k, uint16_t* recent_v, int64_t hkv, int64_t capacity, int64_t flush,
                     int64_t active, int64_t* global_buf, int64_t* logical_buf, int32_t* length,
                     int64_t* page_lengths, int64_t page_size, void* stream) {
    if (hkv <= 0 || flush <= 0 || active < flush || active > capacity || page_size <= 0 || capacity % page_size)
        return R2O_EINVAL;
    launch_recent_shift({{recent_k, recent_v}, {nullptr, nullptr}, hkv, capacity, flush, active - flush,
                         {global_buf, logical_buf}, {0, 0}, length, page_lengths, page_size}, (hipStream_t)stream);
    R2O_CHECK_LAUNCH();
    return R2O_OK;
}

int r2o_ring_flush(const r2o_ring_flush_params* p, void* stream) {
    if (!p || !p->recent_k || !p->recent_v || !p->length || !p->global_buf || !p->logical_buf || !p->page_lengths)
        return R2O_EINVAL;
    if (p->hkv <= 0 || p->flush <= 0 || p->active < p->flush || p->active > p->capacity || p->page_size <= 0 ||
        p->capacity % p->page_size || (p->dtype != 0 && p->dtype != 1))
        return R2O_EINVAL;
    if (!p->k_packed || !p->k_scale || !p->k_zero || (p->k_bits != 4 && p->k_bits != 2) ||
        !(p->superblock == 32 || p->superblock == 64 || p->superblock == 128) || p->k_tail < 0 ||
        p->k_tail >= p->superblock || p->k_start < 0 || p->k_start % p->superblock ||
        p->k_start + p->k_tail + p->flush > p->k_capacity || p->k_superblocks * p->superblock != p->k_capacity)
        return R2O_EINVAL;
    if (!p->v_packed || !p->v_scale || (p->v_bits != 4 && p->v_bits != 2) || p->v_start < 0 ||
        p->v_start + p->flush > p->v_capacity ||
        (p->v_bits == 2 && (!p->v_zero || !(p->v_group == 32 || p->v_group == 64 || p->v_group == 128))))
        return R2O_EINVAL;
    if ((p->dst_global == nullptr) != (p->dst_logical == nullptr) || (p->new_k == nullptr) != (p->new_v == nullptr))
        return R2O_EINVAL;
    const hipStream_t st = (hipStream_t)stream;
    CachePack a{};
    a.key = {p->recent_k, p->capacity, nullptr, p->flush, p->k_tail, p->k_start, p->k_packed, p->k_scale, p->k_zero,
             p->k_operands, p->k_capacity, p->k_superblocks};
    ValuePack& v = p->v_bits == 4 ? a.v4 : a.v2;
    v = {p->recent_v, p->capacity, nullptr, p->flush, p->v_start, p->v_packed, p->v_scale, p->v_zero, p->v_capacity,
         p->v_bits == 4 ? 128 : (int)p->v_group};
    if (p->dst_global) {
        a.index_copies = (int)p->flush;
        a.index_src[0] = p->global_buf;
        a.index_src[1] = p->logical_buf;
        a.index_dst[0] = p->dst_global;
        a.index_dst[1] = p->dst_logical;
    }
    const uintptr_t low = reinterpret_cast<uintptr_t>(p->recent_k) | reinterpret_cast<uintptr_t>(p->recent_v) |
                          reinterpret_cast<uintptr_t>(p->k_packed) | reinterpret_cast<uintptr_t>(p->k_scale) |
                          reinterpret_cast<uintptr_t>(p->v_packed);
    if (low % 16 == 0) {
        launch_pack_cache(a, (int)p->k_bits, p->superblock, p->dtype, p->hkv, st);
    } else {  // rows or arenas off their 16 bytes: the packers by themselves check what they may widen
        if (p->k_bits == 4) launch_pack_keys<4>(a.key, p->superblock, p->dtype, p->hkv, st);
        else launch_pack_keys<2>(a.key, p->superblock, p->dtype, p->hkv, st);
        if (p->v_bits == 4) launch_pack_values<4>(a.v4, p->dtype, p->hkv, st);
        else launch_pack_values<2>(a.v2, p->dtype, p->hkv, st);
        a.v4.n = a.v2.n = 0;
        launch_pack_cache(a, 0, p->superblock, p->dtype, 1, st);  // the index copies
    }
    R2O_CHECK_LAUNCH();
    launch_recent_shift({{p->recent_k, p->recent_v}, {p->new_k, p->new_v}, p->hkv, p->capacity, p->flush,
                         p->active - p->flush, {p->global_buf, p->logical_buf}, {p->new_global, p->new_logical},
                         p->length, p->page_lengths, p->page_size}, st);
    R2O_CHECK_LAUNCH();
    return R2O_OK;
}

int r2o_cache_build(const r2o_cache_build_params* p, void* stream) {
    if (!p || !p->pages || !p->storage || !p->ring_k || !p->ring_v) return R2O_EINVAL;
    if (p->tokens > 0 && (!p->key || !p->value || !p->plan_global || !p->plan_logical)) return R2O_EINVAL;
    if ((p->key_dtype != 0 && p->key_dtype != 1) || (p->value_dtype != 0 && p->value_dtype != 1)) return R2O_EINVAL;
    if (p->hkv <= 0 || p->tokens < 0 || p->n_pages < 0 || p->page_words <= 0 || p->reserve4 < 0 || p->reserve2 < 0 ||
        p->ring_capacity < 0)
        return R2O_EINVAL;
    const int64_t s_fp = p->tier_tokens[0], s_i4 = p->tier_tokens[1], s_i2 = p->tier_tokens[2], s_ev = p->tier_tokens[3];
    if (s_fp < 0 || s_i4 < 0 || s_i2 < 0 || s_ev < 0) return R2O_EINVAL;
    const int64_t n = s_fp + s_i4 + s_i2;
    if (n > p->k_capacity || n > 0x7fffffff || (n > 0 && !p->index) || !p->k_packed) return R2O_EINVAL;
    const bool packed_k = p->k_bits == 4 || p->k_bits == 2;
    if (!packed_k && p->k_bits != 16) return R2O_EINVAL;
    if (packed_k && (!p->k_scale || !p->k_zero || !(p->superblock == 32 || p->superblock == 64 || p->superblock == 128) ||
                     p->k_superblocks * p->superblock != p->k_capacity))
        return R2O_EINVAL;
    if ((s_fp > 0 && !p->fp_v) || s_i4 > p->i4_capacity || (p->i4_capacity > 0 && (!p->i4_v || !p->i4_scale)) ||
        s_i2 > p->i2_capacity || p->i4_capacity < 0 || p->i2_capacity < 0 ||
        (p->i2_capacity > 0 && (!p->i2_v || !p->i2_scale || !p->i2_zero ||
                                !(p->i2_group == 32 || p->i2_group == 64 || p->i2_group == 128))))
        return R2O_EINVAL;
    for (const void* q : {(const void*)p->key, (const void*)p->value, (const void*)p->k_packed, (const void*)p->k_scale,
                          (const void*)p->fp_v, (const void*)p->i4_v, (const void*)p->i2_v, (const void*)p->ring_k,
                          (const void*)p->ring_v})
        if (reinterpret_cast<uintptr_t>(q) % 16) return R2O_EINVAL;
    const hipStream_t st = (hipStream_t)stream;
    const int64_t h = p->hkv, span = n + p->reserve4 + p->reserve2, head = s_fp + s_i4, cap = p->ring_capacity;
    CacheIndex x{};
    x.start = p->pages + p->page_words;
    x.n_pages = p->n_pages;
    x.plan_global = p->plan_global;
    x.plan_logical = p->plan_logical;
    x.index = p->index;
    x.global = p->storage + p->page_words;
    x.logical = x.global + span;
    x.evicted = x.logical + span;
    x.int2_at = head;
    x.reserve4 = p->reserve4;
    x.survivors = n;
    x.page_blocks = (int)blocks_of(p->n_pages, 4);
    int64_t blocks = 0;
    add_fill(x, blocks, p->storage, p->pages, 1, 0, 0, 8 * p->page_words, 0);
    for (int64_t* idx : {x.global, x.logical}) {
        add_fill(x, blocks, idx, nullptr, 1, 0, 8 * head, 8 * (head + p->reserve4), 0xff);
        add_fill(x, blocks, idx, nullptr, 1, 0, 8 * (span - p->reserve2), 8 * span, 0xff);
    }
    add_fill(x, blocks, x.evicted + s_ev, nullptr, 1, 0, 0, 16 * cap, 0xff);
    for (uint16_t* ring : {p->ring_k, p->ring_v}) add_fill(x, blocks, ring, nullptr, 1, 0, 0, h * cap * 256, 0);
    if (packed_k) {
        const int64_t row = p->k_bits * 16, sb = blocks_of(n, p->superblock), zb = p->k_bits == 4 ? 128 : 256;
        add_fill(x, blocks, p->k_packed, nullptr, h, p->k_capacity * row, n * row, p->k_capacity * row, 0);
        add_fill(x, blocks, p->k_scale, nullptr, h, p->k_superblocks * 256, sb * 256, p->k_superblocks * 256, 0);
        add_fill(x, blocks, p->k_zero, nullptr, h, p->k_superblocks * zb, sb * zb, p->k_superblocks * zb, 0);
        if (p->k_operands)
            add_fill(x, blocks, p->k_operands, nullptr, h, p->k_superblocks * 512, sb * 512, p->k_superblocks * 512, 0);
    } else {
        add_fill(x, blocks, p->k_packed, nullptr, h, p->k_capacity * 256, n * 256, p->k_capacity * 256, 0);
    }
    add_fill(x, blocks, p->i4_v, nullptr, h, p->i4_capacity * 64, s_i4 * 64, p->i4_capacity * 64, 0);
    add_fill(x, blocks, p->i4_scale, nullptr, h, p->i4_capacity * 4, s_i4 * 4, p->i4_capacity * 4, 0);
    const int64_t g = p->i2_capacity > 0 ? 128 / p->i2_group : 0;
    add_fill(x, blocks, p->i2_v, nullptr, h, p->i2_capacity * 32, s_i2 * 32, p->i2_capacity * 32, 0);
    add_fill(x, blocks, p->i2_scale, nullptr, h, p->i2_capacity * 2 * g, s_i2 * 2 * g, p->i2_capacity * 2 * g, 0);
    add_fill(x, blocks, p->i2_zero, nullptr, h, p->i2_capacity * g, s_i2 * g, p->i2_capacity * g, 0);
    static_assert(kMaxFills >= 1 + 4 + 1 + 2 + 4 + 2 + 3, "every fill has a place");
    if (blocks + x.page_blocks > 0x7fffffff) return R2O_EINVAL;
    hipLaunchKernelGGL(cache_index_kernel, dim3((unsigned)(x.page_blocks + blocks)), dim3(256), 0, st, x);
    R2O_CHECK_LAUNCH();
    CachePack a{};
    if (packed_k)
        a.key = {p->key, p->tokens, p->index, n, 0, 0, p->k_packed, p->k_scale, p->k_zero, p->k_operands, p->k_capacity,
                 p->k_superblocks};
    else
        a.rows = {p->key, p->tokens, p->index, n, reinterpret_cast<uint16_t*>(p->k_packed), p->k_capacity};
    a.fp = {p->value, p->tokens, p->index, s_fp, p->fp_v, s_fp};
    a.v4 = {p->value, p->tokens, p->index + s_fp, s_i4, 0, p->i4_v, p->i4_scale, nullptr, p->i4_capacity, 128};
    a.v2 = {p->value, p->tokens, p->index + head, s_i2, 0, p->i2_v, p->i2_scale, p->i2_zero, p->i2_capacity, (int)p->i2_group};
    int key_bits = packed_k && n > 0 ? (int)p->k_bits : 0;
    if (key_bits && p->key_dtype != p->value_dtype) {  // one dtype per launch
        if (key_bits == 4) launch_pack_keys<4>(a.key, p->superblock, p->key_dtype, h, st);
        else launch_pack_keys<2>(a.key, p->superblock, p->key_dtype, h, st);
        key_bits = 0;
    }
    launch_pack_cache(a, key_bits, p->superblock, p->value_dtype, h, st);
    R2O_CHECK_LAUNCH();
    return R2O_OK;
}

const char* r2o_build_target(void) { return "gfx950"; }

}  // extern "C"
