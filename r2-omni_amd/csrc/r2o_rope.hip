// Query/key rotation for gfx950, of a prompt or a decode step: Qwen multimodal rotary embedding (mRoPE) or
// Qwen3's RMSNorm + RoPE, each with an optional orthonormal FWHT-128, and the FWHT alone.
//
// A row (128 channels of one (request, head, token)) is 16 lanes of 8 channels, one 16-byte load and store;
// the rotate-half partner (channel +- 64) is lane ^ 8, read by DPP inside the product that uses it.  A wave
// takes 4 tokens and walks a run of heads: cos and sin are loaded once for all of them, and 4 heads' rows
// are in flight at a time.  The stream of rows bounds a prompt, latency a decode step.  Measured on a prompt
// of 32768 tokens, 28 + 4 heads, bf16: mRoPE 480 -> ~118 us (4.6 TB/s; one wave per row before, 2-byte loads
// and its own cos and sin per row), the FWHT of 131072 rows 50 -> 14.8 us (4.5 TB/s; LDS stages before).
//
// mRoPE follows _qwen_qk_mrope_kernel / _qwen_batched_qk_mrope_kernel (triton_qwen_mrope.py:45-211): x *
// cos + rotate_half(x) * sin in fp32, where dimension d takes its cos/sin from axis 0, 1 or 2 of the [3, B,
// S, 128] tables by its position d % 64 within the mRoPE sections, then the optional FWHT, then one
// rounding to the input dtype.  The Qwen3 branch (qwen_sspa_attention.py:1228-1235: q_norm / k_norm,
// apply_rotary_pos_emb, then triton_fwht_128 when keys are Hadamard-rotated) reproduces the rounding of
// every torch op of that sequence:
//   Qwen3RMSNorm (transformers 5.15.0 modeling_qwen3.py): v = mean(x^2) in fp32, n = dtype(x * rsqrt(v +
//   eps)) with rsqrt evaluated as 1 / sqrt (both correctly rounded, as torch's CPU kernel), then
//   w = dtype(weight * n);
//   apply_rotary_pos_emb: y = dtype(dtype(w * cos) + dtype(rotate_half(w) * sin)), rotate_half(w) =
//   (-w[d + 64], w[d - 64]);
//   optional FWHT-128 of y in fp32 (triton_fwht_128), rounded to dtype.
#include <algorithm>
#include <initializer_list>

#include "r2o_common.hpp"

namespace {

enum Kind { kMrope = 0, kQwen3 = 1 };

struct RopeArgs {
    const uint16_t* q;
    const uint16_t* k;
    const uint16_t* v;  // nullable: V rows take the FWHT alone
    uint16_t* q_out;
    uint16_t* k_out;
    uint16_t* v_out;
    const void* cos;
    const void* sin;
    int64_t cs[4];  // cos strides (axis, batch, token, dim) in elements
    int64_t ss[4];  // sin strides
    const uint16_t* q_weight;  // kQwen3: [128] RMSNorm weights, input dtype
    const uint16_t* k_weight;
    float eps;
    int64_t tokens;
    uint32_t items;            // batch * tokens
    int hq, hkv, heads;        // heads: hq + hkv, and hkv more with V rows
    int heads_per_wave;
    int table_code, s0, s1, hadamard;
    int vec_tables;            // a lane's 8 channels are one aligned run of one axis
};

// cos or sin of the lane's channels 8 c8 .. 8 c8 + 7.
__device__ __forceinline__ void load_table(const RopeArgs& a, const void* base, const int64_t (&st)[4], int64_t b,
                                           int64_t token, int c8, float (&x)[8]) {
    const int64_t at = b * st[1] + token * st[2];
    const int d0 = (8 * c8) & 63;
    if (a.vec_tables) {
        const int64_t e = at + (d0 < a.s0 ? 0 : (d0 < a.s0 + a.s1 ? 1 : 2)) * st[0] + 8 * c8;
        if (a.table_code == 2) {
            const r2o_f4* p = reinterpret_cast<const r2o_f4*>(reinterpret_cast<const float*>(base) + e);
            const r2o_f4 lo = r2o_ldg(p), hi = r2o_ldg(p + 1);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                x[i] = lo[i];
                x[i + 4] = hi[i];
            }
        } else {
            const r2o_u4 w = r2o_load8<true>(reinterpret_cast<const uint16_t*>(base) + e);
            if (a.table_code == 0) r2o_unpack8<0>(w, x);
            else r2o_unpack8<1>(w, x);
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int d = d0 + i;
        const int64_t e = at + (d < a.s0 ? 0 : (d < a.s0 + a.s1 ? 1 : 2)) * st[0] + (8 * c8 + i) * st[3];
        if (a.table_code == 2) {
            x[i] = r2o_ldg(reinterpret_cast<const float*>(base) + e);
        } else {
            const uint32_t w = r2o_ldg(reinterpret_cast<const uint16_t*>(base) + e);
            x[i] = a.table_code == 0 ? r2o_bf16_to_f32(w) : r2o_f16_to_f32(w);
        }
    }
}

// Round to the tensor dtype and back: the result of one torch op.
template <int DT>
__device__ __forceinline__ float round_to(float x) {
    return r2o_round_dtype(x, DT);
}

// One row's rotation in place.  sn carries rotate_half's sign (negative below channel 64).
template <int KIND, int DT>
__device__ __forceinline__ void rotate_row(float (&x)[8], const float (&cs)[8], const float (&sn)[8],
                                           const float (&weight)[8], float eps) {
    if constexpr (KIND == kMrope) {
        float y[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] = x[i] * cs[i] + r2o_lane_xor<8>(x[i]) * sn[i];
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = y[i];
    } else {
        // mean of squares: pair sums x[t]^2 + x[t + 64]^2, then a butterfly over t = 8 (c8 % 8) + i from bit 5
        // down to bit 0 (every lane forms the same sums)
        float s[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float sq = __fmul_rn(x[i], x[i]);
            s[i] = __fadd_rn(sq, r2o_lane_xor<8>(sq));
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            s[i] = __fadd_rn(s[i], r2o_lane_xor<4>(s[i]));
            s[i] = __fadd_rn(s[i], r2o_lane_xor<2>(s[i]));
            s[i] = __fadd_rn(s[i], r2o_lane_xor<1>(s[i]));
        }
#pragma unroll
        for (int m = 4; m >= 1; m >>= 1)
#pragma unroll
            for (int i = 0; i < m; ++i) s[i] = __fadd_rn(s[i], s[i + m]);
        const float inv = __fdiv_rn(1.f, __fsqrt_rn(__fadd_rn(__fdiv_rn(s[0], 128.f), eps)));
        float w[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) w[i] = round_to<DT>(__fmul_rn(weight[i], round_to<DT>(__fmul_rn(x[i], inv))));
#pragma unroll
        for (int i = 0; i < 8; ++i)
            x[i] = round_to<DT>(__fadd_rn(round_to<DT>(__fmul_rn(w[i], cs[i])),
                                          round_to<DT>(__fmul_rn(r2o_lane_xor<8>(w[i]), sn[i]))));
    }
}

constexpr int kHeadsInFlight = 4;

// grid (ceil(items / 16), ceil(heads / heads_per_wave)), block 256.  Lanes past the last item work on it
// again and store nothing: the exchanges need every lane of the wave.
template <int KIND, int DT, bool VEC>
__global__ __launch_bounds__(256) void rotate_kernel(RopeArgs a) {
    const int lane = threadIdx.x & 63, c8 = lane & 15;
    const uint32_t item = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 4 + (lane >> 4);
    const bool live = item < a.items;
    const uint32_t at = live ? item : a.items - 1;
    const uint32_t tokens = (uint32_t)a.tokens, b = at / tokens, token = at - b * tokens;
    float cs[8], sn[8], wq[8], wk[8];
    load_table(a, a.cos, a.cs, b, token, c8, cs);
    load_table(a, a.sin, a.ss, b, token, c8, sn);
#pragma unroll
    for (int i = 0; i < 8; ++i) sn[i] = c8 < 8 ? -sn[i] : sn[i];
    if constexpr (KIND == kQwen3) {
        r2o_unpack8<DT>(r2o_load8<VEC>(a.q_weight + 8 * c8), wq);
        r2o_unpack8<DT>(r2o_load8<VEC>(a.k_weight + 8 * c8), wk);
    }
    // element offsets of the lane's channels in head 0 of q and of k / v; heads are tokens * 128 apart
    const int64_t q0 = ((int64_t)b * a.hq * a.tokens + token) * 128 + 8 * c8;
    const int64_t k0 = ((int64_t)b * a.hkv * a.tokens + token) * 128 + 8 * c8;
    auto offset = [&](int h) {  // h is wave-uniform
        return h < a.hq ? q0 + h * a.tokens * 128 : k0 + (h - (h < a.hq + a.hkv ? a.hq : a.hq + a.hkv)) * a.tokens * 128;
    };
    const int h_end = min(a.heads, (int)(blockIdx.y + 1) * a.heads_per_wave);
    for (int h0 = blockIdx.y * a.heads_per_wave; h0 < h_end; h0 += kHeadsInFlight) {
        r2o_u4 raw[kHeadsInFlight];
#pragma unroll
        for (int u = 0; u < kHeadsInFlight; ++u) {
            const int h = min(h0 + u, h_end - 1);
            raw[u] = r2o_load8<VEC>((h < a.hq ? a.q : (h < a.hq + a.hkv ? a.k : a.v)) + offset(h));
        }
#pragma unroll
        for (int u = 0; u < kHeadsInFlight; ++u) {
            const int h = h0 + u;
            if (h >= h_end) break;
            float x[8];
            r2o_unpack8<DT>(raw[u], x);
            const bool is_v = h >= a.hq + a.hkv;
            if (!is_v) rotate_row<KIND, DT>(x, cs, sn, h < a.hq ? wq : wk, a.eps);
            if (is_v || a.hadamard) r2o_fwht_row8(x, c8);
            if (live) r2o_store8<VEC>((h < a.hq ? a.q_out : (is_v ? a.v_out : a.k_out)) + offset(h), r2o_pack8<DT>(x));
        }
    }
}

// The FWHT alone: a wave takes 4 rows per load, kFwhtRows loads in flight.
constexpr int kFwhtRows = 4;

template <int DT, bool VEC>
__global__ __launch_bounds__(256) void fwht128_kernel(const uint16_t* src, uint16_t* dst, int64_t rows) {
    const int lane = threadIdx.x & 63, c8 = lane & 15;
    const int64_t r0 = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * (4 * kFwhtRows) + (lane >> 4);
    r2o_u4 raw[kFwhtRows];
#pragma unroll
    for (int k = 0; k < kFwhtRows; ++k) raw[k] = r2o_load8<VEC>(src + min(r0 + 4 * k, rows - 1) * 128 + 8 * c8);
#pragma unroll
    for (int k = 0; k < kFwhtRows; ++k) {
        float x[8];
        r2o_unpack8<DT>(raw[k], x);
        r2o_fwht_row8(x, c8);
        if (r0 + 4 * k < rows) r2o_store8<VEC>(dst + (r0 + 4 * k) * 128 + 8 * c8, r2o_pack8<DT>(x));
    }
}

bool aligned16(std::initializer_list<const void*> ptrs) {
    for (const void* p : ptrs)
        if (reinterpret_cast<uintptr_t>(p) % 16) return false;  // a null pointer is aligned
    return true;
}

// Heads of a wave: all of them share its cos and sin, but a call of few tokens is spread over the chip
// first.  kFullWaves waves are 8 for each SIMD.
constexpr int64_t kFullWaves = 8192;

template <int KIND>
int launch_rotate(RopeArgs& a, int64_t dtype, int64_t batch, int64_t hq, int64_t hkv, int64_t tokens, hipStream_t stream) {
    const int64_t items = batch * tokens, heads = hq + (a.v ? 2 : 1) * hkv;
    if (heads > 0x7fffffff / 2 || items > 0x7fffffff) return R2O_EINVAL;  // past any GPU's memory
    a.tokens = tokens;
    a.items = (uint32_t)items;
    a.hq = (int)hq;
    a.hkv = (int)hkv;
    a.heads = (int)heads;
    const int64_t token_waves = (items + 3) / 4;
    int64_t per = (heads * token_waves + kFullWaves - 1) / kFullWaves;
    per = std::max<int64_t>(1, std::min(per, heads));
    per = std::max(per, (heads + 65534) / 65535);  // the grid's second dimension
    a.heads_per_wave = (int)per;
    const int piece = a.table_code == 2 ? 4 : 8;  // elements of 16 bytes
    a.vec_tables = a.s0 % 8 == 0 && a.s1 % 8 == 0 && a.cs[3] == 1 && a.ss[3] == 1 && aligned16({a.cos, a.sin});
    for (int i = 0; i < 3; ++i) a.vec_tables = a.vec_tables && a.cs[i] % piece == 0 && a.ss[i] % piece == 0;
    const dim3 grid((unsigned)((items + 15) / 16), (unsigned)((heads + per - 1) / per));
    const bool vec = aligned16({a.q, a.k, a.v, a.q_out, a.k_out, a.v_out, a.q_weight, a.k_weight});
    if (dtype == 0) {
        if (vec) hipLaunchKernelGGL((rotate_kernel<KIND, 0, true>), grid, dim3(256), 0, stream, a);
        else hipLaunchKernelGGL((rotate_kernel<KIND, 0, false>), grid, dim3(256), 0, stream, a);
    } else {
        if (vec) hipLaunchKernelGGL((rotate_kernel<KIND, 1, true>), grid, dim3(256), 0, stream, a);
        else hipLaunchKernelGGL((rotate_kernel<KIND, 1, false>), grid, dim3(256), 0, stream, a);
    }
    R2O_CHECK_LAUNCH();
    return R2O_OK;
}

}  // namespace

extern "C" {

int r2o_qkv_mrope(const uint16_t* q, const uint16_t* k, const uint16_t* v, uint16_t* q_out, uint16_t* k_out,
                  uint16_t* v_out, int64_t dtype, int64_t batch, int64_t hq, int64_t hkv, int64_t tokens,
                  const void* cos, const void* sin, int64_t table_dtype, const int64_t* cos_strides,
                  const int64_t* sin_strides, int64_t section0, int64_t section1, int64_t apply_hadamard,
                  void* stream) {
    if (!q || !k || !q_out || !k_out || !cos || !sin || !cos_strides || !sin_strides) return R2O_EINVAL;
    if ((v == nullptr) != (v_out == nullptr)) return R2O_EINVAL;
    if ((dtype != 0 && dtype != 1) || table_dtype < 0 || table_dtype > 2) return R2O_EINVAL;
    if (batch <= 0 || hq <= 0 || hkv <= 0 || tokens <= 0) return R2O_EINVAL;
    if (section0 < 0 || section1 < 0 || section0 + section1 > 64) return R2O_EINVAL;
    RopeArgs a{};
    a.q = q;
    a.k = k;
    a.v = v;
    a.q_out = q_out;
    a.k_out = k_out;
    a.v_out = v_out;
    a.cos = cos;
    a.sin = sin;
    for (int i = 0; i < 4; ++i) {
        a.cs[i] = cos_strides[i];
        a.ss[i] = sin_strides[i];
    }
    a.table_code = (int)table_dtype;
    a.s0 = (int)section0;
    a.s1 = (int)section1;
    a.hadamard = apply_hadamard ? 1 : 0;
    return launch_rotate<kMrope>(a, dtype, batch, hq, hkv, tokens, (hipStream_t)stream);
}

int r2o_qk_mrope(const uint16_t* q, const uint16_t* k, uint16_t* q_out, uint16_t* k_out, int64_t dtype, int64_t batch,
                 int64_t hq, int64_t hkv, int64_t tokens, const void* cos, const void* sin, int64_t table_dtype,
                 const int64_t* cos_strides, const int64_t* sin_strides, int64_t section0, int64_t section1,
                 int64_t apply_hadamard, void* stream) {
    return r2o_qkv_mrope(q, k, nullptr, q_out, k_out, nullptr, dtype, batch, hq, hkv, tokens, cos, sin, table_dtype,
                         cos_strides, sin_strides, section0, section1, apply_hadamard, stream);
}

int r2o_qkv_norm_rope(const uint16_t* q, const uint16_t* k, const uint16_t* v, uint16_t* q_out, uint16_t* k_out,
                      uint16_t* v_out, int64_t dtype, int64_t batch, int64_t hq, int64_t hkv, int64_t tokens,
                      const uint16_t* q_weight, const uint16_t* k_weight, float eps, const uint16_t* cos,
                      const uint16_t* sin, const int64_t* cos_strides, const int64_t* sin_strides,
                      int64_t apply_hadamard, void* stream) {
    if (!q || !k || !q_out || !k_out || !q_weight || !k_weight || !cos || !sin || !cos_strides || !sin_strides)
        return R2O_EINVAL;
    if ((v == nullptr) != (v_out == nullptr)) return R2O_EINVAL;
    if ((dtype != 0 && dtype != 1) || batch <= 0 || hq <= 0 || hkv <= 0 || tokens <= 0) return R2O_EINVAL;
    if (!(eps >= 0.f)) return R2O_EINVAL;
    RopeArgs a{};
    a.q = q;
    a.k = k;
    a.v = v;
    a.q_out = q_out;
    a.k_out = k_out;
    a.v_out = v_out;
    a.q_weight = q_weight;
    a.k_weight = k_weight;
    a.cos = cos;
    a.sin = sin;
    for (int i = 0; i < 3; ++i) {  // one axis: every channel lies in section 0
        a.cs[i + 1] = cos_strides[i];
        a.ss[i + 1] = sin_strides[i];
    }
    a.s0 = 64;
    a.table_code = (int)dtype;
    a.eps = eps;
    a.hadamard = apply_hadamard ? 1 : 0;
    return launch_rotate<kQwen3>(a, dtype, batch, hq, hkv, tokens, (hipStream_t)stream);
}

int r2o_qk_norm_rope(const uint16_t* q, const uint16_t* k, uint16_t* q_out, uint16_t* k_out, int64_t dtype,
                     int64_t batch, int64_t hq, int64_t hkv, int64_t tokens, const uint16_t* q_weight,
                     const uint16_t* k_weight, float eps, const uint16_t* cos, const uint16_t* sin,
                     const int64_t* cos_strides, const int64_t* sin_strides, int64_t apply_hadamard, void* stream) {
    return r2o_qkv_norm_rope(q, k, nullptr, q_out, k_out, nullptr, dtype, batch, hq, hkv, tokens, q_weight, k_weight,
                             eps, cos, sin, cos_strides, sin_strides, apply_hadamard, stream);
}

int r2o_fwht128(const uint16_t* src, uint16_t* dst, int64_t rows, int64_t dtype, void* stream) {
    if (rows < 0 || rows > 0x7fffffff || (dtype != 0 && dtype != 1)) return R2O_EINVAL;
    if (rows == 0) return R2O_OK;
    const dim3 grid((unsigned)((rows + 16 * kFwhtRows - 1) / (16 * kFwhtRows)));
    const bool vec = aligned16({src, dst});
    const hipStream_t st = (hipStream_t)stream;
    if (dtype == 0) {
        if (vec) hipLaunchKernelGGL((fwht128_kernel<0, true>), grid, dim3(256), 0, st, src, dst, rows);
        else hipLaunchKernelGGL((fwht128_kernel<0, false>), grid, dim3(256), 0, st, src, dst, rows);
    } else {
        if (vec) hipLaunchKernelGGL((fwht128_kernel<1, true>), grid, dim3(256), 0, st, src, dst, rows);
        else hipLaunchKernelGGL((fwht128_kernel<1, false>), grid, dim3(256), 0, st, src, dst, rows);
    }
    R2O_CHECK_LAUNCH();
    return R2O_OK;
}

}  // extern "C"
