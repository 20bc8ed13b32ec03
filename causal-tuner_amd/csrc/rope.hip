// Partial GPT-J rotary embedding for gfx950: the MI355X replacement of the reference's
// Triton kernels `_rotate_pair`, `_rope` and `_owned_qk_rope` (kernels/core_cuda.py:133-189)
// behind `PartialRoPE`, `inverse_rope_tile` and `rotate_owned_qk` (core_cuda.py:192-229).
//
// Layout: x [tokens, heads, head_dim] with ldx elements between tokens (heads * head_dim
// when contiguous), y likewise with ldy; cosine and sine [tokens, half] contiguous,
// half <= head_dim / 2. Channel pairs (2c, 2c+1) with c < half rotate, the rest pass
// through. Per pair, in fp32 with every product rounded to the tensor type first
// (core_cuda.py:136-142, launched without FMA contraction):
//   ec = T(e c), os = T(o s), oc = T(o c), es = T(e s)
//   e' = T(ec - os), o' = T(oc + es)
// The inverse rotation negates the sine. HBM-bound elementwise work: eight channels per lane
// where the layout allows 16-byte accesses, one lane per pair otherwise.

#include "epilogue.hpp"

namespace ct {
namespace {

template <int T>
__device__ __forceinline__ float load_t(const void *p, int64_t i) {
    if constexpr (T == CT_BF16) return bf16_to_f32(static_cast<const uint16_t *>(p)[i]);
    else if constexpr (T == CT_F16) return f16_to_f32(static_cast<const uint16_t *>(p)[i]);
    else return static_cast<const float *>(p)[i];
}

template <int T>
__device__ __forceinline__ void store_t(void *p, int64_t i, float v) {
    if constexpr (T == CT_BF16) static_cast<uint16_t *>(p)[i] = bf16_bits(v);
    else if constexpr (T == CT_F16) static_cast<uint16_t *>(p)[i] = f16_bits(v);
    else static_cast<float *>(p)[i] = v;
}

template <int T, int TC, bool INVERSE>
__device__ __forceinline__ void rotate_pair(const void *x, int64_t xi, void *y, int64_t yi, float c, float s) {
    const float e = load_t<T>(x, xi), o = load_t<T>(x, xi + 1);
    if constexpr (INVERSE) s = -s;
    float e2, o2;
    rope_pair<T>(e, o, c, s, e2, o2);
    store_t<T>(y, yi, e2);
    store_t<T>(y, yi + 1, o2);
}

// Every pair of x -> y (y may be x): rotated channels rotate, the others are copied.
template <int T, int TC, bool INVERSE>
__global__ __launch_bounds__(256) void rope_all(const void *x, void *y, const void *cosine, const void *sine,
                                                int64_t pairs, int64_t heads, int64_t dim2, int64_t half, int64_t ldx,
                                                int64_t ldy) {
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p >= pairs) return;
    const int64_t per = heads * dim2;  // pairs per token
    const int64_t token = p / per, within = p - token * per;
    const int64_t channel = within % dim2;
    const int64_t xi = token * ldx + 2 * within, yi = token * ldy + 2 * within;
    if (channel < half) {
        const int64_t t = token * half + channel;
        rotate_pair<T, TC, INVERSE>(x, xi, y, yi, load_t<TC>(cosine, t), load_t<TC>(sine, t));
    } else if (x != y) {
        store_t<T>(y, yi, load_t<T>(x, xi));
        store_t<T>(y, yi + 1, load_t<T>(x, xi + 1));
    }
}

// Four table values (16 bytes of float32, 8 of a 16-bit type).
template <int TC>
__device__ __forceinline__ void load_trig4(const void *p, int64_t i, float (&v)[4]) {
    if constexpr (TC == CT_F32) {
        const float4 q = *reinterpret_cast<const float4 *>(static_cast<const float *>(p) + i);
        v[0] = q.x, v[1] = q.y, v[2] = q.z, v[3] = q.w;
    } else {
        const uint2 q = *reinterpret_cast<const uint2 *>(static_cast<const uint16_t *>(p) + i);
        const uint32_t w[2] = {q.x, q.y};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint16_t b = (uint16_t)(j & 1 ? w[j / 2] >> 16 : w[j / 2]);
            v[j] = TC == CT_BF16 ? bf16_to_f32(b) : f16_to_f32(b);
        }
    }
}

// rope_all for bf16 in runs of 8 channels (4 pairs that all rotate or all pass): one 16-byte
// load and store per lane, consecutive lanes along a token. Bound by HBM; the pair-per-lane
// kernel issues four times the instructions for 4-byte accesses and 64-bit divisions
// (q's gradient, 8192 x 4096, 134 MB moved: 91 us there, 32 us here).
template <int TC, bool INVERSE>
__global__ __launch_bounds__(256) void rope_all_vec(const uint16_t *x, uint16_t *y, const void *cosine,
                                                    const void *sine, uint32_t runs, uint32_t per, uint32_t dim8,
                                                    int half, int64_t ldx, int64_t ldy) {
    const uint32_t p = blockIdx.x * 256u + threadIdx.x;
    if (p >= runs) return;
    const uint32_t token = p / per, within = p - token * per;
    const int pair = (int)(within % dim8) * 4;
    const bool rotates = pair < half;
    if (!rotates && x == y) return;
    uint4 q = *reinterpret_cast<const uint4 *>(x + token * ldx + 8 * within);
    if (rotates) {
        float c[4], s[4];
        load_trig4<TC>(cosine, (int64_t)token * half + pair, c);
        load_trig4<TC>(sine, (int64_t)token * half + pair, s);
        uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float e2, o2;
            rope_pair<CT_BF16>(bf16_to_f32((uint16_t)w[j]), bf16_to_f32((uint16_t)(w[j] >> 16)), c[j],
                               INVERSE ? -s[j] : s[j], e2, o2);
            w[j] = pack_bf16x2(e2, o2);
        }
        q = make_uint4(w[0], w[1], w[2], w[3]);
    }
    *reinterpret_cast<uint4 *>(y + token * ldy + 8 * within) = q;
}

// Whole runs of 8 channels: both matrices 16-byte aligned with pitches of 8 elements, heads
// and rotated channels in multiples of 8, tables aligned to four values, and run indexes that
// fit 32 bits.
template <int T, int TC>
bool rope_vec_ok(const void *x, const void *y, const void *cosine, const void *sine, int64_t tokens, int64_t heads,
                 int64_t head_dim, int64_t half, int64_t ldx, int64_t ldy) {
    constexpr uintptr_t kTrig = TC == CT_F32 ? 16 : 8;
    return T == CT_BF16 && reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0 &&
           ldx % 8 == 0 && ldy % 8 == 0 && head_dim % 8 == 0 && half % 4 == 0 &&
           reinterpret_cast<uintptr_t>(cosine) % kTrig == 0 && reinterpret_cast<uintptr_t>(sine) % kTrig == 0 &&
           tokens * heads * (head_dim / 8) < (int64_t{1} << 31);
}

// In place, rotated channels only (the owned q/k outputs of a projection group).
template <int T, int TC, bool INVERSE>
__global__ __launch_bounds__(256) void rope_rotated(void *x, const void *cosine, const void *sine, int64_t pairs,
                                                    int64_t heads, int64_t dim2, int64_t half, int64_t ldx) {
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;  // over tokens x heads x half
    if (p >= pairs) return;
    const int64_t channel = p % half;
    const int64_t th = p / half;  // token * heads + head
    const int64_t token = th / heads, head = th - token * heads;
    const int64_t t = token * half + channel;
    const int64_t xi = token * ldx + 2 * (head * dim2 + channel);
    rotate_pair<T, TC, INVERSE>(x, xi, x, xi, load_t<TC>(cosine, t), load_t<TC>(sine, t));
}

template <int T, int TC, bool INVERSE>
hipError_t launch(const void *x, void *y, const void *cosine, const void *sine, int64_t tokens, int64_t heads,
                  int64_t head_dim, int64_t half, bool rotated_only, int64_t ldx, int64_t ldy, hipStream_t s) {
    const int64_t dim2 = head_dim / 2;
    const int64_t pairs = rotated_only ? tokens * heads * half : tokens * heads * dim2;
    if (pairs == 0) return hipSuccess;
    const dim3 grid((unsigned)cdiv(pairs, 256)), block(256);
    if (rotated_only)
        rope_rotated<T, TC, INVERSE><<<grid, block, 0, s>>>(y, cosine, sine, pairs, heads, dim2, half, ldy);
    else if (rope_vec_ok<T, TC>(x, y, cosine, sine, tokens, heads, head_dim, half, ldx, ldy))
        rope_all_vec<TC, INVERSE><<<dim3((unsigned)cdiv(pairs / 4, 256)), block, 0, s>>>(
            static_cast<const uint16_t *>(x), static_cast<uint16_t *>(y), cosine, sine, (uint32_t)(pairs / 4),
            (uint32_t)(heads * dim2 / 4), (uint32_t)(dim2 / 4), (int)half, ldx, ldy);
    else
        rope_all<T, TC, INVERSE><<<grid, block, 0, s>>>(x, y, cosine, sine, pairs, heads, dim2, half, ldx, ldy);
    return hipGetLastError();
}

template <int T, int TC>
hipError_t launch_dir(const void *x, void *y, const void *cosine, const void *sine, int64_t tokens, int64_t heads,
                      int64_t head_dim, int64_t half, bool inverse, bool rotated_only, int64_t ldx, int64_t ldy,
                      hipStream_t s) {
    return inverse ? launch<T, TC, true>(x, y, cosine, sine, tokens, heads, head_dim, half, rotated_only, ldx, ldy, s)
                   : launch<T, TC, false>(x, y, cosine, sine, tokens, heads, head_dim, half, rotated_only, ldx, ldy,
                                          s);
}

template <int T>
hipError_t launch_trig(const void *x, void *y, const void *cosine, const void *sine, int64_t tokens, int64_t heads,
                       int64_t head_dim, int64_t half, bool inverse, bool rotated_only, int trig, int64_t ldx,
                       int64_t ldy, hipStream_t s) {
    switch (trig) {
        case CT_BF16: return launch_dir<T, CT_BF16>(x, y, cosine, sine, tokens, heads, head_dim, half, inverse,
                                                    rotated_only, ldx, ldy, s);
        case CT_F16: return launch_dir<T, CT_F16>(x, y, cosine, sine, tokens, heads, head_dim, half, inverse,
                                                  rotated_only, ldx, ldy, s);
        default: return launch_dir<T, CT_F32>(x, y, cosine, sine, tokens, heads, head_dim, half, inverse,
                                              rotated_only, ldx, ldy, s);
    }
}

bool known_dtype(int d) { return d == CT_F32 || d == CT_F16 || d == CT_BF16; }

}  // namespace
}  // namespace ct

extern "C" int ct_rope(const void *x, void *y, const void *cosine, const void *sine, int64_t tokens, int64_t heads,
                       int64_t head_dim, int64_t half, int64_t ldx, int64_t ldy, int32_t inverse,
                       int32_t rotated_only, int32_t dtype, int32_t trig_dtype, hipStream_t stream) {
    using namespace ct;
    if (tokens < 0 || heads < 0 || head_dim <= 0 || head_dim % 2 || half < 0 || half > head_dim / 2)
        return -CT_EINVAL_SHAPE;
    if (ldx == 0) ldx = heads * head_dim;
    if (ldy == 0) ldy = heads * head_dim;
    if (ldx < heads * head_dim || ldy < heads * head_dim) return -CT_EINVAL_SHAPE;
    if (x == y && ldx != ldy) return -CT_EINVAL_LAYOUT;
    if (!known_dtype(dtype) || !known_dtype(trig_dtype)) return -CT_EINVAL_DTYPE;
    if (tokens == 0 || heads == 0) return 0;
    if (!x || !y || (half > 0 && (!cosine || !sine))) return -CT_EINVAL_POINTER;
    if (rotated_only && x != y) return -CT_EINVAL_LAYOUT;  // rotated-only runs in place
    if (rotated_only && half == 0) return 0;
    hipError_t e;
    switch (dtype) {
        case CT_BF16:
            e = launch_trig<CT_BF16>(x, y, cosine, sine, tokens, heads, head_dim, half, inverse, rotated_only,
                                     trig_dtype, ldx, ldy, stream);
            break;
        case CT_F16:
            e = launch_trig<CT_F16>(x, y, cosine, sine, tokens, heads, head_dim, half, inverse, rotated_only,
                                    trig_dtype, ldx, ldy, stream);
            break;
        default:
            e = launch_trig<CT_F32>(x, y, cosine, sine, tokens, heads, head_dim, half, inverse, rotated_only,
                                    trig_dtype, ldx, ldy, stream);
    }
    return e == hipSuccess ? 0 : (int)e;
}
