// Per-token affine quantizer and the fused quantize + bit-pack encoders.
//
// Restates on the device the reference's TokenQuant chain (utils/compute.py:84-112):
//   scale = T((max - min) * rel),  zero = T(round(T(min / scale))),
//   code  = T(round(T(x / scale))) - zero,     dequant = T(T(code + zero) * scale)
// where T is the 16-bit storage type and every op computes in fp32 and rounds to T, as the
// PyTorch kernels do.  min / max run over all heads and channels of one (batch, token).
#include "pkv_block.hpp"
#include "pkv_runtime.hpp"

#include <algorithm>

namespace pkv {

template <int DT> struct T16;

template <> struct T16<PKV_F16> {
    static __device__ __forceinline__ float from_bits(uint32_t u16) {
        return __half2float(__ushort_as_half((unsigned short)u16));
    }
    static __device__ __forceinline__ uint32_t to_bits(float x) {
        return (uint32_t)__half_as_ushort(__float2half_rn(x));
    }
};

template <> struct T16<PKV_BF16> {
    static __device__ __forceinline__ float from_bits(uint32_t u16) { return __uint_as_float(u16 << 16); }
    static __device__ __forceinline__ uint32_t to_bits(float x) {   // round to nearest even
        uint32_t u = __float_as_uint(x);
        if ((u & 0x7FFFFFFFu) > 0x7F800000u) return (u >> 16) | 0x40u;   // NaN stays NaN
        u += 0x7FFFu + ((u >> 16) & 1u);
        return u >> 16;
    }
};

template <int DT> __device__ __forceinline__ float round_t(float x) {
    return T16<DT>::from_bits(T16<DT>::to_bits(x));
}

// code of x given the token's (scale, zero); all values are T-representable floats.
template <int DT> __device__ __forceinline__ float quant_code(float x, float scale, float zero) {
    const float qv = rintf(round_t<DT>(__fdiv_rn(x, scale)));
    return round_t<DT>(round_t<DT>(qv) - zero);
}

template <int DT> __device__ __forceinline__ void unpack8(const uint4 v, float out[8]) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        out[2 * i] = T16<DT>::from_bits(w[i] & 0xFFFFu);
        out[2 * i + 1] = T16<DT>::from_bits(w[i] >> 16);
    }
}

// ---- per-token scale / zero ------------------------------------------------------------
// grid (T/16, B), 256 threads: 16 lanes per token, 8 channels per lane, loop over heads.
template <int DT>
__global__ void quant_params_kernel(const uint16_t *__restrict__ x, int H, int T, float rel,
                                    uint16_t *__restrict__ scale, uint16_t *__restrict__ zero) {
    const int b = blockIdx.y;
    const int tok = blockIdx.x * 16 + (threadIdx.x >> 4);
    const int l16 = threadIdx.x & 15;
    float mn = INFINITY, mx = -INFINITY;
    if (tok < T) {
        for (int h = 0; h < H; h++) {
            const uint4 v = *reinterpret_cast<const uint4 *>(
                x + (((size_t)b * H + h) * T + tok) * kHeadDim + l16 * 8);
            float f[8];
            unpack8<DT>(v, f);
#pragma unroll
            for (int i = 0; i < 8; i++) {
                mn = fminf(mn, f[i]);
                mx = fmaxf(mx, f[i]);
            }
        }
    }
#pragma unroll
    for (int d = 8; d >= 1; d >>= 1) {
        mn = fminf(mn, __shfl_xor(mn, d, 16));
        mx = fmaxf(mx, __shfl_xor(mx, d, 16));
    }
    if (l16 == 0 && tok < T) {
        const float range = round_t<DT>(mx - mn);
        const float sc = round_t<DT>(range * rel);
        const float z = round_t<DT>(rintf(round_t<DT>(__fdiv_rn(mn, sc))));
        scale[(size_t)b * T + tok] = (uint16_t)T16<DT>::to_bits(sc);
        zero[(size_t)b * T + tok] = (uint16_t)T16<DT>::to_bits(z);
    }
}

// ---- fused quantize + encode: the cell ---------------------------------------------------
// 128 threads work on one block.  Thread = "cell": 16 tokens (one round) x 4 adjacent channels,
// i.e. four packs.  The cell is loaded straight from x (8 bytes per token row, rows of a
// half-wavefront contiguous), quantized and analysed in registers with packed 16-bit arithmetic;
// no code tile is ever formed.
//   K block (64 x 128):  cell (round r = tid / 32, channels 4t..4t+3, t = tid % 32) IS lane t of
//                        unit r, so the packs are emitted where they were computed.
//   V block (128 x 64):  cell (round r = tid / 16, channels 4g..4g+3, g = tid % 16); V units want
//                        lane = channel with the packs of four consecutive rounds, so the pack
//                        records change hands once through LDS.
//
// Exact division without the division sequence.  code = rint(T(x / scale)) - zero needs
// h = RN16(RN32(x / scale)), which equals RN16(x / scale) (24 >= 2 * 11 + 2 bits: double rounding
// is innocuous).  With r = 1 / scale refined to half an ulp once per token,
//   q0 = x * r;  e = fma(-scale, q0, x);  q1 = fma(e, r, q0)
// is within 2^-24 (1 + 2^-20) of the quotient, while a quotient of two 11-bit significands is
// either exactly an fp16 rounding midpoint (then e is exact and q1 hits it exactly, so the tie is
// broken as in the reference) or at least 2^-23 away from every midpoint; so RN16(q1) is the
// reference's value.  bf16 inputs take the plain path (quant_code).
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// Per-token constants: scale, 1 / scale, and for fp16 either
//   sub2 != 0 (zero in [-500, 3000], the usual case): add2 = (c, c) with c = 1536 + (zero & 1) - zero as fp16 and
//             sub2 = (0x6600 + (zero & 1)) in both halves.  h + c is then one correctly rounded fp16 addition whose
//             result lies in [1535.5, 2048), where the spacing is 1: it rounds h - zero to an integer, and because
//             c - zero is even a tie goes to the same side as in rint(h).  The code is the result's bit pattern
//             minus sub2 -- no separate rounding instruction;
//   sub2 == 0: add2 = (-zero, -zero) for the general sequence rint(h) + (-zero).
// bf16: sub2 != 0 (|zero| <= 2^20): add2 = 2^23 - zero as fp32 bits; sub2 == 0: add2 = zero as fp32 bits.
struct TokPar { float s, r; uint32_t add2, sub2; };
template <int DT> __device__ __forceinline__ TokPar token_par(float sc, uint32_t zero_bits, bool general_form = false);

__device__ __forceinline__ uint32_t pk_u16(u16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ u16x2 as_u16x2(uint32_t v) { return __builtin_bit_cast(u16x2, v); }

// codes of four adjacent channels of one token as two pairs of 16-bit integers
// (UNIFORM: every lane of the wavefront holds the same token constants, so the choice of the sequence is a uniform
// branch; otherwise each lane chooses for itself)
template <int DT, bool UNIFORM = true>
__device__ __forceinline__ void quant4(uint2 xw, const TokPar tp, uint32_t &c01, uint32_t &c23) {
    if (DT == PKV_F16) {
        const f16x2 x01 = __builtin_bit_cast(f16x2, xw.x), x23 = __builtin_bit_cast(f16x2, xw.y);
        auto quot = [&](_Float16 xh) -> _Float16 {
            const float f = (float)xh;
            const float q0 = __fmul_rn(f, tp.r);
            const float e = __fmaf_rn(-tp.s, q0, f);
            return (_Float16)__fmaf_rn(e, tp.r, q0);
        };
        const f16x2 h01 = {quot(x01[0]), quot(x01[1])}, h23 = {quot(x23[0]), quot(x23[1])};
        const f16x2 add = __builtin_bit_cast(f16x2, tp.add2);
        if ((UNIFORM ? (uint32_t)__builtin_amdgcn_readfirstlane(tp.sub2) : tp.sub2) != 0u) {
            const u16x2 sub = as_u16x2(tp.sub2);
            c01 = pk_u16((u16x2)(__builtin_bit_cast(u16x2, (f16x2)(h01 + add)) - sub));
            c23 = pk_u16((u16x2)(__builtin_bit_cast(u16x2, (f16x2)(h23 + add)) - sub));
        } else {
            const f16x2 magic = {(_Float16)1024.f, (_Float16)1024.f};    // 1024 + c has c in its low mantissa bits
            const f16x2 d01 = __builtin_elementwise_roundeven(h01) + add, d23 = __builtin_elementwise_roundeven(h23) + add;
            c01 = __builtin_bit_cast(uint32_t, (f16x2)(d01 + magic)) & 0x00FF00FFu;
            c23 = __builtin_bit_cast(uint32_t, (f16x2)(d23 + magic)) & 0x00FF00FFu;
        }
    } else if ((UNIFORM ? (uint32_t)__builtin_amdgcn_readfirstlane(tp.sub2) : tp.sub2) != 0u) {
        // bf16, zero point of moderate size: the same three-instruction quotient (a quotient of two 8-bit
        // significands is either exactly a bf16 rounding midpoint or at least 2^-17 away from every one), rounded to
        // bf16 by the hardware conversion; rint(h) and rint(h) - zero are then exact in fp32 (bf16 values of 256 and
        // above are integers already), so adding 2^23 - zero leaves the code in the low mantissa bits.
        typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
        typedef float f32x2 __attribute__((ext_vector_type(2)));
        auto quot = [&](float f) -> float {
            const float q0 = __fmul_rn(f, tp.r);
            const float e = __fmaf_rn(-tp.s, q0, f);
            return __fmaf_rn(e, tp.r, q0);
        };
        const f32x2 q01 = {quot(__uint_as_float(xw.x << 16)), quot(__uint_as_float(xw.x & 0xFFFF0000u))};
        const f32x2 q23 = {quot(__uint_as_float(xw.y << 16)), quot(__uint_as_float(xw.y & 0xFFFF0000u))};
        const uint32_t h01 = __builtin_bit_cast(uint32_t, __builtin_convertvector(q01, bf16x2));
        const uint32_t h23 = __builtin_bit_cast(uint32_t, __builtin_convertvector(q23, bf16x2));
        const float mz = __uint_as_float(tp.add2);                        // 2^23 - zero
        const uint32_t a = __float_as_uint(rintf(__uint_as_float(h01 << 16)) + mz) & 0xFFu;
        const uint32_t b = __float_as_uint(rintf(__uint_as_float(h01 & 0xFFFF0000u)) + mz) & 0xFFu;
        const uint32_t c = __float_as_uint(rintf(__uint_as_float(h23 << 16)) + mz) & 0xFFu;
        const uint32_t d = __float_as_uint(rintf(__uint_as_float(h23 & 0xFFFF0000u)) + mz) & 0xFFu;
        c01 = a | (b << 16);
        c23 = c | (d << 16);
    } else {
        const float z = __uint_as_float(tp.add2);
        const uint32_t a = (uint32_t)(int)quant_code<DT>(T16<DT>::from_bits(xw.x & 0xFFFFu), tp.s, z) & 0xFFu;
        const uint32_t b = (uint32_t)(int)quant_code<DT>(T16<DT>::from_bits(xw.x >> 16), tp.s, z) & 0xFFu;
        const uint32_t c = (uint32_t)(int)quant_code<DT>(T16<DT>::from_bits(xw.y & 0xFFFFu), tp.s, z) & 0xFFu;
        const uint32_t d = (uint32_t)(int)quant_code<DT>(T16<DT>::from_bits(xw.y >> 16), tp.s, z) & 0xFFu;
        c01 = a | (b << 16);
        c23 = c | (d << 16);
    }
}

// The usual case of quant4 for fp16 (sub2 != 0) on its own, for rounds whose 16 tokens all take it (one test per
// round instead of one branch per token).  The first product x * r reads the fp16 x directly (v_fma_mix_f32 with
// -0 as the addend: x * r + (-0) is the product, sign of zero included), which saves the conversion of x.
__device__ __forceinline__ void quant4_f16_fast(uint2 xw, const TokPar tp, uint32_t &c01, uint32_t &c23) {
    const uint32_t negzero = 0x80000000u;
    float q0[4];
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[1,0,0]" : "=v"(q0[0]) : "v"(xw.x), "v"(tp.r), "s"(negzero));
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(q0[1]) : "v"(xw.x), "v"(tp.r), "s"(negzero));
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[1,0,0]" : "=v"(q0[2]) : "v"(xw.y), "v"(tp.r), "s"(negzero));
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(q0[3]) : "v"(xw.y), "v"(tp.r), "s"(negzero));
    const f16x2 x01 = __builtin_bit_cast(f16x2, xw.x), x23 = __builtin_bit_cast(f16x2, xw.y);
    const float f[4] = {(float)x01[0], (float)x01[1], (float)x23[0], (float)x23[1]};
    _Float16 h[4];
#pragma unroll
    for (int i = 0; i < 4; i++) h[i] = (_Float16)__fmaf_rn(__fmaf_rn(-tp.s, q0[i], f[i]), tp.r, q0[i]);
    const f16x2 h01 = {h[0], h[1]}, h23 = {h[2], h[3]};
    const f16x2 add = __builtin_bit_cast(f16x2, tp.add2);
    const u16x2 sub = as_u16x2(tp.sub2);
    c01 = pk_u16((u16x2)(__builtin_bit_cast(u16x2, (f16x2)(h01 + add)) - sub));
    c23 = pk_u16((u16x2)(__builtin_bit_cast(u16x2, (f16x2)(h23 + add)) - sub));
}

// ---- x -> uint8 code matrix [T, B*H*128] -----------------------------------------------
// grid (T/16, ceil(H / 4), B), 256 threads: 16 lanes per token, 8 channels per lane, up to four heads per thread with
// all of their rows requested before the first is used; the quotient as in the fused encoders (quant4: the lanes of a
// wavefront hold four different tokens, so each chooses its sequence for itself).
constexpr int kQuantHeads = 4;
template <int DT>
__global__ void __launch_bounds__(256) quantize_kernel(const uint16_t *__restrict__ x, int H, int T,
                                                       const uint16_t *__restrict__ scale, const uint16_t *__restrict__ zero,
                                                       uint8_t *__restrict__ codes, uint32_t *max_code_out) {
    const int b = blockIdx.z, h0 = blockIdx.y * kQuantHeads;
    const int B = gridDim.z;
    const int tok = blockIdx.x * 16 + (threadIdx.x >> 4);
    const int l16 = threadIdx.x & 15;
    const int nh = min(kQuantHeads, H - h0);               // uniform
    uint32_t cmax = 0;
    if (tok < T) {
        uint4 v[kQuantHeads];
#pragma unroll
        for (int i = 0; i < kQuantHeads; i++)
            if (i < nh) v[i] = *reinterpret_cast<const uint4 *>(x + (((size_t)b * H + h0 + i) * T + tok) * kHeadDim + l16 * 8);
        const TokPar tp = token_par<DT>(T16<DT>::from_bits(scale[(size_t)b * T + tok]), zero[(size_t)b * T + tok], false);
        const size_t hidden = (size_t)B * H * kHeadDim;
        uint8_t *row = codes + (size_t)tok * hidden + ((size_t)b * H + h0) * kHeadDim + l16 * 8;
#pragma unroll
        for (int i = 0; i < kQuantHeads; i++) {
            if (i < nh) {
                uint32_t a01, a23, b01, b23;
                quant4<DT, false>(make_uint2(v[i].x, v[i].y), tp, a01, a23);
                quant4<DT, false>(make_uint2(v[i].z, v[i].w), tp, b01, b23);
                const uint32_t lo = __builtin_amdgcn_perm(a23, a01, 0x06040200u), hi = __builtin_amdgcn_perm(b23, b01, 0x06040200u);
                const u16x2 m = __builtin_elementwise_max(__builtin_elementwise_max(as_u16x2(a01 & 0x00FF00FFu), as_u16x2(a23 & 0x00FF00FFu)),
                                                          __builtin_elementwise_max(as_u16x2(b01 & 0x00FF00FFu), as_u16x2(b23 & 0x00FF00FFu)));
                cmax = max(cmax, max((uint32_t)m[0], (uint32_t)m[1]));
                *reinterpret_cast<uint2 *>(row + (size_t)i * kHeadDim) = make_uint2(lo, hi);
            }
        }
    }
    if (max_code_out) {
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) cmax = max(cmax, __shfl_xor(cmax, d, 64));
        // a read first: once the largest code has been seen nobody writes any more (a million atomics on one
        // address would cost milliseconds)
        if ((threadIdx.x & 63) == 0 && cmax > __hip_atomic_load(max_code_out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMax(max_code_out, cmax);
    }
}

// ---- parameters and codes in one pass over x, of one tensor or of K and V ---------------
// quant_params_kernel and quantize_kernel in one: grid (T/16, B, tensors), 256 threads, 16 lanes per token, 8 channels per lane.  The
// rows of up to eight heads stay in registers between the two; with more heads the last eight do and the others come again, from
// the L2.  Bound by the memory system, where the pair read x twice in four launches for K and V.
struct QuantSide {
    const uint16_t *x;
    float rel;
    uint16_t *scale, *zero;
    uint8_t *codes;
};
template <int DT>
__global__ void __launch_bounds__(256) quant_codes_kernel(const QuantSide k, const QuantSide v, int H, int T) {
    constexpr int kHeads = 8;
    const QuantSide &sd = blockIdx.z == 0 ? k : v;
    const int b = blockIdx.y, B = gridDim.y;
    const int tok = blockIdx.x * 16 + (threadIdx.x >> 4), l16 = threadIdx.x & 15;
    const int at = min(tok, T - 1);                        // (lanes past the end go along for the exchanges)
    const uint16_t *rows = sd.x + ((size_t)b * H * T + at) * kHeadDim + l16 * 8;
    const size_t head = (size_t)T * kHeadDim;
    uint4 r[kHeads];
    auto load = [&](int h0) {
#pragma unroll
        for (int i = 0; i < kHeads; i++)
            if (h0 + i < H) r[i] = *reinterpret_cast<const uint4 *>(rows + (size_t)(h0 + i) * head);
    };
    const int last = (H - 1) / kHeads * kHeads;
    float mn = INFINITY, mx = -INFINITY;
    for (int h0 = 0; h0 <= last; h0 += kHeads) {
        load(h0);
#pragma unroll
        for (int i = 0; i < kHeads; i++) {
            if (h0 + i < H) {
                float f[8];
                unpack8<DT>(r[i], f);
#pragma unroll
                for (int c = 0; c < 8; c++) {
                    mn = fminf(mn, f[c]);
                    mx = fmaxf(mx, f[c]);
                }
            }
        }
    }
#pragma unroll
    for (int d = 8; d >= 1; d >>= 1) {
        mn = fminf(mn, __shfl_xor(mn, d, 16));
        mx = fmaxf(mx, __shfl_xor(mx, d, 16));
    }
    const float range = round_t<DT>(mx - mn);
    const float sc = round_t<DT>(range * sd.rel);
    const uint32_t zb = T16<DT>::to_bits(rintf(round_t<DT>(__fdiv_rn(mn, sc))));
    const bool in = tok < T;
    if (in && l16 == 0) {
        sd.scale[(size_t)b * T + tok] = (uint16_t)T16<DT>::to_bits(sc);
        sd.zero[(size_t)b * T + tok] = (uint16_t)zb;
    }
    const TokPar tp = token_par<DT>(sc, zb, false);
    uint8_t *row = sd.codes + ((size_t)at * B + b) * (size_t)H * kHeadDim + l16 * 8;
    for (int h0 = last; h0 >= 0; h0 -= kHeads) {
        if (h0 != last) load(h0);
#pragma unroll
        for (int i = 0; i < kHeads; i++) {
            if (in && h0 + i < H) {
                uint32_t a01, a23, b01, b23;
                quant4<DT, false>(make_uint2(r[i].x, r[i].y), tp, a01, a23);
                quant4<DT, false>(make_uint2(r[i].z, r[i].w), tp, b01, b23);
                *reinterpret_cast<uint2 *>(row + (size_t)(h0 + i) * kHeadDim) =
                    make_uint2(__builtin_amdgcn_perm(a23, a01, 0x06040200u), __builtin_amdgcn_perm(b23, b01, 0x06040200u));
            }
        }
    }
}

// ---- uint8 code matrix -> x_hat [B, H, T, 128] -----------------------------------------
// the same grid and thread roles
template <int DT>
__global__ void __launch_bounds__(256) dequantize_kernel(const uint8_t *__restrict__ codes, int H, int T,
                                                         const uint16_t *__restrict__ scale, const uint16_t *__restrict__ zero,
                                                         uint16_t *__restrict__ x) {
    const int b = blockIdx.z, h0 = blockIdx.y * kQuantHeads;
    const int B = gridDim.z;
    const int tok = blockIdx.x * 16 + (threadIdx.x >> 4);
    const int l16 = threadIdx.x & 15;
    const int nh = min(kQuantHeads, H - h0);               // uniform
    if (tok >= T) return;
    const size_t hidden = (size_t)B * H * kHeadDim;
    const uint8_t *row = codes + (size_t)tok * hidden + ((size_t)b * H + h0) * kHeadDim + l16 * 8;
    uint2 c[kQuantHeads];
#pragma unroll
    for (int i = 0; i < kQuantHeads; i++)
        if (i < nh) c[i] = *reinterpret_cast<const uint2 *>(row + (size_t)i * kHeadDim);
    const float sc = T16<DT>::from_bits(scale[(size_t)b * T + tok]);
    const float z = T16<DT>::from_bits(zero[(size_t)b * T + tok]);
#pragma unroll
    for (int i = 0; i < kQuantHeads; i++) {
        if (i < nh) {
            uint32_t out[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const uint32_t w = q < 2 ? c[i].x : c[i].y;
                const float a0 = (float)((w >> (16 * (q & 1))) & 0xFFu);
                const float a1 = (float)((w >> (16 * (q & 1) + 8)) & 0xFFu);
                const uint32_t r0 = T16<DT>::to_bits(round_t<DT>(a0 + z) * sc);
                const uint32_t r1 = T16<DT>::to_bits(round_t<DT>(a1 + z) * sc);
                out[q] = r0 | (r1 << 16);
            }
            *reinterpret_cast<uint4 *>(x + (((size_t)b * H + h0 + i) * T + tok) * kHeadDim + l16 * 8) =
                make_uint4(out[0], out[1], out[2], out[3]);
        }
    }
}

// ---- quantise and dequantise at once ---------------------------------------------------
// A 64-token cut that waits for its partner is attended in the form the streams will give it: parameters, codes and
// dequantised values of n tokens in one launch, K and V in the grid's third dimension.  grid (ceil(n / 16), B, 2), the
// thread roles of quantize_kernel over all heads; the second read of the rows comes from L1 / L2.  Latency-bound: a few
// workgroups, once every 128 tokens (params, quantize and dequantize kernels with their read-back took 70 us a side).
struct QdqSide { const uint16_t *x; uint16_t *out; float rel; };
template <int DT>
__global__ void __launch_bounds__(256) quant_dequant_kernel(const QdqSide k, const QdqSide v, int H, int n, int out_rows) {
    const QdqSide sd = blockIdx.z ? v : k;
    const int b = blockIdx.y, tok = blockIdx.x * 16 + (threadIdx.x >> 4), l16 = threadIdx.x & 15;
    if (tok >= n) return;                                    // (whole rows of 16 lanes)
    float mn = INFINITY, mx = -INFINITY;
    const uint16_t *rows = sd.x + ((size_t)b * H * n + tok) * kHeadDim + l16 * 8;
#pragma unroll 4
    for (int h = 0; h < H; h++) {
        float f[8];
        unpack8<DT>(*reinterpret_cast<const uint4 *>(rows + (size_t)h * n * kHeadDim), f);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            mn = fminf(mn, f[i]);
            mx = fmaxf(mx, f[i]);
        }
    }
#pragma unroll
    for (int d = 8; d >= 1; d >>= 1) {
        mn = fminf(mn, __shfl_xor(mn, d, 16));
        mx = fmaxf(mx, __shfl_xor(mx, d, 16));
    }
    const float sc = round_t<DT>(round_t<DT>(mx - mn) * sd.rel);
    const float z = round_t<DT>(rintf(round_t<DT>(__fdiv_rn(mn, sc))));
    const TokPar tp = token_par<DT>(sc, T16<DT>::to_bits(z), false);
    uint16_t *out = sd.out + ((size_t)b * H * out_rows + tok) * kHeadDim + l16 * 8;
#pragma unroll 2
    for (int h = 0; h < H; h++) {
        const uint4 w = *reinterpret_cast<const uint4 *>(rows + (size_t)h * n * kHeadDim);
        uint32_t c[4], r[4];                                 // codes of adjacent channels as 16-bit pairs
        quant4<DT, false>(make_uint2(w.x, w.y), tp, c[0], c[1]);
        quant4<DT, false>(make_uint2(w.z, w.w), tp, c[2], c[3]);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float a0 = (float)(c[i] & 0xFFu), a1 = (float)((c[i] >> 16) & 0xFFu);
            r[i] = T16<DT>::to_bits(round_t<DT>(a0 + z) * sc) | (T16<DT>::to_bits(round_t<DT>(a1 + z) * sc) << 16);
        }
        *reinterpret_cast<uint4 *>(out + (size_t)h * out_rows * kHeadDim) = make_uint4(r[0], r[1], r[2], r[3]);
    }
}

int launch_quant_dequant(const void *k, const void *v, void *k_out, void *v_out, int dtype, int B, int H, int n, int out_rows, float k_rel,
                         float v_rel, hipStream_t s) {
    const QdqSide ks{(const uint16_t *)k, (uint16_t *)k_out, k_rel}, vs{(const uint16_t *)v, (uint16_t *)v_out, v_rel};
    const dim3 grid((unsigned)((n + 15) / 16), (unsigned)B, 2);
    if (dtype == PKV_F16) quant_dequant_kernel<PKV_F16><<<grid, 256, 0, s>>>(ks, vs, H, n, out_rows);
    else quant_dequant_kernel<PKV_BF16><<<grid, 256, 0, s>>>(ks, vs, H, n, out_rows);
    PKV_HIP_CHECK(hipGetLastError());
    return PKV_OK;
}

// bit_length of both 16-bit halves, at most MOST (larger values mean the codes overflow the format; the launch reports that through
// max_code): the exponent of (2 r + 1) 2^-10 as a half, r read as a subnormal half (r 2^-24 times 2^15, exact).  Four instructions;
// sums of min(r >> k, 1) came out of the compiler as compares and selects of single halves, 24.  (The limit comes first: 0x8000,
// the range of a pack of NaNs of both signs, reads as -0.)
template <int MOST>
__device__ __forceinline__ uint32_t pk_bitlen(uint32_t r) {
    constexpr uint16_t kTop = (1u << MOST) - 1u;
    const u16x2 v = __builtin_elementwise_min(as_u16x2(r), (u16x2){kTop, kTop});
    const f16x2 f = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, v), (f16x2){(_Float16)32768.f, (_Float16)32768.f},
                                              (f16x2){(_Float16)0.0009765625f, (_Float16)0.0009765625f});
    return pk_u16((u16x2)((__builtin_bit_cast(u16x2, f) >> 10) - (u16x2){5, 5}));
}
// Minimum or maximum of 16 words of two codes each, as unsigned integers: what NaN makes of a code may have its top bit set, and
// the packs of such tokens are to be the same in every kernel (v_pk_minimum3_f16 would take three at a time, but by their sign).
template <bool MAX>
__device__ __forceinline__ uint32_t pk_side16(const uint32_t c[16]) {
    auto of = [](u16x2 a, u16x2 b) { return MAX ? __builtin_elementwise_max(a, b) : __builtin_elementwise_min(a, b); };
    u16x2 m[4];
#pragma unroll
    for (int j = 0; j < 4; j++) m[j] = as_u16x2(c[j]);
#pragma unroll
    for (int k = 4; k < 16; k++) m[k & 3] = of(m[k & 3], as_u16x2(c[k]));
    return pk_u16(of(of(m[0], m[1]), of(m[2], m[3])));
}
// 2^len of both halves, as a factor the compiler does not see through: it would make a shift and an addition of every
// multiply-add by it.
__device__ __forceinline__ u16x2 pk_power(uint32_t len2) {
    uint32_t p = pk_u16((u16x2)((u16x2){1, 1} << as_u16x2(len2)));
    asm("" : "+v"(p));
    return as_u16x2(p);
}

// The two packs held in one register pair column: codes c[k] (k = token, two channels per word)
// -> minima, widths and the two 64-bit pack words  sum (c_k - min) << ((15 - k) * len).
__device__ __forceinline__ void build_pair(const uint32_t c[16], uint32_t &mn2, uint32_t &len2, uint32_t &mx2,
                                           uint64_t &w_lo, uint64_t &w_hi) {
    mn2 = pk_side16<false>(c);
    mx2 = pk_side16<true>(c);
    const u16x2 mn = as_u16x2(mn2), mx = as_u16x2(mx2), one = {1, 1};
    len2 = pk_bitlen<4>(pk_u16((u16x2)(mx - mn)));
    const u16x2 p = pk_power(len2);
    // quarter windows (4 tokens, 4 * len <= 16 bits), all arithmetic modulo 2^16 per half:
    //   sum c_k p^(3-k) - min (1 + p + p^2 + p^3)
    const u16x2 rep = ((p + one) * p + one) * p + one;
    const u16x2 mnrep = mn * rep;
    // (the four windows side by side: each step waits for the one before)
    u16x2 w[4];
    uint32_t qw[4];
#pragma unroll
    for (int j = 0; j < 4; j++) w[j] = as_u16x2(c[4 * j]) * p + as_u16x2(c[4 * j + 1]);
#pragma unroll
    for (int j = 0; j < 4; j++) w[j] = w[j] * p + as_u16x2(c[4 * j + 2]);
#pragma unroll
    for (int j = 0; j < 4; j++) w[j] = w[j] * p + as_u16x2(c[4 * j + 3]);
#pragma unroll
    for (int j = 0; j < 4; j++) qw[j] = pk_u16((u16x2)(w[j] - mnrep));
    // 64-bit words: tokens 0..7 above tokens 8..15
    const uint32_t l0 = len2 & 0xFFFFu, l1 = len2 >> 16;
    const uint32_t a0 = ((qw[0] & 0xFFFFu) << (4u * l0)) | (qw[1] & 0xFFFFu), b0 = ((qw[2] & 0xFFFFu) << (4u * l0)) | (qw[3] & 0xFFFFu);
    const uint32_t a1 = ((qw[0] >> 16) << (4u * l1)) | (qw[1] >> 16), b1 = ((qw[2] >> 16) << (4u * l1)) | (qw[3] >> 16);
    w_lo = ((uint64_t)a0 << (8u * l0)) | b0;
    w_hi = ((uint64_t)a1 << (8u * l1)) | b1;
}

// running (min, max) of the 8 values of one 16-byte row chunk
template <int DT>
__device__ __forceinline__ void minmax8(const uint4 v, float &mn, float &mx) {
    if (DT == PKV_F16) {   // packed fp16 comparisons, converted once
        const f16x2 a = __builtin_bit_cast(f16x2, v.x), b = __builtin_bit_cast(f16x2, v.y), c = __builtin_bit_cast(f16x2, v.z),
                    d = __builtin_bit_cast(f16x2, v.w);
        const f16x2 lo = __builtin_elementwise_min(__builtin_elementwise_min(a, b), __builtin_elementwise_min(c, d));
        const f16x2 hi = __builtin_elementwise_max(__builtin_elementwise_max(a, b), __builtin_elementwise_max(c, d));
        mn = fminf(mn, fminf((float)lo[0], (float)lo[1]));
        mx = fmaxf(mx, fmaxf((float)hi[0], (float)hi[1]));
    } else {
        float f[8];
        unpack8<DT>(v, f);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            mn = fminf(mn, f[i]);
            mx = fmaxf(mx, f[i]);
        }
    }
}


// min and max over the 16 lanes of a row of the wavefront (every lane gets the results): the exchanges are DPP
// operands of the min / max instructions themselves (quad permutes, then the half-row and row mirrors).
__device__ __forceinline__ void row16_minmax(float &mn, float &mx) {
    // (written out: the compiler keeps the exchanges as separate moves; a VGPR written by a VALU instruction must be
    // two instructions old before a DPP operand reads it, which the interleaving and the s_nop provide)
    asm("s_nop 1\n\t"
        "v_min_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_max_f32_dpp %1, %1, %1 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 0\n\t"
        "v_min_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_max_f32_dpp %1, %1, %1 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 0\n\t"
        "v_min_f32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
        "v_max_f32_dpp %1, %1, %1 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 0\n\t"
        "v_min_f32_dpp %0, %0, %0 row_mirror row_mask:0xf bank_mask:0xf\n\t"
        "v_max_f32_dpp %1, %1, %1 row_mirror row_mask:0xf bank_mask:0xf"
        : "+v"(mn), "+v"(mx));
}
// packed fp16 min / max as the instructions themselves (the builtins first quieten every operand with an extra
// instruction; the instructions ignore quiet NaNs as the builtins do)
__device__ __forceinline__ f16x2 pk_min_h(f16x2 a, f16x2 b) {
    f16x2 r;
    asm("v_pk_min_f16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ f16x2 pk_max_h(f16x2 a, f16x2 b) {
    f16x2 r;
    asm("v_pk_max_f16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// Where the rows of x lie: elements from one sequence, head and token to the next (channels contiguous, every row on a
// 16-byte boundary).  A cut of a prompt is encoded where it is, also as a transposed projection output.
struct XRows { int64_t sb, sh, st; };

// The rotary embedding of the rows, when the K encoder applies it: cos / sin [.., tokens, 128] by sequence (elements).
struct Rot { const uint16_t *cos, *sin; int64_t sb; };

// Token parameters of one round of the round-major encoders for a group of up to four heads (several of which share
// a workgroup).  256 threads per 16 tokens: thread (tt = token, l16) reads 8 channels of every head; lane l16 == 0
// writes the token's scale and zero and its constants for quant4.  `rows` is x at (sequence, head 0, the round's first
// token) and uniform, so the loads are one 32-bit lane offset on scalar bases; only the rows that exist are
// fetched and compared.
template <int DT>
__device__ __forceinline__ void round_token_params_few(const uint16_t *rows, const XRows xs, int H, int tt, int l16, float rel,
                                                       uint16_t *scale_out, uint16_t *zero_out, TokPar *par_out) {
    const uint32_t lane_off = ((uint32_t)tt * (uint32_t)xs.st + (uint32_t)l16 * 8u) * 2u;          // bytes (row strides are below 2^25 elements)
    uint4 v[4];
    v[0] = *reinterpret_cast<const uint4 *>(reinterpret_cast<const char *>(rows) + lane_off);
#pragma unroll
    for (int i = 1; i < 4; i++)
        if (i < H) v[i] = *reinterpret_cast<const uint4 *>(reinterpret_cast<const char *>(rows + i * xs.sh) + lane_off);
    float mn, mx;
    if (DT == PKV_F16) {
        f16x2 lo, hi;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (i < H) {
                const f16x2 a = __builtin_bit_cast(f16x2, v[i].x), b = __builtin_bit_cast(f16x2, v[i].y),
                            c = __builtin_bit_cast(f16x2, v[i].z), d = __builtin_bit_cast(f16x2, v[i].w);
                const f16x2 l = pk_min_h(pk_min_h(a, b), pk_min_h(c, d)), h = pk_max_h(pk_max_h(a, b), pk_max_h(c, d));
                lo = i ? pk_min_h(lo, l) : l;
                hi = i ? pk_max_h(hi, h) : h;
            }
        }
        mn = fminf((float)lo[0], (float)lo[1]);
        mx = fmaxf((float)hi[0], (float)hi[1]);
    } else {
        mn = INFINITY, mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (i < H) minmax8<DT>(v[i], mn, mx);
    }
    row16_minmax(mn, mx);
    if (l16 == 0) {
        const float range = round_t<DT>(mx - mn);
        const float sc = round_t<DT>(range * rel);
        const uint32_t zb = T16<DT>::to_bits(rintf(round_t<DT>(__fdiv_rn(mn, sc))));
        *scale_out = (uint16_t)T16<DT>::to_bits(sc);
        *zero_out = (uint16_t)zb;
        *par_out = token_par<DT>(sc, zb, false);
    }
}

// `rows` (uniform) is the first of the cell's 16 token rows, `lane_off` the lane's byte offset from it, `row_bytes` (uniform)
// the bytes from row to row: a load is one 32-bit lane offset on a scalar base.  (Rows as immediates of a per-lane 64-bit
// address need the row stride as a constant, and a branch between the two forms took registers: 131 and 149 instead of
// 128 at most in the K kernel, fused K + V encode of 2 x 1 GiB 630 -> 723 us.)
__device__ __forceinline__ void cell_load(const char *rows, int64_t row_bytes, uint32_t lane_off, uint2 xr[16]) {
#pragma unroll
    for (int k = 0; k < 16; k++) xr[k] = *reinterpret_cast<const uint2 *>(rows + k * row_bytes + lane_off);
}

// The rows of a cell with their rotary embedding, every product and the sum rounded to the storage type as the reference's
// chain of elementwise ops does (utils/compute.py:35-43): channel d of the lower half becomes x[d] cos[d] - x[d + 64] sin[d],
// of the upper half x[d] cos[d] + x[d - 64] sin[d].  A lane holds channels 4 t .. 4 t + 3, so the other factor of a pair is
// in the same register of lane t ^ 16: one permlane16_swap and a select.  `cr` / `sr`: the first row's table entries,
// uniform; eight rows of the tables at a time (they come from the caches: every head and sequence reads the same ones).
template <int DT>
__device__ __forceinline__ void cell_rotate(const char *cr, const char *sr, uint32_t lane_off, bool upper, uint2 xr[16]) {
#pragma clang fp contract(off)
    const uint32_t flip = upper ? 0u : 0x80008000u;
#pragma unroll
    for (int k0 = 0; k0 < 16; k0 += 8) {
        uint2 c[8], s[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            c[k] = *reinterpret_cast<const uint2 *>(cr + (k0 + k) * (2 * kHeadDim) + lane_off);
            s[k] = *reinterpret_cast<const uint2 *>(sr + (k0 + k) * (2 * kHeadDim) + lane_off);
        }
#pragma unroll
        for (int k = 0; k < 8; k++) {
            uint32_t own[2] = {xr[k0 + k].x, xr[k0 + k].y}, cc[2] = {c[k].x, c[k].y}, ss[2] = {s[k].x, s[k].y};
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const auto sw = __builtin_amdgcn_permlane16_swap(own[e], own[e], false, false);   // even rows' values, odd rows' values
                const uint32_t other = (upper ? sw[0] : sw[1]) ^ flip;
                if (DT == PKV_F16) {
                    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
                    const h2 a = __builtin_bit_cast(h2, own[e]) * __builtin_bit_cast(h2, cc[e]);
                    const h2 b = __builtin_bit_cast(h2, other) * __builtin_bit_cast(h2, ss[e]);
                    own[e] = __builtin_bit_cast(uint32_t, (h2)(a + b));
                } else {
                    typedef float f2 __attribute__((ext_vector_type(2)));
                    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
                    auto up = [](uint32_t v) -> f2 { return (f2){__uint_as_float(v << 16), __uint_as_float(v & 0xFFFF0000u)}; };
                    auto rn = [](f2 v) -> uint32_t { return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, b2)); };
                    own[e] = rn(up(rn(up(own[e]) * up(cc[e]))) + up(rn(up(other) * up(ss[e]))));
                }
            }
            xr[k0 + k] = make_uint2(own[0], own[1]);
        }
    }
}

// The same where the lanes of a wavefront do not share a base (several groups to a workgroup).
__device__ __forceinline__ void cell_load_lanes(const uint16_t *xc, int64_t st, uint2 xr[16]) {
#pragma unroll
    for (int k = 0; k < 16; k++) xr[k] = *reinterpret_cast<const uint2 *>(xc + k * st);
}

// The same cell from permuted rows: row k is token rows[k] (uniform: the indices come from scalar loads) of the
// tokens that start at `seq`, which is uniform too; `lane_off` is the lane's byte offset inside a token's rows.
__device__ __forceinline__ void cell_load_rows(const uint16_t *seq, const uint32_t *rows, uint32_t last_row, uint32_t lane_off, uint2 xr[16]) {
#pragma unroll
    for (int k = 0; k < 16; k++)                          // (row indices clamped: a damaged order cannot read outside the block)
        xr[k] = *reinterpret_cast<const uint2 *>(reinterpret_cast<const char *>(seq + (size_t)min(rows[k], last_row) * kHeadDim) + lane_off);
}

// The same when the lanes of a wavefront do not share their rows (`rows` differs between lanes; 64-byte aligned): the
// 16 indices are loaded by the lane itself and the row offsets are per-lane 32-bit offsets on the uniform base.
__device__ __forceinline__ void cell_load_rows_lanes(const uint16_t *seq, const uint32_t *rows, uint32_t last_row, uint32_t lane_off, uint2 xr[16]) {
    uint4 idx[4];
#pragma unroll
    for (int q = 0; q < 4; q++) idx[q] = reinterpret_cast<const uint4 *>(rows)[q];
#pragma unroll
    for (int k = 0; k < 16; k++) {
        const uint4 v = idx[k >> 2];
        const uint32_t row = min((k & 3) == 0 ? v.x : (k & 3) == 1 ? v.y : (k & 3) == 2 ? v.z : v.w, last_row);
        xr[k] = *reinterpret_cast<const uint2 *>(reinterpret_cast<const char *>(seq) + (row * (uint32_t)(kHeadDim * 2) + lane_off));
    }
}

// (general_form: the constants of the general sequence whatever the zero point -- for callers whose wavefronts hold
// several tokens and must take one path for all of them)
template <int DT>
__device__ __forceinline__ TokPar token_par(float sc, uint32_t zero_bits, bool general_form) {
    float r = __builtin_amdgcn_rcpf(sc);
    r = __fmaf_rn(__fmaf_rn(-sc, r, 1.f), r, r);
    TokPar tp;
    tp.s = sc;
    tp.r = r;
    tp.sub2 = 0;
    if (DT == PKV_F16) {
        const float z = T16<DT>::from_bits(zero_bits);        // an integer (or inf / nan for degenerate tokens)
        if (!general_form && z >= -500.f && z <= 3000.f) {
            const int zi = (int)z, odd = zi & 1;
            tp.add2 = (uint32_t)__half_as_ushort(__float2half_rn((float)(1536 + odd - zi))) * 0x00010001u;   // exact: |c| < 2048
            tp.sub2 = (uint32_t)(0x6600 + odd) * 0x00010001u;
        } else {
            tp.add2 = (zero_bits ^ 0x8000u) * 0x00010001u;
        }
    } else {
        const float z = T16<DT>::from_bits(zero_bits);        // an integer (or inf / nan for degenerate tokens)
        if (!general_form && fabsf(z) <= 1048576.f) {       // 2^23 - zero and the sums below stay exact
            tp.add2 = __float_as_uint(8388608.f - z);
            tp.sub2 = 1u;
        } else {
            tp.add2 = __float_as_uint(z);
        }
    }
    return tp;
}

// True (uniformly) when all 16 tokens of the round at `par` (LDS) take the usual case of quant4.
__device__ __forceinline__ bool round_all_fast(const TokPar *par) {
    const uint32_t sub2 = par[threadIdx.x & 15].sub2;
    return !__any(sub2 == 0u);
}

// The codes of a loaded cell (rows xr, the 16 tokens' constants at par) as pairs of 16-bit integers.
template <int DT, bool UNIFORM = true>
__device__ __forceinline__ void cell_quant(const uint2 xr[16], const TokPar *par, uint32_t c01[16], uint32_t c23[16]) {
    if (DT == PKV_F16 && round_all_fast(par)) {
#pragma unroll
        for (int k = 0; k < 16; k++) quant4_f16_fast(xr[k], par[k], c01[k], c23[k]);
    } else {
#pragma unroll
        for (int k = 0; k < 16; k++) quant4<DT, UNIFORM>(xr[k], par[k], c01[k], c23[k]);
    }
}

// The four packs of a cell's codes: words, minima, widths.
__device__ __forceinline__ void cell_build(const uint32_t c01[16], const uint32_t c23[16], UnitPacks &u, uint32_t &cmax) {
    uint32_t mn01, mn23, len01, len23, mx01, mx23;
    build_pair(c01, mn01, len01, mx01, u.word[0], u.word[1]);
    build_pair(c23, mn23, len23, mx23, u.word[2], u.word[3]);
    const u16x2 m = __builtin_elementwise_max(as_u16x2(mx01), as_u16x2(mx23));
    cmax = max((uint32_t)m[0], (uint32_t)m[1]);
    u.mn[0] = mn01 & 0xFFFFu; u.mn[1] = mn01 >> 16; u.mn[2] = mn23 & 0xFFFFu; u.mn[3] = mn23 >> 16;
    u.len[0] = len01 & 0xFFFFu; u.len[1] = len01 >> 16; u.len[2] = len23 & 0xFFFFu; u.len[3] = len23 >> 16;
}

// The four packs of a loaded cell (rows xr, the 16 tokens' constants at par): words, minima, widths.  For the round-major
// encoders: with one or three heads the halves of a wavefront serve different groups, hence different tokens, so each lane takes
// its own token's sequence.
template <int DT>
__device__ __forceinline__ void cell_packs(const uint2 xr[16], const TokPar *par, UnitPacks &u, uint32_t &cmax) {
    uint32_t c01[16], c23[16];
    if (DT == PKV_F16 && round_all_fast(par)) {
#pragma unroll
        for (int k = 0; k < 16; k++) quant4_f16_fast(xr[k], par[k], c01[k], c23[k]);
    } else {
#pragma unroll
        for (int k = 0; k < 16; k++) quant4<DT, false>(xr[k], par[k], c01[k], c23[k]);
    }
    uint32_t mn01, mn23, len01, len23, mx01, mx23;
    build_pair(c01, mn01, len01, mx01, u.word[0], u.word[1]);
    build_pair(c23, mn23, len23, mx23, u.word[2], u.word[3]);
    const u16x2 m = __builtin_elementwise_max(as_u16x2(mx01), as_u16x2(mx23));
    cmax = max((uint32_t)m[0], (uint32_t)m[1]);
    u.mn[0] = mn01 & 0xFFFFu; u.mn[1] = mn01 >> 16; u.mn[2] = mn23 & 0xFFFFu; u.mn[3] = mn23 >> 16;
    u.len[0] = len01 & 0xFFFFu; u.len[1] = len01 >> 16; u.len[2] = len23 & 0xFFFFu; u.len[3] = len23 >> 16;
}

// ---- widths 5 and 6 (extension of the format) in the round-major encoders ------------------------------------
// A pack word grows to 16 * len <= 96 bits.  It is kept as two halves of 8 * len bits -- `hi` tokens 0..7, `lo`
// tokens 8..15 -- and since 8 * len bits are len whole bytes, the word's 2 * len bytes in the stream are simply the
// bytes of `lo` followed by the bytes of `hi`.  The halves are assembled from windows of TWO tokens (2 * len <= 12
// bits fit the packed 16-bit arithmetic the quarter windows of the reference's widths use).
struct UnitPacksW {
    uint64_t lo[4], hi[4];
    uint32_t len[4];
    uint32_t mn[4];
    uint32_t off[4];
    uint32_t payload;
};

// four windows of l2 = 2 * len <= 12 bits
__device__ __forceinline__ uint64_t join4(uint32_t e0, uint32_t e1, uint32_t e2, uint32_t e3, uint32_t l2) {
    return ((uint64_t)((e0 << l2) | e1) << (2u * l2)) | ((e2 << l2) | e3);
}

__device__ __forceinline__ void build_pair_wide(const uint32_t c[16], uint32_t &mn2, uint32_t &len2, uint32_t &mx2,
                                                uint64_t &lo_a, uint64_t &hi_a, uint64_t &lo_b, uint64_t &hi_b) {
    mn2 = pk_side16<false>(c);
    mx2 = pk_side16<true>(c);
    const u16x2 mn = as_u16x2(mn2), mx = as_u16x2(mx2), one = {1, 1};
    len2 = pk_bitlen<6>(pk_u16((u16x2)(mx - mn)));
    const u16x2 p = pk_power(len2);
    const u16x2 mnrep = mn * (p + one);
    uint32_t ew[8];                                              // tokens 2j, 2j+1: (c - min) p + (c' - min) < 2^12
#pragma unroll
    for (int j = 0; j < 8; j++) ew[j] = pk_u16((u16x2)(as_u16x2(c[2 * j]) * p + as_u16x2(c[2 * j + 1]) - mnrep));
    const uint32_t l0 = 2u * (len2 & 0xFFFFu), l1 = 2u * (len2 >> 16);
    hi_a = join4(ew[0] & 0xFFFFu, ew[1] & 0xFFFFu, ew[2] & 0xFFFFu, ew[3] & 0xFFFFu, l0);
    lo_a = join4(ew[4] & 0xFFFFu, ew[5] & 0xFFFFu, ew[6] & 0xFFFFu, ew[7] & 0xFFFFu, l0);
    hi_b = join4(ew[0] >> 16, ew[1] >> 16, ew[2] >> 16, ew[3] >> 16, l1);
    lo_b = join4(ew[4] >> 16, ew[5] >> 16, ew[6] >> 16, ew[7] >> 16, l1);
}

__device__ __forceinline__ void cell_build(const uint32_t c01[16], const uint32_t c23[16], UnitPacksW &u, uint32_t &cmax) {
    uint32_t mn01, mn23, len01, len23, mx01, mx23;
    build_pair_wide(c01, mn01, len01, mx01, u.lo[0], u.hi[0], u.lo[1], u.hi[1]);
    build_pair_wide(c23, mn23, len23, mx23, u.lo[2], u.hi[2], u.lo[3], u.hi[3]);
    const u16x2 m = __builtin_elementwise_max(as_u16x2(mx01), as_u16x2(mx23));
    cmax = max((uint32_t)m[0], (uint32_t)m[1]);
    u.mn[0] = mn01 & 0xFFFFu; u.mn[1] = mn01 >> 16; u.mn[2] = mn23 & 0xFFFFu; u.mn[3] = mn23 >> 16;
    u.len[0] = len01 & 0xFFFFu; u.len[1] = len01 >> 16; u.len[2] = len23 & 0xFFFFu; u.len[3] = len23 >> 16;
}

template <int DT>
__device__ __forceinline__ void cell_packs(const uint2 xr[16], const TokPar *par, UnitPacksW &u, uint32_t &cmax) {
    uint32_t c01[16], c23[16];
    if (DT == PKV_F16 && round_all_fast(par)) {
#pragma unroll
        for (int k = 0; k < 16; k++) quant4_f16_fast(xr[k], par[k], c01[k], c23[k]);
    } else {
#pragma unroll
        for (int k = 0; k < 16; k++) quant4<DT, false>(xr[k], par[k], c01[k], c23[k]);
    }
    uint32_t mn01, mn23, len01, len23, mx01, mx23;
    build_pair_wide(c01, mn01, len01, mx01, u.lo[0], u.hi[0], u.lo[1], u.hi[1]);
    build_pair_wide(c23, mn23, len23, mx23, u.lo[2], u.hi[2], u.lo[3], u.hi[3]);
    const u16x2 m = __builtin_elementwise_max(as_u16x2(mx01), as_u16x2(mx23));
    cmax = max((uint32_t)m[0], (uint32_t)m[1]);
    u.mn[0] = mn01 & 0xFFFFu; u.mn[1] = mn01 >> 16; u.mn[2] = mn23 & 0xFFFFu; u.mn[3] = mn23 >> 16;
    u.len[0] = len01 & 0xFFFFu; u.len[1] = len01 >> 16; u.len[2] = len23 & 0xFFFFu; u.len[3] = len23 >> 16;
}

template <bool WIDE> struct PacksOf { typedef UnitPacks type; };
template <> struct PacksOf<true> { typedef UnitPacksW type; };

// the 2 * len bytes of pack k at dst (2-byte aligned, in LDS): one 16-bit store per piece by the lanes whose pack has that piece.
// A longer pack has the pieces of a shorter one, so every compare narrows the execution mask of the one before and the mask
// is put back once per pack.  Written as instructions: the compiler made a branch to a block of its own and one back
// out of every predicated store, 32 of them a round.  It does not see these stores either: packs_put() stands before the barrier behind
// the last ones.  (Behind a lane's last pack the s_nop fills up the five wait states that an exchange between lanes needs after a
// vector instruction wrote the mask.)
// The encoders are bound by the instructions they issue: these stores, the widths and windows above and the minima and maxima
// below (fewer wait states) took 4 % off K, 4 % off V on 16 x 8 x 32768 tokens (fp16, rel 0.1: 322 -> 309, 352 -> 339 us), 3 and 7 % at
// rel 0.05 with its wide packs (329 -> 318, 508 -> 475).
__device__ __forceinline__ uint32_t lds_offset(const void *p) {
    return (uint32_t)reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) void *)p);
}
__device__ __forceinline__ void put_pack(uint16_t *dst, const UnitPacks &u, int k) {
    uint64_t mask;
    asm volatile("s_mov_b64 %0, exec\n\t"
                 "v_cmpx_lt_u32_e32 vcc, 0, %4\n\t"
                 "ds_write_b16 %1, %2\n\t"
                 "v_cmpx_lt_u32_e32 vcc, 1, %4\n\t"
                 "ds_write_b16_d16_hi %1, %2 offset:2\n\t"
                 "v_cmpx_lt_u32_e32 vcc, 2, %4\n\t"
                 "ds_write_b16 %1, %3 offset:4\n\t"
                 "v_cmpx_lt_u32_e32 vcc, 3, %4\n\t"
                 "ds_write_b16_d16_hi %1, %3 offset:6\n\t"
                 "s_mov_b64 exec, %0"
                 : "=&s"(mask)
                 : "v"(lds_offset(dst)), "v"((uint32_t)u.word[k]), "v"((uint32_t)(u.word[k] >> 32)), "v"(u.len[k])
                 : "vcc", "memory");
    if (k == 3) asm volatile("s_nop 2");
}
__device__ __forceinline__ void put_pack(uint16_t *dst, const UnitPacksW &u, int k) {
    const uint32_t s = 8u * u.len[k];                            // (at most 48; without pieces nothing is stored)
    const uint64_t w = u.lo[k] | (u.hi[k] << s);
    uint64_t mask;
    asm volatile("s_mov_b64 %0, exec\n\t"
                 "v_cmpx_lt_u32_e32 vcc, 0, %5\n\t"
                 "ds_write_b16 %1, %2\n\t"
                 "v_cmpx_lt_u32_e32 vcc, 1, %5\n\t"
                 "ds_write_b16_d16_hi %1, %2 offset:2\n\t"
                 "v_cmpx_lt_u32_e32 vcc, 2, %5\n\t"
                 "ds_write_b16 %1, %3 offset:4\n\t"
                 "v_cmpx_lt_u32_e32 vcc, 3, %5\n\t"
                 "ds_write_b16_d16_hi %1, %3 offset:6\n\t"
                 "v_cmpx_lt_u32_e32 vcc, 4, %5\n\t"
                 "ds_write_b16 %1, %4 offset:8\n\t"
                 "v_cmpx_lt_u32_e32 vcc, 5, %5\n\t"
                 "ds_write_b16_d16_hi %1, %4 offset:10\n\t"
                 "s_mov_b64 exec, %0"
                 : "=&s"(mask)
                 : "v"(lds_offset(dst)), "v"((uint32_t)w), "v"((uint32_t)(w >> 32)), "v"((uint32_t)(u.hi[k] >> ((64u - s) & 63u))), "v"(u.len[k])
                 : "vcc", "memory");
    if (k == 3) asm volatile("s_nop 2");
}
__device__ __forceinline__ void packs_put() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// Emit one analysed unit at blk[unit_off] (the K layout: lane t's packs sit where they were computed).
template <class U>
__device__ __forceinline__ void unit_emit_any(uint8_t *blk, uint32_t unit_off, int t, const UnitGeom g, const U &u) {
    uint32_t minsw = 0, lensw = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        minsw |= u.mn[i] << (i * g.W);
        lensw |= u.len[i] << (i * g.LB);
    }
    lds_put_meta(blk + unit_off, t, g.W, minsw);
    lds_put_meta(blk + unit_off + g.mins_bytes, t, g.LB, lensw);
    uint8_t *pay = blk + unit_off + g.mins_bytes + g.lens_bytes;
#pragma unroll
    for (int i = 0; i < 4; i++) put_pack(reinterpret_cast<uint16_t *>(pay + u.off[i]), u, i);
}

// A group is the run of blocks that share one (context block, sequence): H blocks for K, 2 H for V, consecutive in
// stream order.  The encoders below give a workgroup the blocks of up to eight heads of a group.
constexpr int kSubBlocks = 8;

// Wave priorities (s_setprio) of the round-major encoders' phases: the parameter pass goes first, so that its rows
// are requested from HBM as early as possible; forming the packs, the long arithmetic phase, yields to everything
// else.  Worth 3-4 % (0.392 -> 0.377 ms for K, 0.431 -> 0.414 ms for V on 1 GiB of input).
#ifndef PKV_EPRIO_STAT
#define PKV_EPRIO_STAT 3
#define PKV_EPRIO_PACK 0
#define PKV_EPRIO_EMIT 2
#endif

// Copy n bytes (even) from LDS (src 4-byte aligned, readable up to 20 bytes past n) to global memory (dst 2-byte
// aligned) with `N` threads, t = 0 .. N - 1 of them: head to the first 16-byte boundary and tail in 2-byte pieces, the
// body as aligned 16-byte stores fed by aligned LDS reads and byte funnel shifts.
template <int N>
__device__ __forceinline__ void copy_out(uint8_t *dst, const uint8_t *src, uint32_t n, int t) {
    const uint32_t head = min(n, (uint32_t)((16u - (uint32_t)(reinterpret_cast<uintptr_t>(dst) & 15u)) & 15u));
    const uint32_t nq = (n - head) >> 4;
    for (uint32_t i = t; i < (head >> 1); i += N)
        reinterpret_cast<uint16_t *>(dst)[i] = reinterpret_cast<const uint16_t *>(src)[i];
    const uint32_t *src32 = reinterpret_cast<const uint32_t *>(src + (head & ~3u));
    for (uint32_t i = t; i < nq; i += N) {
        const uint32_t *q = src32 + 4 * i;
        const uint32_t d0 = q[0], d1 = q[1], d2 = q[2], d3 = q[3], d4 = q[4];
        uint4 v;
        v.x = __builtin_amdgcn_alignbyte(d1, d0, head);
        v.y = __builtin_amdgcn_alignbyte(d2, d1, head);
        v.z = __builtin_amdgcn_alignbyte(d3, d2, head);
        v.w = __builtin_amdgcn_alignbyte(d4, d3, head);
        *reinterpret_cast<uint4 *>(dst + head + 16 * (size_t)i) = v;
    }
    const uint32_t done = head + 16u * nq;
    for (uint32_t i = t; i < ((n - done) >> 1); i += N)
        reinterpret_cast<uint16_t *>(dst + done)[i] = reinterpret_cast<const uint16_t *>(src + done)[i];
}
__device__ __forceinline__ void copy_out32(uint8_t *dst, const uint8_t *src, uint32_t n, int t) { copy_out<32>(dst, src, n, t); }

// Minimum and maximum of every token of a round over a wavefront's cells.  Lane's cell: rows xr[k] = token
// k, four channels.  The 16 per-token values of a lane are reduced and transposed at once: each step exchanges half
// of the registers with the lane 32, 16, 8, 4 positions away and keeps the other half, so the register count halves
// while the lanes behind a value double -- v_permlane32_swap / v_permlane16_swap trade whole half-wavefronts and
// rows between two registers, the two steps inside a row are DPP moves under bank masks.  Afterwards lane l holds
// token l / 4 (all four lanes of a quad the same): ~120 vector instructions instead of a second pass over the rows.
// (The packed min / max are written as instructions, see pk_min_h; a lane exchange must not read a register that a
// vector instruction wrote less than two instructions earlier, and the compiler does not see into the assembly, so
// these carry their own two wait states, one for four of them where four are independent: with two behind each of the 62 a round
// they held a wavefront for 250 cycles.)
// KEYS: the operands are order keys of bf16 values (bf16_keys), compared as signed 16-bit integers.
template <bool MAX, bool KEYS>
__device__ __forceinline__ uint32_t pk_sel_x(uint32_t a, uint32_t b) {
    uint32_t r;
    if (KEYS) {
        if (MAX) asm("v_pk_max_i16 %0, %1, %2\n\ts_nop 1" : "=v"(r) : "v"(a), "v"(b));
        else asm("v_pk_min_i16 %0, %1, %2\n\ts_nop 1" : "=v"(r) : "v"(a), "v"(b));
    } else {
        if (MAX) asm("v_pk_max_f16 %0, %1, %2\n\ts_nop 1" : "=v"(r) : "v"(a), "v"(b));
        else asm("v_pk_min_f16 %0, %1, %2\n\ts_nop 1" : "=v"(r) : "v"(a), "v"(b));
    }
    return r;
}
// bf16 has no packed min / max: both halves of a word become 16-bit integers that order like the values (negative
// values have their magnitude bits flipped); the map is its own inverse.
__device__ __forceinline__ uint32_t bf16_keys(uint32_t w) {
    typedef short i16x2 __attribute__((ext_vector_type(2)));
    const i16x2 v = __builtin_bit_cast(i16x2, w);
    const i16x2 m = (v >> (short)15) & (short)0x7FFF;
    return __builtin_bit_cast(uint32_t, (i16x2)(v ^ m));
}
// A token's (minimum, maximum) as one word that a packed MINIMUM combines: the minimum in the low half, the negated
// maximum in the high half (fp16: sign bit flipped; bf16: both as order keys, the maximum's complemented).
template <int DT>
__device__ __forceinline__ uint32_t minmax_word(float mn, float mx) {
    if (DT == PKV_F16) return T16<DT>::to_bits(mn) | ((T16<DT>::to_bits(mx) ^ 0x8000u) << 16);
    return bf16_keys(T16<DT>::to_bits(mn) | (T16<DT>::to_bits(mx) << 16)) ^ 0xFFFF0000u;
}
template <int DT>
__device__ __forceinline__ void minmax_unword(uint32_t w, float &mn, float &mx) {
    if (DT != PKV_F16) w = bf16_keys(w ^ 0xFFFF0000u);
    else w ^= 0x80000000u;
    mn = T16<DT>::from_bits(w & 0xFFFFu);
    mx = T16<DT>::from_bits(w >> 16);
}
// Four of them with the wait states once, behind the last: a[i] = min / max(a[i], b[i]).
template <bool MAX, bool KEYS>
__device__ __forceinline__ void pk_sel4(uint32_t &a0, uint32_t &a1, uint32_t &a2, uint32_t &a3, uint32_t b0, uint32_t b1, uint32_t b2, uint32_t b3) {
#define PKV_SEL4(op)                                                                                                                      \
    asm(op " %0, %0, %4\n\t" op " %1, %1, %5\n\t" op " %2, %2, %6\n\t" op " %3, %3, %7\n\ts_nop 1"                                         \
        : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3) : "v"(b0), "v"(b1), "v"(b2), "v"(b3))
    if (KEYS) {
        if (MAX) PKV_SEL4("v_pk_max_i16");
        else PKV_SEL4("v_pk_min_i16");
    } else {
        if (MAX) PKV_SEL4("v_pk_max_f16");
        else PKV_SEL4("v_pk_min_f16");
    }
#undef PKV_SEL4
}
// v[i] = min / max over the two dwords of row xr[first + i], rows first .. first + 3
template <int DT, bool MAX>
__device__ __forceinline__ void rows_sel4(const uint2 xr[16], int first, uint32_t (&v)[4]) {
    constexpr bool KEYS = DT != PKV_F16;
    if (KEYS) {
        uint32_t b[4];
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = bf16_keys(xr[first + i].x), b[i] = bf16_keys(xr[first + i].y);
        pk_sel4<MAX, true>(v[0], v[1], v[2], v[3], b[0], b[1], b[2], b[3]);
    } else {
#define PKV_ROWS4(op)                                                                                                                     \
    asm(op " %0, %4, %5\n\t" op " %1, %6, %7\n\t" op " %2, %8, %9\n\t" op " %3, %10, %11\n\ts_nop 1"                                       \
        : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])                                                                               \
        : "v"(xr[first].x), "v"(xr[first].y), "v"(xr[first + 1].x), "v"(xr[first + 1].y), "v"(xr[first + 2].x), "v"(xr[first + 2].y),        \
          "v"(xr[first + 3].x), "v"(xr[first + 3].y))
        if (MAX) PKV_ROWS4("v_pk_max_f16");
        else PKV_ROWS4("v_pk_min_f16");
#undef PKV_ROWS4
    }
}
// a[i] = min / max after halves of the wavefront (rows of 16) of a[i] and b[i] have changed places
template <bool MAX, bool KEYS, bool HALVES>
__device__ __forceinline__ void swap_sel4(uint32_t (&a)[4], const uint32_t (&b)[4]) {
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const auto r = HALVES ? __builtin_amdgcn_permlane32_swap(a[i], b[i], false, false) : __builtin_amdgcn_permlane16_swap(a[i], b[i], false, false);
        a[i] = (uint32_t)r[0];
        o[i] = (uint32_t)r[1];
    }
    pk_sel4<MAX, KEYS>(a[0], a[1], a[2], a[3], o[0], o[1], o[2], o[3]);
}
// lanes whose bank is in HI_BANKS keep b and meet the partner's b, the others keep a and meet the partner's a;
// CTRL_LO / CTRL_HI: how the low / high banks read their partner
template <bool MAX, bool KEYS, int CTRL_LO, int CTRL_HI, int HI_BANKS>
__device__ __forceinline__ uint32_t row_step_sel(uint32_t a, uint32_t b) {
    const int mine = __builtin_amdgcn_update_dpp((int)a, (int)b, 0xE4, 0xF, HI_BANKS, false);
    int theirs = __builtin_amdgcn_update_dpp(0, (int)a, CTRL_LO, 0xF, 0xF ^ HI_BANKS, false);
    theirs = __builtin_amdgcn_update_dpp(theirs, (int)b, CTRL_HI, 0xF, HI_BANKS, false);
    return pk_sel_x<MAX, KEYS>((uint32_t)mine, (uint32_t)theirs);
}
// one side (minimum or maximum) of cell_token_minmax as packed halves: lane l holds token l / 4, two channel parities
template <int DT, bool MAX>
__device__ __forceinline__ uint32_t cell_token_side(const uint2 xr[16]) {
    constexpr bool KEYS = DT != PKV_F16;
    uint32_t v[4], w[4], q[4];
    rows_sel4<DT, MAX>(xr, 0, v);
    rows_sel4<DT, MAX>(xr, 8, q);
    swap_sel4<MAX, KEYS, true>(v, q);                      // lanes 0..31: token k, lanes 32..63: token k + 8
    rows_sel4<DT, MAX>(xr, 4, w);
    rows_sel4<DT, MAX>(xr, 12, q);
    swap_sel4<MAX, KEYS, true>(w, q);
    swap_sel4<MAX, KEYS, false>(v, w);                     // row rho: token k + 4 rho
#pragma unroll
    for (int k = 0; k < 2; k++) v[k] = row_step_sel<MAX, KEYS, 0x128, 0x128, 0xC>(v[k], v[k + 2]);   // lanes 8..15 of a row: token k + 2 + 4 rho
    const uint32_t r = row_step_sel<MAX, KEYS, 0x104, 0x114, 0xA>(v[0], v[1]);         // banks 1, 3: the odd token; token = lane / 4
    return KEYS ? bf16_keys(r) : r;
}
template <int DT>
__device__ __forceinline__ void cell_token_minmax(const uint2 xr[16], float &mn, float &mx) {
    const uint32_t lo = cell_token_side<DT, false>(xr);
    __builtin_amdgcn_sched_barrier(0);                     // (one side after the other: 16 registers in flight, not 32)
    const uint32_t hi = cell_token_side<DT, true>(xr);
    mn = fminf(T16<DT>::from_bits(lo & 0xFFFFu), T16<DT>::from_bits(lo >> 16));
    mx = fmaxf(T16<DT>::from_bits(hi & 0xFFFFu), T16<DT>::from_bits(hi >> 16));
    asm("s_nop 1\n\t"
        "v_min_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_max_f32_dpp %1, %1, %1 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 0\n\t"
        "v_min_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_max_f32_dpp %1, %1, %1 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf"
        : "+v"(mn), "+v"(mx));
}

// The same for a wavefront whose two halves hold different rounds (lanes 0..31 the tokens of one round, lanes 32..63
// those of the next): the reduction stays inside the halves -- rows, then 8, 4 and 2 lanes -- and lane l ends up
// with token l / 2 of the 32.
template <int DT, bool MAX>
__device__ __forceinline__ uint32_t cell_token_side_halves(const uint2 xr[16], bool odd_pair) {
    constexpr bool KEYS = DT != PKV_F16;
    uint32_t v[4], w[4], q[4];
    rows_sel4<DT, MAX>(xr, 0, v);
    rows_sel4<DT, MAX>(xr, 8, q);
    swap_sel4<MAX, KEYS, false>(v, q);                     // odd rows: token k + 8
    rows_sel4<DT, MAX>(xr, 4, w);
    rows_sel4<DT, MAX>(xr, 12, q);
    swap_sel4<MAX, KEYS, false>(w, q);
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] = row_step_sel<MAX, KEYS, 0x128, 0x128, 0xC>(v[k], w[k]);       // lanes 8..15 of a row: + 4
#pragma unroll
    for (int k = 0; k < 2; k++) v[k] = row_step_sel<MAX, KEYS, 0x104, 0x114, 0xA>(v[k], v[k + 2]);   // banks 1, 3: + 2
    // lanes 2, 3 of a quad: + 1 (no bank mask reaches inside a quad: selects, and the exchange as a quad permute)
    const uint32_t mine = odd_pair ? v[1] : v[0], send = odd_pair ? v[0] : v[1];
    const uint32_t theirs = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)send, 0x4E, 0xF, 0xF, false);
    const uint32_t r = pk_sel_x<MAX, KEYS>(mine, theirs);
    return KEYS ? bf16_keys(r) : r;
}
template <int DT>
__device__ __forceinline__ void cell_token_minmax_halves(const uint2 xr[16], float &mn, float &mx) {
    const bool odd_pair = (threadIdx.x & 2) != 0;
    const uint32_t lo = cell_token_side_halves<DT, false>(xr, odd_pair);
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t hi = cell_token_side_halves<DT, true>(xr, odd_pair);
    mn = fminf(T16<DT>::from_bits(lo & 0xFFFFu), T16<DT>::from_bits(lo >> 16));
    mx = fmaxf(T16<DT>::from_bits(hi & 0xFFFFu), T16<DT>::from_bits(hi >> 16));
    asm("s_nop 1\n\t"
        "v_min_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_max_f32_dpp %1, %1, %1 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf"
        : "+v"(mn), "+v"(mx));
}

constexpr uint64_t kCloseCells = 2048;       // workgroups of one side's launch, at most (encode_closes)
// The end of a launch that closes by itself (ClosedEncode): every workgroup counts itself out, sixteen to a counter and the sixteens on
// one (adding to one address takes 13 ns each, one after the other), and the last one leaves the outcome and clears the state.
// Behind `waitcnt` this wavefront's accesses to the state have arrived.  The output has not: its lines may stay in this XCD's L2 until
// the launch ends, so a host that learned of the end from here could read the stream's old bytes through another stream.
__device__ __forceinline__ void encode_close(const EncodeClose &c, uint32_t &last_of_all) {
    if (c.total == 0) return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t group = blockIdx.x / kCloseGroup, groups = (c.total + kCloseGroup - 1u) / kCloseGroup;
        auto count = [&](uint32_t at) { return __hip_atomic_fetch_add(reinterpret_cast<uint32_t *>(c.count + kCloseStride * at), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u; };
        const bool last = count(1u + group) == min(kCloseGroup, c.total - group * kCloseGroup) && count(0u) == groups;
        if (last) publish_outcomes(c.st, nullptr, c.last, nullptr, c.tag, 0);
        last_of_all = last ? 1u : 0u;
    }
    __syncthreads();
    if (last_of_all == 0u) return;
    // (ordinary stores: nothing reads the state any more before the launch has ended)
    for (uint32_t i = threadIdx.x; i < c.n / 2u; i += blockDim.x) reinterpret_cast<uint4 *>(c.st)[i] = make_uint4(0u, 0u, 0u, 0u);
    if (threadIdx.x == 0 && (c.n & 1u)) reinterpret_cast<uint64_t *>(c.st)[c.n - 1u] = 0;
}

// ---- K, all heads in one workgroup, x read ONCE as cells ----------------------------------------
// The round-major encoder above reads a round's rows twice: once row-wise for the token parameters (the trip that
// goes to HBM and whose latency every round waits out) and again as cells.  Here a round is read as cells only; the
// token minima and maxima come from the cell registers (cell_token_minmax: per wavefront, then four partial
// results per token through LDS, from which every wavefront forms the round's parameters for itself, so a round
// has one barrier), and the next round's cells are requested as soon as this round's are quantized -- into the same
// registers -- so that they travel while the packs are formed and emitted.  For 5..8 heads (one group per
// workgroup); PERM as in the round-major kernel.  Same stream, parameters and block_info as that kernel.
// ROT: the rows get their rotary embedding on the way (cell_rotate) -- a prompt's keys are then read once where they are,
// instead of being rotated into a buffer of their own size first.  The arithmetic costs the encoder 90 us on 512 MiB of
// bf16 (196 -> 287 us, bound by the vector units), the pass it saves took 190.
// The 256 threads `tid` of a workgroup of their own, or of one that holds two such groups (both have one: they meet at the barriers).
struct KCellsLds {
    uint32_t idx;
    uint64_t off;
    uint32_t blk_off[kSubBlocks + 1];
    __attribute__((aligned(16))) TokPar par[4 * 16];       // [wavefront][token of the round]
    float2 mm[2][4][16];                                   // [round parity][wavefront][token]: (min, max)
};
template <int DT, bool WIDE, bool PERM, bool XCH, bool STRIDED, bool ROT>
__device__ __forceinline__ void k_quant_encode_cells(
    const int tid, uint8_t *const gbuf, KCellsLds &lds, const uint16_t *__restrict__ x, int B, int H, int T, const XRows xs, float rel, uint16_t *__restrict__ scale,
    uint16_t *__restrict__ zero, uint8_t *__restrict__ stream, uint64_t capacity, uint32_t *__restrict__ info,
    ScanState *st, int W, uint32_t ngroups, uint32_t bound, uint64_t base, int par_stride,
    const uint32_t *__restrict__ perm, int perm_block, const Stagger stagger, int nsg, uint64_t *xw, const Rot rot) {
    uint64_t &s_off = lds.off;
    uint32_t *const blk_off = lds.blk_off;
    TokPar *const s_par = lds.par;
    auto &s_mm = lds.mm;
    stagger_first_generation(stagger);
    if (tid == 0) lds.idx = atomicAdd(&st->ticket, 1u);
    __syncthreads();
    const uint32_t gidx = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds.idx);
    if (gidx >= ngroups) return;
    // XCH (more than eight heads): runs of eight heads, one workgroup and one ticket each, as in the round-major
    // kernel: a run forms the minima and maxima over its own heads, publishes them per token and collects the others'.
    const int H_all = H;
    const uint32_t sgi = XCH ? gidx % (uint32_t)nsg : 0u;
    const int hbase = XCH ? 8 * (int)sgi : 0;
    if (XCH) H = min(8, H_all - hbase);
    const int j = tid >> 5, t = tid & 31, wave = tid >> 6, lane = tid & 63;
    const uint32_t grp = XCH ? gidx / (uint32_t)nsg : gidx;
    const uint32_t cb = grp / (uint32_t)B, b = grp % (uint32_t)B;
    const size_t tok0 = (size_t)cb * 64;
    const UnitGeom g = unit_geom(W);
    const bool active = j < H;
    const int jc = min(j, H - 1);                          // (a repeated head changes no minimum or maximum)
    const TokPar *my_par = XCH ? s_par : s_par + 16 * wave;
    uint8_t *blk = gbuf + (size_t)j * bound;
    uint32_t my_off = 8u;
    uint32_t cmax_all = 0;
    // (a wavefront holds two heads: rows of the ordinary stride hang off a per-lane pointer, others off the scalar base of
    // the first head)
    const int j0 = STRIDED ? min(2 * __builtin_amdgcn_readfirstlane(wave), H - 1) : jc;
    const char *cells = reinterpret_cast<const char *>(x + b * xs.sb + (hbase + j0) * xs.sh + (int64_t)tok0 * (STRIDED ? xs.st : kHeadDim) + (STRIDED ? 0 : 4 * t));
    const uint32_t cell_off = STRIDED ? ((uint32_t)(jc - j0) * (uint32_t)xs.sh + 4u * (uint32_t)t) * 2u : 0u;
    const int64_t row_bytes = STRIDED ? 2 * xs.st : 2 * kHeadDim;
    // PERM: the rows of a round are tokens perm[...] of the repacking block that holds this context block
    const uint16_t *pseq = x + (((size_t)b * H) * T + (tok0 / (size_t)(PERM ? perm_block : 1)) * (size_t)(PERM ? perm_block : 1)) * kHeadDim;
    const uint32_t plane = (uint32_t)(((size_t)jc * T * kHeadDim + 4 * t) * 2);
    // (bf16 with the wide packs or with the exchange between runs would need more than 128 registers to keep a round
    // in flight: it asks at the top)
    constexpr bool AHEAD = !((WIDE || XCH) && DT != PKV_F16);
    uint2 xr[16];
    if (AHEAD) {
        if (PERM) cell_load_rows(pseq, perm + tok0, (uint32_t)perm_block - 1u, plane, xr);
        else cell_load(cells, row_bytes, cell_off, xr);
    }
#pragma unroll 1
    for (int r = 0; r < 4; r++) {
        if (!AHEAD) {
            if (PERM) cell_load_rows(pseq, perm + tok0 + 16 * r, (uint32_t)perm_block - 1u, plane, xr);
            else cell_load(cells + r * 16 * row_bytes, row_bytes, cell_off, xr);
        }
        __builtin_amdgcn_s_setprio(PKV_EPRIO_STAT);
        if (ROT) {
            const int64_t row = (int64_t)b * rot.sb + (int64_t)(tok0 + 16 * (size_t)r) * kHeadDim;
            uint32_t lt = (uint32_t)t;                     // (what follows from it is formed here, not kept through the loop: bf16 has 128
            asm volatile("" : "+v"(lt));                   // registers in use)
            cell_rotate<DT>(reinterpret_cast<const char *>(rot.cos + row), reinterpret_cast<const char *>(rot.sin + row), 8u * lt, lt >= 16u, xr);
        }
        {
            float mn, mx;
            cell_token_minmax<DT>(xr, mn, mx);
            if ((lane & 3) == 0) s_mm[r & 1][wave][lane >> 2] = make_float2(mn, mx);
        }
        __syncthreads();
        if (XCH) {
            if (wave == 0) {
                const int tk = lane & 15;
                const float2 p0 = s_mm[r & 1][0][tk], p1 = s_mm[r & 1][1][tk], p2 = s_mm[r & 1][2][tk], p3 = s_mm[r & 1][3][tk];
                const float rmn = fminf(fminf(p0.x, p1.x), fminf(p2.x, p3.x)), rmx = fmaxf(fmaxf(p0.y, p1.y), fmaxf(p2.y, p3.y));
                uint64_t *words = xw + ((size_t)(gidx - sgi) * 4 + r) * 16;       // [run][round][token] of this group
                if (lane < 16)
                    __hip_atomic_store(words + (size_t)sgi * 64 + lane, (1ull << 63) | ((uint64_t)T16<DT>::to_bits(rmn) << 16) | (uint64_t)T16<DT>::to_bits(rmx),
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                // lane = (run, token) for up to four runs at a time
                float amn = INFINITY, amx = -INFINITY;
                for (int s0 = 0; s0 < nsg; s0 += 4) {
                    const int run = s0 + (lane >> 4);
                    if (run < nsg) {
                        const uint64_t *wp = words + (size_t)run * 64 + tk;
                        uint64_t w = __hip_atomic_load(wp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        int spins = 0;
                        while ((w >> 63) == 0 && spins < kSpinLimit) {
                            __builtin_amdgcn_s_sleep(8);
                            w = __hip_atomic_load(wp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            spins++;
                        }
                        if ((w >> 63) == 0) atomicExch(&st->error, (uint32_t)PKV_ERR_INTERNAL);     // (bounded wait: the host reports it)
                        amn = fminf(amn, T16<DT>::from_bits((uint32_t)(w >> 16) & 0xFFFFu));
                        amx = fmaxf(amx, T16<DT>::from_bits((uint32_t)w & 0xFFFFu));
                    }
                }
                amn = fminf(amn, __shfl_xor(amn, 16, 64)); amx = fmaxf(amx, __shfl_xor(amx, 16, 64));
                amn = fminf(amn, __shfl_xor(amn, 32, 64)); amx = fmaxf(amx, __shfl_xor(amx, 32, 64));
                if (lane < 16) {
                    const float range = round_t<DT>(amx - amn);
                    const float sc = round_t<DT>(range * rel);
                    const uint32_t zb = T16<DT>::to_bits(rintf(round_t<DT>(__fdiv_rn(amn, sc))));
                    if (sgi == 0) {
                        const size_t tok = (size_t)b * par_stride + tok0 + 16 * r + lane;
                        scale[tok] = (uint16_t)T16<DT>::to_bits(sc);
                        zero[tok] = (uint16_t)zb;
                    }
                    s_par[lane] = token_par<DT>(sc, zb, false);
                }
            }
            __syncthreads();
        } else if (lane < 16) {
            const float2 p0 = s_mm[r & 1][0][lane], p1 = s_mm[r & 1][1][lane], p2 = s_mm[r & 1][2][lane], p3 = s_mm[r & 1][3][lane];
            const float mn = fminf(fminf(p0.x, p1.x), fminf(p2.x, p3.x)), mx = fmaxf(fmaxf(p0.y, p1.y), fmaxf(p2.y, p3.y));
            const float range = round_t<DT>(mx - mn);
            const float sc = round_t<DT>(range * rel);
            const uint32_t zb = T16<DT>::to_bits(rintf(round_t<DT>(__fdiv_rn(mn, sc))));
            if (wave == 0) {
                const size_t tok = (size_t)b * par_stride + tok0 + 16 * r + lane;
                scale[tok] = (uint16_t)T16<DT>::to_bits(sc);
                zero[tok] = (uint16_t)zb;
            }
            s_par[16 * wave + lane] = token_par<DT>(sc, zb, false);
        }
        wave_lds_order();
        __builtin_amdgcn_s_setprio(PKV_EPRIO_PACK);
        uint32_t c01[16], c23[16];
        cell_quant<DT>(xr, my_par, c01, c23);
        if (AHEAD && r < 3) {                              // travels while the packs are formed
            if (PERM) cell_load_rows(pseq, perm + tok0 + 16 * (r + 1), (uint32_t)perm_block - 1u, plane, xr);
            else cell_load(cells + (r + 1) * 16 * row_bytes, row_bytes, cell_off, xr);
        }
        typename PacksOf<WIDE>::type u;
        uint32_t cmax;
        cell_build(c01, c23, u, cmax);
        __builtin_amdgcn_s_setprio(PKV_EPRIO_EMIT);
        pack_offsets(u.len, u.off, u.payload);
        const uint32_t usz = (uint32_t)(g.mins_bytes + g.lens_bytes) + u.payload;
        if (r == 3) {
            // every block's final size is known before its last unit is written: the group's size is published now
            if (active && t == 0) blk_off[j + 1] = my_off + usz;
            if (tid == 0) blk_off[0] = 0;
            __syncthreads();
            if (tid == 0) {
                for (int q = 1; q <= H; q++) blk_off[q] += blk_off[q - 1];
                lookback_publish(st, gidx, blk_off[H]);
            }
        }
        if (active) {
            cmax_all = max(cmax_all, cmax);
            if (t == 0) reinterpret_cast<uint16_t *>(blk)[r] = (uint16_t)(my_off - 8u + usz);
            unit_emit_any(blk, my_off, t, g, u);
            my_off += usz;
        }
    }
    if (__any(cmax_all >= (1u << W))) {   // codes that do not fit W bits are an error the host reports
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) cmax_all = max(cmax_all, __shfl_xor(cmax_all, d, 64));
        if ((tid & 63) == 0) atomicMax(&st->max_code, cmax_all);
    }
    packs_put();
    __syncthreads();
    const uint32_t bytes = blk_off[H];
    if (tid < 64) {
        const uint64_t off = base + lookback_offset(st, gidx, bytes, true);
        if (tid == 0) {
            s_off = off;
            if (gidx == ngroups - 1) __hip_atomic_store(&st->total, off + bytes, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (off + bytes > capacity) atomicExch(&st->error, (uint32_t)PKV_ERR_CAPACITY);
        }
    }
    __syncthreads();
    const uint64_t off = s_off;
    if (off + bytes > capacity) return;
    if (tid < H) {
        const uint32_t first = XCH ? grp * (uint32_t)H_all + (uint32_t)hbase : gidx * (uint32_t)H;      // block index = group * heads + head
        info[2 * (size_t)(first + tid)] = (uint32_t)(off + blk_off[tid]);
        info[2 * (size_t)(first + tid) + 1] = blk_off[tid + 1] - blk_off[tid];
    }
    if (active) copy_out32(stream + off + blk_off[j], blk, my_off, t);
}

template <int DT, bool WIDE, bool PERM, bool XCH = false, bool STRIDED = false, bool ROT = false>
__global__ void __launch_bounds__(256) k_quant_encode_cells_kernel(
    const uint16_t *__restrict__ x, int B, int H, int T, const XRows xs, float rel, uint16_t *__restrict__ scale,
    uint16_t *__restrict__ zero, uint8_t *__restrict__ stream, uint64_t capacity, uint32_t *__restrict__ info,
    ScanState *st, int W, uint32_t ngroups, uint32_t bound, uint64_t base, int par_stride,
    const uint32_t *__restrict__ perm, int perm_block, const Stagger stagger, int nsg, uint64_t *xw, const Rot rot, const EncodeClose c) {
    extern __shared__ __align__(16) uint8_t gbuf[];        // H block slots of `bound` bytes
    __shared__ KCellsLds lds;
    k_quant_encode_cells<DT, WIDE, PERM, XCH, STRIDED, ROT>(threadIdx.x, gbuf, lds, x, B, H, T, xs, rel, scale, zero, stream, capacity,
                                                                   info, st, W, ngroups, bound, base, par_stride, perm, perm_block, stagger,
                                                                   nsg, xw, rot);
    if (!XCH) encode_close(c, lds.idx);                     // (runs that wait for each other are closed by finish_encode)
}

// ---- K, up to four heads: round-major, several groups to a workgroup ---------------------------
// The eight blocks a workgroup of 256 threads owns (block j = tid / 32, lane t = tid % 32) are here the H <= 4 heads
// of gpw = 8 / H (rounded down) consecutive (context block, sequence) groups -- consecutive in the stream too -- so
// that all eight half-wavefronts have a block.  The workgroup goes through its groups ROUND BY ROUND (16 tokens):
// it reads the round's rows row-wise for the token parameters (round_token_params_few, one group after the other),
// then at once re-reads them as cells -- the lines are still in L2 -- quantizes, and emits unit `round` of every
// block behind the units already there.  x crosses HBM once.  Blocks sit in worst-case slots in LDS and are
// compacted by the final copy.  (Five to eight heads, more than eight, and every token order take the cells
// kernel above, which reads a round once.)  `ngroups` counts workgroups, `ngroups_all` groups.
template <int DT, bool WIDE>
__global__ void __launch_bounds__(256) k_quant_encode_rounds_kernel(
    const uint16_t *__restrict__ x, int B, int H, int T, const XRows xs, float rel, uint16_t *__restrict__ scale,
    uint16_t *__restrict__ zero, uint8_t *__restrict__ stream, uint64_t capacity, uint32_t *__restrict__ info,
    ScanState *st, int W, uint32_t ngroups, uint32_t bound, uint64_t base, int par_stride, const Stagger stagger,
    int gpw, uint32_t ngroups_all) {
    extern __shared__ __align__(16) uint8_t gbuf[];        // gpw * H block slots of `bound` bytes
    __shared__ uint32_t s_idx;
    __shared__ uint64_t s_off;
    __shared__ uint32_t blk_off[kSubBlocks + 1];           // byte offset of each block inside the workgroup's bytes
    __shared__ __attribute__((aligned(16))) TokPar s_par[kSubBlocks * 16];      // [group of the workgroup][token of the round]
    const int tid = threadIdx.x;
    stagger_first_generation(stagger);
    if (tid == 0) s_idx = atomicAdd(&st->ticket, 1u);
    __syncthreads();
    const uint32_t gidx = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_idx);   // uniform: the rows' addresses become scalar
    if (gidx >= ngroups) return;
    // half-wavefront j serves head j % H of group gidx * gpw + j / H
    const int j = tid >> 5, t = tid & 31;                 // block and lane of the unit
    const int jg = j / H, jh = j % H;
    const uint32_t grp_first = gidx * (uint32_t)gpw;
    const int ng = (int)min((uint32_t)gpw, ngroups_all - grp_first);          // groups of this workgroup
    const int nblk = ng * H;                              // blocks of this workgroup
    const uint32_t grp = grp_first + (uint32_t)min(jg, ng - 1);
    const uint32_t cb = grp / (uint32_t)B, b = grp % (uint32_t)B;
    const size_t tok0 = (size_t)cb * 64;
    const UnitGeom g = unit_geom(W);
    const bool active = jg < ng && j < gpw * H;
    const TokPar *my_par = s_par + 16 * min(jg, ng - 1);
    uint8_t *blk = gbuf + (size_t)j * bound;
    uint32_t my_off = 8u;                                 // bytes of this block so far (uniform per half-wavefront)
    uint32_t cmax_all = 0;
#pragma unroll 1
    for (int r = 0; r < 4; r++) {
        // token parameters of the round: 16 lanes x 8 channels per token, the heads of one group after the other
        __builtin_amdgcn_s_setprio(PKV_EPRIO_STAT);
        {
            const int tt = tid >> 4, l16 = tid & 15;
            for (int q = 0; q < ng; q++) {
                const uint32_t gq = grp_first + (uint32_t)q;
                const uint32_t cq = gq / (uint32_t)B, bq = gq % (uint32_t)B;
                const size_t tq = (size_t)bq * par_stride + (size_t)cq * 64 + 16 * r + tt;
                round_token_params_few<DT>(x + bq * xs.sb + (int64_t)(cq * 64u + 16u * r) * xs.st, xs, H,
                                           tt, l16, rel, scale + tq, zero + tq, s_par + 16 * q + tt);
            }
        }
        // the same rows again, as cells (issued before the barrier; they hit the lines just fetched)
        uint2 xr[16];
        cell_load_lanes(x + b * xs.sb + jh * xs.sh + (int64_t)(tok0 + 16 * r) * xs.st + 4 * t, xs.st, xr);
        __syncthreads();
        __builtin_amdgcn_s_setprio(PKV_EPRIO_PACK);
        typename PacksOf<WIDE>::type u;
        uint32_t cmax;
        cell_packs<DT>(xr, my_par, u, cmax);
        __syncthreads();                                  // s_par is rewritten by the next round
        __builtin_amdgcn_s_setprio(PKV_EPRIO_EMIT);
        pack_offsets(u.len, u.off, u.payload);            // (all lanes: the scan runs on whole wavefronts)
        const uint32_t usz = (uint32_t)(g.mins_bytes + g.lens_bytes) + u.payload;
        if (r == 3) {
            // every block's final size is known before its last unit is written: the workgroup's size is published
            // now, so that the workgroups behind it in the stream wait that much less for it
            if (active && t == 0) blk_off[j + 1] = my_off + usz;          // sizes first ...
            if (tid == 0) blk_off[0] = 0;
            __syncthreads();
            if (tid == 0) {                                               // ... then their running sum
                for (int q = 1; q <= nblk; q++) blk_off[q] += blk_off[q - 1];
                lookback_publish(st, gidx, blk_off[nblk]);
            }
        }
        if (active) {
            cmax_all = max(cmax_all, cmax);
            if (t == 0) reinterpret_cast<uint16_t *>(blk)[r] = (uint16_t)(my_off - 8u + usz);
            unit_emit_any(blk, my_off, t, g, u);
            my_off += usz;
        }
    }
    if (__any(cmax_all >= (1u << W))) {   // codes that do not fit W bits are an error the host reports
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) cmax_all = max(cmax_all, __shfl_xor(cmax_all, d, 64));
        if ((tid & 63) == 0) atomicMax(&st->max_code, cmax_all);
    }
    packs_put();
    __syncthreads();
    const uint32_t bytes = blk_off[nblk];
    if (tid < 64) {
        const uint64_t off = base + lookback_offset(st, gidx, bytes, true);
        if (tid == 0) {
            s_off = off;
            if (gidx == ngroups - 1) st->total = off + bytes;
            if (off + bytes > capacity) atomicExch(&st->error, (uint32_t)PKV_ERR_CAPACITY);
        }
    }
    __syncthreads();
    const uint64_t off = s_off;
    if (off + bytes > capacity) return;
    if (tid < nblk) {
        const uint32_t first = grp_first * (uint32_t)H;                   // block index = group * H + head
        info[2 * (size_t)(first + tid)] = (uint32_t)(off + blk_off[tid]);
        info[2 * (size_t)(first + tid) + 1] = blk_off[tid + 1] - blk_off[tid];
    }
    if (active) copy_out32(stream + off + blk_off[j], blk, my_off, t);     // each half-wavefront copies its own block
}

// OR the FB-bit fields f[0..3] of four adjacent lanes 4m..4m+3, slot i, into a unit's LSB-first metadata array
// (field of lane c, slot i at bit (4c + i) * FB).  The 16 * FB bits of the four lanes start at byte 2 * FB * m.
__device__ __forceinline__ void meta_or4(uint8_t *arr, int m, int FB, int i, const uint32_t f[4]) {
    if (FB > 4) {                                 // widths 5, 6: 80 / 96 bits of four lanes, plus up to 16 bits of phase
        unsigned __int128 v = 0;
#pragma unroll
        for (int k = 0; k < 4; k++) v |= (unsigned __int128)f[k] << (4 * FB * k + FB * i);
        const uint32_t byte = 2u * (uint32_t)FB * (uint32_t)m;
        uint32_t *w = reinterpret_cast<uint32_t *>(arr + (byte & ~3u));
        v <<= 8u * (byte & 3u);
#pragma unroll
        for (int d = 0; d < 4; d++) {
            const uint32_t piece = (uint32_t)(v >> (32 * d));
            if (piece) atomicOr(w + d, piece);
        }
        return;
    }
    if (FB == 4) {                                // fields on 16-bit lanes: two aligned words, 32-bit arithmetic only
        uint32_t *w = reinterpret_cast<uint32_t *>(arr + 8u * (uint32_t)m);
        atomicOr(w, (f[0] | (f[1] << 16)) << (4 * i));
        atomicOr(w + 1, (f[2] | (f[3] << 16)) << (4 * i));
        return;
    }
    if (FB == 2) {                                // fields on byte lanes: one aligned word
        uint32_t *w = reinterpret_cast<uint32_t *>(arr + 4u * (uint32_t)m);
        atomicOr(w, (f[0] | (f[1] << 8) | (f[2] << 16) | (f[3] << 24)) << (2 * i));
        return;
    }
    // FB == 3: 48 bits at byte 6 m (odd m: two bytes into the word; 48 + 16 bits still fit two words)
    const uint32_t lo = (f[0] | (f[1] << 12)) << (3 * i), hi = (f[2] | (f[3] << 12)) << (3 * i);     // 27 bits each
    uint64_t v = (uint64_t)lo | ((uint64_t)hi << 24);
    const uint32_t byte = 6u * (uint32_t)m;
    uint32_t *w = reinterpret_cast<uint32_t *>(arr + (byte & ~3u));
    v <<= 8u * (byte & 3u);
    atomicOr(w, (uint32_t)v);
    atomicOr(w + 1, (uint32_t)(v >> 32));
}

// Inclusive prefix sum over each run of eight lanes (m = lane % 8) on the DPP data path; `total` receives the run's
// sum in all eight lanes.
__device__ __forceinline__ uint32_t oct_incl_scan(uint32_t v, int m, uint32_t &total) {
    uint32_t x = v;
    const uint32_t u1 = __builtin_amdgcn_update_dpp(0u, x, 0x111, 0xF, 0xF, true);      // row_shr:1
    x += m >= 1 ? u1 : 0u;
    const uint32_t u2 = __builtin_amdgcn_update_dpp(0u, x, 0x112, 0xF, 0xF, true);      // row_shr:2
    x += m >= 2 ? u2 : 0u;
    x += __builtin_amdgcn_update_dpp(0u, x, 0x114, 0xF, 0xA, false);                    // row_shr:4 into lanes 4..7 of a run
    const uint32_t last = __builtin_amdgcn_update_dpp(0u, x, 0xFF, 0xF, 0xF, false);    // every quad: its lane 3
    total = __builtin_amdgcn_update_dpp(last, last, 0x104, 0xF, 0x5, false);            // first quad of a run: the second quad's
    return x;
}

// ---- V, up to four heads: round-major, several groups to a workgroup ---------------------------
// One workgroup of 512 threads owns the 2 H blocks of each of gpw = 8 / H (rounded down) consecutive (128-token
// context block, sequence) groups, H <= 4, and goes through them 32 tokens (two rounds) at a time: read the rows
// row-wise for the token parameters, then at once re-read them as cells -- still in L2 -- quantize and append.
// Thread = (round parity rp, head slot j, cell lane t); head slot j serves head j % H of group gidx * gpw + j / H.
// Its cell (round 2 it + rp, channels 4t..4t+3) holds slot (2 it + rp) % 4 of lanes 4m..4m+3, m = t % 8, of unit
// (warp (t / 8) % 2, segment it / 2) of block 2 j + t / 16.  A unit's payload is slot-major, so the eight threads of
// a (unit, slot) append their packs behind the slots already there; the metadata bit-fields are OR-ed in with LDS
// atomics.  Units sit in worst-case slots in LDS; the final copy compacts them into the stream.  (Five to eight
// heads, more than eight, and every token order take the cells kernel below.)  `ngroups` counts workgroups,
// `ngroups_total` groups.
template <int DT, bool WIDE>
__global__ void __launch_bounds__(512) v_quant_encode_rounds_kernel(
    const uint16_t *__restrict__ x, int B, int H, int T, const XRows xs, float rel, uint16_t *__restrict__ scale,
    uint16_t *__restrict__ zero, uint8_t *__restrict__ stream, uint64_t capacity, uint32_t *__restrict__ info,
    ScanState *st, int W, uint32_t ngroups, uint32_t unit_slot, uint64_t base, int par_stride, const Stagger stagger,
    int gpw, uint32_t ngroups_total) {
    extern __shared__ __align__(16) uint8_t gbuf[];        // 16 blocks x 4 units x unit_slot bytes
    __shared__ uint32_t s_idx;
    __shared__ uint64_t s_off;
    __shared__ uint32_t blk_off[17];                       // byte offset of each block inside the workgroup's bytes
    __shared__ uint32_t s_tot[2][8][4];                    // payload bytes the two rounds of an iteration append per unit
    __shared__ uint16_t s_usz[16][4];                      // bytes of every unit (block, unit index 2 w + sg)
    __shared__ __attribute__((aligned(16))) TokPar s_par[kSubBlocks * 32];      // [group of the workgroup][token of the iteration]
    const int tid = threadIdx.x;
    stagger_first_generation(stagger);
    if (tid == 0) s_idx = atomicAdd(&st->ticket, 1u);
    __syncthreads();
    const uint32_t gidx = s_idx;
    if (gidx >= ngroups) return;
    const int rp = tid >> 8, j = (tid >> 5) & 7, t = tid & 31;
    const int jg = j / H, jh = j % H;
    const uint32_t grp_first = gidx * (uint32_t)gpw;
    const int ng = (int)min((uint32_t)gpw, ngroups_total - grp_first);        // groups of this workgroup
    const int nheads = ng * H;                            // head slots in use
    const uint32_t grp = grp_first + (uint32_t)min(jg, ng - 1);
    const uint32_t cb = grp / (uint32_t)B, b = grp % (uint32_t)B;
    const size_t tok0 = (size_t)cb * 128;
    const UnitGeom g = unit_geom(W);
    const uint32_t meta = (uint32_t)(g.mins_bytes + g.lens_bytes);
    const bool active = jg < ng;
    const TokPar *my_par = s_par + 32 * min(jg, ng - 1) + 16 * rp;
    const int blkid = 2 * j + (t >> 4), w = (t >> 3) & 1, m = t & 7;
    // metadata areas start as zeros (fields are OR-ed in)
    for (uint32_t i = tid; i < 64u * (meta / 4u); i += 512)
        reinterpret_cast<uint32_t *>(gbuf + (size_t)(i / (meta / 4u)) * unit_slot)[i % (meta / 4u)] = 0u;
    uint32_t run_off = 0;                                  // payload bytes of the thread's current unit so far
    uint32_t cmax_all = 0;
#pragma unroll 1
    for (int it = 0; it < 4; it++) {
        // token parameters of the 32 tokens: 16 lanes x 8 channels per token, the heads of one group after the other
        __builtin_amdgcn_s_setprio(PKV_EPRIO_STAT);
        {
            const int tt = tid >> 4, l16 = tid & 15;
            for (int q = 0; q < ng; q++) {
                const uint32_t gq = grp_first + (uint32_t)q;
                const uint32_t cq = gq / (uint32_t)B, bq = gq % (uint32_t)B;
                const size_t tq = (size_t)bq * par_stride + (size_t)cq * 128 + 32 * it + tt;
                round_token_params_few<DT>(x + bq * xs.sb + (int64_t)(cq * 128u + 32u * it) * xs.st, xs,
                                           H, tt, l16, rel, scale + tq, zero + tq, s_par + 32 * q + tt);
            }
        }
        // the same rows again, as cells (issued before the barrier; they hit the lines just fetched)
        uint2 xr[16];
        cell_load_lanes(x + b * xs.sb + jh * xs.sh + (int64_t)(tok0 + 32 * it + 16 * rp) * xs.st + 4 * t, xs.st, xr);
        __syncthreads();
        __builtin_amdgcn_s_setprio(PKV_EPRIO_PACK);
        typename PacksOf<WIDE>::type u;
        uint32_t cmax;
        cell_packs<DT>(xr, my_par, u, cmax);
        // bytes of the thread's four packs, their offsets inside the (unit, slot) and the slot's total
        const uint32_t pb = 2u * (u.len[0] + u.len[1] + u.len[2] + u.len[3]);
        uint32_t tot;
        const uint32_t inc = oct_incl_scan(pb, m, tot);
        if (m == 0) s_tot[rp][j][t >> 3] = tot;
        __syncthreads();                                  // s_par is rewritten by the next iteration; s_tot is published
        __builtin_amdgcn_s_setprio(PKV_EPRIO_EMIT);
        const uint32_t tot_even = s_tot[0][j][t >> 3], tot_odd = s_tot[1][j][t >> 3];
        if (it == 3) {
            // the last units' sizes are known before their packs are written: the workgroup's size is published now,
            // so that the workgroups behind it in the stream wait that much less for it
            if (active && rp == 0 && m == 0) s_usz[blkid][2 * w + 1] = (uint16_t)(meta + run_off + tot_even + tot_odd);
            __syncthreads();
            if (tid == 0) {
                uint32_t run = 0;
                for (int q = 0; q < 2 * nheads; q++) {
                    blk_off[q] = run;
                    run += 8u + s_usz[q][0] + s_usz[q][1] + s_usz[q][2] + s_usz[q][3];
                }
                blk_off[2 * nheads] = run;
                lookback_publish(st, gidx, run);
            }
        }
        if (active) {
            cmax_all = max(cmax_all, cmax);
            const int sg = it >> 1, slot = 2 * (it & 1) + rp;
            uint8_t *unit = gbuf + (size_t)(blkid * 4 + 2 * w + sg) * unit_slot;
            meta_or4(unit, m, g.W, slot, u.mn);
            meta_or4(unit + g.mins_bytes, m, g.LB, slot, u.len);
            uint32_t o = meta + run_off + (rp ? tot_even : 0u) + (inc - pb);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                put_pack(reinterpret_cast<uint16_t *>(unit + o), u, k);
                o += 2u * u.len[k];
            }
        }
        run_off += tot_even + tot_odd;                    // both rounds of the iteration are behind the unit now
        if (it & 1) {                                     // the unit (w, it / 2) is complete
            if (it == 1 && active && rp == 0 && m == 0) s_usz[blkid][2 * w] = (uint16_t)(meta + run_off);
            run_off = 0;
        }
    }
    if (__any(cmax_all >= (1u << W))) {   // codes that do not fit W bits are an error the host reports
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) cmax_all = max(cmax_all, __shfl_xor(cmax_all, d, 64));
        if ((tid & 63) == 0) atomicMax(&st->max_code, cmax_all);
    }
    packs_put();
    __syncthreads();
    const int nblk = 2 * nheads;
    const uint32_t bytes = blk_off[nblk];
    if (tid < 64) {
        const uint64_t off = base + lookback_offset(st, gidx, bytes, true);
        if (tid == 0) {
            s_off = off;
            if (gidx == ngroups - 1) st->total = off + bytes;
            if (off + bytes > capacity) atomicExch(&st->error, (uint32_t)PKV_ERR_CAPACITY);
        }
    }
    __syncthreads();
    const uint64_t off = s_off;
    if (off + bytes > capacity) return;
    if (tid < nblk) {
        const uint32_t first = grp_first * (uint32_t)(2 * H);             // block index = group * 2 H + 2 head + half
        info[2 * (size_t)(first + tid)] = (uint32_t)(off + blk_off[tid]);
        info[2 * (size_t)(first + tid) + 1] = blk_off[tid + 1] - blk_off[tid];
    }
    // half-wavefront q copies block q: the header of cumulative unit sizes, then its four units one after another
    const int q = tid >> 5;
    if (q < nblk) {
        uint8_t *dst = stream + off + blk_off[q];
        uint32_t cum = 0;
#pragma unroll
        for (int un = 0; un < 4; un++) {
            const uint32_t n = s_usz[q][un];
            copy_out32(dst + 8 + cum, gbuf + (size_t)(q * 4 + un) * unit_slot, n, t);
            cum += n;
            if (t == un) reinterpret_cast<uint16_t *>(dst)[un] = (uint16_t)cum;
        }
    }
}

// ---- V, all heads in one workgroup, x read ONCE as cells ----------------------------------------
// The V counterpart of k_quant_encode_cells_kernel: the threads keep the roles of the round-major V encoder (round
// parity rp, head j, cell lane t), but an iteration's 32 tokens are read as cells only, and a wavefront is ONE head
// with both rounds of the iteration (lanes 0..31 the even round, lanes 32..63 the odd one).  Everything a head's
// blocks need from each other -- the payload bytes the even round puts in front of the odd one -- is then an
// exchange between the halves of a wavefront, and the only thing wavefronts share is the token minima and maxima:
// each forms those of its head from the cell registers, the eight partial results per token go through LDS, and
// every wavefront forms the 32 tokens' parameters for itself.  One barrier per iteration.  For 5..8 heads, tokens
// in their own order; same stream, parameters and block_info as the round-major kernel.
// PERM: the tokens in the order of a repacking, as in the round-major kernel; with scale_in / zero_in (the tokens'
// parameters in the order of x, known from the pass that made the order) nothing is left to exchange and an
// iteration has no barrier at all.
// Wide packs: the sixteen blocks' worst cases fill more than half of a CU's LDS, so that one workgroup is resident, and takes
// the two 64-token segments of its blocks side by side, sixteen wavefronts in two iterations instead of eight in four: eight
// wavefronts a CU left it waiting for its loads.  16 x 8 x 32768 tokens of fp16 V at rel 0.05: 475 -> 425 us (bf16 521 -> 463, rel 0.03
// 487 -> 436), from a code matrix 284 -> 225, 3 x 8 x 11008 70.6 -> 60.7 and 44.9 -> 38.2.
__host__ __device__ constexpr int v_cell_segs(bool wide) { return wide ? 2 : 1; }
template <bool WIDE>
struct VCellsLds {
    uint32_t idx;
    uint64_t off;
    uint32_t blk_off[17];
    uint16_t usz[16][4];
    __attribute__((aligned(16))) TokPar par[v_cell_segs(WIDE) * 8 * 32];       // [wavefront][token of the iteration]
    uint32_t mm[2][v_cell_segs(WIDE) * 8][32];                                 // [iteration parity][wavefront][token]: minmax_word
};
template <int DT, bool WIDE, bool PERM, bool XCH, bool STRIDED>
__device__ __forceinline__ void v_quant_encode_cells(
    uint8_t *const gbuf, VCellsLds<WIDE> &lds, const uint16_t *__restrict__ x, int B, int H, int T, const XRows xs, float rel, uint16_t *__restrict__ scale,
    uint16_t *__restrict__ zero, uint8_t *__restrict__ stream, uint64_t capacity, uint32_t *__restrict__ info,
    ScanState *st, int W, uint32_t ngroups, uint32_t unit_slot, uint64_t base, int par_stride,
    const uint32_t *__restrict__ perm, int perm_block, const uint16_t *__restrict__ scale_in,
    const uint16_t *__restrict__ zero_in, const Stagger stagger, int nsg, uint64_t *xw) {
    constexpr int SEGS = v_cell_segs(WIDE), ITS = 4 / SEGS;
    uint64_t &s_off = lds.off;
    uint32_t *const blk_off = lds.blk_off;
    auto &s_usz = lds.usz;
    TokPar *const s_par = lds.par;
    auto &s_mm = lds.mm;
    const int tid = threadIdx.x;
    stagger_first_generation(stagger);
    if (tid == 0) lds.idx = atomicAdd(&st->ticket, 1u);
    __syncthreads();
    const uint32_t gidx = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds.idx);
    if (gidx >= ngroups) return;
    // XCH (more than eight heads): runs of eight heads that exchange the minima and maxima of their heads per token,
    // as in the K kernel; a run's words are [iteration][token of the iteration]
    const int H_all = H;
    const uint32_t sgi = XCH ? gidx % (uint32_t)nsg : 0u;
    const int hbase = XCH ? 8 * (int)sgi : 0;
    if (XCH) H = min(8, H_all - hbase);
    const int wave = tid >> 6, j = wave & 7, seg = wave >> 3, rp = (tid >> 5) & 1, t = tid & 31, lane = tid & 63;
    const uint32_t grp = XCH ? gidx / (uint32_t)nsg : gidx;
    const uint32_t cb = grp / (uint32_t)B, b = grp % (uint32_t)B;
    const size_t tok0 = (size_t)cb * 128;
    const UnitGeom g = unit_geom(W);
    const uint32_t meta = (uint32_t)(g.mins_bytes + g.lens_bytes);
    const bool active = j < H;
    const int jc = min(j, H - 1);
    const TokPar *my_par = s_par + 32 * (XCH ? seg : wave) + 16 * rp;
    const int blkid = 2 * j + (t >> 4), w = (t >> 3) & 1, m = t & 7;
    for (uint32_t i = tid; i < 64u * (meta / 4u); i += 512 * SEGS)                 // metadata areas start as zeros
        reinterpret_cast<uint32_t *>(gbuf + (size_t)(i / (meta / 4u)) * unit_slot)[i % (meta / 4u)] = 0u;
    uint32_t run_off = 0;
    uint32_t cmax_all = 0;
    const char *cells = reinterpret_cast<const char *>(x + b * xs.sb + (hbase + __builtin_amdgcn_readfirstlane(jc)) * xs.sh + (int64_t)tok0 * xs.st);
    const uint32_t cell_off = (16u * (uint32_t)rp * (uint32_t)xs.st + 4u * (uint32_t)t) * 2u;
    const int64_t row_bytes = STRIDED ? 2 * xs.st : 2 * kHeadDim;
    const uint32_t plane = (uint32_t)(((size_t)jc * T * kHeadDim + 4 * t) * 2);
    const bool known = PERM && scale_in != nullptr;              // uniform
    if (known) __syncthreads();                                  // the metadata zeros are in place before the first OR (no barrier below)
#pragma unroll 1
    for (int step = 0; step < ITS; step++) {
        const int it = SEGS == 1 ? step : step + 2 * __builtin_amdgcn_readfirstlane(seg);      // 32 tokens each
        // (no request ahead as in the K kernel: placing the packs holds too many registers to keep 16 rows in flight)
        uint2 xr[16];
        // PERM: (the 32 tokens of an iteration lie in one repacking block: perm_block is a multiple of 64)
        const size_t rb = PERM ? ((tok0 + 32 * it) / (size_t)perm_block) * (size_t)perm_block : 0;
        if (PERM) cell_load_rows_lanes(x + (((size_t)b * H) * T + rb) * kHeadDim, perm + tok0 + 32 * it + 16 * rp, (uint32_t)perm_block - 1u, plane, xr);
        else cell_load(cells + it * 32 * row_bytes, row_bytes, cell_off, xr);
        __builtin_amdgcn_s_setprio(PKV_EPRIO_STAT);
        if (known) {
            if (lane < 32) {
                const uint32_t src = min(perm[tok0 + 32 * it + lane], (uint32_t)perm_block - 1u);
                const uint32_t sb = scale_in[(size_t)b * T + rb + src], zb = zero_in[(size_t)b * T + rb + src];
                if (j == 0) {
                    const size_t tok = (size_t)b * par_stride + tok0 + 32 * it + lane;
                    scale[tok] = (uint16_t)sb;
                    zero[tok] = (uint16_t)zb;
                }
                s_par[32 * wave + lane] = token_par<DT>(T16<DT>::from_bits(sb), zb, false);
            }
        } else {
        {
            float mn, mx;
            cell_token_minmax_halves<DT>(xr, mn, mx);
            if ((lane & 1) == 0) s_mm[it & 1][wave][lane >> 1] = minmax_word<DT>(mn, mx);
        }
        __syncthreads();
        if (XCH) {
            if (j == 0) {
                const int tk = lane & 31;
                uint32_t pw = s_mm[it & 1][8 * seg][tk];
#pragma unroll
                for (int q = 1; q < 8; q++) pw = pk_sel_x<false, DT != PKV_F16>(pw, s_mm[it & 1][8 * seg + q][tk]);
                float rmn, rmx;
                minmax_unword<DT>(pw, rmn, rmx);
                uint64_t *words = xw + (size_t)(gidx - sgi) * 128 + 32 * it;      // [run][iteration][token] of this group
                if (lane < 32)
                    __hip_atomic_store(words + (size_t)sgi * 128 + lane, (1ull << 63) | ((uint64_t)T16<DT>::to_bits(rmn) << 16) | (uint64_t)T16<DT>::to_bits(rmx),
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                // lane = (parity of the run, token)
                float amn = INFINITY, amx = -INFINITY;
                for (int run = lane >> 5; run < nsg; run += 2) {
                    const uint64_t *wp = words + (size_t)run * 128 + tk;
                    uint64_t w = __hip_atomic_load(wp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    int spins = 0;
                    while ((w >> 63) == 0 && spins < kSpinLimit) {
                        __builtin_amdgcn_s_sleep(8);
                        w = __hip_atomic_load(wp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        spins++;
                    }
                    if ((w >> 63) == 0) atomicExch(&st->error, (uint32_t)PKV_ERR_INTERNAL);     // (bounded wait: the host reports it)
                    amn = fminf(amn, T16<DT>::from_bits((uint32_t)(w >> 16) & 0xFFFFu));
                    amx = fmaxf(amx, T16<DT>::from_bits((uint32_t)w & 0xFFFFu));
                }
                amn = fminf(amn, __shfl_xor(amn, 32, 64)); amx = fmaxf(amx, __shfl_xor(amx, 32, 64));
                if (lane < 32) {
                    const float range = round_t<DT>(amx - amn);
                    const float sc = round_t<DT>(range * rel);
                    const uint32_t zb = T16<DT>::to_bits(rintf(round_t<DT>(__fdiv_rn(amn, sc))));
                    if (sgi == 0) {
                        const size_t tok = (size_t)b * par_stride + tok0 + 32 * it + lane;
                        scale[tok] = (uint16_t)T16<DT>::to_bits(sc);
                        zero[tok] = (uint16_t)zb;
                    }
                    s_par[32 * seg + lane] = token_par<DT>(sc, zb, false);
                }
            }
            __syncthreads();
        } else
        if (lane < 32) {
            uint32_t pw = s_mm[it & 1][8 * seg][lane];             // the eight heads' words, combined by packed minima
#pragma unroll
            for (int q = 1; q < 8; q++) pw = pk_sel_x<false, DT != PKV_F16>(pw, s_mm[it & 1][8 * seg + q][lane]);
            float mn, mx;
            minmax_unword<DT>(pw, mn, mx);
            const float range = round_t<DT>(mx - mn);
            const float sc = round_t<DT>(range * rel);
            const uint32_t zb = T16<DT>::to_bits(rintf(round_t<DT>(__fdiv_rn(mn, sc))));
            if (j == 0) {
                const size_t tok = (size_t)b * par_stride + tok0 + 32 * it + lane;
                scale[tok] = (uint16_t)T16<DT>::to_bits(sc);
                zero[tok] = (uint16_t)zb;
            }
            s_par[32 * wave + lane] = token_par<DT>(sc, zb, false);
        }
        }
        wave_lds_order();
        __builtin_amdgcn_s_setprio(PKV_EPRIO_PACK);
        uint32_t c01[16], c23[16];
        cell_quant<DT, false>(xr, my_par, c01, c23);          // (the halves of the wavefront hold different tokens)
        typename PacksOf<WIDE>::type u;
        uint32_t cmax;
        cell_build(c01, c23, u, cmax);
        const uint32_t pb = 2u * (u.len[0] + u.len[1] + u.len[2] + u.len[3]);
        uint32_t tot;
        const uint32_t inc = oct_incl_scan(pb, m, tot);
        __builtin_amdgcn_s_setprio(PKV_EPRIO_EMIT);
        const auto halves = __builtin_amdgcn_permlane32_swap(tot, tot, false, false);      // the even round's total, the odd round's
        const uint32_t tot_even = halves[0], tot_odd = halves[1];
        if (step == ITS - 1) {
            if (active && rp == 0 && m == 0) s_usz[blkid][2 * w + (it >> 1)] = (uint16_t)(meta + run_off + tot_even + tot_odd);
            __syncthreads();
            if (tid == 0) {
                uint32_t run = 0;
                for (int q = 0; q < 2 * H; q++) {
                    blk_off[q] = run;
                    run += 8u + s_usz[q][0] + s_usz[q][1] + s_usz[q][2] + s_usz[q][3];
                }
                blk_off[2 * H] = run;
                lookback_publish(st, gidx, run);
            }
        }
        if (active) {
            cmax_all = max(cmax_all, cmax);
            const int sg = it >> 1, slot = 2 * (it & 1) + rp;
            uint8_t *unit = gbuf + (size_t)(blkid * 4 + 2 * w + sg) * unit_slot;
            meta_or4(unit, m, g.W, slot, u.mn);
            meta_or4(unit + g.mins_bytes, m, g.LB, slot, u.len);
            uint32_t o = meta + run_off + (rp ? tot_even : 0u) + (inc - pb);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                put_pack(reinterpret_cast<uint16_t *>(unit + o), u, k);
                o += 2u * u.len[k];
            }
        }
        run_off += tot_even + tot_odd;
        if (it & 1) {
            if (SEGS == 1 && it == 1 && active && rp == 0 && m == 0) s_usz[blkid][2 * w] = (uint16_t)(meta + run_off);
            run_off = 0;
        }
    }
    if (__any(cmax_all >= (1u << W))) {
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) cmax_all = max(cmax_all, __shfl_xor(cmax_all, d, 64));
        if ((tid & 63) == 0) atomicMax(&st->max_code, cmax_all);
    }
    packs_put();
    __syncthreads();
    const int nblk = 2 * H;
    const uint32_t bytes = blk_off[nblk];
    if (tid < 64) {
        const uint64_t off = base + lookback_offset(st, gidx, bytes, true);
        if (tid == 0) {
            s_off = off;
            if (gidx == ngroups - 1) __hip_atomic_store(&st->total, off + bytes, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (off + bytes > capacity) atomicExch(&st->error, (uint32_t)PKV_ERR_CAPACITY);
        }
    }
    __syncthreads();
    const uint64_t off = s_off;
    if (off + bytes > capacity) return;
    if (tid < nblk) {
        const uint32_t first = XCH ? grp * (uint32_t)(2 * H_all) + (uint32_t)(2 * hbase) : gidx * (uint32_t)nblk;    // block index = group * 2 heads + 2 head + half
        info[2 * (size_t)(first + tid)] = (uint32_t)(off + blk_off[tid]);
        info[2 * (size_t)(first + tid) + 1] = blk_off[tid + 1] - blk_off[tid];
    }
    const int q = (tid >> 5) & 15;
    if (q < nblk) {
        uint8_t *dst = stream + off + blk_off[q];
        uint32_t cum = 0;
#pragma unroll
        for (int un = 0; un < 4; un++) {
            const uint32_t n = s_usz[q][un];
            const bool mine = SEGS == 1 || un >> 1 == seg;
            if (mine) copy_out32(dst + 8 + cum, gbuf + (size_t)(q * 4 + un) * unit_slot, n, t);
            cum += n;
            if (mine && t == un) reinterpret_cast<uint16_t *>(dst)[un] = (uint16_t)cum;
        }
    }
}

template <int DT, bool WIDE, bool PERM, bool XCH = false, bool STRIDED = false>
__global__ void __launch_bounds__(512 * v_cell_segs(WIDE)) v_quant_encode_cells_kernel(
    const uint16_t *__restrict__ x, int B, int H, int T, const XRows xs, float rel, uint16_t *__restrict__ scale,
    uint16_t *__restrict__ zero, uint8_t *__restrict__ stream, uint64_t capacity, uint32_t *__restrict__ info,
    ScanState *st, int W, uint32_t ngroups, uint32_t unit_slot, uint64_t base, int par_stride,
    const uint32_t *__restrict__ perm, int perm_block, const uint16_t *__restrict__ scale_in,
    const uint16_t *__restrict__ zero_in, const Stagger stagger, int nsg, uint64_t *xw, const EncodeClose c) {
    extern __shared__ __align__(16) uint8_t gbuf[];        // 16 blocks x 4 units x unit_slot bytes
    __shared__ VCellsLds<WIDE> lds;
    v_quant_encode_cells<DT, WIDE, PERM, XCH, STRIDED>(gbuf, lds, x, B, H, T, xs, rel, scale, zero, stream, capacity, info, st, W, ngroups,
                                                       unit_slot, base, par_stride, perm, perm_block, scale_in, zero_in, stagger, nsg, xw);
    if (!XCH) encode_close(c, lds.idx);                     // (runs that wait for each other are closed by finish_encode)
}

// ---- K and V in one launch -----------------------------------------------------------------------
// Workgroups of 512 threads, two resident on a CU: one in two takes a group of V as the kernel above, the other two groups of K
// (T is a multiple of 128, so there are twice as many of those).  A launch of its own leaves the chip partly empty at its end or,
// when it is small, all the time, and all its workgroups go through their phases together.  V and K go in turns of 256 (`turns` of
// them each, then the rest of V, the rest of K), so that a CU starts with one of each.
struct CellsSide {
    const uint16_t *x;
    XRows xs;
    float rel;
    uint16_t *scale, *zero;
    uint8_t *stream;
    uint64_t capacity, base;
    uint32_t *info;
    ScanState *st;
    int W;
    uint32_t ngroups, slot;                // K: bytes of a block's slot, V: of a unit's
    const uint16_t *scale_in, *zero_in;
};
template <int DT, bool PERM, bool ROT>
__global__ void __launch_bounds__(512) kv_quant_encode_cells_kernel(const CellsSide k, const CellsSide v, int B, int H, int T, int par_stride,
                                                                    const uint32_t *__restrict__ perm, int perm_block, uint32_t turns, const Rot rot) {
    extern __shared__ __align__(16) uint8_t gbuf[];
    const Stagger stagger{0u, 0u};
    __shared__ union Lds { __device__ Lds() {} VCellsLds<false> v; KCellsLds k[2]; } lds;
    const uint32_t turn = blockIdx.x >> 8;
    if (turn < 2u * turns ? (turn & 1u) == 0u : blockIdx.x - (turns << 9) < v.ngroups - (turns << 8)) {
        v_quant_encode_cells<DT, false, PERM, false, !PERM>(gbuf, lds.v, v.x, B, H, T, v.xs, v.rel, v.scale, v.zero, v.stream, v.capacity, v.info,
                                                            v.st, v.W, v.ngroups, v.slot, v.base, par_stride, perm, perm_block, v.scale_in,
                                                            v.zero_in, stagger, 1, nullptr);
    } else {
        const int half = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8);
        k_quant_encode_cells<DT, false, PERM, false, !PERM, ROT>((int)threadIdx.x & 255, gbuf + (size_t)half * H * k.slot, lds.k[half], k.x,
                                                                       B, H, T, k.xs, k.rel, k.scale, k.zero, k.stream, k.capacity, k.info, k.st,
                                                                       k.W, k.ngroups, k.slot, k.base, par_stride, perm, perm_block, stagger, 1,
                                                                       nullptr, rot);
    }
}

// `rows` (uniform: scalar registers) is the first of the 16 token rows, `lane_off` the lane's byte offset inside a
// row, so that a load is one 32-bit lane offset on a scalar base
__device__ __forceinline__ void code_cell_load(const uint8_t *rows, size_t row_bytes, uint32_t lane_off, uint32_t w[16]) {
#pragma unroll
    for (int k = 0; k < 16; k++) w[k] = *reinterpret_cast<const uint32_t *>(rows + (size_t)k * row_bytes + lane_off);
}
// four codes of a dword as two pairs of 16-bit integers (codes 0, 1 and codes 2, 3)
__device__ __forceinline__ void code_cell_pairs(const uint32_t w[16], uint32_t c01[16], uint32_t c23[16]) {
#pragma unroll
    for (int k = 0; k < 16; k++) {
        c01[k] = __builtin_amdgcn_perm(0u, w[k], 0x0C010C00u);
        c23[k] = __builtin_amdgcn_perm(0u, w[k], 0x0C030C02u);
    }
}

}  // namespace pkv

#include "pkv_quant_once.hpp"

namespace pkv {

// ---- the block codec from a code matrix, as cells --------------------------------------------------------------
// The cells encoders with nothing to quantize: the input is the uint8 code matrix [ctx_len, hidden] of pkv_k_encode /
// pkv_v_encode.  Eight consecutive K blocks (64 x 128) or sixteen consecutive V blocks (128 x 64) of the stream are
// 1024 adjacent channels of one context block, i.e. exactly the group a cells workgroup owns, with the "heads" being
// 128-channel slices of the matrix.  A thread reads its cell as sixteen dwords (four codes of one token each; the 32
// lanes of a half-wavefront one 128-byte line per token), asks for the next round's while it forms and emits this
// round's packs, and no code tile is staged in LDS.  For hidden a multiple of 1024, the reference's block shapes and
// widths up to 6.  Launches of few groups take all tokens of a group at once (code_encode_once_kernel), also with other
// rows of whole runs; pack_group_kernel takes everything else.
template <bool WIDE>
__global__ void __launch_bounds__(256) k_code_cells_kernel(
    const uint8_t *__restrict__ codes, int hidden, uint8_t *__restrict__ stream, uint64_t capacity,
    uint32_t *__restrict__ info, ScanState *st, int W, uint32_t ngroups, uint32_t bound, const Stagger stagger, const EncodeClose c) {
    extern __shared__ __align__(16) uint8_t gbuf[];        // 8 block slots of `bound` bytes
    __shared__ uint32_t s_idx;
    __shared__ uint64_t s_off;
    __shared__ uint32_t blk_off[kSubBlocks + 1];
    const int tid = threadIdx.x;
    stagger_first_generation(stagger);
    if (tid == 0) s_idx = atomicAdd(&st->ticket, 1u);
    __syncthreads();
    const uint32_t gidx = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_idx);
    if (gidx >= ngroups) {
        encode_close(c, s_idx);
        return;
    }
    const int j = tid >> 5, t = tid & 31;                 // block of the group, lane of the unit
    const uint32_t per_row = (uint32_t)hidden / 1024u;    // groups per context block
    const uint32_t cb = gidx / per_row, hg = gidx % per_row;
    const UnitGeom g = unit_geom(W);
    uint8_t *blk = gbuf + (size_t)j * bound;
    uint32_t my_off = 8u;
    const uint8_t *rows = codes + (size_t)cb * 64 * (size_t)hidden + (size_t)hg * 1024;      // uniform
    const uint32_t lane_off = (uint32_t)(j * 128 + 4 * t);
    uint32_t w[16];
    code_cell_load(rows, (size_t)hidden, lane_off, w);
#pragma unroll 1
    for (int r = 0; r < 4; r++) {
        __builtin_amdgcn_s_setprio(PKV_EPRIO_PACK);
        uint32_t c01[16], c23[16];
        code_cell_pairs(w, c01, c23);
        if (r < 3) code_cell_load(rows + (size_t)(r + 1) * 16 * (size_t)hidden, (size_t)hidden, lane_off, w);     // travels while the packs are formed
        typename PacksOf<WIDE>::type u;
        uint32_t cmax;
        cell_build(c01, c23, u, cmax);
        __builtin_amdgcn_s_setprio(PKV_EPRIO_EMIT);
        pack_offsets(u.len, u.off, u.payload);
        const uint32_t usz = (uint32_t)(g.mins_bytes + g.lens_bytes) + u.payload;
        if (r == 3) {                                     // the group's size is known before its last units are written
            if (t == 0) blk_off[j + 1] = my_off + usz;
            if (tid == 0) blk_off[0] = 0;
            __syncthreads();
            if (tid == 0) {
                for (int q = 1; q <= kSubBlocks; q++) blk_off[q] += blk_off[q - 1];
                lookback_publish(st, gidx, blk_off[kSubBlocks]);
            }
        }
        if (t == 0) reinterpret_cast<uint16_t *>(blk)[r] = (uint16_t)(my_off - 8u + usz);
        unit_emit_any(blk, my_off, t, g, u);
        my_off += usz;
    }
    packs_put();
    __syncthreads();
    const uint32_t bytes = blk_off[kSubBlocks];
    if (tid < 64) {
        const uint64_t off = lookback_offset(st, gidx, bytes, true);
        if (tid == 0) {
            s_off = off;
            if (gidx == ngroups - 1) __hip_atomic_store(&st->total, off + bytes, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (off + bytes > capacity) atomicExch(&st->error, (uint32_t)PKV_ERR_CAPACITY);
        }
    }
    __syncthreads();
    const uint64_t off = s_off;
    if (off + bytes <= capacity) {
        if (tid < kSubBlocks) {
            info[2 * (size_t)(gidx * (uint32_t)kSubBlocks + tid)] = (uint32_t)(off + blk_off[tid]);
            info[2 * (size_t)(gidx * (uint32_t)kSubBlocks + tid) + 1] = blk_off[tid + 1] - blk_off[tid];
        }
        copy_out32(stream + off + blk_off[j], blk, my_off, t);
    }
    encode_close(c, s_idx);
}

// V: the thread roles of v_quant_encode_cells_kernel (a wavefront = one 128-channel slice with both rounds of an
// iteration in its halves), no barrier inside an iteration.
template <bool WIDE>
__global__ void __launch_bounds__(512 * v_cell_segs(WIDE)) v_code_cells_kernel(
    const uint8_t *__restrict__ codes, int hidden, uint8_t *__restrict__ stream, uint64_t capacity,
    uint32_t *__restrict__ info, ScanState *st, int W, uint32_t ngroups, uint32_t unit_slot, const Stagger stagger, const EncodeClose c) {
    extern __shared__ __align__(16) uint8_t gbuf[];        // 16 blocks x 4 units x unit_slot bytes
    __shared__ uint32_t s_idx;
    __shared__ uint64_t s_off;
    __shared__ uint32_t blk_off[17];
    __shared__ uint16_t s_usz[16][4];
    constexpr int SEGS = v_cell_segs(WIDE), ITS = 4 / SEGS;
    const int tid = threadIdx.x;
    stagger_first_generation(stagger);
    if (tid == 0) s_idx = atomicAdd(&st->ticket, 1u);
    __syncthreads();
    const uint32_t gidx = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_idx);      // uniform: the rows' addresses become scalar
    if (gidx >= ngroups) {
        encode_close(c, s_idx);
        return;
    }
    const int j = (tid >> 6) & 7, seg = tid >> 9, rp = (tid >> 5) & 1, t = tid & 31;
    const uint32_t per_row = (uint32_t)hidden / 1024u;
    const uint32_t cb = gidx / per_row, hg = gidx % per_row;
    const UnitGeom g = unit_geom(W);
    const uint32_t meta = (uint32_t)(g.mins_bytes + g.lens_bytes);
    const int blkid = 2 * j + (t >> 4), wq = (t >> 3) & 1, m = t & 7;
    for (uint32_t i = tid; i < 64u * (meta / 4u); i += 512 * SEGS)                 // metadata areas start as zeros
        reinterpret_cast<uint32_t *>(gbuf + (size_t)(i / (meta / 4u)) * unit_slot)[i % (meta / 4u)] = 0u;
    uint32_t run_off = 0;
    const uint8_t *rows = codes + (size_t)cb * 128 * (size_t)hidden + (size_t)hg * 1024;      // uniform
    const uint32_t lane_off = (uint32_t)(16 * rp) * (uint32_t)hidden + (uint32_t)(j * 128 + 4 * t);
    __syncthreads();                                       // the metadata zeros are in place before the first OR
#pragma unroll 1
    for (int step = 0; step < ITS; step++) {
        const int it = SEGS == 1 ? step : step + 2 * __builtin_amdgcn_readfirstlane(seg);      // 32 tokens each
        // (no request ahead: with sixteen more registers in flight while the packs are placed the kernel needs 142
        // and a CU holds one workgroup instead of two)
        uint32_t w[16];
        code_cell_load(rows + (size_t)it * 32 * (size_t)hidden, (size_t)hidden, lane_off, w);
        __builtin_amdgcn_s_setprio(PKV_EPRIO_PACK);
        uint32_t c01[16], c23[16];
        code_cell_pairs(w, c01, c23);
        typename PacksOf<WIDE>::type u;
        uint32_t cmax;
        cell_build(c01, c23, u, cmax);
        const uint32_t pb = 2u * (u.len[0] + u.len[1] + u.len[2] + u.len[3]);
        uint32_t tot;
        const uint32_t inc = oct_incl_scan(pb, m, tot);
        __builtin_amdgcn_s_setprio(PKV_EPRIO_EMIT);
        const auto halves = __builtin_amdgcn_permlane32_swap(tot, tot, false, false);      // the even round's total, the odd round's
        const uint32_t tot_even = halves[0], tot_odd = halves[1];
        if (step == ITS - 1) {
            if (rp == 0 && m == 0) s_usz[blkid][2 * wq + (it >> 1)] = (uint16_t)(meta + run_off + tot_even + tot_odd);
            __syncthreads();
            if (tid == 0) {
                uint32_t run = 0;
                for (int q = 0; q < 16; q++) {
                    blk_off[q] = run;
                    run += 8u + s_usz[q][0] + s_usz[q][1] + s_usz[q][2] + s_usz[q][3];
                }
                blk_off[16] = run;
                lookback_publish(st, gidx, run);
            }
        }
        {
            const int sg = it >> 1, slot = 2 * (it & 1) + rp;
            uint8_t *unit = gbuf + (size_t)(blkid * 4 + 2 * wq + sg) * unit_slot;
            meta_or4(unit, m, g.W, slot, u.mn);
            meta_or4(unit + g.mins_bytes, m, g.LB, slot, u.len);
            uint32_t o = meta + run_off + (rp ? tot_even : 0u) + (inc - pb);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                put_pack(reinterpret_cast<uint16_t *>(unit + o), u, k);
                o += 2u * u.len[k];
            }
        }
        run_off += tot_even + tot_odd;
        if (it & 1) {
            if (SEGS == 1 && it == 1 && rp == 0 && m == 0) s_usz[blkid][2 * wq] = (uint16_t)(meta + run_off);
            run_off = 0;
        }
    }
    packs_put();
    __syncthreads();
    const uint32_t bytes = blk_off[16];
    if (tid < 64) {
        const uint64_t off = lookback_offset(st, gidx, bytes, true);
        if (tid == 0) {
            s_off = off;
            if (gidx == ngroups - 1) __hip_atomic_store(&st->total, off + bytes, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (off + bytes > capacity) atomicExch(&st->error, (uint32_t)PKV_ERR_CAPACITY);
        }
    }
    __syncthreads();
    const uint64_t off = s_off;
    if (off + bytes <= capacity) {
        if (tid < 16) {
            info[2 * (size_t)(gidx * 16u + tid)] = (uint32_t)(off + blk_off[tid]);
            info[2 * (size_t)(gidx * 16u + tid) + 1] = blk_off[tid + 1] - blk_off[tid];
        }
        const int q = (tid >> 5) & 15;                         // half-wavefront q copies block q (of two segments each its own)
        uint8_t *dst = stream + off + blk_off[q];
        uint32_t cum = 0;
#pragma unroll
        for (int un = 0; un < 4; un++) {
            const uint32_t n = s_usz[q][un];
            const bool mine = SEGS == 1 || un >> 1 == seg;
            if (mine) copy_out32(dst + 8 + cum, gbuf + (size_t)(q * 4 + un) * unit_slot, n, t);
            cum += n;
            if (mine && t == un) reinterpret_cast<uint16_t *>(dst)[un] = (uint16_t)cum;
        }
    }
    encode_close(c, s_idx);
}

// Launch of the two kernels above (pkv_codec.hip decides when they apply): `st` is a prepared scan state of
// code_cells_words status words, `bound` the worst-case bytes of a block.
static OncePlan code_plan(bool is_k, int ctx_len, int hidden) { return once_plan(is_k, (uint64_t)(ctx_len / (is_k ? 64 : 128)), hidden / kHeadDim, kOnceSmallCodes); }
bool code_cells_serve(bool is_k, int ctx_len, int hidden) {
    if (hidden % 1024 == 0) return true;
    const OncePlan p = hidden % kHeadDim ? OncePlan{0, 0, 0, 0} : code_plan(is_k, ctx_len, hidden);
    return p.threads && hidden / kHeadDim % p.run == 0;    // (code_encode_once_kernel knows whole runs only)
}
static uint32_t code_cells_groups(bool is_k, int ctx_len, int hidden) { return (uint32_t)(ctx_len / (is_k ? 64 : 128)) * (uint32_t)(hidden / 1024); }
// (as encode_closes: K of 1024 channels of 4-bit codes, calls without a size one after the other, us: 4096 rows 13.1 -> 9.8, 16384 13.4 -> 12.7, 32768
// 22.1 -> 21.8, 65536 37.0 -> 36.4, 131072 60.3 -> 60.8; beyond, 262144 rows, 118.4 and 119.0)
uint32_t code_cells_closes(bool is_k, int ctx_len, int hidden) {
    if (const OncePlan p = code_plan(is_k, ctx_len, hidden); p.threads) return p.nwg;
    const uint32_t n = code_cells_groups(is_k, ctx_len, hidden);
    return n <= kCloseCells ? n : 0u;
}
uint32_t code_cells_words(bool is_k, int ctx_len, int hidden) {
    const OncePlan p = code_plan(is_k, ctx_len, hidden);
    return p.threads ? p.nwg : code_cells_groups(is_k, ctx_len, hidden);
}
int launch_code_cells(bool is_k, const uint8_t *codes, int ctx_len, int hidden, int bits, uint32_t bound, uint8_t *stream,
                      uint64_t capacity, uint32_t *info, ScanState *st, const EncodeClose &close, hipStream_t s) {
    const uint32_t ngroups = code_cells_groups(is_k, ctx_len, hidden);
    int rc;
    Stagger sg;
    if (const OncePlan p = code_plan(is_k, ctx_len, hidden); p.threads) {
        OnceSide a{};
        a.codes = codes; a.hidden = hidden;
        a.stream = stream; a.capacity = capacity; a.info = info; a.st = st; a.W = bits;
        a.nruns = p.nruns; a.nwg = p.nwg; a.slot = once_slot(is_k, bits);
        return p.threads == 256 ? once_launch_codes<256>(is_k, a, p.run, close, s) : once_launch_codes<1024>(is_k, a, p.run, close, s);
    } else if (is_k) {
        const uint32_t slot = (bound + 15u) & ~15u;
        const uint32_t lds = (uint32_t)kSubBlocks * slot + 32u;
        auto kern = bits > 4 ? k_code_cells_kernel<true> : k_code_cells_kernel<false>;
        if ((rc = stagger_for(reinterpret_cast<const void *>(kern), 256, lds, ngroups, &sg))) return rc;
        kern<<<ngroups, 256, lds, s>>>(codes, hidden, stream, capacity, info, st, bits, ngroups, slot, sg, close);
    } else {
        const uint32_t unit_slot = (uint32_t)(((bound - 8u) / 4u + 15u) & ~15u);
        const uint32_t lds = 64u * unit_slot + 64u;
        auto kern = bits > 4 ? v_code_cells_kernel<true> : v_code_cells_kernel<false>;
        PKV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        const unsigned threads = 512u * v_cell_segs(bits > 4);
        if ((rc = stagger_for(reinterpret_cast<const void *>(kern), (int)threads, lds, ngroups, &sg))) return rc;
        kern<<<ngroups, threads, lds, s>>>(codes, hidden, stream, capacity, info, st, bits, ngroups, unit_slot, sg, close);
    }
    PKV_HIP_CHECK(hipGetLastError());
    return PKV_OK;
}

// ---- per-token median of the V codes, straight from V -----------------------------------------------------------
// `median_repacking` (utils/compute.py:262-270) orders the tokens of a block by the lower median of each token's
// V codes over ALL channels of all sequences and heads.  This kernel gets those medians without a code matrix: a
// workgroup of 256 threads owns 16 tokens and walks the sequences; thread (token tt, l16) reads 8 channels of every
// head (the parameter pass of the round-major encoders), every lane of a token's row computes the token's scale and
// zero for itself, quantises its 64 values and counts them into a histogram column of its own in LDS
// (hist[level][thread]: one LDS add per value, no two threads on one word).  At the end the columns of a token are
// summed per level and the level that reaches rank (n - 1) / 2 is the median.  H <= 8, code width <= 6 bits.
template <int DT>
__global__ void __launch_bounds__(256, DT == PKV_F16 ? 8 : 4) token_median_from_x_kernel(const uint16_t *__restrict__ x, int B, int H, int T, float rel,
                                                                  int W, uint8_t *__restrict__ median,
                                                                  uint16_t *__restrict__ scale_out, uint16_t *__restrict__ zero_out) {
    extern __shared__ uint32_t hist[];                     // [1 << W][256]
    const int tid = threadIdx.x, tt = tid >> 4, l16 = tid & 15;
    const int levels = 1 << W;
    // workgroups go round-robin over the 8 XCDs: each XCD takes a contiguous eighth of the tokens
    const uint32_t wg = (gridDim.x & 7u) == 0u ? (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3) : blockIdx.x;
    const size_t tok0 = (size_t)wg * 16;
    const uint32_t tok_idx = (uint32_t)tok0 + (uint32_t)tt;
    for (int l = 0; l < levels; l++) hist[l * 256 + tid] = 0u;       // the thread's own column: no barrier needed
    const uint32_t lane_off = (uint32_t)(tt * kHeadDim + l16 * 8) * 2u;
    typedef __attribute__((address_space(3))) uint32_t *lds_u32_ptr;
    const uint32_t col = (uint32_t)reinterpret_cast<uintptr_t>((lds_u32_ptr)hist) + 4u * (uint32_t)tid;    // LDS byte address of the thread's column
    // the rows of sequence b + 1 are requested head by head as soon as the head's values of sequence b have been
    // quantised (into the registers they leave), so the next round trip to memory runs under this sequence's work
    auto load_row = [&](int b, int i) {
        const uint16_t *rows = x + (((size_t)b * H) * T + tok0) * kHeadDim;
        return *reinterpret_cast<const uint4 *>(reinterpret_cast<const char *>(rows + (size_t)min(i, H - 1) * T * kHeadDim) + lane_off);
    };
    uint4 v[8];
    // groups of 16 neighbouring workgroups start at different sequences: with every workgroup on the same sequence
    // at the same time the requests of the whole grid lie 8 MiB-strided rows apart in one 64 MiB range and pile up
    // on a part of the memory channels (0.251 -> 0.233 ms on 16 x 8 x 32768 tokens, with the mapping above)
    const int b_rot = (int)(wg >> 4) % B;
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = load_row(b_rot, i);
    for (int bb = 0; bb < B; bb++) {
        const int b = bb + b_rot < B ? bb + b_rot : bb + b_rot - B;
        const int bn1 = bb + 1 + b_rot;                    // the next sequence (requested while there is one)
        const int bn = bn1 < B ? bn1 : bn1 - B;
        const bool more = bb + 1 < B;
        float mn, mx;
        if (DT == PKV_F16) {
            f16x2 lo[8], hi[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const f16x2 a = __builtin_bit_cast(f16x2, v[i].x), b2 = __builtin_bit_cast(f16x2, v[i].y),
                            c = __builtin_bit_cast(f16x2, v[i].z), d = __builtin_bit_cast(f16x2, v[i].w);
                lo[i] = pk_min_h(pk_min_h(a, b2), pk_min_h(c, d));
                hi[i] = pk_max_h(pk_max_h(a, b2), pk_max_h(c, d));
            }
#pragma unroll
            for (int w = 4; w >= 1; w >>= 1)
#pragma unroll
                for (int i = 0; i < w; i++) {
                    lo[i] = pk_min_h(lo[i], lo[i + w]);
                    hi[i] = pk_max_h(hi[i], hi[i + w]);
                }
            mn = fminf((float)lo[0][0], (float)lo[0][1]);
            mx = fmaxf((float)hi[0][0], (float)hi[0][1]);
        } else {
            mn = INFINITY, mx = -INFINITY;
#pragma unroll
            for (int i = 0; i < 8; i++) minmax8<DT>(v[i], mn, mx);
        }
        row16_minmax(mn, mx);
        const float range = round_t<DT>(mx - mn);
        const float sc = round_t<DT>(range * rel);
        const uint32_t zb = T16<DT>::to_bits(rintf(round_t<DT>(__fdiv_rn(mn, sc))));
        // a wavefront holds four tokens: it takes the usual quantisation sequence when all four can, else the general
        // one for all (quant4 branches on the first lane's constants)
        if (scale_out && l16 == 0) {                       // the parameters pkv_quant_params would write, for the encoder
            // (a uniform row pointer and a 32-bit offset, written out as the store itself: the compiler kept 64-bit
            // per-lane addresses across the loop and spilled them, with a reload and a full wait in every sequence)
            uint16_t *srow = scale_out + (size_t)b * T, *zrow = zero_out + (size_t)b * T;
            const uint32_t boff = 2u * tok_idx, sbits = T16<DT>::to_bits(sc);
            asm volatile("global_store_short %0, %1, %2" : : "v"(boff), "v"(sbits), "s"(srow) : "memory");
            asm volatile("global_store_short %0, %1, %2" : : "v"(boff), "v"(zb), "s"(zrow) : "memory");
        }
        TokPar tp = token_par<DT>(sc, zb, false);
        const bool wave_usual = !__any(tp.sub2 == 0u);
        if (!wave_usual) tp = token_par<DT>(sc, zb, true);
        // count one head's eight codes (four 16-bit pairs): both halves clamped to the top level with one packed
        // operation, then one multiply-add per code forms the byte address of the level's row in the thread's column
        // (v_mad_u32_u16: 16-bit half selected by op_sel, times the row pitch, plus the column's offset)
        auto count = [&](const uint32_t c[4], int i) {
            const uint32_t one = i < H ? 1u : 0u;          // heads beyond H - 1 repeat the last one: counted as nothing
            const u16x2 top = {(unsigned short)(levels - 1), (unsigned short)(levels - 1)};
            const uint32_t pitch = 1024u;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                // (a code that does not fit W bits is counted at the top level; the encoders report it)
                const uint32_t cc = pk_u16(__builtin_elementwise_min(as_u16x2(c[q]), top));
                uint32_t a_lo, a_hi;
                asm("v_mad_u32_u16 %0, %1, %2, %3" : "=v"(a_lo) : "v"(cc), "s"(pitch), "v"(col));
                asm("v_mad_u32_u16 %0, %1, %2, %3 op_sel:[1,0,0,0]" : "=v"(a_hi) : "v"(cc), "s"(pitch), "v"(col));
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Wint-to-pointer-cast"      // the host pass sees a 64-bit pointer here; LDS pointers are 32 bits wide
                __hip_atomic_fetch_add((lds_u32_ptr)a_lo, one, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                __hip_atomic_fetch_add((lds_u32_ptr)a_hi, one, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
#pragma clang diagnostic pop
            }
        };
        // (the branch is per head and uniform, so that the request of the next sequence's row is common code: with
        // one loop per case the rows came back in different registers and were copied at the join)
#pragma unroll
        for (int i = 0; i < 8; i++) {
            uint32_t c[4];
            if (DT == PKV_F16 && wave_usual) {
                quant4_f16_fast(make_uint2(v[i].x, v[i].y), tp, c[0], c[1]);
                quant4_f16_fast(make_uint2(v[i].z, v[i].w), tp, c[2], c[3]);
            } else {
                quant4<DT>(make_uint2(v[i].x, v[i].y), tp, c[0], c[1]);
                quant4<DT>(make_uint2(v[i].z, v[i].w), tp, c[2], c[3]);
            }
            if (more) v[i] = load_row(bn, i);
            count(c, i);
        }
    }
    __syncthreads();
    // thread (tt, l16) sums the columns of token tt for its levels l16 * nper .. (a level per lane up to 16 levels)
    const int nper = levels > 16 ? levels / 16 : 1;
    uint32_t cnt[4] = {0u, 0u, 0u, 0u}, tot = 0;
    for (int sl = 0; sl < nper; sl++) {
        const int l = l16 * nper + sl;
        if (l < levels)
            for (int q = 0; q < 16; q++) cnt[sl] += hist[l * 256 + tt * 16 + ((q + l16) & 15)];
        tot += cnt[sl];
    }
    uint32_t incl = tot;                                   // inclusive scan over the 16 lanes of the token's row
    incl += __builtin_amdgcn_update_dpp(0u, incl, 0x111, 0xF, 0xF, true);
    incl += __builtin_amdgcn_update_dpp(0u, incl, 0x112, 0xF, 0xF, true);
    incl += __builtin_amdgcn_update_dpp(0u, incl, 0x114, 0xF, 0xF, true);
    incl += __builtin_amdgcn_update_dpp(0u, incl, 0x118, 0xF, 0xF, true);
    const uint32_t need = (uint32_t)((size_t)B * H * kHeadDim - 1) / 2u + 1u;      // values at or below the lower median
    uint32_t run = incl - tot;
    int found = -1;
    for (int sl = 0; sl < nper; sl++) {
        run += cnt[sl];
        if (found < 0 && run >= need) found = l16 * nper + sl;
    }
    const uint64_t has = __ballot(found >= 0);
    const uint32_t mine = (uint32_t)(has >> (16 * (tt & 3))) & 0xFFFFu;            // the token's row of the wavefront
    if (found >= 0 && (mine & ((1u << l16) - 1u)) == 0u) median[tok0 + tt] = (uint8_t)found;
}

// medians of the V codes of every token (device array of T bytes) from V itself
static int launch_token_median_from_x(const void *x, int dtype, int B, int H, int T, float rel, int bits, uint8_t *median,
                                      void *scale_out, void *zero_out, hipStream_t s) {
    const size_t lds = (size_t)(1 << bits) * 256 * sizeof(uint32_t);
    auto kern = dtype == PKV_F16 ? token_median_from_x_kernel<PKV_F16> : token_median_from_x_kernel<PKV_BF16>;
    if (lds > 48 * 1024)
        PKV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    kern<<<(unsigned)(T / 16), 256, lds, s>>>((const uint16_t *)x, B, H, T, rel, bits, median, (uint16_t *)scale_out, (uint16_t *)zero_out);
    PKV_HIP_CHECK(hipGetLastError());
    return PKV_OK;
}

static int check_xshape(const void *x, int dtype, int B, int H, int T) {
    PKV_REQUIRE(x != nullptr, PKV_ERR_INVALID, "null pointer argument");
    PKV_REQUIRE(dtype == PKV_F16 || dtype == PKV_BF16, PKV_ERR_UNSUPPORTED, "Unsupported data type");
    PKV_REQUIRE(B > 0 && H > 0 && T > 0, PKV_ERR_INVALID, "sizes must be positive");
    PKV_REQUIRE(B <= 65535 && H <= 65535, PKV_ERR_UNSUPPORTED, "batch / head count above 65535");
    return PKV_OK;
}

// One encode of the fused path: where its tokens are, where they go.
struct EncodeJob {
    const void *x;
    XRows xs;
    float rel;
    int bits;
    uint8_t *stream;
    uint64_t capacity, base;
    uint32_t *info;
    void *scale, *zero;
    int par_stride;
    const uint32_t *perm = nullptr;
    int perm_block = 0;
    const void *scale_in = nullptr, *zero_in = nullptr;
    Rot rot = {nullptr, nullptr, 0};       // K of five heads or more, in their own order
    int polls = kOncePolls;                // (pkv_quant_once.hpp)
};

// 64-bit words of look-back state the job takes: status words (one per ticket), then the words the runs of a group
// exchange: one per (run, token), where a group has more than one.
static uint64_t state_words(bool is_k, int B, int H, int T) {
    const uint64_t ctx_blk = is_k ? 64 : 128, groups = (uint64_t)T / ctx_blk * (uint64_t)B;
    const uint64_t nsub = groups * (uint64_t)(((is_k ? H : 2 * H) + kSubBlocks - 1) / kSubBlocks);
    const uint64_t n = nsub + (H <= kSubBlocks ? 0 : groups * (uint64_t)((H + kSubBlocks - 1) / kSubBlocks) * ctx_blk);
    const OncePlan p = once_plan(is_k, groups, H, kOnceSmall);
    return p.threads ? std::max(n, p.nwg * (p.nruns > 1 ? 1 + ctx_blk : 1)) : n;
}

template <bool IS_K>
static int check_job(EncodeJob &job, int dtype, int B, int H, int T) {
    const void *x = job.x, *scale = job.scale, *zero = job.zero;
    const uint8_t *stream = job.stream;
    const uint32_t *info = job.info, *perm = job.perm;
    const int bits = job.bits, par_stride = job.par_stride, perm_block = job.perm_block;
    const float rel = job.rel;
    const uint64_t base = job.base;
    uint64_t &capacity = job.capacity;
    int rc = check_xshape(x, dtype, B, H, T);
    if (rc) return rc;
    PKV_REQUIRE(stream && info && scale && zero, PKV_ERR_INVALID, "null pointer argument");
    PKV_REQUIRE((reinterpret_cast<uintptr_t>(stream) & 1u) == 0, PKV_ERR_INVALID,
                "compressed_buffer must start at an even address (blocks are written in 2-byte units)");
    PKV_REQUIRE(capacity > 0, PKV_ERR_INVALID, "compressed_buffer must be a non-empty tensor");
    PKV_REQUIRE(bits >= 2 && bits <= 6, PKV_ERR_UNSUPPORTED,
                "not supported: bits_len %d (the fused encoders take 2..6; wider codes go through pkv_quant_params, "
                "pkv_quantize and pkv_{k,v}_encode)", bits);
    PKV_REQUIRE(rel > 0.f, PKV_ERR_INVALID, "quant_scale_rel must be positive");
    const int ctx_blk = IS_K ? 64 : 128, hid_blk = IS_K ? 128 : 64;
    PKV_REQUIRE(T % ctx_blk == 0, PKV_ERR_INVALID, "ctx_len must be divisible by ctx_len_block_size");
    PKV_REQUIRE(par_stride >= T, PKV_ERR_INVALID, "parameter row stride shorter than the token count");
    if (perm) {
        PKV_REQUIRE(H <= kSubBlocks, PKV_ERR_UNSUPPORTED, "not supported: a token order with more than 8 KV heads");
        PKV_REQUIRE(perm_block >= 64 && perm_block % 64 == 0 && T % perm_block == 0, PKV_ERR_INVALID,
                    "the repacking block must be a multiple of 64 tokens that divides ctx_len");
        PKV_REQUIRE((uint64_t)H * (uint64_t)T * 256ull < (1ull << 32), PKV_ERR_UNSUPPORTED,
                    "not supported: a token order on more than 4 GiB of rows per sequence");
    }
    PKV_REQUIRE(base <= capacity, PKV_ERR_INVALID, "stream offset beyond the buffer");
    // block_info holds 32-bit byte offsets (uint32 in the reference too, evaluation/evaluation.py:420-426): a stream
    // that would grow past 4 GiB is reported as a full buffer instead of wrapping its offsets
    if (capacity > (1ull << 32)) capacity = 1ull << 32;
    PKV_REQUIRE(base <= capacity, PKV_ERR_CAPACITY, "stream offset beyond 4 GiB: block_info offsets are 32 bits");
    // (the K cells kernels reach the second head of a wavefront through a 32-bit byte offset, unless the rows are 128 apart and
    // not rotated: those hang off an address per lane)
    const bool offset = IS_K && H > 4 && (job.xs.st != kHeadDim || job.rot.cos);
    PKV_REQUIRE((!offset || job.xs.sh < (1ll << 31) - 128) && job.xs.st < (1 << 25), PKV_ERR_UNSUPPORTED,
                "not supported: 4 GiB or more from one head to the next");
    PKV_REQUIRE(state_words(IS_K, B, H, T) < (1ull << 31), PKV_ERR_UNSUPPORTED, "batch x tokens too large");
    return PKV_OK;
}

// The cells kernel of a width, a type, a token order, a row stride and (K) a rotary embedding.
template <bool IS_K, bool WIDE, int DT>
static auto cells_kernel_of(bool perm, bool xch, bool strided, bool rot) {
    if constexpr (IS_K)
        return perm ? k_quant_encode_cells_kernel<DT, WIDE, true>
               : rot ? (xch ? k_quant_encode_cells_kernel<DT, WIDE, false, true, true, true> : k_quant_encode_cells_kernel<DT, WIDE, false, false, true, true>)
               : xch ? (strided ? k_quant_encode_cells_kernel<DT, WIDE, false, true, true> : k_quant_encode_cells_kernel<DT, WIDE, false, true>)
                     : (strided ? k_quant_encode_cells_kernel<DT, WIDE, false, false, true> : k_quant_encode_cells_kernel<DT, WIDE, false>);
    else
        return perm ? v_quant_encode_cells_kernel<DT, WIDE, true>
                    : xch ? (strided ? v_quant_encode_cells_kernel<DT, WIDE, false, true, true> : v_quant_encode_cells_kernel<DT, WIDE, false, true>)
                          : (strided ? v_quant_encode_cells_kernel<DT, WIDE, false, false, true> : v_quant_encode_cells_kernel<DT, WIDE, false>);
}
template <bool IS_K>
static auto cells_kernel(int bits, int dtype, bool perm, bool xch, bool strided, bool rot = false) {
    if (bits > 4)
        return dtype == PKV_F16 ? cells_kernel_of<IS_K, true, PKV_F16>(perm, xch, strided, rot) : cells_kernel_of<IS_K, true, PKV_BF16>(perm, xch, strided, rot);
    return dtype == PKV_F16 ? cells_kernel_of<IS_K, false, PKV_F16>(perm, xch, strided, rot) : cells_kernel_of<IS_K, false, PKV_BF16>(perm, xch, strided, rot);
}

// The kernels that take a group's tokens at once (pkv_quant_once.hpp), where they serve the job.  (K reaches the second head of
// a wavefront through a 32-bit byte offset.  Groups of up to four heads in bf16 stay with the round-major kernels: those leave a
// NaN out of a token's minimum and maximum, the order keys of the cells do not.  So does V of more than eight heads for the
// other runs of eight, where the keys of all heads meet here.)
static OncePlan once_plan_of(bool is_k, const EncodeJob &job, int dtype, int B, int H, int T) {
    if (job.rot.cos || job.xs.sh >= (1ll << 31) - 128 || (H <= 4 && dtype != PKV_F16 && !job.perm) ||
        (!is_k && H > kSubBlocks && dtype != PKV_F16 && !job.scale_in)) return OncePlan{0, 0, 0, 0};
    return once_plan(is_k, (uint64_t)T / (is_k ? 64 : 128) * (uint64_t)B, H, kOnceSmall);
}
static OnceSide once_side(bool is_k, const EncodeJob &job, const OncePlan &p, int B, int H, int T, ScanState *st) {
    OnceSide a{};
    a.x = (const uint16_t *)job.x; a.xs = job.xs; a.rel = job.rel;
    a.scale = (uint16_t *)job.scale; a.zero = (uint16_t *)job.zero;
    a.stream = job.stream; a.capacity = job.capacity; a.base = job.base; a.info = job.info;
    a.st = st; a.xw = st->status + p.nwg;
    a.B = B; a.H = H; a.T = T; a.W = job.bits; a.par_stride = job.par_stride; a.nruns = p.nruns;
    a.nwg = p.nwg; a.slot = once_slot(is_k, job.bits);
    a.perm = job.perm; a.perm_block = job.perm_block;
    a.scale_in = (const uint16_t *)job.scale_in; a.zero_in = (const uint16_t *)job.zero_in;
    a.polls = job.polls;
    return a;
}

// Workgroups of a launch that closes by itself; 0: finish_encode follows.  The cells kernels of up to eight heads do so up to 2048
// workgroups.  Calls without a size one after the other, a kernel behind -> by itself, 8 heads, fp16, us: K and V of 512 tokens 16.0 -> 12.7 and
// 15.9 -> 12.7 (the host's launch), 4096 15.6 -> 14.4 and 16.0 -> 16.8, 2 x 8192 19.5 -> 19.3 and 21.5 -> 23.0 (what the runs have exchanged is cleared by
// one workgroup), 4 x 8192 32.2 -> 31.5 and 31.3 -> 30.9, 8 x 8192 53.1 -> 52.6 and 47.1 -> 46.4, 16 x 8192 90.1 -> 90.5 and 108.4 -> 97.8.  Beyond, what a
// workgroup waits for at its end costs as much or more (K of 32 x 8192 161.3 and 161.1, of 8 x 65536 304 -> 308), and runs of eight heads
// that wait for each other lose (4 x 32 heads x 16384 179.4 -> 183.2 and 197 -> 199).
static uint32_t encode_closes(bool is_k, const EncodeJob &job, int dtype, int B, int H, int T) {
    if (const OncePlan p = once_plan_of(is_k, job, dtype, B, H, T); p.threads) return p.nwg;
    if ((H <= 4 && !job.perm) || H > kSubBlocks) return 0;
    const uint64_t n = (uint64_t)(T / (is_k ? 64 : 128)) * (uint64_t)B;
    return n <= kCloseCells ? (uint32_t)n : 0u;
}

template <bool IS_K>
static int launch_quant_encode(const EncodeJob &job, int dtype, int B, int H, int T, ScanState *st, const EncodeClose &close, hipStream_t s) {
    const void *x = job.x;
    const XRows xs = job.xs;
    const float rel = job.rel;
    const int bits = job.bits, par_stride = job.par_stride, perm_block = job.perm_block;
    uint8_t *stream = job.stream;
    const uint64_t capacity = job.capacity, base = job.base;
    uint32_t *info = job.info;
    void *scale = job.scale, *zero = job.zero;
    const uint32_t *perm = job.perm;
    const void *scale_in = job.scale_in, *zero_in = job.zero_in;
    const int ctx_blk = IS_K ? 64 : 128, hid_blk = IS_K ? 128 : 64;
    int rc;
    if (const OncePlan p = once_plan_of(IS_K, job, dtype, B, H, T); p.threads) {
        const OnceSide a = once_side(IS_K, job, p, B, H, T, st), none{};
        return p.threads == 256 ? once_launch<256>(IS_K ? a : none, IS_K ? none : a, dtype, close, s) : once_launch<1024>(IS_K ? a : none, IS_K ? none : a, dtype, close, s);
    }
    // One workgroup per run of up to eight heads of a (context block, sequence) group -- K: its up to eight blocks;
    // V: its up to sixteen -- or, with fewer than five heads, per 8 / H groups.
    {
        const int HB = IS_K ? H : 2 * H;
        const uint32_t bound = IS_K ? (uint32_t)k_block_bound(ctx_blk, bits) : (uint32_t)v_block_bound(hid_blk, bits);
        const uint32_t nsub = (uint32_t)(T / ctx_blk) * (uint32_t)B * (uint32_t)((HB + kSubBlocks - 1) / kSubBlocks);
        const int nruns = (H + kSubBlocks - 1) / kSubBlocks;                // runs of eight heads per group
        const uint32_t nruns_all = (uint32_t)(T / ctx_blk) * (uint32_t)B * (uint32_t)nruns;
        if (!IS_K && H <= 8) {               // one workgroup per group of 2 H blocks
            const uint32_t unit_slot = (uint32_t)(((bound - 8u) / 4u + 15u) & ~15u);
            const uint32_t lds = 64u * unit_slot + 64u;
            const uint32_t ngroups_all = (uint32_t)(T / ctx_blk) * (uint32_t)B;
            // up to four heads: 8 / H groups to a workgroup, so that all eight head slots have blocks
            const int gpw = (H <= 4 && !perm) ? kSubBlocks / H : 1;
            const uint32_t ngroups = (ngroups_all + (uint32_t)gpw - 1u) / (uint32_t)gpw;
            // (a token order always comes with gpw == 1, i.e. the cells kernel)
            auto kern = bits > 4 ? (dtype == PKV_F16 ? v_quant_encode_rounds_kernel<PKV_F16, true>
                                                      : v_quant_encode_rounds_kernel<PKV_BF16, true>)
                                 : (dtype == PKV_F16 ? v_quant_encode_rounds_kernel<PKV_F16, false>
                                                      : v_quant_encode_rounds_kernel<PKV_BF16, false>);
            PKV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
            Stagger sg;
            if (gpw == 1) {                         // five to eight heads, or any token order: x read once, as cells
                auto cells = cells_kernel<false>(bits, dtype, perm != nullptr, false, xs.st != kHeadDim);
                PKV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(cells),
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
                const unsigned threads = 512u * v_cell_segs(bits > 4);
                if ((rc = stagger_for(reinterpret_cast<const void *>(cells), (int)threads, lds, ngroups, &sg))) return rc;
                cells<<<ngroups, threads, lds, s>>>((const uint16_t *)x, B, H, T, xs, rel, (uint16_t *)scale, (uint16_t *)zero,
                                                stream, capacity, info, st, bits, ngroups, unit_slot, base, par_stride, perm, perm_block,
                                                (const uint16_t *)scale_in, (const uint16_t *)zero_in, sg, 1, nullptr, close);
            } else {
                if ((rc = stagger_for(reinterpret_cast<const void *>(kern), 512, lds, ngroups, &sg))) return rc;
                kern<<<ngroups, 512, lds, s>>>((const uint16_t *)x, B, H, T, xs, rel, (uint16_t *)scale, (uint16_t *)zero,
                                               stream, capacity, info, st, bits, ngroups, unit_slot, base, par_stride, sg, gpw,
                                               ngroups_all);
            }
        } else if (IS_K && H <= kSubBlocks) {       // nsub == number of groups
            const uint32_t slot = (bound + 15u) & ~15u;
            // up to four heads: 8 / H groups to a workgroup, so that all eight half-wavefronts have a block
            const int gpw = (H <= 4 && !perm) ? kSubBlocks / H : 1;
            const uint32_t nwg = (nsub + (uint32_t)gpw - 1u) / (uint32_t)gpw;
            const uint32_t lds = (uint32_t)(gpw * H) * slot + 32u;
            // (a token order always comes with gpw == 1, i.e. the cells kernel: the round-major kernel serves groups of
            // up to four heads in their own order)
            auto kern = bits > 4 ? (dtype == PKV_F16 ? k_quant_encode_rounds_kernel<PKV_F16, true>
                                                      : k_quant_encode_rounds_kernel<PKV_BF16, true>)
                                 : (dtype == PKV_F16 ? k_quant_encode_rounds_kernel<PKV_F16, false>
                                                      : k_quant_encode_rounds_kernel<PKV_BF16, false>);
            Stagger sg;
            if (gpw == 1) {                         // five to eight heads: x read once, as cells
                auto cells = cells_kernel<true>(bits, dtype, perm != nullptr, false, xs.st != kHeadDim, job.rot.cos != nullptr);
                if ((rc = stagger_for(reinterpret_cast<const void *>(cells), 256, lds, nwg, &sg))) return rc;
                cells<<<nwg, 256, lds, s>>>((const uint16_t *)x, B, H, T, xs, rel, (uint16_t *)scale, (uint16_t *)zero, stream,
                                            capacity, info, st, bits, nwg, slot, base, par_stride, perm, perm_block, sg, 1, nullptr, job.rot, close);
            } else {
                if ((rc = stagger_for(reinterpret_cast<const void *>(kern), 256, lds, nwg, &sg))) return rc;
                kern<<<nwg, 256, lds, s>>>((const uint16_t *)x, B, H, T, xs, rel, (uint16_t *)scale, (uint16_t *)zero, stream,
                                           capacity, info, st, bits, nwg, slot, base, par_stride, sg, gpw, nsub);
            }
        } else if (IS_K) {                           // more than eight heads: runs of eight, one workgroup each, that exchange their minima and maxima
            const uint32_t slot = (bound + 15u) & ~15u;
            const uint32_t lds = (uint32_t)kSubBlocks * slot + 32u;
            const int nsg = (H + kSubBlocks - 1) / kSubBlocks;
            auto kern = cells_kernel<true>(bits, dtype, false, true, xs.st != kHeadDim, job.rot.cos != nullptr);
            Stagger sg;
            if ((rc = stagger_for(reinterpret_cast<const void *>(kern), 256, lds, nsub, &sg))) return rc;
            kern<<<nsub, 256, lds, s>>>((const uint16_t *)x, B, H, T, xs, rel, (uint16_t *)scale, (uint16_t *)zero, stream,
                                        capacity, info, st, bits, nsub, slot, base, par_stride, nullptr, 0, sg, nsg,
                                        st->status + nsub, job.rot, EncodeClose{});
        } else {                                     // V, more than eight heads: the same runs of eight
            const uint32_t unit_slot = (uint32_t)(((bound - 8u) / 4u + 15u) & ~15u);
            const uint32_t lds = 64u * unit_slot + 64u;
            auto kern = cells_kernel<false>(bits, dtype, false, true, xs.st != kHeadDim);
            PKV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
            Stagger sg;
            const unsigned threads = 512u * v_cell_segs(bits > 4);
            if ((rc = stagger_for(reinterpret_cast<const void *>(kern), (int)threads, lds, nruns_all, &sg))) return rc;
            kern<<<nruns_all, threads, lds, s>>>((const uint16_t *)x, B, H, T, xs, rel, (uint16_t *)scale, (uint16_t *)zero,
                                             stream, capacity, info, st, bits, nruns_all, unit_slot, base, par_stride, nullptr, 0,
                                             nullptr, nullptr, sg, nruns, st->status + nruns_all, EncodeClose{});
        }
        PKV_HIP_CHECK(hipGetLastError());
    }
    return PKV_OK;
}

static XRows dense_rows(int H, int T) { return XRows{(int64_t)H * T * kHeadDim, (int64_t)T * kHeadDim, kHeadDim}; }

template <bool IS_K>
static int run_quant_encode(const void *x, int dtype, int B, int H, int T, float rel, int bits,
                            uint8_t *stream, uint64_t capacity, uint64_t base, uint32_t *info, void *scale,
                            void *zero, int par_stride, uint64_t *size_out, float *ms_out, hipStream_t s,
                            const uint32_t *perm = nullptr, int perm_block = 0, const void *scale_in = nullptr,
                            const void *zero_in = nullptr) {
    EncodeJob job{x, dense_rows(H, T), rel, bits, stream, capacity, base, info, scale, zero, par_stride, perm, perm_block, scale_in, zero_in};
    int rc = check_job<IS_K>(job, dtype, B, H, T);
    if (rc) return rc;
    const uint32_t closes = size_out ? 0u : encode_closes(IS_K, job, dtype, B, H, T);
    ClosedEncode ce;
    ScanHandle sh;
    if ((rc = prepare_scan_state((uint32_t)state_words(IS_K, B, H, T) + (closes ? close_words(closes) : 0u), &sh, s, size_out || ms_out))) return rc;
    if (closes && (rc = ce.begin(sh, closes, s))) return rc;
    LaunchTimer tm(s, ms_out != nullptr);
    if ((rc = tm.begin())) return rc;
    if ((rc = launch_quant_encode<IS_K>(job, dtype, B, H, T, sh.st, ce.close, s))) return rc;
    if (closes && (rc = ce.launched(sh))) return rc;
    if ((rc = tm.end(ms_out))) return rc;
    return closes ? PKV_OK : finish_encode(sh, size_out, bits, s);
}

// K and V by the cells kernels in one launch: five to eight heads and codes of up to four bits on both sides, below the four
// generations of V from which the launches of their own are staggered.  B x 8 heads x 8192 tokens, us for a median repacking's
// order and encodes and for the first update of a growing cache (rotary keys), two launches -> one: fp16 B = 4 99.2 -> 84.9 and 130.5 ->
// 118.0, 6 122 -> 117 and 153 -> 140, 8 146 -> 145 and 175 -> 172, 12 227 -> 199 and 259 -> 217, 24 384 -> 347 and 376 -> 347, 32 (8192 and
// 8064 tokens) 435 -> 437 and 449 -> 427; bf16 B = 4 115 -> 93 and 144 -> 126, 8 166 -> 158 and 196 -> 195, 24 428 -> 387 and 434 -> 401, 32 522 ->
// 493; at 8192 tokens, staggered, 414 -> 429 and 484 -> 497.  In turns up to 1024 groups of V, V first beyond (fp16 B = 16 269 -> 259 us in
// turns, but 24 347 -> 359 and 32 427 -> 445).
constexpr uint64_t kBothGroups = 2048, kBothTurns = 1024;
static bool cells_in_one_launch(const EncodeJob job[2], const OncePlan &pk, const OncePlan &pv, int B, int H, int T) {
    return !pk.threads && !pv.threads && H > 4 && H <= kSubBlocks && job[0].bits <= 4 && job[1].bits <= 4 &&
           job[0].xs.sh < (1ll << 31) - 128 && (uint64_t)(T / 128) * (uint64_t)B < kBothGroups;
}
static int launch_cells_both(const EncodeJob job[2], int dtype, int B, int H, int T, ScanState *k_st, ScanState *v_st, hipStream_t s) {
    CellsSide side[2];
    for (int i = 0; i < 2; i++) {
        const EncodeJob &a = job[i];
        const uint32_t bound = i ? ((uint32_t)v_block_bound(64, a.bits) - 8u) / 4u : (uint32_t)k_block_bound(64, a.bits);
        side[i] = CellsSide{(const uint16_t *)a.x, a.xs, a.rel, (uint16_t *)a.scale, (uint16_t *)a.zero, a.stream, a.capacity, a.base, a.info,
                            i ? v_st : k_st, a.bits, (uint32_t)(T / (i ? 128 : 64)) * (uint32_t)B, (bound + 15u) & ~15u,
                            (const uint16_t *)a.scale_in, (const uint16_t *)a.zero_in};
    }
    const uint32_t lds_k = 2u * (uint32_t)H * side[0].slot + 32u, lds_v = 64u * side[1].slot + 64u, lds = lds_k > lds_v ? lds_k : lds_v;
    const bool perm = job[0].perm != nullptr, rot = job[0].rot.cos != nullptr;
    auto pick = [&](auto f16, auto bf16) { return dtype == PKV_F16 ? f16 : bf16; };
    auto kern = perm ? pick(kv_quant_encode_cells_kernel<PKV_F16, true, false>, kv_quant_encode_cells_kernel<PKV_BF16, true, false>)
                : rot ? pick(kv_quant_encode_cells_kernel<PKV_F16, false, true>, kv_quant_encode_cells_kernel<PKV_BF16, false, true>)
                      : pick(kv_quant_encode_cells_kernel<PKV_F16, false, false>, kv_quant_encode_cells_kernel<PKV_BF16, false, false>);
    PKV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const uint32_t vg = side[1].ngroups;
    kern<<<2u * vg, 512, lds, s>>>(side[0], side[1], B, H, T, job[0].par_stride, job[0].perm, job[0].perm_block,
                                   vg <= kBothTurns ? vg >> 8 : 0u, job[0].rot);
    PKV_HIP_CHECK(hipGetLastError());
    return PKV_OK;
}

// K and V (checked jobs) with one wait; in one launch where both take a group's tokens at once.
static int encode_both(const EncodeJob job[2], int dtype, int B, int H, int T, uint64_t *k_size, uint64_t *v_size, hipStream_t s) {
    int rc;
    ScanHandle sh;
    if ((rc = prepare_scan_state((uint32_t)state_words(true, B, H, T), &sh, s, true, (uint32_t)state_words(false, B, H, T)))) return rc;
    const OncePlan pk = once_plan_of(true, job[0], dtype, B, H, T), pv = once_plan_of(false, job[1], dtype, B, H, T);
    if (pk.threads && pk.threads == pv.threads && (job[0].bits > 4) == (job[1].bits > 4)) {
        const OnceSide ks = once_side(true, job[0], pk, B, H, T, sh.st), vs = once_side(false, job[1], pv, B, H, T, sh.second);
        if ((rc = pk.threads == 256 ? once_launch<256>(ks, vs, dtype, EncodeClose{}, s) : once_launch<1024>(ks, vs, dtype, EncodeClose{}, s))) return rc;
    } else if (cells_in_one_launch(job, pk, pv, B, H, T)) {
        if ((rc = launch_cells_both(job, dtype, B, H, T, sh.st, sh.second, s))) return rc;
    } else {
        if ((rc = launch_quant_encode<true>(job[0], dtype, B, H, T, sh.st, EncodeClose{}, s))) return rc;
        if ((rc = launch_quant_encode<false>(job[1], dtype, B, H, T, sh.second, EncodeClose{}, s))) return rc;
    }
    return finish_encode(sh, k_size, job[0].bits, s, v_size, job[1].bits);
}

// The jobs of two sides, checked.  With a token order the rows are dense.
static int append_jobs(EncodeJob job[2], const pkv_append_side *k, const pkv_append_side *v, int dtype, int B, int H, int T, int par_stride,
                       const uint32_t *perm, int perm_block, bool sizes) {
    PKV_REQUIRE(k && v && sizes, PKV_ERR_INVALID, "null pointer argument");
    for (int i = 0; i < 2; i++) {
        const pkv_append_side &a = i ? *v : *k;
        PKV_REQUIRE(a.stride_b >= 0 && a.stride_h >= 0 && a.stride_t >= 0 && a.stride_t < (1 << 25) &&
                        (a.stride_b | a.stride_h | a.stride_t) % 8 == 0 && (reinterpret_cast<uintptr_t>(a.x) & 15u) == 0,
                    PKV_ERR_INVALID, "rows must start on 16-byte boundaries (row stride below 2^25 elements)");
        job[i] = EncodeJob{a.x, perm ? dense_rows(H, T) : XRows{a.stride_b, a.stride_h, a.stride_t}, a.rel, a.bits, a.stream, a.capacity, a.used,
                           a.info_tail, a.scale_tail, a.zero_tail, par_stride, perm, perm_block};
        PKV_REQUIRE((a.cos == nullptr) == (a.sin == nullptr), PKV_ERR_INVALID, "cos and sin go together");
        if (a.cos) {
            PKV_REQUIRE(i == 0 && H > 4 && !perm, PKV_ERR_UNSUPPORTED, "not supported: a rotary embedding other than of K with five heads or more");
            PKV_REQUIRE(a.rot_stride_b >= 0 && a.rot_stride_b % 8 == 0 && ((reinterpret_cast<uintptr_t>(a.cos) | reinterpret_cast<uintptr_t>(a.sin)) & 15u) == 0,
                        PKV_ERR_INVALID, "rows must start on 16-byte boundaries");
            job[i].rot = Rot{(const uint16_t *)a.cos, (const uint16_t *)a.sin, a.rot_stride_b};
        }
        const int rc = i ? check_job<false>(job[i], dtype, B, H, T) : check_job<true>(job[i], dtype, B, H, T);
        if (rc) return rc;
    }
    return PKV_OK;
}

}  // namespace pkv

extern "C" {

int pkv_median_order(const void *v, int dtype, int B, int H, int T, float rel, int bits, int block_size, uint32_t *perm,
                     void *scale_out, void *zero_out, float *ms_out, pkv_stream_t s_) {
    using namespace pkv;
    hipStream_t s = (hipStream_t)s_;
    int rc = check_xshape(v, dtype, B, H, T);
    if (rc) return rc;
    PKV_REQUIRE(perm != nullptr, PKV_ERR_INVALID, "null pointer argument");
    PKV_REQUIRE((scale_out == nullptr) == (zero_out == nullptr), PKV_ERR_INVALID, "scale_out and zero_out go together");
    PKV_REQUIRE(rel > 0.f, PKV_ERR_INVALID, "quant_scale_rel must be positive");
    PKV_REQUIRE(H <= kSubBlocks, PKV_ERR_UNSUPPORTED, "not supported: more than 8 KV heads (order the code matrix with pkv_median_repack)");
    PKV_REQUIRE(bits >= 2 && bits <= 6, PKV_ERR_UNSUPPORTED, "not supported: bits_len %d (2..6)", bits);
    PKV_REQUIRE(block_size > 0 && block_size <= 1024 && T % block_size == 0 && T % 16 == 0, PKV_ERR_INVALID,
                "ctx_len must be divisible by 16 and by a block size of at most 1024 tokens");
    void *scratch = nullptr;
    if ((rc = scratch_get((size_t)T, s, &scratch))) return rc;
    uint8_t *median = static_cast<uint8_t *>(scratch);
    LaunchTimer tm(s, ms_out != nullptr);
    if ((rc = tm.begin())) return rc;
    if ((rc = launch_token_median_from_x(v, dtype, B, H, T, rel, bits, median, scale_out, zero_out, s))) return rc;
    if ((rc = launch_block_order(median, T, block_size, perm, s))) return rc;
    return tm.end(ms_out);
}

int pkv_k_quant_encode_perm(const void *x, int dtype, int B, int H, int T, float rel, int bits, const uint32_t *perm,
                            int perm_block, uint8_t *stream, uint64_t capacity, uint32_t *block_info, void *scale,
                            void *zero, uint64_t *size_out, float *ms_out, pkv_stream_t s) {
    PKV_REQUIRE(perm != nullptr, PKV_ERR_INVALID, "null pointer argument");
    return pkv::run_quant_encode<true>(x, dtype, B, H, T, rel, bits, stream, capacity, 0, block_info, scale, zero, T,
                                       size_out, ms_out, (hipStream_t)s, perm, perm_block);
}

int pkv_v_quant_encode_perm(const void *x, int dtype, int B, int H, int T, float rel, int bits, const uint32_t *perm,
                            int perm_block, const void *scale_in, const void *zero_in, uint8_t *stream, uint64_t capacity,
                            uint32_t *block_info, void *scale, void *zero, uint64_t *size_out, float *ms_out, pkv_stream_t s) {
    PKV_REQUIRE(perm != nullptr, PKV_ERR_INVALID, "null pointer argument");
    PKV_REQUIRE((scale_in == nullptr) == (zero_in == nullptr), PKV_ERR_INVALID, "scale_in and zero_in go together");
    PKV_REQUIRE(scale_in == nullptr || (scale_in != scale && zero_in != zero), PKV_ERR_INVALID,
                "the known parameters (order of x) and the written ones (order of the stream) are different arrays");
    return pkv::run_quant_encode<false>(x, dtype, B, H, T, rel, bits, stream, capacity, 0, block_info, scale, zero, T,
                                        size_out, ms_out, (hipStream_t)s, perm, perm_block, scale_in, zero_in);
}

int pkv_kv_quant_encode_perm(const pkv_append_side *k, const pkv_append_side *v, int dtype, int B, int H, int T, const uint32_t *perm, int perm_block,
                             const void *v_scale_in, const void *v_zero_in, uint64_t *k_size, uint64_t *v_size, pkv_stream_t s_) {
    using namespace pkv;
    PKV_REQUIRE(k && v && k_size && v_size && perm, PKV_ERR_INVALID, "null pointer argument");
    PKV_REQUIRE((v_scale_in == nullptr) == (v_zero_in == nullptr), PKV_ERR_INVALID, "scale_in and zero_in go together");
    PKV_REQUIRE(v_scale_in == nullptr || (v_scale_in != v->scale_tail && v_zero_in != v->zero_tail), PKV_ERR_INVALID,
                "the known parameters (order of x) and the written ones (order of the stream) are different arrays");
    EncodeJob job[2];
    for (int i = 0; i < 2; i++) {
        const pkv_append_side &a = i ? *v : *k;
        job[i] = EncodeJob{a.x, dense_rows(H, T), a.rel, a.bits, a.stream, a.capacity, 0, a.info_tail, a.scale_tail, a.zero_tail, T, perm, perm_block,
                           i ? v_scale_in : nullptr, i ? v_zero_in : nullptr};
        const int rc = i ? check_job<false>(job[i], dtype, B, H, T) : check_job<true>(job[i], dtype, B, H, T);
        if (rc) return rc;
    }
    return encode_both(job, dtype, B, H, T, k_size, v_size, (hipStream_t)s_);
}

int pkv_quant_params(const void *x, int dtype, int B, int H, int T, float rel, void *scale, void *zero,
                     float *ms_out, pkv_stream_t s_) {
    using namespace pkv;
    hipStream_t s = (hipStream_t)s_;
    int rc = check_xshape(x, dtype, B, H, T);
    if (rc) return rc;
    PKV_REQUIRE(scale && zero, PKV_ERR_INVALID, "null pointer argument");
    PKV_REQUIRE(rel > 0.f, PKV_ERR_INVALID, "quant_scale_rel must be positive");
    LaunchTimer tm(s, ms_out != nullptr);
    if ((rc = tm.begin())) return rc;
    const dim3 grid((unsigned)((T + 15) / 16), (unsigned)B);
    if (dtype == PKV_F16)
        quant_params_kernel<PKV_F16><<<grid, 256, 0, s>>>((const uint16_t *)x, H, T, rel, (uint16_t *)scale,
                                                          (uint16_t *)zero);
    else
        quant_params_kernel<PKV_BF16><<<grid, 256, 0, s>>>((const uint16_t *)x, H, T, rel, (uint16_t *)scale,
                                                           (uint16_t *)zero);
    PKV_HIP_CHECK(hipGetLastError());
    return tm.end(ms_out);
}

int pkv_quantize(const void *x, int dtype, int B, int H, int T, const void *scale, const void *zero,
                 uint8_t *codes, uint32_t *max_code_out, float *ms_out, pkv_stream_t s_) {
    using namespace pkv;
    hipStream_t s = (hipStream_t)s_;
    int rc = check_xshape(x, dtype, B, H, T);
    if (rc) return rc;
    PKV_REQUIRE(scale && zero && codes, PKV_ERR_INVALID, "null pointer argument");
    LaunchTimer tm(s, ms_out != nullptr);
    if ((rc = tm.begin())) return rc;
    const dim3 grid((unsigned)((T + 15) / 16), (unsigned)((H + kQuantHeads - 1) / kQuantHeads), (unsigned)B);
    if (dtype == PKV_F16)
        quantize_kernel<PKV_F16><<<grid, 256, 0, s>>>((const uint16_t *)x, H, T, (const uint16_t *)scale,
                                                      (const uint16_t *)zero, codes, max_code_out);
    else
        quantize_kernel<PKV_BF16><<<grid, 256, 0, s>>>((const uint16_t *)x, H, T, (const uint16_t *)scale,
                                                       (const uint16_t *)zero, codes, max_code_out);
    PKV_HIP_CHECK(hipGetLastError());
    return tm.end(ms_out);
}

int pkv_quant_codes(const void *k, const void *v, int dtype, int B, int H, int T, float k_rel, float v_rel, void *k_scale, void *k_zero,
                    uint8_t *k_codes, void *v_scale, void *v_zero, uint8_t *v_codes, pkv_stream_t s_) {
    using namespace pkv;
    hipStream_t s = (hipStream_t)s_;
    int rc = check_xshape(k, dtype, B, H, T);
    if (rc || (v && (rc = check_xshape(v, dtype, B, H, T)))) return rc;
    PKV_REQUIRE(k_scale && k_zero && k_codes && (!v || (v_scale && v_zero && v_codes)), PKV_ERR_INVALID, "null pointer argument");
    PKV_REQUIRE(k_rel > 0.f && (!v || v_rel > 0.f), PKV_ERR_INVALID, "quant_scale_rel must be positive");
    const QuantSide ks{(const uint16_t *)k, k_rel, (uint16_t *)k_scale, (uint16_t *)k_zero, k_codes},
                    vs{(const uint16_t *)v, v_rel, (uint16_t *)v_scale, (uint16_t *)v_zero, v_codes};
    const dim3 grid((unsigned)((T + 15) / 16), (unsigned)B, v ? 2u : 1u);
    if (dtype == PKV_F16) quant_codes_kernel<PKV_F16><<<grid, 256, 0, s>>>(ks, vs, H, T);
    else quant_codes_kernel<PKV_BF16><<<grid, 256, 0, s>>>(ks, vs, H, T);
    PKV_HIP_CHECK(hipGetLastError());
    return PKV_OK;
}

int pkv_dequantize(const uint8_t *codes, int dtype, int B, int H, int T, const void *scale,
                   const void *zero, void *x_out, float *ms_out, pkv_stream_t s_) {
    using namespace pkv;
    hipStream_t s = (hipStream_t)s_;
    int rc = check_xshape(x_out, dtype, B, H, T);
    if (rc) return rc;
    PKV_REQUIRE(scale && zero && codes, PKV_ERR_INVALID, "null pointer argument");
    LaunchTimer tm(s, ms_out != nullptr);
    if ((rc = tm.begin())) return rc;
    const dim3 grid((unsigned)((T + 15) / 16), (unsigned)((H + kQuantHeads - 1) / kQuantHeads), (unsigned)B);
    if (dtype == PKV_F16)
        dequantize_kernel<PKV_F16><<<grid, 256, 0, s>>>(codes, H, T, (const uint16_t *)scale,
                                                        (const uint16_t *)zero, (uint16_t *)x_out);
    else
        dequantize_kernel<PKV_BF16><<<grid, 256, 0, s>>>(codes, H, T, (const uint16_t *)scale,
                                                         (const uint16_t *)zero, (uint16_t *)x_out);
    PKV_HIP_CHECK(hipGetLastError());
    return tm.end(ms_out);
}

int pkv_k_quant_encode(const void *x, int dtype, int B, int H, int T, float rel, int bits, uint8_t *stream,
                       uint64_t capacity, uint32_t *block_info, void *scale, void *zero,
                       uint64_t *size_out, float *ms_out, pkv_stream_t s) {
    return pkv::run_quant_encode<true>(x, dtype, B, H, T, rel, bits, stream, capacity, 0, block_info, scale,
                                       zero, T, size_out, ms_out, (hipStream_t)s);
}

int pkv_v_quant_encode(const void *x, int dtype, int B, int H, int T, float rel, int bits, uint8_t *stream,
                       uint64_t capacity, uint32_t *block_info, void *scale, void *zero,
                       uint64_t *size_out, float *ms_out, pkv_stream_t s) {
    return pkv::run_quant_encode<false>(x, dtype, B, H, T, rel, bits, stream, capacity, 0, block_info, scale,
                                        zero, T, size_out, ms_out, (hipStream_t)s);
}

int pkv_k_quant_encode_append(const void *x, int dtype, int B, int H, int T_new, float rel, int bits,
                               uint8_t *stream, uint64_t capacity, uint64_t stream_used, uint32_t *block_info_tail,
                               void *scale_tail, void *zero_tail, int par_stride, uint64_t *size_out,
                               float *ms_out, pkv_stream_t s) {
    return pkv::run_quant_encode<true>(x, dtype, B, H, T_new, rel, bits, stream, capacity, stream_used,
                                       block_info_tail, scale_tail, zero_tail, par_stride, size_out, ms_out,
                                       (hipStream_t)s);
}

int pkv_v_quant_encode_append(const void *x, int dtype, int B, int H, int T_new, float rel, int bits,
                               uint8_t *stream, uint64_t capacity, uint64_t stream_used, uint32_t *block_info_tail,
                               void *scale_tail, void *zero_tail, int par_stride, uint64_t *size_out,
                               float *ms_out, pkv_stream_t s) {
    return pkv::run_quant_encode<false>(x, dtype, B, H, T_new, rel, bits, stream, capacity, stream_used,
                                        block_info_tail, scale_tail, zero_tail, par_stride, size_out, ms_out,
                                        (hipStream_t)s);
}

int pkv_kv_quant_encode_append(const pkv_append_side *k, const pkv_append_side *v, int dtype, int B, int H, int T_new,
                               int par_stride, uint64_t *k_size, uint64_t *v_size, pkv_stream_t s) {
    using namespace pkv;
    EncodeJob job[2];
    const int rc = append_jobs(job, k, v, dtype, B, H, T_new, par_stride, nullptr, 0, k_size && v_size);
    return rc ? rc : encode_both(job, dtype, B, H, T_new, k_size, v_size, (hipStream_t)s);
}

int pkv_kv_quant_encode_alone(const pkv_append_side *k, const pkv_append_side *v, int dtype, int B, int H, int T_new, int par_stride,
                              const uint32_t *perm, int perm_block, uint64_t *k_size, uint64_t *v_size, pkv_stream_t s) {
    using namespace pkv;
    EncodeJob job[2];
    const int rc = append_jobs(job, k, v, dtype, B, H, T_new, par_stride, perm, perm_block, k_size && v_size);
    if (rc) return rc;
    job[0].polls = job[1].polls = 0;
    return encode_both(job, dtype, B, H, T_new, k_size, v_size, (hipStream_t)s);
}

}  // extern "C"
