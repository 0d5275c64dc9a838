// Fused decompress-attention decode: one query token per sequence attends over a compressed
// K/V cache (plus an optional 16-bit tail window) without materialising K or V.
//
// Fuses the reference's chain  kq_mat_vec_mul -> fused_kq -> softmax -> w * v_scale ->
// wv_mat_vec_mul -> fused_wv  (packkv_cuda_ext/src/kernels.cu:426-535, :632-765,
// src/fused_kernels.cu:13-76, :187-261, models/llama.py:202-209,
// evaluation/evaluation.py:661) and adds batch and GQA-group dimensions.
//
// Work decomposition (flash-decoding): grid (split, kv_head, batch).  A workgroup walks
// 128-token super-tiles = 2 K blocks (64 x 128) + 2 V blocks (128 x 64) of its head and keeps
// an online-softmax state; each split writes (m, l, acc[128]) per query head, a small merge
// kernel combines the splits and the tail window.
#include "pkv_block.hpp"
#include "pkv_runtime.hpp"

#include <mutex>

#ifndef PKV_DYNAMIC_TILES
#define PKV_DYNAMIC_TILES 1
#endif
#ifndef PKV_SPLIT_TARGET
#define PKV_SPLIT_TARGET 1024
#endif

namespace pkv {

constexpr int kTile = 128;              // tokens per super-tile
constexpr int kPartStride = 2 + kHeadDim;  // floats per partial: m, l, acc[128]
typedef float float2v __attribute__((ext_vector_type(2)));
// Rows of q and v_win and results are promised at their elements' alignment only.  The same wide instructions (global
// accesses take any address), without telling the compiler more than that.
typedef uint32_t uint4_at2 __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t uint_at2 __attribute__((aligned(2)));
typedef float float2v_at4 __attribute__((ext_vector_type(2), aligned(4)));
__device__ __forceinline__ uint4 load_uint4(const uint4_at2 *p) {
    const uint4_at2 v = *p;
    return make_uint4(v[0], v[1], v[2], v[3]);
}

__device__ __forceinline__ float a_ld16(const uint16_t *p, size_t i, int dtype) {
    const uint32_t u = p[i];
    return dtype == PKV_F16 ? __half2float(__ushort_as_half((unsigned short)u)) : __uint_as_float(u << 16);
}

__device__ __forceinline__ uint16_t a_st16(float x, int dtype) {
    if (dtype == PKV_F16) return __half_as_ushort(__float2half_rn(x));
    uint32_t u = __float_as_uint(x);
    if ((u & 0x7FFFFFFFu) > 0x7F800000u) return (uint16_t)((u >> 16) | 0x40u);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

struct AttnParams {
    const uint8_t *k_stream;
    const uint32_t *k_info;
    const uint8_t *v_stream;
    const uint32_t *v_info;
    const uint16_t *k_scale, *k_zero, *v_scale, *v_zero;
    const uint16_t *q;
    const uint16_t *k_win, *v_win;
    float *part;          // [B, Hq, nparts, kPartStride]
    uint16_t *out;        // [B, Hq, 128]: written directly by the attention kernel when there is a single partial
    int B, Hq, Hkv, T_c, T_w;
    int Gq;               // query heads per KV head; the kernels are built for the next of 1, 2, 4, 8 and leave the rest idle
    int par_stride;       // tokens per sequence row of the scale / zero arrays (>= T_c)
    int win_stride;       // tokens per (sequence, KV head) row of k_win / v_win (>= T_w)
    int k_bits, v_bits, dtype;
    float sm_scale;
    int tiles_per_split, nsplit, nparts;
    int win_piece;        // window tokens per piece; piece i writes partial nsplit + i
    int win_members;      // async-copy kernel: workgroups of their own per KV head for the pieces; 0: split i takes piece i
    uint32_t k_cap, v_cap, blk_stride;
    uint32_t k_bytes, v_bytes;   // valid bytes of the streams
    int out_f32;          // `out` holds fp32 instead of the 16-bit storage type
    int direct_out;       // a single partial and a 16-bit result: the async-copy kernel writes `out` itself
    int dynamic;          // async-copy kernel: the members of a (sequence, KV head) take tiles from a common counter
    int batch_shift;      // ... in batches of (tiles left >> batch_shift), at least 1 and at most 4
    int merge;            // async-copy kernel: the last workgroup of a (sequence, KV head) to finish merges its partials
    uint32_t *counters;   // [B Hkv] tile counters, [B Hkv] counts of members that are done with them, [B Hkv] workgroups that
                          // have written their partials; zero between launches
};

// x rounded to the 16-bit storage type (nearest even), as fp32.
__device__ __forceinline__ float round16(float x, int dtype) {
    const uint32_t u = a_st16(x, dtype);
    return dtype == PKV_F16 ? __half2float(__ushort_as_half((unsigned short)u)) : __uint_as_float(u << 16);
}

// A partial is written through to memory: the workgroup that merges it may run on another XCD, behind another L2, in the
// same launch (merge_head).
__device__ __forceinline__ void part_store(float *p, float x) { __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// ---- variant 1: decode tiles into LDS, then plain VALU attention --------------------------
// Straightforward and easy to audit; kept as the cross-check for the tuned kernel.
// REF: decompress-then-attend to the letter -- every element is formed as the reference stores it,
// T(T(code + zero) * scale) (utils/compute.py:178), and the dot products run on those values.
template <int G, bool REF>
__global__ void __launch_bounds__(256) attn_tiles_kernel(const AttnParams p) {
    extern __shared__ __align__(16) uint8_t lds[];
    uint8_t *ktile = lds;                                   // [128 tok][128 ch]
    uint8_t *vtile = ktile + kTile * kHeadDim;              // [128 tok][128 ch]
    uint8_t *blkbuf = vtile + kTile * kHeadDim;             // 4 x blk_stride
    float *fl = reinterpret_cast<float *>(blkbuf + 4 * p.blk_stride);
    float *qf = fl;                       // [G][128]
    float *S = qf + G * kHeadDim;         // [G][128]
    float *P = S + G * kTile;             // [G][128]
    float *ks = P + G * kTile;            // [128] x4
    float *kz = ks + kTile, *vs = kz + kTile, *vz = vs + kTile;
    float *st_m = vz + kTile;             // [G] each
    float *st_l = st_m + G, *st_a = st_l + G, *st_z = st_a + G, *qsum = st_z + G;
    __shared__ uint32_t s_phase[4], s_off[4];

    const int split = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
    const int tid = threadIdx.x;
    const int lane32 = tid & 31, hw = tid >> 5;
    const int bh = b * p.Hkv + h;
    const int n_hid_k = p.B * p.Hkv, n_hid_v = 2 * p.B * p.Hkv;
    const UnitGeom gk = unit_geom(p.k_bits), gv = unit_geom(p.v_bits);

    for (int i = tid; i < G * kHeadDim; i += 256)
        qf[i] = i < p.Gq * kHeadDim ? a_ld16(p.q, ((size_t)b * p.Hq + (size_t)h * p.Gq) * kHeadDim + i, p.dtype) : 0.f;
    if (tid < G) { st_m[tid] = -INFINITY; st_l[tid] = 0.f; st_z[tid] = 0.f; }
    __syncthreads();
    if (tid < G) {
        float s = 0.f;
        for (int d = 0; d < kHeadDim; d++) s += qf[tid * kHeadDim + d];
        qsum[tid] = s;
    }
    float acc[G];
#pragma unroll
    for (int g = 0; g < G; g++) acc[g] = 0.f;

    const int n_tiles = p.T_c / kTile;
    const int tile0 = split * p.tiles_per_split;
    const int tile1 = min(n_tiles, tile0 + p.tiles_per_split);
    for (int tau = tile0; tau < tile1; tau++) {
        // 1. stage the four blocks and the per-token quantizer parameters
        for (int j = 0; j < 4; j++) {
            const bool is_k = j < 2;
            const uint32_t bidx = is_k ? (uint32_t)((2 * tau + j) * n_hid_k + bh)
                                       : (uint32_t)(tau * n_hid_v + 2 * bh + (j - 2));
            const uint32_t *info = is_k ? p.k_info : p.v_info;
            const uint8_t *stream = is_k ? p.k_stream : p.v_stream;
            uint32_t off, size;
            block_span(info, bidx, is_k ? p.k_cap : p.v_cap, is_k ? p.k_bytes : p.v_bytes, off, size);
            const uint32_t ph = stage_to_lds(stream + off, size, blkbuf + j * p.blk_stride, tid, 256);
            if (tid == 0) s_phase[j] = ph;
        }
        if (tid < kTile) {
            const size_t ti = (size_t)b * p.par_stride + (size_t)tau * kTile + tid;
            ks[tid] = a_ld16(p.k_scale, ti, p.dtype);
            kz[tid] = a_ld16(p.k_zero, ti, p.dtype);
            vs[tid] = a_ld16(p.v_scale, ti, p.dtype);
            vz[tid] = a_ld16(p.v_zero, ti, p.dtype);
        }
        __syncthreads();
        // 2. unpack: half-wave hw handles K unit (block hw/4, round hw%4) and V unit
        //    (block hw/4 = channel half, segment hw%4)
        {
            const int j = hw >> 2, unit = hw & 3;
            const uint8_t *kb = blkbuf + j * p.blk_stride;
            const uint32_t kph = s_phase[j];
            const uint16_t *kcum = reinterpret_cast<const uint16_t *>(kb + kph);
            const uint32_t kstart = kph + 8u + (unit ? (uint32_t)kcum[unit - 1] : 0u);
            unit_decode<true>(kb, kstart, unit, lane32, gk, ktile + j * 64 * kHeadDim, kHeadDim);
            const uint8_t *vb = blkbuf + (2 + j) * p.blk_stride;
            const uint32_t vph = s_phase[2 + j];
            const uint16_t *vcum = reinterpret_cast<const uint16_t *>(vb + vph);
            const uint32_t vstart = vph + 8u + (unit ? (uint32_t)vcum[unit - 1] : 0u);
            unit_decode<false>(vb, vstart, unit, lane32, gv, vtile + j * 64, kHeadDim);
        }
        __syncthreads();
        // 3. scores: two threads per token, 64 channels each
        {
            const int tok = tid >> 1, half = tid & 1;
            const uint32_t *row = reinterpret_cast<const uint32_t *>(ktile + tok * kHeadDim + half * 64);
            float dot[G];
#pragma unroll
            for (int g = 0; g < G; g++) dot[g] = 0.f;
            const float s_tok = ks[tok], z_tok = kz[tok];
#pragma unroll 4
            for (int i = 0; i < 16; i++) {
                const uint32_t w = row[i];
                float c0 = (float)(w & 0xFFu), c1 = (float)((w >> 8) & 0xFFu),
                      c2 = (float)((w >> 16) & 0xFFu), c3 = (float)(w >> 24);
                if (REF) {
                    c0 = round16(round16(c0 + z_tok, p.dtype) * s_tok, p.dtype);
                    c1 = round16(round16(c1 + z_tok, p.dtype) * s_tok, p.dtype);
                    c2 = round16(round16(c2 + z_tok, p.dtype) * s_tok, p.dtype);
                    c3 = round16(round16(c3 + z_tok, p.dtype) * s_tok, p.dtype);
                }
#pragma unroll
                for (int g = 0; g < G; g++) {
                    const float *qq = qf + g * kHeadDim + half * 64 + 4 * i;
                    dot[g] += qq[0] * c0 + qq[1] * c1 + qq[2] * c2 + qq[3] * c3;
                }
            }
#pragma unroll
            for (int g = 0; g < G; g++) {
                const float d = dot[g] + __shfl_xor(dot[g], 1, 64);
                if (half == 0) S[g * kTile + tok] = REF ? d * p.sm_scale : p.sm_scale * s_tok * (d + z_tok * qsum[g]);
            }
        }
        __syncthreads();
        // 4. online softmax: wavefront w owns query heads w, w+4, ...
        for (int g = tid >> 6; g < G; g += 4) {
            const int lane = tid & 63;
            const float s0 = S[g * kTile + lane], s1 = S[g * kTile + 64 + lane];
            float mx = fmaxf(s0, s1);
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) mx = fmaxf(mx, __shfl_xor(mx, d, 64));
            const float m_old = st_m[g];
            const float m_new = fmaxf(m_old, mx);
            const float p0 = __expf(s0 - m_new), p1 = __expf(s1 - m_new);
            const float w0 = REF ? p0 : p0 * vs[lane], w1 = REF ? p1 : p1 * vs[64 + lane];
            P[g * kTile + lane] = w0;
            P[g * kTile + 64 + lane] = w1;
            float sum = p0 + p1;
            float zs = REF ? 0.f : w0 * vz[lane] + w1 * vz[64 + lane];
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) {
                sum += __shfl_xor(sum, d, 64);
                zs += __shfl_xor(zs, d, 64);
            }
            if (lane == 0) {
                const float alpha = __expf(m_old - m_new);   // exp(-inf) = 0 on the first tile
                st_a[g] = alpha;
                st_m[g] = m_new;
                st_l[g] = st_l[g] * alpha + sum;
                st_z[g] = st_z[g] * alpha + zs;
            }
        }
        __syncthreads();
        // 5. PV: thread = (channel, token half)
        {
            const int ch = tid & 127, half = tid >> 7;
            float part[G];
#pragma unroll
            for (int g = 0; g < G; g++) part[g] = 0.f;
#pragma unroll 8
            for (int t = 0; t < 64; t++) {
                float c = (float)vtile[(half * 64 + t) * kHeadDim + ch];
                if (REF) c = round16(round16(c + vz[half * 64 + t], p.dtype) * vs[half * 64 + t], p.dtype);
#pragma unroll
                for (int g = 0; g < G; g++) part[g] += P[g * kTile + half * 64 + t] * c;
            }
#pragma unroll
            for (int g = 0; g < G; g++) acc[g] = acc[g] * st_a[g] + part[g];
        }
        __syncthreads();
    }
    // combine the two token halves and write the partial
    {
        const int ch = tid & 127, half = tid >> 7;
        float *red = S;   // reuse: [G][128]
        if (half == 1)
            for (int g = 0; g < G; g++) red[g * kTile + ch] = acc[g];
        __syncthreads();
        if (half == 0) {
            for (int g = 0; g < p.Gq; g++) {
                const size_t hq = (size_t)b * p.Hq + (size_t)h * p.Gq + g;
                float *dst = p.part + (hq * p.nparts + split) * kPartStride;
                dst[2 + ch] = acc[g] + red[g * kTile + ch] + st_z[g];
                if (ch == 0) { dst[0] = st_m[g]; dst[1] = st_l[g]; }
            }
        }
    }
}

// ---- matrix-core kernels (variants 0 and 2): shared arithmetic ----------------------------
// K side: every half-wavefront unpacks one round (16 tokens x 128 channels, lane t = channels
// 4t..4t+3) into an int8 tile in LDS laid out [token][channel]; the tile is read back in the
// operand layout of the 16x16 int8 MFMAs (lane = token, 8 consecutive channels per 8-byte read;
// the staged kernel pairs two reads into one v_mfma_i32_16x16x64_i8 operand, the gather kernel
// issues v_mfma_i32_16x16x32_i8 per read) and contracted against q, which is split per query head into three signed 7-bit digits
// (q = qs * (d0 * 2^14 + d1 * 2^7 + d2)), one MFMA row per (digit, head).  Integer arithmetic
// is exact, so the scores carry only the 2^-21 relative rounding of that split.
// V side: lane = channel as in the stream, nothing is transposed.  MFMA number k of a segment
// takes token k of each of the lane's four packs (rounds) as its four contraction slots, so a
// register pair of 16-bit fields is an operand as it stands: the masked field bits are the fp16
// SUBNORMAL delta * 2^-24 (the matrix cores take subnormal inputs exactly), no conversion.  The A
// operand holds the softmax weights (times v_scale) of the 4 query heads, so the per-lane
// accumulators are out[g][channel] and need no cross-lane reduction; pack minima enter through
// one more MFMA against the per-round weight sums (split hi/lo).
typedef int int4v __attribute__((ext_vector_type(4)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef _Float16 half4v __attribute__((ext_vector_type(4)));
typedef unsigned short ushort2v __attribute__((ext_vector_type(2)));

constexpr int kKtStride = 136;         // bytes per token row of the int8 K tile (128 + 8 pad)
constexpr int kKtDw = kKtStride / 4;

__device__ __forceinline__ uint32_t pk_shr16(uint32_t v, uint32_t sh) {
    ushort2v a = __builtin_bit_cast(ushort2v, v), b = __builtin_bit_cast(ushort2v, sh);
    return __builtin_bit_cast(uint32_t, (ushort2v)(a >> b));
}

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_keep(float x) {   // lanes without a valid source keep x
    const int v = __builtin_bit_cast(int, x);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(v, v, CTRL, ROW_MASK, 0xF, false));
}

__device__ __forceinline__ float wave_max(float x) {
    x = fmaxf(x, dpp_keep<0xB1, 0xF>(x));    // quad_perm [1,0,3,2]
    x = fmaxf(x, dpp_keep<0x4E, 0xF>(x));    // quad_perm [2,3,0,1]
    x = fmaxf(x, dpp_keep<0x141, 0xF>(x));   // row_half_mirror
    x = fmaxf(x, dpp_keep<0x140, 0xF>(x));   // row_mirror
    x = fmaxf(x, dpp_keep<0x142, 0xA>(x));   // row_bcast:15 into rows 1 and 3
    x = fmaxf(x, dpp_keep<0x143, 0xC>(x));   // row_bcast:31 into rows 2 and 3
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), 63));
}

__device__ __forceinline__ float row16_sum(float x) {  // every lane gets the sum of its 16-lane row
    x += dpp_keep<0xB1, 0xF>(x);
    x += dpp_keep<0x4E, 0xF>(x);
    x += dpp_keep<0x141, 0xF>(x);
    x += dpp_keep<0x140, 0xF>(x);
    return x;
}

__device__ __forceinline__ float wave_sum(float x) {
    x = row16_sum(x);
    const int v = __builtin_bit_cast(int, x);
    float s = 0.f;
#pragma unroll
    for (int r = 0; r < 4; r++) s += __builtin_bit_cast(float, __builtin_amdgcn_readlane(v, 16 * r));
    return s;
}

// ---- 16-bit tail window ------------------------------------------------------------------------------------------
// Attention of the query heads of KV head (h, b) over tokens [t0, t1) of the uncompressed tail window, written as
// partial `part_idx` (an empty range writes a partial of weight zero).  `lds` provides min(G, 4) * 528 floats.  Called by
// all 256 threads of a workgroup.
// Latency is all there is to it (64 rows of K and V are 32 KB), so a workgroup makes one trip to memory per 64 tokens:
// thread (tt = tid / 16, c = tid % 16) asks for 16 bytes of K and of V of tokens tt, tt + 16, tt + 32, tt + 48, and
// everything until the end stays inside the wavefront -- scores by DPP sums over the 16 lanes of a row, a maximum, sums
// and outputs of the wavefront's own -- so that one barrier, before the four wavefronts' results are combined, is the
// only one.
constexpr int kWinChunk = 64;         // tokens per trip
constexpr int kWinLds = 528;          // floats of LDS per query head: four wavefronts' outputs, maxima and sums
constexpr int kWinPieceLds = 4 * kWinLds * 4;   // LDS every instance of the async-copy kernel has in its two slots

template <bool BF>
__device__ __forceinline__ void cvt_pair(uint32_t w, float &lo, float &hi) {
    if (!BF) {
        lo = __half2float(__ushort_as_half((unsigned short)(w & 0xFFFFu)));
        hi = __half2float(__ushort_as_half((unsigned short)(w >> 16)));
    } else {
        lo = __uint_as_float(w << 16);
        hi = __uint_as_float(w & 0xFFFF0000u);
    }
}
template <bool BF>
__device__ __forceinline__ void cvt8(const uint4 v, float f[8]) {
    cvt_pair<BF>(v.x, f[0], f[1]); cvt_pair<BF>(v.y, f[2], f[3]); cvt_pair<BF>(v.z, f[4], f[5]); cvt_pair<BF>(v.w, f[6], f[7]);
}
// x of this lane and of the lane 32 (16) positions away: the halves (rows) of two registers change places
__device__ __forceinline__ float add_swap32(float a, float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float((uint32_t)r[0]) + __uint_as_float((uint32_t)r[1]);
}
__device__ __forceinline__ float add_swap16(float a, float b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float((uint32_t)r[0]) + __uint_as_float((uint32_t)r[1]);
}

// Heads gb .. gb + G - 1 of the group, G <= 4.
template <int G, bool BF>
__device__ __forceinline__ void window_heads(const AttnParams &p, uint8_t *lds, int h, int b, int gb, int t0, int t1,
                                             int part_idx) {
    float *red = reinterpret_cast<float *>(lds);             // [4 wavefronts][G][128], then maxima and sums [4][G] each
    float *red_m = red + 4 * G * kHeadDim, *red_l = red_m + 4 * G;
    const int tid = threadIdx.x, tt = tid >> 4, c = tid & 15, wave = tid >> 6, lane = tid & 63;
    const size_t row0 = ((size_t)b * p.Hkv + h) * p.win_stride;
    const uint4 *kbase = reinterpret_cast<const uint4 *>(p.k_win + row0 * kHeadDim) + c;
    const uint4_at2 *vbase = reinterpret_cast<const uint4_at2 *>(p.v_win + row0 * kHeadDim) + c;
    float q[G][8], acc[G][8], m[G], l[G];
#pragma unroll
    for (int g = 0; g < G; g++) {
        uint4 w = make_uint4(0u, 0u, 0u, 0u);                // an idle head slot (group of 3 in the kernel of 4, ...)
        if (gb + g < p.Gq) w = load_uint4(reinterpret_cast<const uint4_at2 *>(p.q + ((size_t)b * p.Hq + (size_t)h * p.Gq + gb + g) * kHeadDim) + c);
        cvt8<BF>(w, q[g]);
        m[g] = -INFINITY; l[g] = 0.f;
#pragma unroll
        for (int j = 0; j < 8; j++) acc[g][j] = 0.f;
    }
    for (int base = t0; base < t1; base += kWinChunk) {
        uint4 kr[4], vr[4];
#pragma unroll
        for (int i = 0; i < 4; i++) kr[i] = kbase[(size_t)min(base + 16 * i + tt, t1 - 1) * 16];      // (past the end: the last row again, weight zero)
#pragma unroll
        for (int i = 0; i < 4; i++) vr[i] = load_uint4(vbase + (size_t)min(base + 16 * i + tt, t1 - 1) * 16);
        float s[G][4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float k8[8];
            cvt8<BF>(kr[i], k8);
            const bool in = base + 16 * i + tt < t1;
#pragma unroll
            for (int g = 0; g < G; g++) {
                float d = 0.f;
#pragma unroll
                for (int j = 0; j < 8; j++) d = fmaf(q[g][j], k8[j], d);
                s[g][i] = in ? row16_sum(d) * p.sm_scale : -INFINITY;
            }
        }
#pragma unroll
        for (int g = 0; g < G; g++) {
            const float mx = fmaxf(m[g], wave_max(fmaxf(fmaxf(s[g][0], s[g][1]), fmaxf(s[g][2], s[g][3]))));
            const float ref = mx == -INFINITY ? 0.f : mx;    // a wavefront without tokens: weights of zero, not NaN
            const float alpha = __expf(m[g] - ref);
            m[g] = mx;
            l[g] *= alpha;
#pragma unroll
            for (int j = 0; j < 8; j++) acc[g][j] *= alpha;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                s[g][i] = __expf(s[g][i] - ref);
                l[g] += s[g][i];
            }
        }
        // past the end V is zero as well: weight zero times an infinity of the last row would be NaN.  (The lanes compare
        // again: the masks of the scores, kept until here, would take scalar registers the tiles' loop has not got.)
        int rows = t1 - base - tt;
        asm volatile("" : "+v"(rows));
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float v8[8];
            if (16 * i >= rows) vr[i] = make_uint4(0u, 0u, 0u, 0u);
            cvt8<BF>(vr[i], v8);
#pragma unroll
            for (int g = 0; g < G; g++)
#pragma unroll
                for (int j = 0; j < 8; j++) acc[g][j] = fmaf(s[g][i], v8[j], acc[g][j]);
        }
    }
    // sums over the wavefront's four rows: while there are heads to share out, a step trades half of them with the lanes
    // 32 (16) positions away, so that afterwards a row holds G / 4 heads (all of them when G is 1)
    constexpr int G2 = G >= 2 ? G / 2 : 1, G4 = G >= 4 ? G / 4 : 1;
#pragma unroll
    for (int g = 0; g < G2; g++) {
#pragma unroll
        for (int j = 0; j < 8; j++) acc[g][j] = add_swap32(acc[g][j], acc[G >= 2 ? g + G2 : g][j]);
        l[g] = add_swap32(l[g], l[G >= 2 ? g + G2 : g]);
    }
#pragma unroll
    for (int g = 0; g < G4; g++) {
#pragma unroll
        for (int j = 0; j < 8; j++) acc[g][j] = add_swap16(acc[g][j], acc[G >= 4 ? g + G4 : g][j]);
        l[g] = add_swap16(l[g], l[G >= 4 ? g + G4 : g]);
    }
    const int g0 = (G >= 2 ? (lane >> 5) * G2 : 0) + (G >= 4 ? ((lane >> 4) & 1) * G4 : 0);
    if (G >= 4 || (lane & (G == 2 ? 16 : 48)) == 0) {
#pragma unroll
        for (int g = 0; g < G4; g++) {
            float4v *dst = reinterpret_cast<float4v *>(red + (wave * G + g0 + g) * kHeadDim + 8 * c);
            dst[0] = (float4v){acc[g][0], acc[g][1], acc[g][2], acc[g][3]};
            dst[1] = (float4v){acc[g][4], acc[g][5], acc[g][6], acc[g][7]};
            if (c == 0) red_l[wave * G + g0 + g] = l[g];
        }
    }
    if (lane == 0) {
#pragma unroll
        for (int g = 0; g < G; g++) red_m[wave * G + g] = m[g];
    }
    __syncthreads();
    for (int i = tid; i < min(G, p.Gq - gb) * kHeadDim; i += 256) {
        const int g = i >> 7, ch = i & (kHeadDim - 1);
        const float M = fmaxf(fmaxf(red_m[g], red_m[G + g]), fmaxf(red_m[2 * G + g], red_m[3 * G + g]));
        const float ref = M == -INFINITY ? 0.f : M;
        float num = 0.f, den = 0.f;
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const float e = __expf(red_m[w * G + g] - ref);
            num = fmaf(e, red[(w * G + g) * kHeadDim + ch], num);
            den = fmaf(e, red_l[w * G + g], den);
        }
        const size_t hq = (size_t)b * p.Hq + (size_t)h * p.Gq + gb + g;
        if (p.direct_out) {                                  // the only partial: the result itself
            p.out[hq * kHeadDim + ch] = a_st16(num / den, p.dtype);
            continue;
        }
        float *dst = p.part + (hq * p.nparts + part_idx) * kPartStride;
        part_store(dst + 2 + ch, num);
        if (ch == 0) { part_store(dst, M); part_store(dst + 1, den); }
    }
}

// (groups of eight heads in two halves: their queries and sums together need 170 registers)
template <int G, bool BF>
__device__ __forceinline__ void window_body(const AttnParams &p, uint8_t *lds, int h, int b, int t0, int t1, int part_idx) {
    if constexpr (G <= 4) {
        window_heads<G, BF>(p, lds, h, b, 0, t0, t1, part_idx);
    } else {
#pragma unroll 1
        for (int gb = 0; gb < p.Gq; gb += 4) {
            if (gb) __syncthreads();                         // the first half's results are read
            window_heads<4, BF>(p, lds, h, b, gb, t0, t1, part_idx);
        }
    }
}

// The window in pieces of its own: grid (Hkv, B, pieces), partial nsplit + piece.
template <int G, bool BF>
__global__ void __launch_bounds__(256) attn_window_kernel(const AttnParams p) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[kWinPieceLds];
    const int t0 = (int)blockIdx.z * p.win_piece;
    window_body<G, BF>(p, lds, blockIdx.x, blockIdx.y, t0, min(t0 + p.win_piece, p.T_w), p.nsplit + (int)blockIdx.z);
}

// ---- merge of a head's partials by the last of its `arrivals` workgroups to get here (async-copy kernel) ----
// Saves the launch of the merge kernel, its run and the gap in front of it.  The price is three trips past the L2s -- a
// workgroup's stores, its count, the last one's read of all partials -- and that the counts on one address retire one
// after the other.  merge_pays says where the price is lower.  4-bit fp16 steps, us per step in a graph of 40 (launched
// one by one the host takes about 12.7 us for two launches and 10 for one, so that there every step below that gains),
// with the merge launch -> merged here; `pairs` = sequences x KV heads:
//   several tiles a workgroup, 4 to 8 workgroups a head: always.  Groups of 4: 128 pairs x 256 tiles 116.0 -> 114.7, x 32
//     24.7 -> 23.8, 256 x 32 38.6 -> 37.1; groups of 8: 128 x 16 22.9 -> 22.5, 256 x 64 86.4 -> 84.8
//   one tile each, when all workgroups of a head arrive at once and nothing hides the trips: groups of 8 never (two heads a
//     wavefront one after the other: 8 pairs x 6 tiles 10.8 -> 11.5, 128 x 2 11.2 -> 11.8); else up to 14 pairs (14 x 8 9.0 ->
//     9.3, but 12.6 -> 9.9 one by one; 8 x 4 8.8 -> 8.7) and from 72 on (72 x 8 11.2 -> 11.0, 128 x 4 10.3 -> 9.9; groups of
//     1: 128 x 8 11.3 -> 10.8); in between up to four workgroups (32 x 4 9.0 -> 9.2, groups of 1 8.3 -> 8.1, but 32 x 8 9.0 ->
//     10.0, 64 x 8 10.0 -> 11.0), with groups of 4 and more than 32 pairs three (64 x 3 9.0 -> 9.4, x 4 9.1 -> 9.7).
//   32 workgroups a head (32 heads x 4096 tokens) 15.5 -> 16.5, 24 (3 x 8 x 11008 + 137) 25.2 -> 27.2 (both before a member's
//     last tile became a step of its own): hence at most eight.
// Every workgroup has written its partials through to memory (part_store) and waited for that before it counts itself;
// the reader's loads go past its own L2.  No workgroup waits for another.  Lane = two adjacent channels; a wavefront merges
// a head of its own when the group has four or more, otherwise the wavefronts share a head's partials and meet in LDS.
constexpr int kMergeArrivals = 8;
static bool merge_pays(int G, int pairs, int nsplit, int tiles_per_split) {
    if (tiles_per_split > 1) return true;
    return G <= 4 && (pairs <= 14 || pairs >= 72 || nsplit <= (G == 4 && pairs > 32 ? 3 : 4));
}
template <int G>
__device__ __forceinline__ void merge_head(const AttnParams &p, uint8_t *lds, int h, int b, uint32_t arrivals) {
    constexpr int WPH = G >= 4 ? 1 : 4 / G;          // wavefronts per head
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    volatile uint32_t *last = reinterpret_cast<volatile uint32_t *>(lds);
    float2v *sums = reinterpret_cast<float2v *>(lds + 16);        // [4 wavefronts][64 lanes]
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");             // this wavefront's partials have reached memory
    __syncthreads();
    if (tid == 0) {
        uint32_t *count = p.counters + 2 * p.B * p.Hkv + b * p.Hkv + h;
        const bool all = __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u == arrivals;
        if (all) __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *last = all ? 1u : 0u;
    }
    __syncthreads();
    if (*last == 0u) return;
    const int sub = wave % WPH;
    for (int g = wave / WPH; g < p.Gq; g += 4 / WPH) {
        const size_t hq = (size_t)b * p.Hq + (size_t)h * p.Gq + g;
        const float *base = p.part + hq * p.nparts * kPartStride;
        // lane <-> partial (at most two per workgroup): maximum, weights, denominator
        const uint64_t ml = __hip_atomic_load(reinterpret_cast<const uint64_t *>(base + (size_t)min(lane, p.nparts - 1) * kPartStride),
                                              __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint64_t *col = reinterpret_cast<const uint64_t *>(base + 2) + lane;
        constexpr int kRows = 2 * kMergeArrivals / WPH;
        uint64_t v[kRows];
#pragma unroll
        for (int u = 0; u < kRows; u++)
            v[u] = __hip_atomic_load(col + (size_t)min(sub + WPH * u, p.nparts - 1) * (kPartStride / 2), __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_AGENT);
        const bool there = lane < p.nparts;
        const float m = there ? __uint_as_float((uint32_t)ml) : -INFINITY, l = there ? __uint_as_float((uint32_t)(ml >> 32)) : 0.f;
        const float w = __expf(m - wave_max(m));
        const float den = wave_sum(w * l);
        float2v num = {0.f, 0.f};
#pragma unroll
        for (int u = 0; u < kRows; u++) {
            const int at = sub + WPH * u;
            const float wu = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w), at));
            if (at < p.nparts) {
                num[0] = fmaf(wu, __uint_as_float((uint32_t)v[u]), num[0]);
                num[1] = fmaf(wu, __uint_as_float((uint32_t)(v[u] >> 32)), num[1]);
            }
        }
        if constexpr (WPH > 1) {                     // (one pass of this loop: the group has G = 4 / WPH heads)
            sums[tid] = num;
            __syncthreads();
            if (sub) return;
#pragma unroll
            for (int i = 1; i < WPH; i++) num += sums[tid + 64 * i];
        }
        if (p.out_f32) {
            reinterpret_cast<float2v_at4 *>(reinterpret_cast<float *>(p.out) + hq * kHeadDim)[lane] = num / den;
        } else {
            const uint32_t lo = a_st16(num[0] / den, p.dtype), hi = a_st16(num[1] / den, p.dtype);
            reinterpret_cast<uint_at2 *>(p.out + hq * kHeadDim)[lane] = lo | (hi << 16);
        }
    }
}

// ---- merge of the per-split partials: grid (Hq, B), 256 threads, nparts floats of dynamic LDS ----
// Partials are read in parallel: thread <-> partial for the maxima and weights, then thread <-> (parity of the
// partial, channel) for the weighted sum, four rows in flight.
__global__ void __launch_bounds__(256) attn_merge_kernel(const float *__restrict__ part, uint16_t *__restrict__ out,
                                                         int Hq, int nparts, int dtype, int out_f32) {
    extern __shared__ float w_s[];                   // weight of every partial
    __shared__ float red[8];
    __shared__ __attribute__((aligned(8))) float part_num[3 * kHeadDim];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const size_t hq = (size_t)blockIdx.y * Hq + blockIdx.x;
    const float *base = part + hq * nparts * kPartStride;
    float mx = -INFINITY;
    for (int s = tid; s < nparts; s += 256) mx = fmaxf(mx, base[(size_t)s * kPartStride]);
    mx = wave_max(mx);
    if (lane == 0) red[wave] = mx;
    __syncthreads();
    const float M = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    float den = 0.f;
    for (int s = tid; s < nparts; s += 256) {
        const float w = __expf(base[(size_t)s * kPartStride] - M);
        w_s[s] = w;
        den += w * base[(size_t)s * kPartStride + 1];
    }
    den = wave_sum(den);
    if (lane == 0) red[4 + wave] = den;
    __syncthreads();
    den = (red[4] + red[5]) + (red[6] + red[7]);
    // weighted sum: wavefront = every fourth partial, lane = two adjacent channels (rows are 8-byte aligned), eight
    // loads in flight per lane -- a long list of partials (small batches spread one head over many splits) is a
    // chain of dependent round trips otherwise
    const float2v *col = reinterpret_cast<const float2v *>(base + 2) + lane;
    float2v num = {0.f, 0.f};
    int s = wave;
    for (; s + 28 < nparts; s += 32) {
        float2v v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = col[(size_t)(s + 4 * u) * (kPartStride / 2)];
#pragma unroll
        for (int u = 0; u < 8; u++) num += w_s[s + 4 * u] * v[u];
    }
    if (s < nparts) {                                  // the last, partial batch: still one round trip
        float2v v[8];
        float w[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int idx = min(s + 4 * u, nparts - 1);
            v[u] = col[(size_t)idx * (kPartStride / 2)];
            w[u] = w_s[idx];
        }
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (s + 4 * u < nparts) num += w[u] * v[u];      // (not a weight of zero: the last partial may hold an infinity)
    }
    if (wave) reinterpret_cast<float2v *>(part_num + (wave - 1) * kHeadDim)[lane] = num;
    __syncthreads();
    if (wave == 0) {
#pragma unroll
        for (int w = 0; w < 3; w++) num += reinterpret_cast<const float2v *>(part_num + w * kHeadDim)[lane];
        if (out_f32) {
            reinterpret_cast<float2v_at4 *>(reinterpret_cast<float *>(out) + hq * kHeadDim)[lane] = num / den;
        } else {
            const uint32_t lo = a_st16(num[0] / den, dtype), hi = a_st16(num[1] / den, dtype);
            reinterpret_cast<uint_at2 *>(out + hq * kHeadDim)[lane] = lo | (hi << 16);
        }
    }
}

}  // namespace pkv
#include "pkv_attn_direct.hpp"
namespace pkv {

template <int G, int KW, int VW>
static int launch_direct(const AttnParams &p, hipStream_t s) {
    constexpr int GP = ((G + 3) / 4) * 4;
    const uint32_t lds_bytes = 8u * 16u * kKtStride + kRing * 16u * 4u + GP * kTile * 2u + 2u * GP * 8u * 2u + 6u * 8u * 4u;
    const dim3 grid((unsigned)p.nsplit, (unsigned)p.Hkv, (unsigned)p.B);
    if (p.dtype == PKV_BF16)
        attn_direct_kernel<G, KW, VW, true><<<grid, 256, lds_bytes, s>>>(p);
    else
        attn_direct_kernel<G, KW, VW, false><<<grid, 256, lds_bytes, s>>>(p);
    PKV_HIP_CHECK(hipGetLastError());
    return PKV_OK;
}

}  // namespace pkv
#include "pkv_attn_dma.hpp"
namespace pkv {

template <int G, int KW, int VW>
static int launch_dma(const AttnParams &p, hipStream_t s) {
    static_assert(dma_lds_bytes<G, KW, VW>() >= kWinPieceLds, "window pieces borrow the slots");
    const dim3 grid((unsigned)(p.nsplit + p.win_members) * (unsigned)p.Hkv * (unsigned)p.B);
    if (p.dtype == PKV_BF16)
        attn_dma_kernel<G, KW, VW, true><<<grid, 256, 0, s>>>(p);
    else
        attn_dma_kernel<G, KW, VW, false><<<grid, 256, 0, s>>>(p);
    PKV_HIP_CHECK(hipGetLastError());
    return PKV_OK;
}

// PKV_ATTN_MINIMAL (kernel development only): instantiate the 4-bit kernels for groups of 4 and 1 alone; every other
// shape is refused.  Cuts the compile of this file from minutes to seconds.
template <int G>
static int launch_dma_bits(const AttnParams &p, hipStream_t s) {
#ifdef PKV_ATTN_MINIMAL
#if PKV_ATTN_MINIMAL == 55     // (-DPKV_ATTN_MINIMAL=55: the 5-bit kernel instead, =33: the 3-bit kernel)
    if constexpr (G == 4) { if (p.k_bits == 5 && p.v_bits == 5) return launch_dma<G, 5, 5>(p, s); }
#elif PKV_ATTN_MINIMAL == 33
    if constexpr (G == 4) { if (p.k_bits == 3 && p.v_bits == 3) return launch_dma<G, 3, 3>(p, s); }
#else
    if constexpr (G == 4 || G == 1) { if (p.k_bits == 4 && p.v_bits == 4) return launch_dma<G, 4, 4>(p, s); }
#endif
    PKV_REQUIRE(false, PKV_ERR_UNSUPPORTED, "minimal build: 4-bit codes and groups of 4 only");
#else
    switch (p.k_bits * 8 + p.v_bits) {
        case 2 * 8 + 2: return launch_dma<G, 2, 2>(p, s);
        case 2 * 8 + 3: return launch_dma<G, 2, 3>(p, s);
        case 2 * 8 + 4: return launch_dma<G, 2, 4>(p, s);
        case 3 * 8 + 2: return launch_dma<G, 3, 2>(p, s);
        case 3 * 8 + 3: return launch_dma<G, 3, 3>(p, s);
        case 3 * 8 + 4: return launch_dma<G, 3, 4>(p, s);
        case 4 * 8 + 2: return launch_dma<G, 4, 2>(p, s);
        case 4 * 8 + 3: return launch_dma<G, 4, 3>(p, s);
        case 5 * 8 + 5: return launch_dma<G, 5, 5>(p, s);       // the extension widths 5 and 6, for K, V or both
        case 6 * 8 + 6: return launch_dma<G, 6, 6>(p, s);
        case 5 * 8 + 4: return launch_dma<G, 5, 4>(p, s);
        case 4 * 8 + 5: return launch_dma<G, 4, 5>(p, s);
        case 6 * 8 + 5: return launch_dma<G, 6, 5>(p, s);
        case 5 * 8 + 6: return launch_dma<G, 5, 6>(p, s);
        case 6 * 8 + 4: return launch_dma<G, 6, 4>(p, s);
        case 4 * 8 + 6: return launch_dma<G, 4, 6>(p, s);
        default: return launch_dma<G, 4, 4>(p, s);
    }
#endif
}

template <int G>
static int launch_direct_bits(const AttnParams &p, hipStream_t s) {
#ifdef PKV_ATTN_MINIMAL
    PKV_REQUIRE(false, PKV_ERR_UNSUPPORTED, "minimal build: the asynchronous-copy kernel only");
#else
    switch (p.k_bits * 8 + p.v_bits) {
        case 2 * 8 + 2: return launch_direct<G, 2, 2>(p, s);
        case 2 * 8 + 3: return launch_direct<G, 2, 3>(p, s);
        case 2 * 8 + 4: return launch_direct<G, 2, 4>(p, s);
        case 3 * 8 + 2: return launch_direct<G, 3, 2>(p, s);
        case 3 * 8 + 3: return launch_direct<G, 3, 3>(p, s);
        case 3 * 8 + 4: return launch_direct<G, 3, 4>(p, s);
        case 4 * 8 + 2: return launch_direct<G, 4, 2>(p, s);
        case 4 * 8 + 3: return launch_direct<G, 4, 3>(p, s);
        default: return launch_direct<G, 4, 4>(p, s);
    }
#endif
}

template <int G>
static int launch_attn(const AttnParams &p, int variant, bool aligned16, bool ref_rounding, uint16_t *out, hipStream_t s) {
    PKV_REQUIRE(variant >= 0 && variant <= 2, PKV_ERR_INVALID, "variant must be 0, 1 or 2");
    // variant 0: asynchronous-copy kernel (needs 16-byte aligned streams; otherwise, and as
    // variant 2, the kernel that gathers straight from global memory); variant 1: plain VALU kernel
    if (p.T_c > 0 && variant == 0 && aligned16) {
        const int rc = launch_dma_bits<G>(p, s);
        if (rc) return rc;
    } else if (p.T_c > 0 && (variant == 0 || variant == 2)) {
        const int rc = launch_direct_bits<G>(p, s);
        if (rc) return rc;
    } else if (p.T_c > 0) {
        const uint32_t lds_bytes = 2u * kTile * kHeadDim + 4u * p.blk_stride +
                                   (uint32_t)sizeof(float) * (G * kHeadDim + 2 * G * kTile + 4 * kTile + 5 * G);
        const dim3 grid((unsigned)p.nsplit, (unsigned)p.Hkv, (unsigned)p.B);
        const void *fn = ref_rounding ? reinterpret_cast<const void *>(attn_tiles_kernel<G, true>)
                                      : reinterpret_cast<const void *>(attn_tiles_kernel<G, false>);
        PKV_HIP_CHECK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes));
        if (ref_rounding)
            attn_tiles_kernel<G, true><<<grid, 256, lds_bytes, s>>>(p);
        else
            attn_tiles_kernel<G, false><<<grid, 256, lds_bytes, s>>>(p);
        PKV_HIP_CHECK(hipGetLastError());
    }
    const bool dma_path = p.T_c > 0 && variant == 0 && aligned16;
    if (p.T_w > 0 && !dma_path) {
        const dim3 grid((unsigned)p.Hkv, (unsigned)p.B, (unsigned)((p.T_w + p.win_piece - 1) / p.win_piece));
        if (p.dtype == PKV_BF16) attn_window_kernel<G, true><<<grid, 256, 0, s>>>(p);
        else attn_window_kernel<G, false><<<grid, 256, 0, s>>>(p);
        PKV_HIP_CHECK(hipGetLastError());
    }
    // (a single partial is the result, and the async-copy kernel merges short lists itself)
    if (!((dma_path || p.T_c == 0) && p.direct_out) && !p.merge) {
        attn_merge_kernel<<<dim3((unsigned)p.Hq, (unsigned)p.B), 256, (size_t)p.nparts * sizeof(float), s>>>(
            p.part, out, p.Hq, p.nparts, p.dtype, p.out_f32);
        PKV_HIP_CHECK(hipGetLastError());
    }
    return PKV_OK;
}

}  // namespace pkv

// ---- partials without an allocation --------------------------------------------------------------
// pkv_attn_decode_noalloc keeps the per-split partials in this array instead of library-allocated memory.  Every
// GPU the library runs on holds its own copy, at its own address, until the process ends.  In host code the name
// below is only a handle for hipGetSymbolAddress: the device address it yields (per device) is what kernels get.
#define PKV_ATTN_STATIC_SCRATCH_BYTES (8u << 20)
static __device__ __align__(256) unsigned char scratch[PKV_ATTN_STATIC_SCRATCH_BYTES];
// layout: partials, then the tile counters of the async-copy kernel (zero at load, left at zero by every launch)
static constexpr size_t kStaticPartBytes = (size_t)PKV_ATTN_STATIC_SCRATCH_BYTES - (size_t)pkv::kAttnCounters * sizeof(uint32_t);

namespace pkv {
namespace {
constexpr int kStaticMaxDevices = 16;
void *g_static_part[kStaticMaxDevices];          // device address of `scratch` on each device, once looked up
std::mutex g_static_mu;

// Device address of this device's copy of `scratch` (looked up once per device, with that device current).
int static_scratch_ptr(void **out) {
    int dev = 0;
    PKV_HIP_CHECK(hipGetDevice(&dev));
    PKV_REQUIRE(dev >= 0 && dev < kStaticMaxDevices, PKV_ERR_INVALID, "device index %d out of range", dev);
    std::lock_guard<std::mutex> lock(g_static_mu);
    if (!g_static_part[dev]) {
        void *ptr = nullptr;
        PKV_HIP_CHECK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        PKV_REQUIRE(ptr != nullptr, PKV_ERR_HIP, "hipGetSymbolAddress returned a null address");
        g_static_part[dev] = ptr;
    }
    *out = g_static_part[dev];
    return PKV_OK;
}

}  // namespace
static int attn_decode_impl(const pkv_attn_args *a, float *ms_out, hipStream_t s, bool static_partials);
}  // namespace pkv

extern "C" int pkv_attn_decode(const pkv_attn_args *a, float *ms_out, pkv_stream_t s_) {
    return pkv::attn_decode_impl(a, ms_out, (hipStream_t)s_, false);
}

extern "C" int pkv_attn_decode_noalloc(const pkv_attn_args *a, pkv_stream_t s_) {
    return pkv::attn_decode_impl(a, nullptr, (hipStream_t)s_, true);
}

int pkv::attn_decode_impl(const pkv_attn_args *a, float *ms_out, hipStream_t s, bool static_partials) {
    PKV_REQUIRE(a != nullptr, PKV_ERR_INVALID, "null pointer argument");
    PKV_REQUIRE(a->dtype == PKV_F16 || a->dtype == PKV_BF16, PKV_ERR_UNSUPPORTED, "Unsupported data type");
    PKV_REQUIRE(a->B > 0 && a->Hq > 0 && a->Hkv > 0 && a->Hq % a->Hkv == 0, PKV_ERR_INVALID,
                "need B, Hq, Hkv > 0 and Hq divisible by Hkv");
    PKV_REQUIRE(a->B <= 65535 && a->Hkv <= 65535, PKV_ERR_UNSUPPORTED, "batch / head count above 65535");
    PKV_REQUIRE(a->T_c >= 0 && a->T_w >= 0 && a->T_c + a->T_w > 0, PKV_ERR_INVALID, "empty cache");
    PKV_REQUIRE(a->T_c % kTile == 0, PKV_ERR_INVALID, "compressed length must be a multiple of 128 tokens");
    PKV_REQUIRE(a->T_w <= 2048, PKV_ERR_UNSUPPORTED, "tail window longer than 2048 tokens");
    PKV_REQUIRE(a->q && a->out, PKV_ERR_INVALID, "null pointer argument");
    PKV_REQUIRE((a->flags & ~(PKV_ATTN_REF_ROUNDING | PKV_ATTN_OUT_F32)) == 0, PKV_ERR_INVALID, "unknown flag bits");
    const bool ref_rounding = (a->flags & PKV_ATTN_REF_ROUNDING) != 0;
    PKV_REQUIRE(!ref_rounding || a->variant == 1, PKV_ERR_INVALID,
                "PKV_ATTN_REF_ROUNDING is a mode of the plain kernel (variant 1)");
    if (a->T_c > 0) {
        PKV_REQUIRE(a->k_stream && a->k_info && a->v_stream && a->v_info && a->k_scale && a->k_zero &&
                        a->v_scale && a->v_zero,
                    PKV_ERR_INVALID, "null pointer argument");
        PKV_REQUIRE(a->k_bits >= 2 && a->k_bits <= kMaxBits && a->v_bits >= 2 && a->v_bits <= kMaxBits, PKV_ERR_UNSUPPORTED,
                    "not supported: bits_len outside 2..8");
        PKV_REQUIRE(a->k_bytes > 0 && a->v_bytes > 0 && a->k_bytes < (1ull << 32) && a->v_bytes < (1ull << 32),
                    PKV_ERR_INVALID, "stream sizes must be in 1 .. 4 GiB - 1");
    }
    const int par_stride = a->par_stride ? a->par_stride : a->T_c, win_stride = a->win_stride ? a->win_stride : a->T_w;
    PKV_REQUIRE(par_stride >= a->T_c && win_stride >= a->T_w, PKV_ERR_INVALID, "row stride shorter than the row");
    PKV_REQUIRE((uint64_t)a->B * (uint64_t)par_stride < (1ull << 28), PKV_ERR_UNSUPPORTED,
                "batch x compressed tokens above 2^28");
    PKV_REQUIRE((uint64_t)(a->T_c / 64) * (uint64_t)a->B * (uint64_t)a->Hkv < (1ull << 27), PKV_ERR_UNSUPPORTED,
                "more than 2^27 blocks per stream");
    if (a->T_w > 0) {
        PKV_REQUIRE(a->k_win && a->v_win, PKV_ERR_INVALID, "null pointer argument");
        PKV_REQUIRE((reinterpret_cast<uintptr_t>(a->k_win) & 15u) == 0, PKV_ERR_INVALID,
                    "k_win must be 16-byte aligned");
    }
    const int Gq = a->Hq / a->Hkv;
    PKV_REQUIRE(Gq <= 8, PKV_ERR_UNSUPPORTED, "not supported: more than 8 query heads per KV head");
    const int G = Gq <= 2 ? Gq : Gq <= 4 ? 4 : 8;      // groups of 3 and of 5..7 run the kernels of 4 and 8 with idle head slots

    AttnParams p;
    p.k_stream = a->k_stream; p.k_info = a->k_info; p.v_stream = a->v_stream; p.v_info = a->v_info;
    p.k_scale = (const uint16_t *)a->k_scale; p.k_zero = (const uint16_t *)a->k_zero;
    p.v_scale = (const uint16_t *)a->v_scale; p.v_zero = (const uint16_t *)a->v_zero;
    p.q = (const uint16_t *)a->q;
    p.k_win = (const uint16_t *)a->k_win; p.v_win = (const uint16_t *)a->v_win;
    p.B = a->B; p.Hq = a->Hq; p.Hkv = a->Hkv; p.T_c = a->T_c; p.T_w = a->T_w;
    p.Gq = Gq;
    p.par_stride = par_stride; p.win_stride = win_stride;
    p.k_bits = a->k_bits; p.v_bits = a->v_bits; p.dtype = a->dtype; p.sm_scale = a->sm_scale;
    // the matrix-core kernels take the reference's widths and, in the asynchronous-copy kernel, the extension widths
    // 5 and 6 (the other side then 4, 5 or 6); any other combination with an extension width runs the plain kernel
    const bool narrow = a->T_c == 0 || (a->k_bits <= 4 && a->v_bits <= 4);
    const bool wide_fast = !narrow && a->k_bits >= 4 && a->v_bits >= 4 && a->k_bits <= 6 && a->v_bits <= 6 && a->variant == 0;
    const bool aligned16 = (narrow || wide_fast) &&
                           ((reinterpret_cast<uintptr_t>(a->k_stream) | reinterpret_cast<uintptr_t>(a->v_stream)) & 15u) == 0;
    const bool dma_path = a->T_c > 0 && a->variant == 0 && aligned16;
    const int n_tiles = a->T_c / kTile, pairs = a->B * a->Hkv;
    // The tail window goes in pieces of 64 tokens, one trip to memory each, to workgroups of their own -- in the
    // async-copy kernel's launch while they are at most a quarter of the workgroups that are resident at once (the tiles
    // keep the rest: 8 sequences x 4096 tokens), otherwise every split takes a share of the window behind its tiles (32
    // sequences: 69 us, the share being 40 tokens of a 160-token window); other paths give it a kernel of its own, with longer
    // pieces once there are more than four per CU (or more partials than the static array holds).
    int nsplit = 0, tps = 0, win_members = (a->T_w + kWinChunk - 1) / kWinChunk;
    if (n_tiles > 0) {
        // Members per (sequence, KV head): about PKV_SPLIT_TARGET workgroups in all for the reference's widths -- four resident on each of 256
        // CUs.  When the heads do not divide that number, rounding the members up leaves a few workgroups over that
        // only start once others have finished, each with a full share of tiles (12 sequences x 8 heads: 11 members,
        // 1056 workgroups, 115 us per step against 99 us with 10 members); so both roundings are priced as
        // generations x tiles per member and the cheaper one is taken, the finer cut on a tie.
        // (as many members as are resident at once; groups of eight query heads run three workgroups per CU: 156 against
        // 165 us with four.)  Width 5 runs three, but two when that is the cheaper cut: with three a tile takes 1.3 times as
        // long and a member's start half a tile more, and up to eight members merge by themselves (merge_head).  5-bit
        // steps, three -> two: 32 pairs x 64 tiles (22 members of three tiles, 16 of four) 19.95 -> 19.0 us, 64 x 64 (six, eight)
        // 30.8 -> 29.3; the other way round 24 x 86 with a window (three, five) 20.3 and 21.7, 256 x 64 83 and 94, 128 x 256 149 and 168.
        const int bits = a->k_bits > a->v_bits ? a->k_bits : a->v_bits;
        const int most = !dma_path && bits == 5 && G <= 4 ? 2 : PKV_DMA_RESIDENT(bits, G), least = bits == 5 && most == 3 ? 2 : most;
        if (dma_path && 4 * (int64_t)pairs * win_members > PKV_SPLIT_TARGET / 4 * most) win_members = 0;
        long best_cost = -1;
        for (int per_cu = most; per_cu >= least; per_cu--) {
            const int target = PKV_SPLIT_TARGET / 4 * per_cu - (dma_path ? pairs * win_members : 0);
            for (int up = 1; up >= 0; up--) {
                int want = up ? (target + pairs - 1) / pairs : target / pairs;
                if (want < 1) want = 1;
                if (want > n_tiles) want = n_tiles;
                const int t = (n_tiles + want - 1) / want, n = (n_tiles + t - 1) / t;
                const long each = per_cu > least ? 13l * t + 5 : 10l * t;
                const long cost = (((long)pairs * n + target - 1) / target) * each;
                if (best_cost < 0 || cost < best_cost) { best_cost = cost; tps = t; nsplit = n; }
            }
        }
    }
    const bool shared_window = dma_path && win_members == 0 && a->T_w > 0;      // every split writes a piece, empty or not
    if (a->T_w > 0 && !dma_path) {
        int64_t most = PKV_SPLIT_TARGET / pairs;
        const int64_t room = (int64_t)(kStaticPartBytes / ((size_t)a->B * a->Hq * kPartStride * sizeof(float))) - nsplit;
        if (room < most) most = room;
        if (most < win_members) win_members = most < 1 ? 1 : (int)most;
    }
    p.tiles_per_split = tps; p.nsplit = nsplit;
    p.win_piece = a->T_w > 0 ? (a->T_w + (shared_window ? nsplit : win_members) - 1) / (shared_window ? nsplit : win_members) : 0;
    p.win_members = dma_path ? win_members : 0;
    p.nparts = nsplit + (shared_window ? nsplit : a->T_w > 0 ? (a->T_w + p.win_piece - 1) / p.win_piece : 0);
    p.k_cap = a->T_c > 0 ? (uint32_t)k_block_bound(64, a->k_bits) : 0;
    p.v_cap = a->T_c > 0 ? (uint32_t)v_block_bound(64, a->v_bits) : 0;
    const uint32_t cap = p.k_cap > p.v_cap ? p.k_cap : p.v_cap;
    p.blk_stride = ((cap + 14u + 15u) & ~15u) + 32u;
    p.k_bytes = (uint32_t)a->k_bytes; p.v_bytes = (uint32_t)a->v_bytes;   // up to 14 bytes of phase in front, slack behind
    p.out = (uint16_t *)a->out;
    p.out_f32 = (a->flags & PKV_ATTN_OUT_F32) ? 1 : 0;
    p.direct_out = p.nparts == 1 && !p.out_f32;
    // The async-copy kernel balances the members of a head through two counters per head (with one member there is
    // nothing to balance).
    // Tiles by counter pay when a member has many tiles (the first five are its own anyway): short launches -- a few
    // tiles per member, the small-batch decode steps -- only get the counters' atomic round trips on top (batch 1,
    // 32768 tokens: 46 us against 19 us with fixed shares).  And only up to eight members per head: every member asks
    // its head's counter once per tile, and atomics on one address retire one after the other -- with 16 members a
    // step of batch 8 x 65536 tokens takes 172 us against 126 us with fixed shares, with 64 (batch 2 x 131072) 206
    // against 67 us; at 4 and 8 members the counters are worth 1-2 %.
    p.dynamic = PKV_DYNAMIC_TILES && dma_path && nsplit > 1 && nsplit <= 8 && tps >= 12 && 2 * a->B * a->Hkv <= kAttnCounters;
    p.batch_shift = 1;                     // a member asks for 1 / (2 nsplit) of what is left: ceil(log2(2 nsplit))
    while ((1 << p.batch_shift) < 2 * nsplit) p.batch_shift++;
    // few workgroups a head: the last of them merges (merge_head)
    p.merge = dma_path && p.nparts > 1 && nsplit + win_members <= kMergeArrivals && merge_pays(G, pairs, nsplit, tps) &&
              3 * (int64_t)a->B * a->Hkv <= kAttnCounters;
    p.counters = nullptr;
    // Partials and counters: the stream's own scratch, or the static array -- for pkv_attn_decode_noalloc, and for a
    // stream that is capturing a graph before it has scratch of its own.
    void *part = nullptr, *static_part = nullptr;
    const size_t part_bytes = (size_t)a->B * a->Hq * p.nparts * kPartStride * sizeof(float);
    int rc = static_scratch_ptr(&static_part);     // looked up on the first call on a device, while nothing is capturing
    if (rc) return rc;
    bool use_static = static_partials;
    if (!use_static) {
        rc = scratch_get(part_bytes, s, &part);
        if (rc == PKV_OK && (p.dynamic || p.merge)) {
            rc = attn_counters_get(s, &p.counters);
            if (rc == PKV_ERR_CAPTURING && !p.dynamic) { p.merge = 0; rc = PKV_OK; }     // a merge launch needs no counters
        }
        if (rc == PKV_ERR_CAPTURING && part_bytes <= kStaticPartBytes) use_static = true;
        else if (rc) return rc == PKV_ERR_CAPTURING ? PKV_ERR_HIP : rc;
    }
    if (use_static) {
        PKV_REQUIRE(part_bytes <= kStaticPartBytes, PKV_ERR_UNSUPPORTED,
                    "pkv_attn_decode_noalloc: %zu bytes of partials (batch %d x %d query heads x %d partials) exceed the "
                    "%zu bytes the static buffer has for them; use pkv_attn_decode", part_bytes, a->B, a->Hq, p.nparts,
                    kStaticPartBytes);
        part = static_part;
        p.counters = reinterpret_cast<uint32_t *>(static_cast<unsigned char *>(part) + kStaticPartBytes);
    }
    p.part = (float *)part;

    LaunchTimer tm(s, ms_out != nullptr);
    if ((rc = tm.begin())) return rc;
    const int variant = narrow || (wide_fast && aligned16) ? a->variant : 1;
    switch (G) {
        case 1: rc = launch_attn<1>(p, variant, aligned16, ref_rounding, (uint16_t *)a->out, s); break;
        case 2: rc = launch_attn<2>(p, variant, aligned16, ref_rounding, (uint16_t *)a->out, s); break;
        case 4: rc = launch_attn<4>(p, variant, aligned16, ref_rounding, (uint16_t *)a->out, s); break;
        default: rc = launch_attn<8>(p, variant, aligned16, ref_rounding, (uint16_t *)a->out, s); break;
    }
    if (rc) return rc;
    return tm.end(ms_out);
}
