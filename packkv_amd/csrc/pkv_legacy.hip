// The reference's four GPU ops, generalised to any head count and any hidden_dim that is a
// multiple of the block width, with fp32 accumulation (the reference accumulates in 16 bit,
// include/type_traits.h:26-58):
//   kq_mat_vec_mul  packkv_cuda_ext/src/kernels.cu:426-535   (K unpack fused with q . code)
//   wv_mat_vec_mul  packkv_cuda_ext/src/kernels.cu:632-765   (V unpack fused with w . code)
//   fused_kq        packkv_cuda_ext/src/fused_kernels.cu:13-76
//   fused_wv        packkv_cuda_ext/src/fused_kernels.cu:187-261
#include "pkv_block.hpp"
#include "pkv_runtime.hpp"

#include <initializer_list>

namespace pkv {

__device__ __forceinline__ float ld16(const uint16_t *p, size_t i, int dtype) {
    const uint32_t u = p[i];
    return dtype == PKV_F16 ? __half2float(__ushort_as_half((unsigned short)u)) : __uint_as_float(u << 16);
}

__device__ __forceinline__ uint16_t st16(float x, int dtype) {
    if (dtype == PKV_F16) return __half_as_ushort(__float2half_rn(x));
    uint32_t u = __float_as_uint(x);
    if ((u & 0x7FFFFFFFu) > 0x7F800000u) return (uint16_t)((u >> 16) | 0x40u);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

// A wavefront decodes a block by itself: the block's bytes go to an LDS slot of its own, its two halves parse a unit each
// (unit_fields) and the codes meet q or w in registers as they come out -- no code tile, no barrier.  What bounds both
// kernels is instruction issue (about 300 vector instructions per wavefront and pair of units: windows, shifts and masks
// 1.75 per code pair, minima 0.5, products 1 per code) behind the chain block_info -> block bytes -> parse; with a workgroup
// of two wavefronts per block the chain had a barrier between its links, the tile was written and read back, and a code
// cost a conversion.
// f.x .. f.w times the four codes c01 | c23 as unit_fields hands them out, i.e. codes times 2^-24 read from halves: products
// exact, fp32 sums.  The factors come 2^24 times as large, so that the products are those of the codes: with the sum scaled
// back instead, products of bf16 factors below 2^-102 fell among the subnormals and lost bits.  Factors of 2^100 and more
// could overflow: where a row holds one (or a NaN), a code is scaled instead, one more instruction each (BIG).
constexpr float kFieldUnit = 16777216.f, kFieldMost = 0x1p100f;      // 2^24
typedef _Float16 half_pair __attribute__((ext_vector_type(2)));
template <bool BIG>
__device__ __forceinline__ float field(_Float16 c) { return BIG ? (float)c * kFieldUnit : (float)c; }
template <bool BIG>
__device__ __forceinline__ float dot4(uint32_t c01, uint32_t c23, const float4 f) {
    const half_pair a = __builtin_bit_cast(half_pair, c01), b = __builtin_bit_cast(half_pair, c23);
    float s = field<BIG>(a[1]) * f.y;
    s = fmaf(field<BIG>(a[0]), f.x, s);
    s = fmaf(field<BIG>(b[0]), f.z, s);
    return fmaf(field<BIG>(b[1]), f.w, s);
}
template <bool BIG>
__device__ __forceinline__ float dot4(uint32_t c01, uint32_t c23, const float4 f, float acc) {
    const half_pair a = __builtin_bit_cast(half_pair, c01), b = __builtin_bit_cast(half_pair, c23);
    acc = fmaf(field<BIG>(a[0]), f.x, acc);
    acc = fmaf(field<BIG>(a[1]), f.y, acc);
    acc = fmaf(field<BIG>(b[0]), f.z, acc);
    return fmaf(field<BIG>(b[1]), f.w, acc);
}
// True (uniform) when one of the wavefront's factors, `N` a lane, is too large for 2^24 times itself, or NaN.
template <int N>
__device__ __forceinline__ bool factors_big(const float (&f)[N]) {
    bool big = false;
#pragma unroll
    for (int i = 0; i < N; i++) big = big || !(fabsf(f[i]) < kFieldMost);
    return __any(big);
}

// K . q: wavefront per K block (`wpw` of them to a workgroup, `slot` bytes of LDS each), a half per round, lane = four
// channels.  A token's 32 sums of four channels are turned through LDS so that a lane adds sixteen of them, one after the
// other from the lowest channel on: kq comes out of sums that nearly cancel (q . code against the zero points), so a last
// bit here that changed with the order of the sum would show there.
// 65536 tokens x 8 heads at 4 bits: 15.4 us, 17.4 with a workgroup and a code tile per block (medians of 300 launches in
// kernel traces, in the reference's sequence of four ops with two inputs in turn; these and those below).
constexpr int kKqTok = 20, kKqRow = 16 * kKqTok + 16;      // floats from token to token and from row of lanes to row: no bank conflicts
template <int W>
__global__ void __launch_bounds__(256) kq_kernel(const uint8_t *__restrict__ stream, uint64_t stream_bytes, const uint32_t *__restrict__ info,
                                                 const uint16_t *__restrict__ q, uint16_t *__restrict__ kq_out, int ctx_len,
                                                 int hidden_dim, int ctx_blk, int nunits, uint32_t blk_cap, uint32_t slot,
                                                 uint32_t nblocks, int dtype, int q_interleaved, LaunchStamp started) {
    launch_started(started);
    extern __shared__ __align__(16) uint8_t lds[];
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t b = blockIdx.x * (blockDim.x >> 6) + wave;
    if (b >= nblocks) return;
    uint8_t *blk = lds + wave * slot;
    const int lane = threadIdx.x & 63, t = lane & 31, half = lane >> 5, l16 = lane & 15;
    float *turn = reinterpret_cast<float *>(blk + slot - 4 * 4 * kKqRow) + (lane >> 4) * kKqRow;
    const uint32_t n_hid = (uint32_t)hidden_dim / kHeadDim, cb = b / n_hid, hb = b % n_hid;
    uint32_t off, size;
    block_span(info, b, blk_cap, stream_bytes, off, size);
    const uint32_t phase = stage_to_lds(stream + off, size, blk, lane, 64);
    float qf[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {      // (interleaved as in evaluation/evaluation.py:465-468)
        const int src = !q_interleaved ? 4 * t + i : i < 2 ? 2 * t + i : 64 + 2 * t + (i - 2);
        qf[i] = ld16(q, (size_t)hb * kHeadDim + src, dtype);
    }
    const bool big = factors_big(qf);
    const float unit_q = big ? 1.f : kFieldUnit;
    const float4 q4 = make_float4(qf[0] * unit_q, qf[1] * unit_q, qf[2] * unit_q, qf[3] * unit_q);
    wave_lds_order();
    const uint16_t *cum = reinterpret_cast<const uint16_t *>(blk + phase);      // (phase is even)
#pragma unroll 1
    for (int u0 = 0; u0 < nunits; u0 += 2) {
        const int unit = min(u0 + half, nunits - 1);      // (an odd last round: both halves decode it, the first one writes)
        const uint32_t start = phase + 2u * (uint32_t)nunits + (unit ? (uint32_t)cum[unit - 1] : 0u);
        if (big) unit_fields<W>(blk, start, t, [&](int k, uint32_t c01, uint32_t c23) { turn[kKqTok * k + l16] = dot4<true>(c01, c23, q4); });
        else unit_fields<W>(blk, start, t, [&](int k, uint32_t c01, uint32_t c23) { turn[kKqTok * k + l16] = dot4<false>(c01, c23, q4); });
        wave_lds_order();
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float4 v = *reinterpret_cast<const float4 *>(turn + kKqTok * l16 + 4 * i);
            s = ((s + v.x) + v.y) + v.z;
            s += v.w;
        }
        wave_lds_order();
        s += __shfl_xor(s, 16, 64);
        if ((lane & 16) == 0 && u0 + half < nunits) kq_out[(size_t)hb * ctx_len + (size_t)cb * ctx_blk + 16 * unit + l16] = st16(s, dtype);
    }
}

// w . V: wavefront per V block, four context blocks of one column of blocks to a workgroup; a half per 64-token segment,
// lane = channel, so a channel's sum over the tokens stays in its lane.  The weights lie in LDS as floats, [segment][token of
// the pack][round], one 16-byte broadcast per four codes.  The halves and then the workgroup's blocks are added before the
// one atomic per channel.
// 65536 tokens x 8 heads at 3 bits: 14.8 us, 21.2 with a code tile per block and an atomic per channel and block.
constexpr int kWvWaves = 4;
template <int W>
__global__ void __launch_bounds__(64 * kWvWaves) wv_kernel(const uint8_t *__restrict__ stream, uint64_t stream_bytes, const uint32_t *__restrict__ info,
                                                           const uint16_t *__restrict__ w, float *__restrict__ wv_out, int ctx_len,
                                                           int hidden_dim, int hid_blk, uint32_t blk_cap, uint32_t slot, int dtype,
                                                           LaunchStamp started) {
    launch_started(started);
    extern __shared__ __align__(16) uint8_t lds[];
    __shared__ __align__(16) float ws[kWvWaves][128];
    __shared__ float part[kWvWaves][kHeadDim];
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63, t = lane & 31, seg = lane >> 5;
    const uint32_t n_hid = (uint32_t)(hidden_dim / hid_blk), n_ctx = (uint32_t)(ctx_len / 128);
    const uint32_t hb = blockIdx.x % n_hid, cb = blockIdx.x / n_hid * kWvWaves + wave;
    const int npair = hid_blk / kLanes;                    // unit = 2 * pair + segment
    if (cb < n_ctx) {
        uint8_t *blk = lds + wave * slot;
        const uint32_t head = (hb * (uint32_t)hid_blk) / kHeadDim;
        uint32_t off, size;
        block_span(info, cb * n_hid + hb, blk_cap, stream_bytes, off, size);
        const uint32_t phase = stage_to_lds(stream + off, size, blk, lane, 64);
        float wf[2];
#pragma unroll
        for (int i = 0; i < 2; i++) wf[i] = ld16(w, (size_t)head * ctx_len + (size_t)cb * 128 + lane + 64 * i, dtype);
        const bool big = factors_big(wf);
#pragma unroll
        for (int i = 0; i < 2; i++)                        // segment i, round lane / 16, token lane % 16 of the pack
            ws[wave][64 * i + 4 * (lane & 15) + (lane >> 4)] = wf[i] * (big ? 1.f : kFieldUnit);
        wave_lds_order();
        const uint16_t *cum = reinterpret_cast<const uint16_t *>(blk + phase);  // (phase is even)
#pragma unroll 1
        for (int p = 0; p < npair; p++) {
            uint32_t at = 64u * (uint32_t)seg;
            asm volatile("" : "+v"(at));                   // (the weights are read where they are used: kept in registers they would take 64)
            const float4 *w4 = reinterpret_cast<const float4 *>(ws[wave] + at);
            const int unit = 2 * p + seg;
            const uint32_t start = phase + 4u * (uint32_t)npair + (unit ? (uint32_t)cum[unit - 1] : 0u);
            float acc[4] = {0.f, 0.f, 0.f, 0.f};
            if (big) unit_fields<W>(blk, start, t, [&](int k, uint32_t c01, uint32_t c23) { acc[k & 3] = dot4<true>(c01, c23, w4[k], acc[k & 3]); });
            else unit_fields<W>(blk, start, t, [&](int k, uint32_t c01, uint32_t c23) { acc[k & 3] = dot4<false>(c01, c23, w4[k], acc[k & 3]); });
            const float s = (acc[0] + acc[1]) + (acc[2] + acc[3]);
            const float both = s + __shfl_xor(s, 32, 64);
            if (seg == 0) part[wave][kLanes * p + t] = both;
        }
    } else {
        for (int c = lane; c < hid_blk; c += 64) part[wave][c] = 0.f;
    }
    __syncthreads();
    if ((int)threadIdx.x < hid_blk) {
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < kWvWaves; i++) s += part[i][threadIdx.x];
        atomicAdd(wv_out + (size_t)hb * hid_blk + threadIdx.x, s);
    }
}

__device__ __forceinline__ float wave_sum_f32(float x) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) x += __shfl_xor(x, d, 64);
    return x;
}

// Four adjacent 16-bit values from `i` on, as they lie: one 8-byte load where `vec` says that every row starts on an 8-byte
// boundary and ends on a multiple of four (uniform), else one by one, zero past the end.
struct Raw4 {
    uint16_t u[4];
};
__device__ __forceinline__ Raw4 ld4(const uint16_t *p, size_t row, int i, int n, bool vec) {
    Raw4 r = {{0, 0, 0, 0}};
    if (vec) {
        if (i < n) *reinterpret_cast<uint2 *>(r.u) = *reinterpret_cast<const uint2 *>(p + row + i);
    } else {
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (i + k < n) r.u[k] = p[row + i + k];
    }
    return r;
}
static bool rows_of_fours(int n, std::initializer_list<const void *> ptrs) {
    uintptr_t a = 0;
    for (const void *p : ptrs) a |= reinterpret_cast<uintptr_t>(p);
    return n % 4 == 0 && (a & 7u) == 0;
}

// grid = (ceil(N / 1024), M), 256 threads: every workgroup forms the row's sum of q itself (K values) and finishes 1024
// columns, four per thread, which are on their way meanwhile.
__global__ void __launch_bounds__(256) fused_kq_kernel(uint16_t *__restrict__ out, const uint16_t *__restrict__ q,
                                                       const uint16_t *__restrict__ zero, const uint16_t *__restrict__ scale,
                                                       const uint16_t *__restrict__ t, int K, int N, int dtype, bool vec, LaunchStamp started) {
    launch_started(started);
    __shared__ float red[4];
    const int m = blockIdx.y;
    const int n = blockIdx.x * 1024 + 4 * (int)threadIdx.x;
    const size_t row = (size_t)m * N;
    const Raw4 z = ld4(zero, 0, n, N, vec), tt = ld4(t, row, n, N, vec), sc = ld4(scale, 0, n, N, vec);
    float s = 0.f;
    for (int d = threadIdx.x; d < K; d += 256) s += ld16(q, (size_t)m * K + d, dtype);
    s = wave_sum_f32(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    const float sm = (red[0] + red[1]) + (red[2] + red[3]);
    Raw4 o;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float u = sm * ld16(z.u, i, dtype) + ld16(tt.u, i, dtype);
        o.u[i] = st16(u * ld16(sc.u, i, dtype), dtype);
    }
    if (vec) {
        if (n < N) *reinterpret_cast<uint2 *>(out + row + n) = *reinterpret_cast<const uint2 *>(o.u);
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (n + i < N) out[row + n + i] = o.u[i];
    }
}

// Row sums of w * zero * scale in two steps: grid (ceil(N / 1024), M) partial sums, then one workgroup per row
// adds the partials and finishes the D outputs.  (65536 columns x 8 rows: 3.4 us for the partial sums; 8.0 with 4096 columns
// a workgroup, read one value at a time.)
constexpr int kWvPart = 1024;
__global__ void __launch_bounds__(256) fused_wv_partial_kernel(const uint16_t *__restrict__ w, const uint16_t *__restrict__ zero,
                                                               const uint16_t *__restrict__ scale, float *__restrict__ part,
                                                               int N, int dtype, bool vec, LaunchStamp started) {
    launch_started(started);
    __shared__ float red[4];
    const int m = blockIdx.y, n = blockIdx.x * kWvPart + 4 * (int)threadIdx.x;
    const Raw4 a = ld4(w, (size_t)m * N, n, N, vec), z = ld4(zero, 0, n, N, vec), sc = ld4(scale, 0, n, N, vec);
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (n + i < N) s += ld16(a.u, i, dtype) * ld16(z.u, i, dtype) * ld16(sc.u, i, dtype);
    s = wave_sum_f32(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) part[(size_t)m * gridDim.x + blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

__global__ void __launch_bounds__(256) fused_wv_kernel(uint16_t *__restrict__ out, const float *__restrict__ part, int nparts,
                                                       const uint16_t *__restrict__ term1, int D, int dtype) {
    __shared__ float red[4];
    const int m = blockIdx.x;
    float s = 0.f;
    for (int i = threadIdx.x; i < nparts; i += 256) s += part[(size_t)m * nparts + i];
    s = wave_sum_f32(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    const float c = (red[0] + red[1]) + (red[2] + red[3]);
    for (int d = threadIdx.x; d < D; d += 256)
        out[(size_t)m * D + d] = st16(c + ld16(term1, (size_t)m * D + d, dtype), dtype);
}

static int check_dtype(int dtype) {
    PKV_REQUIRE(dtype == PKV_F16 || dtype == PKV_BF16, PKV_ERR_UNSUPPORTED, "Unsupported data type");
    return PKV_OK;
}

}  // namespace pkv

extern "C" {

int pkv_kq_mat_vec_mul(const uint8_t *stream, uint64_t stream_bytes, const uint32_t *block_info, const void *q, void *kq_out,
                       int ctx_len, int hidden_dim, int ctx_blk, int hid_blk, int bits, int dtype,
                       int q_interleaved, float *ms_out, pkv_stream_t s_) {
    using namespace pkv;
    hipStream_t s = (hipStream_t)s_;
    int rc = check_dtype(dtype);
    if (rc) return rc;
    PKV_REQUIRE(stream && block_info && q && kq_out, PKV_ERR_INVALID, "null pointer argument");
    PKV_REQUIRE(stream_bytes > 0 && stream_bytes < (1ull << 32), PKV_ERR_INVALID, "stream size must be in 1 .. 4 GiB - 1");
    PKV_REQUIRE(bits >= 2 && bits <= 4 && hid_blk == kHeadDim && ctx_blk > 0 && ctx_blk % kPackTok == 0 &&
                    ctx_blk <= 256 && ctx_len > 0 && ctx_len % ctx_blk == 0 && hidden_dim > 0 &&
                    hidden_dim % hid_blk == 0,
                PKV_ERR_UNSUPPORTED, "no such case");
    const int nunits = ctx_blk / kPackTok;
    const uint32_t cap = (uint32_t)k_block_bound(ctx_blk, bits);
    const int nblocks = (ctx_len / ctx_blk) * (hidden_dim / hid_blk);
    const uint32_t slot = ((cap + 15u) & ~15u) + 32u + 4u * 4u * kKqRow;      // at most 23.7 KB: 256 tokens at 4 bits
    const uint32_t wpw = slot * 4u <= 65536u ? 4u : 65536u / slot;
    StampedLaunch tm(s, ms_out != nullptr);
    if ((rc = tm.begin())) return rc;
    auto kern = bits == 2 ? kq_kernel<2> : bits == 3 ? kq_kernel<3> : kq_kernel<4>;
    kern<<<((uint32_t)nblocks + wpw - 1u) / wpw, 64u * wpw, wpw * slot, s>>>(
        stream, stream_bytes, block_info, (const uint16_t *)q, (uint16_t *)kq_out, ctx_len, hidden_dim, ctx_blk, nunits, cap,
        slot, (uint32_t)nblocks, dtype, q_interleaved, tm.stamp());
    PKV_HIP_CHECK(hipGetLastError());
    return tm.end(ms_out);
}

int pkv_wv_mat_vec_mul(const uint8_t *stream, uint64_t stream_bytes, const uint32_t *block_info, const void *w, float *wv_out,
                       int ctx_len, int hidden_dim, int ctx_blk, int hid_blk, int bits, int dtype,
                       float *ms_out, pkv_stream_t s_) {
    using namespace pkv;
    hipStream_t s = (hipStream_t)s_;
    int rc = check_dtype(dtype);
    if (rc) return rc;
    PKV_REQUIRE(stream && block_info && w && wv_out, PKV_ERR_INVALID, "null pointer argument");
    PKV_REQUIRE(stream_bytes > 0 && stream_bytes < (1ull << 32), PKV_ERR_INVALID, "stream size must be in 1 .. 4 GiB - 1");
    PKV_REQUIRE(bits >= 2 && bits <= 4 && ctx_blk == 128 && (hid_blk == 32 || hid_blk == 64 || hid_blk == 128) &&
                    ctx_len > 0 && ctx_len % ctx_blk == 0 && hidden_dim > 0 && hidden_dim % kHeadDim == 0,
                PKV_ERR_UNSUPPORTED, "no such case");
    const uint32_t cap = (uint32_t)v_block_bound(hid_blk, bits);
    const uint32_t slot = ((cap + 15u) & ~15u) + 32u;           // at most 9.2 KB: 128 channels at 4 bits
    const uint32_t rows = (uint32_t)(ctx_len / ctx_blk + kWvWaves - 1) / kWvWaves;
    StampedLaunch tm(s, ms_out != nullptr);
    if ((rc = tm.begin())) return rc;
    auto kern = bits == 2 ? wv_kernel<2> : bits == 3 ? wv_kernel<3> : wv_kernel<4>;
    kern<<<rows * (uint32_t)(hidden_dim / hid_blk), 64 * kWvWaves, kWvWaves * slot, s>>>(
        stream, stream_bytes, block_info, (const uint16_t *)w, wv_out, ctx_len, hidden_dim, hid_blk, cap, slot, dtype, tm.stamp());
    PKV_HIP_CHECK(hipGetLastError());
    return tm.end(ms_out);
}

int pkv_fused_kq(void *our_kq, const void *q, const void *k_zero, const void *k_scale, const void *t, int M,
                 int K, int N, int dtype, float *ms_out, pkv_stream_t s_) {
    using namespace pkv;
    hipStream_t s = (hipStream_t)s_;
    int rc = check_dtype(dtype);
    if (rc) return rc;
    PKV_REQUIRE(our_kq && q && k_zero && k_scale && t, PKV_ERR_INVALID, "null pointer argument");
    PKV_REQUIRE(M > 0 && K > 0 && N > 0, PKV_ERR_INVALID, "sizes must be positive");
    PKV_REQUIRE(M <= 65535, PKV_ERR_UNSUPPORTED, "more than 65535 rows");
    StampedLaunch tm(s, ms_out != nullptr);
    if ((rc = tm.begin())) return rc;
    fused_kq_kernel<<<dim3((unsigned)((N + 1023) / 1024), (unsigned)M), 256, 0, s>>>(
        (uint16_t *)our_kq, (const uint16_t *)q, (const uint16_t *)k_zero, (const uint16_t *)k_scale,
        (const uint16_t *)t, K, N, dtype, rows_of_fours(N, {our_kq, k_zero, k_scale, t}), tm.stamp());
    PKV_HIP_CHECK(hipGetLastError());
    return tm.end(ms_out);
}

int pkv_fused_wv(void *our_wv, const void *w, const void *v_zero, const void *v_scale, const void *term1,
                 int M, int N, int D, int dtype, float *ms_out, pkv_stream_t s_) {
    using namespace pkv;
    hipStream_t s = (hipStream_t)s_;
    int rc = check_dtype(dtype);
    if (rc) return rc;
    PKV_REQUIRE(our_wv && w && v_zero && v_scale && term1, PKV_ERR_INVALID, "null pointer argument");
    PKV_REQUIRE(M > 0 && N > 0 && D > 0, PKV_ERR_INVALID, "sizes must be positive");
    PKV_REQUIRE(M <= 65535, PKV_ERR_UNSUPPORTED, "more than 65535 rows");
    const int nparts = (N + kWvPart - 1) / kWvPart;
    void *scratch = nullptr;
    if ((rc = scratch_get((size_t)M * nparts * sizeof(float), s, &scratch))) return rc;
    StampedLaunch tm(s, ms_out != nullptr);
    if ((rc = tm.begin())) return rc;
    fused_wv_partial_kernel<<<dim3((unsigned)nparts, (unsigned)M), 256, 0, s>>>(
        (const uint16_t *)w, (const uint16_t *)v_zero, (const uint16_t *)v_scale, (float *)scratch, N, dtype,
        rows_of_fours(N, {w, v_zero, v_scale}), tm.stamp());
    fused_wv_kernel<<<M, 256, 0, s>>>((uint16_t *)our_wv, (const float *)scratch, nparts, (const uint16_t *)term1,
                                      D, dtype);
    PKV_HIP_CHECK(hipGetLastError());
    return tm.end(ms_out);
}

}  // extern "C"
