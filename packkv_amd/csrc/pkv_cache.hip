// The decode step's write into the cache's 16-bit window: rotary embedding of the new K rows and the copy of the
// new K and V rows behind the rows already there, in one launch.
//
// Reference: the cache applies the rotary embedding to the incoming keys itself
// (models/cache/packkv_quant.py:59-60, `apply_rotary_pos_emb_single`, utils/compute.py:35-43:
// (t * cos) + (rotate_half(t) * sin) with rotate_half(t) = cat(-t[64:], t[:64])) and appends keys and values to its
// buffer with torch.cat (packkv_quant.py:62-83).  The three elementwise operations run in the 16-bit storage type --
// each computes in fp32 and rounds its result -- so the kernel rounds both products and the sum, and its rows are
// bit for bit what the reference's chain of kernels produces.
#include "pkv_common.hpp"
#include "pkv_runtime.hpp"

// Every product and sum below is rounded on its own, as separate kernels would round them: no fused multiply-add
// may be formed across them (the compiler narrows the fp32 arithmetic on 16-bit values to 16-bit instructions,
// which is exact, and would then be free to contract them).
#pragma clang fp contract(off)

namespace pkv {

template <int DT> __device__ __forceinline__ float ld16(const uint16_t *p) {
    return DT == PKV_F16 ? __half2float(__ushort_as_half(*p)) : __uint_as_float((uint32_t)*p << 16);
}
template <int DT> __device__ __forceinline__ uint16_t rn16(float x) {
    if (DT == PKV_F16) return __half_as_ushort(__float2half_rn(x));
    uint32_t u = __float_as_uint(x);
    if ((u & 0x7FFFFFFFu) > 0x7F800000u) return (uint16_t)((u >> 16) | 0x40u);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
template <int DT> __device__ __forceinline__ float rt(float x) {
    const uint16_t b = rn16<DT>(x);
    return ld16<DT>(&b);
}

// grid (n, H, B), 64 threads: thread d owns channels d and d + 64 of one (sequence, head, new token)
template <int DT>
__global__ void __launch_bounds__(64) window_append_kernel(const uint16_t *__restrict__ k_new, const uint16_t *__restrict__ v_new,
                                                           const uint16_t *__restrict__ cos, const uint16_t *__restrict__ sin,
                                                           long sb, long sh, long st, long rot_sb, uint16_t *__restrict__ k_win,
                                                           uint16_t *__restrict__ v_win, int H, int n, int win_pos, int win_stride) {
    const int tok = blockIdx.x, h = blockIdx.y, b = blockIdx.z, d = threadIdx.x;
    const size_t src = (size_t)b * sb + (size_t)h * sh + (size_t)tok * st;
    const size_t dst = (((size_t)b * H + h) * win_stride + win_pos + tok) * kHeadDim;
    v_win[dst + d] = v_new[src + d];
    v_win[dst + d + 64] = v_new[src + d + 64];
    if (cos == nullptr) {
        k_win[dst + d] = k_new[src + d];
        k_win[dst + d + 64] = k_new[src + d + 64];
        return;
    }
    const size_t rot = (size_t)b * rot_sb + (size_t)tok * kHeadDim;
    if (DT == PKV_F16) {     // correctly rounded 16-bit multiplies and adds are exactly the reference's fp32-then-round ops
        const _Float16 *kp = reinterpret_cast<const _Float16 *>(k_new) + src, *cp = reinterpret_cast<const _Float16 *>(cos) + rot,
                       *sp = reinterpret_cast<const _Float16 *>(sin) + rot;
        _Float16 *op = reinterpret_cast<_Float16 *>(k_win) + dst;
        const _Float16 k0 = kp[d], k1 = kp[d + 64];
        const _Float16 a0 = k0 * cp[d], b0 = -k1 * sp[d], a1 = k1 * cp[d + 64], b1 = k0 * sp[d + 64];
        op[d] = a0 + b0;
        op[d + 64] = a1 + b1;
        return;
    }
    const float k0 = ld16<DT>(k_new + src + d), k1 = ld16<DT>(k_new + src + d + 64);
    const float c0 = ld16<DT>(cos + rot + d), c1 = ld16<DT>(cos + rot + d + 64);
    const float s0 = ld16<DT>(sin + rot + d), s1 = ld16<DT>(sin + rot + d + 64);
    k_win[dst + d] = rn16<DT>(rt<DT>(k0 * c0) + rt<DT>(-k1 * s0));
    k_win[dst + d + 64] = rn16<DT>(rt<DT>(k1 * c1) + rt<DT>(k0 * s1));
}

// ---- a cut: tokens leave the window for the streams --------------------------------------------------------------
// The tokens at hand are, in order, the originals of a pending 64-token cut, the window's rows behind it and the new
// tokens (keys with their rotary embedding).  The first `stage` of them go to the encoder, the next `pend_out` are the
// new pending cut, the rest are the new window rows behind it; a window is written into a buffer of its own, so nothing
// is read after it was overwritten.  Replaces the reference's chain of cat / slice / rotary elementwise kernels
// (models/cache/packkv_quant.py:59-83), which went over a prompt seven times.
// Tokens [first, first + 32 gridDim.x), heads [heads * blockIdx.y, + heads), one sequence per blockIdx.z; eight threads
// per token, each with channels 8 c .. 8 c + 7 of both halves of a row, so that a rotary pair meets in one thread and
// every access is 16 bytes; cos and sin are read once for all heads of the workgroup.  Bound by the memory system: the
// first update of 32 sequences x 8 heads x 8192 tokens (bf16, rotary; 537 MB a side) takes 669 us with both encodes,
// 3046 us with the chain of torch kernels; with heads beside each other in a token's row 662 against 3663 us.
struct CutParams {
    const uint16_t *k_new, *v_new, *cos, *sin, *k_pend, *v_pend, *k_win, *v_win;
    uint16_t *k_stage, *v_stage, *k_pend_out, *v_pend_out, *k_win_out, *v_win_out;
    int64_t sb, sh, st, rot_sb;
    int H, pend, held, total, stage, pend_out, win_stride, first, heads;
};

template <int DT>
__device__ __forceinline__ void rotate8(uint4 &lo, uint4 &hi, const uint4 c0, const uint4 c1, const uint4 s0, const uint4 s1) {
    if (DT == PKV_F16) {
        typedef _Float16 h8 __attribute__((ext_vector_type(8)));
        const h8 k0 = __builtin_bit_cast(h8, lo), k1 = __builtin_bit_cast(h8, hi);
        const h8 a0 = k0 * __builtin_bit_cast(h8, c0), b0 = -k1 * __builtin_bit_cast(h8, s0);
        const h8 a1 = k1 * __builtin_bit_cast(h8, c1), b1 = k0 * __builtin_bit_cast(h8, s1);
        lo = __builtin_bit_cast(uint4, (h8)(a0 + b0));
        hi = __builtin_bit_cast(uint4, (h8)(a1 + b1));
        return;
    }
    typedef unsigned short u8v __attribute__((ext_vector_type(8)));
    typedef float f8 __attribute__((ext_vector_type(8)));
    typedef __bf16 b8 __attribute__((ext_vector_type(8)));
    auto up = [](uint4 v) -> f8 { return __builtin_convertvector(__builtin_bit_cast(b8, v), f8); };
    auto rn = [](f8 v) -> f8 { return __builtin_convertvector(__builtin_convertvector(v, b8), f8); };
    const f8 k0 = up(lo), k1 = up(hi);
    const f8 r0 = rn(k0 * up(c0)) + rn(-k1 * up(s0)), r1 = rn(k1 * up(c1)) + rn(k0 * up(s1));
    lo = __builtin_bit_cast(uint4, __builtin_convertvector(r0, b8));
    hi = __builtin_bit_cast(uint4, __builtin_convertvector(r1, b8));
}

template <int DT>
__global__ void __launch_bounds__(256) cut_kernel(const CutParams p) {
    const int i = p.first + (int)blockIdx.x * 32 + ((int)threadIdx.x >> 3), c = threadIdx.x & 7, b = blockIdx.z;
    if (i >= p.total) return;
    const bool fresh = i >= p.held;                          // a new token; before it the window, before that the pending cut
    const bool rotary = fresh && p.cos != nullptr;
    uint4 c0, c1, s0, s1;
    if (rotary) {
        const size_t at = (size_t)b * p.rot_sb + (size_t)(i - p.held) * kHeadDim;
        const uint4 *cp = reinterpret_cast<const uint4 *>(p.cos + at), *sp = reinterpret_cast<const uint4 *>(p.sin + at);
        c0 = cp[c]; c1 = cp[c + 8]; s0 = sp[c]; s1 = sp[c + 8];
    }
    const int h1 = min(p.H, ((int)blockIdx.y + 1) * p.heads);
#pragma unroll 2
    for (int h = (int)blockIdx.y * p.heads; h < h1; h++) {
        const size_t bh = (size_t)b * p.H + h;
        const uint16_t *ks, *vs;
        if (fresh) {
            const int64_t at = b * p.sb + h * p.sh + (int64_t)(i - p.held) * p.st;
            ks = p.k_new + at; vs = p.v_new + at;
        } else if (i < p.pend) {
            ks = p.k_pend + (bh * 64 + i) * kHeadDim; vs = p.v_pend + (bh * 64 + i) * kHeadDim;
        } else {
            ks = p.k_win + (bh * p.win_stride + i) * kHeadDim; vs = p.v_win + (bh * p.win_stride + i) * kHeadDim;
        }
        uint16_t *kd, *vd;
        if (i < p.stage) {
            kd = p.k_stage ? p.k_stage + (bh * p.stage + i) * kHeadDim : nullptr;
            vd = p.v_stage ? p.v_stage + (bh * p.stage + i) * kHeadDim : nullptr;
        } else if (i < p.stage + p.pend_out) {
            kd = p.k_pend_out + (bh * 64 + (i - p.stage)) * kHeadDim; vd = p.v_pend_out + (bh * 64 + (i - p.stage)) * kHeadDim;
        } else {
            kd = p.k_win_out + (bh * p.win_stride + (i - p.stage)) * kHeadDim; vd = p.v_win_out + (bh * p.win_stride + (i - p.stage)) * kHeadDim;
        }
        if (kd) {
            uint4 lo = reinterpret_cast<const uint4 *>(ks)[c], hi = reinterpret_cast<const uint4 *>(ks)[c + 8];
            if (rotary) rotate8<DT>(lo, hi, c0, c1, s0, s1);
            reinterpret_cast<uint4 *>(kd)[c] = lo;
            reinterpret_cast<uint4 *>(kd)[c + 8] = hi;
        }
        if (vd) {
            const uint4 lo = reinterpret_cast<const uint4 *>(vs)[c], hi = reinterpret_cast<const uint4 *>(vs)[c + 8];
            reinterpret_cast<uint4 *>(vd)[c] = lo;
            reinterpret_cast<uint4 *>(vd)[c + 8] = hi;
        }
    }
}

}  // namespace pkv

extern "C" {

int pkv_window_cut(const pkv_cut_args *a, pkv_stream_t s_) {
    using namespace pkv;
    hipStream_t s = (hipStream_t)s_;
    PKV_REQUIRE(a && a->k_new && a->v_new && a->k_win_out && a->v_win_out, PKV_ERR_INVALID, "null pointer argument");
    PKV_REQUIRE((a->cos == nullptr) == (a->sin == nullptr), PKV_ERR_INVALID, "cos and sin go together");
    PKV_REQUIRE(a->dtype == PKV_F16 || a->dtype == PKV_BF16, PKV_ERR_UNSUPPORTED, "Unsupported data type");
    PKV_REQUIRE(a->B > 0 && a->H > 0 && a->n > 0 && a->B <= 65535 && a->H <= 65535, PKV_ERR_INVALID, "sizes must be positive (batch, heads <= 65535)");
    PKV_REQUIRE((a->pend == 0 || a->pend == 64) && (a->pend_out == 0 || a->pend_out == 64) && a->buf >= 0 && a->stage >= 0, PKV_ERR_INVALID,
                "a pending cut is 64 tokens");
    const int64_t total = (int64_t)a->pend + a->buf + a->n;
    PKV_REQUIRE(total < (1ll << 31) && (int64_t)a->stage + a->pend_out <= total && total - a->stage <= a->win_stride && a->pend + a->buf <= a->win_stride,
                PKV_ERR_INVALID, "the rows do not fit the window (%d rows)", a->win_stride);
    PKV_REQUIRE(a->pend == 0 || (a->k_pend && a->v_pend), PKV_ERR_INVALID, "null pointer argument");
    PKV_REQUIRE(a->pend_out == 0 || (a->k_pend_out && a->v_pend_out && a->k_pend_out != a->k_pend && a->v_pend_out != a->v_pend && a->k_rel > 0.f && a->v_rel > 0.f),
                PKV_ERR_INVALID, "a pending cut needs buffers of its own and positive relative scales");
    PKV_REQUIRE(a->pend + a->buf == 0 || (a->k_win && a->v_win && a->k_win != a->k_win_out && a->v_win != a->v_win_out), PKV_ERR_INVALID,
                "the new window is written into buffers of its own");
    // what is encoded in place must be new tokens (their rotary embedding is then the encoder's work)
    PKV_REQUIRE(a->stage == 0 || ((a->k_stage && a->v_stage) || a->pend + a->buf == 0), PKV_ERR_INVALID,
                "staged tokens need a buffer unless they are new");
    PKV_REQUIRE(a->stride_b >= 0 && a->stride_h >= 0 && a->stride_t >= 0 && a->rot_stride_b >= 0 &&
                    (a->stride_b | a->stride_h | a->stride_t | a->rot_stride_b) % 8 == 0, PKV_ERR_INVALID, "strides must be multiples of 8");
    const void *ptrs[] = {a->k_new, a->v_new, a->cos, a->sin, a->k_pend, a->v_pend, a->k_win, a->v_win, a->k_stage, a->v_stage,
                          a->k_pend_out, a->v_pend_out, a->k_win_out, a->v_win_out};
    for (const void *ptr : ptrs)
        PKV_REQUIRE((reinterpret_cast<uintptr_t>(ptr) & 15u) == 0, PKV_ERR_INVALID, "buffers must be 16-byte aligned");
    CutParams p;
    p.k_new = (const uint16_t *)a->k_new; p.v_new = (const uint16_t *)a->v_new; p.cos = (const uint16_t *)a->cos; p.sin = (const uint16_t *)a->sin;
    p.k_pend = (const uint16_t *)a->k_pend; p.v_pend = (const uint16_t *)a->v_pend; p.k_win = (const uint16_t *)a->k_win; p.v_win = (const uint16_t *)a->v_win;
    p.k_stage = (uint16_t *)a->k_stage; p.v_stage = (uint16_t *)a->v_stage;
    p.k_pend_out = (uint16_t *)a->k_pend_out; p.v_pend_out = (uint16_t *)a->v_pend_out;
    p.k_win_out = (uint16_t *)a->k_win_out; p.v_win_out = (uint16_t *)a->v_win_out;
    p.sb = a->stride_b; p.sh = a->stride_h; p.st = a->stride_t; p.rot_sb = a->rot_stride_b;
    p.H = a->H; p.pend = a->pend; p.held = a->pend + a->buf; p.total = (int)total; p.stage = a->stage; p.pend_out = a->pend_out;
    p.win_stride = a->win_stride;
    p.first = a->k_stage || a->v_stage ? 0 : a->stage;       // nothing to stage: the encoder reads those tokens where they are
    const int blocks = (p.total - p.first + 31) / 32;
    if (blocks > 0) {
        // all heads in one workgroup while that leaves four workgroups per CU; one head each for short runs
        p.heads = (int64_t)blocks * a->B >= 1024 ? a->H : 1;
        const dim3 grid((unsigned)blocks, (unsigned)((a->H + p.heads - 1) / p.heads), (unsigned)a->B);
        if (a->dtype == PKV_F16) cut_kernel<PKV_F16><<<grid, 256, 0, s>>>(p);
        else cut_kernel<PKV_BF16><<<grid, 256, 0, s>>>(p);
        PKV_HIP_CHECK(hipGetLastError());
    }
    if (a->pend_out) return launch_quant_dequant(a->k_pend_out, a->v_pend_out, a->k_win_out, a->v_win_out, a->dtype, a->B, a->H, a->pend_out,
                                                 a->win_stride, a->k_rel, a->v_rel, s);
    return PKV_OK;
}

int pkv_window_append(const void *k_new, const void *v_new, const void *cos, const void *sin, int dtype, int B, int H,
                      int n, int64_t stride_b, int64_t stride_h, int64_t stride_t, int64_t rot_stride_b, void *k_win,
                      void *v_win, int win_pos, int win_stride, pkv_stream_t s_) {
    using namespace pkv;
    hipStream_t s = (hipStream_t)s_;
    PKV_REQUIRE(k_new && v_new && k_win && v_win, PKV_ERR_INVALID, "null pointer argument");
    PKV_REQUIRE((cos == nullptr) == (sin == nullptr), PKV_ERR_INVALID, "cos and sin go together");
    PKV_REQUIRE(dtype == PKV_F16 || dtype == PKV_BF16, PKV_ERR_UNSUPPORTED, "Unsupported data type");
    PKV_REQUIRE(B > 0 && H > 0 && n > 0 && B <= 65535 && H <= 65535, PKV_ERR_INVALID, "sizes must be positive (batch, heads <= 65535)");
    PKV_REQUIRE(win_pos >= 0 && win_stride > 0 && win_pos + n <= win_stride, PKV_ERR_INVALID,
                "the new rows do not fit the window (%d + %d > %d)", win_pos, n, win_stride);
    PKV_REQUIRE(stride_b >= 0 && stride_h >= 0 && stride_t >= 0 && rot_stride_b >= 0, PKV_ERR_INVALID, "negative stride");
    const dim3 grid((unsigned)n, (unsigned)H, (unsigned)B);
    if (dtype == PKV_F16)
        window_append_kernel<PKV_F16><<<grid, 64, 0, s>>>((const uint16_t *)k_new, (const uint16_t *)v_new, (const uint16_t *)cos,
                                                          (const uint16_t *)sin, (long)stride_b, (long)stride_h, (long)stride_t,
                                                          (long)rot_stride_b, (uint16_t *)k_win, (uint16_t *)v_win, H, n, win_pos,
                                                          win_stride);
    else
        window_append_kernel<PKV_BF16><<<grid, 64, 0, s>>>((const uint16_t *)k_new, (const uint16_t *)v_new, (const uint16_t *)cos,
                                                           (const uint16_t *)sin, (long)stride_b, (long)stride_h, (long)stride_t,
                                                           (long)rot_stride_b, (uint16_t *)k_win, (uint16_t *)v_win, H, n, win_pos,
                                                           win_stride);
    PKV_HIP_CHECK(hipGetLastError());
    return PKV_OK;
}

}  // extern "C"
