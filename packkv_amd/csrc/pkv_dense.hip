// The dense view of a compressed cache: K and V [B, H, T_c + T_w, 128] in the storage type, the compressed tokens
// dequantised as the reference stores them, T(T(code + zero) * scale) (utils/compute.py:173-179), then the rows of the
// 16-bit window -- what the reference's `update` returns (models/cache/packkv_quant.py:84-85).
//
// One launch, K and V in the grid's second dimension.  A workgroup of 256 threads owns 128 tokens of one (sequence,
// head): two K blocks (64 x 128) or the two V blocks of the head (128 x 64), staged into LDS as aligned 16-byte chunks.
// A K lane dequantises its four adjacent channels in registers and a half-wavefront stores whole 256-byte rows; a V
// lane owns one channel, so V codes turn through a 16 KB tile in LDS and leave as 16 bytes per lane.  Workgroups behind
// the tiles copy the window, 64 rows each.
// Bound by the memory system: 16 sequences x 8 heads x 8192 tokens of 4-bit codes take 119 us, 5.4 TB/s read and
// written (5-bit 126 us), the rate of a large device copy; unpacking to a code matrix and dequantising that took 243 us,
// and the concatenation with the window came on top.  Two sequences x 3072 tokens: 17 us against 52 us.
#include "pkv_block.hpp"
#include "pkv_runtime.hpp"

namespace pkv {

constexpr int kDenseTile = 128;      // tokens per workgroup
constexpr int kDenseWinRows = 64;    // window rows per workgroup

struct DenseSide {
    const uint8_t *stream;
    const uint32_t *info;
    const uint16_t *scale, *zero, *win;
    uint16_t *out;
    uint64_t bytes;
    uint32_t cap;                    // worst-case bytes of a block
    int bits;
};
struct DenseParams {
    DenseSide side[2];               // K, V
    int H, BH, n_tiles, T_c, T_w, par_stride, win_stride;
    uint32_t blk_stride;
};

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// A token's (scale, zero), ready for dequant4: fp16 in both halves of a word each, bf16 as fp32 bits.
template <int DT>
__device__ __forceinline__ uint2 dense_par(uint32_t scale_bits, uint32_t zero_bits) {
    if (DT == PKV_F16) return make_uint2(scale_bits * 0x00010001u, zero_bits * 0x00010001u);
    return make_uint2(scale_bits << 16, zero_bits << 16);
}
// Four codes (one per byte) of one token.  fp16: 0x6400 | code is 1024 + code, all steps are single correctly rounded
// 16-bit operations (code + zero and the product are exact in fp32, so rounding them once is what the reference's
// fp32-then-round elementwise kernels do).  bf16: fp32 with the hardware's round-to-nearest-even conversion.
template <int DT>
__device__ __forceinline__ uint2 dequant4(uint32_t c4, uint2 par) {
    if (DT == PKV_F16) {
        const f16x2 k1024 = {(_Float16)1024.f, (_Float16)1024.f};
        const f16x2 s = __builtin_bit_cast(f16x2, par.x), z = __builtin_bit_cast(f16x2, par.y);
        const f16x2 lo = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, c4, 0x04010400u)) - k1024;
        const f16x2 hi = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, c4, 0x04030402u)) - k1024;
        const f16x2 zl = lo + z, zh = hi + z;
        return make_uint2(__builtin_bit_cast(uint32_t, (f16x2)(zl * s)), __builtin_bit_cast(uint32_t, (f16x2)(zh * s)));
    }
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    const float s = __uint_as_float(par.x), z = __uint_as_float(par.y);
    uint32_t out[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const f32x2 a = {(float)((c4 >> (16 * i)) & 0xFFu) + z, (float)((c4 >> (16 * i + 8)) & 0xFFu) + z};
        const uint32_t r = __builtin_bit_cast(uint32_t, __builtin_convertvector(a, bf16x2));
        const f32x2 m = {__uint_as_float(r << 16) * s, __uint_as_float(r & 0xFFFF0000u) * s};
        out[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(m, bf16x2));
    }
    return make_uint2(out[0], out[1]);
}

template <int DT>
__global__ void __launch_bounds__(256) dense_view_kernel(const DenseParams p) {
    extern __shared__ __align__(16) uint8_t lds[];           // two staged blocks | V: the code tile
    __shared__ uint2 s_par[kDenseTile];
    const bool is_k = blockIdx.y == 0;
    const DenseSide &sd = p.side[blockIdx.y];
    const int tid = threadIdx.x;
    const uint32_t item = blockIdx.x / (uint32_t)p.BH, bh = blockIdx.x % (uint32_t)p.BH;
    uint16_t *rows = sd.out + (size_t)bh * (size_t)(p.T_c + p.T_w) * kHeadDim;
    if (item >= (uint32_t)p.n_tiles) {                       // a piece of the window
        const int r0 = (int)(item - (uint32_t)p.n_tiles) * kDenseWinRows, n16 = min(kDenseWinRows, p.T_w - r0) * (kHeadDim / 8);
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
        const u32x4 *src = reinterpret_cast<const u32x4 *>(sd.win + ((size_t)bh * p.win_stride + r0) * kHeadDim);
        u32x4 *dst = reinterpret_cast<u32x4 *>(rows + (size_t)(p.T_c + r0) * kHeadDim);
        u32x4 v[4];      // (filled whatever n16 is: an array filled under conditions went through scratch memory)
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = src[min(tid + 256 * i, n16 - 1)];
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (tid + 256 * i < n16) dst[tid + 256 * i] = v[i];
        return;
    }
    const int j = tid >> 7, t = tid & 31, u = (tid >> 5) & 3;
    if (tid < kDenseTile) {
        const size_t at = (size_t)(bh / (uint32_t)p.H) * p.par_stride + (size_t)item * kDenseTile + tid;
        s_par[tid] = dense_par<DT>(sd.scale[at], sd.zero[at]);
    }
    const uint32_t b = is_k ? (2u * item + (uint32_t)j) * (uint32_t)p.BH + bh : 2u * (item * (uint32_t)p.BH + bh) + (uint32_t)j;
    uint8_t *blk = lds + (uint32_t)j * p.blk_stride;
    uint32_t off, size;
    block_span(sd.info, b, sd.cap, sd.bytes, off, size);
    const uint32_t phase = stage_to_lds(sd.stream + off, size, blk, tid & 127, 128);
    __syncthreads();
    const UnitGeom g = unit_geom(sd.bits);
    const uint16_t *cum = reinterpret_cast<const uint16_t *>(blk + phase);
    const uint32_t start = min(phase + 8u + (u ? (uint32_t)cum[u - 1] : 0u), sd.cap);      // (a damaged header stays inside the slot)
    uint16_t *tile_rows = rows + (size_t)item * kDenseTile * kHeadDim;
    if (is_k) {
        const int tok0 = 64 * j + kPackTok * u;
        unit_codes(blk, start, t, g, [&](int k, uint32_t c4) {
            *reinterpret_cast<uint2 *>(tile_rows + (size_t)(tok0 + k) * kHeadDim + 4 * t) = dequant4<DT>(c4, s_par[tok0 + k]);
        });
        return;
    }
    uint8_t *tile = lds + 2u * p.blk_stride;
    unit_decode<false>(blk, start, 4 * j + u, t, g, tile, kHeadDim);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kDenseTile / 16; i++) {              // 16 rows of 128 codes per step, eight codes per thread
        const int tok = 16 * i + (tid >> 4), c = tid & 15;
        const uint2 c8 = *reinterpret_cast<const uint2 *>(tile + tok * kHeadDim + 8 * c);
        const uint2 par = s_par[tok];
        const uint2 a = dequant4<DT>(c8.x, par), d = dequant4<DT>(c8.y, par);
        *reinterpret_cast<uint4 *>(tile_rows + (size_t)tok * kHeadDim + 8 * c) = make_uint4(a.x, a.y, d.x, d.y);
    }
}

}  // namespace pkv

extern "C" int pkv_dense_view(const pkv_attn_args *a, void *k_out, void *v_out, pkv_stream_t s_) {
    using namespace pkv;
    hipStream_t s = (hipStream_t)s_;
    PKV_REQUIRE(a && k_out && v_out, PKV_ERR_INVALID, "null pointer argument");
    PKV_REQUIRE(a->dtype == PKV_F16 || a->dtype == PKV_BF16, PKV_ERR_UNSUPPORTED, "Unsupported data type");
    PKV_REQUIRE(a->B > 0 && a->Hkv > 0 && a->T_c >= 0 && a->T_w >= 0 && a->T_c + a->T_w > 0, PKV_ERR_INVALID, "empty cache");
    PKV_REQUIRE(a->T_c % kDenseTile == 0, PKV_ERR_INVALID, "compressed length must be a multiple of 128 tokens");
    DenseParams p;
    p.H = a->Hkv;
    p.BH = a->B * a->Hkv;
    p.n_tiles = a->T_c / kDenseTile;
    p.T_c = a->T_c; p.T_w = a->T_w;
    p.par_stride = a->par_stride ? a->par_stride : a->T_c;
    p.win_stride = a->win_stride ? a->win_stride : a->T_w;
    PKV_REQUIRE(p.par_stride >= a->T_c && p.win_stride >= a->T_w, PKV_ERR_INVALID, "row stride shorter than the row");
    PKV_REQUIRE(((reinterpret_cast<uintptr_t>(k_out) | reinterpret_cast<uintptr_t>(v_out)) & 15u) == 0, PKV_ERR_INVALID,
                "outputs must be 16-byte aligned");
    if (a->T_c > 0) {
        PKV_REQUIRE(a->k_stream && a->k_info && a->v_stream && a->v_info && a->k_scale && a->k_zero && a->v_scale && a->v_zero,
                    PKV_ERR_INVALID, "null pointer argument");
        PKV_REQUIRE(a->k_bits >= 2 && a->k_bits <= kMaxBits && a->v_bits >= 2 && a->v_bits <= kMaxBits, PKV_ERR_UNSUPPORTED,
                    "not supported: bits_len outside 2..8");
        PKV_REQUIRE(a->k_bytes > 0 && a->v_bytes > 0 && a->k_bytes < (1ull << 32) && a->v_bytes < (1ull << 32), PKV_ERR_INVALID,
                    "stream sizes must be in 1 .. 4 GiB - 1");
    }
    if (a->T_w > 0)
        PKV_REQUIRE(a->k_win && a->v_win && ((reinterpret_cast<uintptr_t>(a->k_win) | reinterpret_cast<uintptr_t>(a->v_win)) & 15u) == 0,
                    PKV_ERR_INVALID, "window tensors must be present and 16-byte aligned");
    const uint32_t k_cap = a->T_c ? (uint32_t)k_block_bound(64, a->k_bits) : 0u, v_cap = a->T_c ? (uint32_t)v_block_bound(64, a->v_bits) : 0u;
    p.side[0] = DenseSide{a->k_stream, a->k_info, (const uint16_t *)a->k_scale, (const uint16_t *)a->k_zero, (const uint16_t *)a->k_win,
                          (uint16_t *)k_out, a->k_bytes, k_cap, a->k_bits};
    p.side[1] = DenseSide{a->v_stream, a->v_info, (const uint16_t *)a->v_scale, (const uint16_t *)a->v_zero, (const uint16_t *)a->v_win,
                          (uint16_t *)v_out, a->v_bytes, v_cap, a->v_bits};
    // a slot holds a block at any phase and what the last pack's 16-byte read takes along
    p.blk_stride = (((k_cap > v_cap ? k_cap : v_cap) + 15u) & ~15u) + 32u;
    const uint64_t items = (uint64_t)p.n_tiles + (uint64_t)((a->T_w + kDenseWinRows - 1) / kDenseWinRows);
    PKV_REQUIRE(items * (uint64_t)p.BH < (1ull << 31), PKV_ERR_UNSUPPORTED, "batch x tokens too large");
    const uint32_t lds = 2u * p.blk_stride + kDenseTile * kHeadDim;
    const dim3 grid((unsigned)(items * (uint64_t)p.BH), 2);
    if (a->dtype == PKV_F16) dense_view_kernel<PKV_F16><<<grid, 256, lds, s>>>(p);
    else dense_view_kernel<PKV_BF16><<<grid, 256, lds, s>>>(p);
    PKV_HIP_CHECK(hipGetLastError());
    return PKV_OK;
}
