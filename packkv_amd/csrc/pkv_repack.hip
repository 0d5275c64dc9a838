// Token repacking and the analytic pack-size model on the device.
//
// Reference (utils/compute.py): `median_repacking` (:262-270) reorders the tokens of every quantisation block,
// jointly for K and V across all heads and sequences, by descending median of the token's V codes;
// `bit_pack` (:272-297) prices a code matrix as  sum over packs of pack_len * bit_length(max - min)  payload bits
// plus (W + ceil(log2(W + 1))) metadata bits per pack, W = ceil(log2(#distinct codes)).  Both work on the uint8
// code matrix [ctx_len, hidden] (channel = (b * H + h) * 128 + d), the layout the codecs consume.
//
// Tie order: the reference sorts with torch.sort(descending=True) without stable=True, which leaves the order
// of equal medians to the backend.  Here ties keep their original order (a stable descending sort).
#include "pkv_common.hpp"
#include "pkv_runtime.hpp"
#include "pkv_block.hpp"

#include <map>
#include <mutex>

namespace pkv {

typedef unsigned short ushort2v __attribute__((ext_vector_type(2)));

// ---- lower median of every token row: one wavefront per token ----
// Rows of up to 16384 codes below 128 stay in registers (16 bytes x 16 per lane) and the median is found by
// bisection on the value: a step counts the bytes above the probe with three word-wide instructions per four codes
// ((x | 0x80) - (probe + 1) keeps bit 7 of a byte exactly when the byte is above the probe; no borrow crosses bytes
// while both are at most 128).  Other rows use a 256-bin histogram in LDS (slow when few values dominate: equal
// addresses serialise the LDS atomics).
__global__ void __launch_bounds__(256) token_median_kernel(const uint8_t *__restrict__ codes, int ctx_len, int hidden,
                                                           uint8_t *__restrict__ median) {
    __shared__ uint32_t hist[4][256];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int tok = blockIdx.x * 4 + wave;
    if (tok >= ctx_len) return;                                   // whole wavefronts leave; no workgroup barrier below
    const uint4 *row = reinterpret_cast<const uint4 *>(codes + (size_t)tok * hidden);
    const int nchunks = hidden / 16;
    const uint32_t k = (uint32_t)(hidden - 1) / 2u;               // torch.median: the lower of the two middle values
    if (nchunks <= 16 * 64) {
        uint32_t w[64];
        uint32_t high = 0u;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int c = lane + 64 * i;
            const uint4 v = c < nchunks ? row[c] : make_uint4(0x7F7F7F7Fu, 0x7F7F7F7Fu, 0x7F7F7F7Fu, 0x7F7F7F7Fu);
            w[4 * i] = v.x; w[4 * i + 1] = v.y; w[4 * i + 2] = v.z; w[4 * i + 3] = v.w;
            high |= v.x | v.y | v.z | v.w;
        }
        if (__ballot((high & 0x80808080u) != 0u) == 0ull) {
            const uint32_t n_pad = (uint32_t)(16 * 64 * 16 - hidden);   // padding bytes hold 127: above every probe
            uint32_t lo = 0u, hi = 127u;
            while (lo < hi) {
                const uint32_t mid = (lo + hi) >> 1;
                const uint32_t cmpw = (mid + 1u) * 0x01010101u;
                uint32_t above = 0u;
#pragma unroll
                for (int i = 0; i < 64; i++)
                    above += (uint32_t)__builtin_popcount(((w[i] | 0x80808080u) - cmpw) & 0x80808080u);
                above = wave_sum_u32(above) - n_pad;
                if ((uint32_t)hidden - above >= k + 1u) hi = mid; else lo = mid + 1u;   // codes <= mid reach rank k
            }
            if (lane == 0) median[tok] = (uint8_t)lo;
            return;
        }
    }
    uint32_t *h = hist[wave];
    for (int i = lane; i < 256; i += 64) h[i] = 0u;
    wave_lds_order();
    for (int c = lane; c < nchunks; c += 64) {
        const uint4 v = row[c];
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int kk = 0; kk < 4; kk++) atomicAdd(&h[(w[i] >> (8 * kk)) & 0xFFu], 1u);
    }
    wave_lds_order();
    // lane l owns bins 4l..4l+3
    const uint32_t c0 = h[4 * lane], c1 = h[4 * lane + 1], c2 = h[4 * lane + 2], c3 = h[4 * lane + 3];
    const uint32_t mine = c0 + c1 + c2 + c3;
    uint32_t inc = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t up = __shfl_up(inc, d, 64);
        if (lane >= d) inc += up;
    }
    const uint32_t before = inc - mine;
    if (before <= k && k < inc) {
        uint32_t bin = 4 * lane, run = before + c0;
        if (k >= run) { bin++; run += c1; }
        if (k >= run) { bin++; run += c2; }
        if (k >= run) bin++;
        median[tok] = (uint8_t)bin;
    }
}

// ---- order of the tokens of every block: descending median, ties in original order ----
// perm[blk * bs + r] = index inside the block of the token that moves to position r.
__global__ void block_order_kernel(const uint8_t *__restrict__ median, int block_size, uint32_t *__restrict__ perm) {
    extern __shared__ uint8_t m_s[];
    const int i = threadIdx.x;
    const size_t base = (size_t)blockIdx.x * block_size;
    if (i < block_size) m_s[i] = median[base + i];
    __syncthreads();
    if (i >= block_size) return;
    const uint32_t mine = m_s[i];
    uint32_t rank = 0;
    for (int j = 0; j < block_size; j++) {
        const uint32_t o = m_s[j];
        rank += (o > mine) || (o == mine && j < i);
    }
    perm[base + rank] = (uint32_t)i;
}

int launch_block_order(const uint8_t *median, int ctx_len, int block_size, uint32_t *perm, hipStream_t s) {
    const int threads = (block_size + 63) / 64 * 64;
    block_order_kernel<<<(unsigned)(ctx_len / block_size), threads, (size_t)block_size, s>>>(median, block_size, perm);
    PKV_HIP_CHECK(hipGetLastError());
    return PKV_OK;
}

// ---- greedy order of the tokens of every block: one workgroup of 1024 threads per block ----
// `greedy_repacking` (utils/compute.py:210-260): a block's N tokens are rows of D2 = 2 * hidden codes (K half, then
// V half).  Every pack starts from the remaining token with the largest cosine to the rounded mean of the remaining
// tokens and then takes, pack_len - 1 times, the remaining token whose addition costs the fewest payload bits,
// sum over channels of bit_length(max - min).  All of it is integer work here: the bit counts are exact, the
// bits already spent are common to all candidates (so the new total decides), and the cosines are compared exactly
// (codes are non-negative and the mean is common: cos_a > cos_b  <=>  dot_a^2 |b|^2 > dot_b^2 |a|^2, 128-bit
// products).  Ties go to the earlier token -- the order the reference's argmax / argmin see on a CPU backend;
// the reference itself leaves them, and fp32 near-ties of the cosine, to the backend.
//
// LDS: running minimum and maximum per channel (D2 bytes each; the mean borrows the maximum's array), one cost or
// one (dot, norm) pair per token, and the alive flags.  A wavefront prices whole tokens (tokens wave, wave + 16, ..),
// its lanes stride over the row 16 channels at a time; every wavefront then finds the winner for itself from the
// LDS array, so a pick costs two barriers.
constexpr int kGreedyThreads = 1024;
constexpr int kGreedyMaxTokens = 256;

__device__ __forceinline__ uint32_t bytes_even(uint32_t x) { return x & 0x00FF00FFu; }          // bytes 0, 2 -> 16-bit lanes
__device__ __forceinline__ uint32_t bytes_odd(uint32_t x) { return (x >> 8) & 0x00FF00FFu; }    // bytes 1, 3
__device__ __forceinline__ uint32_t pk_max_u16(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(ushort2v, a), __builtin_bit_cast(ushort2v, b)));
}
__device__ __forceinline__ uint32_t pk_min_u16(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(ushort2v, a), __builtin_bit_cast(ushort2v, b)));
}
// bit_length of a value below 256 held in byte `B` of x: the exponent of its float (frexp: 0 -> 0, 1 -> 1, 2..3 -> 2, ..)
template <int B>
__device__ __forceinline__ uint32_t byte_bit_length(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_frexp_expf((float)((x >> (8 * B)) & 0xFFu));
}
// sum over the four bytes of bit_length(max(x, mx) - min(x, mn))
__device__ __forceinline__ uint32_t range_bits4(uint32_t x, uint32_t mn, uint32_t mx) {
    const uint32_t re = pk_max_u16(bytes_even(x), bytes_even(mx)) - pk_min_u16(bytes_even(x), bytes_even(mn));
    const uint32_t ro = pk_max_u16(bytes_odd(x), bytes_odd(mx)) - pk_min_u16(bytes_odd(x), bytes_odd(mn));
    return byte_bit_length<0>(re) + byte_bit_length<2>(re) + byte_bit_length<0>(ro) + byte_bit_length<2>(ro);
}
__device__ __forceinline__ uint32_t bytes_min4(uint32_t a, uint32_t b) {
    return pk_min_u16(bytes_even(a), bytes_even(b)) | (pk_min_u16(bytes_odd(a), bytes_odd(b)) << 8);
}
__device__ __forceinline__ uint32_t bytes_max4(uint32_t a, uint32_t b) {
    return pk_max_u16(bytes_even(a), bytes_even(b)) | (pk_max_u16(bytes_odd(a), bytes_odd(b)) << 8);
}
__device__ __forceinline__ uint32_t dot_bytes4(uint32_t a, uint32_t b) {      // sum of the four byte products
    return (a & 0xFFu) * (b & 0xFFu) + ((a >> 8) & 0xFFu) * ((b >> 8) & 0xFFu) + ((a >> 16) & 0xFFu) * ((b >> 16) & 0xFFu) +
           (a >> 24) * (b >> 24);
}
__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long x) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) x += __shfl_xor(x, d, 64);
    return x;
}
// cos_a > cos_b for non-negative vectors with a common second operand: (dot, squared norm) pairs, exact
__device__ __forceinline__ bool cos_greater(unsigned long long dot_a, unsigned long long nx_a, unsigned long long dot_b,
                                            unsigned long long nx_b) {
    if (nx_a == 0) return false;                 // a is the zero vector: cosine 0, never above a non-negative cosine
    if (nx_b == 0) return dot_a > 0;
    const unsigned long long pa = dot_a * dot_a, pb = dot_b * dot_b;          // < 2^63 for rows of up to 2^16 bytes
    const unsigned long long lhs_hi = __umul64hi(pa, nx_b), lhs_lo = pa * nx_b;
    const unsigned long long rhs_hi = __umul64hi(pb, nx_a), rhs_lo = pb * nx_a;
    return lhs_hi > rhs_hi || (lhs_hi == rhs_hi && lhs_lo > rhs_lo);
}

__global__ void __launch_bounds__(kGreedyThreads) greedy_order_kernel(const uint8_t *__restrict__ k_codes,
                                                                      const uint8_t *__restrict__ v_codes, int hidden,
                                                                      int block_size, int pack_len,
                                                                      uint32_t *__restrict__ perm) {
    extern __shared__ __attribute__((aligned(16))) uint8_t g_lds[];
    const int D2 = 2 * hidden, n16 = D2 / 16, h16 = hidden / 16;
    uint4 *mn = reinterpret_cast<uint4 *>(g_lds), *mx = mn + n16;                 // [D2] bytes each
    unsigned long long *key_dot = reinterpret_cast<unsigned long long *>(mx + n16);   // [256]
    unsigned long long *key_nx = key_dot + kGreedyMaxTokens;                           // [256]
    uint32_t *cost = reinterpret_cast<uint32_t *>(key_nx + kGreedyMaxTokens);        // [2][256]
    uint8_t *alive = reinterpret_cast<uint8_t *>(cost + 2 * kGreedyMaxTokens);        // [256]

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int N = block_size;
    const size_t row0 = (size_t)blockIdx.x * N;
    // 16 channels `c16` of token `tok`: K half first, then V half
    auto row16 = [&](int tok, int c16) -> uint4 {
        const uint8_t *base = c16 < h16 ? k_codes + (row0 + tok) * (size_t)hidden + 16 * (size_t)c16
                                        : v_codes + (row0 + tok) * (size_t)hidden + 16 * (size_t)(c16 - h16);
        return *reinterpret_cast<const uint4 *>(base);
    };
    if (tid < kGreedyMaxTokens) alive[tid] = tid < N;
    __syncthreads();

    int n_alive = N, picked = 0, flip = 0;
    for (int pk = 0; pk < N / pack_len; pk++) {
        // ---- seed: rounded mean of the remaining tokens (into mx), then the best cosine ----
        for (int c16 = tid; c16 < n16; c16 += kGreedyThreads) {
            uint32_t sum[16];
#pragma unroll
            for (int i = 0; i < 16; i++) sum[i] = 0;
            for (int tok = 0; tok < N; tok++) {
                if (!alive[tok]) continue;
                const uint4 x = row16(tok, c16);
                const uint32_t w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
                for (int i = 0; i < 16; i++) sum[i] += (w[i >> 2] >> (8 * (i & 3))) & 0xFFu;
            }
            uint32_t m[4] = {0, 0, 0, 0};
#pragma unroll
            for (int i = 0; i < 16; i++)      // mean(dim=1).round(): fp32 quotient, round half to even
                m[i >> 2] |= (uint32_t)rintf((float)sum[i] / (float)n_alive) << (8 * (i & 3));
            mx[c16] = make_uint4(m[0], m[1], m[2], m[3]);
        }
        __syncthreads();
        for (int tok = wave; tok < N; tok += kGreedyThreads / 64) {
            if (!alive[tok]) continue;
            unsigned long long dot = 0, nx = 0;
            for (int c16 = lane; c16 < n16; c16 += 64) {
                const uint4 x = row16(tok, c16), m = mx[c16];
                dot += dot_bytes4(x.x, m.x) + dot_bytes4(x.y, m.y) + dot_bytes4(x.z, m.z) + dot_bytes4(x.w, m.w);
                nx += dot_bytes4(x.x, x.x) + dot_bytes4(x.y, x.y) + dot_bytes4(x.z, x.z) + dot_bytes4(x.w, x.w);
            }
            dot = wave_sum_u64(dot);
            nx = wave_sum_u64(nx);
            if (lane == 0) { key_dot[tok] = dot; key_nx[tok] = nx; }
        }
        __syncthreads();
        int sel = -1;
        {   // every wavefront finds the winner itself: lane-local scan in token order, then a reduction that
            // prefers the earlier token on equal cosines
            unsigned long long bd = 0, bn = 0;
            for (int tok = lane; tok < N; tok += 64) {
                if (!alive[tok]) continue;
                if (sel < 0 || cos_greater(key_dot[tok], key_nx[tok], bd, bn)) { sel = tok; bd = key_dot[tok]; bn = key_nx[tok]; }
            }
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) {
                const int os = __shfl_xor(sel, d, 64);
                const unsigned long long od = __shfl_xor(bd, d, 64), on = __shfl_xor(bn, d, 64);
                if (os >= 0 && (sel < 0 || cos_greater(od, on, bd, bn) || (!cos_greater(bd, bn, od, on) && os < sel))) {
                    sel = os; bd = od; bn = on;
                }
            }
        }
        __syncthreads();                          // everyone has read the mean and the alive flags
        for (int c16 = tid; c16 < n16; c16 += kGreedyThreads) {
            const uint4 x = row16(sel, c16);
            mn[c16] = x;
            mx[c16] = x;
        }
        if (tid == 0) { alive[sel] = 0; perm[row0 + picked] = (uint32_t)sel; }
        picked++;
        n_alive--;
        __syncthreads();

        // ---- the pack's other tokens: fewest bits after the pick ----
        for (int j = 1; j < pack_len; j++) {
            uint32_t *cst = cost + flip * kGreedyMaxTokens;
            flip ^= 1;
            for (int tok = wave; tok < N; tok += kGreedyThreads / 64) {
                if (!alive[tok]) continue;
                uint32_t bits = 0;
                for (int c16 = lane; c16 < n16; c16 += 64) {
                    const uint4 x = row16(tok, c16), lo = mn[c16], hi = mx[c16];
                    bits += range_bits4(x.x, lo.x, hi.x) + range_bits4(x.y, lo.y, hi.y) + range_bits4(x.z, lo.z, hi.z) +
                            range_bits4(x.w, lo.w, hi.w);
                }
                bits = wave_sum_u32(bits);
                if (lane == 0) cst[tok] = bits;
            }
            __syncthreads();
            uint32_t best = 0xFFFFFFFFu;           // (cost, token) in one word: the minimum is the first cheapest token
            for (int tok = lane; tok < N; tok += 64)
                if (alive[tok]) best = min(best, (cst[tok] << 8) | (uint32_t)tok);
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) best = min(best, (uint32_t)__shfl_xor(best, d, 64));
            sel = (int)(best & 0xFFu);
            __syncthreads();                      // everyone has read the alive flags
            for (int c16 = tid; c16 < n16; c16 += kGreedyThreads) {
                const uint4 x = row16(sel, c16), lo = mn[c16], hi = mx[c16];
                mn[c16] = make_uint4(bytes_min4(lo.x, x.x), bytes_min4(lo.y, x.y), bytes_min4(lo.z, x.z), bytes_min4(lo.w, x.w));
                mx[c16] = make_uint4(bytes_max4(hi.x, x.x), bytes_max4(hi.y, x.y), bytes_max4(hi.z, x.z), bytes_max4(hi.w, x.w));
            }
            if (tid == 0) { alive[sel] = 0; perm[row0 + picked] = (uint32_t)sel; }
            picked++;
            n_alive--;
            __syncthreads();
        }
    }
}

// ---- greedy order of blocks of up to 64 tokens: the block's rows stay in registers, sliced by channel ----
// A workgroup of 512 threads holds 4096 channels of all the tokens of a block (thread = 8 adjacent channels, one
// dword pair per token, in registers for the whole block), so a pick re-reads nothing from memory; rows of up to
// 2048 channels take workgroups of 256 threads, two per CU.  The workgroups that cover a block form a group: every step (a seed or a pick) each member
// sums its slice per token (every thread leaves its sums in LDS, eight threads per pair of tokens add them up),
// publishes the sums as (step number << 32 | value) words -- a pick: one word per pair of tokens, two 16-bit sums;
// a seed: dot product and squared norm per token -- reads the words of all members and finds the winner for itself.
// The words of two consecutive steps live in two buffers, and a member can be at most one step ahead of another, so
// a word is never overwritten before it was read.  Workgroups take tickets in the order they start and a group is a
// run of consecutive tickets: whenever a member waits, the members it waits for run already or start as soon as a
// complete group ahead of them leaves; the launch never holds more groups than fit the device.  The waits are
// bounded all the same (kGreedySpinLimit, error word of the state).
//
// The remaining tokens occupy register slots 0 .. n_alive - 1 (the winner's slot takes the rows of the last slot;
// lane l of every wavefront knows which token slot l holds), so a step walks a prefix of the slots without a test
// per token and two tokens are priced side by side.
//
// Pricing a token: min and max as packed 16-bit lanes, r = max - min, then bit_length(r) is the exponent of
// (2 r + 1) 2^-10 as a half: one packed fma on r read as a subnormal half (r 2^-24 * 2^15 + 2^-10, exact), the
// exponent fields masked and added by a sum of absolute differences -- 3.7 vector instructions per channel.  The
// constant bias of the exponent (5 per channel) is common to all tokens.  A step of a group of eight wide
// workgroups takes ~6.5 us on an MI355X: 3.8 us of pricing at the full rate of the vector ALUs, the rest the sums,
// the exchange, the winner and the slot move, which nothing overlaps.
// A member whose slice of a block holds no code above 15 looks its costs up instead (greedy_narrow, eight channels to a thread; its
// sums lack the bias, which is common to all tokens and so may differ from member to member).  us a launch, codes of 5 bits and
// of 4: 128 blocks x 4096 channels 306 and 159, 512 x 2048 (256 threads) 319 and 170, 32 x 8192 365 and 223 (two members), 128 x 32768 1590
// and 960 (eight).  Before there was a second path both took the time of the first.
constexpr int kSlicedThreadsWide = 512;                 // one workgroup per CU, two wavefronts per SIMD: rows of two or more slices
constexpr int kSlicedThreadsNarrow = 256;               // two workgroups per CU: rows of up to 2048 channels in more than 256 blocks
                                                        // (fewer blocks, and rows of up to 1024: greedy_order_block_kernel)
constexpr int kSlicedTokens = 64;
constexpr int kGreedySpinLimit = 1 << 22;
// words per row of the per-thread sums: runs of 32 threads, each + 4, then + 4

typedef _Float16 half2v __attribute__((ext_vector_type(2)));

// Even / odd bytes of a dword as 16-bit lanes, with the mask and the byte selector as operands: the kernel below
// makes these two constants opaque once per step, so that nothing derived from the packed rows -- which stay in
// registers for a whole block -- is kept in registers of its own from step to step.
__device__ __forceinline__ uint32_t even_bytes(uint32_t x, uint32_t mask_00ff00ff) { return x & mask_00ff00ff; }
__device__ __forceinline__ uint32_t odd_bytes(uint32_t x, uint32_t sel_0c030c01) { return __builtin_amdgcn_perm(0u, x, sel_0c030c01); }

// Two tokens (a, b), 8 channels each: sums of the exponent fields, << 10.  Stage by stage over the eight independent
// chains, so that no instruction waits for the one before it.
__device__ __forceinline__ void price8x2(uint32_t x0a, uint32_t x1a, uint32_t x0b, uint32_t x1b, const uint32_t (&mn)[4],
                                         const uint32_t (&mx)[4], uint32_t k_even, uint32_t k_odd, uint32_t &sum_a, uint32_t &sum_b) {
    const uint32_t v[8] = {even_bytes(x0a, k_even), even_bytes(x0b, k_even), odd_bytes(x0a, k_odd), odd_bytes(x0b, k_odd),
                           even_bytes(x1a, k_even), even_bytes(x1b, k_even), odd_bytes(x1a, k_odd), odd_bytes(x1b, k_odd)};
    ushort2v hi[8], lo[8];
    uint32_t e[8];
#pragma unroll
    for (int i = 0; i < 8; i++) hi[i] = __builtin_elementwise_max(__builtin_bit_cast(ushort2v, v[i]), __builtin_bit_cast(ushort2v, mx[i >> 1]));
#pragma unroll
    for (int i = 0; i < 8; i++) lo[i] = __builtin_elementwise_min(__builtin_bit_cast(ushort2v, v[i]), __builtin_bit_cast(ushort2v, mn[i >> 1]));
#pragma unroll
    for (int i = 0; i < 8; i++) hi[i] -= lo[i];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const half2v f = __builtin_elementwise_fma(__builtin_bit_cast(half2v, hi[i]), (half2v){(_Float16)32768.0f, (_Float16)32768.0f},
                                                   (half2v){(_Float16)0.0009765625f, (_Float16)0.0009765625f});
        e[i] = __builtin_bit_cast(uint32_t, f);
    }
#pragma unroll
    for (int i = 0; i < 8; i++) e[i] &= 0x7C007C00u;
    sum_a = __builtin_amdgcn_sad_u16(e[0], 0u, 0u);
    sum_b = __builtin_amdgcn_sad_u16(e[1], 0u, 0u);
#pragma unroll
    for (int i = 1; i < 4; i++) {
        sum_a = __builtin_amdgcn_sad_u16(e[2 * i], 0u, sum_a);
        sum_b = __builtin_amdgcn_sad_u16(e[2 * i + 1], 0u, sum_b);
    }
}

// data-parallel-primitive moves between the lanes of a row of 16 (0x100 | n: from lane + n, 0x110 | n: from lane - n,
// 0x142 / 0x143: lane 15 / 31 to the following rows, below 0x100: a permutation of every four lanes)
template <int CTRL, int ROW_MASK, bool ZERO_FILL>
__device__ __forceinline__ uint32_t lane_move(uint32_t old, uint32_t src) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)src, CTRL, ROW_MASK, 0xF, ZERO_FILL);
}
__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v) {      // the minimum over the wavefront, uniform
    v = min(v, lane_move<0x111, 0xF, false>(0xFFFFFFFFu, v));
    v = min(v, lane_move<0x112, 0xF, false>(0xFFFFFFFFu, v));
    v = min(v, lane_move<0x114, 0xF, false>(0xFFFFFFFFu, v));
    v = min(v, lane_move<0x118, 0xF, false>(0xFFFFFFFFu, v));
    v = min(v, lane_move<0x142, 0xA, false>(0xFFFFFFFFu, v));
    v = min(v, lane_move<0x143, 0xC, false>(0xFFFFFFFFu, v));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
__device__ __forceinline__ uint32_t quad_sum(uint32_t v) {          // every lane: the sum over its four lanes
    v += lane_move<0xB1, 0xF, false>(0u, v);
    return v + lane_move<0x4E, 0xF, false>(0u, v);
}
__device__ __forceinline__ uint32_t sum8_down(uint32_t v) {         // lanes 0, 8, ..: the sum over lanes l .. l + 7
    v += lane_move<0x101, 0xF, true>(0u, v);
    v += lane_move<0x102, 0xF, true>(0u, v);
    return v + lane_move<0x104, 0xF, true>(0u, v);
}

// Word `idx` of the 128 published words of the members first, first + stride, ..: up to four loads in flight, all of
// them repeated until every word carries the step number.  `take(w)` gets the low halves.
template <typename F>
__device__ __forceinline__ void gather_words(const uint64_t *words, uint32_t idx, uint32_t first, uint32_t stride, uint32_t members,
                                             uint32_t seq, ScanState *st, F &&take) {
    for (uint32_t m0 = first; m0 < members; m0 += 4 * stride) {
        const uint64_t *p = words + (size_t)m0 * 128 + idx;
        const bool on1 = m0 + stride < members, on2 = m0 + 2 * stride < members, on3 = m0 + 3 * stride < members;
        const uint64_t *p1 = on1 ? p + (size_t)stride * 128 : p, *p2 = on2 ? p + (size_t)2 * stride * 128 : p,
                       *p3 = on3 ? p + (size_t)3 * stride * 128 : p;
        uint64_t w0, w1, w2, w3;
        int spins = 0;
        do {
            w0 = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            w1 = __hip_atomic_load(p1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            w2 = __hip_atomic_load(p2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            w3 = __hip_atomic_load(p3, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } while (((uint32_t)(w0 >> 32) != seq || (uint32_t)(w1 >> 32) != seq || (uint32_t)(w2 >> 32) != seq ||
                  (uint32_t)(w3 >> 32) != seq) && ++spins < kGreedySpinLimit);
        if (spins >= kGreedySpinLimit) st->error = (uint32_t)PKV_ERR_INTERNAL;
        take((uint32_t)w0);
        if (on1) take((uint32_t)w1);
        if (on2) take((uint32_t)w2);
        if (on3) take((uint32_t)w3);
    }
}

// The rows of a thread: 64 slots as two vectors of 32 registers, which the slot move indexes with a uniform run-time
// index (register-indexed moves); every other access is by constant.
typedef uint32_t u32x32 __attribute__((ext_vector_type(32)));

template <int THREADS, int CHANNELS>
constexpr int greedy_narrow_words() { return 256 * 4 + 2 * 64 * (THREADS / 64) * (CHANNELS / 4); }

// Codes of at most four bits, where every one of a block is below 16.  A channel's four codes of four tokens lie in one register,
// and what a code costs -- bit_length of the pack's range once it has joined -- is looked up there: a channel's table of 16
// bytes (one of 136 for its minimum and maximum so far, read from LDS after every pick) serves four tokens with two byte
// permutes, one vector instruction a token and channel against 3.0.  A code c >= 8 is kept as 0x80 | (c - 8): as a selector
// that is out of the lower half's range, and 0xFF comes out; with its top bit flipped it selects from the upper half, and the
// codes below 8 are out of range.  So each lookup finds one cost and one 0xFF, which is a constant -1 of the whole register,
// carries included.
__device__ __forceinline__ uint32_t code_selectors(uint32_t x) { return (x & 0x07070707u) | ((x & 0x08080808u) << 4); }
__device__ __forceinline__ uint32_t selector_codes(uint32_t s, uint32_t low = 0x07070707u, uint32_t shift = 4u) { return (s & low) | ((s >> shift) & 0x08080808u); }
// Bytes [row][column] of four registers the other way round.
__device__ __forceinline__ void transpose4(const uint32_t a0, const uint32_t a1, const uint32_t a2, const uint32_t a3, uint32_t (&x)[4]) {
    const uint32_t l01 = __builtin_amdgcn_perm(a1, a0, 0x05010400u), h01 = __builtin_amdgcn_perm(a1, a0, 0x07030602u);
    const uint32_t l23 = __builtin_amdgcn_perm(a3, a2, 0x05010400u), h23 = __builtin_amdgcn_perm(a3, a2, 0x07030602u);
    x[0] = __builtin_amdgcn_perm(l23, l01, 0x05040100u);
    x[1] = __builtin_amdgcn_perm(l23, l01, 0x07060302u);
    x[2] = __builtin_amdgcn_perm(h23, h01, 0x05040100u);
    x[3] = __builtin_amdgcn_perm(h23, h01, 0x07060302u);
}
// Half of a reduction that shares its results out: lanes l and l ^ 32 (16, or by a move within a row) each give away one of two values
// and keep the sum of the other.  a's sum ends up where the lane's bit is clear (`upper` false), b's where it is set.
__device__ __forceinline__ uint32_t halve32(uint32_t a, uint32_t b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    return (uint32_t)r[0] + (uint32_t)r[1];
}
__device__ __forceinline__ uint32_t halve16(uint32_t a, uint32_t b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    return (uint32_t)r[0] + (uint32_t)r[1];
}
template <int CTRL>
__device__ __forceinline__ uint32_t halve_row(uint32_t a, uint32_t b, bool upper) {
    return (upper ? b : a) + lane_move<CTRL, 0xF, true>(0u, upper ? a : b);
}
constexpr int kRor8 = 0x128, kHalfMirror = 0x141, kXor2 = 0x4E, kXor1 = 0xB1;     // lanes l ^ 8, l ^ 7, l ^ 2, l ^ 1

// The better of this lane's vector and of the one a move brings (none: its own again): larger dot^2 / norm, by cross products,
// then lower tag.  32 bits: dot and norm stay below 2^19 (2048 channels), the products below 2^57.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ void best_cosine(uint32_t &dot, uint32_t &norm, uint32_t &tag) {
    const uint32_t d = lane_move<CTRL, ROW_MASK, false>(dot, dot), n = lane_move<CTRL, ROW_MASK, false>(norm, norm),
                   t = lane_move<CTRL, ROW_MASK, false>(tag, tag);
    const unsigned long long theirs = (unsigned long long)d * d * norm, own = (unsigned long long)dot * dot * n;
    const bool take = theirs > own || (theirs == own && t < tag);
    dot = take ? d : dot;
    norm = take ? n : norm;
    tag = take ? t : tag;
}
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ unsigned long long lane_move64(unsigned long long x) {
    const uint32_t lo = lane_move<CTRL, ROW_MASK, false>((uint32_t)x, (uint32_t)x),
                   hi = lane_move<CTRL, ROW_MASK, false>((uint32_t)(x >> 32), (uint32_t)(x >> 32));
    return ((unsigned long long)hi << 32) | lo;
}
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ void best_cosine(unsigned long long &dot, unsigned long long &norm, uint32_t &tag) {
    const unsigned long long d = lane_move64<CTRL, ROW_MASK>(dot), n = lane_move64<CTRL, ROW_MASK>(norm);
    const uint32_t t = lane_move<CTRL, ROW_MASK, false>(tag, tag);
    const unsigned __int128 theirs = (unsigned __int128)(d * d) * norm, own = (unsigned __int128)(dot * dot) * n;
    const bool take = theirs > own || (theirs == own && t < tag);
    dot = take ? d : dot;
    norm = take ? n : norm;
    tag = take ? t : tag;
}

typedef uint32_t u32x16 __attribute__((ext_vector_type(16)));

// CHANNELS adjacent channels to a thread, 4 or 8; `rows(q, v)`: v[i][t] = dword i of token 4 q + t's, called in order.  One barrier a step: a wavefront adds its
// channels up by itself -- 64 tokens in sixteen registers of byte sums, halved six times -- and leaves a sum per token; behind
// the barrier every wavefront adds the wavefronts' sums of all tokens (lane = token slot) and finds the winner.  The sums of two
// steps in turn lie in two buffers.  Where several workgroups hold a block the sums go through GROUP, with a second barrier.  About 1.5 us a step of 2048 channels, half of it
// vector instructions of two wavefronts a SIMD, the rest the latency of that chain; tables read only where a range has changed
// were slower (104 us a launch against 98), cosines compared in 128 bits by shuffles 108.
struct NoGroup {
    static constexpr bool kMany = false;
};
template <int THREADS, int CHANNELS, typename ROWS, typename GROUP>
__device__ __forceinline__ void greedy_narrow(ROWS &&rows, uint32_t *lds, int N, int pack_len, GROUP &&group, uint32_t *__restrict__ perm) {
    constexpr int kWaves = THREADS / 64, kDwords = CHANNELS / 4;
    typedef typename std::remove_reference<GROUP>::type Group;
    static_assert(CHANNELS == 4 || CHANNELS == 8, "byte sums of a lane's channels");
    static_assert(kWaves == 4 || kWaves == 8, "a lane reads the wavefronts' sums 16 bytes at a time");
    uint4 *table = reinterpret_cast<uint4 *>(lds);             // [minimum][maximum]: the cost of every code
    uint32_t *sums = lds + 256 * 4;                            // [2][64 tokens or 32 pairs][wavefront][kDwords]
    static_assert(greedy_narrow_words<THREADS, CHANNELS>() == 256 * 4 + 2 * 64 * kWaves * kDwords, "LDS");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool bit1 = lane & 2, bit2 = lane & 4, bit3 = lane & 8;
    if (tid < 256) {
        const int lo = tid >> 4, hi = max(tid & 15, lo);
        uint32_t w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int v = 0; v < 16; v++) w[v >> 2] |= (32u - (uint32_t)__clz(max(hi, v) - min(lo, v))) << (8 * (v & 3));
        table[tid] = make_uint4(w[0], w[1], w[2], w[3]);
    }
    u32x16 x[CHANNELS];                                        // x[c][q]: channel c of the tokens in slots 4 q .. 4 q + 3
#pragma unroll
    for (int q = 0; q < kSlicedTokens / 4; q++) {
        uint32_t v[kDwords][4];
        rows(q, v);
#pragma unroll
        for (int i = 0; i < kDwords; i++) {
            uint32_t by_channel[4];
            transpose4(v[i][0], v[i][1], v[i][2], v[i][3], by_channel);
#pragma unroll
            for (int c = 0; c < 4; c++) x[4 * i + c][q] = code_selectors(by_channel[c]);
        }
    }
    __syncthreads();
    // where a lane leaves its wavefront's sums and which it reads (lane = slot): see the halvings below
    const int pick_quad = (lane >> 5) | ((lane >> 3) & 2) | (kDwords == 1 ? (lane >> 1) & 4 : lane & 4) | ((lane << 2) & 8);
    const int pick_odd = kDwords == 1 ? (lane >> 2) & 1 : (lane >> 3) & 1, pick_word = (2 * pick_quad + pick_odd) * kWaves + wave;
    const int seed_word = ((int)(__brev((uint32_t)lane) >> 26) * kWaves + wave) * kDwords;
    const int pick_read = (2 * (lane >> 2) + (lane & 1)) * kWaves, pick_half = (lane & 2) << 3;
    uint32_t orig = (uint32_t)lane, order = 0u;                // the token in slot `lane`; the token picked as number `lane`
    int n_alive = N, in_pack = 0;
    uint32_t mn[2 * kDwords], mx[2 * kDwords];                 // ranges of channels (0, 2), (1, 3), (4, 6), (5, 7), as 16-bit lanes
    uint32_t cost[CHANNELS][4];                                // [channel]: its table
    for (int step = 0; step < N; step++) {
        const bool seed = in_pack == 0;
        in_pack = in_pack + 1 == pack_len ? 0 : in_pack + 1;
        uint32_t *buf = sums + (step & 1) * 64 * kWaves * kDwords;
        int sel;
        if (seed) {
            // ---- seed: rounded mean of the remaining tokens, then the best cosine ----
            uint32_t sum[CHANNELS] = {};
#pragma unroll
            for (int q = 0; q < kSlicedTokens / 4; q++) {
                if (4 * q < n_alive) {
                    const uint32_t live = n_alive - 4 * q >= 4 ? 0x01010101u : 0x01010101u >> (8 * (4 * q + 4 - n_alive));
#pragma unroll
                    for (int c = 0; c < CHANNELS; c++) sum[c] = __builtin_amdgcn_udot4(selector_codes(x[c][q]), live, sum[c], false);
                }
            }
            const float na = (float)n_alive;                   // mean(dim=1).round(): fp32 quotient, round half to even
            uint32_t mean[kDwords];
#pragma unroll
            for (int i = 0; i < kDwords; i++)
                mean[i] = (uint32_t)rintf((float)sum[4 * i] / na) | ((uint32_t)rintf((float)sum[4 * i + 1] / na) << 8) |
                          ((uint32_t)rintf((float)sum[4 * i + 2] / na) << 16) | ((uint32_t)rintf((float)sum[4 * i + 3] / na) << 24);
            // dot product and squared norm as 16-bit lanes: at most 4 x 15 x 15 a lane and four channels, 57600 a wavefront
            uint32_t g8[8], low = 0x07070707u, shift = 4u;
            asm volatile("" : "+s"(low), "+s"(shift));         // (the codes anew: those of the mean's sums would be kept in registers)
#pragma unroll
            for (int g = 0; g < 8; g++) {
                g8[g] = 0u;
                if (8 * g < n_alive) {
                    uint32_t v[8];
#pragma unroll
                    for (int q = 0; q < 2; q++) {
                        uint32_t dot[4] = {}, norm[4] = {};
#pragma unroll
                        for (int i = 0; i < kDwords; i++) {
                            uint32_t by_token[4];
                            transpose4(selector_codes(x[4 * i][2 * g + q], low, shift), selector_codes(x[4 * i + 1][2 * g + q], low, shift),
                                       selector_codes(x[4 * i + 2][2 * g + q], low, shift), selector_codes(x[4 * i + 3][2 * g + q], low, shift), by_token);
#pragma unroll
                            for (int t = 0; t < 4; t++) {
                                dot[t] = __builtin_amdgcn_udot4(by_token[t], mean[i], dot[t], false);
                                norm[t] = __builtin_amdgcn_udot4(by_token[t], by_token[t], norm[t], false);
                            }
                        }
#pragma unroll
                        for (int t = 0; t < 4; t++) v[4 * q + t] = dot[t] | (norm[t] << 16);
                    }
                    const uint32_t a = halve16(halve32(v[0], v[1]), halve32(v[2], v[3])), b = halve16(halve32(v[4], v[5]), halve32(v[6], v[7]));
                    g8[g] = halve_row<kRor8>(a, b, bit3);
                }
            }
            uint32_t g4[4];
#pragma unroll
            for (int i = 0; i < 4; i++) g4[i] = halve_row<kHalfMirror>(g8[2 * i], g8[2 * i + 1], bit2);
            const uint32_t g2a = halve_row<kXor2>(g4[0], g4[1], bit1), g2b = halve_row<kXor2>(g4[2], g4[3], bit1);
            // (slot: the lane's number with its bits in reverse)
            if constexpr (kDwords == 1) {
                buf[seed_word] = halve_row<kXor1>(g2a, g2b, lane & 1);
            } else {                                           // half a wavefront's sums fill 16 bits: the last halving in 32
                const uint32_t own = lane & 1 ? g2b : g2a, got = lane_move<kXor1, 0xF, true>(0u, lane & 1 ? g2a : g2b);
                *reinterpret_cast<uint2 *>(buf + seed_word) = make_uint2((own & 0xFFFFu) + (got & 0xFFFFu), (own >> 16) + (got >> 16));
            }
            __syncthreads();
            uint32_t dot = 0u, norm = 0u;
            if (lane < n_alive) {
#pragma unroll
                for (int i = 0; i < kWaves * kDwords; i += 4) {
                    const uint4 w = *reinterpret_cast<const uint4 *>(buf + lane * kWaves * kDwords + i);
                    if constexpr (kDwords == 1) {
                        dot += (w.x & 0xFFFFu) + (w.y & 0xFFFFu) + (w.z & 0xFFFFu) + (w.w & 0xFFFFu);
                        norm += (w.x >> 16) + (w.y >> 16) + (w.z >> 16) + (w.w >> 16);
                    } else {
                        dot += w.x + w.z;
                        norm += w.y + w.w;
                    }
                }
            }
            // equal cosines: the earlier token.  A zero vector has cosine 0; slots that are empty as well, and lose every tie.
            uint32_t tag = lane < n_alive ? (orig << 8) | (uint32_t)lane : 0x8000u | (uint32_t)lane;
            if constexpr (Group::kMany) {
                unsigned long long all_dot = dot, all_norm = norm;
                group.seeds(lane, wave, n_alive, all_dot, all_norm);
                all_norm = all_norm ? all_norm : 1ull;
                best_cosine<0x111, 0xF>(all_dot, all_norm, tag);
                best_cosine<0x112, 0xF>(all_dot, all_norm, tag);
                best_cosine<0x114, 0xF>(all_dot, all_norm, tag);
                best_cosine<0x118, 0xF>(all_dot, all_norm, tag);
                best_cosine<0x142, 0xA>(all_dot, all_norm, tag);
                best_cosine<0x143, 0xC>(all_dot, all_norm, tag);
            } else {
                norm = max(norm, 1u);
                best_cosine<0x111, 0xF>(dot, norm, tag);
                best_cosine<0x112, 0xF>(dot, norm, tag);
                best_cosine<0x114, 0xF>(dot, norm, tag);
                best_cosine<0x118, 0xF>(dot, norm, tag);
                best_cosine<0x142, 0xA>(dot, norm, tag);
                best_cosine<0x143, 0xC>(dot, norm, tag);
            }
            sel = __builtin_amdgcn_readlane((int)tag, 63) & 0xFF;
        } else {
            // ---- the pack's other tokens: fewest bits after the pick ----
            uint32_t h32[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                h32[i] = 0u;
                if (8 * i < n_alive) {
                    // (slots past the last one are priced as well: bounded sums nobody reads)
                    uint32_t s[2];
#pragma unroll
                    for (int q = 0; q < 2; q++) {
                        s[q] = CHANNELS;                       // the channels' 0xFFs
#pragma unroll
                        for (int c = 0; c < CHANNELS; c++) {
                            const uint32_t at = x[c][2 * i + q];
                            s[q] += __builtin_amdgcn_perm(cost[c][1], cost[c][0], at) + __builtin_amdgcn_perm(cost[c][3], cost[c][2], at ^ 0x80808080u);
                        }
                    }
                    h32[i] = halve32(s[0], s[1]);
                }
            }
            // bytes of at most 4 CHANNELS a lane, twice as much after each halving up to 128, then 16-bit lanes
            uint32_t h16[4], wa, wb;
#pragma unroll
            for (int j = 0; j < 4; j++) h16[j] = halve16(h32[2 * j], h32[2 * j + 1]);
            if constexpr (kDwords == 1) {
                const uint32_t za = halve_row<kRor8>(h16[0], h16[1], bit3), zb = halve_row<kRor8>(h16[2], h16[3], bit3);
                wa = halve_row<kHalfMirror>(bytes_even(za), bytes_odd(za), bit2);
                wb = halve_row<kHalfMirror>(bytes_even(zb), bytes_odd(zb), bit2);
            } else {
                uint32_t z[4];
#pragma unroll
                for (int j = 0; j < 4; j++) z[j] = halve_row<kRor8>(bytes_even(h16[j]), bytes_odd(h16[j]), bit3);
                wa = halve_row<kHalfMirror>(z[0], z[1], bit2);
                wb = halve_row<kHalfMirror>(z[2], z[3], bit2);
            }
            uint32_t u = halve_row<kXor2>(wa, wb, bit1);
            u += lane_move<kXor1, 0xF, true>(0u, u);
            if ((lane & 1) == 0) buf[pick_word] = u;           // slots 4 quad + odd and, in the upper half, + 2
            __syncthreads();
            uint32_t a = 0u;
#pragma unroll
            for (int i = 0; i < kWaves; i += 4) {
                const uint4 w = *reinterpret_cast<const uint4 *>(buf + pick_read + i);
                a += w.x + w.y + w.z + w.w;
            }
            a = (a >> pick_half) & 0xFFFFu;
            if constexpr (Group::kMany) group.picks(lane, wave, n_alive, a);
            // (cost, token) in one word: the minimum is the first cheapest token
            const uint32_t key = lane < n_alive ? (a << 8) | orig : 0xFFFFFFFFu;
            const uint32_t best = wave_min_u32(key);
            sel = (int)__builtin_ctzll(__ballot(key == best));
        }
        // the winner in slot `sel` leaves: its codes widen the pack's ranges and the last slot moves into `sel`
        const int last = n_alive - 1;
        const uint32_t tok = (uint32_t)__builtin_amdgcn_readlane((int)orig, sel);
        const uint32_t moved = (uint32_t)__builtin_amdgcn_readlane((int)orig, last);
        if (lane == sel) orig = moved;
        if (lane == step) order = tok;
        const int lq = last >> 2, sq = sel >> 2;
        const uint32_t sb = (uint32_t)sel & 3u, keep = ~(0xFFu << (8 * sb));
        const uint32_t take = (0x07060504u & keep) | (((uint32_t)last & 3u) << (8 * sb)), pair = sb | ((4u + sb) << 16) | 0x0C000C00u;
        uint32_t w[CHANNELS];
#pragma unroll
        for (int c = 0; c < CHANNELS; c++) {
            const uint32_t l = x[c][lq];
            w[c] = x[c][sq];
            x[c][sq] = __builtin_amdgcn_perm(w[c], l, take);
        }
        n_alive--;
#pragma unroll
        for (int i = 0; i < 2 * kDwords; i++) {
            const int c = 4 * (i >> 1) + (i & 1);
            const uint32_t codes = selector_codes(__builtin_amdgcn_perm(w[c + 2], w[c], pair));
            mn[i] = seed ? codes : pk_min_u16(mn[i], codes);
            mx[i] = seed ? codes : pk_max_u16(mx[i], codes);
        }
#pragma unroll
        for (int c = 0; c < CHANNELS; c++) {
            const int i = 2 * (c >> 2) + (c & 1);
            const uint32_t at = (mn[i] << 8) | (mx[i] << 4);              // bytes into the table, a 16-bit lane a channel
            const uint4 t = *reinterpret_cast<const uint4 *>(reinterpret_cast<const uint8_t *>(table) + ((at >> (c & 2) * 8) & 0xFF0u));
            cost[c][0] = t.x; cost[c][1] = t.y; cost[c][2] = t.z; cost[c][3] = t.w;
        }
    }
    if (perm && wave == 0 && lane < N) perm[lane] = order;
}

// The sums of a group's members: published and gathered as greedy_order_sliced_kernel's comment says, by members that look costs
// up and by those that compute them alike.
template <int THREADS>
struct SliceGroup {
    static constexpr bool kMany = true;
    static constexpr int kRuns = THREADS / 32, kSeedParts = THREADS / 128;
    uint64_t *xw;
    uint32_t members, mem, seq;
    int flip;
    ScanState *st;
    uint32_t (*s_tot)[64];                           // [kRuns]
    unsigned long long (*s_tot64)[128];              // [kSeedParts]
    __device__ __forceinline__ void publish(uint32_t word, uint32_t value) const {
        __hip_atomic_store(xw + ((size_t)flip * members + mem) * 128 + word, ((uint64_t)seq << 32) | value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // value v = tid & 127 of the members q = tid >> 7, q + kSeedParts, ..
    __device__ __forceinline__ void gather_seeds(int n_alive) {
        const int v = threadIdx.x & 127, q = threadIdx.x >> 7;
        unsigned long long a = 0ull;
        if (v < 2 * n_alive)
            gather_words(xw + (size_t)flip * members * 128, (uint32_t)v, (uint32_t)q, (uint32_t)kSeedParts, members, seq, st,
                         [&](uint32_t w) { a += w; });
        s_tot64[q][v] = a;
        flip ^= 1;
    }
    // pair k = tid & 31 of the members q = tid >> 5, q + kRuns, ..
    __device__ __forceinline__ void gather_picks(int n_alive) {
        const int k = threadIdx.x & 31, q = threadIdx.x >> 5;
        uint32_t a_lo = 0u, a_hi = 0u;
        if (2 * k < n_alive)
            gather_words(xw + (size_t)flip * members * 128, (uint32_t)k, (uint32_t)q, (uint32_t)kRuns, members, seq, st,
                         [&](uint32_t w) { a_lo += w & 0xFFFFu; a_hi += w >> 16; });
        s_tot[q][2 * k] = a_lo;
        s_tot[q][2 * k + 1] = a_hi;
        flip ^= 1;
    }
    // this member's sums of the token in slot `lane` -> the group's
    __device__ __forceinline__ void seeds(int lane, int wave, int n_alive, unsigned long long &dot, unsigned long long &norm) {
        seq++;
        if (members == 1) return;
        if (wave == 0 && lane < n_alive) {
            publish(2 * lane, (uint32_t)dot);
            publish(2 * lane + 1, (uint32_t)norm);
        }
        gather_seeds(n_alive);
        __syncthreads();
        dot = norm = 0ull;
        if (lane < n_alive) {
#pragma unroll
            for (int q = 0; q < kSeedParts; q++) { dot += s_tot64[q][2 * lane]; norm += s_tot64[q][2 * lane + 1]; }
        }
    }
    __device__ __forceinline__ void picks(int lane, int wave, int n_alive, uint32_t &cost) {
        seq++;
        if (members == 1) return;
        const uint32_t next = lane_move<0xB1, 0xF, true>(0u, cost);
        if (wave == 0 && (lane & 1) == 0 && lane < n_alive) publish(lane >> 1, cost | (next << 16));
        gather_picks(n_alive);
        __syncthreads();
        cost = 0u;
        for (int q = 0; q < (int)min(members, (uint32_t)kRuns); q++) cost += s_tot[q][lane];
    }
};

template <int THREADS>
__global__ void __launch_bounds__(THREADS, 2)
greedy_order_sliced_kernel(const uint8_t *__restrict__ k_codes, const uint8_t *__restrict__ v_codes, int hidden, int N,
                           int pack_len, uint32_t nblocks, uint32_t members, uint32_t groups,
                           uint32_t *__restrict__ perm, ScanState *st) {
    constexpr int kRuns = THREADS / 32, kPartStride = kRuns * 36 + 4, kSeedParts = THREADS / 128;
    __shared__ __attribute__((aligned(16))) uint32_t s_part[32 * kPartStride];   // picks: [pair of slots][thread], padded
    __shared__ uint32_t s_seed[128 * 32];            // seeds: [2 * slot + (0: dot, 1: squared norm)][adder]
    __shared__ uint32_t s_tot[kRuns][64];            // picks: sums over the members q, q + kRuns, ..
    __shared__ unsigned long long s_tot64[kSeedParts][128];   // seeds: sums over the members q, q + kSeedParts, ..
    __shared__ uint32_t s_ticket;
    const int tid = threadIdx.x, lane = tid & 63;
    if (tid == 0) s_ticket = atomicAdd(&st->ticket, 1u);
    __syncthreads();
    const uint32_t ticket = s_ticket;
    const uint32_t grp = ticket / members, mem = ticket - grp * members;
    if (grp >= groups) return;
    uint64_t *xw = st->status + (size_t)grp * 2 * members * 128;      // [buffer][member][128]
    const int D2 = 2 * hidden;
    const int ch = ((int)mem * THREADS + tid) * 8;                    // first of the thread's 8 channels
    const bool have = ch < D2;
    const uint8_t *col = ch < hidden ? k_codes + ch : v_codes + (have ? ch - hidden : 0);
    const uint32_t channels = have ? ~0u : 0u;
    SliceGroup<THREADS> group{xw, members, mem, 0u, 0, st, s_tot, s_tot64};

    for (uint32_t blk = grp; blk < nblocks; blk += groups) {
        const size_t row0 = (size_t)blk * N;
        // codes of at most four bits are looked up, by each member as its own slice allows
        // (the rows are gone through twice, each time with an address that moves on: 64 of them kept would be spilled.  Slots past
        // the block hold its last row, which is never alive there; threads without channels read some and drop it: no branch)
        const uint8_t *at;
        int left;
        auto from_the_top = [&]() {
            uint64_t first = row0 * (size_t)hidden;
            left = N;
            asm volatile("" : "+s"(first), "+s"(left));
            at = col + first;
        };
        auto next_row = [&]() {
            uint2 v = *reinterpret_cast<const uint2 *>(at);
            v.x &= channels;
            v.y &= channels;
            left--;
            at += left > 0 ? hidden : 0;
            return v;
        };
        uint32_t any = 0u;
        from_the_top();
#pragma unroll 16
        for (int t = 0; t < N; t++) {
            const uint2 v = next_row();
            any |= v.x | v.y;
        }
        from_the_top();
        if (!__syncthreads_or((any & 0xF0F0F0F0u) != 0u)) {
            greedy_narrow<THREADS, 8>(
                [&](int q, uint32_t (&v)[2][4]) {
#pragma unroll
                    for (int t = 0; t < 4; t++) {
                        const uint2 r = next_row();
                        v[0][t] = r.x;
                        v[1][t] = r.y;
                    }
                    if (q & 1) __builtin_amdgcn_sched_barrier(0);      // (no more than eight rows on their way: there are no registers for all)
                }, s_part, N, pack_len, group,
                                      mem == 0 ? perm + row0 : nullptr);
            continue;
        }
        int own = tid;                               // (what follows from it is formed here: kept through the other path it was spilled)
        asm volatile("" : "+v"(own));
        const int adder = (own >> 2) & 31;           // the LDS word that takes the sums of the thread's four lanes
        const bool quad_first = (own & 3) == 0;
        // a thread's word in a row of s_part and, as a reader, where the 32 words it adds start: rows and runs of 32 are
        // padded so that the 16-byte reads of a wavefront spread over all banks
        const int part_word = (own >> 5) * 36 + (own & 31), part_read = (own / kRuns) * kPartStride + (own % kRuns) * 36;
        u32x32 x0v[2], x1v[2];
#define x0(t) x0v[(t) >> 5][(t) & 31]
#define x1(t) x1v[(t) >> 5][(t) & 31]
#pragma unroll
        for (int t = 0; t < kSlicedTokens; t++) {
            const uint2 v = next_row();
            x0(t) = v.x;
            x1(t) = v.y;
        }
        uint32_t orig = (uint32_t)lane;          // the token in slot `lane`
        int n_alive = N, picked = 0;
        uint32_t mn[4], mx[4];       // even / odd bytes of dword 0, even / odd bytes of dword 1, as 16-bit lanes

        for (int step = 0; step < N / pack_len * pack_len; step++) {
            const bool seed = step % pack_len == 0;
            int sel = -1;
            uint32_t k_even = 0x00FF00FFu, k_odd = 0x0C030C01u, k_zero = 0u;     // opaque from here on: see even_bytes
            asm volatile("" : "+s"(k_even), "+s"(k_odd), "+v"(k_zero));
            if (seed) {
            // ---- seed: rounded mean of the remaining tokens, then the best cosine ----
            uint32_t sum[4] = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int t8 = 0; t8 < kSlicedTokens; t8 += 8) {
                if (t8 < n_alive) {
#pragma unroll
                    for (int t = t8; t < t8 + 8; t++)
                        if (t < n_alive) {
                            sum[0] += even_bytes(x0(t), k_even); sum[1] += odd_bytes(x0(t), k_odd);
                            sum[2] += even_bytes(x1(t), k_even); sum[3] += odd_bytes(x1(t), k_odd);
                        }
                }
            }
            uint32_t mean[2];
#pragma unroll
            for (int d = 0; d < 2; d++) {      // mean(dim=1).round(): fp32 quotient, round half to even
                const float na = (float)n_alive;
                const uint32_t e_lo = (uint32_t)rintf((float)(sum[2 * d] & 0xFFFFu) / na), e_hi = (uint32_t)rintf((float)(sum[2 * d] >> 16) / na);
                const uint32_t o_lo = (uint32_t)rintf((float)(sum[2 * d + 1] & 0xFFFFu) / na), o_hi = (uint32_t)rintf((float)(sum[2 * d + 1] >> 16) / na);
                mean[d] = e_lo | (o_lo << 8) | (e_hi << 16) | (o_hi << 24);
            }
            for (int i = tid; i < 128 * 32; i += THREADS) s_seed[i] = 0u;
            __syncthreads();
#pragma unroll
            for (int t8 = 0; t8 < kSlicedTokens; t8 += 8) {
                if (t8 < n_alive) {
#pragma unroll
                    for (int t = t8; t < t8 + 8; t++)
                        if (t < n_alive) {
                            const uint32_t dot = quad_sum(__builtin_amdgcn_udot4(x0(t), mean[0], __builtin_amdgcn_udot4(x1(t), mean[1], 0u, false), false));
                            const uint32_t nx = quad_sum(__builtin_amdgcn_udot4(x0(t), x0(t), __builtin_amdgcn_udot4(x1(t), x1(t), k_zero, false), false));
                            if (quad_first) {
                                atomicAdd(&s_seed[(2 * t) * 32 + adder], dot);
                                atomicAdd(&s_seed[(2 * t + 1) * 32 + adder], nx);
                            }
                        }
                }
            }
            __syncthreads();
            group.seq++;
            {   // value v: two or four adjacent threads add 16 or 8 adders each
                const int v = tid / kSeedParts, part = tid % kSeedParts;
                uint32_t a = 0u;
#pragma unroll
                for (int i = 0; i < 32 / kSeedParts; i++) a += s_seed[v * 32 + part * (32 / kSeedParts) + i];
                a += lane_move<0xB1, 0xF, false>(0u, a);
                if (kSeedParts == 4) a += lane_move<0x4E, 0xF, false>(0u, a);
                if (part == 0 && v < 2 * n_alive) {
                    if (members > 1) group.publish((uint32_t)v, a);
                    else s_tot64[0][v] = a;
                }
            }
            if (members > 1) group.gather_seeds(n_alive);
            __syncthreads();
            {
                unsigned long long bd = 0, bn = 0;
                uint32_t bo = orig;
                if (lane < n_alive) {
                    sel = lane;
                    bd = s_tot64[0][2 * lane];
                    bn = s_tot64[0][2 * lane + 1];
                    if (members > 1) {
#pragma unroll
                        for (int q = 1; q < kSeedParts; q++) { bd += s_tot64[q][2 * lane]; bn += s_tot64[q][2 * lane + 1]; }
                    }
                }
#pragma unroll
                for (int d = 32; d >= 1; d >>= 1) {      // equal cosines: the earlier token
                    const int os = __shfl_xor(sel, d, 64);
                    const uint32_t oo = __shfl_xor(bo, d, 64);
                    const unsigned long long od = __shfl_xor(bd, d, 64), on = __shfl_xor(bn, d, 64);
                    if (os >= 0 && (sel < 0 || cos_greater(od, on, bd, bn) || (!cos_greater(bd, bn, od, on) && oo < bo))) {
                        sel = os; bo = oo; bd = od; bn = on;
                    }
                }
                sel = __builtin_amdgcn_readfirstlane(sel);
            }
            } else {
            // ---- the pack's other tokens: fewest bits after the pick ----
#pragma unroll
                for (int k4 = 0; k4 < kSlicedTokens / 2; k4 += 4) {
                    if (2 * k4 < n_alive) {
#pragma unroll
                        for (int k = k4; k < k4 + 4; k++)
                            if (2 * k < n_alive) {
                                // (with an odd count the slot past the last one is priced as well: a bounded sum nobody reads)
                                uint32_t a0, a1;
                                price8x2(x0(2 * k), x1(2 * k), x0(2 * k + 1), x1(2 * k + 1), mn, mx, k_even, k_odd, a0, a1);
                                s_part[k * kPartStride + part_word] = (a0 >> 10) | (a1 << 6);   // sums of fields at bit 10: a 16-bit lane per slot
                            }
                    }
                }
                __syncthreads();
                group.seq++;
                {   // pair k: kRuns adjacent threads add 32 words each
                    const int k = tid / kRuns, part = tid % kRuns;
                    const uint4 *src = reinterpret_cast<const uint4 *>(s_part + part_read);
                    uint32_t a = 0u;
#pragma unroll
                    for (int i = 0; i < 8; i++) {
                        const uint4 w = src[i];
                        a += w.x + w.y + w.z + w.w;
                    }
                    a = sum8_down(a);
                    if (kRuns == 16) a += lane_move<0x108, 0xF, true>(0u, a);
                    if (part == 0 && 2 * k < n_alive) {
                        if (members > 1) {      // both slots of the pair in one word
                            group.publish((uint32_t)k, a);
                        } else {
                            s_tot[0][2 * k] = a & 0xFFFFu;
                            s_tot[0][2 * k + 1] = a >> 16;
                        }
                    }
                }
                if (members > 1) group.gather_picks(n_alive);
                __syncthreads();
                uint32_t key = 0xFFFFFFFFu;            // (cost, token) in one word: the minimum is the first cheapest token
                if (lane < n_alive) {
                    uint32_t a = s_tot[0][lane];
                    if (members > 1) {
#pragma unroll
                        for (int q = 1; q < kRuns; q++) a += s_tot[q][lane];
                    }
                    key = (a << 8) | orig;
                }
                const uint32_t best = wave_min_u32(key);
                sel = (int)__builtin_ctzll(__ballot(key == best));
            }
            // the winner in slot `sel` leaves: its rows widen the pack's ranges and the last slot moves into `sel`
            const int last = n_alive - 1;
            const uint32_t tok = (uint32_t)__builtin_amdgcn_readlane((int)orig, sel);
            const uint32_t moved = (uint32_t)__builtin_amdgcn_readlane((int)orig, last);
            if (lane == sel) orig = moved;
            // (both halves of the slot arrays are read and written at the index modulo 32, with what they hold unless
            // the slot lies in them: no branch, so the arrays stay where they are)
            const int li = last & 31, si = sel & 31;
            const uint32_t la0 = x0v[0][li], la1 = x1v[0][li], lb0 = x0v[1][li], lb1 = x1v[1][li];
            const uint32_t l0 = last < 32 ? la0 : lb0, l1 = last < 32 ? la1 : lb1;
            const uint32_t sa0 = x0v[0][si], sa1 = x1v[0][si], sb0 = x0v[1][si], sb1 = x1v[1][si];
            const uint32_t w0 = sel < 32 ? sa0 : sb0, w1 = sel < 32 ? sa1 : sb1;
            x0v[0][si] = sel < 32 ? l0 : sa0;
            x1v[0][si] = sel < 32 ? l1 : sa1;
            x0v[1][si] = sel < 32 ? sb0 : l0;
            x1v[1][si] = sel < 32 ? sb1 : l1;
            if (mem == 0 && tid == 0) perm[row0 + picked] = tok;
            picked++;
            n_alive--;
            if (seed) {
                mn[0] = mx[0] = even_bytes(w0, k_even); mn[1] = mx[1] = odd_bytes(w0, k_odd);
                mn[2] = mx[2] = even_bytes(w1, k_even); mn[3] = mx[3] = odd_bytes(w1, k_odd);
            } else {
                mn[0] = pk_min_u16(mn[0], even_bytes(w0, k_even)); mx[0] = pk_max_u16(mx[0], even_bytes(w0, k_even));
                mn[1] = pk_min_u16(mn[1], odd_bytes(w0, k_odd)); mx[1] = pk_max_u16(mx[1], odd_bytes(w0, k_odd));
                mn[2] = pk_min_u16(mn[2], even_bytes(w1, k_even)); mx[2] = pk_max_u16(mx[2], even_bytes(w1, k_even));
                mn[3] = pk_min_u16(mn[3], odd_bytes(w1, k_odd)); mx[3] = pk_max_u16(mx[3], odd_bytes(w1, k_odd));
            }
        }
    }
}

// ---- the same for rows of up to 2048 channels, K and V together: one workgroup holds a block by itself ----
// Four channels to a thread, and with nobody to exchange sums with there is no state, no ticket and no closing launch.  What a
// step consists of is the chain price -> sums -> winner -> move.  Codes of any width are priced as 16-bit lanes (greedy_block_wide:
// even and odd bytes apart, two registers a token, 3.0 vector instructions a channel and token), codes of four bits by looking
// them up (greedy_narrow).  256 blocks of 64 tokens, a launch: x 2048 channels 182 us wide and 99 narrow, x 1024 channels
// (256 threads) 142 and 70; 1024 blocks of the latter 342 and 182.
__device__ __forceinline__ void price4x2(uint32_t ea, uint32_t oa, uint32_t eb, uint32_t ob, const uint32_t (&mn)[2], const uint32_t (&mx)[2],
                                         uint32_t &sum_a, uint32_t &sum_b) {
    const uint32_t v[4] = {ea, eb, oa, ob};
    ushort2v hi[4], lo[4];
    uint32_t e[4];
#pragma unroll
    for (int i = 0; i < 4; i++) hi[i] = __builtin_elementwise_max(__builtin_bit_cast(ushort2v, v[i]), __builtin_bit_cast(ushort2v, mx[i >> 1]));
#pragma unroll
    for (int i = 0; i < 4; i++) lo[i] = __builtin_elementwise_min(__builtin_bit_cast(ushort2v, v[i]), __builtin_bit_cast(ushort2v, mn[i >> 1]));
#pragma unroll
    for (int i = 0; i < 4; i++) hi[i] -= lo[i];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const half2v f = __builtin_elementwise_fma(__builtin_bit_cast(half2v, hi[i]), (half2v){(_Float16)32768.0f, (_Float16)32768.0f},
                                                   (half2v){(_Float16)0.0009765625f, (_Float16)0.0009765625f});
        e[i] = __builtin_bit_cast(uint32_t, f);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) e[i] &= 0x7C007C00u;
    sum_a = __builtin_amdgcn_sad_u16(e[2], 0u, __builtin_amdgcn_sad_u16(e[0], 0u, 0u));
    sum_b = __builtin_amdgcn_sad_u16(e[3], 0u, __builtin_amdgcn_sad_u16(e[1], 0u, 0u));
}

template <int THREADS>
constexpr int greedy_block_words() { return 32 * (THREADS / 32 * 36 + 4) + 128 * 32 + 64 + 128; }

// Codes of any width: `raw` = the thread's four channels of every token, as loaded; `perm` = the block's order.
template <int THREADS>
__device__ __forceinline__ void greedy_block_wide(const uint32_t (&raw)[kSlicedTokens], uint32_t *lds, int N, int pack_len, uint32_t *__restrict__ perm) {
    constexpr int kRuns = THREADS / 32, kPartStride = kRuns * 36 + 4, kSeedParts = THREADS / 128;
    uint32_t *s_part = lds;                          // picks: [pair of slots][thread], padded
    uint32_t *s_seed = s_part + 32 * kPartStride;    // seeds: [2 * slot + (0: dot, 1: squared norm)][adder]
    uint32_t *s_tot = s_seed + 128 * 32, *s_key = s_tot + 64;
    static_assert(32 * kPartStride + 128 * 32 + 64 + 128 == greedy_block_words<THREADS>(), "LDS");
    const int tid = threadIdx.x, lane = tid & 63;
    const int adder = (tid >> 2) & 31;               // the LDS word that takes the sums of the thread's four lanes
    const bool quad_first = (tid & 3) == 0;
    const int part_word = (tid >> 5) * 36 + (tid & 31), part_read = (tid / kRuns) * kPartStride + (tid % kRuns) * 36;
    u32x32 ev[2], ov[2];
#define xe(t) ev[(t) >> 5][(t) & 31]
#define xo(t) ov[(t) >> 5][(t) & 31]
#pragma unroll
    for (int t = 0; t < kSlicedTokens; t++) {
        xe(t) = bytes_even(raw[t]);
        xo(t) = bytes_odd(raw[t]);
    }
    uint32_t orig = (uint32_t)lane;                  // the token in slot `lane`
    int n_alive = N, picked = 0;
    uint32_t mn[2], mx[2];
    for (int step = 0; step < N / pack_len * pack_len; step++) {
        const bool seed = step % pack_len == 0;
        int sel = -1;
        if (seed) {
            // ---- seed: rounded mean of the remaining tokens, then the best cosine ----
            uint32_t sum[2] = {0u, 0u};
#pragma unroll
            for (int t8 = 0; t8 < kSlicedTokens; t8 += 8) {
                if (t8 < n_alive) {
#pragma unroll
                    for (int t = t8; t < t8 + 8; t++)
                        if (t < n_alive) { sum[0] += xe(t); sum[1] += xo(t); }
                }
            }
            const float na = (float)n_alive;           // mean(dim=1).round(): fp32 quotient, round half to even
            const uint32_t mean = (uint32_t)rintf((float)(sum[0] & 0xFFFFu) / na) | ((uint32_t)rintf((float)(sum[1] & 0xFFFFu) / na) << 8) |
                                  ((uint32_t)rintf((float)(sum[0] >> 16) / na) << 16) | ((uint32_t)rintf((float)(sum[1] >> 16) / na) << 24);
            for (int i = tid; i < 128 * 32; i += THREADS) s_seed[i] = 0u;
            __syncthreads();
#pragma unroll
            for (int t8 = 0; t8 < kSlicedTokens; t8 += 8) {
                if (t8 < n_alive) {
#pragma unroll
                    for (int t = t8; t < t8 + 8; t++)
                        if (t < n_alive) {
                            const uint32_t x = xe(t) | (xo(t) << 8);
                            const uint32_t dot = quad_sum(__builtin_amdgcn_udot4(x, mean, 0u, false)), nx = quad_sum(__builtin_amdgcn_udot4(x, x, 0u, false));
                            if (quad_first) {
                                atomicAdd(&s_seed[(2 * t) * 32 + adder], dot);
                                atomicAdd(&s_seed[(2 * t + 1) * 32 + adder], nx);
                            }
                        }
                }
            }
            __syncthreads();
            {   // value v: two or four adjacent threads add 16 or 8 adders each
                const int v = tid / kSeedParts, part = tid % kSeedParts;
                uint32_t a = 0u;
#pragma unroll
                for (int i = 0; i < 32 / kSeedParts; i++) a += s_seed[v * 32 + part * (32 / kSeedParts) + i];
                a += lane_move<0xB1, 0xF, false>(0u, a);
                if (kSeedParts == 4) a += lane_move<0x4E, 0xF, false>(0u, a);
                if (part == 0) s_key[v] = a;
            }
            __syncthreads();
            unsigned long long bd = 0, bn = 0;
            uint32_t bo = orig;
            if (lane < n_alive) {
                sel = lane;
                bd = s_key[2 * lane];
                bn = s_key[2 * lane + 1];
            }
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) {        // equal cosines: the earlier token
                const int os = __shfl_xor(sel, d, 64);
                const uint32_t oo = __shfl_xor(bo, d, 64);
                const unsigned long long od = __shfl_xor(bd, d, 64), on = __shfl_xor(bn, d, 64);
                if (os >= 0 && (sel < 0 || cos_greater(od, on, bd, bn) || (!cos_greater(bd, bn, od, on) && oo < bo))) {
                    sel = os; bo = oo; bd = od; bn = on;
                }
            }
            sel = __builtin_amdgcn_readfirstlane(sel);
        } else {
            // ---- the pack's other tokens: fewest bits after the pick ----
#pragma unroll
            for (int k4 = 0; k4 < kSlicedTokens / 2; k4 += 4) {
                if (2 * k4 < n_alive) {
#pragma unroll
                    for (int k = k4; k < k4 + 4; k++)
                        if (2 * k < n_alive) {
                            // (with an odd count the slot past the last one is priced as well: a bounded sum nobody reads)
                            uint32_t a0, a1;
                            price4x2(xe(2 * k), xo(2 * k), xe(2 * k + 1), xo(2 * k + 1), mn, mx, a0, a1);
                            s_part[k * kPartStride + part_word] = (a0 >> 10) | (a1 << 6);   // sums of fields at bit 10: a 16-bit lane per slot
                        }
                }
            }
            __syncthreads();
            {   // pair k: kRuns adjacent threads add 32 words each
                const int k = tid / kRuns, part = tid % kRuns;
                const uint4 *src = reinterpret_cast<const uint4 *>(s_part + part_read);
                uint32_t a = 0u;
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const uint4 w = src[i];
                    a += w.x + w.y + w.z + w.w;
                }
                a = sum8_down(a);
                if (kRuns == 16) a += lane_move<0x108, 0xF, true>(0u, a);
                if (part == 0 && 2 * k < n_alive) {
                    s_tot[2 * k] = a & 0xFFFFu;
                    s_tot[2 * k + 1] = a >> 16;
                }
            }
            __syncthreads();
            // (cost, token) in one word: the minimum is the first cheapest token
            const uint32_t key = lane < n_alive ? (s_tot[lane] << 8) | orig : 0xFFFFFFFFu;
            const uint32_t best = wave_min_u32(key);
            sel = (int)__builtin_ctzll(__ballot(key == best));
        }
        // the winner in slot `sel` leaves: its rows widen the pack's ranges and the last slot moves into `sel`
        const int last = n_alive - 1;
        const uint32_t tok = (uint32_t)__builtin_amdgcn_readlane((int)orig, sel);
        const uint32_t moved = (uint32_t)__builtin_amdgcn_readlane((int)orig, last);
        if (lane == sel) orig = moved;
        // (both halves of the slot arrays are read and written at the index modulo 32, with what they hold unless
        // the slot lies in them: no branch, so the arrays stay where they are)
        const int li = last & 31, si = sel & 31;
        const uint32_t la0 = ev[0][li], la1 = ov[0][li], lb0 = ev[1][li], lb1 = ov[1][li];
        const uint32_t l0 = last < 32 ? la0 : lb0, l1 = last < 32 ? la1 : lb1;
        const uint32_t sa0 = ev[0][si], sa1 = ov[0][si], sb0 = ev[1][si], sb1 = ov[1][si];
        const uint32_t w0 = sel < 32 ? sa0 : sb0, w1 = sel < 32 ? sa1 : sb1;
        ev[0][si] = sel < 32 ? l0 : sa0;
        ov[0][si] = sel < 32 ? l1 : sa1;
        ev[1][si] = sel < 32 ? sb0 : l0;
        ov[1][si] = sel < 32 ? sb1 : l1;
        if (tid == 0) perm[picked] = tok;
        picked++;
        n_alive--;
        mn[0] = seed ? w0 : pk_min_u16(mn[0], w0);
        mx[0] = seed ? w0 : pk_max_u16(mx[0], w0);
        mn[1] = seed ? w1 : pk_min_u16(mn[1], w1);
        mx[1] = seed ? w1 : pk_max_u16(mx[1], w1);
    }
#undef xe
#undef xo
}

template <int THREADS>
__global__ void __launch_bounds__(THREADS, 2)
greedy_order_block_kernel(const uint8_t *__restrict__ k_codes, const uint8_t *__restrict__ v_codes, int hidden, int N, int pack_len,
                          uint32_t *__restrict__ perm) {
    __shared__ __attribute__((aligned(16))) uint32_t lds[greedy_block_words<THREADS>()];
    const int ch = (int)threadIdx.x * 4;
    const uint8_t *col = ch < hidden ? k_codes + ch : v_codes + (ch - hidden);
    const bool have = ch < 2 * hidden;
    const size_t row0 = (size_t)blockIdx.x * N;
    uint32_t raw[kSlicedTokens], any = 0u;
#pragma unroll
    for (int t = 0; t < kSlicedTokens; t++) {
        raw[t] = 0u;
        if (t < N && have) raw[t] = *reinterpret_cast<const uint32_t *>(col + (row0 + t) * (size_t)hidden);
    }
#pragma unroll
    for (int t = 0; t < kSlicedTokens; t++) any |= raw[t];
    if (__syncthreads_or((any & 0xF0F0F0F0u) != 0u)) greedy_block_wide<THREADS>(raw, lds, N, pack_len, perm + row0);
    else greedy_narrow<THREADS, 4>(
        [&](int q, uint32_t (&v)[1][4]) {
#pragma unroll
            for (int t = 0; t < 4; t++) v[0][t] = raw[4 * q + t];
        }, lds, N, pack_len, NoGroup{}, perm + row0);
}

// ---- out row r = in row perm[r], for K and V at once: grid (ctx_len), 256 threads ----
__global__ void __launch_bounds__(256) gather_rows_kernel(const uint8_t *__restrict__ k_in, const uint8_t *__restrict__ v_in,
                                                          uint8_t *__restrict__ k_out, uint8_t *__restrict__ v_out,
                                                          const uint32_t *__restrict__ perm, int block_size, int hidden) {
    const size_t r = blockIdx.x;
    const size_t src = r - r % (size_t)block_size + perm[r];
    const uint4 *ks = reinterpret_cast<const uint4 *>(k_in + src * hidden), *vs = reinterpret_cast<const uint4 *>(v_in + src * hidden);
    uint4 *kd = reinterpret_cast<uint4 *>(k_out + r * hidden), *vd = reinterpret_cast<uint4 *>(v_out + r * hidden);
    for (int c = threadIdx.x; c < hidden / 16; c += 256) {
        kd[c] = ks[c];
        vd[c] = vs[c];
    }
}

// ---- analytic size: sum of bit_length(max - min) over packs, and which code values occur ----
// State between the workgroups of a launch: words of the stream's look-back state, zero before and after it.
struct PackSizeState {
    unsigned long long sum;             // workgroups that are done << kPackSizeDone | sum of the pack widths so far
    unsigned long long present[4];      // bit v: code v occurs
};
constexpr int kPackSizeDone = 52;       // fewer than 2^12 workgroups; 2^52 bits are 2^49 bytes of codes at the very least

// 256 or 1024 threads per workgroup, a grid-stride walk over the items (pack, 4 WORDS adjacent channels), the channel chunk
// running fastest so that a wavefront reads whole rows; 16 / WORDS rows in flight per thread; minima and maxima as packed
// 16-bit lanes (even and odd bytes of every dword apart).  One atomic per workgroup: same-address atomics retire
// one after the other, so their number, not the bytes, would set the time of a grid with a workgroup per pack -- and the
// wavefronts of a CU share a workgroup of 1024 (one presence table to clear, one atomic) rather than having one each of four.
// Random 4-bit codes, packs of 16, a call's kernel time: 32768 x 16384 codes 113 us (174 with up to 2048 workgroups of 256
// threads and 16 channels a thread), 16384 x 4096 31 (60.6), 16384 x 1024 19.6 (21.1), 256 x 512 9.4 (12.6).
// Bound by instruction issue: 7 vector instructions per dword for the ranges and 8 for the presence flags (a
// register bit mask for values below 32 instead of the LDS flags costs the same).
// The last workgroup to finish hands the result to the waiting host thread (a tagged slot in pinned memory) and leaves
// the state clear: a launch to zero the result, a copy and a stream synchronisation around it, and a pair of events,
// made a call 55 us around a kernel of 12 (16384 tokens x 8 heads of fp16 K and V, greedy record: 641 -> 388 us, with the sizes
// before the repacking counted once).  Everything crosses workgroups by atomics that are complete before the workgroup's one
// addition to `sum` (which also counts it done): no fence, no cached read of another workgroup's data.
typedef unsigned short pk_u16x2 __attribute__((ext_vector_type(2)));

// One or two matrices of one shape (K and V: blockIdx.y), whose last workgroups report apart; with PERM the rows of a block of
// `block_size` tokens (a multiple of the pack) in the order of a repacking: row r of block b is row perm[b * block_size + r] of it, so that
// a repacked matrix need not be written to be priced (16384 x 2 x 1024 codes: 27.1 us a call; written first, 25.5 and 11 for the gather).
constexpr int kPackSizeMost = 2, kPackSizeWords = 3;       // matrices of a launch, words of a slot for each
static_assert(kPackSizeMost * kPackSizeWords <= kSlotWords, "a slot holds the results of a launch: the next one is another thread's");
struct PackSizeJob {
    const uint8_t *codes[kPackSizeMost];
    PackSizeState *st;                   // one for each matrix
    unsigned long long *slot;            // kPackSizeWords words for each matrix
    const uint32_t *perm;
    int block_size;
};
template <int WORDS, bool PERM>
__global__ void __launch_bounds__(1024) pack_size_kernel(const PackSizeJob job, int hidden, int pack_len, size_t n_items, uint32_t tag) {
    const uint8_t *__restrict__ codes = job.codes[blockIdx.y];
    PackSizeState *st = job.st + blockIdx.y;
    unsigned long long *slot = job.slot + kPackSizeWords * blockIdx.y;
    // a presence word per (code value, lane % 32): a lane marks its own column, so the marks of a wavefront never
    // share a bank however few values the matrix holds (one word per value made every mark a same-address conflict)
    __shared__ __align__(16) uint32_t seen[256 * 32];
    __shared__ unsigned long long wsum[16];
    for (int i = threadIdx.x; i < 256 * 32 / 4; i += blockDim.x) reinterpret_cast<uint4 *>(seen)[i] = make_uint4(0u, 0u, 0u, 0u);
    __syncthreads();
    uint32_t *col = seen + (threadIdx.x & 31);
    const uint32_t chunks = (uint32_t)hidden / (4u * WORDS);
    struct Words { uint32_t w[WORDS]; };
    constexpr int kRows = 16 / WORDS;
    unsigned long long lens = 0;
    for (size_t item = (size_t)blockIdx.x * blockDim.x + threadIdx.x; item < n_items; item += (size_t)gridDim.x * blockDim.x) {
        const size_t pack = item / chunks;
        const uint32_t chunk = (uint32_t)(item - pack * chunks);
        const size_t tok0 = pack * (size_t)pack_len;
        // PERM: the block's first row; the pack's entries of the order
        const size_t row0 = PERM ? tok0 / (size_t)job.block_size * (size_t)job.block_size : tok0;
        const uint8_t *p = codes + row0 * hidden + (size_t)chunk * (4 * WORDS);
        const uint32_t *order = PERM ? job.perm + tok0 : nullptr;
        pk_u16x2 mn[2 * WORDS], mx[2 * WORDS];
#pragma unroll
        for (int i = 0; i < 2 * WORDS; i++) { mn[i] = (pk_u16x2){255, 255}; mx[i] = (pk_u16x2){0, 0}; }
        auto load = [&](int row) -> Words {
            const uint8_t *at = p + (size_t)(PERM ? (int)min(order[row], (uint32_t)job.block_size - 1u) : row) * hidden;
            if constexpr (WORDS == 4) return __builtin_bit_cast(Words, *reinterpret_cast<const uint4 *>(at));
            else return Words{{*reinterpret_cast<const uint32_t *>(at)}};
        };
        auto take = [&](const Words v) {
            const uint32_t *w = v.w;
#pragma unroll
            for (int i = 0; i < WORDS; i++) {
                const pk_u16x2 e = __builtin_bit_cast(pk_u16x2, w[i] & 0x00FF00FFu);
                const pk_u16x2 o = __builtin_bit_cast(pk_u16x2, (w[i] >> 8) & 0x00FF00FFu);
                mn[2 * i] = __builtin_elementwise_min(mn[2 * i], e);
                mx[2 * i] = __builtin_elementwise_max(mx[2 * i], e);
                mn[2 * i + 1] = __builtin_elementwise_min(mn[2 * i + 1], o);
                mx[2 * i + 1] = __builtin_elementwise_max(mx[2 * i + 1], o);
                col[32u * e[0]] = 1u;
                col[32u * e[1]] = 1u;
                col[32u * o[0]] = 1u;
                col[32u * o[1]] = 1u;
            }
        };
        int k = 0;
        for (; k + kRows <= pack_len; k += kRows) {
            Words v[kRows];
#pragma unroll
            for (int u = 0; u < kRows; u++) v[u] = load(k + u);
#pragma unroll
            for (int u = 0; u < kRows; u++) take(v[u]);
        }
        for (; k < pack_len; k++) take(load(k));
        uint32_t l = 0;
#pragma unroll
        for (int i = 0; i < 2 * WORDS; i++) {
            const pk_u16x2 r = mx[i] - mn[i];
#pragma unroll
            for (int hlf = 0; hlf < 2; hlf++)
                l += r[hlf] ? 32u - (uint32_t)__builtin_clz((uint32_t)r[hlf]) : 0u;   // bit_length = ceil(log2(range + 1))
        }
        lens += l;
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) lens += __shfl_xor(lens, d, 64);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = lens;
    __syncthreads();
    if (threadIdx.x < 256) {   // value threadIdx.x: any of its 32 columns (read rotated, so that the threads of a wavefront spread over the banks)
        uint32_t any = 0u;
#pragma unroll 8
        for (int c = 0; c < 32; c++) any |= seen[32 * threadIdx.x + ((c + threadIdx.x) & 31)];
        const unsigned long long mine = __ballot(any != 0u);
        if ((threadIdx.x & 63) == 0) {
            // (most workgroups find what they saw already marked: a load in parallel instead of one more atomic in line)
            unsigned long long *word = st->present + (threadIdx.x >> 6);
            if (mine & ~__hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                __hip_atomic_fetch_or(word, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");            // this wavefront's marks have reached memory
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long mine = 1ull << kPackSizeDone;
        for (uint32_t i = 0; i < blockDim.x / 64u; i++) mine += wsum[i];
        const unsigned long long all = __hip_atomic_fetch_add(&st->sum, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + mine;
        if ((all >> kPackSizeDone) == gridDim.x) {
            const unsigned long long total = all & ((1ull << kPackSizeDone) - 1ull), t = (unsigned long long)tag << 34;
            uint32_t n = 0;
            for (int i = 0; i < 4; i++) {
                n += (uint32_t)__popcll(__hip_atomic_load(st->present + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                __hip_atomic_store(st->present + i, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            __hip_atomic_store(&st->sum, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(slot, (total & 0xFFFFFFFFull) | t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            __hip_atomic_store(slot + 1, (total >> 32) | t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            __hip_atomic_store(slot + 2, (unsigned long long)n | t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

static int pack_sizes(const uint8_t *const *codes, int n, const uint32_t *perm, int block_size, int ctx_len, int hidden_dim, int pack_len,
                      uint64_t *len_sum_out, uint32_t *n_unique_out, float *ms_out, hipStream_t s) {
    PKV_REQUIRE(n >= 1 && n <= kPackSizeMost, PKV_ERR_INVALID, "one or two matrices");
    PKV_REQUIRE(len_sum_out && n_unique_out, PKV_ERR_INVALID, "null pointer argument");
    for (int i = 0; i < n; i++) PKV_REQUIRE(codes[i], PKV_ERR_INVALID, "null pointer argument");
    PKV_REQUIRE(ctx_len > 0 && hidden_dim > 0 && pack_len > 0, PKV_ERR_INVALID, "sizes must be positive");
    for (int i = 0; i < n; i++)
        PKV_REQUIRE(hidden_dim % 16 == 0 && (reinterpret_cast<uintptr_t>(codes[i]) & 15u) == 0, PKV_ERR_INVALID,
                    "hidden_dim must be a multiple of 16 and the code matrix 16-byte aligned");
    PKV_REQUIRE(ctx_len % pack_len == 0, PKV_ERR_INVALID, "ctx_len must be divisible by the pack length");
    PKV_REQUIRE(!perm || (block_size > 0 && block_size % pack_len == 0 && ctx_len % block_size == 0), PKV_ERR_INVALID,
                "with a token order, ctx_len must be divisible by the block size and that by the pack length");
    int rc;
    OutcomeSlot slot;
    if ((rc = slot.take(s))) return rc;
    ScanHandle sh;
    if ((rc = prepare_scan_state((uint32_t)(n * sizeof(PackSizeState) / 8), &sh, s, true))) return rc;
    LaunchTimer tm(s, ms_out != nullptr);
    if ((rc = tm.begin())) return rc;
    // 16 channels to a thread once that fills the chip (two workgroups of 1024 per CU); below, 4 channels, and small
    // workgroups while there is not one of 1024 for every CU (1024 x 1024 codes: 10.0 us, 12.8 with 16 channels a thread).  At
    // most one of 1024 a CU: a second one clears and scans a presence table of its own and adds once more to the one sum (K and V
    // of 16384 tokens, a call: 1024 channels 25.5 us, 28.4 with twice the workgroups; 2048 33.6, 40.7; 4096 43.4, 45.7; 16384 112, 117).
    const size_t wide = (size_t)(ctx_len / pack_len) * (size_t)(hidden_dim / 16);
    const bool large = n * wide >= 512u * 1024u;
    const size_t n_items = large ? wide : 4 * wide;
    const unsigned threads = n * n_items <= 256u * 256u ? 256u : 1024u;
    const size_t wanted = (n_items + threads - 1) / threads, most = 256u / (unsigned)n;
    PackSizeJob job{{codes[0], codes[n - 1]}, reinterpret_cast<PackSizeState *>(sh.st), (unsigned long long *)slot.words, perm, block_size};
    auto kern = perm ? (large ? pack_size_kernel<4, true> : pack_size_kernel<1, true>) : (large ? pack_size_kernel<4, false> : pack_size_kernel<1, false>);
    kern<<<dim3((unsigned)(wanted < most ? wanted : most), (unsigned)n), threads, 0, s>>>(job, hidden_dim, pack_len, n_items, slot.tag);
    PKV_HIP_CHECK(hipGetLastError());
    if ((rc = scan_state_cleared(sh, s))) return rc;
    if ((rc = tm.end(ms_out))) return rc;
    uint64_t v[kPackSizeMost * kPackSizeWords];
    if ((rc = slot.wait(kPackSizeWords * n, s, v))) return rc;
    for (int i = 0; i < n; i++) {
        const uint64_t *r = v + kPackSizeWords * i;
        len_sum_out[i] = r[0] | r[1] << 32;
        n_unique_out[i] = (uint32_t)r[2];
    }
    return PKV_OK;
}

}  // namespace pkv

extern "C" {

int pkv_bit_pack_size(const uint8_t *codes, int ctx_len, int hidden_dim, int pack_len, uint64_t *len_sum_out,
                      uint32_t *n_unique_out, float *ms_out, pkv_stream_t s) {
    const uint8_t *one[1] = {codes};
    return pkv::pack_sizes(one, 1, nullptr, 0, ctx_len, hidden_dim, pack_len, len_sum_out, n_unique_out, ms_out, (hipStream_t)s);
}

int pkv_bit_pack_size_pair(const uint8_t *k_codes, const uint8_t *v_codes, const uint32_t *perm, int block_size, int ctx_len, int hidden_dim,
                           int pack_len, uint64_t len_sum_out[2], uint32_t n_unique_out[2], pkv_stream_t s) {
    const uint8_t *both[2] = {k_codes, v_codes};
    return pkv::pack_sizes(both, 2, perm, block_size, ctx_len, hidden_dim, pack_len, len_sum_out, n_unique_out, nullptr, (hipStream_t)s);
}

int pkv_median_repack(const uint8_t *k_codes, const uint8_t *v_codes, uint8_t *k_out, uint8_t *v_out, uint32_t *perm,
                      int ctx_len, int hidden_dim, int block_size, float *ms_out, pkv_stream_t s_) {
    using namespace pkv;
    hipStream_t s = (hipStream_t)s_;
    PKV_REQUIRE(k_codes && v_codes && perm && (k_out != nullptr) == (v_out != nullptr), PKV_ERR_INVALID, "null pointer argument");
    PKV_REQUIRE(k_codes != k_out && v_codes != v_out, PKV_ERR_INVALID, "repacking cannot run in place");
    PKV_REQUIRE(ctx_len > 0 && hidden_dim > 0 && block_size > 0, PKV_ERR_INVALID, "sizes must be positive");
    PKV_REQUIRE(hidden_dim % 16 == 0 && ((reinterpret_cast<uintptr_t>(k_codes) | reinterpret_cast<uintptr_t>(v_codes) |
                                          reinterpret_cast<uintptr_t>(k_out) | reinterpret_cast<uintptr_t>(v_out)) & 15u) == 0,
                PKV_ERR_INVALID, "hidden_dim must be a multiple of 16 and the code matrices 16-byte aligned");
    PKV_REQUIRE(block_size <= 1024 && ctx_len % block_size == 0, PKV_ERR_INVALID,
                "ctx_len must be divisible by a block size of at most 1024 tokens");
    void *scratch = nullptr;
    int rc = scratch_get((size_t)ctx_len, s, &scratch);
    if (rc) return rc;
    uint8_t *median = static_cast<uint8_t *>(scratch);
    LaunchTimer tm(s, ms_out != nullptr);
    if ((rc = tm.begin())) return rc;
    token_median_kernel<<<(unsigned)((ctx_len + 3) / 4), 256, 0, s>>>(v_codes, ctx_len, hidden_dim, median);
    const int threads = (block_size + 63) / 64 * 64;
    block_order_kernel<<<(unsigned)(ctx_len / block_size), threads, (size_t)block_size, s>>>(median, block_size, perm);
    if (k_out) gather_rows_kernel<<<(unsigned)ctx_len, 256, 0, s>>>(k_codes, v_codes, k_out, v_out, perm, block_size, hidden_dim);
    PKV_HIP_CHECK(hipGetLastError());
    return tm.end(ms_out);
}

int pkv_greedy_repack(const uint8_t *k_codes, const uint8_t *v_codes, uint8_t *k_out, uint8_t *v_out, uint32_t *perm,
                      int ctx_len, int hidden_dim, int block_size, int pack_len, float *ms_out, pkv_stream_t s_) {
    using namespace pkv;
    hipStream_t s = (hipStream_t)s_;
    PKV_REQUIRE(k_codes && v_codes && perm && (k_out != nullptr) == (v_out != nullptr), PKV_ERR_INVALID, "null pointer argument");
    PKV_REQUIRE(k_codes != k_out && v_codes != v_out, PKV_ERR_INVALID, "repacking cannot run in place");
    const bool rows = k_out != nullptr;               // without outputs: the order only
    PKV_REQUIRE(ctx_len > 0 && hidden_dim > 0 && block_size > 0 && pack_len > 0, PKV_ERR_INVALID, "sizes must be positive");
    PKV_REQUIRE(hidden_dim % 16 == 0 && ((reinterpret_cast<uintptr_t>(k_codes) | reinterpret_cast<uintptr_t>(v_codes) |
                                          reinterpret_cast<uintptr_t>(k_out) | reinterpret_cast<uintptr_t>(v_out)) & 15u) == 0,
                PKV_ERR_INVALID, "hidden_dim must be a multiple of 16 and the code matrices 16-byte aligned");
    PKV_REQUIRE(block_size <= kGreedyMaxTokens && ctx_len % block_size == 0, PKV_ERR_INVALID,
                "ctx_len must be divisible by a block size of at most 256 tokens");
    PKV_REQUIRE(block_size % pack_len == 0, PKV_ERR_INVALID,
                "block_size must be a multiple of pack_len (the reference drops the tokens of an incomplete pack)");
    const uint32_t nblocks = (uint32_t)(ctx_len / block_size);
    // blocks of up to 64 tokens: register-resident channel slices, as many groups of workgroups as fit the device;
    int rc;
    // K and V rows of up to 1024 channels together: a workgroup of 256 threads to a block.  Up to 2048: one of 512, while the blocks do
    // not outnumber the CUs (5-bit codes: 256 blocks 235 -> 204 us, the gather included; 512 blocks 345 against 390: two workgroups of the
    // sliced kernel on a CU fill each other's gaps; 4-bit codes, without a gather: 256 blocks 102, 512 in the sliced kernel 170).
    const bool small = 2 * (size_t)hidden_dim <= 4u * kSlicedThreadsNarrow;
    if (block_size <= kSlicedTokens && (small || (2 * (size_t)hidden_dim <= 4u * kSlicedThreadsWide && nblocks <= 256u))) {
        LaunchTimer tm(s, ms_out != nullptr);
        if ((rc = tm.begin())) return rc;
        if (small)
            greedy_order_block_kernel<kSlicedThreadsNarrow><<<nblocks, kSlicedThreadsNarrow, 0, s>>>(k_codes, v_codes, hidden_dim, block_size, pack_len, perm);
        else
            greedy_order_block_kernel<kSlicedThreadsWide><<<nblocks, kSlicedThreadsWide, 0, s>>>(k_codes, v_codes, hidden_dim, block_size, pack_len, perm);
        if (rows) gather_rows_kernel<<<(unsigned)ctx_len, 256, 0, s>>>(k_codes, v_codes, k_out, v_out, perm, block_size, hidden_dim);
        PKV_HIP_CHECK(hipGetLastError());
        return tm.end(ms_out);
    }
    // rows of more than one narrow slice go to the wide workgroups, which have a CU to themselves: two members of a
    // group on one CU, or another group's member in the same phase, would price at half speed and hold up their group
    const bool wide = 2 * (size_t)hidden_dim > 8u * kSlicedThreadsNarrow;
    const uint32_t slice = 8u * (wide ? kSlicedThreadsWide : kSlicedThreadsNarrow);
    uint32_t members = (uint32_t)((2 * (size_t)hidden_dim + slice - 1) / slice), groups = 0;
    if (block_size <= kSlicedTokens) {
        int dev = 0;
        PKV_HIP_CHECK(hipGetDevice(&dev));
        static std::mutex mu;
        static std::map<std::pair<int, bool>, uint32_t> resident;      // workgroups of the sliced kernel that fit the device at once
        std::lock_guard<std::mutex> lock(mu);
        auto it = resident.find({dev, wide});
        if (it == resident.end()) {
            int cus = 0, per_cu = 0;
            PKV_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
            if (wide)
                PKV_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(
                    &per_cu, reinterpret_cast<const void *>(greedy_order_sliced_kernel<kSlicedThreadsWide>), kSlicedThreadsWide, 0));
            else
                PKV_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(
                    &per_cu, reinterpret_cast<const void *>(greedy_order_sliced_kernel<kSlicedThreadsNarrow>), kSlicedThreadsNarrow, 0));
            it = resident.emplace(std::make_pair(dev, wide), (uint32_t)(cus > 0 && per_cu > 0 ? cus * per_cu : 0)).first;
        }
        groups = it->second / members;
        if (groups > nblocks) groups = nblocks;
    }
    if (groups > 0) {
        ScanHandle sh;
        if ((rc = prepare_scan_state(groups * 2u * members * 128u, &sh, s, ms_out != nullptr))) return rc;
        ScanState *st = sh.st;
        LaunchTimer tm(s, ms_out != nullptr);
        if ((rc = tm.begin())) return rc;
        if (wide)
            greedy_order_sliced_kernel<kSlicedThreadsWide><<<groups * members, kSlicedThreadsWide, 0, s>>>(
                k_codes, v_codes, hidden_dim, block_size, pack_len, nblocks, members, groups, perm, st);
        else
            greedy_order_sliced_kernel<kSlicedThreadsNarrow><<<groups * members, kSlicedThreadsNarrow, 0, s>>>(
                k_codes, v_codes, hidden_dim, block_size, pack_len, nblocks, members, groups, perm, st);
        if (rows) gather_rows_kernel<<<(unsigned)ctx_len, 256, 0, s>>>(k_codes, v_codes, k_out, v_out, perm, block_size, hidden_dim);
        PKV_HIP_CHECK(hipGetLastError());
        if ((rc = tm.end(ms_out))) return rc;
        uint64_t none = 0;                             // a timed call waits for the kernels: it looks at the error word too
        rc = finish_encode(sh, ms_out ? &none : nullptr, 0, s);
        PKV_REQUIRE(rc != PKV_ERR_INTERNAL, PKV_ERR_INTERNAL, "greedy order: a workgroup waited too long for the sums of its group");
        if (rc) return rc;
        return PKV_OK;
    }
    // longer blocks: the cost word holds (bits << 8 | token): bits <= 8 * 2 * hidden_dim must stay below 2^24
    const size_t lds = 4 * (size_t)hidden_dim + kGreedyMaxTokens * (8 + 8 + 8 + 1);
    PKV_REQUIRE(hidden_dim <= 32768 && lds <= 160 * 1024, PKV_ERR_UNSUPPORTED,
                "not supported: the greedy order of blocks of more than 64 tokens keeps 4 * hidden_dim bytes in LDS (hidden_dim <= 32768)");
    if (lds > 48 * 1024)
        PKV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(greedy_order_kernel),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    LaunchTimer tm(s, ms_out != nullptr);
    if ((rc = tm.begin())) return rc;
    greedy_order_kernel<<<nblocks, kGreedyThreads, lds, s>>>(k_codes, v_codes, hidden_dim, block_size, pack_len, perm);
    if (rows) gather_rows_kernel<<<(unsigned)ctx_len, 256, 0, s>>>(k_codes, v_codes, k_out, v_out, perm, block_size, hidden_dim);
    PKV_HIP_CHECK(hipGetLastError());
    return tm.end(ms_out);
}

}  // extern "C"
