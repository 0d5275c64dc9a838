// The encoders for launches that do not fill the chip: a group's tokens all at once.
//
// The cells encoders (pkv_quant.hip) walk a group -- 64 tokens for K, 128 for V -- round by round: with several workgroups
// on a CU the rounds of one hide the latency of another.  While there are few groups nothing hides anything: a group costs
// four times the chain load -> token parameters -> packs -> emit, and one CU issues all of its instructions.  Here every
// 16 (K) or 32 (V) tokens of a group have wavefronts of their own, and a group's heads are dealt to workgroups in runs of
// `R`, so that the chain is gone through once and the work spreads over the CUs.  The runs exchange the minima and maxima of
// their tokens through memory, as the runs of eight heads do in the cells kernels.  Same stream, parameters and block_info.
//
// Two sizes: 256 threads, two heads of K or one of V, and 1024 threads, eight heads of K or four of V.  K and V of one call
// share a launch, K's workgroups first.
#pragma once

namespace pkv {

constexpr int kOnceSleep = 4;  // back-off of the waits, in units of 64 cycles: a few hundred workgroups at most poll
// Polls before a wavefront stops waiting for the other runs of its group.  They take tickets after its own too and may not
// have started -- another stream's kernel can hold the CUs that they need, for as long as it likes -- so it then reads the
// rows of the whole group itself (once_exchange).  A few tenths of a millisecond; where nothing else runs a run's words are
// there after a few microseconds.
constexpr int kOncePolls = 512;

// One side of a launch.
struct OnceSide {
    const uint16_t *x;
    XRows xs;
    float rel;
    uint16_t *scale, *zero;
    uint8_t *stream;
    uint64_t capacity, base;
    uint32_t *info;
    ScanState *st;
    uint64_t *xw;              // the words the runs of a group exchange, [group][run][token]
    int B, H, T, W, par_stride, nruns;
    uint32_t nwg, slot;        // workgroups; LDS bytes of a block (K) or unit (V)
    const uint32_t *perm;
    int perm_block;
    const uint16_t *scale_in, *zero_in;
    int polls;                 // kOncePolls; 0: never wait for another run
    const uint8_t *codes;      // the block codec: a code matrix [T, hidden] instead of x
    int hidden;
};
template <int NT> struct OnceRun {                         // heads of a run
    static constexpr int K = NT / 128, V = NT / 256;
};
template <int NT> struct OnceLds {
    uint64_t off;
    uint32_t idx;
    uint32_t blk_off[9];
    uint16_t usz[8][4];                                                 // [block][unit]
    uint32_t tot[4][4][4];                                              // V: payload bytes of [32 tokens][head][unit of the head]
    float2 mm[4][4][16];                                                // K: (min, max) [round][wavefront][token]; V: words [32 tokens][head][token]
    __attribute__((aligned(16))) TokPar par[NT / 64 * 32];              // [wavefront][token of its rounds]
};

// The workgroup's ticket; every thread of it calls.
template <int NT>
__device__ __forceinline__ uint32_t once_ticket(OnceLds<NT> &l, ScanState *st) {
    if (threadIdx.x == 0) l.idx = atomicAdd(&st->ticket, 1u);
    __syncthreads();
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)l.idx);
}

// A 32-bit value per token of a wavefront (token lane / LANES, the same value in the LANES lanes) combined over all runs of the
// group: `words` holds [run][stride] of them.  The wavefronts that `publish` store their run's.  `add(value)` is called for one run
// after the other, a LANES-th of them in each lane.  False (uniform) where a run was not there after `polls` looks: what was
// added is then no result, and the caller forms the value from the rows of all runs.
template <int LANES, class Add>
__device__ __forceinline__ bool once_exchange(uint64_t *words, uint32_t stride, uint32_t run, int nruns, bool publish, uint32_t mine, int polls, Add add) {
    const int lane = threadIdx.x & 63, tk = lane / LANES, part = lane % LANES;
    if (publish && part == 0)
        __hip_atomic_store(words + (size_t)run * stride + tk, (1ull << 63) | (uint64_t)mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    bool there = polls > 0;
    for (int q = part; q < nruns && there; q += LANES) {
        const uint64_t *wp = words + (size_t)q * stride + tk;
        uint64_t w = __hip_atomic_load(wp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        while ((w >> 63) == 0 && polls > 0) {
            __builtin_amdgcn_s_sleep(kOnceSleep);
            w = __hip_atomic_load(wp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            polls--;
        }
        there = (w >> 63) != 0;
        if (there) add((uint32_t)w);
    }
    return __all(there);
}

// (the sixteen row addresses are formed where they are used: kept for the rare path they took 30 registers)
__device__ __forceinline__ int once_opaque(int head) {
    asm volatile("" : "+s"(head));
    return head;
}

// Token parameters from the minimum and maximum; the lanes that `write` store them.
template <int DT>
__device__ __forceinline__ TokPar once_params(float mn, float mx, float rel, bool write, uint16_t *scale, uint16_t *zero, size_t tok) {
    const float range = round_t<DT>(mx - mn);
    const float sc = round_t<DT>(range * rel);
    const uint32_t zb = T16<DT>::to_bits(rintf(round_t<DT>(__fdiv_rn(mn, sc))));
    if (write) {
        scale[tok] = (uint16_t)T16<DT>::to_bits(sc);
        zero[tok] = (uint16_t)zb;
    }
    return token_par<DT>(sc, zb, false);
}

// Offsets of the workgroup's `nblk` blocks from their units' sizes (lane = block, first wavefront), the sum published.
template <int NT>
__device__ __forceinline__ void once_sizes(OnceLds<NT> &l, ScanState *st, uint32_t idx, int nblk) {
    const int lane = threadIdx.x & 63;
    uint32_t sz = 0;
    if (lane < nblk) sz = 8u + l.usz[lane][0] + l.usz[lane][1] + l.usz[lane][2] + l.usz[lane][3];
    const uint32_t incl = half_incl_scan(sz);
    if (lane < nblk) l.blk_off[lane + 1] = incl;
    if (lane == 0) l.blk_off[0] = 0;
    if (lane == nblk - 1) lookback_publish(st, idx, incl);
}

// The workgroup's place in the stream, by its first wavefront; then block_info.  False where the stream does not fit.
template <int NT>
__device__ __forceinline__ bool once_place(OnceLds<NT> &l, const OnceSide &a, uint32_t idx, uint32_t first, int nblk) {
    const uint32_t bytes = (uint32_t)__builtin_amdgcn_readfirstlane((int)l.blk_off[nblk]);
    if (threadIdx.x < 64) {
        const uint64_t off = a.base + lookback_offset<kOnceSleep>(a.st, idx, bytes, true);
        if (threadIdx.x == 0) {
            l.off = off;
            if (idx == a.nwg - 1) __hip_atomic_store(&a.st->total, off + bytes, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (off + bytes > a.capacity) atomicExch(&a.st->error, (uint32_t)PKV_ERR_CAPACITY);
        }
    }
    __syncthreads();
    if (l.off + bytes > a.capacity) return false;
    const uint32_t tid = threadIdx.x;
    if (tid < (uint32_t)nblk) {
        a.info[2 * (size_t)(first + tid)] = (uint32_t)(l.off + l.blk_off[tid]);
        a.info[2 * (size_t)(first + tid) + 1] = l.blk_off[tid + 1] - l.blk_off[tid];
    }
    return true;
}

__device__ __forceinline__ void once_max_code(ScanState *st, uint32_t cmax, int W) {
    if (__any(cmax >= (1u << W))) {   // codes that do not fit W bits are an error the host reports
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) cmax = max(cmax, __shfl_xor(cmax, d, 64));
        if ((threadIdx.x & 63) == 0) atomicMax(&st->max_code, cmax);
    }
}

// K: thread = (round, head of the run, lane of the unit).  The codes of a cell to the `nblk` blocks from `first` on.
template <int NT, bool WIDE>
__device__ __forceinline__ void k_write_once(const OnceSide &a, OnceLds<NT> &l, uint8_t *gbuf, uint32_t idx, int nblk, uint32_t first,
                                             const uint32_t c01[16], const uint32_t c23[16], bool checked) {
    constexpr int R = OnceRun<NT>::K;
    const int tid = threadIdx.x, j = (tid >> 5) % R, r = tid / (32 * R), t = tid & 31;
    const UnitGeom g = unit_geom(a.W);
    typename PacksOf<WIDE>::type u;
    uint32_t cmax;
    cell_build(c01, c23, u, cmax);
    pack_offsets(u.len, u.off, u.payload);
    const uint32_t usz = (uint32_t)(g.mins_bytes + g.lens_bytes) + u.payload;
    if (t == 0) l.usz[j][r] = (uint16_t)usz;
    __syncthreads();
    if (tid < 64) once_sizes(l, a.st, idx, nblk);
    if (j < nblk) {
        uint8_t *blk = gbuf + (size_t)j * a.slot;
        uint32_t at = 8u;
#pragma unroll
        for (int q = 0; q < 3; q++) at += q < r ? l.usz[j][q] : 0u;
        if (t == 0) reinterpret_cast<uint16_t *>(blk)[r] = (uint16_t)(at - 8u + usz);
        unit_emit_any(blk, at, t, g, u);
    }
    if (checked) once_max_code(a.st, j < nblk ? cmax : 0u, a.W);
    packs_put();
    __syncthreads();
    if (!once_place(l, a, idx, first, nblk)) return;
    const int q = tid >> 7;                                // 128 threads copy a block
    if (q < nblk) copy_out<128>(a.stream + l.off + l.blk_off[q], gbuf + (size_t)q * a.slot, l.blk_off[q + 1] - l.blk_off[q], tid & 127);
}

template <int NT, int DT, bool WIDE, bool PERM>
__device__ __forceinline__ void k_encode_once(const OnceSide &a, OnceLds<NT> &l, uint8_t *gbuf) {
    constexpr int R = OnceRun<NT>::K, WPR = R / 2;         // wavefronts of a round
    const uint32_t idx = once_ticket(l, a.st);
    if (idx >= a.nwg) return;
    const uint32_t run = idx % (uint32_t)a.nruns, grp = idx / (uint32_t)a.nruns;
    const int hbase = R * (int)run, H = min(R, a.H - hbase);
    const uint32_t cb = grp / (uint32_t)a.B, b = grp % (uint32_t)a.B;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = wave / WPR, wr = wave % WPR;
    const int lane = tid & 63, t = tid & 31;
    const size_t tok0 = (size_t)cb * 64 + 16 * (size_t)r;
    uint2 xr[16];
    auto load = [&](int head) {                            // heads `head` and the one after it in the halves (a repeated head changes no minimum or maximum)
        const int j0 = min(head, a.H - 1), jc = min(head + (lane >> 5), a.H - 1);
        if (PERM) {
            const size_t blk0 = (size_t)cb * 64 / (size_t)a.perm_block * (size_t)a.perm_block;
            cell_load_rows(a.x + ((size_t)b * a.H * a.T + blk0) * kHeadDim, a.perm + tok0, (uint32_t)a.perm_block - 1u,
                           (uint32_t)(((size_t)jc * a.T * kHeadDim + 4 * t) * 2), xr);
        } else {
            cell_load(reinterpret_cast<const char *>(a.x + b * a.xs.sb + j0 * a.xs.sh + (int64_t)tok0 * a.xs.st), 2 * a.xs.st,
                      ((uint32_t)(jc - j0) * (uint32_t)a.xs.sh + 4u * (uint32_t)t) * 2u, xr);
        }
    };
    load(hbase + 2 * wr);
    float mn, mx;                                          // of token lane / 4
    cell_token_minmax<DT>(xr, mn, mx);
    if (WPR > 1) {
        if ((lane & 3) == 0) l.mm[r][wr][lane >> 2] = make_float2(mn, mx);
        __syncthreads();
#pragma unroll
        for (int q = 0; q < WPR; q++) {
            const float2 p = l.mm[r][q][lane >> 2];
            mn = q ? fminf(mn, p.x) : p.x;
            mx = q ? fmaxf(mx, p.y) : p.y;
        }
    }
    if (a.nruns > 1) {
        const uint32_t mine = T16<DT>::to_bits(mn) << 16 | T16<DT>::to_bits(mx);
        // (NaN drops out of minima and maxima; a token that is nothing else keeps what the cells kernels make of it)
        const float mn0 = a.H <= 8 ? NAN : INFINITY, mx0 = a.H <= 8 ? NAN : -INFINITY;
        mn = mn0, mx = mx0;
        if (once_exchange<4>(a.xw + (size_t)grp * a.nruns * 64 + 16 * r, 64, run, a.nruns, wr == 0, mine, a.polls, [&](uint32_t w) {
                mn = fminf(mn, T16<DT>::from_bits(w >> 16));
                mx = fmaxf(mx, T16<DT>::from_bits(w & 0xFFFFu));
            })) {
#pragma unroll
            for (int d = 1; d < 4; d <<= 1) {
                mn = fminf(mn, __shfl_xor(mn, d, 64));
                mx = fmaxf(mx, __shfl_xor(mx, d, 64));
            }
        } else {
            mn = mn0, mx = mx0;
#pragma unroll 1
            for (int h = 0; h < a.H; h += 2) {
                load(once_opaque(h));
                float hmn, hmx;
                cell_token_minmax<DT>(xr, hmn, hmx);
                mn = fminf(mn, hmn);
                mx = fmaxf(mx, hmx);
            }
            load(once_opaque(hbase + 2 * wr));
        }
    }
    TokPar *par = l.par + 32 * wave;
    const TokPar tp = once_params<DT>(mn, mx, a.rel, (lane & 3) == 0 && wr == 0 && run == 0, a.scale, a.zero, (size_t)b * a.par_stride + tok0 + (lane >> 2));
    if ((lane & 3) == 0) par[lane >> 2] = tp;
    wave_lds_order();
    uint32_t c01[16], c23[16];
    cell_quant<DT>(xr, par, c01, c23);
    k_write_once<NT, WIDE>(a, l, gbuf, idx, H, grp * (uint32_t)a.H + (uint32_t)hbase, c01, c23, true);      // block index = group * heads + head
}

// V: a wavefront is 32 tokens of one head, the two rounds in its halves.  Its codes to the 2 H blocks from `first` on.
template <int NT>
__device__ __forceinline__ void v_clear_once(const OnceSide &a, uint8_t *gbuf) {      // metadata areas start as zeros
    const UnitGeom g = unit_geom(a.W);
    const uint32_t words = (uint32_t)(g.mins_bytes + g.lens_bytes) / 4u;
    for (uint32_t i = threadIdx.x; i < 8u * OnceRun<NT>::V * words; i += NT)
        reinterpret_cast<uint32_t *>(gbuf + (size_t)(i / words) * a.slot)[i % words] = 0u;
}
template <int NT, bool WIDE>
__device__ __forceinline__ void v_write_once(const OnceSide &a, OnceLds<NT> &l, uint8_t *gbuf, uint32_t idx, int H, uint32_t first,
                                             const uint32_t c01[16], const uint32_t c23[16], bool checked) {
    constexpr int R = OnceRun<NT>::V;
    const int tid = threadIdx.x, wave = tid >> 6, it = wave / R, j = wave % R, lane = tid & 63, rp = lane >> 5, t = lane & 31;
    const int seg = it >> 1, slot = 2 * (it & 1) + rp, blkid = 2 * j + (t >> 4), w = (t >> 3) & 1, m = t & 7, nblk = 2 * H;
    const UnitGeom g = unit_geom(a.W);
    const uint32_t meta = (uint32_t)(g.mins_bytes + g.lens_bytes);
    typename PacksOf<WIDE>::type u;
    uint32_t cmax;
    cell_build(c01, c23, u, cmax);
    const uint32_t pb = 2u * (u.len[0] + u.len[1] + u.len[2] + u.len[3]);
    uint32_t tot;
    const uint32_t inc = oct_incl_scan(pb, m, tot);
    const auto halves = __builtin_amdgcn_permlane32_swap(tot, tot, false, false);      // the even round's total, the odd round's
    if (rp == 0 && m == 0) l.tot[it][j][t >> 3] = halves[0] + halves[1];
    __syncthreads();
    if (tid < 8 * R) {                                     // unit (block, 2 warp + segment)
        const int q = tid >> 2, un = tid & 3, sg = un & 1, at = 2 * (q & 1) + (un >> 1);
        l.usz[q][un] = (uint16_t)(meta + l.tot[2 * sg][q >> 1][at] + l.tot[2 * sg + 1][q >> 1][at]);
    }
    if (tid < 64) {
        wave_lds_order();
        once_sizes(l, a.st, idx, nblk);
    }
    if (j < H) {
        uint8_t *unit = gbuf + (size_t)(blkid * 4 + 2 * w + seg) * a.slot;
        meta_or4(unit, m, g.W, slot, u.mn);
        meta_or4(unit + g.mins_bytes, m, g.LB, slot, u.len);
        uint32_t o = meta + ((it & 1) ? l.tot[it - 1][j][t >> 3] : 0u) + (rp ? (uint32_t)halves[0] : 0u) + (inc - pb);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            put_pack(reinterpret_cast<uint16_t *>(unit + o), u, k);
            o += 2u * u.len[k];
        }
    }
    if (checked) once_max_code(a.st, j < H ? cmax : 0u, a.W);
    packs_put();
    __syncthreads();
    if (!once_place(l, a, idx, first, nblk)) return;
    // a half-wavefront copies a unit, the first of a block its header of cumulative unit sizes
    for (int i = tid >> 5; i < 4 * nblk; i += NT / 32) {
        const int q = i >> 2, un = i & 3;
        uint8_t *dst = a.stream + l.off + l.blk_off[q];
        uint32_t cum = 0;
#pragma unroll
        for (int k = 0; k < 3; k++) cum += k < un ? l.usz[q][k] : 0u;
        const uint32_t n = l.usz[q][un];
        copy_out<32>(dst + 8 + cum, gbuf + (size_t)i * a.slot, n, tid & 31);
        if (t == 0) reinterpret_cast<uint16_t *>(dst)[un] = (uint16_t)(cum + n);
    }
}

template <int NT, int DT, bool WIDE, bool PERM>
__device__ __forceinline__ void v_encode_once(const OnceSide &a, OnceLds<NT> &l, uint8_t *gbuf) {
    constexpr int R = OnceRun<NT>::V;
    v_clear_once<NT>(a, gbuf);
    const uint32_t idx = once_ticket(l, a.st);
    if (idx >= a.nwg) return;
    const uint32_t run = idx % (uint32_t)a.nruns, grp = idx / (uint32_t)a.nruns;
    const int hbase = R * (int)run, H = min(R, a.H - hbase);
    const uint32_t cb = grp / (uint32_t)a.B, b = grp % (uint32_t)a.B;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), it = wave / R, j = wave % R;
    const int lane = tid & 63, rp = lane >> 5, t = lane & 31;
    const size_t tok = (size_t)cb * 128 + 32 * (size_t)it;
    const size_t rb = PERM ? tok / (size_t)a.perm_block * (size_t)a.perm_block : 0;      // (32 tokens lie in one repacking block)
    uint2 xr[16];
    auto load = [&](int head) {
        if (PERM)
            cell_load_rows_lanes(a.x + ((size_t)b * a.H * a.T + rb) * kHeadDim, a.perm + tok + 16 * rp, (uint32_t)a.perm_block - 1u,
                                 (uint32_t)(((size_t)head * a.T * kHeadDim + 4 * t) * 2), xr);
        else
            cell_load(reinterpret_cast<const char *>(a.x + b * a.xs.sb + head * a.xs.sh + (int64_t)tok * a.xs.st), 2 * a.xs.st,
                      (16u * (uint32_t)rp * (uint32_t)a.xs.st + 4u * (uint32_t)t) * 2u, xr);
    };
    load(hbase + min(j, H - 1));
    TokPar *par = l.par + 32 * wave;
    const size_t ptok = (size_t)b * a.par_stride + tok + (lane >> 1);                    // of token lane / 2
    const bool write = (lane & 1) == 0 && j == 0 && run == 0;
    if (PERM && a.scale_in != nullptr) {                   // the tokens' parameters come with the order
        const uint32_t src = min(a.perm[tok + (lane >> 1)], (uint32_t)a.perm_block - 1u);
        const uint32_t sb = a.scale_in[(size_t)b * a.T + rb + src], zb = a.zero_in[(size_t)b * a.T + rb + src];
        if (write) {
            a.scale[ptok] = (uint16_t)sb;
            a.zero[ptok] = (uint16_t)zb;
        }
        if ((lane & 1) == 0) par[lane >> 1] = token_par<DT>(T16<DT>::from_bits(sb), zb, false);
    } else {
        float mn, mx;
        cell_token_minmax_halves<DT>(xr, mn, mx);
        uint32_t pw = minmax_word<DT>(mn, mx);             // combined by packed minima
        if (R > 1) {
            uint32_t (*mm)[R][32] = reinterpret_cast<uint32_t (*)[R][32]>(l.mm);
            if ((lane & 1) == 0) mm[it][j][lane >> 1] = pw;
            __syncthreads();
            pw = mm[it][0][lane >> 1];
#pragma unroll
            for (int q = 1; q < R; q++) pw = pk_sel_x<false, DT != PKV_F16>(pw, mm[it][q][lane >> 1]);
        }
        if (a.nruns > 1) {
            const uint32_t mine = pw;
            if (once_exchange<2>(a.xw + (size_t)grp * a.nruns * 128 + 32 * it, 128, run, a.nruns, j == 0, mine, a.polls,
                                 [&](uint32_t w) { pw = pk_sel_x<false, DT != PKV_F16>(pw, w); })) {
                pw = pk_sel_x<false, DT != PKV_F16>(pw, (uint32_t)__shfl_xor((int)pw, 1, 64));
            } else {
                pw = mine;
#pragma unroll 1
                for (int h = 0; h < a.H; h++) {
                    load(once_opaque(h));
                    cell_token_minmax_halves<DT>(xr, mn, mx);
                    pw = pk_sel_x<false, DT != PKV_F16>(pw, minmax_word<DT>(mn, mx));
                }
                load(once_opaque(hbase + min(j, H - 1)));
            }
        }
        minmax_unword<DT>(pw, mn, mx);
        if (a.H > 8) mn = fminf(mn, INFINITY), mx = fmaxf(mx, -INFINITY);      // (a token of NaN only, as above)
        const TokPar tp = once_params<DT>(mn, mx, a.rel, write, a.scale, a.zero, ptok);
        if ((lane & 1) == 0) par[lane >> 1] = tp;
    }
    wave_lds_order();
    uint32_t c01[16], c23[16];
    cell_quant<DT, false>(xr, par + 16 * rp, c01, c23);    // (the halves of the wavefront hold different tokens)
    v_write_once<NT, WIDE>(a, l, gbuf, idx, H, grp * (uint32_t)(2 * a.H) + (uint32_t)(2 * hbase), c01, c23, true);      // block index = group * 2 heads + 2 head + half
}

template <int NT, int DT, bool WIDE, bool PERM>
__global__ void __launch_bounds__(NT) quant_encode_once_kernel(const OnceSide k, const OnceSide v, const EncodeClose c) {
    extern __shared__ __align__(16) uint8_t gbuf[];
    __shared__ OnceLds<NT> l;
    if (blockIdx.x < k.nwg) k_encode_once<NT, DT, WIDE, PERM>(k, l, gbuf);
    else v_encode_once<NT, DT, WIDE, PERM>(v, l, gbuf);
    encode_close(c, l.idx);
}

// The block codec from a code matrix: the "heads" are 128-channel slices of it, nothing to quantise and nothing to exchange.
template <int NT, bool IS_K, bool WIDE>
__global__ void __launch_bounds__(NT) code_encode_once_kernel(const OnceSide a, const EncodeClose c) {
    extern __shared__ __align__(16) uint8_t gbuf[];
    __shared__ OnceLds<NT> l;
    constexpr int R = IS_K ? OnceRun<NT>::K : OnceRun<NT>::V;
    if (!IS_K) v_clear_once<NT>(a, gbuf);
    const uint32_t idx = once_ticket(l, a.st);
    if (idx >= a.nwg) {
        encode_close(c, l.idx);
        return;
    }
    const uint32_t cb = idx / (uint32_t)a.nruns, hg = idx % (uint32_t)a.nruns;
    const int tid = threadIdx.x, t = tid & 31;
    const uint8_t *rows = a.codes + (size_t)cb * (IS_K ? 64 : 128) * (size_t)a.hidden + (size_t)hg * (128 * R);
    uint32_t w[16], c01[16], c23[16];
    if constexpr (IS_K) {
        const int r = __builtin_amdgcn_readfirstlane(tid / (32 * R));
        code_cell_load(rows + (size_t)(16 * r) * (size_t)a.hidden, (size_t)a.hidden, (uint32_t)((tid >> 5) % R * 128 + 4 * t), w);
        code_cell_pairs(w, c01, c23);
        k_write_once<NT, WIDE>(a, l, gbuf, idx, R, idx * (uint32_t)R, c01, c23, false);
    } else {
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        code_cell_load(rows + (size_t)(32 * (wave / R)) * (size_t)a.hidden, (size_t)a.hidden,
                       (uint32_t)(16 * ((tid >> 5) & 1)) * (uint32_t)a.hidden + (uint32_t)(wave % R * 128 + 4 * t), w);
        code_cell_pairs(w, c01, c23);
        v_write_once<NT, WIDE>(a, l, gbuf, idx, R, idx * (uint32_t)(2 * R), c01, c23, false);
    }
    encode_close(c, l.idx);
}

// ---- which launches, and their shapes ----------------------------------------------------------------------------

// Kernel times without the closing (encode_close) by the number of workgroups (trace; fp16, 4-bit codes, 8 heads; cells kernel | 1024 threads | 256 threads):
//   tokens         512                 4096                 8192             16384            32768
//   K           17.9 | 12.7 |  8.8   18.3 | 13.0 | 12.0   19.1 | 14.2 | 18   22.3 | 17.6 | 31   30.6 | 37 | 54 us
//   V           23.9 | 14.9 | 10.5   25.0 | 15.8 | 13.7   25.5 | 16.8 | 19   27.0 | 20.0 | 32   31.3 | 38 | 55
//   K codes     10.8 |  7.4 |  5.6   11.2 |  7.6 |  8.6   12.0 |  8.4 | 13   14.0 | 10.8 | 22   21.3 | 19 | 39
//   V codes     12.3 |  7.6 |  5.8   13.4 |  8.0 |  9.3   13.8 |  8.9 | 14   15.1 | 11.5 | 23   18.5 | 19 | 37
// What grows with the workgroups is their tickets (about 13 ns each: atomics on one address) and, past one workgroup a CU, a
// second generation that waits for the first.  So: 256 threads up to 256 workgroups (128 where there is nothing to
// quantise), then 1024 threads up to 256 workgroups, then the kernels that walk.
constexpr uint64_t kOnceSmall = 256, kOnceSmallCodes = 128, kOnceBig = 256;
struct OncePlan {
    int threads;               // 0: the launch takes the other encoders
    int run;                   // heads of a workgroup
    int nruns;
    uint32_t nwg;
};
// `groups` = (context block, sequence) pairs of `heads` heads.
static OncePlan once_plan(bool is_k, uint64_t groups, int heads, uint64_t small_limit) {
    OncePlan p{0, 0, 0, 0};
    const int small = is_k ? OnceRun<256>::K : OnceRun<256>::V, big = is_k ? OnceRun<1024>::K : OnceRun<1024>::V;
    if (groups * (uint64_t)((heads + small - 1) / small) <= small_limit) p.threads = 256, p.run = small;
    else if (groups * (uint64_t)((heads + big - 1) / big) <= kOnceBig) p.threads = 1024, p.run = big;
    else return p;
    p.nruns = (heads + p.run - 1) / p.run;
    p.nwg = (uint32_t)(groups * (uint64_t)p.nruns);
    return p;
}
static uint32_t once_slot(bool is_k, int bits) {
    const uint32_t n = is_k ? (uint32_t)k_block_bound(64, bits) : ((uint32_t)v_block_bound(64, bits) - 8u) / 4u;
    return (n + 15u) & ~15u;
}
static uint32_t once_lds(bool is_k, int run, uint32_t slot) { return (uint32_t)run * slot * (is_k ? 1u : 8u) + 64u; }

template <int NT>
static int once_launch_codes(bool is_k, const OnceSide &a, int run, const EncodeClose &c, hipStream_t s) {
    const bool wide = a.W > 4;
    auto kern = is_k ? (wide ? code_encode_once_kernel<NT, true, true> : code_encode_once_kernel<NT, true, false>)
                     : (wide ? code_encode_once_kernel<NT, false, true> : code_encode_once_kernel<NT, false, false>);
    const uint32_t lds = once_lds(is_k, run, a.slot);
    PKV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    kern<<<a.nwg, NT, lds, s>>>(a, c);
    PKV_HIP_CHECK(hipGetLastError());
    return PKV_OK;
}

template <int NT, int DT, bool WIDE>
static auto once_kernel_of(bool perm) { return perm ? quant_encode_once_kernel<NT, DT, WIDE, true> : quant_encode_once_kernel<NT, DT, WIDE, false>; }
template <int NT>
static auto once_kernel(int bits, int dtype, bool perm) {
    if (bits > 4) return dtype == PKV_F16 ? once_kernel_of<NT, PKV_F16, true>(perm) : once_kernel_of<NT, PKV_BF16, true>(perm);
    return dtype == PKV_F16 ? once_kernel_of<NT, PKV_F16, false>(perm) : once_kernel_of<NT, PKV_BF16, false>(perm);
}
// K and V, either of them without workgroups; widths on the same side of 4, with a token order both or neither.
template <int NT>
static int once_launch(const OnceSide &k, const OnceSide &v, int dtype, const EncodeClose &c, hipStream_t s) {
    auto kern = once_kernel<NT>(k.nwg ? k.W : v.W, dtype, (k.nwg ? k.perm : v.perm) != nullptr);
    const uint32_t lk = k.nwg ? once_lds(true, OnceRun<NT>::K, k.slot) : 0u, lv = v.nwg ? once_lds(false, OnceRun<NT>::V, v.slot) : 0u;
    const uint32_t lds = lk > lv ? lk : lv;
    PKV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    kern<<<k.nwg + v.nwg, NT, lds, s>>>(k, v, c);
    PKV_HIP_CHECK(hipGetLastError());
    return PKV_OK;
}

}  // namespace pkv
