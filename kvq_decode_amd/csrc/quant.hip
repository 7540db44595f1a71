// KIVI quantization of the paged KV cache for gfx950: bulk (prefill) and on-append
// (decode). No reference code exists for this (README.md:16 "not started"); the format
// follows the reference's byte model (src/bpt/roofline.py:6-9): asymmetric fp16 scale and
// zero, K per channel over groups of k_group tokens, V per token. Every code is bit-exact
// with the float32 specification; it and the arithmetic are in quant_math.h.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "kvq_internal.h"
#include "quant_math.h"

#pragma clang fp contract(off)

namespace kvq {

namespace {

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return min(max(v, lo), hi); }

// One store of 8 values' codes (4 or 8 bytes), aligned because code rows are 16-byte aligned.
// NT: the streaming policy, for the bulk quantizer, whose codes nothing reads back soon.
template <int FMT, bool NT = false>
__device__ __forceinline__ void store8(uint8_t* dst, const Codes8<FMT>& c) {
    if constexpr (FMT == KVQ_KV_INT4) {
        if constexpr (NT) __builtin_nontemporal_store(c.w[0], (uint32_t*)dst);
        else *(uint32_t*)dst = c.w[0];
    } else {
        const u2q w = {c.w[0], c.w[1]};
        if constexpr (NT) __builtin_nontemporal_store(w, (u2q*)dst);
        else *(u2q*)dst = w;
    }
}

// Physical block of page `page` of sequence b, or -1 when the block-table entry lies
// outside [0, num_blocks). The write paths neither read nor write a row whose page is
// outside the pool (the fp16 append skips such slots the same way), so a bad table entry
// cannot redirect codes or pairs into another sequence's block.
__device__ __forceinline__ int phys_of(const QuantParams& p, int b, int page) {
    const int e = p.bt[(int64_t)b * p.bt_sb + page];
    return (e >= 0 && e < p.num_blocks) ? e : -1;
}

// Tokens of sequence b the bulk quantizer covers: seq_lens[b], limited to the slots its
// block-table row addresses.
__device__ __forceinline__ int seq_len_of(const QuantParams& p, int b) {
    return clampi(p.seq_lens[b], 0, p.max_blocks * p.block_size);
}

// The append's sequence length: seq_lens[b] counts the new token, at position
// seq_lens[b] - 1. A length below 1 or past the block table's last slot has no slot for
// that token; the append then writes nothing for the sequence (-1).
__device__ __forceinline__ int append_len_of(const QuantParams& p, int b) {
    const int n = p.seq_lens[b];
    return (n >= 1 && n <= p.max_blocks * p.block_size) ? n : -1;
}

// Min / max over aligned lane groups without LDS (exact operations, so the order of the
// combination does not change the result): within a 16-lane row by DPP - quad_perm xor 1
// and xor 2; row_half_mirror, where each quad already holds its own result, so lane i
// meeting lane 7 - i combines the two quads of a half; row_ror:8 - and across rows by
// v_permlane16_swap / v_permlane32_swap (xor 16 / xor 32), whose two results are the lane's
// own value and its partner's.
template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, false));
}
template <int O>  // xor lane offset 1, 2, 4 (within 8-lane halves), 8, 16 or 32
__device__ __forceinline__ void minmax_xor(float& mn, float& mx) {
    if constexpr (O == 16 || O == 32) {
        const auto a = O == 16 ? __builtin_amdgcn_permlane16_swap(__float_as_uint(mn), __float_as_uint(mn), false, false)
                               : __builtin_amdgcn_permlane32_swap(__float_as_uint(mn), __float_as_uint(mn), false, false);
        const auto b = O == 16 ? __builtin_amdgcn_permlane16_swap(__float_as_uint(mx), __float_as_uint(mx), false, false)
                               : __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
        mn = fminf(__uint_as_float(a[0]), __uint_as_float(a[1]));
        mx = fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
    } else {
        constexpr int CTRL = O == 1 ? 0xB1 : O == 2 ? 0x4E : O == 4 ? 0x141 : 0x128;
        mn = fminf(mn, dpp<CTRL>(mn));
        mx = fmaxf(mx, dpp<CTRL>(mx));
    }
}

// Packed-half min / max of 8 channels across the lanes l ^ O, O = 8, 16 or 32 (v_pk_min_f16 /
// v_pk_max_f16 order +-0 and skip NaN as the f32 instructions do, on all pairs:
// tests/gpu_checks/quant_math_check.hip).
template <int O>
__device__ __forceinline__ h8q xor_lanes(h8q v, bool swap_hi) {
    u4q x = __builtin_bit_cast(u4q, v), y;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if constexpr (O == 8) {  // row_ror:8
            y[j] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x[j], 0x128, 0xf, 0xf, false);
        } else {
            const auto a = O == 16 ? __builtin_amdgcn_permlane16_swap(x[j], x[j], false, false)
                                   : __builtin_amdgcn_permlane32_swap(x[j], x[j], false, false);
            y[j] = swap_hi ? a[1] : a[0];
        }
    }
    return __builtin_bit_cast(h8q, y);
}
template <int O>
__device__ __forceinline__ void minmax8_xor(h8q& mn, h8q& mx) {
    if constexpr (O == 8) {
        mn = __builtin_elementwise_min(mn, xor_lanes<8>(mn, false));
        mx = __builtin_elementwise_max(mx, xor_lanes<8>(mx, false));
    } else {  // the swap's two results are the lane's own value and its partner's
        mn = __builtin_elementwise_min(xor_lanes<O>(mn, false), xor_lanes<O>(mn, true));
        mx = __builtin_elementwise_max(xor_lanes<O>(mx, false), xor_lanes<O>(mx, true));
    }
}

// Streaming 16-byte read of the fp16 source, which the quantizer reads once.
__device__ __forceinline__ h8q load_nt(const _Float16* src) {
    return __builtin_nontemporal_load((const h8q*)src);
}

// (scale, zero) pairs of 8 consecutive channels: two 16-byte stores.
__device__ __forceinline__ void store_pairs8(_Float16* dst, const ScaleZero* q) {
    *(u4q*)dst = u4q{q[0].sz, q[1].sz, q[2].sz, q[3].sz};
    *(u4q*)(dst + 8) = u4q{q[4].sz, q[5].sz, q[6].sz, q[7].sz};
}

// K groups of one wave (at head dim 256: of two, 128 channels each): the whole groups within
// kSmallSpan tokens, or one larger group.
constexpr int kSmallSpan = 64;
__host__ __device__ inline int k_groups_per_wave(int k_group) {
    return k_group <= kSmallSpan ? kSmallSpan / k_group : 1;
}

// K, bulk: one wave per (group, 128 channels of a kv head, sequence): the group's rows in
// slabs of 128, 8 chunks of 16 rows (a chunk lies in one page). A load instruction covers RPI
// whole rows (PC lanes of 16 bytes each): lane (ri, c) owns channels 8c .. 8c + 7 of rows
// RPI i + ri. A slab's rows stay in registers (KC loads in flight) between the min / max pass
// and the encode pass, so a group of up to 128 tokens reads its source once; longer groups
// re-read all but the last slab. Pages are wave-uniform: the slab's block-table entries are
// loaded once (lane j: chunk j's) and read back by v_readlane, and an address is a scalar
// base per chunk plus the lane's offset. Where a slab is cut short or a page lies outside the
// pool, the missing rows are replaced by rows of the group that count, which leave its min /
// max as they are, and are not written. Min / max run on packed halves, over the rows in
// registers and then across the RPI lanes that share channels: no LDS, no barrier. Row limits
// are compared with ri itself: RPI i + ri, kept in registers over the loops, would spill. Codes go
// to each token's page slot, the pairs to the group's first page; a group whose first page
// lies outside the pool could not be read back and writes nothing.
template <int FMT, int D>
__device__ __forceinline__ void quant_k_group(const QuantParams& p, int kvh, int grp, int half,
                                              int b) {
    constexpr int CW = D < 128 ? D : 128;  // channels of a wave
    constexpr int PC = CW / 8, RPI = 64 / PC, KC = 128 / RPI, CI = 16 / RPI;
    const int lane = threadIdx.x & 63, c = lane % PC, ri = lane / PC;
    const int n = seq_len_of(p, b);
    // the launch's spare waves first: their groups may start past 2^31
    if (grp >= p.max_groups) return;
    const int t0 = grp * p.k_group, t1 = (int)min((uint32_t)t0 + (uint32_t)p.k_group, (uint32_t)n);
    if (t0 >= t1) return;  // uniform over the wave
    const int last = t1 - t0 - 1;  // the group's last row
    const int bmask = p.block_size - 1;
    // lane j: the page of chunk j & 7 of the slab from row s0 on (-1: outside the pool)
    auto slab_pages = [&](int s0) {
        return phys_of(p, b, (t0 + min(s0 + 16 * (lane & 7), last)) >> p.bs_shift);
    };
    int pages = slab_pages(0);
    const int lead = __builtin_amdgcn_readlane(pages, 0);
    if (lead < 0) return;
    const int ch = half * CW + 8 * c;  // the lane's first channel
    const _Float16* src = p.k_src + (int64_t)kvh * p.s_sh + ch;
    const int64_t row_off = (int64_t)ri * p.s_stok;

    h8q rows[KC];
    auto fill = [&](int s0) {
        if (s0 + 127 <= last && __ballot(pages < 0) == 0) {  // a whole slab
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const _Float16* base = src + (int64_t)__builtin_amdgcn_readlane(pages, k) * p.s_sblk +
                                       (int64_t)((t0 + s0 + 16 * k) & bmask) * p.s_stok;
#pragma unroll
                for (int i = 0; i < CI; ++i) {
                    rows[CI * k + i] = load_nt(base + RPI * i * p.s_stok + row_off);
                    // one load's address registers at a time
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        } else {
            for (int k = 0; k < 8; ++k) {
                int ph = __builtin_amdgcn_readlane(pages, k), r0 = s0 + 16 * k;
                if (ph < 0 || r0 > last) {  // rows that count: the group's first chunk
                    ph = lead;
                    r0 = 0;
                }
                const _Float16* base = src + (int64_t)ph * p.s_sblk + (int64_t)((t0 + r0) & bmask) * p.s_stok;
#pragma unroll
                for (int kk = 0; kk < 8; ++kk) {
                    if (kk != k) continue;  // static register indices
#pragma unroll
                    for (int i = 0; i < CI; ++i)
                        rows[CI * kk + i] = load_nt(base + (int64_t)(RPI * i + min(ri, last - r0 - RPI * i)) * p.s_stok);
                }
            }
        }
    };
    const int last_slab = last / 128;
    h8q mn, mx;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        mn[e] = (_Float16)INFINITY;
        mx[e] = (_Float16)-INFINITY;
    }
    for (int s = 0;;) {
        fill(128 * s);
#pragma unroll
        for (int i = 0; i < KC; ++i) {
            mn = __builtin_elementwise_min(mn, rows[i]);
            mx = __builtin_elementwise_max(mx, rows[i]);
        }
        if (s == last_slab) break;
        pages = slab_pages(128 * ++s);
    }
    if constexpr (PC <= 8) minmax8_xor<8>(mn, mx);
    minmax8_xor<16>(mn, mx);
    minmax8_xor<32>(mn, mx);
    ScaleZero q[8];
    uint32_t live[2];
#pragma unroll
    for (int e = 0; e < 8; ++e) q[e] = make_params<FMT>((float)mn[e], (float)mx[e]);
    live_masks<FMT>(q, live);
    if (ri == 0) store_pairs8(p.k_scale + 2 * (((int64_t)lead * p.kv_heads + kvh) * D + ch), q);

    constexpr int CB = FMT == KVQ_KV_INT4 ? 4 : 8;  // code bytes per lane and row
    uint8_t* dst = p.k_codes + (int64_t)kvh * p.k_sh + ch / 8 * CB + (int64_t)ri * p.k_stok;
    for (int s = last_slab;;) {  // the slab in registers first
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int ph = __builtin_amdgcn_readlane(pages, k), r0 = 128 * s + 16 * k;
            if (ph < 0 || r0 > last) continue;  // uniform
            uint8_t* base = dst + (int64_t)ph * p.k_sblk + (int64_t)((t0 + r0) & bmask) * p.k_stok;
#pragma unroll
            for (int i = 0; i < CI; ++i) {
                const Codes8<FMT> w = encode8<FMT, 1>(rows[CI * k + i], q, live);
                if (ri <= last - r0 - RPI * i) store8<FMT, true>(base + RPI * i * p.k_stok, w);
            }
        }
        if (--s < 0) break;
        pages = slab_pages(128 * s);
        fill(128 * s);
    }
}

// K, bulk, groups of up to kSmallSpan tokens: one wave per (whole groups of that many tokens
// together, 128 channels of a kv head, sequence). The rows are loaded all at once, as
// quant_k_group's slab, and then group by group reduced and encoded from their registers. A chunk
// past the sequence or in a page outside the pool is skipped in every pass (uniform over the
// wave); the rows past the sequence in its last chunk are replaced by its last row and not
// written.
// Bound by HBM on large inputs, as the other groups (16 x 8192 tokens, 8 kv heads, D = 128, INT8,
// groups of 16: 172 us, of 128: 165), and else by the chain of loads, reductions and stores, which
// grows with the groups of a wave: 64 tokens and not 128, which halve the waves of a short batch
// and at D >= 128 spill 26 registers (64: four waves per SIMD without spills). 64 sequences of 10 to 577 tokens, D = 256, INT8,
// groups of 16: 65 us; one wave per group loading its 16 rows 74, eight groups one after the other
// on a wave, each with a slab's loads, 304.
template <int FMT, int D>
__device__ __forceinline__ void quant_k_small(const QuantParams& p, int kvh, int span, int half,
                                              int b) {
    constexpr int CW = D < 128 ? D : 128;  // channels of a wave
    constexpr int PC = CW / 8, RPI = 64 / PC, CI = 16 / RPI, NC = kSmallSpan / 16, KC = NC * CI;
    const int lane = threadIdx.x & 63, c = lane % PC, ri = lane / PC;
    const int n = seq_len_of(p, b);
    const int per = k_groups_per_wave(p.k_group), len = per * p.k_group, gc = p.k_group / 16;
    if ((int64_t)span * len >= n) return;  // uniform over the wave
    const int t0 = span * len, last = min(len, n - t0) - 1;  // the span's last row
    const int bmask = p.block_size - 1;
    // lane j: the page of chunk j % NC (-1: outside the pool, or no chunk of the span)
    int pages = phys_of(p, b, (t0 + min(16 * (lane % NC), last)) >> p.bs_shift);
    if (16 * (lane % NC) > last) pages = -1;
    const int ch = half * CW + 8 * c;  // the lane's first channel
    const _Float16* src = p.k_src + (int64_t)kvh * p.s_sh + ch;
    h8q rows[KC];
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        const int ph = __builtin_amdgcn_readlane(pages, k);
        if (ph < 0) continue;
        const _Float16* base = src + (int64_t)ph * p.s_sblk + (int64_t)((t0 + 16 * k) & bmask) * p.s_stok;
#pragma unroll
        for (int i = 0; i < CI; ++i)
            rows[CI * k + i] = load_nt(base + (int64_t)min(RPI * i + ri, last - 16 * k) * p.s_stok);
    }
    constexpr int CB = FMT == KVQ_KV_INT4 ? 4 : 8;  // code bytes per lane and row
    uint8_t* dst = p.k_codes + (int64_t)kvh * p.k_sh + ch / 8 * CB + (int64_t)ri * p.k_stok;
    for (int c0 = 0; 16 * c0 <= last; c0 += gc) {  // the group of chunks c0 .. c0 + gc - 1
        const int lead = __builtin_amdgcn_readlane(pages, c0);
        if (lead < 0) continue;
        h8q mn, mx;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            mn[e] = (_Float16)INFINITY;
            mx[e] = (_Float16)-INFINITY;
        }
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            if (k < c0 || k >= c0 + gc || __builtin_amdgcn_readlane(pages, k) < 0) continue;
#pragma unroll
            for (int i = 0; i < CI; ++i) {
                mn = __builtin_elementwise_min(mn, rows[CI * k + i]);
                mx = __builtin_elementwise_max(mx, rows[CI * k + i]);
            }
        }
        if constexpr (PC <= 8) minmax8_xor<8>(mn, mx);
        minmax8_xor<16>(mn, mx);
        minmax8_xor<32>(mn, mx);
        ScaleZero q[8];
        uint32_t live[2];
#pragma unroll
        for (int e = 0; e < 8; ++e) q[e] = make_params<FMT>((float)mn[e], (float)mx[e]);
        live_masks<FMT>(q, live);
        if (ri == 0) store_pairs8(p.k_scale + 2 * (((int64_t)lead * p.kv_heads + kvh) * D + ch), q);
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            const int ph = __builtin_amdgcn_readlane(pages, k);
            if (k < c0 || k >= c0 + gc || ph < 0) continue;
            uint8_t* base = dst + (int64_t)ph * p.k_sblk + (int64_t)((t0 + 16 * k) & bmask) * p.k_stok;
#pragma unroll
            for (int i = 0; i < CI; ++i) {
                const Codes8<FMT> w = encode8<FMT, 1>(rows[CI * k + i], q, live);
                if (RPI * i + ri <= last - 16 * k) store8<FMT, true>(base + RPI * i * p.k_stok, w);
            }
        }
    }
}

// V: one token row (D channels of one kv head) per D/8 lanes, each lane 8 channels. Bulk:
// kVIter row blocks of RPI = 512 / D rows per wave, all loads issued before the first row
// is encoded (16 blocks at D >= 128: as many bytes in flight as half a K slab, which the
// register file, sized for the K waves of the same launch, has room for); a block's pages (its own and its V group's first) are wave-uniform, read back
// from one block-table load as in quant_k_group. Min / max: packed over the lane's 8 values,
// then across the row's lanes by DPP. The codes go to the token's page slot, its (scale,
// zero) pair to index t % VG of its V group's first page (VG = 2^vg_shift tokens); a row is
// written only when both pages lie in the pool. The pairs of the wave's rows are gathered
// lane by lane (lane (g, i): row block i's row g) and stored by one instruction.
template <int D>
constexpr int kVIter = D == 64 ? 8 : 16;

// (scale, zero) of one row from the 8 values each of its D/8 lanes holds.
template <int FMT, int D>
__device__ __forceinline__ ScaleZero v_params(h8q v) {
    constexpr int LPR = D / 8;
    typedef _Float16 h4q __attribute__((ext_vector_type(4)));
    const h4q a = __builtin_shufflevector(v, v, 0, 1, 2, 3), b = __builtin_shufflevector(v, v, 4, 5, 6, 7);
    const h4q n4 = __builtin_elementwise_min(a, b), x4 = __builtin_elementwise_max(a, b);
    const h2q n2 = __builtin_elementwise_min(__builtin_shufflevector(n4, n4, 0, 1), __builtin_shufflevector(n4, n4, 2, 3));
    const h2q x2 = __builtin_elementwise_max(__builtin_shufflevector(x4, x4, 0, 1), __builtin_shufflevector(x4, x4, 2, 3));
    float mn = fminf((float)n2[0], (float)n2[1]), mx = fmaxf((float)x2[0], (float)x2[1]);
    // the row's LPR lanes (aligned lane groups of one wave)
    minmax_xor<1>(mn, mx);
    minmax_xor<2>(mn, mx);
    minmax_xor<4>(mn, mx);
    if constexpr (LPR >= 16) minmax_xor<8>(mn, mx);
    if constexpr (LPR >= 32) minmax_xor<16>(mn, mx);
    return make_params<FMT>(mn, mx);
}

template <int FMT, int D>
__device__ __forceinline__ void quant_v_tile(const QuantParams& p, int kvh, int tile, int b) {
    constexpr int LPR = D / 8, RPI = 64 / LPR, NI = kVIter<D>, ROWS = NI * RPI;
    const int lane = threadIdx.x & 63, c = lane % LPR, ri = lane / LPR;
    const int n = seq_len_of(p, b);
    if ((int64_t)tile * ROWS >= n) return;  // uniform over the wave
    const int r0 = tile * ROWS;             // the wave's first row
    const int last = min(ROWS, n - r0) - 1, last_blk = last / RPI;
    const int bmask = p.block_size - 1, vg = 1 << p.vg_shift;
    // lane j: page pg0 + j, pg0 the first page of the first row's V group
    const int pg0 = (r0 >> p.vg_shift) << (p.vg_shift - p.bs_shift);
    const int pages = phys_of(p, b, min(pg0 + lane, (r0 + last) >> p.bs_shift));
    const _Float16* src = p.v_src + (int64_t)kvh * p.s_sh + 8 * c;
    int phys[NI], vlead[NI];
    h8q rows[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int t = r0 + RPI * i;  // first row of the block
        phys[i] = __builtin_amdgcn_readlane(pages, (t >> p.bs_shift) - pg0);
        vlead[i] = __builtin_amdgcn_readlane(
            pages, ((t >> p.vg_shift) << (p.vg_shift - p.bs_shift)) - pg0);
        if (i > last_blk || vlead[i] < 0) phys[i] = -1;
        if (phys[i] >= 0) {  // uniform
            const int row = min(ri, last - RPI * i);
            rows[i] = load_nt(src + (int64_t)phys[i] * p.s_sblk +
                              (int64_t)(t & bmask) * p.s_stok + (int64_t)row * p.s_stok);
        }
    }
    constexpr int CB = FMT == KVQ_KV_INT4 ? 4 : 8;
    uint8_t* dst = p.v_codes + (int64_t)kvh * p.v_sh + CB * c + (int64_t)ri * p.v_stok;
    uint32_t pair = 0;
    int64_t pair_at = -1;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        if (phys[i] < 0) continue;  // uniform
        const int t = r0 + RPI * i;
        const ScaleZero q = v_params<FMT, D>(rows[i]);
        const uint32_t live = q.flat() ? 0u : ~0u;
        const Codes8<FMT> w = encode8<FMT, 0>(rows[i], &q, &live);
        const bool mine = ri <= last - RPI * i;
        uint8_t* row = dst + (int64_t)phys[i] * p.v_sblk + (int64_t)(t & bmask) * p.v_stok;
        if (mine) store8<FMT, true>(row, w);
        if (c == i && mine) {  // c < D/8, at least NI lanes a row
            pair = q.sz;
            pair_at = (((int64_t)vlead[i] * p.kv_heads + kvh) << p.vg_shift) + ((t + ri) & (vg - 1));
        }
    }
    if (pair_at >= 0) *(uint32_t*)(p.v_scale + 2 * pair_at) = pair;
}

// The newest token's V row (append), on the D/8 lanes c of one wave.
template <int FMT, int D>
__device__ __forceinline__ void quant_v_append(const QuantParams& p, int kvh, int b, int c) {
    const h8q v = *(const h8q*)(p.v_new + ((int64_t)b * p.kv_heads + kvh) * D + 8 * c);
    const int n = append_len_of(p, b);
    if (n < 1) return;
    // the barrier of quant_k_append, met here after the same first round trip (a sequence
    // without a slot returns before it in both roles)
    asm volatile("" ::"s"(n) : "memory");
    __builtin_amdgcn_s_barrier();
    const int t = n - 1;
    const int phys = phys_of(p, b, t >> p.bs_shift);
    const int vlead = phys_of(p, b, (t >> p.vg_shift) << (p.vg_shift - p.bs_shift));
    if (phys < 0 || vlead < 0) return;
    const ScaleZero q = v_params<FMT, D>(v);
    const uint32_t live = q.flat() ? 0u : ~0u;
    constexpr int CB = FMT == KVQ_KV_INT4 ? 4 : 8;
    store8<FMT>(p.v_codes + (int64_t)phys * p.v_sblk + (int64_t)(t & (p.block_size - 1)) * p.v_stok +
                    (int64_t)kvh * p.v_sh + CB * c,
                encode8<FMT, 0>(v, &q, &live));
    if (c == 0) {
        const int64_t sz = (((int64_t)vlead * p.kv_heads + kvh) << p.vg_shift) +
                           (t & ((1 << p.vg_shift) - 1));
        *(uint32_t*)(p.v_scale + 2 * sz) = q.sz;
    }
}

// Codes of one K row's 8 channels 8c .. 8c + 7 under (scale, zero) q, into the row's slot.
template <int FMT>
__device__ __forceinline__ void emit_k_row(const QuantParams& p, int kvh, int c, int t,
                                           int phys, h8q v, const ScaleZero* q,
                                           const uint32_t* live) {
    constexpr int CB = FMT == KVQ_KV_INT4 ? 4 : 8;
    store8<FMT>(p.k_codes + (int64_t)phys * p.k_sblk + (int64_t)(t & (p.block_size - 1)) * p.k_stok +
                    (int64_t)kvh * p.k_sh + CB * c,
                encode8<FMT, 1>(v, q, live));
}

// Append, K: the group holding the newest token (position n - 1, row r = (n - 1) % k_group
// of the group that starts at t0). The residual [B][Hkv][k_group + 2][D] keeps the
// group's fp16 rows and, in rows k_group and k_group + 1, their running per-channel min
// and max (exact in fp16: min / max of fp16 values). Four waves; lane (c, slice) owns
// channels 8c .. 8c + 7; every lane loads the new row and its channels' stored min / max
// together with the sequence length (none of them depends on it), so the group's new
// (scale, zero) pairs are known one memory round trip in (r == 0 starts the group from the new
// row alone). The new row is encoded with them. The group's earlier rows are re-encoded only
// in the 8-channel slices whose min or max moved (a code depends on its row and its channel's
// pair only): a token moves a channel's range with probability 2 / (r + 1), so 16 r slices
// move early in a group and about 2 of its 16 late. The moved slices' parameters are packed
// through LDS, per wave, and the 256 lanes take (row, moved slice) items, so that no lane
// idles beside a slice that did not move. Measured over the 128 appends of a group (64
// sequences, 8 kv heads, INT8): 5.3 us, against 7.6 with each slice's own 16 lanes re-encoding
// it, up to 8 rows each, and V in workgroups of its own (10.8 with the earlier encoder). What
// is left is the launch and two dependent memory round trips. The slice's first lane writes
// the pairs (when they moved), the min / max rows and the new residual row. A group whose
// first page lies outside the pool writes nothing; rows whose page lies outside are not
// written. Appends are sequential: the residual holds rows 0 .. r - 1 of the group and their
// min / max (from the appends of positions t0 .. n - 2, or from init_k_residual).
constexpr int kAppendWaves = 4;  // of the K role

template <int FMT, int D>
__device__ __forceinline__ void quant_k_append(const QuantParams& p, int kvh, int b) {
    constexpr int LPR = D / 8, THREADS = 64 * kAppendWaves, CACHE = 4;
    // a wave's moved slices: 8 parameters each, and the slice's index
    __shared__ __attribute__((aligned(16))) ScaleZero sm_q[kAppendWaves][LPR][8];
    __shared__ int sm_c[kAppendWaves][LPR];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = threadIdx.x % LPR;
    const int64_t head = (int64_t)b * p.kv_heads + kvh;
    _Float16* res = p.k_resid + head * (p.k_group + 2) * D;
    const h8q kn = *(const h8q*)(p.k_new + head * D + 8 * c);
    const h8q smn = *(const h8q*)(res + (int64_t)p.k_group * D + 8 * c);
    const h8q smx = *(const h8q*)(res + (int64_t)(p.k_group + 1) * D + 8 * c);
    const int n = append_len_of(p, b);
    if (n < 1) return;
    const int t0 = ((n - 1) / p.k_group) * p.k_group, r = n - 1 - t0;
    const int lead = phys_of(p, b, t0 >> p.bs_shift);
    const int phys_new = phys_of(p, b, (n - 1) >> p.bs_shift);
    float mn[8], mx[8];
    bool moved = r == 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float x = (float)kn[e];
        const float omn = r == 0 ? INFINITY : (float)smn[e];
        const float omx = r == 0 ? -INFINITY : (float)smx[e];
        mn[e] = fminf(omn, x);
        mx[e] = fmaxf(omx, x);
        moved = moved || mn[e] != omn || mx[e] != omx;
    }
    ScaleZero q[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) q[e] = make_params<FMT>(mn[e], mx[e]);
    // slices c of the wave's first LPR lanes (the other lanes repeat them)
    const uint64_t mask = __ballot(moved) & (~0ull >> (64 - LPR));
    const int nm = __popcll(mask);
    // every wave has read the stored min / max (the mask follows from them) before one of them
    // writes the new ones: a wave that read those would take no slice for moved
    asm volatile("" ::"s"(mask) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (nm > 0 && r > 0) {  // uniform: re-encode rows 0 .. r - 1 of the moved slices
        if (lane < LPR && moved) {
            const int at = __popcll(mask & ((1ull << lane) - 1));
#pragma unroll
            for (int e = 0; e < 8; ++e) sm_q[wave][at][e] = q[e];
            sm_c[wave][at] = c;
        }
        __builtin_amdgcn_wave_barrier();  // the wave's LDS operations run in order
        // item (row, slice): slices in the lane index's low bits, rounded to a power of two
        const int sh = nm > 1 ? 32 - __builtin_clz(nm - 1) : 0, item = threadIdx.x & ((1 << sh) - 1);
        const int row0 = threadIdx.x >> sh, step = THREADS >> sh;
        if (item < nm) {
            const int mc = sm_c[wave][item];
            for (int base = row0; base < r; base += step * CACHE) {
                h8q rows[CACHE];
                int ph[CACHE];
#pragma unroll
                for (int i = 0; i < CACHE; ++i) {  // loads first, at clamped rows
                    const int t = min(base + i * step, r - 1);
                    ph[i] = phys_of(p, b, (t0 + t) >> p.bs_shift);
                    rows[i] = *(const h8q*)(res + (int64_t)t * D + 8 * mc);
                }
                if (lead < 0) break;
                ScaleZero mq[8];
                uint32_t live[2];
#pragma unroll
                for (int e = 0; e < 8; ++e) mq[e] = sm_q[wave][item][e];
                live_masks<FMT>(mq, live);
#pragma unroll
                for (int i = 0; i < CACHE; ++i) {
                    const int t = base + i * step;
                    if (t < r && ph[i] >= 0)
                        emit_k_row<FMT>(p, kvh, mc, t0 + t, ph[i], rows[i], mq, live);
                }
            }
        }
    }
    if (threadIdx.x < LPR && lead >= 0) {
        uint32_t live[2];
        live_masks<FMT>(q, live);
        if (phys_new >= 0) emit_k_row<FMT>(p, kvh, c, n - 1, phys_new, kn, q, live);
        h8q nmn, nmx;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            nmn[e] = (_Float16)mn[e];
            nmx[e] = (_Float16)mx[e];
        }
        *(h8q*)(res + (int64_t)r * D + 8 * c) = kn;
        *(h8q*)(res + (int64_t)p.k_group * D + 8 * c) = nmn;
        *(h8q*)(res + (int64_t)(p.k_group + 1) * D + 8 * c) = nmx;
        if (moved)  // (scale, zero) pairs of channels 8c .. 8c + 7, in the group's first page
            store_pairs8(p.k_scale + 2 * (((int64_t)lead * p.kv_heads + kvh) * D + 8 * c), q);
    }
}

// Bulk, one launch: the K groups and the V row tiles of every (kv head, sequence), in 4-wave
// workgroups; per (kv head, sequence) kb K and vb V workgroups, alternating through the grid
// (of every kb + vb consecutive, kb are K), so that both kinds are in flight together and the
// launch has one tail. Groups and tiles past a sequence's end return at once. The kv heads of
// one tile run on one XCD (workgroup i runs on XCD i % 8): their source rows are adjacent in
// the token-major cache.
//
// Bound by HBM, reads and writes mixed: without the arithmetic it takes 96 to 98% of the
// time, and FP8 moves 4.9 TB/s where a plain copy moves 4.8. Measured (us per call, 8 kv
// heads, D = 128): INT4, 8 sequences of 1000 to 16400 tokens, 128.5 -> 78.3; FP8, 16 x 8192,
// 218.4 -> 163.0, against two kernels (K, then V) at about 20 VALU instructions per value. Of
// that, with the arithmetic above: one launch 98.6 / 186.6; 3 waves per SIMD (168 VGPRs, 172
// without the attribute) 88.8 / 181.9; streaming stores 86.9 / 173.2; 16 V row blocks per wave
// instead of 8 83.9 / 172.5 (32: 90.7); the XCD order 83.4 / 166.1; fewer registers (s and z
// in one) 82.5 / 164.5, (row limits, no loop over groups) 79.1 / 163.0. 4 waves per SIMD spill
// (126.9 / 256.1). All V workgroups after the K ones: 86.2 / 165.8.
//
// SMALL: K groups of up to kSmallSpan tokens, a kernel of its own for its registers.
template <int FMT, int D, bool SMALL>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3)))
void quant_bulk_kernel(const QuantParams p, int kb, int vb) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int b = blockIdx.y, nb = kb + vb, whole = nb / 8 * 8;
    int kvh, j;  // the j-th workgroup of (kvh, b)
    if ((int)blockIdx.x < whole * p.kv_heads) {
        kvh = blockIdx.x / 8 % p.kv_heads;
        j = blockIdx.x / 8 / p.kv_heads * 8 + blockIdx.x % 8;
    } else {
        const int i = blockIdx.x - whole * p.kv_heads;
        kvh = i % p.kv_heads;
        j = whole + i / p.kv_heads;
    }
    const int k0 = (int)((int64_t)j * kb / nb), k1 = (int)((int64_t)(j + 1) * kb / nb);
    if (k1 > k0) {
        constexpr int PER = D > 128 ? D / 128 : 1;  // waves per group or span
        const int w = 4 * k0 + wave;
        if constexpr (SMALL) quant_k_small<FMT, D>(p, kvh, w / PER, w % PER, b);
        else quant_k_group<FMT, D>(p, kvh, w / PER, w % PER, b);
    } else {
        quant_v_tile<FMT, D>(p, kvh, 4 * (j - k0) + wave, b);
    }
}

// Append in one launch: workgroup (kv head, sequence); its first four waves re-quantize the
// K group holding the newest token, the first D/8 lanes of the fifth quantize the newest V
// row. The two roles write disjoint memory (K codes, pairs and residual; V codes and pairs).
template <int FMT, int D>
__global__ __launch_bounds__(64 * (kAppendWaves + 1)) void quant_append_kernel(const QuantParams p) {
    // a scalar branch: the roles' barriers are met by whole waves
    if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) < kAppendWaves) {
        quant_k_append<FMT, D>(p, blockIdx.x, blockIdx.y);
    } else if (threadIdx.x < 64 * kAppendWaves + D / 8) {
        quant_v_append<FMT, D>(p, blockIdx.x, blockIdx.y, threadIdx.x - 64 * kAppendWaves);
    }
}

template <int FMT, int D, bool APPEND>
hipError_t launch_fmt_d(const QuantParams& p, hipStream_t stream) {
    if (APPEND) {
        hipLaunchKernelGGL((quant_append_kernel<FMT, D>), dim3(p.kv_heads, p.batch),
                           dim3(64 * (kAppendWaves + 1)), 0, stream, p);
        return hipGetLastError();
    }
    constexpr int PER = D > 128 ? D / 128 : 1, VROWS = 4 * kVIter<D> * (512 / D);
    const int per = k_groups_per_wave(p.k_group);
    const int kb = (PER * ((p.max_groups + per - 1) / per) + 3) / 4;
    const int vb = (int)(((int64_t)p.max_blocks * p.block_size + VROWS - 1) / VROWS);
    if (int64_t(p.kv_heads) * (int64_t(kb) + vb) > INT32_MAX) return hipErrorInvalidConfiguration;
    const auto kernel = p.k_group <= kSmallSpan ? quant_bulk_kernel<FMT, D, true> : quant_bulk_kernel<FMT, D, false>;
    hipLaunchKernelGGL(kernel, dim3(p.kv_heads * (kb + vb), p.batch), dim3(256), 0, stream, p, kb, vb);
    return hipGetLastError();
}

template <int FMT, bool APPEND>
hipError_t launch_fmt(const QuantParams& p, hipStream_t stream) {
    switch (p.head_dim) {  // the quantized formats' head dims (decode reads these)
        case 64: return launch_fmt_d<FMT, 64, APPEND>(p, stream);
        case 128: return launch_fmt_d<FMT, 128, APPEND>(p, stream);
        case 256: return launch_fmt_d<FMT, 256, APPEND>(p, stream);
        default: return hipErrorInvalidValue;
    }
}

template <bool APPEND>
hipError_t launch_any(const QuantParams& p, int kv_format, hipStream_t stream) {
    switch (kv_format) {
        case KVQ_KV_INT8: return launch_fmt<KVQ_KV_INT8, APPEND>(p, stream);
        case KVQ_KV_FP8_E4M3: return launch_fmt<KVQ_KV_FP8_E4M3, APPEND>(p, stream);
        case KVQ_KV_INT4: return launch_fmt<KVQ_KV_INT4, APPEND>(p, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

hipError_t launch_quantize_cache(const QuantParams& p, int kv_format, hipStream_t stream) {
    return launch_any<false>(p, kv_format, stream);
}

hipError_t launch_quantize_append(const QuantParams& p, int kv_format, hipStream_t stream) {
    return launch_any<true>(p, kv_format, stream);
}

}  // namespace kvq
