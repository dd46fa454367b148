// Block-sparse attention for few query rows against a long K/V ("decode") on gfx950 (MI355X).
//
// Same function as the forward (sparse_attention with BLOCK_Q = Sq, sparseattention/sparse_attn_kernel.py:74-146,
// :10-63) for Sq <= 32: there is one Q tile per (b, h), so the forward's one-workgroup-per-Q-tile launch would
// leave the device empty and walk each list serially.  Here the list of a (b, h) is cut into `nsplit` ranges of
// 32-key chunks, one workgroup each; inside a workgroup the four waves take chunks in turn, every wave with a
// K/V stream of its own (no barrier in the loop) and its own online-softmax state for all query rows; waves, then
// workgroups, are merged by the usual rescaling.  The kernel is HBM-bound: every K and V byte of an executed tile is
// read once, 2 flop per byte and query row.
//
// Per chunk of 32 keys a wave
//   * holds K as MFMA operand (lane = key, 8 x 16 bytes of its row half; the contraction order is permuted the same way in Q, which
//     costs nothing), from whole rows after a way through LDS or, where decode_key_rows says so, straight from global memory,
//   * receives V in its own LDS stage by direct loads (swizzled rows, transposing reads: fwd_common.h),
//   * computes S^T = K . Q^T (32 keys x 32 query rows, rows past Sq are padding), masks PARTIAL tiles from the bool
//     mask, updates the lagging reference value, P = exp2(S^T - m), O^T += V^T . P^T, row sums by a small MFMA,
// while the loads of its next chunk (and the list index of the one after) are in flight.
#include "fwd_common.h"

namespace sa {

namespace {

constexpr int kDecodeWaves = 4;

// Where K comes as whole rows.  Two workgroups with the 16 rows that this takes of each wave's share have all of a compute unit's LDS,
// none is left for lists made in the kernel.  us, K per lane | as rows, K and V not in a cache (a call's own are a layer's of many):
//   D = 128  B1 H32 Sk8192 Sq1 36.5 | 33.1  Sq8 38.3 | 34.4   B4 H16 Sk8192 Sq1 50.6 | 48.0   B4 H16 Sk32768 Sq1 165.8 | 163.1
//            B8 H32 Sk32768 Sq1 647 | 624 (6.9 TB/s; a linear streaming read runs at 7.1)   B8 H16 Sk16384 Sq16 gathered 90.3 | 83.6
//   D = 64   B1 H32 Sk2048 Sq8 13.5 | 11.9   B4 H16 Sk32768 Sq1 90.3 | 85.9   Sq32 97.3 | 93.3
// and nowhere slower but at BLOCK_K = 16 (B8 H32 Sk4096 Sq1 87.7 | 90.2), whose rows come from two places.
// Called again and again on the same K and V, which nothing else has pushed out, K per lane is faster up to 512 MiB of them (D = 128, Sq1,
// per lane | rows; behind it the same call on K and V from a rotation of 1.5 GiB): B1 H32 Sk2048 14.1 | 14.6 (16.0 | 15.9),
// B4 H16 Sk8192 45.8 | 47.9 (51.8 | 50.2), B8 H32 Sk2048 45.8 | 48.0 (51.0 | 49.4), Sk4096 83.1 | 90.2 (93.8 | 91.4), Sk8192 174 |
// 170 (176.6 | 173): loads with the streaming hint find less of what the last call left.  A program's layers have K and V of
// their own, so the rule goes by the rotation.
constexpr bool decode_key_rows(bool b16, bool dm) { return !b16 && !dm; }

template <int D, bool KR>
constexpr int decode_smem_bytes() {
    // per wave two V stages of 32 rows and, where K comes as whole rows, 16 rows of it
    constexpr int stream = kDecodeWaves * (2 * 32 + (KR ? 16 : 0)) * D * 2;
    constexpr int merge = kDecodeWaves * 32 * (D + 2) * 4 + 16;   // per wave 32 rows of D + 2 floats; the parts of a plane
    static_assert(kDecodeMergeRows <= kDecodeWaves * 32, "LDS holds the parts that the last workgroup merges");
    static_assert(kDecodeMergeFew <= kArrivalMost, "a plane's workgroups have place in its count");
    return stream > merge ? stream : merge;
}

// Merge of partial rows: `n` parts of (D values, reference value m, row sum l) at `part + i * stride` floats; this
// thread owns NV consecutive values starting at d0.  Returns the merged reference value and sum, values in out[].
template <int NV>
__device__ __forceinline__ void merge_parts(const float *part, int n, int64_t stride, int D, int d0, float (&out)[NV],
                                            float &M, float &L) {
    M = kNegInf;
    for (int i = 0; i < n; i++) M = fmaxf(M, part[i * stride + D]);
    L = 0.f;
#pragma unroll
    for (int j = 0; j < NV; j++) out[j] = 0.f;
    if (M == kNegInf) return;  // no part saw an attended key
    for (int i = 0; i < n; i++) {
        const float *pp = part + i * stride;
        const float w = __builtin_amdgcn_exp2f(pp[D] - M);  // 0 for parts without an attended key (m = -inf)
        L += w * pp[D + 1];
#pragma unroll
        for (int j = 0; j < NV; j++) out[j] += w * pp[d0 + j];
    }
}

// DM: the workgroup's own lists, behind the V stages: a bit per mask entry, then FULL and PARTIAL tiles (16 bit each).
constexpr int kDirectBits = kDecodeDirectEntries / 8;
constexpr int kDirectList = kDecodeDirectEntries / 32;  // entries of one list at most
constexpr int kDirectBytes = kDirectBits + 2 * 2 * kDirectList;

// The byte of a bool mask as a bit: bits 0..3 for the four bytes of w (any non-zero byte attends).
__device__ __forceinline__ uint32_t bits_of4(uint32_t w) {
    w |= w >> 4;
    w |= w >> 2;
    w |= w >> 1;
    return ((w & 0x01010101u) * 0x01020408u >> 24) & 15u;
}

// PK: the mask entries of PARTIAL tiles come bit-packed from p.packed (sa_mask_pack_partial with BQ = Sq) instead of from
// the bool mask.  B16: BLOCK_K = 16, two list entries per chunk of 32 keys (else BLOCK_K >= 32, BLOCK_K/32 chunks per
// entry).  DM: no lists given; every workgroup reads the plane's mask (at most kDecodeDirectEntries bytes, mostly from a
// cache) and makes the lists that the classification would have made in LDS, in the same order: results are bit-identical.
// One launch instead of two where both are mostly latency, and three allocations less: with the lists made first / here, bf16,
// D = 128, three quarters of the keys attended: B4 H32 Sq1 Sk2048 28.0 / 24.1 us, B1 H8 Sq1 Sk512 12.5 / 10.3, at the bound
// B8 H32 Sq1 Sk32768 496 / 477, B8 H16 Sq32 Sk1024 26.3 / 25.1; nowhere slower than the runs differ.
template <int DT, int D, bool PK, bool B16, bool DM>
__global__ __launch_bounds__(kDecodeWaves * 64, 2) void sparse_decode_kernel(const DecodeParams p) {
    using E = Elem<DT>;
    constexpr int ROWB = D * 2;
    constexpr int VBUF = 32 * ROWB;   // one chunk of V
    constexpr int RPI = 1024 / ROWB;  // rows written by one wave-wide direct load
    constexpr int NLD = 32 / RPI;     // direct loads per chunk
    constexpr int PPR = ROWB / 16;
    constexpr int NC = D / 16, NDB = D / 32;
    constexpr bool KR = decode_key_rows(B16, DM);  // K comes as whole rows
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l32 = lane & 31, hh = lane >> 5;
    const int bh = (int)(blockIdx.x / (unsigned)p.nsplit), split = (int)(blockIdx.x - (unsigned)bh * (unsigned)p.nsplit);
    const int b = bh / p.H, h = bh - b * p.H;

    // query row of this lane (rows past Sq are padding: zero queries, row 0's mask, never stored)
    const bool live = l32 < p.Sq;
    const int qrow = live ? l32 : 0;
    // Q^T operand: lane (l32, hh) keeps d = (D/2) hh + 8c .. +7 of its row for step c (K uses the same order, so each lane's K
    // bytes are contiguous).  Requested first of all, with the counts or the mask, and scaled once behind the requests for the first chunk:
    // requested and scaled in front of them it was a memory round trip of its own (B4 H32 Sq1 Sk2048 with a new mask 22.6 -> 21.8 us a
    // call, B8 H16 Sq16 Sk16384 gathered 90.5 -> 89.4).
    u32x4 qf[NC];
    {
        const uint16_t *qp = p.q + b * p.qs[0] + h * p.qs[1] + (int64_t)qrow * p.qs[2] + (D / 2) * hh;
#pragma unroll
        for (int c = 0; c < NC; c++) qf[c] = *(const u32x4 *)(qp + 8 * c);
    }

    const uint16_t *kbase = p.k + b * p.ks[0] + h * p.ks[1];
    const uint16_t *vbase = p.v + b * p.vs[0] + h * p.vs[1];
    const int32_t *fid = DM ? nullptr : p.full_ids + b * p.fis[0] + h * p.fis[1];
    const int32_t *pid = DM ? nullptr : p.part_ids + b * p.pis[0] + h * p.pis[1];
    // Counts and tile indices are clamped to what Sk holds (the reference guards every K/V and mask load with
    // kv_offset < SEQLEN_K, sparse_attn_kernel.py:35,39,60): stale or foreign metadata then gives wrong numbers, never
    // an access outside K, V or the mask.
    const int nKt = p.Sk >> p.lbk;
    int F = DM ? 0 : min(max(p.full_lens[b * p.fls[0] + h * p.fls[1]], 0), nKt);
    int NE = DM ? 0 : F + min(max(p.part_lens[b * p.pls[0] + h * p.pls[1]], 0), nKt - F);
    const int nCh = p.Sk >> 5;  // (DM) chunks of a row
    uint32_t *const bits = reinterpret_cast<uint32_t *>(smem + decode_smem_bytes<D, KR>());  // (DM) [Sq][nCh]
    uint16_t *const list = reinterpret_cast<uint16_t *>(smem + decode_smem_bytes<D, KR>() + kDirectBits);  // FULL, then PARTIAL
    if constexpr (DM) {
        const uint8_t *m0 = p.mask + b * p.ms[0] + h * p.ms[1];
        const int ppr = 2 * nCh, pieces = p.Sq * ppr;  // of 16 entries
        for (int i0 = tid; i0 < pieces; i0 += 4 * 256) {
            u32x4 x[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int i = min(i0 + 256 * j, pieces - 1), r = i / ppr;
                x[j] = *(const u32x4 *)(m0 + r * p.ms[2] + 16 * (i - r * ppr));
            }
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (i0 + 256 * j < pieces)
                    reinterpret_cast<uint16_t *>(bits)[i0 + 256 * j] = (uint16_t)(bits_of4(x[j].x) | (bits_of4(x[j].y) << 4) |
                                                                                  (bits_of4(x[j].z) << 8) | (bits_of4(x[j].w) << 12));
        }
        __syncthreads();
        // a lane per tile; every wave counts, the first one writes
        const int words = p.BK >> 5;  // of a row of a tile
        int P = 0;
        for (int c0 = 0; c0 < nKt; c0 += 64) {
            const int c = c0 + lane;
            uint32_t any = 0u, all = ~0u;
            if (c < nKt)
                for (int r = 0; r < p.Sq; r++)
                    for (int w = 0; w < words; w++) {
                        const uint32_t x = bits[r * nCh + c * words + w];
                        any |= x;
                        all &= x;
                    }
            const bool is_part = any != 0u && all != ~0u, is_full = any != 0u && !is_part;
            const uint64_t full = __builtin_amdgcn_ballot_w64(is_full), part = __builtin_amdgcn_ballot_w64(is_part);
            const uint64_t below = (1ull << lane) - 1ull;
            if (wave == 0 && is_full) list[F + __popcll(full & below)] = (uint16_t)c;
            if (wave == 0 && is_part) list[kDirectList + P + __popcll(part & below)] = (uint16_t)c;
            F += __popcll(full);
            P += __popcll(part);
        }
        NE = F + P;
        __syncthreads();
    }
    constexpr int EPC = B16 ? 2 : 1;   // list entries per chunk
    const int sh = B16 ? 0 : p.lbk - 5;  // chunks per list entry, log2
    const int T = B16 ? (NE + 1) >> 1 : NE << sh;
    // this workgroup's chunks [t_lo, t_hi); this wave takes t_lo + wave, + 4, ...
    const int t_lo = (int)((unsigned)T * (unsigned)split / (unsigned)p.nsplit),
              t_hi = (int)((unsigned)T * (unsigned)(split + 1) / (unsigned)p.nsplit);  // T * nsplit < 2^31 (checked by the caller)
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);

    const uint8_t *mrow = PK || DM ? nullptr : p.mask + b * p.ms[0] + h * p.ms[1] + (int64_t)qrow * p.ms[2];
    // this row's bits in the packed tile of a PARTIAL slot: BK/8 bytes per row, Sq rows per tile
    const int64_t tile_bytes = (int64_t)p.Sq * (p.BK >> 3);
    const uint8_t *prow = PK ? p.packed + b * p.pks[0] + h * p.pks[1] + (int64_t)qrow * (p.BK >> 3) : nullptr;


    // online-softmax state of this lane's query row (see sparse_fwd_kernel.h); scores start from 0 here and the
    // reference value is subtracted before the exponential
    float m_ref = 0.f;
    float raise_above = -3.0e38f;
    f32x4 acc_l = {0.f, 0.f, 0.f, 0.f};
    const uint32_t sel1 = (((lane >> 4) ^ lane) & 1) == 0 ? E::ones4().x : 0u;
    const u32x4 sum_sel = {sel1, sel1, sel1, sel1};
    f32x16 acc[NDB];
#pragma unroll
    for (int db = 0; db < NDB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[db][i] = 0.f;

    // V: transposing-read offsets and direct-load source offsets, as in sparse_fwd_kernel.h with one wave per chunk
    int voff[NDB];
    {
        const int tr_row = 4 * hh + ((lane & 15) >> 2);
        const int x = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
        const int sw = v_swizzle<D>(tr_row) >> 2;
#pragma unroll
        for (int db = 0; db < NDB; db++) voff[db] = tr_row * ROWB + 64 * (db ^ sw) + 16 * x + 8 * (lane & 1);
    }
    const int ld_r0 = lane / PPR, ld_slot = lane % PPR;
    uint32_t ld_voff[NLD];
#pragma unroll
    for (int i = 0; i < NLD; i++) {
        const int r = RPI * i + ld_r0;
        ld_voff[i] = (uint32_t)((r * p.vs[2] + 8 * (ld_slot ^ v_swizzle<D>(r))) * 2);
    }
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const SA_LDS uint8_t *)smem);
    uint8_t *const vmine = smem + wave_u * 2 * VBUF;
    const uint32_t vmine_lds = lds0 + wave_u * 2 * VBUF;
    // KR: K is read as whole rows like V, 1 KiB per wave instruction, so that its loads can carry the streaming hint too (a lane
    // that reads its own key's row takes 16 bytes of a line at a time, and with the hint the line is gone after the first ones), and
    // crosses the lanes through 16 rows of LDS: the same operand, so results are bit-identical (decode_key_rows).
    uint8_t *const kmine = smem + kDecodeWaves * 2 * VBUF + wave_u * 16 * ROWB;
    const int64_t kr_lane = (int64_t)ld_r0 * p.ks[2] + 8 * ld_slot;

    // list entries of chunk t (clamped into the row of tiles; an entry past the count reads as entry 0 and is masked out)
    auto idx_load = [&](int t, int(&idx)[EPC]) {
        if constexpr (DM) {
            const int e = t >> sh;
            idx[0] = list[e < F ? e : kDirectList + e - F];
            return;
        }
#pragma unroll
        for (int j = 0; j < EPC; j++) {
            const int e0 = B16 ? 2 * t + j : (t >> sh);
            const int e = e0 < NE ? e0 : 0;
            const int v = e < F ? fid[(int64_t)e * p.fis[2]] : pid[(int64_t)(e - F) * p.pis[2]];
            idx[j] = min(max(v, 0), nKt - 1);
        }
    };
    // first key column of every entry of chunk t
    auto cols_of = [&](int t, const int(&idx)[EPC], int(&col)[EPC]) {
#pragma unroll
        for (int j = 0; j < EPC; j++)
            col[j] = (__builtin_amdgcn_readfirstlane(idx[j]) << p.lbk) + (B16 ? 0 : ((t & ((1 << sh) - 1)) << 5));
    };
    // what chunk t's entries are: bit j = entry j exists, bit 4 + j = it is PARTIAL
    auto flags_of = [&](int t) -> unsigned {
        unsigned f = 0u;
#pragma unroll
        for (int j = 0; j < EPC; j++) {
            const int e = B16 ? 2 * t + j : (t >> sh);
            if (e < NE) f |= (1u << j) | (e >= F ? (16u << j) : 0u);
        }
        return f;
    };
    constexpr unsigned ALL = (1u << EPC) - 1u;
    constexpr int NMW = PK || DM ? EPC : 4;  // mask words per lane and chunk
    // everything chunk t needs from memory: K into registers, V into LDS stage `st`, mask words if it has a PARTIAL entry
    auto issue = [&](int t, const int(&col)[EPC], int st, u32x4(&kf)[NC], uint32_t(&mk)[NMW]) {
        if constexpr (KR) {
            static_assert(NLD == NC, "a chunk of K is as many registers either way");
#pragma unroll
            for (int i = 0; i < NLD; i++) {
                kf[i] = __builtin_nontemporal_load((const u32x4 *)(kbase + (int64_t)(col[0] + RPI * i) * p.ks[2] + kr_lane));
            }
        } else {
            const int kcol = B16 ? ((l32 < 16 ? col[0] : col[EPC - 1]) - (l32 & 16)) : col[0];  // (+ l32: this lane's key)
            const uint16_t *kp = kbase + (int64_t)(kcol + l32) * p.ks[2] + (D / 2) * hh;
#pragma unroll
            for (int c = 0; c < NC; c++) kf[c] = *(const u32x4 *)(kp + 8 * c);
        }
#pragma unroll
        for (int i = 0; i < NLD; i++) {
            // rows [RPI i, RPI i + RPI) of the chunk: with BLOCK_K = 16 the second half belongs to the second entry
            const int vcol = B16 ? (RPI * i < 16 ? col[0] : col[EPC - 1] - 16) : col[0];
            dma16<true>(vbase + (int64_t)vcol * p.vs[2], ld_voff[i], vmine_lds + st * VBUF + RPI * i * ROWB);
        }
        const unsigned fl = flags_of(t);
        if (fl >> 4) {
            if constexpr (DM) {
                mk[0] = bits[qrow * nCh + (col[0] >> 5)];
            } else if constexpr (PK) {
#pragma unroll
                for (int j = 0; j < EPC; j++) {
                    const int e = B16 ? 2 * t + j : (t >> sh);
                    const uint8_t *a = prow + (int64_t)((fl >> (4 + j)) & 1u ? e - F : 0) * tile_bytes;
                    if constexpr (B16) mk[j] = *(const uint16_t *)a;
                    else mk[j] = *(const uint32_t *)(a + 4 * (t & ((1 << sh) - 1)));
                }
            } else {
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const int64_t cc = (B16 ? (g < 2 ? col[0] + 8 * g : col[EPC - 1] + 8 * (g - 2)) : col[0] + 8 * g) + 4 * hh;
                    if (p.mask_vec4) {
                        mk[g] = *(const uint32_t *)(mrow + cc);
                    } else {
                        const uint8_t *m0 = mrow + cc * p.ms[3];
                        mk[g] = (uint32_t)m0[0] | ((uint32_t)m0[p.ms[3]] << 8) | ((uint32_t)m0[2 * p.ms[3]] << 16) |
                                ((uint32_t)m0[3 * p.ms[3]] << 24);
                    }
                }
            }
        }
    };
    // one chunk: scores, mask, softmax update, O^T += V^T . P^T
    auto compute = [&](int t, int st, const u32x4(&kf)[NC], const uint32_t(&mk)[NMW]) __attribute__((always_inline)) {
        f32x16 s;
#pragma unroll
        for (int i = 0; i < 16; i++) s[i] = 0.f;
        u32x4 ka[NC];  // the A operand: lane (l32, hh) holds d = (D/2) hh + 8c .. +7 of key l32
        if constexpr (KR) {
            // Lanes read what others have written and overwrite what others have read.  A wave's operations on LDS take effect in
            // their order, so nothing waits here; the fence keeps the compiler, which sees one lane, to that order.
            const int r = l32 & 15;
            auto in_order = [] {
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            };
            in_order();
#pragma unroll
            for (int i = 0; i < NLD / 2; i++) {
                const int w = RPI * i + ld_r0;
                *(u32x4 *)(kmine + w * ROWB + 16 * (ld_slot ^ k_swizzle<D>(w))) = kf[i];
            }
            in_order();
#pragma unroll
            for (int c = 0; c < NC; c++) ka[c] = *(const u32x4 *)(kmine + r * ROWB + 16 * ((NC * hh + c) ^ k_swizzle<D>(r)));
            in_order();
#pragma unroll
            for (int i = 0; i < NLD / 2; i++) {
                const int w = RPI * i + ld_r0;
                *(u32x4 *)(kmine + w * ROWB + 16 * (ld_slot ^ k_swizzle<D>(w))) = kf[NLD / 2 + i];
            }
            in_order();
#pragma unroll
            for (int c = 0; c < NC; c++) {
                const u32x4 x = *(const u32x4 *)(kmine + r * ROWB + 16 * ((NC * hh + c) ^ k_swizzle<D>(r)));
                ka[c] = l32 < 16 ? ka[c] : x;
            }
        } else {
#pragma unroll
            for (int c = 0; c < NC; c++) ka[c] = kf[c];
        }
#pragma unroll
        for (int c = 0; c < NC; c++) s = E::mfma(ka[c], qf[c], s);
        const unsigned fl = flags_of(t);
        if (fl != ALL) {  // a PARTIAL entry, or (BLOCK_K = 16) a second entry past the end of the list
            if constexpr (PK || DM) {
                // bit k of w: key k of the chunk; FULL entries count as all ones, missing ones as zero
                uint32_t w;
                if constexpr (B16) {
                    const uint32_t w0 = (fl & 16u) ? (mk[0] & 0xffffu) : ((fl & 1u) ? 0xffffu : 0u);
                    const uint32_t w1 = (fl & 32u) ? (mk[EPC - 1] & 0xffffu) : ((fl & 2u) ? 0xffffu : 0u);
                    w = w0 | (w1 << 16);
                } else {
                    w = (fl & 16u) ? mk[0] : ((fl & 1u) ? ~0u : 0u);
                }
                w >>= 4 * hh;  // this lane's keys are 8g + 4hh + jj
#pragma unroll
                for (int g = 0; g < 4; g++)
#pragma unroll
                    for (int jj = 0; jj < 4; jj++)
                        if (((w >> (8 * g + jj)) & 1u) == 0u) s[4 * g + jj] = kNegInf;
            } else {
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const int j = B16 ? (g >> 1) : 0;
                    const uint32_t w = ((fl >> (4 + j)) & 1u) ? mk[g] : (((fl >> j) & 1u) ? 0x01010101u : 0u);
#pragma unroll
                    for (int jj = 0; jj < 4; jj++)
                        if (((w >> (8 * jj)) & 0xffu) == 0u) s[4 * g + jj] = kNegInf;
                }
            }
        }
        float mx = kNegInf;
#pragma unroll
        for (int i = 0; i < 16; i++) mx = fmaxf(mx, s[i]);
        mx = half_swap_max(mx);
        const float rel = mx - m_ref;
        const bool raise = rel > raise_above;  // false for rows without an attended key so far (mx = -inf)
        if (__builtin_amdgcn_ballot_w64(raise) != 0ull) {
            const float a = raise ? (raise_above == kMaxSlack ? __builtin_amdgcn_exp2f(-rel) : 0.f) : 1.f;
            m_ref = raise ? mx : m_ref;
            raise_above = raise ? kMaxSlack : raise_above;
#pragma unroll
            for (int i = 0; i < 2; i++) acc_l[i] *= a;
#pragma unroll
            for (int db = 0; db < NDB; db++)
#pragma unroll
                for (int i = 0; i < 16; i++) acc[db][i] *= a;
        }
        uint32_t pw[8];
#pragma unroll
        for (int i = 0; i < 16; i += 2)
            pw[i >> 1] = E::pack2(__builtin_amdgcn_exp2f(s[i] - m_ref), __builtin_amdgcn_exp2f(s[i + 1] - m_ref));
        const uint8_t *vb_ = vmine + st * VBUF;
#pragma unroll
        for (int kc = 0; kc < 2; kc++) {
            const u32x4 pk4 = u32x4{pw[4 * kc], pw[4 * kc + 1], pw[4 * kc + 2], pw[4 * kc + 3]};
#pragma unroll
            for (int db = 0; db < NDB; db++) {
                const uint8_t *vp = vb_ + 16 * kc * ROWB + voff[db];
                const u32x2 lo = E::tr_read(vp), hi = E::tr_read(vp + 8 * ROWB);
                acc[db] = E::mfma(u32x4{lo.x, lo.y, hi.x, hi.y}, pk4, acc[db]);
            }
            acc_l = E::mfma16(sum_sel, pk4, acc_l);
        }
    };

    // ---- this wave's chunk stream: chunk t computes while chunk t + 4 loads and the index of t + 8 is fetched ----
    {
        u32x4 kf[2][NC];
        uint32_t mk[2][NMW];
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int g = 0; g < NMW; g++) mk[j][g] = 0u;
        int t = t_lo + wave_u;
        int idxs[2][EPC] = {};  // idxs[s]: list indices of the chunk that goes into stage s next
        if (t < t_hi) {
            idx_load(t, idxs[0]);
            if (t + kDecodeWaves < t_hi) idx_load(t + kDecodeWaves, idxs[1]);
            int col[EPC];
            cols_of(t, idxs[0], col);
            issue(t, col, 0, kf[0], mk[0]);
        }
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int e = 0; e < 4; e++) qf[c][e] = live ? E::scale2(qf[c][e], p.scale) : 0u;
        for (; t < t_hi; t += 2 * kDecodeWaves) {
            static_for<2>([&](auto jc) {
                constexpr int j = decltype(jc)::value;
                const int tt = t + j * kDecodeWaves;  // the chunk in stage j
                if (tt >= t_hi) return;
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // chunk tt has landed, and the index of the next
                // (the compiler accounts for these loads here, where it costs nothing, instead of in front of their
                // first use, where its wait would take the direct loads of the next chunk along)
#pragma unroll
                for (int c = 0; c < NC; c++) asm volatile("" ::"v"(kf[j][c]));
#pragma unroll
                for (int g = 0; g < NMW; g++) asm volatile("" ::"v"(mk[j][g]));
#pragma unroll
                for (int e = 0; e < EPC; e++) asm volatile("" ::"v"(idxs[j ^ 1][e]));
                const int tn = tt + kDecodeWaves;
                if (tn < t_hi) {
                    int col_n[EPC];
                    cols_of(tn, idxs[j ^ 1], col_n);
                    if (tn + kDecodeWaves < t_hi) idx_load(tn + kDecodeWaves, idxs[j]);
                    issue(tn, col_n, j ^ 1, kf[j ^ 1], mk[j ^ 1]);
                }
                compute(tt, j, kf[j], mk[j]);
            });
        }
    }

    // ---- merge the four waves through LDS (the V stages are free once every wave is done) ----
    __syncthreads();
    float *const part = reinterpret_cast<float *>(smem);
    constexpr int PST = D + 2;  // floats per row of a part
    {
        float *mine = part + (wave * 32 + l32) * PST;
#pragma unroll
        for (int db = 0; db < NDB; db++)
#pragma unroll
            for (int g = 0; g < 4; g++)
#pragma unroll
                for (int jj = 0; jj < 4; jj++) mine[32 * db + 8 * g + 4 * hh + jj] = acc[db][4 * g + jj];
        if (hh == 0) {
            mine[D] = raise_above == kMaxSlack ? m_ref : kNegInf;
            mine[D + 1] = l32 < 16 ? acc_l[0] : acc_l[1];
        }
    }
    __syncthreads();
    // n parts in LDS, `stride` floats apart, added up: a wave takes rows, four floats per lane
    constexpr int LPR = D / 4, RPW = 64 / LPR;  // lanes per row, rows side by side
    const int l = lane & (LPR - 1), r0 = lane / LPR;
    auto add_up = [&](const float *parts, int n, int stride, int first, int step, auto &&leave) {
#pragma unroll 1
        for (int row = first; row < p.Sq; row += step) {
            float out[4], M, L;
            merge_parts<4>(parts + row * PST, n, stride, D, 4 * l, out, M, L);
            leave(row, f32x4{out[0], out[1], out[2], out[3]}, M, L);
        }
    };
    const int first = wave_u * RPW + r0, step = kDecodeWaves * RPW;
    auto to_output = [&](int row, f32x4 x, float M, float L) {
        const float inv = L > 0.f ? 1.f / L : 0.f;
        if (p.lse != nullptr && l == 0)
            p.lse[b * p.lses[0] + h * p.lses[1] + row * p.lses[2]] =
                L > 0.f ? (M + __builtin_amdgcn_logf(L)) * 0.69314718056f : kNegInf;
        *(u32x2 *)(p.o + b * p.os[0] + h * p.os[1] + (int64_t)row * p.os[2] + 4 * l) =
            u32x2{E::pack2(x.x * inv, x.y * inv), E::pack2(x.z * inv, x.w * inv)};
    };
    if (p.nsplit == 1) {
        add_up(part, kDecodeWaves, 32 * PST, first, step, to_output);
        return;
    }
    const uint32_t part_bytes = (uint32_t)(p.Sq * PST * 4);
    uint8_t *const plane_parts = reinterpret_cast<uint8_t *>(p.ws) + (int64_t)bh * p.nsplit * part_bytes;
    const HandOver mine(plane_parts + (int64_t)split * part_bytes, part_bytes);
    add_up(part, kDecodeWaves, 32 * PST, first, step, [&](int row, f32x4 x, float M, float L) {
        mine.put((uint32_t)(4 * (row * PST + 4 * l)), x);
        if (l == 0) mine.put((uint32_t)(4 * (row * PST + D)), f32x2{M, L});
    });
    if (p.arrivals == nullptr) return;

    // ---- the last workgroup of the plane brings all parts to LDS as they lie in memory, and adds them up ----
    // A launch of its own for that costs its 3 us on an idle device and two more memory round trips: B4 H32 Sq1 Sk2048 with a new mask
    // 25.8 -> 23.3 us a call, B8 H16 Sq16 Sk16384 gathered 86.4 -> 85.3, B8 H32 Sq1 Sk32768 651 -> 649 (D = 128, bf16).  With the parts
    // read into registers row by row instead, in unrolled code that every compute unit fetches for the first time here: 24.3, 92.2.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();  // every wave's rows have been handed over, and LDS has been read
    if (tid == 0) *reinterpret_cast<int *>(smem) = arrives_last(p.arrivals + bh, p.tag, p.nsplit);
    __syncthreads();
    const bool last = __builtin_amdgcn_readfirstlane(*reinterpret_cast<int *>(smem)) != 0;
    if (!last) return;
    __syncthreads();
    // (rows are a multiple of 8 bytes; the 8 in front of a plane that starts between two pieces of 16 are the plane's before it,
    // the up to 8 behind the last plane the counters')
    const uint32_t lead = (uint32_t)(uintptr_t)plane_parts & 8u, bytes = p.nsplit * part_bytes + lead;
    for (uint32_t at = 1024u * wave_u; at < bytes; at += 1024u * kDecodeWaves)
        if (at + 16u * lane < bytes) dma16<false, true>(plane_parts - lead + at, 16u * lane, lds0 + at);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    float *const all = part + lead / 4;
    add_up(all, p.nsplit, p.Sq * PST, first, step, to_output);
}

// Merge of the nsplit partial results of every (b, h) in a launch of its own, where that is sooner (decode_merges_in_launch) or the
// workspace has no place for the counters: grid B*H, 256 threads, 8 per query row.
template <int DT, int D>
__global__ __launch_bounds__(256) void decode_merge_kernel(const DecodeParams p) {
    using E = Elem<DT>;
    constexpr int NV = D / 8, PST = D + 2;
    const int tid = threadIdx.x, bh = blockIdx.x;
    const int b = bh / p.H, h = bh - b * p.H;
    const int q = tid >> 3, d0 = (tid & 7) * NV;
    if (q >= p.Sq) return;
    float out[NV], M, L;
    merge_parts<NV>(p.ws + ((int64_t)bh * p.nsplit * p.Sq + q) * PST, p.nsplit, (int64_t)p.Sq * PST, D, d0, out, M, L);
    const float inv = L > 0.f ? 1.f / L : 0.f;
    if (p.lse != nullptr && (tid & 7) == 0)
        p.lse[b * p.lses[0] + h * p.lses[1] + q * p.lses[2]] =
            L > 0.f ? (M + __builtin_amdgcn_logf(L)) * 0.69314718056f : kNegInf;
    uint16_t *orow = p.o + b * p.os[0] + h * p.os[1] + (int64_t)q * p.os[2] + d0;
#pragma unroll
    for (int j = 0; j < NV; j += 2) *(uint32_t *)(orow + j) = E::pack2(out[j] * inv, out[j + 1] * inv);
}

// The same for more than kDecodeMergeFew parts: one wave per query row, four per workgroup.  Eight lanes share a part (two
// neighbouring floats of every 16 each, so a part is read in runs of 64 bytes), eight parts go side by side and kMergeBatch
// reads of each are in flight.  The parts lie in a cache and are few: all of this is latency, and the kernel above, which
// walks them one after the other, took most of a call with many (bf16, D = 128, Sq1; classification, decode and merge):
// 128 parts (B1 H4 Sk32768) 76.9 -> 19.5 us, 22 parts (B2 H12 Sq4 Sk8192) 40.6 -> 31.1, 16 parts (B1 H32 Sk32768) 78.7 -> 72.5.
// Around the line (decode and merge in a graph, us, kernel above | this one):
//   parts                2             4             5             6             8             9            16
//   B1 H8  Sq1  Sk4096   30.3 | 30.9   20.2 | 19.7   18.9 | 17.8   18.9 | 17.3   17.5 | 14.8   17.8 | 14.5   18.5 | 12.0
//   B4 H16 Sq1  Sk4096   39.8 | 40.6   28.6 | 28.2   34.6 | 33.3   32.3 | 30.3   30.9 | 27.8   36.7 | 33.4   39.2 | 31.6
//   B4 H8  Sq16 Sk4096   39.1 | 39.8   26.0 | 25.4   24.1 | 23.0   23.1 | 21.3   22.6 | 19.6   26.9 | 23.7   28.0 | 20.5
// so from five parts on this one is faster at these sizes; the line stands at eight, where the order of the sum has been so far.
// With 2 ... 4 parts the exchanges between lanes cost more than they save: 2 parts (B1 H8 Sk512) 12.5 -> 14.4, 4 parts (B8 H16
// Sq32 Sk1024) 26.3 -> 29.6.
constexpr int kMergeBatch = 4;
template <int DT, int D>
__global__ __launch_bounds__(256) void decode_merge_many_kernel(const DecodeParams p) {
    using E = Elem<DT>;
    constexpr int NP = D / 16, PST = D + 2;
    const int lane = threadIdx.x & 63, l8 = lane & 7, grp = lane >> 3;
    const int64_t row = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (row >= (int64_t)p.B * p.H * p.Sq) return;
    const int bh = (int)(row / p.Sq), q = (int)(row - (int64_t)bh * p.Sq);
    const int b = bh / p.H, h = bh - b * p.H;
    const int64_t stride = (int64_t)p.Sq * PST;
    const float *const part = p.ws + ((int64_t)bh * p.nsplit * p.Sq + q) * PST;
    float M = kNegInf;
    for (int i = lane; i < p.nsplit; i += 64) M = fmaxf(M, part[i * stride + D]);
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) M = fmaxf(M, __shfl_xor(M, s));
    float L = 0.f;
    f32x2 out[NP];
#pragma unroll
    for (int c = 0; c < NP; c++) out[c] = f32x2{0.f, 0.f};
    if (M != kNegInf) {  // else no part saw an attended key
        for (int i0 = grp; i0 < p.nsplit; i0 += 8 * kMergeBatch) {
            f32x2 ml[kMergeBatch], x[kMergeBatch][NP];
#pragma unroll
            for (int i = 0; i < kMergeBatch; i++) {
                // (past the last part: the last one again, left out below: a weight of 0 would turn an infinity into NaN)
                const float *pp = part + min(i0 + 8 * i, p.nsplit - 1) * stride;
                ml[i] = *(const f32x2 *)(pp + D);
#pragma unroll
                for (int c = 0; c < NP; c++) x[i][c] = *(const f32x2 *)(pp + 16 * c + 2 * l8);
            }
#pragma unroll
            for (int i = 0; i < kMergeBatch; i++) {
                if (i0 + 8 * i >= p.nsplit) break;
                // 0 for parts without an attended key (m = -inf)
                const float w = __builtin_amdgcn_exp2f(ml[i].x - M);
                L += w * ml[i].y;
#pragma unroll
                for (int c = 0; c < NP; c++) {
                    out[c].x += w * x[i][c].x;
                    out[c].y += w * x[i][c].y;
                }
            }
        }
#pragma unroll
        for (int s = 8; s < 64; s <<= 1) {
            L += __shfl_xor(L, s);
#pragma unroll
            for (int c = 0; c < NP; c++) {
                out[c].x += __shfl_xor(out[c].x, s);
                out[c].y += __shfl_xor(out[c].y, s);
            }
        }
    }
    if (grp != 0) return;
    const float inv = L > 0.f ? 1.f / L : 0.f;
    if (p.lse != nullptr && l8 == 0)
        p.lse[b * p.lses[0] + h * p.lses[1] + q * p.lses[2]] =
            L > 0.f ? (M + __builtin_amdgcn_logf(L)) * 0.69314718056f : kNegInf;
    uint16_t *orow = p.o + b * p.os[0] + h * p.os[1] + (int64_t)q * p.os[2] + 2 * l8;
#pragma unroll
    for (int c = 0; c < NP; c++) *(uint32_t *)(orow + 16 * c) = E::pack2(out[c].x * inv, out[c].y * inv);
}

// Merge of n attention results over disjoint key ranges: o = sum_i exp(lse_i - lse) o_i, lse = log sum_i exp(lse_i).
// One thread per 8 output elements.
template <int DT>
__global__ __launch_bounds__(256) void merge_parts_kernel(const MergeParams p) {
    using E = Elem<DT>;
    const int per_row = p.D / 8;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t row = idx / per_row;
    const int part = (int)(idx - row * per_row);
    if (row >= (int64_t)p.B * p.H * p.Sq) return;
    const int q = (int)(row % p.Sq);
    const int bh = (int)(row / p.Sq);
    const int b = bh / p.H, h = bh - b * p.H;
    const float *lp = p.lse_parts + b * p.lps[1] + h * p.lps[2] + (int64_t)q * p.lps[3];
    float M = kNegInf;
    for (int i = 0; i < p.n; i++) M = fmaxf(M, lp[i * p.lps[0]]);
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    float L = 0.f;
    if (M != kNegInf) {
        for (int i = 0; i < p.n; i++) {
            const float w = __expf(lp[i * p.lps[0]] - M);  // 0 for parts whose keys this row does not attend to
            L += w;
            const u32x4 x = *(const u32x4 *)(p.o_parts + i * p.ops[0] + b * p.ops[1] + h * p.ops[2] +
                                             (int64_t)q * p.ops[3] + 8 * part);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t xe = x[e];
                if constexpr (DT == 0) {
                    acc[2 * e] += w * __uint_as_float(xe << 16);
                    acc[2 * e + 1] += w * __uint_as_float(xe & 0xffff0000u);
                } else {
                    const f16x2 hx = __builtin_bit_cast(f16x2, xe);
                    acc[2 * e] += w * (float)hx.x;
                    acc[2 * e + 1] += w * (float)hx.y;
                }
            }
        }
    }
    const float inv = L > 0.f ? 1.f / L : 0.f;
    u32x4 out;
#pragma unroll
    for (int e = 0; e < 4; e++) out[e] = E::pack2(acc[2 * e] * inv, acc[2 * e + 1] * inv);
    *(u32x4 *)(p.o + b * p.os[0] + h * p.os[1] + (int64_t)q * p.os[2] + 8 * part) = out;
    if (p.lse != nullptr && part == 0)
        p.lse[b * p.lses[0] + h * p.lses[1] + (int64_t)q * p.lses[2]] = L > 0.f ? M + __logf(L) : kNegInf;
}

template <int DT, int D, bool PK, bool B16, bool DM = false>
hipError_t launch_decode_kind(const DecodeParams &p, hipStream_t stream) {
    constexpr int smem = decode_smem_bytes<D, decode_key_rows(B16, DM)>() + (DM ? kDirectBytes : 0);
    auto kern = sparse_decode_kernel<DT, D, PK, B16, DM>;
    static unsigned long long attr_done = 0;  // devices on which this kernel may use `smem` bytes of LDS
    if (const hipError_t e0 = allow_dynamic_smem(kern, smem, attr_done); e0 != hipSuccess) return e0;
    hipLaunchKernelGGL(kern, dim3((unsigned)p.nsplit * (unsigned)(p.B * p.H)), dim3(kDecodeWaves * 64), smem, stream, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || p.nsplit == 1 || p.arrivals != nullptr) return e;
    const unsigned rows = (unsigned)p.B * p.H * p.Sq;  // (at most 65535 planes of 32 rows)
    if (p.nsplit > kDecodeMergeFew) hipLaunchKernelGGL((decode_merge_many_kernel<DT, D>), dim3((rows + 3) / 4), dim3(256), 0, stream, p);
    else hipLaunchKernelGGL((decode_merge_kernel<DT, D>), dim3(p.B * p.H), dim3(256), 0, stream, p);
    return hipGetLastError();
}

template <int DT, int D>
hipError_t launch_decode_one(const DecodeParams &p, hipStream_t stream) {
    if (p.full_ids == nullptr) return launch_decode_kind<DT, D, false, false, true>(p, stream);
    const bool pk = p.packed != nullptr, b16 = p.BK == 16;
    if (pk) return b16 ? launch_decode_kind<DT, D, true, true>(p, stream) : launch_decode_kind<DT, D, true, false>(p, stream);
    return b16 ? launch_decode_kind<DT, D, false, true>(p, stream) : launch_decode_kind<DT, D, false, false>(p, stream);
}

}  // namespace

hipError_t launch_merge_parts(const MergeParams &p, int dtype, hipStream_t stream) {
    const int64_t threads = (int64_t)p.B * p.H * p.Sq * (p.D / 8);
    const unsigned grid = (unsigned)((threads + 255) / 256);
    if (dtype == 0) hipLaunchKernelGGL((merge_parts_kernel<0>), dim3(grid), dim3(256), 0, stream, p);
    else if (dtype == 1) hipLaunchKernelGGL((merge_parts_kernel<1>), dim3(grid), dim3(256), 0, stream, p);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_decode(const DecodeParams &p, int dtype, int D, hipStream_t stream) {
    if (dtype == 0 && D == 128) return launch_decode_one<0, 128>(p, stream);
    if (dtype == 0 && D == 64) return launch_decode_one<0, 64>(p, stream);
    if (dtype == 1 && D == 128) return launch_decode_one<1, 128>(p, stream);
    if (dtype == 1 && D == 64) return launch_decode_one<1, 64>(p, stream);
    return hipErrorInvalidValue;
}

}  // namespace sa
