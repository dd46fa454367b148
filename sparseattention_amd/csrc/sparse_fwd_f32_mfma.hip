// Block-sparse attention forward for float32 q, k, v, o on the matrix unit (v_mfma_f32_32x32x2_f32), gfx950.
//
// Same function as sparse_fwd_kernel (the Triton kernels sparse_attention_kernel / _sparse_inner,
// sparseattention/sparse_attn_kernel.py:74-146 and :10-63, which take the element type of their inputs, :98-101, :145),
// in float32 throughout: nothing is rounded below float32, P enters the P.V product as it leaves the exponential.
// The plain vector-unit kernel of sparse_fwd_f32.hip stays for the sizes this one does not have.
//
// One workgroup per (Q tile of BQ = 32 NW rows, b, h); wave w owns query rows [32w, 32w+32).  The list (FULL tiles,
// then PARTIAL tiles) is consumed 32 keys at a time through two LDS stages of K and V rows, filled by direct loads
// global -> LDS one chunk ahead; the mask words of a chunk and the raw list travel the same way, so the loop holds no
// load the compiler knows of and one "s_waitcnt vmcnt(0)" per chunk covers everything.
//
// MFMA operands (lane = 32 hh + l32; every instruction contracts over 2 indices, one per lane half):
//   S^T = K . Q^T   A = K: lane (l32, hh) supplies key l32, d = (D/2) hh + c in step c (its half row is contiguous:
//                   one 16-byte LDS read feeds four steps); B = Q^T in registers with the same order of d.
//                   The result leaves lane (l32, hh) holding query l32 and keys 8g + 4hh + j in register 4g + j.
//   O^T = V^T . P^T step (g, j) contracts over the two keys 8g + j and 8g + 4 + j: B = P^T is register 4g + j of
//                   the scores as it stands (lane half hh holds key 8g + 4hh + j), A = V^T: lane (l32, hh) reads
//                   V[key 8g + 4hh + j][32 db + l32], 32 consecutive floats per lane half.
// LDS rows are unpadded (a direct load writes 64 lanes x 16 bytes contiguously); the 16-byte pieces of a row are
// XORed with the row's low four bits for K (the 16 rows read together fall into 16 bank groups) and with 8 * bit 2 of
// the row for V (the two lane halves read rows four apart: they fall into different halves of the banks).
//
// Online softmax in the reference's order (sparse_attn_kernel.py:53-58): row maximum, rescale, exponentials, row sum,
// accumulate; exp2 units with the scale folded into Q.  Rows that attend to nothing give 0.
#include "fwd_common.h"

namespace sa {

namespace {

constexpr int kF32ListCap = 1024;  // list entries kept in LDS (the launcher refuses longer rows of tiles)
constexpr int f32_groups(int NW, bool SP) { return SP && NW <= 2 ? 2 : 1; }
// LDS of a group of NW waves: [K, two stages][V, two stages][mask words, two stages][list]
template <int D, int NW>
constexpr int f32_group_bytes = 4 * 32 * D * 4 + 2 * NW * 1024 + kF32ListCap * 4;

// MODE 0: BK = 16 (two list entries per chunk), MODE 1: BK = 32, MODE 2: BK >= 64 (BK/32 chunks per entry).
// PK: mask entries of PARTIAL tiles from the bit-packed tiles; else from the bool mask (key stride 1, rows and base
// 16-byte aligned: checked by the launcher).
// SP: lists shared by up to p.nsplit workgroups (fwd_split_share).
// KG: groups of NW waves that share out a part's chunks, each with stages of its own, in step; their rows meet in LDS.  Two where lists are
// shared and NW <= 2 would leave two of the four SIMDs idle (144 KiB of LDS at D = 128, one workgroup a compute unit: fwd_split_plan).
// By chunks, not by entries: of an entry of two chunks (BLOCK_K 64) one group had both, 8 tiles of 32 chunks at D = 64 15.2 -> 12.6 us.
// A small launch is a chain: B1 H4 S512 D64 with half of the 32 x 32 blocks (32 Q tiles, about 9 chunks each, parts of two) takes 11.1 us a
// pass, where two waves per part, lists by way of LDS and a second launch for the merge took 15.7.  Time stamps with both lists read whole
// beside the counts (11.2 us; callers' rows may end with the list): queries, counts and lists 1.2 us, first K and V at 2.3, products and
// softmax 3.0, the groups' rows 0.4, parts handed over 0.7, all arrived 0.8, parts read and added 2.1.
// Registers for two waves per SIMD (D = 64: results stay out of the accumulation registers; causal B2 H16 S2048 235 -> 226 us), but not at
// D = 128 with two waves a workgroup: registers that fill a SIMD keep the waves of two workgroups on different ones (339 us against 592).
template <int D, int NW, int MODE, bool PK, bool SP, bool SD>
__global__ __launch_bounds__(NW * f32_groups(NW, SP) * 64, D == 128 && NW * f32_groups(NW, SP) <= 2 ? 1 : 2) void sparse_fwd_f32_mfma_kernel(const FwdParams p) {
    constexpr int KG = f32_groups(NW, SP);
    constexpr int ROWB = D * 4, PPR = ROWB / 16;  // bytes and 16-byte pieces per K/V row
    constexpr int KBUF = 32 * ROWB;               // one stage of K (or V): 32 rows
    constexpr int MBUF = NW * 1024;               // one stage of mask words: 64 lanes x 16 bytes per wave
    constexpr int OFF_V = 2 * KBUF, OFF_M = 4 * KBUF, OFF_L = OFF_M + 2 * MBUF, GROUP = f32_group_bytes<D, NW>;
    constexpr int EPC = MODE == 0 ? 2 : 1;
    constexpr int LBKC = MODE == 0 ? 4 : 5;
    constexpr int RPI = 1024 / ROWB;   // rows per direct load
    constexpr int NLD = 32 / RPI / NW; // direct loads per wave and chunk, each for K and for V
    static_assert(32 % (RPI * NW) == 0, "staging layout");

    extern __shared__ __attribute__((aligned(1024))) uint8_t smem0[];
    const int grp = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / (NW * 64));
    uint8_t *const smem = smem0 + grp * GROUP;
    int *const ring = reinterpret_cast<int *>(smem + OFF_L);

    const int tid = KG == 1 ? threadIdx.x : threadIdx.x % (NW * 64), lane = tid & 63, wave = tid >> 6;
    const int l32 = lane & 31, hh = lane >> 5;
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);
    // Workgroup -> (b, h, Q tile) as in sparse_fwd_kernel: the hardware hands consecutive workgroup ids to the 8 XCDs
    // in turn; the remap gives every XCD whole planes (so that the Q tiles sharing a K/V plane meet in one L2 and every
    // XCD gets the same mix of long and short lists), planes two at a time with their Q tiles interleaved, last Q tile
    // first; or more planes side by side (SD, fwd_spread).
    int b, h, qt, s0 = 0;  // s0: this workgroup's part of a shared list
    {
        const int total = p.nQ * p.B * p.H, per = total >> 3;
        int lin = blockIdx.x;
        if constexpr (SP) {  // the first parts of all tiles, then the second ones, ...
            s0 = lin / total;
            lin -= s0 * total;
        }
        int bh;
        if constexpr (SD) {
            int i = blockIdx.x >> 3, group = 0;
            if ((i >> 5) == 1 && (i | 31) < per) i ^= 31;
            int n = 8 * i + (blockIdx.x & 7);
            if (p.spread != p.B * p.H) {
                group = n / (p.spread * p.nQ);
                n -= group * (p.spread * p.nQ);
            }
            int below = n / p.spread;
            bh = group * p.spread + n - below * p.spread;
            if ((p.spread & 4) != 0 && (below | 1) < p.nQ) below ^= (below >> 1) & 1;
            qt = p.nQ - 1 - below;
        } else {
            if (lin < (per << 3)) lin = (lin & 7) * per + (lin >> 3);
            int pair = lin / (2 * p.nQ);
            const int r = lin - pair * 2 * p.nQ;
            if (((p.B * p.H) & 15) == 0) {
                const int ppx = (p.B * p.H) >> 4;
                const int x = pair / ppx;
                pair = (pair - x * ppx) * 8 + x;
            }
            const bool paired = 2 * pair + 1 < p.B * p.H;
            bh = 2 * pair + (paired ? (r & 1) : 0);
            qt = p.nQ - 1 - (paired ? (r >> 1) : r);
        }
        b = bh / p.H;
        h = bh - b * p.H;
    }
    const int qrow = qt * (NW * 32) + wave * 32 + l32;

    const float *const kbase = reinterpret_cast<const float *>(p.k) + b * p.ks[0] + h * p.ks[1];
    const float *const vbase = reinterpret_cast<const float *>(p.v) + b * p.vs[0] + h * p.vs[1];
    const int32_t *fid = p.full_ids + b * p.fis[0] + h * p.fis[1] + qt * p.fis[2];
    const int32_t *pid = p.part_ids + b * p.pis[0] + h * p.pis[1] + qt * p.pis[2];
    // Queries and counts travel together.
    f32x4 q_in[D / 8];
    {
        const float *qp = reinterpret_cast<const float *>(p.q) + b * p.qs[0] + h * p.qs[1] + (int64_t)qrow * p.qs[2] + (D / 2) * hh;
#pragma unroll
        for (int c = 0; c < D / 8; c++) q_in[c] = *(const f32x4 *)(qp + 4 * c);
    }
    int cnt[2];
    const int32_t *const cnt_addr[2] = {p.full_lens + (b * p.fls[0] + h * p.fls[1] + qt * p.fls[2]),
                                        p.part_lens + (b * p.pls[0] + h * p.pls[1] + qt * p.pls[2])};
    scalar_gather(cnt_addr, cnt);
    int F = min(min(max(cnt[0], 0), p.nK), kF32ListCap);
    int NE = F + min(min(max(cnt[1], 0), p.nK - F), kF32ListCap - F);
    int share = 1, p_lo = 0;
    if constexpr (SP) {
        share = fwd_split_share(NE, p.lbk, 5, p.split_least, p.split_chunks, p.nsplit);
        if (s0 >= share) return;
        const int e_lo = fwd_split_first(NE, p.lbk, 5, s0, share), e_hi = fwd_split_first(NE, p.lbk, 5, s0 + 1, share);
        p_lo = max(e_lo - F, 0);
        fid += (int64_t)min(e_lo, F) * p.fis[3];
        pid += (int64_t)p_lo * p.pis[3];
        F = min(max(F - e_lo, 0), e_hi - e_lo);
        NE = e_hi - e_lo;
    }
    const bool in_lanes = SP && NE <= 64;  // a part of at most 64 entries: one per lane, no way by LDS
    // this group's chunks, t_lo .. t_lo + T - 1 of the part's (an entry of several chunks is shared out too), and those of the longest group
    const int T_part = MODE == 2 ? (NE << (p.lbk - 5)) : ((NE + EPC - 1) / EPC);
    const int t_lo = T_part * grp / KG, T = T_part * (grp + 1) / KG - t_lo, T_all = (T_part + KG - 1) / KG;
    int lane_entry = 0;
    if (in_lanes && lane < NE) lane_entry = lane < F ? fid[(int64_t)lane * p.fis[3]] : pid[(int64_t)(lane - F) * p.pis[3]];
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const SA_LDS uint8_t *)smem);

    // ---- per-lane constants ------------------------------------------------------------------------------------
    const int koff0 = l32 * ROWB + 16 * ((hh * (PPR / 2)) ^ (l32 & 15));  // read i of the row half: koff0 ^ (16 i)
    const int voff0 = 4 * hh * ROWB + 128 * hh + 16 * (l32 >> 2) + 4 * (l32 & 3);  // d block db: ^ (128 db); key: + row * ROWB
    // direct loads: load n (0 .. 32/RPI - 1) fills rows [RPI n, RPI n + RPI) of a stage, lane -> row n RPI + ld_r, LDS
    // piece ld_slot, which holds the source piece ld_slot ^ swizzle(row)
    const int ld_r = lane / PPR, ld_slot = lane % PPR;
    const int64_t ld_kbase = ((int64_t)ld_r * p.ks[2]) * 4, ld_vbase = ((int64_t)ld_r * p.vs[2]) * 4;
    const int64_t tile_bytes = (int64_t)(NW * 4) * p.BK;
    const uint8_t *const pbase = PK ? p.packed + b * p.pks[0] + h * p.pks[1] + ((int64_t)qt * p.nK + p_lo) * tile_bytes : nullptr;
    const uint8_t *const mrow0 = PK ? nullptr : p.mask + b * p.ms[0] + h * p.ms[1] + (int64_t)(qt * (NW * 32)) * p.ms[2];

    struct Plan {
        int col[EPC];    // first key column of every entry of the chunk
        int slot[EPC];   // its slot among the PARTIAL entries (0 when it is not PARTIAL)
        unsigned flags;  // bit j: entry j exists; bit 4 + j: it is PARTIAL
    };
    auto plan_entry = [&](Plan &pl, int j, int e, int idx, int sub) {
        const bool exists = e < NE && (unsigned)idx < (unsigned)p.nK;
        const bool partial = exists && e >= F;
        pl.col[j] = exists ? ((MODE == 2 ? (idx << p.lbk) : (idx << LBKC)) + 32 * sub) : 0;
        pl.slot[j] = partial ? e - F : 0;
        pl.flags |= (exists ? 1u : 0u) << j | (partial ? 16u : 0u) << j;
    };
    auto plan_of = [&](int t, Plan &pl) {  // chunk t of the part
        pl.flags = 0u;
#pragma unroll
        for (int j = 0; j < EPC; j++) {
            const int e = MODE == 2 ? (t >> (p.lbk - 5)) : t * EPC + j;
            const int sub = MODE == 2 ? (t & ((1 << (p.lbk - 5)) - 1)) : 0;
            plan_entry(pl, j, e, in_lanes ? __builtin_amdgcn_readlane(lane_entry, min(e, 63)) : __builtin_amdgcn_readfirstlane(ring[min(e, kF32ListCap - 1)]), sub);
        }
    };
    // all direct loads of a chunk into stage `buf`
    auto stage_chunk = [&](int buf, const Plan &pl, int t) {
#pragma unroll
        for (int i = 0; i < NLD; i++) {
            const int n = NW * i + wave_u;  // this load's place in the chunk
            const int row0 = RPI * n;
            const int j = MODE == 0 ? (row0 >> 4) : 0;
            const int in_entry = MODE == 0 ? (row0 & 15) : row0;
            const int kswz = (row0 & 15) ^ 0, vswz = 8 * ((row0 >> 2) & 1);
            // (rows row0 .. row0 + RPI - 1 differ from row0 in bits that ld_r supplies: RPI <= 4 divides 16 and 4)
            const int col = (MODE == 0 && j ? pl.col[EPC - 1] : pl.col[0]) + in_entry;
            const uint8_t *ks_ = reinterpret_cast<const uint8_t *>(kbase + (int64_t)col * p.ks[2]) + ld_kbase +
                                 16 * (ld_slot ^ ((kswz | ld_r) & 15));
            const uint8_t *vs_ = reinterpret_cast<const uint8_t *>(vbase + (int64_t)col * p.vs[2]) + ld_vbase +
                                 16 * (ld_slot ^ (vswz ^ (8 * ((ld_r >> 2) & 1))));
            dma16_lane(ks_, lds0 + buf * KBUF + row0 * ROWB);
            dma16_lane(vs_, lds0 + OFF_V + buf * KBUF + row0 * ROWB);
        }
        // mask words of this wave's 32 rows
        const uint32_t mdst = lds0 + OFF_M + buf * MBUF + wave_u * 1024;
        if constexpr (PK) {
            // one dword per lane: the row's 32 bits of the chunk (BK = 16: lane half hh takes entry hh's dword that holds
            // rows 2r, 2r + 1)
            const int r = wave * 32 + l32;
            const uint8_t *src;
            if constexpr (MODE == 0) src = pbase + (int64_t)(hh ? pl.slot[EPC - 1] : pl.slot[0]) * tile_bytes + (r & ~1) * 2;
            else if constexpr (MODE == 1) src = pbase + (int64_t)pl.slot[0] * tile_bytes + r * 4;
            else src = pbase + (int64_t)pl.slot[0] * tile_bytes + (int64_t)r * (p.BK >> 3) + 4 * (t & ((1 << (p.lbk - 5)) - 1));
            dma4_lane(src, mdst);
        } else {
            // 16 mask bytes per lane: keys 16 hh .. 16 hh + 15 of the chunk (BK = 16: entry hh)
            const int col = MODE == 0 ? (hh ? pl.col[EPC - 1] : pl.col[0]) : pl.col[0] + 16 * hh;
            dma16_lane(mrow0 + (int64_t)(wave * 32 + l32) * p.ms[2] + col, mdst);
        }
    };

    // ---- state ----
    float m_i = kNegInf, l_i = 0.f;  // of this lane's query row; l_i over this lane half's keys only
    f32x16 acc[D / 32];
#pragma unroll
    for (int db = 0; db < D / 32; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[db][i] = 0.f;

    // Q^T operand: d = (D/2) hh + c for step c, scaled once (softmax scale / ln 2)
    float qf[D / 2];
    auto scale_q = [&]() {
#pragma unroll
        for (int c = 0; c < D / 2; c++) qf[c] = q_in[c / 4][c % 4] * p.scale;
    };
    if (T_all > 0) {
        if (!in_lanes) {
            // the list: wave w brings entries 64 w + lane, 64 (w + NW) + lane, ...
            for (int base = 64 * wave_u; base < NE; base += 64 * NW) {
                const int e = min(base + lane, NE - 1);
                const int32_t *src = e < F ? fid + (int64_t)e * p.fis[3] : pid + (int64_t)(e - F) * p.pis[3];
                dma4_lane(src, lds0 + OFF_L + 4 * base);
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
        }
        Plan pl;
        if (T > 0) {  // (KG > 1: a part of one chunk is the other group's)
            plan_of(t_lo, pl);
            stage_chunk(0, pl, t_lo);
        }
        unsigned fl_cur = T > 0 ? pl.flags : 0u;
        scale_q();
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();

        auto chunk = [&](auto buf_c, int tc) {
            constexpr int BUF = decltype(buf_c)::value;
            // the next chunk goes to the other stage (past the last chunk the last one once more: in a long loop cheaper than the
            // branch, 1 %, but a part of one chunk would wait for it)
            unsigned fl_next = 0u;
            if (!SP || tc + 1 < T) {
                const int tn = t_lo + (tc + 1 < T ? tc + 1 : T - 1);
                Plan pn;
                plan_of(tn, pn);
                stage_chunk(BUF ^ 1, pn, tn);
                fl_next = pn.flags;
            }

            // ---- S^T = K . Q^T ----
            const uint8_t *kb_ = smem + BUF * KBUF;
            f32x16 s;
#pragma unroll
            for (int i = 0; i < 16; i++) s[i] = 0.f;
            int kbo = koff0;
            asm volatile("" : "+v"(kbo));
            // (SP: operand reads three bundles ahead, pinned, where each was waited for as it was issued: the products and softmax of a lone
            // chunk 3.2 -> 2.95 us; in the plain form, whose waves cover for each other, 1 % slower)
            constexpr int kAheadK = SP ? 3 : 0;
            f32x4 kf[PPR / 2];
            auto k_read = [&](int i) { kf[i] = *(const f32x4 *)(kb_ + (kbo ^ (16 * i))); };
#pragma unroll
            for (int i = 0; i < kAheadK; i++) k_read(i);
            if constexpr (SP) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < PPR / 2; i++) {
                if (i + kAheadK < PPR / 2) k_read(i + kAheadK);
#pragma unroll
                for (int e = 0; e < 4; e++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[i][e], qf[4 * i + e], s, 0, 0, 0);
                if constexpr (SP) __builtin_amdgcn_sched_barrier(0);
            }

            // ---- mask (chunks with a PARTIAL or missing entry only) ----
            constexpr unsigned ALL = (1u << EPC) - 1u;
            if (fl_cur != ALL) {
                const uint8_t *mb_ = smem + OFF_M + BUF * MBUF + wave * 1024;
                if constexpr (PK) {
                    uint32_t w;
                    if constexpr (MODE == 0) {
                        const uint32_t a = *(const uint32_t *)(mb_ + 4 * l32), c2 = *(const uint32_t *)(mb_ + 128 + 4 * l32);
                        const int sh = 16 * (l32 & 1);
                        const uint32_t w0 = (fl_cur & 16u) ? ((a >> sh) & 0xffffu) : ((fl_cur & 1u) ? 0xffffu : 0u);
                        const uint32_t w1 = (fl_cur & 32u) ? ((c2 >> sh) & 0xffffu) : ((fl_cur & 2u) ? 0xffffu : 0u);
                        w = w0 | (w1 << 16);
                    } else {
                        const uint32_t a = *(const uint32_t *)(mb_ + 4 * l32);
                        w = (fl_cur & 16u) ? a : ((fl_cur & 1u) ? ~0u : 0u);
                    }
                    w >>= 4 * hh;
#pragma unroll
                    for (int g = 0; g < 4; g++)
#pragma unroll
                        for (int jj = 0; jj < 4; jj++)
                            if (((w >> (8 * g + jj)) & 1u) == 0u) s[4 * g + jj] = kNegInf;
                } else {
                    // the row's 32 bytes: keys 0..15 in the first 512 bytes of the wave's slice, 16..31 in the second
#pragma unroll
                    for (int g = 0; g < 4; g++) {
                        const int j = MODE == 0 ? (g >> 1) : 0;  // list entry of this group of keys
                        const bool exists = (fl_cur >> j) & 1u, partial = (fl_cur >> (4 + j)) & 1u;
                        const uint32_t raw = *(const uint32_t *)(mb_ + 512 * (g >> 1) + 16 * l32 + 8 * (g & 1) + 4 * hh);
                        const uint32_t w = partial ? raw : (exists ? 0x01010101u : 0u);
#pragma unroll
                        for (int jj = 0; jj < 4; jj++)
                            if (((w >> (8 * jj)) & 0xffu) == 0u) s[4 * g + jj] = kNegInf;
                    }
                }
            }

            // ---- online softmax (sparse_attn_kernel.py:53-58) ----
            float mx = kNegInf;
#pragma unroll
            for (int i = 0; i < 16; i++) mx = fmaxf(mx, s[i]);
            mx = half_swap_max(mx);
            const float m_new = fmaxf(m_i, mx);
            const float m_use = m_new == kNegInf ? 0.f : m_new;          // a row that has seen no key yet
            const float alpha = m_i == kNegInf ? 0.f : __builtin_amdgcn_exp2f(m_i - m_use);
            m_i = m_new;
            float psum = 0.f;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                s[i] = __builtin_amdgcn_exp2f(s[i] - m_use);
                psum += s[i];
            }
            l_i = l_i * alpha + psum;
            if (__builtin_amdgcn_ballot_w64(alpha != 1.f) != 0ull) {
#pragma unroll
                for (int db = 0; db < D / 32; db++)
#pragma unroll
                    for (int i = 0; i < 16; i++) acc[db][i] *= alpha;
            }

            // ---- O^T += V^T . P^T ----
            const uint8_t *vb_ = smem + OFF_V + BUF * KBUF;
            int vbo = voff0;
            asm volatile("" : "+v"(vbo));
#pragma unroll
            for (int g = 0; g < 4; g++)
#pragma unroll
                for (int j = 0; j < 4; j++)
#pragma unroll
                    for (int db = 0; db < D / 32; db++) {
                        const float vv = *(const float *)(vb_ + (8 * g + j) * ROWB + (vbo ^ (128 * db)));
                        acc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv, s[4 * g + j], acc[db], 0, 0, 0);
                    }
            fl_cur = fl_next;
        };
        auto step = [&](auto buf_c, int tc) {
            if (KG == 1 || tc < T) chunk(buf_c, tc);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the next chunk has landed
            __syncthreads();                                   // and every wave is done with this one
        };
        for (int t = 0; t < T_all; t += 2) {
            step(std::integral_constant<int, 0>{}, t);
            if (t + 1 < T_all) step(std::integral_constant<int, 1>{}, t + 1);
        }
    }

    // ---- the groups' rows, the parts' rows, O = acc / l (sparse_attn_kernel.py:144); rows without a key give 0 ----
    const uint32_t lu = __float_as_uint(l_i);
    const auto sw = __builtin_amdgcn_permlane32_swap(lu, lu, false, false);
    float l_tot = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
    auto finish = [&](auto g_c) {
        constexpr int G = decltype(g_c)::value, NB = D / 32 / KG;  // this group's blocks of 32 columns: G NB ...
        f32x16 o[NB];
#pragma unroll
        for (int d = 0; d < NB; d++) o[d] = acc[G * NB + d];
        if constexpr (KG > 1) {
            // each group leaves the other's columns in its own stages, which nobody reads any more, its rows' state in its list
            static_assert(KG == 2 && NW * 32 * D * 2 <= 4 * KBUF && NW * 32 * 8 <= kF32ListCap * 4, "what a group leaves fits its LDS");
            const uint32_t at = wave_u * (NB * 4096) + 16 * lane, st_at = OFF_L + (wave_u * 32 + l32) * 8;
#pragma unroll
            for (int d = 0; d < NB; d++)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const f32x16 &a = acc[(1 - G) * NB + d];
                    *(f32x4 *)(smem + at + 1024 * (4 * d + g)) = f32x4{a[4 * g], a[4 * g + 1], a[4 * g + 2], a[4 * g + 3]};
                }
            if (hh == 0) *(f32x2 *)(smem + st_at) = f32x2{m_i, l_tot};
            __syncthreads();
            const uint8_t *const other = smem0 + (1 - G) * GROUP;
            const f32x2 st = *(const f32x2 *)(other + st_at);
            const float M = fmaxf(m_i, st.x), M0 = M == kNegInf ? 0.f : M;
            const float mine = __builtin_amdgcn_exp2f(m_i - M0), its = __builtin_amdgcn_exp2f(st.x - M0);
            // (the first group's values first, whichever group adds)
            auto add = [&](float a, float x) { return G == 0 ? __builtin_fmaf(a, mine, its * x) : __builtin_fmaf(x, its, mine * a); };
            l_tot = add(l_tot, st.y);
#pragma unroll
            for (int d = 0; d < NB; d++)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const f32x4 x = *(const f32x4 *)(other + at + 1024 * (4 * d + g));
#pragma unroll
                    for (int e = 0; e < 4; e++) o[d][4 * g + e] = add(o[d][4 * g + e], x[e]);
                }
            m_i = M;
        }
        if (SP && share > 1) {
            const int64_t tile = (int64_t)(b * p.H + h) * p.nQ + qt, first = tile * p.nsplit;
            constexpr uint32_t rows_step = NW * 32 * D * 4, state_step = NW * 32 * 8;
            const HandOver rows(p.ws + first * (rows_step / 4), p.nsplit * rows_step), state(p.ws_ml + first * (state_step / 4), p.nsplit * state_step);
            const uint32_t rows_at = wave_u * (32 * D * 4) + G * NB * 4096 + 16 * lane, state_at = (wave_u * 32 + l32) * 8;
#pragma unroll
            for (int d = 0; d < NB; d++)
#pragma unroll
                for (int g = 0; g < 4; g++)
                    rows.put(s0 * rows_step + rows_at + 1024 * (4 * d + g), f32x4{o[d][4 * g], o[d][4 * g + 1], o[d][4 * g + 2], o[d][4 * g + 3]});
            if (G == 0 && hh == 0) state.put(s0 * state_step + state_at, f32x2{m_i, l_tot});
            if (p.tag == 0) return;
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();  // every wave's rows have been handed over, and LDS has been read
            if (threadIdx.x < 64) {
                const bool all = all_arrived(p.arrivals(NW * 32) + first, p.tag, s0, share);
                if (threadIdx.x == 0) *reinterpret_cast<int *>(smem0) = all;
            }
            __syncthreads();
            if (__builtin_amdgcn_readfirstlane(*reinterpret_cast<int *>(smem0)) == 0) return;
            add_parts<NB, NB == 1 ? 8 : (NB == 2 ? 3 : 2)>(rows, rows_at, rows_step, state, state_at, state_step, share, o, m_i, l_tot);
        }
        const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
        if (G == 0 && p.lse != nullptr && hh == 0)
            p.lse[b * p.lses[0] + h * p.lses[1] + (int64_t)qrow * p.lses[2]] =
                l_tot > 0.f ? (m_i + __builtin_amdgcn_logf(l_tot)) * 0.69314718056f : kNegInf;
        float *orow = reinterpret_cast<float *>(p.o) + b * p.os[0] + h * p.os[1] + (int64_t)qrow * p.os[2] + 4 * hh + 32 * G * NB;
#pragma unroll
        for (int d = 0; d < NB; d++)
#pragma unroll
            for (int g = 0; g < 4; g++)
                *(f32x4 *)(orow + 32 * d + 8 * g) = f32x4{o[d][4 * g] * inv, o[d][4 * g + 1] * inv, o[d][4 * g + 2] * inv, o[d][4 * g + 3] * inv};
    };
    if (KG == 1 || grp == 0) finish(std::integral_constant<int, 0>{});
    else finish(std::integral_constant<int, KG - 1>{});
}

template <int D, int NW, int MODE, bool PK, bool SP, bool SD>
hipError_t launch_lists(const FwdParams &p, hipStream_t stream) {
    constexpr int smem = f32_groups(NW, SP) * f32_group_bytes<D, NW>;
    auto kern = sparse_fwd_f32_mfma_kernel<D, NW, MODE, PK, SP, SD>;
    static unsigned long long attr_done = 0;
    if (const hipError_t e0 = allow_dynamic_smem(kern, smem, attr_done); e0 != hipSuccess) return e0;
    hipLaunchKernelGGL(kern, dim3((unsigned)p.nQ * (unsigned)(p.B * p.H) * (unsigned)(SP ? p.nsplit : 1)),
                       dim3(f32_groups(NW, SP) * NW * 64), smem, stream, p);
    return hipGetLastError();
}

template <int D, int NW, int MODE, bool PK>
hipError_t launch_one(const FwdParams &p, hipStream_t stream) {
    if (p.nsplit > 1) return launch_lists<D, NW, MODE, PK, true, false>(p, stream);
    if constexpr (NW > 1) {
        if (p.spread != 0) return launch_lists<D, NW, MODE, PK, false, true>(p, stream);
    }
    return launch_lists<D, NW, MODE, PK, false, false>(p, stream);
}

template <int D, int NW, bool PK>
hipError_t launch_mode(const FwdParams &p, hipStream_t stream) {
    if (p.BK == 16) return launch_one<D, NW, 0, PK>(p, stream);
    if (p.BK == 32) return launch_one<D, NW, 1, PK>(p, stream);
    return launch_one<D, NW, 2, PK>(p, stream);
}

template <int D, bool PK>
hipError_t launch_bq(const FwdParams &p, int BQ, hipStream_t stream) {
    switch (BQ) {
        case 32:
            // (a lone wave issues all 32 direct loads of a chunk itself; at D = 128 their addresses overflow the scalar
            // registers, and the vector-unit kernel serves that size)
            if constexpr (D > 64) return hipErrorInvalidValue;
            else return launch_mode<D, 1, PK>(p, stream);
        case 64: return launch_mode<D, 2, PK>(p, stream);
        case 128: return launch_mode<D, 4, PK>(p, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

// Whether the matrix-unit kernel takes this float32 call: head dim 64 or 128, BLOCK_Q 32 (head dim 64 only) / 64 / 128, BLOCK_K a power of
// two >= 16 with at most kF32ListCap tiles per row, K/V rows 16-byte aligned, and either packed PARTIAL tiles or a
// bool mask whose rows can be fetched 16 bytes at a time.
bool fwd_f32_mfma_has(const FwdParams &p, int D, int BQ) {
    if ((D != 64 && D != 128) || (BQ != 32 && BQ != 64 && BQ != 128) || (D == 128 && BQ == 32)) return false;
    // (the kernels shift by p.lbk: it must be the logarithm of BLOCK_K)
    if (p.BK < 16 || (p.BK & (p.BK - 1)) || p.lbk < 4 || (1 << p.lbk) != p.BK || p.nK > kF32ListCap) return false;
    if (p.packed != nullptr) return true;
    return p.mask != nullptr && p.ms[3] == 1 && ((uintptr_t)p.mask & 15) == 0 && p.ms[0] % 16 == 0 && p.ms[1] % 16 == 0 &&
           p.ms[2] % 16 == 0;
}

hipError_t launch_fwd_f32_mfma(const FwdParams &p, int D, int BQ, hipStream_t stream) {
    if (!fwd_f32_mfma_has(p, D, BQ)) return hipErrorInvalidValue;
    const hipError_t e = p.packed != nullptr ? (D == 64 ? launch_bq<64, true>(p, BQ, stream) : launch_bq<128, true>(p, BQ, stream))
                                             : (D == 64 ? launch_bq<64, false>(p, BQ, stream) : launch_bq<128, false>(p, BQ, stream));
    return e != hipSuccess || p.nsplit <= 1 || p.tag != 0 ? e : launch_fwd_merge(p, 2, D, BQ, stream);
}

}  // namespace sa
