// Backward pass of the block-sparse attention on gfx950 (MI355X): dQ, dK, dV from dO.
//
// The reference has no backward pass ("Backwards pass + decode kernels", README.md:65); the function differentiated
// is its forward, o = softmax(q k^T * scale + (mask ? 0 : -inf)) v (sparse_attn_kernel.py:149-185), with the row
// log-sum-exp the forward hands out (FwdParams::lse):
//     P = exp(S - lse),  dV = P^T dO,  dP = dO V^T,  dS = P o (dP - rowsum(dO o O)),  dQ = scale dS K,  dK = scale dS^T Q.
//
// Three ways to the gradients, by head dim and size (launch_bwd):
//   D = 64                      sparse_bwd_kernel: a pass for dK and dV together and one for dQ, in one launch
//   D = 128                     sparse_bwd_kernel: a pass each for dK, dQ and dV, in one launch
//   D = 128, bwd_ds_group > 0   sparse_bwd_keys_kernel: dK, dV and dS from one pass over the keys, dS stored;
//                               sparse_bwd_queries_kernel: dQ from the stored dS (bwd_dq_tile)
// All but the last are forms of bwd_tile.  A workgroup owns a tile of 128 RESIDENT rows (queries for dQ, keys for dK
// and dV), 32 per wave, whose operands stay in registers, and walks the list of 64-row tiles of the STREAMED side
// (keys for dQ, queries for dK/dV) that the mask leaves for it: FULL tiles, then PARTIAL ones, as in the forward; for
// dK/dV the lists are those of the transposed mask.  Per 32 streamed rows:
//     S^T  = Y . X^T        Y streamed (K | Q | Q), X resident and pre-scaled (Q | K | K)       -> P^T = exp2(S^T - L)
//     dP^T = Z . G^T        Z streamed (V | dO | -), G resident (dO | V | -)                    -> dS^T = P^T o (dP^T - Delta)
//     acc^T += Y^T . dS^T   (dQ, dK)      or      acc^T += Z^T . P^T   (dV)
// L and Delta belong to the query: per lane when queries are resident, per score register (read from LDS) when they
// are streamed.  Streamed chunks of 64 rows arrive by direct loads global -> LDS in two stages, one barrier per chunk.
// A chunk buffer is read both ways - row-wise as MFMA A operand (ds_read_b128) and transposed (ds_read_b64_tr_b16) -
// so the 16-byte pieces of a row are swizzled with a function of the row that keeps both patterns free of bank
// conflicts (bwd_swizzle).
#include "fwd_common.h"
#include "places.h"

namespace sa {

namespace {

constexpr int kBwdListCap = 2048;  // list entries kept in LDS (streamed length up to 131072)

// XOR applied to the 16-byte piece index of LDS row `row`.
// D = 128 (16 pieces per row, rows 256 bytes apart): bits 0-1 and 2-3 of the row swapped.  16 consecutive rows get 16
// different values (row-wise reads of one piece), and the 4 rows of a transposing read get 4 different 64-byte groups.
// D = 64 (8 pieces, rows 128 bytes apart, so rows of equal parity share their banks): row bit 1 goes to bit 2, bits
// 3 and 2 to bits 1 and 0.  The 8 rows of equal parity among 16 get 8 different values, and the two rows of equal
// parity in a transposing read get different 64-byte groups.
template <int D>
__device__ __forceinline__ int bwd_swizzle(int row) {
    if constexpr (D == 128) return ((row & 3) << 2) | ((row >> 2) & 3);
    else return (((row >> 1) & 1) << 2) | (((row >> 3) & 1) << 1) | ((row >> 2) & 1);
}

// LDS offset of a lane's transposing read of rows 4hh + j, j = 0..3, of d block 0; rows + 8 of them: ^ bwd_tr_rows8, d
// block db: ^ 64 db, rows + 16: + 16 rows.
template <int D>
__device__ __forceinline__ int bwd_tr_base(int lane) {
    const int hh = lane >> 5, j = (lane & 15) >> 2, x = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
    const int grp = D == 128 ? j : (j >> 1);  // the 64-byte-group part of bwd_swizzle(4hh + j); its piece part is hh
    return (4 * hh + j) * D * 2 + 64 * grp + 16 * (x ^ hh) + 8 * (lane & 1);
}
template <int D>
constexpr int bwd_tr_rows8 = 8 * D * 2 + 32;

// What a workgroup makes of its resident tile.
constexpr int kDQ = 0;   // queries resident
constexpr int kDK = 1;   // keys resident, as for the following
constexpr int kDV = 2;
constexpr int kDKV = 3;  // both from one walk: S and P once instead of twice (D = 64, where two accumulators leave room for
                         // more waves per SIMD, and D = 128 where dS is stored)

// LDS, two stages of each: [Y][Z][stats: 64 L then 64 Delta floats][mask: 8 bytes per resident row][list]
template <int D, bool PK>
struct BwdLds {
    static constexpr int NS = 2;
    static constexpr int CBUF = 64 * D * 2;  // one streamed chunk of one tensor
    static constexpr int Z0 = NS * CBUF, STAT0 = 2 * NS * CBUF, MASK0 = STAT0 + NS * 512, LIST0 = MASK0 + (PK ? NS * 1024 : 0);
    static constexpr int bytes = LIST0 + kBwdListCap * 4;
};

// Workgroup -> (plane of the pass, resident tile) as in sparse_fwd_kernel: consecutive workgroup ids go to the 8 XCDs in
// turn, so each XCD gets a contiguous range of the plane-major order (the tiles that share K/V or Q/dO meet in one L2),
// planes two at a time with their tiles interleaved, the tile that is heaviest under causal-like masks first
// (the last queries, the first keys: p.first_tile_first).
struct BwdPlace {
    int plane, rt;
};
template <class P>
__device__ __forceinline__ BwdPlace bwd_place_in_order(const P &p, int lin) {  // lin: in the plane-major order
    int pair = lin / (2 * p.nR);
    const int pr = lin - pair * 2 * p.nR;
    if ((p.planes & 15) == 0) {  // every eighth pair of planes to an XCD: masks that differ per batch element load them alike
        const int ppx = p.planes >> 4;
        const int x = pair / ppx;
        pair = (pair - x * ppx) * 8 + x;
    }
    const bool paired = 2 * pair + 1 < p.planes;
    const int order = paired ? (pr >> 1) : pr;
    return {2 * pair + (paired ? (pr & 1) : 0), p.first_tile_first ? order : p.nR - 1 - order};
}
__device__ __forceinline__ BwdPlace bwd_place(const BwdParams &p, int lin, int total) {
    const int per = total >> 3;
    if (p.spread != 0) {
        const SidePlace at = side_place(8 * side_turn(lin >> 3, per) + (lin & 7), p.spread, p.planes, p.nR);
        return {at.plane, p.first_tile_first ? at.order : p.nR - 1 - at.order};
    }
    return bwd_place_in_order(p, lin < (per << 3) ? (lin & 7) * per + (lin >> 3) : lin);
}

// out = acc * scale; acc holds the transposed tile: lane (row l32, hh), register 4g + jj of block db is
// d = 32 db + 8g + 4hh + jj.  A lane's 8-byte pieces would make every store instruction touch 32 rows, so the wave's 32
// rows go through a private slice `ob` of the (now idle) chunk buffers, rows 16 bytes apart from the banks' period, and
// leave as whole rows, 16 bytes per lane.  o0: the wave's first row, rows os2 elements apart.
template <int D>
constexpr int bwd_out_row = D * 2 + 16;
template <int DT, int D>
__device__ __forceinline__ void bwd_store_rows(const f32x16 (&a)[D / 32], float scale, uint8_t *ob, uint16_t *o0, int64_t os2, int lane) {
    using E = Elem<DT>;
    constexpr int OROW = bwd_out_row<D>, PPR = D / 8;  // 16-byte pieces per row
    const int l32 = lane & 31, hh = lane >> 5;
#pragma unroll
    for (int db = 0; db < D / 32; db++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const u32x2 w = {E::pack2(a[db][4 * g] * scale, a[db][4 * g + 1] * scale),
                             E::pack2(a[db][4 * g + 2] * scale, a[db][4 * g + 3] * scale)};
            *(u32x2 *)(ob + l32 * OROW + 2 * (32 * db + 8 * g + 4 * hh)) = w;
        }
#pragma unroll
    for (int i = 0; i < 32 * PPR / 64; i++) {
        const int idx = 64 * i + lane, r = idx / PPR, pc = idx % PPR;
        const u32x4 x = *(const u32x4 *)(ob + r * OROW + 16 * pc);
        // (written once, whole rows: a streaming store leaves the streamed operands' lines in L2 alone)
        __builtin_nontemporal_store(x, (u32x4 *)(o0 + (int64_t)r * os2 + 8 * pc));
    }
}

// PK: the mask entries of PARTIAL tiles come bit-packed from p.packed, else from the bool mask.  DS (DSM 1; 2: past L2): dS, rounded as it
// enters dK's product, is stored for bwd_dq_tile too (D = 128: both accumulators, K and V take 192 of 256 registers, so that
// S, dP and the reads on their way share the rest: see `phase`).  K then stays unscaled and S - L is scaled in float32 (a rounded
// scale K would give dQ another P than the rounded scale Q of the forward: 3 % more error, this is less than before).
// ORD: the counts come with the tile's place in the order (bwd_sort_tiles), F << 9 | T.
template <int DT, int D, int KIND, bool PK, int PASS, int DSM = 0, bool ORD = false>
__device__ __forceinline__ void bwd_tile(const BwdParams p, int lin, int total, uint8_t *smem, int counts = 0) {
    using E = Elem<DT>;
    static_assert(D == 128 || D == 64, "head dim");
    constexpr bool DS = DSM != 0;
    constexpr int ROWB = D * 2;
    using Lds = BwdLds<D, PK>;
    constexpr int NS = Lds::NS, CBUF = Lds::CBUF, Z0 = Lds::Z0, STAT0 = Lds::STAT0, MASK0 = Lds::MASK0;
    constexpr int NC = D / 16, NDB = D / 32;
    constexpr int PPR = ROWB / 16;   // 16-byte pieces per row
    constexpr int RPI = 64 / PPR;    // rows per wave-wide direct load (1 KiB)
    constexpr int NLD = 16 / RPI;    // direct loads per wave per chunk and tensor
    constexpr bool LANE_STATS = KIND == kDQ;                // queries are the resident side
    constexpr bool OUT_P = KIND == kDV;                     // P and Z enter the output product, nothing else is needed
    constexpr bool BOTH = KIND == kDKV;
    constexpr int NMW = PK ? 1 : 8;                         // mask words per lane and chunk in registers (PK: in LDS)
    int *const ent = reinterpret_cast<int *>(smem + Lds::LIST0);

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l32 = lane & 31, hh = lane >> 5;
    const BwdPlace at = bwd_place(p, lin, total);
    const int plane = at.plane, rt = at.rt, bh = p.plane0 + plane;
    const int b = bh / p.H, h = bh - b * p.H;
    const int rrow = rt * 128 + wave * 32 + l32;

    const uint16_t *ybase = p.y + b * p.ys[0] + h * p.ys[1];
    const uint16_t *zbase = p.z + b * p.zs[0] + h * p.zs[1];
    const int32_t *fid = p.full_ids + b * p.fis[0] + h * p.fis[1] + rt * p.fis[2];
    const int32_t *pid = p.part_ids + b * p.pis[0] + h * p.pis[1] + rt * p.pis[2];
    const uint8_t *mrow = PK ? nullptr : p.mask + b * p.ms[0] + h * p.ms[1] + (int64_t)rrow * p.mrs;
    // packed tiles: 8 bytes per row, 1024 per tile, nS tiles per resident tile; a lane's four bytes of its wave's 32 rows
    const uint8_t *prow = PK ? p.packed + b * p.pks[0] + h * p.pks[1] + (int64_t)rt * p.nS * 1024 : nullptr;
    const float *statL = p.stat_l + b * p.sts[0] + h * p.sts[1];
    const float *statD = p.stat_d + b * p.sts[0] + h * p.sts[1];
    // bytes from a query's L to its Delta (both live in one workspace, less than 4 GiB apart)
    const uint32_t stat_gap = (uint32_t)((const uint8_t *)p.stat_d - (const uint8_t *)p.stat_l);

    // resident operands: lane (l32, hh) keeps d = 16c + 8hh .. +7 of its row; X carries the softmax scale / ln 2
    u32x4 xf[NC], gf[OUT_P ? 1 : NC];
    {
        const uint16_t *xp = p.x + b * p.xs[0] + h * p.xs[1] + (int64_t)rrow * p.xs[2] + 8 * hh;
#pragma unroll
        for (int c = 0; c < NC; c++) {
            xf[c] = *(const u32x4 *)(xp + 16 * c);
#pragma unroll
            for (int e = 0; e < 4; e++)
                if constexpr (!DS) xf[c][e] = E::scale2(xf[c][e], p.scale);
        }
        if constexpr (!OUT_P) {
            const uint16_t *gp = p.g + b * p.gs[0] + h * p.gs[1] + (int64_t)rrow * p.gs[2] + 8 * hh;
#pragma unroll
            for (int c = 0; c < NC; c++) gf[c] = *(const u32x4 *)(gp + 16 * c);
        }
    }
    float laneL = 0.f, laneD = 0.f;
    if constexpr (LANE_STATS) {
        laneL = statL[(int64_t)rrow * p.sts[2]];
        laneD = statD[(int64_t)rrow * p.sts[2]];
    }
    // Counts and tile indices are clamped to the nS streamed tiles there are (the reference guards every K/V and mask
    // load with kv_offset < SEQLEN_K, sparse_attn_kernel.py:35,39,60): stale or foreign metadata then gives wrong
    // numbers, never an access outside the tensors or past the list's LDS copy (nS <= kBwdListCap, checked by the host).
    int F, T;  // chunks = list entries
    if constexpr (ORD) {
        F = counts >> 9;
        T = counts & 511;
    } else {
        int cnt[2];
        const int32_t *const cnt_addr[2] = {p.full_lens + (b * p.fls[0] + h * p.fls[1] + rt * p.fls[2]),
                                            p.part_lens + (b * p.pls[0] + h * p.pls[1] + rt * p.pls[2])};
        scalar_gather(cnt_addr, cnt);
        F = min(max(cnt[0], 0), p.nS);
        T = F + min(max(cnt[1], 0), p.nS - F);
    }
    f32x16 acc[NDB], acc2[BOTH ? NDB : 1];  // acc2: dV beside dK
#pragma unroll
    for (int db = 0; db < NDB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            acc[db][i] = 0.f;
            if constexpr (BOTH) acc2[db][i] = 0.f;
        }

    // LDS offsets inside a chunk buffer: row-wise operand reads (row 32kb + l32, piece 2c + hh) and transposing
    // reads (rows 16kc + 4hh + j and + 8 of a 32-row block, 32-wide d block db), both through bwd_swizzle.  The
    // swizzle being an XOR, so are the steps from one piece, row group or d block to the next.
    const int nbase = l32 * ROWB + 16 * (hh ^ bwd_swizzle<D>(l32));
    const int tbase = bwd_tr_base<D>(lane);
    // direct loads: load i of this wave fills rows RPI (4i + wave) .. + RPI - 1 of the chunk; the lane writes LDS
    // piece lane % PPR of its row and therefore fetches the swizzled source piece
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const SA_LDS uint8_t *)smem);
    // (rows 4 RPI apart have the same swizzle, so the loads differ by a scalar)
    const int ld_row = RPI * wave_u + lane / PPR, ld_piece = (lane % PPR) ^ bwd_swizzle<D>(ld_row);
    const uint32_t ld_yoff = (uint32_t)((ld_row * p.ys[2] + 8 * ld_piece) * 2);
    const uint32_t ld_zoff = (uint32_t)((ld_row * p.zs[2] + 8 * ld_piece) * 2);

    // the tile's list (FULL entries, then PARTIAL ones) as first streamed rows
    for (int e = tid; e < T; e += 256) {
        const int idx = e < F ? fid[(int64_t)e * p.fis[3]] : pid[(int64_t)(e - F) * p.pis[3]];
        ent[e] = min(max(idx, 0), p.nS - 1) << 6;
    }
    __syncthreads();

    // where this wave's keys' dS of the 64 queries from ent[t] goes: 4 KiB in a row
    const int64_t ds_row = (int64_t)p.nR * 2 * 16384;  // all keys of 128 queries
    uint8_t *const ds0 = DS ? p.ds + (int64_t)plane * (p.nS >> 1) * ds_row + (2 * rt + (wave_u >> 1)) * 16384 + (wave_u & 1) * 8192 : nullptr;
    auto ds_out = [&](int t) {
        const int row = __builtin_amdgcn_readfirstlane(ent[t]);
        return ds0 + (row >> 7) * ds_row + ((row & 64) << 6);
    };

    // everything chunk t needs from memory, into stage st
    auto issue = [&](int t, int st, uint32_t(&mk)[NMW]) {
        int ln = lane;
        if constexpr (DS) asm volatile("" : "+v"(ln));
        const int col = __builtin_amdgcn_readfirstlane(ent[t]);
#pragma unroll
        for (int i = 0; i < NLD; i++) {
            const uint32_t dst = 1024 * (4 * i + wave_u);  // RPI rows per load
            dma16(ybase + (int64_t)(col + 4 * RPI * i) * p.ys[2], ld_yoff, lds0 + st * CBUF + dst);
            dma16(zbase + (int64_t)(col + 4 * RPI * i) * p.zs[2], ld_zoff, lds0 + Z0 + st * CBUF + dst);
        }
        if constexpr (!LANE_STATS) {
            if (wave_u == 0 && ln < 32) {  // 64 L values, then 64 Delta values, 16 bytes per lane (row stride 1)
                const uint32_t off = (ln < 16 ? 0u : stat_gap) + 16u * (ln & 15);
                dma16(statL + col, off, lds0 + STAT0 + st * 512);
            }
        }
        if (t >= F) {
            if constexpr (PK) {  // the rows' bits of the tile in slot t - F, every wave those of its own rows
                dma4(prow + (int64_t)(t - F) * 1024 + wave_u * 256, 4 * ln, lds0 + MASK0 + st * 1024 + wave_u * 256);
            } else {
#pragma unroll
                for (int kb = 0; kb < 2; kb++)
#pragma unroll
                    for (int g = 0; g < 4; g++) {
                        const int64_t cc = col + 32 * kb + 8 * g + 4 * hh;
                        if (p.mask_vec4) {
                            mk[4 * kb + g] = *(const uint32_t *)(mrow + cc);
                        } else {
                            const uint8_t *m0 = mrow + cc * p.mcs;
                            mk[4 * kb + g] = (uint32_t)m0[0] | ((uint32_t)m0[p.mcs] << 8) | ((uint32_t)m0[2 * p.mcs] << 16) |
                                             ((uint32_t)m0[3 * p.mcs] << 24);
                        }
                    }
            }
        }
    };

    auto compute = [&](int t, int st, const uint32_t(&mk)[NMW]) {
        // Two accumulators of D = 128 leave no register over: the offsets are made anew from their bases per phase (kept,
        // they spill), and no phase's reads move into another.
        uint32_t nb = lds0 + nbase, tb0 = lds0 + tbase, sb = lds0 + STAT0 + 16 * hh;
        int ln = lane;
        auto phase = [&] {
            if constexpr (DS) {
                __builtin_amdgcn_sched_barrier(0);
                asm volatile("" : "+v"(nb), "+v"(tb0), "+v"(ln));
                sb = lds0 + STAT0 + 16 * (ln >> 5);
            }
        };
        constexpr int kAhead = 4;
        auto paced = [] {  // operand reads this far ahead of the products
            if constexpr (DS) {
                __builtin_amdgcn_sched_group_barrier(0x100, 4 + kAhead, 0);
                static_for<NC - kAhead>([](auto) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                });
                __builtin_amdgcn_sched_group_barrier(0x008, kAhead, 0);
            }
        };
        phase();
        constexpr auto lds = [](uint32_t a) { return (const SA_LDS uint8_t *)(uintptr_t)a; };
        const uint32_t yb = st * CBUF, zb = Z0 + st * CBUF;
        static_for<2>([&](auto kb_c) {
            constexpr int kb = decltype(kb_c)::value;
            // the products start from -L and -Delta where those come with the streamed rows, from zero where they are the lane's
            f32x16 s, dp;
            auto start = [&](f32x16 &a, int which) {
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    f32x4 x = {0.f, 0.f, 0.f, 0.f};
                    if constexpr (!LANE_STATS) x = *(const SA_LDS f32x4 *)lds(sb + st * 512 + 256 * which + 128 * kb + 32 * g);
#pragma unroll
                    for (int jj = 0; jj < 4; jj++) a[4 * g + jj] = x[jj];
                }
            };
            start(s, 0);
#pragma unroll
            for (int c = 0; c < NC; c++) s = E::mfma(*(const SA_LDS u32x4 *)lds((nb ^ (32 * c)) + yb + 32 * kb * ROWB), xf[c], s);
            if constexpr (DS) asm volatile("" : "+v"(s));
            paced();
            phase();
            if constexpr (!OUT_P) {
                start(dp, 1);
#pragma unroll
                for (int c = 0; c < NC; c++) dp = E::mfma(*(const SA_LDS u32x4 *)lds((nb ^ (32 * c)) + zb + 32 * kb * ROWB), gf[c], dp);
            }
            if constexpr (DS) asm volatile("" : "+v"(s), "+v"(dp));
            paced();
            phase();
            if (t >= F) {
                // w: bit 8g + jj says whether this lane's entry (streamed row 32kb + 8g + 4hh + jj) attends
                uint32_t w;
                if constexpr (PK) {  // bit k of the packed word: streamed row 32kb + k
                    w = *(const SA_LDS uint32_t *)lds(lds0 + MASK0 + st * 1024 + wave_u * 256 + 8 * (ln & 31) + 4 * kb) >> (4 * (ln >> 5));
                } else {  // one byte per entry: the non-zero bytes of each dword become four bits
                    w = 0u;
#pragma unroll
                    for (int g = 0; g < 4; g++) {
                        const uint32_t m = mk[4 * kb + g];
                        const uint32_t nz = ((((m & 0x7f7f7f7fu) + 0x7f7f7f7fu) | m) >> 7) & 0x01010101u;
                        w |= ((nz * 0x01020408u) >> 24) << (8 * g);
                    }
                }
#pragma unroll
                for (int g = 0; g < 4; g++)
#pragma unroll
                    for (int jj = 0; jj < 4; jj++)
                        if (((w >> (8 * g + jj)) & 1u) == 0u) s[4 * g + jj] = kNegInf;
            }
            // P^T = exp2(S^T - L) and, unless OUT_P, dS^T = P^T o (dP^T - Delta); rounded to the input type
            uint32_t pw[8], pp[BOTH ? 8 : 1];
#pragma unroll
            for (int g = 0; g < 4; g++) {
                float w[4], pv[4];
#pragma unroll
                for (int jj = 0; jj < 4; jj++) {
                    const float pr = __builtin_amdgcn_exp2f(LANE_STATS ? s[4 * g + jj] + laneL : DS ? s[4 * g + jj] * p.scale : s[4 * g + jj]);
                    pv[jj] = pr;
                    w[jj] = OUT_P ? pr : pr * (LANE_STATS ? dp[4 * g + jj] + laneD : dp[4 * g + jj]);
                }
                pw[2 * g] = E::pack2(w[0], w[1]);
                pw[2 * g + 1] = E::pack2(w[2], w[3]);
                if constexpr (BOTH) {
                    pp[2 * g] = E::pack2(pv[0], pv[1]);
                    pp[2 * g + 1] = E::pack2(pv[2], pv[3]);
                }
            }
            if constexpr (DS) {  // (the order of the pieces: bwd_dq_tile)
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    uint8_t *const to = ds_out(t) + 2048 * kb + 1024 * c + (uint32_t)((32 * (ln & 31) + 16 * (ln >> 5)) ^ (128 * c));
                    const u32x4 x = {pw[4 * c], pw[4 * c + 1], pw[4 * c + 2], pw[4 * c + 3]};
                    if constexpr (DSM == 2) __builtin_nontemporal_store(x, (u32x4 *)to);
                    else *(u32x4 *)to = x;
                }
            }
            phase();
            const uint32_t tb = (OUT_P ? zb : yb) + 32 * kb * ROWB;
            static_for<2>([&](auto kc_c) {
                constexpr int kc = decltype(kc_c)::value;
                const u32x4 pk4 = u32x4{pw[4 * kc], pw[4 * kc + 1], pw[4 * kc + 2], pw[4 * kc + 3]};
#pragma unroll
                for (int db = 0; db < NDB; db++) {
                    const u32x2 lo = E::tr_read(lds((tb0 ^ (64 * db)) + tb + 16 * kc * ROWB));
                    const u32x2 hi = E::tr_read(lds((tb0 ^ (64 * db) ^ bwd_tr_rows8<D>) + tb + 16 * kc * ROWB));
                    acc[db] = E::mfma(u32x4{lo.x, lo.y, hi.x, hi.y}, pk4, acc[db]);
                }
                phase();
                if constexpr (BOTH) {
                    const uint32_t vb = zb + 32 * kb * ROWB;
                    const u32x4 pp4 = u32x4{pp[4 * kc], pp[4 * kc + 1], pp[4 * kc + 2], pp[4 * kc + 3]};
#pragma unroll
                    for (int db = 0; db < NDB; db++) {
                        const u32x2 lo = E::tr_read(lds((tb0 ^ (64 * db)) + vb + 16 * kc * ROWB));
                        const u32x2 hi = E::tr_read(lds((tb0 ^ (64 * db) ^ bwd_tr_rows8<D>) + vb + 16 * kc * ROWB));
                        acc2[db] = E::mfma(u32x4{lo.x, lo.y, hi.x, hi.y}, pp4, acc2[db]);
                    }
                }
                phase();
            });
        });
    };

    {
        uint32_t mk[NS][NMW];
#pragma unroll
        for (int j = 0; j < NS; j++)
#pragma unroll
            for (int i = 0; i < NMW; i++) mk[j][i] = 0u;
        // The resident operands were requested before the list and have landed with it.  "Used" here, they are no loads any
        // more to the compiler, whose wait in front of their first use in the loop would take the direct loads of the
        // chunks behind along, in every trip.
#pragma unroll
        for (int c = 0; c < NC; c++) asm volatile("" : "+v"(xf[c]));
        if constexpr (!OUT_P) {
#pragma unroll
            for (int c = 0; c < NC; c++) asm volatile("" : "+v"(gf[c]));
        }
        if constexpr (LANE_STATS) asm volatile("" : "+v"(laneL), "+v"(laneD));
        if (T > 0) issue(0, 0, mk[0]);
        if constexpr (DS) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        for (int t0 = 0; t0 < T; t0 += NS) {
            static_for<NS>([&](auto jc) {
                constexpr int j = decltype(jc)::value, jn = j ^ 1;
                const int t = t0 + j;
                if (t >= T) return;
                // own pieces of chunk t and its mask words; four stores of dS came after their requests
                if constexpr (DS) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
                else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                if constexpr (!PK) {
#pragma unroll
                    for (int i = 0; i < NMW; i++) asm volatile("" ::"v"(mk[j][i]));
                }
                __syncthreads();  // everyone's pieces; and everyone is done with the other stage
                if (t + 1 < T) issue(t + 1, jn, mk[jn]);
                compute(t, j, mk[j]);
            });
        }
    }

    __syncthreads();  // every wave is done with the chunk buffers
    static_assert(4 * 32 * bwd_out_row<D> <= 2 * NS * CBUF, "the rows of the four waves fit the chunk buffers");
    uint8_t *const ob = smem + wave_u * 32 * bwd_out_row<D>;
    int ln = lane;
    if constexpr (DS) asm volatile("" : "+v"(ln));
    // Where the rows go is read from the argument block only now (the pointer passes through an asm statement): held in
    // scalar registers through the loop these strides had others spilled.
    typedef const __attribute__((address_space(4))) BwdLaunch *ArgPtr;
    ArgPtr args = (ArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(args));
    auto store = [&](const f32x16(&a)[NDB], float scale, uint16_t *out, int64_t os0, int64_t os1, int64_t os2) {
        bwd_store_rows<DT, D>(a, scale, ob, out + b * os0 + h * os1 + (int64_t)(rt * 128 + wave_u * 32) * os2, os2, ln);
    };
    store(acc, args->pass[PASS].out_scale, args->pass[PASS].out, args->pass[PASS].outs[0], args->pass[PASS].outs[1], args->pass[PASS].outs[2]);
    if constexpr (BOTH)  // (a wave's slice is its own: its reads above come first)
        store(acc2, 1.f, args->pass[PASS].out2, args->pass[PASS].outs2[0], args->pass[PASS].outs2[1], args->pass[PASS].outs2[2]);
}

// dQ from the dS that the pass over the keys stored: dQ^T += K^T . dS^T, one product instead of three, bound by the reads
// of dS (B8 H16 S4096 causal: 2.2 GB in 487 us, 4.5 TB/s, and 312 us with the same dS from L2, so neither the products nor the
// loads into LDS bound it; every key: 4.3 GB in 741 us, 5.8 TB/s).  128 queries per workgroup, 32 per wave; a chunk of 64 keys is
// 16 KiB of K, shared, and 4 KiB of dS per wave.  More of dS on its way does not help (causal: a fifth wave for K, which leaves
// LDS for 80 instead of 48 KiB of dS per compute unit, +9 us; dS through registers, 96 ... 160 KiB, +30 ... +100 us; the next
// step's requests behind this one's LDS reads +5 us; two stages and four workgroups per compute unit +30 us).
// dS lies as [plane][128 queries][64 keys][halves of 32 keys][32 queries][32 keys]: what a workgroup here reads in a step is 8 KiB
// in a row, and what a wave of the key pass stores of a chunk 4 KiB (pieces of 2 KiB 4 KiB apart before: causal 498 -> 493 us).  Where
// there is more of it than the caches hold (kDsFar) it is stored past L2, where Q and dO are read again and again (key pass 1156 -> 1141 us,
// reads from beyond L2 1.4 -> 0.76 GB; this pass 493 -> 487), and the planes are walked from the last one the key pass wrote, whose dS the
// memory-side cache still holds (520 -> 498).  All three together: every key 941 -> 741 us.  In the 2 KiB of the last two,
// key k's queries 8g + 4h .. + 3 are the 8 bytes at 1024 (g / 2) + ((32 k + 16 h) ^ 128 (g / 2)) + 8 (g & 1): the key
// pass stores 1 KiB per instruction, and a transposing read (four keys, two groups of 16 queries) meets no bank twice.
// A block that the key pass did not visit holds whatever the memory held: none of its entries attends, so it lies in
// PARTIAL tiles only, where the entries that do not attend are set to zero here.
template <int D>
struct BwdDqLds {
    static constexpr int NST = 4, SBUF = 32 * D * 2;  // stages, and bytes of K in one; of dS as many at D = 128
    static constexpr int DS0 = NST * SBUF, MASK0 = DS0 + NST * 8192, LIST0 = MASK0 + 4096, bytes = LIST0 + kBwdListCap * 2;
};
template <int DT, int D>
__device__ __forceinline__ void bwd_dq_tile(const BwdParams &p, int lin, int total, uint8_t *smem) {
    using E = Elem<DT>;
    using Lds = BwdDqLds<D>;
    constexpr int ROWB = D * 2, NDB = D / 32, PPR = ROWB / 16, RPI = 64 / PPR, SLD = 8 / RPI;
    constexpr int NST = Lds::NST, SBUF = Lds::SBUF, DS0 = Lds::DS0, MASK0 = Lds::MASK0;
    uint16_t *const ent = reinterpret_cast<uint16_t *>(smem + Lds::LIST0);
    const int tid = threadIdx.x, lane = tid & 63, wave_u = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, hh = lane >> 5;
    const BwdPlace at = bwd_place(p, lin, total);
    const int plane = p.far ? p.planes - 1 - at.plane /* (last written first) */ : at.plane, rt = at.rt, bh = p.plane0 + plane;
    const int b = bh / p.H, h = bh - b * p.H;
    const uint16_t *ybase = p.y + b * p.ys[0] + h * p.ys[1];
    const int32_t *fid = p.full_ids + b * p.fis[0] + h * p.fis[1] + rt * p.fis[2];
    const int32_t *pid = p.part_ids + b * p.pis[0] + h * p.pis[1] + rt * p.pis[2];
    const uint8_t *prow = p.packed + b * p.pks[0] + h * p.pks[1] + (int64_t)rt * p.nS * 1024 + wave_u * 256;
    const uint8_t *dsbase = p.ds + ((int64_t)plane * p.nR + rt) * p.nS * 16384 + wave_u * 2048;
    int cnt[2];  // (clamped as in bwd_tile)
    const int32_t *const cnt_addr[2] = {p.full_lens + (b * p.fls[0] + h * p.fls[1] + rt * p.fls[2]),
                                        p.part_lens + (b * p.pls[0] + h * p.pls[1] + rt * p.pls[2])};
    scalar_gather(cnt_addr, cnt);
    const int F = min(max(cnt[0], 0), p.nS);
    const int T = F + min(max(cnt[1], 0), p.nS - F);
    f32x16 acc[NDB];
#pragma unroll
    for (int db = 0; db < NDB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[db][i] = 0.f;
    const int tbase = bwd_tr_base<D>(lane);
    const int cq = (lane >> 4) & 1;
    const int dbase = 1024 * cq + 128 * (hh ^ cq) + 32 * ((lane & 15) >> 2) + 16 * (lane & 1) + 8 * ((lane >> 1) & 1);
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const SA_LDS uint8_t *)smem);
    const int ld_row = RPI * wave_u + lane / PPR, ld_piece = (lane % PPR) ^ bwd_swizzle<D>(ld_row);
    const uint32_t ld_yoff = (uint32_t)((ld_row * p.ys[2] + 8 * ld_piece) * 2);
    for (int e = tid; e < T; e += 256) {
        const int idx = e < F ? fid[(int64_t)e * p.fis[3]] : pid[(int64_t)(e - F) * p.pis[3]];
        ent[e] = (uint16_t)min(max(idx, 0), p.nS - 1);
    }
    __syncthreads();
    // Steps of 32 keys, two per list entry.
    const int64_t ytile = 64 * p.ys[2], yhalf = 32 * p.ys[2], yload = 4 * RPI * p.ys[2];
    auto issue = [&](int u, int st) {
        const int t = u >> 1, kt = __builtin_amdgcn_readfirstlane(ent[t]);
        const uint8_t *dsp = dsbase + (int64_t)kt * 16384 + (u & 1) * 8192;
        if (t >= F && (u & 1) == 0) dma4(prow + (int64_t)(t - F) * 1024, 4 * lane, lds0 + MASK0 + (t & 3) * 1024 + wave_u * 256);
#pragma unroll
        for (int i = 0; i < 2; i++) dma16<true>(dsp + 1024 * i, 16 * lane, lds0 + DS0 + st * 8192 + wave_u * 2048 + 1024 * i);
        const uint16_t *yp = ybase + kt * ytile + ((u & 1) ? yhalf : 0);
#pragma unroll
        for (int i = 0; i < SLD; i++) dma16(yp + i * yload, ld_yoff, lds0 + st * SBUF + 1024 * (4 * i + wave_u));
    };
    auto compute = [&](int u, int st) {
        const uint8_t *yb = smem + st * SBUF, *db_ = smem + DS0 + st * 8192 + wave_u * 2048 + dbase;
        u32x4 x[2];  // dS^T of keys 16kc ..
#pragma unroll
        for (int kc = 0; kc < 2; kc++) {
            const u32x2 lo = E::tr_read(db_ + 512 * kc), hi = E::tr_read(db_ + 512 * kc + 256);
            x[kc] = u32x4{lo.x, lo.y, hi.x, hi.y};
        }
        const int t = u >> 1;
        if (t >= F) {  // bit k of the packed word: key k of the step
            const uint32_t w = *(const uint32_t *)(smem + MASK0 + (t & 3) * 1024 + wave_u * 256 + 8 * l32 + 4 * (u & 1)) >> (4 * hh);
#pragma unroll
            for (int kc = 0; kc < 2; kc++)
#pragma unroll
                for (int d = 0; d < 4; d++) {
                    const uint32_t two = w >> (16 * kc + 8 * (d >> 1) + 2 * (d & 1));
                    x[kc][d] &= ((two & 1u) ? 0xffffu : 0u) | ((two & 2u) ? 0xffff0000u : 0u);
                }
        }
#pragma unroll
        for (int kc = 0; kc < 2; kc++)
#pragma unroll
            for (int db = 0; db < NDB; db++) {
                const uint8_t *tb = yb + 16 * kc * ROWB;
                const u32x2 klo = E::tr_read(tb + (tbase ^ (64 * db)));
                const u32x2 khi = E::tr_read(tb + (tbase ^ (64 * db) ^ bwd_tr_rows8<D>));
                acc[db] = E::mfma(u32x4{klo.x, klo.y, khi.x, khi.y}, x[kc], acc[db]);
            }
    };
    const int U = 2 * T;
#pragma unroll
    for (int u = 0; u < NST - 1; u++)
        if (u < U) issue(u, u);
    for (int u0 = 0; u0 < U; u0 += NST) {
        static_for<NST>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            const int u = u0 + j;
            if (u >= U) return;
            // own pieces of step u: behind them are the loads of at most two steps, four or (with mask words) five each
            if (u + 2 < U) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * (2 + SLD)) : "memory");
            else if (u + 1 < U) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 + SLD) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();  // everyone's pieces; and everyone is done with the stage of step u - 1
            if (u + NST - 1 < U) issue(u + NST - 1, (j + NST - 1) % NST);
            compute(u, j);
        });
    }
    __syncthreads();
    bwd_store_rows<DT, D>(acc, p.out_scale, smem + wave_u * 32 * bwd_out_row<D>,
                          p.out + b * p.outs[0] + h * p.outs[1] + (int64_t)(rt * 128 + wave_u * 32) * p.outs[2], p.outs[2], lane);
}

// D = 64 with packed tiles: three workgroups per compute unit (168 registers, 43 KB of LDS; a third stage of the chunks
// beside two of them instead: 2 ... 14 % slower).  Both passes of B4 H12 S2048 documents: 125 us as three launches with dK
// and dV apart, 80 us now; causal B8 H12 S4096 910 -> 753 us; D = 128 causal B4 H16 S2048 358 -> 315, B2 H8 S1024 97 -> 41 us.
// All passes in one launch: a launch each would leave the device to the last tiles of every pass, and passes of fewer tiles
// than workgroup slots would run one after the other (B2 H8 S1024: 128 tiles a pass on 512 slots).  The passes whose
// tiles take longest come first; every pass starts at a multiple of eight workgroups, so that the plane-to-XCD mapping of
// bwd_tile holds for each.
// ORD: the tiles come by falling cost (l.order).
template <int DT, int D, bool PK, bool ORD>
__global__ __launch_bounds__(256, D == 64 && PK ? 3 : 2) void sparse_bwd_kernel(const BwdLaunch l) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    const int id = blockIdx.x;
    int pass = 0, lin = id, counts = 0;  // lin: workgroup of its pass, as bwd_place takes it
    if constexpr (ORD) {
        const int e = __builtin_amdgcn_readfirstlane(l.order[(id & 7) * l.slots + (id >> 3)]);
        pass = e >> 29;
        lin = (e >> 18 & 2047) * 8 + (id & 7);
        counts = e & 0x3ffff;
    } else if (D != 64 && id >= l.first[2]) {
        pass = 2;
        lin = id - l.first[2];
    } else if (id >= l.first[1]) {
        pass = 1;
        lin = id - l.first[1];
    }
    if (pass == 0) {
        if (lin < l.tiles[0]) bwd_tile<DT, D, D == 64 ? kDKV : kDK, PK, 0, 0, ORD>(l.pass[0], lin, l.tiles[0], smem, counts);
    } else if (D == 64 || pass == 1) {
        if (lin < l.tiles[1]) bwd_tile<DT, D, kDQ, PK, 1, 0, ORD>(l.pass[1], lin, l.tiles[1], smem, counts);
    } else {
        if constexpr (D != 64) bwd_tile<DT, D, kDV, PK, 2, 0, ORD>(l.pass[2], lin, l.tiles[2], smem, counts);
    }
}

// dK, dV and dS from one walk over the keys' lists.  FAR: dS is larger than the caches (kDsFar) and stored past L2.
template <int DT, bool FAR>
__global__ __launch_bounds__(256, 2) void sparse_bwd_keys_kernel(const BwdLaunch l) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    bwd_tile<DT, 128, kDKV, true, 0, FAR ? 2 : 1>(l.pass[0], blockIdx.x, l.tiles[0], smem);
}

// dQ from the stored dS.  LDS: [K, four stages][dS, four stages][mask words of four entries][list]
template <int DT, int D>
__global__ __launch_bounds__(256, 2) void sparse_bwd_queries_kernel(const BwdParams p, int tiles) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    bwd_dq_tile<DT, D>(p, blockIdx.x, tiles, smem);
}

// Per query row: -Delta = -sum_d dO o O, and -L = -lse / ln 2 (-inf for rows that attended to nothing, so that their
// P = exp2(S - L) is 0).  D/8 lanes per row, 8 elements each.
// In front of them, where the passes take their tiles by falling cost, eight workgroups sort one XCD's tiles each: a counting sort over
// 32 classes of cost by eighths of the XCD's tiles, the passes one after the other in the order of planes (neighbours share operands; within
// one in any order: each tile's result is its own).  A tile's counts go with its place, so that its start is no read longer.
constexpr int kCosts = 256, kOrderMost = 2048;
__device__ __forceinline__ void bwd_sort_tiles(const BwdOrderParams &o, int xcd) {
    __shared__ int32_t entry[kOrderMost];
    __shared__ uint16_t cost[kOrderMost];
    __shared__ int count[kCosts], of_wave[4], least_of[3], most_of[3];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (tid < 3) {
        least_of[tid] = 0x7fffffff;
        most_of[tid] = 0;
    }
    count[tid] = 0;
    __syncthreads();
    {  // one pass per wave (its arguments are scalars then), the passes' tiles one after the other
        const int pass = wave % o.n, waves = (4 - pass + o.n - 1) / o.n;
        const BwdOrderParams::Pass &q = o.pass[pass];
        const int tiles = q.planes * q.nR >> 3;
        int first = 0, least = 0x7fffffff, most = 0;
        for (int n = 0; n < pass; n++) first += o.pass[n].planes * o.pass[n].nR >> 3;
        for (int k = 64 * (wave / o.n) + lane; k < tiles; k += 64 * waves) {
            const BwdPlace at = bwd_place_in_order(q, xcd * tiles + k);
            const int b = at.plane / q.H, h = at.plane - b * q.H;
            const int f = q.full_lens[b * q.fls[0] + h * q.fls[1] + at.rt * q.fls[2]], m = q.part_lens[b * q.pls[0] + h * q.pls[1] + at.rt * q.pls[2]];
            const int F = min(max(f, 0), q.nS), T = F + min(max(m, 0), q.nS - F);  // (clamped as in bwd_tile; below 512: bwd_order_bytes)
            const int c = min(q.fixed + q.per_entry * T, 0xffff);
            cost[first + k] = (uint16_t)c;
            entry[first + k] = pass << 29 | k << 18 | F << 9 | T;
            least = min(least, c);
            most = max(most, c);
        }
#pragma unroll
        for (int s = 1; s < 64; s <<= 1) {
            least = min(least, __shfl_xor(least, s));
            most = max(most, __shfl_xor(most, s));
        }
        if (lane == 0) {
            atomicMin(&least_of[pass], least);
            atomicMax(&most_of[pass], most);
        }
    }
    __syncthreads();
    bool alike = true;  // lists of about one length: the order of planes, whose neighbours share operands, is the better one
    for (int n = 0; n < o.n; n++) alike = alike && 4 * (most_of[n] - least_of[n]) <= most_of[n];
    if (alike) {
        for (int i = tid; i < o.slots; i += 256) o.order[xcd * o.slots + i] = entry[i];
        return;
    }
    const int most = max(max(most_of[0], most_of[1]), most_of[2]);
    auto cls = [&](int i) { return 8 * (31 - (int)((unsigned)cost[i] * 31u / (unsigned)most)) + 8 * i / o.slots; };
    for (int i = tid; i < o.slots; i += 256) atomicAdd(&count[cls(i)], 1);
    __syncthreads();
    const int mine = count[tid];
    int upto = mine;  // of the wave's classes up to this one
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
        const int x = __shfl_up(upto, s);
        if (lane >= s) upto += x;
    }
    if (lane == 63) of_wave[tid >> 6] = upto;
    __syncthreads();
    for (int w = 0; w < tid >> 6; w++) upto += of_wave[w];
    count[tid] = upto - mine;
    __syncthreads();
    for (int i = tid; i < o.slots; i += 256) o.order[xcd * o.slots + atomicAdd(&count[cls(i)], 1)] = entry[i];
}
template <int DT, int D, bool ORD>
__global__ __launch_bounds__(256) void bwd_prepare_kernel(const BwdPrepParams p) {
    constexpr int LPR = D / 8;  // lanes per row
    int block = blockIdx.x;
    if constexpr (ORD) {
        if (block < 8) return bwd_sort_tiles(p.order, block);
        block -= 8;
    }
    const int64_t row = (int64_t)block * (256 / LPR) + threadIdx.x / LPR;
    const int part = threadIdx.x % LPR;
    if (row >= (int64_t)p.B * p.H * p.Sq) return;
    const int q = (int)(row % p.Sq);
    const int bh = (int)(row / p.Sq);
    const int b = bh / p.H, h = bh - b * p.H;
    // (read once, whole rows: streaming loads, which this device serves faster than loads that keep their lines in L2)
    const u32x4 a = __builtin_nontemporal_load((const u32x4 *)(p.o + b * p.os[0] + h * p.os[1] + (int64_t)q * p.os[2] + 8 * part));
    const u32x4 g = __builtin_nontemporal_load((const u32x4 *)(p.d_o + b * p.dos[0] + h * p.dos[1] + (int64_t)q * p.dos[2] + 8 * part));
    float sum = 0.f;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const uint32_t ae = a[e], ge = g[e];  // (a bit cast applied to the vector element itself reads element 0)
        if constexpr (DT == 0) {
            sum += __uint_as_float(ae << 16) * __uint_as_float(ge << 16);
            sum += __uint_as_float(ae & 0xffff0000u) * __uint_as_float(ge & 0xffff0000u);
        } else {
            const f16x2 x = __builtin_bit_cast(f16x2, ae), y = __builtin_bit_cast(f16x2, ge);
            sum += (float)x.x * (float)y.x + (float)x.y * (float)y.y;
        }
    }
#pragma unroll
    for (int m = LPR / 2; m >= 1; m >>= 1) sum += __shfl_xor(sum, m, LPR);
    if (part == 0) {
        const float lse = p.lse[b * p.ls[0] + h * p.ls[1] + (int64_t)q * p.ls[2]];
        p.stat_l[row] = lse == kNegInf ? kNegInf : lse * p.l_mul;
        p.stat_d[row] = -sum;
    }
}

template <int DT, int D, bool PK, bool ORD>
hipError_t launch_bwd_one(const BwdParams &dq, const BwdParams &dk, const BwdParams &dv, const BwdOrderParams &ord, hipStream_t stream) {
    constexpr int smem = BwdLds<D, PK>::bytes;
    auto kern = sparse_bwd_kernel<DT, D, PK, ORD>;
    static unsigned long long attr_done = 0;
    if (const hipError_t e0 = allow_dynamic_smem(kern, smem, attr_done); e0 != hipSuccess) return e0;
    BwdLaunch l{};
    const BwdParams *order[3] = {&dk, &dq, &dv};
    constexpr int n = D == 64 ? 2 : 3;
    int next = 0;
    for (int i = 0; i < n; i++) {
        l.pass[i] = *order[i];
        l.tiles[i] = order[i]->nR * order[i]->B * order[i]->H;
        l.first[i] = next;
        next += (l.tiles[i] + 7) & ~7;
    }
    if (D == 64) {
        l.pass[0].out2 = dv.out;
        for (int i = 0; i < 3; i++) l.pass[0].outs2[i] = dv.outs[i];
    }
    if constexpr (ORD) {
        l.order = ord.order;
        l.slots = ord.slots;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)(ORD ? 8 * l.slots : l.first[n - 1] + l.tiles[n - 1])), dim3(256), smem, stream, l);
    return hipGetLastError();
}

// The planes in groups of `group`, whose dS takes its turn in the workspace.  (The key tiles of a group in one launch with the
// query tiles of the group before, dealt out evenly: 2 ... 15 % slower than launches of their own, with 2 ... 8 groups.)
template <int DT, bool FAR>
hipError_t launch_bwd_ds(const BwdParams &dq, const BwdParams &dk, const BwdParams &dv, uint8_t *ds, int group, hipStream_t stream) {
    constexpr int smem = BwdLds<128, true>::bytes;
    auto kern = sparse_bwd_keys_kernel<DT, FAR>;
    static unsigned long long attr_done = 0;
    if (const hipError_t e0 = allow_dynamic_smem(kern, smem, attr_done); e0 != hipSuccess) return e0;
    auto kern_q = sparse_bwd_queries_kernel<DT, 128>;
    static unsigned long long attr_done_q = 0;
    if (const hipError_t e0 = allow_dynamic_smem(kern_q, BwdDqLds<128>::bytes, attr_done_q); e0 != hipSuccess) return e0;
    const int planes = dq.B * dq.H;
    for (int p0 = 0; p0 < planes; p0 += group) {
        BwdLaunch l{};
        l.pass[0] = dk;
        l.pass[0].out2 = dv.out;
        for (int c = 0; c < 3; c++) l.pass[0].outs2[c] = dv.outs[c];
        BwdParams q = dq;
        for (BwdParams *p : {&l.pass[0], &q}) {
            p->plane0 = p0;
            p->planes = planes - p0 < group ? planes - p0 : group;
            p->ds = ds;
            p->far = FAR;
            p->spread = bwd_spread(p->planes, dq.nR > dk.nR ? dq.nR : dk.nR);
        }
        l.tiles[0] = l.pass[0].planes * dk.nR;
        hipLaunchKernelGGL(kern, dim3((unsigned)l.tiles[0]), dim3(256), smem, stream, l);
        if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
        hipLaunchKernelGGL(kern_q, dim3((unsigned)(q.planes * q.nR)), dim3(256), BwdDqLds<128>::bytes, stream, q, q.planes * q.nR);
        if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <int DT, int D>
hipError_t launch_prepare_one(const BwdPrepParams &p, hipStream_t stream) {
    const int64_t rows = (int64_t)p.B * p.H * p.Sq;
    constexpr int RPB = 256 / (D / 8);  // rows per workgroup
    const unsigned blocks = (unsigned)((rows + RPB - 1) / RPB);
    if (p.order.n > 0) hipLaunchKernelGGL((bwd_prepare_kernel<DT, D, true>), dim3(8 + blocks), dim3(256), 0, stream, p);
    else hipLaunchKernelGGL((bwd_prepare_kernel<DT, D, false>), dim3(blocks), dim3(256), 0, stream, p);
    return hipGetLastError();
}

}  // namespace

// dS through memory: a pass over the keys (S, dP, dK, dV) and one over the queries (dQ), against one launch of three passes
// and 8 products.  It needs the device filled twice over by the key tiles alone (two workgroups on each of 256 compute units):
// causal, D = 128, backward with prepare in us, dS | three passes (by falling cost where that is their order):
//   256 key tiles  B1 H32 S1024  68 |  58   B1 H8  S4096  206 |  191   B2 H8 S2048 113 | 93
//   512            B8 H32 S256   48 |  55   B4 H16 S1024   98 |   97   B2 H16 S2048 165 | 154   B1 H16 S4096 259 | 283   B1 H8 S8192 511 | 666
//                  there every key B2 H16 S2048 212 | 262, random blocks 128 | 158, a window of 512 82 | 99, documents of 64 to 1024 103 | 85
//   1024           B8 H32 S512  116 | 134   B4 H16 S2048  266 |  317   B2 H16 S4096 434 | 541
//   4096           B8 H16 S4096 1719 | 2148, documents 551 | 747
// D = 64 stays with its two passes: dS is as large there and its two products half as long.
int bwd_ds_group(int B, int H, int Sq, int Sk, int D, size_t bytes) {
    constexpr int64_t kLeastTiles = 512;  // key tiles of a group
    if (D != 128) return 0;
    const size_t plane = (size_t)Sq * Sk * 2;
    const int64_t planes = (int64_t)B * H;
    int64_t n = (int64_t)(bytes / plane);
    if (n > planes) n = planes;
    if (n * (Sk / 128) < kLeastTiles) return 0;
    const int64_t groups = (planes + n - 1) / n;
    n = (planes + groups - 1) / groups;  // groups of even size
    return n * (Sk / 128) < kLeastTiles ? 0 : (int)n;
}

// dS of a group of more bytes, four times the memory-side cache, goes past L2 and is read from the planes written last (bwd_dq_tile).  Backward
// with prepare in us, dS through the caches in the order of planes | past them:
//   0.27 GB  B2 H16 S2048 causal 154 | 172, every key 209 | 206     0.54  B1 H16 S4096 causal 248 | 258, window of 1024 keys 116 | 123
//   1.07     B1 H8 S8192 window of 2048 205 | 209, B2 H16 S4096 causal 438 | 421, documents 153 | 158, every key 846 | 820
//   1.6      B3 H16 S4096 causal 691 | 660, documents 234 | 226     2.1  B4 H16 S4096 causal 884 | 859, documents 299 | 287
//   4.3      B8 H16 S4096 causal 1743 | 1700, documents 557 | 547, every key 3103 | 2935
constexpr int64_t kDsFar = (int64_t)1 << 30;

// At most 4 GiB, a seventieth of the device's memory.
size_t bwd_ds_bytes(int B, int H, int Sq, int Sk, int D) {
    return (size_t)Sq * Sk * 2 * bwd_ds_group(B, H, Sq, Sk, D, (size_t)4 << 30);
}

// Tiles by falling cost.  In the order of planes the last ones to start are as likely long as short: of 1536 tiles (B4 H12 S2048 D64, packed
// documents) on 768 slots one of 15 entries started at 31 us and ended the launch at 60, where the work is 40 us of every slot.
// More workgroups than run at once by a quarter (256 compute units; three each at D = 64 with packed tiles, else two), lists of eight entries
// or more, at D = 128 of sixteen, eighths of equal size, at most kOrderMost tiles a XCD.  So many query tiles that their statistics take as
// long as the sort (prepare 5.1 -> 6.1 us at 256 query tiles of D = 128, 7.1 -> 7.3 at 768 of D = 64).  Planes of a XCD that its L2 nearly holds
// (8 MiB), since the tiles at work are of all of them; and two planes or more, three where they are long, since a XCD with one has all its
// long tiles at work on one part of it.  Backward with statistics, us, planes | cost:
//   D = 64   documents B4 H12 S2048 70.7 | 57.9, B8 H12 S1024 70.9 | 57.7, B4 H17 S1024 58.2 | 44.7, B8 H24 S512 50.7 | 46.8, B2 H12 S4096 74.0 | 62.7
//            causal B4 H12 S2048 120 | 105, B4 H17 S1024 56.5 | 48.0   blocks B4 H12 S2048 111 | 101   every key 177 | 179, B8 H12 S1024 96.5 | 97.7
//            window of a quarter B4 H12 S2048 68.5 | 65.8, B8 H12 S1024 49.6 | 49.4, B8 H24 S512 40.1 | 40.4, of 64 keys there 35.2 | 37.1
//            from a bool mask (with a transposed copy) documents B2 H12 S4096 91.5 | 76.4, causal 232 | 216
//            left as it is: causal B1 H8 S8192 301 | 348, window of half B2 H8 S4096 97.7 | 102, documents from a bool mask there 79.1 | 90.3
//   D = 128  documents B4 H8 S1024 51.6 | 47.3, B2 H12 S2048 70.8 | 65.3   causal B4 H8 S1024 54.1 | 49.9, B2 H12 S2048 134 | 120, B1 H16 S3072 175 | 161
//            every key B4 H8 S1024 74.2 | 74.1, window of a quarter 39.2 | 40.2   (B1 H64 S512, left as it is: 45.0 | 46.1, window 32.3 | 33.9)
size_t bwd_order_bytes(int B, int H, int Sq, int Sk, int D) {
    const int64_t planes = (int64_t)B * H, tq = planes * (Sq / 128), tk = planes * (Sk / 128), all = tq + tk * (D == 64 ? 1 : 2);
    const int shortest = Sq < Sk ? Sq : Sk, longest = Sq < Sk ? Sk : Sq;
    if (tq % 8 || tk % 8 || all <= (D == 64 ? 960 : 640) || all > 8 * kOrderMost) return 0;
    if (shortest < (D == 64 ? 512 : 1024) || tq < (D == 64 ? 384 : 192) || planes < (longest > 3072 ? 24 : 16)) return 0;
    if ((planes + 7) / 8 * 2 * ((int64_t)Sq + Sk) * D * 2 > (8 << 20)) return 0;
    return (size_t)all * 4;
}
BwdOrderParams bwd_order(const BwdParams &dq, const BwdParams &dk, const BwdParams &dv, int D, int32_t *order) {
    BwdOrderParams o{};
    const BwdParams *passes[3] = {&dk, &dq, &dv};  // (as launch_bwd_one has them)
    o.n = D == 64 ? 2 : 3;
    o.order = order;
    for (int i = 0; i < o.n; i++) {
        const BwdParams &p = *passes[i];
        BwdOrderParams::Pass &q = o.pass[i];
        q.full_lens = p.full_lens;
        q.part_lens = p.part_lens;
        for (int c = 0; c < 3; c++) {
            q.fls[c] = p.fls[c];
            q.pls[c] = p.pls[c];
        }
        q.nR = p.nR;
        q.nS = p.nS;
        q.planes = p.planes;
        q.H = p.H;
        q.first_tile_first = p.first_tile_first;
        // (quarters of a microsecond: of the pass that makes dK and dV 2.5 an entry and 5 besides, of dQ 1.75 and 3.5; products 4 : 3 : 2)
        q.per_entry = D == 64 ? (i == 0 ? 10 : 7) : (i == 2 ? 6 : 9);
        q.fixed = 2 * q.per_entry;
        o.slots += p.planes * p.nR / 8;
    }
    return o;
}

hipError_t launch_bwd(const BwdParams &dq, const BwdParams &dk, const BwdParams &dv, int dtype, int D, uint8_t *ds, int group, const BwdOrderParams &order, hipStream_t stream) {
    if (group > 0) {
        const bool far = (int64_t)group * dq.nR * dk.nR * (128 * 128 * 2) > kDsFar;
        if (dtype == 0) return far ? launch_bwd_ds<0, true>(dq, dk, dv, ds, group, stream) : launch_bwd_ds<0, false>(dq, dk, dv, ds, group, stream);
        return far ? launch_bwd_ds<1, true>(dq, dk, dv, ds, group, stream) : launch_bwd_ds<1, false>(dq, dk, dv, ds, group, stream);
    }
    const bool pk = dq.packed != nullptr && dk.packed != nullptr;  // (with only one of them the mask is there too)
#define SA_BWD(DT, DD) \
    if (dtype == DT && D == DD) \
        return pk ? (order.n > 0 ? launch_bwd_one<DT, DD, true, true>(dq, dk, dv, order, stream) : launch_bwd_one<DT, DD, true, false>(dq, dk, dv, order, stream)) \
                  : (order.n > 0 ? launch_bwd_one<DT, DD, false, true>(dq, dk, dv, order, stream) : launch_bwd_one<DT, DD, false, false>(dq, dk, dv, order, stream))
    SA_BWD(0, 128);
    SA_BWD(0, 64);
    SA_BWD(1, 128);
    SA_BWD(1, 64);
#undef SA_BWD
    return hipErrorInvalidValue;
}

hipError_t launch_bwd_prepare(const BwdPrepParams &p, int dtype, int D, hipStream_t stream) {
    if (dtype == 0 && D == 128) return launch_prepare_one<0, 128>(p, stream);
    if (dtype == 0 && D == 64) return launch_prepare_one<0, 64>(p, stream);
    if (dtype == 1 && D == 128) return launch_prepare_one<1, 128>(p, stream);
    if (dtype == 1 && D == 64) return launch_prepare_one<1, 64>(p, stream);
    return hipErrorInvalidValue;
}

}  // namespace sa
