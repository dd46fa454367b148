// Internal declarations shared by the C-ABI translation unit and the kernel translation units.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sa {

// ---- mask classification -------------------------------------------------------------------------
struct ClassifyParams {
    const uint8_t *mask;
    int64_t sb, sh, sq, sk;  // mask strides in bytes over the DISTINCT planes (sb/sh unused when uB/uH == 1)
    uint8_t *cls;            // [uB*uH, nQ, nK] class bytes: 0 empty, 1 partial, 2 full
    int uB, uH;              // distinct planes along b and h
    int Sq, Sk, BQ, BK, nQ, nK;
    int lbk;                 // log2(BK) (wide kernel only)
};

struct CompactParams {
    const uint8_t *cls;
    int uH;                // distinct planes along h in cls
    int bcast_b, bcast_h;  // 1: every output plane along that dimension reads class plane 0
    int oB, oH;            // output planes to write
    int nQ, nK;
    int32_t *full_ids, *full_lens, *part_ids, *part_lens;
    int64_t fis[4], fls[3], pis[4], pls[3];  // output strides in elements
};

// Bit-packing of the PARTIAL tiles: tile (qt, slot) of a distinct plane is the slot-th entry of that Q tile's
// PARTIAL list; its BQ x BK mask entries become BQ*BK/8 bytes, row-major, entry (r, c) in bit (c & 7) of byte
// (r*BK + c) >> 3.
struct PackParams {
    const uint8_t *mask;
    int64_t sb, sh, sq, sk;  // mask strides in bytes over the distinct planes
    const int32_t *part_ids, *part_lens;
    int64_t pis[4], pls[3];  // list strides in elements, indexed with the distinct-plane coordinates
    uint8_t *packed;
    int64_t ob, oh;  // bytes between the packed planes along b and h
    int uB, uH;
    int BQ, BK, nQ, nK;
    int vec8;  // 1: key stride 1 and every row segment 8-byte aligned, so 8 entries load as one qword
};

// Classification, compaction and (packed not null) packing in one launch, a workgroup per Q tile (classify_rows_kernel).
struct ClassifyRowsParams {
    ClassifyParams c;  // (cls unused)
    CompactParams l;
    uint8_t *packed;
    int64_t ob, oh;
};
// The rule: mask_classify.hip.  The mask must suit the wide kernel, `packed` and its plane strides even addresses.
bool classify_rows_has(const ClassifyParams &p, int copies, bool packing);
hipError_t launch_classify_rows(const ClassifyRowsParams &p, hipStream_t stream);

// Q tiles dealt out to G persistent workgroups (G a multiple of 8, G/8 <= 64).  Workgroup g = 8*j + x is taken
// to run on XCD x (hardware hands consecutive workgroup ids to the XCDs in turn) and gets Q tiles of the x-th
// eighth of the (b,h)-major order, so that the tiles sharing a K/V plane meet in one L2.
// sched: int32 [G][R+1][4]; entry 0 of a row = {count, 0, 0, 0}, entries 1..count = {(b << 16) | h, qt, F, P}.
struct ScheduleParams {
    const int32_t *full_lens, *part_lens;
    int64_t fls[3], pls[3];
    int B, H, nQ;
    int G, R;
    int lbk;  // log2(BK): chunks of 64 keys per entry = BK/64, entries per chunk = 64/BK
    int pairs;  // 1: two Q tiles per workgroup, one workgroup per pair of tiles (G = number of pairs, R = 2)
    int32_t *sched;
};

// Check of caller-supplied lists against the nK tiles a row of tiles has; *flag collects error bits (never cleared here).
struct ValidateParams {
    const int32_t *full_ids, *full_lens, *part_ids, *part_lens;
    int64_t fis[4], fls[3], pis[4], pls[3];
    int B, H, nQ, nK;
    int32_t *flag;
};
hipError_t launch_validate(const ValidateParams &p, hipStream_t stream);

hipError_t launch_classify(const ClassifyParams &p, bool wide, hipStream_t stream);
hipError_t launch_schedule(const ScheduleParams &p, hipStream_t stream);
hipError_t launch_compact(const CompactParams &p, hipStream_t stream);
hipError_t launch_pack(const PackParams &p, hipStream_t stream);

// ---- masks given by a formula ---------------------------------------------------------------------
// Entry (b, q, k) attends when any term holds; a term is the AND of the conditions its flags switch on.
constexpr int kMaxMaskTerms = 8;
constexpr int kTermBack = 1;      // (q + offset) - k < back
constexpr int kTermAhead = 2;     // k - (q + offset) < ahead
constexpr int kTermQRange = 4;    // q_lo <= q < q_hi
constexpr int kTermKRange = 8;    // k_lo <= k < k_hi
constexpr int kTermSameDoc = 16;  // doc_q[b][q] == doc_k[b][k]
// A term as the kernels evaluate it: for query row q it admits the keys of
//   [max(q + a, k_lo), min(q + b, k_hi))   when q_lo <= q < q_hi, none otherwise,
// and of those the keys of q's document when `doc` is set.  a, b are clamped to +-2^30 and the ranges to the
// mask's extent on the host, so that with Sq, Sk <= 2^29 everything stays inside int32.
struct MaskTerm {
    int32_t a, b, k_lo, k_hi, q_lo, q_hi, doc;
};
struct TermsParams {
    MaskTerm terms[kMaxMaskTerms];
    int n_terms;
    const int32_t *doc_q, *doc_k;  // [uB, Sq] and [uB, Sk] document numbers, or null
    int64_t dqs[2], dks[2];        // their strides in elements
    int uB;                        // distinct planes (the mask never depends on the head)
    int Sq, Sk, BQ, BK, lbk, nQ, nK;
    // the lists: oH planes along the head, and along the batch all oB planes from the one distinct plane (oB_all) or
    // the distinct plane's own
    int oB_all, oB, oH;
    int32_t *full_ids, *full_lens, *part_ids, *part_lens;
    int64_t fis[4], fls[3], pis[4], pls[3];
    uint8_t *packed;  // PackParams layout, or null
    int64_t ob;       // bytes between packed planes along b
};
// Masks made by one launch: the two tilings of a backward are short of workgroups one by one.
struct TermsBatch {
    TermsParams of[2];
};
hipError_t launch_mask_terms(const TermsBatch &b, int n, hipStream_t stream);

// ---- block-sparse forward ------------------------------------------------------------------------
struct FwdParams {
    const uint16_t *q, *k, *v;
    uint16_t *o;
    const uint8_t *mask;
    const int32_t *full_ids, *full_lens, *part_ids, *part_lens;
    int64_t qs[3], ks[3], vs[3], os[3];  // b, h, s strides in elements (d stride is 1)
    int64_t ms[4];                        // mask strides in bytes
    int64_t fis[4], fls[3], pis[4], pls[3];
    int B, H, Sq, Sk, nQ;
    int BK, lbk;    // KV tile width and its log2
    int mask_vec4;  // 1: mask columns are contiguous and 4-byte aligned, so 4 entries load as one dword
    // Bit-packed PARTIAL tiles (PackParams layout), or null: then the mask itself is read.
    const uint8_t *packed;
    int64_t pks[2];  // bytes between packed planes along b and h (0 where the mask is broadcast)
    int nK;          // KV tiles per row of tiles (slots per Q tile in `packed`)
    int spread;      // planes taken together, their Q tiles side by side from the last one down (fwd_spread), or 0: two by two
    // Schedule of persistent workgroups (ScheduleParams layout), or null: then one workgroup per Q tile.
    const int32_t *sched;
    int sched_G, sched_R;  // workgroups, and entries per row after the header entry
    float scale;    // softmax scale / ln 2
    // 0, or the group size G of the rotated walk of the FULL entries (sparse_fwd_kernel, one workgroup per Q tile):
    // Q tile qt starts 2 * (G - 1 - qt mod G) chunks into its FULL entries.
    int rot;
    // Optional second output: natural-log sum of exp(scaled score) over the attended keys of every query row
    // (-inf for rows without one), or null.
    float *lse;
    int64_t lses[3];  // b, h, row strides in elements
    // Lists shared by up to nsplit > 1 workgroups each (fwd_split_share), or nsplit <= 1: the workgroups' partial results,
    //   ws    [B*H*nQ][nsplit][BQ/32][D/8][64 lanes][4] floats: unnormalised rows in the order the registers hold them
    //   ws_ml [B*H*nQ][nsplit][BQ][2] floats: reference value (-inf: no attended key) and sum of every row
    int nsplit, split_chunks;  // split_chunks: chunks of one part (the last ones may be shorter)
    int split_least;           // lists of up to this many chunks are not shared
    int halves;                // 1: every list in two halves by the waves of one workgroup (fwd_in_halves)
    float *ws, *ws_ml;
    // Ragged sizes: the tile grid (Sq, Sk, nQ, nK, lists, packed tiles) is that of a padded mask, the tensors have Sq_in
    // and Sk_in rows, which stand q0 and k0 rows into the grid, of D_in elements (a multiple of 8, at most the kernel's D).
    int ragged;
    int q0, k0, Sq_in, Sk_in, D_in;
    // The launch's number where the last workgroup of a shared list to arrive adds the parts up (all_arrived), or 0: then a second
    // launch does (launch_fwd_merge).  The words it knows that by, [B*H*nQ][nsplit], lie behind ws_ml.  (The arguments stay within
    // 512 bytes with the grid's size behind them: 16 more, and one more miss at the start made a launch of 22.5 us 0.3 us longer.)
    uint64_t tag;
    __host__ __device__ uint64_t *arrivals(int BQ) const { return reinterpret_cast<uint64_t *>(ws_ml + (int64_t)B * H * nQ * nsplit * BQ * 2); }
};
static_assert(sizeof(FwdParams) + 3 * sizeof(uint32_t) <= 512, "the forward's arguments with the grid's size behind them");

// How many workgroups share a list of NE entries of 2^lbk keys, walked in chunks of 2^lck keys, and the first entry of
// part s of them (s = share: the end of the list).  Entries of one chunk stay together.
__host__ __device__ inline int fwd_split_share(int NE, int lbk, int lck, int split_least, int split_chunks, int nsplit) {
    const int le = lck > lbk ? lck - lbk : 0, lc = lbk > lck ? lbk - lck : 0;
    const int groups = (NE + (1 << le) - 1) >> le;
    if ((groups << lc) <= split_least) return 1;
    const int parts = ((groups << lc) + split_chunks - 1) / split_chunks;
    const int most = groups < nsplit ? groups : nsplit;
    return parts < most ? (parts > 1 ? parts : 1) : (most > 1 ? most : 1);
}
__host__ __device__ inline int fwd_split_first(int NE, int lbk, int lck, int s, int share) {
    const int le = lck > lbk ? lck - lbk : 0;
    const unsigned groups = (unsigned)(NE + (1 << le) - 1) >> le;
    const int e = (int)(groups * (unsigned)s / (unsigned)share) << le;
    return e < NE ? e : NE;
}
// Whether the last workgroup of a shared list to arrive adds up its parts (all_arrived), else a second launch does: sparse_fwd_merge.hip.
bool fwd_merges_in_launch(int tiles, int nsplit, int BQ, int D, int dtype);
// The rule for nsplit, split_chunks and split_least: sparse_fwd_merge.hip.
// chunks 0: every list has one assistant (fwd_assists, sparse_fwd_kernel<..., AS>), which takes the end of it where it is `least` longer.
struct FwdSplitPlan {
    int nsplit = 1, chunks = 1 << 30, least = 0;
};
bool fwd_assists(int64_t planes, int nQ, int Sk, int BQ, int BK, int D, int dtype, int cus);
constexpr int kAssistLeast = 8;
FwdSplitPlan fwd_split_plan(int tiles, int Sk, int BQ, int D, int dtype, int cus);
// FwdParams::spread of a launch: sparse_fwd_merge.hip.
int fwd_spread(int64_t planes, int nQ, int BQ, int64_t plane_bytes, int cus);
// Whether a launch walks its lists in two halves (sparse_fwd_kernel<..., TW>) where they are not shared: sparse_fwd_merge.hip.
bool fwd_in_halves(int64_t tiles, int Sk, int BQ, int BK, int D, int dtype, int cus);
// There: chunks up to which the form without halves is no slower, if every list is known to be as short.
int fwd_halves_least(int BQ, int D);
// Adds up the parts of shared lists (dtype 2: float32 output).
hipError_t launch_fwd_merge(const FwdParams &p, int dtype, int D, int BQ, hipStream_t stream);

// dtype: 0 bf16, 1 fp16.  Returns hipErrorInvalidValue when no instantiation matches (D, BQ).
hipError_t launch_fwd(const FwdParams &p, int dtype, int D, int BQ, hipStream_t stream);
// The forward for short lists (sparse_fwd_c32.hip): three workgroups per compute unit, 32 keys per step.  It exists
// for bf16 / fp16, D = 128, BLOCK_Q = 128, bit-packed PARTIAL tiles, no schedule (fwd_c32_has), and cuts lists at
// 256 entries.  Results agree with launch_fwd within rounding (the keys meet the online softmax in other groupings).
bool fwd_c32_has(const FwdParams &p, int dtype, int D, int BQ);
hipError_t launch_fwd_c32(const FwdParams &p, int dtype, int D, int BQ, hipStream_t stream);
// float32 q, k, v, o (the pointers of FwdParams then address floats; strides stay in elements): any BQ from 1 to 256
// (to 128 at D = 256), any BK; reads the packed tiles when given, else the mask; no schedules.
hipError_t launch_fwd_f32(const FwdParams &p, int D, int BQ, hipStream_t stream);
// The same on the matrix unit (sparse_fwd_f32_mfma.hip) for the sizes it has (fwd_f32_mfma_has); launch_fwd_f32 takes
// it whenever it can.
bool fwd_f32_mfma_has(const FwdParams &p, int D, int BQ);
hipError_t launch_fwd_f32_mfma(const FwdParams &p, int D, int BQ, hipStream_t stream);

// Few query rows against a long K/V (decode): one Q tile of Sq <= 32 rows per (b, h), its list of KV tiles split
// over `nsplit` workgroups whose partial results a second kernel merges.
// The most entries a plane's mask may have for a decode without lists, and the widest tiles: bits and lists lie in LDS, every
// workgroup of the plane reads the whole mask, and a lane goes over a tile.
constexpr int kDecodeDirectEntries = 32768;
constexpr int kDecodeDirectBK = 256;
// Whether the last workgroup of a plane to arrive merges its parts (else a second launch does).  It does where that is sooner: the
// workgroups of a plane count in one word, half a microsecond each, and one workgroup adds up all rows.  us, second launch -> last
// workgroup, lists made in the call:
//   parts of one row  8  14.5 -> 12.3   16  29.0 -> 34.8   32  14.6 -> 23.6   64  33.4 -> 53.8
//   rows, D = 128     8 x 4 16.8 -> 15.2   8 x 8 18.7 -> 16.1   8 x 16 26.7 -> 23.6   2 x 16 13.7 -> 13.5   2 x 32 15.4 -> 16.0
//   rows, D = 64      8 x 4 12.2 -> 10.6   8 x 8 12.7 -> 13.5   8 x 16 14.5 -> 15.2   2 x 16 10.4 -> 10.3   2 x 32 12.0 -> 12.4
// Up to kDecodeMergeFew parts both add a row's parts up one after the other: the same bits.
constexpr int kDecodeMergeFew = 8;
constexpr int kDecodeMergeRows = 128;  // partial rows of a plane that LDS holds
inline bool decode_merges_in_launch(int64_t nsplit, int64_t Sq, int D) {
    return nsplit > 1 && nsplit <= kDecodeMergeFew && Sq <= 16 && nsplit * Sq <= (D == 128 ? kDecodeMergeRows : 32);
}
struct DecodeParams {
    const uint16_t *q, *k, *v;
    uint16_t *o;
    const uint8_t *mask;
    const int32_t *full_ids, *full_lens, *part_ids, *part_lens;  // all null: the tiles are found in the mask
    int64_t qs[3], ks[3], vs[3], os[3];  // b, h, s strides in elements (d stride is 1)
    int64_t ms[4];                        // mask strides in bytes
    int64_t fis[3], fls[2], pis[3], pls[2];  // b, h (and entry) strides of the lists of the one Q tile
    int B, H, Sq, Sk;
    int BK, lbk;    // KV tile width (a power of two >= 16) and its log2
    int mask_vec4;  // 1: mask columns are contiguous and 4-byte aligned
    // Bit-packed PARTIAL tiles of the one Q tile (PackParams layout with BQ = Sq), or null: then the mask itself is read.
    const uint8_t *packed;
    int64_t pks[2];  // bytes between packed planes along b and h
    int nsplit;     // workgroups per (b, h)
    float *ws;      // [B*H][nsplit][Sq][D + 2] floats: unnormalised rows, then reference value and row sum
    // [B*H] words by which the last workgroup of a plane to arrive knows that it is the one to merge (arrives_last), or null:
    // then a second launch merges.
    uint64_t *arrivals;
    uint64_t tag;   // the launch's number
    float scale;    // softmax scale / ln 2
    float *lse;     // optional second output as in FwdParams, or null
    int64_t lses[3];
};
hipError_t launch_decode(const DecodeParams &p, int dtype, int D, hipStream_t stream);

// Merge of n attention results computed over disjoint key ranges (outputs and row log-sum-exps).
struct MergeParams {
    const uint16_t *o_parts;  // [n,B,H,Sq,D]
    const float *lse_parts;   // [n,B,H,Sq]
    uint16_t *o;
    float *lse;               // optional
    int64_t ops[4], lps[4];   // part, b, h, row strides in elements (d stride is 1)
    int64_t os[3], lses[3];
    int n, B, H, Sq, D;
};
hipError_t launch_merge_parts(const MergeParams &p, int dtype, hipStream_t stream);

// ---- backward ------------------------------------------------------------------------------------
// One pass of the backward kernel (sparse_bwd.hip): tiles of 128 resident rows walk their lists of 64-row streamed
// tiles.  dQ: resident q (x = q, g = dO), streamed keys (y = k, z = v), statistics per resident row.
// dK / dV: resident keys (x = k, g = v), streamed queries (y = q, z = dO), statistics per streamed row, lists and
// mask strides of the transposed mask.  D = 64 or 128.
struct BwdParams {
    const uint16_t *x, *g, *y, *z;
    uint16_t *out;
    int64_t xs[3], gs[3], ys[3], zs[3], outs[3];  // b, h, row strides in elements (d stride is 1)
    const uint8_t *mask;
    int64_t ms[2];     // mask strides along b and h in bytes
    int64_t mrs, mcs;  // mask strides along the resident and the streamed rows in bytes
    int mask_vec4;     // 1: mcs == 1 and 4-byte aligned rows
    // Bit-packed PARTIAL tiles of this pass's tiling (PackParams layout, tiles of 128 x 64), or null: then `mask`.
    const uint8_t *packed;
    int64_t pks[2];    // bytes between packed planes along b and h
    int nS;            // streamed tiles per resident tile (slots in `packed`)
    const int32_t *full_ids, *full_lens, *part_ids, *part_lens;  // per resident tile, streamed tiles of 64
    int64_t fis[4], fls[3], pis[4], pls[3];
    const float *stat_l, *stat_d;  // per query: -lse / ln 2 (-inf for dead rows) and -rowsum(dO o O)
    int64_t sts[3];                // their b, h, row strides in elements (row stride 1 when queries are streamed)
    int B, H, nR;                  // nR: resident tiles
    int first_tile_first;          // launch order of a plane's tiles: 0 last tile first (queries), 1 first tile first (keys)
    float scale;                   // softmax scale / ln 2 (folded into x)
    float out_scale;               // softmax scale for dQ and dK, 1 for dV
    uint16_t *out2;                // dV, where one pass makes both
    int64_t outs2[3];
    int plane0, planes;            // the pass covers planes plane0 .. plane0 + planes - 1 of the B * H
    uint8_t *ds;                   // workspace of dS of these planes (bwd_dq_tile), Sq * Sk elements each
    int far;                       // 1: dS of these planes is larger than the caches (kDsFar)
    int spread;                    // planes taken together, their tiles side by side (bwd_spread), or 0: two by two
};
// The passes of one launch: workgroup first[i] + t has tile t of pass i.
struct BwdLaunch {
    BwdParams pass[3];
    int first[3], tiles[3];
    // null, or [8][slots]: workgroup 8 j + x has the j-th of XCD x's tiles by falling cost: pass << 29 | its place in the XCD's share << 18 |
    // its FULL entries << 9 | all its entries
    const int32_t *order;
    int slots;
};
// How the tiles of a launch come by falling cost (bwd_prepare_kernel makes the order from the lists' lengths).
struct BwdOrderParams {
    int n;  // passes, or 0: no order
    struct Pass {
        const int32_t *full_lens, *part_lens;
        int64_t fls[3], pls[3];
        int nR, nS, planes, H, first_tile_first;
        int fixed, per_entry;  // cost of a tile, and of an entry of its list
    } pass[3];
    int slots;
    int32_t *order;
};
// The rule for it (sparse_bwd.hip): bytes of `order`, 0 where the tiles stay in the order of planes.
size_t bwd_order_bytes(int B, int H, int Sq, int Sk, int D);
BwdOrderParams bwd_order(const BwdParams &dq, const BwdParams &dk, const BwdParams &dv, int D, int32_t *order);
// group > 0 (D = 128 and both packed buffers): dS of that many planes at a time goes through `ds`, and dQ is made from it.
hipError_t launch_bwd(const BwdParams &dq, const BwdParams &dk, const BwdParams &dv, int dtype, int D, uint8_t *ds, int group, const BwdOrderParams &order, hipStream_t stream);
// The rule for group: sparse_bwd.hip.  bytes: what the workspace holds besides the statistics.
int bwd_ds_group(int B, int H, int Sq, int Sk, int D, size_t bytes);
// Bytes of dS that are worth their place, 0 where none are.
size_t bwd_ds_bytes(int B, int H, int Sq, int Sk, int D);

struct BwdPrepParams {
    const uint16_t *o, *d_o;
    const float *lse;
    int64_t os[3], dos[3], ls[3];
    float *stat_l, *stat_d;  // [B*H*Sq] each, contiguous
    float l_mul;             // stat_l = lse * l_mul: -1 / ln 2, or -1 / (ln 2 scale) where the kernel scales S - L
    int B, H, Sq;
    BwdOrderParams order;
};
hipError_t launch_bwd_prepare(const BwdPrepParams &p, int dtype, int D, hipStream_t stream);

}  // namespace sa
