// Tile classification and bit-packing of an attention mask that is given by a formula, on gfx950 (MI355X).
//
// The reference parses a materialised bool tensor (sparseattention/mask_utils.py:47-82) and names masks defined
// algebraically, without materialisation and its memory cost, as the first thing that could come next
// (README.md:12, :63).  Here the mask of entry (b, q, k) is the OR of up to kMaxMaskTerms terms, each the AND of
// the conditions its flags switch on:
//
//   BACK      (q + offset) - k < back        (how far behind the diagonal a key may lie)
//   AHEAD     k - (q + offset) < ahead       (ahead = 1: causal)
//   Q_RANGE   q_lo <= q < q_hi
//   K_RANGE   k_lo <= k < k_hi
//   SAME_DOC  doc_q[b][q] == doc_k[b][k]
//
// One kernel, mask_terms_kernel, makes the lists (as classify + compact do for a tensor mask, mask_classify.hip) and the
// PARTIAL tiles at one bit per entry in the layout of pack_partial_kernel, so the forward and the backward run without
// any mask tensor.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.h"

namespace sa {

namespace {

constexpr int kThreads = 512;
constexpr int kWaves = kThreads / 64;
constexpr int kStrips = 1024;             // strips of 64 keys decided per batch
constexpr int kTiles = kStrips * 64 / 16; // most tiles a round holds in LDS
constexpr int kRows = 1024;               // query rows whose documents LDS holds (Q tiles of more read memory again)
constexpr int kKeys = 2048;               // keys whose documents LDS holds: the last that the rows of the Q tile reach
constexpr int kByRow = 255;               // (in kept_at) a strip whose entries follow from its document alone
constexpr int kKept = 16, kKeptRows = 128; // strips whose words LDS holds, of Q tiles of up to so many rows

// Brings the arguments' lines into the scalar cache under one wait.  They are read here and there as the kernel gets to them, and a
// line that is not there yet is a round trip of its own each time.
__device__ __forceinline__ void warm_arguments(int which) {
    static_assert(sizeof(TermsParams) > 7 * 64 && sizeof(TermsParams) <= 8 * 64, "a load for each of the lines");
    const uint64_t at = (uint64_t)(uintptr_t)__builtin_amdgcn_kernarg_segment_ptr() + (uint64_t)(__builtin_amdgcn_readfirstlane(which) * (int)sizeof(TermsParams));
    int l[8];
    asm volatile(
        "s_load_dword %0, %8, 0x0\n\ts_load_dword %1, %8, 0x40\n\ts_load_dword %2, %8, 0x80\n\ts_load_dword %3, %8, 0xc0\n\t"
        "s_load_dword %4, %8, 0x100\n\ts_load_dword %5, %8, 0x140\n\ts_load_dword %6, %8, 0x180\n\ts_load_dword %7, %8, 0x1c0\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&s"(l[0]), "=&s"(l[1]), "=&s"(l[2]), "=&s"(l[3]), "=&s"(l[4]), "=&s"(l[5]), "=&s"(l[6]), "=&s"(l[7])
        : "s"(at));
}

// For one query row a term admits an interval of keys (and of those the keys of the row's document).
__device__ __forceinline__ void term_interval(const MaskTerm &m, int q, int &lo, int &hi) {
    lo = max(q + m.a, m.k_lo);
    hi = min(q + m.b, m.k_hi);
    if (q < m.q_lo || q >= m.q_hi) hi = lo;
}

// bits [a, b) of a 64-bit word, 0 <= a, b <= 64
__device__ __forceinline__ uint64_t bit_range(int a, int b) {
    return b > a ? (~0ull >> (64 - (b - a))) << a : 0ull;
}

// The documents of 64 neighbouring keys (lane = key) as runs of one number: `starts` has a bit at the first key of
// every run.  Packed documents have one to three runs in 64 keys; unsorted numbers, up to 64, only cost more steps.
__device__ __forceinline__ uint64_t run_starts(int dk) {
    const int lane = threadIdx.x & 63;
    const int before = __builtin_amdgcn_update_dpp(dk, dk, 0x138, 0xf, 0xf, false);  // (wave_shr 1: the lane before)
    return __ballot(lane == 0 || dk != before);
}

// The mask entries of this lane's query row q against the keys ks .. ks + n - 1 (n <= 64; lane i holds the document of
// key ks + i in dk), bit i = key ks + i; lo, hi: the row's interval of the first term.  All lanes of the wave have to be active.
__device__ __forceinline__ uint64_t row_word(const TermsParams &p, int q, int lo, int hi, int ks, int n, int dq, int dk, uint64_t starts) {
    uint64_t same = ~0ull;
    if (p.doc_q && p.doc_k) {
        same = 0ull;
        for (uint64_t m = starts; m != 0ull;) {
            const int i = __builtin_ctzll(m);
            m &= m - 1ull;
            const int d = __builtin_amdgcn_readlane(dk, i);
            same |= dq == d ? bit_range(i, m ? __builtin_ctzll(m) : 64) : 0ull;
        }
    }
    uint64_t word = 0ull;
    for (int t = 0;;) {
        const uint64_t w = bit_range(min(max(lo - ks, 0), 64), min(max(hi - ks, 0), 64));
        word |= p.terms[t].doc ? w & same : w;
        if (++t >= p.n_terms) break;
        term_interval(p.terms[t], q, lo, hi);
    }
    return word & bit_range(0, n);
}

// Smallest and largest of x over the 16 lanes of a row, and over the wave, in every lane (all lanes active): by DPP and lane swaps, a
// few cycles each, where __shfl_xor goes through LDS.
template <int CTRL>
__device__ __forceinline__ int from_lane(int x) { return __builtin_amdgcn_update_dpp(x, x, CTRL, 0xf, 0xf, false); }
__device__ __forceinline__ void range_of_row(int &lo, int &hi) {
    auto step = [&](int lo2, int hi2) {
        lo = min(lo, lo2);
        hi = max(hi, hi2);
    };
    step(from_lane<0x128>(lo), from_lane<0x128>(hi));  // row_ror 8, 4, 2, 1
    step(from_lane<0x124>(lo), from_lane<0x124>(hi));
    step(from_lane<0x122>(lo), from_lane<0x122>(hi));
    step(from_lane<0x121>(lo), from_lane<0x121>(hi));
}
__device__ __forceinline__ void range_of_wave(int &lo, int &hi) {
    range_of_row(lo, hi);
    const auto l16 = __builtin_amdgcn_permlane16_swap(lo, lo, false, false), h16 = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
    lo = min((int)l16[0], (int)l16[1]);
    hi = max((int)h16[0], (int)h16[1]);
    const auto l32 = __builtin_amdgcn_permlane32_swap(lo, lo, false, false), h32 = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
    lo = min((int)l32[0], (int)l32[1]);
    hi = max((int)h32[0], (int)h32[1]);
}

// grid (nQ, distinct planes, masks), 512 threads: a workgroup makes everything of one Q tile, so nothing goes through memory
// between classification, lists and packed tiles.  Per round of at most kTiles tiles:
//   A  a strip of 64 keys is decided from the first and the last row of the Q tile where it can be (both ends of a
//      row's interval move right, or stay, as q grows): no term reaches it, or one term covers it from every row,
//      document conditions judged by the ranges of the document numbers on both sides.  16 lanes read a strip's documents,
//      then a thread decides a strip.  Of one term, where the rows have two documents or more, the strips that lie in the first or
//      the last of them are PARTIAL by that alone, and an entry is whether its row has the strip's document.
//   B  the other strips, a wave per strip and 64 rows: lane = query row, one 64-bit word of entries per row (row_word), and two
//      ballots per tile tell whether some entry attends and whether some does not.
//   C  a wave per list compacts the tiles' states by ballot and popcount.
//   D  the PARTIAL tiles' words are stored, a wave per strip: those of the first kKept strips of B wait in LDS, the others are
//      made again.
// Latency bound (a few dependent reads of documents and arguments, a few barriers; a word is a few dozen instructions per 64 rows and
// strip): arguments and documents are requested at once at the start, documents of rows and keys stay in LDS.  Against
// classification with one key per lane and one row per step, compaction and packing as three kernels that evaluated the
// terms per entry (launches back to back in a graph): causal documents B4 S2048 tiles 128x64 71 -> 10.3 us, B4 S16384
// tiles 128x32 352 -> 44 us, window and prefix at S32768 149 -> 9.5 us.  1024 threads: 10.4 / 49 / 10.5 us.
// The two tilings of a backward come from one launch: few Q tiles each (B4 S2048: 64 workgroups).  One tiling | both, traced, causal
// documents of 64 ... 1024, before and with documents and words in LDS, wide loads of them, ranges by DPP, a thread per strip and the
// strips decided by one document: B4 S2048 11.2 | 11.4 -> 9.2 | 9.3 us, B4 S16384 21.7 | 36.0 -> 15.1 | 25.0, B1 S32768 29.5 | 34.8 ->
// 16.0 | 20.9.  Of the 9.2 us 1.7 are an empty launch, 0.7 arguments, 2.6 A, 1.3 B, 0.8 C and 2.1 the stores with the end of the launch.
__global__ __launch_bounds__(kThreads) void mask_terms_kernel(const TermsBatch batch) {
    warm_arguments(blockIdx.z);
    const TermsParams &p = batch.of[blockIdx.z];
    if ((int)blockIdx.x >= p.nQ || (int)blockIdx.y >= p.uB) return;
    __shared__ unsigned state[kTiles / 4];  // a byte per tile, bit 0: some entry attends, bit 1: some entry does not
    __shared__ uint16_t part[kTiles];       // the PARTIAL tiles of the round, in order
    __shared__ uint16_t todo[kStrips];      // strips that step A left open
    __shared__ uint8_t kept_at[kStrips];    // 1 + place in `todo` of a strip whose words are kept, kByRow, or 0
    __shared__ int n_todo, sh_min[kWaves], sh_max[kWaves], row_doc[kRows];
    __shared__ __attribute__((aligned(16))) int key_doc[kKeys];
    __shared__ union {
        int range[kStrips][2];                // (A) smallest and largest document of a strip
        uint64_t words[kKept][kKeptRows];     // (B, D)
    } u;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int qt = blockIdx.x, ub = blockIdx.y;
    const int q0 = qt * p.BQ, q1 = q0 + p.BQ - 1;
    const int32_t *dqp = p.doc_q ? p.doc_q + (int64_t)ub * p.dqs[0] : nullptr;
    const int32_t *dkp = p.doc_k ? p.doc_k + (int64_t)ub * p.dks[0] : nullptr;
    const bool docs = dqp && dkp;

    // the keys that some row of the tile reaches under some term: documents of strips outside are not read
    int reach_lo = INT32_MAX, reach_hi = INT32_MIN;
    for (int t = 0; t < p.n_terms; t++) {
        const MaskTerm &m = p.terms[t];
        const int r0 = max(q0, m.q_lo), r1 = min(q1, m.q_hi - 1);
        if (r0 > r1) continue;
        reach_lo = min(reach_lo, max(r0 + m.a, m.k_lo));
        reach_hi = max(reach_hi, min(r1 + m.b, m.k_hi));
    }
    const int unit = p.BK < 64 ? p.BK : 64;  // keys of one strip that belong to one tile
    const int per_strip = 64 / unit;         // tiles a strip reaches: 4, 2 or 1
    const int lsp = p.lbk > 6 ? p.lbk - 6 : 0;  // log2 of the strips a tile reaches
    const int round = p.BK < 64 ? kStrips * per_strip : max(1, kStrips >> lsp);
    const bool keep_words = p.BQ <= kKeptRows && lsp <= 10;  // (one batch of strips a round)
    auto reached = [&](int ks) { return ks < reach_hi && min(ks + 64, p.Sk) > reach_lo; };
    // The documents of the keys of one strip, four to a lane, 16 lanes: requested a pass ahead, the first ones with those of the rows.
    constexpr int kPass = kThreads / 16;
    const int strip_of_thread = (int)threadIdx.x / 16;
    // (Sk is a multiple of 16: a lane's four keys exist together)
    const bool by_four = p.dks[1] == 1 && ((uintptr_t)dkp & 15) == 0;
    int4 d_next = {};
    auto request_keys = [&](int ks, bool in) {
        const int k = ks + 4 * (lane & 15);
        if (!in || k >= p.Sk || !reached(ks)) return;
        if (by_four) {
            d_next = *reinterpret_cast<const int4 *>(dkp + k);
        } else {
            const int32_t *const at = dkp + (int64_t)k * p.dks[1];
            d_next = int4{at[0], at[p.dks[1]], at[2 * p.dks[1]], at[3 * p.dks[1]]};
        }
    };
    if (docs) {
        const int strips = (int)min((int64_t)kStrips, ((int64_t)min(round, p.nK) * p.BK + 63) >> 6);
        request_keys(64 * strip_of_thread, strip_of_thread < strips);
        int lo = INT32_MAX, hi = INT32_MIN;
        for (int r = threadIdx.x; r < p.BQ; r += kThreads) {
            const int d = dqp[(int64_t)(q0 + r) * p.dqs[1]];
            if (r < kRows) row_doc[r] = d;
            lo = min(lo, d);
            hi = max(hi, d);
        }
        range_of_wave(lo, hi);
        if (lane == 0) {
            sh_min[wave] = lo;
            sh_max[wave] = hi;
        }
    }

    auto doc_of_row = [&](int r) {
        return !docs || r >= p.BQ ? 0 : (r < kRows ? row_doc[r] : dqp[(int64_t)(q0 + r) * p.dqs[1]]);
    };
    int doc_base = 0;  // key_doc holds the keys [doc_base, doc_base + kKeys) of strips that some row reaches
    auto doc_of_key = [&](int ks, int n) {
        if (!docs) return 0;
        if ((unsigned)(ks - doc_base) < (unsigned)kKeys) return key_doc[ks - doc_base + min(lane, n - 1)];
        return lane < n ? dkp[(int64_t)(ks + lane) * p.dks[1]] : 0;
    };
    auto mark = [&](int tile, unsigned bits) { atomicOr(&state[tile >> 2], bits << (8 * (tile & 3))); };

    int qmin = INT32_MAX, qmax = INT32_MIN;
    int nf = 0, np = 0;
    for (int tile0 = 0; tile0 < p.nK; tile0 += round) {
        const int tiles = min(round, p.nK - tile0);
        const int64_t k_begin = (int64_t)tile0 * p.BK, k_stop = (int64_t)(tile0 + tiles) * p.BK;
        for (int i = threadIdx.x; i < (tiles + 3) / 4; i += kThreads) state[i] = 0u;
        for (int64_t kb = k_begin; kb < k_stop; kb += kStrips * 64) {
            const int strips = (int)(min((int64_t)(kStrips * 64), k_stop - kb) + 63) >> 6;
            if (threadIdx.x == 0) n_todo = 0;
            // A
            if (docs) {
                doc_base = max((int)kb, ((min(max(reach_hi, (int)kb), (int)kb + 64 * strips) + 63) & ~63) - kKeys);
                if (kb != 0) request_keys((int)kb + 64 * strip_of_thread, strip_of_thread < strips);
                for (int s0 = 0; s0 < strips; s0 += kPass) {
                    const int s = s0 + strip_of_thread, ks = (int)kb + 64 * s;
                    const int4 d = d_next;
                    request_keys(ks + 64 * kPass, s + kPass < strips);
                    const int k = ks + 4 * (lane & 15);
                    const bool in = s < strips && k < p.Sk;
                    int lo = in ? min(min(d.x, d.y), min(d.z, d.w)) : INT32_MAX;
                    int hi = in ? max(max(d.x, d.y), max(d.z, d.w)) : INT32_MIN;
                    if (in && (unsigned)(ks - doc_base) < (unsigned)kKeys) *reinterpret_cast<int4 *>(key_doc + (k - doc_base)) = d;
                    range_of_row(lo, hi);
                    if (s < strips && (lane & 15) == 0) {
                        u.range[s][0] = lo;
                        u.range[s][1] = hi;
                    }
                }
            }
            __syncthreads();
            if (docs && tile0 == 0 && kb == 0) {
#pragma unroll
                for (int w = 0; w < kWaves; w++) {
                    qmin = min(qmin, sh_min[w]);
                    qmax = max(qmax, sh_max[w]);
                }
            }
            for (int s = threadIdx.x; s < strips; s += kThreads) {
                const int ks = (int)kb + 64 * s, ke = min(ks + 64, p.Sk);
                bool apart = false, one = false, edge = false;
                if (docs) {  // (of strips that no row reaches the numbers are not the keys': no term asks for them below)
                    const int kmin = u.range[s][0], kmax = u.range[s][1];
                    apart = qmax < kmin || kmax < qmin;
                    one = qmin == qmax && kmin == kmax && qmin == kmin;
                    edge = kmin == kmax && qmin != qmax && (kmin == qmin || kmin == qmax);
                }
                bool none = true, whole = false, by_row = false;
                for (int t = 0; t < p.n_terms; t++) {
                    const MaskTerm &m = p.terms[t];
                    const int r0 = max(q0, m.q_lo), r1 = min(q1, m.q_hi - 1);  // rows of the tile the term speaks about
                    if (r0 > r1 || (m.doc && apart)) continue;
                    int lo0, hi0, lo1, hi1;
                    term_interval(m, r0, lo0, hi0);
                    term_interval(m, r1, lo1, hi1);
                    // hi(q) <= hi1 and lo(q) >= lo0 on these rows
                    if (hi1 > ks && lo0 < ke) none = false;
                    const bool covers = r0 == q0 && r1 == q1 && lo1 <= ks && hi0 >= ke;
                    if ((!m.doc || one) && covers) whole = true;
                    // keys of one document that some rows have and others have not: all of them or none, row by row
                    if (m.doc && edge && covers && p.n_terms == 1) by_row = true;
                }
                int at = 0;
                if (none || whole || by_row) {
                    const int t0 = ((ks - (int)k_begin) >> p.lbk);
                    for (int j = 0; j < per_strip && t0 + j < tiles; j++) mark(t0 + j, by_row ? 3u : (whole ? 1u : 2u));
                    at = by_row ? kByRow : 0;
                } else {
                    at = atomicAdd(&n_todo, 1) + 1;
                    todo[at - 1] = (uint16_t)s;
                    if (at > kKept) at = 0;
                }
                kept_at[s] = keep_words ? (uint8_t)at : (uint8_t)0;
            }
            __syncthreads();
            // B: a wave takes 64 rows of a strip at a time, wherever it can the same rows of every strip it takes
            const int open = __builtin_amdgcn_readfirstlane(n_todo), groups = (p.BQ + 63) >> 6;
            auto strip_of = [&](int i) { return (int)kb + 64 * __builtin_amdgcn_readfirstlane((int)todo[i]); };
            int i = 0, g = wave, i_step = 0, g_step = kWaves;
            for (; g >= groups; g -= groups) i++;
            for (; g_step >= groups; g_step -= groups) i_step++;
            int ks_next = 0, dk_next = 0;
            if (i < open) {
                ks_next = strip_of(i);
                dk_next = doc_of_key(ks_next, min(64, p.Sk - ks_next));
            }
            int dq, lo, hi;
            auto take_rows = [&]() {
                dq = doc_of_row(64 * g + lane);
                term_interval(p.terms[0], q0 + 64 * g + lane, lo, hi);
            };
            for (take_rows(); i < open;) {
                const int ks = ks_next, dk = dk_next;
                const int n = min(64, p.Sk - ks);
                int i2 = i + i_step, g2 = g + g_step;
                if (g2 >= groups) {
                    g2 -= groups;
                    i2++;
                }
                if (i2 != i && i2 < open) {  // (the next strip's documents travel under this one's words)
                    ks_next = strip_of(i2);
                    dk_next = doc_of_key(ks_next, min(64, p.Sk - ks_next));
                }
                const uint64_t starts = docs ? run_starts(dk) : 0ull;
                const int row = 64 * g + lane;
                const bool in = row < p.BQ;
                const uint64_t w = row_word(p, q0 + row, lo, hi, ks, n, dq, dk, starts);
                if (keep_words && i < kKept && in) u.words[i][row] = w;
                const int t0 = ((ks - (int)k_begin) >> p.lbk);
                for (int j = 0; j < per_strip && t0 + j < tiles; j++) {
                    const uint64_t field = bit_range(j * unit, (j + 1) * unit);
                    const unsigned any = __ballot(in && (w & field) != 0ull) != 0ull;
                    const unsigned gap = __ballot(in && (w & field) != field) != 0ull;
                    if (lane == 0) mark(t0 + j, any | (gap << 1));
                }
                i = i2;
                if (g2 != g) {
                    g = g2;
                    take_rows();
                }
            }
            __syncthreads();
        }
        // C: even waves the FULL list, odd ones the PARTIAL list, of every fourth output plane each
        const int planes = (p.oB_all ? p.oB : 1) * p.oH;
        const unsigned want = (wave & 1) ? 3u : 1u;
        const uint64_t below = (1ull << lane) - 1ull;
        int found = 0;
        for (int pl = wave >> 1; pl < max(planes, kWaves / 2); pl += kWaves / 2) {
            const int b = p.oB_all ? pl / p.oH : ub, h = p.oB_all ? pl % p.oH : pl;
            int32_t *ids = (wave & 1) ? p.part_ids + b * p.pis[0] + h * p.pis[1] + qt * p.pis[2]
                                      : p.full_ids + b * p.fis[0] + h * p.fis[1] + qt * p.fis[2];
            const int64_t step = (wave & 1) ? p.pis[3] : p.fis[3];
            const int before = (wave & 1) ? np : nf;
            found = 0;
            for (int t0 = 0; t0 < tiles; t0 += 64) {
                const bool is = t0 + lane < tiles && reinterpret_cast<const uint8_t *>(state)[t0 + lane] == want;
                const uint64_t bits = __ballot(is);
                const int at = found + __popcll(bits & below);
                if (is && pl < planes) ids[(int64_t)(before + at) * step] = tile0 + t0 + lane;
                if (is && wave == 1 && pl == 0) part[at] = (uint16_t)(t0 + lane);
                found += __popcll(bits);
            }
        }
        if (lane == 0 && wave < 2) sh_min[wave] = found;
        __syncthreads();
        // D
        const int n_part = sh_min[1];
        if (p.packed) {
            const int64_t tile_bytes = (int64_t)p.BQ * p.BK / 8;
            const int row_bytes = p.BK / 8, strips = n_part << lsp;
            uint8_t *out_q = p.packed + (int64_t)ub * p.ob + ((int64_t)qt * p.nK + np) * tile_bytes;
            auto first_key = [&](int i) { return (tile0 + (int)part[i >> lsp]) * p.BK + 64 * (i & ((1 << lsp) - 1)); };
            for (int i = wave; i < strips; i += kWaves) {
                const int ks = first_key(i);
                const int kept = keep_words ? __builtin_amdgcn_readfirstlane((int)kept_at[(ks - (int)k_begin) >> 6]) : 0;
                int dk = 0;
                uint64_t starts = 0ull;
                if (docs && (kept == 0 || kept == kByRow)) {
                    dk = doc_of_key(ks, unit);
                    if (kept == kByRow) dk = __builtin_amdgcn_readfirstlane(dk);
                    else starts = run_starts(dk);
                }
                uint8_t *out_s = out_q + (i >> lsp) * tile_bytes + 8 * (i & ((1 << lsp) - 1));
                for (int r = lane; r < ((p.BQ + 63) & ~63); r += 64) {
                    uint64_t w;
                    if (kept == kByRow) {
                        w = doc_of_row(r) == dk ? ~0ull : 0ull;
                    } else if (kept != 0) {
                        w = u.words[kept - 1][min(r, kKeptRows - 1)] >> (ks & 63);  // (of rows past the tile's end nothing is stored)
                    } else {
                        int lo, hi;
                        term_interval(p.terms[0], q0 + r, lo, hi);
                        w = row_word(p, q0 + r, lo, hi, ks, unit, doc_of_row(r), dk, starts);
                    }
                    uint8_t *out = out_s + (int64_t)r * row_bytes;
                    if (r < p.BQ) {
                        if (unit == 16) {
                            *(uint16_t *)out = (uint16_t)w;
                        } else if (unit == 64) {
                            __builtin_memcpy(__builtin_assume_aligned(out, 4), &w, 8);
                        } else {
                            *(uint32_t *)out = (uint32_t)w;
                        }
                    }
                }
            }
        }
        nf += sh_min[0];
        np += n_part;
        __syncthreads();  // (the next round clears `state` and writes sh_min again)
    }
    const int planes = (p.oB_all ? p.oB : 1) * p.oH;
    for (int pl = threadIdx.x; pl < planes; pl += kThreads) {
        const int b = p.oB_all ? pl / p.oH : ub, h = p.oB_all ? pl % p.oH : pl;
        p.full_lens[b * p.fls[0] + h * p.fls[1] + qt * p.fls[2]] = nf;
        p.part_lens[b * p.pls[0] + h * p.pls[1] + qt * p.pls[2]] = np;
    }
}

}  // namespace

hipError_t launch_mask_terms(const TermsBatch &b, int n, hipStream_t stream) {
    unsigned nQ = 0, planes = 0;
    for (int i = 0; i < n; i++) {
        nQ = b.of[i].nQ > (int)nQ ? b.of[i].nQ : nQ;
        planes = b.of[i].uB > (int)planes ? b.of[i].uB : planes;
    }
    hipLaunchKernelGGL(mask_terms_kernel, dim3(nQ, planes, n), dim3(kThreads), 0, stream, b);
    return hipGetLastError();
}

}  // namespace sa
