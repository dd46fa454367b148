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
    const int before = __shfl_up(dk, 1);
    return __ballot(lane == 0 || dk != before);
}

// The mask entries of this lane's query row q against the keys ks .. ks + n - 1 (n <= 64; lane i holds the document of
// key ks + i in dk), bit i = key ks + i.  All lanes of the wave have to be active.
__device__ __forceinline__ uint64_t row_word(const TermsParams &p, int q, int ks, int n, int dq, int dk, uint64_t starts) {
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
    for (int t = 0; t < p.n_terms; t++) {
        int lo, hi;
        term_interval(p.terms[t], q, lo, hi);
        const uint64_t w = bit_range(min(max(lo - ks, 0), 64), min(max(hi - ks, 0), 64));
        word |= p.terms[t].doc ? w & same : w;
    }
    return word & bit_range(0, n);
}

// grid (nQ, distinct planes, masks), 512 threads: a workgroup makes everything of one Q tile, so nothing goes through memory
// between classification, lists and packed tiles.  Per round of at most kTiles tiles:
//   A  a strip of 64 keys is decided from the first and the last row of the Q tile where it can be (both ends of a
//      row's interval move right, or stay, as q grows): no term reaches it, or one term covers it from every row,
//      document conditions judged by the ranges of the document numbers on both sides (16 lanes read a strip's).
//   B  the other strips, a wave each: lane = query row, one 64-bit word of entries per row (row_word), and two ballots
//      per tile tell whether some entry attends and whether some does not.
//   C  a wave per list compacts the tiles' states by ballot and popcount.
//   D  the PARTIAL tiles' words are made again, a wave per strip, and stored: they cost less than keeping them.
// Latency bound (a few dependent reads of documents; a word is a few dozen instructions per 64 rows and strip), so the
// documents of the rows stay in LDS and those of the next strip are requested under the words of this one.  Against
// classification with one key per lane and one row per step, compaction and packing as three kernels that evaluated the
// terms per entry (launches back to back in a graph): causal documents B4 S2048 tiles 128x64 71 -> 10.3 us, B4 S16384
// tiles 128x32 352 -> 44 us, window and prefix at S32768 149 -> 9.5 us.  1024 threads: 10.4 / 49 / 10.5 us.
// The two tilings of a backward come from one launch: few Q tiles each (B4 S2048: 64 workgroups), and most of a launch is the start
// of a compute unit that has none of the code yet.  Causal documents B4 S2048 20.0 -> 10.6 us, B8 S4096 24.5 -> 14.8, B1 S32768 53 -> 33.
__global__ __launch_bounds__(kThreads) void mask_terms_kernel(const TermsBatch batch) {
    const TermsParams &p = batch.of[blockIdx.z];
    if ((int)blockIdx.x >= p.nQ || (int)blockIdx.y >= p.uB) return;
    __shared__ unsigned state[kTiles];  // bit 0: some entry attends, bit 1: some entry does not
    __shared__ uint16_t part[kTiles];   // the PARTIAL tiles of the round, in order
    __shared__ uint16_t todo[kStrips];  // strips that step A left open
    __shared__ int n_todo, sh_min[kWaves], sh_max[kWaves], row_doc[kRows];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int qt = blockIdx.x, ub = blockIdx.y;
    const int q0 = qt * p.BQ, q1 = q0 + p.BQ - 1;
    const int32_t *dqp = p.doc_q ? p.doc_q + (int64_t)ub * p.dqs[0] : nullptr;
    const int32_t *dkp = p.doc_k ? p.doc_k + (int64_t)ub * p.dks[0] : nullptr;
    const bool docs = dqp && dkp;

    int qmin = INT32_MAX, qmax = INT32_MIN;
    if (docs) {
        for (int r = threadIdx.x; r < p.BQ; r += kThreads) {
            const int d = dqp[(int64_t)(q0 + r) * p.dqs[1]];
            if (r < kRows) row_doc[r] = d;
            qmin = min(qmin, d);
            qmax = max(qmax, d);
        }
#pragma unroll
        for (int sh = 32; sh >= 1; sh >>= 1) {
            qmin = min(qmin, __shfl_xor(qmin, sh));
            qmax = max(qmax, __shfl_xor(qmax, sh));
        }
        if (lane == 0) {
            sh_min[wave] = qmin;
            sh_max[wave] = qmax;
        }
        __syncthreads();
#pragma unroll
        for (int w = 0; w < kWaves; w++) {
            qmin = min(qmin, sh_min[w]);
            qmax = max(qmax, sh_max[w]);
        }
    }

    auto doc_of_row = [&](int r) {
        return !docs || r >= p.BQ ? 0 : (r < kRows ? row_doc[r] : dqp[(int64_t)(q0 + r) * p.dqs[1]]);
    };
    auto doc_of_key = [&](int ks, int n) { return docs && lane < n ? dkp[(int64_t)(ks + lane) * p.dks[1]] : 0; };

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
    int nf = 0, np = 0;
    for (int tile0 = 0; tile0 < p.nK; tile0 += round) {
        const int tiles = min(round, p.nK - tile0);
        const int64_t k_begin = (int64_t)tile0 * p.BK, k_stop = (int64_t)(tile0 + tiles) * p.BK;
        for (int i = threadIdx.x; i < tiles; i += kThreads) state[i] = 0u;
        for (int64_t kb = k_begin; kb < k_stop; kb += kStrips * 64) {
            const int strips = (int)(min((int64_t)(kStrips * 64), k_stop - kb) + 63) >> 6;
            if (threadIdx.x == 0) n_todo = 0;
            __syncthreads();
            // A
            const int group = docs ? 16 : 1;
            for (int s0 = 0; s0 < strips; s0 += kThreads / group) {
                const int s = s0 + (int)threadIdx.x / group;
                const int ks = (int)kb + 64 * s, ke = min(ks + 64, p.Sk);
                bool apart = false, one = false;
                if (docs && ks < reach_hi && ke > reach_lo) {
                    int kmin = INT32_MAX, kmax = INT32_MIN;
                    if (s < strips) {
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            const int k = ks + 16 * i + (lane & 15);
                            if (k < ke) {
                                const int d = dkp[(int64_t)k * p.dks[1]];
                                kmin = min(kmin, d);
                                kmax = max(kmax, d);
                            }
                        }
                    }
#pragma unroll
                    for (int sh = 8; sh >= 1; sh >>= 1) {
                        kmin = min(kmin, __shfl_xor(kmin, sh));
                        kmax = max(kmax, __shfl_xor(kmax, sh));
                    }
                    apart = qmax < kmin || kmax < qmin;
                    one = qmin == qmax && kmin == kmax && qmin == kmin;
                }
                if (s >= strips || (int)threadIdx.x % group != 0) continue;
                bool none = true, whole = false;
                for (int t = 0; t < p.n_terms; t++) {
                    const MaskTerm &m = p.terms[t];
                    const int r0 = max(q0, m.q_lo), r1 = min(q1, m.q_hi - 1);  // rows of the tile the term speaks about
                    if (r0 > r1 || (m.doc && apart)) continue;
                    int lo0, hi0, lo1, hi1;
                    term_interval(m, r0, lo0, hi0);
                    term_interval(m, r1, lo1, hi1);
                    // hi(q) <= hi1 and lo(q) >= lo0 on these rows
                    if (hi1 > ks && lo0 < ke) none = false;
                    if ((!m.doc || one) && r0 == q0 && r1 == q1 && lo1 <= ks && hi0 >= ke) whole = true;
                }
                if (none || whole) {
                    const int t0 = ((ks - (int)k_begin) >> p.lbk);
                    for (int j = 0; j < per_strip && t0 + j < tiles; j++) atomicOr(&state[t0 + j], whole ? 1u : 2u);
                } else {
                    todo[atomicAdd(&n_todo, 1)] = (uint16_t)s;
                }
            }
            __syncthreads();
            // B
            const int open = n_todo;
            int dk_next = wave < open ? doc_of_key((int)kb + 64 * (int)todo[wave], min(64, p.Sk - ((int)kb + 64 * (int)todo[wave]))) : 0;
            for (int i = wave; i < open; i += kWaves) {
                const int ks = (int)kb + 64 * (int)todo[i];
                const int n = min(64, p.Sk - ks);
                const int dk = dk_next;
                if (i + kWaves < open) {  // (the next strip's documents travel under this one's words)
                    const int kn = (int)kb + 64 * (int)todo[i + kWaves];
                    dk_next = doc_of_key(kn, min(64, p.Sk - kn));
                }
                const uint64_t starts = docs ? run_starts(dk) : 0ull;
                uint64_t some = 0ull, every = ~0ull;
                for (int r0 = 0; r0 < p.BQ; r0 += 64) {
                    const int q = q0 + r0 + lane;
                    const bool in = r0 + lane < p.BQ;
                    const uint64_t w = row_word(p, q, ks, n, doc_of_row(r0 + lane), dk, starts);
                    some |= in ? w : 0ull;
                    every &= in ? w : ~0ull;
                }
                const int t0 = ((ks - (int)k_begin) >> p.lbk);
                for (int j = 0; j < per_strip && t0 + j < tiles; j++) {
                    const uint64_t field = bit_range(j * unit, (j + 1) * unit);
                    const unsigned any = __ballot((some & field) != 0ull) != 0ull;
                    const unsigned gap = __ballot((every & field) != field) != 0ull;
                    if (lane == 0) atomicOr(&state[t0 + j], any | (gap << 1));
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
                const bool is = t0 + lane < tiles && state[t0 + lane] == want;
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
            int dk_next = wave < strips ? doc_of_key(first_key(wave), unit) : 0;
            for (int i = wave; i < strips; i += kWaves) {
                const int ks = first_key(i), dk = dk_next;
                if (i + kWaves < strips) dk_next = doc_of_key(first_key(i + kWaves), unit);
                const uint64_t starts = docs ? run_starts(dk) : 0ull;
                uint8_t *out_s = out_q + (i >> lsp) * tile_bytes + 8 * (i & ((1 << lsp) - 1));
                for (int r = lane; r < ((p.BQ + 63) & ~63); r += 64) {
                    const uint64_t w = row_word(p, q0 + r, ks, unit, doc_of_row(r), dk, starts);
                    uint8_t *out = out_s + (int64_t)r * row_bytes;
                    if (r < p.BQ) {
                        if (unit == 16) {
                            *(uint16_t *)out = (uint16_t)w;
                        } else {
                            ((uint32_t *)out)[0] = (uint32_t)w;
                            if (unit == 64) ((uint32_t *)out)[1] = (uint32_t)(w >> 32);
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
