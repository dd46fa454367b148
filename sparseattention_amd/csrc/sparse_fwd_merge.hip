// Lists shared by several workgroups (FwdParams::nsplit): when they are, and the sum of their parts.
#include "fwd_common.h"

namespace sa {

namespace {

// One wave per (Q tile, 32 rows, 32 of the D columns), four per workgroup: the parts' rows in the register order they were
// left in (lane (l32, hh): row l32, columns 8g + 4hh + j), so every read is a run of 1 KiB.  The rows are the launch's
// own output of a moment ago, past the L2s and mostly still in the memory-side cache; the reads of kBatch parts are in flight together.
constexpr int kBatch = 4;
template <int DT, int D>
__global__ __launch_bounds__(256) void fwd_merge_kernel(const FwdParams p, int lck, int NW) {
    constexpr int NDB = D / 32;
    const int lane = threadIdx.x & 63, l32 = lane & 31, hh = lane >> 5;
    const int id = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int db = id % NDB, rb = (id / NDB) % NW;
    const int tile = id / (NDB * NW);
    if (tile >= p.B * p.H * p.nQ) return;
    const int bh = tile / p.nQ, qt = tile - bh * p.nQ;
    const int b = bh / p.H, h = bh - b * p.H;
    const int F = min(max(p.full_lens[b * p.fls[0] + h * p.fls[1] + qt * p.fls[2]], 0), p.nK);
    const int NE = F + min(max(p.part_lens[b * p.pls[0] + h * p.pls[1] + qt * p.pls[2]], 0), p.nK - F);
    const int share = fwd_split_share(NE, p.lbk, lck, p.split_least, p.split_chunks, p.nsplit);
    if (share <= 1) return;  // written by the workgroup that had the whole list

    const int64_t part0 = (int64_t)tile * p.nsplit;
    const float *const ml = p.ws_ml + 2 * (part0 * (NW * 32) + rb * 32 + l32);
    const float *const wo = p.ws + (part0 * NW + rb) * (32 * D) + 1024 * db + 4 * lane;
    float M = kNegInf, L = 0.f;
    f32x4 sum[4];
#pragma unroll
    for (int g = 0; g < 4; g++) sum[g] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int i0 = 0; i0 < share; i0 += kBatch) {
        // (past the last part: the last one again, left out of the sums below: a weight of 0 would turn an infinity into NaN)
        f32x2 st[kBatch];
        f32x4 x[kBatch][4];
#pragma unroll
        for (int i = 0; i < kBatch; i++) st[i] = *(const f32x2 *)(ml + (int64_t)min(i0 + i, share - 1) * (NW * 64));
#pragma unroll
        for (int i = 0; i < kBatch; i++)
#pragma unroll
            for (int g = 0; g < 4; g++)
                x[i][g] = *(const f32x4 *)(wo + (int64_t)min(i0 + i, share - 1) * NW * (32 * D) + 256 * g);
        float Mn = M;
#pragma unroll
        for (int i = 0; i < kBatch; i++) Mn = fmaxf(Mn, st[i].x);
        const float M0 = Mn == kNegInf ? 0.f : Mn;  // (no part so far saw an attended key: every weight is 0)
        const float keep = __builtin_amdgcn_exp2f(M - M0);
        auto add = [&](int i, float old) {  // (fma by name, so that both forms below round alike)
            const float w = __builtin_amdgcn_exp2f(st[i].x - M0);
            L = i == 0 ? __builtin_fmaf(L, old, w * st[i].y) : __builtin_fmaf(w, st[i].y, L);
#pragma unroll
            for (int g = 0; g < 4; g++)
#pragma unroll
                for (int e = 0; e < 4; e++) sum[g][e] = i == 0 ? __builtin_fmaf(sum[g][e], old, w * x[i][g][e]) : __builtin_fmaf(w, x[i][g][e], sum[g][e]);
        };
        add(0, keep);
        if (i0 + kBatch <= share) {  // (a batch of its own for the usual case: a branch per part cost 0.4 us of a 17 us call)
#pragma unroll
            for (int i = 1; i < kBatch; i++) add(i, 1.f);
        } else {
#pragma unroll
            for (int i = 1; i < kBatch - 1; i++)
                if (i0 + i < share) add(i, 1.f);
        }
        M = Mn;
    }
    const float inv = L > 0.f ? 1.f / L : 0.f;
    const int row = (qt * NW + rb) * 32 + l32;
    if (p.lse != nullptr && db == 0 && hh == 0)
        p.lse[b * p.lses[0] + h * p.lses[1] + (int64_t)row * p.lses[2]] =
            L > 0.f ? (M + __builtin_amdgcn_logf(L)) * 0.69314718056f : kNegInf;
    const int64_t at = b * p.os[0] + h * p.os[1] + (int64_t)row * p.os[2] + 32 * db + 4 * hh;
#pragma unroll
    for (int g = 0; g < 4; g++) {
        if constexpr (DT == 2) {
            *(f32x4 *)(reinterpret_cast<float *>(p.o) + at + 8 * g) = f32x4{sum[g][0] * inv, sum[g][1] * inv, sum[g][2] * inv, sum[g][3] * inv};
        } else {
            using E = Elem<DT == 2 ? 0 : DT>;
            *(u32x2 *)(p.o + at + 8 * g) = u32x2{E::pack2(sum[g][0] * inv, sum[g][1] * inv), E::pack2(sum[g][2] * inv, sum[g][3] * inv)};
        }
    }
}

}  // namespace

// When lists are shared.  A compute unit takes two workgroups of these kernels, so up to 2 * cus of them run at once, and a
// launch of half as many or fewer Q tiles leaves slots empty while each list is walked by one workgroup.  A chunk of 64
// keys takes a workgroup 0.95 us while it has its compute unit to itself and 1.5 us beside another one (D = 128).  The host
// goes by Sk; the lengths are on the device, and a launch pays 2 to 3 us for a merge that finds nothing to do.  us at D = 128,
// bf16, every list as long as stated, one workgroup per list | shared (and "alone" in such a launch: with that merge):
//   parts of 8 chunks, up to cus / 4 tiles
//       8 tiles   8 chunks  12.1 | alone 14.0    12  15.9 | 14.2    32  34.1 | 17.3    256  240 | 31
//      64 tiles   4 chunks   9.0 | alone 11.5    12  16.7 | 19.9    16  20.0 | 21.2    24  27.4 | 24.1    64  63.9 | 32.6
//   parts of 16 chunks, up to cus / 2 tiles, lists of more than 8 + tiles / 8 chunks (beside each other workgroups take half as
//   long again: two of 9 chunks are no faster than one of 18)
//      65 tiles  16 chunks  19.8 | alone 22.8    17  21.1 | 22.6    20  23.5 | 23.6    64  63.8 | 36.2
//      96 tiles  17 chunks  21.2 | 25.1          20  23.6 | 26.3    24  27.4 | 28.2    64  64.1 | 39.4
//     128 tiles  16 chunks  20.3 | alone 22.9    17  21.1 | 27.2    24  27.2 | 30.5    28  31.0 | 32.1    64  64.8 | 46.3
//   parts of 48 chunks, up to cus tiles, where a second workgroup per compute unit is all there is to gain (and lists are not
//   walked in halves, see fwd_in_halves)
//     192 tiles  32 chunks  35.1 | alone 38.2    49  51.8 | 52.0    64  67.3 | 62.4   128 125.5 | 107.5
//     256 tiles  48 chunks  55.9 | alone 58.0    49  56.9 | 62.0    64  72.7 | 74.8   128 135.3 | 130.1   256  288 | 239
// From 257 tiles on every slot has work.  Sk below 32 chunks is not shared, whatever the lists (32 chunks, Sk = 2048: 8 tiles
// 33.6 | 17.0, 64 tiles 34.7 | 26.3, 128 tiles 35.2 | 33.6; 16 chunks: the tables above, as lists of a longer Sk).
// float32: a chunk of 32 keys keeps the matrix unit busy for 1.7 us (D = 64) or 3.4 us, so two chunks are worth a part
// (32 tiles of 16 chunks at D = 64: 46 -> 11.4 us, 256 of 32 at D = 128, BLOCK_Q 64: 158 -> 93 us).  At D = 128, BLOCK_Q 64 the two groups of
// a workgroup take a compute unit's LDS: parts for one workgroup a unit where those fill seven eighths of the units.  Every list that
// long, us, parts for two workgroups a unit | one:
//    16 tiles of 64 chunks 35.8 | 23.7   32 of 16 16.8 | 16.6, of 32 30.0 | 21.4, of 128 56.7 | 50.9   48 of 32 39.1 | 28.9   64 of 64 55.8 | 49.0
//   128 of 32 55.2 | 48.2, of 128 166 | 161   and three quarters of them: 96 of 16 35.5 | 28.5, of 64 81.6 | 85.0, of 128 138 | 160
// Sk above 4096 is not shared there: a row's
// keys are added up one after the other in one workgroup, 1.2e-6 from the result at 4096 keys and 3.3e-6 at 32768, and shared
// lists (4e-7 and 7e-7) would move the result by that much.
FwdSplitPlan fwd_split_plan(int tiles, int Sk, int BQ, int D, int dtype, int cus) {
    FwdSplitPlan plan;
    if (D > 128 || (BQ != 32 && BQ != 64 && BQ != 128) || (dtype == 2 && ((D == 128 && BQ == 32) || Sk > 4096))) return plan;
    const int lck = dtype == 2 ? 5 : 6;
    const int chunks = (Sk + (1 << lck) - 1) >> lck;  // of the longest list there can be
    const int part = dtype == 2 ? 2 : (4 * tiles <= cus ? 8 : (2 * tiles <= cus ? 16 : 48));
    const bool lone = dtype == 2 && D == 128 && BQ == 64 && 2 * tiles <= cus && 8 * (cus / tiles * tiles) >= 7 * cus;
    const int most = lone ? cus / tiles : 2 * cus / tiles, parts = (chunks + part - 1) / part;
    const int n = parts < most ? parts : most;
    if (n < 2 || chunks < (dtype == 2 ? 4 : 32)) return plan;
    plan.nsplit = n < 32 ? n : 32;
    plan.chunks = part;
    plan.least = part == 16 ? 8 + tiles / 8 : part;
    return plan;
}

// One workgroup reads all parts of its Q tile, where a second launch spreads them over the device: in the launch up to 256 KiB a tile.
// float32, us, second launch | last workgroup (parts x KiB a part, every list that long):
//   8 x 16  32 tiles 13.3 | 11.7    32 x 8  8 tiles 19.8 | 17.5    8 x 32  32 tiles 18.5 | 17.3
//   32 x 16  16 tiles 25.2 | 24.9, 8 tiles 21.0 | 20.7, 4 tiles 20.2 | 20.4    16 x 32  16 tiles 20.1 | 20.0    8 x 64  16 tiles 21.9 | 23.6
//   32 x 32  8 tiles 29.2 | 33.6, 4 tiles 25.0 | 29.6    16 x 64  16 tiles 28.9 | 30.6    32 x 64  4 tiles 38.0 | 50.7
// bf16, where one wave reads 32 rows of every part: up to four parts, of 64 KiB only where there are more than 16 tiles to add up side by side
//   4 x 64  128 tiles of up to 256 chunks 136.0 | 132.8, 128 72.3 | 68.8, 64 45.3 | 42.0, 25 28.7 | 25.8; 64 tiles of 32 22.7 | 21.3, 32 tiles 20.6 | 18.7
//   4 x 32  128 tiles, D = 64, of up to 256 79.3 | 76.8, BLOCK_Q 64 of up to 128 58.3 | 58.1    4 x 16  128 tiles of up to 128 45.9 | 41.5
//   8 x 32  8 tiles of 64, D = 64 14.4 | 14.8, 64 tiles of up to 128 29.4 | 29.3, BLOCK_Q 64 36.8 | 38.2, 16 tiles of 64 21.0 | 21.9
//   4 x 64  of 32 chunks  8 tiles 16.4 | 17.6   16 tiles 17.5 | 17.9   32 tiles 20.4 | 18.7   64 tiles 25.2 | 21.2
// For a second launch too parts are stored past L2 (HandOver): a launch whose parts lie in the L2s ends with writing them back.  bf16, us, a kernel
// of its own without the adding up and with stores through L2 | this one: 64 tiles of 64 chunks, BLOCK_Q 64, D = 64 22.5 | 20.6, D = 128
// 27.0 | 25.7; 32 tiles of 256, D = 64 30.5 | 27.6; 16 tiles of 128, BLOCK_Q 128 24.8 | 23.7; it loses at 8 tiles of 128, BLOCK_Q 64, D = 64 16.3 | 17.3.
bool fwd_merges_in_launch(int tiles, int nsplit, int BQ, int D, int dtype) {
    const int64_t bytes = (int64_t)nsplit * BQ * D * 4;
    return bytes <= 256 * 1024 && (dtype == 2 || (nsplit <= 4 && (bytes <= 128 * 1024 || tiles > 16)));
}

// When a list is walked in two halves by one workgroup of twice the waves (sparse_fwd_kernel<..., TW>): from half as many Q tiles
// as compute units on, up to as many.  A compute unit has one workgroup then, which leaves half of its registers and LDS
// idle, at BLOCK_Q = 64 two of its four SIMDs too.  No workspace, no second launch; but a long list stays on its compute unit,
// where parts of it would go to units whose own lists are short.  bf16 and fp16, us, D = 128 where not said:
//   BLOCK_Q 128, Sk of 49 to 72 chunks, or 96 where every compute unit has a tile.  Shared by two with a merge | halves, lists that
//   grow evenly from an eighth of the keys to all ("causal") and lists of all keys:
//       136 tiles  causal  64 chunks 63.0 | 51.6   72 60.5 | 56.6   80 61.3 | 61.7    96 70.8 | 72.3    all  96 73.6 | 73.4
//       192 tiles  causal  64        58.9 | 51.7   72 57.5 | 57.4   96 71.7 | 73.0   192 122.6 | 138.4  all  96 83.3 | 79.0   192 148.8 | 148.8
//       240 tiles  causal  64        62.1 | 54.0   72 61.1 | 60.3   88 69.8 | 72.5   192 134.7 | 147.2  all  96 95.9 | 90.8
//       256 tiles  causal  64        62.0 | 54.9   80 69.3 | 67.4   96 79.0 | 78.9   192 146.6 | 149.5  all  96 99.9 | 94.2   192 178.9 | 178.9
//       D = 64     causal  224 tiles 72 chunks 41.5 | 41.8   88 45.9 | 49.0    256 tiles  72 41.9 | 42.1   96 52.9 | 53.3
//       256 tiles  window 64  12.5 | 10.5   256  15.1 | 13.1   900, BLOCK_K 32  26.6 | 22.9
//   (with shorter rows the launch had no merge to save, and lists of up to 16 chunks would pay up to 1.4 us for the wider workgroup,
//   fwd_halves_least; longer ones gain little: causal Sk 1024 21.4 | 20.2, every key of 2048 39.2 | 36.7)
//   BLOCK_Q 64, one workgroup per list (Sk up to 48 chunks) or shared by two with a merge | halves
//       256 tiles  causal  16 chunks 24.5 | 17.8   64, D = 64 51.1 | 34.8   256 203.0 | 197.4   all 128 104.6 | 96.6
//                  window 256  12.2 | 12.0   window 64 (lists of two chunks)  9.1 | 9.5
//       160 tiles  causal Sk 1280  30.7 | 20.6   window 500  17.6 | 14.7
//       192 tiles  causal  128 100.6 | 96.5   256 191.0 | 185.4         (D = 64: 77.3 | 72.6, 145.9 | 139.5)
//       224 tiles  causal   96  76.1 | 74.3   128  98.3 | 99.8   256 188.3 | 193.0   (D = 64: 80.2 | 72.4, 141.3 | 140.3)
//       240 tiles  causal   96  76.2 | 75.5   128  99.2 | 104.2  256 188.2 | 201.3
// Up to two thirds as many tiles as compute units lists of more than 96 chunks are shared by three workgroups (BLOCK_Q 128, 136 tiles of
// 8192 keys: 78.1 | 88.9).
bool fwd_in_halves(int64_t tiles, int Sk, int BQ, int BK, int D, int dtype, int cus) {
    if (dtype == 2 || (D != 64 && D != 128) || BK < 32 || 2 * tiles <= cus || tiles > cus) return false;
    if (BQ == 128) return Sk > 48 * 64 && Sk <= (tiles == cus ? 96 : 72) * 64;
    if (BQ != 64 || Sk < 1024) return false;
    if (Sk <= 96 * 64) return true;
    return 3 * tiles > 2 * cus && (D == 64 || 4 * tiles <= 3 * cus || tiles == cus);
}

// When every list has an assistant (sparse_fwd_kernel<..., AS>): up to one Q tile of 128 rows a compute unit, more than half as many, where neither
// parts by the length of Sk nor halves serve.  A unit has one workgroup then, which takes 0.95 us a chunk, and the longest list ends the
// launch.  The second workgroups of the grid land on the units in the order of the first ones, so which tile an assistant sits beside is known, and
// the two lists' lengths say what it takes: half the difference, from eight chunks on (less does not pay for the meeting of the parts, 3 us), or
// on a unit of its own half the list, where that is longer than the longest that has to share.  Both workgroups decide alike from the same
// counts.  us, one workgroup a list | with assistants, bf16:
//   causal     256 tiles  D = 128  16 chunks 22.5 | 21.1   20 24.2 | 20.2 (160 tiles)   32 36.8 | 29.0   D = 64  32 26.2 | 20.6
//              192 tiles  16 20.7 | 18.4   48 50.3 | 35.1
//   documents of 64 ... 1024  256 tiles 32 chunks 22.2 | 20.1, D = 64 16.5 | 14.7   192 tiles 16 17.5 | 15.9   160 tiles 20 17.4 | 15.8
// Lists with nothing to assist pay for the place and the counts of the tile beside, about 0.4 us, and for second workgroups that end at once, about 0.3.  Where
// the lists are known to be alike they get none (sa_fwd_split_uneven_keys); where nothing is known:
//   every key  256 tiles 16 22.3 | 23.0   32 38.2 | 39.8, D = 64 27.4 | 27.3   192 tiles 16 21.1 | 21.6   48 50.8 | 51.8
//   blocks of 128 keys, a half empty, three masks  16 18.2 | 19.3, 17.4 | 18.5, 19.6 | 20.3   32 28.8 | 29.6, 27.3 | 26.3, 25.4 | 26.4   192 tiles 48 40.8 | 35.6, 34.5 | 34.9, 36.5 | 35.3
//   window of 200 keys  16 12.4 | 13.2   32 12.5 | 13.1, D = 64 9.5 | 9.8   192 tiles 48 12.2 | 12.4   of 1000 keys  32 23.6 | 25.4   192 tiles 48 23.8 | 24.0
//   16 chunks at D = 64: causal 16.7 | 15.9, every key 17.7 | 18.4.  12 chunks: causal 17.1 | 17.5.
// A whole call on a fresh causal mask of S1024 26.9 | 24.8, on another device 27.0 | 25.6.  Other bits than one workgroup a list gives, since each part's P is rounded against a reference value
// of its own.  The error against float64 is less in all of 46 cases (nine shapes, causal, documents and blocks, both types), by 0.003 to 0.07 %: causal S1024
// bf16 2.4710e-3 | 2.4701e-3, S2048 fp16 3.1557e-4 | 3.1547e-4.
// From 49 chunks on halves stay: causal 64 chunks of S4096 54.1 | 46.6, but every key 68.0 | 77.6, causal Sq 2048 Sk 4096 61.0 | 66.9.
bool fwd_assists(int64_t planes, int nQ, int Sk, int BQ, int BK, int D, int dtype, int cus) {
    const int64_t tiles = planes * nQ;
    const int chunks = (Sk + 63) / 64;
    return dtype != 2 && (D == 64 || D == 128) && BQ == 128 && BK >= 32 && cus == 256 && planes % 8 == 0 && 2 * tiles > cus && tiles <= cus && chunks >= (D == 64 ? 24 : 16) && chunks <= 48;
}

// A caller who knows that all lists are short does without the wider workgroup: us, one workgroup of half the waves | halves, 256 tiles,
// every list as long as stated (kept whole by the first half up to 10 chunks, at BLOCK_Q 64 up to 4: sparse_fwd_kernel's LEAST)
//   BLOCK_Q 128          4 chunks  9.7 | 10.8    8 13.6 | 14.9   12 18.0 | 19.0   14 20.5 | 21.1   16 22.4 | 22.6   20 26.6 | 26.2
//                D = 64  4 chunks  7.5 |  8.2    8 10.4 | 10.7   13 13.2 | 13.5   14 13.9 | 13.8   16 15.3 | 15.0   20 18.1 | 17.2
//   BLOCK_Q 64           2 chunks  7.8 |  8.4    4 10.2 | 10.9    5 11.4 | 11.5    6 12.5 | 11.6    8 15.0 | 12.9
//                D = 64  2 chunks  6.0 |  6.6    4  7.8 |  8.4    5  8.7 |  9.1    6  9.4 |  9.0    8 11.1 | 10.0
int fwd_halves_least(int BQ, int D) { return BQ == 64 ? 5 : (D == 64 ? 13 : 16); }

// How many planes are walked together (an XCD has an eighth of them, see below), their Q tiles side by side from the last one down.  An XCD's first 32 workgroups
// go to its 32 compute units, the next 32 to the same ones: with planes two by two and 16 Q tiles a plane the second workgroup of a unit has
// the first one's Q tile in another plane, under a causal mask (or the documents of one batch element) a list as long, and the
// units of the longest lists finish last, alone.  Side by side the longest lists of all planes go to different units, and the second 32 the
// other way round (sparse_fwd_kernel), so that a unit's two lists add up to about the same.  us, two by two | side by side:
//   causal      512 tiles  B2 H16 S2048 52.0 | 46.7   D = 64 34.7 | 30.0   B1 H16 S4096 86.5 | 80.6   B1 H8 S8192 158.4 | 147.4
//               768  B4 H12 S2048 66.7 | 59.5, D = 64 44.8 | 36.5     1024  B4 H16 S2048 85.1 | 75.8   B8 H16 S1024 56.1 | 47.8
//   documents   768  54.8 | 51.0, D = 64 28.5 | 23.1   1024  65.8 | 62.6   B8 H16 S1024, D = 64 32.1 | 25.8   B2 H32, BLOCK_Q 64 41.6 | 31.9
//   every key   512  67.5 | 66.7   768 102.6 | 103.5   1024  123.3 | 123.7   blocks  512 43.7 | 45.1   768 64.0 | 64.6   1024 80.1 | 80.0
// As many as leave their K and V in the XCD's 4 MiB of L2, two by two | those | more of them:
//   1024 tiles, 1 MiB a plane, causal 85.1 | 75.8 | 73.3, blocks 80.1 | 80.0 | 82.9, every key 123.3 | 123.7 | 125.0
//   2048 tiles, 1 MiB, causal 151.9 | 145.0 | 147.9, blocks 105.0 | 101.0 | 113.0, documents 137.3 | 135.8 | 140.8
//   2048 tiles, 1/2 MiB, causal 96.6 | 92.0 | 99.2, documents 87.3 | 84.4 | 87.7; D = 64 91.8 | 85.0 | 84.2, documents 84.1 | 81.0 | 80.0
//   4096 tiles, 2 MiB (two fit), causal 493.9 | - | 499.4, blocks 316.8 | - | 338.9, documents 315.2 | - | 348.1
// An odd number of planes an XCD cannot be taken two by two (two XCDs shared a pair, one its long lists): then up to 6 MiB, else one by one.
//   B1 H24 S4096 causal 113.9 | 105.5, blocks 114.7 | 113.9, documents 62.3 | 57.8   B3 H24 311 | 282, 276 | 280, 137 | 124
//   one by one  B5 H8 S4096 187 | 179, blocks 166.3 | 166.2, documents 87.8 | 82.3   B1 H8 S16384 537 | 460, documents 69 | 75
//   (documents of one plane an XCD go either way by mask, -26 ... +20 % over 63 of them at S8192 ... 32768, -1.8 % in the mean)
// Planes that are an odd number of fours (12 heads, 4 heads) took two by two leave one XCD the long lists of a pair and another its short ones; side
// by side a plane's Q tiles go to two XCDs in turn, by twos:
//   causal B3 H12 S2048 60.9 | 54.4   B1 H4 S16384 347 | 304   B1 H12 S8192 D = 64 137 | 132   B1 H12 S4096 84.3 | 81.4   B5 H12 S1024 31.3 | 30.9
//   documents B3 H12 S2048 37.2 | 34.3   B5 H12 S1024 29.8 | 27.9   blocks 87.5 | 86.0, 36.3 | 38.1   every key 98.8 | 99.3
//   window of 500 keys B3 H12 S2048 37.4 | 38.4   B1 H12 S8192 D = 64 25.3 | 27.4 (one by one, not by twos: 24.1 | 25.8 for 25.0 | 25.8 at S4096)
//   (on another device 36.3 | 35.0, 24.1 | 25.1, of 1000 keys B3 H12 S2048 46.2 | 41.1: no reason to leave windows out where they are known)
//   float32 B3 H12 S1152 D = 64 causal 154.5 | 110.8, documents 125.6 | 108.5
// float32, whose chunks keep the matrix unit busy four to eight times as long: causal B2 H16 S1024 D64 144.2 | 88.9, B4 H12 148.8 | 108.0,
// B1 H8 S4096 479 | 321, BLOCK_Q 128 B3 H8 S2048 281 | 199; documents B2 H16 S1024 120.7 | 89.2; every key 144.5 | 144.3; D = 128 B1 H16 S2048 313 | 311.
int fwd_spread(int64_t planes, int nQ, int BQ, int64_t plane_bytes, int cus) {
    if (planes % 4 != 0 || planes * nQ <= cus || (BQ != 64 && BQ != 128)) return 0;  // (BLOCK_Q 32 B4 H8 S2048 causal 106.9 | 108.1)
    const int unit = planes % 8 != 0 ? 4 : 8;
    const int64_t each = planes / unit, most = (each % 2 != 0 ? 6 << 20 : 4 << 20) / (plane_bytes > 0 ? plane_bytes : 1);
    if (each <= 2) return (int)planes;
    int64_t n = most < each ? most : each;
    while (n > 1 && each % n != 0) n--;
    return n > 2 ? (int)(unit * n) : (each % 2 != 0 ? unit : 0);
}

hipError_t launch_fwd_merge(const FwdParams &p, int dtype, int D, int BQ, hipStream_t stream) {
    const int NW = BQ / 32, lck = dtype == 2 ? 5 : 6;
    const int64_t waves = (int64_t)p.B * p.H * p.nQ * NW * (D / 32);
    const dim3 grid((unsigned)((waves + 3) / 4)), block(256);
#define SA_MERGE(DT, DD) \
    if (dtype == DT && D == DD) hipLaunchKernelGGL((fwd_merge_kernel<DT, DD>), grid, block, 0, stream, p, lck, NW)
    SA_MERGE(0, 64);
    else SA_MERGE(0, 128);
    else SA_MERGE(1, 64);
    else SA_MERGE(1, 128);
    else SA_MERGE(2, 64);
    else SA_MERGE(2, 128);
    else return hipErrorInvalidValue;
#undef SA_MERGE
    return hipGetLastError();
}

}  // namespace sa
