// Lists shared by several workgroups (FwdParams::nsplit): when they are, and the sum of their parts.
#include "fwd_common.h"

namespace sa {

namespace {

// One wave per (Q tile, 32 rows, 32 of the D columns), four per workgroup: the parts' rows in the register order they were
// left in (lane (l32, hh): row l32, columns 8g + 4hh + j), so every read is a run of 1 KiB.  The rows are the launch's
// own output of a moment ago and mostly still in a cache; the reads of kBatch parts are in flight together.
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
    const int share = fwd_split_share(NE, p.lbk, lck, p.split_chunks, p.nsplit);
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
        L *= keep;
#pragma unroll
        for (int g = 0; g < 4; g++)
#pragma unroll
            for (int e = 0; e < 4; e++) sum[g][e] *= keep;
#pragma unroll
        for (int i = 0; i < kBatch; i++) {
            if (i0 + i >= share) break;
            const float w = __builtin_amdgcn_exp2f(st[i].x - M0);
            L += w * st[i].y;
#pragma unroll
            for (int g = 0; g < 4; g++)
#pragma unroll
                for (int e = 0; e < 4; e++) sum[g][e] += w * x[i][g][e];
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
// keys takes a workgroup 0.95 us while it has its compute unit to itself and 1.5 us beside another one (D = 128); the
// partial results and their merge cost 4 us plus 12 ns per part.  With few tiles parts of 8 chunks pay for that (64 tiles
// of 16 chunks: 20.4 -> 18.7 us; 8 tiles of 256: 240 -> 31), up to 128 tiles 24 chunks do (128 tiles of 32: 38 -> 33 us,
// of 64: 69 -> 47, of 256: 255 -> 142; parts of 8 made lists of 18 slower, 25 -> 31 us), and between 128 and 256 tiles,
// where a second workgroup per compute unit is all there is to gain, only long lists (256 tiles of 64: 82 -> 75 us, of
// 256: 288 -> 239; of 16: 21 -> 28).  From 257 tiles on every slot has work.  The lengths are on the device: the host
// goes by Sk, and where the lists turn out short (a window) a launch pays 3 to 4 us for the merge that finds nothing.
// float32: a chunk of 32 keys keeps the matrix unit busy for 1.7 us (D = 64) or 3.4 us, so two chunks are worth a part
// (32 tiles of 16 chunks at D = 64: 46 -> 16 us, 256 of 32 at D = 128: 158 -> 95 us).  There the keys of a row are added
// up one after the other, which costs 1.2e-6 of the result at 4096 keys and 3.3e-6 at 32768, shared lists 4e-7 and
// 7e-7; longer rows than 4096 keys stay with the one order of addition, so that a result does not move by more than
// float32 sums may (1.5e-6).
void fwd_split_plan(int tiles, int Sk, int BQ, int D, int dtype, int cus, int *nsplit, int *split_chunks) {
    *nsplit = 1;
    *split_chunks = 1 << 30;
    if (D > 128 || (BQ != 32 && BQ != 64 && BQ != 128) || (dtype == 2 && ((D == 128 && BQ == 32) || Sk > 4096))) return;
    const int lck = dtype == 2 ? 5 : 6;
    const int chunks = (Sk + (1 << lck) - 1) >> lck;  // of the longest list there can be
    const int part = dtype == 2 ? 2 : (4 * tiles <= cus ? 8 : (2 * tiles <= cus ? 16 : 48));
    const int most = 2 * cus / tiles, parts = (chunks + part - 1) / part;
    const int n = parts < most ? parts : most;
    if (n < 2 || chunks < (dtype == 2 ? 4 : 32)) return;
    *nsplit = n < 32 ? n : 32;
    *split_chunks = part;
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
