// Tile classification of a boolean attention mask on gfx950 (MI355X).
//
// Replaces the Triton kernel _compute_mask_inner (sparseattention/mask_utils.py:47-82), which walks the
// KV tiles of one Q-tile row serially and loads 32-byte row segments.  Here the work is split in two:
//
//   classify_wide_kernel / classify_generic_kernel
//       one class byte per (plane, Q tile, KV tile): 0 = empty, 1 = partial, 2 = full.  The wide kernel
//       streams the mask with 16-byte loads, 1 KiB contiguous per wave per row, and every byte of a
//       distinct plane is read exactly once.
//   compact_kernel
//       one wave per (b, h, Q tile): ballot + popcount prefix over the class bytes, writing the two
//       ascending index lists and their counts (mask_utils.py:72-82).
//   pack_partial_kernel (optional, no counterpart in the reference)
//       one bit per entry of every PARTIAL tile, so that the forward reads BQ*BK/8 contiguous bytes per
//       partial tile instead of BQ row segments of the mask (sparse_attn_kernel.py:42-46).
//   classify_rows_kernel
//       all three in one launch, for masks of few bytes per Q tile and for large ones of many Q tiles.
//
// A byte != 0 counts as "attend", so masks that were viewed from uint8 storage behave like torch.sum.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.h"

namespace sa {

namespace {

// 0x80 in every byte of x that is non-zero.
__device__ __forceinline__ uint32_t nonzero_bytes(uint32_t x) {
    return (((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x) & 0x80808080u;
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kWideCols = 1024;  // mask columns covered by one workgroup: 64 lanes x 16 bytes
constexpr int kRowUnroll = 8;    // independent 16-byte loads in flight per lane

// grid (ceil(Sk/1024), nQ, distinct planes), 256 threads.  The four waves of a workgroup take rows
// w, w+4, ... of the same BQ x 1024 slab, so consecutive lanes always read consecutive 16-byte
// pieces of one mask row; the per-wave results meet in LDS.
__global__ __launch_bounds__(256) void classify_wide_kernel(const ClassifyParams p) {
    __shared__ unsigned long long sh_all[4];
    __shared__ unsigned long long sh_any[4];

    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int qt = blockIdx.y;
    const int plane = blockIdx.z;
    const int ub = plane / p.uH, uh = plane - ub * p.uH;
    const int col = blockIdx.x * kWideCols + lane * 16;
    const bool in_range = col < p.Sk;

    uint32_t any = 0u, all = 0x80808080u;
    if (in_range) {
        const uint8_t *base = p.mask + (int64_t)ub * p.sb + (int64_t)uh * p.sh + (int64_t)qt * p.BQ * p.sq + col;
        int r = wave;
        for (; r + 4 * (kRowUnroll - 1) < p.BQ; r += 4 * kRowUnroll) {
            u32x4 v[kRowUnroll];
#pragma unroll
            for (int u = 0; u < kRowUnroll; u++)
                v[u] = __builtin_nontemporal_load((const u32x4 *)(base + (int64_t)(r + 4 * u) * p.sq));
#pragma unroll
            for (int u = 0; u < kRowUnroll; u++) {
                any |= v[u].x | v[u].y | v[u].z | v[u].w;
                all &= nonzero_bytes(v[u].x) & nonzero_bytes(v[u].y) & nonzero_bytes(v[u].z) & nonzero_bytes(v[u].w);
            }
        }
        for (; r < p.BQ; r += 4) {
            const u32x4 v = __builtin_nontemporal_load((const u32x4 *)(base + (int64_t)r * p.sq));
            any |= v.x | v.y | v.z | v.w;
            all &= nonzero_bytes(v.x) & nonzero_bytes(v.y) & nonzero_bytes(v.z) & nonzero_bytes(v.w);
        }
    }
    const unsigned long long ball_all = __ballot(all == 0x80808080u);
    const unsigned long long ball_any = __ballot(any != 0u);
    if (lane == 0) {
        sh_all[wave] = ball_all;
        sh_any[wave] = ball_any;
    }
    __syncthreads();

    const int tiles = kWideCols >> p.lbk;  // KV tiles per slab, <= 64
    const int t = threadIdx.x;
    if (t < tiles) {
        const int kt = blockIdx.x * tiles + t;
        if (kt < p.nK) {
            const unsigned long long a = sh_all[0] & sh_all[1] & sh_all[2] & sh_all[3];
            const unsigned long long o = sh_any[0] | sh_any[1] | sh_any[2] | sh_any[3];
            const int lpt = p.BK >> 4;  // lanes per tile
            const unsigned long long field = lpt == 64 ? ~0ull : (((1ull << lpt) - 1ull) << (t * lpt));
            const uint8_t cls = (a & field) == field ? 2 : ((o & field) != 0ull ? 1 : 0);
            p.cls[((int64_t)plane * p.nQ + qt) * p.nK + kt] = cls;
        }
    }
}

// One thread per tile, any strides, any tile shape.
__global__ __launch_bounds__(256) void classify_generic_kernel(const ClassifyParams p) {
    const int64_t total = (int64_t)p.uB * p.uH * p.nQ * p.nK;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= total) return;
    const int kt = (int)(t % p.nK);
    const int qt = (int)((t / p.nK) % p.nQ);
    const int plane = (int)(t / ((int64_t)p.nK * p.nQ));
    const int ub = plane / p.uH, uh = plane - ub * p.uH;
    const uint8_t *base = p.mask + (int64_t)ub * p.sb + (int64_t)uh * p.sh + (int64_t)qt * p.BQ * p.sq +
                          (int64_t)kt * p.BK * p.sk;
    int64_t count = 0;
    for (int r = 0; r < p.BQ; r++) {
        const uint8_t *row = base + (int64_t)r * p.sq;
        for (int c = 0; c < p.BK; c++) count += row[(int64_t)c * p.sk] != 0;
    }
    p.cls[t] = count == (int64_t)p.BQ * p.BK ? 2 : (count > 0 ? 1 : 0);
}

// One wave per (b, h, Q tile) row of the outputs; 4 rows per workgroup.
__global__ __launch_bounds__(256) void compact_kernel(const CompactParams p) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= (int64_t)p.oB * p.oH * p.nQ) return;
    const int qt = (int)(row % p.nQ);
    const int h = (int)((row / p.nQ) % p.oH);
    const int b = (int)(row / ((int64_t)p.nQ * p.oH));
    const int ub = p.bcast_b ? 0 : b, uh = p.bcast_h ? 0 : h;
    const uint8_t *cls = p.cls + (((int64_t)ub * p.uH + uh) * p.nQ + qt) * p.nK;
    int32_t *fid = p.full_ids + b * p.fis[0] + h * p.fis[1] + qt * p.fis[2];
    int32_t *pid = p.part_ids + b * p.pis[0] + h * p.pis[1] + qt * p.pis[2];
    const unsigned long long below = (1ull << lane) - 1ull;
    int nf = 0, np = 0;
    for (int k0 = 0; k0 < p.nK; k0 += 64) {
        const int kt = k0 + lane;
        const int c = kt < p.nK ? cls[kt] : 0;
        const unsigned long long bf = __ballot(c == 2);
        const unsigned long long bp = __ballot(c == 1);
        if (c == 2) fid[(int64_t)(nf + __popcll(bf & below)) * p.fis[3]] = kt;
        if (c == 1) pid[(int64_t)(np + __popcll(bp & below)) * p.pis[3]] = kt;
        nf += __popcll(bf);
        np += __popcll(bp);
    }
    if (lane == 0) {
        p.full_lens[b * p.fls[0] + h * p.fls[1] + qt * p.fls[2]] = nf;
        p.part_lens[b * p.pls[0] + h * p.pls[1] + qt * p.pls[2]] = np;
    }
}

// grid (slot lanes, nQ, distinct planes), 256 threads.  Workgroup x takes a run of consecutive PARTIAL slots of its Q
// tile, at least four: neighbouring tiles share the 128-byte lines of the mask rows (four tiles of 32 keys per line),
// and the workgroups of one Q tile run on different XCDs, each with an L2 of its own.  A thread makes one output
// byte at a time from 8 neighbouring mask entries of one row.
// The lists may be a caller's own: the count is clamped to the nK slots a Q tile has in `packed`, and a slot whose
// index lies outside [0, nK) is left untouched, so neither the reads of the mask nor the writes of `packed` leave
// their tensors whatever the lists hold.
__global__ __launch_bounds__(256) void pack_partial_kernel(const PackParams p) {
    const int qt = blockIdx.y;
    const int plane = blockIdx.z;
    const int ub = plane / p.uH, uh = plane - ub * p.uH;
    const int len = min(max(p.part_lens[ub * p.pls[0] + uh * p.pls[1] + qt * p.pls[2]], 0), p.nK);
    const int32_t *ids = p.part_ids + ub * p.pis[0] + uh * p.pis[1] + qt * p.pis[2];
    const int bpr = p.BK >> 3;                 // output bytes per tile row
    const int tile_bytes = p.BQ * bpr;
    const uint8_t *rows = p.mask + (int64_t)ub * p.sb + (int64_t)uh * p.sh + (int64_t)qt * p.BQ * p.sq;
    uint8_t *out_q = p.packed + (int64_t)ub * p.ob + (int64_t)uh * p.oh + (int64_t)qt * p.nK * tile_bytes;
    const int per = max(4, (len + (int)gridDim.x - 1) / (int)gridDim.x);
    const int slot_end = min(len, ((int)blockIdx.x + 1) * per);
    for (int slot = blockIdx.x * per; slot < slot_end; slot++) {
        const int id = ids[(int64_t)slot * p.pis[3]];
        if ((unsigned)id >= (unsigned)p.nK) continue;  // (uniform over the workgroup)
        const int64_t col0 = (int64_t)id * p.BK;
        uint8_t *out = out_q + (int64_t)slot * tile_bytes;
        for (int o = threadIdx.x; o < tile_bytes; o += 256) {
            const int r = o / bpr, cb = o - r * bpr;
            const uint8_t *src = rows + (int64_t)r * p.sq + (col0 + 8 * cb) * p.sk;
            uint32_t lo, hi;
            if (p.vec8) {
                const uint2 w = *(const uint2 *)src;
                lo = w.x;
                hi = w.y;
            } else {
                lo = hi = 0u;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    lo |= (uint32_t)src[(int64_t)i * p.sk] << (8 * i);
                    hi |= (uint32_t)src[(int64_t)(4 + i) * p.sk] << (8 * i);
                }
            }
            // 0x80 per non-zero byte -> one bit per byte, entry i of the group in bit i
            const uint32_t a = nonzero_bytes(lo) >> 7, b = nonzero_bytes(hi) >> 7;
            // (bits 0, 8, 16, 24 times 2^21 + 2^14 + 2^7 + 1 meet in bits 21..24, without carries)
            const uint32_t nib_lo = ((a * 0x00204081u) >> 21) & 0xfu, nib_hi = ((b * 0x00204081u) >> 21) & 0xfu;
            out[o] = (uint8_t)(nib_lo | (nib_hi << 4));
        }
    }
}

// The three steps above in one launch, a launch's latency each for masks of few bytes per Q tile: grid (nQ, distinct planes),
// a workgroup of eight waves (SLAB: sixteen) makes everything of one Q tile and the tiles' states stay in LDS.
//   rows     16 bytes per lane and row, as classify_wide_kernel; column blocks of 64 lanes are dealt to the waves, and where
//            there are fewer than eight of them the rows of one are shared by several waves.  Rows of 16, 32 .. 512 bytes
//            go several to a wave instruction.
//   lists    wave 0 writes the FULL list, wave 1 the PARTIAL one, wave 2 + 3 the next output plane's ...
//   packing  16 mask bytes (just read and in L2, in the form for small slabs) become 16 bits per thread and step.
// SLAB is the form for slabs of megabytes, bound by HBM: sixteen waves, each with two column blocks side by side and eight rows of
// both in flight, so that a workgroup has up to 256 KiB requested and reads its slab from front to back, by streaming loads.  1 GiB
// of a window's mask with lists and packed tiles 190 -> 166 us (6.5 TB/s), all PARTIAL 816 -> 434 us: PARTIAL tiles are read a second
// time, when the whole slab has been read, from beyond the L2s (a slab is as large as one, and some 32 workgroups share it).
constexpr int kRowsTiles = 2048;           // KV tiles of a Q tile that LDS holds
constexpr int64_t kSmallSlab = 512 * 1024;  // mask bytes of a Q tile past which it is the SLAB form
template <bool SLAB>
__global__ __launch_bounds__(SLAB ? 1024 : 512) void classify_rows_kernel(const ClassifyRowsParams a) {
    constexpr int kRowsThreads = SLAB ? 1024 : 512, kRowsWaves = kRowsThreads / 64;
    __shared__ unsigned state[kRowsTiles];  // bit 0: some entry attends, bit 1: some entry does not
    __shared__ uint16_t part[kRowsTiles];   // the PARTIAL tiles, in order
    __shared__ int sh_np;
    const ClassifyParams &p = a.c;
    const CompactParams &l = a.l;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int qt = blockIdx.x, plane = blockIdx.y;
    const int ub = plane / p.uH, uh = plane - ub * p.uH;
    const uint8_t *rows = p.mask + (int64_t)ub * p.sb + (int64_t)uh * p.sh + (int64_t)qt * p.BQ * p.sq;
    for (int i = tid; i < p.nK; i += kRowsThreads) state[i] = 0u;
    __syncthreads();
    if constexpr (SLAB) {
        const int pieces = p.Sk >> 4, blocks = (pieces + 63) >> 6;
        for (int cb = wave; cb < blocks; cb += 2 * kRowsWaves) {
            // (a lane without a piece of its own, or a wave without a second block, reads the row's last one again)
            const int piece[2] = {cb * 64 + lane, (cb + kRowsWaves) * 64 + lane};
            const uint8_t *const base[2] = {rows + 16 * min(piece[0], pieces - 1), rows + 16 * min(piece[1], pieces - 1)};
            uint32_t any[2] = {0u, 0u}, all[2] = {0x80808080u, 0x80808080u};
            const bool two = cb + kRowsWaves < blocks;
            auto fold = [&](int i, const u32x4 &v) {
                any[i] |= v.x | v.y | v.z | v.w;
                all[i] &= nonzero_bytes(v.x) & nonzero_bytes(v.y) & nonzero_bytes(v.z) & nonzero_bytes(v.w);
            };
            int r = 0;
            for (; r + kRowUnroll <= p.BQ; r += kRowUnroll) {
                u32x4 v[2][kRowUnroll];
#pragma unroll
                for (int u = 0; u < kRowUnroll; u++) {
                    v[0][u] = __builtin_nontemporal_load((const u32x4 *)(base[0] + (int64_t)(r + u) * p.sq));
                    if (two) v[1][u] = __builtin_nontemporal_load((const u32x4 *)(base[1] + (int64_t)(r + u) * p.sq));
                }
#pragma unroll
                for (int u = 0; u < kRowUnroll; u++) {
                    fold(0, v[0][u]);
                    if (two) fold(1, v[1][u]);
                }
            }
            for (; r < p.BQ; r++) {
                fold(0, __builtin_nontemporal_load((const u32x4 *)(base[0] + (int64_t)r * p.sq)));
                if (two) fold(1, __builtin_nontemporal_load((const u32x4 *)(base[1] + (int64_t)r * p.sq)));
            }
#pragma unroll
            for (int i = 0; i < 2; i++)
                if (piece[i] < pieces) atomicOr(&state[(16 * piece[i]) >> p.lbk], (any[i] != 0u ? 1u : 0u) | (all[i] != 0x80808080u ? 2u : 0u));
        }
    } else {
        const int pieces = p.Sk >> 4;  // 16-byte pieces of a row
        const int per_row = pieces < 64 && (pieces & (pieces - 1)) == 0 ? pieces : 64;
        const int rpi = 64 / per_row, sub = lane / per_row;  // rows of one wave instruction, and this lane's
        const int blocks = (pieces + per_row - 1) / per_row;
        const int groups = min(blocks, kRowsWaves), share = kRowsWaves / groups;  // waves that share a column block
        if (wave < groups * share) {
            const int step = share * rpi;
            for (int cb = wave / share; cb < blocks; cb += groups) {
                const int piece = cb * per_row + lane % per_row;
                if (piece >= pieces) continue;
                const uint8_t *base = rows + 16 * piece;
                uint32_t any = 0u, all = 0x80808080u;
                int r = (wave % share) * rpi + sub;
                const bool mine = r < p.BQ;
                for (; r + step * (kRowUnroll - 1) < p.BQ; r += step * kRowUnroll) {
                    u32x4 v[kRowUnroll];
#pragma unroll
                    for (int u = 0; u < kRowUnroll; u++) v[u] = *(const u32x4 *)(base + (int64_t)(r + step * u) * p.sq);
#pragma unroll
                    for (int u = 0; u < kRowUnroll; u++) {
                        any |= v[u].x | v[u].y | v[u].z | v[u].w;
                        all &= nonzero_bytes(v[u].x) & nonzero_bytes(v[u].y) & nonzero_bytes(v[u].z) & nonzero_bytes(v[u].w);
                    }
                }
                for (; r < p.BQ; r += step) {
                    const u32x4 v = *(const u32x4 *)(base + (int64_t)r * p.sq);
                    any |= v.x | v.y | v.z | v.w;
                    all &= nonzero_bytes(v.x) & nonzero_bytes(v.y) & nonzero_bytes(v.z) & nonzero_bytes(v.w);
                }
                if (mine) atomicOr(&state[(16 * piece) >> p.lbk], (any != 0u ? 1u : 0u) | (all != 0x80808080u ? 2u : 0u));
            }
        }
    }
    __syncthreads();
    // even waves the FULL list, odd ones the PARTIAL list, of every (kRowsWaves / 2)-th output plane each
    {
        const int nb = l.bcast_b ? l.oB : 1, nh = l.bcast_h ? l.oH : 1;
        const unsigned want = (wave & 1) ? 3u : 1u;
        const unsigned long long below = (1ull << lane) - 1ull;
        for (int pl = wave >> 1; pl < nb * nh; pl += kRowsWaves / 2) {
            const int b = l.bcast_b ? pl / nh : ub, h = l.bcast_h ? pl % nh : uh;
            int32_t *ids = (wave & 1) ? l.part_ids + b * l.pis[0] + h * l.pis[1] + qt * l.pis[2] : l.full_ids + b * l.fis[0] + h * l.fis[1] + qt * l.fis[2];
            const int64_t step = (wave & 1) ? l.pis[3] : l.fis[3];
            int found = 0;
            for (int k0 = 0; k0 < p.nK; k0 += 64) {
                const bool is = k0 + lane < p.nK && state[k0 + lane] == want;
                const unsigned long long bits = __ballot(is);
                const int at = found + __popcll(bits & below);
                if (is) ids[(int64_t)at * step] = k0 + lane;
                if (is && wave == 1 && pl == 0) part[at] = (uint16_t)(k0 + lane);
                found += __popcll(bits);
            }
            if (lane == 0) {
                if (wave & 1) l.part_lens[b * l.pls[0] + h * l.pls[1] + qt * l.pls[2]] = found;
                else l.full_lens[b * l.fls[0] + h * l.fls[1] + qt * l.fls[2]] = found;
                if (wave == 1 && pl == 0) sh_np = found;
            }
        }
    }
    if (a.packed == nullptr) return;
    __syncthreads();
    const int per_tile = p.BQ << (p.lbk - 4);  // 16-byte pieces of a tile
    const int64_t total = (int64_t)sh_np * per_tile;
    uint16_t *out = (uint16_t *)(a.packed + (int64_t)ub * a.ob + (int64_t)uh * a.oh + (int64_t)qt * p.nK * per_tile * 2);
    for (int64_t i = tid; i < total; i += kRowsThreads) {
        const int slot = (int)i / per_tile, w = (int)i - slot * per_tile;
        const int r = w >> (p.lbk - 4), c = w & ((1 << (p.lbk - 4)) - 1);
        const u32x4 v = *(const u32x4 *)(rows + (int64_t)r * p.sq + (int64_t)part[slot] * p.BK + 16 * c);
        unsigned bits = 0u;
#pragma unroll
        for (int e = 0; e < 4; e++) bits |= ((((nonzero_bytes(v[e]) >> 7) * 0x00204081u) >> 21) & 0xfu) << (4 * e);
        out[i] = (uint16_t)bits;
    }
}

// One wave per (b, h, Q tile) row of the lists: bit 0 of *flag when a count is negative or the two counts exceed nK,
// bit 1 when a FULL index inside its count lies outside [0, nK), bit 2 the same for a PARTIAL index.
__global__ __launch_bounds__(256) void validate_lists_kernel(const ValidateParams p) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= (int64_t)p.B * p.H * p.nQ) return;
    const int qt = (int)(row % p.nQ);
    const int h = (int)((row / p.nQ) % p.H);
    const int b = (int)(row / ((int64_t)p.nQ * p.H));
    const int nf = p.full_lens[b * p.fls[0] + h * p.fls[1] + qt * p.fls[2]];
    const int np = p.part_lens[b * p.pls[0] + h * p.pls[1] + qt * p.pls[2]];
    int bad = (nf < 0 || np < 0 || (int64_t)nf + np > p.nK) ? 1 : 0;
    const int32_t *fid = p.full_ids + b * p.fis[0] + h * p.fis[1] + qt * p.fis[2];
    const int32_t *pid = p.part_ids + b * p.pis[0] + h * p.pis[1] + qt * p.pis[2];
    const int cf = nf < 0 ? 0 : (nf > p.nK ? p.nK : nf), cp = np < 0 ? 0 : (np > p.nK ? p.nK : np);  // slots that exist
    for (int e = lane; e < cf; e += 64)
        if ((unsigned)fid[(int64_t)e * p.fis[3]] >= (unsigned)p.nK) bad |= 2;
    for (int e = lane; e < cp; e += 64)
        if ((unsigned)pid[(int64_t)e * p.pis[3]] >= (unsigned)p.nK) bad |= 4;
    if (bad) atomicOr(p.flag, bad);
}

}  // namespace

hipError_t launch_validate(const ValidateParams &p, hipStream_t stream) {
    const int64_t rows = (int64_t)p.B * p.H * p.nQ;
    hipLaunchKernelGGL(validate_lists_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, stream, p);
    return hipGetLastError();
}

hipError_t launch_pack(const PackParams &p, hipStream_t stream) {
    const int lanes = p.nK < 8 ? p.nK : 8;
    hipLaunchKernelGGL(pack_partial_kernel, dim3(lanes, p.nQ, p.uB * p.uH), dim3(256), 0, stream, p);
    return hipGetLastError();
}

// One workgroup reads a Q tile's whole slab of the mask, so the slab must be small, or there must be many of them.  us for
// lists and packed tiles, three launches | one (launches back to back in a graph):
//   slab 2 KiB x 4 workgroups (decode, four lengths)  6.2 | 4.0    32 KiB x 8 (Sk 32768)      7.4 | 5.4
//   128 KiB x 8 (causal S1024)                        9.4 | 5.7    128 KiB x 8, all PARTIAL  12.1 | 9.6
//   512 KiB x 128 (causal S8192)                     19.0 | 13.5   512 KiB x 256, all PARTIAL 97 | 51
//   256 KiB x 64, all PARTIAL                        17.7 | 15.9   256 KiB x 512, all PARTIAL 76 | 42
// and beyond the rule 256 KiB x 16 causal 9.8 | 6.9 but all PARTIAL 12.5 | 15.6, 2 MiB x 4 10.3 | 23.5.
// Larger slabs (the SLAB form).  A compute unit runs one workgroup, so a launch takes rounds of 256, and one that is hardly begun costs as
// much as a full one; a wave takes 1024 columns, so rows must be long enough for half of the sixteen waves.  Lists alone:
//   1 MiB (128 x 8192)  x 192 35.5 | 30.3   x 256 46.0 | 40.5   x 272 49.7 | 58.8   x 320 57.1 | 62.1   x 384 67.6 | 65.7   x 768 128.7 | 120.6
//   2 MiB (128 x 16384) x 192 76.2 | 63.8   x 257 100 | 113     x 320 121 | 125     x 384 143 | 132
//   4 MiB (128 x 32768) x 192 136 | 148     x 240 168 | 172     x 256 182 | 169     and packed: causal 196 | 171, all PARTIAL 833 | 432
//   64 rows: 1 MiB x 512 84.1 | 86.3        2 MiB x 300 112 | 127   x 512 182 | 170     4 MiB x 192 135 | 147   x 256 169 | 167
// Half a round reads as fast as three launches read a mask from the memory-side cache (256 MiB), and saves two of them:
//   1 MiB x 128 24.9 | 25.5, packed, causal 31.4 | 26.2   2 MiB x 128 54.0 | 52.4, packed 62.1 | 52.9   4 MiB x 128 93.3 | 97.4
// (with lists of 32 planes each its own, which three launches spread over the device, 2 MiB x 128 55.2 | 58.0).  Packed tiles of 64 Ki entries
// and more: a Q tile has few PARTIAL ones, and each is one workgroup's in the packing launch, so the one launch is always the faster one where
// there are some: 256 x 1024 tiles of 32768 keys x 128, causal 255 | 190, window 334 | 209, of 16384 keys x 300, causal 408 | 265; where there
// are none, or all are, up to 13 % slower (176 | 184, 538 | 562; 207 | 234).
bool classify_rows_has(const ClassifyParams &p, int copies, bool packing) {
    const int64_t slab = (int64_t)p.BQ * p.Sk, workgroups = (int64_t)p.nQ * p.uB * p.uH;
    if (p.nK > kRowsTiles) return false;
    if (slab <= kSmallSlab) return slab <= 128 * 1024 || slab <= workgroups * 8192;
    if (slab > INT32_MAX || p.Sk < 8 * kWideCols || workgroups < 128) return false;
    constexpr int64_t kMiB = 1 << 20;
    const int64_t slots = (workgroups + 255) / 256 * 256;  // of the rounds the launch takes
    if (packing && p.BQ * p.BK >= 64 * 1024) return true;
    if (slab >= 4 * kMiB) return workgroups >= 256 && 10 * workgroups >= 9 * slots;
    if (p.BQ < 128) return slab >= 2 * kMiB && 10 * workgroups >= 9 * slots;
    if (workgroups >= 192) return 4 * workgroups >= 3 * slots;
    return copies <= 8 && (slab <= kMiB ? packing : slab <= 2 * kMiB && workgroups * slab >= 256 * kMiB);
}

hipError_t launch_classify_rows(const ClassifyRowsParams &p, hipStream_t stream) {
    const dim3 grid(p.c.nQ, p.c.uB * p.c.uH);
    if ((int64_t)p.c.BQ * p.c.Sk > kSmallSlab) hipLaunchKernelGGL(classify_rows_kernel<true>, grid, dim3(1024), 0, stream, p);
    else hipLaunchKernelGGL(classify_rows_kernel<false>, grid, dim3(512), 0, stream, p);
    return hipGetLastError();
}

hipError_t launch_classify(const ClassifyParams &p, bool wide, hipStream_t stream) {
    if (wide) {
        const dim3 grid((p.Sk + kWideCols - 1) / kWideCols, p.nQ, p.uB * p.uH);
        hipLaunchKernelGGL(classify_wide_kernel, grid, dim3(256), 0, stream, p);
    } else {
        const int64_t total = (int64_t)p.uB * p.uH * p.nQ * p.nK;
        hipLaunchKernelGGL(classify_generic_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, p);
    }
    return hipGetLastError();
}

hipError_t launch_compact(const CompactParams &p, hipStream_t stream) {
    const int64_t rows = (int64_t)p.oB * p.oH * p.nQ;
    hipLaunchKernelGGL(compact_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, stream, p);
    return hipGetLastError();
}

}  // namespace sa
